// Per-(kz, kx) profile network for the plane Couette corrector guess:
// training and inference on the matrix cores (bf16 operands, FP32
// accumulation, v_mfma_f32_16x16x16_bf16), no reference counterpart.
//
// One sample is one Fourier mode (kz, kx) at one step.  Its input is the
// wall-normal profile of the first and second differences of the nonlinear
// term, D1 = N^n - N^{n-1} and D2 = N^n - 2 N^{n-1} + N^{n-2} (3 components,
// real and imaginary parts, Ny points each: 12 Ny values, each difference
// scaled by its RMS), then dt k^2 / Re, kx / k_max and kz / k_max, zero
// padded to `din` (a multiple of 32).  Its output is the profile of the
// residual of quadratic extrapolation, N(u*) - (3 N^n - 3 N^{n-1} + N^{n-2})
// (6 Ny values) scaled by w = 1 / (1 + c dt k^2 / Re) and 1 / s_out: the
// corrector's fixed point u* = S(u^n; N(u*)) is the converged state of the
// step, so N(u*) = N^{n+1} and the training pairs come from the solver's own
// history.  Network: din -> H -> H -> dout, SiLU, weights FP32 (Adam) and
// bf16 copies for the matrix cores.
//
// Every layer, forward and backward, is one bf16 GEMM (pn_tile) with a fused
// epilogue: bias + pre-activation store + SiLU (forward), the loss and its
// gradient (output layer), or the SiLU derivative (backward); the weight and
// bias gradients are GEMMs over the batch.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "context.hpp"
#include "dft.hpp"

namespace dnsmi {

typedef short pv4s __attribute__((ext_vector_type(4)));
typedef float pv4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t pn_bf16(float f) {
  const uint32_t u = __float_as_uint(f);
  return (uint16_t)((u + (((u >> 16) & 1u) + 0x7FFFu)) >> 16);
}
__device__ __forceinline__ float pn_silu(float z) { return z / (1.0f + __expf(-z)); }
__device__ __forceinline__ float pn_dsilu(float z) {
  const float s = 1.0f / (1.0f + __expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

// ------------------------------------------------------------------ GEMM
// C (M x N) = op(A) (M x K) op(B) (K x N), bf16 operands, FP32 accumulation.
// An operand is stored either with k contiguous (AK: A[m lda + k], BK:
// B[n ldb + k]) or with k strided (A[k lda + m], B[k ldb + n]).  Epilogue on
// v = acc (+ bias[n]):
//   EPI_LINEAR  C = v
//   EPI_SILU    C = v (the pre-activation, if C is given), Cb = bf16(silu(v))
//   EPI_DSILU   Cb = bf16(acc * silu'(Z[m][n])) (no bias)
//   EPI_LOSS    d = v - Z[m][n]: Cb = bf16(2 d scale), and the tile's sum of
//               d^2 into lossp[tile]
//   EPI_PART    C = acc for one of `splits` ranges of K (each C_split apart
//               of the next), and as row M the column sums of op(B): the
//               weight gradients and, below them, the bias gradients
//
// A workgroup of four waves takes a BM x BN tile, K in chunks of 64 through
// two LDS buffers, each chunk's global loads issued two chunks ahead into
// registers: at the layers' sizes (K = 256 .. 3104, one tile per CU) the loop
// is bound by the latency of those loads, not by the matrix cores.  The
// 16 x 16 x 16 products of one output are accumulated in ascending k in every
// tile shape, so an output does not depend on the tile (or the batch) it is
// computed in; only EPI_PART splits K.
//
// LDS: row r of an operand holds its 64 k as eight 16-byte slots; slot
// 4 h + g is what lane group g (lane / 16) feeds to two successive products,
// k = 32 h + 4 g .. + 3 and 32 h + 16 + 4 g .. + 3, so one 16-byte read serves
// both.  Rows and their slots are permuted (pn_at) so that the 16 rows of a
// product, and the rows that a strided operand's four-k groups scatter to,
// spread over all 64 banks.  Measured at 2048 x 3104 -> 256: 18 us against 182
// us for element-wise loads through one buffer.
enum { EPI_LINEAR = 0, EPI_SILU = 1, EPI_DSILU = 2, EPI_LOSS = 3, EPI_PART = 4 };

struct GemmArgs {
  int M, N, K;
  const uint16_t* A;
  int lda;
  const uint16_t* B;
  int ldb;
  float* C;
  int ldc;
  uint16_t* Cb;
  int ldcb;
  const float* bias;
  const float* Z;
  int ldz;
  float scale;
  float* lossp;
  int splits;
  long long C_split;
};

constexpr int kPnK = 64;  // k per LDS chunk

// LDS word of 16-byte slot `slot` of row `row`.
__device__ __forceinline__ int pn_at(int row, int slot) {
  return (row ^ (((row >> 2) ^ (row >> 3)) & 1)) * kPnK + 8 * (slot ^ (((row >> 1) ^ (row >> 4)) & 7));
}

// Operand rows [r0, r0 + R) of chunk [k0, k0 + 64) into registers.  Thread
// layout: k contiguous, 16-byte pieces, eight threads to a row; k strided,
// 4 k x R / 16 rows, 16 threads along the rows.
//
// A chunk whose elements all exist: from the chunk's first element (uniform)
// at a thread's fixed byte offsets, with no branch or select that would wait
// for the loads, and no alignment of their own (memcpy: an unaligned global
// load is one instruction on gfx950).  Rows past the matrix read its last
// row (k contiguous): their outputs are not stored.
template <int R, int T>
__device__ __forceinline__ int pn_strided_row(int tid) { return R * 16 / T * (tid % (T / 16)); }
template <int T>
__device__ __forceinline__ int pn_strided_k(int tid) {
  return T == 256 ? 4 * ((tid >> 6) + 4 * ((tid >> 4) & 3))
                  : 4 * (((tid >> 6) & 3) + 8 * (tid >> 8) + 4 * ((tid >> 5) & 1));
}
template <int R, bool KC, int T>
struct PnOffsets {
  static constexpr int n = KC ? R * 8 / T : 4;
  uint32_t at[n];
  __device__ __forceinline__ PnOffsets(int ld, int r0, int rows, int tid) {
#pragma unroll
    for (int i = 0; i < n; ++i) {
      if constexpr (KC)
        at[i] = 2u * ((uint32_t)min(i * (T / 8) + (tid >> 3), rows - 1 - r0) * ld + 8 * (tid & 7));
      else
        at[i] = 2u * ((uint32_t)(pn_strided_k<T>(tid) + i) * ld + pn_strided_row<R, T>(tid));
    }
  }
};
template <int R, bool KC, int T>
__device__ __forceinline__ void pn_load(uint32_t (&v)[R * 32 / T], const uint16_t* __restrict__ p, int ld, int r0,
                                        int k0, const PnOffsets<R, KC, T>& o) {
  const char* base = reinterpret_cast<const char*>(p + (KC ? (size_t)r0 * ld + k0 : (size_t)k0 * ld + r0));
  constexpr int n = PnOffsets<R, KC, T>::n, W = R * 32 / T / n;
#pragma unroll
  for (int i = 0; i < n; ++i) __builtin_memcpy(&v[i * W], base + o.at[i], 4 * W);
}

// Any chunk, element by element: zero for k >= kend, the last row's values
// past the rows.
template <int R, bool KC, int T>
__device__ __forceinline__ void pn_load_edge(uint32_t (&v)[R * 32 / T], const uint16_t* __restrict__ p, int ld, int r0,
                                             int rows, int k0, int kend, int tid) {
  if constexpr (KC) {
    const int k = k0 + 8 * (tid & 7);
#pragma unroll
    for (int i = 0; i < R * 8 / T; ++i) {
      const uint16_t* q = p + (size_t)min(r0 + i * (T / 8) + (tid >> 3), rows - 1) * ld;
      uint16_t h[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) h[e] = q[min(k + e, kend - 1)];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[4 * i + e] = (k + 2 * e < kend ? h[2 * e] : 0u) | (uint32_t)(k + 2 * e + 1 < kend ? h[2 * e + 1] : 0u) << 16;
    }
  } else {
    constexpr int NB = R * 16 / T;
    const int r = r0 + pn_strided_row<R, T>(tid);
    const int k = k0 + pn_strided_k<T>(tid);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint16_t* q = p + (size_t)min(k + e, kend - 1) * ld;
      uint16_t h[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i) h[i] = q[min(r + i, rows - 1)];
#pragma unroll
      for (int i = 0; i < NB / 2; ++i)
        v[e * (NB / 2) + i] = k + e < kend ? h[2 * i] | (uint32_t)h[2 * i + 1] << 16 : 0u;
    }
  }
}

template <int R, bool KC, int T>
__device__ __forceinline__ void pn_store(const uint32_t (&v)[R * 32 / T], uint16_t* __restrict__ lds, int tid) {
  if constexpr (KC) {
    const int h = tid & 7, slot = 4 * (h >> 2) + 2 * (h & 1), half = (h & 3) >> 1;
#pragma unroll
    for (int i = 0; i < R * 8 / T; ++i) {
      const int r = i * (T / 8) + (tid >> 3);
      *reinterpret_cast<uint2*>(lds + pn_at(r, slot) + 4 * half) = uint2{v[4 * i], v[4 * i + 1]};
      *reinterpret_cast<uint2*>(lds + pn_at(r, slot + 1) + 4 * half) =
          uint2{v[4 * i + 2], v[4 * i + 3]};
    }
  } else {
    constexpr int NB = R * 16 / T;
    const int kb = pn_strided_k<T>(tid) / 4;
    const int slot = 4 * (kb >> 3) + (kb & 3), half = (kb >> 2) & 1;
#pragma unroll
    for (int e = 0; e < NB; ++e) {
      const int r = pn_strided_row<R, T>(tid) + e;
      const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;  // the odd or even halves of two rows
      const uint32_t lo = __builtin_amdgcn_perm(v[1 * (NB / 2) + e / 2], v[e / 2], sel);
      const uint32_t hi = __builtin_amdgcn_perm(v[3 * (NB / 2) + e / 2], v[2 * (NB / 2) + e / 2], sel);
      *reinterpret_cast<uint2*>(lds + pn_at(r, slot) + 4 * half) = uint2{lo, hi};
    }
  }
}

// Two successive 16 x 16 x 16 operands of one lane.
union PnFrag {
  uint4 q;
  pv4s s[2];
};

// Tile t of the product (n fastest), or, EPI_PART, part t / tiles of tile
// t % tiles.  smem: 2 (BM + BN) 64 bf16 words.
template <int BM, int BN, bool AK, bool BK, int EPI, int T, int S>
__device__ __forceinline__ void pn_tile(const GemmArgs& g, int t, uint16_t* __restrict__ smem) {
  constexpr int WN = T / 128;                     // 2 x WN waves
  constexpr int TM = BM / 32, TN = BN / 16 / WN;  // 16 x 16 products per wave
  const int nt = (g.N + BN - 1) / BN;
  int k0 = 0, kend = g.K, part = 0;
  if constexpr (EPI == EPI_PART) {
    const int tiles = nt * ((g.M + BM - 1) / BM);
    part = t / tiles;
    t -= part * tiles;
    const int per = ((g.K + kPnK - 1) / kPnK + g.splits - 1) / g.splits * kPnK;
    k0 = part * per;
    kend = k0 + per < g.K ? k0 + per : g.K;
  }
  // where k is strided, the last tile along the rows is moved back to lie
  // inside the matrix, and leaves what the tile before it computes too
  const int mt = t / nt * BM, ntl = (t - t / nt * nt) * BN;
  const int m0 = !AK && g.M >= BM ? min(mt, g.M - BM) : mt;
  const int n0 = !BK && g.N >= BN ? min(ntl, g.N - BN) : ntl;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, grp = lane >> 4, l16 = lane & 15;
  const int wm = wave / WN * (BM / 2), wn = wave % WN * (BN / WN);
  pv4f acc[TM][TN], cs[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    cs[j] = pv4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[i][j] = pv4f{0.f, 0.f, 0.f, 0.f};
  }
  // column sums of op(B): products with a row of ones, in the tiles of the
  // first row of waves
  const bool sums = EPI == EPI_PART && mt == 0 && wm == 0;
  const pv4s ones = {0x3F80, 0x3F80, 0x3F80, 0x3F80};
  constexpr int kBuf = (BM + BN) * kPnK;
  auto compute = [&](int buf) {
    const uint16_t* As = smem + buf * kBuf;
    const uint16_t* Bs = As + BM * kPnK;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      PnFrag a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int r = wm + i * 16 + l16;
        a[i].q = *reinterpret_cast<const uint4*>(As + pn_at(r, 4 * h + grp));
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int r = wn + j * 16 + l16;
        b[j].q = *reinterpret_cast<const uint4*>(Bs + pn_at(r, 4 * h + grp));
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i].s[s], b[j].s[s], acc[i][j], 0, 0, 0);
        if (sums) {
#pragma unroll
          for (int j = 0; j < TN; ++j)
            cs[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ones, b[j].s[s], cs[j], 0, 0, 0);
        }
      }
    }
  };
  // the chunks whose elements all exist: while chunk c is multiplied, c + 1 ..
  // c + S - 1 are in registers or on their way, and c + S is asked for (past
  // the end: the last one again)
  const bool narrow = (!AK && g.M < BM) || (!BK && g.N < BN);
  const int nk = narrow || kend <= k0 ? 0 : (kend - k0) / kPnK;
  if (nk > 0) {
    const PnOffsets<BM, AK, T> oa(g.lda, m0, g.M, tid);
    const PnOffsets<BN, BK, T> ob(g.ldb, n0, g.N, tid);
    uint32_t va[S][BM * 32 / T], vb[S][BN * 32 / T];
    auto load = [&](int c, int set) {
      const int k = k0 + min(c, nk - 1) * kPnK;
      pn_load<BM, AK, T>(va[set], g.A, g.lda, m0, k, oa);
      pn_load<BN, BK, T>(vb[set], g.B, g.ldb, n0, k, ob);
      __builtin_amdgcn_sched_barrier(0);  // else they sink behind the products that are to hide them
    };
    auto store = [&](int buf, int set) {
      pn_store<BM, AK, T>(va[set], smem + buf * kBuf, tid);
      pn_store<BN, BK, T>(vb[set], smem + buf * kBuf + BM * kPnK, tid);
    };
#pragma unroll
    for (int u = 0; u < S; ++u) load(u, u);
    store(0, 0);
    __syncthreads();
    int c = 0;
    for (; c + S < nk; c += S) {
#pragma unroll
      for (int u = 0; u < S; ++u) {
        load(c + u + S, u);
        compute(u & 1);
        store((u + 1) & 1, (u + 1) % S);
        __syncthreads();
      }
    }
#pragma unroll
    for (int u = 0; u < S; ++u)
      if (c + u < nk) {
        compute(u & 1);
        if (u + 1 < S) store((u + 1) & 1, u + 1);
        __syncthreads();
      }
  }
  // the last, partial chunk of K (of a matrix narrower than the tile: all)
  for (int k = k0 + nk * kPnK; k < kend; k += kPnK) {
    uint32_t va[BM * 32 / T], vb[BN * 32 / T];
    pn_load_edge<BM, AK, T>(va, g.A, g.lda, m0, g.M, k, kend, tid);
    pn_load_edge<BN, BK, T>(vb, g.B, g.ldb, n0, g.N, k, kend, tid);
    pn_store<BM, AK, T>(va, smem, tid);
    pn_store<BN, BK, T>(vb, smem + BM * kPnK, tid);
    __syncthreads();
    compute(0);
    __syncthreads();
  }
  // lane holds D[4 (lane / 16) + q][lane % 16] of each 16 x 16 tile
  float sq = 0.f;
  float* C = g.C;
  if constexpr (EPI == EPI_PART) C += part * g.C_split;
  // what the epilogue reads, all asked for before the first store (a load
  // behind a store would wait for it): rows and columns past the end read
  // the last one's
  float bias[TN], z[TM][TN][4];
  if constexpr (EPI == EPI_LINEAR || EPI == EPI_SILU || EPI == EPI_LOSS) {
#pragma unroll
    for (int j = 0; j < TN; ++j) bias[j] = g.bias[min(n0 + wn + j * 16 + l16, g.N - 1)];
  }
  if constexpr (EPI == EPI_DSILU || EPI == EPI_LOSS) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float* zr = g.Z + (size_t)min(m0 + wm + i * 16 + 4 * grp + q, g.M - 1) * g.ldz;
#pragma unroll
        for (int j = 0; j < TN; ++j) z[i][j][q] = zr[min(n0 + wn + j * 16 + l16, g.N - 1)];
      }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int m = m0 + wm + i * 16 + 4 * grp + q;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + wn + j * 16 + l16;
        float v = acc[i][j][q];
        [[maybe_unused]] uint16_t h = 0;
        const bool mine = m < g.M && n < g.N && m >= mt && n >= ntl;
        if constexpr (EPI == EPI_DSILU) h = pn_bf16(v * pn_dsilu(z[i][j][q]));
        if constexpr (EPI == EPI_LINEAR || EPI == EPI_SILU || EPI == EPI_LOSS) v += bias[j];
        if constexpr (EPI == EPI_SILU) h = pn_bf16(pn_silu(v));
        if constexpr (EPI == EPI_LOSS) {
          const float d = v - z[i][j][q];
          sq += mine ? d * d : 0.f;
          h = pn_bf16(2.0f * d * g.scale);
        }
        if (mine) {
          if constexpr (EPI == EPI_LINEAR || EPI == EPI_PART) C[(size_t)m * g.ldc + n] = v;
          if constexpr (EPI == EPI_SILU) {
            if (C) C[(size_t)m * g.ldc + n] = v;
          }
          if constexpr (EPI == EPI_SILU || EPI == EPI_DSILU || EPI == EPI_LOSS) g.Cb[(size_t)m * g.ldcb + n] = h;
        }
      }
    }
  if constexpr (EPI == EPI_PART) {
    if (sums && grp == 0) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + wn + j * 16 + l16;
        if (n < g.N) C[(size_t)g.M * g.ldc + n] = cs[j][0];
      }
    }
  }
  if constexpr (EPI == EPI_LOSS) {
    // fixed-order sum over the tile (LDS is free: the loop ended in a barrier)
    float* red = reinterpret_cast<float*>(smem);
    for (int o = 32; o > 0; o >>= 1) sq += __shfl_down(sq, o, 64);
    if (lane == 0) red[wave] = sq;
    __syncthreads();
    if (tid == 0) {
      float v = 0.f;
      for (int w = 0; w < T / 64; ++w) v += red[w];
      g.lossp[t] = v;
    }
  }
}

// Workgroups go to the 8 XCDs in turn; renumbered so that each XCD takes one
// contiguous range of tiles, whose shared operand rows then meet in its L2.
__device__ __forceinline__ int pn_xcd(int b, int G) {
  const int q = G / 8, r = G % 8, x = b % 8, i = b / 8;
  return x * q + (x < r ? x : r) + i;
}

template <int BM, int BN, int EPI, int T, int S>
__global__ void __launch_bounds__(T, 2) k_pn_layer(GemmArgs g) {
  __shared__ __align__(16) uint16_t smem[2 * (BM + BN) * kPnK];
  pn_tile<BM, BN, true, false, EPI, T, S>(g, pn_xcd(blockIdx.x, gridDim.x), smem);
}

// out[i] = sum over `parts` of part[q stride + i], in order.
struct SumArgs {
  const float* part;
  int parts;
  long long stride, n;
  float* out;
  float scale;
};

// One backward launch, its independent pieces side by side so that small
// ones fill the chip together: tiles of dZ = (dY W^T) silu'(Z) in the first
// nz workgroups, (tile, part)s of a weight gradient in the next nw, the sum
// of an earlier launch's parts in the next ns, and the loss in the last one.
struct BackArgs {
  GemmArgs z, w;
  SumArgs s, loss;
  int nz, nw, ns;
};
constexpr int kSumPer = 4;  // elements per thread of the sum, all in flight

template <int BN>
__global__ void __launch_bounds__(256, 2) k_pn_back(BackArgs a) {
  __shared__ __align__(16) uint16_t smem[2 * (64 + BN) * kPnK];
  int b = blockIdx.x;
  if (b < a.nz) return pn_tile<32, 64, true, true, EPI_DSILU, 256, 2>(a.z, pn_xcd(b, a.nz), smem);
  b -= a.nz;
  if (b < a.nw) return pn_tile<64, BN, false, false, EPI_PART, 256, 2>(a.w, b, smem);
  b -= a.nw;
  if (b < a.ns) {
    const long long i0 = (long long)b * kSumPer * 256 + threadIdx.x;
    float v[kSumPer] = {};
    for (int q = 0; q < a.s.parts; ++q) {
      const float* p = a.s.part + q * a.s.stride;
#pragma unroll
      for (int e = 0; e < kSumPer; ++e) v[e] += p[min(i0 + e * 256, a.s.n - 1)];
    }
#pragma unroll
    for (int e = 0; e < kSumPer; ++e)
      if (i0 + e * 256 < a.s.n) a.s.out[i0 + e * 256] = v[e];
    return;
  }
  float v = 0.f;
  for (long long i = threadIdx.x; i < a.loss.n; i += 256) v += a.loss.part[i];
  float* red = reinterpret_cast<float*>(smem);
  red[threadIdx.x] = v;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) *a.loss.out = red[0] * a.loss.scale;
}

static int pn_tiles(int M, int N, int BM, int BN) { return (int)(((long long)M + BM - 1) / BM * ((N + BN - 1) / BN)); }

// Tile of a layer: 64 x 128 (eight waves), the fewest operand bytes per
// product, where that still gives most of the 256 CUs a workgroup; else 32 x
// 64 (four).  8128 x 3104 -> 256, 254 workgroups of 64 x 128: 36 us, 64 x 64
// tiles 40 us, 64 x 128 in four waves 39 us; 2048 x 3104 -> 256: 18 us in 256
// workgroups of 32 x 64, where 64 x 128 would fill 64 CUs.
static bool pn_large(int M, int N) { return N >= 128 && pn_tiles(M, N, 64, 128) >= 208; }
static int pn_layer_tiles(int M, int N) { return pn_large(M, N) ? pn_tiles(M, N, 64, 128) : pn_tiles(M, N, 32, 64); }

// Chunks in flight (S): four where K is long (the input layer: 36 -> 34 us at
// 8128 x 3104 -> 256, 20 -> 18 at 2048), else two (the output layer, four
// chunks of K: 26 against 35 us at 8128 x 256 -> 1536, whose extra loads
// bring nothing).
template <int EPI, int S>
static void pn_layer_s(const GemmArgs& g, hipStream_t s) {
  const dim3 grid(pn_layer_tiles(g.M, g.N));
  if (pn_large(g.M, g.N))
    hipLaunchKernelGGL((k_pn_layer<64, 128, EPI, 512, S>), grid, dim3(512), 0, s, g);
  else
    hipLaunchKernelGGL((k_pn_layer<32, 64, EPI, 256, S>), grid, dim3(256), 0, s, g);
}
template <int EPI>
static int pn_layer(const GemmArgs& g, hipStream_t s) {
  if (g.K >= 1024)
    pn_layer_s<EPI, 4>(g, s);
  else
    pn_layer_s<EPI, 2>(g, s);
  return hipGetLastError() == hipSuccess ? DNSMI_OK : DNSMI_EHIP;
}

static int pn_back(const BackArgs& a, hipStream_t s) {
  const int n = a.nz + a.nw + a.ns + (a.loss.out ? 1 : 0);
  if (!n) return DNSMI_OK;
  if (a.w.N >= 128)
    hipLaunchKernelGGL(k_pn_back<128>, dim3(n), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(k_pn_back<64>, dim3(n), dim3(256), 0, s, a);
  return hipGetLastError() == hipSuccess ? DNSMI_OK : DNSMI_EHIP;
}

// ------------------------------------------------------------------ layout
// Parameters (FP32): W1 (din, H) | b1 (H) | W2 (H, H) | b2 (H) | W3 (H, dout) |
// b3 (dout), row-major.  bf16 copies of W1, W2, W3 in the same layout.
struct PNet {
  int din, H, dout;
  __host__ __device__ long long w1() const { return 0; }
  __host__ __device__ long long b1() const { return (long long)din * H; }
  __host__ __device__ long long w2() const { return b1() + H; }
  __host__ __device__ long long b2() const { return w2() + (long long)H * H; }
  __host__ __device__ long long w3() const { return b2() + H; }
  __host__ __device__ long long b3() const { return w3() + (long long)H * dout; }
  __host__ __device__ long long n() const { return b3() + dout; }
};

// bf16 copies of the parameters, four per thread.
__global__ void __launch_bounds__(256) k_pn_cast(const float* __restrict__ p, long long n, uint16_t* __restrict__ wb) {
  const long long i = 4 * ((long long)blockIdx.x * blockDim.x + threadIdx.x);
  if (i + 4 <= n) {
    float f[4];
    uint16_t h[4];
    __builtin_memcpy(f, p + i, 16);
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = pn_bf16(f[e]);
    __builtin_memcpy(wb + i, h, 8);
  } else {
    for (long long e = i; e < n; ++e) wb[e] = pn_bf16(p[e]);
  }
}

__global__ void k_pn_adam(float* __restrict__ prm, const float* __restrict__ g, float* __restrict__ m,
                          float* __restrict__ v, long long P, float lr, float c1, float c2) {
  const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  const float gi = g[p];
  const float mi = 0.9f * m[p] + 0.1f * gi;
  const float vi = 0.999f * v[p] + 0.001f * gi * gi;
  m[p] = mi;
  v[p] = vi;
  prm[p] -= lr * (mi / c1) / (sqrtf(vi / c2) + 1e-8f);
}

static bool pn_ok(const PNet& n) { return n.din > 0 && n.din % 32 == 0 && n.H > 0 && n.H % 64 == 0 && n.dout > 0; }

// The hidden layers of B samples: X (B, din) bf16 -> H1, H2 (bf16), with the
// pre-activations Z1, Z2 (FP32) where they are given (training).
static int pn_hidden(const PNet& net, int B, const uint16_t* X, const uint16_t* wb, const float* prm, float* Z1,
                     float* Z2, uint16_t* H1, uint16_t* H2, hipStream_t s) {
  GemmArgs g{};
  g.M = B;
  g.N = net.H;
  g.K = net.din;
  g.A = X;
  g.lda = net.din;
  g.B = wb + net.w1();
  g.ldb = net.H;
  g.C = Z1;
  g.ldc = net.H;
  g.Cb = H1;
  g.ldcb = net.H;
  g.bias = prm + net.b1();
  int rc = pn_layer<EPI_SILU>(g, s);
  if (rc) return rc;
  g.K = net.H;
  g.A = H1;
  g.lda = net.H;
  g.B = wb + net.w2();
  g.C = Z2;
  g.Cb = H2;
  g.bias = prm + net.b2();
  return pn_layer<EPI_SILU>(g, s);
}

// The output layer's product, up to its epilogue.
static GemmArgs pn_out(const PNet& net, int B, const uint16_t* H2, const uint16_t* wb, const float* prm) {
  GemmArgs g{};
  g.M = B;
  g.N = net.dout;
  g.K = net.H;
  g.A = H2;
  g.lda = net.H;
  g.B = wb + net.w3();
  g.ldb = net.dout;
  g.bias = prm + net.b3();
  return g;
}

static int pn_cast(const PNet& net, const float* prm, uint16_t* wb, hipStream_t s) {
  hipLaunchKernelGGL(k_pn_cast, dim3((unsigned)((net.n() + 1023) / 1024)), dim3(256), 0, s, prm, net.n(), wb);
  return hipGetLastError() == hipSuccess ? DNSMI_OK : DNSMI_EHIP;
}

int pnet_forward(int din, int H, int dout, int B, const uint16_t* X, const float* prm, uint16_t* wb, uint16_t* wh,
                 float* Y, hipStream_t s) {
  const PNet net{din, H, dout};
  if (!pn_ok(net) || B <= 0) return DNSMI_EINVAL;
  uint16_t* H1 = wh;
  uint16_t* H2 = H1 + (size_t)B * H;
  int rc = pn_cast(net, prm, wb, s);
  if (rc) return rc;
  if ((rc = pn_hidden(net, B, X, wb, prm, nullptr, nullptr, H1, H2, s))) return rc;
  GemmArgs g = pn_out(net, B, H2, wb, prm);
  g.C = Y;
  g.ldc = dout;
  return pn_layer<EPI_LINEAR>(g, s);
}

// A weight gradient G (M + 1 rows: the weights', then the bias's) = [P | 1]^T
// Q over the batch, P (B, M), Q (B, N): up to `want` workgroups by splitting
// the batch into parts of equal numbers of 64-sample chunks (the last part
// takes what is left), two chunks each at least where the batch has them, as
// far as `room` floats of scratch hold the parts (one part needs none and goes
// straight to G).
struct WGrad {
  GemmArgs g;
  int blocks;
  SumArgs sum;
  int sum_blocks;
  long long used;  // floats of scratch
};

static WGrad pn_wgrad(int M, int N, int B, const uint16_t* P, const uint16_t* Q, float* G, float* scratch,
                      long long room, int want) {
  WGrad r{};
  // 128 columns a tile only where the matrix has them: a narrower one is loaded
  // element by element throughout (pn_tile).  Gradient of 8128 samples, 256 ->
  // 126 outputs: 121 us in tiles of 128, 103 us of 64.
  const int tiles = pn_tiles(M, N, 64, N >= 128 ? 128 : 64);
  const long long n = (long long)(M + 1) * N;
  long long parts = want / tiles;
  if (parts > (B + 127) / 128) parts = (B + 127) / 128;
  if (parts > room / n) parts = room / n;
  if (parts < 1) parts = 1;
  // the chunks of a part rounded up leave the last parts none: as many parts
  // as have some (pn_tile divides the batch the same way)
  const long long chunks = ((long long)B + kPnK - 1) / kPnK, per = (chunks + parts - 1) / parts;
  parts = (chunks + per - 1) / per;
  r.g.M = M;
  r.g.N = N;
  r.g.K = B;
  r.g.A = P;
  r.g.lda = M;
  r.g.B = Q;
  r.g.ldb = N;
  r.g.ldc = N;
  r.g.splits = (int)parts;
  r.g.C = parts > 1 ? scratch : G;
  r.g.C_split = n;
  r.blocks = tiles * (int)parts;
  if (parts > 1) {
    r.sum = {scratch, (int)parts, n, n, G, 1.0f};
    r.sum_blocks = (int)((n + 256 * kSumPer - 1) / (256 * kSumPer));
    r.used = parts * n;
  }
  return r;
}

// dZ = (dQ W^T) silu'(Z), dQ (B, K), W (N, K) row-major.
static GemmArgs pn_dz(int B, int N, int K, const uint16_t* dQ, const uint16_t* W, const float* Z, uint16_t* dZ) {
  GemmArgs g{};
  g.M = B;
  g.N = N;
  g.K = K;
  g.A = dQ;
  g.lda = K;
  g.B = W;
  g.ldb = K;
  g.Cb = dZ;
  g.ldcb = N;
  g.Z = Z;
  g.ldz = N;
  return g;
}

// Gradient of L = (1/(B dout)) sum (Y - T)^2 into grad (FP32), loss into
// *loss (may be null).  Eight launches: the cast, three layers (the last one
// forms dY and the loss in its epilogue; Y itself is never stored), then
//   dZ2, parts of dW3 | dZ1, parts of dW2, sum of dW3, loss | parts of dW1,
//   sum of dW2 | sum of dW1
// each bias gradient in its weights' launch.  The parts live where the B x
// dout outputs would (wf): dW3's and dW1's at its start, dW2's behind them,
// the loss's at its end.
// 2048 x (3104 -> 256 -> 256 -> 1536): 73 us, against 3670 us with one GEMM,
// column sum (one thread per column) or loss sum (one thread) per launch and
// the batch never split.
int pnet_grad(int din, int H, int dout, int B, const uint16_t* X, const float* T, const float* prm,
              uint16_t* wb, float* wf, uint16_t* wh, float* grad, float* loss, hipStream_t s) {
  const PNet net{din, H, dout};
  if (!pn_ok(net) || B <= 0) return DNSMI_EINVAL;
  float* Z1 = wf;
  float* Z2 = Z1 + (size_t)B * H;
  float* scratch = Z2 + (size_t)B * H;
  uint16_t* H1 = wh;
  uint16_t* H2 = H1 + (size_t)B * H;
  uint16_t* dZ = H2 + (size_t)B * H;
  uint16_t* dY = dZ + (size_t)B * H;
  int rc = pn_cast(net, prm, wb, s);
  if (rc) return rc;
  if ((rc = pn_hidden(net, B, X, wb, prm, Z1, Z2, H1, H2, s))) return rc;
  const long long ny = (long long)B * dout;
  const int nl = pn_layer_tiles(B, dout);  // <= ny: a tile holds at least one output
  GemmArgs g = pn_out(net, B, H2, wb, prm);
  g.Z = T;
  g.ldz = dout;
  g.scale = 1.0f / (float)ny;
  g.Cb = dY;
  g.ldcb = dout;
  g.lossp = scratch + ny - nl;
  if ((rc = pn_layer<EPI_LOSS>(g, s))) return rc;
  constexpr int kFill = 512;  // workgroups that fill the chip (two per CU)
  const long long room = ny - nl;
  const int nz = pn_tiles(B, H, 32, 64);
  const WGrad w2 = pn_wgrad(H, H, B, H1, dZ, grad + net.w2(), nullptr, room / 4, kFill - nz > 128 ? kFill - nz : 128);
  float* tail = scratch + room - w2.used;
  const WGrad w3 = pn_wgrad(H, dout, B, H2, dY, grad + net.w3(), scratch, room - w2.used, kFill - nz > 256 ? kFill - nz : 256);
  const WGrad w1 = pn_wgrad(din, H, B, X, H2, grad + net.w1(), scratch, room - w2.used, kFill);
  BackArgs a{};
  a.z = pn_dz(B, H, dout, dY, wb + net.w3(), Z2, dZ);
  a.nz = nz;
  a.w = w3.g;
  a.nw = w3.blocks;
  if ((rc = pn_back(a, s))) return rc;
  // dZ1 goes into the H2 slot (its last reader was dW3)
  a = BackArgs{};
  a.z = pn_dz(B, H, H, dZ, wb + net.w2(), Z1, H2);
  a.nz = nz;
  a.w = w2.g;
  if (w2.sum_blocks) a.w.C = tail;
  a.nw = w2.blocks;
  a.s = w3.sum;
  a.ns = w3.sum_blocks;
  if (loss) a.loss = {scratch + ny - nl, 1, 0, nl, loss, 1.0f / (float)ny};
  if ((rc = pn_back(a, s))) return rc;
  a = BackArgs{};
  a.w = w1.g;
  a.nw = w1.blocks;
  a.s = w2.sum;
  a.s.part = tail;
  a.ns = w2.sum_blocks;
  if ((rc = pn_back(a, s))) return rc;
  a = BackArgs{};
  a.s = w1.sum;
  a.ns = w1.sum_blocks;
  return pn_back(a, s);
}

int pnet_adam(long long P, float* prm, const float* g, float* m, float* v, int step, float lr,
              hipStream_t s) {
  const float c1 = 1.0f - powf(0.9f, (float)step), c2 = 1.0f - powf(0.999f, (float)step);
  hipLaunchKernelGGL(k_pn_adam, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, s, prm, g, m, v, P, lr, c1, c2);
  return hipGetLastError() == hipSuccess ? DNSMI_OK : DNSMI_EHIP;
}

// ------------------------------------------------------------------ features
struct PFeat {
  const double* kx;  // per kx index (Nkx)
  const double* kz;  // per kz index (Nkz)
  int Nkx, Ny, din;
  long long M;  // modes
  double kmax, dt, re, c;
  float s_1, s_2, s_out;
};

__device__ __forceinline__ double pf_k2(const PFeat& a, long long m) {
  const double kx = a.kx[m % a.Nkx], kz = a.kz[m / a.Nkx];
  return kx * kx + kz * kz;
}

// One thread per (sample, component, y): D1, D2 of the profile (the older
// terms rounded to FP32, as the guess's history keeps them) into X, and
// with nnext the weighted third difference into T.  X rows: [c][re,im][y]
// for D1, then for D2, then dt k^2 / Re, kx / k_max, kz / k_max, zeros.
__global__ void k_pn_features(PFeat a, const cx<double>* __restrict__ nm2, const cx<double>* __restrict__ nm1,
                              const cx<double>* __restrict__ ncur, const cx<double>* __restrict__ nnext,
                              const long long* __restrict__ modes, int ns, uint16_t* __restrict__ X,
                              float* __restrict__ T) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long per = 3LL * a.Ny;
  if (i >= (long long)ns * per) return;
  const int smp = (int)(i / per);
  const int r = (int)(i - (long long)smp * per);
  const int c = r / a.Ny, y = r - c * a.Ny;
  const long long m = modes[smp];
  const long long e = ((long long)c * a.M + m) * a.Ny + y;
  const cx<double> cu = ncur[e];
  const float h1x = (float)nm1[e].x, h1y = (float)nm1[e].y;
  const float h2x = (float)nm2[e].x, h2y = (float)nm2[e].y;
  const double d1x = cu.x - (double)h1x, d1y = cu.y - (double)h1y;
  const double d2x = (cu.x - 2.0 * (double)h1x) + (double)h2x, d2y = (cu.y - 2.0 * (double)h1y) + (double)h2y;
  uint16_t* xr = X + (size_t)smp * a.din;
  const int o = 2 * c * a.Ny + y;
  xr[o] = pn_bf16((float)d1x * a.s_1);
  xr[o + a.Ny] = pn_bf16((float)d1y * a.s_1);
  xr[6 * a.Ny + o] = pn_bf16((float)d2x * a.s_2);
  xr[6 * a.Ny + o + a.Ny] = pn_bf16((float)d2y * a.s_2);
  if (r == 0) {
    const double k2 = pf_k2(a, m);
    xr[12 * a.Ny] = pn_bf16((float)fmin(a.dt * k2 / a.re, 8.0));
    xr[12 * a.Ny + 1] = pn_bf16((float)(a.kx[m % a.Nkx] / a.kmax));
    xr[12 * a.Ny + 2] = pn_bf16((float)(a.kz[m / a.Nkx] / a.kmax));
    for (int f = 12 * a.Ny + 3; f < a.din; ++f) xr[f] = 0;
  }
  if (T && nnext) {
    const double w = 1.0 / (1.0 + a.dt * a.c * pf_k2(a, m) / a.re);
    const cx<double> p2 = nm2[e], p1 = nm1[e], x = nnext[e];
    const double d3x = (x.x - 3 * cu.x) + (3 * p1.x - p2.x), d3y = (x.y - 3 * cu.y) + (3 * p1.y - p2.y);
    float* tr = T + (size_t)smp * (6 * a.Ny);
    tr[o] = (float)(w * d3x / a.s_out);
    tr[o + a.Ny] = (float)(w * d3y / a.s_out);
  }
}

// The same input rows for the guess: every mode, from N^n (FP64) and the
// FP32 history h1 = N^{n-1}, h2 = N^{n-2} ((re, im) pairs, walls layout).
__global__ void k_pn_features_hist(PFeat a, const cx<double>* __restrict__ ncur, const float2* __restrict__ h1,
                                   const float2* __restrict__ h2, uint16_t* __restrict__ X) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long per = 3LL * a.Ny;
  if (i >= a.M * per) return;
  const long long m = i / per;
  const int r = (int)(i - m * per);
  const int c = r / a.Ny, y = r - c * a.Ny;
  const long long e = ((long long)c * a.M + m) * a.Ny + y;
  const cx<double> cu = ncur[e];
  const float2 p1 = h1[e], p2 = h2[e];
  const double d1x = cu.x - (double)p1.x, d1y = cu.y - (double)p1.y;
  const double d2x = (cu.x - 2.0 * (double)p1.x) + (double)p2.x, d2y = (cu.y - 2.0 * (double)p1.y) + (double)p2.y;
  uint16_t* xr = X + (size_t)m * a.din;
  const int o = 2 * c * a.Ny + y;
  xr[o] = pn_bf16((float)d1x * a.s_1);
  xr[o + a.Ny] = pn_bf16((float)d1y * a.s_1);
  xr[6 * a.Ny + o] = pn_bf16((float)d2x * a.s_2);
  xr[6 * a.Ny + o + a.Ny] = pn_bf16((float)d2y * a.s_2);
  if (r == 0) {
    const double k2 = pf_k2(a, m);
    xr[12 * a.Ny] = pn_bf16((float)fmin(a.dt * k2 / a.re, 8.0));
    xr[12 * a.Ny + 1] = pn_bf16((float)(a.kx[m % a.Nkx] / a.kmax));
    xr[12 * a.Ny + 2] = pn_bf16((float)(a.kz[m / a.Nkx] / a.kmax));
    for (int f = 12 * a.Ny + 3; f < a.din; ++f) xr[f] = 0;
  }
}

// Guess: next (= the quadratic extrapolation N_ext, FP64) += s_out Y / w per
// point, Y the network's output for every mode in order.
__global__ void k_pn_apply(PFeat a, const float* __restrict__ Y, cx<double>* __restrict__ next) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long per = 3LL * a.Ny;
  if (i >= a.M * per) return;
  const long long m = i / per;
  const int r = (int)(i - m * per);
  const int c = r / a.Ny, y = r - c * a.Ny;
  const double inv_w = 1.0 + a.dt * a.c * pf_k2(a, m) / a.re;
  const float* yr = Y + (size_t)m * (6 * a.Ny);
  const int o = 2 * c * a.Ny + y;
  const long long e = ((long long)c * a.M + m) * a.Ny + y;
  cx<double> v = next[e];
  v.x += (double)a.s_out * (double)yr[o] * inv_w;
  v.y += (double)a.s_out * (double)yr[o + a.Ny] * inv_w;
  next[e] = v;
}

static PFeat pfeat(Ctx* c, int din, float s_1, float s_2, float s_out) {
  PFeat a{};
  a.kx = c->kx;
  a.kz = c->kz;
  a.Nkx = c->Nx1;
  a.Ny = c->ny;
  a.din = din;
  a.M = (long long)c->Nz1 * c->Nx1;
  const double kxm = 2 * kPi / c->cfg.lx * (c->nx / 2), kzm = 2 * kPi / c->cfg.lz * (c->nz / 2);
  a.kmax = fmax(kxm, kzm);
  a.dt = c->cfg.dt;
  a.re = c->cfg.re;
  a.c = c->cfg.implicitness;
  a.s_1 = s_1;
  a.s_2 = s_2;
  a.s_out = s_out;
  return a;
}

int pnet_features(Ctx* c, const double* nm2, const double* nm1, const double* ncur, const double* nnext,
                  const long long* modes, int ns, int din, float s_1, float s_2, float s_out, uint16_t* X,
                  float* T, hipStream_t s) {
  if (!c->walls) return c->fail(DNSMI_EINVAL, "profile network: plane Couette contexts only");
  if (din < 12 * c->ny + 3 || din % 32) return c->fail(DNSMI_EINVAL, "profile network: din must be >= 12 ny + 3 and a multiple of 32");
  if (ns == 0) return DNSMI_OK;
  const PFeat a = pfeat(c, din, s_1, s_2, s_out);
  const long long n = (long long)ns * 3 * c->ny;
  hipLaunchKernelGGL(k_pn_features, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a,
                     reinterpret_cast<const cx<double>*>(nm2), reinterpret_cast<const cx<double>*>(nm1),
                     reinterpret_cast<const cx<double>*>(ncur), reinterpret_cast<const cx<double>*>(nnext),
                     modes, ns, X, T);
  return check_launch(c, "profile features");
}

int walls_guess_rhs(Ctx* c, const double* state, double* rhs, hipStream_t s);
int walls_predict(Ctx* c, const double* state, const double* rhs, double* pred, hipStream_t s);
int extrap_walls(Ctx* c, const double* n0, const float* h1, float* h2, double* next, const uint16_t* wb,
                 const float* bias, int H, float s_1, float s_2, float s_out, int mode, hipStream_t s);

// The plane Couette guess with the profile network: N^n (plain; the first
// corrector pass records the split reference), the network's input from N^n
// and the FP32 history,
// its output, then N_ext = quadratic extrapolation + s_out Y / w into
// rhs_prev (h2 <- N^n) and pred = the predictor's solve fed with N_ext.
// Caller-owned buffers, M = the number of modes: wb (the bf16 weight
// copies, one word per parameter), X (M din bf16 words), wh (2 H M bf16 words),
// Y (M dout floats).
int guess_walls_profile(Ctx* c, const double* state, double* pred, double* rhs_prev, const float* h1, float* h2,
                        int din, int H, int dout, const float* prm, uint16_t* wb, uint16_t* X, uint16_t* wh,
                        float* Y, float s_1, float s_2, float s_out, hipStream_t s) {
  if (!c->walls) return c->fail(DNSMI_EINVAL, "profile network: plane Couette contexts only");
  if (dout != 6 * c->ny) return c->fail(DNSMI_EINVAL, "profile network: dout must be 6 ny");
  const long long M = (long long)c->Nz1 * c->Nx1;
  if (M >= (1LL << 31)) return c->fail(DNSMI_EINVAL, "profile network: too many modes");
  int rc = walls_guess_rhs(c, state, c->rhs0, s);
  if (rc) return rc;
  const PFeat a = pfeat(c, din, s_1, s_2, s_out);
  const unsigned nb = (unsigned)((M * 3 * c->ny + 255) / 256);
  // the input reads h1, h2 before the extrapolation overwrites h2
  hipLaunchKernelGGL(k_pn_features_hist, dim3(nb), dim3(256), 0, s, a, reinterpret_cast<const cx<double>*>(c->rhs0),
                     reinterpret_cast<const float2*>(h1), reinterpret_cast<const float2*>(h2), X);
  if ((rc = check_launch(c, "profile input"))) return rc;
  if ((rc = pnet_forward(din, H, dout, (int)M, X, prm, wb, wh, Y, s)))
    return c->fail(rc, "profile network forward");
  if ((rc = extrap_walls(c, c->rhs0, h1, h2, rhs_prev, nullptr, nullptr, 32, s_1, s_2, s_out, 3, s))) return rc;
  hipLaunchKernelGGL(k_pn_apply, dim3(nb), dim3(256), 0, s, a, Y, reinterpret_cast<cx<double>*>(rhs_prev));
  if ((rc = check_launch(c, "profile apply"))) return rc;
  return walls_predict(c, state, rhs_prev, pred, s);
}

}  // namespace dnsmi
