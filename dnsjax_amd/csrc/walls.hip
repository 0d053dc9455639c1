// Plane Couette (wall-bounded) path, gfx950.
//
// Set-up (host C++, once per context; geometries/cartesian.py:575-801,
// fd.py:21-108): CGL grid, Fornberg D1/D2 stencils, per-mode Lk (Neumann)
// and Hk (Dirichlet) band matrices factored with partial pivoting in the
// LAPACK ab layout (dgbtf2 order of operations), homogeneous solutions
// p_i, v_i, q_i and the 2x2 influence matrix inverse, y-quadrature
// weights.  Per-mode tables are stored mode-fastest ([j][row][mode]) so a
// wavefront whose lanes are consecutive (kz, kx) modes reads them
// coalesced.
//
// Per step:
//   RHS (flows/plane_couette.py:274-289): WT1 FD curl + transpose
//   (3,Nkz,Nkx,Ny) -> 6 fields (Ny,Nkz,Nkx); z-inverse; the shared x pass
//   with base flow U = y; the shared z-forward; WT5 transpose back.
//   IMM (flows/plane_couette.py:376-504): divergence, the pressure's Lk
//   solve, the three velocity solves with Hk, wall divergence, alpha = -M^-1 d,
//   correction and the quadrature-weighted norm partials: one launch whose
//   workgroups take two modes of one k^2 class each, band solves as chains of
//   matrix-core products (k_imm_fused); the same in five launches, or with
//   sequential sweeps, where the modes are too few or the columns too long.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdint>
#include <cstring>
#include <string>
#include <thread>
#include <unordered_map>
#include <vector>

#include "context.hpp"
#include "dft.hpp"
#include "passes.hpp"

namespace dnsmi {

// Influence-matrix work vectors (complex, [vec][mode][y]): f_hat, the
// pressure, the three R_c / velocity columns, three forward-sweep results.
enum ImmVec { V_F = 0, V_P = 1, V_R = 2, V_T = 5, V_COUNT = 8 };
constexpr int kImmT = 128;  // threads per mode in the parallel phases

struct WallTables {
  int p = 0, Ny = 0, Nkz = 0, Nkx = 0, M = 0;
  int curl_ty = 32;  // y points per curl workgroup (walls_curl_ty)
  // device
  double* d1w = nullptr;  // (Ny, p+1)
  double *d1t = nullptr, *d2t = nullptr;  // the same as (p+1, Ny), (p+2, Ny): lanes along y read adjacent words
  int* d1j0 = nullptr;    // (Ny)
  double* d2w = nullptr;  // (Ny, p+2)
  int* d2j0 = nullptr;
  double* qw = nullptr;   // quadrature weight / Ly, (Ny)
  double* lk_ab = nullptr;  // [j][row][mode]
  int* lk_piv = nullptr;    // [j][mode]
  double* hk_ab = nullptr;
  int* hk_piv = nullptr;
  double* vq = nullptr;   // [map][y][4]: v1, v2, q1, q2 of a k^2 class
  int* umode = nullptr;   // per mode: its k^2 class (map)
  double* minv = nullptr;  // [4][mode]
  double* mkx = nullptr;   // per mode
  double* mkz = nullptr;
  double* scratch = nullptr;  // IMM work vectors, complex [vec][mode][y]
  // chunk maps of the band solves (chunked sweeps), one per distinct k^2,
  // (map_word); sched = the modes, with their maps, in the order
  // the chunked solve takes them (items of two modes of one map)
  double *lk_fmap = nullptr, *lk_bmap = nullptr, *hk_fmap = nullptr, *hk_bmap = nullptr;
  int2* sched = nullptr;  // (mode, map) per slot, two slots per item
  int items = 0;
  int U = 0;              // distinct k^2 values
  // host copies: the y grid, and each mode's class (walls_table reads the
  // device tables back in the reference layouts through it)
  std::vector<double> h_ys;
  std::vector<int> h_umode;
};

inline int walls_curl_ty(int Ny, int M);  // the curl kernel's tile height

// ------------------------------------------------------------------ host set-up
// Fornberg (1998), SIAM Rev. 40, 685-691: weights of derivatives 0..m at z
// on nodes x[0..n].
static void fornberg(double z, const double* x, int n1, int m, std::vector<double>& C) {
  const int n = n1 - 1;
  C.assign((size_t)n1 * (m + 1), 0.0);
  auto at = [&](int i, int k) -> double& { return C[(size_t)i * (m + 1) + k]; };
  at(0, 0) = 1.0;
  double c1 = 1.0, c4 = x[0] - z;
  for (int i = 1; i <= n; ++i) {
    const int mn = std::min(i, m);
    double c2 = 1.0;
    const double c5 = c4;
    c4 = x[i] - z;
    for (int j = 0; j < i; ++j) {
      const double c3 = x[i] - x[j];
      c2 *= c3;
      if (j == i - 1) {
        for (int k = mn; k > 0; --k) at(i, k) = c1 * (k * at(i - 1, k - 1) - c5 * at(i - 1, k)) / c2;
        at(i, 0) = -c1 * c5 * at(i - 1, 0) / c2;
      }
      for (int k = mn; k > 0; --k) at(j, k) = (c4 * at(j, k) - k * at(j, k - 1)) / c3;
      at(j, 0) = c4 * at(j, 0) / c3;
    }
    c1 = c2;
  }
}

struct Stencil {
  int width;
  std::vector<double> w;  // (Ny, width)
  std::vector<int> j0;    // (Ny)
};

// fd.py:68-108: D1 with p+1 points, D2 with p+2 points, one-sided at walls.
static void build_stencils(const std::vector<double>& y, int p, Stencil& d1, Stencil& d2) {
  const int Ny = (int)y.size();
  d1.width = p + 1;
  d2.width = p + 2;
  d1.w.assign((size_t)Ny * d1.width, 0.0);
  d2.w.assign((size_t)Ny * d2.width, 0.0);
  d1.j0.assign(Ny, 0);
  d2.j0.assign(Ny, 0);
  std::vector<double> C;
  for (int i = 0; i < Ny; ++i) {
    int j0 = std::max(0, std::min(i - d1.width / 2, Ny - d1.width));
    fornberg(y[i], &y[j0], d1.width, 1, C);
    d1.j0[i] = j0;
    for (int k = 0; k < d1.width; ++k) d1.w[(size_t)i * d1.width + k] = C[(size_t)k * 2 + 1];
    j0 = std::max(0, std::min(i - d2.width / 2, Ny - d2.width));
    fornberg(y[i], &y[j0], d2.width, 2, C);
    d2.j0[i] = j0;
    for (int k = 0; k < d2.width; ++k) d2.w[(size_t)i * d2.width + k] = C[(size_t)k * 3 + 2];
  }
}

// Dense row i of a stencil operator, as a function (j -> value).
static double stencil_at(const Stencil& s, int i, int j) {
  const int k = j - s.j0[i];
  return (k >= 0 && k < s.width) ? s.w[(size_t)i * s.width + k] : 0.0;
}

// LAPACK band storage: A(i, j) = ab[(kl + ku + i - j) * n + j] (row-major
// rows of length n here), 2 kl + ku + 1 rows.
struct Band {
  int n, kl, ku, rows;
  std::vector<double> ab;
  std::vector<int> piv;
  Band(int n_, int kl_, int ku_) : n(n_), kl(kl_), ku(ku_), rows(2 * kl_ + ku_ + 1) {
    ab.assign((size_t)rows * n, 0.0);
    piv.assign(n, 0);
  }
  double& at(int i, int j) { return ab[(size_t)(kl + ku + i - j) * n + j]; }
  double& raw(int r, int j) { return ab[(size_t)r * n + j]; }
};

// Partial-pivoting band LU in the order of LAPACK's unblocked dgbtf2
// (the routine dgbtrf uses when its block size exceeds kl): pivot = first
// largest |a| in the column, reciprocal-scaled multipliers, rank-1 update
// up to the last column touched so far.  Returns 0 or the 1-based index of
// a zero pivot.
static int band_lu(Band& B) {
  const int n = B.n, kl = B.kl, ku = B.ku, kv = kl + ku;
  int ju = 0, info = 0;
  for (int j = 0; j < n; ++j) {
    const int km = std::min(kl, n - 1 - j);
    int jp = 0;
    double best = std::fabs(B.raw(kv, j));
    for (int i = 1; i <= km; ++i) {
      const double a = std::fabs(B.raw(kv + i, j));
      if (a > best) {
        best = a;
        jp = i;
      }
    }
    B.piv[j] = j + jp;
    if (B.raw(kv + jp, j) != 0.0) {
      ju = std::max(ju, std::min(j + ku + jp, n - 1));
      if (jp != 0)
        for (int c = j; c <= ju; ++c) std::swap(B.at(j, c), B.at(j + jp, c));
      if (km > 0) {
        const double r = 1.0 / B.raw(kv, j);
        for (int i = 1; i <= km; ++i) B.raw(kv + i, j) *= r;
        for (int c = j + 1; c <= ju; ++c) {
          const double t = -B.at(j, c);
          if (t != 0.0)
            for (int i = 1; i <= km; ++i) B.at(j + i, c) += B.raw(kv + i, j) * t;
        }
      }
    } else if (info == 0) {
      info = j + 1;
    }
  }
  return info;
}

// dgbtrs('N') on one real right-hand side, as the device sweep does it.
static void band_solve(const Band& B, std::vector<double>& b) {
  const int n = B.n, kl = B.kl, ku = B.ku, kuu = kl + ku;
  auto raw = [&](int r, int j) { return B.ab[(size_t)r * n + j]; };
  for (int j = 0; j < n - 1; ++j) {
    const int pj = B.piv[j];
    std::swap(b[j], b[pj]);
    for (int i = 1; i <= kl && j + i < n; ++i) b[j + i] -= raw(kl + ku + i, j) * b[j];
  }
  for (int j = n - 1; j >= 0; --j) {
    const double x = b[j] / raw(kl + ku, j);
    b[j] = x;
    for (int i = 1; i <= kuu && j - i >= 0; ++i) b[j - i] -= raw(kuu - i, j) * x;
  }
}

// Chunk maps of the band solves: a chunk of B rows, with the rows its steps
// reach (kl after it forward, kl + ku before it back), is a window of at most
// 16 rows, or of 32 where a back window's reach leaves 16 too little (p >= 6).
// B is a multiple of four rows, so that the rows a window keeps move by whole
// registers of the matrix cores' operands (chunk_chain).
//
// mx, a mixed context: 16 rows, in windows of up to 32.  There the iterate is
// rounded to FP32 at the start of every evaluation, where a change in its last
// bit can send an element to the other neighbour: 1e-7 of the RMS in an
// element of the nonlinear term, 1e-10 of the whole.  So the mixed form keeps
// one order of operations to the bit: chunks of 16 rows, each of a map's sums
// over the window's rows in ascending order (v_mfma_f64_16x16x4_f64 is four
// fused multiply-adds in ascending k), and the right-hand sides' terms one by
// one (imm_fhat_mx_at, imm_r_at).  Its maps take 72 words per row of the
// column where the FP64 contexts' take 53 (p = 4; p = 6: 80 and 70), and one step
// of 128 x 256 x 128, p = 6, 317 us where theirs takes 302.
__host__ __device__ constexpr int chunk_tiles(int p, bool back, bool mx) { return mx || (back && p >= 6) ? 2 : 1; }
__host__ __device__ constexpr int chunk_keep(int p, bool back) { return back ? 2 * p : p; }
__host__ __device__ constexpr int chunk_rows(int p, bool back, bool mx) {
  return mx ? 16 : 16 * chunk_tiles(p, back, mx) - (chunk_keep(p, back) + 3) / 4 * 4;
}
__host__ __device__ constexpr int chunk_window(int p, bool back, bool mx) {
  return chunk_rows(p, back, mx) + chunk_keep(p, back);
}
// rows that a window's registers hold: the window up to a multiple of four
__host__ __device__ constexpr int chunk_span(int p, bool back, bool mx) {
  return (chunk_window(p, back, mx) + 3) / 4 * 4;
}
__host__ __device__ constexpr int chunk_count(int n, int p, bool back, bool mx) {
  return (n + chunk_rows(p, back, mx) - 1) / chunk_rows(p, back, mx);
}
// A map's words, in the order the products take them (map of chunk c, class
// u at (c U + u) words): operand e of lane (g = lane / 16, r = lane % 16) at
// map_word(e, lane), two operands side by side, so that a wavefront's load
// is 1 KB of consecutive words.  One tile: e = k / 4, entry (t = r, k = 4 e +
// g).  Two: first the operands of rows 16 + r (high_operands), then those of
// rows r (low_operands), of which a back map's k >= 16 are zero by construction
// (it is lower triangular) and left out.  A mixed context's back map is the
// identity in rows and columns >= 16 (its steps eliminate with rows < 16 only):
// those columns are left out too, and the window's rows added at their place in
// the sum (chunk_chain), the same value to the bit: one step of 128 x 256 x 128,
// p = 6, 360 us with them, 317 us without.
__host__ __device__ constexpr int high_operands(int p, bool back, bool mx) {
  return chunk_tiles(p, back, mx) == 1 ? 0 : back && mx ? 4 : chunk_span(p, back, mx) / 4;
}
__host__ __device__ constexpr int low_operands(int p, bool back, bool mx) {
  return back || !mx ? 4 : chunk_span(p, back, mx) / 4;
}
// Longest column of the chunked solves: the five-launch form's H_k solve keeps
// six of them with their zero rows (chunk_lds) in LDS, at most 65392 bytes for
// every Ny up to here.
constexpr int kChunkNy = 650;
__host__ __device__ constexpr int map_operands(int p, bool back, bool mx) {
  return high_operands(p, back, mx) + low_operands(p, back, mx);
}
__host__ __device__ constexpr int map_words(int p, bool back, bool mx) { return 64 * map_operands(p, back, mx); }
__host__ __device__ constexpr int map_word(int e, int lane) { return ((e >> 1) * 64 + lane) * 2 + (e & 1); }
// entry (t, k) of word i
__host__ __device__ inline void map_entry(int i, int high, int& t, int& k) {
  const int e = (i >> 7) * 2 + (i & 1), lane = (i & 127) >> 1;
  t = (lane & 15) + (e < high ? 16 : 0);
  k = 4 * (e < high ? e : e - high) + (lane >> 4);
}

// Chunk maps of one band solve (the operation order of band_solve): forward
// chunk c applies the steps j in [cB, min(cB + B, n - 1)) (row swap,
// elimination) to the window of rows cB + t, t < W = B + kl; its map is those
// row operations applied to the identity.  Back chunk c, top row T = n - 1 -
// cB, applies the steps j = T, T - 1, ... (at most B, j >= 0: divide by the
// diagonal, eliminate upwards) to the window of rows T - t, t < W = B + kl +
// ku.  Written as map u of U; `raw(r, j)` reads the factored band, `piv(j)`
// the pivot row.  Returns false if an entry left out is not what it is taken for
// (it cannot be, by the argument above; the check keeps the layout honest).
template <typename Raw, typename Piv>
static bool chunk_maps(int n, int p, bool mx, int u, int U, Raw raw, Piv piv, double* F, double* G) {
  const int kl = p, kuu = 2 * p;
  bool ok = true;
  std::vector<double> X;
  auto write = [&](bool back, int c, double* out) {
    const int W = chunk_window(p, back, mx), words = map_words(p, back, mx), high = high_operands(p, back, mx);
    const int klow = 4 * low_operands(p, back, mx);  // columns that rows 0 .. 15 keep, and the others
    const int khigh = 4 * high;
    double* m = out + ((size_t)c * U + u) * words;
    for (int i = 0; i < words; ++i) {
      int t, k;
      map_entry(i, high, t, k);
      m[i] = t < W && k < W ? X[(size_t)t * W + k] : 0.0;
    }
    for (int t = 0; t < W; ++t)
      for (int k = t < 16 ? klow : khigh; k < W; ++k) ok = ok && X[(size_t)t * W + k] == (t == k ? 1.0 : 0.0);
  };
  for (int c = 0; c < chunk_count(n, p, false, mx); ++c) {
    const int B = chunk_rows(p, false, mx), W = chunk_window(p, false, mx), j0 = c * B;
    X.assign((size_t)W * W, 0.0);
    for (int t = 0; t < W; ++t) X[(size_t)t * W + t] = 1.0;
    for (int j = j0; j < std::min(j0 + B, n - 1); ++j) {
      const int tj = j - j0, tp = piv(j) - j0;
      if (tp != tj)
        for (int k = 0; k < W; ++k) std::swap(X[(size_t)tj * W + k], X[(size_t)tp * W + k]);
      for (int i = 1; i <= kl && j + i < n; ++i) {
        const double l = raw(kuu + i, j);
        for (int k = 0; k < W; ++k) X[(size_t)(tj + i) * W + k] -= l * X[(size_t)tj * W + k];
      }
    }
    write(false, c, F);
  }
  for (int c = 0; c < chunk_count(n, p, true, mx); ++c) {
    const int B = chunk_rows(p, true, mx), W = chunk_window(p, true, mx), T = n - 1 - c * B;
    X.assign((size_t)W * W, 0.0);
    for (int t = 0; t < W; ++t) X[(size_t)t * W + t] = 1.0;
    for (int j = T; j > T - B && j >= 0; --j) {
      const int tj = T - j;
      const double dg = raw(kuu, j);
      for (int k = 0; k < W; ++k) X[(size_t)tj * W + k] /= dg;
      for (int i = 1; i <= kuu && j - i >= 0; ++i) {
        const double l = raw(kuu - i, j);
        for (int k = 0; k < W; ++k) X[(size_t)(tj + i) * W + k] -= l * X[(size_t)tj * W + k];
      }
    }
    write(true, c, G);
  }
  return ok;
}

// Linear weights of the y quadrature, divided by Ly.  Odd Ny: the
// non-uniform composite Simpson rule (geometries/cartesian.py:125-140).
// Even Ny (the reference exits there): Simpson panels over the first Ny-4
// intervals plus the exact integral of the cubic through the last four
// points.
static std::vector<double> quadrature_weights(const std::vector<double>& y, double Ly) {
  const int n = (int)y.size();
  std::vector<double> w(n, 0.0);
  const int m = (n % 2 == 1) ? n : n - 3;
  for (int i = 0; i + 2 < m; i += 2) {
    const double h0 = y[i + 1] - y[i], h1 = y[i + 2] - y[i + 1];
    const double hs = h0 + h1, hp = h0 * h1, r = h0 / h1;
    w[i] += hs / 6 * (2 - 1 / r);
    w[i + 1] += hs / 6 * (hs * hs / hp);
    w[i + 2] += hs / 6 * (2 - r);
  }
  if (n % 2 == 0) {
    // solve V w = moments, V[m][i] = (x_i - a)^m, on the last 4 points
    const double a = y[n - 4], b = y[n - 1];
    double V[4][5];
    for (int r = 0; r < 4; ++r) {
      for (int i = 0; i < 4; ++i) V[r][i] = std::pow(y[n - 4 + i] - a, r);
      V[r][4] = std::pow(b - a, r + 1) / (r + 1);
    }
    for (int c = 0; c < 4; ++c) {  // Gaussian elimination with partial pivoting
      int pr = c;
      for (int r = c + 1; r < 4; ++r)
        if (std::fabs(V[r][c]) > std::fabs(V[pr][c])) pr = r;
      for (int k = 0; k < 5; ++k) std::swap(V[c][k], V[pr][k]);
      for (int r = c + 1; r < 4; ++r) {
        const double f = V[r][c] / V[c][c];
        for (int k = c; k < 5; ++k) V[r][k] -= f * V[c][k];
      }
    }
    double x[4];
    for (int r = 3; r >= 0; --r) {
      double s = V[r][4];
      for (int k = r + 1; k < 4; ++k) s -= V[r][k] * x[k];
      x[r] = s / V[r][r];
    }
    for (int i = 0; i < 4; ++i) w[n - 4 + i] += x[i];
  }
  for (double& v : w) v /= Ly;
  return w;
}

template <typename V>
static int upload_vec(Ctx* c, V** dst, const std::vector<V>& v) {
  *dst = static_cast<V*>(c->alloc(v.size() * sizeof(V)));
  if (!*dst) return c->fail(DNSMI_ENOMEM, "device allocation failed");
  const hipError_t e = hipMemcpy(*dst, v.data(), v.size() * sizeof(V), hipMemcpyHostToDevice);
  if (e != hipSuccess) return c->fail(DNSMI_EHIP, hipGetErrorString(e));
  return DNSMI_OK;
}

static int walls_autotune(Ctx* c);

// ------------------------------------------------------------------ set-up on the GPU
// The per-class tables of geometries/cartesian.py:575-801 built on the GPU:
// the band LU of L_k and H_k (band_lu), the homogeneous solutions and M^-1
// (the band_solve / D1 sequence of walls_setup's class loop) and the chunk
// maps (chunk_maps), with the host code's operations in its order and every
// product, sum and quotient rounded on its own as the host computes them
// (contraction into FMA is switched off in these kernels), so the tables
// equal the host set-up's bit for bit.  One workgroup of one wavefront per
// k^2 class (and matrix, and chunk); a class's band lives in LDS while it is
// factored and used.
struct GpuSetup {
  int n, kl, ku, rows, U, W1, W2;  // W1, W2: widths of the D1 and D2 stencils
  int mx;                          // chunk maps of a mixed context
  const double* d1w;
  const int* d1j0;
  const double* d2w;
  const int* d2j0;
  const double* k2;  // [U]
  double dt, cc, nu;
  double* band;  // [2][U][rows][n], raw(r, j) at r * n + j; L_k then H_k
  int* piv;      // [2][U][n]
  int* flag;     // [0]: a zero pivot, [1]: a chunk-map entry left out of the packing is not zero
  double* vq;    // [U][n][4]
  double* minv;  // [U][4]
};

__device__ inline double setup_stencil(const double* w, const int* j0, int W, int i, int j) {
  const int k = j - j0[i];
  return (k >= 0 && k < W) ? w[i * W + k] : 0.0;
}

// d1_apply of walls_setup: s += w_k v_(j0 + k), k ascending, from 0.
__device__ inline double setup_d1(const GpuSetup& g, const double* v, int i) {
#pragma clang fp contract(off)
  double s = 0.0;
  for (int k = 0; k < g.W1; ++k) {
    const double t = g.d1w[i * g.W1 + k] * v[g.d1j0[i] + k];
    s = s + t;
  }
  return s;
}

// Build and factor L_k (blockIdx.y = 0) or H_k (1) of class blockIdx.x.
__global__ void __launch_bounds__(64) k_setup_lu(GpuSetup g) {
#pragma clang fp contract(off)
  extern __shared__ double ab[];  // rows x n
  const int u = blockIdx.x, which = blockIdx.y, lane = threadIdx.x;
  const int n = g.n, kl = g.kl, ku = g.ku, kv = kl + ku, rows = g.rows;
  const double k2 = g.k2[u];
  for (int e = lane; e < rows * n; e += 64) ab[e] = 0.0;
  __syncthreads();
  for (int i = lane; i < n; i += 64) {
    const int jlo = i - kl > 0 ? i - kl : 0, jhi = i + ku < n - 1 ? i + ku : n - 1;
    for (int j = jlo; j <= jhi; ++j) {
      const double lraw = setup_stencil(g.d2w, g.d2j0, g.W2, i, j) - (i == j ? k2 : 0.0);
      double v;
      if (which == 0) {
        v = lraw;
        if (i == 0) v = (k2 == 0.0) ? (j == 0 ? 1.0 : 0.0) : setup_stencil(g.d1w, g.d1j0, g.W1, 0, j);
        if (i == n - 1) v = setup_stencil(g.d1w, g.d1j0, g.W1, n - 1, j);
      } else {
        const double cn = g.cc * g.nu;
        const double t = cn * lraw;
        v = (i == j ? 1.0 / g.dt : 0.0) - t;
        if (i == 0 || i == n - 1) v = (i == j) ? 1.0 : 0.0;
      }
      ab[(kv + i - j) * n + j] = v;
    }
  }
  __syncthreads();
  int ju = 0;
  bool zero = false;
  int* piv = g.piv + (size_t)(which * g.U + u) * n;
  for (int j = 0; j < n; ++j) {
    const int km = kl < n - 1 - j ? kl : n - 1 - j;
    int jp = 0;
    double best = fabs(ab[kv * n + j]);
    for (int i = 1; i <= km; ++i) {
      const double a = fabs(ab[(kv + i) * n + j]);
      if (a > best) {
        best = a;
        jp = i;
      }
    }
    const double pv = ab[(kv + jp) * n + j];
    if (lane == 0) piv[j] = j + jp;
    __syncthreads();
    if (pv == 0.0) {
      zero = true;
      continue;
    }
    const int jr = j + ku + jp < n - 1 ? j + ku + jp : n - 1;
    ju = ju > jr ? ju : jr;
    if (jp != 0) {
      for (int c = j + lane; c <= ju; c += 64) {
        const double a0 = ab[(kv + j - c) * n + c];
        ab[(kv + j - c) * n + c] = ab[(kv + j + jp - c) * n + c];
        ab[(kv + j + jp - c) * n + c] = a0;
      }
      __syncthreads();
    }
    if (km > 0) {
      const double r = 1.0 / ab[kv * n + j];
      if (lane >= 1 && lane <= km) ab[(kv + lane) * n + j] = ab[(kv + lane) * n + j] * r;
      __syncthreads();
      const int nc = ju - j;
      for (int e = lane; e < nc * km; e += 64) {
        const int q = e / km, i = 1 + e - q * km, c = j + 1 + q;
        const double t = -ab[(kv + j - c) * n + c];
        if (t != 0.0) {
          const double prod = ab[(kv + i) * n + j] * t;
          ab[(kv + j + i - c) * n + c] = ab[(kv + j + i - c) * n + c] + prod;
        }
      }
      __syncthreads();
    }
  }
  if (zero && lane == 0) g.flag[0] = 1;
  double* out = g.band + (size_t)(which * g.U + u) * rows * n;
  for (int e = lane; e < rows * n; e += 64) out[e] = ab[e];
}

// band_solve on the vectors v + q n (q < nvec), one per 16 lanes, with the
// factored band ab and pivots pl in LDS.
__device__ inline void setup_solve(const GpuSetup& g, const double* ab, const int* pl, double* v, int nvec) {
#pragma clang fp contract(off)
  const int n = g.n, kl = g.kl, kv = g.kl + g.ku, lane = threadIdx.x;
  const int q = lane >> 4, t = lane & 15;
  const bool act = q < nvec;
  double* b = v + (act ? q : 0) * n;
  for (int j = 0; j < n - 1; ++j) {
    if (act && t == 0) {
      const int pj = pl[j];
      const double x = b[j];
      b[j] = b[pj];
      b[pj] = x;
    }
    __syncthreads();
    if (act && t >= 1 && t <= kl && j + t < n) {
      const double prod = ab[(kv + t) * n + j] * b[j];
      b[j + t] = b[j + t] - prod;
    }
    __syncthreads();
  }
  for (int j = n - 1; j >= 0; --j) {
    if (act && t == 0) b[j] = b[j] / ab[kv * n + j];
    __syncthreads();
    const int i = t + 1;
    if (act && i <= kv && j - i >= 0) {
      const double prod = ab[(kv - i) * n + j] * b[j];
      b[j - i] = b[j - i] - prod;
    }
    __syncthreads();
  }
}

// Homogeneous solutions and M^-1 of class blockIdx.x: p_1,2 = L^-1 e_(0, n-1);
// v_1,2 = H^-1 (-D1 p_1,2 with zero wall rows); q_1,2 = H^-1 (p_1,2 with
// zero wall rows); M = D1 v at the walls.
__global__ void __launch_bounds__(64) k_setup_homog(GpuSetup g) {
#pragma clang fp contract(off)
  extern __shared__ double sm[];
  const int u = blockIdx.x, lane = threadIdx.x, n = g.n, rows = g.rows;
  double* ab = sm;               // rows x n
  double* v = sm + rows * n;     // four vectors of n
  int* pl = reinterpret_cast<int*>(v + 4 * n);
  for (int which = 0; which < 2; ++which) {
    const double* src = g.band + (size_t)(which * g.U + u) * rows * n;
    const int* ps = g.piv + (size_t)(which * g.U + u) * n;
    for (int e = lane; e < rows * n; e += 64) ab[e] = src[e];
    for (int e = lane; e < n; e += 64) pl[e] = ps[e];
    if (which == 0)
      for (int e = lane; e < 2 * n; e += 64) v[e] = (e == 0 || e == 2 * n - 1) ? 1.0 : 0.0;
    __syncthreads();
    setup_solve(g, ab, pl, v, which == 0 ? 2 : 4);
    if (which == 0) {
      // r_1,2 = -D1 p_1,2 (zero on the walls) into vectors 2, 3; then the
      // walls of p_1,2 zeroed in place: the four H_k right-hand sides
      for (int i = lane; i < n; i += 64) {
        const bool wall = i == 0 || i == n - 1;
        v[2 * n + i] = wall ? 0.0 : -setup_d1(g, v, i);
        v[3 * n + i] = wall ? 0.0 : -setup_d1(g, v + n, i);
      }
      __syncthreads();
      if (lane == 0) v[0] = v[n - 1] = v[n] = v[2 * n - 1] = 0.0;
      __syncthreads();
    }
  }
  if (lane == 0) {
    const double m00 = setup_d1(g, v + 2 * n, 0), m01 = setup_d1(g, v + 3 * n, 0);
    const double m10 = setup_d1(g, v + 2 * n, n - 1), m11 = setup_d1(g, v + 3 * n, n - 1);
    double mi[4];
    if (g.k2[u] == 0.0) {
      mi[0] = mi[1] = mi[2] = 0.0;
      mi[3] = 1.0 / m11;
    } else {
      const double a = m00 * m11, b = m01 * m10;
      const double det = a - b;
      mi[0] = m11 / det;
      mi[1] = -m01 / det;
      mi[2] = -m10 / det;
      mi[3] = m00 / det;
    }
    for (int q = 0; q < 4; ++q) g.minv[u * 4 + q] = mi[q];
  }
  for (int j = lane; j < n; j += 64) {
    double* w = g.vq + ((size_t)u * n + j) * 4;
    w[0] = v[2 * n + j];
    w[1] = v[3 * n + j];
    w[2] = v[j];
    w[3] = v[n + j];
  }
}

// Chunk map of chunk blockIdx.x, class blockIdx.y; blockIdx.z: 0 L_k
// forward, 1 L_k back, 2 H_k forward, 3 H_k back (chunk_maps' steps).
__global__ void __launch_bounds__(64) k_setup_maps(GpuSetup g, double* lf, double* lb, double* hf, double* hb) {
#pragma clang fp contract(off)
  constexpr int WMAX = 32;
  __shared__ double X[WMAX * WMAX];
  const int c = blockIdx.x, u = blockIdx.y, which = blockIdx.z >> 1;
  const bool back = blockIdx.z & 1;
  const int lane = threadIdx.x, n = g.n, kl = g.kl, kuu = g.kl + g.ku;
  const bool mx = g.mx;
  if (c >= chunk_count(n, kl, back, mx)) return;
  const double* ab = g.band + (size_t)(which * g.U + u) * g.rows * n;
  const int* pv = g.piv + (size_t)(which * g.U + u) * n;
  const int B = chunk_rows(kl, back, mx), W = chunk_window(kl, back, mx);
  for (int e = lane; e < W * W; e += 64) X[e] = (e / W == e % W) ? 1.0 : 0.0;
  __syncthreads();
  const int j0 = c * B;
  if (!back) {
    const int jend = j0 + B < n - 1 ? j0 + B : n - 1;
    for (int j = j0; j < jend; ++j) {
      const int tj = j - j0, tp = pv[j] - j0;
      if (tp != tj) {
        for (int k = lane; k < W; k += 64) {
          const double x = X[tj * W + k];
          X[tj * W + k] = X[tp * W + k];
          X[tp * W + k] = x;
        }
        __syncthreads();
      }
      for (int e = lane; e < kl * W; e += 64) {
        const int i = 1 + e / W, k = e % W;
        if (j + i < n) {
          const double prod = ab[(kuu + i) * n + j] * X[tj * W + k];
          X[(tj + i) * W + k] = X[(tj + i) * W + k] - prod;
        }
      }
      __syncthreads();
    }
  } else {
    const int T = n - 1 - j0;
    for (int j = T; j > T - B && j >= 0; --j) {
      const int tj = T - j;
      const double dg = ab[kuu * n + j];
      for (int k = lane; k < W; k += 64) X[tj * W + k] = X[tj * W + k] / dg;
      __syncthreads();
      for (int e = lane; e < kuu * W; e += 64) {
        const int i = 1 + e / W, k = e % W;
        if (j - i >= 0) {
          const double prod = ab[(kuu - i) * n + j] * X[tj * W + k];
          X[(tj + i) * W + k] = X[(tj + i) * W + k] - prod;
        }
      }
      __syncthreads();
    }
  }
  const int words = map_words(kl, back, mx), high = high_operands(kl, back, mx);
  const int klow = 4 * low_operands(kl, back, mx), khigh = 4 * high;
  double* F = (which == 0 ? (back ? lb : lf) : (back ? hb : hf)) + ((size_t)c * g.U + u) * words;
  for (int i = lane; i < words; i += 64) {
    int t, k;
    map_entry(i, high, t, k);
    F[i] = t < W && k < W ? X[t * W + k] : 0.0;
  }
  bool bad = false;
  for (int e = lane; e < W * W; e += 64) {
    const int t = e / W, k = e % W;
    bad = bad || (k >= (t < 16 ? klow : khigh) && X[e] != (t == k ? 1.0 : 0.0));
  }
  if (bad) g.flag[1] = 1;
}

// Per-mode tables from the per-class ones: band factors [j][row][mode],
// pivots [j][mode], M^-1 [4][mode].
__global__ void __launch_bounds__(256) k_setup_scatter(GpuSetup g, const int* __restrict__ umode, int M,
                                                       double* lk_ab, double* hk_ab, int* lk_piv, int* hk_piv,
                                                       double* minv) {
  const long long nab = (long long)g.n * g.rows * M, npv = (long long)g.n * M;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < nab; e += (long long)gridDim.x * blockDim.x) {
    const int m = (int)(e % M);
    const long long jr = e / M;
    const int r = (int)(jr % g.rows), j = (int)(jr / g.rows), u = umode[m];
    lk_ab[e] = g.band[((size_t)u * g.rows + r) * g.n + j];
    hk_ab[e] = g.band[((size_t)(g.U + u) * g.rows + r) * g.n + j];
    if (e < npv) {
      const int mm = (int)(e % M), jj = (int)(e / M), uu = umode[mm];
      lk_piv[e] = g.piv[(size_t)uu * g.n + jj];
      hk_piv[e] = g.piv[(size_t)(g.U + uu) * g.n + jj];
    }
    if (e < 4LL * M) {
      const int mm = (int)(e % M), q = (int)(e / M);
      minv[e] = g.minv[umode[mm] * 4 + q];
    }
  }
}

// LDS bytes of the set-up kernels (the GPU set-up runs where both fit 64 KiB).
static size_t setup_lds_lu(int n, int rows) { return (size_t)rows * n * sizeof(double); }
static size_t setup_lds_homog(int n, int rows) {
  return ((size_t)rows * n + 4ull * n) * sizeof(double) + (size_t)n * sizeof(int);
}

int walls_setup(Ctx* c) {
  const dnsmi_config& g = c->cfg;
  if (g.nx % 2 || g.nz % 2 || g.nx < 4 || g.nz < 4 || g.ny < 5)
    return c->fail(DNSMI_EINVAL, "walls: nx, nz even >= 4 and ny >= 5");
  // the y grid is fixed on [-1, 1] (parameters.py:190-191)
  if (g.ly != 2.0) return c->fail(DNSMI_EINVAL, "walls: ly must be 2 (the channel is y in [-1, 1])");
  if (g.oversampling_factor != 3) return c->fail(DNSMI_EINVAL, "oversampling_factor must be 3");
  const int p = g.fd_order;
  if (p != 2 && p != 4 && p != 6 && p != 8) return c->fail(DNSMI_EINVAL, "fd_order must be 2, 4, 6 or 8");
  if (g.ny < p + 3) return c->fail(DNSMI_EINVAL, "ny too small for fd_order");
  c->nx = g.nx;
  c->ny = g.ny;
  c->nz = g.nz;
  c->Nx1 = g.nx / 2;
  c->Nz1 = g.nz - 1;
  c->Ny1 = g.ny;
  c->Px = 3 * g.nx / 2;
  c->Pz = 3 * g.nz / 2;
  c->Py = g.ny;
  if (!supported_length(c->Px) || !supported_length(c->Pz))
    return c->fail(DNSMI_EINVAL, "padded lengths must be one of 12,16,24,32,48,64,72,96,128,144,192");
  const int Ny = g.ny, Nkz = c->Nz1, Nkx = c->Nx1, M = Nkz * Nkx;
  c->spec_elems = 3LL * M * Ny;
  WallTables* t = new WallTables();
  c->wt = t;
  t->p = p;
  t->Ny = Ny;
  t->Nkz = Nkz;
  t->Nkx = Nkx;
  t->M = M;
  // forced variants (tile_cols != 0): bit 64 selects the 64-row curl tiles
  t->curl_ty = g.tile_cols != 0 ? ((g.variants & 64) ? 64 : 32) : walls_curl_ty(Ny, M);
  c->curl_rows = t->curl_ty;

  // buffers: WT1 out (6,Ny,Nkz,Nkx) | z-inverse out (6,Ny,Pz,Nkx) | x-pass out
  // (3,Ny,Pz,Nkx) | z-forward out (3,Ny,Nkz,Nkx)
  const size_t cxs = 16;  // FP64-sized in the mixed form too: escalated passes run in FP64
  const size_t a1 = 6ull * Ny * Nkz * Nkx, a3 = 3ull * Ny * c->Pz * Nkx;
  const size_t b2 = 6ull * Ny * c->Pz * Nkx, b4 = 3ull * Ny * Nkz * Nkx;
  c->bufA_bytes = std::max(a1, a3) * cxs;
  c->bufB_bytes = std::max(b2, b4) * cxs;
  c->bufA = c->alloc(c->bufA_bytes);
  c->bufB = c->alloc(c->bufB_bytes);
  c->rhs0 = static_cast<double*>(c->alloc(c->spec_elems * 16));
  c->nref = c->rhs0;
  if (c->split) {
    // n_ref apart from rhs0, which the corrector uses as scratch
    c->nref = static_cast<double*>(c->alloc(c->spec_elems * 16));
    c->uref = static_cast<double*>(c->alloc(c->spec_elems * 16));
    c->xref = static_cast<float*>(c->alloc(6ull * Ny * c->Pz * c->Px * sizeof(float)));
    if (!c->nref || !c->uref || !c->xref) return c->fail(DNSMI_ENOMEM, "device allocation failed");
  }
  c->max_partials = M + 1024;  // the IMM writes one norm partial per mode
  c->partials = static_cast<double*>(c->alloc(sizeof(double) * c->max_partials));
  t->scratch = static_cast<double*>(c->alloc((size_t)V_COUNT * Ny * M * 16));
  if (!c->bufA || !c->bufB || !c->rhs0 || !c->partials || !t->scratch)
    return c->fail(DNSMI_ENOMEM, "device allocation failed");
  int rc = setup_twiddles(c);
  if (rc) return rc;

  const std::vector<double> kx = real_wavenumbers(g.nx, g.lx);
  const std::vector<double> kz = complex_wavenumbers(g.nz, g.lz);
  if ((rc = upload_doubles(c, &c->kx, kx))) return rc;
  if ((rc = upload_doubles(c, &c->kz, kz))) return rc;

  // CGL grid and base flow U = y (flows/plane_couette.py:73-108)
  std::vector<double> y(Ny);
  for (int j = 0; j < Ny; ++j) y[j] = -std::cos((double)j * kPi / (double)(Ny - 1));
  t->h_ys = y;
  // the y grid in the ky slot: the learned guess's coordinate of a point
  if ((rc = upload_doubles(c, &c->ky, y))) return rc;
  std::vector<double> base(3 * Ny, 0.0), cbase(3 * Ny, 0.0), nbase(3 * Ny, 0.0);
  for (int j = 0; j < Ny; ++j) {
    base[j] = y[j];
    cbase[2 * Ny + j] = -1.0;
    nbase[1 * Ny + j] = y[j] * 1.0;
  }
  if ((rc = upload_doubles(c, &c->base, base))) return rc;
  if ((rc = upload_doubles(c, &c->cbase, cbase))) return rc;
  if ((rc = upload_doubles(c, &c->nbase, nbase))) return rc;

  Stencil d1, d2;
  build_stencils(y, p, d1, d2);
  if ((rc = upload_vec(c, &t->d1w, d1.w))) return rc;
  if ((rc = upload_vec(c, &t->d1j0, d1.j0))) return rc;
  auto transposed = [&](const Stencil& d) {
    std::vector<double> w(d.w.size());
    for (int i = 0; i < Ny; ++i)
      for (int k = 0; k < d.width; ++k) w[(size_t)k * Ny + i] = d.w[(size_t)i * d.width + k];
    return w;
  };
  if ((rc = upload_vec(c, &t->d1t, transposed(d1)))) return rc;
  if ((rc = upload_vec(c, &t->d2t, transposed(d2)))) return rc;
  if ((rc = upload_vec(c, &t->d2w, d2.w))) return rc;
  if ((rc = upload_vec(c, &t->d2j0, d2.j0))) return rc;
  if ((rc = upload_vec(c, &t->qw, quadrature_weights(y, g.ly)))) return rc;

  // per-mode IMM tables (geometries/cartesian.py:704-779)
  const int kl = p, ku = p, rows = 3 * p + 1;
  const double dt = g.dt, cc = g.implicitness, nu = 1.0 / g.re;
  // L_k and H_k depend on the mode only through k^2: modes with the same
  // k^2 (bit for bit) share every per-mode table, computed once per class
  // (at the class's first mode, first[u]) and copied to the others
  std::vector<int> umode(M), first;
  std::vector<double> mkx(M), mkz(M), k2u;
  {
    std::unordered_map<uint64_t, int> key;
    for (int iz = 0; iz < Nkz; ++iz)
      for (int ix = 0; ix < Nkx; ++ix) {
        const int m = iz * Nkx + ix;
        const double k2 = kx[ix] * kx[ix] + kz[iz] * kz[iz];
        mkx[m] = kx[ix];
        mkz[m] = kz[iz];
        uint64_t b;
        std::memcpy(&b, &k2, sizeof b);
        const auto it = key.emplace(b, (int)first.size());
        if (it.second) {
          first.push_back(m);
          k2u.push_back(k2);
        }
        umode[m] = it.first->second;
      }
  }
  const int U = (int)first.size();
  t->U = U;
  t->h_umode = umode;
  if ((rc = upload_vec(c, &t->umode, umode))) return rc;
  // the chunk maps of the L_k and H_k solves, one per class (not when the
  // sequential sweeps are requested)
  const bool mx = c->fp32_primary;
  const size_t nf = (size_t)chunk_count(Ny, p, false, mx) * U * map_words(p, false, mx),
               nb = (size_t)chunk_count(Ny, p, true, mx) * U * map_words(p, true, mx);
  const bool maps_fit = nf < (1ull << 28) && nb < (1ull << 28) && Ny <= kChunkNy;
  const bool forced = g.tile_cols != 0;  // the variant bits choose the form
  if (forced && (g.variants & 8) == 0 && !maps_fit)
    return c->fail(DNSMI_EINVAL,
                   "chunk maps exceed 2^28 words or their LDS staging 64 KiB: use the sequential band solve");
  const bool want_maps = maps_fit && !(forced && (g.variants & 8) != 0);
  // on the GPU unless asked for on the host, or a class's band and vectors
  // do not fit the set-up kernels' 64 KiB of LDS (or the classes a grid's
  // y dimension)
  const bool on_gpu = !g.setup_on_host && setup_lds_homog(Ny, rows) <= 65536 && U <= 65535;
  const auto t0 = std::chrono::steady_clock::now();
  if (on_gpu) {
    GpuSetup gs{};
    gs.n = Ny;
    gs.kl = kl;
    gs.ku = ku;
    gs.rows = rows;
    gs.U = U;
    gs.mx = mx;
    gs.W1 = d1.width;
    gs.W2 = d2.width;
    gs.d1w = t->d1w;
    gs.d1j0 = t->d1j0;
    gs.d2w = t->d2w;
    gs.d2j0 = t->d2j0;
    gs.dt = dt;
    gs.cc = cc;
    gs.nu = nu;
    double* k2d = nullptr;
    if ((rc = upload_vec(c, &k2d, k2u))) return rc;
    gs.k2 = k2d;
    gs.band = static_cast<double*>(c->alloc(2ull * U * rows * Ny * sizeof(double)));
    gs.piv = static_cast<int*>(c->alloc(2ull * U * Ny * sizeof(int)));
    gs.flag = static_cast<int*>(c->alloc(2 * sizeof(int)));
    gs.minv = static_cast<double*>(c->alloc(4ull * U * sizeof(double)));
    t->vq = static_cast<double*>(c->alloc(4ull * U * Ny * sizeof(double)));
    t->lk_ab = static_cast<double*>(c->alloc((size_t)Ny * rows * M * sizeof(double)));
    t->hk_ab = static_cast<double*>(c->alloc((size_t)Ny * rows * M * sizeof(double)));
    t->lk_piv = static_cast<int*>(c->alloc((size_t)Ny * M * sizeof(int)));
    t->hk_piv = static_cast<int*>(c->alloc((size_t)Ny * M * sizeof(int)));
    t->minv = static_cast<double*>(c->alloc(4ull * M * sizeof(double)));
    if (!gs.band || !gs.piv || !gs.flag || !gs.minv || !t->vq || !t->lk_ab || !t->hk_ab || !t->lk_piv ||
        !t->hk_piv || !t->minv)
      return c->fail(DNSMI_ENOMEM, "device allocation failed");
    gs.vq = t->vq;
    if (hipMemset(gs.flag, 0, 2 * sizeof(int)) != hipSuccess) return c->fail(DNSMI_EHIP, "memset");
    hipLaunchKernelGGL(k_setup_lu, dim3(U, 2), dim3(64), setup_lds_lu(Ny, rows), nullptr, gs);
    if ((rc = check_launch(c, "setup_lu"))) return rc;
    hipLaunchKernelGGL(k_setup_homog, dim3(U), dim3(64), setup_lds_homog(Ny, rows), nullptr, gs);
    if ((rc = check_launch(c, "setup_homog"))) return rc;
    if (want_maps) {
      for (double** m : {&t->lk_fmap, &t->hk_fmap})
        if (!(*m = static_cast<double*>(c->alloc(nf * sizeof(double)))))
          return c->fail(DNSMI_ENOMEM, "device allocation failed");
      for (double** m : {&t->lk_bmap, &t->hk_bmap})
        if (!(*m = static_cast<double*>(c->alloc(nb * sizeof(double)))))
          return c->fail(DNSMI_ENOMEM, "device allocation failed");
      hipLaunchKernelGGL(k_setup_maps, dim3(std::max(chunk_count(Ny, p, false, mx), chunk_count(Ny, p, true, mx)), U, 4),
                         dim3(64), 0, nullptr, gs, t->lk_fmap, t->lk_bmap, t->hk_fmap, t->hk_bmap);
      if ((rc = check_launch(c, "setup_maps"))) return rc;
    }
    const long long nab = (long long)Ny * rows * M;
    const int sb = (int)std::min<long long>((nab + 255) / 256, 65536);
    hipLaunchKernelGGL(k_setup_scatter, dim3(sb), dim3(256), 0, nullptr, gs, t->umode, M, t->lk_ab,
                       t->hk_ab, t->lk_piv, t->hk_piv, t->minv);
    if ((rc = check_launch(c, "setup_scatter"))) return rc;
    int flag[2] = {0, 0};
    if (hipMemcpy(flag, gs.flag, sizeof flag, hipMemcpyDeviceToHost) != hipSuccess)
      return c->fail(DNSMI_EHIP, "set-up: read flags");
    for (void* q : {(void*)k2d, (void*)gs.band, (void*)gs.piv, (void*)gs.flag, (void*)gs.minv}) c->release(q);
    if (flag[0]) return c->fail(DNSMI_ESINGULAR, "banded LU hit a zero pivot");
    if (flag[1]) return c->fail(DNSMI_EINVAL, "chunk maps: nonzero entry outside the window's tiles");
  } else {
    std::vector<double> lk_ab((size_t)Ny * rows * M), hk_ab((size_t)Ny * rows * M);
    std::vector<int> lk_piv((size_t)Ny * M), hk_piv((size_t)Ny * M);
    std::vector<double> minv(4ull * M), vq((size_t)U * Ny * 4);
    auto copy_mode = [&](int m, int r) {
      for (int j = 0; j < Ny; ++j) {
        for (int q = 0; q < rows; ++q) {
          lk_ab[((size_t)j * rows + q) * M + m] = lk_ab[((size_t)j * rows + q) * M + r];
          hk_ab[((size_t)j * rows + q) * M + m] = hk_ab[((size_t)j * rows + q) * M + r];
        }
        lk_piv[(size_t)j * M + m] = lk_piv[(size_t)j * M + r];
        hk_piv[(size_t)j * M + m] = hk_piv[(size_t)j * M + r];
      }
      for (int q = 0; q < 4; ++q) minv[(size_t)q * M + m] = minv[(size_t)q * M + r];
    };
    for (int m = 0; m < M; ++m) {
      if (first[umode[m]] != m) {
        copy_mode(m, first[umode[m]]);
        continue;
      }
      const double k2 = k2u[umode[m]];
      Band L(Ny, kl, ku), H(Ny, kl, ku);
      for (int i = 0; i < Ny; ++i) {
        for (int j = std::max(0, i - kl); j <= std::min(Ny - 1, i + ku); ++j) {
          const double d2ij = stencil_at(d2, i, j);
          const double lraw = d2ij - (i == j ? k2 : 0.0);
          double lv = lraw;
          if (i == 0) lv = (k2 == 0.0) ? (j == 0 ? 1.0 : 0.0) : stencil_at(d1, 0, j);
          if (i == Ny - 1) lv = stencil_at(d1, Ny - 1, j);
          L.at(i, j) = lv;
          double hv = (i == j ? 1.0 / dt : 0.0) - cc * nu * lraw;
          if (i == 0 || i == Ny - 1) hv = (i == j) ? 1.0 : 0.0;
          H.at(i, j) = hv;
        }
      }
      // D1 rows of the walls are p+1 wide and lie inside the band by
      // construction (one-sided stencils start at the wall).
      if (band_lu(L) != 0 || band_lu(H) != 0)
        return c->fail(DNSMI_ESINGULAR, "banded LU hit a zero pivot");
      std::vector<double> p1(Ny, 0.0), p2(Ny, 0.0);
      p1[0] = 1.0;
      p2[Ny - 1] = 1.0;
      band_solve(L, p1);
      band_solve(L, p2);
      auto d1_apply = [&](const std::vector<double>& v, int i) {
        double s = 0.0;
        for (int k = 0; k < d1.width; ++k) s += d1.w[(size_t)i * d1.width + k] * v[d1.j0[i] + k];
        return s;
      };
      std::vector<double> r1(Ny), r2(Ny);
      for (int i = 0; i < Ny; ++i) {
        r1[i] = -d1_apply(p1, i);
        r2[i] = -d1_apply(p2, i);
      }
      r1[0] = r1[Ny - 1] = r2[0] = r2[Ny - 1] = 0.0;
      band_solve(H, r1);
      band_solve(H, r2);
      std::vector<double> s1 = p1, s2 = p2;
      s1[0] = s1[Ny - 1] = s2[0] = s2[Ny - 1] = 0.0;
      band_solve(H, s1);
      band_solve(H, s2);
      const double M00 = d1_apply(r1, 0), M01 = d1_apply(r2, 0);
      const double M10 = d1_apply(r1, Ny - 1), M11 = d1_apply(r2, Ny - 1);
      double Mi[4];
      if (k2 == 0.0) {
        Mi[0] = Mi[1] = Mi[2] = 0.0;
        Mi[3] = 1.0 / M11;
      } else {
        const double det = M00 * M11 - M01 * M10;
        Mi[0] = M11 / det;
        Mi[1] = -M01 / det;
        Mi[2] = -M10 / det;
        Mi[3] = M00 / det;
      }
      for (int q = 0; q < 4; ++q) minv[(size_t)q * M + m] = Mi[q];
      for (int j = 0; j < Ny; ++j) {
        for (int r = 0; r < rows; ++r) {
          lk_ab[((size_t)j * rows + r) * M + m] = L.raw(r, j);
          hk_ab[((size_t)j * rows + r) * M + m] = H.raw(r, j);
        }
        lk_piv[(size_t)j * M + m] = L.piv[j];
        hk_piv[(size_t)j * M + m] = H.piv[j];
        double* w = &vq[((size_t)umode[m] * Ny + j) * 4];
        w[0] = r1[j];
        w[1] = r2[j];
        w[2] = s1[j];
        w[3] = s2[j];
      }
    }
    if ((rc = upload_vec(c, &t->lk_ab, lk_ab))) return rc;
    if ((rc = upload_vec(c, &t->hk_ab, hk_ab))) return rc;
    if (want_maps) {  // built in parallel on the host threads
      std::vector<double> lf(nf), lb(nb), hf(nf), hb(nb);
      const int nth = (int)std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
      std::vector<char> ok(nth, 1);
      auto work = [&](int w) {
        for (int u = w; u < U; u += nth) {
          const int m = first[u];
          auto lraw = [&](int r, int j) { return lk_ab[((size_t)j * rows + r) * M + m]; };
          auto lpiv = [&](int j) { return lk_piv[(size_t)j * M + m]; };
          auto hraw = [&](int r, int j) { return hk_ab[((size_t)j * rows + r) * M + m]; };
          auto hpiv = [&](int j) { return hk_piv[(size_t)j * M + m]; };
          const bool a = chunk_maps(Ny, p, mx, u, U, lraw, lpiv, lf.data(), lb.data());
          const bool b = chunk_maps(Ny, p, mx, u, U, hraw, hpiv, hf.data(), hb.data());
          if (!a || !b) ok[w] = 0;
        }
      };
      std::vector<std::thread> pool;
      for (int w = 1; w < nth; ++w) pool.emplace_back(work, w);
      work(0);
      for (auto& th : pool) th.join();
      for (char o : ok)
        if (!o) return c->fail(DNSMI_EINVAL, "chunk maps: nonzero entry outside the window's tiles");
      if ((rc = upload_vec(c, &t->lk_fmap, lf))) return rc;
      if ((rc = upload_vec(c, &t->lk_bmap, lb))) return rc;
      if ((rc = upload_vec(c, &t->hk_fmap, hf))) return rc;
      if ((rc = upload_vec(c, &t->hk_bmap, hb))) return rc;
    }
    if ((rc = upload_vec(c, &t->lk_piv, lk_piv))) return rc;
    if ((rc = upload_vec(c, &t->hk_piv, hk_piv))) return rc;
    if ((rc = upload_vec(c, &t->vq, vq))) return rc;
    if ((rc = upload_vec(c, &t->minv, minv))) return rc;
  }
  if (hipDeviceSynchronize() != hipSuccess) return c->fail(DNSMI_EHIP, "set-up: synchronise");
  const double setup_ms =
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  char note[96];
  std::snprintf(note, sizeof note, "imm_setup=%s(%.1f ms) curl_rows=%d ", on_gpu ? "gpu" : "host", setup_ms,
                t->curl_ty);
  if (want_maps) {
    // the chunked solves' items: two modes of one class (one map), the second
    // marked absent (its complement) where a class's count is odd
    std::vector<int> order(M);
    for (int m = 0; m < M; ++m) order[m] = m;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return umode[a] < umode[b]; });
    std::vector<int2> sched;
    for (int i = 0; i < M;) {
      const int m = order[i], u = umode[m];
      const bool two = i + 1 < M && umode[order[i + 1]] == u;
      sched.push_back(make_int2(m, u));
      sched.push_back(make_int2(two ? order[i + 1] : ~m, u));
      i += two ? 2 : 1;
    }
    t->items = (int)(sched.size() / 2);
    if ((rc = upload_vec(c, &t->sched, sched))) return rc;
  }
  if ((rc = upload_vec(c, &t->mkx, mkx))) return rc;
  if ((rc = upload_vec(c, &t->mkz, mkz))) return rc;
  if (!forced && !maps_fit) {  // the autotuner has one form to choose
    c->sweep_seq = true;
    c->tuning = std::string(note) + "band_solve=sequential(chunk maps exceed 2^28 words or 64 KiB LDS) ";
    return DNSMI_OK;
  }
  if (!forced) {
    rc = walls_autotune(c);
    c->tuning = std::string(note) + c->tuning;
    return rc;
  }
  c->tuning = note;
  return DNSMI_OK;
}

void walls_release(Ctx* c) {
  delete c->wt;
  c->wt = nullptr;
}

// ------------------------------------------------------------------ RHS kernels
// WT1: FD curl + transpose.  In: u (3, M, Ny) with M = Nkz*Nkx modes, FP64.
// Out: V (6, Ny, Nkz, Nkx) in T: u_x, u_y, u_z, w_x = D1 u_z - i kz u_y,
// i kz u_x, -D1 u_x (the i kx parts of w_y, w_z are added by the x pass).
// A block handles TY y-points x kTM modes; loads run along y, stores
// along the mode index.  The curl's tiles are taller than the transposes'
// (kTY): each re-reads a halo of S1 rows on either side, so taller tiles
// re-read less but make fewer workgroups (walls_curl_ty chooses).
constexpr int kTY = 16, kTM = 16;

// The curl's tile height: 64 rows where that still gives at least four
// workgroups per CU (128 x 256 x 128: 2032; the RHS 356 against 386 us
// FP64, 211 against 240 us mixed), else 32 (64 x 128 x 64: 252 workgroups
// of 64 rows would leave CUs idle; 64 against 73 us).
inline int walls_curl_ty(int Ny, int M) {
  const long long blocks64 = (long long)((Ny + 63) / 64) * ((M + kTM - 1) / kTM);
  return blocks64 >= 4 * 256 ? 64 : 32;
}

// EM (EvalMode): EV_RECORD also copies u to ucopy (u_ref); EV_INC takes the
// curl of d = u - uref, formed in FP64.
template <typename T, int S1, int EM, int TY>
__global__ void __launch_bounds__(TY* kTM)
    k_walls_curl_t(const cx<double>* __restrict__ u, cx<T>* __restrict__ v,
                   const double* __restrict__ d1w, const int* __restrict__ d1j0,
                   const double* __restrict__ mkz, int Ny, int M, const int* __restrict__ act,
                   const cx<double>* __restrict__ uref, cx<double>* __restrict__ ucopy) {
  if (act && *act == 0) return;
  constexpr int HALO = S1;
  __shared__ cx<double> tile[3][kTM][TY + 2 * HALO + 1];
  const int ntile_y = (Ny + TY - 1) / TY;
  const int y0 = (blockIdx.x % ntile_y) * TY;
  const int m0 = (blockIdx.x / ntile_y) * kTM;
  const int ylo = max(0, y0 - HALO);
  const int yhi = min(Ny, y0 + TY + HALO);
  const int span = yhi - ylo;
  const size_t comp = (size_t)M * Ny;
  // load: lanes along y
  for (int e = threadIdx.x; e < 3 * kTM * span; e += blockDim.x) {
    const int c = e / (kTM * span);
    const int r = e - c * kTM * span;
    const int mi = r / span, yi = r - mi * span;
    const int m = m0 + mi;
    cx<double> val{0, 0};
    if (m < M) {
      const size_t e = c * comp + (size_t)m * Ny + ylo + yi;
      val = u[e];
      if constexpr (EM == EV_RECORD) {
        const int yy = ylo + yi;  // the tile's own rows (not its halo)
        if (yy >= y0 && yy < y0 + TY) ucopy[e] = val;
      }
      if constexpr (EM == EV_INC) {
        const cx<double> r = uref[e];
        val = {val.x - r.x, val.y - r.y};
      }
    }
    tile[c][mi][yi] = val;
  }
  __syncthreads();
  const int mi = threadIdx.x % kTM, yi = threadIdx.x / kTM;
  const int m = m0 + mi, y = y0 + yi;
  if (m >= M || y >= Ny) return;
  const cx<double> ux = tile[0][mi][y - ylo], uy = tile[1][mi][y - ylo], uz = tile[2][mi][y - ylo];
  cx<double> dux{0, 0}, duz{0, 0};
  const int j0 = d1j0[y];
#pragma unroll
  for (int k = 0; k < S1; ++k) {
    const double w = d1w[y * S1 + k];
    const cx<double> a = tile[0][mi][j0 + k - ylo], b = tile[2][mi][j0 + k - ylo];
    dux.x += w * a.x;
    dux.y += w * a.y;
    duz.x += w * b.x;
    duz.y += w * b.y;
  }
  const double k = mkz[m];
  // flows/plane_couette.py:257-271
  const cx<double> wx = {duz.x + k * uy.y, duz.y - k * uy.x};  // dy w - i kz v
  const cx<double> wyp = {-k * ux.y, k * ux.x};                // i kz u
  const cx<double> wzp = {-dux.x, -dux.y};                     // -dy u
  const size_t f = (size_t)Ny * M;
  const size_t o = (size_t)y * M + m;
  v[0 * f + o] = {static_cast<T>(ux.x), static_cast<T>(ux.y)};
  v[1 * f + o] = {static_cast<T>(uy.x), static_cast<T>(uy.y)};
  v[2 * f + o] = {static_cast<T>(uz.x), static_cast<T>(uz.y)};
  v[3 * f + o] = {static_cast<T>(wx.x), static_cast<T>(wx.y)};
  v[4 * f + o] = {static_cast<T>(wyp.x), static_cast<T>(wyp.y)};
  v[5 * f + o] = {static_cast<T>(wzp.x), static_cast<T>(wzp.y)};
}

// z-inverse of NF independent fields: (NF, Ny, Nkz, Nkx) -> (NF, Ny, Pz, Nkx).
template <typename T, int P, int TC, int NF>
__global__ void __launch_bounds__(TC * ColPlan<P>::threads)
    k_z_inverse_plain(const cx<T>* __restrict__ in, cx<T>* __restrict__ out,
                      const cx<T>* __restrict__ tw, int nz, int Ny, int Nx1,
                      const int* __restrict__ act) {
  if (act && *act == 0) return;
  constexpr int N1 = ColPlan<P>::N1, N2 = ColPlan<P>::N2;
  __shared__ cx<T> lds[TC * P];
  __shared__ cx<T> tws[P];
  for (int i = threadIdx.x; i < P; i += blockDim.x) tws[i] = tw[i];
  __syncthreads();
  const int tid = threadIdx.x, col = tid % TC, j_ = tid / TC;
  const int ntile = (Nx1 + TC - 1) / TC;
  const int y = blockIdx.x / ntile;
  const int kx = (blockIdx.x - y * ntile) * TC + col;
  const bool ok = kx < Nx1;
  const int Nz1 = nz - 1;
  const size_t in_f = (size_t)Ny * Nz1 * Nx1;
  const size_t in_off = (size_t)y * Nz1 * Nx1 + kx;
  const size_t out_f = (size_t)Ny * P * Nx1;
  const size_t out_off = (size_t)y * P * Nx1 + kx;
#pragma unroll 1
  for (int f = blockIdx.y; f < NF; f += gridDim.y) {  // one field per workgroup row
    const int j = opaque(j_);
    if (j < N2) {
      cx<T> x[N1];
#pragma unroll
      for (int a = 0; a < N1; ++a) {
        const int s = Pad<P>::stored_in(N2 * a, N2, j);
        x[a] = (ok && s >= 0) ? in[f * in_f + in_off + (size_t)s * Nx1] : cx<T>{0, 0};
      }
      step_a_store<P, N1, N2, +1, TC>(x, j, col, lds, tws);
    }
    __syncthreads();
    if (j < N1 && ok) {
      cx<T> o[N2];
      step_b_load<P, N1, N2, +1, TC>(o, j, col, lds);
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) out[f * out_f + out_off + (size_t)(j + N1 * k2) * Nx1] = o[k2];
    }
    __syncthreads();
  }
}

// WT5: (3, Ny, Nkz, Nkx) T -> rhs (3, M, Ny) FP64, tiled transpose; with
// nref (split evaluations) rhs = nref + the transformed increment; with
// nref_out (a recording evaluation) rhs is also copied there.
template <typename T>
__global__ void __launch_bounds__(kTY* kTM)
    k_walls_to_spec(const cx<T>* __restrict__ w, cx<double>* __restrict__ rhs, int Ny, int M,
                    const int* __restrict__ act, const cx<double>* __restrict__ nref,
                    cx<double>* __restrict__ nref_out) {
  if (act && *act == 0) return;
  __shared__ cx<double> tile[kTY][kTM + 1];
  const int ntile_y = (Ny + kTY - 1) / kTY;
  const int c = blockIdx.y;
  const int y0 = (blockIdx.x % ntile_y) * kTY;
  const int m0 = (blockIdx.x / ntile_y) * kTM;
  const size_t f = (size_t)Ny * M;
  {
    const int mi = threadIdx.x % kTM, yi = threadIdx.x / kTM;
    const int m = m0 + mi, y = y0 + yi;
    if (m < M && y < Ny) {
      const cx<T> v = w[c * f + (size_t)y * M + m];
      tile[yi][mi] = {static_cast<double>(v.x), static_cast<double>(v.y)};
    }
  }
  __syncthreads();
  const int yi = threadIdx.x % kTY, mi = threadIdx.x / kTY;
  const int m = m0 + mi, y = y0 + yi;
  if (m < M && y < Ny) {
    const size_t e = c * f + (size_t)m * Ny + y;
    cx<double> r = tile[yi][mi];
    if (nref) r = {nref[e].x + r.x, nref[e].y + r.y};
    rhs[e] = r;
    if (nref_out) nref_out[e] = r;
  }
}

// ------------------------------------------------------------------ IMM kernel
struct ImmArgs {
  const cx<double>* un;   // velocity_n (3, M, Ny)
  const cx<double>* uj;   // velocity_j
  const cx<double>* nn;   // nonlin_n
  const cx<double>* nj;   // nonlin_j
  cx<double>* out;        // velocity_new (may alias un or uj)
  cx<double>* corr;       // correction (may be null)
  double* partials;       // per-block sum of quadrature-weighted k_metric |delta|^2
  const double *d1w, *d2w, *qw;  // stencil weights as [k][y]
  const double *lk_ab, *hk_ab;
  const int *lk_piv, *hk_piv;
  const double* vq;    // [map][y][4]: v1, v2, q1, q2
  const int* umode;    // per mode: its map
  const double *minv, *mkx, *mkz;
  cx<double>* scratch;  // work vectors [vec][mode][y]
  const int* act;       // if set and 0: the launch is skipped
  int Ny, M, Nkx;
  double dt, c, nu;
};

// The influence-matrix step in five phases.  The right-hand sides of the
// banded systems are generated in parallel over (mode, y) (one workgroup
// per mode, lanes along y: the fields' rows are contiguous in y), the
// sequential band sweeps run one thread per (mode, right-hand side) on
// precomputed rows with their loads issued a batch of rows ahead of the
// recurrence, and the assembly is parallel again.  Work vectors are
// [vec][mode][y]; per mode the arithmetic is the one-thread-per-mode
// formulation's, operation for operation.

// Work vector v, mode m: element y at [y * VS] from the returned pointer.
// The rows are contiguous in y (VS = 1): the parallel phases' lanes run
// along y; a sweep lane walks its own row.
constexpr int VS = 1;
__device__ __forceinline__ cx<double>* svec(const ImmArgs& a, int v, int m) {
  return a.scratch + ((size_t)v * a.M + m) * a.Ny;
}
__device__ __forceinline__ cx<double> ikm(double k, cx<double> z) { return {-k * z.y, k * z.x}; }

// D1 (S = p + 1 points) / D2 (S = p + 2) stencils: row y's weights, and their
// sum over a row r (global or LDS) whose element y is at r[y * stride].  The
// first point is build_stencils' j0, computed: a load of it would stand
// before every stencil's reads.
template <int S>
struct Weights {
  double w[S];
  int j0;
  __device__ __forceinline__ Weights() {}
  __device__ __forceinline__ Weights(const double* t, int Ny, int y) {
    j0 = max(0, min(y - S / 2, Ny - S));
#pragma unroll
    for (int k = 0; k < S; ++k) w[k] = t[(size_t)k * Ny + y];
  }
  __device__ __forceinline__ cx<double> operator()(const cx<double>* r, size_t stride = 1) const {
    cx<double> s{0, 0};
#pragma unroll
    for (int k = 0; k < S; ++k) {
      const cx<double> v = r[(j0 + k) * stride];
      s.x += w[k] * v.x;
      s.y += w[k] * v.y;
    }
    return s;
  }
};

// Per-row arithmetic of the parallel phases, shared by the five-launch
// form and the fused form (so both compute the same values, bit for bit).
// `row` = m Ny, `comp` = M Ny; the rows the stencils read are in LDS.

// c N_j + (1 - c) N_n at element e of a field (phases 1 and 3).
__device__ __forceinline__ cx<double> imm_n_at(const ImmArgs& a, size_t e) {
  const cx<double> j = a.nj[e], n = a.nn[e];
  const double g = 1.0 - a.c;
  return {__builtin_fma(a.c, j.x, g * n.x), __builtin_fma(a.c, j.y, g * n.y)};
}

// d_hat^n at row y (phase 1): i kx u_x + D1 u_y + i kz u_z; un1 = u^n_y's
// row, ux and uz the other components there.
template <int PO>
__device__ __forceinline__ cx<double> imm_dhat_at(const Weights<PO + 1>& d1, const cx<double>* un1, cx<double> ux,
                                                  cx<double> uz, double kx, double kz) {
  const cx<double> dv = d1(un1);
  const cx<double> t0 = ikm(kx, ux), t2 = ikm(kz, uz);
  return {(t0.x + dv.x) + t2.x, (t0.y + dv.y) + t2.y};
}

// f_hat at row y (phase 1), zero on the walls; dh = d_hat^n's row, nc1 the
// y row of c N_j + (1 - c) N_n, ncx and ncz its other components at y.
template <int PO>
__device__ __forceinline__ cx<double> imm_fhat_at(const ImmArgs& a, const Weights<PO + 1>& d1,
                                                  const Weights<PO + 2>& d2, const cx<double>* dh,
                                                  const cx<double>* nc1, cx<double> ncx, cx<double> ncz, double kx,
                                                  double kz, double k2, int y) {
  const bool wall = y <= 0 || y >= a.Ny - 1;
  const double idt = 1.0 / a.dt, g = (1 - a.c) * a.nu;
  const cx<double> d = dh[y];
  const cx<double> dv = d1(nc1);
  const cx<double> t0 = ikm(kx, ncx), t2 = ikm(kz, ncz);
  const cx<double> dn = {(t0.x + dv.x) + t2.x, (t0.y + dv.y) + t2.y};
  const cx<double> d2d = d2(dh);
  const cx<double> lkd = {d2d.x - k2 * d.x, d2d.y - k2 * d.y};
  return wall ? cx<double>{0, 0} : cx<double>{(idt * d.x + dn.x) + g * lkd.x, (idt * d.y + dn.y) + g * lkd.y};
}

// A mixed context's f_hat at row y: N_j's and N_n's divergences apart and
// combined last, d / dt a division.  nj1 and nn1 are the y rows of N_j and
// N_n, n = {N_j x, N_j z, N_n x, N_n z} at y.
template <int PO>
__device__ __forceinline__ cx<double> imm_fhat_mx_at(const ImmArgs& a, const Weights<PO + 1>& d1,
                                                     const Weights<PO + 2>& d2, const cx<double>* dh,
                                                     const cx<double>* nj1, const cx<double>* nn1,
                                                     const cx<double> (&n)[4], double kx, double kz, double k2,
                                                     int y) {
  const bool wall = y <= 0 || y >= a.Ny - 1;
  const double dt = a.dt, cc = a.c, g = (1 - a.c) * a.nu;
  const cx<double> d = dh[y];
  const cx<double> dvj = d1(nj1), dvn = d1(nn1);
  const cx<double> aj = ikm(kx, n[0]), cj = ikm(kz, n[1]), an = ikm(kx, n[2]), cn = ikm(kz, n[3]);
  const cx<double> divj = {(aj.x + dvj.x) + cj.x, (aj.y + dvj.y) + cj.y};
  const cx<double> divn = {(an.x + dvn.x) + cn.x, (an.y + dvn.y) + cn.y};
  const cx<double> d2d = d2(dh);
  const cx<double> lkd = {d2d.x - k2 * d.x, d2d.y - k2 * d.y};
  return wall ? cx<double>{0, 0}
              : cx<double>{((d.x / dt + cc * divj.x) + (1 - cc) * divn.x) + g * lkd.x,
                           ((d.y / dt + cc * divj.y) + (1 - cc) * divn.y) + g * lkd.y};
}

// R_c at row y for the three components (phase 3), zero on the walls; pp =
// the p_P row, ur = the rows of u^n (component c at ur + c ld); nc = c N_j +
// (1 - c) N_n at y, or in a mixed context (MX) N_j there and nn = N_n, added
// one by one.
template <int PO, bool MX>
__device__ __forceinline__ void imm_r_at(const ImmArgs& a, const Weights<PO + 1>& d1, const Weights<PO + 2>& d2,
                                         const cx<double>* pp, const cx<double>* ur, int ld,
                                         const cx<double> (&nc)[3], const cx<double> (&nn)[3], double kx, double kz,
                                         double k2, int y, cx<double> (&r)[3]) {
  const bool wall = y <= 0 || y >= a.Ny - 1;
  const double idt = 1.0 / a.dt, g = (1.0 - a.c) * a.nu;
  const cx<double> p = pp[y];
  const cx<double> dpp[3] = {ikm(kx, p), d1(pp), ikm(kz, p)};
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const cx<double>* unc = ur + c * ld;
    const cx<double> u = unc[y];
    const cx<double> du = d2(unc);
    const cx<double> l = {du.x - k2 * u.x, du.y - k2 * u.y};
    const cx<double> hm = {idt * u.x + g * l.x, idt * u.y + g * l.y};
    if constexpr (MX)
      r[c] = {((hm.x - dpp[c].x) + a.c * nc[c].x) + (1 - a.c) * nn[c].x,
              ((hm.y - dpp[c].y) + a.c * nc[c].y) + (1 - a.c) * nn[c].y};
    else
      r[c] = {(hm.x - dpp[c].x) + nc[c].x, (hm.y - dpp[c].y) + nc[c].y};
    if (wall) r[c] = {0, 0};
  }
}

// alpha = -M^-1 (wall divergence of v_arb) with the k^2 = 0 gauge (phase 5);
// va = v_arb's row (element y at va[y * vs]).
template <int PO>
__device__ __forceinline__ void imm_alpha(const ImmArgs& a, int m, const cx<double>* va, size_t vs,
                                          cx<double>& al1, cx<double>& al2) {
  const int Ny = a.Ny;
  const size_t M = a.M;
  const double kx = a.mkx[m], kz = a.mkz[m];
  cx<double> dw0 = Weights<PO + 1>(a.d1w, Ny, 0)(va, vs), dw1 = Weights<PO + 1>(a.d1w, Ny, Ny - 1)(va, vs);
  if (kx * kx + kz * kz == 0.0) dw0 = {0, 0};
  const double m00 = a.minv[0 * M + m], m01 = a.minv[1 * M + m];
  const double m10 = a.minv[2 * M + m], m11 = a.minv[3 * M + m];
  al1 = {-(m00 * dw0.x + m01 * dw1.x), -(m00 * dw0.y + m01 * dw1.y)};
  al2 = {-(m10 * dw0.x + m11 * dw1.x), -(m10 * dw0.y + m11 * dw1.y)};
}

// Row y of the assembly (phase 5): the corrected velocity into out (and the
// correction into corr); returns k_metric |delta|^2 of the row (before its
// quadrature weight).  ua, va, wa: v_arb's rows (stride vs).
__device__ __forceinline__ double imm_assemble_at(const ImmArgs& a, int m, size_t row, size_t comp, double kx,
                                                  double kz, double4 w, const cx<double> (&uj)[3],
                                                  const cx<double>* ua, const cx<double>* va,
                                                  const cx<double>* wa, size_t vs, cx<double> al1,
                                                  cx<double> al2, int y) {
  const double km = (m % a.Nkx == 0) ? 1.0 : 2.0;
  const double v1 = w.x, v2 = w.y, q1 = w.z, q2 = w.w;
  const cx<double> vv = va[(size_t)y * vs];
  const cx<double> vn = {(vv.x + al1.x * v1) + al2.x * v2, (vv.y + al1.y * v1) + al2.y * v2};
  const cx<double> q = {al1.x * q1 + al2.x * q2, al1.y * q1 + al2.y * q2};
  const cx<double> uu = ua[(size_t)y * vs], ww = wa[(size_t)y * vs];
  const cx<double> iq_x = ikm(kx, q), iq_z = ikm(kz, q);
  const cx<double> nw[3] = {{uu.x - iq_x.x, uu.y - iq_x.y}, vn, {ww.x - iq_z.x, ww.y - iq_z.y}};
  double s = 0.0;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const size_t idx = c * comp + row + y;
    const cx<double> d = {nw[c].x - uj[c].x, nw[c].y - uj[c].y};
    a.out[idx] = nw[c];
    if (a.corr) a.corr[idx] = d;
    s += km * (d.x * d.x) + km * (d.y * d.y);
  }
  return s;
}

// Phase 1 (flows/plane_couette.py:427-445): d_hat^n into LDS, then f_hat
// (zero on the walls) -> V_F.
template <int PO, bool MX>
__global__ void __launch_bounds__(kImmT) k_imm_fhat(ImmArgs a) {
  if (a.act && *a.act == 0) return;
  // LDS: d_hat, then the y rows of u^n and c N_j + (1 - c) N_n, or N_j and
  // N_n (the D1 stencils' operands, read once from HBM)
  extern __shared__ cx<double> dh[];
  const int m = blockIdx.x, Ny = a.Ny;
  const size_t comp = (size_t)a.M * Ny, row = (size_t)m * Ny;
  const double kx = a.mkx[m], kz = a.mkz[m];
  const double k2 = kx * kx + kz * kz;
  cx<double>* un1 = dh + Ny;
  cx<double>* nc1 = dh + 2 * Ny;
  [[maybe_unused]] cx<double>* nn1 = dh + 3 * Ny;
  for (int y = threadIdx.x; y < Ny; y += blockDim.x) {
    un1[y] = a.un[comp + row + y];
    if constexpr (MX) {
      nc1[y] = a.nj[comp + row + y];
      nn1[y] = a.nn[comp + row + y];
    } else {
      nc1[y] = imm_n_at(a, comp + row + y);
    }
  }
  __syncthreads();
  for (int y = threadIdx.x; y < Ny; y += blockDim.x)
    dh[y] = imm_dhat_at<PO>(Weights<PO + 1>(a.d1w, Ny, y), un1, a.un[row + y], a.un[2 * comp + row + y], kx, kz);
  __syncthreads();
  cx<double>* f = svec(a, V_F, m);
  for (int y = threadIdx.x; y < Ny; y += blockDim.x) {
    const Weights<PO + 1> d1(a.d1w, Ny, y);
    const Weights<PO + 2> d2(a.d2w, Ny, y);
    if constexpr (MX) {
      const cx<double> n[4] = {a.nj[row + y], a.nj[2 * comp + row + y], a.nn[row + y], a.nn[2 * comp + row + y]};
      f[y * VS] = imm_fhat_mx_at<PO>(a, d1, d2, dh, nc1, nn1, n, kx, kz, k2, y);
    } else {
      f[y * VS] = imm_fhat_at<PO>(a, d1, d2, dh, nc1, imm_n_at(a, row + y), imm_n_at(a, 2 * comp + row + y), kx, kz,
                                  k2, y);
    }
  }
}

// Phases 2 and 4: solve ab x = rhs per (mode, right-hand side r =
// blockIdx.y) with the LU factors and pivots in LAPACK band layout
// (mode-fastest).  Forward sweep rhs vector vin + r -> vtmp + r, back
// substitution -> vout + r.  Loads of U rows are issued before their
// recurrence steps.
template <int PO>
struct SweepBatch {
  static constexpr int value = PO <= 2 ? 32 : (PO <= 4 ? 16 : 8);
};

// Lanes per sweep workgroup (one wave; 16-lane workgroups over 4x the CUs
// measured slower: a sweep is bound by its chain of batch latencies).
constexpr int kSweepLanes = 64;

template <int PO>
__global__ void __launch_bounds__(kSweepLanes)
    k_band_sweeps(ImmArgs a, const double* __restrict__ ab, const int* __restrict__ piv, int vin,
                  int vtmp, int vout) {
  if (a.act && *a.act == 0) return;
  constexpr int KL = PO, KU = PO, KUU = 2 * PO, ROWS = 3 * PO + 1, U = SweepBatch<PO>::value;
  const int m = blockIdx.x * kSweepLanes + threadIdx.x;
  if (m >= a.M) return;
  const int r = blockIdx.y, Ny = a.Ny, M = a.M;
  // rin and out may be the same vector (the H sweeps solve in place): the
  // forward sweep only reads rin and writes tmp, the back substitution only
  // reads tmp and writes out, so each sweep's pointers are restrict within
  // its own scope (a batch's loads need not wait for the previous stores).
  {
    const cx<double>* __restrict__ rin = svec(a, vin + r, m);
    cx<double>* __restrict__ tmp = svec(a, vtmp + r, m);
    cx<double> w[KL + 1];
#pragma unroll
    for (int i = 0; i <= KL; ++i) w[i] = (i < Ny) ? rin[(size_t)i * VS] : cx<double>{0, 0};
    for (int j0 = 0; j0 < Ny - 1; j0 += U) {
      int dd[U];
      double L[U][KL];
      cx<double> nf[U];
      // Loads from clamped (always valid) rows with no branches, so that the
      // whole batch is in flight at once; the guards apply at use.
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = j0 + u;
        const int jj = j < Ny - 2 ? j : Ny - 2;
        dd[u] = piv[(size_t)jj * M + m] - j;
        const double* col = ab + (size_t)jj * ROWS * M + m;
#pragma unroll
        for (int i = 1; i <= KL; ++i) L[u][i - 1] = col[(size_t)(KL + KU + i) * M];
        const int jf = j + KL + 1 < Ny ? j + KL + 1 : Ny - 1;
        nf[u] = rin[(size_t)jf * VS];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = j0 + u;
        if (j < Ny - 1) {
          const cx<double> w0 = w[0];
#pragma unroll
          for (int i = 1; i <= KL; ++i)
            if (dd[u] == i) {
              w[0] = w[i];
              w[i] = w0;
            }
#pragma unroll
          for (int i = 1; i <= KL; ++i) {
            if (j + i < Ny) {
              const double l = L[u][i - 1];
              w[i].x -= l * w[0].x;
              w[i].y -= l * w[0].y;
            }
          }
          tmp[(size_t)j * VS] = w[0];
#pragma unroll
          for (int i = 0; i < KL; ++i) w[i] = w[i + 1];
          w[KL] = (j + KL + 1 < Ny) ? nf[u] : cx<double>{0, 0};
        }
      }
    }
    tmp[(size_t)(Ny - 1) * VS] = w[0];
  }
  {
    const cx<double>* __restrict__ tmp = svec(a, vtmp + r, m);
    cx<double>* __restrict__ out = svec(a, vout + r, m);
    cx<double> z[KUU + 1];
#pragma unroll
    for (int i = 0; i <= KUU; ++i) z[KUU - i] = (Ny - 1 - i >= 0) ? tmp[(size_t)(Ny - 1 - i) * VS] : cx<double>{0, 0};
    for (int j0 = Ny - 1; j0 >= 0; j0 -= U) {
      double dg[U], Uv[U][KUU];
      cx<double> nz[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = j0 - u;
        const double* col = ab + (size_t)(j > 0 ? j : 0) * ROWS * M + m;
        dg[u] = col[(size_t)(KL + KU) * M];
#pragma unroll
        for (int i = 1; i <= KUU; ++i) Uv[u][i - 1] = col[(size_t)(KUU - i) * M];
        nz[u] = tmp[(size_t)(j - KUU - 1 > 0 ? j - KUU - 1 : 0) * VS];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = j0 - u;
        if (j >= 0) {
          const cx<double> x = {z[KUU].x / dg[u], z[KUU].y / dg[u]};
          out[(size_t)j * VS] = x;
#pragma unroll
          for (int i = 1; i <= KUU; ++i) {
            if (j - i >= 0) {
              const double uu = Uv[u][i - 1];
              z[KUU - i].x -= uu * x.x;
              z[KUU - i].y -= uu * x.y;
            }
          }
#pragma unroll
          for (int i = KUU; i > 0; --i) z[i] = z[i - 1];
          z[0] = (j - KUU - 1 >= 0) ? nz[u] : cx<double>{0, 0};
        }
      }
    }
  }
}

// Phases 2 and 4, chunked form: the same solves through the precomputed
// chunk maps (chunk_maps), on the FP64 matrix cores.  A wavefront takes two
// modes of one k^2 class: its right-hand sides, real and imaginary parts
// apart, are the columns of a matrix (4 of 16 for L_k, 12 of 16 for H_k), and
// a chunk is (map) x (window) in 16-row tiles of v_mfma_f64_16x16x4_f64.  Lane
// (g = lane / 16, col = lane % 16) holds rows 4 i + g of a tile's result and
// row 4 q + g of its k step q: a result is the next chunk's operand as it
// stands, the rows that stay in the window moving by whole registers, so the
// chain over the chunks never leaves the registers.  Rows entering the window
// come from the LDS rows the solve works in (in place: a chunk's results
// overwrite rows that have left the window), and results go back there, off
// the chain.
//
// Bound, with the maps in a cache near by: the products, 27 ns each and one per
// SIMD at a time, 128 + 156 of them for a solve at Ny = 256, p = 6 (7.6 us; in
// the whole step the maps' way there sets the pace, k_imm_fused), where broadcasting the window to
// one lane per map row through LDS took 50 FMA steps behind 150 LDS reads per
// 16 rows (1.5 us).  Windows of 16 rows (12 to 8 new ones each) take fewer
// products per row than two-tile ones of 16 new rows (p = 4: 0.83 against
// 1.25), and operands in load order cost the vector memory path a quarter of
// what gathering them from packed columns did (25 cycles per load on each CU,
// four solving wavefronts: 1000 to 1400 cycles per 16 rows, more loads in
// flight only made it worse).
typedef double wd4 __attribute__((ext_vector_type(4)));

// The LDS rows of a solve belong to one wavefront, whose LDS operations
// complete in issue order.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// LDS vectors of a solve: Ny rows each between zero rows, so that a window
// that reaches past either end reads zeros without a test: as many as the last
// chunk's window has behind its direction's end, the next vector's first ones
// serving the one before.  Vector v starts at v ld + pad; ld = 4 mod 16 keeps
// the columns of a wavefront's reads (four rows of each) on different banks.
__host__ __device__ inline int chunk_pad(int Ny, int p, bool mx) {
  const int f = chunk_span(p, false, mx) - 1 - (Ny - 1) % chunk_rows(p, false, mx);
  const int b = chunk_span(p, true, mx) - 1 - (Ny - 1) % chunk_rows(p, true, mx);
  return f > b ? f : b;
}
__host__ __device__ inline int chunk_ld(int Ny, int p, bool mx) { return (Ny + chunk_pad(Ny, p, mx) + 11) / 16 * 16 + 4; }
__host__ __device__ inline int chunk_lds(int Ny, int p, bool mx, int vectors) {
  return vectors * chunk_ld(Ny, p, mx) + chunk_pad(Ny, p, mx);
}
// Zeros over all rows that are no vector's.
__device__ __forceinline__ void chunk_zero(cx<double>* lds, int Ny, int p, bool mx, int vectors) {
  const int pad = chunk_pad(Ny, p, mx), ld = chunk_ld(Ny, p, mx), gap = ld - Ny;
  for (int v = 0; v < vectors; ++v)
    for (int i = threadIdx.x; i < gap; i += blockDim.x) {
      const int row = v * ld + (i < pad ? i : Ny + i);
      lds[row] = cx<double>{0, 0};
    }
  for (int i = threadIdx.x; i < pad; i += blockDim.x) lds[vectors * ld + i] = cx<double>{0, 0};
}

// Chunk c's operands e, e + 1 of this lane (chunks past the last repeat it).
struct MapChunk {
  const double2* p;
  __device__ __forceinline__ MapChunk(const double* __restrict__ map, int U, int u, int words, int c, int nC, int lane)
      : p(reinterpret_cast<const double2*>(map + ((size_t)(c < nC ? c : nC - 1) * U + u) * words) + lane) {}
  __device__ __forceinline__ double2 operator()(int pair) const { return p[pair * 64]; }
};

// Chunks of maps in registers, loaded that many less one ahead: eight words a
// lane each in one-tile windows, 16 to 24 in two-tile ones.
template <int PO, bool BACK, bool MX>
struct ChunkMaps {
  static constexpr int R = chunk_tiles(PO, BACK, MX) == 1 ? 4 : 3, N = map_operands(PO, BACK, MX);
  double f[R][N];
  // the first R - 1 chunks'
  __device__ __forceinline__ void start(const double* __restrict__ map, int U, int u, int lane, int Ny) {
#pragma unroll
    for (int q = 0; q < R - 1; ++q) {
      const MapChunk m(map, U, u, map_words(PO, BACK, MX), q, chunk_count(Ny, PO, BACK, MX), lane);
#pragma unroll
      for (int e = 0; e < N / 2; ++e) {
        const double2 v = m(e);
        f[q][2 * e] = v.x;
        f[q][2 * e + 1] = v.y;
      }
    }
  }
};

// The chunks of one direction.  Window position t <-> row o + s t (o the
// chunk's first row, s = 1 forward, -1 back), the last KEEP rows stay in the
// window from one chunk to the next.  pc: the lane's column (element y at
// pc[2 y]: one part of a complex row); lanes past the columns repeat one, and
// store its values again.  Window rows are read one chunk ahead, a chunk's
// results stored one behind.
//
// The k steps of rows that were in LDS come first in each sum, those of the
// rows kept from the chunk before last, and a second tile (whose rows are the
// kept ones) before the first: a result's latency passes behind products that
// do not need it.  Behind each product (64 cycles of the matrix core) stands
// its share of the loads and stores, pinned there: in front of the products
// they cost half as much again.  A mixed context's k steps are in ascending
// order (chunk_tiles).
template <int PO, bool BACK, bool MX>
__device__ __forceinline__ void chunk_chain(const double* __restrict__ map, int U, int u, int lane, int Ny, double* pc,
                                            ChunkMaps<PO, BACK, MX>& maps) {
  constexpr int TILES = chunk_tiles(PO, BACK, MX), B = chunk_rows(PO, BACK, MX), KEEP = chunk_keep(PO, BACK);
  constexpr int R = ChunkMaps<PO, BACK, MX>::R, N = ChunkMaps<PO, BACK, MX>::N;
  constexpr int NH = high_operands(PO, BACK, MX), NL = low_operands(PO, BACK, MX);
  constexpr int WR = chunk_span(PO, BACK, MX) / 4, KR = (KEEP + 3) / 4, BR = B / 4, S = BACK ? -1 : 1;
  static_assert(KR + BR == WR, "kept and new rows fill the window's registers");
  static_assert(NH <= WR && NL <= WR && BR <= NH + NL && N / 2 <= NH + NL, "each product's operand, load and store");
  const int g = lane >> 4, nC = chunk_count(Ny, PO, BACK, MX);
  double* pg = pc + 2 * ((BACK ? Ny - 1 : 0) + S * g);  // this lane group's row of the first chunk
  double w[WR], done[BR];                               // the window; chunk c - 1's results
#pragma unroll
  for (int i = 0; i < WR; ++i) w[i] = pg[2 * S * 4 * i];
#pragma unroll
  for (int i = 0; i < BR; ++i) done[i] = 0.0;
  auto step = [&](int c, double(&fc)[N], double(&pf)[N]) {
    const MapChunk m(map, U, u, map_words(PO, BACK, MX), c + R - 1, nC, lane);
    // (the last chunk asks for its own rows again; chunk 0 stores zeros over
    // rows that the window holds and chunk 1 stores)
    double* in = pg + 2 * S * min(c + 1, nC - 1) * B;
    double* out = pg + 2 * S * max(c - 1, 0) * B;
    double fresh[WR];
    wd4 acc[TILES];
#pragma unroll
    for (int i = 0; i < TILES; ++i) acc[i] = wd4{0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < NH + NL; ++e) {
      // product e: tile, k step q, operand of the map
      const int tile = e < NH ? 1 : 0, K = tile ? NH : NL, i = tile ? e : e - NH;
      const int kr = !MX && KR < K ? KR : 0, q = i < K - kr ? kr + i : i - (K - kr);
      acc[tile] = __builtin_amdgcn_mfma_f64_16x16x4f64(fc[tile ? q : NH + q], w[q], acc[tile], 0, 0, 0);
      if (e < N / 2) {
        const double2 v = m(e);
        pf[2 * e] = v.x;
        pf[2 * e + 1] = v.y;
      }
      if (e < BR) out[2 * S * 4 * e] = done[e < BR ? e : 0];
      if (KR + e < WR) fresh[KR + e < WR ? KR + e : 0] = in[2 * S * 4 * (KR + e)];
      if (e == 0 && KEEP % 4 != 0) fresh[KR - 1] = in[2 * S * 4 * (KR - 1)];
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (MX && BACK) {  // rows and columns >= 16: the identity
#pragma unroll
      for (int i = 0; i < KR; ++i) acc[1][i] += w[BR + i];
    }
#pragma unroll
    for (int i = 0; i < BR; ++i) done[i] = acc[i >> 2][i & 3];
#pragma unroll
    for (int i = 0; i < WR; ++i) {
      const int o = i + BR < WR ? i + BR : 0;
      const double kept = acc[o >> 2][o & 3];
      w[i] = 4 * i + 4 <= KEEP ? kept : 4 * i >= KEEP ? fresh[i] : (4 * i + g < KEEP ? kept : fresh[i]);
    }
  };
  int c = 0;
  for (; c + R <= nC; c += R) {
#pragma unroll
    for (int q = 0; q < R; ++q) step(c + q, maps.f[q], maps.f[(q + R - 1) % R]);
  }
#pragma unroll
  for (int q = 0; q < R - 1; ++q)
    if (c + q < nC) step(c + q, maps.f[q], maps.f[(q + R - 1) % R]);
#pragma unroll
  for (int i = 0; i < BR; ++i)
    if ((nC - 1) * B + 4 * i + g < Ny) pg[2 * S * ((nC - 1) * B + 4 * i)] = done[i];
}

// Band solve of this wavefront's columns, in place; maps: the forward maps,
// started.
template <int PO, bool MX>
__device__ __forceinline__ void chunk_solve(const double* __restrict__ fmap, const double* __restrict__ bmap, int U,
                                            int u, int lane, int Ny, double* pc, ChunkMaps<PO, false, MX>& maps) {
  ChunkMaps<PO, true, MX> back;
  back.start(bmap, U, u, lane, Ny);
  wave_sync();
  chunk_chain<PO, false, MX>(fmap, U, u, lane, Ny, pc, maps);
  wave_sync();
  chunk_chain<PO, true, MX>(bmap, U, u, lane, Ny, pc, back);
  wave_sync();
}

// A launch's workgroups go to the 8 XCDs (each with its own L2) in turn:
// renumbered so that each XCD takes one contiguous range of items, where
// neighbouring modes (grouped by k^2) share chunk-map cache lines.
__device__ __forceinline__ int xcd_block(int b, int G) {
  constexpr int X = 8;
  const int q = G / X, r = G % X, x = b % X, i = b / X;
  return x * q + (x < r ? x : r) + i;
}

// The lane's column of a solve with NR right-hand sides per mode: modes at
// sh + half hs, right-hand sides ld apart, real and imaginary part.
template <int NR>
__device__ __forceinline__ double* chunk_column(cx<double>* sh, int hs, int ld, int lane) {
  const int v = min((lane & 15) >> 1, 2 * NR - 1);
  return reinterpret_cast<double*>(sh + (v / NR) * hs + (v % NR) * ld) + (lane & 1);
}

// The item's two modes come as (mode, map), the second (a class with an odd
// count) perhaps marked absent: then it repeats the first and stores nothing.
__device__ __forceinline__ int2 sched_mode(const int2* __restrict__ sched, int slot, bool& live) {
  int2 mu = sched[slot];
  live = mu.x >= 0;
  if (!live) mu.x = ~mu.x;
  return mu;
}

template <int PO, int NR, bool MX>
__global__ void __launch_bounds__(64, 2)
    k_band_chunks(ImmArgs a, const double* __restrict__ fmap, const double* __restrict__ bmap,
                  const int2* __restrict__ sched, int U, int vin, int vout) {
  if (a.act && *a.act == 0) return;
  extern __shared__ cx<double> lds[];  // chunk_lds(Ny, PO, MX, 2 NR): [2][NR][ld]
  const int Ny = a.Ny, M = a.M, ld = chunk_ld(Ny, PO, MX), lane = threadIdx.x;
  cx<double>* sh = lds + chunk_pad(Ny, PO, MX);
  const int item = xcd_block(blockIdx.x, gridDim.x);
  const size_t vs = (size_t)M * Ny;  // between work vectors (VS = 1: rows contiguous)
  bool live[2];
  int2 mu[2];
  for (int h = 0; h < 2; ++h) mu[h] = sched_mode(sched, 2 * item + h, live[h]);
  ChunkMaps<PO, false, MX> maps;
  maps.start(fmap, U, mu[0].y, lane, Ny);
  chunk_zero(lds, Ny, PO, MX, 2 * NR);
  // the right-hand sides, all in flight (rows past the end load and store the
  // last one again)
  for (int i0 = 0; i0 < Ny; i0 += 4 * 64) {
    cx<double> v[4][2 * NR];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 2 * NR; ++r)
        v[q][r] = a.scratch[((size_t)vin * M + mu[r / NR].x) * Ny + (r % NR) * vs + min(i0 + q * 64 + lane, Ny - 1)];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 2 * NR; ++r) sh[r * ld + min(i0 + q * 64 + lane, Ny - 1)] = v[q][r];
  }
  chunk_solve<PO, MX>(fmap, bmap, U, mu[0].y, lane, Ny, chunk_column<NR>(sh, NR * ld, ld, lane), maps);
  for (int i = lane; i < Ny; i += 64)
#pragma unroll
    for (int r = 0; r < 2 * NR; ++r)
      if (live[r / NR]) a.scratch[((size_t)vout * M + mu[r / NR].x) * Ny + (r % NR) * vs + i] = sh[r * ld + i];
}

// The whole influence-matrix step of two modes of one k^2 class in one
// workgroup, two wavefronts: everything between the fields and the new
// velocity stays in four LDS rows per mode and in registers.  Each wavefront
// does the parallel phases of its mode (lanes along y, YP points each, whose
// u^n_x, u^n_z and c N_j + (1 - c) N_n wait in registers through the L_k
// solve: the fields are read once); one of them the solves of both.  The
// per-row arithmetic and the solves are those of the five-launch form (same
// values, bit for bit); eight work vectors' round trips through memory and
// four launches go.
//
// Traffic: 15 vector components, and a class's maps for every two modes (1140
// bytes per point at p = 6, where the fields of both are 480).  The maps' way from the
// caches is the bound, not the products, which would take 15 us per item (two
// solves) at Ny = 256, p = 6; four items per CU (36 KB of LDS, 256 registers) put one
// solving wavefront on each SIMD (the first wavefronts of a CU's workgroups
// start on different ones).  One predictor, with the sequence of launches that
// was the fastest before: 128 x 256 x 128, p = 6, five launches 623 us, so
// 296 us; 64 x 128 x 64, p = 4, two launches (solve and parallel phases by
// each wavefront) 68 us, so 27 us; 48 x 65 x 32, p = 4: 35 us, so 12 us.
// Mixed contexts (MX; chunk_tiles): 128 x 256 x 128, p = 6, 563 us, so 317 us.
constexpr int kImmRows = 4;       // LDS rows per mode
// Largest Ny of the one-launch form.  LDS (8 rows, 40 KB) and points per lane
// would reach 320; five points a lane (from 257) already spill up to 53
// registers, and longer columns have neither been measured nor taken.
constexpr int kImmFusedNy = 278;

template <int PO, int YP, bool MX>
__global__ void __launch_bounds__(128, 2)
    k_imm_fused(ImmArgs a, const double* __restrict__ lf, const double* __restrict__ lb,
                const double* __restrict__ hf, const double* __restrict__ hb, const int2* __restrict__ sched, int U) {
  if (a.act && *a.act == 0) return;
  extern __shared__ cx<double> lds[];  // chunk_lds(Ny, PO, MX, 2 kImmRows): [2][kImmRows][ld]
  const int Ny = a.Ny, M = a.M, ld = chunk_ld(Ny, PO, MX), hs = kImmRows * ld;
  cx<double>* sh = lds + chunk_pad(Ny, PO, MX);
  const int lane = threadIdx.x & 63, half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int item = xcd_block(blockIdx.x, gridDim.x);
  const bool solver = half == 0;
  bool live;
  const int2 mu = sched_mode(sched, 2 * item + half, live);
  const int m = mu.x, u = __builtin_amdgcn_readfirstlane(mu.y);
  ChunkMaps<PO, false, MX> maps;
  if (solver) maps.start(lf, U, u, lane, Ny);
  chunk_zero(lds, Ny, PO, MX, 2 * kImmRows);
  cx<double>* r0 = sh + half * hs;
  cx<double>*r1 = r0 + ld, *r2 = r0 + 2 * ld, *r3 = r0 + 3 * ld;
  const size_t comp = (size_t)M * Ny, row = (size_t)m * Ny;
  const double kx = a.mkx[m], kz = a.mkz[m];
  const double k2 = kx * kx + kz * kz;
  // phase 1: u^n_y in r1, c N_j + (1 - c) N_n (y) in r0, d_hat in r2, f_hat in
  // r3; mixed: N_j (y) in r0, N_n (y) in r3 until f_hat replaces it, and the
  // fields are read again where the other components are needed
  cx<double> ux[YP], uz[YP];
  [[maybe_unused]] cx<double> nc[YP][3], fh[YP];
#pragma unroll
  for (int j = 0; j < YP; ++j) {
    const int y = min(lane + 64 * j, Ny - 1);
    ux[j] = a.un[row + y];
    uz[j] = a.un[2 * comp + row + y];
    r1[y] = a.un[comp + row + y];
    if constexpr (MX) {
      r0[y] = a.nj[comp + row + y];
      r3[y] = a.nn[comp + row + y];
    } else {
#pragma unroll
      for (int c = 0; c < 3; ++c) nc[j][c] = imm_n_at(a, c * comp + row + y);
      r0[y] = nc[j][1];
    }
  }
  // weights of G rows at a time: all their loads in flight, within the registers
  constexpr int G = YP < 2 ? YP : 2;
  wave_sync();
#pragma unroll
  for (int j0 = 0; j0 < YP; j0 += G) {
    Weights<PO + 1> d1[G];
#pragma unroll
    for (int j = 0; j < G && j0 + j < YP; ++j) d1[j] = Weights<PO + 1>(a.d1w, Ny, min(lane + 64 * (j0 + j), Ny - 1));
#pragma unroll
    for (int j = 0; j < G && j0 + j < YP; ++j)
      r2[min(lane + 64 * (j0 + j), Ny - 1)] = imm_dhat_at<PO>(d1[j], r1, ux[j0 + j], uz[j0 + j], kx, kz);
    __builtin_amdgcn_sched_barrier(0);
  }
  wave_sync();
#pragma unroll
  for (int j0 = 0; j0 < YP; j0 += G) {
    Weights<PO + 1> d1[G];
    Weights<PO + 2> d2[G];
    [[maybe_unused]] cx<double> n[G][4];
#pragma unroll
    for (int j = 0; j < G && j0 + j < YP; ++j) {
      int y = min(lane + 64 * (j0 + j), Ny - 1);
      if (YP > G) y = opaque(y);
      d1[j] = Weights<PO + 1>(a.d1w, Ny, y);
      d2[j] = Weights<PO + 2>(a.d2w, Ny, y);
      if constexpr (MX) {
        n[j][0] = a.nj[row + y];
        n[j][1] = a.nj[2 * comp + row + y];
        n[j][2] = a.nn[row + y];
        n[j][3] = a.nn[2 * comp + row + y];
      }
    }
#pragma unroll
    for (int j = 0; j < G && j0 + j < YP; ++j) {
      const int y = min(lane + 64 * (j0 + j), Ny - 1);
      if constexpr (MX)
        fh[j0 + j] = imm_fhat_mx_at<PO>(a, d1[j], d2[j], r2, r0, r3, n[j], kx, kz, k2, y);
      else
        r3[y] = imm_fhat_at<PO>(a, d1[j], d2[j], r2, r0, nc[j0 + j][0], nc[j0 + j][2], kx, kz, k2, y);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  wave_sync();
  // u^n's rows in r0, r1, r2 (phase 1's other rows are read)
#pragma unroll
  for (int j = 0; j < YP; ++j) {
    const int y = min(lane + 64 * j, Ny - 1);
    r0[y] = ux[j];
    r2[y] = uz[j];
    if constexpr (MX) r3[y] = fh[j];
  }
  __syncthreads();
  // phase 2: p_P in r3
  if (solver) {
    chunk_solve<PO, MX>(lf, lb, U, u, lane, Ny, chunk_column<1>(sh + 3 * ld, hs, ld, lane), maps);
    maps.start(hf, U, u, lane, Ny);
  }
  // phase 3: R_c in r0, r1, r2 (through registers: the stencils read them)
  {
    cx<double> r[YP][3];
#pragma unroll
    for (int j0 = 0; j0 < YP; j0 += G) {
      Weights<PO + 1> e1[G];
      Weights<PO + 2> e2[G];
      [[maybe_unused]] cx<double> nj[G][3], nn[G][3];
#pragma unroll
      for (int j = 0; j < G && j0 + j < YP; ++j) {
        // opaque: else phase 1's weights wait in registers through the solve
        const int y = opaque(min(lane + 64 * (j0 + j), Ny - 1));
        e1[j] = Weights<PO + 1>(a.d1w, Ny, y);
        e2[j] = Weights<PO + 2>(a.d2w, Ny, y);
        if constexpr (MX) {
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            nj[j][c] = a.nj[c * comp + row + y];
            nn[j][c] = a.nn[c * comp + row + y];
          }
        }
      }
      if (j0 == 0) __syncthreads();  // p_P is there
#pragma unroll
      for (int j = 0; j < G && j0 + j < YP; ++j)
        imm_r_at<PO, MX>(a, e1[j], e2[j], r3, r0, ld, MX ? nj[j] : nc[j0 + j], nn[j], kx, kz, k2,
                         min(lane + 64 * (j0 + j), Ny - 1), r[j0 + j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    wave_sync();
#pragma unroll
    for (int j = 0; j < YP; ++j)
#pragma unroll
      for (int c = 0; c < 3; ++c) r0[c * ld + min(lane + 64 * j, Ny - 1)] = r[j][c];
  }
  __syncthreads();
  // phase 4: the arbitrary velocity in r0, r1, r2
  if (solver) chunk_solve<PO, MX>(hf, hb, U, u, lane, Ny, chunk_column<3>(sh, hs, ld, lane), maps);
  // phase 5, its operands asked for before the barrier (the wavefront that
  // does not solve has them by then)
  double4 vq[YP];
  cx<double> uj[YP][3];
  double qw[YP];
#pragma unroll
  for (int j = 0; j < YP; ++j) {
    const int y = opaque(min(lane + 64 * j, Ny - 1));
    vq[j] = reinterpret_cast<const double4*>(a.vq)[(size_t)u * Ny + y];
#pragma unroll
    for (int c = 0; c < 3; ++c) uj[j][c] = a.uj[c * comp + row + y];
    qw[j] = a.qw[y];
  }
  __syncthreads();
  if (!live) return;
  cx<double> al1, al2;
  imm_alpha<PO>(a, m, r1, 1, al1, al2);
  double acc = 0.0;
#pragma unroll
  for (int j = 0; j < YP; ++j) {
    const int y = lane + 64 * j;
    if (y < Ny) acc += qw[j] * imm_assemble_at(a, m, row, comp, kx, kz, vq[j], uj[j], r0, r1, r2, 1, al1, al2, y);
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
  if (lane == 0 && a.partials) a.partials[m] = acc;
}

// Phase 3 (flows/plane_couette.py:449-472): R_c for the three components
// (zero on the walls) -> V_R + c, with the pressure row in LDS.
template <int PO, bool MX>
__global__ void __launch_bounds__(kImmT) k_imm_rc(ImmArgs a) {
  if (a.act && *a.act == 0) return;
  // LDS: the p_P row, then the rows of u^n (the D2 stencils' operands)
  extern __shared__ cx<double> pp[];
  const int m = blockIdx.x, Ny = a.Ny;
  const size_t comp = (size_t)a.M * Ny, row = (size_t)m * Ny;
  const double kx = a.mkx[m], kz = a.mkz[m];
  const double k2 = kx * kx + kz * kz;
  const cx<double>* P = svec(a, V_P, m);
  cx<double>* ur = pp + Ny;  // [c][y]
  for (int y = threadIdx.x; y < Ny; y += blockDim.x) {
    pp[y] = P[y * VS];
#pragma unroll
    for (int c = 0; c < 3; ++c) ur[c * Ny + y] = a.un[c * comp + row + y];
  }
  __syncthreads();
  for (int y = threadIdx.x; y < Ny; y += blockDim.x) {
    cx<double> nc[3], nn[3], r[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const size_t e = c * comp + row + y;
      if constexpr (MX) {
        nc[c] = a.nj[e];
        nn[c] = a.nn[e];
      } else {
        nc[c] = imm_n_at(a, e);
      }
    }
    imm_r_at<PO, MX>(a, Weights<PO + 1>(a.d1w, Ny, y), Weights<PO + 2>(a.d2w, Ny, y), pp, ur, Ny, nc, nn, kx, kz, k2,
                     y, r);
#pragma unroll
    for (int c = 0; c < 3; ++c) svec(a, V_R + c, m)[y * VS] = r[c];
  }
}

// Phase 5 (flows/plane_couette.py:476-504): alpha = -M^-1 (wall divergence
// of v_arb), the corrected velocity, the correction, and this mode's
// quadrature-weighted k_metric |delta|^2 into partials[m].
template <int PO>
__global__ void __launch_bounds__(kImmT) k_imm_final(ImmArgs a) {
  if (a.act && *a.act == 0) return;
  __shared__ double red[kImmT / 64];
  const int m = blockIdx.x, Ny = a.Ny, M = a.M;
  const size_t comp = (size_t)M * Ny, row = (size_t)m * Ny;
  const double kx = a.mkx[m], kz = a.mkz[m];
  const cx<double>* ua = svec(a, V_R + 0, m);
  const cx<double>* va = svec(a, V_R + 1, m);
  const cx<double>* wa = svec(a, V_R + 2, m);
  cx<double> al1, al2;
  imm_alpha<PO>(a, m, va, VS, al1, al2);
  double acc = 0.0;
  for (int y = threadIdx.x; y < Ny; y += blockDim.x) {
    const double4 w = reinterpret_cast<const double4*>(a.vq)[(size_t)a.umode[m] * Ny + y];
    const cx<double> uj[3] = {a.uj[row + y], a.uj[comp + row + y], a.uj[2 * comp + row + y]};
    acc += a.qw[y] * imm_assemble_at(a, m, row, comp, kx, kz, w, uj, ua, va, wa, VS, al1, al2, y);
  }
  const double s = block_sum(acc, red);
  if (threadIdx.x == 0 && a.partials) a.partials[m] = s;
}

// Quadrature-weighted norm of a field in (3, M, Ny) layout.
__global__ void __launch_bounds__(256)
    k_walls_norm(const cx<double>* __restrict__ f, const double* __restrict__ qw, int Ny, int M,
                 int Nkx, double* __restrict__ partials) {
  __shared__ double red[4];
  const long long n = (long long)M * Ny;
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  double acc = 0.0;
  if (i < n) {
    const int m = (int)(i / Ny), y = (int)(i - (long long)m * Ny);
    const double km = (m % Nkx == 0) ? 1.0 : 2.0;
    double s = 0.0;
    for (int c = 0; c < 3; ++c) {
      const cx<double> d = f[c * n + i];
      s += km * (d.x * d.x) + km * (d.y * d.y);
    }
    acc = qw[y] * s;
  }
  const double s = block_sum(acc, red);
  if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// ------------------------------------------------------------------ launchers
template <typename T, int EM, int TY>
static void launch_walls_curl_ty(Ctx* c, const cx<double>* u, cx<T>* A, hipStream_t s) {
  WallTables* t = c->wt;
  const cx<double>* uref = reinterpret_cast<const cx<double>*>(c->uref);
  cx<double>* ucopy = reinterpret_cast<cx<double>*>(c->uref);
  const dim3 grid(((t->Ny + TY - 1) / TY) * ((t->M + kTM - 1) / kTM));
  switch (t->p) {
#define CURL(PO)                                                                                \
  case PO:                                                                                      \
    hipLaunchKernelGGL((k_walls_curl_t<T, PO + 1, EM, TY>), grid, dim3(TY * kTM), 0, s, u, A,   \
                       t->d1w, t->d1j0, t->mkz, t->Ny, t->M, c->act, uref, ucopy);              \
    break;
    CURL(2) CURL(4) CURL(6) CURL(8)
#undef CURL
    default: break;
  }
}
template <typename T, int EM>
static void launch_walls_curl(Ctx* c, const cx<double>* u, cx<T>* A, hipStream_t s) {
  if (c->wt->curl_ty == 64)
    launch_walls_curl_ty<T, EM, 64>(c, u, A, s);
  else
    launch_walls_curl_ty<T, EM, 32>(c, u, A, s);
}

// em: EvalMode; EV_RECORD / EV_INC only in FP32 with the reference buffers.
template <typename T>
static int walls_rhs_t(Ctx* c, const double* state, double* rhs, hipStream_t s, int em) {
  WallTables* t = c->wt;
  const int Ny = t->Ny, M = t->M;
  cx<T>* A = static_cast<cx<T>*>(c->bufA);
  cx<T>* B = static_cast<cx<T>*>(c->bufB);
  const cx<T>* twz = static_cast<const cx<T>*>(c->fp32 ? c->tw32[2] : c->tw64[2]);
  const int ntile_y = (Ny + kTY - 1) / kTY, ntile_m = (M + kTM - 1) / kTM;
  {
    ProfScope ps(c, KID_W_Z_INVERSE, s);
    const cx<double>* u = reinterpret_cast<const cx<double>*>(state);
    if (t->p != 2 && t->p != 4 && t->p != 6 && t->p != 8) return c->fail(DNSMI_EINVAL, "fd_order");
    if (em == EV_PLAIN)
      launch_walls_curl<T, EV_PLAIN>(c, u, A, s);
    else if constexpr (std::is_same<T, float>::value) {
      if (em == EV_RECORD)
        launch_walls_curl<T, EV_RECORD>(c, u, A, s);
      else
        launch_walls_curl<T, EV_INC>(c, u, A, s);
    }
    int rc = check_launch(c, "walls_curl");
    if (rc) return rc;
    const int ntile = (c->Nx1 + 16 - 1) / 16;
    switch (c->Pz) {
#define X(P)                                                                                    \
  case P:                                                                                       \
    hipLaunchKernelGGL((k_z_inverse_plain<T, P, 16, 6>), dim3(Ny * ntile, 6),                   \
                       dim3(16 * ColPlan<P>::threads), 0, s, A, B, twz, c->nz, Ny, c->Nx1,     \
                       c->act);                                                                 \
    break;
      DNSMI_FOR_EACH_P(X)
#undef X
      default: return c->fail(DNSMI_EINVAL, "unsupported padded z length");
    }
    rc = check_launch(c, "walls_z_inverse");
    if (rc) return rc;
  }
  int rc = launch_x_pass<T>(c, B, A, c->base, c->cbase, c->nbase, Ny, KID_W_X_NONLINEAR, s, em);
  if (rc) return rc;
  rc = launch_z_forward_buf<T>(c, A, B, Ny, KID_W_Z_FORWARD, s);
  if (rc) return rc;
  {
    ProfScope ps(c, KID_W_Z_FORWARD, s);
    hipLaunchKernelGGL((k_walls_to_spec<T>), dim3(ntile_y * ntile_m, 3), dim3(kTY * kTM), 0, s, B,
                       reinterpret_cast<cx<double>*>(rhs), Ny, M, c->act,
                       em == EV_INC ? reinterpret_cast<const cx<double>*>(c->nref) : nullptr,
                       em == EV_RECORD ? reinterpret_cast<cx<double>*>(c->nref) : nullptr);
  }
  return check_launch(c, "walls_to_spec");
}

// One evaluation in the context's current precision (see EvalMode; EV_INC
// without a recorded reference records one, every FP64 evaluation is
// EV_PLAIN).
static int walls_rhs_mode(Ctx* c, const double* state, double* rhs, hipStream_t s, int em) {
  if (em == EV_INC && !c->ref_valid) em = EV_RECORD;
  if (!c->fp32 || !c->split) em = EV_PLAIN;
  if (!c->fp32) return walls_rhs_t<double>(c, state, rhs, s, EV_PLAIN);
  const int rc = walls_rhs_t<float>(c, state, rhs, s, em);
  if (rc == DNSMI_OK && em == EV_RECORD) c->ref_valid = true;
  return rc;
}

int walls_get_rhs(Ctx* c, const double* state, double* rhs, hipStream_t s) {
  return walls_rhs_mode(c, state, rhs, s, EV_PLAIN);
}

// N(state), the first evaluation of a guessed step: plain, after which the
// step's first corrector evaluation records the split reference.
int walls_guess_rhs(Ctx* c, const double* state, double* rhs, hipStream_t s) {
  c->ref_valid = false;
  return walls_rhs_mode(c, state, rhs, s, EV_PLAIN);
}

// The launches of one step; MX: a mixed context's.
template <int PO, bool MX>
static int launch_imm(Ctx* c, const ImmArgs& a, hipStream_t s) {
  WallTables* t = c->wt;
  const int Ny = t->Ny;
  const size_t row = (size_t)Ny * sizeof(cx<double>);
  const dim3 gm(t->M), gc(t->items);
  if (c->imm_fused && !c->sweep_seq) {
    if (Ny > kImmFusedNy) return c->fail(DNSMI_EINVAL, "imm: ny too large for the fused form");
    const size_t lds = (size_t)chunk_lds(Ny, PO, MX, 2 * kImmRows) * sizeof(cx<double>);
    auto fused = [&](auto yp) {
      hipLaunchKernelGGL((k_imm_fused<PO, decltype(yp)::value, MX>), gc, dim3(128), lds, s, a, t->lk_fmap, t->lk_bmap,
                         t->hk_fmap, t->hk_bmap, t->sched, t->U);
    };
    if (Ny <= 64) fused(std::integral_constant<int, 1>{});
    else if (Ny <= 128) fused(std::integral_constant<int, 2>{});
    else if (Ny <= 256) fused(std::integral_constant<int, 4>{});
    else fused(std::integral_constant<int, 5>{});
    return DNSMI_OK;
  }
  // solves of nr right-hand sides per mode
  auto solve = [&](auto nr, const double* ab, const int* piv, const double* fmap, const double* bmap, int vin,
                   int vout) {
    constexpr int NR = decltype(nr)::value;
    if (c->sweep_seq)
      hipLaunchKernelGGL(k_band_sweeps<PO>, dim3((t->M + kSweepLanes - 1) / kSweepLanes, NR), dim3(kSweepLanes), 0, s,
                         a, ab, piv, vin, (int)V_T, vout);
    else  // per workgroup two modes' vectors in LDS
      hipLaunchKernelGGL((k_band_chunks<PO, NR, MX>), gc, dim3(64),
                         (size_t)chunk_lds(Ny, PO, MX, 2 * NR) * sizeof(cx<double>), s, a, fmap, bmap, t->sched, t->U,
                         vin, vout);
  };
  hipLaunchKernelGGL((k_imm_fhat<PO, MX>), gm, dim3(kImmT), (MX ? 4 : 3) * row, s, a);
  solve(std::integral_constant<int, 1>{}, t->lk_ab, t->lk_piv, t->lk_fmap, t->lk_bmap, (int)V_F, (int)V_P);
  hipLaunchKernelGGL((k_imm_rc<PO, MX>), gm, dim3(kImmT), 4 * row, s, a);
  solve(std::integral_constant<int, 3>{}, t->hk_ab, t->hk_piv, t->hk_fmap, t->hk_bmap, (int)V_R, (int)V_R);
  hipLaunchKernelGGL(k_imm_final<PO>, gm, dim3(kImmT), 0, s, a);
  return DNSMI_OK;
}

// `out` may alias un or uj: a mode's new velocity is stored by the workgroup
// that read the mode's rows (phase 5 reads a point of uj and then stores it),
// after the last of its reads of u^n.  In the one-launch form all of those,
// the absent second mode's repeats of the first one's rows among them, come
// before the barriers in front of phase 5; the five-launch form's are in
// earlier launches.
static int walls_imm(Ctx* c, const double* un, const double* uj, const double* nn,
                     const double* nj, double* out, double* corr, double* err, hipStream_t s) {
  WallTables* t = c->wt;
  const int nb = t->M;  // one norm partial per mode
  if (nb > c->max_partials) return c->fail(DNSMI_EINVAL, "imm: too many blocks");
  ImmArgs a{};
  a.un = reinterpret_cast<const cx<double>*>(un);
  a.uj = reinterpret_cast<const cx<double>*>(uj);
  a.nn = reinterpret_cast<const cx<double>*>(nn);
  a.nj = reinterpret_cast<const cx<double>*>(nj);
  a.out = reinterpret_cast<cx<double>*>(out);
  a.corr = reinterpret_cast<cx<double>*>(corr);
  a.partials = c->partials;
  a.d1w = t->d1t;
  a.d2w = t->d2t;
  a.qw = t->qw;
  a.lk_ab = t->lk_ab;
  a.hk_ab = t->hk_ab;
  a.lk_piv = t->lk_piv;
  a.hk_piv = t->hk_piv;
  a.vq = t->vq;
  a.umode = t->umode;
  a.minv = t->minv;
  a.mkx = t->mkx;
  a.mkz = t->mkz;
  a.scratch = reinterpret_cast<cx<double>*>(t->scratch);
  a.act = c->act;
  a.Ny = t->Ny;
  a.M = t->M;
  a.Nkx = t->Nkx;
  a.dt = c->cfg.dt;
  a.c = c->cfg.implicitness;
  a.nu = 1.0 / c->cfg.re;
  {
    if (!c->sweep_seq && !t->lk_fmap) return c->fail(DNSMI_EINVAL, "imm: chunk maps not built");
    ProfScope ps(c, KID_W_IMM, s);
    if (4 * (size_t)t->Ny * sizeof(cx<double>) > 65536 || (!c->sweep_seq && t->Ny > kChunkNy))
      return c->fail(DNSMI_EINVAL, "imm: ny too large for the per-mode LDS rows");
    int rc = DNSMI_OK;
    switch (t->p) {
#define IMM(PO)                                                                       \
  case PO:                                                                            \
    rc = c->fp32_primary ? launch_imm<PO, true>(c, a, s) : launch_imm<PO, false>(c, a, s); \
    break;
      IMM(2) IMM(4) IMM(6) IMM(8)
#undef IMM
      default: return c->fail(DNSMI_EINVAL, "fd_order");
    }
    if (rc) return rc;
  }
  int rc = check_launch(c, "imm");
  if (rc || !err) return rc;
  return finalize_norm(c, nb, err, s);
}

// Chooses the band-solve form by timing one influence-matrix step of each
// on zeroed buffers (both forms are exact solves of the same systems).
static int walls_autotune(Ctx* c) {
  if (hipMemset(c->rhs0, 0, c->spec_elems * 16) != hipSuccess ||
      hipMemset(c->bufA, 0, c->spec_elems * 16) != hipSuccess)
    return c->fail(DNSMI_EHIP, "autotune: memset");
  // zero fields in, the new velocity into a buffer of its own (in place, the
  // second call would no longer start from zeros); bufA is transform scratch,
  // unused here
  double* z = c->rhs0;
  double* o = static_cast<double*>(c->bufA);
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)
    return c->fail(DNSMI_EHIP, "autotune: events");
  // a form that cannot run here (nonzero return) never wins
  auto time_imm = [&](bool seq, bool fused) {
    c->sweep_seq = seq;
    c->imm_fused = fused;
    if (walls_imm(c, z, z, z, z, o, nullptr, nullptr, nullptr) != DNSMI_OK)  // warm-up
      return (double)INFINITY;
    (void)hipEventRecord(e0, nullptr);
    for (int i = 0; i < 3; ++i)
      if (walls_imm(c, z, z, z, z, o, nullptr, nullptr, nullptr) != DNSMI_OK) return (double)INFINITY;
    (void)hipEventRecord(e1, nullptr);
    (void)hipEventSynchronize(e1);
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    return ms / 3.0;
  };
  // three alternating rounds, each form's best kept: a single round is
  // swayed by clock ramps and a profiler's first-launch costs, which fall
  // on whichever form runs first
  double tc = INFINITY, tf = INFINITY, ts = INFINITY;
  for (int round = 0; round < 3; ++round) {
    tc = std::min(tc, time_imm(false, false));
    tf = std::min(tf, time_imm(false, true));
    ts = std::min(ts, time_imm(true, false));
  }
  if (!(ts < INFINITY)) return c->fail(DNSMI_EINVAL, "autotune: the sequential band solve failed: " + c->err);
  c->err.clear();
  c->sweep_seq = ts < tc && ts < tf;
  c->imm_fused = !c->sweep_seq && tf < tc;
  if (c->sweep_seq) {  // the chunk maps are not needed any more
    WallTables* t = c->wt;
    for (double** p : {&t->lk_fmap, &t->lk_bmap, &t->hk_fmap, &t->hk_bmap}) {
      c->release(*p);
      *p = nullptr;
    }
    c->release(t->sched);
    t->sched = nullptr;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  char buf[160];
  snprintf(buf, sizeof buf, "band_solve=%s(chunked %.1f us, fused %.1f us, sequential %.1f us) ",
           c->sweep_seq ? "sequential" : (c->imm_fused ? "fused" : "chunked"), 1e3 * tc, 1e3 * tf, 1e3 * ts);
  c->tuning = buf;
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? DNSMI_OK : c->fail(DNSMI_EHIP, std::string("autotune: ") + hipGetErrorString(e));
}

int walls_predict(Ctx* c, const double* state, const double* rhs, double* pred, hipStream_t s) {
  return walls_imm(c, state, state, rhs, rhs, pred, nullptr, nullptr, s);
}

int walls_correct(Ctx* c, const double* state_prev, const double* pred_in,
                  const double* rhs_prev, const double* rhs_next, double* pred_out,
                  double* corr, hipStream_t s) {
  return walls_imm(c, state_prev, pred_in, rhs_prev, rhs_next, pred_out, corr, nullptr, s);
}

int walls_norm(Ctx* c, const double* corr, double* err, hipStream_t s) {
  WallTables* t = c->wt;
  const long long n = (long long)t->M * t->Ny;
  const int nb = (int)((n + 255) / 256);
  if (nb > c->max_partials) return c->fail(DNSMI_EINVAL, "norm: too many blocks");
  {
    ProfScope ps(c, KID_W_NORM, s);
    hipLaunchKernelGGL(k_walls_norm, dim3(nb), dim3(256), 0, s,
                       reinterpret_cast<const cx<double>*>(corr), t->qw, t->Ny, t->M, t->Nkx,
                       c->partials);
  }
  int rc = check_launch(c, "walls_norm");
  if (rc) return rc;
  return finalize_norm(c, nb, err, s);
}

int extrap_walls(Ctx* c, const double* n0, const float* h1, float* h2, double* next,
                 const uint16_t* wb, const float* bias, int H, float s_1, float s_2, float s_out,
                 int mode, hipStream_t s);

// Wall-bounded corrector guess (no reference counterpart).  The walls
// corrector's fixed point is u* = S(u^n; N(u*)) with S the influence-matrix
// solve (the explicit term is the previous evaluation,
// flows/plane_couette.py:534-539), so the guess is the predictor's solve
// (flows/plane_couette.py:507-519) fed with an extrapolated nonlinear term
// N_ext = N^n + dN (extrap_walls: dN = 0, D1, D1 + D2, or D1 + D2 plus the
// network's residual, D1, D2 the differences of N over the FP32 history
// h1 = N^{n-1}, h2 = N^{n-2}; h2 <- N^n).  rhs_prev <- N_ext, and the
// reference's iterate_correction continues from (pred, rhs_prev).
int guess_walls(Ctx* c, const double* state, double* pred, double* rhs_prev, const float* h1,
                float* h2, const uint16_t* wb, const float* bias, int H, float s_1, float s_2,
                float s_out, int mode, hipStream_t s) {
  if (mode < 0 || mode > 3) return c->fail(DNSMI_EINVAL, "guess: mode must be 0, 1, 2 or 3");
  if (mode == 2 && H != 32 && H != 64)
    return c->fail(DNSMI_EINVAL, "guess: hidden width must be 32 or 64");
  // N^n; the first corrector pass from the guess records the split reference
  int rc = walls_guess_rhs(c, state, c->rhs0, s);
  if (rc) return rc;
  if ((rc = extrap_walls(c, c->rhs0, h1, h2, rhs_prev, wb, bias, H, s_1, s_2, s_out, mode, s)))
    return rc;
  return walls_predict(c, state, rhs_prev, pred, s);
}

// The predictor's evaluation N(u^n) is plain; the first corrector
// evaluation N(u^1) records the split reference (mixed form), so every later
// increment is of the corrector's own size.
int walls_predict_and_correct(Ctx* c, const double* state, double* pred, double* rhs_next,
                              double* err, hipStream_t s) {
  double* n0 = c->rhs0;
  int rc = walls_rhs_mode(c, state, n0, s, EV_PLAIN);
  if (rc) return rc;
  if ((rc = walls_imm(c, state, state, n0, n0, pred, nullptr, nullptr, s))) return rc;
  c->ref_valid = false;
  if ((rc = walls_rhs_mode(c, pred, rhs_next, s, EV_RECORD))) return rc;
  return walls_imm(c, state, pred, n0, rhs_next, pred, nullptr, err, s);
}

int walls_iterate_correction(Ctx* c, const double* state_prev, double* pred,
                             const double* rhs_prev, double* rhs_next, double* err,
                             hipStream_t s) {
  // N_n := rhs_prev, the previous evaluation (flows/plane_couette.py:534-539)
  if ((const void*)rhs_next == (const void*)rhs_prev) {
    int rc = walls_rhs_mode(c, pred, c->rhs0, s, EV_INC);
    if (rc) return rc;
    if ((rc = walls_imm(c, state_prev, pred, rhs_prev, c->rhs0, pred, nullptr, err, s))) return rc;
    const hipError_t e = hipMemcpyAsync(rhs_next, c->rhs0, c->spec_elems * 16,
                                        hipMemcpyDeviceToDevice, s);
    return e == hipSuccess ? DNSMI_OK : c->fail(DNSMI_EHIP, hipGetErrorString(e));
  }
  int rc = walls_rhs_mode(c, pred, rhs_next, s, EV_INC);
  if (rc) return rc;
  return walls_imm(c, state_prev, pred, rhs_prev, rhs_next, pred, nullptr, err, s);
}

// The set-up tables in the reference layouts (for tests), read back from the
// device: which = 0 Lk_ab, 1 Hk_ab (mode, row, y), 2 v1, 3 q1 (mode, y),
// 4 M_inv (mode, 2, 2), 5 ys; 6 Lk_piv, 7 Hk_piv (mode, y; ints written as
// doubles); 8 .. 11 the chunk maps as stored (L_k forward, L_k back,
// H_k forward, H_k back; empty without them); 12 the per-class homogeneous
// solutions as stored ([class][y][4]); 13 the word counts of 8 .. 11 and
// the number of k^2 classes.
int walls_table(Ctx* c, int which, double* out, long long n) {
  WallTables* t = c->wt;
  if (!t) return c->fail(DNSMI_EINVAL, "not a wall-bounded context");
  const int Ny = t->Ny, M = t->M, rows = 3 * t->p + 1, U = t->U;
  auto fetch = [&](const void* src, size_t bytes, void* dst) {
    return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost) == hipSuccess;
  };
  auto want = [&](long long k) { return n == k ? DNSMI_OK : c->fail(DNSMI_EINVAL, "table size mismatch"); };
  int rc;
  switch (which) {
    case 0:
    case 1: {
      if ((rc = want((long long)M * rows * Ny))) return rc;
      std::vector<double> d((size_t)Ny * rows * M);
      if (!fetch(which == 0 ? t->lk_ab : t->hk_ab, d.size() * sizeof(double), d.data()))
        return c->fail(DNSMI_EHIP, "read table");
      for (int m = 0; m < M; ++m)
        for (int r = 0; r < rows; ++r)
          for (int j = 0; j < Ny; ++j) out[((size_t)m * rows + r) * Ny + j] = d[((size_t)j * rows + r) * M + m];
      return DNSMI_OK;
    }
    case 2:
    case 3:
    case 12: {
      std::vector<double> d(4ull * U * Ny);
      if (!fetch(t->vq, d.size() * sizeof(double), d.data())) return c->fail(DNSMI_EHIP, "read table");
      if (which == 12) {
        if ((rc = want((long long)d.size()))) return rc;
        std::copy(d.begin(), d.end(), out);
        return DNSMI_OK;
      }
      if ((rc = want((long long)M * Ny))) return rc;
      const int q = which == 2 ? 0 : 2;  // v1 = H^-1(-D1 p1), q1 = H^-1(p1)
      for (int m = 0; m < M; ++m)
        for (int j = 0; j < Ny; ++j) out[(size_t)m * Ny + j] = d[((size_t)t->h_umode[m] * Ny + j) * 4 + q];
      return DNSMI_OK;
    }
    case 4: {
      if ((rc = want(4LL * M))) return rc;
      std::vector<double> d(4ull * M);
      if (!fetch(t->minv, d.size() * sizeof(double), d.data())) return c->fail(DNSMI_EHIP, "read table");
      for (int m = 0; m < M; ++m)
        for (int q = 0; q < 4; ++q) out[(size_t)m * 4 + q] = d[(size_t)q * M + m];
      return DNSMI_OK;
    }
    case 5:
      if ((rc = want((long long)t->h_ys.size()))) return rc;
      std::copy(t->h_ys.begin(), t->h_ys.end(), out);
      return DNSMI_OK;
    case 6:
    case 7: {
      if ((rc = want((long long)M * Ny))) return rc;
      std::vector<int> d((size_t)Ny * M);
      if (!fetch(which == 6 ? t->lk_piv : t->hk_piv, d.size() * sizeof(int), d.data()))
        return c->fail(DNSMI_EHIP, "read table");
      for (int m = 0; m < M; ++m)
        for (int j = 0; j < Ny; ++j) out[(size_t)m * Ny + j] = d[(size_t)j * M + m];
      return DNSMI_OK;
    }
    case 8:
    case 9:
    case 10:
    case 11: {
      const bool back = which == 9 || which == 11;
      const size_t words = (size_t)chunk_count(Ny, t->p, back, c->fp32_primary) * U * map_words(t->p, back, c->fp32_primary);
      const double* src = which == 8 ? t->lk_fmap : which == 9 ? t->lk_bmap : which == 10 ? t->hk_fmap : t->hk_bmap;
      if (!src) return want(0);
      if ((rc = want((long long)words))) return rc;
      if (!fetch(src, words * sizeof(double), out)) return c->fail(DNSMI_EHIP, "read table");
      return DNSMI_OK;
    }
    case 13: {  // the words of tables 8 .. 11 (0 where absent), then the class count
      if ((rc = want(5))) return rc;
      out[4] = U;
      const double* maps[4] = {t->lk_fmap, t->lk_bmap, t->hk_fmap, t->hk_bmap};
      for (int i = 0; i < 4; ++i) {
        const bool back = i % 2 != 0, mx = c->fp32_primary;
        out[i] = maps[i] ? (double)((size_t)chunk_count(Ny, t->p, back, mx) * U * map_words(t->p, back, mx)) : 0.0;
      }
      return DNSMI_OK;
    }
    default: return c->fail(DNSMI_EINVAL, "unknown table");
  }
}

}  // namespace dnsmi
