// Triply periodic RHS pipeline and spectral updates, gfx950.
//
// One RHS evaluation (flows/monochromatic.py:366-386 via rhs.py:34-92 and
// fft.py:291-408) is five passes over HBM, each a batch of independent
// length-P transforms done as register-DFT / LDS / register-DFT:
//   K1 y-inverse  (pad ky, curl prep)   u (3,Ny1,Nz1,Nx1) f64 -> W1 (5,Py,Nz1,Nx1)
//   K2 z-inverse  (pad kz, curl)        W1 -> W2 (6,Py,Pz,Nx1)
//   K3 x pass     (c2r, u x w + base-flow terms, r2c, truncate)
//                                      W2 -> W3 (3,Py,Pz,Nx1)
//   K4 z-forward  (truncate kz)         W3 -> W4 (3,Py,Nz1,Nx1)
//   K5 y-forward  (truncate ky) + Leray projection + fused epilogue:
//        plain RHS / Euler predictor / CN corrector with FP64 norm partials.
// W1..W4 hold T = double (plain) or float (mixed) complex; the state, the
// RHS, the projection, the Helmholtz multiply and the norm stay FP64.
//
// The curl is split across passes: K1 transforms u and i*ky*u_{x,z} (the
// only factors that vary along y), K2 applies the i*kz factors before its
// transforms, K3 applies the i*kx factors on the kx bins before its c2r.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <string>
#include <type_traits>
#include <vector>

#include "context.hpp"
#include "ctl.hpp"
#include "dft.hpp"
#include "passes.hpp"

namespace dnsmi {

// K5 epilogues.  The carry forms keep B = ildt_2 (ldt_1 u^n + (1 - c) N^n)
// in the RHS buffer instead of N: the predictor writes it beside u^1, and a
// corrector pass is then u <- B + c ildt_2 N(u), the reference's fixed-point
// iteration in its full form (the incremental form u + c ildt_2 (N(u) -
// N_prev) telescopes to it), reading B and the iterate and writing the
// iterate only.
enum { MODE_RHS = 0, MODE_PREDICT = 1, MODE_CORRECT = 2, MODE_PREDICT_CARRY = 3, MODE_CORRECT_CARRY = 4 };

struct StepArgs {
  const double* state;     // MODE_PREDICT: u^n
  const double* rhs_prev;  // MODE_CORRECT: N_prev; MODE_CORRECT_CARRY: B
  double* pred;            // MODE_PREDICT: out; MODE_CORRECT: in/out
  double* rhs_out;         // N of this evaluation
  double* partials;        // MODE_CORRECT: per-block sum k_metric |delta|^2
  const int* act;          // if set and 0: the whole launch is skipped
  const double* nref;      // EV_INC: N(u_ref), added to the projected increment
                           // (carry form: B + c ildt_2 N(u_ref), in place of B)
  double* nref_out;        // EV_RECORD: receives a copy of N (the new N(u_ref))
                           // (carry form: B + c ildt_2 N(u_ref), the new iterate)
  double dt, c, re;
};

// Argument structs of the FFT-pass kernels: each kernel is launched with
// one (K(args)) or, batched over the members of an ensemble, reads member
// blockIdx.z's from a device table (K_b(table)); complex arrays are passed
// untyped and cast to the kernel's precision.
struct YInvArgs {
  const void* u;
  void* w1;
  const void* tw;
  const double* ky;
  int ny, Nz1, Nx1;
  const int* act;
  const void* uref;
  void* ucopy;
};
struct ZInvArgs {
  const void* w1;
  void* w2;
  const void* tw;
  const double* kz;
  int nz, Py, Nx1;
  const int* act;
  int stream_out;  // non-temporal stores of the output (an autotuned choice)
};
struct XArgs {
  const void* w2;
  void* w3;
  const void* tw;
  const double* kx;
  const double *base, *cbase, *nbase;
  int nx, Py, Pz, ybs;
  const int* act;
  float* xref;
};
struct ZFwdArgs {
  const void* w3;
  void* w4;
  const void* tw;
  int nz, Py, Nx1;
  const int* act;
};
struct YFwdArgs {
  const void* w4;
  const void* tw;
  const double *kx, *ky, *kz;
  int ny, Nz1, Nx1;
  StepArgs s;
};


template <typename T>
__device__ __forceinline__ cx<T> to_t(cx<double> d) {
  return {static_cast<T>(d.x), static_cast<T>(d.y)};
}

// ------------------------------------------------------------------ K1
// EM (EvalMode): EV_RECORD also copies u to ucopy (u_ref); EV_INC transforms
// d = u - uref, formed in FP64 before the rounding to T.
template <typename T, int P, int TC, bool PADY, int EM>
__device__ __forceinline__ void y_inverse_body(const cx<double>* __restrict__ u, cx<T>* __restrict__ w1,
                const cx<T>* __restrict__ tw, const double* __restrict__ ky, int ny, int Nz1,
                int Nx1, const int* __restrict__ act, const cx<double>* __restrict__ uref,
                cx<double>* __restrict__ ucopy) {
  if (act && *act == 0) return;
  constexpr int N1 = ColPlan<P>::N1, N2 = ColPlan<P>::N2;
  __shared__ cx<T> lds[TC * P];
  __shared__ cx<T> tws[P];
  for (int i = threadIdx.x; i < P; i += blockDim.x) tws[i] = tw[i];
  __syncthreads();
  const int tid = threadIdx.x, col = tid % TC, j_ = tid / TC;
  const int ntile = (Nx1 + TC - 1) / TC;
  const int kz = blockIdx.x / ntile;
  const int kx = (blockIdx.x - kz * ntile) * TC + col;
  const bool ok = kx < Nx1;
  const size_t plane = (size_t)Nz1 * Nx1;
  const size_t in_comp = (size_t)(ny - 1) * plane;
  const size_t out_f = (size_t)P * plane;
  const size_t off = (size_t)kz * Nx1 + kx;
  // pass 0: u_x -> F0 = Y(u_x), F4 = Y(i ky u_x); pass 1: u_z -> F2, F3;
  // pass 2: u_y -> F1.
#pragma unroll 1
  for (int pass = blockIdx.y; pass < 3; pass += gridDim.y) {
    const int j = opaque(j_);
    const int c = pass == 0 ? 0 : (pass == 1 ? 2 : 1);
    const int fa = c;
    const int fb = pass == 0 ? 4 : 3;
    cx<T> xa[N1], xb[N1];
    if (j < N2) {
#pragma unroll
      for (int a = 0; a < N1; ++a) {
        const int s = PadN<P, PADY ? 2 * P / 3 : P>::stored_in(N2 * a, N2, j);
        cx<T> v{0, 0}, vk{0, 0};
        if (ok && s >= 0) {
          const size_t e = c * in_comp + (size_t)s * plane + off;
          cx<double> d = u[e];
          if constexpr (EM == EV_RECORD) ucopy[e] = d;
          if constexpr (EM == EV_INC) {
            const cx<double> r = uref[e];
            d = {d.x - r.x, d.y - r.y};
          }
          const double k = ky[s];
          v = to_t<T>(d);
          vk = {static_cast<T>(-k * d.y), static_cast<T>(k * d.x)};
        }
        xa[a] = v;
        xb[a] = vk;
      }
      step_a_store<P, N1, N2, +1, TC>(xa, j, col, lds, tws);
    }
    __syncthreads();
    if (j < N1 && ok) {
      cx<T> y[N2];
      step_b_load<P, N1, N2, +1, TC>(y, j, col, lds);
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) w1[fa * out_f + (size_t)(j + N1 * k2) * plane + off] = y[k2];
    }
    __syncthreads();
    if (pass < 2) {
      if (j < N2) step_a_store<P, N1, N2, +1, TC>(xb, j, col, lds, tws);
      __syncthreads();
      if (j < N1 && ok) {
        cx<T> y[N2];
        step_b_load<P, N1, N2, +1, TC>(y, j, col, lds);
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2)
          w1[fb * out_f + (size_t)(j + N1 * k2) * plane + off] = y[k2];
      }
      __syncthreads();
    }
  }
}
template <typename T, int P, int TC, bool PADY, int EM>
__global__ void __launch_bounds__(TC * ColPlan<P>::threads) k_y_inverse(YInvArgs a) {
  y_inverse_body<T, P, TC, PADY, EM>(static_cast<const cx<double>*>(a.u), static_cast<cx<T>*>(a.w1), static_cast<const cx<T>*>(a.tw), a.ky, a.ny, a.Nz1, a.Nx1, a.act, static_cast<const cx<double>*>(a.uref), static_cast<cx<double>*>(a.ucopy));
}
template <typename T, int P, int TC, bool PADY, int EM>
__global__ void __launch_bounds__(TC * ColPlan<P>::threads) k_y_inverse_b(const YInvArgs* __restrict__ t) {
  const YInvArgs a = t[blockIdx.z];
  y_inverse_body<T, P, TC, PADY, EM>(static_cast<const cx<double>*>(a.u), static_cast<cx<T>*>(a.w1), static_cast<const cx<T>*>(a.tw), a.ky, a.ny, a.Nz1, a.Nx1, a.act, static_cast<const cx<double>*>(a.uref), static_cast<cx<double>*>(a.ucopy));
}


// ------------------------------------------------------------------ K2
template <typename T, int P, int TC>
__device__ __forceinline__ void z_inverse_body(const cx<T>* __restrict__ w1, cx<T>* __restrict__ w2, const cx<T>* __restrict__ tw,
                const double* __restrict__ kz_tab, int nz, int Py, int Nx1, const int* __restrict__ act, bool nt) {
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
  const size_t in_f = (size_t)Py * Nz1 * Nx1;
  const size_t in_off = (size_t)y * Nz1 * Nx1 + kx;
  const size_t out_f = (size_t)Py * P * Nx1;
  const size_t out_off = (size_t)y * P * Nx1 + kx;
  // outputs: 0 u_x, 1 u_y, 2 u_z, 3 w_x, 4 Z(i kz Yu_x), 5 Z(-Y(i ky u_x))
#pragma unroll 1
  for (int pass = blockIdx.y; pass < 4; pass += gridDim.y) {
    const int j = opaque(j_);
    cx<T> xa[N1], xb[N1];
    if (j < N2) {
#pragma unroll
      for (int a = 0; a < N1; ++a) {
        const int s = Pad<P>::stored_in(N2 * a, N2, j);
        cx<T> va{0, 0}, vb{0, 0};
        if (ok && s >= 0) {
          const T k = static_cast<T>(kz_tab[s]);
          const size_t e = in_off + (size_t)s * Nx1;
          if (pass == 0) {
            const cx<T> f0 = w1[0 * in_f + e];
            va = f0;
            vb = {-k * f0.y, k * f0.x};
          } else if (pass == 1) {
            const cx<T> f1 = w1[1 * in_f + e];
            const cx<T> f3 = w1[3 * in_f + e];
            va = f1;
            vb = {f3.x + k * f1.y, f3.y - k * f1.x};
          } else if (pass == 2) {
            va = w1[2 * in_f + e];
          } else {
            const cx<T> f4 = w1[4 * in_f + e];
            va = {-f4.x, -f4.y};
          }
        }
        xa[a] = va;
        xb[a] = vb;
      }
      step_a_store<P, N1, N2, +1, TC>(xa, j, col, lds, tws);
    }
    const int fa = pass == 0 ? 0 : (pass == 1 ? 1 : (pass == 2 ? 2 : 5));
    const int fb = pass == 0 ? 4 : 3;
    __syncthreads();
    if (j < N1 && ok) {
      cx<T> o[N2];
      step_b_load<P, N1, N2, +1, TC>(o, j, col, lds);
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2)
        st_out(&w2[fa * out_f + out_off + (size_t)(j + N1 * k2) * Nx1], o[k2], nt);
    }
    __syncthreads();
    if (pass < 2) {
      if (j < N2) step_a_store<P, N1, N2, +1, TC>(xb, j, col, lds, tws);
      __syncthreads();
      if (j < N1 && ok) {
        cx<T> o[N2];
        step_b_load<P, N1, N2, +1, TC>(o, j, col, lds);
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2)
          st_out(&w2[fb * out_f + out_off + (size_t)(j + N1 * k2) * Nx1], o[k2], nt);
      }
      __syncthreads();
    }
  }
}
template <typename T, int P, int TC>
__global__ void __launch_bounds__(TC * ColPlan<P>::threads) k_z_inverse(ZInvArgs a) {
  z_inverse_body<T, P, TC>(static_cast<const cx<T>*>(a.w1), static_cast<cx<T>*>(a.w2), static_cast<const cx<T>*>(a.tw), a.kz, a.nz, a.Py, a.Nx1, a.act, a.stream_out != 0);
}
template <typename T, int P, int TC>
__global__ void __launch_bounds__(TC * ColPlan<P>::threads) k_z_inverse_b(const ZInvArgs* __restrict__ t) {
  const ZInvArgs a = t[blockIdx.z];
  z_inverse_body<T, P, TC>(static_cast<const cx<T>*>(a.w1), static_cast<cx<T>*>(a.w2), static_cast<const cx<T>*>(a.tw), a.kz, a.nz, a.Py, a.Nx1, a.act, a.stream_out != 0);
}


// K1 / K2, sequential form: one transform in flight per pass (fewer live
// registers, higher occupancy); an input used by two outputs is read twice,
// the second time from L2.  Same outputs as the paired forms above.
template <typename T, int P, int TC, bool PADY, int EM>
__device__ __forceinline__ void y_inverse_seq_body(const cx<double>* __restrict__ u, cx<T>* __restrict__ w1,
                    const cx<T>* __restrict__ tw, const double* __restrict__ ky, int ny, int Nz1,
                    int Nx1, const int* __restrict__ act, const cx<double>* __restrict__ uref,
                    cx<double>* __restrict__ ucopy) {
  if (act && *act == 0) return;
  constexpr int N1 = ColPlan<P>::N1, N2 = ColPlan<P>::N2;
  __shared__ cx<T> lds[TC * P];
  __shared__ cx<T> tws[P];
  for (int i = threadIdx.x; i < P; i += blockDim.x) tws[i] = tw[i];
  __syncthreads();
  const int tid = threadIdx.x, col = tid % TC, j_ = tid / TC;
  const int ntile = (Nx1 + TC - 1) / TC;
  const int kz = blockIdx.x / ntile;
  const int kx = (blockIdx.x - kz * ntile) * TC + col;
  const bool ok = kx < Nx1;
  const size_t plane = (size_t)Nz1 * Nx1;
  const size_t in_comp = (size_t)(ny - 1) * plane;
  const size_t out_f = (size_t)P * plane;
  const size_t off = (size_t)kz * Nx1 + kx;
  // pass -> (input component, multiply by i ky, output field)
#pragma unroll 1
  for (int pass = blockIdx.y; pass < 5; pass += gridDim.y) {
    const int j = opaque(j_);
    const int c = pass < 2 ? 0 : (pass < 4 ? 2 : 1);
    const bool iky = (pass == 1 || pass == 3);
    const int f = pass == 0 ? 0 : (pass == 1 ? 4 : (pass == 2 ? 2 : (pass == 3 ? 3 : 1)));
    if (j < N2) {
      cx<T> x[N1];
#pragma unroll
      for (int a = 0; a < N1; ++a) {
        const int s = PadN<P, PADY ? 2 * P / 3 : P>::stored_in(N2 * a, N2, j);
        cx<T> v{0, 0};
        if (ok && s >= 0) {
          const size_t e = c * in_comp + (size_t)s * plane + off;
          cx<double> d = u[e];
          if constexpr (EM == EV_RECORD) {
            if (!iky) ucopy[e] = d;  // each component is read by one such pass
          }
          if constexpr (EM == EV_INC) {
            const cx<double> r = uref[e];
            d = {d.x - r.x, d.y - r.y};
          }
          if (iky) {
            const double k = ky[s];
            v = {static_cast<T>(-k * d.y), static_cast<T>(k * d.x)};
          } else {
            v = to_t<T>(d);
          }
        }
        x[a] = v;
      }
      step_a_store<P, N1, N2, +1, TC>(x, j, col, lds, tws);
    }
    __syncthreads();
    if (j < N1 && ok) {
      cx<T> y[N2];
      step_b_load<P, N1, N2, +1, TC>(y, j, col, lds);
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) w1[f * out_f + (size_t)(j + N1 * k2) * plane + off] = y[k2];
    }
    __syncthreads();
  }
}
template <typename T, int P, int TC, bool PADY, int EM>
__global__ void __launch_bounds__(TC * ColPlan<P>::threads) k_y_inverse_seq(YInvArgs a) {
  y_inverse_seq_body<T, P, TC, PADY, EM>(static_cast<const cx<double>*>(a.u), static_cast<cx<T>*>(a.w1), static_cast<const cx<T>*>(a.tw), a.ky, a.ny, a.Nz1, a.Nx1, a.act, static_cast<const cx<double>*>(a.uref), static_cast<cx<double>*>(a.ucopy));
}
template <typename T, int P, int TC, bool PADY, int EM>
__global__ void __launch_bounds__(TC * ColPlan<P>::threads) k_y_inverse_seq_b(const YInvArgs* __restrict__ t) {
  const YInvArgs a = t[blockIdx.z];
  y_inverse_seq_body<T, P, TC, PADY, EM>(static_cast<const cx<double>*>(a.u), static_cast<cx<T>*>(a.w1), static_cast<const cx<T>*>(a.tw), a.ky, a.ny, a.Nz1, a.Nx1, a.act, static_cast<const cx<double>*>(a.uref), static_cast<cx<double>*>(a.ucopy));
}


template <typename T, int P, int TC>
__device__ __forceinline__ void z_inverse_seq_body(const cx<T>* __restrict__ w1, cx<T>* __restrict__ w2,
                    const cx<T>* __restrict__ tw, const double* __restrict__ kz_tab, int nz, int Py,
                    int Nx1, const int* __restrict__ act, bool nt) {
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
  const size_t in_f = (size_t)Py * Nz1 * Nx1;
  const size_t in_off = (size_t)y * Nz1 * Nx1 + kx;
  const size_t out_f = (size_t)Py * P * Nx1;
  const size_t out_off = (size_t)y * P * Nx1 + kx;
  // pass: 0 Z(F0)->0, 1 Z(i kz F0)->4, 2 Z(F1)->1, 3 Z(F3 - i kz F1)->3,
  //       4 Z(F2)->2, 5 Z(-F4)->5
#pragma unroll 1
  for (int pass = blockIdx.y; pass < 6; pass += gridDim.y) {
    const int j = opaque(j_);
    const int fo = pass == 0 ? 0 : (pass == 1 ? 4 : (pass == 2 ? 1 : (pass == 3 ? 3 : (pass == 4 ? 2 : 5))));
    if (j < N2) {
      cx<T> x[N1];
#pragma unroll
      for (int a = 0; a < N1; ++a) {
        const int s = Pad<P>::stored_in(N2 * a, N2, j);
        cx<T> v{0, 0};
        if (ok && s >= 0) {
          const T k = static_cast<T>(kz_tab[s]);
          const size_t e = in_off + (size_t)s * Nx1;
          if (pass == 0) {
            v = w1[0 * in_f + e];
          } else if (pass == 1) {
            const cx<T> f0 = w1[0 * in_f + e];
            v = {-k * f0.y, k * f0.x};
          } else if (pass == 2) {
            v = w1[1 * in_f + e];
          } else if (pass == 3) {
            const cx<T> f1 = w1[1 * in_f + e];
            const cx<T> f3 = w1[3 * in_f + e];
            v = {f3.x + k * f1.y, f3.y - k * f1.x};
          } else if (pass == 4) {
            v = w1[2 * in_f + e];
          } else {
            const cx<T> f4 = w1[4 * in_f + e];
            v = {-f4.x, -f4.y};
          }
        }
        x[a] = v;
      }
      step_a_store<P, N1, N2, +1, TC>(x, j, col, lds, tws);
    }
    __syncthreads();
    if (j < N1 && ok) {
      cx<T> o[N2];
      step_b_load<P, N1, N2, +1, TC>(o, j, col, lds);
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2)
        st_out(&w2[fo * out_f + out_off + (size_t)(j + N1 * k2) * Nx1], o[k2], nt);
    }
    __syncthreads();
  }
}
template <typename T, int P, int TC>
__global__ void __launch_bounds__(TC * ColPlan<P>::threads) k_z_inverse_seq(ZInvArgs a) {
  z_inverse_seq_body<T, P, TC>(static_cast<const cx<T>*>(a.w1), static_cast<cx<T>*>(a.w2), static_cast<const cx<T>*>(a.tw), a.kz, a.nz, a.Py, a.Nx1, a.act, a.stream_out != 0);
}
template <typename T, int P, int TC>
__global__ void __launch_bounds__(TC * ColPlan<P>::threads) k_z_inverse_seq_b(const ZInvArgs* __restrict__ t) {
  const ZInvArgs a = t[blockIdx.z];
  z_inverse_seq_body<T, P, TC>(static_cast<const cx<T>*>(a.w1), static_cast<cx<T>*>(a.w2), static_cast<const cx<T>*>(a.tw), a.kz, a.nz, a.Py, a.Nx1, a.act, a.stream_out != 0);
}


// ------------------------------------------------------------------ K3
// One row (fixed y, z) per N1 threads; R rows per workgroup.  Inverse plan
// (N1, N2), forward plan (N2, N1): the inverse's output distribution
// x = j + N1 k2 is exactly the forward's input distribution, so the
// physical values never leave registers.
template <int N1, int N2>
struct XRow {
  static constexpr int a = RowLds<N1, N2>::value, b = RowLds<N2, N1>::value;
  static constexpr int value = a > b ? a : b;
};

// Waves per SIMD the x pass asks for: three for FP64 at P <= 96, whose rows
// fit 168 registers (the plane Couette x pass at P = 96 has 2304 waves:
// at two per SIMD the last 256 would run as a second, nearly empty round).
template <typename T, int P>
struct XWaves {
  static constexpr int value = (sizeof(T) == 8 && P <= 96) ? 3 : 2;
};

// The nonlinear term is formed in two stages to bound the live registers:
// after the (u_z, w_y) and (u_y, w_z) transforms, component 0 is complete
// and is transformed and stored; the (u_x, w_x) transform then completes
// components 1 and 2.  At most four physical fields are held at once.
//
// EM (EvalMode, FP32 only): EV_RECORD also stores each row's total velocity
// and vorticity U + u, W + w (the reference's physical fields) to xref,
// lane-major: field f, row r, lane j, point k2 at ((f rows + r) P + j N2 + k2).
// EV_INC takes the transformed fields as the increment d, w_d over u_ref
// (no base flow added) and forms dN = U x w_d + d x (W + w_d) with U, W
// read back from xref: every FP32 product is then of increment size.
template <typename T, int P, int R, int EM>
__device__ __forceinline__ void x_nonlinear_body(const cx<T>* __restrict__ w2, cx<T>* __restrict__ w3,
                  const cx<T>* __restrict__ tw, const double* __restrict__ kx_tab,
                  const double* __restrict__ base, const double* __restrict__ cbase,
                  const double* __restrict__ /* nbase: U x curl U, implied */, int nx, int Py,
                  int Pz, int ybase_stride, const int* __restrict__ act,
                  float* __restrict__ xref) {
  static_assert(EM == EV_PLAIN || sizeof(T) == 4, "split evaluations are FP32 only");
  if (act && *act == 0) return;
  constexpr int N1 = Plan<P>::N1, N2 = Plan<P>::N2;
  constexpr int ROW = XRow<N1, N2>::value;
  // 64 % N1 == 0: each row's N1 lanes sit in one wavefront
  constexpr bool kWaveRows = 64 % N1 == 0;
  __shared__ cx<T> lds[R * ROW];
  __shared__ cx<T> tab_i[N1 * N2];  // inverse plan (N1, N2)
  __shared__ cx<T> tab_f[N2 * N1];  // forward plan (N2, N1)
  fill_plan_twiddles<N1, N2>(tab_i, tw);
  fill_plan_twiddles<N2, N1>(tab_f, tw);
  __syncthreads();
  const int tid = threadIdx.x, r = tid / N1, j_ = tid - r * N1;
  const int nrows = Py * Pz;
  const int row = blockIdx.x * R + r;
  const bool ok = row < nrows;
  const int yrow = ok ? row / Pz : 0;
  constexpr int Nx1 = Pad<P>::half;  // nx / 2
  const size_t fstride = (size_t)nrows * Nx1;
  const cx<T>* in = w2 + (size_t)(ok ? row : 0) * Nx1;
  cx<T>* out = w3 + (size_t)(ok ? row : 0) * Nx1;
  cx<T>* rl = lds + r * ROW;
  const T inv = static_cast<T>(1.0 / P);

  // Inverse transform of one (u, w) pair into physical values re/im, in
  // three parts so a pair's loads can be issued while the previous pair is
  // transformed.  load_pair: the row's 16 lanes load the pair's modes
  // coalesced (kx = j + N1 i), 2 Nx1 / N1 values per lane.  stage_pair: the
  // combined input z_m = X_m + i Y_m (X_{P-k} = conj X_k) goes to the row's
  // LDS.  inverse_pair: the step-A lanes read theirs from there.  Step A's
  // output reuses the buffer: within a wavefront its reads complete before
  // its writes, and rows that span wavefronts synchronise in between.
  constexpr int PER = (Nx1 + N1 - 1) / N1;
  struct PairIn {
    cx<T> X[PER], G[PER];
    T kk[PER];
  };
  auto load_pair = [&](int pair, PairIn& q) {
    const int j = opaque(j_);
    const int fx = pair == 0 ? 2 : (pair == 1 ? 1 : 0);
    const int fg = pair == 0 ? 4 : (pair == 1 ? 5 : 3);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int k = j + N1 * i;
      if (Nx1 % N1 == 0 || k < Nx1) {
        q.kk[i] = static_cast<T>(kx_tab[k]);
        q.X[i] = in[fx * fstride + k];
        q.G[i] = in[fg * fstride + k];
      }
    }
  };
  auto stage_pair = [&](int pair, const PairIn& q) {
    const int j = opaque(j_);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int k = j + N1 * i;
      if (Nx1 % N1 == 0 || k < Nx1) {
        const T kk = q.kk[i];
        cx<T> X = q.X[i], Y;
        const cx<T> g = q.G[i];
        if (pair == 0)  // (u_z, w_y = Z(i kz Yu_x) - i kx u_z)
          Y = {g.x + kk * X.y, g.y - kk * X.x};
        else if (pair == 1)  // (u_y, w_z = Z(-Y(i ky u_x)) + i kx u_y)
          Y = {g.x - kk * X.y, g.y + kk * X.x};
        else  // (u_x, w_x)
          Y = g;
        if (k == 0) {  // irfft ignores the imaginary part of the DC bin
          X.y = 0;
          Y.y = 0;
        }
        rl[k] = {X.x - Y.y, X.y + Y.x};
        if (k != 0) rl[P - k] = {X.x + Y.y, Y.x - X.y};
      }
    }
  };
  auto inverse_pair = [&](int pair, T* re, T* im) {
    row_sync<kWaveRows>();
    const int j = opaque(j_);
    cx<T> z[N1];
    if (j < N2) {
#pragma unroll
      for (int a = 0; a < N1; ++a) {
        // padded index m = N2 a + j: the lane range's position relative to
        // the zero band is fixed at compile time per (unrolled) a
        const int lo = N2 * a, hi = N2 * a + N2 - 1;
        const bool none = Pad<P>::zero(lo, hi), pos = hi < Nx1, neg = lo > P - Nx1;
        const int m = lo + j;
        const bool live = !none && (pos || neg || m < Nx1 || m > P - Nx1);
        z[a] = live ? rl[m] : cx<T>{0, 0};
      }
    }
    if constexpr (!kWaveRows) __syncthreads();
    if (j < N2) row_step_a_store_tab<P, N1, N2, +1>(z, j, rl, tab_i);
    row_sync<kWaveRows>();
    cx<T> o[N2];
    row_step_b_load<P, N1, N2, +1>(o, j, rl);
    // total velocity and vorticity: u + U and w + curl U, component
    // (2, 1), (1, 2), (0, 0) for pairs 0, 1, 2 (increments: d and w_d alone)
    const int cu = pair == 0 ? 2 : (pair == 1 ? 1 : 0);
    const int cw = pair == 0 ? 1 : (pair == 1 ? 2 : 0);
    if constexpr (EM == EV_INC) {
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) {
        re[k2] = o[k2].x;
        im[k2] = o[k2].y;
      }
    } else {
      const int yr = opaque(yrow);
      const T Uc = static_cast<T>(base[cu * ybase_stride + yr]);
      const T Cc = static_cast<T>(cbase[cw * ybase_stride + yr]);
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) {
        re[k2] = o[k2].x + Uc;
        im[k2] = o[k2].y + Cc;
      }
    }
    if constexpr (EM == EV_RECORD) {
      if (ok) {
        const size_t fs = (size_t)nrows * P;
        float* xr = xref + (size_t)row * P + opaque(j_) * N2;
        float* pu = xr + cu * fs;
        float* pw = xr + (3 + cw) * fs;
        if constexpr (N2 % 4 == 0) {
#pragma unroll
          for (int i = 0; i < N2 / 4; ++i) {
            reinterpret_cast<float4*>(pu)[i] = {re[4 * i], re[4 * i + 1], re[4 * i + 2], re[4 * i + 3]};
            reinterpret_cast<float4*>(pw)[i] = {im[4 * i], im[4 * i + 1], im[4 * i + 2], im[4 * i + 3]};
          }
        } else {
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2) {
            pu[k2] = re[k2];
            pw[k2] = im[k2];
          }
        }
      }
    }
    row_sync<kWaveRows>();
  };

  // Forward transform of one real component, truncated to kx < nx/2.
  auto forward_store = [&](int c, const T* v_re) {
    const int j = opaque(j_);
    {
      cx<T> v[N2];
#pragma unroll
      for (int a = 0; a < N2; ++a) v[a] = {v_re[a], 0};
      row_step_a_store_tab<P, N2, N1, -1>(v, j, rl, tab_f);
    }
    row_sync<kWaveRows>();
    if (j < N2 && ok) {
      cx<T> o[N1];
      row_step_b_load<P, N2, N1, -1>(o, j, rl);
#pragma unroll
      for (int k2 = 0; k2 < N1; ++k2) {
        const int k = j + N2 * k2;
        // N2 k2 >= Nx1: truncated for every lane (those DFT outputs are dead)
        if (N2 * k2 < Nx1 && k < Nx1) out[c * fstride + k] = cscale(o[k2], inv);
      }
    }
    row_sync<kWaveRows>();
  };

  // u' x w' + (u' x curl U + U x w') + U x curl U   (rhs.py:80-88) is
  // formed as (u' + U) x (w' + curl U): the base-flow tables satisfy
  // nbase = U x curl U (the tilt rotates U and curl U together and leaves
  // (0, U dU/dy, 0) unchanged; plane Couette: (y,0,0) x (0,0,-1) = (0,y,0)),
  // so the product is the same sum of four terms with no per-row constants
  // held across the passes.
  T uz[N2], wy[N2], uy[N2], wz[N2];
  PairIn q;
  load_pair(0, q);
  stage_pair(0, q);
  load_pair(1, q);
  inverse_pair(0, uz, wy);
  stage_pair(1, q);
  load_pair(2, q);
  inverse_pair(1, uy, wz);
  // EV_INC: the reference fields of this lane's points (rows past the end
  // read row 0's, like the inputs), N2 consecutive floats per field, read
  // four at a time where N2 allows
  const size_t xfs = (size_t)nrows * P;
  const float* xr = EM == EV_INC ? xref + (size_t)(ok ? row : 0) * P + j_ * N2 : nullptr;
  auto ref_row = [&](int f, T (&v)[N2]) {
    const float* p = xr + f * xfs;
    if constexpr (N2 % 4 == 0) {
#pragma unroll
      for (int i = 0; i < N2 / 4; ++i) {
        const float4 t = reinterpret_cast<const float4*>(p)[i];
        v[4 * i] = t.x;
        v[4 * i + 1] = t.y;
        v[4 * i + 2] = t.z;
        v[4 * i + 3] = t.w;
      }
    } else {
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) v[k2] = p[k2];
    }
  };
  // EV_INC: the reference fields component 0 reads (U_y, U_z, W_y, W_z)
  // stay in registers for components 1 and 2, so each is read once
  constexpr int KR = EM == EV_INC ? N2 : 1;
  T Uy[KR], Uz[KR], Wy[KR], Wz[KR];
  {
    T nl0[N2];
    if constexpr (EM == EV_INC) {
      ref_row(1, Uy);
      ref_row(2, Uz);
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) nl0[k2] = Uy[k2] * wz[k2] - Uz[k2] * wy[k2];
      ref_row(4, Wy);
      ref_row(5, Wz);
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2)
        nl0[k2] += uy[k2] * (Wz[k2] + wz[k2]) - uz[k2] * (Wy[k2] + wy[k2]);
    } else {
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) {
        nl0[k2] = uy[k2] * wz[k2] - uz[k2] * wy[k2];
      }
    }
    forward_store(0, nl0);
  }
  stage_pair(2, q);
  // Components 1 and 2 are real: one complex transform of nl1 + i nl2,
  // separated by Hermitian symmetry, X1[k] = (Z[k] + conj Z[P-k]) / 2 and
  // X2[k] = (Z[k] - conj Z[P-k]) / 2i.  Z[P-k] for k < Nx1 lives in another
  // lane of the row (lane (N2 - j) mod N2), so the needed high outputs are
  // exchanged through the row's LDS.
  {
    cx<T> v[N2];
    {
      T ux[N2], wx[N2];
      inverse_pair(2, ux, wx);
      if constexpr (EM == EV_INC) {
        // (U + u_ref) x w_d, then d x (W + w_ref + w_d); U_y, U_z, W_y, W_z
        // kept from component 0
        {
          T Ux[N2];
          ref_row(0, Ux);
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2) {
            v[k2].x = Uz[k2] * wx[k2] - Ux[k2] * wz[k2];
            v[k2].y = Ux[k2] * wy[k2];
          }
        }
        {
          T Wx[N2];
          ref_row(3, Wx);
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2) {
            v[k2].y -= Uy[k2] * wx[k2];
            v[k2].x += uz[k2] * (Wx[k2] + wx[k2]);
            v[k2].y -= uy[k2] * (Wx[k2] + wx[k2]);
          }
        }
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) {
          v[k2].x -= ux[k2] * (Wz[k2] + wz[k2]);
          v[k2].y += ux[k2] * (Wy[k2] + wy[k2]);
        }
      } else {
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) {
          v[k2].x = uz[k2] * wx[k2] - ux[k2] * wz[k2];
          v[k2].y = ux[k2] * wy[k2] - uy[k2] * wx[k2];
        }
      }
    }
    const int j = opaque(j_);
    row_step_a_store_tab<P, N2, N1, -1>(v, j, rl, tab_f);
    row_sync<kWaveRows>();
    cx<T> o[N1];
    if (j < N2) row_step_b_load<P, N2, N1, -1>(o, j, rl);
    row_sync<kWaveRows>();
    // publish Z[k] for the partners' indices: k = j + N2 k2 with k2 >= KH
    constexpr int KH = N1 - 1 - (Nx1 - 1) / N2;
    if (j < N2) {
#pragma unroll
      for (int k2 = KH; k2 < N1; ++k2) rl[j + N2 * k2] = o[k2];
      if (j == 0) rl[0] = o[0];
    }
    row_sync<kWaveRows>();
    if (j < N2 && ok) {
#pragma unroll
      for (int k2 = 0; k2 < N1; ++k2) {
        const int k = j + N2 * k2;
        if (N2 * k2 < Nx1 && k < Nx1) {
          const cx<T> z = o[k2], w = rl[k == 0 ? 0 : P - k];
          const cx<T> x1 = {(z.x + w.x) * (T)0.5, (z.y - w.y) * (T)0.5};
          const cx<T> x2 = {(z.y + w.y) * (T)0.5, (w.x - z.x) * (T)0.5};
          out[1 * fstride + k] = cscale(x1, inv);
          out[2 * fstride + k] = cscale(x2, inv);
        }
      }
    }
  }
}
template <typename T, int P, int R, int EM>
__global__ void __launch_bounds__(R * Plan<P>::N1, (EM == EV_INC ? 3 : XWaves<T, P>::value)) k_x_nonlinear(XArgs a) {
  x_nonlinear_body<T, P, R, EM>(static_cast<const cx<T>*>(a.w2), static_cast<cx<T>*>(a.w3), static_cast<const cx<T>*>(a.tw), a.kx, a.base, a.cbase, a.nbase, a.nx, a.Py, a.Pz, a.ybs, a.act, a.xref);
}
template <typename T, int P, int R, int EM>
__global__ void __launch_bounds__(R * Plan<P>::N1, (EM == EV_INC ? 3 : XWaves<T, P>::value)) k_x_nonlinear_b(const XArgs* __restrict__ t) {
  const XArgs a = t[blockIdx.z];
  x_nonlinear_body<T, P, R, EM>(static_cast<const cx<T>*>(a.w2), static_cast<cx<T>*>(a.w3), static_cast<const cx<T>*>(a.tw), a.kx, a.base, a.cbase, a.nbase, a.nx, a.Py, a.Pz, a.ybs, a.act, a.xref);
}


// K3, split form (N2 even): 2 N1 threads per row.  The inverse step B
// (a DFT-N2 per k1) is split by decimation in frequency between the thread
// pair (k1, h): z_b = (y_b +- y_{b+N2/2}) w^{b h}, a DFT-(N2/2), outputs
// k2 = 2m + h.  Each thread then holds N2/2 physical points per field
// (half of the plain form), at x = (k1 + N1 h) + 2 N1 m, which is the input
// distribution of the forward plan (N2/2, 2 N1); its step B (DFT-2N1) is
// split the same way.  Both threads of a pair read the whole LDS column.
template <typename T, int P, int R>
__device__ __forceinline__ void x_nonlinear_split_body(const cx<T>* __restrict__ w2, cx<T>* __restrict__ w3,
                        const cx<T>* __restrict__ tw, const double* __restrict__ kx_tab,
                        const double* __restrict__ base, const double* __restrict__ cbase,
                        const double* __restrict__ nbase, int nx, int Py, int Pz,
                        int ybase_stride, const int* __restrict__ act) {
  if (act && *act == 0) return;
  constexpr int N1 = Plan<P>::N1, N2 = Plan<P>::N2;
  static_assert(N2 % 2 == 0, "split x pass needs an even second factor");
  constexpr int H2 = N2 / 2;    // points per field per thread
  constexpr int TPR = 2 * N1;   // threads per row
  constexpr int F1 = H2, F2 = TPR, G2 = F2 / 2;  // forward plan (F1, F2)
  constexpr int ROWA = N1 * (N2 + 1), ROWB = F1 * (F2 + 1);
  constexpr int ROW = ROWA > ROWB ? ROWA : ROWB;
  __shared__ cx<T> lds[R * ROW];
  __shared__ cx<T> tws[P];
  for (int i = threadIdx.x; i < P; i += blockDim.x) tws[i] = tw[i];
  __syncthreads();
  const int tid = threadIdx.x, r = tid / TPR, t = tid - r * TPR;
  const int k1 = t >> 1, h = t & 1;
  const int nrows = Py * Pz;
  const int row = blockIdx.x * R + r;
  const bool ok = row < nrows;
  const int yrow = ok ? row / Pz : 0;
  const int Nx1 = nx / 2;
  const size_t fstride = (size_t)nrows * Nx1;
  const cx<T>* in = w2 + (size_t)(ok ? row : 0) * Nx1;
  cx<T>* rl = lds + r * ROW;

  T ux[H2], uy[H2], uz[H2], wx[H2], wy[H2], wz[H2];
#pragma unroll
  for (int pair = 0; pair < 3; ++pair) {
    if (t < N2) {
      cx<T> z[N1];
#pragma unroll
      for (int a = 0; a < N1; ++a) {
        const int m = N2 * a + t;
        int k = -1;
        bool cj = false;
        if (m < Nx1) {
          k = m;
        } else if (m > P - Nx1) {
          k = P - m;
          cj = true;
        }
        cx<T> X{0, 0}, Y{0, 0};
        if (ok && k >= 0) {
          const T kk = static_cast<T>(kx_tab[k]);
          if (pair == 0) {
            X = in[2 * fstride + k];
            const cx<T> g = in[4 * fstride + k];
            Y = {g.x + kk * X.y, g.y - kk * X.x};
          } else if (pair == 1) {
            X = in[1 * fstride + k];
            const cx<T> g = in[5 * fstride + k];
            Y = {g.x - kk * X.y, g.y + kk * X.x};
          } else {
            X = in[0 * fstride + k];
            Y = in[3 * fstride + k];
          }
          if (k == 0) {
            X.y = 0;
            Y.y = 0;
          }
        }
        z[a] = cj ? cx<T>{X.x + Y.y, Y.x - X.y} : cx<T>{X.x - Y.y, X.y + Y.x};
      }
      row_step_a_store<P, N1, N2, +1>(z, t, rl, tws);
    }
    __syncthreads();
    {
      cx<T> zz[H2];
      const cx<T>* col = rl + k1 * (N2 + 1);
#pragma unroll
      for (int b = 0; b < H2; ++b) {
        const cx<T> y0 = col[b], y1 = col[b + H2];
        zz[b] = h ? twiddle_const<N2, +1>(csub(y0, y1), b) : cadd(y0, y1);
      }
      Dft<H2, +1, T>::run(zz);
#pragma unroll
      for (int m = 0; m < H2; ++m) {
        if (pair == 0) {
          uz[m] = zz[m].x;
          wy[m] = zz[m].y;
        } else if (pair == 1) {
          uy[m] = zz[m].x;
          wz[m] = zz[m].y;
        } else {
          ux[m] = zz[m].x;
          wx[m] = zz[m].y;
        }
      }
    }
    __syncthreads();
  }

  const T U0 = static_cast<T>(base[0 * ybase_stride + yrow]);
  const T U1 = static_cast<T>(base[1 * ybase_stride + yrow]);
  const T U2 = static_cast<T>(base[2 * ybase_stride + yrow]);
  const T C0 = static_cast<T>(cbase[0 * ybase_stride + yrow]);
  const T C1 = static_cast<T>(cbase[1 * ybase_stride + yrow]);
  const T C2 = static_cast<T>(cbase[2 * ybase_stride + yrow]);
  const T B0 = static_cast<T>(nbase[0 * ybase_stride + yrow]);
  const T B1 = static_cast<T>(nbase[1 * ybase_stride + yrow]);
  const T B2 = static_cast<T>(nbase[2 * ybase_stride + yrow]);
  T nl[3][H2];
#pragma unroll
  for (int m = 0; m < H2; ++m) {
    const T a0 = ux[m], a1 = uy[m], a2 = uz[m];
    const T b0 = wx[m], b1 = wy[m], b2 = wz[m];
    nl[0][m] = (a1 * b2 - a2 * b1) + (((a1 * C2 - a2 * C1) + (U1 * b2 - U2 * b1)) + B0);
    nl[1][m] = (a2 * b0 - a0 * b2) + (((a2 * C0 - a0 * C2) + (U2 * b0 - U0 * b2)) + B1);
    nl[2][m] = (a0 * b1 - a1 * b0) + (((a0 * C1 - a1 * C0) + (U0 * b1 - U1 * b0)) + B2);
  }

  const T inv = static_cast<T>(1.0 / P);
  cx<T>* out = w3 + (size_t)(ok ? row : 0) * Nx1;
  const int bq = k1 + N1 * h;  // forward input column: x = bq + F2 m
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    {
      cx<T> v[F1];
#pragma unroll
      for (int m = 0; m < F1; ++m) v[m] = {nl[c][m], 0};
      row_step_a_store<P, F1, F2, -1>(v, bq, rl, tws);
    }
    __syncthreads();
    if (t < 2 * F1 && ok) {
      const int kf = t >> 1, hh = t & 1;
      const cx<T>* col = rl + kf * (F2 + 1);
      cx<T> zz[G2];
#pragma unroll
      for (int b = 0; b < G2; ++b) {
        const cx<T> y0 = col[b], y1 = col[b + G2];
        zz[b] = hh ? twiddle_const<F2, -1>(csub(y0, y1), b) : cadd(y0, y1);
      }
      Dft<G2, -1, T>::run(zz);
#pragma unroll
      for (int m = 0; m < G2; ++m) {
        const int k = kf + F1 * (2 * m + hh);
        if (k < Nx1) out[c * fstride + k] = cscale(zz[m], inv);
      }
    }
    __syncthreads();
  }
}
template <typename T, int P, int R>
__global__ void __launch_bounds__(R * 2 * Plan<P>::N1) k_x_nonlinear_split(XArgs a) {
  x_nonlinear_split_body<T, P, R>(static_cast<const cx<T>*>(a.w2), static_cast<cx<T>*>(a.w3), static_cast<const cx<T>*>(a.tw), a.kx, a.base, a.cbase, a.nbase, a.nx, a.Py, a.Pz, a.ybs, a.act);
}
template <typename T, int P, int R>
__global__ void __launch_bounds__(R * 2 * Plan<P>::N1) k_x_nonlinear_split_b(const XArgs* __restrict__ t) {
  const XArgs a = t[blockIdx.z];
  x_nonlinear_split_body<T, P, R>(static_cast<const cx<T>*>(a.w2), static_cast<cx<T>*>(a.w3), static_cast<const cx<T>*>(a.tw), a.kx, a.base, a.cbase, a.nbase, a.nx, a.Py, a.Pz, a.ybs, a.act);
}


// ------------------------------------------------------------------ K4
template <typename T, int P, int TC>
__device__ __forceinline__ void z_forward_body(const cx<T>* __restrict__ w3, cx<T>* __restrict__ w4, const cx<T>* __restrict__ tw,
                int nz, int Py, int Nx1, const int* __restrict__ act) {
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
  const size_t in_f = (size_t)Py * P * Nx1;
  const size_t in_off = (size_t)y * P * Nx1 + kx;
  const size_t out_f = (size_t)Py * Nz1 * Nx1;
  const size_t out_off = (size_t)y * Nz1 * Nx1 + kx;
  const T inv = static_cast<T>(1.0 / P);
#pragma unroll 1
  for (int c = blockIdx.y; c < 3; c += gridDim.y) {
    const int j = opaque(j_);
    if (j < N2) {
      cx<T> x[N1];
#pragma unroll
      for (int a = 0; a < N1; ++a)
        x[a] = ok ? w3[c * in_f + in_off + (size_t)(N2 * a + j) * Nx1] : cx<T>{0, 0};
      step_a_store<P, N1, N2, -1, TC>(x, j, col, lds, tws);
    }
    __syncthreads();
    if (j < N1 && ok) {
      cx<T> o[N2];
      step_b_load<P, N1, N2, -1, TC>(o, j, col, lds);
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) {
        const int s = Pad<P>::stored_in(N1 * k2, N1, j);
        if (s >= 0) w4[c * out_f + out_off + (size_t)s * Nx1] = cscale(o[k2], inv);
      }
    }
    __syncthreads();
  }
}
template <typename T, int P, int TC>
__global__ void __launch_bounds__(TC * ColPlan<P>::threads) k_z_forward(ZFwdArgs a) {
  z_forward_body<T, P, TC>(static_cast<const cx<T>*>(a.w3), static_cast<cx<T>*>(a.w4), static_cast<const cx<T>*>(a.tw), a.nz, a.Py, a.Nx1, a.act);
}
template <typename T, int P, int TC>
__global__ void __launch_bounds__(TC * ColPlan<P>::threads) k_z_forward_b(const ZFwdArgs* __restrict__ t) {
  const ZFwdArgs a = t[blockIdx.z];
  z_forward_body<T, P, TC>(static_cast<const cx<T>*>(a.w3), static_cast<cx<T>*>(a.w4), static_cast<const cx<T>*>(a.tw), a.nz, a.Py, a.Nx1, a.act);
}


// ------------------------------------------------------------------ K5
// The epilogue's operands at one mode: what the mode of the pass combines
// with the projected N, for the three components.
template <int MODE>
struct YOps {
  cx<double> a[3];  // state, N_prev or B
  cx<double> p[3];  // the iterate
  cx<double> r[3];  // N(u_ref) of an increment
  __device__ __forceinline__ void load(const StepArgs& g, size_t pos, size_t comp) {
    constexpr bool predict = MODE == MODE_PREDICT || MODE == MODE_PREDICT_CARRY;
    constexpr bool correct = MODE == MODE_CORRECT || MODE == MODE_CORRECT_CARRY;
    const double* pa = predict ? g.state : (MODE == MODE_CORRECT_CARRY && g.nref ? g.nref : g.rhs_prev);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const size_t idx = c * comp + pos;
      if constexpr (predict || correct) a[c] = reinterpret_cast<const cx<double>*>(pa)[idx];
      if constexpr (correct) p[c] = reinterpret_cast<const cx<double>*>(g.pred)[idx];
      if constexpr (MODE == MODE_RHS || MODE == MODE_PREDICT || MODE == MODE_CORRECT)
        if (g.nref) r[c] = reinterpret_cast<const cx<double>*>(g.nref)[idx];
    }
  }
};

// One mode: the projection of N and the pass's update of the three
// components.  Returns the mode's share of the norm.
template <int MODE>
__device__ __forceinline__ double y_epilogue(const StepArgs& args, const YOps<MODE>& cur, cx<double> n0,
                                             cx<double> n1, cx<double> n2, double kxv, double kyv, double kzv,
                                             double km, bool mean, size_t pos, size_t comp) {
  double acc = 0.0;
  const double lapl = -((kxv * kxv + kyv * kyv) + kzv * kzv);
  const double il = lapl < 0 ? 1.0 / lapl : 0.0;
  // div = i kx N0 + i ky N1 + i kz N2 ; p = inv_lapl * div
  const cx<double> dv = {((-kxv * n0.y) + (-kyv * n1.y)) + (-kzv * n2.y),
                         ((kxv * n0.x) + (kyv * n1.x)) + (kzv * n2.x)};
  const cx<double> pr = {il * dv.x, il * dv.y};
  const double kk[3] = {kxv, kyv, kzv};
  const cx<double> nn[3] = {n0, n1, n2};
  const double ldt1 = mean ? 0.0 : 1.0 / args.dt + (1.0 - args.c) * lapl / args.re;
  const double ildt2 = mean ? 0.0 : 1.0 / (1.0 / args.dt - args.c * lapl / args.re);
  cx<double>* pd = reinterpret_cast<cx<double>*>(args.pred);
  cx<double>* rout = reinterpret_cast<cx<double>*>(args.rhs_out);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    // rhs = N - i k p (increments: N(u_ref) + P[dN])
    cx<double> rh = {nn[c].x + kk[c] * pr.y, nn[c].y - kk[c] * pr.x};
    const size_t idx = c * comp + pos;
    if constexpr (MODE == MODE_CORRECT_CARRY) {
      // u <- B + c ildt_2 N(u); increments: (B + c ildt_2 N(u_ref)) + c ildt_2 P[dN]
      const cx<double> base = cur.a[c], p0 = cur.p[c];
      const double ci = args.c * ildt2;
      const cx<double> un = {base.x + ci * rh.x, base.y + ci * rh.y};
      const cx<double> d = {un.x - p0.x, un.y - p0.y};
      pd[idx] = un;
      if (args.nref_out) reinterpret_cast<cx<double>*>(args.nref_out)[idx] = un;
      acc += km * (d.x * d.x) + km * (d.y * d.y);
      continue;
    }
    if constexpr (MODE == MODE_PREDICT_CARRY) {
      const cx<double> u = cur.a[c];
      pd[idx] = {(u.x * ldt1 + rh.x) * ildt2, (u.y * ldt1 + rh.y) * ildt2};
      const double cm = 1.0 - args.c;
      rout[idx] = {(u.x * ldt1 + cm * rh.x) * ildt2, (u.y * ldt1 + cm * rh.y) * ildt2};
      continue;
    }
    if (args.nref) rh = {cur.r[c].x + rh.x, cur.r[c].y + rh.y};
    if (args.nref_out) reinterpret_cast<cx<double>*>(args.nref_out)[idx] = rh;
    if constexpr (MODE == MODE_PREDICT) {
      const cx<double> u = cur.a[c];
      pd[idx] = {(u.x * ldt1 + rh.x) * ildt2, (u.y * ldt1 + rh.y) * ildt2};
    } else if constexpr (MODE == MODE_CORRECT) {
      const cx<double> np = cur.a[c], p0 = cur.p[c];
      const cx<double> d = {args.c * (rh.x - np.x) * ildt2, args.c * (rh.y - np.y) * ildt2};
      pd[idx] = {p0.x + d.x, p0.y + d.y};
      acc += km * (d.x * d.x) + km * (d.y * d.y);
    }
    rout[idx] = rh;
  }
  return acc;
}

// A third of the workgroup per component: the three transforms run side by
// side, meet in LDS, and the projection and epilogue then go over the modes
// with all threads, three components to a thread, the next mode's operands
// loaded before this one's results are stored.
//
// The pass has one workgroup per column tile (62 at 32^3, 508 at 128^3), so
// below the largest grids it is bound by one workgroup's chain of memory round
// trips: three transforms and 36 epilogue loads one behind the other in the
// serial form (below), one transform and at most three modes here.  A launch,
// serial and side by side: 32^3 FP64 11.1 and 5.7 us, 64^3 FP64 15.8 and 7.9,
// 96 x 64 x 48 FP32 23.5 and 11.0, sixteen 48^3 FP32 54.5 and 40.9; 128^3 FP32
// moves its 224 MB at memory speed either way (55.0 and 56.8 us).
template <typename T, int P, int TC, int MODE, bool PADY>
__device__ __forceinline__ void y_forward_body(const cx<T>* __restrict__ w4, const cx<T>* __restrict__ tw,
                const double* __restrict__ kx_tab, const double* __restrict__ ky_tab,
                const double* __restrict__ kz_tab, int ny, int Nz1, int Nx1, StepArgs args) {
  if (args.act && *args.act == 0) return;
  constexpr int N1 = ColPlan<P>::N1, N2 = ColPlan<P>::N2;
  constexpr int NM = PADY ? 2 * P / 3 : P;    // ny
  constexpr int G = 3 * N2;                   // threads of one column
  constexpr int IT = (NM - 1 + G - 1) / G;    // modes of one thread
  __shared__ cx<T> lds[3 * TC * P];
  __shared__ cx<T> tws[P];
  __shared__ double red[16];
  for (int i = threadIdx.x; i < P; i += blockDim.x) tws[i] = tw[i];
  __syncthreads();
  const int tid = threadIdx.x, col = tid % TC, g = tid / TC;
  const int tc = g / N2, j = g - tc * N2;
  const int ntile = (Nx1 + TC - 1) / TC;
  const int kz = blockIdx.x / ntile;
  const int kx = (blockIdx.x - kz * ntile) * TC + col;
  const bool ok = kx < Nx1;
  const size_t plane = (size_t)Nz1 * Nx1;
  const size_t in_f = (size_t)P * plane;
  const size_t off = (size_t)kz * Nx1 + kx;
  const size_t comp = (size_t)(ny - 1) * plane;
  const T inv = static_cast<T>(1.0 / P);
  cx<T>* lc = lds + tc * (TC * P);
  {
    cx<T> x[N1];
#pragma unroll
    for (int a = 0; a < N1; ++a)
      x[a] = ok ? w4[tc * in_f + (size_t)(N2 * a + j) * plane + off] : cx<T>{0, 0};
    step_a_store<P, N1, N2, -1, TC>(x, j, col, lc, tws);
  }
  YOps<MODE> cur;
  if (ok && g < NM - 1) cur.load(args, (size_t)g * plane + off, comp);
  __syncthreads();
  {
    cx<T> R[N2];
    if (j < N1) step_b_load<P, N1, N2, -1, TC>(R, j, col, lc);
    __syncthreads();
    if (j < N1) {
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2)
        if (!PadN<P, NM>::zero(N1 * k2, N1 * k2 + N1 - 1)) lc[(j + N1 * k2) * TC + col] = cscale(R[k2], inv);
    }
  }
  __syncthreads();

  double acc = 0.0;
  const double kxv = ok ? kx_tab[kx] : 0.0, kzv = kz_tab[kz];
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int s = g + it * G;
    YOps<MODE> nxt;
    if (it + 1 < IT && ok && s + G < NM - 1) nxt.load(args, (size_t)(s + G) * plane + off, comp);
    if (ok && s < NM - 1) {
      const int m = s < NM / 2 ? s : s + (P - NM + 1);
      const cx<T>* l = lds + m * TC + col;
      acc += y_epilogue<MODE>(args, cur, {l[0].x, l[0].y}, {l[TC * P].x, l[TC * P].y},
                              {l[2 * TC * P].x, l[2 * TC * P].y}, kxv, ky_tab[s], kzv, kx == 0 ? 1.0 : 2.0,
                              s == 0 && kz == 0 && kx == 0, (size_t)s * plane + off, comp);
    }
    cur = nxt;
  }
  if (MODE == MODE_CORRECT || MODE == MODE_CORRECT_CARRY) {
    const double s = block_sum(acc, red);
    if (threadIdx.x == 0) args.partials[blockIdx.x] = s;
  }
}
template <typename T, int P, int TC, int MODE, bool PADY>
__global__ void __launch_bounds__(3 * TC * ColPlan<P>::threads) k_y_forward(YFwdArgs a) {
  y_forward_body<T, P, TC, MODE, PADY>(static_cast<const cx<T>*>(a.w4), static_cast<const cx<T>*>(a.tw), a.kx, a.ky, a.kz, a.ny, a.Nz1, a.Nx1, a.s);
}
template <typename T, int P, int TC, int MODE, bool PADY>
__global__ void __launch_bounds__(3 * TC * ColPlan<P>::threads) k_y_forward_b(const YFwdArgs* __restrict__ t) {
  const YFwdArgs a = t[blockIdx.z];
  y_forward_body<T, P, TC, MODE, PADY>(static_cast<const cx<T>*>(a.w4), static_cast<const cx<T>*>(a.tw), a.kx, a.ky, a.kz, a.ny, a.Nz1, a.Nx1, a.s);
}


// The components one behind the other in one tile's LDS, the results in
// registers.
template <typename T, int P, int TC, int MODE, bool PADY>
__device__ __forceinline__ void y_forward_serial_body(const cx<T>* __restrict__ w4, const cx<T>* __restrict__ tw,
                const double* __restrict__ kx_tab, const double* __restrict__ ky_tab,
                const double* __restrict__ kz_tab, int ny, int Nz1, int Nx1, StepArgs args) {
  if (args.act && *args.act == 0) return;
  constexpr int N1 = ColPlan<P>::N1, N2 = ColPlan<P>::N2;
  __shared__ cx<T> lds[TC * P];
  __shared__ cx<T> tws[P];
  __shared__ double red[16];
  for (int i = threadIdx.x; i < P; i += blockDim.x) tws[i] = tw[i];
  __syncthreads();
  const int tid = threadIdx.x, col = tid % TC, j = tid / TC;
  const int ntile = (Nx1 + TC - 1) / TC;
  const int kz = blockIdx.x / ntile;
  const int kx = (blockIdx.x - kz * ntile) * TC + col;
  const bool ok = kx < Nx1;
  const size_t plane = (size_t)Nz1 * Nx1;
  const size_t in_f = (size_t)P * plane;
  const size_t off = (size_t)kz * Nx1 + kx;
  const size_t comp = (size_t)(ny - 1) * plane;
  const T inv = static_cast<T>(1.0 / P);
  cx<T> R[3][N2];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (j < N2) {
      cx<T> x[N1];
#pragma unroll
      for (int a = 0; a < N1; ++a)
        x[a] = ok ? w4[c * in_f + (size_t)(N2 * a + j) * plane + off] : cx<T>{0, 0};
      step_a_store<P, N1, N2, -1, TC>(x, j, col, lds, tws);
    }
    __syncthreads();
    if (j < N1) {
      step_b_load<P, N1, N2, -1, TC>(R[c], j, col, lds);
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) R[c][k2] = cscale(R[c][k2], inv);
    }
    __syncthreads();
  }

  double acc = 0.0;
  if (j < N1 && ok) {
    const double kxv = kx_tab[kx], kzv = kz_tab[kz];
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) {
      const int s = PadN<P, PADY ? 2 * P / 3 : P>::stored_in(N1 * k2, N1, j);
      if (s < 0) continue;
      YOps<MODE> ops;
      ops.load(args, (size_t)s * plane + off, comp);
      acc += y_epilogue<MODE>(args, ops, {R[0][k2].x, R[0][k2].y}, {R[1][k2].x, R[1][k2].y},
                              {R[2][k2].x, R[2][k2].y}, kxv, ky_tab[s], kzv, kx == 0 ? 1.0 : 2.0,
                              s == 0 && kz == 0 && kx == 0, (size_t)s * plane + off, comp);
    }
  }
  if (MODE == MODE_CORRECT || MODE == MODE_CORRECT_CARRY) {
    const double s = block_sum(acc, red);
    if (threadIdx.x == 0) args.partials[blockIdx.x] = s;
  }
}
template <typename T, int P, int TC, int MODE, bool PADY>
__global__ void __launch_bounds__(TC * ColPlan<P>::threads) k_y_forward_serial(YFwdArgs a) {
  y_forward_serial_body<T, P, TC, MODE, PADY>(static_cast<const cx<T>*>(a.w4), static_cast<const cx<T>*>(a.tw), a.kx, a.ky, a.kz, a.ny, a.Nz1, a.Nx1, a.s);
}
template <typename T, int P, int TC, int MODE, bool PADY>
__global__ void __launch_bounds__(TC * ColPlan<P>::threads) k_y_forward_serial_b(const YFwdArgs* __restrict__ t) {
  const YFwdArgs a = t[blockIdx.z];
  y_forward_serial_body<T, P, TC, MODE, PADY>(static_cast<const cx<T>*>(a.w4), static_cast<const cx<T>*>(a.tw), a.kx, a.ky, a.kz, a.ny, a.Nz1, a.Nx1, a.s);
}


// ------------------------------------------------------------------ pointwise
struct PointArgs {
  const double* a;  // state / pred_in / correction
  const double* b;  // rhs / rhs_prev
  const double* c2; // rhs_next
  double* out;      // pred_out / state out
  double* out2;     // correction out
  double* partials;
  double dt, c, re;
  int ny, Nz1, Nx1;
  long long n;  // complex elements per component
};

enum { PW_PREDICT = 0, PW_CORRECT = 1, PW_NORM = 2, PW_DIVFREE = 3, PW_DIVFREE_NORM = 4 };

struct PwArgs {
  PointArgs p;
  const double *kx, *ky, *kz;
};
struct ZmArgs {
  double* u;
  long long n;
};
struct FinArgs {
  const double* partials;
  int n;
  double* err;
  const int* act;
  StepCtl* ctl;
  CtlRule rule;
};

template <int OP>
__device__ __forceinline__ void pointwise_body(PointArgs p, const double* __restrict__ kx_tab, const double* __restrict__ ky_tab,
                const double* __restrict__ kz_tab) {
  __shared__ double red[16];
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  double acc = 0.0;
  if (i < p.n) {
    const int kx = (int)(i % p.Nx1);
    const long long t = i / p.Nx1;
    const int kz = (int)(t % p.Nz1);
    const int s = (int)(t / p.Nz1);
    const double kxv = kx_tab[kx], kyv = ky_tab[s], kzv = kz_tab[kz];
    const double km = kx == 0 ? 1.0 : 2.0;
    const double lapl = -((kxv * kxv + kyv * kyv) + kzv * kzv);
    const bool mean = (s == 0 && kz == 0 && kx == 0);
    const cx<double>* A = reinterpret_cast<const cx<double>*>(p.a);
    const cx<double>* B = reinterpret_cast<const cx<double>*>(p.b);
    const cx<double>* C = reinterpret_cast<const cx<double>*>(p.c2);
    cx<double>* O = reinterpret_cast<cx<double>*>(p.out);
    cx<double>* O2 = reinterpret_cast<cx<double>*>(p.out2);
    if (OP == PW_PREDICT || OP == PW_CORRECT) {
      const double ldt1 = mean ? 0.0 : 1.0 / p.dt + (1.0 - p.c) * lapl / p.re;
      const double ildt2 = mean ? 0.0 : 1.0 / (1.0 / p.dt - p.c * lapl / p.re);
      for (int c = 0; c < 3; ++c) {
        const long long idx = c * p.n + i;
        if (OP == PW_PREDICT) {
          const cx<double> u = A[idx], r = B[idx];
          O[idx] = {(u.x * ldt1 + r.x) * ildt2, (u.y * ldt1 + r.y) * ildt2};
        } else {
          const cx<double> pr = A[idx], np = B[idx], nn = C[idx];
          const cx<double> d = {p.c * (nn.x - np.x) * ildt2, p.c * (nn.y - np.y) * ildt2};
          O[idx] = {pr.x + d.x, pr.y + d.y};
          if (O2) O2[idx] = d;
        }
      }
    } else if (OP == PW_NORM) {
      for (int c = 0; c < 3; ++c) {
        const cx<double> d = A[c * p.n + i];
        acc += km * (d.x * d.x) + km * (d.y * d.y);
      }
    } else {
      // u - grad(inv_lapl div u); mean mode zeroed (flows/monochromatic.py:516-560)
      const double il = lapl < 0 ? 1.0 / lapl : 0.0;
      const cx<double> u0 = A[i], u1 = A[p.n + i], u2 = A[2 * p.n + i];
      const cx<double> dv = {((-kxv * u0.y) + (-kyv * u1.y)) + (-kzv * u2.y),
                             ((kxv * u0.x) + (kyv * u1.x)) + (kzv * u2.x)};
      const cx<double> pr = {il * dv.x, il * dv.y};
      const double kk[3] = {kxv, kyv, kzv};
      const cx<double> uu[3] = {u0, u1, u2};
      for (int c = 0; c < 3; ++c) {
        const cx<double> corr = {kk[c] * pr.y, -kk[c] * pr.x};  // -(i k p)
        cx<double> v = {uu[c].x + corr.x, uu[c].y + corr.y};
        if (OP == PW_DIVFREE_NORM) acc += km * (corr.x * corr.x) + km * (corr.y * corr.y);
        if (mean) v = {0.0, 0.0};
        O[c * p.n + i] = v;
      }
    }
  }
  if (OP == PW_NORM || OP == PW_DIVFREE_NORM) {
    const double s = block_sum(acc, red);
    if (threadIdx.x == 0) p.partials[blockIdx.x] = s;
  }
}
template <int OP>
__global__ void __launch_bounds__(256) k_pointwise(PwArgs a) {
  pointwise_body<OP>(a.p, a.kx, a.ky, a.kz);
}
template <int OP>
__global__ void __launch_bounds__(256) k_pointwise_b(const PwArgs* __restrict__ t) {
  const PwArgs a = t[blockIdx.z];
  pointwise_body<OP>(a.p, a.kx, a.ky, a.kz);
}


__device__ __forceinline__ void zero_mean_body(double* __restrict__ u, long long n) {
  if (threadIdx.x < 6) u[2 * (threadIdx.x / 2) * n + (threadIdx.x & 1)] = 0.0;
}
__global__ void __launch_bounds__(64) k_zero_mean(ZmArgs a) {
  zero_mean_body(a.u, a.n);
}
__global__ void __launch_bounds__(64) k_zero_mean_b(const ZmArgs* __restrict__ t) {
  const ZmArgs a = t[blockIdx.z];
  zero_mean_body(a.u, a.n);
}


// The norm from its per-block partials, summed in a fixed order.  With a
// control block (the corrector slots of a device step, whose err it writes)
// it then applies the corrector rule, one launch instead of two.  Every
// thread reads *act before the reduction's barriers, so the rule's update of
// `active` (the same word) cannot race with that read.
__device__ __forceinline__ void finalize_norm_body(const double* __restrict__ partials, int n,
                                                       double* err, const int* act, StepCtl* ctl,
                                                       CtlRule rule) {
  if (act && *act == 0) return;
  __shared__ double red[16];
  // eight loads in flight per thread: one behind the other, each waits out a
  // round trip to memory
  constexpr int U = 8;
  double v = 0.0;
  for (int i0 = threadIdx.x; i0 < n; i0 += U * blockDim.x) {
    double w[U];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int i = i0 + q * (int)blockDim.x;
      w[q] = i < n ? partials[i] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < U; ++q) v += w[q];
  }
  const double s = block_sum(v, red);
  if (threadIdx.x == 0) {
    const double e = sqrt(s);
    *err = e;
    if (ctl) ctl_after_iteration(ctl, rule, e);
  }
}
__global__ void __launch_bounds__(1024) k_finalize_norm(FinArgs a) {
  finalize_norm_body(a.partials, a.n, a.err, a.act, a.ctl, a.rule);
}
__global__ void __launch_bounds__(1024) k_finalize_norm_b(const FinArgs* __restrict__ t) {
  const FinArgs a = t[blockIdx.z];
  finalize_norm_body(a.partials, a.n, a.err, a.act, a.ctl, a.rule);
}


int finalize_norm(Ctx* c, int nblocks, double* err_dev, hipStream_t s) {
  ProfScope ps(c, KID_FINALIZE, s);
  StepCtl* ctl = c->fuse_ctl ? reinterpret_cast<StepCtl*>(c->ctl) : nullptr;
  // A workgroup of 1024 once 256 threads would take a second round of loads:
  // the 8128 partials of 128 x 256 x 128 plane Couette 14.5 -> 4.5 us; up to
  // 2048 the launch's 4 us are one round trip and the sum, whichever the size.
  launch(c, &k_finalize_norm, &k_finalize_norm_b, dim3(1), dim3(nblocks > 2048 ? 1024 : 256), s,
         FinArgs{c->partials, nblocks, err_dev, c->act, ctl, c->rule});
  return check_launch(c, "finalize_norm");
}

// ------------------------------------------------------------------ launchers
template <typename T>
struct Bufs {
  cx<T>* A;
  cx<T>* B;
  const cx<T>* twx;
  const cx<T>* twy;
  const cx<T>* twz;
};

template <typename T>
static Bufs<T> bufs_of(Ctx* c) {
  const int slot = std::is_same<T, float>::value ? 1 : 0;
  void* const* tw = slot ? c->tw32 : c->tw64;
  return {static_cast<cx<T>*>(c->bufA), static_cast<cx<T>*>(c->bufB),
          static_cast<const cx<T>*>(tw[0]), static_cast<const cx<T>*>(tw[1]),
          static_cast<const cx<T>*>(tw[2])};
}

// Columns per workgroup of the y/z passes: 16 (the default) or 8, chosen
// per context by the autotuner (c->tile_cols); kTCMin sizes the buffers
// that scale with the number of column tiles.
constexpr int kTC = 16, kTCMin = 8;

// Calls f(std::integral_constant<int, TC>) for the context's column tile.
template <typename F>
static void with_tc(const Ctx* c, F&& f) {
  if (c->tile_cols == 8)
    f(std::integral_constant<int, 8>{});
  else
    f(std::integral_constant<int, kTC>{});
}
constexpr int kRows = 16;  // rows per workgroup of the x pass
constexpr int kCUs = 256;   // compute units of the chip

template <typename T, int P, int EM, int TC>
static void launch_y_inverse_p(Ctx* c, dim3 grid, const cx<double>* u, cx<T>* w1, const cx<T>* tw,
                               hipStream_t s) {
  const dim3 blk(TC * ColPlan<P>::threads);
  const bool pady = c->Py != c->ny;  // y padded by the 3/2 rule
  const YInvArgs a{u, w1, tw, c->ky, c->ny, c->Nz1, c->Nx1, c->act, c->uref, c->uref};
  if (c->yinv_seq && pady)
    launch(c, &k_y_inverse_seq<T, P, TC, true, EM>, &k_y_inverse_seq_b<T, P, TC, true, EM>, grid, blk, s, a);
  else if (c->yinv_seq)
    launch(c, &k_y_inverse_seq<T, P, TC, false, EM>, &k_y_inverse_seq_b<T, P, TC, false, EM>, grid, blk, s, a);
  else if (pady)
    launch(c, &k_y_inverse<T, P, TC, true, EM>, &k_y_inverse_b<T, P, TC, true, EM>, grid, blk, s, a);
  else
    launch(c, &k_y_inverse<T, P, TC, false, EM>, &k_y_inverse_b<T, P, TC, false, EM>, grid, blk, s, a);
}

template <typename T>
static int launch_y_inverse(Ctx* c, const double* state, hipStream_t s, int em = EV_PLAIN) {
  Bufs<T> b = bufs_of<T>(c);
  const int ntile = (c->Nx1 + c->tile_cols - 1) / c->tile_cols;
  // one pass per workgroup (grid.y): the passes read different inputs and
  // write different outputs, and Nz1 * ntile workgroups alone underfill the GPU
  const dim3 grid(c->Nz1 * ntile, c->yinv_seq ? 5 : 3);
  const cx<double>* u = reinterpret_cast<const cx<double>*>(state);
  if (em != EV_PLAIN && (!std::is_same<T, float>::value || !c->uref))
    return c->fail(DNSMI_EINVAL, "split evaluation without FP32 reference buffers");
  ProfScope ps(c, KID_Y_INVERSE, s);
  switch (c->Py) {
#define X(P)                                                                    \
  case P:                                                                       \
    with_tc(c, [&](auto tcv) {                                                  \
      constexpr int TC = decltype(tcv)::value;                                  \
      if (em == EV_PLAIN)                                                       \
        launch_y_inverse_p<T, P, EV_PLAIN, TC>(c, grid, u, b.A, b.twy, s);      \
      else if constexpr (std::is_same<T, float>::value) {                       \
        if (em == EV_RECORD)                                                    \
          launch_y_inverse_p<T, P, EV_RECORD, TC>(c, grid, u, b.A, b.twy, s);   \
        else                                                                    \
          launch_y_inverse_p<T, P, EV_INC, TC>(c, grid, u, b.A, b.twy, s);      \
      }                                                                         \
    });                                                                         \
    break;
    DNSMI_FOR_EACH_P(X)
#undef X
    default: return c->fail(DNSMI_EINVAL, "unsupported padded y length");
  }
  return check_launch(c, "y_inverse");
}

template <typename T>
static int launch_z_inverse(Ctx* c, hipStream_t s) {
  Bufs<T> b = bufs_of<T>(c);
  const int ntile = (c->Nx1 + c->tile_cols - 1) / c->tile_cols;
  const dim3 grid(c->Py * ntile, c->zinv_seq ? 6 : 4);  // one pass per workgroup
  ProfScope ps(c, KID_Z_INVERSE, s);
  switch (c->Pz) {
#define X(P)                                                                                    \
  case P:                                                                                       \
    with_tc(c, [&](auto tcv) {                                                                  \
      constexpr int TC = decltype(tcv)::value;                                                  \
      const ZInvArgs a{b.A, b.B, b.twz, c->kz, c->nz, c->Py, c->Nx1, c->act, c->zinv_nt};      \
      if (c->zinv_seq)                                                                          \
        launch(c, &k_z_inverse_seq<T, P, TC>, &k_z_inverse_seq_b<T, P, TC>, grid,               \
               dim3(TC * ColPlan<P>::threads), s, a);                                           \
      else                                                                                      \
        launch(c, &k_z_inverse<T, P, TC>, &k_z_inverse_b<T, P, TC>, grid,                       \
               dim3(TC * ColPlan<P>::threads), s, a);                                           \
    });                                                                                         \
    break;
    DNSMI_FOR_EACH_P(X)
#undef X
    default: return c->fail(DNSMI_EINVAL, "unsupported padded z length");
  }
  return check_launch(c, "z_inverse");
}

template <int P>
struct XSplit {
  static constexpr bool value = Plan<P>::N2 % 2 == 0;  // split form available
  static constexpr int tpr = value ? 2 * Plan<P>::N1 : Plan<P>::N1;
  static constexpr int rows = (256 / tpr) > 0 ? 256 / tpr : 1;
};

template <typename T, int P>
static void launch_x_len(Ctx* c, const Bufs<T>& b, const cx<T>* xin, cx<T>* xout,
                         const double* base, const double* cbase, const double* nbase, int ny,
                         int em, hipStream_t s) {
  constexpr int R = XSplit<P>::rows;
  const int nrows = ny * c->Pz;
  const dim3 grid((nrows + R - 1) / R);
  bool split = false;
  if constexpr (XSplit<P>::value) split = c->xpass_split && em == EV_PLAIN;
  const XArgs a{xin, xout, b.twx, c->kx, base, cbase, nbase, c->nx, ny, c->Pz, ny, c->act, c->xref};
  if (split) {
    if constexpr (XSplit<P>::value)
      launch(c, &k_x_nonlinear_split<T, P, R>, &k_x_nonlinear_split_b<T, P, R>, grid,
             dim3(R * XSplit<P>::tpr), s, a);
  } else {
    constexpr int R1 = kRows;
    const dim3 grid1((nrows + R1 - 1) / R1), blk(R1 * Plan<P>::N1);
    if (em == EV_PLAIN) {
      launch(c, &k_x_nonlinear<T, P, R1, EV_PLAIN>, &k_x_nonlinear_b<T, P, R1, EV_PLAIN>, grid1, blk, s, a);
    } else if constexpr (std::is_same<T, float>::value) {
      if (em == EV_RECORD)
        launch(c, &k_x_nonlinear<T, P, R1, EV_RECORD>, &k_x_nonlinear_b<T, P, R1, EV_RECORD>, grid1, blk, s, a);
      else
        launch(c, &k_x_nonlinear<T, P, R1, EV_INC>, &k_x_nonlinear_b<T, P, R1, EV_INC>, grid1, blk, s, a);
    }
  }
}

// x pass over rows (y, z) of W[f][y][z][kx]: periodic (y = padded grid) and
// wall-bounded (y = the grid points) share it; the base flow profiles are
// given per y.  em: EvalMode (FP32 contexts with reference buffers only).
template <typename T>
int launch_x_pass(Ctx* c, const cx<T>* xin, cx<T>* xout, const double* base, const double* cbase,
                  const double* nbase, int ny, int kid, hipStream_t s, int em) {
  if (em != EV_PLAIN && (!std::is_same<T, float>::value || !c->xref))
    return c->fail(DNSMI_EINVAL, "split evaluation without FP32 reference buffers");
  Bufs<T> b = bufs_of<T>(c);
  ProfScope ps(c, kid, s);
  switch (c->Px) {
#define X(P)                                                                \
  case P:                                                                   \
    launch_x_len<T, P>(c, b, xin, xout, base, cbase, nbase, ny, em, s);    \
    break;
    DNSMI_FOR_EACH_P(X)
#undef X
    default: return c->fail(DNSMI_EINVAL, "unsupported padded x length");
  }
  return check_launch(c, "x_nonlinear");
}
template int launch_x_pass<double>(Ctx*, const cx<double>*, cx<double>*, const double*,
                                   const double*, const double*, int, int, hipStream_t, int);
template int launch_x_pass<float>(Ctx*, const cx<float>*, cx<float>*, const double*,
                                  const double*, const double*, int, int, hipStream_t, int);

template <typename T>
static int launch_x_nonlinear(Ctx* c, hipStream_t s, int em = EV_PLAIN) {
  Bufs<T> b = bufs_of<T>(c);
  return launch_x_pass<T>(c, b.B, b.A, c->base, c->cbase, c->nbase, c->Py, KID_X_NONLINEAR, s, em);
}

// z forward over columns (y, kx) of W[c][y][z][kx] -> W[c][y][kz][kx]; ny is
// the number of y planes (padded y for periodic, grid points for walls).
template <typename T>
int launch_z_forward_buf(Ctx* c, const cx<T>* in, cx<T>* out, int ny, int kid, hipStream_t s) {
  Bufs<T> b = bufs_of<T>(c);
  const int ntile = (c->Nx1 + c->tile_cols - 1) / c->tile_cols;
  const dim3 grid(ny * ntile, 3);  // one component per workgroup
  ProfScope ps(c, kid, s);
  switch (c->Pz) {
#define X(P)                                                                                   \
  case P:                                                                                      \
    with_tc(c, [&](auto tcv) {                                                                 \
      constexpr int TC = decltype(tcv)::value;                                                 \
      launch(c, &k_z_forward<T, P, TC>, &k_z_forward_b<T, P, TC>, grid,                         \
             dim3(TC * ColPlan<P>::threads), s, ZFwdArgs{in, out, b.twz, c->nz, ny, c->Nx1, c->act}); \
    });                                                                                        \
    break;
    DNSMI_FOR_EACH_P(X)
#undef X
    default: return c->fail(DNSMI_EINVAL, "unsupported padded z length");
  }
  return check_launch(c, "z_forward");
}
template int launch_z_forward_buf<double>(Ctx*, const cx<double>*, cx<double>*, int, int,
                                          hipStream_t);
template int launch_z_forward_buf<float>(Ctx*, const cx<float>*, cx<float>*, int, int,
                                         hipStream_t);

template <typename T>
static int launch_z_forward(Ctx* c, hipStream_t s) {
  Bufs<T> b = bufs_of<T>(c);
  return launch_z_forward_buf<T>(c, b.A, b.B, c->Py, KID_Z_FORWARD, s);
}

template <typename T, int P, int TC, int MODE, bool PADY>
static void launch_y_forward_p(Ctx* c, int nb, const YFwdArgs& a, hipStream_t s) {
  // Three components of 16 FP64 columns that take more than half a CU's LDS
  // leave one workgroup to it: with more workgroups than CUs nothing overlaps
  // one's transforms with another's loads, and the serial form is the faster
  // one.  FP64 step at 128^3 (508 workgroups): 839 us serial, 865 us side by
  // side; 64 x 128^2 (254): 437 and 415 us.  FP32 tiles leave two workgroups to
  // a CU; from 144 rows on the serial form is the faster one where nearly all
  // of those places are taken: mixed step at 128^3 (508) 708 and 715 us, 128 x
  // 96 x 128 562 and 568 us from a guess, but 128 x 128 x 96 (380) 547 and 540
  // us and 96 x 64 x 96 and 128 x 64 x 128 (285, 508; 96 rows) within 0.6 %.
  //
  // nb is one member's workgroups, in a batch too: the two forms sum the norm in
  // different orders, and a member's error equals its eager run's to the bit.
  // That costs large batches (16 x 64^3 FP64: 3446 us serial, 3480 us side by
  // side) what it gains small ones (4 x 32^3 FP64: 315 and 294 us).
  constexpr size_t tile = 3 * TC * P * sizeof(cx<T>);
  constexpr bool fp64 = std::is_same<T, double>::value;
  if constexpr (tile > (fp64 ? 80 : 50) * 1024) {
    if (nb > (fp64 ? kCUs : kCUs * 3 / 2)) {
      launch(c, &k_y_forward_serial<T, P, TC, MODE, PADY>, &k_y_forward_serial_b<T, P, TC, MODE, PADY>, dim3(nb),
             dim3(TC * ColPlan<P>::threads), s, a);
      return;
    }
  }
  launch(c, &k_y_forward<T, P, TC, MODE, PADY>, &k_y_forward_b<T, P, TC, MODE, PADY>, dim3(nb),
         dim3(3 * TC * ColPlan<P>::threads), s, a);
}

template <typename T, int MODE>
static int launch_y_forward(Ctx* c, const StepArgs& a, hipStream_t s, int* nblocks) {
  Bufs<T> b = bufs_of<T>(c);
  const int ntile = (c->Nx1 + c->tile_cols - 1) / c->tile_cols;
  const int nb = c->Nz1 * ntile;
  if (nblocks) *nblocks = nb;
  if ((MODE == MODE_CORRECT || MODE == MODE_CORRECT_CARRY) && nb > c->max_partials)
    return c->fail(DNSMI_EINVAL, "y_forward: too many blocks");
  ProfScope ps(c, KID_Y_FORWARD, s);
  const YFwdArgs ya{b.B, b.twy, c->kx, c->ky, c->kz, c->ny, c->Nz1, c->Nx1, a};
  switch (c->Py) {
#define X(P)                                                                                   \
  case P:                                                                                      \
    with_tc(c, [&](auto tcv) {                                                                 \
      constexpr int TC = decltype(tcv)::value;                                                 \
      if (c->Py != c->ny)                                                                      \
        launch_y_forward_p<T, P, TC, MODE, true>(c, nb, ya, s);                                \
      else                                                                                     \
        launch_y_forward_p<T, P, TC, MODE, false>(c, nb, ya, s);                               \
    });                                                                                        \
    break;
    DNSMI_FOR_EACH_P(X)
#undef X
    default: return c->fail(DNSMI_EINVAL, "unsupported padded y length");
  }
  return check_launch(c, "y_forward");
}

template <typename T, int MODE>
static int periodic_rhs_t(Ctx* c, const double* state, const StepArgs& a, hipStream_t s,
                          int* nblocks, int em) {
  int rc;
  if ((rc = launch_y_inverse<T>(c, state, s, em))) return rc;
  if ((rc = launch_z_inverse<T>(c, s))) return rc;
  if ((rc = launch_x_nonlinear<T>(c, s, em))) return rc;
  if ((rc = launch_z_forward<T>(c, s))) return rc;
  return launch_y_forward<T, MODE>(c, a, s, nblocks);
}

// One evaluation of N(state) in the context's current precision.  em: see
// EvalMode; EV_INC records a reference first when none is valid (the step's
// first corrector evaluation), and adds n_ref through a.nref; FP64 passes
// are always EV_PLAIN.
template <int MODE>
static int periodic_rhs_mode(Ctx* c, const double* state, StepArgs a, hipStream_t s,
                             int* nblocks, int em = EV_PLAIN) {
  if (em == EV_INC && !c->ref_valid) em = EV_RECORD;
  if (!c->fp32 || !c->split) em = EV_PLAIN;
  a.nref = em == EV_INC ? c->nref : nullptr;
  a.nref_out = em == EV_RECORD ? c->nref : nullptr;
  if (!c->fp32) return periodic_rhs_t<double, MODE>(c, state, a, s, nblocks, EV_PLAIN);
  const int rc = periodic_rhs_t<float, MODE>(c, state, a, s, nblocks, em);
  if (rc == DNSMI_OK && em == EV_RECORD) c->ref_valid = true;
  return rc;
}

static StepArgs step_args(Ctx* c) {
  StepArgs a{};
  a.dt = c->cfg.dt;
  a.c = c->cfg.implicitness;
  a.re = c->cfg.re;
  a.partials = c->partials;
  a.act = c->act;
  return a;
}

int periodic_get_rhs(Ctx* c, const double* state, double* rhs, hipStream_t s) {
  StepArgs a = step_args(c);
  a.rhs_out = rhs;
  return periodic_rhs_mode<MODE_RHS>(c, state, a, s, nullptr);
}

// N(state) into rhs, the first evaluation of a guessed step: a plain
// evaluation, after which the step's first corrector evaluation records the
// reference of the split evaluations.
int periodic_guess_rhs(Ctx* c, const double* state, double* rhs, hipStream_t s) {
  StepArgs a = step_args(c);
  a.rhs_out = rhs;
  c->ref_valid = false;
  return periodic_rhs_mode<MODE_RHS>(c, state, a, s, nullptr, EV_PLAIN);
}

// The split evaluations of a step are increments over its first corrector
// iterate: the predictor's evaluation N(u^n) is plain, the first corrector
// evaluation N(u^1) records u_ref = u^1 (so every later increment is of the
// corrector's own size, far smaller than u^1 - u^n).
int periodic_predict_and_correct(Ctx* c, const double* state, double* pred, double* rhs_next,
                                 double* err, hipStream_t s) {
  StepArgs a = step_args(c);
  a.state = state;
  a.pred = pred;
  a.rhs_out = c->rhs0;
  int rc = periodic_rhs_mode<MODE_PREDICT>(c, state, a, s, nullptr, EV_PLAIN);
  if (rc) return rc;
  StepArgs b = step_args(c);
  b.rhs_prev = c->rhs0;
  b.pred = pred;
  b.rhs_out = rhs_next;
  int nb = 0;
  c->ref_valid = false;
  rc = periodic_rhs_mode<MODE_CORRECT>(c, pred, b, s, &nb, EV_RECORD);
  if (rc) return rc;
  return finalize_norm(c, nb, err, s);
}

// The carry forms of predict_and_correct and iterate_correction (see the K5
// epilogue modes): `carry` receives B from the predictor and is read by
// every corrector pass; split evaluations keep B + c ildt_2 N(u_ref) in
// n_ref.  A pass reads B and the iterate and writes the iterate (3 S, where
// the incremental form also reads N_prev and writes N: 4 S).
int periodic_predict_and_correct_carry(Ctx* c, const double* state, double* pred, double* carry,
                                       double* err, hipStream_t s) {
  StepArgs a = step_args(c);
  a.state = state;
  a.pred = pred;
  a.rhs_out = carry;
  int rc = periodic_rhs_mode<MODE_PREDICT_CARRY>(c, state, a, s, nullptr, EV_PLAIN);
  if (rc) return rc;
  StepArgs b = step_args(c);
  b.rhs_prev = carry;
  b.pred = pred;
  int nb = 0;
  c->ref_valid = false;
  rc = periodic_rhs_mode<MODE_CORRECT_CARRY>(c, pred, b, s, &nb, EV_RECORD);
  if (rc) return rc;
  return finalize_norm(c, nb, err, s);
}

int periodic_iterate_correction_carry(Ctx* c, double* pred, const double* carry, double* err, hipStream_t s) {
  StepArgs b = step_args(c);
  b.rhs_prev = carry;
  b.pred = pred;
  int nb = 0;
  int rc = periodic_rhs_mode<MODE_CORRECT_CARRY>(c, pred, b, s, &nb, EV_INC);
  if (rc) return rc;
  return finalize_norm(c, nb, err, s);
}

int periodic_iterate_correction(Ctx* c, double* pred, const double* rhs_prev, double* rhs_next,
                                double* err, hipStream_t s) {
  StepArgs b = step_args(c);
  b.rhs_prev = rhs_prev;
  b.pred = pred;
  b.rhs_out = rhs_next;
  int nb = 0;
  int rc = periodic_rhs_mode<MODE_CORRECT>(c, pred, b, s, &nb, EV_INC);
  if (rc) return rc;
  return finalize_norm(c, nb, err, s);
}

static PointArgs point_args(Ctx* c) {
  PointArgs p{};
  p.dt = c->cfg.dt;
  p.c = c->cfg.implicitness;
  p.re = c->cfg.re;
  p.ny = c->ny;
  p.Nz1 = c->Nz1;
  p.Nx1 = c->Nx1;
  p.n = (long long)c->Ny1 * c->Nz1 * c->Nx1;
  p.partials = c->partials;
  return p;
}

static int pw_blocks(const PointArgs& p) { return (int)((p.n + 255) / 256); }

int periodic_predict(Ctx* c, const double* state, const double* rhs, double* pred,
                     hipStream_t s) {
  PointArgs p = point_args(c);
  p.a = state;
  p.b = rhs;
  p.out = pred;
  ProfScope ps(c, KID_POINTWISE, s);
  launch(c, &k_pointwise<PW_PREDICT>, &k_pointwise_b<PW_PREDICT>, dim3(pw_blocks(p)), dim3(256), s,
         PwArgs{p, c->kx, c->ky, c->kz});
  return check_launch(c, "predict");
}

int periodic_correct(Ctx* c, const double* pred_in, const double* rhs_prev,
                     const double* rhs_next, double* pred_out, double* corr, hipStream_t s) {
  PointArgs p = point_args(c);
  p.a = pred_in;
  p.b = rhs_prev;
  p.c2 = rhs_next;
  p.out = pred_out;
  p.out2 = corr;
  ProfScope ps(c, KID_POINTWISE, s);
  launch(c, &k_pointwise<PW_CORRECT>, &k_pointwise_b<PW_CORRECT>, dim3(pw_blocks(p)), dim3(256), s,
         PwArgs{p, c->kx, c->ky, c->kz});
  return check_launch(c, "correct");
}

int periodic_norm(Ctx* c, const double* corr, double* err, hipStream_t s) {
  PointArgs p = point_args(c);
  p.a = corr;
  const int nb = pw_blocks(p);
  if (nb > c->max_partials) return c->fail(DNSMI_EINVAL, "norm: too many blocks");
  ProfScope ps(c, KID_POINTWISE, s);
  launch(c, &k_pointwise<PW_NORM>, &k_pointwise_b<PW_NORM>, dim3(nb), dim3(256), s, PwArgs{p, c->kx, c->ky, c->kz});
  int rc = check_launch(c, "norm");
  if (rc) return rc;
  return finalize_norm(c, nb, err, s);
}

int periodic_correct_velocity(Ctx* c, double* state, double* err, hipStream_t s) {
  PointArgs p = point_args(c);
  p.a = state;
  p.out = state;
  const int nb = pw_blocks(p);
  if (!c->cfg.correct_divergence) {
    // only the mean mode is zeroed (a kernel, not a memset, so that the
    // call can sit inside a captured graph)
    if (err) return c->fail(DNSMI_EINVAL, "measure_corrections needs correct_divergence");
    ProfScope ps(c, KID_POINTWISE, s);
    launch(c, &k_zero_mean, &k_zero_mean_b, dim3(1), dim3(64), s, ZmArgs{state, p.n});
    return check_launch(c, "zero_mean");
  }
  if (err) {
    if (nb > c->max_partials) return c->fail(DNSMI_EINVAL, "too many blocks");
    ProfScope ps(c, KID_POINTWISE, s);
    launch(c, &k_pointwise<PW_DIVFREE_NORM>, &k_pointwise_b<PW_DIVFREE_NORM>, dim3(nb), dim3(256), s,
           PwArgs{p, c->kx, c->ky, c->kz});
    int rc = check_launch(c, "correct_velocity");
    if (rc) return rc;
    return finalize_norm(c, nb, err, s);
  }
  ProfScope ps(c, KID_POINTWISE, s);
  launch(c, &k_pointwise<PW_DIVFREE>, &k_pointwise_b<PW_DIVFREE>, dim3(nb), dim3(256), s,
         PwArgs{p, c->kx, c->ky, c->kz});
  return check_launch(c, "correct_velocity");
}

// ------------------------------------------------------------------ set-up
bool supported_length(int P) {
  switch (P) {
#define X(P_) case P_:
    DNSMI_FOR_EACH_P(X)
#undef X
    return true;
    default: return false;
  }
}

template <typename T>
static std::vector<cx<T>> host_twiddles(int P) {
  std::vector<cx<T>> t(P);
  for (int m = 0; m < P; ++m) {
    const CosSin v = ct_unit(m, P);
    t[m] = {static_cast<T>(v.c), static_cast<T>(v.s)};
  }
  return t;
}

static int upload(Ctx* c, void** dst, const void* src, size_t bytes) {
  *dst = c->alloc(bytes);
  if (!*dst) return c->fail(DNSMI_ENOMEM, "device allocation failed");
  hipError_t e = hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice);
  if (e != hipSuccess) return c->fail(DNSMI_EHIP, hipGetErrorString(e));
  return DNSMI_OK;
}

int setup_twiddles(Ctx* c) {
  const int Ps[3] = {c->Px, c->Py, c->Pz};
  for (int a = 0; a < 3; ++a) {
    if (!Ps[a]) continue;
    auto t64 = host_twiddles<double>(Ps[a]);
    auto t32 = host_twiddles<float>(Ps[a]);
    int rc = upload(c, &c->tw64[a], t64.data(), t64.size() * sizeof(t64[0]));
    if (rc) return rc;
    rc = upload(c, &c->tw32[a], t32.data(), t32.size() * sizeof(t32[0]));
    if (rc) return rc;
  }
  return DNSMI_OK;
}

int upload_doubles(Ctx* c, double** dst, const std::vector<double>& v) {
  return upload(c, reinterpret_cast<void**>(dst), v.data(), v.size() * sizeof(double));
}

// Harmonics (operators.py:18-56) times 2 pi / L, in the reference's
// operation order ((h * 2) * pi / L).
std::vector<double> real_wavenumbers(int n, double L) {
  std::vector<double> k(n / 2);
  for (int i = 0; i < n / 2; ++i) k[i] = (double)(i * 2) * kPi / L;
  return k;
}
std::vector<double> complex_wavenumbers(int n, double L) {
  std::vector<double> k(n - 1);
  for (int i = 0; i < n - 1; ++i) {
    const int h = i < n / 2 ? i : i - (n - 1);
    k[i] = (double)(h * 2) * kPi / L;
  }
  return k;
}

// ------------------------------------------------------------------ autotuner
// Every variant below computes the same result; at context creation each
// alternative is timed on the context's own work buffers (HIP events, a
// warm-up launch then `reps` launches) and the fastest is kept.  The choices
// are readable through dnsmi_tuning().
template <typename F>
static double time_launches(F&& launch, int reps) {
  hipEvent_t a = nullptr, b = nullptr;
  if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess) return 1e30;
  launch();
  (void)hipEventRecord(a, nullptr);
  for (int i = 0; i < reps; ++i) launch();
  (void)hipEventRecord(b, nullptr);
  float ms = 0.f;
  if (hipEventSynchronize(b) != hipSuccess || hipEventElapsedTime(&ms, a, b) != hipSuccess) ms = 1e30f;
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  return ms;
}

template <typename T>
static int periodic_autotune_t(Ctx* c) {
  const int reps = 3;
  std::string log;
  // each variant timed in three alternating rounds, the best round kept
  // (a single round is swayed by clock ramps and a profiler's first-launch
  // costs, which fall on whichever variant runs first)
  auto pick = [&](const char* what, bool& flag, auto&& launch) {
    double t0 = 1e30, t1 = 1e30;
    for (int round = 0; round < 3; ++round) {
      flag = false;
      t0 = std::min(t0, time_launches(launch, reps));
      flag = true;
      t1 = std::min(t1, time_launches(launch, reps));
    }
    flag = t1 < t0;
    char buf[160];
    snprintf(buf, sizeof buf, "%s=%s(%.1f/%.1f us) ", what, flag ? "alt" : "base",
             1e3 * t0 / reps, 1e3 * t1 / reps);
    log += buf;
  };
  const double* state = c->rhs0;  // zeroed scratch stands in for a state
  pick("y_inverse_seq", c->yinv_seq, [&] { launch_y_inverse<T>(c, state, nullptr); });
  pick("z_inverse_seq", c->zinv_seq, [&] { launch_z_inverse<T>(c, nullptr); });
  bool split_ok = false;
  switch (c->Px) {
#define X(P) case P: split_ok = XSplit<P>::value; break;
    DNSMI_FOR_EACH_P(X)
#undef X
    default: break;
  }
  if (split_ok) pick("x_split", c->xpass_split, [&] { launch_x_nonlinear<T>(c, nullptr); });
  // the column tile of the y and z passes: one whole RHS with 16 and with 8
  {
    double* out = static_cast<double*>(c->alloc(c->spec_elems * 16));
    if (!out) return c->fail(DNSMI_ENOMEM, "autotune: device allocation failed");
    StepArgs a = step_args(c);
    a.rhs_out = out;
    auto rhs = [&] { periodic_rhs_t<T, MODE_RHS>(c, state, a, nullptr, nullptr, EV_PLAIN); };
    double t16 = 1e30, t8 = 1e30;
    for (int round = 0; round < 3; ++round) {
      c->tile_cols = kTC;
      t16 = std::min(t16, time_launches(rhs, reps));
      c->tile_cols = kTCMin;
      t8 = std::min(t8, time_launches(rhs, reps));
    }
    c->tile_cols = t8 < t16 ? kTCMin : kTC;
    char buf[160];
    snprintf(buf, sizeof buf, "tile_cols=%d(16: %.1f / 8: %.1f us) ", c->tile_cols, 1e3 * t16 / reps,
             1e3 * t8 / reps);
    log += buf;
    // non-temporal stores of the z-inverse output: they keep the caches for
    // the lines that pass still reads, but the next pass then reads all of
    // its input from memory, so the choice is timed over a whole RHS.  FP64
    // only: the FP32 output (half the bytes) is read back from the caches
    // by the x pass, and in FP32 the isolated timings are near ties that
    // the stepping loop, with its recorded reference fields, does not bear
    // out.
    double tp = 1e30, tn = 1e30;
    if (sizeof(T) == 8) {
      for (int round = 0; round < 3; ++round) {
        c->zinv_nt = false;
        tp = std::min(tp, time_launches(rhs, reps));
        c->zinv_nt = true;
        tn = std::min(tn, time_launches(rhs, reps));
      }
    }
    c->zinv_nt = tn < tp;
    c->release(out);
    if (sizeof(T) == 8)
      snprintf(buf, sizeof buf, "z_inverse_stream=%s(%.1f/%.1f us) ", c->zinv_nt ? "alt" : "base",
               1e3 * tp / reps, 1e3 * tn / reps);
    else
      snprintf(buf, sizeof buf, "z_inverse_stream=base(fp32) ");
    log += buf;
  }
  c->tuning = log;
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? DNSMI_OK : c->fail(DNSMI_EHIP, std::string("autotune: ") + hipGetErrorString(e));
}

int periodic_autotune(Ctx* c) {
  if (hipMemset(c->bufA, 0, c->bufA_bytes) != hipSuccess ||
      hipMemset(c->bufB, 0, c->bufB_bytes) != hipSuccess ||
      hipMemset(c->rhs0, 0, c->spec_elems * 16) != hipSuccess)
    return c->fail(DNSMI_EHIP, "autotune: memset");
  return c->fp32 ? periodic_autotune_t<float>(c) : periodic_autotune_t<double>(c);
}

int periodic_setup(Ctx* c) {
  const dnsmi_config& g = c->cfg;
  if (g.nx % 2 || g.ny % 2 || g.nz % 2 || g.nx < 4 || g.ny < 4 || g.nz < 4)
    return c->fail(DNSMI_EINVAL, "nx, ny, nz must be even and >= 4");
  if (g.oversampling_factor != 3) return c->fail(DNSMI_EINVAL, "oversampling_factor must be 3");
  c->nx = g.nx;
  c->ny = g.ny;
  c->nz = g.nz;
  c->Nx1 = g.nx / 2;
  c->Ny1 = g.ny - 1;
  c->Nz1 = g.nz - 1;
  c->Px = 3 * g.nx / 2;
  c->Pz = 3 * g.nz / 2;
  c->Py = g.oversample_y ? 3 * g.ny / 2 : g.ny;
  if (!supported_length(c->Px) || !supported_length(c->Py) || !supported_length(c->Pz))
    return c->fail(DNSMI_EINVAL, "padded lengths must be one of 12,16,24,32,48,64,72,96,128,144,192");
  c->spec_elems = 3LL * c->Ny1 * c->Nz1 * c->Nx1;
  // FP64-sized in the mixed form too: its escalated passes run in FP64
  const size_t cxs = 16;
  const size_t w1 = 5ull * c->Py * c->Nz1 * c->Nx1, w3 = 3ull * c->Py * c->Pz * c->Nx1;
  const size_t w2 = 6ull * c->Py * c->Pz * c->Nx1, w4 = 3ull * c->Py * c->Nz1 * c->Nx1;
  c->bufA_bytes = (w1 > w3 ? w1 : w3) * cxs;
  c->bufB_bytes = (w2 > w4 ? w2 : w4) * cxs;
  c->bufA = c->alloc(c->bufA_bytes);
  c->bufB = c->alloc(c->bufB_bytes);
  c->rhs0 = static_cast<double*>(c->alloc(c->spec_elems * 16));
  if (c->split) {
    c->nref = static_cast<double*>(c->alloc(c->spec_elems * 16));
    c->uref = static_cast<double*>(c->alloc(c->spec_elems * 16));
    c->xref = static_cast<float*>(c->alloc(6ull * c->Py * c->Pz * c->Px * sizeof(float)));
    if (!c->nref || !c->uref || !c->xref) return c->fail(DNSMI_ENOMEM, "device allocation failed");
  }
  const long long per_comp = (long long)c->Ny1 * c->Nz1 * c->Nx1;
  // norm partials (one per y-forward block) and the statistics' two per
  // 256-mode block, whichever is larger
  const long long stats_partials = 2 * ((per_comp + 255) / 256);
  const long long norm_partials = (per_comp + 255) / 256 + (long long)c->Nz1 * ((c->Nx1 + kTCMin - 1) / kTCMin);
  c->max_partials = (int)((stats_partials > norm_partials ? stats_partials : norm_partials) + 1024);
  c->partials = static_cast<double*>(c->alloc(sizeof(double) * c->max_partials));
  if (!c->bufA || !c->bufB || !c->rhs0 || !c->partials)
    return c->fail(DNSMI_ENOMEM, "device allocation failed");
  int rc = setup_twiddles(c);
  if (rc) return rc;
  if ((rc = upload_doubles(c, &c->kx, real_wavenumbers(g.nx, g.lx)))) return rc;
  if ((rc = upload_doubles(c, &c->ky, complex_wavenumbers(g.ny, g.ly)))) return rc;
  if ((rc = upload_doubles(c, &c->kz, complex_wavenumbers(g.nz, g.lz)))) return rc;

  // Base flow on the padded y grid (flows/monochromatic.py:116-208):
  // U_x = sin(2 pi y / Ly) (Kolmogorov) or cos (Waleffe), evaluated as the
  // inverse real transform of the single harmonic q_f = 1.
  const int Py = c->Py;
  std::vector<double> base(3 * Py, 0.0), dbase(3 * Py, 0.0), cbase(3 * Py, 0.0),
      nbase(3 * Py, 0.0);
  if (g.system == DNSMI_KOLMOGOROV || g.system == DNSMI_WALEFFE) {
    const double kf = 2 * kPi / g.ly;
    for (int y = 0; y < Py; ++y) {
      const CosSin t = ct_unit(y, Py);
      // irfft of coefficient -0.5j (sin) or 0.5 (cos) at q_f = 1, times 2
      base[y] = g.system == DNSMI_KOLMOGOROV ? t.s : t.c;
      dbase[y] = g.system == DNSMI_KOLMOGOROV ? kf * t.c : -kf * t.s;
    }
  } else if (g.system != DNSMI_DECAYING_BOX) {
    return c->fail(DNSMI_EINVAL, "not a periodic system");
  }
  for (int y = 0; y < Py; ++y) {
    cbase[2 * Py + y] = -dbase[y];
    nbase[1 * Py + y] = base[y] * dbase[y];
  }
  const double tilt = kPi * g.tilt_degree / 180.0;
  if (tilt != 0.0) {
    const double sn = std::sin(tilt), cs = std::cos(tilt);
    for (int y = 0; y < Py; ++y) {
      base[2 * Py + y] = sn * base[y];
      base[y] *= cs;
      cbase[0 * Py + y] = -sn * cbase[2 * Py + y];
      cbase[2 * Py + y] *= cs;
    }
  }
  if ((rc = upload_doubles(c, &c->base, base))) return rc;
  if ((rc = upload_doubles(c, &c->cbase, cbase))) return rc;
  if ((rc = upload_doubles(c, &c->nbase, nbase))) return rc;
  if (c->cfg.tile_cols == 0) return periodic_autotune(c);
  return DNSMI_OK;
}

}  // namespace dnsmi
