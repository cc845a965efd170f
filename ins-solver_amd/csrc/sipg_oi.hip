// Over-integrated variable-coefficient SIPG operator (the reference's
// FactorPoissonMatrixFreeDiagOI{2D,3D}, selected by [pressure-solve] over_int,
// src/solvers/2d/mp_ins_solver.cpp:98-100,580-600): the coefficient is given at the cubature
// points of the cells (kv) and of their faces (ks), and every integral of the operator is taken
// with those rules (oi.h). Element-centric like the nodal operator: a trace pass stores, for
// every face point of every cell, u and T = sJ k n.grad u (own outward normal); the element
// pass gathers the neighbour's values at the matching point (a permutation of the symmetric
// face rule), then
//
//   out_i = sum_q wv_q kv_q grad phi_i . Kt grad u (x_q)                    (volume, Kt = J grad xi grad xi^T)
//         + sum_f sum_q ws_q [ phi_i F + (beta_f . grad phi_i) sig ](x_fq)   (faces)
//   F = (tauS [u] - (T- - T+)) / 2,  sig = -ks [u] / 2,  beta_f = Kt alpha_f = sJ grad xi . n
//
// Dirichlet ghost u+ = -u-, T+ = -T- (vmf_2d_mult_avg_jump.h:32-38); Neumann faces none.
#include <hip/hip_runtime.h>

#include <stdexcept>
#include <string>

#include "dg_layout.h"
#include "kernels.h"
#include "reduce.h"
#include "sipg_cell.h"

namespace insp {

namespace {

// Points of the rules (oi.h): triangle volume / 3D faces 3, 6, 12, 16; edges 2N+1; tetrahedron
// volume (N+2)^3.
constexpr int oi_nv(int dim, int N) {
  return dim == 2 ? (N == 1 ? 3 : N == 2 ? 6 : N == 3 ? 12 : 16) : (N + 2) * (N + 2) * (N + 2);
}
constexpr int oi_ns(int dim, int N) {
  return dim == 2 ? 2 * N + 1 : (N == 1 ? 3 : N == 2 ? 6 : N == 3 ? 12 : 16);
}

template <int DIM, int N>
struct OiL {
  static constexpr int Np = DIM == 2 ? (N + 1) * (N + 2) / 2 : (N + 1) * (N + 2) * (N + 3) / 6;
  static constexpr int Nf = DIM + 1, nv = oi_nv(DIM, N), ns = oi_ns(DIM, N);
  static constexpr int off_GV = 0, off_wv = off_GV + DIM * nv * Np, off_IS = off_wv + nv;
  static constexpr int off_GS = off_IS + Nf * ns * Np, off_ws = off_GS + Nf * DIM * ns * Np;
  static constexpr int size = off_ws + ns;
  static constexpr int nperm = DIM == 2 ? 2 : 6;
};

inline void check(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    throw std::runtime_error(std::string("kernel launch failed: ") + what + ": " + hipGetErrorString(e));
}

template <int DIM, typename T>
__device__ __forceinline__ void face_beta(const T* K, int f, T* beta) {
#pragma unroll
  for (int s = 0; s < DIM; ++s) {
    T b = 0;
#pragma unroll
    for (int r = 0; r < DIM; ++r) b += (T)face_alpha(DIM, f, r) * K[kidx(DIM, r, s)];
    beta[s] = b;
  }
}

template <int DIM, int N, typename T>
__global__ void __launch_bounds__(256)
k_trace_oi(int64_t E, int64_t stride, const T* __restrict__ u, const double* __restrict__ Kt,
           const T* __restrict__ ks, const T* __restrict__ Cp, T* __restrict__ tU, T* __restrict__ tT) {
  using L = OiL<DIM, N>;
  const cptr<T> C = as_const(Cp);
  const int64_t e = xcd_block() * blockDim.x + threadIdx.x;
  if (e >= E) return;
  constexpr int NK = DIM == 2 ? 3 : 6;
  T uu[L::Np], K[NK];
#pragma unroll
  for (int m = 0; m < L::Np; ++m) uu[m] = u[m * stride + e];
#pragma unroll
  for (int k = 0; k < NK; ++k) K[k] = (T)Kt[k * stride + e];
#pragma unroll
  for (int f = 0; f < L::Nf; ++f) {
    T beta[DIM];
    face_beta<DIM>(K, f, beta);
    for (int q = 0; q < L::ns; ++q) {
      T U = 0, Tn = 0;
#pragma unroll
      for (int m = 0; m < L::Np; ++m) U = fma(C[L::off_IS + (f * L::ns + q) * L::Np + m], uu[m], U);
#pragma unroll
      for (int s = 0; s < DIM; ++s) {
        T g = 0;
#pragma unroll
        for (int m = 0; m < L::Np; ++m) g = fma(C[L::off_GS + ((f * DIM + s) * L::ns + q) * L::Np + m], uu[m], g);
        Tn = fma(beta[s], g, Tn);
      }
      const int64_t idx = (int64_t)(f * L::ns + q) * stride + e;
      tU[idx] = U;
      tT[idx] = ks[idx] * Tn;
    }
  }
}

template <int DIM, int N, typename T>
__global__ void __launch_bounds__(256)
k_apply_oi(int64_t E, int64_t stride, const T* __restrict__ u, const T* __restrict__ tU,
           const T* __restrict__ tT, const double* __restrict__ Kt, const double* __restrict__ tauS,
           const int* __restrict__ nbr, const int* __restrict__ code, const int* __restrict__ bctype,
           const T* __restrict__ kv, const T* __restrict__ ks, const T* __restrict__ Cp,
           const int* __restrict__ qmapp, T* __restrict__ out, double* __restrict__ partial) {
  using L = OiL<DIM, N>;
  const cptr<T> C = as_const(Cp);
  const cptr<int> qmap = as_const(qmapp);
  const int64_t e = xcd_block() * blockDim.x + threadIdx.x;
  double dotv = 0.0;
  if (e < E) {
    constexpr int NK = DIM == 2 ? 3 : 6;
    T uu[L::Np], acc[L::Np], K[NK];
#pragma unroll
    for (int m = 0; m < L::Np; ++m) {
      uu[m] = u[m * stride + e];
      acc[m] = 0;
    }
#pragma unroll
    for (int k = 0; k < NK; ++k) K[k] = (T)Kt[k * stride + e];
    // volume: k at the cubature points
    for (int q = 0; q < L::nv; ++q) {
      T g[DIM];
#pragma unroll
      for (int s = 0; s < DIM; ++s) {
        T a = 0;
#pragma unroll
        for (int m = 0; m < L::Np; ++m) a = fma(C[L::off_GV + (s * L::nv + q) * L::Np + m], uu[m], a);
        g[s] = a;
      }
      const T wk = C[L::off_wv + q] * kv[(int64_t)q * stride + e];
#pragma unroll
      for (int r = 0; r < DIM; ++r) {
        T h = 0;
#pragma unroll
        for (int s = 0; s < DIM; ++s) h = fma(K[kidx(DIM, r, s)], g[s], h);
        h *= wk;
#pragma unroll
        for (int i = 0; i < L::Np; ++i) acc[i] = fma(C[L::off_GV + (r * L::nv + q) * L::Np + i], h, acc[i]);
      }
    }
    // faces at the face points
#pragma unroll
    for (int f = 0; f < L::Nf; ++f) {
      const int nb = nbr[f * stride + e];
      int mode = 0, fn = 0, p = 0;
      if (nb >= 0) {
        const int c = code[f * stride + e];
        fn = c / L::nperm;
        p = c - fn * L::nperm;
      } else {
        mode = bctype[-nb - 1] == 0 ? 1 : 2;
      }
      if (mode == 2) continue;
      T beta[DIM];
      face_beta<DIM>(K, f, beta);
      const T ts = (T)tauS[f * stride + e];
      for (int q = 0; q < L::ns; ++q) {
        const int64_t own = (int64_t)(f * L::ns + q) * stride + e;
        const T Um = tU[own], Tm = tT[own];
        T Up, Tp;
        if (mode == 0) {
          const int64_t nidx = (int64_t)(fn * L::ns + qmap[p * L::ns + q]) * stride + nb;
          Up = tU[nidx];
          Tp = tT[nidx];
        } else {
          Up = -Um;
          Tp = -Tm;
        }
        const T w = C[L::off_ws + q];
        const T jump = Um - Up;
        const T F = w * (T)0.5 * (ts * jump - (Tm - Tp));
        const T sig = w * (T)-0.5 * ks[own] * jump;
#pragma unroll
        for (int i = 0; i < L::Np; ++i) {
          T dn = 0;
#pragma unroll
          for (int s = 0; s < DIM; ++s) dn = fma(beta[s], C[L::off_GS + ((f * DIM + s) * L::ns + q) * L::Np + i], dn);
          acc[i] = fma(C[L::off_IS + (f * L::ns + q) * L::Np + i], F, fma(dn, sig, acc[i]));
        }
      }
    }
#pragma unroll
    for (int i = 0; i < L::Np; ++i) {
      out[i * stride + e] = acc[i];
      dotv += (double)uu[i] * (double)acc[i];
    }
  }
  if (partial) {
    const double t = block_sum1<256>(dotv);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
  }
}

// The same two passes with four waves to a cell (as sipg_split.h does for the nodal operator: 64 cells a
// block, the waves' parts of A u meet in LDS): wave w takes face w, a share of the volume points that
// balances the waves, and with them a quarter of the serial chain of an over-integrated cell (64 volume
// and 24 face points at 3D order 2). The neighbour's point is fetched one point ahead. FP64 calls, one
// thread per cell / four waves: 3D order 2, 29k cells 79.7 / 35.4 us, 1.05M 632 / 559; 3D order 3, 48k
// 293 / 104, 664k 1410 / 1026; 3D order 4, 35k 724 / 360, 384k 2644 / 2103; 2D order 4, 20k 53.6 / 28.2,
// 1.28M 584 / 589: the longer a cell's chain, the more even a full chip gains, so it is taken at every
// size.
template <int DIM, int N>
struct OiShare {
  int b[5];
  constexpr OiShare() : b{} {
    using L = OiL<DIM, N>;
    const int col = 2 * DIM * L::Np, face = L::ns * L::Np * (DIM + 2);
    int done = 0;
    for (int w = 0; w < 4; ++w) {
      b[w] = done;
      const int faces_left = (L::Nf > w ? L::Nf - w : 0) * face;
      int take = (((L::nv - done) * col + faces_left) / (4 - w) - (w < L::Nf ? face : 0) + col / 2) / col;
      if (take < 0) take = 0;
      if (w == 3 || done + take > L::nv) take = L::nv - done;
      done += take;
    }
    b[4] = L::nv;
  }
};

template <int DIM, int N, typename T>
__global__ void __launch_bounds__(256)
k_trace_oi_split(int64_t E, int64_t stride, const T* __restrict__ u, const double* __restrict__ Kt,
                 const T* __restrict__ ks, const T* __restrict__ Cp, T* __restrict__ tU, T* __restrict__ tT) {
  using L = OiL<DIM, N>;
  constexpr int NK = DIM == 2 ? 3 : 6, NQ = L::Nf * L::ns;
  const cptr<T> C = as_const(Cp);
  const int64_t e = xcd_block() * 64 + (threadIdx.x & 63);
  if (e >= E) return;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  T uu[L::Np], K[NK];
#pragma unroll
  for (int m = 0; m < L::Np; ++m) uu[m] = u[m * stride + e];
#pragma unroll
  for (int k = 0; k < NK; ++k) K[k] = (T)Kt[k * stride + e];
  // point g of the cell's Nf * ns, a quarter of them to a wave
  for (int g = NQ * w / 4; g < NQ * (w + 1) / 4; ++g) {
    const int f = g / L::ns, q = g - f * L::ns;
    T beta[DIM];
#pragma unroll
    for (int s = 0; s < DIM; ++s) {
      T b = 0;
#pragma unroll
      for (int r = 0; r < DIM; ++r) {
        T al = 0;
#pragma unroll
        for (int k = 0; k < L::Nf; ++k) al = f == k ? (T)face_alpha(DIM, k, r) : al;
        b = fma(al, K[kidx(DIM, r, s)], b);
      }
      beta[s] = b;
    }
    T U = 0, Tn = 0;
#pragma unroll
    for (int m = 0; m < L::Np; ++m) U = fma(C[L::off_IS + g * L::Np + m], uu[m], U);
#pragma unroll
    for (int s = 0; s < DIM; ++s) {
      T d = 0;
#pragma unroll
      for (int m = 0; m < L::Np; ++m) d = fma(C[L::off_GS + ((f * DIM + s) * L::ns + q) * L::Np + m], uu[m], d);
      Tn = fma(beta[s], d, Tn);
    }
    const int64_t idx = (int64_t)g * stride + e;
    tU[idx] = U;
    tT[idx] = ks[idx] * Tn;
  }
}

template <int DIM, int N, typename T, int W>
__device__ __forceinline__ void
oi_quarter(int64_t e, int64_t stride, const T* __restrict__ u, const T* __restrict__ tU,
           const T* __restrict__ tT, const double* __restrict__ Kt, const double* __restrict__ tauS,
           const int* __restrict__ nbr, const int* __restrict__ bctype, const T* __restrict__ kv,
           const T* __restrict__ ks, cptr<T> C, cptr<int> qmap, T (&acc)[OiL<DIM, N>::Np]) {
  using L = OiL<DIM, N>;
  constexpr int NK = DIM == 2 ? 3 : 6;
  constexpr OiShare<DIM, N> share;
  constexpr bool has_face = W < L::Nf;
  constexpr int F0 = has_face ? W : 0;
  int nb = 0;
  T ts = 0;
  if constexpr (has_face) {
    nb = nbr[F0 * stride + e];
    ts = (T)tauS[F0 * stride + e];
  }
  T uu[L::Np], K[NK];
#pragma unroll
  for (int m = 0; m < L::Np; ++m) {
    uu[m] = u[m * stride + e];
    acc[m] = 0;
  }
#pragma unroll
  for (int k = 0; k < NK; ++k) K[k] = (T)Kt[k * stride + e];
  int mode = 2;  // 0 interior, 1 Dirichlet, 2 no terms
  int64_t own = 0, nbase = 0;
  cptr<int> map = qmap;
  if constexpr (has_face) {
    mode = nb >= 0 ? 0 : (bctype[-nb - 1] == 0 ? 1 : 2);
    const int c = nb & 31, fn = nb >= 0 ? c / L::nperm : F0, p = nb >= 0 ? c - fn * L::nperm : 0;
    own = (int64_t)F0 * L::ns * stride + e;
    nbase = (int64_t)fn * L::ns * stride + (nb >= 0 ? (int64_t)(nb >> 5) : e);
    map = qmap + p * L::ns;
  }
  // values of the first face point, in flight during the volume term
  T Um = 0, Tm = 0, Up = 0, Tp = 0, kq = 0;
  auto fetch = [&](int q) {
    const int64_t n = nbase + (int64_t)map[q] * stride, o = own + (int64_t)q * stride;
    Um = tU[o];
    Tm = tT[o];
    kq = ks[o];
    Up = tU[n];
    Tp = tT[n];
  };
  if constexpr (has_face) fetch(0);
  T kn = share.b[W] < share.b[W + 1] ? kv[(int64_t)share.b[W] * stride + e] : (T)0;
#pragma unroll 1
  for (int q = share.b[W]; q < share.b[W + 1]; ++q) {
    const T wk = C[L::off_wv + q] * kn;
    kn = kv[(int64_t)(q + 1 < share.b[W + 1] ? q + 1 : q) * stride + e];
    T g[DIM];
#pragma unroll
    for (int s = 0; s < DIM; ++s) {
      T a = 0;
#pragma unroll
      for (int m = 0; m < L::Np; ++m) a = fma(C[L::off_GV + (s * L::nv + q) * L::Np + m], uu[m], a);
      g[s] = a;
    }
#pragma unroll
    for (int r = 0; r < DIM; ++r) {
      T h = 0;
#pragma unroll
      for (int s = 0; s < DIM; ++s) h = fma(K[kidx(DIM, r, s)], g[s], h);
      h *= wk;
#pragma unroll
      for (int i = 0; i < L::Np; ++i) acc[i] = fma(C[L::off_GV + (r * L::nv + q) * L::Np + i], h, acc[i]);
    }
  }
  if constexpr (has_face) {
    if (mode == 2) return;
    T beta[DIM];
    face_beta<DIM>(K, F0, beta);
#pragma unroll 1
    for (int q = 0; q < L::ns; ++q) {
      const T um = Um, tm = Tm, k = kq;
      const T up = mode == 0 ? Up : -um, tp = mode == 0 ? Tp : -tm;
      fetch(q + 1 < L::ns ? q + 1 : q);
      const T wq = C[L::off_ws + q];
      const T jump = um - up;
      const T F = wq * (T)0.5 * (ts * jump - (tm - tp));
      const T sig = wq * (T)-0.5 * k * jump;
      T bs[DIM];
#pragma unroll
      for (int s = 0; s < DIM; ++s) bs[s] = beta[s] * sig;
#pragma unroll
      for (int i = 0; i < L::Np; ++i) {
        T a = fma(C[L::off_IS + (F0 * L::ns + q) * L::Np + i], F, acc[i]);
#pragma unroll
        for (int s = 0; s < DIM; ++s) a = fma(C[L::off_GS + ((F0 * DIM + s) * L::ns + q) * L::Np + i], bs[s], a);
        acc[i] = a;
      }
    }
  }
}

template <int DIM, int N, typename T>
__global__ void __launch_bounds__(256)
k_apply_oi_split(int64_t E, int64_t stride, const T* __restrict__ u, const T* __restrict__ tU,
                 const T* __restrict__ tT, const double* __restrict__ Kt, const double* __restrict__ tauS,
                 const int* __restrict__ nbr, const int* __restrict__ bctype, const T* __restrict__ kv,
                 const T* __restrict__ ks, const T* __restrict__ Cp, const int* __restrict__ qmapp,
                 T* __restrict__ out, double* __restrict__ partial) {
  using L = OiL<DIM, N>;
  __shared__ T part[4][L::Np][64];
  const cptr<T> C = as_const(Cp);
  const cptr<int> qmap = as_const(qmapp);
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t e = xcd_block() * 64 + lane;
  if (e < E) {
    T acc[L::Np];
    switch (w) {
      case 0: oi_quarter<DIM, N, T, 0>(e, stride, u, tU, tT, Kt, tauS, nbr, bctype, kv, ks, C, qmap, acc); break;
      case 1: oi_quarter<DIM, N, T, 1>(e, stride, u, tU, tT, Kt, tauS, nbr, bctype, kv, ks, C, qmap, acc); break;
      case 2: oi_quarter<DIM, N, T, 2>(e, stride, u, tU, tT, Kt, tauS, nbr, bctype, kv, ks, C, qmap, acc); break;
      default: oi_quarter<DIM, N, T, 3>(e, stride, u, tU, tT, Kt, tauS, nbr, bctype, kv, ks, C, qmap, acc); break;
    }
#pragma unroll
    for (int i = 0; i < L::Np; ++i) part[w][i][lane] = acc[i];
  }
  __syncthreads();
  double dotv = 0.0;
  if (e < E) {
    for (int i = w; i < L::Np; i += 4) {
      const T a = (part[0][i][lane] + part[1][i][lane]) + (part[2][i][lane] + part[3][i][lane]);
      out[i * stride + e] = a;
      dotv += (double)u[i * stride + e] * (double)a;
    }
  }
  if (partial) {
    const double t = block_sum1<256>(dotv);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
  }
}

// Exact diagonal of the over-integrated operator.
template <int DIM, int N>
__global__ void __launch_bounds__(256)
k_diag_oi(int64_t E, int64_t stride, const double* __restrict__ Kt, const double* __restrict__ tauS,
          const int* __restrict__ nbr, const int* __restrict__ bctype, const double* __restrict__ kv,
          const double* __restrict__ ks, const double* __restrict__ C, double* __restrict__ diag) {
  using L = OiL<DIM, N>;
  const int64_t e = xcd_block() * blockDim.x + threadIdx.x;
  if (e >= E) return;
  constexpr int NK = DIM == 2 ? 3 : 6;
  double K[NK];
  for (int k = 0; k < NK; ++k) K[k] = Kt[k * stride + e];
  for (int i = 0; i < L::Np; ++i) {
    double d = 0;
    for (int q = 0; q < L::nv; ++q) {
      double g[DIM];
      for (int s = 0; s < DIM; ++s) g[s] = C[L::off_GV + (s * L::nv + q) * L::Np + i];
      double a = 0;
      for (int r = 0; r < DIM; ++r)
        for (int s = 0; s < DIM; ++s) a += g[r] * K[kidx(DIM, r, s)] * g[s];
      d += C[L::off_wv + q] * kv[(int64_t)q * stride + e] * a;
    }
    for (int f = 0; f < L::Nf; ++f) {
      const int nb = nbr[f * stride + e];
      double scale = 0.5;
      if (nb < 0) {
        if (bctype[-nb - 1] != 0) continue;
        scale = 1.0;
      }
      double beta[DIM];
      face_beta<DIM>(K, f, beta);
      const double ts = tauS[f * stride + e];
      for (int q = 0; q < L::ns; ++q) {
        const double phi = C[L::off_IS + (f * L::ns + q) * L::Np + i];
        double dn = 0;
        for (int s = 0; s < DIM; ++s) dn += beta[s] * C[L::off_GS + ((f * DIM + s) * L::ns + q) * L::Np + i];
        d += scale * C[L::off_ws + q] *
             (ts * phi * phi - 2.0 * ks[(int64_t)(f * L::ns + q) * stride + e] * phi * dn);
      }
    }
    diag[i * stride + e] = d;
  }
}

dim3 grid_oi(int64_t E) {
  const int64_t nb = (E + 255) / 256;
  return dim3((unsigned)nb);
}

}  // namespace

#define INSP_OI_DISPATCH(dim, N, CALL)                                  \
  do {                                                                  \
    if ((dim) == 2) {                                                   \
      switch (N) {                                                      \
        case 1: { constexpr int D_ = 2, N_ = 1; CALL; } break;          \
        case 2: { constexpr int D_ = 2, N_ = 2; CALL; } break;          \
        case 3: { constexpr int D_ = 2, N_ = 3; CALL; } break;          \
        case 4: { constexpr int D_ = 2, N_ = 4; CALL; } break;          \
        default: throw std::runtime_error("unsupported order");         \
      }                                                                 \
    } else {                                                            \
      switch (N) {                                                      \
        case 1: { constexpr int D_ = 3, N_ = 1; CALL; } break;          \
        case 2: { constexpr int D_ = 3, N_ = 2; CALL; } break;          \
        case 3: { constexpr int D_ = 3, N_ = 3; CALL; } break;          \
        case 4: { constexpr int D_ = 3, N_ = 4; CALL; } break;          \
        default: throw std::runtime_error("unsupported order");         \
      }                                                                 \
    }                                                                   \
  } while (0)

bool oi_shape_matches(int dim, int N, int nv, int ns, int table_size) {
  bool ok = false;
  INSP_OI_DISPATCH(dim, N, ok = (OiL<D_, N_>::nv == nv && OiL<D_, N_>::ns == ns && OiL<D_, N_>::size == table_size));
  return ok;
}

template <typename T>
int launch_apply_oi(const MeshView& m, const LevelView& l, const OiView<T>& o, const T* u, T* out,
                    hipStream_t s, double* partial) {
  if (m.E == 0) return 0;
  // four waves to a cell wherever the neighbour words are packed (meshes below 2^26 cells)
  if (m.nbc) {
    const dim3 grid((unsigned)four_wave_blocks(m.E));
    INSP_OI_DISPATCH(m.dim, l.N,
                     hipLaunchKernelGGL((k_trace_oi_split<D_, N_, T>), grid, dim3(256), 0, s, m.E, m.stride, u,
                                        m.Kt, o.ks, o.C, o.tU, o.tT));
    check("k_trace_oi_split");
    INSP_OI_DISPATCH(m.dim, l.N,
                     hipLaunchKernelGGL((k_apply_oi_split<D_, N_, T>), grid, dim3(256), 0, s, m.E, m.stride, u,
                                        o.tU, o.tT, m.Kt, l.tauS, m.nbc, m.bctype, o.kv, o.ks, o.C, o.qmap, out,
                                        partial));
    check("k_apply_oi_split");
    return (int)grid.x;
  }
  INSP_OI_DISPATCH(m.dim, l.N,
                   hipLaunchKernelGGL((k_trace_oi<D_, N_, T>), grid_oi(m.E), dim3(256), 0, s, m.E, m.stride, u,
                                      m.Kt, o.ks, o.C, o.tU, o.tT));
  check("k_trace_oi");
  INSP_OI_DISPATCH(m.dim, l.N,
                   hipLaunchKernelGGL((k_apply_oi<D_, N_, T>), grid_oi(m.E), dim3(256), 0, s, m.E, m.stride, u,
                                      o.tU, o.tT, m.Kt, l.tauS, m.nbr, m.code, m.bctype, o.kv, o.ks, o.C,
                                      o.qmap, out, partial));
  check("k_apply_oi");
  return apply_blocks(m.E);
}

void launch_diag_oi(const MeshView& m, const LevelView& l, const OiView<double>& o, double* diag,
                    hipStream_t s) {
  if (m.E == 0) return;
  INSP_OI_DISPATCH(m.dim, l.N,
                   hipLaunchKernelGGL((k_diag_oi<D_, N_>), grid_oi(m.E), dim3(256), 0, s, m.E, m.stride, m.Kt,
                                      l.tauS, m.nbr, m.bctype, o.kv, o.ks, o.C, diag));
  check("k_diag_oi");
}

template int launch_apply_oi<double>(const MeshView&, const LevelView&, const OiView<double>&, const double*,
                                     double*, hipStream_t, double*);
template int launch_apply_oi<float>(const MeshView&, const LevelView&, const OiView<float>&, const float*,
                                    float*, hipStream_t, double*);

}  // namespace insp
