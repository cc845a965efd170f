// Kernels of the passes that give a cell to four waves (sipg_split.h); sipg_split.hip launches them,
// those of 3D order 4 from a source file of their own, as they compile slowest.
#pragma once

#include <hip/hip_runtime.h>

#include <stdexcept>
#include <string>

#include "reduce.h"
#include "sipg_split.h"
#include "split_passes.h"

namespace insp {
namespace split {

inline void check(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    throw std::runtime_error(std::string("kernel launch failed: ") + what + ": " + hipGetErrorString(e));
}

constexpr int kCells = 64;  // cells of a block
inline dim3 grid_split(int64_t E) { return dim3((unsigned)four_wave_blocks(E)); }

template <int DIM, int N, typename T, bool VAR>
__global__ void __launch_bounds__(256)
k_trace_split(int64_t E, int64_t stride, const T* __restrict__ u, const double* __restrict__ Kt,
              const T* __restrict__ kfac, const T* __restrict__ C, T* __restrict__ tr, int64_t cs,
              int64_t ts) {
  u += blockIdx.y * cs;  // component blockIdx.y of a vector
  tr += blockIdx.y * ts;
  constexpr int Np = op_layout(DIM, N).Np;
  const int64_t e = xcd_block() * kCells + (threadIdx.x & 63);
  if (e >= E) return;
  T uu[Np];
#pragma unroll
  for (int m = 0; m < Np; ++m) uu[m] = u[m * stride + e];
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const cptr<T> Cc = as_const(C);
  switch (w) {
    case 0: trace_quarter<DIM, N, T, VAR, 0>(e, stride, uu, Kt, kfac, Cc, tr); break;
    case 1: trace_quarter<DIM, N, T, VAR, 1>(e, stride, uu, Kt, kfac, Cc, tr); break;
    case 2: trace_quarter<DIM, N, T, VAR, 2>(e, stride, uu, Kt, kfac, Cc, tr); break;
    default: trace_quarter<DIM, N, T, VAR, 3>(e, stride, uu, Kt, kfac, Cc, tr); break;
  }
}

template <int DIM, int N, typename T, bool VAR>
__global__ void __launch_bounds__(256)
k_apply_split(int64_t E, int64_t stride, const T* __restrict__ u, const T* __restrict__ tr,
              const double* __restrict__ Kt, const double* __restrict__ tauS,
              const int* __restrict__ nbr, const int* __restrict__ bctype,
              const T* __restrict__ kfac, const T* __restrict__ C, const int* __restrict__ tab,
              MassTerm<T> mass, T* __restrict__ out, double* __restrict__ partial) {
  __shared__ T part[4][op_layout(DIM, N).Np][64];
  const int64_t e = xcd_block() * kCells + (threadIdx.x & 63);
  const double dotv = apply_split<DIM, N, T, VAR>(e, e < E, stride, u, tr, Kt, tauS, nbr, bctype, kfac,
                                                  as_const(C), tab, mass, out, NoSlip{}, part);
  if (partial) {
    const double t = block_sum1<256>(dotv);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
  }
}

// Component blockIdx.y of the vector (velocity) operator with slip faces; kfac may be null (k = 1).
template <int DIM, int N>
__global__ void __launch_bounds__(256)
k_vec_split(int64_t E, int64_t stride, const double* __restrict__ u, const double* __restrict__ tr,
            const double* __restrict__ Kt, const double* __restrict__ tauS, const int* __restrict__ nbr,
            const int* __restrict__ bctype, const double* __restrict__ kfac, const double* __restrict__ C,
            const int* __restrict__ tab, MassTerm<double> mass, const double* __restrict__ bn, int64_t cs,
            int64_t ts, int64_t bs, double* __restrict__ out, double* __restrict__ partial) {
  __shared__ double part[4][op_layout(DIM, N).Np][64];
  const int c = blockIdx.y;
  const int64_t e = xcd_block() * kCells + (threadIdx.x & 63);
  const SlipFaces<double> slip{u, tr, cs, ts, bn, c};
  const double dotv = apply_split<DIM, N, double, 2>(e, e < E, stride, u + c * cs, tr + c * ts, Kt, tauS, nbr,
                                                     bctype + c * bs, kfac, as_const(C), tab, mass,
                                                     out + c * cs, slip, part);
  if (partial) {
    const double t = block_sum1<256>(dotv);
    if (threadIdx.x == 0) partial[blockIdx.y * gridDim.x + blockIdx.x] = t;
  }
}

template <int DIM, int N, typename T, bool VAR>
__global__ void __launch_bounds__(256)
k_cheb_split(int64_t E, int64_t stride, const T* __restrict__ u, const T* __restrict__ tr,
             const double* __restrict__ Kt, const double* __restrict__ tauS,
             const int* __restrict__ nbr, const int* __restrict__ bctype,
             const T* __restrict__ kfac, const T* __restrict__ C, const int* __restrict__ tab,
             const T* __restrict__ f, const T* __restrict__ inv, const T* prev, T* x_next, T c1, T c2) {
  __shared__ T part[4][op_layout(DIM, N).Np][64];
  const int64_t e = xcd_block() * kCells + (threadIdx.x & 63);
  (void)apply_split<DIM, N, T, VAR>(e, e < E, stride, u, tr, Kt, tauS, nbr, bctype, kfac, as_const(C),
                                    tab, MassTerm<T>{}, ChebOut<T>{f, inv, prev, x_next, c1, c2},
                                    NoSlip{}, part);
}


template <int DIM, int N, typename T>
void trace(const MeshView& m, const LevelView& l, const T* u, const T* kfac, T* tr, hipStream_t s, int ncomp,
           int64_t cs, int64_t ts) {
  const T* C = static_cast<const T*>(l.C);
  dim3 grid = grid_split(m.E);
  grid.y = (unsigned)ncomp;
  if (kfac)
    hipLaunchKernelGGL((k_trace_split<DIM, N, T, true>), grid, dim3(256), 0, s, m.E, m.stride, u, m.Kt, kfac, C,
                       tr, cs, ts);
  else
    hipLaunchKernelGGL((k_trace_split<DIM, N, T, false>), grid, dim3(256), 0, s, m.E, m.stride, u, m.Kt, kfac,
                       C, tr, cs, ts);
  check("k_trace_split");
}

template <int DIM, int N, typename T>
void apply(const MeshView& m, const LevelView& l, const T* u, const T* tr, const T* kfac,
           const MassView<T>& mv, T* out, hipStream_t s, double* partial) {
  const T* C = static_cast<const T*>(l.C);
  const MassTerm<T> mass{m.J, mv.mm, mv.mmc, mv.on()};
#define INSP_CALL(V)                                                                                   \
  hipLaunchKernelGGL((k_apply_split<DIM, N, T, V>), grid_split(m.E), dim3(256), 0, s, m.E, m.stride, u, \
                     tr, m.Kt, l.tauS, m.nbc, m.bctype, kfac, C, l.tab, mass, out, partial)
  if (kfac) INSP_CALL(true);
  else INSP_CALL(false);
#undef INSP_CALL
  check("k_apply_split");
}

template <int DIM, int N, typename T>
void cheb(const MeshView& m, const LevelView& l, const T* u, const T* tr, const T* kfac, const T* f,
          const T* inv, const T* prev, T* x_next, T c1, T c2, hipStream_t s) {
  const T* C = static_cast<const T*>(l.C);
#define INSP_CALL(V)                                                                                  \
  hipLaunchKernelGGL((k_cheb_split<DIM, N, T, V>), grid_split(m.E), dim3(256), 0, s, m.E, m.stride, u, \
                     tr, m.Kt, l.tauS, m.nbc, m.bctype, kfac, C, l.tab, f, inv, prev, x_next, c1, c2)
  if (kfac) INSP_CALL(true);
  else INSP_CALL(false);
#undef INSP_CALL
  check("k_cheb_split");
}

template <int DIM, int N>
void vec(const MeshView& m, const LevelView& l, int ncomp, const double* u, const double* tr,
         const double* kfac, const MassView<double>& mv, const double* bn, int64_t cs, int64_t ts, int64_t bs,
         double* out, hipStream_t s, double* partial) {
  dim3 grid = grid_split(m.E);
  grid.y = (unsigned)ncomp;
  hipLaunchKernelGGL((k_vec_split<DIM, N>), grid, dim3(256), 0, s, m.E, m.stride, u, tr, m.Kt, l.tauS, m.nbc,
                     m.bctype, kfac, l.C64, l.tab, MassTerm<double>{m.J, mv.mm, mv.mmc, mv.on()}, bn, cs, ts,
                     bs, out, partial);
  check("k_vec_split");
}

// DECL is extern where the instantiations are compiled elsewhere, and empty there.
#define INSP_SPLIT_INST(DECL, DIM, N, T)                                                                \
  DECL template void trace<DIM, N, T>(const MeshView&, const LevelView&, const T*, const T*, T*,        \
                                      hipStream_t, int, int64_t, int64_t);                                                     \
  DECL template void apply<DIM, N, T>(const MeshView&, const LevelView&, const T*, const T*, const T*,  \
                                      const MassView<T>&, T*, hipStream_t, double*);                    \
  DECL template void cheb<DIM, N, T>(const MeshView&, const LevelView&, const T*, const T*, const T*,   \
                                     const T*, const T*, const T*, T*, T, T, hipStream_t);

#define INSP_SPLIT_VEC(DECL, DIM, N)                                                                    \
  DECL template void vec<DIM, N>(const MeshView&, const LevelView&, int, const double*, const double*,  \
                                 const double*, const MassView<double>&, const double*, int64_t, int64_t, \
                                 int64_t, double*, hipStream_t, double*);

}  // namespace split
}  // namespace insp
