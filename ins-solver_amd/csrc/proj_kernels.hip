// Pressure projection around the solve: the gradient of the pressure with a central
// flux and the velocity update of the projection step.
//
//   grad_h p = sum_r grad(xi_r) D_r p + LIFT_f (fscale_f n_f (p* - p-)),  p* = (p- + p+)/2
//   uTT = uT - dt grad_h p                                  (ins_2d_proj_rhs.h:1-10)
//
// The gradient is the toolkit's DGMesh::grad_with_central_flux (called at
// src/solvers/2d/ins_solver.cpp:337, code not vendored): the textbook strong form with a
// central flux; on boundary faces p* = p- (no face term). fscale_f n_f = sum_r alpha_fr
// grad(xi_r) for a straight-sided simplex, so only grad(xi) is stored per cell. One
// thread per cell; the neighbour's face values are gathered by index and permutation.
#include <hip/hip_runtime.h>

#include <stdexcept>
#include <string>

#include "dg_layout.h"
#include "kernels.h"
#include "sipg_cell.h"

namespace insp {

namespace {

// One thread per cell, one node of the result at a time: t_r = (D_r p)_i + sum_f alpha_fr s_fi with
// s_fi = sum_j LIFT_i,fj (p* - p-)_fj, then component x is sum_r d xi_r / d x_x t_r. The face term
// of component x carries the factor fscale_f n_fx = sum_r alpha_fr d xi_r / d x_x, so D_r p and the
// lifted jumps are formed once for all components (a component at a time formed them again for
// each: 6000 instead of 2300 FMAs per cell at 3D order 3) and nothing but p and the jumps stays in
// registers. The loads go in rounds: neighbour words, node maps, then every neighbour value.
// 31^3 x 6 cells, order 3, FP64, device vectors: 2209 us per call with staged copies and a component
// at a time (344 us of it this kernel), 106 us per call now.
//
// uT and the outputs may be the same arrays component by component: a thread reads an entry of uT
// right before it writes the result there. Threads past the last cell clear the outputs' padding.
template <int DIM, int N>
__global__ void __launch_bounds__(256)
k_grad_central(int64_t E, int64_t stride, const double* __restrict__ G, const int* __restrict__ nbr,
               const int* __restrict__ code, const double* __restrict__ C, const int* __restrict__ tab,
               const double* __restrict__ lift, const double* __restrict__ p, double dt,
               const double* u0, const double* u1, const double* u2, double* o0, double* o1,
               double* o2) {
  constexpr OpLayout L = op_layout(DIM, N);
  constexpr int Np = L.Np, Nfp = L.Nfp, Nf = L.Nf, NF = Nf * Nfp;
  constexpr FmaskTable FM = make_fmask(DIM, N);
  const cptr<double> Cc = as_const(C);
  const cptr<double> Lc = as_const(lift);
  const int64_t e = xcd_block() * blockDim.x + threadIdx.x;
  if (e >= stride) return;
  if (e >= E) {
    for (int i = 0; i < Np; ++i) {
      o0[i * stride + e] = 0.0;
      o1[i * stride + e] = 0.0;
      if constexpr (DIM == 3) o2[i * stride + e] = 0.0;
    }
    return;
  }
  int nb[Nf], base[Nf];
#pragma unroll
  for (int f = 0; f < Nf; ++f) {
    nb[f] = nbr[f * stride + e];
    base[f] = code[f * stride + e];
  }
  double pp[Np];
#pragma unroll
  for (int m = 0; m < Np; ++m) pp[m] = p[m * stride + e];
  double g[DIM][DIM];  // g[r][x] = d xi_r / d x_x
#pragma unroll
  for (int r = 0; r < DIM; ++r)
#pragma unroll
    for (int x = 0; x < DIM; ++x) g[r][x] = G[(r * DIM + x) * stride + e];
  // p* - p-; a boundary face reads the cell's own values, so its jump is zero
  double jump[NF];
#pragma unroll
  for (int f = 0; f < Nf; ++f) {
    const bool in = nb[f] >= 0;
    const int64_t q = in ? (int64_t)nb[f] : e;
    const int tbase = L.tab_nbr + (f * Nf * L.nperm + (in ? base[f] : 0)) * Nfp;
    int pk[Nfp];
#pragma unroll
    for (int j = 0; j < Nfp; ++j) pk[j] = tab[tbase + j] >> 6;
#pragma unroll
    for (int j = 0; j < Nfp; ++j) jump[f * Nfp + j] = p[(int64_t)pk[j] * stride + q];
#pragma unroll
    for (int j = 0; j < Nfp; ++j) {
      const double own = pp[FM.v[f * Nfp + j]];
      jump[f * Nfp + j] = in ? 0.5 * (jump[f * Nfp + j] - own) : 0.0;
    }
  }
#pragma unroll 1
  for (int i = 0; i < Np; ++i) {
    const int64_t k = i * stride + e;
    double ux[DIM];
    ux[0] = u0 ? u0[k] : 0.0;
    ux[1] = u1 ? u1[k] : 0.0;
    if constexpr (DIM == 3) ux[2] = u2 ? u2[k] : 0.0;
    double t[DIM];
#pragma unroll
    for (int r = 0; r < DIM; ++r) {
      double d = 0;
#pragma unroll
      for (int m = 0; m < Np; ++m) d = fma(Cc[L.off_D + (r * Np + i) * Np + m], pp[m], d);
      t[r] = d;
    }
#pragma unroll
    for (int f = 0; f < Nf; ++f) {
      double s = 0;
#pragma unroll
      for (int j = 0; j < Nfp; ++j) s = fma(Lc[i * NF + f * Nfp + j], jump[f * Nfp + j], s);
#pragma unroll
      for (int r = 0; r < DIM; ++r)
        if (face_alpha(DIM, f, r) != 0.0) t[r] = fma(face_alpha(DIM, f, r), s, t[r]);
    }
    double o[DIM];
#pragma unroll
    for (int x = 0; x < DIM; ++x) {
      double a = 0;
#pragma unroll
      for (int r = 0; r < DIM; ++r) a = fma(g[r][x], t[r], a);
      o[x] = a;
    }
    o0[k] = u0 ? ux[0] - dt * o[0] : o[0];
    o1[k] = u1 ? ux[1] - dt * o[1] : o[1];
    if constexpr (DIM == 3) o2[k] = u2 ? ux[2] - dt * o[2] : o[2];
  }
}

}  // namespace

void launch_grad_central(int dim, int N, int64_t E, int64_t stride, const double* G, const int* nbr,
                         const int* code, const double* C64, const int* tab, const double* lift,
                         const double* p, double dt, const double* const u[3], double* const out[3],
                         hipStream_t s) {
  if (E == 0) return;
  const dim3 grid((unsigned)((stride + 255) / 256)), block(256);  // the padding is cleared too
#define INSP_GRAD(D, NN)                                                                          \
  hipLaunchKernelGGL((k_grad_central<D, NN>), grid, block, 0, s, E, stride, G, nbr, code, C64,  \
                     tab, lift, p, dt, u[0], u[1], u[2], out[0], out[1], out[2])
  if (dim == 2) {
    switch (N) {
      case 1: INSP_GRAD(2, 1); break;
      case 2: INSP_GRAD(2, 2); break;
      case 3: INSP_GRAD(2, 3); break;
      case 4: INSP_GRAD(2, 4); break;
      default: throw std::runtime_error("unsupported order");
    }
  } else {
    switch (N) {
      case 1: INSP_GRAD(3, 1); break;
      case 2: INSP_GRAD(3, 2); break;
      case 3: INSP_GRAD(3, 3); break;
      case 4: INSP_GRAD(3, 4); break;
      default: throw std::runtime_error("unsupported order");
    }
  }
#undef INSP_GRAD
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess)
    throw std::runtime_error(std::string("k_grad_central launch failed: ") + hipGetErrorString(err));
}

}  // namespace insp
