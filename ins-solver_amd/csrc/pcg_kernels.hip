#include "pcg_kernels.h"

#include <cmath>
#include <stdexcept>
#include <string>

#include "dg_layout.h"
#include "reduce.h"
#include "sipg_cell.h"

namespace insp {

namespace {

constexpr int kBlock = 256;

// The step's sums |r|^2, r.z, r.(z - z_old): value k as n partials (n = 1: the value) at p + k * stride.
struct PcgSums {
  const double* p;
  int n, stride;
};

inline void check(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    throw std::runtime_error(std::string("kernel launch failed: ") + what + ": " + hipGetErrorString(e));
}

__device__ __forceinline__ double safe_div(double a, double b) { return b != 0.0 ? a / b : 0.0; }

// K sums of partials by the whole block, stride apart; every thread gets them, in an order that
// depends on n alone.
template <int K>
__device__ __forceinline__ void totals(const double* __restrict__ p, int n, int64_t stride, double (&v)[K]) {
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = 0.0;
  if (n == 1) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = p[k * stride];
    return;
  }
  for (int i = threadIdx.x; i < n; i += 2 * kBlock) {
    const int j = i + kBlock;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const double a = p[k * stride + i], b = j < n ? p[k * stride + j] : 0.0;
      v[k] += a + b;
    }
  }
  __shared__ double sh[K][kBlock / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    v[k] = wave_sum(v[k]);
    if (lane == 0) sh[k][w] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K; ++k) {
    double t = 0;
#pragma unroll
    for (int i = 0; i < kBlock / 64; ++i) t += sh[k][i];
    v[k] = t;
  }
  __syncthreads();
}

__device__ __forceinline__ void put3(const double (&v)[3], int64_t block, int64_t stride, double* partial) {
  __shared__ double sh[3][kBlock / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double t = wave_sum(v[k]);
    if (lane == 0) sh[k][w] = t;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double t = 0;
#pragma unroll
    for (int i = 0; i < kBlock / 64; ++i) t += sh[threadIdx.x][i];
    partial[threadIdx.x * stride + block] = t;
  }
}

// The three sums where there are too many partials to fold.
__global__ void __launch_bounds__(kBlock) k_pcg_sums(PcgSums sums, double* __restrict__ out) {
  double v[3];
  totals<3>(sums.p, sums.n, sums.stride, v);
  if (threadIdx.x < 3) out[threadIdx.x] = threadIdx.x == 0 ? v[0] : threadIdx.x == 1 ? v[1] : v[2];
}

__global__ void k_pcg_start(double* st) {
  if (threadIdx.x == 0) {
    st[P_IT] = 0.0;
    st[P_STOP0] = st[P_STOP1] = (double)PCG_RUNNING;
  }
}

// Length of the step; the first block keeps p.Ap for the direction pass. False once stopped (the same
// for every wave: only the direction pass stops).
__device__ __forceinline__ bool step_length(const Parts& pap, double* st, const PcgTurn& t, bool first, double* a) {
  if (!pcg_running(st, t)) return false;
  double v[1];
  totals<1>(pap.p, pap.n, 0, v);
  if (first && threadIdx.x == 0) st[P_PAP] = v[0];
  *a = safe_div(st[t.rz], v[0]);
  return true;
}

// One stream instead of three (x and r; the preconditioner; the two inner products): 64 instead of 96
// bytes per entry. Two entries per access.
__global__ void __launch_bounds__(kBlock)
k_pcg_jacobi(int64_t n2, double2* __restrict__ x, double2* __restrict__ r, double2* __restrict__ z,
             const double2* __restrict__ p, const double2* __restrict__ Ap, const double2* __restrict__ inv,
             Parts pap, double* st, PcgTurn t, double* __restrict__ partial) {
  double a;
  if (!step_length(pap, st, t, blockIdx.x == 0, &a)) return;
  double v[3] = {0.0, 0.0, 0.0};
  auto one = [&](double& xi, double& ri, double& zi, double pi, double api, double di) {
    xi = fma(a, pi, xi);
    ri = fma(-a, api, ri);
    const double zn = di * ri;
    v[0] += ri * ri;
    v[1] += ri * zn;
    v[2] += ri * (zn - zi);
    zi = zn;
  };
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n2; i += (int64_t)gridDim.x * kBlock) {
    const double2 pi = p[i], ai = Ap[i], di = inv[i];
    double2 xi = x[i], ri = r[i], zi = z[i];
    one(xi.x, ri.x, zi.x, pi.x, ai.x, di.x);
    one(xi.y, ri.y, zi.y, pi.y, ai.y, di.y);
    x[i] = xi;
    r[i] = ri;
    z[i] = zi;
  }
  put3(v, blockIdx.x, gridDim.x, partial);
}

// One thread per cell: its new residual stays in registers for the inverse mass matrix (wave-uniform
// rows through the scalar cache). 8 instead of 11 vectors through memory.
template <int NP>
__global__ void __launch_bounds__(kBlock)
k_pcg_inv_mass(int64_t E, int64_t stride, int64_t cs, double* __restrict__ x, double* __restrict__ r,
               double* __restrict__ z, const double* __restrict__ p, const double* __restrict__ Ap,
               const double* __restrict__ J, const double* __restrict__ Minv, double scale,
               const double* __restrict__ recp, Parts pap, double* st, PcgTurn t, double* __restrict__ partial) {
  double a;
  const int64_t block = blockIdx.y * (int64_t)gridDim.x + blockIdx.x;
  if (!step_length(pap, st, t, block == 0, &a)) return;
  const cptr<double> Mi = as_const(Minv);
  const int64_t c0 = blockIdx.y * cs;
  double v[3] = {0.0, 0.0, 0.0};
  // (no loop over cells: the compiler keeps Minv of a loop in spilled scalar registers)
  const int64_t e = blockIdx.x * (int64_t)kBlock + threadIdx.x;
  if (e < E) {
    double rr[NP];
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      const int64_t k = c0 + j * stride + e;
      x[k] = fma(a, p[k], x[k]);
      rr[j] = fma(-a, Ap[k], r[k]);
      r[k] = rr[j];
      v[0] += rr[j] * rr[j];
    }
    const double inv_j = 1.0 / J[e];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int64_t k = c0 + i * stride + e;
      double s = 0;
#pragma unroll
      for (int j = 0; j < NP; ++j) s = fma(Mi[i * NP + j], rr[j], s);
      s *= inv_j;
      const double zn = recp ? s / recp[i * stride + e] : s * scale;
      v[1] += rr[i] * zn;
      v[2] += rr[i] * (zn - z[k]);
      z[k] = zn;
    }
  }
  put3(v, block, (int64_t)gridDim.x * gridDim.y, partial);
}

// Every block forms the same sums and takes the same decision; the first one writes it down, into slots
// that no wave of this launch reads (PcgTurn): all waves of a block go the same way to its barriers.
__global__ void __launch_bounds__(kBlock)
k_pcg_direction(int64_t n2, double2* __restrict__ p, const double2* __restrict__ z, PcgSums sums, double* st,
                PcgTurn t, double tol) {
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  if (!pcg_running(st, t)) {
    if (first) pcg_keep_stop(st, t);
    return;
  }
  const double ro = st[t.rz], pap = st[P_PAP];
  double v[3];
  totals<3>(sums.p, sums.n, sums.stride, v);
  const PcgStop why = pcg_decide(v[0], pap, tol);
  if (first) pcg_record(st, t, v[0], v[1], why);
  if (why != PCG_RUNNING) return;
  const double beta = safe_div(v[2], ro);
  const int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x;
  if (i >= n2) return;
  double2 pi = p[i];
  const double2 zi = z[i];
  pi.x = fma(beta, pi.x, zi.x);
  pi.y = fma(beta, pi.y, zi.y);
  p[i] = pi;
}

}  // namespace

void pcg_start(double* st, hipStream_t s) {
  hipLaunchKernelGGL(k_pcg_start, dim3(1), dim3(64), 0, s, st);
  check("k_pcg_start");
}

int pcg_update_jacobi(int64_t n, double* x, double* r, double* z, const double* p, const double* Ap,
                      const double* inv, Parts pap, double* st, const PcgTurn& t, double* partial, hipStream_t s) {
  const int nb = (int)pcg_stream_blocks(n / 2);
  auto v2 = [](const double* q) { return reinterpret_cast<const double2*>(q); };
  hipLaunchKernelGGL(k_pcg_jacobi, dim3(nb), dim3(kBlock), 0, s, n / 2, reinterpret_cast<double2*>(x),
                     reinterpret_cast<double2*>(r), reinterpret_cast<double2*>(z), v2(p), v2(Ap), v2(inv), pap,
                     st, t, partial);
  check("k_pcg_jacobi");
  return nb;
}

int pcg_update_inv_mass(int np, int ncomp, int64_t E, int64_t stride, int64_t cs, double* x, double* r,
                        double* z, const double* p, const double* Ap, const double* J, const double* Minv,
                        double scale, const double* recp, Parts pap, double* st, const PcgTurn& t, double* partial,
                        hipStream_t s) {
  const dim3 grid((unsigned)((E + kBlock - 1) / kBlock), (unsigned)ncomp);
#define INSP_IM(NP)                                                                                         \
  case NP:                                                                                                  \
    hipLaunchKernelGGL((k_pcg_inv_mass<NP>), grid, dim3(kBlock), 0, s, E, stride, cs, x, r, z, p, Ap, J, Minv, \
                       scale, recp, pap, st, t, partial);                                                   \
    break
  switch (np) {
    INSP_IM(3);
    INSP_IM(4);
    INSP_IM(6);
    INSP_IM(10);
    INSP_IM(15);
    INSP_IM(20);
    INSP_IM(35);
    default: throw std::runtime_error("unsupported number of nodes");
  }
#undef INSP_IM
  check("k_pcg_inv_mass");
  return (int)(grid.x * grid.y);
}

void pcg_direction(int64_t n, double* p, const double* z, int nb, const double* partial, double* st,
                   const PcgTurn& t, double tol, hipStream_t s) {
  PcgSums sums{partial, nb, nb};
  const int64_t n2 = n / 2, blocks = (n2 + kBlock - 1) / kBlock;
  if (!pcg_fold_pays(nb, blocks)) {
    hipLaunchKernelGGL(k_pcg_sums, dim3(1), dim3(kBlock), 0, s, sums, st + P_SUM);
    check("k_pcg_sums");
    sums = PcgSums{st + P_SUM, 1, 1};
  }
  hipLaunchKernelGGL(k_pcg_direction, dim3((unsigned)blocks), dim3(kBlock), 0, s, n2,
                     reinterpret_cast<double2*>(p), reinterpret_cast<const double2*>(z), sums, st, t, tol);
  check("k_pcg_direction");
}

}  // namespace insp
