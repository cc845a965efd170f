// Element pass with one thread per cell that adds the mass term of the viscous operator in the same pass
// (apply_cell with MASS): a pass of its own read u and A u and wrote A u again (40 us beside an element
// pass of 190 us on 384,000 cells at order 3).
#include <hip/hip_runtime.h>

#include <stdexcept>
#include <string>

#include "dg_layout.h"
#include "kernels.h"
#include "reduce.h"
#include "sipg_cell.h"

namespace insp {

namespace {

template <int DIM, int N, bool VAR>
__global__ void __launch_bounds__(256)
k_apply_mass(int64_t E, int64_t stride, const double* __restrict__ u, const double* __restrict__ tr,
             const double* __restrict__ Kt, const double* __restrict__ tauS, const int* __restrict__ nbr,
             const int* __restrict__ bctype, const double* __restrict__ kfac, const double* __restrict__ C,
             const int* __restrict__ tab, MassTerm<double> mass, double* __restrict__ out,
             double* __restrict__ partial) {
  const int64_t e = xcd_block() * blockDim.x + threadIdx.x;
  double dotv = 0.0;
  if (e < E)
    dotv = apply_cell<DIM, N, double, VAR, true, double*, NoSlip, true>(
        e, stride, u, tr, Kt, tauS, nbr, nullptr, bctype, kfac, as_const(C), as_const(tab), out, NoSlip{},
        mass);
  if (partial) {
    const double t = block_sum1<256>(dotv);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
  }
}

}  // namespace

// Not at 3D order 4, where two waves per SIMD hide neither the column's loads nor the longer chain: mult with a
// coefficient and a factor per node, 279,936 cells, 1018 us in the element pass, 763 after it.
bool apply_mass_pays(const MeshView& m, const LevelView& l) {
  return m.nbc && l.N >= 2 && !(m.dim == 3 && l.N == 4);
}

void launch_apply_mass(const MeshView& m, const LevelView& l, const double* u, const double* tr,
                       const double* kfac, const MassView<double>& mv, double* out, hipStream_t s,
                       double* partial) {
  if (!apply_mass_pays(m, l)) throw std::invalid_argument("element pass with mass term: order 2 and up, packed words");
  if (m.E == 0) return;
  const double* C = static_cast<const double*>(l.C);
  const MassTerm<double> mass{m.J, mv.mm, mv.mmc, true};
  const dim3 grid((unsigned)apply_blocks(m.E));
#define INSP_M(D, NN)                                                                                   \
  do {                                                                                                  \
    if (kfac)                                                                                           \
      hipLaunchKernelGGL((k_apply_mass<D, NN, true>), grid, dim3(256), 0, s, m.E, m.stride, u, tr, m.Kt, \
                         l.tauS, m.nbc, m.bctype, kfac, C, l.tab, mass, out, partial);                  \
    else                                                                                                \
      hipLaunchKernelGGL((k_apply_mass<D, NN, false>), grid, dim3(256), 0, s, m.E, m.stride, u, tr,     \
                         m.Kt, l.tauS, m.nbc, m.bctype, kfac, C, l.tab, mass, out, partial);            \
  } while (0)
  switch (m.dim * 8 + l.N) {
    case 18: INSP_M(2, 2); break;
    case 19: INSP_M(2, 3); break;
    case 20: INSP_M(2, 4); break;
    case 26: INSP_M(3, 2); break;
    case 27: INSP_M(3, 3); break;
    default: throw std::runtime_error("unsupported order");
  }
#undef INSP_M
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw std::runtime_error(std::string("k_apply_mass launch failed: ") + hipGetErrorString(e));
}

}  // namespace insp
