// Launches of the passes that give a cell to four waves (sipg_split.h).
#include <hip/hip_runtime.h>

#include "sipg_split_kernels.h"

namespace insp {

namespace split {
INSP_SPLIT_INST(extern, 3, 3, double)
INSP_SPLIT_INST(extern, 3, 3, float)
INSP_SPLIT_INST(extern, 3, 4, double)
INSP_SPLIT_INST(extern, 3, 4, float)
INSP_SPLIT_VEC(extern, 2, 2)
INSP_SPLIT_VEC(extern, 2, 3)
INSP_SPLIT_VEC(extern, 2, 4)
INSP_SPLIT_VEC(extern, 3, 2)
INSP_SPLIT_VEC(extern, 3, 3)
INSP_SPLIT_VEC(extern, 3, 4)
}  // namespace split

namespace {
#define INSP_SPLIT_N(dim, N, CALL)                               \
  switch ((dim) * 8 + (N)) {                                     \
    case 18: { constexpr int D_ = 2, N_ = 2; CALL; } break;      \
    case 19: { constexpr int D_ = 2, N_ = 3; CALL; } break;      \
    case 20: { constexpr int D_ = 2, N_ = 4; CALL; } break;      \
    case 26: { constexpr int D_ = 3, N_ = 2; CALL; } break;      \
    case 27: { constexpr int D_ = 3, N_ = 3; CALL; } break;      \
    case 28: { constexpr int D_ = 3, N_ = 4; CALL; } break;      \
    default: throw std::runtime_error("unsupported order");      \
  }
}  // namespace

namespace {
constexpr int64_t kFill = 1 << 16;  // cells that give every SIMD one wave of 64
}

bool split_trace(const MeshView& m, const LevelView& l) {
  if (!m.nbc) return false;
  if (m.dim == 2) return l.N == 4 && m.E <= 3 * kFill;
  return l.N == 4 || (l.N == 3 && m.E <= 6 * kFill) || (l.N == 2 && m.E <= 3 * kFill);
}

bool split_apply(const MeshView& m, const LevelView& l, bool fp32) {
  if (!m.nbc || l.N < 2) return false;
  if (m.dim == 2) return m.E <= (l.N == 4 ? 3 * kFill : kFill);
  if (l.N == 2) return m.E <= 12 * kFill;
  if (l.N == 3) return m.E <= (fp32 ? 2 * kFill : kFill + kFill / 2);
  return m.E <= (fp32 ? kFill + kFill / 2 : kFill);
}

int split_blocks(int64_t E) { return (int)split::grid_split(E).x; }

template <typename T>
void launch_trace_split(const MeshView& m, const LevelView& l, const T* u, const T* kfac, T* tr,
                        hipStream_t s, int ncomp, int64_t cs, int64_t ts) {
  if (m.E == 0) return;
  INSP_SPLIT_N(m.dim, l.N, (split::trace<D_, N_, T>(m, l, u, kfac, tr, s, ncomp, cs, ts)))
}

template <typename T>
void launch_apply_split(const MeshView& m, const LevelView& l, const T* u, const T* tr, const T* kfac,
                        const MassView<T>& mass, T* out, hipStream_t s, double* partial) {
  if (m.E == 0) return;
  INSP_SPLIT_N(m.dim, l.N, (split::apply<D_, N_, T>(m, l, u, tr, kfac, mass, out, s, partial)))
}

template <typename T>
void launch_cheb_split(const MeshView& m, const LevelView& l, const T* u, const T* tr, const T* kfac,
                       const T* f, const T* inv, const T* prev, T* x_next, T c1, T c2, hipStream_t s) {
  if (m.E == 0) return;
  INSP_SPLIT_N(m.dim, l.N, (split::cheb<D_, N_, T>(m, l, u, tr, kfac, f, inv, prev, x_next, c1, c2, s)))
}

void launch_vec_split(const MeshView& m, const LevelView& l, int ncomp, const double* u, const double* tr,
                      const double* kfac, const MassView<double>& mass, const double* bnormal, int64_t cs,
                      int64_t ts, int64_t bs, double* out, hipStream_t s, double* partial) {
  if (m.E == 0) return;
  INSP_SPLIT_N(m.dim, l.N, (split::vec<D_, N_>(m, l, ncomp, u, tr, kfac, mass, bnormal, cs, ts, bs, out, s, partial)))
}

#define INSP_INST(T)                                                                                   \
  template void launch_trace_split<T>(const MeshView&, const LevelView&, const T*, const T*, T*,       \
                                      hipStream_t, int, int64_t, int64_t);                                                    \
  template void launch_apply_split<T>(const MeshView&, const LevelView&, const T*, const T*, const T*, \
                                      const MassView<T>&, T*, hipStream_t, double*);                   \
  template void launch_cheb_split<T>(const MeshView&, const LevelView&, const T*, const T*, const T*,  \
                                     const T*, const T*, const T*, T*, T, T, hipStream_t);
INSP_INST(double)
INSP_INST(float)

}  // namespace insp
