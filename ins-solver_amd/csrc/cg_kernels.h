// Kernels of the order-1 Jacobi-CG (the coarse solve of the p-multigrid cycle). A sum over the mesh
// is left as partial sums, one per block of its producer, and every block of the next kernel adds
// them for itself, in one order: no kernel in between that adds them up.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"
#include "partials.h"

namespace insp {

// A sum as n partials (n = 1: the value itself).
struct Parts {
  const double* p;
  int n;
};
// Scalar slots of the iteration: r.z of the last and of this iteration (they trade places), p.Ap, and
// the step length of the direction that x still lacks.
struct CgSlots {
  double* scal;
  int rz_old, rz_new, pap, asave;
};

// x = 0, z = p = inv b; partials of b.z. Returns their number. n is even, every vector 16-byte
// aligned (as below).
template <typename T>
int cg_init(int64_t n, const T* b, const T* inv, T* x, T* z, T* p, double* partial, hipStream_t s);
// z -= (rz_old / pap) inv Ap, with p.Ap from its partials; stores it in slot pap; partials of
// r.z = sum z^2 / inv (entries with inv = 0 add nothing). Returns their number.
template <typename T>
int cg_update_z(int64_t n, T* z, const T* Ap, const T* inv, Parts pap, const CgSlots& c, double* partial,
                hipStream_t s);
// p_next = z + (rz_new / rz_old) p, rz_new from its partials; slot rz_new and asave = rz_old / pap
// stored.
template <typename T>
void cg_update_p(int64_t n, T* p_next, const T* p, const T* z, Parts rz, const CgSlots& c, hipStream_t s);
// x += asave p0 + (rz_old / pap) p1, then p0 = z + (rz_new / rz_old) p1 (slot rz_new stored) unless
// last.
template <typename T>
void cg_update_x2p(int64_t n, T* x, T* p0, const T* p1, const T* z, Parts rz, const CgSlots& c, bool last,
                   hipStream_t s);
// x += (rz_old / pap) p
template <typename T>
void cg_update_x(int64_t n, T* x, const T* p, const CgSlots& c, hipStream_t s);

// The order-1 operator on the next direction, which it forms itself: p_next = z + (rz_new / rz_old) p
// (z and p of the cell and of its neighbours are read), Ap = A p_next, partials of p_next.Ap
// (apply_blocks(E)). It also brings x up to date where x2: x += asave p_next(before) + (rz_old / pap) p,
// else asave = rz_old / pap is stored; slot rz_new is stored. cells: vectors, words, penalties cell by
// cell (3D); otherwise in rows, with the packed words.
template <typename T>
void launch_p1_direction(const MeshView& m, const LevelView& l, bool cells, const T* z, const T* p,
                         T* p_next, T* Ap, T* x, bool x2, const T* kfac, Parts rz, const CgSlots& c,
                         double* partial, hipStream_t s);
// Where it is taken instead of an update of p and an apply.
bool p1_direction_pays(const MeshView& m);

}  // namespace insp
