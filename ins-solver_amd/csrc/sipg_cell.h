// Per-cell bodies of the SIPG operator kernels (trace pass, element pass, the
// one-pass order-1 element pass), shared by the single-solve and the batched
// kernels. See sipg_kernels.hip for the formulation and its reference citations.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "dg_layout.h"
#include "kernels.h"
#include "reduce.h"

namespace insp {

// Blocks are dispatched round-robin over the 8 XCDs of an MI355X. Give each
// XCD a contiguous range of cells so that neighbour gathers hit its own L2.
__device__ __forceinline__ int64_t xcd_block() {
  const int nb = gridDim.x, b = blockIdx.x;
  const int q = nb >> 3, rem = nb & 7, x = b & 7, k = b >> 3;
  return (int64_t)(x * q + (x < rem ? x : rem) + k);
}

// Operator tables (matrices and index tables) are read-only for a whole launch and the
// same for every lane: reading them through the constant address space lets the compiler
// fetch them with scalar loads into SGPRs whether the pointer came from a kernel argument
// or from a problem descriptor.
template <typename T>
using cptr = const __attribute__((address_space(4))) T*;
template <typename T>
__device__ __forceinline__ cptr<T> as_const(const T* p) {
  return (cptr<T>)p;
}

// Coefficient at an index: VAR 0 = constant 1, 1 = from kfac, 2 = from kfac when it is
// not null (decided per problem at run time; one code path for both).
template <int VAR, typename T>
__device__ __forceinline__ T kval(const T* __restrict__ kfac, int64_t idx) {
  if constexpr (VAR == 0) return (T)1;
  else if constexpr (VAR == 1) return kfac[idx];
  else return kfac ? kfac[idx] : (T)1;
}

// Mass term of the viscous operator, J M (mm o u) (per node from mm, else the constant mmc), where on.
template <typename T>
struct MassTerm {
  const double* J = nullptr;
  const T* mm = nullptr;
  T mmc = 0;
  bool on = false;
};

// Its node columns one after the other, in the volume term's loop over them. The column's value is
// loaded again (registers have no run-time index) one column ahead, so that its wait lies behind a
// column's arithmetic; the unrolled form keeps all of M in spilled scalar registers.
template <typename T>
struct MassColumns {
  const MassTerm<T>& m;
  const T* __restrict__ u;
  int64_t e, stride;
  T Je, next;
  __device__ __forceinline__ T load(int j) const {
    return (m.mm ? m.mm[j * stride + e] : m.mmc) * u[j * stride + e];
  }
  __device__ __forceinline__ MassColumns(const MassTerm<T>& mass, const T* __restrict__ uu, int64_t cell,
                                         int64_t st, int j0, bool on)
      : m(mass), u(uu), e(cell), stride(st), Je(on ? (T)mass.J[cell] : (T)0), next(on ? load(j0) : (T)0) {}
  // acc += column j; j1: the end of the loop
  template <int Np>
  __device__ __forceinline__ void add(int j, int j1, cptr<T> __restrict__ row, T (&acc)[Np]) {
    const T v = Je * next;
    next = load(j + 1 < j1 ? j + 1 : j);
#pragma unroll
    for (int i = 0; i < Np; ++i) acc[i] = fma(row[i], v, acc[i]);
  }
};

// Trace pass for one cell: T = sJ n.(k grad u) at every face node. Per node h = k K grad u is
// formed once; a face's trace is sum_r alpha_{f,r} h_r with the compile-time face coefficients
// (one row of h, or the sum of its rows on the slanted face), so no per-face coefficient table
// stays live across the node loop.
template <int DIM, int N, typename T, int VAR>
__device__ __forceinline__ void
trace_cell(int64_t e, int64_t stride, const T* __restrict__ u, const double* __restrict__ Kt,
           const T* __restrict__ kfac, cptr<T> __restrict__ C, T* __restrict__ tr) {
  constexpr OpLayout L = op_layout(DIM, N);
  constexpr int Np = L.Np, Nfp = L.Nfp, Nf = L.Nf;
  constexpr FmaskTable FM = make_fmask(DIM, N);
  T uu[Np];
#pragma unroll
  for (int m = 0; m < Np; ++m) uu[m] = u[m * stride + e];
  T K[L.NK];
#pragma unroll
  for (int k = 0; k < L.NK; ++k) K[k] = (T)Kt[k * stride + e];
#pragma unroll
  for (int p = 0; p < Np; ++p) {
    T g[DIM];
#pragma unroll
    for (int s = 0; s < DIM; ++s) {
      T a = 0;
#pragma unroll
      for (int m = 0; m < Np; ++m) a = fma(C[L.off_D + (s * Np + p) * Np + m], uu[m], a);
      g[s] = a;
    }
    const T kp = kval<VAR>(kfac, p * stride + e);
    T h[DIM];
#pragma unroll
    for (int r = 0; r < DIM; ++r) {
      T a = 0;
#pragma unroll
      for (int s = 0; s < DIM; ++s) a = fma(K[kidx(DIM, r, s)], g[s], a);
      h[r] = kp * a;
    }
#pragma unroll
    for (int f = 0; f < Nf; ++f)
#pragma unroll
      for (int j = 0; j < Nfp; ++j)
        if (FM.v[f * Nfp + j] == p) {
          T v = 0;
#pragma unroll
          for (int r = 0; r < DIM; ++r)
            if (face_alpha(DIM, f, r) != 0.0) v += (T)face_alpha(DIM, f, r) * h[r];
          tr[(int64_t)(f * Nfp + j) * stride + e] = v;
        }
  }
}

// Where the element pass leaves (A u) at flat index k: stored as it is, or consumed by a
// functor out(k, (A u)_k, u_k).
template <typename T>
__device__ __forceinline__ void store_out(T* __restrict__ o, int64_t k, T acc, T) {
  o[k] = acc;
}
template <typename T, class O>
__device__ __forceinline__ void store_out(const O& o, int64_t k, T acc, T u) {
  o(k, acc, u);
}

// One Chebyshev step taken in place of the store, in three-term form: res = D^-1 (f - A x),
// x_next = x + c1 (x - x_prev) + c2 res (x_prev not read when c1 = 0, zero when null). x_next goes
// to another buffer than x (the pass still reads x); it may be x_prev's, each entry being read
// before it is written by the same thread.
template <typename T>
struct ChebOut {
  const T* f;
  const T* inv;
  const T* prev;
  T* x_next;
  T c1, c2;
  __device__ __forceinline__ void operator()(int64_t k, T acc, T u) const {
    const T res = inv[k] * (f[k] - acc);
    T di = c2 * res;
    if (c1 != (T)0) di = fma(c1, prev ? u - prev[k] : u, di);
    x_next[k] = u + di;
  }
};

// Whether the element pass loads a whole face at a time: 2D, and 3D up to order 3 in FP32 and order 2 in
// FP64. 3D faces of order 4, and of order 3 in FP64, go one node at a time: larger rounds cost a wave
// per SIMD and measured slower (64^3x6 tets, FP64 order 3: 731 us per element pass one node at a
// time, 774 us two at a time, 1021 us whole faces; 48^3x6, FP64 order 4: 1116 us one at a time, 1322
// us five). With the loads of a node issued a node ahead: FP64 order 3, 384,000 cells 184 -> 161 us,
// 64^3x6 745 -> 666 us; order 4, 384,000 cells 584 -> 534 us.
constexpr bool whole_faces(int dim, int N, int bytes) {
  return !(dim == 3 && (N == 4 || (N == 3 && bytes == 8)));
}

// Whether a pass that takes the face nodes one by one fetches a node ahead. With slip faces at order 3 the
// second node's values cost the third wave per SIMD (187 instead of 167 registers): 196,608 cells 140 us
// per component without, 236 with. At order 4 there are two waves either way.
template <class Slip>
constexpr bool node_ahead(int N) {
  return !(Slip::enabled && N == 3);
}

// The terms of face node j of face f (volume node p), from its own and the neighbour's value and trace and
// its coefficient: into acc, or (FOLD) the symmetry term's face mass product into sv. (Written out in a lambda
// it spilled up to 244 scalar registers at 2D order 2: Chebyshev step, 180,000 cells, FP64 with a
// coefficient 16.3 -> 13.7 us, FP32 11.3 -> 9.9.)
template <int DIM, int N, typename T, bool FOLD, class Slip>
__device__ __forceinline__ void
face_node(int f, int j, int p, int64_t e, int64_t stride, int mode, int nb, T ts, T umj, T tm, T up, T Tp, T k,
          const T (&beta)[DIM], cptr<T> __restrict__ C, const Slip& slip, T (&acc)[op_layout(DIM, N).Np],
          T (&sv)[op_layout(DIM, N).Nfp]) {
  constexpr OpLayout L = op_layout(DIM, N);
  constexpr int Np = L.Np, Nfp = L.Nfp;
  constexpr FmaskTable FM = make_fmask(DIM, N);
  if constexpr (Slip::enabled) {
    if (mode == 3) {
      const double* n = slip.bn + (int64_t)(-nb - 1) * DIM;
      T su = 0, st = 0;
#pragma unroll
      for (int d = 0; d < DIM; ++d) {
        su = fma((T)n[d], slip.u0[d * slip.cstride + p * stride + e], su);
        st = fma((T)n[d], slip.tr0[d * slip.tstride + (int64_t)(f * Nfp + j) * stride + e], st);
      }
      umj = (T)n[slip.comp] * su;
      tm = (T)n[slip.comp] * st;
    }
  }
  const T upj = mode == 0 ? up : -umj;
  const T tpj = mode == 0 ? Tp : -tm;
  const T jump = umj - upj;
  const T F = (T)0.5 * (ts * jump - (tm - tpj));
  T sig = (T)-0.5 * jump;
  sig *= k;
#pragma unroll
  for (int i = 0; i < Nfp; ++i) {
    const T mf = C[L.off_MfT + (f * Nfp + j) * Nfp + i];
    acc[FM.v[f * Nfp + i]] = fma(mf, F, acc[FM.v[f * Nfp + i]]);
    if constexpr (FOLD) sv[i] = fma(mf, sig, sv[i]);
  }
  if constexpr (!FOLD) {
#pragma unroll
    for (int r = 0; r < DIM; ++r) {
      const T bs = beta[r] * sig;
#pragma unroll
      for (int i = 0; i < Np; ++i)
        acc[i] = fma(C[L.off_Wt + ((f * DIM + r) * Nfp + j) * Np + i], bs, acc[i]);
    }
  }
}

// One cell of the element pass; returns u.(A u) over the cell. PACK: nbr holds the packed
// words (neighbour << 5) | code, -(bface+1) on the boundary, and code is not read.
template <int DIM, int N, typename T, int VAR, bool PACK = false, class Out = T*,
          class Slip = NoSlip, bool MASS = false>
__device__ __forceinline__ double
apply_cell(int64_t e, int64_t stride, const T* __restrict__ u, const T* __restrict__ tr,
           const double* __restrict__ Kt, const double* __restrict__ tauS,
           const int* __restrict__ nbr, const int* __restrict__ code,
           const int* __restrict__ bctype, const T* __restrict__ kfac, cptr<T> __restrict__ C,
           cptr<int> __restrict__ tab, Out out, const Slip& slip = Slip{},
           const MassTerm<T>& mass = MassTerm<T>{}) {
  constexpr OpLayout L = op_layout(DIM, N);
  constexpr int Np = L.Np, Nfp = L.Nfp, Nf = L.Nf;
  constexpr FmaskTable FM = make_fmask(DIM, N);
  T uu[Np], acc[Np];
#pragma unroll
  for (int m = 0; m < Np; ++m) {
    uu[m] = u[m * stride + e];
    acc[m] = 0;
  }
  T K[L.NK];
#pragma unroll
  for (int k = 0; k < L.NK; ++k) K[k] = (T)Kt[k * stride + e];
  int nbf[Nf], cf[Nf];
  T tsf[Nf];
#pragma unroll
  for (int f = 0; f < Nf; ++f) {
    if constexpr (PACK) {
      const int w = nbr[f * stride + e];
      nbf[f] = w >= 0 ? w >> 5 : w;
      cf[f] = w & 31;
    } else {
      nbf[f] = nbr[f * stride + e];
      cf[f] = nbf[f] >= 0 ? code[f * stride + e] : 0;
    }
    tsf[f] = (T)tauS[f * stride + e];
  }

  // Volume term, one node column at a time.
  MassColumns<T> mc(mass, u, e, stride, 0, MASS);
  for (int j = 0; j < Np; ++j) {
    T g[DIM];
#pragma unroll
    for (int s = 0; s < DIM; ++s) {
      T a = 0;
#pragma unroll
      for (int m = 0; m < Np; ++m) a = fma(C[L.off_D + (s * Np + j) * Np + m], uu[m], a);
      g[s] = a;
    }
    T kj = 1;
    kj = kval<VAR>(kfac, j * stride + e);
#pragma unroll
    for (int r = 0; r < DIM; ++r) {
      T h = 0;
#pragma unroll
      for (int s = 0; s < DIM; ++s) h = fma(K[kidx(DIM, r, s)], g[s], h);
      h *= kj;
#pragma unroll
      for (int i = 0; i < Np; ++i) acc[i] = fma(C[L.off_Bt + (r * Np + j) * Np + i], h, acc[i]);
    }
    if constexpr (MASS) mc.add(j, Np, C + L.off_M + j * Np, acc);
  }

  // Face terms. Where the registers allow it a face's loads are issued in two rounds before its
  // arithmetic: the cell's own traces with the node map of the shared face, then the neighbour's
  // values and traces at the mapped nodes; the loops unroll completely and the cell's own face-node
  // values come from registers. Otherwise the nodes go one at a time. A boundary face reads the
  // cell's own entries in the second round and does not use them.
  constexpr bool whole = whole_faces(DIM, N, (int)sizeof(T));
#pragma unroll
  for (int f = 0; f < Nf; ++f) {
    T beta[DIM];
#pragma unroll
    for (int s = 0; s < DIM; ++s) {
      T b = 0;
#pragma unroll
      for (int r = 0; r < DIM; ++r) b += (T)face_alpha(DIM, f, r) * K[kidx(DIM, r, s)];
      beta[s] = b;
    }
    const int nb = nbf[f];
    int mode = 0;  // 0 interior, 1 Dirichlet, 2 Neumann (or other: no terms), 3 slip
    if (nb < 0) {
      const int bt = bctype[-nb - 1];
      mode = bt == 0 ? 1 : (Slip::enabled && bt == 2 ? 3 : 2);
    }
    if (mode == 2) continue;
    const int64_t q = nb >= 0 ? (int64_t)nb : e;
    const int tbase = L.tab_nbr + (f * Nf * L.nperm + (nb >= 0 ? cf[f] : 0)) * Nfp;
    const T ts = tsf[f];
    // FP32 order 3 in 3D lifts the symmetry term through the face mass and the rows of D_r
    // (fewer coefficient loads, 0.47 vs 0.51 ms on 262k cells); elsewhere the extra live
    // registers cost more than the loads saved (FP64 order 4 spills), so the D_r^T EMAT_f
    // table is read per face node.
    constexpr bool fold = sizeof(T) == 4 && DIM == 3 && N == 3;
    T sv[Nfp];
#pragma unroll
    for (int i = 0; i < Nfp; ++i) sv[i] = 0;
    auto node = [&](int j, int p, T um, T tm, T up, T Tp, T k) {
      face_node<DIM, N, T, fold>(f, j, p, e, stride, mode, nb, ts, um, tm, up, Tp, k, beta, C, slip, acc, sv);
    };
    if constexpr (whole) {
      T Tm[Nfp], up[Nfp], Tp[Nfp];
      int pk[Nfp];
#pragma unroll
      for (int j = 0; j < Nfp; ++j) {
        Tm[j] = tr[(int64_t)(f * Nfp + j) * stride + e];
        pk[j] = tab[tbase + j];
      }
#pragma unroll
      for (int j = 0; j < Nfp; ++j) {
        up[j] = u[(int64_t)(pk[j] >> 6) * stride + q];
        Tp[j] = tr[(int64_t)(pk[j] & 63) * stride + q];
      }
#pragma unroll
      for (int j = 0; j < Nfp; ++j)
        node(j, FM.v[f * Nfp + j], uu[FM.v[f * Nfp + j]], Tm[j], up[j], Tp[j],
             kval<VAR>(kfac, FM.v[f * Nfp + j] * stride + e));
    } else {
      // one node at a time, where node_ahead its loads issued during the node before and the node map's entry
      // during the one before that
      struct Node {
        int p;
        T um, Tm, up, Tp, k;
      };
      auto load = [&](int j, int pk) {
        Node x;
        x.p = tab[L.tab_fmask + f * Nfp + j];
        x.um = u[x.p * stride + e];
        x.Tm = tr[(int64_t)(f * Nfp + j) * stride + e];
        x.k = kval<VAR>(kfac, x.p * stride + e);
        x.up = u[(int64_t)(pk >> 6) * stride + q];
        x.Tp = tr[(int64_t)(pk & 63) * stride + q];
        return x;
      };
      if constexpr (!node_ahead<Slip>(N)) {
#pragma unroll 1
        for (int j = 0; j < Nfp; ++j) {
          const Node x = load(j, tab[tbase + j]);
          node(j, x.p, x.um, x.Tm, x.up, x.Tp, x.k);
        }
      } else {
        Node cur = load(0, tab[tbase]);
        int pk = tab[tbase + 1];
#pragma unroll 1
        for (int j = 0; j < Nfp; ++j) {
          const Node nxt = load(j + 1 < Nfp ? j + 1 : j, pk);
          pk = tab[tbase + (j + 2 < Nfp ? j + 2 : Nfp - 1)];
          node(j, cur.p, cur.um, cur.Tm, cur.up, cur.Tp, cur.k);
          cur = nxt;
        }
      }
    }
    // symmetry term sum_r beta_r D_r^T (EMAT_f sig): the face mass first, then the rows
    // of D_r at the face nodes
    if constexpr (fold) {
#pragma unroll
      for (int l = 0; l < Nfp; ++l) {
        const int m = FM.v[f * Nfp + l];
#pragma unroll
        for (int r = 0; r < DIM; ++r) {
          const T w = beta[r] * sv[l];
#pragma unroll
          for (int i = 0; i < Np; ++i) acc[i] = fma(C[L.off_D + (r * Np + m) * Np + i], w, acc[i]);
        }
      }
    }
  }
  double dotv = 0.0;
#pragma unroll
  for (int i = 0; i < Np; ++i) {
    store_out(out, (int64_t)i * stride + e, acc[i], uu[i]);
    dotv += (double)uu[i] * (double)acc[i];
  }
  return dotv;
}

// Order 1 in one pass: the gradient of a P1 cell is constant, so the neighbour's
// flux trace k n.grad(u) is recomputed from its Np nodal values and metric instead
// of being stored by a trace pass. Same operator as apply_cell. The face coefficients
// alpha_{f,r} (face_alpha) are 1 for every r on the slanted face f = DIM-1 and -1 for one r
// on the others: r = DIM-1-f before the slanted face, DIM-f after it.
constexpr bool face_alpha_is_rows(int dim) {
  for (int f = 0; f <= dim; ++f)
    for (int r = 0; r < dim; ++r) {
      const int row = f < dim - 1 ? dim - 1 - f : dim - f;
      const double want = f == dim - 1 ? 1.0 : (r == row ? -1.0 : 0.0);
      if (face_alpha(dim, f, r) != want) return false;
    }
  return true;
}
static_assert(face_alpha_is_rows(2) && face_alpha_is_rows(3), "face coefficient rows");

// Entry i (0 <= i < n) of a small register array, selected by a chain of compares. The chain
// starts from zero rather than from v[0], so that no select has two array entries as its
// operands: the compiler would turn such a select into a load through a selected address and
// move the array to scratch memory.
template <int n, typename T>
__device__ __forceinline__ T pick(const T (&v)[n], int i) {
  T r = (T)0;
#pragma unroll
  for (int k = 0; k < n; ++k) r = i == k ? v[k] : r;
  return r;
}

// PACK: nbr holds one word per face, (neighbour << 5) | code inside the mesh and the
// boundary index -(bface+1) on the boundary, and code is not read.
//
// Loads are issued in two rounds, so that a wave waits for memory twice per cell instead of
// several times per face: first everything addressed by the cell index (neighbour words,
// nodal values, metric, penalties), then everything addressed by a neighbour index (the
// neighbour's nodal values and whole metric, and the node map of the shared face). A
// boundary face reads the cell's own entries in the second round and does not use them.
// Where the order-1 element pass finds the neighbour's node at a face node: in the operator's
// integer table (TabNodes: one load per face node), or in bit fields passed with the launch
// (BitNodes: no load, and no registers held while the other loads are in flight).
struct TabNodes {};
struct BitNodes {
  P1NodeBits b;
};

// What the order-1 pass holds of a cell and its neighbours after its loads.
template <int DIM, typename T>
struct P1Loads {
  static constexpr OpLayout L = op_layout(DIM, 1);
  static constexpr int Np = L.Np, Nfp = L.Nfp, Nf = L.Nf, NK = L.NK;
  int nb[Nf], c[Nf];                       // neighbour or -(bface+1), its code
  T uu[Np], kk[Np], K[NK], ts[Nf];         // values, coefficient, metric, penalties
  T un[Nf][Np], kn[Nf][NK], fn_k[Nf][Np];  // the neighbours' values, metric, coefficient
  int nd[Nf][Nfp], bt[Nf];                 // neighbour's node at each face node; boundary type
  // the cell behind face f, or the cell itself
  __device__ __forceinline__ int64_t at(int f, int64_t e) const { return nb[f] >= 0 ? (int64_t)nb[f] : e; }
};

// Nodal values of cell q of an order-1 vector: in rows, or (VCM, 3D) cell by cell ([E][Np], 16 or 32
// bytes per cell).
template <int Np, bool VCM, typename T>
__device__ __forceinline__ void p1_values(const T* __restrict__ u, int64_t stride, int64_t q, T* dst) {
  if constexpr (VCM) {
    static_assert(Np == 4, "cell-by-cell values: 3D order 1");
    if constexpr (sizeof(T) == 8) {
      const double2* uq = reinterpret_cast<const double2*>(u) + q * 2;
      const double2 a = uq[0], b = uq[1];
      dst[0] = a.x; dst[1] = a.y; dst[2] = b.x; dst[3] = b.y;
    } else {
      const float4 a = reinterpret_cast<const float4*>(u)[q];
      dst[0] = a.x; dst[1] = a.y; dst[2] = a.z; dst[3] = a.w;
    }
  } else {
#pragma unroll
    for (int m = 0; m < Np; ++m) dst[m] = u[m * stride + q];
  }
}

template <int Np, bool VCM, typename T>
__device__ __forceinline__ void p1_store(T* o, int64_t stride, int64_t e, const T (&v)[Np]) {
  if constexpr (VCM) {
    static_assert(Np == 4, "cell-by-cell values: 3D order 1");
    if constexpr (sizeof(T) == 8) {
      double2* oq = reinterpret_cast<double2*>(o) + e * 2;
      oq[0] = make_double2(v[0], v[1]);
      oq[1] = make_double2(v[2], v[3]);
    } else {
      reinterpret_cast<float4*>(o)[e] = make_float4(v[0], v[1], v[2], v[3]);
    }
  } else {
#pragma unroll
    for (int m = 0; m < Np; ++m) o[m * stride + e] = v[m];
  }
}

// Two-bit field c of w (c < 6 in 2D, < 24 in 3D), by 32-bit shifts. With one 64-bit shift the 2D order-1 apply
// gave wrong results in about one wave of 2000 (125,000 cells, other ones on every launch); its v_lshrrev_b64
// had the amount in the last VGPR of the wave's allocation (v79 of 80). That the instruction was the cause is
// inferred: 32-bit shifts also change the register allocation. (gfx90a has this fault, and LLVM keeps such
// amounts out of that register there.)
template <int DIM>
__device__ __forceinline__ int node_field(unsigned long long w, int c) {
  const unsigned lo = (unsigned)w, hi = (unsigned)(w >> 32);
  if constexpr (DIM == 2) return (int)((lo >> (2 * c)) & 3u);
  else return (int)(((c < 16 ? lo : hi) >> ((2 * c) & 31)) & 3u);
}

// Both rounds of loads. VCM: u holds the values, nbr the packed words and tauS the penalties cell by
// cell ([E][4]); the coefficient stays in rows. KAOS: Kt holds the metric cell by cell ([E][NK]).
template <int DIM, typename T, int VAR, bool PACK, class Nodes, bool KAOS, bool VCM>
__device__ __forceinline__ void
p1_load(int64_t e, int64_t stride, const T* __restrict__ u, const double* __restrict__ Kt,
        const double* __restrict__ tauS, const int* __restrict__ nbr, const int* __restrict__ code,
        const int* __restrict__ bctype, const T* __restrict__ kfac, cptr<int> __restrict__ tab,
        const Nodes& nodes, P1Loads<DIM, T>& P) {
  constexpr OpLayout L = op_layout(DIM, 1);
  constexpr int Np = L.Np, Nfp = L.Nfp, Nf = L.Nf, NK = L.NK;
  static_assert(!VCM || PACK, "cell-by-cell values: packed words");
  int wcell[Nf];
  if constexpr (VCM) {
    const int4 w4 = reinterpret_cast<const int4*>(nbr)[e];
    wcell[0] = w4.x; wcell[1] = w4.y; wcell[2] = w4.z; wcell[3] = w4.w;
  }
#pragma unroll
  for (int f = 0; f < Nf; ++f) {
    if constexpr (PACK) {
      const int w = VCM ? wcell[f] : nbr[f * stride + e];
      P.nb[f] = w >= 0 ? w >> 5 : w;
      P.c[f] = w >= 0 ? (w & 31) : 0;
    } else {
      P.nb[f] = nbr[f * stride + e];
      P.c[f] = P.nb[f] >= 0 ? code[f * stride + e] : 0;
    }
  }
  p1_values<Np, VCM>(u, stride, e, P.uu);
#pragma unroll
  for (int m = 0; m < Np; ++m) P.kk[m] = kval<VAR>(kfac, m * stride + e);
  static_assert(!KAOS || NK % 2 == 0, "the cell-by-cell metric is read in pairs");
  auto metric = [&](int64_t q, T* dst) {
    if constexpr (KAOS) {
      const double2* kq = reinterpret_cast<const double2*>(Kt) + q * (NK / 2);
#pragma unroll
      for (int k = 0; k < NK / 2; ++k) {
        const double2 v = kq[k];
        dst[2 * k] = (T)v.x;
        dst[2 * k + 1] = (T)v.y;
      }
    } else {
#pragma unroll
      for (int k = 0; k < NK; ++k) dst[k] = (T)Kt[k * stride + q];
    }
  };
  metric(e, P.K);
  if constexpr (VCM) {
    const double2* tq = reinterpret_cast<const double2*>(tauS) + e * 2;
    const double2 t01 = tq[0], t23 = tq[1];
    P.ts[0] = (T)t01.x; P.ts[1] = (T)t01.y; P.ts[2] = (T)t23.x; P.ts[3] = (T)t23.y;
  } else {
#pragma unroll
    for (int f = 0; f < Nf; ++f) P.ts[f] = (T)tauS[f * stride + e];
  }
  // round 2
#pragma unroll
  for (int f = 0; f < Nf; ++f) {
    const bool in = P.nb[f] >= 0;
    const int64_t q = P.at(f, e);
    const int cf = in ? P.c[f] : 0;
    p1_values<Np, VCM>(u, stride, q, P.un[f]);
#pragma unroll
    for (int m = 0; m < Np; ++m) P.fn_k[f][m] = kval<VAR>(kfac, m * stride + q);
    metric(q, P.kn[f]);
#pragma unroll
    for (int j = 0; j < Nfp; ++j) {
      if constexpr (std::is_same<Nodes, BitNodes>::value)
        P.nd[f][j] = node_field<DIM>(nodes.b.w[DIM == 3 ? 0 : f][j], cf);  // 3D: the same row for every face
      else
        P.nd[f][j] = tab[L.tab_nbr + (f * Nf * L.nperm + cf) * Nfp + j] >> 6;
    }
    P.bt[f] = in ? 0 : bctype[-P.nb[f] - 1];
  }
}

// The arithmetic: acc = (A u) at the cell's nodes; returns u.(A u) over the cell.
template <int DIM, typename T, int VAR, class Slip>
__device__ __forceinline__ double
p1_compute(int64_t e, int64_t stride, const P1Loads<DIM, T>& P, const Slip& slip,
           T (&acc)[op_layout(DIM, 1).Np]) {
  constexpr OpLayout L = op_layout(DIM, 1);
  constexpr int Np = L.Np, Nfp = L.Nfp, Nf = L.Nf;
  constexpr FmaskTable FM = make_fmask(DIM, 1);
  const auto& nb = P.nb;
  const auto& c = P.c;
  const auto& uu = P.uu;
  const auto& kk = P.kk;
  const auto& K = P.K;
  const auto& ts = P.ts;
  const auto& un = P.un;
  const auto& kn = P.kn;
  const auto& fn_k = P.fn_k;
  const auto& nd = P.nd;
  const auto& bt = P.bt;
#pragma unroll
  for (int m = 0; m < Np; ++m) acc[m] = 0;
  // P1: grad phi_i is constant, so Bt[r][j][i] = dphi_ri m_j and Wt[f][r][j][i] = dphi_ri w_j
  // (m, w: column sums of the mass and face mass). The volume term and every face's symmetry
  // term collapse into one vector V: acc_i += sum_r dphi_ri V_r at the end, with
  // V = (sum_j m_j k_j) h + sum_f beta_f sum_j w_j sig_fj.
  // c_f: the face mass factor; c_s = -w/2 with the face mass column sum w = c_f (Nfp + 1)
  constexpr T c_m = (T)p1_mass_colsum(DIM), c_f = (T)p1_face_mass_c(DIM),
              c_s = (T)(-0.5 * p1_face_mass_c(DIM) * (Nfp + 1));
  double dotv = 0.0;
  T g[DIM];
#pragma unroll
  for (int s = 0; s < DIM; ++s) g[s] = (T)0.5 * (uu[s + 1] - uu[0]);
  T h[DIM];
#pragma unroll
  for (int r = 0; r < DIM; ++r) {
    T a = 0;
#pragma unroll
    for (int s = 0; s < DIM; ++s) a = fma(K[kidx(DIM, r, s)], g[s], a);
    h[r] = a;
  }
  T V[DIM];
  {
    T ks = kk[0];
#pragma unroll
    for (int j = 1; j < Np; ++j) ks += kk[j];
    const T mk = c_m * ks;
#pragma unroll
    for (int r = 0; r < DIM; ++r) V[r] = mk * h[r];
  }
#pragma unroll
  for (int f = 0; f < Nf; ++f) {
    T beta[DIM];
    T tm0 = 0;
#pragma unroll
    for (int s = 0; s < DIM; ++s) {
      T b = 0;
#pragma unroll
      for (int r = 0; r < DIM; ++r) b += (T)face_alpha(DIM, f, r) * K[kidx(DIM, r, s)];
      beta[s] = b;
      tm0 = fma(b, g[s], tm0);
    }
    // 0 interior, 1 Dirichlet, 2 Neumann (or other: no terms), 3 slip
    const int mode = nb[f] >= 0 ? 0 : (bt[f] == 0 ? 1 : (Slip::enabled && bt[f] == 2 ? 3 : 2));
    if (mode == 2) continue;
    // the neighbour's flux trace sum_s (sum_r alpha_{fn,r} K_n[r][s]) (grad u_n)_s, constant on
    // a P1 cell; alpha_{fn,r} is selected per lane from the compile-time face table
    T tn0 = 0;
    if (mode == 0) {
      const int fn = c[f] / L.nperm;
      T gn[DIM];
#pragma unroll
      for (int s = 0; s < DIM; ++s) gn[s] = (T)0.5 * (un[f][s + 1] - un[f][0]);
#pragma unroll
      for (int r = 0; r < DIM; ++r) {
        T al = (T)face_alpha(DIM, 0, r);
#pragma unroll
        for (int k = 1; k < Nf; ++k) al = fn == k ? (T)face_alpha(DIM, k, r) : al;
        T t = 0;
#pragma unroll
        for (int s = 0; s < DIM; ++s) t = fma(kn[f][kidx(DIM, r, s)], gn[s], t);
        tn0 = fma(al, t, tn0);
      }
    }
    // slip: n_c (n.U) at the face nodes and n_c sum_d n_d (beta.grad u_d), the gradients of
    // the components recomputed from their nodal values (constant on a P1 cell)
    T nc = 0, sm0 = 0;
    const double* bnv = nullptr;
    if constexpr (Slip::enabled) {
      if (mode == 3) {
        bnv = slip.bn + (int64_t)(-nb[f] - 1) * DIM;
        nc = (T)bnv[slip.comp];
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
          const T* ud = slip.u0 + d * slip.cstride;
          const T u0 = ud[e];
          T t = 0;
#pragma unroll
          for (int s2 = 0; s2 < DIM; ++s2) t = fma(beta[s2], (T)0.5 * (ud[(s2 + 1) * stride + e] - u0), t);
          sm0 = fma((T)bnv[d], t, sm0);
        }
      }
    }
    T F[Nfp], Fs = 0, S = 0;
#pragma unroll
    for (int j = 0; j < Nfp; ++j) {
      const int p = FM.v[f * Nfp + j];
      T um = uu[p];
      T Tm = kk[p] * tm0;
      if constexpr (Slip::enabled) {
        if (mode == 3) {
          T su = 0;
#pragma unroll
          for (int d = 0; d < DIM; ++d) su = fma((T)bnv[d], slip.u0[d * slip.cstride + p * stride + e], su);
          um = nc * su;
          Tm = kk[p] * nc * sm0;
        }
      }
      T up, Tp;
      if (mode == 0) {
        up = pick(un[f], nd[f][j]);
        Tp = (VAR == 0 ? (T)1 : pick(fn_k[f], nd[f][j])) * tn0;
      } else {
        up = -um;
        Tp = -Tm;
      }
      const T jump = um - up;
      F[j] = (T)0.5 * (ts[f] * jump - (Tm - Tp));
      Fs += F[j];
      S = fma(jump, kk[p], S);
    }
    // face mass c (1 + delta_ij): sum_j M_ij F_j = c (F_i + sum_j F_j); sig_j = -jump_j k_j / 2
#pragma unroll
    for (int i = 0; i < Nfp; ++i) acc[FM.v[f * Nfp + i]] = fma(c_f, F[i] + Fs, acc[FM.v[f * Nfp + i]]);
    const T sw = c_s * S;
#pragma unroll
    for (int r = 0; r < DIM; ++r) V[r] = fma(beta[r], sw, V[r]);
  }
  {
    T v0 = V[0];
#pragma unroll
    for (int r = 1; r < DIM; ++r) v0 += V[r];
    acc[0] = fma((T)-0.5, v0, acc[0]);
#pragma unroll
    for (int r = 0; r < DIM; ++r) acc[r + 1] = fma((T)0.5, V[r], acc[r + 1]);
  }
#pragma unroll
  for (int i = 0; i < Np; ++i) dotv += (double)uu[i] * (double)acc[i];
  return dotv;
}

template <int DIM, typename T, int VAR, bool PACK = false, class Out = T*, class Slip = NoSlip,
          class Nodes = TabNodes, bool KAOS = false, bool VCM = false>
__device__ __forceinline__ double
apply_p1_cell(int64_t e, int64_t stride, const T* __restrict__ u, const double* __restrict__ Kt,
              const double* __restrict__ tauS, const int* __restrict__ nbr,
              const int* __restrict__ code, const int* __restrict__ bctype,
              const T* __restrict__ kfac, cptr<T> __restrict__ C, cptr<int> __restrict__ tab,
              Out out, const Slip& slip = Slip{}, const Nodes& nodes = Nodes{}) {
  constexpr int Np = op_layout(DIM, 1).Np;
  (void)C;
  P1Loads<DIM, T> P;
  p1_load<DIM, T, VAR, PACK, Nodes, KAOS, VCM>(e, stride, u, Kt, tauS, nbr, code, bctype, kfac, tab,
                                               nodes, P);
  T acc[Np];
  const double dotv = p1_compute<DIM, T, VAR>(e, stride, P, slip, acc);
  if constexpr (VCM) {
    static_assert(std::is_same<Out, T*>::value, "cell-by-cell values: plain output");
    p1_store<Np, true>(out, stride, e, acc);
  } else {
#pragma unroll
    for (int i = 0; i < Np; ++i) store_out(out, (int64_t)i * stride + e, acc[i], P.uu[i]);
  }
  return dotv;
}

}  // namespace insp
