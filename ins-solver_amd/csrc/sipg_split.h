// Trace and element passes that give a cell to four waves: a block of 256 threads owns 64 cells, lane
// l of every wave the same cell. The waves share out the node columns of the volume term and the
// faces (2D: three waves a face each, the fourth more columns), accumulate their parts of A u and add
// them through LDS in a fixed order. Matrices stay wave-uniform (each wave reads other rows of them),
// as in the passes with one thread per cell (sipg_cell.h), whose operator this is; a cell's serial
// chain is a quarter as long and there are four times the waves.
#pragma once

#include <type_traits>

#include "sipg_cell.h"

namespace insp {

// First node column of wave w: the columns that balance the waves' work, counted in FMAs.
template <int DIM, int N>
struct SplitCols {
  int b[5];
  constexpr SplitCols() : b{} {
    constexpr OpLayout L = op_layout(DIM, N);
    const int col = 2 * DIM * L.Np, face = L.Nfp * (L.Nfp + DIM * L.Np);
    int done = 0;
    for (int w = 0; w < 4; ++w) {
      b[w] = done;
      const int has = w < L.Nf ? face : 0;
      // what is left over goes in equal parts to the waves that are left
      int faces_left = 0;
      for (int v = w; v < L.Nf; ++v) faces_left += face;
      const int left = (L.Np - done) * col + faces_left;
      int take = (left / (4 - w) - has + col / 2) / col;
      if (take < 0) take = 0;
      if (w == 3 || done + take > L.Np) take = L.Np - done;
      done += take;
    }
    b[4] = L.Np;
  }
};

// Traces at the face nodes among the volume nodes p of the wave (a quarter of them).
template <int DIM, int N, typename T, int VAR, int W>
__device__ __forceinline__ void
trace_quarter(int64_t e, int64_t stride, const T (&uu)[op_layout(DIM, N).Np],
              const double* __restrict__ Kt, const T* __restrict__ kfac, cptr<T> __restrict__ C,
              T* __restrict__ tr) {
  constexpr OpLayout L = op_layout(DIM, N);
  constexpr int Np = L.Np, Nfp = L.Nfp, Nf = L.Nf;
  constexpr FmaskTable FM = make_fmask(DIM, N);
  T K[L.NK];
#pragma unroll
  for (int k = 0; k < L.NK; ++k) K[k] = (T)Kt[k * stride + e];
#pragma unroll
  for (int p = W; p < Np; p += 4) {
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

// Volume term of the node columns [j0, j1), and their mass term.
template <int DIM, int N, typename T, int VAR>
__device__ __forceinline__ void
volume_columns(int64_t e, int64_t stride, int j0, int j1, const T (&uu)[op_layout(DIM, N).Np],
               const T (&K)[op_layout(DIM, N).NK], const T* __restrict__ u, const T* __restrict__ kfac,
               cptr<T> __restrict__ C, const MassTerm<T>& mass, T (&acc)[op_layout(DIM, N).Np]) {
  constexpr OpLayout L = op_layout(DIM, N);
  constexpr int Np = L.Np;
  MassColumns<T> mc(mass, u, e, stride, j0, mass.on);
#pragma unroll 1
  for (int j = j0; j < j1; ++j) {
    T g[DIM];
#pragma unroll
    for (int s = 0; s < DIM; ++s) {
      T a = 0;
#pragma unroll
      for (int m = 0; m < Np; ++m) a = fma(C[L.off_D + (s * Np + j) * Np + m], uu[m], a);
      g[s] = a;
    }
    const T kj = kval<VAR>(kfac, j * stride + e);
#pragma unroll
    for (int r = 0; r < DIM; ++r) {
      T h = 0;
#pragma unroll
      for (int s = 0; s < DIM; ++s) h = fma(K[kidx(DIM, r, s)], g[s], h);
      h *= kj;
#pragma unroll
      for (int i = 0; i < Np; ++i) acc[i] = fma(C[L.off_Bt + (r * Np + j) * Np + i], h, acc[i]);
    }
    if (mass.on) mc.add(j, j1, C + L.off_M + j * Np, acc);
  }
}

// One wave's part of (A u) on a cell: face W (if it has one) and its node columns. The face's loads
// are issued before the volume term where the registers allow it (PRE), so that the gathers are in
// flight during it; nbr holds the packed words.
template <int DIM, int N, typename T, int VAR, int W, class Slip>
__device__ __forceinline__ void
apply_quarter(int64_t e, int64_t stride, const T* __restrict__ u, const T* __restrict__ tr,
              const double* __restrict__ Kt, const double* __restrict__ tauS,
              const int* __restrict__ nbr, const int* __restrict__ bctype,
              const T* __restrict__ kfac, cptr<T> __restrict__ C, const int* __restrict__ tab,
              const MassTerm<T>& mass, const Slip& slip, T (&acc)[op_layout(DIM, N).Np]) {
  constexpr OpLayout L = op_layout(DIM, N);
  constexpr int Np = L.Np, Nfp = L.Nfp, Nf = L.Nf;
  constexpr FmaskTable FM = make_fmask(DIM, N);
  constexpr SplitCols<DIM, N> cols;
  static_assert(cols.b[W] < cols.b[W + 1], "every wave has a column");
  constexpr bool has_face = W < Nf;
  constexpr int F0 = has_face ? W : 0;
  int nb = 0;
  T ts = 0;
  if constexpr (has_face) {
    nb = nbr[F0 * stride + e];
    ts = (T)tauS[F0 * stride + e];
  }
  T uu[Np];
#pragma unroll
  for (int m = 0; m < Np; ++m) {
    uu[m] = u[m * stride + e];
    acc[m] = 0;
  }
  T K[L.NK];
#pragma unroll
  for (int k = 0; k < L.NK; ++k) K[k] = (T)Kt[k * stride + e];
  if constexpr (!has_face) {
    volume_columns<DIM, N, T, VAR>(e, stride, cols.b[W], cols.b[W + 1], uu, K, u, kfac, C, mass, acc);
    return;
  }
  const bool in = nb >= 0;
  int mode = 0;  // 0 interior, 1 Dirichlet, 2 Neumann (or other: no terms), 3 slip
  if (!in) {
    const int bt = bctype[-nb - 1];
    mode = bt == 0 ? 1 : (Slip::enabled && bt == 2 ? 3 : 2);
  }
  const int64_t q = in ? (int64_t)(nb >> 5) : e;
  const int* map = tab + L.tab_nbr + (F0 * Nf * L.nperm + (in ? nb & 31 : 0)) * Nfp;
  constexpr bool PRE = (3 * Nfp + 2 * Np) * (int)sizeof(T) / 4 <= 130;
  constexpr int CH = PRE || Nfp % 5 != 0 ? Nfp : 5;  // face nodes per round of loads
  T Tm[CH], up[CH], Tp[CH];
  auto gather = [&](auto J0) {
    constexpr int j0 = decltype(J0)::value;
    int pk[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      pk[j] = map[j0 + j];
      Tm[j] = tr[(int64_t)(F0 * Nfp + j0 + j) * stride + e];
    }
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      up[j] = u[(int64_t)(pk[j] >> 6) * stride + q];
      Tp[j] = tr[(int64_t)(pk[j] & 63) * stride + q];
    }
  };
  if constexpr (PRE) gather(std::integral_constant<int, 0>{});
  volume_columns<DIM, N, T, VAR>(e, stride, cols.b[W], cols.b[W + 1], uu, K, u, kfac, C, mass, acc);
  if (mode == 2) return;
  T beta[DIM];
#pragma unroll
  for (int s = 0; s < DIM; ++s) {
    T b = 0;
#pragma unroll
    for (int r = 0; r < DIM; ++r) b += (T)face_alpha(DIM, F0, r) * K[kidx(DIM, r, s)];
    beta[s] = b;
  }
  auto lift = [&](auto J0) {
    constexpr int j0 = decltype(J0)::value;
#pragma unroll
    for (int jj = 0; jj < CH; ++jj) {
      const int j = j0 + jj;
      const int p = FM.v[F0 * Nfp + j];
      T umj = uu[p], tm = Tm[jj];
      if constexpr (Slip::enabled) {
        if (mode == 3) {
          const double* n = slip.bn + (int64_t)(-nb - 1) * DIM;
          T su = 0, st = 0;
#pragma unroll
          for (int d = 0; d < DIM; ++d) {
            su = fma((T)n[d], slip.u0[d * slip.cstride + p * stride + e], su);
            st = fma((T)n[d], slip.tr0[d * slip.tstride + (int64_t)(F0 * Nfp + j) * stride + e], st);
          }
          umj = (T)n[slip.comp] * su;
          tm = (T)n[slip.comp] * st;
        }
      }
      const T upj = mode == 0 ? up[jj] : -umj;
      const T tpj = mode == 0 ? Tp[jj] : -tm;
      const T jump = umj - upj;
      const T F = (T)0.5 * (ts * jump - (tm - tpj));
      const T sig = (T)-0.5 * jump * kval<VAR>(kfac, p * stride + e);
#pragma unroll
      for (int i = 0; i < Nfp; ++i)
        acc[FM.v[F0 * Nfp + i]] = fma(C[L.off_MfT + (F0 * Nfp + j) * Nfp + i], F, acc[FM.v[F0 * Nfp + i]]);
#pragma unroll
      for (int r = 0; r < DIM; ++r) {
        const T bs = beta[r] * sig;
#pragma unroll
        for (int i = 0; i < Np; ++i)
          acc[i] = fma(C[L.off_Wt + ((F0 * DIM + r) * Nfp + j) * Np + i], bs, acc[i]);
      }
    }
  };
  auto round = [&](auto J0) {
    if constexpr (!PRE) gather(J0);
    lift(J0);
  };
  round(std::integral_constant<int, 0>{});
  if constexpr (CH < Nfp) round(std::integral_constant<int, CH>{});
  if constexpr (2 * CH < Nfp) round(std::integral_constant<int, 2 * CH>{});
  static_assert(3 * CH >= Nfp, "rounds of a face");
}

// Element pass of 64 cells by the 256 threads of a block: the waves' parts meet in LDS (part), then
// wave w adds and writes rows w, w+4, ... of every cell. Returns the thread's share of u.(A u).
template <int DIM, int N, typename T, int VAR, class Out, class Slip>
__device__ __forceinline__ double
apply_split(int64_t e, bool live, int64_t stride, const T* __restrict__ u, const T* __restrict__ tr,
            const double* __restrict__ Kt, const double* __restrict__ tauS,
            const int* __restrict__ nbr, const int* __restrict__ bctype, const T* __restrict__ kfac,
            cptr<T> __restrict__ C, const int* __restrict__ tab, const MassTerm<T>& mass, Out out,
            const Slip& slip, T (*part)[op_layout(DIM, N).Np][64]) {
  constexpr int Np = op_layout(DIM, N).Np;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (live) {
    T acc[Np];
    switch (w) {
      case 0: apply_quarter<DIM, N, T, VAR, 0>(e, stride, u, tr, Kt, tauS, nbr, bctype, kfac, C, tab, mass, slip, acc); break;
      case 1: apply_quarter<DIM, N, T, VAR, 1>(e, stride, u, tr, Kt, tauS, nbr, bctype, kfac, C, tab, mass, slip, acc); break;
      case 2: apply_quarter<DIM, N, T, VAR, 2>(e, stride, u, tr, Kt, tauS, nbr, bctype, kfac, C, tab, mass, slip, acc); break;
      default: apply_quarter<DIM, N, T, VAR, 3>(e, stride, u, tr, Kt, tauS, nbr, bctype, kfac, C, tab, mass, slip, acc); break;
    }
#pragma unroll
    for (int i = 0; i < Np; ++i) part[w][i][lane] = acc[i];
  }
  __syncthreads();
  double dotv = 0.0;
  if (live) {
#pragma unroll
    for (int i0 = 0; i0 < Np; i0 += 4) {
      const int i = i0 + w;
      if (i < Np) {
        const T a = (part[0][i][lane] + part[1][i][lane]) + (part[2][i][lane] + part[3][i][lane]);
        const T ui = u[i * stride + e];
        store_out(out, (int64_t)i * stride + e, a, ui);
        dotv += (double)ui * (double)a;
      }
    }
  }
  return dotv;
}

}  // namespace insp
