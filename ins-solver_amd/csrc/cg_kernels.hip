#include "cg_kernels.h"

#include <algorithm>
#include <stdexcept>
#include <string>

#include "reduce.h"
#include "refelem.h"
#include "sipg_cell.h"

namespace insp {

namespace {

inline void check(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    throw std::runtime_error(std::string("kernel launch failed: ") + what + ": " + hipGetErrorString(e));
}

constexpr int kBlock = kPartBlock;

// Sum of the partials, by the whole block; every thread gets it. Four loads in flight per thread,
// added in an order that depends on n alone, so all blocks and all kernels form the same value.
__device__ __forceinline__ double total(const Parts& q) {
  if (q.n == 1) return q.p[0];
  double a[4] = {0.0, 0.0, 0.0, 0.0};
  for (int i = threadIdx.x; i < q.n; i += 4 * kBlock) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = i + u * kBlock;
      if (j < q.n) a[u] += q.p[j];
    }
  }
  return block_sum1<kBlock>((a[0] + a[1]) + (a[2] + a[3]));
}

__device__ __forceinline__ double safe_div(double a, double b) { return b != 0.0 ? a / b : 0.0; }

// Two entries per access: 16 bytes FP64, 8 bytes FP32.
template <typename T> struct Pair2;
template <> struct Pair2<double> { using type = double2; };
template <> struct Pair2<float> { using type = float2; };
template <typename T> using V2 = typename Pair2<T>::type;
template <typename T>
__device__ __forceinline__ V2<T> ld2(const T* p, int64_t i) { return reinterpret_cast<const V2<T>*>(p)[i]; }
template <typename T>
__device__ __forceinline__ void st2(T* p, int64_t i, const V2<T>& v) { reinterpret_cast<V2<T>*>(p)[i] = v; }

__device__ __forceinline__ void put_partial(double v, double* partial) {
  const double t = block_sum1<kBlock>(v);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

template <typename T, int PER>
__global__ void __launch_bounds__(kBlock)
k_cg_init(int64_t n2, const T* __restrict__ b, const T* __restrict__ inv, T* __restrict__ x,
          T* __restrict__ z, T* __restrict__ p, double* __restrict__ partial) {
  double v = 0.0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int64_t i = (blockIdx.x * (int64_t)PER + k) * kBlock + threadIdx.x;
    if (i < n2) {
      const V2<T> bi = ld2(b, i), di = ld2(inv, i);
      V2<T> zi, xi;
      zi.x = di.x * bi.x;
      zi.y = di.y * bi.y;
      xi.x = xi.y = (T)0;
      st2(x, i, xi);
      st2(z, i, zi);
      st2(p, i, zi);
      v += (double)bi.x * (double)zi.x;
      v += (double)bi.y * (double)zi.y;
    }
  }
  put_partial(v, partial);
}

// The vectors are loaded before the partials are added, so that the two waits overlap.
template <typename T, int PER>
__global__ void __launch_bounds__(kBlock)
k_cg_z(int64_t n2, T* __restrict__ z, const T* __restrict__ Ap, const T* __restrict__ inv, Parts pap,
       CgSlots c, double* __restrict__ partial) {
  V2<T> zi[PER], ai[PER], di[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int64_t i = (blockIdx.x * (int64_t)PER + k) * kBlock + threadIdx.x;
    if (i < n2) {
      zi[k] = ld2(z, i);
      ai[k] = ld2(Ap, i);
      di[k] = ld2(inv, i);
    }
  }
  const double rz = c.scal[c.rz_old];
  const double pa = total(pap);
  if (blockIdx.x == 0 && threadIdx.x == 0) c.scal[c.pap] = pa;
  const T a = (T)safe_div(rz, pa);
  double v = 0.0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int64_t i = (blockIdx.x * (int64_t)PER + k) * kBlock + threadIdx.x;
    if (i < n2) {
      const V2<T> d = di[k];
      V2<T> o;
      o.x = fma(-a * d.x, ai[k].x, zi[k].x);
      o.y = fma(-a * d.y, ai[k].y, zi[k].y);
      st2(z, i, o);
      const double zx = (double)o.x, zy = (double)o.y;
      v += d.x != (T)0 ? zx * zx / (double)d.x : 0.0;
      v += d.y != (T)0 ? zy * zy / (double)d.y : 0.0;
    }
  }
  put_partial(v, partial);
}

template <typename T, int PER>
__global__ void __launch_bounds__(kBlock)
k_cg_p(int64_t n2, T* __restrict__ p_next, const T* __restrict__ p, const T* __restrict__ z, Parts rz,
       CgSlots c) {
  V2<T> pi[PER], zi[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int64_t i = (blockIdx.x * (int64_t)PER + k) * kBlock + threadIdx.x;
    if (i < n2) {
      pi[k] = ld2(p, i);
      zi[k] = ld2(z, i);
    }
  }
  const double ro = c.scal[c.rz_old];
  const double rn = total(rz);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    c.scal[c.rz_new] = rn;
    c.scal[c.asave] = safe_div(ro, c.scal[c.pap]);  // no block reads either in this launch
  }
  const T beta = (T)safe_div(rn, ro);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int64_t i = (blockIdx.x * (int64_t)PER + k) * kBlock + threadIdx.x;
    if (i < n2) {
      V2<T> o;
      o.x = fma(beta, pi[k].x, zi[k].x);
      o.y = fma(beta, pi[k].y, zi[k].y);
      st2(p_next, i, o);
    }
  }
}

template <typename T, int PER>
__global__ void __launch_bounds__(kBlock)
k_cg_x2p(int64_t n2, T* __restrict__ x, T* __restrict__ p0, const T* __restrict__ p1,
         const T* __restrict__ z, Parts rz, CgSlots c, bool last) {
  V2<T> q0[PER], q1[PER], xi[PER], zi[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int64_t i = (blockIdx.x * (int64_t)PER + k) * kBlock + threadIdx.x;
    if (i < n2) {
      q0[k] = ld2(p0, i);
      q1[k] = ld2(p1, i);
      xi[k] = ld2(x, i);
      if (!last) zi[k] = ld2(z, i);
    }
  }
  const double ro = c.scal[c.rz_old];
  const T a0 = (T)c.scal[c.asave];
  const T a1 = (T)safe_div(ro, c.scal[c.pap]);
  T beta = (T)0;
  if (!last) {
    const double rn = total(rz);
    if (blockIdx.x == 0 && threadIdx.x == 0) c.scal[c.rz_new] = rn;
    beta = (T)safe_div(rn, ro);
  }
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int64_t i = (blockIdx.x * (int64_t)PER + k) * kBlock + threadIdx.x;
    if (i < n2) {
      V2<T> o;
      o.x = fma(a1, q1[k].x, fma(a0, q0[k].x, xi[k].x));
      o.y = fma(a1, q1[k].y, fma(a0, q0[k].y, xi[k].y));
      st2(x, i, o);
      if (!last) {
        o.x = fma(beta, q1[k].x, zi[k].x);
        o.y = fma(beta, q1[k].y, zi[k].y);
        st2(p0, i, o);
      }
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(kBlock)
k_cg_x(int64_t n2, T* __restrict__ x, const T* __restrict__ p, CgSlots c) {
  const int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x;
  if (i >= n2) return;
  const T a = (T)safe_div(c.scal[c.rz_old], c.scal[c.pap]);
  const V2<T> pi = ld2(p, i);
  V2<T> xi = ld2(x, i);
  xi.x = fma(a, pi.x, xi.x);
  xi.y = fma(a, pi.y, xi.y);
  st2(x, i, xi);
}

// The gathers (both vectors, metric, words) are issued before the partials of r.z are added; the
// neighbours' directions are formed as beta arrives. p_next may hold the direction before p: its
// entries are read by the thread that writes them.
template <int DIM, typename T, bool VAR, bool KAOS, bool VCM>
__global__ void __launch_bounds__(256)
k_p1_direction(int64_t E, int64_t stride, const T* __restrict__ z, const T* __restrict__ p, T* p_next,
               T* __restrict__ Ap, T* __restrict__ x, bool x2, const double* __restrict__ Kt,
               const double* __restrict__ tauS, const int* __restrict__ nbr,
               const int* __restrict__ bctype, const T* __restrict__ kfac, const int* __restrict__ tab,
               Parts rz, CgSlots c, double* __restrict__ partial, P1NodeBits bits) {
  constexpr OpLayout L = op_layout(DIM, 1);
  constexpr int Np = L.Np, Nf = L.Nf;
  const int64_t e = xcd_block() * blockDim.x + threadIdx.x;
  const bool live = e < E;
  P1Loads<DIM, T> P;
  T po[Np], pn[Nf][Np], pp[Np], xx[Np];
  if (live) {
    p1_load<DIM, T, VAR, true, BitNodes, KAOS, VCM>(e, stride, z, Kt, tauS, nbr, nullptr, bctype, kfac,
                                                    as_const(tab), BitNodes{bits}, P);
    p1_values<Np, VCM>(p, stride, e, po);
#pragma unroll
    for (int f = 0; f < Nf; ++f) p1_values<Np, VCM>(p, stride, P.at(f, e), pn[f]);
    if (x2) {
      p1_values<Np, VCM>((const T*)p_next, stride, e, pp);
      p1_values<Np, VCM>((const T*)x, stride, e, xx);
    }
  }
  const double ro = c.scal[c.rz_old], pa = c.scal[c.pap];
  const double a0 = x2 ? c.scal[c.asave] : 0.0;
  const double rn = total(rz);
  const double a1 = safe_div(ro, pa);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    c.scal[c.rz_new] = rn;  // no block reads it in this launch
    if (!x2) c.scal[c.asave] = a1;
  }
  double dotv = 0.0;
  if (live) {
    const T beta = (T)safe_div(rn, ro);
    if (x2) {
#pragma unroll
      for (int i = 0; i < Np; ++i) xx[i] = fma((T)a1, po[i], fma((T)a0, pp[i], xx[i]));
      p1_store<Np, VCM>(x, stride, e, xx);
    }
#pragma unroll
    for (int i = 0; i < Np; ++i) P.uu[i] = fma(beta, po[i], P.uu[i]);
#pragma unroll
    for (int f = 0; f < Nf; ++f)
#pragma unroll
      for (int i = 0; i < Np; ++i) P.un[f][i] = fma(beta, pn[f][i], P.un[f][i]);
    p1_store<Np, VCM>(p_next, stride, e, P.uu);
    T acc[Np];
    dotv = p1_compute<DIM, T, VAR>(e, stride, P, NoSlip{}, acc);
    p1_store<Np, VCM>(Ap, stride, e, acc);
  }
  put_partial(dotv, partial);
}

int blocks(int64_t n2, int per) { return (int)cg_blocks(n2, per); }

}  // namespace

#define INSP_PER(n2, CALL)                       \
  do {                                           \
    switch (cg_pairs(n2)) {                      \
      case 1: { constexpr int P_ = 1; CALL; } break; \
      case 2: { constexpr int P_ = 2; CALL; } break; \
      default: { constexpr int P_ = 4; CALL; }   \
    }                                            \
  } while (0)

template <typename T>
int cg_init(int64_t n, const T* b, const T* inv, T* x, T* z, T* p, double* partial, hipStream_t s) {
  const int64_t n2 = n / 2;
  const int nb = blocks(n2, cg_pairs(n2));
  INSP_PER(n2, hipLaunchKernelGGL((k_cg_init<T, P_>), dim3(nb), dim3(kBlock), 0, s, n2, b, inv, x, z, p, partial));
  check("k_cg_init");
  return nb;
}

template <typename T>
int cg_update_z(int64_t n, T* z, const T* Ap, const T* inv, Parts pap, const CgSlots& c, double* partial,
                hipStream_t s) {
  const int64_t n2 = n / 2;
  const int nb = blocks(n2, cg_pairs(n2));
  INSP_PER(n2, hipLaunchKernelGGL((k_cg_z<T, P_>), dim3(nb), dim3(kBlock), 0, s, n2, z, Ap, inv, pap, c, partial));
  check("k_cg_z");
  return nb;
}

template <typename T>
void cg_update_p(int64_t n, T* p_next, const T* p, const T* z, Parts rz, const CgSlots& c, hipStream_t s) {
  const int64_t n2 = n / 2;
  const int nb = blocks(n2, cg_pairs(n2));
  INSP_PER(n2, hipLaunchKernelGGL((k_cg_p<T, P_>), dim3(nb), dim3(kBlock), 0, s, n2, p_next, p, z, rz, c));
  check("k_cg_p");
}

template <typename T>
void cg_update_x2p(int64_t n, T* x, T* p0, const T* p1, const T* z, Parts rz, const CgSlots& c, bool last,
                   hipStream_t s) {
  const int64_t n2 = n / 2;
  const int nb = blocks(n2, cg_pairs(n2));
  INSP_PER(n2, hipLaunchKernelGGL((k_cg_x2p<T, P_>), dim3(nb), dim3(kBlock), 0, s, n2, x, p0, p1, z, rz, c, last));
  check("k_cg_x2p");
}

template <typename T>
void cg_update_x(int64_t n, T* x, const T* p, const CgSlots& c, hipStream_t s) {
  const int64_t n2 = n / 2;
  hipLaunchKernelGGL((k_cg_x<T>), dim3(blocks(n2, 1)), dim3(kBlock), 0, s, n2, x, p, c);
  check("k_cg_x");
}

// With more cells the gathers of two vectors per neighbour lose. us per coarse iteration, update and apply /
// direction pass, FP64, k = 1: 2D 1,800 cells 11.4 / 9.4, 65k 12.9 / 10.5; 3D 3k 12.2 / 10.5, 64k 14.4 /
// 12.8, 132k 21.0 / 22.4, 547k 58.5 / 68.9 (two thirds of the apply's waves fit beside the second set of
// neighbour values). The other forms cross later. Per two iterations (FP32: one), 3D 93,750 cells:
// FP64 32.0 / 30.0, with a coefficient 34.0 / 32.4, FP32 13.6 / 11.5, with a coefficient 14.7 / 12.5; 162,000:
// 41.6 / 43.1, 46.4 / 45.9, 16.3 / 14.8, 17.0 / 18.1; 2D 260,642: 40.7 / 38.8, 44.7 / 43.4, 16.2 / 15.0, 16.7 / 15.6.
bool p1_direction_pays(const MeshView& m) {
  return m.nbc && m.E <= (m.dim == 2 ? int64_t(1) << 18 : (int64_t(1) << 16) + (int64_t(1) << 15));
}

template <typename T>
void launch_p1_direction(const MeshView& m, const LevelView& l, bool cells, const T* z, const T* p,
                         T* p_next, T* Ap, T* x, bool x2, const T* kfac, Parts rz, const CgSlots& c,
                         double* partial, hipStream_t s) {
  if (l.N != 1 || !m.nbc || (cells && (m.dim != 3 || !m.Ka || !m.nbc_cells || !l.tau_cells)))
    throw std::invalid_argument("order-1 direction pass: order 1, packed words");
  if (p == p_next || z == p_next) throw std::invalid_argument("order-1 direction pass: p_next must be apart");
  if (m.E == 0) return;
  const P1NodeBits& bits = p1_node_bits(m.dim);
  const dim3 grid((unsigned)apply_blocks(m.E));
#define INSP_DIR(D, V, A, C_)                                                                            \
  hipLaunchKernelGGL((k_p1_direction<D, T, V, A, C_>), grid, dim3(256), 0, s, m.E, m.stride, z, p, p_next, \
                     Ap, x, x2, A ? m.Ka : m.Kt, C_ ? l.tau_cells : l.tauS, C_ ? m.nbc_cells : m.nbc,     \
                     m.bctype, kfac, l.tab, rz, c, partial, bits)
  if (m.dim == 2) { if (kfac) INSP_DIR(2, true, false, false); else INSP_DIR(2, false, false, false); }
  else if (cells) { if (kfac) INSP_DIR(3, true, true, true); else INSP_DIR(3, false, true, true); }
  else { if (kfac) INSP_DIR(3, true, false, false); else INSP_DIR(3, false, false, false); }
#undef INSP_DIR
  check("k_p1_direction");
}

#define INSP_INST(T)                                                                                      \
  template int cg_init<T>(int64_t, const T*, const T*, T*, T*, T*, double*, hipStream_t);                 \
  template int cg_update_z<T>(int64_t, T*, const T*, const T*, Parts, const CgSlots&, double*, hipStream_t); \
  template void cg_update_p<T>(int64_t, T*, const T*, const T*, Parts, const CgSlots&, hipStream_t);      \
  template void cg_update_x2p<T>(int64_t, T*, T*, const T*, const T*, Parts, const CgSlots&, bool,        \
                                 hipStream_t);                                                            \
  template void cg_update_x<T>(int64_t, T*, const T*, const CgSlots&, hipStream_t);                       \
  template void launch_p1_direction<T>(const MeshView&, const LevelView&, bool, const T*, const T*, T*,   \
                                       T*, T*, bool, const T*, Parts, const CgSlots&, double*, hipStream_t);
INSP_INST(double)
INSP_INST(float)

}  // namespace insp
