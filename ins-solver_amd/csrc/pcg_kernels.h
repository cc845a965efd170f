// Preconditioned CG iterations of the Jacobi and inverse-mass solvers, FP64 (the flexible form,
// beta = r.(z - z_old) / (r.z)_old: cg_compute_beta_pre_flex.h, viscous_solver.cpp:158-266): one pass
// updates x and r, preconditions and leaves the three sums of the step, one forms the next direction
// and decides whether to stop. After the stop both leave everything as it is, so iterations may be
// launched ahead of the host's look at the state.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <string>

#include "cg_kernels.h"
#include "pcg_state.h"
#include "vec_kernels.h"

namespace insp {

void pcg_start(double* st, hipStream_t s);  // running, no iterations done
// x += a p, r -= a Ap, z = inv r with a = r.z / p.Ap; partials of |r|^2, r.z and r.(z - z_old), as many
// as it returns of each, one after the other.
int pcg_update_jacobi(int64_t n, double* x, double* r, double* z, const double* p, const double* Ap,
                      const double* inv, Parts pap, double* st, const PcgTurn& t, double* partial, hipStream_t s);
// The same with z = scale (J M)^-1 r, or ((J M)^-1 r)_i / recp_i, on ncomp vectors cs apart.
int pcg_update_inv_mass(int np, int ncomp, int64_t E, int64_t stride, int64_t cs, double* x, double* r,
                        double* z, const double* p, const double* Ap, const double* J, const double* Minv,
                        double scale, const double* recp, Parts pap, double* st, const PcgTurn& t, double* partial,
                        hipStream_t s);
// Counts the iteration and stops it at |r| <= tol or on a breakdown, else p = z + beta p, from the nb
// partials of each of the step's sums.
void pcg_direction(int64_t n, double* p, const double* z, int nb, const double* partial, double* st,
                   const PcgTurn& t, double tol, hipStream_t s);

// Entries up to which iterations are launched ahead: up to about 100 us each (2D order 3, 2048 cells: 20 us).
constexpr int64_t kAheadEntries = int64_t(1) << 20;

struct PcgEnd {
  int iterations = 0, stop = PCG_RUNNING;
  double rr = 0;
};

// Launches iterations (step(k)) until one stops the run or `limit` are done: on short iterations (`ahead`)
// several to a look at the state and the next ones before it (pcg_batch, pcg_looks), otherwise one by
// one, each with its look.
template <class Step>
PcgEnd pcg_drive(int limit, bool ahead, const double* st, double* host, hipEvent_t (&ev)[2], hipStream_t s,
                 Step&& step) {
  auto ok = [](hipError_t e) {
    if (e != hipSuccess) throw std::runtime_error(std::string("conjugate gradients: ") + hipGetErrorString(e));
  };
  PcgEnd end;
  int done = 0, out = 0, head = 0, tail = 0;
  for (;;) {
    if (done < limit && out < (ahead ? pcg_looks(done) : 1)) {
      const int m = std::min(ahead ? pcg_batch(done) : 1, limit - done);
      for (int k = 0; k < m; ++k) step(done + k);
      done += m;
      ok(hipMemcpyAsync(host + tail * P_COUNT, st, P_COUNT * sizeof(double), hipMemcpyDeviceToHost, s));
      ok(hipEventRecord(ev[tail], s));
      tail ^= 1;
      ++out;
      continue;
    }
    if (out == 0) return end;
    ok(hipEventSynchronize(ev[head]));
    const double* h = host + head * P_COUNT;
    end.iterations = (int)h[P_IT];
    end.stop = pcg_stopped(h);
    end.rr = h[P_RR];
    head ^= 1;
    --out;
    if (end.stop != PCG_RUNNING) return end;
  }
}

}  // namespace insp
