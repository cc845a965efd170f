// State of a run of the fused conjugate gradients (pcg_kernels.h) and what its launches read and write of
// it. Plain functions, so that the order of the accesses can be checked on the CPU.
#pragma once

#include <cmath>

#if defined(__HIPCC__)
#define INSP_HD __host__ __device__ __forceinline__
#else
#define INSP_HD inline
#endif

namespace insp {

// r.z and the stop of this and of the next iteration (each pair trades places), p.Ap and |r|^2 of the last
// one, the iterations done, and sums added by a kernel of their own.
enum PcgSlot { P_RZ0 = 0, P_RZ1 = 1, P_PAP = 2, P_RR = 3, P_IT = 4, P_STOP0 = 5, P_STOP1 = 6, P_SUM = 8, P_COUNT = 12 };
enum PcgStop { PCG_RUNNING = 0, PCG_TOL = 1, PCG_BREAKDOWN = 2 };

// Slots of one iteration. Every wave of its launches reads rz and stop, which none of them writes: a wave
// that started late sees what the first one saw. The direction pass writes rz_next and stop_next.
struct PcgTurn {
  int rz, rz_next, stop, stop_next;
};
inline PcgTurn pcg_turn(int k) {
  const int a = k % 2, b = 1 - a;
  return PcgTurn{P_RZ0 + a, P_RZ0 + b, P_STOP0 + a, P_STOP0 + b};
}

INSP_HD bool pcg_running(const double* st, const PcgTurn& t) { return st[t.stop] == (double)PCG_RUNNING; }

// What |r|^2 and p.Ap of an iteration decide.
INSP_HD PcgStop pcg_decide(double rr, double pap, double tol) {
  if (!(pap > 0.0) || !std::isfinite(rr) || !std::isfinite(pap)) return PCG_BREAKDOWN;
  return std::sqrt(rr) <= tol ? PCG_TOL : PCG_RUNNING;
}

// The end of a running iteration, written by one thread, and of one after the stop.
INSP_HD void pcg_record(double* st, const PcgTurn& t, double rr, double rz, PcgStop why) {
  st[P_IT] += 1.0;
  st[P_RR] = rr;
  st[t.rz_next] = rz;
  st[t.stop_next] = (double)why;
}
INSP_HD void pcg_keep_stop(double* st, const PcgTurn& t) { st[t.stop_next] = st[t.stop]; }

// Why the run stopped, from the state after any number of iterations.
inline PcgStop pcg_stopped(const double* st) {
  return (PcgStop)(int)(st[P_STOP0] != (double)PCG_RUNNING ? st[P_STOP0] : st[P_STOP1]);
}

// Launching iterations ahead of the host's look at the state: how many to a look after `done` of them, and how
// many looks may be open. What is launched past the end runs its applies in vain, so it may only be a
// part of what the run has needed: none up to three iterations, then at most a quarter of them and two.
// A look costs about 20 us to wake the host and refill the queue where nothing runs meanwhile.
// 3D order 2, 93,750 cells, inverse mass, us per solve, a look after each iteration of unfused passes / sixteen
// ahead from the start / this: 1 iteration 279 / 783 / 235, 5 683 / 847 / 518, 10 1177 / 1224 / 839, 96
// 9588 / 5619 / 5545.
inline int pcg_batch(int done) { return done < 56 ? 1 + done / 8 : 8; }
inline int pcg_looks(int done) { return done < 4 ? 1 : 2; }

}  // namespace insp
