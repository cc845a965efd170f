// The state of a fused conjugate gradient run (pcg_state.h) under the orders in which a launch's waves may
// come to it: a wave reads the state before and after the first block's thread has written it, and
// must see the same; a run of iterations with several launched after its end; and how many a run that ends
// after any number of iterations launches in vain.
#include "pcg_state.h"

#include <cstdio>
#include <initializer_list>
#include <limits>

using namespace insp;

static int bad = 0;
static void expect(bool ok, const char* what, int k) {
  if (ok) return;
  ++bad;
  std::printf("%s (iteration %d)\n", what, k);
}

int main() {
  const double nan = std::numeric_limits<double>::quiet_NaN(), inf = std::numeric_limits<double>::infinity();
  expect(pcg_decide(4.0, 1.0, 1.0) == PCG_RUNNING && pcg_decide(1.0, 1.0, 1.0) == PCG_TOL, "tolerance", 0);
  expect(pcg_decide(0.0, 0.0, 1.0) == PCG_BREAKDOWN && pcg_decide(0.0, -1.0, 1.0) == PCG_BREAKDOWN, "p.Ap", 0);
  expect(pcg_decide(nan, 1.0, 1.0) == PCG_BREAKDOWN && pcg_decide(inf, 1.0, 1.0) == PCG_BREAKDOWN, "|r|^2", 0);
  expect(pcg_decide(1.0, nan, 1.0) == PCG_BREAKDOWN && pcg_decide(1.0, inf, 1.0) == PCG_BREAKDOWN, "p.Ap", 0);
  for (int end = 1; end <= 9; ++end)
    for (PcgStop why : {PCG_TOL, PCG_BREAKDOWN}) {
      double st[P_COUNT] = {};
      st[P_RZ0] = 100.0;
      for (int k = 0; k < end + 7; ++k) {
        const PcgTurn t = pcg_turn(k);
        // a wave of another block, before the first block has come to its end
        const bool run_early = pcg_running(st, t);
        const double rz_early = st[t.rz];
        if (run_early) pcg_record(st, t, 50.0 + k, 101.0 + k, k + 1 == end ? why : PCG_RUNNING);
        else pcg_keep_stop(st, t);
        // and one after
        expect(pcg_running(st, t) == run_early, "a late wave sees another stop", k);
        expect(st[t.rz] == rz_early, "a late wave sees another r.z", k);
        expect(run_early == (k < end), "stop", k);
        if (k < end) expect(rz_early == 100.0 + k, "r.z of the iteration", k);
        // what the host reads after this iteration
        expect(pcg_stopped(st) == (k + 1 < end ? PCG_RUNNING : why), "the host's stop", k);
        expect(st[P_IT] == (k + 1 < end ? k + 1 : end), "iterations done", k);
        expect(st[P_RR] == 50.0 + (k + 1 < end ? k : end - 1), "|r|^2 of the last one", k);
      }
    }
  for (int end = 1; end <= 2000; ++end) {
    int done = 0, seen = 0, open[2] = {0, 0}, out = 0;  // iterations launched, looked at, and in each open look
    while (seen < end) {
      if (out < pcg_looks(done)) {
        expect(out < 2, "open looks", end);
        done += open[out++] = pcg_batch(done);
      } else {
        seen += open[0];
        open[0] = open[1];
        --out;
      }
    }
    expect(done - end <= (end <= 3 ? 0 : 2 + end / 4) && done - end <= 15, "launched in vain", end);
  }
  std::printf(bad ? "%d failures\n" : "ok\n", bad);
  return bad != 0;
}
