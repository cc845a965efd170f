// Counts of the partial sums against the room kept for them (partials.h), for every order of the finest
// and of the coarsest level and meshes of 10^2 to 10^7 cells.
#include "partials.h"

#include <cstdio>

int main() {
  using namespace insp;
  int bad = 0;
  for (int dim = 2; dim <= 3; ++dim)
    for (int N = 1; N <= 4; ++N)
      for (double e = 1e2; e < 1.01e7; e *= 1.02) {
        const int64_t E = (int64_t)e | 1;
        int64_t stride = (E + 63) / 64 * 64;
        if ((stride / 64) % 2 == 0) stride += 64;
        auto nodes = [&](int k) { return dim == 2 ? (k + 1) * (k + 2) / 2 : (k + 1) * (k + 2) * (k + 3) / 6; };
        const int64_t half = partials_half(E, nodes(N) * stride);
        auto fits = [&](const char* what, int64_t count) {
          if (count <= half) return;
          if (bad++ < 20) std::printf("%s: dim %d order %d, %lld cells: %lld partials, room %lld\n", what, dim, N,
                                      (long long)E, (long long)count, (long long)half);
        };
        for (int c = 1; c <= N; ++c) fits("coarse CG stream", cg_stream_blocks(nodes(c) * stride));
        fits("element pass, one thread per cell", one_thread_blocks(E));
        fits("element pass, four waves", four_wave_blocks(E));
        fits("inverse-mass step", 3 * one_thread_blocks(E));
        fits("vector kernels", 4 * kRedBlocks);
      }
  std::printf(bad ? "%d counts do not fit\n" : "ok\n", bad);
  return bad != 0;
}
