// Which memory the passes take in place (caller_memory.h).
#include "caller_memory.h"

#include <cstdio>

using namespace insp;

int main() {
  int bad = 0;
  auto expect = [&](bool got, bool want, const char* what) {
    if (got != want) ++bad, std::printf("%s\n", what);
  };
  CallerMemory m;
  m.device = true;
  m.gpu = 1;
  m.base = 4096;
  m.size = 800;
  expect(in_place(m, 1, 4096, 800), true, "a whole allocation");
  expect(in_place(m, 1, 4104, 792), true, "its end");
  expect(in_place(m, 1, 4096, 801), false, "one byte past its end");
  expect(in_place(m, 1, 4104, 800), false, "a shifted vector past its end");
  expect(in_place(m, 1, 4096 + 808, 8), false, "a vector behind it");
  expect(in_place(m, 1, 4088, 8), false, "a vector before it");
  expect(in_place(m, 1, 4096, ~(size_t)0), false, "a length that overflows");
  expect(in_place(m, 0, 4096, 800), false, "another GPU's memory");
  m.device = false;
  expect(in_place(m, 1, 4096, 800), false, "host memory");
  expect(in_place(CallerMemory{}, 0, 4096, 8), false, "unknown memory");
  std::printf(bad ? "%d failures\n" : "ok\n", bad);
  return bad != 0;
}
