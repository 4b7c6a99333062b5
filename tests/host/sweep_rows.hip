// Strips of the deep TV's passes (strip_rows / strips_across in sweep.h), on the
// CPU: for every "H W T n" on the command line one line with the rows of a strip
// and the strips of a frame in each pass, for a device of 1024 SIMDs.
#include <cstdio>
#include <cstdlib>

#include "sweep.h"

int main(int argc, char** argv) {
  using namespace scigap::sweep;
  for (int i = 1; i + 3 < argc; i += 4) {
    const int H = std::atoi(argv[i]), W = std::atoi(argv[i + 1]), T = std::atoi(argv[i + 2]);
    const int updates = std::atoi(argv[i + 3]) - 1;
    const int passes = (updates + kMaxPass - 1) / kMaxPass, low = updates / passes;
    const int R = strip_rows(H, W, T, low, 1024);
    std::printf("%d", R);
    for (int c = 0; c < passes; ++c)
      std::printf(" %d", strips_across(W, low + (c < updates % passes ? 1 : 0)) * ((H + R - 1) / R));
    std::printf("\n");
  }
  std::printf("inline %d\n", kInlineStrips);
  return 0;
}
