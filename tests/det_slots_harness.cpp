// Host build of slots_repeat (fdtdx_amd/csrc/kernels.h) for the CPU tests: for window and the entries of
// time_to_idx given as arguments, prints 1 when two steps less than `window` apart share a slot, else 0.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../fdtdx_amd/csrc/kernels.h"

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  std::vector<int32_t> tti;
  for (int a = 2; a < argc; ++a) tti.push_back(atoi(argv[a]));
  printf("%d\n", (int)fdtdx::slots_repeat(tti.data(), (int)tti.size(), atoi(argv[1])));
  return 0;
}
