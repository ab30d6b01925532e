// Prints the large-M launch choices of csrc/mm_choice.hpp, compiled and run by tests/test_mm_choice.py: for argv
// cfg, ntiles, k steps, compute units, one line "first last id splits" per run of rows (33 .. 8192) with one choice.
#include <cstdio>
#include <cstdlib>

#include "mm_choice.hpp"

using namespace fdllm;

int main(int argc, char** argv) {
  if (argc != 5) return 1;
  const int cfg = atoi(argv[1]), ntiles = atoi(argv[2]), ks = atoi(argv[3]);
  MmPolicy pol;
  pol.cus = atoi(argv[4]);
  int first = 33, id0 = -1, split0 = 0;
  for (int M = 33; M <= 8193; ++M) {
    int id = -1, split = 0;
    if (M <= 8192) {
      id = mm_choice(cfg, M, ntiles, ks, pol);
      const MmInfo b = mm_info(id);
      split = ks % b.kss ? 0 : mm_split(cfg, id, M, ntiles, ks / b.kss, pol);  // 0: the streaming kernel
    }
    if (id != id0 || split != split0) {
      if (id0 >= 0) std::printf("%d %d %d %d\n", first, M - 1, id0, split0);
      first = M;
      id0 = id;
      split0 = split;
    }
  }
  return 0;
}
