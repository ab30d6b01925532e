// Prints the prefill attention's form (csrc/prefill_form.hpp), compiled and run by tests/test_prefill_form.py: argv
// rows, query heads, kv heads, compute units, FDLLM_PREFILL_PAIR, FDLLM_PREFILL_HPW -> "whole paired".
#include <cstdio>
#include <cstdlib>

#include "prefill_form.hpp"

int main(int argc, char** argv) {
  if (argc != 7) return 1;
  const fdllm::PrefillForm f =
      fdllm::prefill_form(atoi(argv[1]), atoi(argv[2]), atoi(argv[3]), atoi(argv[4]), atoi(argv[5]), atoi(argv[6]));
  std::printf("%d %d\n", f.whole, f.paired);
  return 0;
}
