// Host driver for the rule that sends a grouped GEMM to the few-rows kernels
// (few_rows_rule.h): reads "kind rows copies N K cus" lines and prints the tile
// height taken for each (0: the 256-row kernels).  Built and run by
// tests/test_few_rows_rule.py with the host compiler.
#include <cstdio>

#include "few_rows_rule.h"

int main() {
  int kind;
  long long rows, copies, N, K, cus;
  while (std::scanf("%d %lld %lld %lld %lld %lld", &kind, &rows, &copies, &N, &K, &cus) == 6)
    std::printf("%d\n", pmx::few_rows_tiling(kind, rows, copies, N, K, cus));
  return 0;
}
