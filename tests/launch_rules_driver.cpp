// Host driver for tests/test_launch_rules.py: the launch rules of
// fhe-mamba_amd/csrc/launch_rules.hpp on lines of
//   mid S1 TILES NSRC NDST LDS   -> waves, LDS bytes of 4, 8, 16 waves
//   digits ND LIMBS N COUNT 0    -> 1 if finished inside ModDown
//   rescale S1 TILES L 0 0       -> 1 if by the column kernel, its waves
#include <cstdio>
#include <cstring>

#include "launch_rules.hpp"

int main() {
  char op[16];
  unsigned a, b, c, d, e;
  while (scanf("%15s %u %u %u %u %u", op, &a, &b, &c, &d, &e) == 6) {
    if (!strcmp(op, "mid"))
      printf("%u %u %u %u\n", fhe::mid_waves(a, b, c, d, e), fhe::mid_lds_bytes(a, c, d, 4),
             fhe::mid_lds_bytes(a, c, d, 8), fhe::mid_lds_bytes(a, c, d, 16));
    else if (!strcmp(op, "digits"))
      printf("%d\n", (int)fhe::finish_digits_in_moddown(a, b, c, d));
    else if (!strcmp(op, "rescale"))
      printf("%d %u\n", (int)fhe::rescale_by_columns(a, b, c), fhe::rescale_waves(a, b, c));
    else
      return 2;
  }
  return 0;
}
