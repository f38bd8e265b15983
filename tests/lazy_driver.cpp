// Host driver for tests/test_lazy_butterflies.py: the NTT butterflies of
// fhe-mamba_amd/csrc/modarith.hpp on records of little-endian uint64.
//   lazy_driver fwd LIM RED   q x y w      -> x' y'
//   lazy_driver inv LIM BX BY q x y w      -> x' y' bx' by'
//   lazy_driver schedule LIM B S           -> S (bound, reduces) pairs, then
//                                             the output bound (text)
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "modarith.hpp"

using namespace fhe;

int main(int argc, char** argv) {
  if (argc < 4) return 2;
  const int lim = atoi(argv[2]);
  if (!strcmp(argv[1], "schedule")) {
    const int b = atoi(argv[3]), S = atoi(argv[4]);
    for (int beta = S - 1; beta >= 0; --beta)
      printf("%d %d\n", fwd_bound(lim, b, S, beta), (int)fwd_reduces(lim, b, S, beta));
    printf("%d 0\n", fwd_bound(lim, b, S, -1));
    return 0;
  }
  uint64_t r[4];
  while (fread(r, 8, 4, stdin) == 4) {
    const uint64_t q = r[0], w = r[3], wp = host_shoup(w, q);
    const LazyMod m{4 * q, 8 * q, 0 - q, 0 - (uint64_t)(lim / 2) * q, 1};
    uint64_t out[4] = {r[1], r[2], 0, 0};
    if (!strcmp(argv[1], "fwd")) {
      fwd_butterfly(out[0], out[1], w, wp, m, atoi(argv[3]) != 0);
    } else {
      int bx = atoi(argv[3]), by = atoi(argv[4]);
      inv_butterfly(out[0], out[1], w, wp, m, lim, bx, by);
      out[2] = bx;
      out[3] = by;
    }
    fwrite(out, 8, 4, stdout);
  }
  return 0;
}
