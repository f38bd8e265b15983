// The plain transforms over poly sets, digit buffers and pointer tables, in
// two passes of ntt_body.hpp (one for N <= 2^12).
#include "ntt_body.hpp"

namespace fhe {
namespace {

template <int LIM, int S, int KIND, bool INV, class Map>
__global__ void __launch_bounds__(max_threads<KIND>())
    ntt_pass(uint64_t* __restrict__ data, size_t poly_stride, const ModConst* __restrict__ mc,
             const uint64_t* __restrict__ tw_all, uint32_t log_n, Map map, uint32_t s_other) {
  ntt_body<LIM, S, KIND, INV, KIND == SINGLE ? RHO_SINGLE : RHO_PLAIN, PlainStore, PlainLoad, Map>(
      data, poly_stride, mc, tw_all, log_n, map, s_other, PlainStore{});
}

template <int S, int KIND, bool INV, class Map>
void launch_pass(Context& c, uint64_t* data, uint32_t npoly, size_t poly_stride, uint32_t nlimb,
                 Map map, uint32_t s_other) {
  using G = Geo<S, KIND == SINGLE ? RHO_SINGLE : RHO_PLAIN>;
  const uint32_t lines = KIND == SINGLE ? 1 : 256 / G::TPL;
  const uint32_t threads = KIND == SINGLE ? G::TPL : 256;
  // COLS has N2 = 2^s_other lines per limb, BLOCKS has N1 = 2^s_other.
  const uint32_t tiles = KIND == SINGLE ? 1 : (1u << s_other) / lines;
  dim3 grid(tiles, npoly, nlimb);
  const char* const PASS_NAME =
      KIND == SINGLE ? (INV ? "ntt_inv_single" : "ntt_fwd_single")
      : KIND == COLS ? (INV ? "ntt_inv_cols" : "ntt_fwd_cols")
                     : (INV ? "ntt_inv_blocks" : "ntt_fwd_blocks");
  with_lim(c, [&](auto lim) {
    FHE_LAUNCH(c, PASS_NAME, (ntt_pass<decltype(lim)::value, S, KIND, INV, Map>), grid,
               dim3(threads), 0, data, poly_stride, c.d_const, INV ? c.d_tw_inv : c.d_tw_fwd,
               c.log_n, map, s_other);
  });
}

template <bool INV, class Map = LimbMap>
void launch_single(Context& c, uint64_t* data, uint32_t npoly, size_t ps, uint32_t nlimb, Map map) {
  switch (c.log_n) {
#define CASE(S) \
  case S: launch_pass<S, SINGLE, INV>(c, data, npoly, ps, nlimb, map, 0); break;
    CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11) CASE(12)
#undef CASE
    default: throw ArgError("unsupported ring dimension");
  }
}

template <bool INV, class Map = LimbMap>
void launch_cols(Context& c, uint32_t s1, uint32_t s2, uint64_t* data, uint32_t npoly, size_t ps,
                 uint32_t nlimb, Map map) {
  switch (s1) {
#define CASE(S) \
  case S: launch_pass<S, COLS, INV>(c, data, npoly, ps, nlimb, map, s2); break;
    CASE(7) CASE(8) CASE(9)
#undef CASE
    default: throw ArgError("unsupported column pass");
  }
}

template <bool INV, class Map = LimbMap>
void launch_blocks(Context& c, uint32_t s1, uint32_t s2, uint64_t* data, uint32_t npoly, size_t ps,
                   uint32_t nlimb, Map map) {
  switch (s2) {
#define CASE(S) \
  case S: launch_pass<S, BLOCKS, INV>(c, data, npoly, ps, nlimb, map, s1); break;
    CASE(6) CASE(7) CASE(8)
#undef CASE
    default: throw ArgError("unsupported block pass");
  }
}

}  // namespace

void ntt_forward_digits(Context& c, uint64_t* digits, uint32_t count, uint32_t nd,
                        uint32_t nq) {
  if (count == 0 || nd == 0 || nq == 0) return;
  if (nq > c.L) throw ArgError("ModUp level out of range");
  if ((uint64_t)count * nd > 65535) throw ArgError("too many digits in one launch");
  const uint32_t ne = nq + c.K;
  // The last digit is the narrowest and so has the most converted limbs.
  const uint32_t w_last = nq - (nd - 1) * c.alpha;
  const uint32_t slots = ne - w_last;
  const DigitMap map{c.alpha, nq, c.L, ne, nd};
  const size_t ps = (size_t)ne * c.n;
  const uint32_t npoly = count * nd;
  if (c.log_n <= 12) {
    launch_single<false>(c, digits, npoly, ps, slots, map);
    return;
  }
  const uint32_t s1 = (c.log_n + 1) / 2, s2 = c.log_n / 2;
  launch_cols<false>(c, s1, s2, digits, npoly, ps, slots, map);
  launch_blocks<false>(c, s1, s2, digits, npoly, ps, slots, map);
}

void ntt_cols(Context& c, uint64_t* data, uint32_t npoly, size_t poly_stride, uint32_t nlimb,
              LimbMap map, bool inverse) {
  const uint32_t s1 = (c.log_n + 1) / 2, s2 = c.log_n / 2;
  if (inverse)
    launch_cols<true>(c, s1, s2, data, npoly, poly_stride, nlimb, map);
  else
    launch_cols<false>(c, s1, s2, data, npoly, poly_stride, nlimb, map);
}

void ntt_forward(Context& c, uint64_t* data, uint32_t npoly, size_t poly_stride, uint32_t nlimb,
                 LimbMap map) {
  if (npoly == 0 || nlimb == 0) return;
  if (npoly > 65535 || nlimb > 65535) throw ArgError("too many polys or limbs in one launch");
  if (c.log_n <= 12) {
    launch_single<false>(c, data, npoly, poly_stride, nlimb, map);
    return;
  }
  const uint32_t s1 = (c.log_n + 1) / 2, s2 = c.log_n / 2;
  launch_cols<false>(c, s1, s2, data, npoly, poly_stride, nlimb, map);
  launch_blocks<false>(c, s1, s2, data, npoly, poly_stride, nlimb, map);
}

void ntt_forward_table(Context& c, uint64_t* const* table, uint32_t npoly, uint32_t nlimb) {
  if (npoly == 0 || nlimb == 0) return;
  if (npoly > 65535 || nlimb > c.L + c.K) throw ArgError("too many polys or limbs in one launch");
  const TableMap map{table};
  if (c.log_n <= 12) {
    launch_single<false>(c, nullptr, npoly, 0, nlimb, map);
    return;
  }
  const uint32_t s1 = (c.log_n + 1) / 2, s2 = c.log_n / 2;
  launch_cols<false>(c, s1, s2, nullptr, npoly, 0, nlimb, map);
  launch_blocks<false>(c, s1, s2, nullptr, npoly, 0, nlimb, map);
}

void ntt_inverse(Context& c, uint64_t* data, uint32_t npoly, size_t poly_stride, uint32_t nlimb,
                 LimbMap map) {
  if (npoly == 0 || nlimb == 0) return;
  if (npoly > 65535 || nlimb > 65535) throw ArgError("too many polys or limbs in one launch");
  if (c.log_n <= 12) {
    launch_single<true>(c, data, npoly, poly_stride, nlimb, map);
    return;
  }
  const uint32_t s1 = (c.log_n + 1) / 2, s2 = c.log_n / 2;
  launch_blocks<true>(c, s1, s2, data, npoly, poly_stride, nlimb, map);
  launch_cols<true>(c, s1, s2, data, npoly, poly_stride, nlimb, map);
}

}  // namespace fhe
