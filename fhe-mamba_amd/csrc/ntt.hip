// The plain transforms over poly sets, digit buffers and pointer tables, in
// two passes of ntt_body.hpp (one for N <= 2^12).
#include "ntt_body.hpp"

namespace fhe {
namespace {

// Input of a forward transform as signed 64-bit coefficients [npoly][N]: |x|
// mod q from the quotient estimate mulhi(|x|, floor(2^64 / q)), at most one
// low, so below 2q, and its complement in 2q for negative x.  The lifted
// residues are never in memory: 16 plaintexts of 34 limbs at N=2^16 took a
// kernel of 112 us to write them and a first pass of 153, now 111 in all.
struct SignedLoad {
  static constexpr bool kLoad = true;
  const int64_t* coef;
  const ModConst* mc;
  uint32_t n, mod0;
  __device__ __forceinline__ uint64_t get(size_t g, uint64_t q) const {
    const int64_t x = coef[(size_t)blockIdx.y * n + g];
    const uint64_t a = x < 0 ? 0 - (uint64_t)x : (uint64_t)x;
    const uint64_t r = a - mulhi64(a, mc[mod0 + blockIdx.z].mu64) * q;
    return x < 0 ? 2 * q - r : r;
  }
};
// Input of an inverse transform of one poly, read from another buffer.
struct FromLoad {
  static constexpr bool kLoad = true;
  const uint64_t* src;
  uint32_t n;
  __device__ __forceinline__ uint64_t get(size_t g, uint64_t) const {
    return src[(size_t)blockIdx.z * n + g];
  }
};

template <int LIM, int S, int KIND, bool INV, class Map, class Load>
__global__ void __launch_bounds__(max_threads<KIND>())
    ntt_pass(uint64_t* __restrict__ data, size_t poly_stride, const ModConst* __restrict__ mc,
             const uint64_t* __restrict__ tw_all, uint32_t log_n, Map map, uint32_t s_other,
             const Load load) {
  ntt_body<LIM, S, KIND, INV, KIND == SINGLE ? RHO_SINGLE : RHO_PLAIN, PlainStore, Load, Map>(
      data, poly_stride, mc, tw_all, log_n, map, s_other, PlainStore{}, load);
}

template <int S, int KIND, bool INV, class Map, class Load>
void launch_pass(Context& c, uint64_t* data, uint32_t npoly, size_t poly_stride, uint32_t nlimb,
                 Map map, uint32_t s_other, const Load& load) {
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
  auto go = [&](auto lim) {
    FHE_LAUNCH(c, PASS_NAME, (ntt_pass<decltype(lim)::value, S, KIND, INV, Map, Load>), grid,
               dim3(threads), 0, data, poly_stride, c.d_const, INV ? c.d_tw_inv : c.d_tw_fwd,
               c.log_n, map, s_other, load);
  };
  // rings below 2^10 (tests of tiny parameters) share the narrow range
  if constexpr (KIND == SINGLE && S < 10)
    go(std::integral_constant<int, 8>{});
  else
    with_lim(c, go);
}

template <bool INV, class Map = LimbMap, class Load = PlainLoad>
void launch_single(Context& c, uint64_t* data, uint32_t npoly, size_t ps, uint32_t nlimb, Map map,
                   const Load& load = Load{}) {
  switch (c.log_n) {
#define CASE(S) \
  case S: launch_pass<S, SINGLE, INV>(c, data, npoly, ps, nlimb, map, 0, load); break;
    CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11) CASE(12)
#undef CASE
    default: throw ArgError("unsupported ring dimension");
  }
}

template <bool INV, class Map = LimbMap, class Load = PlainLoad>
void launch_cols(Context& c, uint32_t s1, uint32_t s2, uint64_t* data, uint32_t npoly, size_t ps,
                 uint32_t nlimb, Map map, const Load& load = Load{}) {
  switch (s1) {
#define CASE(S) \
  case S: launch_pass<S, COLS, INV>(c, data, npoly, ps, nlimb, map, s2, load); break;
    CASE(7) CASE(8) CASE(9)
#undef CASE
    default: throw ArgError("unsupported column pass");
  }
}

template <bool INV, class Map = LimbMap, class Load = PlainLoad>
void launch_blocks(Context& c, uint32_t s1, uint32_t s2, uint64_t* data, uint32_t npoly, size_t ps,
                   uint32_t nlimb, Map map, const Load& load = Load{}) {
  switch (s2) {
#define CASE(S) \
  case S: launch_pass<S, BLOCKS, INV>(c, data, npoly, ps, nlimb, map, s1, load); break;
    CASE(6) CASE(7) CASE(8)
#undef CASE
    default: throw ArgError("unsupported block pass");
  }
}

template <class Map>
void forward_signed(Context& c, const int64_t* coef, uint64_t* data, uint32_t npoly, size_t ps,
                    uint32_t nlimb, Map map, uint32_t mod0) {
  if (npoly == 0 || nlimb == 0) return;
  if (npoly > 65535 || mod0 + nlimb > c.L + c.K)
    throw ArgError("too many polys or limbs in one launch");
  const SignedLoad load{coef, c.d_const, c.n, mod0};
  if (c.log_n <= 12) {
    launch_single<false>(c, data, npoly, ps, nlimb, map, load);
    return;
  }
  const uint32_t s1 = (c.log_n + 1) / 2, s2 = c.log_n / 2;
  launch_cols<false>(c, s1, s2, data, npoly, ps, nlimb, map, load);
  launch_blocks<false>(c, s1, s2, data, npoly, ps, nlimb, map);
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

void ntt_forward_signed(Context& c, const int64_t* coef, uint64_t* data, uint32_t npoly,
                        size_t poly_stride, uint32_t nlimb, uint32_t limb0) {
  forward_signed(c, coef, data, npoly, poly_stride, nlimb, LimbMap::contiguous(limb0), limb0);
}

void ntt_forward_signed_table(Context& c, const int64_t* coef, uint64_t* const* table,
                              uint32_t npoly, uint32_t nlimb) {
  forward_signed(c, coef, nullptr, npoly, 0, nlimb, TableMap{table}, 0);
}

void ntt_inverse_from(Context& c, const uint64_t* src, uint64_t* data, uint32_t nlimb) {
  if (nlimb == 0) return;
  if (nlimb > c.L + c.K) throw ArgError("too many limbs in one launch");
  const FromLoad load{src, c.n};
  const LimbMap map = LimbMap::contiguous(0);
  if (c.log_n <= 12) {
    launch_single<true>(c, data, 1, 0, nlimb, map, load);
    return;
  }
  const uint32_t s1 = (c.log_n + 1) / 2, s2 = c.log_n / 2;
  launch_blocks<true>(c, s1, s2, data, 1, 0, nlimb, map, load);
  launch_cols<true>(c, s1, s2, data, 1, 0, nlimb, map);
}

}  // namespace fhe
