// Rescale as four passes of ntt_body.hpp.
#include "rescale_parts.hpp"

namespace fhe {
namespace {

// ---- Rescale in four launches (ring dimensions 2^13 .. 2^17) ----
// The rescale's passes run radix 8 (RHO_EPILOGUE: eight lines of 2^S
// words, 17 KB of LDS and ~60 VGPRs per 256-lane workgroup), so one
// ciphertext's launch fits the chip in one round of workgroups.
// The inverse NTT of the last limb reads it from the input (LastLimbLoad);
// the forward column pass lifts it to modulus i as it loads (LiftLoad:
// x mod q_i, minus q_l mod q_i in the upper half, the centred lift); the
// last forward pass stores (a_i - t_i) * q_l^-1 (RescaleStore).
template <int LIM, int S>
__global__ void __launch_bounds__(256)
    ntt_pass_rescale_in(uint64_t* __restrict__ last, const ModConst* __restrict__ mc,
                        const uint64_t* __restrict__ tw_all, uint32_t log_n, uint32_t s_other,
                        const RescalePtrs ptrs, uint32_t npoly, size_t poly_words, uint32_t l) {
  ntt_body<LIM, S, BLOCKS, true, RHO_EPILOGUE, PlainStore, LastLimbLoad>(
      last, (size_t)1 << log_n, mc, tw_all, log_n, LimbMap::contiguous(l), s_other,
      PlainStore{}, LastLimbLoad{ptrs.a, npoly, poly_words, (size_t)l << log_n});
}

template <int LIM, int S>
__global__ void __launch_bounds__(256)
    ntt_pass_rescale_lift(uint64_t* __restrict__ t, size_t poly_stride,
                          const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                          uint32_t log_n, uint32_t s_other, const LiftLoad ld) {
  ntt_body<LIM, S, COLS, false, RHO_EPILOGUE, PlainStore, LiftLoad>(
      t, poly_stride, mc, tw_all, log_n, LimbMap::contiguous(0), s_other, PlainStore{}, ld);
}

template <int LIM, int S>
__global__ void __launch_bounds__(256)
    ntt_pass_rescale_out(uint64_t* __restrict__ t, size_t poly_stride,
                         const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                         uint32_t log_n, uint32_t s_other, const RescalePtrs ptrs,
                         const uint64_t* __restrict__ rs, uint32_t l, uint32_t L,
                         uint32_t npoly) {
  ntt_body<LIM, S, BLOCKS, false, RHO_EPILOGUE, RescaleStore>(
      t, poly_stride, mc, tw_all, log_n, LimbMap::contiguous(0), s_other,
      RescaleStore{ptrs.a, ptrs.out, rs, 1u << log_n, l, L, npoly});
}

// The rescale's inverse column pass over the last limb (radix 8, as the
// other rescale passes): launch poly y's single limb, modulus l.
template <int LIM, int S>
__global__ void __launch_bounds__(256)
    ntt_pass_rescale_cols(uint64_t* __restrict__ data, size_t poly_stride,
                          const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                          uint32_t log_n, uint32_t s_other, uint32_t l) {
  ntt_body<LIM, S, COLS, true, RHO_EPILOGUE, PlainStore, PlainLoad, LimbMap>(
      data, poly_stride, mc, tw_all, log_n, LimbMap::contiguous(l), s_other, PlainStore{});
}

}  // namespace

static void rescale_launch(Context& c, uint64_t* const* outs, const uint64_t* const* as,
                           uint32_t count, uint32_t npoly, uint32_t nq);

void rescale_fused(Context& c, uint64_t* out, const uint64_t* a, uint32_t npoly, uint32_t nq) {
  rescale_fused_many(c, &out, &a, 1, npoly, nq);
}

void rescale_fused_many(Context& c, uint64_t* const* outs, const uint64_t* const* as,
                        uint32_t count, uint32_t npoly, uint32_t nq) {
  if (c.log_n < 13 || c.log_n > 17) throw ArgError("fused rescale needs N = 2^13 .. 2^17");
  if (nq < 2 || npoly == 0 || npoly > 65535) throw ArgError("rescale: bad shape");
  for (uint32_t r0 = 0; r0 < count;) {
    const uint32_t b = rescale_batch(count - r0, npoly);
    rescale_launch(c, outs + r0, as + r0, b, npoly, nq);
    r0 += b;
  }
}

// One launch set over `count` <= RESCALE_MAX inputs of npoly polys each.
static void rescale_launch(Context& c, uint64_t* const* outs, const uint64_t* const* as,
                           uint32_t count, uint32_t npoly, uint32_t nq) {
  const uint32_t l = nq - 1, n = c.n, np = count * npoly;
  const uint32_t s1 = (c.log_n + 1) / 2, s2 = c.log_n / 2;
  RescalePtrs ptrs{};
  for (uint32_t r = 0; r < count; ++r) {
    ptrs.a[r] = as[r];
    ptrs.out[r] = outs[r];
  }
  Scratch last(c, (size_t)np * n), t(c, (size_t)np * l * n);
  const LiftLoad lift{last.p, c.d_const, c.d_rescale, n, l, c.L, c.mods[l] >> 1};
  switch (c.log_n) {
#define CASE(LN, A, B)                                                                        \
  case LN: {                                                                                  \
    using GB = Geo<B, RHO_EPILOGUE>;                                                          \
    using GA = Geo<A, RHO_EPILOGUE>;                                                          \
    const uint32_t tb = (1u << s1) / (256 / GB::TPL), ta = (1u << s2) / (256 / GA::TPL);      \
    with_lim(c, [&](auto lim) {                                                               \
      constexpr int LIM = decltype(lim)::value;                                               \
      FHE_LAUNCH(c, "ntt_inv_blocks_rescale", (ntt_pass_rescale_in<LIM, B>),                  \
                 dim3(tb, np, 1), dim3(256), 0, last.p, c.d_const, c.d_tw_inv, c.log_n, s1,   \
                 ptrs, npoly, (size_t)nq * n, l);                                             \
      FHE_LAUNCH(c, "ntt_inv_cols_rescale", (ntt_pass_rescale_cols<LIM, A>),                  \
                 dim3(ta, np, 1), dim3(256), 0, last.p, (size_t)n, c.d_const, c.d_tw_inv,     \
                 c.log_n, s2, l);                                                             \
      FHE_LAUNCH(c, "ntt_fwd_cols_rescale", (ntt_pass_rescale_lift<LIM, A>),                  \
                 dim3(ta, np, l), dim3(256), 0, t.p, (size_t)l * n, c.d_const, c.d_tw_fwd,    \
                 c.log_n, s2, lift);                                                          \
      FHE_LAUNCH(c, "ntt_fwd_blocks_rescale", (ntt_pass_rescale_out<LIM, B>),                 \
                 dim3(tb, np, l), dim3(256), 0, t.p, (size_t)l * n, c.d_const, c.d_tw_fwd,    \
                 c.log_n, s1, ptrs, c.d_rescale, l, c.L, npoly);                              \
    });                                                                                       \
    return;                                                                                   \
  }
    CASE(13, 7, 6) CASE(14, 7, 7) CASE(15, 8, 7) CASE(16, 8, 8) CASE(17, 9, 8)
#undef CASE
    default: throw ArgError("unsupported ring dimension");
  }
}

}  // namespace fhe
