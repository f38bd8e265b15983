// Key switching and rescale for rings of at most 2^12: one workgroup
// transforms a limb, so a call is a handful of short launches and its time is
// their count and each one's chain of sub-passes.  The basis conversions are
// formed by the forward transforms as they load, which leaves four launches
// to a key switch and two to a rescale.
#include "key_product.hpp"
#include "rescale_parts.hpp"

namespace fhe {
namespace {

// Basis conversion as a forward transform loads: target limb blockIdx.z's
// value at position g from the coefficient-form sources, y = REDC(sum_i
// [x_i qhat_inv_i]_{s_i} qhat_mont_ik).  At most SMALL_MAX_SRC sources: the
// 128-bit sum then needs one reduction (8 q < 2^64), and recomputing the
// sources' products in every target's workgroup costs less than the launch
// that would share them.
constexpr uint32_t SMALL_MAX_SRC = 8;
struct SmallPlan {
  const uint64_t* qhat_inv;   // [nsrc][2]
  const uint64_t* qhat_mont;  // [nsrc][ndst]
  uint32_t nsrc, ndst, src_limb, src_mod;
};
constexpr int SMALL_MAXPLAN = 8;
// Launch poly p converts by plan p % nplan the limbs src_limb ... of source
// group p / nplan (src_limbs limbs each).
struct SmallConv {
  const uint64_t* src;
  const ModConst* mc;
  SmallPlan plan[SMALL_MAXPLAN];
  uint32_t nplan, src_limbs, n;
};
struct ConvLoad {
  static constexpr bool kLoad = true;
  static constexpr bool kBulk = true;
  const SmallConv& a;
  uint32_t mod;
  __device__ __forceinline__ uint64_t get(size_t, uint64_t) const { return 0; }
  template <int R>
  __device__ __forceinline__ void bulk(const size_t (&g)[R], uint64_t (&x)[R]) const {
    const SmallPlan& pl = a.plan[blockIdx.y % a.nplan];
    const uint64_t* s =
        a.src + ((size_t)(blockIdx.y / a.nplan) * a.src_limbs + pl.src_limb) * a.n;
    Acc128 acc[R];
    for (uint32_t i = 0; i < pl.nsrc; ++i, s += a.n) {
      const uint64_t qi = a.mc[pl.src_mod + i].q;
      const uint64_t f = pl.qhat_inv[2 * i], fs = pl.qhat_inv[2 * i + 1];
      const uint64_t c = pl.qhat_mont[(size_t)i * pl.ndst + blockIdx.z];
      uint64_t v[R];
#pragma unroll
      for (int k = 0; k < R; ++k) v[k] = s[g[k]];
#pragma unroll
      for (int k = 0; k < R; ++k) acc[k].mac(shoup(v[k], f, fs, qi), c);
    }
    const uint64_t q = a.mc[mod].q, qn = a.mc[mod].qinv_neg;
#pragma unroll
    for (int k = 0; k < R; ++k) x[k] = redc(acc[k].hi, acc[k].lo, q, qn);
  }
};

template <int LIM, int S>
__global__ void __launch_bounds__(max_threads<SINGLE>())
    small_modup_in(uint64_t* __restrict__ coef, size_t poly_stride,
                   const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                   uint32_t log_n, const SrcPtrs src, uint64_t* digits, uint32_t alpha,
                   uint32_t nd, uint32_t ne) {
  ntt_body<LIM, S, SINGLE, true, RHO_SINGLE, PlainStore, SrcLoad<true>>(
      coef, poly_stride, mc, tw_all, log_n, LimbMap::contiguous(0), 0, PlainStore{},
      SrcLoad<true>{src.p, 1u << log_n, digits, alpha, nd, ne});
}

template <int LIM, int S>
__global__ void __launch_bounds__(max_threads<SINGLE>())
    small_modup_out(uint64_t* __restrict__ digits, size_t poly_stride,
                    const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                    uint32_t log_n, DigitMap map, const SmallConv conv) {
  uint32_t pos, mod;
  if (!map.resolve(blockIdx.y, blockIdx.z, pos, mod)) return;
  ntt_body<LIM, S, SINGLE, false, RHO_SINGLE, PlainStore, ConvLoad, DigitMap>(
      digits, poly_stride, mc, tw_all, log_n, map, 0, PlainStore{}, ConvLoad{conv, mod});
}

template <int LIM, int S, int ND>
__global__ void __launch_bounds__(max_threads<SINGLE>())
    small_ksk(uint64_t* __restrict__ data, size_t poly_stride, const ModConst* __restrict__ mc,
              const uint64_t* __restrict__ tw_all, uint32_t log_n, const ModDownEpi epi) {
  ntt_body<LIM, S, SINGLE, true, RHO_SINGLE, PlainStore, KskLoad<ND>>(
      data, poly_stride, mc, tw_all, log_n, LimbMap::contiguous(epi.L), 0, PlainStore{},
      KskLoad<ND>{epi, 1u << log_n});
}

// CONV: the input is converted from conv's sources, else read from y.
template <int LIM, int S, int ND, bool CONV>
__global__ void __launch_bounds__(max_threads<SINGLE>())
    small_moddown(uint64_t* __restrict__ y, size_t poly_stride, const ModConst* __restrict__ mc,
                  const uint64_t* __restrict__ tw_all, uint32_t log_n, const ModDownEpi epi,
                  const SmallConv conv) {
  const EpiStore<ND> st{epi, 1u << log_n, log_n};
  if constexpr (CONV)
    ntt_body<LIM, S, SINGLE, false, RHO_SINGLE, EpiStore<ND>, ConvLoad>(
        y, poly_stride, mc, tw_all, log_n, LimbMap::contiguous(0), 0, st,
        ConvLoad{conv, blockIdx.z});
  else
    ntt_body<LIM, S, SINGLE, false, RHO_SINGLE, EpiStore<ND>>(
        y, poly_stride, mc, tw_all, log_n, LimbMap::contiguous(0), 0, st);
}

// Rescale: the last limb to coefficient form, then every other limb's centred
// lift, transform and (a - t) q_l^-1.
template <int LIM, int S>
__global__ void __launch_bounds__(max_threads<SINGLE>())
    small_rescale_in(uint64_t* __restrict__ last, const ModConst* __restrict__ mc,
                     const uint64_t* __restrict__ tw_all, uint32_t log_n, const RescalePtrs ptrs,
                     uint32_t npoly, size_t poly_words, uint32_t l) {
  ntt_body<LIM, S, SINGLE, true, RHO_SINGLE, PlainStore, LastLimbLoad>(
      last, (size_t)1 << log_n, mc, tw_all, log_n, LimbMap::contiguous(l), 0, PlainStore{},
      LastLimbLoad{ptrs.a, npoly, poly_words, (size_t)l << log_n});
}

template <int LIM, int S>
__global__ void __launch_bounds__(max_threads<SINGLE>())
    small_rescale_out(const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                      uint32_t log_n, const LiftLoad ld, const RescalePtrs ptrs,
                      const uint64_t* __restrict__ rs, uint32_t l, uint32_t L, uint32_t npoly) {
  ntt_body<LIM, S, SINGLE, false, RHO_SINGLE, RescaleStore, LiftLoad>(
      nullptr, 0, mc, tw_all, log_n, LimbMap::contiguous(0), 0,
      RescaleStore{ptrs.a, ptrs.out, rs, 1u << log_n, l, L, npoly}, ld);
}

// f(lim, S, fixed): ring size and lazy range as compile-time constants.  The
// smallest rings (below 2^10, tests of tiny parameters) share the narrow
// range and run-time digit counts.
template <class F>
void with_ring(const Context& c, F&& f) {
  switch (c.log_n) {
#define TINY(S)                                                                            \
  case S:                                                                                  \
    f(std::integral_constant<int, 8>{}, std::integral_constant<int, S>{}, std::false_type{}); \
    return;
#define RING(S)                                                                            \
  case S:                                                                                  \
    with_lim(c, [&](auto lim) { f(lim, std::integral_constant<int, S>{}, std::true_type{}); }); \
    return;
    TINY(4) TINY(5) TINY(6) TINY(7) TINY(8) TINY(9) RING(10) RING(11) RING(12)
#undef TINY
#undef RING
    default: throw ArgError("unsupported ring dimension");
  }
}
SmallPlan small_plan(const ConvPlan& pl, uint32_t src_limb, uint32_t src_mod) {
  return SmallPlan{pl.d_qhat_inv, pl.d_qhat_mont, pl.nsrc, pl.ndst, src_limb, src_mod};
}

}  // namespace

bool small_modup_ok(const Context& c, uint32_t nq) {
  return c.log_n <= 12 && c.alpha <= SMALL_MAX_SRC && num_digits(c, nq) <= SMALL_MAXPLAN;
}
bool small_moddown_ok(const Context& c) {
  return c.log_n <= 12 && c.K >= 1 && c.K <= SMALL_MAX_SRC;
}

void small_modup(Context& c, const uint64_t* const* as, uint32_t count, uint32_t nq,
                 uint64_t* digits) {
  const uint32_t ne = nq + c.K, nd = num_digits(c, nq);
  const uint32_t w_last = nq - (nd - 1) * c.alpha;  // the narrowest digit
  for (uint32_t r0 = 0; r0 < count; r0 += MODUP_MAX_CT) {
    const uint32_t b = count - r0 < (uint32_t)MODUP_MAX_CT ? count - r0 : MODUP_MAX_CT;
    uint64_t* const dig = digits + (size_t)r0 * nd * ne * c.n;
    Scratch coef(c, (size_t)b * nq * c.n);
    SrcPtrs sp{};
    for (uint32_t i = 0; i < b; ++i) sp.p[i] = as[r0 + i];
    SmallConv conv{};
    conv.src = coef.p;
    conv.mc = c.d_const;
    conv.nplan = nd;
    conv.src_limbs = nq;
    conv.n = c.n;
    for (uint32_t d = 0; d < nd; ++d) {
      const uint32_t s0 = d * c.alpha, e0 = s0 + c.alpha < nq ? s0 + c.alpha : nq;
      conv.plan[d] = small_plan(c.modup_plan(s0, e0, nq), s0, s0);
    }
    const DigitMap map{c.alpha, nq, c.L, ne, nd};
    with_ring(c, [&](auto lim, auto s, auto) {
      constexpr int LIM = decltype(lim)::value, S = decltype(s)::value;
      const dim3 threads(Geo<S, RHO_SINGLE>::TPL);
      FHE_LAUNCH(c, "ntt_inv_single_modup", (small_modup_in<LIM, S>), dim3(1, b, nq), threads, 0,
                 coef.p, (size_t)nq * c.n, c.d_const, c.d_tw_inv, c.log_n, sp, dig, c.alpha, nd,
                 ne);
      FHE_LAUNCH(c, "ntt_fwd_single_modup", (small_modup_out<LIM, S>),
                 dim3(1, b * nd, ne - w_last), threads, 0, dig, (size_t)ne * c.n, c.d_const,
                 c.d_tw_fwd, c.log_n, map, conv);
    });
  }
}

void small_ring_ksk(Context& c, uint64_t* ext_p, uint32_t npoly, const ModDownEpi& epi) {
  with_ring(c, [&](auto lim, auto s, auto fixed) {
    constexpr int LIM = decltype(lim)::value, S = decltype(s)::value;
    with_digits<decltype(fixed)::value>(epi.nd, [&](auto nd) {
      FHE_LAUNCH(c, "ntt_inv_single_ksk", (small_ksk<LIM, S, decltype(nd)::value>),
                 dim3(1, npoly, c.K), dim3(Geo<S, RHO_SINGLE>::TPL), 0, ext_p,
                 (size_t)c.K * c.n, c.d_const, c.d_tw_inv, c.log_n, epi);
    });
  });
}

static void small_moddown_launch(Context& c, uint64_t* y, uint32_t npoly, uint32_t nq,
                                 const ModDownEpi& epi, const SmallConv* conv) {
  with_ring(c, [&](auto lim, auto s, auto fixed) {
    constexpr int LIM = decltype(lim)::value, S = decltype(s)::value;
    with_digits<decltype(fixed)::value>(epi.nd, [&](auto nd) {
      constexpr int ND = decltype(nd)::value;
      const dim3 grid(1, npoly, nq), threads(Geo<S, RHO_SINGLE>::TPL);
      if (conv)
        FHE_LAUNCH(c, "ntt_fwd_single_moddown", (small_moddown<LIM, S, ND, true>), grid, threads,
                   0, y, (size_t)nq * c.n, c.d_const, c.d_tw_fwd, c.log_n, epi, *conv);
      else
        FHE_LAUNCH(c, "ntt_fwd_single_moddown", (small_moddown<LIM, S, ND, false>), grid, threads,
                   0, y, (size_t)nq * c.n, c.d_const, c.d_tw_fwd, c.log_n, epi, SmallConv{});
    });
  });
}

void small_ring_moddown(Context& c, uint64_t* y, uint32_t npoly, uint32_t nq,
                        const ModDownEpi& epi) {
  small_moddown_launch(c, y, npoly, nq, epi, nullptr);
}

void small_ring_moddown_conv(Context& c, const uint64_t* ext_p, uint32_t npoly, uint32_t nq,
                             const ConvPlan& pl, const ModDownEpi& epi) {
  SmallConv conv{};
  conv.src = ext_p;
  conv.mc = c.d_const;
  conv.nplan = 1;
  conv.src_limbs = c.K;
  conv.n = c.n;
  conv.plan[0] = small_plan(pl, 0, c.L);
  small_moddown_launch(c, nullptr, npoly, nq, epi, &conv);
}

void small_rescale(Context& c, uint64_t* const* outs, const uint64_t* const* as, uint32_t count,
                   uint32_t npoly, uint32_t nq) {
  const uint32_t l = nq - 1, n = c.n;
  if (nq < 2 || npoly == 0 || npoly > 65535) throw ArgError("rescale: bad shape");
  for (uint32_t r0 = 0; r0 < count;) {
    const uint32_t b = rescale_batch(count - r0, npoly), np = b * npoly;
    RescalePtrs ptrs{};
    for (uint32_t r = 0; r < b; ++r) {
      ptrs.a[r] = as[r0 + r];
      ptrs.out[r] = outs[r0 + r];
    }
    Scratch last(c, (size_t)np * n);
    const LiftLoad lift{last.p, c.d_const, c.d_rescale, n, l, c.L, c.mods[l] >> 1};
    with_ring(c, [&](auto lim, auto s, auto) {
      constexpr int LIM = decltype(lim)::value, S = decltype(s)::value;
      const dim3 threads(Geo<S, RHO_SINGLE>::TPL);
      FHE_LAUNCH(c, "ntt_inv_single_rescale", (small_rescale_in<LIM, S>), dim3(1, np, 1), threads,
                 0, last.p, c.d_const, c.d_tw_inv, c.log_n, ptrs, npoly, (size_t)nq * n, l);
      FHE_LAUNCH(c, "ntt_fwd_single_rescale", (small_rescale_out<LIM, S>), dim3(1, np, l), threads,
                 0, c.d_const, c.d_tw_fwd, c.log_n, lift, ptrs, c.d_rescale, l, c.L, npoly);
    });
    r0 += b;
  }
}

}  // namespace fhe
