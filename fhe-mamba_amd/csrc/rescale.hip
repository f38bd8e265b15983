// Rescale in three launches, or four passes of ntt_body.hpp.
#include "rescale_parts.hpp"

namespace fhe {
namespace {

// ---- Rescale, ring dimensions 2^13 .. 2^17 ----
// The passes run radix 8 (RHO_EPILOGUE: eight lines of 2^S words and 17 KB of
// LDS per 256-lane workgroup), so one ciphertext's launch fits the chip in
// one round of workgroups.  The inverse NTT of the last limb reads it from
// the input (LastLimbLoad); the last forward pass stores (a_i - t_i) * q_l^-1
// (RescaleStore).  Between them, for moduli in the wide lazy range, one
// kernel per column does the inverse column stages of the last limb, its
// centred lift and the forward column stages of every other limb
// (k_rescale_mid, blocked layout on both sides): three launches.  For other
// moduli, and where rescale_by_columns says so, an inverse column pass and a
// forward one that lifts as it loads (LiftLoad): four.

// One workgroup per (launch poly, column) tile, nw waves, LPW column lines a
// wave.  The first line's wave takes the last limb to centred coefficients v
// in LDS; then each line in flight lifts and transforms one target limb after
// another.  v + lift_k >= 0 for lift_k the least multiple of q_k not below
// q_l / 2; where that is q_k itself the sum is below 2 q_k and needs no
// reduction, as for the primes of one chain.
template <int S1, int S2>
__device__ __forceinline__ void rescale_mid_body(
    const uint64_t* __restrict__ last, uint64_t* __restrict__ t,
    const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_inv,
    const uint64_t* __restrict__ tw_fwd, const uint64_t* __restrict__ rs, uint32_t l, uint32_t L,
    uint32_t tile, uint32_t nw, uint64_t* lds) {
  constexpr int M = 1 << S1, TPL = mid_lanes_per_line<S1>(), R = M / TPL;
  constexpr int RHO = R == 4 ? 2 : 3, LPW = 64 / TPL, NSP = (S1 + RHO - 1) / RHO;
  constexpr uint32_t PITCH = mid_pitch<S1>(), N2 = 1u << S2;
  constexpr size_t N = (size_t)M << S2;
  const uint32_t p = tile / N2, col = tile % N2, nl = nw * LPW;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63, sub = lane / TPL, tau = lane % TPL;
  const uint32_t first = wave * LPW + sub;
  uint64_t* const src = lds;
  uint64_t* const line = lds + (size_t)(1 + first) * PITCH;
  uint64_t x[R], twx[2][R - 1], twy[2][R - 1];

  if (first == 0) {
    const uint64_t q = mc[l].q, half = q >> 1;
    const LazyMod lm = lazy_mod<16>(mc[l]);
    const uint64_t* __restrict__ tw = tw_inv + (size_t)l * N * 2;
    int bnd[R];
    const uint64_t* g = last + (size_t)p * N + blocked_off<S2>(R * tau, col);
#pragma unroll
    for (int v = 0; v < R; ++v) x[v] = g[v];
    fetch_twiddles<S1, RHO, true, 0, LPW == 1>(tw, 1, tau, twx[0], twy[0]);
    static_for<NSP>([&](auto spc) {
      constexpr int sp = decltype(spc)::value;
      using W = SubPass<S1, RHO, true, sp>;
      constexpr int w = W::w;
      const uint32_t thi = (tau >> w) << (w + RHO), tlo = tau & ((1u << w) - 1);
      if (sp > 0) {
#pragma unroll
        for (int v = 0; v < R; ++v) x[v] = src[lds_idx(0, thi | ((uint32_t)v << w) | tlo, 0)];
      }
      if constexpr (sp + 1 < NSP)
        fetch_twiddles<S1, RHO, true, sp + 1, LPW == 1>(tw, 1, tau, twx[(sp + 1) & 1],
                                                        twy[(sp + 1) & 1]);
#pragma unroll
      for (int v = 0; v < R; ++v) bnd[v] = 8;
#pragma unroll
      for (int k = 0; k < RHO; ++k) {
        const int beta = w + k, d = 1 << k;
        if (beta < W::blo || beta > W::bhi) continue;
#pragma unroll
        for (int v = 0; v < R; ++v) {
          if (v & d) continue;
          const int ti = twiddle_at<RHO>(k, v);
          inv_butterfly(x[v], x[v + d], twx[sp & 1][ti], twy[sp & 1][ti], lm, 16, bnd[v],
                        bnd[v + d]);
        }
      }
      if (sp == NSP - 1) {
        const uint64_t f = mc[l].ninv, fs = mc[l].ninv_sh;
#pragma unroll
        for (int v = 0; v < R; ++v) {
          const uint64_t z = reduce_4q(shoup_acc(0, x[v], f, fs, lm.neg_q, lm.one), q);
          x[v] = z > half ? z - q : z;
        }
      }
      wave_lds_sync();
#pragma unroll
      for (int v = 0; v < R; ++v) src[lds_idx(0, thi | ((uint32_t)v << w) | tlo, 0)] = x[v];
      wave_lds_sync();
    });
  }
  __syncthreads();

  for (uint32_t k = first; k < l; k += nl) {
    const LazyMod lm = lazy_mod<16>(mc[k]);
    const uint64_t lift = rs[((size_t)l * L + k) * 4 + 3];
    const uint64_t* __restrict__ tw = tw_fwd + (size_t)k * N * 2;
    fetch_twiddles<S1, RHO, false, 0, LPW == 1>(tw, 1, tau, twx[0], twy[0]);
    static_for<NSP>([&](auto spc) {
      constexpr int sp = decltype(spc)::value;
      using W = SubPass<S1, RHO, false, sp>;
      constexpr int w = W::w;
      const uint32_t thi = (tau >> w) << (w + RHO), tlo = tau & ((1u << w) - 1);
      if constexpr (sp + 1 < NSP)
        fetch_twiddles<S1, RHO, false, sp + 1, LPW == 1>(tw, 1, tau, twx[(sp + 1) & 1],
                                                         twy[(sp + 1) & 1]);
#pragma unroll
      for (int v = 0; v < R; ++v) {
        const uint32_t u = lds_idx(0, thi | ((uint32_t)v << w) | tlo, 0);
        x[v] = sp == 0 ? src[u] + lift : line[u];
      }
      if (sp == 0 && lift != mc[k].q) {
#pragma unroll
        for (int v = 0; v < R; ++v) x[v] = reduce_est(x[v], lm.neg_q, mc[k].rq);
      }
#pragma unroll
      for (int j = RHO - 1; j >= 0; --j) {
        const int beta = w + j, d = 1 << j;
        if (beta > W::bhi) continue;
#pragma unroll
        for (int v = 0; v < R; ++v) {
          if (v & d) continue;
          const int ti = twiddle_at<RHO>(j, v);
          fwd_butterfly(x[v], x[v + d], twx[sp & 1][ti], twy[sp & 1][ti], lm,
                        fwd_reduces(16, 2, S1, beta));
        }
      }
      if (sp < NSP - 1) {
        wave_lds_sync();
#pragma unroll
        for (int v = 0; v < R; ++v) line[lds_idx(0, thi | ((uint32_t)v << w) | tlo, 0)] = x[v];
        wave_lds_sync();
      } else {
        uint64_t* g = t + ((size_t)p * l + k) * N + blocked_off<S2>(R * tau, col);
#pragma unroll
        for (int v = 0; v < R; ++v) g[v] = x[v];
      }
    });
  }
}

template <int S1, int S2>
__global__ void __launch_bounds__(S1 == 9 ? 512 : 1024)
    __attribute__((amdgpu_waves_per_eu(S1 == 9 ? 4 : 8, 8)))
    k_rescale_mid(const uint64_t* __restrict__ last, uint64_t* __restrict__ t,
                  const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_inv,
                  const uint64_t* __restrict__ tw_fwd, const uint64_t* __restrict__ rs, uint32_t l,
                  uint32_t L) {
  extern __shared__ uint64_t lds_dyn[];
  // tiles in XCD order, as in k_convert_mid
  const uint32_t per = gridDim.x / 8;
  const uint32_t tile = (blockIdx.x % 8) * per + blockIdx.x / 8;
  rescale_mid_body<S1, S2>(last, t, mc, tw_inv, tw_fwd, rs, l, L, tile, blockDim.x / 64, lds_dyn);
}

template <int LIM, int S>
__global__ void __launch_bounds__(256)
    ntt_pass_rescale_in(uint64_t* __restrict__ last, const ModConst* __restrict__ mc,
                        const uint64_t* __restrict__ tw_all, uint32_t log_n, uint32_t s_other,
                        const RescalePtrs ptrs, uint32_t npoly, size_t poly_words, uint32_t l) {
  ntt_body<LIM, S, BLOCKS, true, RHO_EPILOGUE, PlainStore, LastLimbLoad, LimbMap, false,
           LIM == 16>(
      last, (size_t)1 << log_n, mc, tw_all, log_n, LimbMap::contiguous(l), s_other,
      PlainStore{}, LastLimbLoad{ptrs.a, npoly, poly_words, (size_t)l << log_n});
}

template <int S>
__global__ void __launch_bounds__(256)
    ntt_pass_rescale_lift(uint64_t* __restrict__ t, size_t poly_stride,
                          const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                          uint32_t log_n, uint32_t s_other, const LiftLoad ld) {
  ntt_body<8, S, COLS, false, RHO_EPILOGUE, PlainStore, LiftLoad>(
      t, poly_stride, mc, tw_all, log_n, LimbMap::contiguous(0), s_other, PlainStore{}, ld);
}

template <int LIM, int S>
__global__ void __launch_bounds__(256)
    ntt_pass_rescale_out(uint64_t* __restrict__ t, size_t poly_stride,
                         const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                         uint32_t log_n, uint32_t s_other, const RescalePtrs ptrs,
                         const uint64_t* __restrict__ rs, uint32_t l, uint32_t L,
                         uint32_t npoly) {
  ntt_body<LIM, S, BLOCKS, false, RHO_EPILOGUE, RescaleStore, PlainLoad, LimbMap, LIM == 16>(
      t, poly_stride, mc, tw_all, log_n, LimbMap::contiguous(0), s_other,
      RescaleStore{ptrs.a, ptrs.out, rs, 1u << log_n, l, L, npoly});
}

// The rescale's inverse column pass over the last limb (radix 8, as the
// other rescale passes): launch poly y's single limb, modulus l.
template <int S>
__global__ void __launch_bounds__(256)
    ntt_pass_rescale_cols(uint64_t* __restrict__ data, size_t poly_stride,
                          const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                          uint32_t log_n, uint32_t s_other, uint32_t l) {
  ntt_body<8, S, COLS, true, RHO_EPILOGUE, PlainStore, PlainLoad, LimbMap>(
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
  // The column kernel reduces a lifted value below q_l + q_k by reduce_est.
  bool mid = c.lazy16;
  for (uint32_t k = 0; k < l; ++k) mid = mid && c.mods[l] / c.mods[k] < (1u << 17);
  switch (c.log_n) {
#define CASE(LN, A, B)                                                                        \
  case LN: {                                                                                  \
    using GB = Geo<B, RHO_EPILOGUE>;                                                          \
    using GA = Geo<A, RHO_EPILOGUE>;                                                          \
    const uint32_t tb = (1u << s1) / (256 / GB::TPL), ta = (1u << s2) / (256 / GA::TPL);      \
    auto in = [&](auto lim) {                                                                 \
      FHE_LAUNCH(c, "ntt_inv_blocks_rescale", (ntt_pass_rescale_in<decltype(lim)::value, B>), \
                 dim3(tb, np, 1), dim3(256), 0, last.p, c.d_const, c.d_tw_inv, c.log_n, s1,   \
                 ptrs, npoly, (size_t)nq * n, l);                                             \
    };                                                                                        \
    auto out = [&](auto lim) {                                                                \
      FHE_LAUNCH(c, "ntt_fwd_blocks_rescale", (ntt_pass_rescale_out<decltype(lim)::value, B>), \
                 dim3(tb, np, l), dim3(256), 0, t.p, (size_t)l * n, c.d_const, c.d_tw_fwd,    \
                 c.log_n, s1, ptrs, c.d_rescale, l, c.L, npoly);                              \
    };                                                                                        \
    if (mid && rescale_by_columns(A, np << B, l)) {                                           \
      const uint32_t nw = rescale_waves(A, np << B, l);                                       \
      in(std::integral_constant<int, 16>{});                                                  \
      FHE_LAUNCH(c, "k_rescale_mid", (k_rescale_mid<A, B>), dim3(np << B), dim3(64 * nw),     \
                 rescale_lds_bytes(A, nw), last.p, t.p, c.d_const, c.d_tw_inv, c.d_tw_fwd,    \
                 c.d_rescale, l, c.L);                                                        \
      out(std::integral_constant<int, 16>{});                                                 \
      return;                                                                                 \
    }                                                                                         \
    in(std::integral_constant<int, 8>{});                                                     \
    FHE_LAUNCH(c, "ntt_inv_cols_rescale", (ntt_pass_rescale_cols<A>), dim3(ta, np, 1),        \
               dim3(256), 0, last.p, (size_t)n, c.d_const, c.d_tw_inv, c.log_n, s2, l);       \
    FHE_LAUNCH(c, "ntt_fwd_cols_rescale", (ntt_pass_rescale_lift<A>), dim3(ta, np, l),        \
               dim3(256), 0, t.p, (size_t)l * n, c.d_const, c.d_tw_fwd, c.log_n, s2, lift);   \
    out(std::integral_constant<int, 8>{});                                                    \
    return;                                                                                   \
  }
    CASE(13, 7, 6) CASE(14, 7, 7) CASE(15, 8, 7) CASE(16, 8, 8) CASE(17, 9, 8)
#undef CASE
    default: throw ArgError("unsupported ring dimension");
  }
}

}  // namespace fhe
