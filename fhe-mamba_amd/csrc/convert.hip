// The conversion middle kernel of ModUp and ModDown, and ModUp's own passes.
#include "ntt_body.hpp"

namespace fhe {
namespace {

// First inverse pass of a fused ModUp: c1 of each ciphertext -> coef
// (blocked layout).
template <int S>
__global__ void __launch_bounds__(256)
    ntt_pass_modup_in(uint64_t* __restrict__ coef, size_t poly_stride,
                      const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                      uint32_t log_n, uint32_t s_other, const SrcPtrs src, uint64_t* digits,
                      uint32_t alpha, uint32_t nd, uint32_t ne) {
  ntt_body<16, S, BLOCKS, true, RHO_EPILOGUE, PlainStore, SrcLoad, LimbMap, false, true>(
      coef, poly_stride, mc, tw_all, log_n, LimbMap::contiguous(0), s_other, 0, PlainStore{},
      SrcLoad{src.p, 1u << log_n, digits, alpha, nd, ne});
}

// Last forward pass of a fused ModUp over the digits' converted limbs
// (blocked layout in, standard out).
template <int S>
__global__ void __launch_bounds__(256)
    ntt_pass_modup_out(uint64_t* __restrict__ digits, size_t poly_stride,
                       const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                       uint32_t log_n, DigitMap map, uint32_t s_other) {
  ntt_body<16, S, BLOCKS, false, RHO_EPILOGUE, PlainStore, PlainLoad, DigitMap, true, false>(
      digits, poly_stride, mc, tw_all, log_n, map, s_other, 1, PlainStore{});
}

// ---- Fused middle of a batched ModDown, ring dimensions 2^13 .. 2^17 ----
//
// One workgroup per (poly, column u): the last S1 inverse stages of the K
// P limbs (the column stages; the first pass wrote the blocked P limbs), the
// scaling by N^-1 * [P/p_t]^-1 folded into one Shoup product, the fast
// conversion P -> Q_l (30-bit split MACs, one REDC per output, constants in
// Montgomery form with -P^-1 folded in), and the first S1 forward stages of
// every Q limb, written to the blocked y.  This replaces an inverse column
// pass, a conversion and a forward column pass, and the three round trips
// of the P limbs and y through HBM between them.
//
// Each column line of M = 2^S1 rows belongs to TPL = min(64, M / 4) lanes of
// one wavefront (radix M / TPL per lane), so its sub-passes exchange through
// LDS with wavefront-level ordering only; the four waves of a workgroup meet
// at a single barrier, once the converted sources are in LDS.  With one line
// per wave the modulus, its twiddles and the conversion constants are
// wavefront-uniform.  Stage order, twiddle indices and lazy ranges are those
// of the column passes of ntt_body.  Workgroups have NW waves: 4 for large
// batches, 8 when a launch has too few (poly, column) tiles to fill the
// chip, which halves each workgroup's serial line count and doubles the
// waves in flight.

template <int S1>
constexpr uint32_t mid_pitch() {
  return (1u << S1) + (1u << S1) / 16 + 1;
}
template <int S1>
constexpr int mid_lanes_per_line() {
  return (1 << S1) / 4 < 64 ? (1 << S1) / 4 : 64;
}
template <int S1, int NW>
constexpr int mid_lines() {  // lines in flight per workgroup of NW waves
  return NW * (64 / mid_lanes_per_line<S1>());
}

// What one (poly, column) tile converts.  Poly p of the launch uses plan
// p % nplan; its sources are limbs src_limb0 .. src_limb0 + nsrc - 1 of
// source group p / nplan (moduli src_mod0 + t), its targets the limbs
// pos(k) = k < skip_at ? k : k + skip_len of output group p, target k in
// the plan's constant order having modulus pos < qlimbs ? pos : L + pos -
// qlimbs (Q limbs, then P limbs).  ModDown: one plan, sources the K P limbs
// of ext poly p, targets Q limbs 0..nq-1 of y poly p.  ModUp: one plan per
// digit d, sources the digit's limbs of ciphertext p / nd, targets the
// rest of Q_l + P in the digit buffer's order (the digit's own limbs
// skipped), which is the order of Context::modup_plan's targets.
constexpr int MID_MAXPLAN = 8;
struct MidPlan {
  const uint64_t* src_scale;  // [nsrc][2]: [Q/q_t]^-1 N^-1 mod q_t (Shoup)
  const uint64_t* qhat_mont;  // [nsrc][ndst], Montgomery form w.r.t. the target
  const uint64_t* qhat_mont30;  // [nsrc][ndst], qhat_mont * 2^30 mod the target
  uint32_t nsrc, ndst, src_mod0, src_limb0, skip_at, skip_len, qlimbs;
};
struct MidArgs {
  const uint64_t* src;        // blocked, inverse block stages done, [0, 4q)
  uint64_t* out;              // blocked, forward column stages done, [0, 8q)
  size_t src_group_words, out_group_words;
  MidPlan plan[MID_MAXPLAN];
  uint32_t nplan, L;
};

// One group of at most eight conversion sources i0 .. i1 - 1 for target k:
// T_g = t + u 2^64 == sum_i v_i c_ik (mod t_k), from sources held as 30-bit
// halves (vl, vh) and the Montgomery-form tables c and c' = c 2^30 mod t_k
// split into 30-bit halves: v c == vl c + vh c', so b0 = sum vl cl + vh dl
// and b1 = sum vl ch + vh dh (each below 16 2^60 = 2^64) give T_g = b0 +
// b1 2^30, whose high word u is at most 2^30.
template <int R, uint32_t VSTEP, uint32_t PITCH, class CU64>
__device__ __forceinline__ void conv_group(const uint64_t* sbase, CU64* qhat_mont,
                                           CU64* qhat_mont30, uint32_t nq, uint32_t k,
                                           uint32_t i0, uint32_t i1, uint64_t (&t)[R],
                                           uint64_t (&u)[R]) {
  constexpr uint32_t M30 = (1u << 30) - 1;
  uint64_t b0[R], b1[R];
#pragma unroll
  for (int v = 0; v < R; ++v) b0[v] = b1[v] = 0;
  for (uint32_t i = i0; i < i1; ++i) {
    const uint64_t cv = qhat_mont[(size_t)i * nq + k];
    const uint64_t dv = qhat_mont30[(size_t)i * nq + k];
    const uint64_t* sl = sbase + (size_t)i * PITCH;
    uint64_t sv[R];
#pragma unroll
    for (int v = 0; v < R; ++v) sv[v] = sl[v * VSTEP];
    // the constants' and all R elements' reads in flight before the first
    // product: one wait a source
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t cl = (uint32_t)cv & M30, ch = (uint32_t)(cv >> 30);
    const uint32_t dl = (uint32_t)dv & M30, dh = (uint32_t)(dv >> 30);
#pragma unroll
    for (int v = 0; v < R; ++v) {
      const uint32_t vl = (uint32_t)sv[v], vh = (uint32_t)(sv[v] >> 32);
      b0[v] += (uint64_t)vl * cl + (uint64_t)vh * dl;
      b1[v] += (uint64_t)vl * ch + (uint64_t)vh * dh;
    }
  }
#pragma unroll
  for (int v = 0; v < R; ++v) {
    const uint64_t m = b1[v] << 30;
    t[v] = b0[v] + m;
    u[v] = (b1[v] >> 34) + (t[v] < m);
  }
}

// Body for (poly, column) tile `tile` with (K + NL) PITCH words of lds.
template <int S1, int S2, int NW>
__device__ __forceinline__ void convert_mid_body(const MidArgs& a, const ModConst* __restrict__ mc,
                                                 const uint64_t* __restrict__ tw_inv,
                                                 const uint64_t* __restrict__ tw_fwd,
                                                 uint32_t tile, uint64_t* lds_dyn) {
  constexpr int M = 1 << S1, TPL = mid_lanes_per_line<S1>(), R = M / TPL;
  constexpr int RHO = R == 4 ? 2 : 3, LPW = 64 / TPL, NL = mid_lines<S1, NW>();
  constexpr int NSP = (S1 + RHO - 1) / RHO;
  constexpr uint32_t PITCH = mid_pitch<S1>(), N2 = 1u << S2;
  constexpr size_t N = (size_t)M << S2;
  constexpr uint32_t M30 = (1u << 30) - 1;
  static_assert(R * TPL == M && (1 << RHO) == R, "column split");
  const uint32_t p = tile / N2, col = tile % N2;
  const MidPlan& pl = a.plan[p % a.nplan];
  const uint32_t K = pl.nsrc, nq = pl.ndst;
  const uint64_t* const ext = a.src + (size_t)(p / a.nplan) * a.src_group_words +
                              (size_t)pl.src_limb0 * N;
  uint64_t* const y = a.out + (size_t)p * a.out_group_words;
  // The conversion tables are read-only for the whole launch: reading them
  // through the constant address space lets uniform loads use the scalar
  // cache, as for kernel-argument tables.
  typedef const uint64_t __attribute__((address_space(4))) cu64;
  cu64* const src_scale = (cu64*)pl.src_scale;
  cu64* const qhat_mont = (cu64*)pl.qhat_mont;
  cu64* const qhat_mont30 = (cu64*)pl.qhat_mont30;
  uint64_t* const src = lds_dyn;
  uint64_t* const work = lds_dyn + (size_t)K * PITCH;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63, sub = lane / TPL, tau = lane % TPL;
  const uint32_t first = wave * LPW + sub;

  // Inverse column stages of the P limbs; each limb is one line of src.
  for (uint32_t t = first; t < K; t += NL) {
    const uint32_t midx = pl.src_mod0 + t;
    const uint64_t q = mc[midx].q;
    const LazyMod lm = lazy_mod<16>(mc[midx]);
    const uint64_t* __restrict__ tw = tw_inv + (size_t)midx * N * 2;
    uint64_t* const line = src + (size_t)t * PITCH;
    uint64_t x[R];
    int bnd[R];  // bounds of x in q
    // First window (bits 0 .. RHO-1): rows R tau + v, one blocked run.
    const uint64_t* g = ext + (size_t)t * N + blocked_off<S2>(R * tau, col);
#pragma unroll
    for (int v = 0; v < R; ++v) x[v] = g[v];
#pragma unroll
    for (int sp = 0; sp < NSP; ++sp) {
      const int lo = RHO * sp;
      const int w = lo + RHO <= S1 ? lo : S1 - RHO;
      const int bhi = lo + RHO <= S1 ? lo + RHO - 1 : S1 - 1;
      const uint32_t thi = (tau >> w) << (w + RHO), tlo = tau & ((1u << w) - 1);
      if (sp > 0) {
#pragma unroll
        for (int v = 0; v < R; ++v) x[v] = line[lds_idx(0, thi | ((uint32_t)v << w) | tlo, 0)];
      }
#pragma unroll
      for (int v = 0; v < R; ++v) bnd[v] = 8;
#pragma unroll
      for (int beta = lo; beta <= bhi; ++beta) {
        const int d = 1 << (beta - w);
#pragma unroll
        for (int v = 0; v < R; ++v) {
          if (v & d) continue;
          const uint32_t u = thi | ((uint32_t)v << w) | tlo;
          const uint32_t ti = (1u << (S1 - 1 - beta)) | (u >> (beta + 1));
          const uint64_t wv = tw[2 * ti], ws = tw[2 * ti + 1];
          inv_butterfly(x[v], x[v + d], wv, ws, lm, 16, bnd[v], bnd[v + d]);
        }
      }
      if (sp == NSP - 1) {
        // v_t = x N^-1 [P/p_t]^-1 mod p_t, stored as 30-bit halves.
        const uint64_t f = src_scale[2 * t], fs = src_scale[2 * t + 1];
#pragma unroll
        for (int v = 0; v < R; ++v) {
          const uint64_t z = reduce_4q(shoup_lazy4(x[v], f, fs, q), q);
          x[v] = ((uint64_t)(uint32_t)(z >> 30) << 32) | ((uint32_t)z & M30);
        }
      }
      wave_lds_sync();
#pragma unroll
      for (int v = 0; v < R; ++v) line[lds_idx(0, thi | ((uint32_t)v << w) | tlo, 0)] = x[v];
      wave_lds_sync();
    }
  }
  __syncthreads();

  // Conversion into the Q limbs, one line of `work` per line in flight, then
  // their forward column stages.
  uint64_t* const line = work + (size_t)first * PITCH;
  for (uint32_t k = first; k < nq; k += NL) {
    const uint32_t kpos = k < pl.skip_at ? k : k + pl.skip_len;
    const uint32_t kmod = kpos < pl.qlimbs ? kpos : a.L + (kpos - pl.qlimbs);
    const uint64_t q = mc[kmod].q, qn = mc[kmod].qinv;
    const LazyMod lm = lazy_mod<16>(mc[kmod]);
    const uint64_t* __restrict__ tw = tw_fwd + (size_t)kmod * N * 2;
    uint64_t x[R];
    {
      // First forward window (bits S1-RHO .. S1-1): rows thi | v << w | tlo.
      constexpr int w = S1 - RHO;
      // With w >= 4 the row fields do not interact with the u / 16 padding:
      // lds_idx(thi | v << w | tlo) = lds_idx(thi | tlo) + v * VSTEP, so one
      // address register serves a source line's R reads (immediate offsets).
      static_assert(w >= 4, "padding split");
      constexpr uint32_t VSTEP = (1u << w) + (1u << (w - 4));
      const uint32_t thi = (tau >> w) << (w + RHO), tlo = tau & ((1u << w) - 1);
      const uint64_t* const sbase = src + lds_idx(0, thi | tlo, 0);
      // Sources in groups of at most eight (conv_group); the groups' sum T
      // (K <= 16: T >> 64 < 2^32 < t) takes one Montgomery reduction.
      uint64_t tl[R], th[R];  // T = tl + th 2^64
      const uint32_t k1 = K < 8 ? K : 8;
      conv_group<R, VSTEP, PITCH>(sbase, qhat_mont, qhat_mont30, nq, k, 0, k1, tl, th);
      if (K > 8) {
        uint64_t t2[R], u2[R];
        conv_group<R, VSTEP, PITCH>(sbase, qhat_mont, qhat_mont30, nq, k, 8, K, t2, u2);
#pragma unroll
        for (int v = 0; v < R; ++v) {
          tl[v] += t2[v];
          th[v] += u2[v] + (tl[v] < t2[v]);
        }
      }
#pragma unroll
      for (int v = 0; v < R; ++v) x[v] = redc_lazy(th[v], tl[v], q, qn);  // (0, 2q)
    }
#pragma unroll
    for (int sp = 0; sp < NSP; ++sp) {
      const int hi = S1 - RHO * sp;
      const int w = hi >= RHO ? hi - RHO : 0;
      const int bhi = hi - 1;
      const uint32_t thi = (tau >> w) << (w + RHO), tlo = tau & ((1u << w) - 1);
      if (sp > 0) {
#pragma unroll
        for (int v = 0; v < R; ++v) x[v] = line[lds_idx(0, thi | ((uint32_t)v << w) | tlo, 0)];
      }
#pragma unroll
      for (int beta = bhi; beta >= w; --beta) {
        const int d = 1 << (beta - w);
#pragma unroll
        for (int v = 0; v < R; ++v) {
          if (v & d) continue;
          const uint32_t u = thi | ((uint32_t)v << w) | tlo;
          const uint32_t ti = (1u << (S1 - 1 - beta)) | (u >> (beta + 1));
          const uint64_t wv = tw[2 * ti], ws = tw[2 * ti + 1];
          fwd_butterfly(x[v], x[v + d], wv, ws, lm, fwd_reduces(16, 2, S1, beta));
        }
      }
      if (sp < NSP - 1) {
        wave_lds_sync();
#pragma unroll
        for (int v = 0; v < R; ++v) line[lds_idx(0, thi | ((uint32_t)v << w) | tlo, 0)] = x[v];
        wave_lds_sync();
      } else {
        // Last window (bits 0 .. RHO-1): rows R tau + v, one blocked run.
        uint64_t* g = y + (size_t)kpos * N + blocked_off<S2>(R * tau, col);
#pragma unroll
        for (int v = 0; v < R; ++v) g[v] = x[v];
      }
    }
  }
}

template <int S1, int S2, int NW>
__global__ void __launch_bounds__(64 * NW)
    k_convert_mid(const MidArgs a, const ModConst* __restrict__ mc,
                  const uint64_t* __restrict__ tw_inv, const uint64_t* __restrict__ tw_fwd) {
  extern __shared__ uint64_t lds_dyn[];
  // Tiles in XCD order: workgroup i runs on XCD i % 8, and each XCD takes a
  // contiguous range of (poly, column) tiles, so neighbouring columns, which
  // share cache lines of the blocked layout, meet in one L2.
  const uint32_t per = gridDim.x / 8;
  const uint32_t tile = (blockIdx.x % 8) * per + blockIdx.x / 8;
  convert_mid_body<S1, S2, NW>(a, mc, tw_inv, tw_fwd, tile, lds_dyn);
}

template <int S1, int NW>
size_t mid_lds_bytes(uint32_t K) {
  return (size_t)(K + mid_lines<S1, NW>()) * mid_pitch<S1>() * 8;
}

// Launches with fewer (poly, column) tiles than this use 8-wave workgroups.
constexpr uint32_t MID_SMALL_TILES = 4096;
// Launches of at most this many tiles (one ciphertext's ModUp or ModDown)
// use 16-wave workgroups.
constexpr uint32_t MID_TINY_TILES = 1024;

template <int S1, int S2>
void launch_mid(Context& c, const char* name, const MidArgs& a, uint32_t npoly,
                uint32_t max_src) {
  const uint32_t tiles = npoly << S2;
  if (tiles <= MID_TINY_TILES && mid_lds_bytes<S1, 16>(max_src) <= c.lds_per_block) {
    FHE_LAUNCH(c, name, (k_convert_mid<S1, S2, 16>), dim3(tiles), dim3(1024),
               (mid_lds_bytes<S1, 16>(max_src)), a, c.d_const, c.d_tw_inv, c.d_tw_fwd);
    return;
  }
  if (tiles < MID_SMALL_TILES && mid_lds_bytes<S1, 8>(max_src) <= c.lds_per_block) {
    FHE_LAUNCH(c, name, (k_convert_mid<S1, S2, 8>), dim3(tiles), dim3(512),
               (mid_lds_bytes<S1, 8>(max_src)), a, c.d_const, c.d_tw_inv, c.d_tw_fwd);
    return;
  }
  FHE_LAUNCH(c, name, (k_convert_mid<S1, S2, 4>), dim3(tiles), dim3(256),
             (mid_lds_bytes<S1, 4>(max_src)), a, c.d_const, c.d_tw_inv, c.d_tw_fwd);
}

// The target order of `pl` must be the one MidPlan describes (checked).
MidPlan mid_plan(const Context& c, const ConvPlan& pl, uint32_t src_mod0, uint32_t src_limb0,
                 uint32_t skip_at, uint32_t skip_len, uint32_t qlimbs) {
  for (uint32_t k = 0; k < pl.ndst; ++k) {
    const uint32_t pos = k < skip_at ? k : k + skip_len;
    if (pl.dst_idx[k] != (pos < qlimbs ? pos : c.L + (pos - qlimbs)))
      throw ArgError("conversion plan target order");
  }
  return MidPlan{pl.d_src_scale, pl.d_qhat_mont, pl.d_qhat_mont30, pl.nsrc, pl.ndst,
                 src_mod0, src_limb0, skip_at, skip_len, qlimbs};
}

bool mid_lds_fits(const Context& c, uint32_t nsrc) {
  switch (c.log_n) {
    case 13: case 14: return mid_lds_bytes<7, 4>(nsrc) <= c.lds_per_block;
    case 15: case 16: return mid_lds_bytes<8, 4>(nsrc) <= c.lds_per_block;
    case 17: return mid_lds_bytes<9, 4>(nsrc) <= c.lds_per_block;
    default: return false;
  }
}

// Every modulus of the launch in [2^33, 2^60): the fused kernels' lazy
// ranges (16q < 2^64) and reduce_est's quotient estimate (q >= 2^33).
bool below_2_60_all(const Context& c, uint32_t nq) {
  auto ok = [](uint64_t m) { return m < (1ull << 60) && m >= (1ull << 33); };
  for (uint32_t i = 0; i < nq; ++i)
    if (!ok(c.mods[i])) return false;
  for (uint32_t t = 0; t < c.K; ++t)
    if (!ok(c.mods[c.L + t])) return false;
  return true;
}

}  // namespace

bool convert_mid_ok(const Context& c, uint32_t nq, uint32_t nsrc) {
  return below_2_60_all(c, nq) && mid_lds_fits(c, nsrc);
}

void moddown_mid(Context& c, const uint64_t* ext_p, uint64_t* y, uint32_t npoly, uint32_t nq,
                 const ConvPlan& pl) {
  MidArgs a{};
  a.src = ext_p;
  a.out = y;
  a.src_group_words = (size_t)c.K * c.n;
  a.out_group_words = (size_t)nq * c.n;
  a.plan[0] = mid_plan(c, pl, c.L, 0, nq, 0, nq);
  a.nplan = 1;
  a.L = c.L;
  switch (c.log_n) {
#define CASE(LN, A, B) \
  case LN: launch_mid<A, B>(c, "k_moddown_mid", a, npoly, c.K); return;
    CASE(13, 7, 6) CASE(14, 7, 7) CASE(15, 8, 7) CASE(16, 8, 8) CASE(17, 9, 8)
#undef CASE
    default: throw ArgError("unsupported ring dimension");
  }
}

bool modup_fused_ok(const Context& c, uint32_t nq, uint32_t count) {
  if (c.log_n < 13 || c.log_n > 17 || c.K == 0 || c.alpha == 0 || c.alpha > 16) return false;
  if (nq == 0 || nq > c.L || count == 0 || count > (uint32_t)MODUP_MAX_CT) return false;
  const uint32_t nd = num_digits(c, nq);
  if (nd > (uint32_t)MID_MAXPLAN || (uint64_t)count * nd > 65535) return false;
  return convert_mid_ok(c, nq, c.alpha);
}

void modup_fused(Context& c, const uint64_t* const* as, uint32_t count, uint32_t nq,
                 uint64_t* digits) {
  if (!modup_fused_ok(c, nq, count)) throw ArgError("fused ModUp does not apply");
  const size_t n = c.n;
  const uint32_t ne = nq + c.K, nd = num_digits(c, nq);
  Scratch coef(c, (size_t)count * nq * n);
  SrcPtrs sp{};
  for (uint32_t i = 0; i < count; ++i) sp.p[i] = as[i];
  MidArgs a{};
  a.src = coef.p;
  a.out = digits;
  a.src_group_words = (size_t)nq * n;
  a.out_group_words = (size_t)ne * n;
  a.nplan = nd;
  a.L = c.L;
  uint32_t max_src = 0;
  for (uint32_t d = 0; d < nd; ++d) {
    const uint32_t s0 = d * c.alpha, e0 = s0 + c.alpha < nq ? s0 + c.alpha : nq;
    a.plan[d] = mid_plan(c, c.modup_plan(s0, e0, nq), s0, s0, s0, e0 - s0, nq);
    max_src = max_src > e0 - s0 ? max_src : e0 - s0;
  }
  // The last digit is the narrowest and so has the most converted limbs.
  const uint32_t w_last = nq - (nd - 1) * c.alpha;
  const DigitMap map{c.alpha, nq, c.L, ne, nd};
  const uint32_t s1 = (c.log_n + 1) / 2;
  switch (c.log_n) {
#define CASE(LN, A, B)                                                                        \
  case LN: {                                                                                  \
    using G = Geo<B, RHO_EPILOGUE>;                                                           \
    const uint32_t tiles = (1u << s1) / (256 / G::TPL);                                       \
    FHE_LAUNCH(c, "ntt_inv_blocks_modup", (ntt_pass_modup_in<B>), dim3(tiles, count, nq),     \
               dim3(256), 0, coef.p, (size_t)nq * n, c.d_const, c.d_tw_inv, c.log_n, s1, sp,  \
               digits, c.alpha, nd, ne);                                                      \
    launch_mid<A, B>(c, "k_modup_mid", a, count * nd, max_src);                               \
    FHE_LAUNCH(c, "ntt_fwd_blocks_modup", (ntt_pass_modup_out<B>),                            \
               dim3(tiles, count * nd, ne - w_last), dim3(256), 0, digits, (size_t)ne * n,    \
               c.d_const, c.d_tw_fwd, c.log_n, map, s1);                                      \
    break;                                                                                    \
  }
    CASE(13, 7, 6) CASE(14, 7, 7) CASE(15, 8, 7) CASE(16, 8, 8) CASE(17, 9, 8)
#undef CASE
    default: throw ArgError("unsupported ring dimension");
  }
}

}  // namespace fhe
