// The conversion middle kernel of ModUp and ModDown, and ModUp's own passes.

#include "ntt_body.hpp"

namespace fhe {
namespace {

// First inverse pass of a fused ModUp: c1 of each ciphertext -> coef
// (blocked layout).
template <int S, bool KEEP>
__global__ void __launch_bounds__(256)
    ntt_pass_modup_in(uint64_t* __restrict__ coef, size_t poly_stride,
                      const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                      uint32_t log_n, uint32_t s_other, const SrcPtrs src, uint64_t* digits,
                      uint32_t alpha, uint32_t nd, uint32_t ne) {
  ntt_body<16, S, BLOCKS, true, RHO_EPILOGUE, PlainStore, SrcLoad<KEEP>, LimbMap, false, true>(
      coef, poly_stride, mc, tw_all, log_n, LimbMap::contiguous(0), s_other, PlainStore{},
      SrcLoad<KEEP>{src.p, 1u << log_n, digits, alpha, nd, ne});
}

// Last forward pass of a fused ModUp over the digits' converted limbs
// (blocked layout in, standard out).
template <int S>
__global__ void __launch_bounds__(256)
    ntt_pass_modup_out(uint64_t* __restrict__ digits, size_t poly_stride,
                       const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                       uint32_t log_n, DigitMap map, uint32_t s_other) {
  ntt_body<16, S, BLOCKS, false, RHO_EPILOGUE, PlainStore, PlainLoad, DigitMap, true, false>(
      digits, poly_stride, mc, tw_all, log_n, map, s_other, PlainStore{});
}

// ---- Fused middle of ModUp and of a batched ModDown, N = 2^13 .. 2^17 ----
//
// One workgroup per (poly, column u): the last S1 inverse stages of the
// source limbs (the column stages; the first pass wrote them in the blocked
// layout), the scaling by N^-1 * [Q/q_t]^-1 folded into one Shoup product, the
// fast basis conversion, and the first S1 forward stages of every target
// limb, written blocked.  This replaces an inverse column pass, a conversion
// and a forward column pass, and the round trips through HBM between them.
//
// Each column line of M = 2^S1 rows belongs to TPL = min(64, M / 4) lanes of
// one wavefront (radix M / TPL per lane), so its sub-passes exchange through
// LDS with wavefront-level ordering only.  With one line per wave the modulus
// and its constants are wavefront-uniform.  Targets go in batches of one line
// per line in flight: the workgroup converts a batch into the lines, meets,
// and each wavefront transforms its own.
//
// The conversion y_k = sum_i v_i c_ik mod t_k is a contraction over the
// sources, done on the int8 matrix units.  v_i is held as eight balanced bytes
// s_ia (v = sum_a s_ia 2^8a, s in [-128, 127]), and the table holds the
// balanced bytes of C_iak = c_ik 2^8a 2^32 mod t_k, so
//   T_k = sum_ia s_ia C_iak = sum_b 2^8b S_kb,   S_kb = sum_ia s_ia byte_b(C_iak)
// with |S_kb| <= 8 K 2^14 <= 2^21 exact in 32 bits: v_mfma_i32_32x32x32_i8
// gives the eight sums of four targets (32 rows) at 32 column rows (32
// columns) from four sources a step.  One 32-bit Montgomery step of the about
// 75-bit T_k, T_k + m t_k = 2^32 r, leaves r = sum_i v_i c_ik in (0, 3 t_k)
// after adding t_k.  Per output that is 19 VALU instructions whatever the number
// of sources, where 64-bit multiply-adds took 4 a source and 25.
constexpr uint32_t MAX_CONV_SRC = 16;

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
  const int8_t* bytes;        // ConvPlan::d_bytes
  uint32_t nsrc, ndst, src_mod0, src_limb0, skip_at, skip_len, qlimbs;
};
struct MidArgs {
  const uint64_t* src;        // blocked, inverse block stages done, below 8q
  uint64_t* out;              // blocked, forward column stages done, below 12q
  size_t src_group_words, out_group_words;
  MidPlan plan[MID_MAXPLAN];
  uint32_t nplan, L;
};

// Target constants of the conversion, in LDS.
struct MidTarget {
  uint64_t q;
  uint32_t qinv_neg;  // -q^-1 mod 2^32
  uint32_t pad_;
};
static_assert(sizeof(MidTarget) == 16, "mid_lds_bytes");

// Body for (poly, column) tile `tile` of a workgroup of nw waves (a multiple
// of 4), with mid_lds_bytes of lds.
template <int S1, int S2>
__device__ __forceinline__ void convert_mid_body(const MidArgs& a, const ModConst* __restrict__ mc,
                                                 const uint64_t* __restrict__ tw_inv,
                                                 const uint64_t* __restrict__ tw_fwd,
                                                 uint32_t tile, uint32_t nw, uint64_t* lds_dyn) {
  constexpr int M = 1 << S1, TPL = mid_lanes_per_line<S1>(), R = M / TPL;
  constexpr int RHO = R == 4 ? 2 : 3, LPW = 64 / TPL;
  constexpr int NSP = (S1 + RHO - 1) / RHO;
  constexpr uint32_t PITCH = mid_pitch<S1>(), N2 = 1u << S2;
  constexpr size_t N = (size_t)M << S2;
  static_assert(R * TPL == M && (1 << RHO) == R, "column split");
  const uint32_t nl = nw * LPW;
  const uint32_t p = tile / N2, col = tile % N2;
  const MidPlan& pl = a.plan[p % a.nplan];
  const uint32_t K = pl.nsrc, nq = pl.ndst;
  const uint64_t* const ext = a.src + (size_t)(p / a.nplan) * a.src_group_words +
                              (size_t)pl.src_limb0 * N;
  uint64_t* const y = a.out + (size_t)p * a.out_group_words;
  // The tables are read-only for the whole launch: reading them through the
  // constant address space lets uniform loads use the scalar cache, as for
  // kernel-argument tables.
  typedef const uint64_t __attribute__((address_space(4))) cu64;
  cu64* const src_scale = (cu64*)pl.src_scale;
  const uint32_t groups = (nq + 3) / 4;  // of four targets
  MidTarget* const tgt = reinterpret_cast<MidTarget*>(lds_dyn);
  uint64_t* const src = lds_dyn + (size_t)groups * 4 * (sizeof(MidTarget) / 8);
  uint64_t* const work = src + (size_t)K * PITCH;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63, sub = lane / TPL, tau = lane % TPL;
  const uint32_t first = wave * LPW + sub;
  auto target_mod = [&](uint32_t k, uint32_t& kpos) {
    kpos = k < pl.skip_at ? k : k + pl.skip_len;
    return kpos < pl.qlimbs ? kpos : a.L + (kpos - pl.qlimbs);
  };

  for (uint32_t k = threadIdx.x; k < 4 * groups; k += 64 * nw) {
    uint32_t kpos;
    const uint32_t m = target_mod(k < nq ? k : nq - 1, kpos);
    tgt[k] = MidTarget{mc[m].q, (uint32_t)mc[m].qinv_neg, 0};
  }

  // Inverse column stages of the source limbs; each limb is one line of src.
  for (uint32_t t = first; t < K; t += nl) {
    const uint32_t midx = pl.src_mod0 + t;
    const uint64_t q = mc[midx].q;
    const LazyMod lm = lazy_mod<16>(mc[midx]);
    const uint64_t* __restrict__ tw = tw_inv + (size_t)midx * N * 2;
    uint64_t* const line = src + (size_t)t * PITCH;
    uint64_t x[R], twx[2][R - 1], twy[2][R - 1];
    int bnd[R];  // bounds of x in q
    // First window (bits 0 .. RHO-1): rows R tau + v, one blocked run.
    const uint64_t* g = ext + (size_t)t * N + blocked_off<S2>(R * tau, col);
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
        for (int v = 0; v < R; ++v) x[v] = line[lds_idx(0, thi | ((uint32_t)v << w) | tlo, 0)];
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
        // v_t = x N^-1 [Q/q_t]^-1 mod q_t as balanced bytes: adding 128 to
        // every byte with carries leaves byte_a + 128 in byte a.
        const uint64_t f = src_scale[2 * t], fs = src_scale[2 * t + 1];
#pragma unroll
        for (int v = 0; v < R; ++v) {
          const uint64_t z = reduce_4q(shoup_acc(0, x[v], f, fs, lm.neg_q, lm.one), q);
          x[v] = (z + 0x8080808080808080ull) ^ 0x8080808080808080ull;
        }
      }
      wave_lds_sync();
#pragma unroll
      for (int v = 0; v < R; ++v) line[lds_idx(0, thi | ((uint32_t)v << w) | tlo, 0)] = x[v];
      wave_lds_sync();
    });
  }
  __syncthreads();

  // Batches of nl targets.  The conversion's work units are (four targets, 32
  // rows); each wave takes UPW consecutive ones of one group of four targets.
  constexpr uint32_t BLKS = M / 32, UPW = LPW * M / 128;
  static_assert(UPW >= 1 && BLKS % UPW == 0, "conversion units");
  typedef int v4i __attribute__((ext_vector_type(4)));
  typedef int v16i __attribute__((ext_vector_type(16)));
  typedef unsigned long long v2u __attribute__((ext_vector_type(2)));
  const uint32_t ksteps = (K + 3) / 4, half = lane >> 5, col32 = lane & 31;
  const uint32_t ugrp = wave * UPW / BLKS, ublk = wave * UPW % BLKS;
  uint64_t* const line = work + (size_t)first * PITCH;
  // 1 and 2^16 as values the compiler does not know: products with them are
  // multiply-adds that sign- or zero-extend their 32-bit operand for free.
  const int one = (int)mc[0].one, c16 = one << 16;
  // The units of one group of four targets from KS four-source steps.
  // Sources past K are lines of other data: they meet zero table bytes.
  auto convert = [&](auto ksc, uint32_t tg) {
    constexpr int KS = decltype(ksc)::value;
    const v4i* const tab = reinterpret_cast<const v4i*>(pl.bytes) + (size_t)tg * KS * 64 + lane;
    v4i ab[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) ab[ks] = tab[ks * 64];
    MidTarget mt[2];
#pragma unroll
    for (int o = 0; o < 2; ++o) mt[o] = tgt[4 * tg + 2 * half + o];
#pragma unroll
    for (uint32_t u = 0; u < UPW; ++u) {
      const uint32_t idx = lds_idx(0, 32 * (ublk + u) + col32, 0);
      const uint64_t* const sp = src + 2 * half * PITCH + idx;
      v16i acc = {};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const v2u sv = {sp[4 * ks * PITCH], sp[(4 * ks + 1) * PITCH]};
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(ab[ks], __builtin_bit_cast(v4i, sv), acc, 0,
                                                    0, 0);
      }
      uint64_t* const dst = work + (4 * ugrp + 2 * half) * PITCH + idx;
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        const int p01 = acc[8 * o] + (acc[8 * o + 1] << 8);
        const int p23 = acc[8 * o + 2] + (acc[8 * o + 3] << 8);
        const int p45 = acc[8 * o + 4] + (acc[8 * o + 5] << 8);
        const int p67 = acc[8 * o + 6] + (acc[8 * o + 7] << 8);
        // T = lo + 2^32 (hi - q);  m t = -lo mod 2^32, and the carry of lo +
        // m t out of its low word is that of m t + 2^32 - 1 (none for lo = 0)
        const int64_t lo = (int64_t)p01 * one + (int64_t)p23 * c16;
        int64_t hi = (int64_t)mt[o].q + (int64_t)p45 * one;
        hi += (int64_t)p67 * c16;
        const uint32_t q0 = (uint32_t)mt[o].q, q1 = (uint32_t)(mt[o].q >> 32);
        const uint32_t m = (uint32_t)lo * mt[o].qinv_neg;
        const uint64_t mq0 = (uint64_t)m * q0 + 0xffffffffull;
        uint64_t r = (uint64_t)(hi + (int64_t)(int32_t)(lo >> 32) * one);
        r += (mq0 >> 32) * (uint32_t)one;
        r += (uint64_t)m * q1;
        dst[o * PITCH] = r;
      }
    }
  };
  for (uint32_t k0 = 0; k0 < nq; k0 += nl) {
    const uint32_t tg = k0 / 4 + ugrp;
    if (tg < groups) {
      switch (ksteps) {
        case 1: convert(std::integral_constant<int, 1>{}, tg); break;
        case 2: convert(std::integral_constant<int, 2>{}, tg); break;
        case 3: convert(std::integral_constant<int, 3>{}, tg); break;
        default: convert(std::integral_constant<int, 4>{}, tg); break;
      }
    }
    const uint32_t k = k0 + first;
    uint32_t kpos;
    const uint32_t kmod = target_mod(k < nq ? k : nq - 1, kpos);
    const LazyMod lm = lazy_mod<16>(mc[kmod]);
    const uint64_t* __restrict__ tw = tw_fwd + (size_t)kmod * N * 2;
    uint64_t x[R], twx[2][R - 1], twy[2][R - 1];
    fetch_twiddles<S1, RHO, false, 0, LPW == 1>(tw, 1, tau, twx[0], twy[0]);
    __syncthreads();
    if (k < nq) {
      static_for<NSP>([&](auto spc) {
        constexpr int sp = decltype(spc)::value;
        using W = SubPass<S1, RHO, false, sp>;
        constexpr int w = W::w;
        const uint32_t thi = (tau >> w) << (w + RHO), tlo = tau & ((1u << w) - 1);
        if constexpr (sp + 1 < NSP)
          fetch_twiddles<S1, RHO, false, sp + 1, LPW == 1>(tw, 1, tau, twx[(sp + 1) & 1],
                                                           twy[(sp + 1) & 1]);
#pragma unroll
        for (int v = 0; v < R; ++v) x[v] = line[lds_idx(0, thi | ((uint32_t)v << w) | tlo, 0)];
#pragma unroll
        for (int k = RHO - 1; k >= 0; --k) {
          const int beta = w + k, d = 1 << k;
          if (beta > W::bhi) continue;
#pragma unroll
          for (int v = 0; v < R; ++v) {
            if (v & d) continue;
            const int ti = twiddle_at<RHO>(k, v);
            fwd_butterfly(x[v], x[v + d], twx[sp & 1][ti], twy[sp & 1][ti], lm,
                          fwd_reduces(16, 3, S1, beta));
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
      });
    }
    if (k0 + nl < nq) __syncthreads();  // the next batch overwrites the lines
  }
}

// Register budget: seven waves per SIMD (72 VGPRs, no spill) at N2 = 256 keep
// three workgroups on a CU: 1514 us for the 30-rotation step against 1530 at
// six and 1593 at eight (spills).
template <int S1, int S2>
__global__ void __launch_bounds__(64 * mid_max_waves(S1))
    __attribute__((amdgpu_waves_per_eu(mid_waves_per_simd(S1), 8)))
    k_convert_mid(const MidArgs a, const ModConst* __restrict__ mc,
                  const uint64_t* __restrict__ tw_inv, const uint64_t* __restrict__ tw_fwd) {
  extern __shared__ __align__(16) uint64_t lds_dyn[];
  // Tiles in XCD order: workgroup i runs on XCD i % 8, and each XCD takes a
  // contiguous range of (poly, column) tiles, so neighbouring columns, which
  // share cache lines of the blocked layout, meet in one L2.
  const uint32_t per = gridDim.x / 8;
  const uint32_t tile = (blockIdx.x % 8) * per + blockIdx.x / 8;
  convert_mid_body<S1, S2>(a, mc, tw_inv, tw_fwd, tile, blockDim.x / 64, lds_dyn);
}

template <int S1, int S2>
void launch_mid(Context& c, const char* name, const MidArgs& a, uint32_t npoly,
                uint32_t max_src, uint32_t max_dst) {
  const uint32_t tiles = npoly << S2;
  const uint32_t nw = mid_waves(S1, tiles, max_src, max_dst, c.lds_per_block);
  FHE_LAUNCH(c, name, (k_convert_mid<S1, S2>), dim3(tiles), dim3(64 * nw),
             mid_lds_bytes(S1, max_src, max_dst, nw), a, c.d_const, c.d_tw_inv, c.d_tw_fwd);
}

// The target order of `pl` must be the one MidPlan describes (checked).
MidPlan mid_plan(const Context& c, const ConvPlan& pl, uint32_t src_mod0, uint32_t src_limb0,
                 uint32_t skip_at, uint32_t skip_len, uint32_t qlimbs) {
  for (uint32_t k = 0; k < pl.ndst; ++k) {
    const uint32_t pos = k < skip_at ? k : k + skip_len;
    if (pl.dst_idx[k] != (pos < qlimbs ? pos : c.L + (pos - qlimbs)))
      throw ArgError("conversion plan target order");
  }
  return MidPlan{pl.d_src_scale, pl.d_bytes, pl.nsrc,  pl.ndst, src_mod0,
                 src_limb0,      skip_at,    skip_len, qlimbs};
}

bool mid_lds_fits(const Context& c, uint32_t nsrc, uint32_t ndst) {
  return c.log_n >= 13 && c.log_n <= 17 &&
         mid_lds_bytes((c.log_n + 1) / 2, nsrc, ndst, 4) <= c.lds_per_block;
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
  return nsrc <= MAX_CONV_SRC && below_2_60_all(c, nq) && mid_lds_fits(c, nsrc, nq + c.K);
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
  case LN: launch_mid<A, B>(c, "k_moddown_mid", a, npoly, c.K, nq); return;
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

static void modup_passes(Context& c, const uint64_t* const* as, uint32_t count, uint32_t nq,
                         uint64_t* digits, bool raw) {
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
    if (raw)                                                                                  \
      FHE_LAUNCH(c, "ntt_inv_blocks_modup", (ntt_pass_modup_in<B, false>),                    \
                 dim3(tiles, count, nq), dim3(256), 0, coef.p, (size_t)nq * n, c.d_const,     \
                 c.d_tw_inv, c.log_n, s1, sp, nullptr, c.alpha, nd, ne);                      \
    else                                                                                      \
      FHE_LAUNCH(c, "ntt_inv_blocks_modup", (ntt_pass_modup_in<B, true>),                     \
                 dim3(tiles, count, nq), dim3(256), 0, coef.p, (size_t)nq * n, c.d_const,     \
                 c.d_tw_inv, c.log_n, s1, sp, digits, c.alpha, nd, ne);                       \
    launch_mid<A, B>(c, "k_modup_mid", a, count * nd, max_src, nq + c.K);                     \
    if (!raw)                                                                                 \
      FHE_LAUNCH(c, "ntt_fwd_blocks_modup", (ntt_pass_modup_out<B>),                          \
                 dim3(tiles, count * nd, ne - w_last), dim3(256), 0, digits, (size_t)ne * n,  \
                 c.d_const, c.d_tw_fwd, c.log_n, map, s1);                                    \
    break;                                                                                    \
  }
    CASE(13, 7, 6) CASE(14, 7, 7) CASE(15, 8, 7) CASE(16, 8, 8) CASE(17, 9, 8)
#undef CASE
    default: throw ArgError("unsupported ring dimension");
  }
}

void modup_fused(Context& c, const uint64_t* const* as, uint32_t count, uint32_t nq,
                 uint64_t* digits) {
  modup_passes(c, as, count, nq, digits, false);
}
void modup_raw(Context& c, const uint64_t* const* as, uint32_t count, uint32_t nq,
               uint64_t* digits) {
  modup_passes(c, as, count, nq, digits, true);
}

}  // namespace fhe
