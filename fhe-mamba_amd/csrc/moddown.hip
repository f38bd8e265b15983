// ModDown: the P-limb key products with the first inverse pass, and the last
// forward pass with the key-product epilogue.
#include "key_product.hpp"

namespace fhe {
namespace {

// First inverse pass of ModDown fed by KskLoad.
// BLK: BLOCKS pass of the fused ModDown (moduli below 2^60), writing the
// blocked layout.
template <int LIM, int S, int ND, bool BLK>
__global__ void __launch_bounds__(256)
    ntt_pass_ksk(uint64_t* __restrict__ data, size_t poly_stride, const ModConst* __restrict__ mc,
                 const uint64_t* __restrict__ tw_all, uint32_t log_n, uint32_t s_other,
                 const ModDownEpi epi) {
  ntt_body<LIM, S, BLOCKS, true, RHO_EPILOGUE, PlainStore, KskLoad<ND>, LimbMap, false, BLK>(
      data, poly_stride, mc, tw_all, log_n, LimbMap::contiguous(epi.L), s_other, PlainStore{},
      KskLoad<ND>{epi, 1u << log_n});
}

// BLK: pass of the fused ModDown (moduli below 2^60), y read from the
// blocked layout.
template <int LIM, int S, int ND, bool BLK>
__global__ void __launch_bounds__(256)
    ntt_pass_moddown(uint64_t* __restrict__ data, size_t poly_stride,
                     const ModConst* __restrict__ mc, const uint64_t* __restrict__ tw_all,
                     uint32_t log_n, uint32_t s_other, const ModDownEpi epi) {
  ntt_body<LIM, S, BLOCKS, false, RHO_EPILOGUE, EpiStore<ND>, PlainLoad, LimbMap, BLK>(
      data, poly_stride, mc, tw_all, log_n, LimbMap::contiguous(0), s_other,
      EpiStore<ND>{epi, 1u << log_n, log_n});
}

// Last forward pass of a batched ModDown over the blocked y, both polys of
// each key switch in one workgroup (ND = 1..7 digits, every modulus in
// [2^33, 2^60)).  Eight wavefronts; lane tid holds the same R = 4 positions of row
// `line` in both polys (radix 4: one row per wavefront at N2 = 256, two or
// four at 128 / 64), so the digits' words and the twiddles are loaded once
// for both key products and both transforms, and the Galois target index is
// computed once for both stores.  The workgroup's rows are one blocked
// group (LINES = BLO).  Stage order, twiddle indices and lazy ranges are
// those of ntt_body's forward BLOCKS pass; the epilogue is EpiStore's:
// out_b[d(s)] = sum_j digit_j[s] key_j,b[s] (REDC) + add_b[s] + y_b[s].
// Lazy ranges: y arrives below 12q as from any forward pass and leaves the last
// stage below 12q; the key sum (redc_lazy, below 2q) plus the addend (below
// q) plus that is below 15q, reduced once by reduce_est.
// The key products are formed after the transform, with the stores: the
// butterflies then hold only the transform's values, and up to three digits
// the kernel fits 64 VGPRs, four 8-wave workgroups per CU (0.84 -> 0.80 ms
// for 30 key switches at N=2^16, 24 limbs, 3 digits, against forming them
// first and keeping them in registers).
//
// RAW: a key switch's own digits (modup_raw), whose last forward pass runs here
// too, two digits at a time through the same tile before y's; the finished
// words stay in registers for the products.  Each round's loads are issued
// ahead of the transform before them.  The digits' own pass over memory, and
// the copy of their own limbs, are gone; this kernel and the P-limb one stay
// bound by their reads, and by two 8-wave workgroups a CU (105-123 VGPRs;
// three with spills were 12-20% slower over the whole key switch).  N=2^16, us:
// relinearize + rescale of 37 limbs, 3 digits: the pass 41, ModDown's 52 + 24
// before; 0, 68 + 33 now; 6 rotations of 21 limbs, 2 digits: 95, 119 + 68
// before; 0, 150 + 107 now.
// Rows per workgroup of the paired passes (one blocked group) and the LDS
// words of their two-poly tile.
template <int S>
constexpr uint32_t pair_lines() {
  return 512u >> (S - 2);
}
template <int S>
constexpr uint32_t pair_lds_words() {
  return 2 * pair_lines<S>() * ((1u << S) + (1u << S) / 16 + 1);
}

// The forward block stages of H <= 2 blocked row groups src[h] (LINES rows)
// of one modulus, with shared twiddles: the groups, fetched by fetch_group,
// go to LDS, word p = u * LINES + row; the result, below 12q as from any pass,
// is left there, each wavefront's rows written by it.  next() issues the loads
// of what follows.  Every wavefront must be done with the tile before the call.
__device__ __forceinline__ void fetch_group(ulonglong2 (&v)[2], const uint64_t* src) {
#pragma unroll
  for (int k = 0; k < 2; ++k)
    v[k] = *reinterpret_cast<const ulonglong2*>(src + (uint32_t)k * 1024u + 2 * threadIdx.x);
}
template <int S, int H, class Next>
__device__ __forceinline__ void forward_groups(uint64_t* const (&lds)[2],
                                               const ulonglong2 (&in)[2][2], const Next& next,
                                               const uint64_t* __restrict__ tw, uint32_t twbase,
                                               uint32_t tau, uint32_t line, const LazyMod& lm) {
  constexpr int RHO = 2, R = 4, TPL = 1 << (S - RHO), LINES = 512 / TPL;
  constexpr int NSP = (S + RHO - 1) / RHO;
  constexpr uint32_t LEN = 1u << S, PITCH = LEN + LEN / 16 + 1;
  const uint32_t tid = threadIdx.x;
#pragma unroll
  for (int h = 0; h < H; ++h) {
#pragma unroll
    for (int k = 0; k < R; k += 2) {
      const uint32_t p = (uint32_t)k * 512u + 2 * tid;
      lds[h][lds_idx(p % LINES, p / LINES, PITCH)] = in[h][k / 2].x;
      lds[h][lds_idx((p + 1) % LINES, (p + 1) / LINES, PITCH)] = in[h][k / 2].y;
    }
  }
  __syncthreads();
  next();

  uint64_t x[H][R];
  uint64_t twx[2][R - 1], twy[2][R - 1];
  fetch_twiddles<S, RHO, false, 0, TPL == 64>(tw, twbase, tau, twx[0], twy[0]);
  static_for<NSP>([&](auto spc) {
    constexpr int sp = decltype(spc)::value;
    using W = SubPass<S, RHO, false, sp>;
    constexpr int w = W::w;
    const uint32_t thi = (tau >> w) << (w + RHO), tlo = tau & ((1u << w) - 1);
    if (sp > 0) wave_lds_sync();
#pragma unroll
    for (int v = 0; v < R; ++v) {
      const uint32_t u = thi | ((uint32_t)v << w) | tlo;
#pragma unroll
      for (int h = 0; h < H; ++h) x[h][v] = lds[h][lds_idx(line, u, PITCH)];
    }
    if constexpr (sp + 1 < NSP)
      fetch_twiddles<S, RHO, false, sp + 1, TPL == 64>(tw, twbase, tau, twx[(sp + 1) & 1],
                                                       twy[(sp + 1) & 1]);
#pragma unroll
    for (int k = RHO - 1; k >= 0; --k) {
      const int beta = w + k, d = 1 << k;
      if (beta > W::bhi) continue;
#pragma unroll
      for (int v = 0; v < R; ++v) {
        if (v & d) continue;
        const int ti = twiddle_at<RHO>(k, v);
        const uint64_t wv = twx[sp & 1][ti], ws = twy[sp & 1][ti];
#pragma unroll
        for (int h = 0; h < H; ++h)
          fwd_butterfly(x[h][v], x[h][v + d], wv, ws, lm,
                        fwd_reduces(16, fwd_pass_bound(16), S, beta));
      }
    }
    wave_lds_sync();
#pragma unroll
    for (int v = 0; v < R; ++v) {
      const uint32_t u = thi | ((uint32_t)v << w) | tlo;
#pragma unroll
      for (int h = 0; h < H; ++h) lds[h][lds_idx(line, u, PITCH)] = x[h][v];
    }
  });
  wave_lds_sync();
}

// Position k of lane tid in the workgroup's rows, as the key products and
// stores take them: two adjacent pairs in its wavefront's own run of rows.
__device__ __forceinline__ uint32_t pair_staged(uint32_t tid, int k) {
  return (tid >> 6) * 256u + (uint32_t)(k >> 1) * 128u + 2 * (tid & 63) + (k & 1);
}

// The last forward pass of M digits that ModUp left before it: dst[j] = words
// at positions pair_staged of digit j's group (src(j), blocked), reduced.  Two
// digits at a time through the tile, which the caller may overwrite on return.
template <int S, int M, class Src, class Next>
__device__ __forceinline__ void finish_digits(uint64_t* const (&lds)[2], ulonglong2 (&in)[2][2],
                                              const Src& src, const Next& next,
                                              const uint64_t* __restrict__ tw, uint32_t twbase,
                                              uint32_t tau, uint32_t line, const LazyMod& lm,
                                              float rq, ulonglong2 (&dst)[M][2]) {
  constexpr uint32_t LEN = 1u << S, PITCH = LEN + LEN / 16 + 1;
  static_for<(M + 1) / 2>([&](auto rd) {
    constexpr int j0 = 2 * decltype(rd)::value, H = M - j0 < 2 ? 1 : 2;
    if constexpr (j0 == 0) {
#pragma unroll
      for (int h = 0; h < H; ++h) fetch_group(in[h], src(h));
    }
    forward_groups<S, H>(
        lds, in,
        [&] {
          if constexpr (j0 + 2 >= M) {
            next();
          } else {
            constexpr int HN = M - j0 - 2 < 2 ? 1 : 2;
#pragma unroll
            for (int h = 0; h < HN; ++h) fetch_group(in[h], src(j0 + 2 + h));
          }
        },
        tw, twbase, tau, line, lm);
#pragma unroll
    for (int h = 0; h < H; ++h) {
#pragma unroll
      for (int k = 0; k < 4; k += 2) {
        const uint32_t p = pair_staged(threadIdx.x, k);
        dst[j0 + h][k / 2] = ulonglong2{
            reduce_est(lds[h][lds_idx(p >> S, p & (LEN - 1), PITCH)], lm.neg_q, rq),
            reduce_est(lds[h][lds_idx((p + 1) >> S, (p + 1) & (LEN - 1), PITCH)], lm.neg_q, rq)};
      }
    }
    __syncthreads();
  });
}

// Body of the paired epilogue for the workgroup at row group bx of limb i of
// key switch r, with its tile in lds (pair_lds_words<S>() words).
template <int S, int ND, bool RAW>
__device__ __forceinline__ void moddown_pair_body(const uint64_t* __restrict__ y,
                                                  const ModConst* __restrict__ mc,
                                                  const uint64_t* __restrict__ tw_all,
                                                  uint32_t log_n, uint32_t s_other,
                                                  const ModDownEpi& e, uint32_t bx, uint32_t r,
                                                  uint32_t i, uint64_t* lds_base) {
  constexpr int RHO = 2, R = 4, TPL = 1 << (S - RHO), LINES = 512 / TPL;
  constexpr uint32_t LEN = 1u << S, PITCH = LEN + LEN / 16 + 1;
  static_assert(TPL <= 64 && LINES * TPL == 512 && ND > 0 && ND <= 7, "pair epilogue");
  uint64_t* const lds[2] = {lds_base, lds_base + LINES * PITCH};
  const uint32_t n = 1u << log_n, tid = threadIdx.x;
  const uint64_t q = mc[i].q;
  const LazyMod lm = lazy_mod<16>(mc[i]);
  const float rq = mc[i].rq;
  const uint64_t* __restrict__ tw = tw_all + (size_t)i * n * 2;
  const size_t ps = (size_t)e.nq * n, wg0 = ((size_t)bx * LINES) << S;
  const uint32_t tau = tid % TPL, line = tid / TPL;
  const uint32_t twbase = (1u << s_other) + bx * LINES + line;
  // RAW: digit j's words are formed here from ModUp's intermediate (its own
  // limb, which needs no transform, comes from the source poly).  Slot j < M
  // holds the converted digits in order, the last slot the limb's own digit.
  constexpr int M = RAW ? ND - 1 : 0;
  const size_t dstride = (size_t)e.ne * n;
  const uint32_t own = RAW ? i / e.alpha : 0;
  auto digit_of = [&](int slot) -> uint32_t {
    return !RAW ? slot : slot == M ? own : (uint32_t)slot + ((uint32_t)slot >= own ? 1u : 0u);
  };
  ulonglong2 up[RAW && M > 0 ? M : 1][2];
  ulonglong2 in[2][2];
  auto fetch_y = [&] {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      fetch_group(in[h], y + (size_t)(2 * r + h) * ps + (size_t)i * n + wg0);
  };
  if constexpr (RAW && M > 0)
    finish_digits<S, M>(
        lds, in,
        [&](int j) { return e.digits[r] + digit_of(j) * dstride + (size_t)i * n + wg0; },
        fetch_y, tw, twbase, tau, line, lm, rq, up);
  else
    fetch_y();
  forward_groups<S, 2>(lds, in, [] {}, tw, twbase, tau, line, lm);

  // Key products of both polys at this lane's positions, the digits' words
  // read once (16-byte loads, two positions each), plus the transform, out
  // through the inverse Galois permutation.
  const uint32_t gi = e.ginv[r];
  uint64_t* const out0 = e.out[r] + (size_t)i * n;
  uint64_t* const out1 = e.out[r] + ((size_t)e.nq + i) * n;
  const size_t kstride = 2 * e.kl;
  const uint64_t* const a0 = e.add[r][0];
  const uint64_t* const a1 = e.add[r][1];
  const uint64_t qn = e.mc[i].qinv;
#pragma unroll
  for (int k = 0; k < R; k += 2) {
    const size_t s0 = wg0 + pair_staged(tid, k);
    const uint64_t* dg = (RAW ? e.own[r] : e.digits[r]) + (size_t)i * n + s0;
    const uint64_t* kr = e.key[r] + (size_t)i * n + s0;
    ulonglong2 d[ND], k0[ND], k1[ND];
#pragma unroll
    for (int j = 0; j < ND; ++j) {
      const uint64_t* kj = kr + digit_of(j) * kstride;
      if (j < M)
        d[j] = up[j < M ? j : 0][k / 2];
      else
        d[j] = *reinterpret_cast<const ulonglong2*>(dg + (RAW ? 0 : j * dstride));
      k0[j] = load_stream2(kj);
      k1[j] = load_stream2(kj + e.kl);
    }
    const ulonglong2 av = *reinterpret_cast<const ulonglong2*>(a0 ? a0 + (size_t)i * n + s0 : dg);
    uint64_t pre[2][2];
    key_comb2_lazy<ND>(d, k0, q, qn, pre[0][0], pre[0][1]);
    key_comb2_lazy<ND>(d, k1, q, qn, pre[1][0], pre[1][1]);
    if (a0) {
      pre[0][0] += av.x;
      pre[0][1] += av.y;
    }
    if (a1) {
      const ulonglong2 bv = *reinterpret_cast<const ulonglong2*>(a1 + (size_t)i * n + s0);
      pre[1][0] += bv.x;
      pre[1][1] += bv.y;
    }
    // Positions s (even) and s + 1 = s ^ 1 land on d(s) and d(s) ^ 1: the
    // automorphism maps brev(s) + N/2 to its image plus N/2 (mod N), so the
    // pair stays an aligned pair, swapped when d(s) is odd (16-byte stores).
    const uint32_t p = pair_staged(tid, k);
    const uint32_t s = (uint32_t)wg0 + p;
    uint32_t dst = s;
    if (gi != 1) {
      // 32-bit wrap-around is exact here: only the product mod 2N matters.
      const uint32_t jj = brev_bits(s, log_n);
      const uint32_t ex = ((2u * jj + 1u) * gi) & (2u * n - 1u);
      dst = brev_bits((ex - 1u) >> 1, log_n);
    }
    const uint32_t l0 = lds_idx(p >> S, p & (LEN - 1), PITCH);
    const uint32_t l1 = lds_idx((p + 1) >> S, (p + 1) & (LEN - 1), PITCH);
    const uint64_t a0v = reduce_est(pre[0][0] + lds[0][l0], lm.neg_q, rq);
    const uint64_t a1v = reduce_est(pre[0][1] + lds[0][l1], lm.neg_q, rq);
    const uint64_t b0v = reduce_est(pre[1][0] + lds[1][l0], lm.neg_q, rq);
    const uint64_t b1v = reduce_est(pre[1][1] + lds[1][l1], lm.neg_q, rq);
    const bool odd = dst & 1u;
    const size_t d2 = dst & ~1u;
    *reinterpret_cast<ulonglong2*>(out0 + d2) = odd ? ulonglong2{a1v, a0v} : ulonglong2{a0v, a1v};
    *reinterpret_cast<ulonglong2*>(out1 + d2) = odd ? ulonglong2{b1v, b0v} : ulonglong2{b0v, b1v};
  }
}

template <int S, int ND, bool RAW>
__global__ void __launch_bounds__(512)
    __attribute__((amdgpu_waves_per_eu(RAW                 ? 4
                                       : ND <= 3 && S >= 7 ? 6
                                       : ND == 4 && S >= 7 ? 8
                                                           : 1,
                                       8)))
    ntt_pass_moddown_pair(const uint64_t* __restrict__ y, const ModConst* __restrict__ mc,
                          const uint64_t* __restrict__ tw_all, uint32_t log_n, uint32_t s_other,
                          const ModDownEpi e) {
  __shared__ uint64_t lds[pair_lds_words<S>()];
  moddown_pair_body<S, ND, RAW>(y, mc, tw_all, log_n, s_other, e, blockIdx.x, blockIdx.y, blockIdx.z,
                           lds);
}

// First inverse pass of a batched ModDown with both polys of each key
// switch in one workgroup (the counterpart of ntt_pass_moddown_pair; ND =
// 1..7 digits, every modulus below 2^60): lane tid forms the P-limb key
// products of both polys at the same positions, the digits' words read
// once, runs the first S2 inverse stages of both polys with shared
// twiddles, and the workgroup stores its rows (one blocked group) to the
// blocked layout, below 8q; N^-1 is applied later.
// Up to three digits it fits 64 VGPRs without spills, so four 8-wave
// workgroups share a CU (LDS allows four; measured 2% faster than three at
// N=2^16, 24 limbs).
// Body for the workgroup at row group bx of P limb t of key switch r, with
// its tile in lds (pair_lds_words<S>() words).
template <int S, int ND, bool RAW>
__device__ __forceinline__ void ksk_pair_body(uint64_t* __restrict__ ext, size_t ps,
                                              const ModConst* __restrict__ mc,
                                              const uint64_t* __restrict__ tw_all,
                                              const uint64_t* __restrict__ tw_fwd, uint32_t log_n,
                                              uint32_t s_other, const ModDownEpi& e, uint32_t bx,
                                              uint32_t r, uint32_t t, uint64_t* lds_base) {
  constexpr int RHO = 2, R = 4, TPL = 1 << (S - RHO), LINES = 512 / TPL;
  constexpr int NSP = (S + RHO - 1) / RHO;
  constexpr uint32_t LEN = 1u << S, PITCH = LEN + LEN / 16 + 1;
  static_assert(TPL <= 64 && LINES * TPL == 512 && ND > 0 && ND <= 7, "pair ksk pass");
  uint64_t* const lds[2] = {lds_base, lds_base + LINES * PITCH};
  const uint32_t n = 1u << log_n, tid = threadIdx.x;
  const uint32_t midx = e.L + t;
  const uint64_t q = mc[midx].q;
  const LazyMod lm = lazy_mod<16>(mc[midx]);
  const uint64_t* __restrict__ tw = tw_all + (size_t)midx * n * 2;
  const size_t wg0 = ((size_t)bx * LINES) << S;
  const uint32_t tau = tid % TPL, line = tid / TPL;
  const uint32_t twbase = (1u << s_other) + bx * LINES + line;
  // RAW: the digits' last forward pass, here and not in a pass of its own.
  const size_t dstride = (size_t)e.ne * n;
  ulonglong2 up[RAW ? ND : 1][2];
  ulonglong2 in[2][2];
  if constexpr (RAW)
    finish_digits<S, ND>(
        lds, in,
        [&](int j) { return e.digits[r] + j * dstride + (size_t)(e.nq + t) * n + wg0; }, [] {},
        tw_fwd + (size_t)midx * n * 2, twbase, tau, line, lm, mc[midx].rq, up);

  // P-limb key products of both polys into LDS (this wavefront's rows), in
  // (0, 2q) as the first inverse stage accepts them.
  {
    const size_t kstride = 2 * e.kl;
    const uint64_t qn = e.mc[midx].qinv;
#pragma unroll
    for (int k = 0; k < R; k += 2) {
      const uint32_t p = pair_staged(tid, k);
      const size_t s = wg0 + p;
      const uint64_t* dg = e.digits[r] + (size_t)(e.nq + t) * n + s;
      const uint64_t* kr = e.key[r] + (size_t)midx * n + s;
      ulonglong2 d[ND], k0[ND], k1[ND];
#pragma unroll
      for (int j = 0; j < ND; ++j) {
        d[j] = RAW ? up[RAW ? j : 0][k / 2]
                   : *reinterpret_cast<const ulonglong2*>(dg + j * dstride);
        k0[j] = load_stream2(kr + j * kstride);
        k1[j] = load_stream2(kr + e.kl + j * kstride);
      }
      uint64_t v0, v1;
      const uint32_t l0 = lds_idx(p >> S, p & (LEN - 1), PITCH);
      const uint32_t l1 = lds_idx((p + 1) >> S, (p + 1) & (LEN - 1), PITCH);
      key_comb2_lazy<ND>(d, k0, q, qn, v0, v1);
      lds[0][l0] = v0;
      lds[0][l1] = v1;
      key_comb2_lazy<ND>(d, k1, q, qn, v0, v1);
      lds[1][l0] = v0;
      lds[1][l1] = v1;
    }
  }

  uint64_t x[2][R];
  int bnd[2][R];  // bounds of x in q
  uint64_t twx[2][R - 1], twy[2][R - 1];
  fetch_twiddles<S, RHO, true, 0, TPL == 64>(tw, twbase, tau, twx[0], twy[0]);
  static_for<NSP>([&](auto spc) {
    constexpr int sp = decltype(spc)::value;
    using W = SubPass<S, RHO, true, sp>;
    constexpr int w = W::w;
    const uint32_t thi = (tau >> w) << (w + RHO), tlo = tau & ((1u << w) - 1);
    wave_lds_sync();
#pragma unroll
    for (int v = 0; v < R; ++v) {
      const uint32_t u = thi | ((uint32_t)v << w) | tlo;
      x[0][v] = lds[0][lds_idx(line, u, PITCH)];
      x[1][v] = lds[1][lds_idx(line, u, PITCH)];
      bnd[0][v] = bnd[1][v] = sp == 0 ? 2 : 8;
    }
    if constexpr (sp + 1 < NSP)
      fetch_twiddles<S, RHO, true, sp + 1, TPL == 64>(tw, twbase, tau, twx[(sp + 1) & 1],
                                                      twy[(sp + 1) & 1]);
#pragma unroll
    for (int k = 0; k < RHO; ++k) {
      const int beta = w + k, d = 1 << k;
      if (beta < W::blo || beta > W::bhi) continue;
#pragma unroll
      for (int v = 0; v < R; ++v) {
        if (v & d) continue;
        const int ti = twiddle_at<RHO>(k, v);
        const uint64_t wv = twx[sp & 1][ti], ws = twy[sp & 1][ti];
#pragma unroll
        for (int h = 0; h < 2; ++h)
          inv_butterfly(x[h][v], x[h][v + d], wv, ws, lm, 16, bnd[h][v], bnd[h][v + d]);
      }
    }
    wave_lds_sync();
#pragma unroll
    for (int v = 0; v < R; ++v) {
      const uint32_t u = thi | ((uint32_t)v << w) | tlo;
      lds[0][lds_idx(line, u, PITCH)] = x[0][v];
      lds[1][lds_idx(line, u, PITCH)] = x[1][v];
    }
  });
  __syncthreads();

  // The blocked group of both polys, word p = u * LINES + row, two adjacent
  // words per lane (16-byte stores).
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    uint64_t* __restrict__ dst = ext + (size_t)(2 * r + h) * ps + (size_t)t * n + wg0;
#pragma unroll
    for (int k = 0; k < R; k += 2) {
      const uint32_t p = (uint32_t)k * 512u + 2 * tid;
      *reinterpret_cast<ulonglong2*>(dst + p) =
          ulonglong2{lds[h][lds_idx(p % LINES, p / LINES, PITCH)],
                     lds[h][lds_idx((p + 1) % LINES, (p + 1) / LINES, PITCH)]};
    }
  }
}

template <int S, int ND, bool RAW>
__global__ void __launch_bounds__(512)
    __attribute__((amdgpu_waves_per_eu(RAW ? 4 : ND <= 4 ? 8 : 1, 8)))
    ntt_pass_ksk_pair(uint64_t* __restrict__ ext, size_t ps, const ModConst* __restrict__ mc,
                      const uint64_t* __restrict__ tw_all, const uint64_t* __restrict__ tw_fwd,
                      uint32_t log_n, uint32_t s_other, const ModDownEpi e) {
  __shared__ uint64_t lds[pair_lds_words<S>()];
  ksk_pair_body<S, ND, RAW>(ext, ps, mc, tw_all, tw_fwd, log_n, s_other, e, blockIdx.x, blockIdx.y,
                            blockIdx.z, lds);
}

// f(LIM): the blocked form belongs to the fused ModDown, whose moduli all suit
// the wide lazy range.
template <bool BLK, class F>
void with_pass_lim(const Context& c, F&& f) {
  if constexpr (BLK)
    f(std::integral_constant<int, 16>{});
  else
    with_lim(c, f);
}

// npoly is even: polys 2 r and 2 r + 1 belong to key switch r.
template <int S, bool BLK = false>
void launch_moddown(Context& c, uint64_t* y, uint32_t npoly, uint32_t nq, uint32_t s_other,
                    const ModDownEpi& epi) {
  using G = Geo<S, RHO_EPILOGUE>;
  const uint32_t tiles = (1u << s_other) / (256 / G::TPL);
  const char* name = "ntt_fwd_blocks_moddown";
  if constexpr (BLK) {
    // Both polys of each key switch in one workgroup (blocked y, digits
    // 1..7): rows per workgroup = one blocked group.
    const dim3 grid((1u << s_other) / pair_lines<S>(), npoly / 2, nq);
#define CASE(D, RAW)                                                                         \
  case D:                                                                                    \
    FHE_LAUNCH(c, name, (ntt_pass_moddown_pair<S, D, RAW>), grid, dim3(512), 0, y, c.d_const, \
               c.d_tw_fwd, c.log_n, s_other, epi);                                           \
    return;
    if (epi.raw) {
      switch (epi.nd) {
        CASE(1, true) CASE(2, true) CASE(3, true) CASE(4, true)
      }
    } else {
      switch (epi.nd) {
        CASE(1, false) CASE(2, false) CASE(3, false) CASE(4, false) CASE(5, false)
        CASE(6, false) CASE(7, false)
      }
    }
#undef CASE
  }
  with_digits<!BLK>(epi.nd, [&](auto nd) {  // blocked: eight digits
    with_pass_lim<BLK>(c, [&](auto lim) {
      FHE_LAUNCH(c, name, (ntt_pass_moddown<decltype(lim)::value, S, decltype(nd)::value, BLK>),
                 dim3(tiles, npoly, nq), dim3(256), 0, y, (size_t)nq * c.n, c.d_const,
                 c.d_tw_fwd, c.log_n, s_other, epi);
    });
  });
}

template <int S, bool BLK = false>
void launch_ksk(Context& c, uint64_t* ext, uint32_t npoly, uint32_t s_other,
                const ModDownEpi& epi) {
  using G = Geo<S, RHO_EPILOGUE>;
  const uint32_t tiles = (1u << s_other) / (256 / G::TPL);
  const char* name = "ntt_inv_blocks_ksk";
  const size_t ps = (size_t)c.K * c.n;
  if constexpr (BLK) {
    // Both polys of each key switch in one workgroup (blocked output, digits
    // 1..7, no final scaling): rows per workgroup = one blocked group.
    const dim3 grid((1u << s_other) / pair_lines<S>(), npoly / 2, c.K);
#define CASE(D, RAW)                                                                        \
  case D:                                                                                   \
    FHE_LAUNCH(c, name, (ntt_pass_ksk_pair<S, D, RAW>), grid, dim3(512), 0, ext, ps,        \
               c.d_const, c.d_tw_inv, c.d_tw_fwd, c.log_n, s_other, epi);                   \
    return;
    if (epi.raw) {
      switch (epi.nd) {
        CASE(1, true) CASE(2, true) CASE(3, true) CASE(4, true)
      }
    } else {
      switch (epi.nd) {
        CASE(1, false) CASE(2, false) CASE(3, false) CASE(4, false) CASE(5, false)
        CASE(6, false) CASE(7, false)
      }
    }
#undef CASE
  }
  with_digits<!BLK>(epi.nd, [&](auto nd) {  // blocked: eight digits
    with_pass_lim<BLK>(c, [&](auto lim) {
      FHE_LAUNCH(c, name, (ntt_pass_ksk<decltype(lim)::value, S, decltype(nd)::value, BLK>),
                 dim3(tiles, npoly, c.K), dim3(256), 0, ext, ps, c.d_const, c.d_tw_inv, c.log_n,
                 s_other, epi);
    });
  });
}

}  // namespace

bool moddown_fused_ok(const Context& c, uint32_t nq) {
  if (c.log_n < 13 || c.log_n > 17 || c.K == 0 || c.K > 16) return false;
  if (nq == 0 || nq > c.L) return false;
  return convert_mid_ok(c, nq, c.K);
}

void moddown_fused(Context& c, uint64_t* ext_p, uint64_t* y, uint32_t npoly, uint32_t nq,
                   const ConvPlan& pl, const ModDownEpi& epi) {
  if (npoly == 0) return;
  if (npoly > 2 * MAX_KS_BATCH) throw ArgError("ModDown batch too large");
  if (!moddown_fused_ok(c, nq)) throw ArgError("fused ModDown does not apply");
  if (npoly % 2) throw ArgError("ModDown takes both polys of each key switch");
  if (epi.raw && epi.nd > RAW_MAX_DIGITS)
    throw ArgError("digits without their last pass do not apply");
  const uint32_t s1 = (c.log_n + 1) / 2;
  switch (c.log_n) {
#define CASE(LN, B)                                                \
  case LN:                                                         \
    launch_ksk<B, true>(c, ext_p, npoly, s1, epi);         \
    moddown_mid(c, ext_p, y, npoly, nq, pl);                       \
    launch_moddown<B, true>(c, y, npoly, nq, s1, epi);     \
    return;
    CASE(13, 6) CASE(14, 7) CASE(15, 7) CASE(16, 8) CASE(17, 8)
#undef CASE
    default: throw ArgError("unsupported ring dimension");
  }
}

void ntt_inverse_ksk(Context& c, uint64_t* ext_p, uint32_t npoly, const ModDownEpi& epi) {
  if (npoly == 0 || c.K == 0) return;
  if (npoly > 2 * MAX_KS_BATCH) throw ArgError("key-switch batch too large");
  if (c.log_n <= 12) {
    small_ring_ksk(c, ext_p, npoly, epi);
    return;
  }
  const uint32_t s1 = (c.log_n + 1) / 2, s2 = c.log_n / 2;
  switch (s2) {
#define CASE(S) \
  case S: launch_ksk<S>(c, ext_p, npoly, s1, epi); break;
    CASE(6) CASE(7) CASE(8)
#undef CASE
    default: throw ArgError("unsupported block pass");
  }
  ntt_cols(c, ext_p, npoly, (size_t)c.K * c.n, c.K, LimbMap::contiguous(c.L), true);
}

void ntt_forward_moddown(Context& c, uint64_t* y, uint32_t npoly, uint32_t nq,
                         const ModDownEpi& epi) {
  if (npoly == 0 || nq == 0) return;
  if (npoly > 2 * MAX_KS_BATCH) throw ArgError("ModDown batch too large");
  if (c.log_n <= 12) {
    small_ring_moddown(c, y, npoly, nq, epi);
    return;
  }
  const uint32_t s1 = (c.log_n + 1) / 2, s2 = c.log_n / 2;
  ntt_cols(c, y, npoly, (size_t)nq * c.n, nq, LimbMap::contiguous(0), false);
  switch (s2) {
#define CASE(S) \
  case S: launch_moddown<S>(c, y, npoly, nq, s1, epi); return;
    CASE(6) CASE(7) CASE(8)
#undef CASE
    default: throw ArgError("unsupported block pass");
  }
}

}  // namespace fhe
