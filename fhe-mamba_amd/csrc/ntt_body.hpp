// Negacyclic RNS NTT / inverse NTT for gfx950.
//
// Forward transform = OpenFHE's ForwardTransformToBitReverseInPlace (the
// transform behind every FIDESlib NTT_ launch the reference makes,
// experiments/ntt_warp_tail/probe.cu:58-66): Cooley-Tukey stages with
// twiddles psi^brv(m+i), output slot i holding a(psi^(2 brv(i) + 1)).
// The inverse runs Gentleman-Sande stages with psi^-brv(m+i), then N^-1.
//
// Structure.  For N = 2^logN with logN >= 13 the transform is split into
// two launches over "lines":
//   COLS   line c in [0, N2): elements c + N2*u, u in [0, N1)  (stages that
//          pair elements at distance >= N2; S1 = ceil(logN/2) stages)
//   BLOCKS line b in [0, N1): elements b*N2 + u, u in [0, N2)  (the last
//          S2 = floor(logN/2) stages)
// Rings with logN <= 12 use one launch (SINGLE) per limb, radix 8.  Plain
// two-launch passes hold 16 elements a thread and run 4 stages at a time
// (radix 16), the passes fused with other work 8 and 3 (RHO_EPILOGUE);
// sub-passes exchange through an LDS tile padded by one word per 16 words,
// which keeps both the stride-1 and the stride-16 access patterns free of
// bank conflicts.  Workgroups are 256 threads (4096 elements and ~35 KB LDS
// at radix 16).
//
// What bounds a pass: over a large batch the memory path (64 ciphertexts x 2
// polys x 24 limbs at N=2^16: 3.22 GB a pass, 0.575 ms at the 5.6 TB/s of a
// plain copy, 0.65-0.8 ms measured), for one ciphertext the latency of a
// workgroup's chain of loads, exchanges and butterflies.
//
// Arithmetic: Harvey lazy butterflies on an approximate-quotient Shoup product
// whose bounds are tracked at compile time (fwd_butterfly, inv_butterfly and
// LIM in modarith.hpp); the final launch reduces to [0, q).
//
// Grid: (tiles per limb, poly, limb).  The limb index is the slowest grid
// dimension so consecutive workgroups share one modulus and its twiddle
// table stays hot in L2.
#pragma once

#include "launch_rules.hpp"
#include "ops.hpp"

#include <type_traits>
#include <utility>

namespace fhe {
namespace {

enum Kind { SINGLE = 0, COLS = 1, BLOCKS = 2 };

// RHO stages per sub-pass, radix 2^RHO per thread.  Plain passes are
// ALU-bound and use radix 16 (two sub-passes for 8 stages); the ModDown
// epilogue pass uses radix 8 in its two-launch form: half the LDS and
// registers per wave, so twice the waves to cover its extra global loads.
constexpr int RHO_PLAIN = 4, RHO_EPILOGUE = 3;
// One-launch rings (N <= 2^12) give a limb to one workgroup, so a launch is
// bound by that workgroup's chain of sub-passes: radix 8 over 512 lanes at
// N = 2^12, twice the waves of radix 16.
constexpr int RHO_SINGLE = 3;
template <int KIND>
constexpr int max_threads() {
  return KIND == SINGLE ? 1 << (12 - RHO_SINGLE) : 256;
}

template <int S, int RHO_>
struct Geo {
  static constexpr int RHO = RHO_;
  static constexpr int TPL = 1 << (S - RHO);  // threads per line
  static constexpr int LEN = 1 << S;
  static constexpr int PITCH = LEN + LEN / 16 + 1;
};

__device__ __forceinline__ uint32_t lds_idx(uint32_t line, uint32_t u, uint32_t pitch) {
  return line * pitch + u + (u >> 4);
}

// Base of launch poly p: data + p * poly_stride, or the table's entry for
// polys held in separate allocations.
template <class Map>
__device__ __forceinline__ uint64_t* poly_base(const Map&, uint64_t* data, size_t poly_stride,
                                               uint32_t p) {
  return data + (size_t)p * poly_stride;
}
__device__ __forceinline__ uint64_t* poly_base(const TableMap& m, uint64_t*, size_t, uint32_t p) {
  return m.table[p];
}

// Final stores go through `store.fin(base, offset_in_limb, value, t, q)`,
// with t = store.pre(offset_in_limb, q) when Store::kPre.
// The first pass's input comes from `load.get(offset_in_limb, q)` instead
// of data when Load::kLoad.
struct PlainLoad {
  static constexpr bool kLoad = false;
  __device__ __forceinline__ uint64_t get(size_t, uint64_t) const { return 0; }
};

// LDS writes of this wavefront before the call are seen by its reads after
// the call (LDS executes a wavefront's instructions in order; this keeps the
// compiler from moving accesses across).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// f(integral_constant 0) ... f(integral_constant N - 1): a loop whose index
// is a compile-time constant, so that the register arrays its body indexes
// by it stay registers.
template <class F, int... I>
__device__ __forceinline__ void static_for_seq(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_seq(std::make_integer_sequence<int, N>{}, f);
}

// Sub-pass SP of an S-stage pass: the window [w, w + RHO) of line-local index
// bits that a thread holds, and the stage bits [blo, bhi] done there.
template <int S, int RHO, bool INV, int SP>
struct SubPass {
  static constexpr int hi = S - RHO * SP, lo = RHO * SP;
  static constexpr int w = INV ? (lo + RHO <= S ? lo : S - RHO) : (hi >= RHO ? hi - RHO : 0);
  static constexpr int blo = INV ? lo : w;
  static constexpr int bhi = INV ? (lo + RHO <= S ? lo + RHO - 1 : S - 1) : hi - 1;
};

// The twiddle pairs of sub-pass SP for the thread tau of a line whose stage
// beta uses indices (twbase << (S - 1 - beta)) | (u >> (beta + 1)): stage
// beta's R >> (beta - w + 1) distinct pairs go to entries twiddle_at(beta - w,
// 0), ... .  In the window of the line's top stages they do not depend on tau;
// LINE_UNIFORM (every lane of the wavefront works on lines with one
// twbase) then reads them through the scalar cache.
template <int RHO>
__device__ __forceinline__ constexpr int twiddle_at(int k, int v) {
  return ((1 << RHO) >> (k + 1)) - 1 + (v >> (k + 1));
}
template <int S, int RHO, bool INV, int SP, bool LINE_UNIFORM>
__device__ __forceinline__ void fetch_twiddles(const uint64_t* __restrict__ tw, uint32_t twbase,
                                               uint32_t tau,
                                               uint64_t (&tx)[(1 << RHO) - 1],
                                               uint64_t (&ty)[(1 << RHO) - 1]) {
  using W = SubPass<S, RHO, INV, SP>;
  constexpr int R = 1 << RHO, w = W::w;
  const uint32_t thi = (tau >> w) << (w + RHO);
  constexpr bool scalar = LINE_UNIFORM && w + RHO >= S;
#pragma unroll
  for (int k = 0; k < RHO; ++k) {
#pragma unroll
    for (int g = 0; g < R / 2; ++g) {
      const int beta = w + k, at = twiddle_at<RHO>(k, g << (k + 1));
      if (g >= (R >> (k + 1)) || beta < W::blo || beta > W::bhi) continue;
      if (scalar) {
        typedef const uint64_t __attribute__((address_space(4))) cu64t;
        const uint32_t ti =
            __builtin_amdgcn_readfirstlane((twbase << (S - 1 - beta)) | (uint32_t)g);
        tx[at] = ((cu64t*)tw)[2 * ti];
        ty[at] = ((cu64t*)tw)[2 * ti + 1];
      } else {
        const uint32_t ti = (twbase << (S - 1 - beta)) | ((thi >> (beta + 1)) + (uint32_t)g);
        const ulonglong2 v = *reinterpret_cast<const ulonglong2*>(tw + 2 * ti);
        tx[at] = v.x;
        ty[at] = v.y;
      }
    }
  }
}

// Load::kBulk: bulk(g, x) forms a thread's R input values at once.
template <class Load, class = void>
struct bulk_load : std::false_type {};
template <class Load>
struct bulk_load<Load, std::enable_if_t<Load::kBulk>> : std::true_type {};

template <int LIM>
__device__ __forceinline__ LazyMod lazy_mod(const ModConst& m) {
  static_assert(LIM == 8 || LIM == 16, "lazy range");
  return LazyMod{4 * m.q, 8 * m.q, m.neg_q, LIM == 16 ? m.neg_q8 : m.neg_q4, m.one};
}

// BLK_IN / BLK_OUT (BLOCKS kind): the first pass's input / the last pass's
// output uses the blocked layout described with blocked_off below.  A
// workgroup's tile then still occupies the words [wg0, wg0 + LINES * LEN),
// in the order p = u * LINES + line, and is staged through LDS whatever the
// window.
//
// BLOCKS launches keep every line inside one wavefront (TPL <= 64 lanes, LPW
// = 64 / TPL lines per wave), so their sub-passes exchange through LDS with
// wavefront-level ordering only, and staging of a contiguous window is done
// per wavefront over its own lines (two adjacent words per lane, one
// 1024-byte run per instruction; 8-byte accesses measured 4% slower in the
// inverse block pass).  Only blocked-layout staging, which interleaves the
// lines of the whole workgroup word by word, keeps a workgroup barrier.
struct PlainStore;
template <int LIM, int S, int KIND, bool INV, int RHO_, class Store, class Load = PlainLoad,
          class Map = LimbMap, bool BLK_IN = false, bool BLK_OUT = false>
__device__ __forceinline__ void ntt_body(uint64_t* __restrict__ data, size_t poly_stride,
                                         const ModConst* __restrict__ mc,
                                         const uint64_t* __restrict__ tw_all, uint32_t log_n,
                                         Map map, uint32_t s_other, const Store& store, const Load& load = Load{}) {
  using G = Geo<S, RHO_>;
  constexpr int RHO = G::RHO;
  constexpr int R = 1 << RHO;
  constexpr int LINES = KIND == SINGLE ? 1 : 256 / G::TPL;
  constexpr int NSP = (S + RHO - 1) / RHO;
  __shared__ uint64_t lds[LINES * G::PITCH];

  const uint32_t n = 1u << log_n;
  // Workgroup-uniform: a slot without work exits before any barrier.
  uint32_t pos, midx;
  if (!map.resolve(blockIdx.y, blockIdx.z, pos, midx)) return;
  const uint64_t q = mc[midx].q;
  const LazyMod lm = lazy_mod<LIM>(mc[midx]);
  // Bound (in q) of this pass's input: below 4q (canonical in all the
  // library's own calls) for the first pass of a transform, else what the
  // first pass leaves.
  constexpr bool FIRST = KIND == SINGLE || (KIND == COLS) != INV;
  constexpr bool LAST = KIND == SINGLE || (KIND == COLS) == INV;
  constexpr int B0 = FIRST ? 4 : INV ? LIM / 2 : fwd_pass_bound(LIM);
  static_assert(INV || fwd_bound(LIM, B0, S, -1) <= fwd_pass_bound(LIM), "forward bound");
  const uint64_t* __restrict__ tw = tw_all + (size_t)midx * n * 2;
  uint64_t* __restrict__ base = poly_base(map, data, poly_stride, blockIdx.y) + (size_t)pos * n;

  const uint32_t tid = threadIdx.x;
  uint32_t line, tau;
  if (KIND == COLS) {
    line = tid % LINES;
    tau = tid / LINES;
  } else {
    tau = tid % G::TPL;
    line = tid / G::TPL;
  }
  const uint32_t gline = blockIdx.x * LINES + line;
  const uint32_t twbase = KIND == BLOCKS ? (1u << s_other) + gline : 1u;
  constexpr bool WL = KIND == BLOCKS;
  static_assert(!WL || G::TPL <= 64, "a block line spans one wavefront");
  // Staged position k of this thread: per wavefront (WL) or per workgroup.
  // PAIR (every BLOCKS launch): a lane stages two adjacent positions at a
  // time, so plain staged loads and stores are 16-byte accesses: staged
  // position k is
  // wave * 64R + (k / 2) * 128 + 2 * lane + k % 2.
  constexpr bool PAIR = WL;
  constexpr bool PLAIN_ST = std::is_same<Store, PlainStore>::value;
  auto staged = [&](int k) -> uint32_t {
    if (PAIR)
      return (tid >> 6) * (64u * R) + (uint32_t)(k >> 1) * 128u + 2 * (tid & 63) + (k & 1);
    return WL ? (tid >> 6) * (64u * R) + (uint32_t)k * 64u + (tid & 63)
              : (uint32_t)k * blockDim.x + tid;
  };
  auto sync_lines = [&]() {
    if (WL) wave_lds_sync();
    else __syncthreads();
  };

  uint64_t x[R];
  int bnd[R];  // bounds of x in q (compile-time values once unrolled)
  uint64_t pre[Store::kPre ? R : 1];

  // Twiddles are issued a sub-pass ahead where registers allow (radix 8, or a
  // current window whose own twiddles are scalar), else just before the exchange
  // that precedes their use: their latency is then paid once a sub-pass and
  // not once a butterfly (64-ciphertext batch at N=2^16, 24 limbs: column
  // passes 0.77 / 0.93 -> 0.66 / 0.72 ms).
  uint64_t twx[2][R - 1], twy[2][R - 1];
  auto fetch_tw = [&](auto sp) {
    constexpr int SP = decltype(sp)::value;
    fetch_twiddles<S, RHO, INV, SP, KIND != BLOCKS>(tw, twbase, tau, twx[SP & 1], twy[SP & 1]);
  };

  static_for<NSP>([&](auto spc) {
    constexpr int sp = decltype(spc)::value;
    using W = SubPass<S, RHO, INV, sp>;
    constexpr int w = W::w;
    const uint32_t thi = (tau >> w) << (w + RHO), tlo = tau & ((1u << w) - 1);
    // In BLOCKS / SINGLE launches a window at bit 0 gives each thread 16
    // consecutive words; global traffic for such a window goes through LDS
    // so that lanes touch consecutive addresses.
    constexpr bool contiguous = KIND != COLS && w == 0;
    if constexpr (sp == 0) fetch_tw(std::integral_constant<int, 0>{});

    if (sp == 0 && (contiguous || BLK_IN)) {
      const size_t wg0 = ((size_t)blockIdx.x * LINES) << S;
      if constexpr (PAIR && !Load::kLoad && !BLK_IN) {
#pragma unroll
        for (int k = 0; k < R; k += 2) {
          const uint32_t p = staged(k);
          const ulonglong2 v2 = *reinterpret_cast<const ulonglong2*>(base + wg0 + p);
          lds[lds_idx(p >> S, p & (G::LEN - 1), G::PITCH)] = v2.x;
          lds[lds_idx((p + 1) >> S, (p + 1) & (G::LEN - 1), G::PITCH)] = v2.y;
        }
      } else {
#pragma unroll
        for (int k = 0; k < R; ++k) {
          const uint32_t p = BLK_IN ? (uint32_t)k * blockDim.x + tid : staged(k);
          const uint32_t li = BLK_IN ? lds_idx(p % LINES, p / LINES, G::PITCH)
                                     : lds_idx(p >> S, p & (G::LEN - 1), G::PITCH);
          lds[li] = Load::kLoad ? load.get(wg0 + p, q) : base[wg0 + p];
        }
      }
      if (BLK_IN) __syncthreads();
      else sync_lines();
#pragma unroll
      for (int v = 0; v < R; ++v) {
        const uint32_t u = thi | ((uint32_t)v << w) | tlo;
        x[v] = lds[lds_idx(line, u, G::PITCH)];
      }
    } else if (sp == 0) {
      size_t g[R];
#pragma unroll
      for (int v = 0; v < R; ++v) {
        const uint32_t u = thi | ((uint32_t)v << w) | tlo;
        g[v] = KIND == COLS ? gline + ((size_t)u << s_other) : ((size_t)gline << S) + u;
      }
      if constexpr (bulk_load<Load>::value) {
        load.bulk(g, x);
      } else {
#pragma unroll
        for (int v = 0; v < R; ++v) x[v] = Load::kLoad ? load.get(g[v], q) : base[g[v]];
      }
    } else {
      sync_lines();
#pragma unroll
      for (int v = 0; v < R; ++v) {
        const uint32_t u = thi | ((uint32_t)v << w) | tlo;
        x[v] = lds[lds_idx(line, u, G::PITCH)];
      }
    }
    // Store-side terms for this thread's final positions, loaded ahead of the
    // butterflies: with the first sub-pass when the final window is
    // contiguous (staged positions do not depend on the window), else with
    // the last one.
    constexpr bool kFinalContig = !INV && KIND != COLS;
    if (Store::kPre && LAST && sp == (kFinalContig ? 0 : NSP - 1)) {
      const size_t wg0 = ((size_t)blockIdx.x * LINES) << S;
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const uint32_t u = thi | ((uint32_t)k << w) | tlo;
        const size_t g = kFinalContig ? wg0 + staged(k)
                         : KIND == COLS ? gline + ((size_t)u << s_other)
                                        : ((size_t)gline << S) + u;
        pre[Store::kPre ? k : 0] = store.pre(g, q);
      }
    }

    constexpr bool early = R <= 8 || (KIND != BLOCKS && w + RHO >= S);
    constexpr std::integral_constant<int, sp + 1> next{};
    if constexpr (sp + 1 < NSP && early) fetch_tw(next);

    if (!INV) {
#pragma unroll
      for (int k = RHO - 1; k >= 0; --k) {
        const int beta = w + k, d = 1 << k;
        if (beta > W::bhi) continue;
#pragma unroll
        for (int v = 0; v < R; ++v) {
          if (v & d) continue;
          const int ti = twiddle_at<RHO>(k, v);
          fwd_butterfly(x[v], x[v + d], twx[sp & 1][ti], twy[sp & 1][ti], lm,
                        fwd_reduces(LIM, B0, S, beta));
        }
      }
    } else {
      // Every element of a later sub-pass may be any of the previous one's.
#pragma unroll
      for (int v = 0; v < R; ++v) bnd[v] = sp == 0 ? B0 : LIM / 2;
#pragma unroll
      for (int k = 0; k < RHO; ++k) {
        const int beta = w + k, d = 1 << k;
        if (beta < W::blo || beta > W::bhi) continue;
#pragma unroll
        for (int v = 0; v < R; ++v) {
          if (v & d) continue;
          const int ti = twiddle_at<RHO>(k, v);
          const bool scaled = LAST && beta == S - 1;
          inv_butterfly(x[v], x[v + d], scaled ? mc[midx].wninv : twx[sp & 1][ti],
                        scaled ? mc[midx].wninv_sh : twy[sp & 1][ti], lm, LIM, bnd[v],
                        bnd[v + d]);
        }
      }
    }

    if (sp == NSP - 1) {
      if constexpr (LAST && !INV) {
#pragma unroll
        for (int v = 0; v < R; ++v)
          x[v] = LIM == 16 ? reduce_est(x[v], lm.neg_q, mc[midx].rq) : reduce_8q(x[v], q);
      }
      if constexpr (LAST && INV) {
        // N^-1: the last stage's products carry it in their twiddle, so only
        // its sums (the lower half of the window) are still to be scaled.
        const uint64_t ni = mc[midx].ninv, nis = mc[midx].ninv_sh;
#pragma unroll
        for (int v = 0; v < R; ++v) {
          if (v < R / 2) x[v] = shoup_acc(0, x[v], ni, nis, lm.neg_q, lm.one);
          x[v] = lazy_sub(lazy_sub(x[v], lm.neg_q + lm.neg_q), lm.neg_q);
        }
      }
      if (contiguous || BLK_OUT) {
        if (sp > 0 || NSP == 1) sync_lines();
#pragma unroll
        for (int v = 0; v < R; ++v) {
          const uint32_t u = thi | ((uint32_t)v << w) | tlo;
          lds[lds_idx(line, u, G::PITCH)] = x[v];
        }
        if (BLK_OUT) __syncthreads();
        else sync_lines();
        const size_t wg0 = ((size_t)blockIdx.x * LINES) << S;
        if constexpr (PAIR && PLAIN_ST && !BLK_OUT) {
#pragma unroll
          for (int k = 0; k < R; k += 2) {
            const uint32_t p = staged(k);
            *reinterpret_cast<ulonglong2*>(base + wg0 + p) =
                ulonglong2{lds[lds_idx(p >> S, p & (G::LEN - 1), G::PITCH)],
                           lds[lds_idx((p + 1) >> S, (p + 1) & (G::LEN - 1), G::PITCH)]};
          }
        } else {
#pragma unroll
          for (int k = 0; k < R; ++k) {
            const uint32_t p = BLK_OUT ? (uint32_t)k * blockDim.x + tid : staged(k);
            const uint32_t li = BLK_OUT ? lds_idx(p % LINES, p / LINES, G::PITCH)
                                        : lds_idx(p >> S, p & (G::LEN - 1), G::PITCH);
            store.fin(base, wg0 + p, lds[li], pre[Store::kPre ? k : 0], q);
          }
        }
      } else {
#pragma unroll
        for (int v = 0; v < R; ++v) {
          const uint32_t u = thi | ((uint32_t)v << w) | tlo;
          const size_t g =
              KIND == COLS ? gline + ((size_t)u << s_other) : ((size_t)gline << S) + u;
          store.fin(base, g, x[v], pre[Store::kPre ? v : 0], q);
        }
      }
    } else {
      if constexpr (sp + 1 < NSP && !early) fetch_tw(next);
      if (sp > 0 || (KIND != COLS && INV)) sync_lines();
#pragma unroll
      for (int v = 0; v < R; ++v) {
        const uint32_t u = thi | ((uint32_t)v << w) | tlo;
        lds[lds_idx(line, u, G::PITCH)] = x[v];
      }
    }
  });
}

// Store functors of the last pass.  kPre: the store adds a term t(s) that
// does not depend on the transform (pre), loaded for all of a thread's
// positions before the last sub-pass so its global loads overlap the
// butterflies; fin then writes f(y, t).
struct PlainStore {
  static constexpr bool kPre = false;
  __device__ __forceinline__ uint64_t pre(size_t, uint64_t) const { return 0; }
  __device__ __forceinline__ void fin(uint64_t* base, size_t g, uint64_t v, uint64_t,
                                      uint64_t) const {
    base[g] = v;
  }
};

__device__ __forceinline__ uint32_t brev_bits(uint32_t x, uint32_t bits) {
  return __brev(x) >> (32 - bits);
}

// Blocked limb layout of ModDown's intermediates (P limbs between the first
// inverse pass and the fused middle kernel, y between that kernel and the
// last forward pass).  With the split index s = b * N2 + u (row b < N1,
// column u < N2 = 2^S2), rows are grouped by BLO, the line count of a radix-8
// block-pass workgroup:
//   offset(b, u) = (b / BLO) * BLO * N2 + u * BLO + b % BLO.
// A block-pass workgroup (BLO consecutive rows, all columns) then touches
// one contiguous BLO * N2 run, and a column (all rows, one u) is N1 / BLO
// runs of BLO words.
template <int S2>
constexpr int blocked_rows() {
  return 256 >> (S2 - RHO_EPILOGUE);
}

template <int S2>
__device__ __forceinline__ size_t blocked_off(uint32_t b, uint32_t u) {
  constexpr uint32_t BLO = blocked_rows<S2>();
  return (size_t)(b / BLO) * ((size_t)BLO << S2) + (size_t)u * BLO + (b % BLO);
}

// Column lines in kernels that keep whole columns in LDS (launch_rules.hpp).
template <int S1>
constexpr uint32_t mid_pitch() {
  return column_pitch(S1);
}
template <int S1>
constexpr int mid_lanes_per_line() {
  return column_lanes(S1);
}

// ModUp input: limb blockIdx.z of ciphertext blockIdx.y's c1, read from the
// caller's polys (the first inverse pass reads them in place of a copy).
// Each word is read once by the pass, which also stores it as the word of
// its digit's own limb ([ct][d][ne][N], d = limb / alpha) when KEEP: the
// digits keep c1's own limbs as they are.
constexpr int MODUP_MAX_CT = 32;
template <bool KEEP>
struct SrcLoad {
  static constexpr bool kLoad = true;
  const uint64_t* const* src;  // MODUP_MAX_CT entries in kernel arguments
  uint32_t n;
  uint64_t* digits;
  uint32_t alpha, nd, ne;
  __device__ __forceinline__ uint64_t get(size_t g, uint64_t) const {
    const uint32_t ct = blockIdx.y, i = blockIdx.z;
    const uint64_t v = src[ct][(size_t)i * n + g];
    if (KEEP) digits[(((size_t)ct * nd + i / alpha) * ne + i) * n + g] = v;
    return v;
  }
};
struct SrcPtrs {
  const uint64_t* p[MODUP_MAX_CT];
};

// f(16) where every modulus of the context suits the wide lazy range, else
// f(8), as a compile-time constant.
template <class F>
void with_lim(const Context& c, F&& f) {
  if (c.lazy16)
    f(std::integral_constant<int, 16>{});
  else
    f(std::integral_constant<int, 8>{});
}

}  // namespace
}  // namespace fhe
