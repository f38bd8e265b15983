// The key inner product as the input of ModDown's first inverse pass
// (KskLoad) and as the epilogue of its last forward pass (EpiStore).
#pragma once

#include "ntt_body.hpp"

namespace fhe {
namespace {

// Switching-key words are read once per launch: their loads are marked
// non-temporal so that they do not displace the digits, which every key
// switch of the batch re-reads, from the caches (measured ~1% faster on the
// ModDown passes; non-temporal stores of the outputs were slower).
__device__ __forceinline__ uint64_t load_stream(const uint64_t* p) {
  return __builtin_nontemporal_load(p);
}
__device__ __forceinline__ ulonglong2 load_stream2(const uint64_t* p) {
  typedef unsigned long long v2u __attribute__((ext_vector_type(2)));
  const v2u v = __builtin_nontemporal_load(reinterpret_cast<const v2u*>(p));
  ulonglong2 r;
  r.x = v.x;
  r.y = v.y;
  return r;
}

// Key inner product sum_j d_j k_j reduced once by REDC (keys in Montgomery
// form).
template <int ND>
__device__ __forceinline__ uint64_t key_dot(const uint64_t* dg, size_t dstride, const uint64_t* kr,
                                            size_t kstride, uint32_t nd_rt, uint64_t q,
                                            uint64_t qinv_neg) {
  Acc128 acc;
  if (ND > 0) {
#pragma unroll
    for (int j = 0; j < ND; ++j) acc.mac(dg[j * dstride], load_stream(kr + j * kstride));
  } else {
    for (uint32_t j = 0; j < nd_rt; ++j) acc.mac(dg[j * dstride], load_stream(kr + j * kstride));
  }
  return redc(acc.hi, acc.lo, q, qinv_neg);
}

// The sums of two adjacent positions, every modulus below 2^60 and 1 .. 7
// digits: operands split at bit 30 and accumulated carry-free in three 64-bit
// sums with v_mad_u64_u32, T = a0 + a1 2^30 + a2 2^60.  The reduction is left
// lazy, each sum in (0, 2q) (T < nd q^2 keeps T's high word below q for nd q <
// 2^64).
template <int ND>
__device__ __forceinline__ void key_comb2_lazy(const ulonglong2* d, const ulonglong2* k,
                                               uint64_t q, uint64_t qinv, uint64_t& t0,
                                               uint64_t& t1) {
  static_assert(ND > 0 && ND <= 7, "split key products");
  constexpr uint32_t M30 = (1u << 30) - 1;
  uint64_t a0[2] = {0, 0}, a1[2] = {0, 0}, a2[2] = {0, 0};
#pragma unroll
  for (int j = 0; j < ND; ++j) {
    const uint64_t dd[2] = {d[j].x, d[j].y}, kk[2] = {k[j].x, k[j].y};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t dl = (uint32_t)dd[h] & M30, dh = (uint32_t)(dd[h] >> 30);
      const uint32_t kl = (uint32_t)kk[h] & M30, kh = (uint32_t)(kk[h] >> 30);
      a0[h] += (uint64_t)dl * kl;
      a1[h] += (uint64_t)dl * kh;
      a1[h] += (uint64_t)dh * kl;
      a2[h] += (uint64_t)dh * kh;
    }
  }
  uint64_t t[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint64_t m1 = a1[h] << 30, m2 = a2[h] << 60;
    const uint64_t lo = a0[h] + m1;
    uint64_t hi = (a1[h] >> 34) + (a2[h] >> 4) + (lo < m1);
    const uint64_t lo2 = lo + m2;
    hi += lo2 < m2;
    t[h] = redc_lazy(hi, lo2, q, qinv);
  }
  t0 = t[0];
  t1 = t[1];
}

// ModDown epilogue (see ModDownEpi): the value at evaluation slot s goes to
// slot d(s) of the output, d being the inverse Galois permutation.  ND > 0
// fixes the digit count at compile time (ND = 0: e.nd at run time).
template <int ND>
struct EpiStore {
  static constexpr bool kPre = true;
  const ModDownEpi& e;
  uint32_t n, log_n;
  // Q-limb key inner product plus the addend at position s.
  __device__ __forceinline__ uint64_t pre(size_t s, uint64_t q) const {
    const uint32_t p = blockIdx.y, r = p >> 1, b = p & 1, i = blockIdx.z;
    const uint64_t* dg = e.digits[r] + (size_t)i * n + s;
    const uint64_t* kr = e.key[r] + (size_t)b * e.kl + (size_t)i * n + s;
    const size_t dstride = (size_t)e.ne * n, kstride = 2 * e.kl;
    uint64_t t = key_dot<ND>(dg, dstride, kr, kstride, e.nd, q, e.mc[i].qinv_neg);
    const uint64_t* add = e.add[r][b];
    if (add) t = add_mod(t, add[(size_t)i * n + s], q);
    return t;
  }
  __device__ __forceinline__ void fin(uint64_t*, size_t s, uint64_t y, uint64_t t,
                                      uint64_t q) const {
    const uint32_t p = blockIdx.y, r = p >> 1, b = p & 1, i = blockIdx.z;
    const uint64_t res = add_mod(t, y, q);
    uint32_t d = (uint32_t)s;
    const uint32_t gi = e.ginv[r];
    if (gi != 1) {
      // 32-bit wrap-around is exact here: only the product mod 2N matters.
      const uint32_t j = brev_bits((uint32_t)s, log_n);
      const uint32_t ex = ((2u * j + 1u) * gi) & (2u * n - 1u);
      d = brev_bits((ex - 1u) >> 1, log_n);
    }
    e.out[r][((size_t)b * e.nq + i) * n + d] = res;
  }
};

// P-limb key inner product as the input of ModDown's inverse NTT: launch
// poly p is key switch r = p / 2, component b = p % 2, limb t is P limb t.
template <int ND>
struct KskLoad {
  static constexpr bool kLoad = true;
  const ModDownEpi& e;
  uint32_t n;
  __device__ __forceinline__ uint64_t get(size_t s, uint64_t q) const {
    const uint32_t p = blockIdx.y, r = p >> 1, b = p & 1, t = blockIdx.z;
    const uint64_t* dg = e.digits[r] + (size_t)(e.nq + t) * n + s;
    const uint64_t* kr = e.key[r] + (size_t)b * e.kl + (size_t)(e.L + t) * n + s;
    const size_t dstride = (size_t)e.ne * n, kstride = 2 * e.kl;
    return key_dot<ND>(dg, dstride, kr, kstride, e.nd, q, e.mc[e.L + t].qinv_neg);
  }
};

// f(ND): the digit counts with kernels of their own when FIXED, 0 (run time)
// for the others.
template <bool FIXED, class F>
void with_digits(uint32_t nd, F&& f) {
  if constexpr (FIXED) {
    switch (nd) {
      case 1: f(std::integral_constant<int, 1>{}); return;
      case 2: f(std::integral_constant<int, 2>{}); return;
      case 3: f(std::integral_constant<int, 3>{}); return;
      default: break;
    }
  }
  f(std::integral_constant<int, 0>{});
}

}  // namespace
}  // namespace fhe
