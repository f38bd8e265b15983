// Load and store functors of the rescale's passes.  One launch set rescales
// up to RESCALE_MAX inputs of npoly polys each: launch poly y is poly y %
// npoly of input y / npoly, whose addresses come from a table in the kernel
// arguments.
#pragma once

#include <algorithm>

#include "ntt_body.hpp"

namespace fhe {
namespace {

constexpr int RESCALE_MAX = 16;
struct RescalePtrs {
  const uint64_t* a[RESCALE_MAX];
  uint64_t* out[RESCALE_MAX];
};
struct LastLimbLoad {
  static constexpr bool kLoad = true;
  const uint64_t* const* a;  // RESCALE_MAX entries in kernel arguments
  uint32_t npoly;
  size_t poly_words, last_off;
  __device__ __forceinline__ uint64_t get(size_t g, uint64_t) const {
    const uint32_t y = blockIdx.y;
    return a[y / npoly][(size_t)(y % npoly) * poly_words + last_off + g];
  }
};
struct LiftLoad {
  static constexpr bool kLoad = true;
  const uint64_t* last;  // [npoly][N], coefficient form mod q_l, in [0, q_l)
  const ModConst* mc;
  const uint64_t* rs;
  uint32_t n, l, L;
  uint64_t half;         // q_l >> 1
  __device__ __forceinline__ uint64_t get(size_t g, uint64_t q) const {
    const uint32_t i = blockIdx.z;
    const uint64_t x = last[(size_t)blockIdx.y * n + g];
    const uint64_t r = reduce_2q(x - mulhi64(x, mc[i].mu64) * q, q);
    return x > half ? sub_mod(r, rs[((size_t)l * L + i) * 4], q) : r;
  }
};
struct RescaleStore {
  static constexpr bool kPre = true;
  const uint64_t* const* a;  // RESCALE_MAX entries in kernel arguments
  uint64_t* const* out;
  const uint64_t* rs;
  uint32_t n, l, L, npoly;
  __device__ __forceinline__ uint64_t pre(size_t s, uint64_t) const {
    const uint32_t y = blockIdx.y;
    return a[y / npoly][((size_t)(y % npoly) * (l + 1) + blockIdx.z) * n + s];
  }
  __device__ __forceinline__ void fin(uint64_t*, size_t s, uint64_t y, uint64_t x,
                                      uint64_t q) const {
    const uint32_t i = blockIdx.z, p = blockIdx.y;
    const uint64_t* c = rs + ((size_t)l * L + i) * 4;
    out[p / npoly][((size_t)(p % npoly) * l + i) * n + s] = shoup(x + q - y, c[1], c[2], q);
  }
};

// Inputs of the next launch set out of `left`, npoly polys each.
inline uint32_t rescale_batch(uint32_t left, uint32_t npoly) {
  return std::min<uint32_t>({left, (uint32_t)RESCALE_MAX, 65535u / npoly});
}

}  // namespace
}  // namespace fhe
