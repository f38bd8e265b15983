// CKKS encode / decode on the GPU.
//
// Encode = OpenFHE CKKSPackedEncoding::Encode as restated by the
// reference's GPU encoder (native/fideslib_stage0/src/gpu_special_fft.cu):
//   special inverse FFT over `slots` values (butterfly order and twiddle
//   table of gpu_special_fft.cu:12-22, :99-108 and
//   patches/openfhe-v1.4.2-inverse-fft-plan.patch:18-60), bit reversal,
//   division by slots, multiplication by the scale, llround (ties away from
//   zero), placement of the 2*slots real/imaginary coefficients at stride
//   N / (2 slots), signed RNS lift into each limb
//   (fideslib_plaintext_rns.cu:11-23), forward NTT.
// Decode = inverse NTT, centred CRT (balanced mixed-radix / Garner, so no
// big integers), division by the scale, forward special FFT.
//
// All floating-point operations are plain IEEE double add/sub/mul/div; the
// library is compiled with -ffp-contract=off so none fuse into FMAs, which
// keeps the encoder's rounding identical to the CPU definition.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "ops.hpp"

namespace fhe {
namespace {

constexpr int TPB = 256;

inline uint32_t ilog2(uint32_t x) {
  uint32_t l = 0;
  while ((1u << l) < x) ++l;
  return l;
}

// Twiddle (cos, sin) pairs come from one glibc sincos() call per angle: that
// is what gcc-built OpenFHE evaluates for its (cos(angle), sin(angle))
// table (gcc fuses the pair), and sincos() differs from separate cos()/sin()
// in the last bit for a few angles.
inline void host_sincos(double a, double* s, double* c) { ::sincos(a, s, c); }

std::pair<double*, double*> fft_tables(Context& c, uint32_t slots) {
  std::lock_guard<std::mutex> g(c.fft_mu);
  auto it = c.fft_tables.find(slots);
  if (it != c.fft_tables.end()) return it->second;
  const uint32_t m = 4 * slots;
  std::vector<uint32_t> rot(slots);
  uint32_t p = 1;
  for (uint32_t j = 0; j < slots; ++j) {
    rot[j] = p;
    p = (uint32_t)(((uint64_t)p * 5) % m);
  }
  const size_t cnt = slots > 1 ? slots - 1 : 1;
  std::vector<double> inv(2 * cnt, 0.0), fwd(2 * cnt, 0.0);
  for (uint32_t len = 2; len <= slots; len <<= 1) {
    const uint32_t h = len / 2, lenq = 4 * len, gap = m / lenq;
    for (uint32_t j = 0; j < h; ++j) {
      const double ai = 2.0 * M_PI * ((lenq - rot[j] % lenq) * gap) / m;
      const double af = 2.0 * M_PI * ((rot[j] % lenq) * gap) / m;
      host_sincos(ai, &inv[2 * (h - 1 + j) + 1], &inv[2 * (h - 1 + j)]);
      host_sincos(af, &fwd[2 * (h - 1 + j) + 1], &fwd[2 * (h - 1 + j)]);
    }
  }
  double *di = nullptr, *df = nullptr;
  note_alloc();
  note_alloc();
  hip_check(hipMalloc(&di, inv.size() * 8), "hipMalloc fft");
  hip_check(hipMalloc(&df, fwd.size() * 8), "hipMalloc fft");
  hip_check(hipMemcpy(di, inv.data(), inv.size() * 8, hipMemcpyHostToDevice), "fft table");
  hip_check(hipMemcpy(df, fwd.data(), fwd.size() * 8, hipMemcpyHostToDevice), "fft table");
  c.fft_tables[slots] = {di, df};
  return {di, df};
}

// One butterfly of the special inverse FFT: (a, b) -> (a + b, (a - b) w), and
// of the forward one: (u, b) -> (u + b w, u - b w).
__device__ __forceinline__ void fft_inv_butterfly(double2& a, double2& b, double2 w) {
  const double vr = a.x - b.x, vi = a.y - b.y;
  a = make_double2(a.x + b.x, a.y + b.y);
  b = make_double2(vr * w.x - vi * w.y, vi * w.x + vr * w.y);
}
__device__ __forceinline__ void fft_fwd_butterfly(double2& u, double2& b, double2 w) {
  const double vr = b.x * w.x - b.y * w.y, vi = b.y * w.x + b.x * w.y;
  b = make_double2(u.x - vr, u.y - vi);
  u = make_double2(u.x + vr, u.y + vi);
}

// The transforms run in two kernels, each bound by the latency of its chain of
// dependent stages: the stages with len <= FFT_BLOCK pair elements inside
// aligned blocks of FFT_BLOCK values, one workgroup a block in LDS, one
// butterfly a lane and stage with every stage's twiddle loaded up front; the
// longer ones pair elements a multiple of slots / 2^T apart, 2^T values a lane
// in registers (32768 slots, forward, us: 12.4 + 4 x 4.4 as a block kernel of
// 256 lanes and a kernel a stage, 7.5 + 4.2 as this).  The butterflies and the order of each
// element's are those of the radix-2 definition, hence the same roundings.
constexpr uint32_t FFT_BLOCK = 2048;

// Values of one-slot vectors.
__global__ void k_real_to_complex(double2* v, const double* v_in, uint32_t count) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < count) v[k] = make_double2(v_in[k], 0.0);
}

// Stages len = 2^LOG, ..., 2 (inverse) or 2, ..., 2^LOG (forward) on blocks of
// 2^LOG values.  v_in: the inverse transform's input as real values.
template <int LOG, bool INV>
__global__ void __launch_bounds__(1024)
    k_fft_block(double2* v, const double* v_in, const double* tw) {
  constexpr uint32_t top = 1u << LOG;
  __shared__ double2 x[top];
  const uint32_t t = threadIdx.x;
  const size_t g0 = (size_t)blockIdx.x * top;
  const double2* const tw2 = reinterpret_cast<const double2*>(tw);
  double2 w[LOG];
#pragma unroll
  for (int s = 0; s < LOG; ++s) w[s] = tw2[(1u << s) - 1 + (t & ((1u << s) - 1))];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t k = t + h * (top / 2);
    x[k] = v_in ? make_double2(v_in[g0 + k], 0.0) : v[g0 + k];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < LOG; ++i) {
    const int s = INV ? LOG - 1 - i : i;  // h = len / 2 = 2^s
    const uint32_t h = 1u << s, a = ((t >> s) << (s + 1)) | (t & (h - 1));
    double2 p = x[a], q = x[a + h];
    if (INV)
      fft_inv_butterfly(p, q, w[s]);
    else
      fft_fwd_butterfly(p, q, w[s]);
    x[a] = p;
    x[a + h] = q;
    __syncthreads();
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) v[g0 + t + h * (top / 2)] = x[t + h * (top / 2)];
}

// The T longest stages (len = slots, ..., slots / 2^(T-1) for the inverse, the
// other way round for the forward transform) of vector blockIdx.y.
template <int T, bool INV>
__global__ void __launch_bounds__(64)
    k_fft_top(double2* v, const double* v_in, const double* tw, uint32_t slots) {
  const uint32_t B = slots >> T, t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= B) return;
  v += (size_t)blockIdx.y * slots;
  const double2* const tw2 = reinterpret_cast<const double2*>(tw);
  double2 x[1 << T];
#pragma unroll
  for (int k = 0; k < 1 << T; ++k)
    x[k] = v_in ? make_double2(v_in[(size_t)blockIdx.y * slots + t + k * B], 0.0) : v[t + k * B];
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const int s = INV ? T - 1 - i : i;  // pairs k, k + 2^s: h = 2^s B
#pragma unroll
    for (int k = 0; k < 1 << T; ++k) {
      if (k & (1 << s)) continue;
      const double2 w = tw2[((1u << s) * B - 1) + t + (k & ((1 << s) - 1)) * B];
      if (INV)
        fft_inv_butterfly(x[k], x[k + (1 << s)], w);
      else
        fft_fwd_butterfly(x[k], x[k + (1 << s)], w);
    }
  }
#pragma unroll
  for (int k = 0; k < 1 << T; ++k) v[t + k * B] = x[k];
}

__device__ __forceinline__ uint32_t brev_bits(uint32_t x, uint32_t bits) {
  return bits ? __brev(x) >> (32 - bits) : 0;
}

// Round slot i of the transformed vector (read through the bit reversal) to
// its real / imaginary coefficient of vector blockIdx.y; the other
// coefficients of the slot's two gap blocks are zero.
__global__ void k_round(const double2* v, int64_t* coef, uint32_t slots, uint32_t bits,
                        uint32_t gap, uint32_t n, double scale, int* status) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= slots) return;
  v += (size_t)blockIdx.y * slots;
  coef += (size_t)blockIdx.y * n;
  const double2 x = v[brev_bits(i, bits)];
  const double a = (x.x / (double)slots) * scale, b = (x.y / (double)slots) * scale;
  const double lim = 4611686018427387904.0;  // 2^62
  if (!isfinite(a) || !isfinite(b) || fabs(a) >= lim || fabs(b) >= lim) {
    if (status) atomicOr(status, 1);
    return;
  }
  coef[(size_t)i * gap] = llround(a);
  coef[(size_t)(i + slots) * gap] = llround(b);
  for (uint32_t z = 1; z < gap; ++z) {
    coef[(size_t)i * gap + z] = 0;
    coef[(size_t)(i + slots) * gap + z] = 0;
  }
}

// Balanced Garner reconstruction of coefficient positions i*gap, i < 2 slots,
// then division by the scale; writes complex slot inputs of the forward FFT
// at bit-reversed positions.  Digit a_j, once known, is taken out of every
// later residue, x_i = (x_i - a_j) q_j^-1 mod q_i: one Shoup product of
// x_i - a_j plus a multiple of q_i.  The steps j are a chain, the updates of
// one step are not: a workgroup holds 64 coefficients' residues in LDS and its
// CRT_WAVES wavefronts share each step's limbs, one barrier a step.  Bound by
// the latency of that chain (32768 slots, 24 limbs: 186 us with one residue
// after the other and hardware division, 63 with one wavefront a workgroup,
// 37 as this).
constexpr uint32_t CRT_WAVES = 4;
__global__ void __launch_bounds__(64 * CRT_WAVES)
    k_crt_decode(const uint64_t* coef, double2* v, const ModConst* mc, const uint64_t* garner,
                 uint32_t n, uint32_t nlimb, uint32_t L, uint32_t slots, uint32_t bits,
                 uint32_t gap, double scale) {
  extern __shared__ uint64_t xs[];  // [nlimb][64]
  const uint32_t t = blockIdx.x * 64 + (threadIdx.x & 63);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool valid = t < 2 * slots;
  uint64_t* const x = xs + (threadIdx.x & 63);
  for (uint32_t i = wave; i < nlimb; i += CRT_WAVES)
    x[i * 64] = valid ? coef[(size_t)i * n + (size_t)t * gap] : 0;
  for (uint32_t j = 0; j + 1 < nlimb; ++j) {
    __syncthreads();
    const uint64_t r = x[j * 64], qj = mc[j].q;
    const uint64_t a = r > (qj >> 1) ? r - qj : r;  // balanced, as a signed word
#pragma unroll 2
    for (uint32_t i = j + 1 + ((wave - j - 1) & (CRT_WAVES - 1)); i < nlimb; i += CRT_WAVES) {
      const uint64_t* g = garner + ((size_t)i * L + j) * 2;
      x[i * 64] = shoup(x[i * 64] + mc[i].lift60 - a, g[0], g[1], mc[i].q);
    }
  }
  __syncthreads();
  if (wave != 0 || !valid) return;
  double val = 0.0;
  for (int i = (int)nlimb - 1; i >= 0; --i) {
    const uint64_t r = x[i * 64], q = mc[i].q;
    const double d = (double)(int64_t)(r > (q >> 1) ? r - q : r);
    val = i == (int)nlimb - 1 ? d : val * (double)q + d;
  }
  val = val / scale;
  const uint32_t slot = t < slots ? t : t - slots;
  double* dst = reinterpret_cast<double*>(v + brev_bits(slot, bits));
  dst[t < slots ? 0 : 1] = val;
}

template <bool INV>
void launch_fft_block(Context& c, double2* v, const double* v_in, const double* tw, uint32_t log,
                      uint32_t nblk) {
  const char* name = INV ? "k_fft_inv_block" : "k_fft_fwd_block";
  if (log == 0) {
    if (v_in)
      FHE_LAUNCH(c, "k_real_to_complex", k_real_to_complex, dim3((nblk + 63) / 64), dim3(64), 0, v,
                 v_in, nblk);
    return;
  }
  switch (log) {
#define CASE(G)                                                                               \
  case G:                                                                                     \
    FHE_LAUNCH(c, name, (k_fft_block<G, INV>), dim3(nblk), dim3(1u << (G - 1)), 0, v, v_in, tw); \
    return;
    CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11)
#undef CASE
    default: throw ArgError("unsupported slot count");
  }
}
template <bool INV>
void launch_fft_top(Context& c, double2* v, const double* v_in, const double* tw, uint32_t slots,
                    uint32_t log, uint32_t nvec) {
  const char* name = INV ? "k_fft_inv_top" : "k_fft_fwd_top";
  switch (log) {
#define CASE(T)                                                                              \
  case T:                                                                                    \
    FHE_LAUNCH(c, name, (k_fft_top<T, INV>), dim3((slots >> T) / 64, nvec), dim3(64), 0, v, \
               v_in, tw, slots);                                                             \
    return;
    CASE(1) CASE(2) CASE(3) CASE(4) CASE(5)
#undef CASE
    default: throw ArgError("unsupported slot count");
  }
}

// The special FFT of nvec contiguous vectors of `slots` values each, in v; the
// inverse one may take its input as real values v_in instead.  The block
// kernel's blocks never straddle two vectors (their size divides slots), so
// it runs over the batch as one array.
// One slot is its own transform.
void run_stages_inv(Context& c, double2* v, const double* v_in, const double* tw, uint32_t slots,
                    uint32_t nvec) {
  const uint32_t log = ilog2(slots), blk = slots < FFT_BLOCK ? log : ilog2(FFT_BLOCK);
  const uint32_t top = log - blk;
  if (top) launch_fft_top<true>(c, v, v_in, tw, slots, top, nvec);
  launch_fft_block<true>(c, v, top ? nullptr : v_in, tw, blk, nvec * (slots >> blk));
}
void run_stages_fwd(Context& c, double2* v, const double* tw, uint32_t slots) {
  if (slots < 2) return;
  const uint32_t log = ilog2(slots), blk = slots < FFT_BLOCK ? log : ilog2(FFT_BLOCK);
  launch_fft_block<false>(c, v, nullptr, tw, blk, slots >> blk);
  if (log > blk) launch_fft_top<false>(c, v, nullptr, tw, slots, log - blk, 1);
}

void check_slots(const Context& c, uint32_t slots) {
  if (slots == 0 || (slots & (slots - 1)) || slots > c.n / 2)
    throw ArgError("slots must be a power of two <= N/2");
}

}  // namespace

// Copies `count` values (real parts alone when im is null) into dst, zeros
// up to `slots`, and whether some |z|^2 does not stay below lim2 (NaN and
// infinities do not).
static bool stage_values(double* dst, const double* re, const double* im, uint32_t count,
                         uint32_t slots, double lim2) {
  int over = 0;
  if (im) {
    for (uint32_t j = 0; j < count; ++j) {
      const double a = re[j], b = im[j];
      dst[2 * j] = a;
      dst[2 * j + 1] = b;
      over |= !(a * a + b * b < lim2);
    }
    std::memset(dst + 2 * (size_t)count, 0, 2 * (size_t)(slots - count) * sizeof(double));
  } else {
    for (uint32_t j = 0; j < count; ++j) {
      const double a = re[j];
      dst[j] = a;
      over |= !(a * a < lim2);
    }
    std::memset(dst + count, 0, (size_t)(slots - count) * sizeof(double));
  }
  return over != 0;
}

bool encode(Context& c, const double* re, const double* im, uint32_t count, uint32_t slots,
            double scale, uint32_t nlimb, uint64_t* out) {
  check_slots(c, slots);
  if (count > slots) throw ArgError("more values than slots");
  if (nlimb == 0 || nlimb > c.L) throw ArgError("bad limb count");
  if (!(scale > 0) || !std::isfinite(scale)) throw ArgError("scale must be positive");
  const uint32_t parts = im ? 2 : 1;
  const size_t bytes = parts * (size_t)slots * sizeof(double);
  const auto tw = fft_tables(c, slots);
  // real inputs are uploaded to where the rounded coefficients go afterwards
  Scratch v(c, 2 * (size_t)slots), coef(c, c.n), st(c, 1);
  // Range bound: each inverse-FFT stage maps (a, b) to (a + b, (a - b) w)
  // with |w| = 1, so an output's modulus is at most the sum of the inputs'
  // and, after the division by slots, at most the largest input modulus.
  // Inputs whose bound times the scale stays below 2^62 (the margin 2^-20
  // is far above the transform's rounding) cannot fail k_round's range
  // check, so nothing waits for the device; other inputs read the check's
  // status back, which waits for the stream.
  const double lim = 4611686018427387904.0 * (1.0 - 0x1p-20) / scale;
  const double lim2 = lim * lim;
  bool checked = !(lim2 < INFINITY);
  double* const dst = reinterpret_cast<double*>(im ? v.p : coef.p);
  {
    std::lock_guard<std::mutex> g(c.staging_mu);
    Context::Staging& sg = c.staging_slot(bytes);
    checked |= stage_values(static_cast<double*>(sg.host), re, im, count, slots, lim2);
    hip_check(hipMemcpyAsync(dst, sg.host, bytes, hipMemcpyHostToDevice, c.stream),
              "encode upload");
    hip_check(hipEventRecord(sg.done, c.stream), "encode staging event");
  }
  if (checked) hip_check(hipMemsetAsync(st.p, 0, 8, c.stream), "encode status");
  double2* const vv = reinterpret_cast<double2*>(v.p);
  int64_t* const cf = reinterpret_cast<int64_t*>(coef.p);
  run_stages_inv(c, vv, im ? nullptr : dst, tw.first, slots, 1);
  const uint32_t threads = slots < TPB ? slots : TPB;
  FHE_LAUNCH(c, "k_round", k_round, dim3((slots + threads - 1) / threads), dim3(threads), 0, vv,
             cf, slots, ilog2(slots), c.n / (2 * slots), c.n, scale,
             checked ? reinterpret_cast<int*>(st.p) : nullptr);
  if (checked) {
    int status = 0;
    hip_check(hipMemcpyAsync(&status, st.p, sizeof(int), hipMemcpyDeviceToHost, c.stream),
              "encode status");
    hip_check(hipStreamSynchronize(c.stream), "encode sync");
    if (status) return false;
  }
  ntt_forward_signed(c, cf, out, 1, 0, nlimb, 0);
  return true;
}

bool encode_many(Context& c, const double* re, const double* im, uint32_t count, uint32_t nvec,
                 uint32_t slots, double scale, uint32_t nlimb, uint64_t* const* outs) {
  check_slots(c, slots);
  if (count > slots) throw ArgError("more values than slots");
  if (nlimb == 0 || nlimb > c.L) throw ArgError("bad limb count");
  if (!(scale > 0) || !std::isfinite(scale)) throw ArgError("scale must be positive");
  const double lim = 4611686018427387904.0 * (1.0 - 0x1p-20) / scale;
  const double lim2 = lim * lim;
  const auto tw = fft_tables(c, slots);
  // Up to kChunk vectors share one staging copy and one set of launches:
  // the pointer table (padded to 16 bytes) and then the vectors' values.
  constexpr uint32_t kChunk = 16;
  for (uint32_t r0 = 0; r0 < nvec; r0 += kChunk) {
    const uint32_t m = nvec - r0 < kChunk ? nvec - r0 : kChunk;
    const size_t tab_words = (m + 1) & ~1u, vec_words = (im ? 2 : 1) * (size_t)slots;
    const size_t words = tab_words + m * vec_words;
    bool over = !(lim2 < INFINITY);
    // real inputs are uploaded to where the rounded coefficients go afterwards
    const size_t coef_words = m * (size_t)c.n, fft_words = m * 2 * (size_t)slots;
    Scratch buf(c, tab_words + (im ? fft_words : coef_words)), other(c, im ? coef_words : fft_words);
    uint64_t* const vals = buf.p + tab_words;
    {
      std::lock_guard<std::mutex> g(c.staging_mu);
      Context::Staging& sg = c.staging_slot(words * 8);
      uint64_t* host = static_cast<uint64_t*>(sg.host);
      for (uint32_t r = 0; r < m; ++r) host[r] = reinterpret_cast<uint64_t>(outs[r0 + r]);
      double* hv = reinterpret_cast<double*>(host + tab_words);
      for (uint32_t r = 0; r < m && !over; ++r)
        over = stage_values(hv + r * vec_words, re + (size_t)(r0 + r) * count,
                            im ? im + (size_t)(r0 + r) * count : nullptr, count, slots, lim2);
      if (!over) {
        hip_check(hipMemcpyAsync(buf.p, host, words * 8, hipMemcpyHostToDevice, c.stream),
                  "encode upload");
        hip_check(hipEventRecord(sg.done, c.stream), "encode staging event");
      }
    }
    if (over) {
      // Values that may not fit take the checked single path, which
      // reports the first vector that fails.
      for (uint32_t r = r0; r < r0 + m; ++r)
        if (!encode(c, re + (size_t)r * count, im ? im + (size_t)r * count : nullptr, count, slots,
                    scale, nlimb, outs[r]))
          return false;
      continue;
    }
    double2* const v = reinterpret_cast<double2*>(im ? vals : other.p);
    int64_t* const cf = reinterpret_cast<int64_t*>(im ? other.p : vals);
    const double* const in = im ? nullptr : reinterpret_cast<const double*>(vals);
    run_stages_inv(c, v, in, tw.first, slots, m);
    const uint32_t threads = slots < TPB ? slots : TPB;
    FHE_LAUNCH(c, "k_round", k_round, dim3((slots + threads - 1) / threads, m), dim3(threads), 0,
               v, cf, slots, ilog2(slots), c.n / (2 * slots), c.n, scale, nullptr);
    ntt_forward_signed_table(c, cf, reinterpret_cast<uint64_t* const*>(buf.p), m, nlimb);
  }
  return true;
}

void decode(Context& c, const uint64_t* pt, uint32_t nlimb, uint32_t slots, double scale,
            double* re, double* im) {
  check_slots(c, slots);
  if (nlimb == 0 || nlimb > c.L) throw ArgError("bad limb count");
  const auto tw = fft_tables(c, slots);
  Scratch coef(c, (size_t)nlimb * c.n), v(c, 2 * (size_t)slots);
  double2* const vv = reinterpret_cast<double2*>(v.p);
  ntt_inverse_from(c, pt, coef.p, nlimb);
  FHE_LAUNCH(c, "k_crt_decode", k_crt_decode, dim3((2 * slots + 63) / 64), dim3(64 * CRT_WAVES),
             (size_t)nlimb * 64 * 8, coef.p, vv, c.d_const, c.d_garner, c.n, nlimb, c.L,
             slots, ilog2(slots), c.n / (2 * slots), scale);
  run_stages_fwd(c, vv, tw.second, slots);
  // The transform is waited for before the staging buffer is taken, which is
  // held for the length of the copy alone.
  hip_check(hipStreamSynchronize(c.stream), "decode sync");
  const size_t bytes = 2 * (size_t)slots * sizeof(double);
  std::lock_guard<std::mutex> g(c.staging_mu);
  Context::Staging& sg = c.staging_slot(bytes);
  hip_check(hipMemcpyAsync(sg.host, v.p, bytes, hipMemcpyDeviceToHost, c.stream),
            "decode download");
  hip_check(hipEventRecord(sg.done, c.stream), "decode staging event");
  hip_check(hipStreamSynchronize(c.stream), "decode download");
  const double* const host = static_cast<const double*>(sg.host);
  if (im) {
    for (uint32_t j = 0; j < slots; ++j) {
      re[j] = host[2 * j];
      im[j] = host[2 * j + 1];
    }
  } else {
    for (uint32_t j = 0; j < slots; ++j) re[j] = host[2 * j];
  }
}

}  // namespace fhe
