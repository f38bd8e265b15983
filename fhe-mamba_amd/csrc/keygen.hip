// Client-side key material, encryption and decryption on the GPU.
//
// Mirrors OpenFHE's KeyGen / EvalMultKeyGen / EvalRotateKeyGen / Encrypt /
// Decrypt as called by the reference (native/fideslib_stage0/src/
// packed_fideslib.cpp:1080-1083, :204-205, :1227) with this library's
// sampling streams (sampling.hpp; ChaCha20 unless the context was switched
// to the seeded parity family):
//   public key      b = -a s + e over Q, a uniform in evaluation form
//   switching key   digit j: b_j = -a_j s_new + e_j + [P]_{q_i} s_old on the
//                   Q limbs of digit j (KeySwitchHYBRID key generation)
//   Galois key k    s_old = s, s_new = s(X^{k^-1})
//   relin key       s_old = s^2, s_new = s
//   encryption      (pk_b v + e0 + m, pk_a v + e1), v ternary
// Uniform residues and the small samples (v, e) are drawn on the GPU, each
// lane a block of the counter-based stream, and lifted by the transforms'
// first pass; the secret is the caller's, in host memory.  Drawn on the host
// the three samples of an encryption were 450 us of its 527 (N=2^16, 24
// limbs), most of them with the device idle.
#include <cstring>

#include "ops.hpp"
#include "sampling.hpp"

namespace fhe {
namespace {

constexpr int TPB = 256;

inline uint32_t tpb_for(const Context& c) { return c.n < TPB ? c.n : TPB; }

// Small samples drawn by one launch: stream p gives out[p][0..n), ternary or
// centred binomial (the host definitions of both are in sampling.hpp).
constexpr uint32_t MAX_DRAWS = 3;
struct SmallDraws {
  Stream s[MAX_DRAWS];
  uint32_t ternary;  // bit p: stream p is ternary
};

// Words 8t .. 8t+7 of stream blockIdx.y: one ChaCha20 block a thread.
__global__ void k_small_samples(int64_t* out, uint32_t n, SmallDraws d) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, p = blockIdx.y;
  const Stream& s = d.s[p];
  const bool ternary = (d.ternary >> p) & 1;
  uint64_t w[8];
  if (s.secure) {
    stream_block(s, t, w);
  } else {
    for (int i = 0; i < 8; ++i) w[i] = draw(s.sm_key, 8ull * t + i);
  }
  int64_t* o = out + (size_t)p * n + 8ull * t;
  for (int i = 0; i < 8; ++i) o[i] = ternary ? ternary_from(w[i]) : cbd_from(w[i]);
}

void launch_small(Context& c, int64_t* out, const SmallDraws& d, uint32_t count) {
  const uint32_t blocks = c.n / 8, tpb = blocks < 64 ? blocks : 64;
  FHE_LAUNCH(c, "k_small_samples", k_small_samples, dim3(blocks / tpb, count), dim3(tpb), 0, out,
             c.n, d);
}

// Centred binomial errors of stream (seed, tag, index) in evaluation form
// over the first nlimb moduli.
void errors_to_eval(Context& c, uint64_t seed, uint64_t tag, uint64_t index, uint32_t nlimb,
                    uint64_t* out) {
  Scratch coef(c, c.n);
  int64_t* const cf = reinterpret_cast<int64_t*>(coef.p);
  SmallDraws d{};
  d.s[0] = make_stream(c.sampling, seed, tag, index);
  launch_small(c, cf, d, 1);
  ntt_forward_signed(c, cf, out, 1, 0, nlimb, 0);
}

// Calls that draw randomness or read the caller's host memory cannot be
// replayed from a graph.
void refuse_capture(Context& c, const char* what) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  hip_check(hipStreamIsCapturing(c.stream, &st), what);
  if (st != hipStreamCaptureStatusNone) hip_check(hipErrorStreamCaptureUnsupported, what);
}

// out[j][e] = uniform mod q_{mod0+j} from words 2e, 2e+1 of stream
// (seed, tag, index_base | j); each thread draws four consecutive samples
// (one ChaCha20 block).  `base` carries the family, the call key and the
// tag; the limb's index goes into the nonce here.
__global__ void k_uniform(uint64_t* out, const ModConst* mc, uint32_t n, Stream base,
                          uint64_t seed, uint64_t tag, uint64_t index_base, uint32_t mod0) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  const uint64_t q = mc[mod0 + j].q;
  uint64_t w[8];
  if (base.secure) {
    Stream s = base;
    s.nonce[1] = (uint32_t)(index_base | j);
    stream_block(s, t, w);
  } else {
    const uint64_t key = stream_key(seed, tag, index_base | j);
    for (int i = 0; i < 8; ++i) w[i] = draw(key, 8ull * t + i);
  }
  uint64_t* o = out + (size_t)j * n + 4ull * t;
  for (int i = 0; i < 4; ++i) o[i] = uniform_from(w[2 * i], w[2 * i + 1], q);
}

void launch_uniform(Context& c, uint64_t* out, uint32_t nlimb, uint64_t seed, uint64_t tag,
                    uint64_t index_base, uint32_t mod0) {
  const Stream base = make_stream(c.sampling, seed, tag, 0);
  const uint32_t quads = c.n / 4, tpb = quads < TPB ? quads : TPB;
  FHE_LAUNCH(c, "k_uniform", k_uniform, dim3(quads / tpb, nlimb), dim3(tpb), 0, out, c.d_const,
             c.n, base, seed, tag, index_base, mod0);
}

// b = e - a * s (+ f * s_old on limbs [f_begin, f_end)); all [nlimb][N], f a
// per-limb factor array.
__global__ void k_key_combine(uint64_t* b, const uint64_t* a, const uint64_t* s,
                              const uint64_t* e, const uint64_t* s_old, const uint64_t* f,
                              uint32_t f_begin, uint32_t f_end, const ModConst* mc, uint32_t n) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  const ModConst m = mc[j];
  const size_t o = (size_t)j * n + x;
  uint64_t v = sub_mod(e[o], mul_mod(a[o], s[o], m), m.q);
  if (j >= f_begin && j < f_end) v = add_mod(v, mul_mod(f[j], s_old[o], m), m.q);
  b[o] = v;
}

// ct0 = b v + e0 + m, ct1 = a v + e1 over nq limbs.
__global__ void k_encrypt(uint64_t* ct, const uint64_t* pk, const uint64_t* v, const uint64_t* e0,
                          const uint64_t* e1, const uint64_t* msg, const ModConst* mc, uint32_t n,
                          uint32_t nq, uint32_t L) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
  const ModConst m = mc[i];
  const size_t o = (size_t)i * n + x;
  const uint64_t b = pk[o], a = pk[(size_t)L * n + o];
  ct[o] = add_mod(add_mod(mul_mod(b, v[o], m), e0[o], m.q), msg[o], m.q);
  ct[(size_t)nq * n + o] = add_mod(mul_mod(a, v[o], m), e1[o], m.q);
}

// m = sum_p ct_p s^p.
__global__ void k_decrypt(uint64_t* msg, const uint64_t* ct, const uint64_t* s, const ModConst* mc,
                          uint32_t n, uint32_t nq, uint32_t npoly) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
  const ModConst m = mc[i];
  const size_t o = (size_t)i * n + x;
  uint64_t acc = ct[o], sp = s[o];
  for (uint32_t p = 1; p < npoly; ++p) {
    acc = add_mod(acc, mul_mod(ct[(size_t)p * nq * n + o], sp, m), m.q);
    sp = mul_mod(sp, s[o], m);
  }
  msg[o] = acc;
}

__global__ void k_square(uint64_t* out, const uint64_t* a, const ModConst* mc, uint32_t n) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
  const size_t o = (size_t)i * n + x;
  out[o] = mul_mod(a[o], a[o], mc[i]);
}

}  // namespace

void sample_secret_host(Context& c, uint64_t seed, int64_t* out) {
  sample_ternary(make_stream(c.sampling, seed, TAG_SECRET, 0), out, c.n);
}
void sample_sparse_secret_host(Context& c, uint64_t seed, int64_t* out, uint32_t h) {
  sample_sparse_ternary(make_stream(c.sampling, seed, TAG_SECRET, 0), out, c.n, h);
}

void signed_to_eval(Context& c, const int64_t* coef_host, uint32_t idx0, uint32_t nlimb,
                    uint64_t* out) {
  refuse_capture(c, "secret upload");
  const size_t bytes = (size_t)c.n * 8;
  Scratch coef(c, c.n);
  {
    // staged in pinned memory, so that nothing waits for the stream here and
    // the caller's array is free when this returns
    std::lock_guard<std::mutex> g(c.staging_mu);
    Context::Staging& sg = c.staging_slot(bytes);
    std::memcpy(sg.host, coef_host, bytes);
    hip_check(hipMemcpyAsync(coef.p, sg.host, bytes, hipMemcpyHostToDevice, c.stream),
              "secret upload");
    hip_check(hipEventRecord(sg.done, c.stream), "secret staging event");
  }
  ntt_forward_signed(c, reinterpret_cast<const int64_t*>(coef.p), out, 1, 0, nlimb, idx0);
}

void keygen_public(Context& c, const int64_t* s_coef, uint64_t seed, uint64_t* pk) {
  const size_t n = c.n;
  Scratch s(c, c.L * n), e(c, c.L * n);
  signed_to_eval(c, s_coef, 0, c.L, s.p);
  errors_to_eval(c, seed, TAG_PK_E, 0, c.L, e.p);
  uint64_t* a = pk + (size_t)c.L * n;
  launch_uniform(c, a, c.L, seed, TAG_PK_A, 0, 0);
  FHE_LAUNCH(c, "k_key_combine", k_key_combine, dim3(c.n / tpb_for(c), c.L), dim3(tpb_for(c)), 0, pk, a, s.p, e.p, nullptr, nullptr, 0u, 0u, c.d_const, c.n);
  hip_check(hipStreamSynchronize(c.stream), "keygen sync");
}

void keygen_switch(Context& c, const uint64_t* s_old, const uint64_t* s_new, uint64_t seed,
                   uint64_t tag, uint64_t* key) {
  const size_t n = c.n;
  const uint32_t nm = c.L + c.K;
  Scratch e(c, nm * n);
  for (uint32_t j = 0; j < c.dnum; ++j) {
    const uint32_t s = j * c.alpha, end = s + c.alpha < c.L ? s + c.alpha : c.L;
    errors_to_eval(c, seed, tag + TAG_KSK_E, j, nm, e.p);
    uint64_t* b = key + ((size_t)j * 2) * nm * n;
    uint64_t* a = b + (size_t)nm * n;
    launch_uniform(c, a, nm, seed, tag + TAG_KSK_A, (uint64_t)j << 16, 0);
    FHE_LAUNCH(c, "k_key_combine", k_key_combine, dim3(c.n / tpb_for(c), nm), dim3(tpb_for(c)), 0, b, a, s_new, e.p, s_old, c.d_keyfac_out, s, end, c.d_const, c.n);
  }
  hip_check(hipStreamSynchronize(c.stream), "keygen sync");
}

void keygen_galois(Context& c, const int64_t* s_coef, uint32_t galois, uint64_t seed,
                   uint64_t* key) {
  const uint32_t nm = c.L + c.K;
  Scratch s(c, (size_t)nm * c.n), sp(c, (size_t)nm * c.n);
  signed_to_eval(c, s_coef, 0, nm, s.p);
  automorph(c, sp.p, s.p, 1, nm, galois_inverse(galois, c.n));
  keygen_switch(c, s.p, sp.p, seed, TAG_GALOIS + ((uint64_t)galois << 3), key);
}

void keygen_relin(Context& c, const int64_t* s_coef, uint64_t seed, uint64_t* key) {
  const uint32_t nm = c.L + c.K;
  Scratch s(c, (size_t)nm * c.n), s2(c, (size_t)nm * c.n);
  signed_to_eval(c, s_coef, 0, nm, s.p);
  FHE_LAUNCH(c, "k_square", k_square, dim3(c.n / tpb_for(c), nm), dim3(tpb_for(c)), 0, s2.p, s.p, c.d_const, c.n);
  keygen_switch(c, s2.p, s.p, seed, TAG_RELIN, key);
}

void encrypt_pk(Context& c, const uint64_t* pk, const uint64_t* m, uint32_t nq, uint64_t seed,
                uint64_t* ct) {
  refuse_capture(c, "encrypt");
  const size_t n = c.n;
  Scratch coef(c, MAX_DRAWS * n), ve(c, MAX_DRAWS * nq * n);
  int64_t* const cf = reinterpret_cast<int64_t*>(coef.p);
  SmallDraws d{};
  d.s[0] = make_stream(c.sampling, seed, TAG_ENC_V, 0);
  d.s[1] = make_stream(c.sampling, seed, TAG_ENC_E, 0);
  d.s[2] = make_stream(c.sampling, seed, TAG_ENC_E, 1);
  d.ternary = 1;
  launch_small(c, cf, d, 3);
  ntt_forward_signed(c, cf, ve.p, 3, nq * n, nq, 0);
  const uint64_t *v = ve.p, *e0 = v + nq * n, *e1 = e0 + nq * n;
  FHE_LAUNCH(c, "k_encrypt", k_encrypt, dim3(c.n / tpb_for(c), nq), dim3(tpb_for(c)), 0, ct, pk, v, e0, e1, m, c.d_const, c.n, nq, c.L);
}

void decrypt(Context& c, const uint64_t* ct, uint32_t npoly, uint32_t nq, const int64_t* s_coef,
             uint64_t* m) {
  Scratch s(c, (size_t)nq * c.n);
  signed_to_eval(c, s_coef, 0, nq, s.p);
  FHE_LAUNCH(c, "k_decrypt", k_decrypt, dim3(c.n / tpb_for(c), nq), dim3(tpb_for(c)), 0, m, ct, s.p, c.d_const, c.n, nq, npoly);
}

}  // namespace fhe
