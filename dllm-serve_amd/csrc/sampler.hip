// K8 / K9: the low-confidence remasking sampler of the diffusion runner.
//
// K8 (smx_row_kernel) reduces each row of bf16 logits
// [M, V] to what `x0_p, x0 = torch.max(F.softmax(logits, -1), -1)` returns
// (dllmserve/engine/model_runner.py:862-863,886-887):
//   m  = max_j l_j,  s = sum_j exp(l_j - m)                      (f32)
//   P_j = bf16(exp(l_j - m) / s)                                  (the bf16 probabilities)
//   x0_p = max_j P_j = bf16(1 / s),  x0 = min { j : P_j == x0_p }
// in one read of the logits.  A probability can only round to x0_p when its
// logit is within 2^-6 of m, and bf16 logits below m are that close to it
// only when |m| <= 2; so x0 is the first index of the maximal logit unless
// |m| <= 2, in which case the columns before that index are rescanned for an
// earlier one whose rounded probability ties.
//
// Layout: one workgroup per row, or several for few rows (smx_splits); each
// thread streams every NT-th 16-byte chunk, the next batch's loads in flight,
// and keeps a record {m, s, first index of m}; the records are merged across
// the workgroup (and across a row's workgroups by a second launch) and one
// wavefront finishes the row (the tie rescan included).  HBM-bound: 2 V bytes
// per row, read once.  256 rows of 126464: 16.4 -> 14.3 us (4.5 TB/s).
//
// With a per-row temperature T > 0 the row is first transformed as the
// reference's add_gumbel_noise does (model_runner.py:592-600):
//   v_j = bf16(exp(f64 l_j) / (-log u_j)^T),   u_j uniform in [0, 1) (f64)
// and the softmax-max runs over v.  u_j comes from a counter-based generator
// (SplitMix64 of seed + (c + 1) * 0x9E3779B97F4A7C15, c = (row_base + row) *
// V + j, top 53 bits), so a row's draws do not depend on how rows are
// grouped into launches; torch's own generator stream is not reproduced.
//
// K9 (lowconf_unmask_kernel) is the per-sequence unmasking step that follows
// (model_runner.py:895-949): in the sequence's window of token positions,
// count the masked ones, unmask k = min(ceil(nmask / steps_remain), nmask) of
// them -- the window's first position first when the first-token rule
// applies -- and the rest in order of confidence (descending, ties to the
// lower position, which is the set torch.topk returns).  One wavefront (windows
// of up to 1024 positions, keys in registers) or workgroup (keys in LDS) per
// sequence; the k-th largest (confidence, position) key is found by a
// bitwise search.
#include "common.h"

#include <limits.h>

namespace dllm {

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kUnmaskMaxWin = 8192;  // SamplingParams caps gen_length at 8192

__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Merge partial (m2, s2, i2) into (m, s, i).  An empty partial is
// (-inf, 0, INT_MAX).  Symmetric, so butterfly reductions agree on all lanes.
__device__ __forceinline__ void smx_merge(float& m, float& s, int& i, float m2, float s2, int i2) {
  const float mn = fmaxf(m, m2);
  const float a = (m == mn) ? s : s * fexp2((m - mn) * kLog2e);
  const float b = (m2 == mn) ? s2 : s2 * fexp2((m2 - mn) * kLog2e);
  i = (m > m2) ? i : (m2 > m) ? i2 : min(i, i2);
  s = a + b;
  m = mn;
}

__device__ __forceinline__ void smx_wave_reduce(float& m, float& s, int& i) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float m2 = __uint_as_float(lane_xor(__float_as_uint(m), off));
    const float s2 = __uint_as_float(lane_xor(__float_as_uint(s), off));
    const int i2 = (int)lane_xor((uint32_t)i, off);
    smx_merge(m, s, i, m2, s2, i2);
  }
}

__device__ __forceinline__ uint64_t splitmix64_at(uint64_t seed, uint64_t c) {
  uint64_t z = seed + (c + 1) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// exp(l) / (-log u)^T in f64, rounded to f32 and then to bf16 (the value the
// reference stores back into its bf16 logits), returned as f32.
__device__ __forceinline__ float gumbel_value(float l, double T, uint64_t seed, uint64_t c) {
  const double u = (double)(splitmix64_at(seed, c) >> 11) * 0x1.0p-53;
  const double nl = -log(u);
  const double g = T == 1.0 ? nl : pow(nl, T);
  const double v = exp((double)l) / g;
  return bf16_bits_to_f32(f64_to_bf16_bits_2step(v));
}

__device__ __forceinline__ void smx_unpack(u32x4_t v, float (&f)[8]) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    f[2 * w] = __uint_as_float(v[w] << 16);
    f[2 * w + 1] = __uint_as_float(v[w] & 0xffff0000u);
  }
}

// Fold U chunks of 8 logits (chunk u = columns 8 (c + u step) ..) into the
// running (m, s, i).  A thread's chunks arrive in increasing column order, so
// a tie with the running max keeps the earlier index.  One test of the maximum
// for all 8 U logits.
template <int U>
__device__ __forceinline__ void smx_batch(const u32x4_t (&v)[U], int c, int step, float& m, float& s, int& i) {
  float f[U][8];
#pragma unroll
  for (int u = 0; u < U; ++u) smx_unpack(v[u], f[u]);
  float cm = f[0][0];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int k = 0; k < 8; ++k) cm = fmaxf(cm, f[u][k]);
  if (cm > m) {
    int at = 0;
#pragma unroll
    for (int u = U - 1; u >= 0; --u)
#pragma unroll
      for (int k = 7; k >= 0; --k)
        if (f[u][k] == cm) at = 8 * (c + u * step) + k;
    s *= fexp2((m - cm) * kLog2e);
    m = cm;
    i = at;
  }
  if (m != -INFINITY) {
    float e0 = 0.f, e1 = 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int k = 0; k < 8; k += 2) {
        e0 += fexp2((f[u][k] - m) * kLog2e);
        e1 += fexp2((f[u][k + 1] - m) * kLog2e);
      }
    s += e0 + e1;
  }
}

// The noisy rows.  v = exp(l) / E^T, E = -log u, takes ~160 instructions of
// f64 per logit, but next to the row's maximum only few values count: one that
// lies kNoiseGap below any other value of the row adds exp(-kNoiseGap) < 2^-158
// of that value's own term to the sum of exponentials -- nothing in f32 -- and
// is not the maximum.  A cheap bound tells most of them: with h = the high 32
// bits of the draw, E >= 1 - u > (2^32 - 1 - h) 2^-32, hence
//   log2 v < l log2(e) - T (log2(2^32 - 1 - h) - 32).
// A threshold follows from a value that the row is known to hold: at first from
// lower bounds over a wavefront's first chunk, then from the largest value that
// any wavefront of the workgroup has computed (in LDS).  A logit whose bound is
// below it is left out, all others (infinite and NaN bounds included) are
// computed in f64 as before, the ones with the lanes' largest bounds first.
// Bounded by the integer hash (two 64-bit products per logit, six quarter-rate
// multiplies).  256 x 126464 logits at temperature 1 on an MI355X: 154 us
// without the bound, 42 us with one logarithm per logit and a threshold per
// wavefront, 35.6 us now.
constexpr float kNoiseGap = 110.0f;

// High word of the draw's SplitMix64 product, z1 = seed + (counter + 1) * golden;
// the generator's last step xors its own top bit into the word's lowest one.
__device__ __forceinline__ uint32_t noise_high(uint64_t z1) {
  uint64_t z = z1;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z ^= z >> 27;
  const uint32_t lo = (uint32_t)z, hi = (uint32_t)(z >> 32);
  return __umulhi(lo, 0x133111EBu) + lo * 0x94D049BBu + hi * 0x133111EBu;  // of z * 0x94D049BB133111EB
}

// log2 of the bound above for one logit with h = hi.
__device__ __forceinline__ float noise_bound_log2(float l, float T, uint32_t hi) {
  const uint32_t h = hi ^ (hi >> 31);
  const float lg = __builtin_amdgcn_logf((float)~h) - 32.0f;  // log2; -inf when ~h is 0
  return __builtin_fmaf(l, kLog2e, -T * lg);
}

// log2 of a lower bound of the value: E <= -log(h 2^-32) (1e-5 for the rounding
// of the logarithm near h = 2^32), and half a bf16 step down.
__device__ __forceinline__ float noise_floor_log2(float l, float T, uint32_t hi) {
  const uint32_t h = hi ^ (hi >> 31);
  const float E = 0.69314718f * (32.0f - __builtin_amdgcn_logf((float)h)) + 1e-5f;  // inf when h is 0
  return __builtin_fmaf(l, kLog2e, -T * __builtin_amdgcn_logf(E)) - (0.01f + 1e-3f * T);
}

// log2 below which a bound means "kNoiseGap below m_w, or less" (m_w: a value
// of the row).  The slack covers the bound's f32 rounding (log2 terms below
// 2^9, T times one of at most 32) and the rounding of v to bf16 (2^-8); up to
// 2^127 only, so that every value that may overflow is computed.
__device__ __forceinline__ float noise_threshold(float m_w, float T) {
  const float d = m_w - kNoiseGap;
  return d > 1.0f ? fminf(__builtin_amdgcn_logf(d), 127.0f) - (0.02f + 1e-4f * T) : -INFINITY;
}

__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x = fmaxf(x, __uint_as_float(lane_xor(__float_as_uint(x), off)));
  return x;
}

// Fold 8 logits of a row with temperature T into (m, s, i); rc + e0 = counter
// of the first.  thr: the wavefront's threshold.  All 64 lanes call it; those
// with `live` false hold no logits.  False: there is no threshold, and nothing
// was folded.
__device__ __forceinline__ bool smx_noisy_chunk(u32x4_t v, int e0, bool live, double T, float inv_T, uint64_t seed,
                                                uint64_t rc, float& m, float& s, int& i, float& thr,
                                                uint32_t* best) {
  float f[8], b[8];
  uint32_t hi[8];
  smx_unpack(v, f);
  const float Tf = (float)T;
  // One limit for the chunk: a logit up to its largest one has a bound below thr
  // unless log2(2^32 - 1 - h) <= 32 + (lmax log2(e) - thr) / T, so that each
  // logit costs its hash and one comparison (a NaN logit makes the maximum, and
  // with it the limit, NaN: everything passes).
  float lmax = f[0];
#pragma unroll
  for (int k = 1; k < 8; ++k) lmax = __builtin_elementwise_maximum(lmax, f[k]);
  const float x = __builtin_amdgcn_exp2f(32.0f + (lmax * kLog2e - thr) * inv_T);
  // thr's slack covers the rounding of the difference, the factor that of the sum
  // and of exp2; two more for the xored bit and the conversion
  const uint32_t lim = x < 4.2e9f ? (uint32_t)(x * 1.002f) + 2u : 0xffffffffu;
  uint64_t z = seed + (rc + (uint64_t)e0 + 1) * 0x9E3779B97F4A7C15ull;
  bool any = false;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    hi[k] = noise_high(z);
    z += 0x9E3779B97F4A7C15ull;
    any |= ~hi[k] <= lim;
  }
  if (!__builtin_amdgcn_ballot_w64(live && any)) return true;
  if (thr == -INFINITY) {  // the wavefront knows no value yet
    float lb = -INFINITY;
#pragma unroll
    for (int k = 0; k < 8; ++k) lb = fmaxf(lb, noise_floor_log2(f[k], Tf, hi[k]));
    thr = noise_threshold(__builtin_amdgcn_exp2f(fminf(wave_max(live ? lb : -INFINITY), 126.0f)), Tf);
    if (thr == -INFINITY) return false;
  }
  uint32_t pend = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    b[k] = noise_bound_log2(f[k], Tf, hi[k]);
    pend |= !(b[k] < thr) ? 1u << k : 0u;
  }
  if (!live) pend = 0;
  while (__builtin_amdgcn_ballot_w64(pend != 0)) {  // each turn clears one bit of every lane that has any
    bool raised = false;
    if (pend != 0) {
      int at = -1;
      float bb = 0.f, l = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const bool take = ((pend >> k) & 1u) && (at < 0 || !(b[k] <= bb));
        at = take ? k : at;
        bb = take ? b[k] : bb;
        l = take ? f[k] : l;
      }
      pend &= ~(1u << at);
      const float x = gumbel_value(l, T, seed, rc + (uint64_t)(e0 + at));
      if (x > m) {
        s = s * fexp2((m - x) * kLog2e) + fexp2((x - x) * kLog2e);
        m = x;
        i = e0 + at;
        raised = true;
      } else if (m != -INFINITY) {
        s += fexp2((x - m) * kLog2e);
        if (x == m) i = min(i, e0 + at);
      }
    }
    if (__builtin_amdgcn_ballot_w64(raised)) {
      const float m_w = wave_max(m);
      thr = fmaxf(thr, noise_threshold(m_w, Tf));
      if ((threadIdx.x & 63) == 0 && m_w > 0.f) atomicMax(best, __float_as_uint(m_w));  // ordered like the value
#pragma unroll
      for (int k = 0; k < 8; ++k) pend &= b[k] < thr ? ~(1u << k) : ~0u;
    }
  }
  return true;
}

// The same for a chunk without a threshold (no value above kNoiseGap is known: a
// small vocabulary, a low temperature, normalised logits): nothing can be left
// out, so all eight are computed, without bounds and one after the other in
// straight code.  On an MI355X, in us, with no bounds anywhere / all through the
// bounds / as it is: 256 x 126464 normal logits of sigma 0.3 at temperature 0.4
// 322 / 444 / 350, of sigma 1 322 / 157 / 136, 256 x 4096 of sigma 1 at 0.4 17.5 /
// 22.7 / 18.9, 1024 x 32000 330 / 290 / 234.
__device__ __forceinline__ void smx_plain_chunk(u32x4_t v, int e0, bool live, double T, uint64_t seed, uint64_t rc,
                                                float& m, float& s, int& i, float& thr, uint32_t* best) {
  float f[8];
  smx_unpack(v, f);
  const uint64_t c0 = rc + (uint64_t)e0;
#pragma unroll
  for (int k = 0; k < 8; ++k) f[k] = gumbel_value(f[k], T, seed, c0 + (uint64_t)k);
  float cm = f[0];
#pragma unroll
  for (int k = 1; k < 8; ++k) cm = fmaxf(cm, f[k]);
  const bool raised = live && cm > m;
  if (raised) {
    s *= fexp2((m - cm) * kLog2e);
    m = cm;
#pragma unroll
    for (int k = 7; k >= 0; --k) i = f[k] == cm ? e0 + k : i;
  }
  if (live && m != -INFINITY) {
    float e[2] = {0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 8; ++k) e[k & 1] += fexp2((f[k] - m) * kLog2e);
    s += e[0] + e[1];
  }
  if (__builtin_amdgcn_ballot_w64(raised)) {
    const float m_w = wave_max(m);
    thr = fmaxf(thr, noise_threshold(m_w, (float)T));
    if ((threadIdx.x & 63) == 0 && m_w > 0.f) atomicMax(best, __float_as_uint(m_w));
  }
}

struct SmxArgs {
  const uint16_t* logits;
  int64_t ld;       // elements between rows
  int M;
  int V;
  int chunks;       // V / 8
  int64_t* x0;
  uint16_t* x0p;
  const double* temp;  // per-row temperature (nullable: no transform)
  uint64_t seed;
  int64_t row_base;
  int n_split;         // workgroups per row
  float* rec;          // [M][n_split][3] records (n_split > 1)
};

// Fold columns [8 c0, 8 c1) of one row into the thread's running (m, s, i):
// thread t takes chunks c0 + t, c0 + t + NT, ..., four 16-byte loads of the
// next batch in flight beside the batch that is summed.
template <int NT>
__device__ __forceinline__ void smx_scan(const SmxArgs& a, int row, int c0, int c1, float& m, float& s, int& idx) {
  constexpr int U = 4;
  const uint16_t* base = a.logits + (int64_t)row * a.ld;
  const u32x4_t ninf = {0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u};
  const int nb = (c1 - c0 + U * NT - 1) / (U * NT);
  if (nb <= 0) return;
  int c = c0 + (int)threadIdx.x;
  u32x4_t v[U];
  // chunks past the end re-read the last one and are replaced by -inf below
#pragma unroll
  for (int u = 0; u < U; ++u) v[u] = ld128_stream(base + 8 * (int64_t)min(c + u * NT, c1 - 1));
  for (int b = 1; b < nb; ++b) {
    u32x4_t w[U];
#pragma unroll
    for (int u = 0; u < U; ++u) w[u] = ld128_stream(base + 8 * (int64_t)min(c + (U + u) * NT, c1 - 1));
    smx_batch<U>(v, c, NT, m, s, idx);
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = w[u];
    c += U * NT;
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (c + u * NT >= c1) v[u] = ninf;
  smx_batch<U>(v, c, NT, m, s, idx);
}

// The same for a row with temperature T > 0 (smx_noisy_chunk).  Whole
// wavefronts walk together: their lanes share a threshold.
template <int NT>
__device__ __forceinline__ void smx_scan_noisy(const SmxArgs& a, int row, int c0, int c1, float& m, float& s,
                                               int& idx) {
  const uint16_t* base = a.logits + (int64_t)row * a.ld;
  const u32x4_t ninf = {0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u};
  const double T = a.temp[row];
  const uint64_t rc = (uint64_t)(a.row_base + row) * (uint64_t)a.V;
  float thr = -INFINITY;
  bool plain = false;  // no threshold was found, nothing can be left out
  const float inv_T = 1.0f / (float)T;
  const int lead = (int)(threadIdx.x & 63);
  __shared__ uint32_t best;  // the largest value computed, as bits (0: none)
  if (threadIdx.x == 0) best = 0;
  __syncthreads();
  // one chunk at a time, the next one's load in flight: the chunk's code with its
  // f64 functions is long, and a second copy of it costs instruction fetches
  auto load = [&](int c) { return c < c1 ? ld128_stream(base + 8 * (int64_t)c) : ninf; };
  int c = c0 + (int)threadIdx.x;
  u32x4_t v = load(c);
#pragma unroll 1
  for (; c - lead < c1; c += NT) {
    const u32x4_t next = load(c + NT);
    const float known = __uint_as_float(__hip_atomic_load(&best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
    if (known > 0.f) thr = fmaxf(thr, noise_threshold(known, (float)T));
    plain = plain && thr == -INFINITY;
    if (!plain) plain = !smx_noisy_chunk(v, 8 * c, c < c1, T, inv_T, a.seed, rc, m, s, idx, thr, &best);
    if (plain) smx_plain_chunk(v, 8 * c, c < c1, T, a.seed, rc, m, s, idx, thr, &best);
    v = next;
  }
}

// Merge the workgroup's per-thread records; every thread returns the result.
template <int NT>
__device__ __forceinline__ void smx_block_reduce(float& m, float& s, int& idx) {
  __shared__ float red_m[NT / 64];
  __shared__ float red_s[NT / 64];
  __shared__ int red_i[NT / 64];
  smx_wave_reduce(m, s, idx);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) {
    red_m[wave] = m;
    red_s[wave] = s;
    red_i[wave] = idx;
  }
  __syncthreads();
  m = -INFINITY;
  s = 0.f;
  idx = INT_MAX;
  if (lane < NT / 64) {
    m = red_m[lane];
    s = red_s[lane];
    idx = red_i[lane];
  }
  smx_wave_reduce(m, s, idx);
}

// x0 / x0_p of one row from its merged (m, s, first index of m), by one
// wavefront: the probability of the maximum is bf16(1/s); when |m| <= 2 an
// earlier column may round to the same probability, so the columns before
// the first maximum are rescanned for the earliest such one.
__device__ void smx_finish(const SmxArgs& a, int row, float m, float s, int idx) {
  const int lane = threadIdx.x & 63;
  const uint32_t P = f32_to_bf16_bits(1.0f / s);
  int best = idx;
  if (fabsf(m) <= 2.0f && idx != INT_MAX && idx > 0) {
    // earliest column j < idx with bf16(exp(v_j - m) / s) == P
    const uint16_t* base = a.logits + (int64_t)row * a.ld;
    const float thr = m - 0.015625f;
    int found = INT_MAX;
    const int nch = (idx + 7) >> 3;
    const double T = a.temp ? a.temp[row] : 0.0;
    const uint64_t rc = (uint64_t)(a.row_base + row) * (uint64_t)a.V;
    for (int c = lane; c < nch; c += 64) {
      const u32x4_t v = ld128(base + 8 * (int64_t)c);
#pragma unroll
      for (int k = 7; k >= 0; --k) {
        const uint32_t w = v[k >> 1];
        float f = (k & 1) ? __uint_as_float(w & 0xffff0000u) : __uint_as_float(w << 16);
        if (T > 0.0) f = gumbel_value(f, T, a.seed, rc + (uint64_t)(8 * c + k));
        const int j = 8 * c + k;
        if (j < idx && f >= thr && f32_to_bf16_bits(expf(f - m) / s) == P) found = min(found, j);
      }
    }
    found = min(found, (int)lane_xor((uint32_t)found, 32));
    found = min(found, (int)lane_xor((uint32_t)found, 16));
    found = min(found, (int)lane_xor((uint32_t)found, 8));
    found = min(found, (int)lane_xor((uint32_t)found, 4));
    found = min(found, (int)lane_xor((uint32_t)found, 2));
    found = min(found, (int)lane_xor((uint32_t)found, 1));
    best = min(best, found);
  }
  if (lane == 0) {
    a.x0[row] = best == INT_MAX ? 0 : best;
    a.x0p[row] = (uint16_t)P;
  }
}

// One workgroup per row (n_split = 1: scan, merge and finish in one launch) or
// n_split of them, each a range of the row's chunks; their records (m, s, i)
// then go to `rec` and smx_merge_kernel finishes the rows.
template <bool GUMBEL, int NT>
__global__ __launch_bounds__(NT) void smx_row_kernel(SmxArgs a) {
  const int row = blockIdx.x / a.n_split;
  const int sp = blockIdx.x - row * a.n_split;
  const int per = (a.chunks + a.n_split - 1) / a.n_split;
  const int c0 = sp * per, c1 = min(a.chunks, c0 + per);
  float m = -INFINITY, s = 0.f;
  int idx = INT_MAX;
  if (GUMBEL && a.temp[row] > 0.0)
    smx_scan_noisy<NT>(a, row, c0, c1, m, s, idx);
  else
    smx_scan<NT>(a, row, c0, c1, m, s, idx);
  smx_block_reduce<NT>(m, s, idx);
  if (a.n_split > 1) {
    if (threadIdx.x == 0) {
      float* r = a.rec + 3 * (int64_t)blockIdx.x;
      r[0] = m;
      r[1] = s;
      r[2] = __int_as_float(idx);
    }
  } else if ((threadIdx.x >> 6) == 0) {
    smx_finish(a, row, m, s, idx);
  }
}

// The records of a row's n_split (at most 64) ranges merged, one wavefront per row.
__global__ __launch_bounds__(256) void smx_merge_kernel(SmxArgs a) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= a.M) return;
  float m = -INFINITY, s = 0.f;
  int idx = INT_MAX;
  if (lane < a.n_split) {
    const float* r = a.rec + 3 * ((int64_t)row * a.n_split + lane);
    m = r[0];
    s = r[1];
    idx = __float_as_int(r[2]);
  }
  smx_wave_reduce(m, s, idx);
  smx_finish(a, row, m, s, idx);
}

// Workgroups per row.  A CU takes in at most ~26 KB a microsecond, ~10 us for a
// row of 253 KB, so few rows are spread over several CUs; the second launch
// (~2.5 us) pays for that up to 64 rows, and with noise, whose integer hash
// keeps a CU busy for 35 us a row, wherever CUs would stay idle.  Measured at
// 126464 logits per row, one workgroup a row against the split: 8 rows 12.3 /
// 7.8, 32 12.5 / 8.5, 64 12.3 / 9.8, 96 12.4 / 11.6, 128 12.6 / 12.1 us (not
// split); with noise 8 rows 35 / 10.9, 64 35 / 19.9, 128 35 / 26.0 us.  A range
// is at least 512 chunks (noise: 256; twice and four times as many ranges:
// 20.8 and 21.7 us at 64 rows).
static int smx_splits(int M, int V, bool noisy) {
  if (M <= 0) return 1;
  int n = noisy ? min(32, 256 / M) : M <= 64 ? min(8, 256 / M) : 1;
  n = min(n, V / 8 / (noisy ? 256 : 512));
  return n < 1 ? 1 : n;
}

// ---- K9 ---------------------------------------------------------------------

struct UnmaskArgs {
  int64_t* tokens;
  int64_t n_tokens;       // elements of tokens (bounds guard)
  const int32_t* params;  // [n_seq][5]: tok_off, win_len, row_off, steps_remain, first_rule
  const int64_t* x0;
  const uint16_t* conf;
  int64_t n_rows;         // rows of x0 / conf (bounds guard)
  int64_t mask_id;
  int max_win;
  int32_t* n_unmasked;    // nullable
};

// Order-preserving map of bf16 bits to 16-bit unsigned (-0 equals +0).
__device__ __forceinline__ uint32_t conf_order(uint32_t b) {
  if (b == 0x8000u) b = 0;
  return (b & 0x8000u) ? (~b & 0xffffu) : (b | 0x8000u);
}

__device__ __forceinline__ int block_sum(int v, int* red) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += (int)lane_xor((uint32_t)v, off);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}

__global__ __launch_bounds__(256) void lowconf_unmask_kernel(UnmaskArgs a) {
  __shared__ uint32_t keys[kUnmaskMaxWin];
  __shared__ int red[4];
  const int b = blockIdx.x;
  const int32_t* p = a.params + 5 * (int64_t)b;
  const int64_t tok_off = p[0];
  const int n = min(min(p[1], a.max_win), kUnmaskMaxWin);
  const int64_t r0 = p[2];
  const int sr = p[3];
  const bool first_rule = p[4] != 0;
  const int tid = threadIdx.x;
  const bool valid = n > 0 && tok_off >= 0 && tok_off + n <= a.n_tokens && r0 >= 0 && r0 + n <= a.n_rows;
  if (!valid) {  // uniform per workgroup
    if (a.n_unmasked && tid == 0) a.n_unmasked[b] = 0;
    return;
  }
  int64_t* tok = a.tokens + tok_off;
  int cnt = 0;
  for (int j = tid; j < n; j += 256) {
    const bool masked = tok[j] == a.mask_id;
    keys[j] = masked ? ((conf_order(a.conf[r0 + j]) << 16) | (0xffffu - (uint32_t)j)) : 0u;
    cnt += masked;
  }
  const int nmask = block_sum(cnt, red);  // its barriers also publish keys[]
  // steps_remain <= 0: nothing is unmasked (the reference divides by it)
  int k = sr > 0 ? min((nmask + sr - 1) / sr, nmask) : 0;
  const int k_total = k;
  if (first_rule && k > 0 && keys[0] != 0u) {
    __syncthreads();  // every thread has read keys[0]
    if (tid == 0) {
      tok[0] = a.x0[r0];
      keys[0] = 0u;
    }
    --k;
    __syncthreads();
  }
  if (k > 0) {
    uint32_t T = 0;
    for (int bit = 31; bit >= 0; --bit) {
      const uint32_t cand = T | (1u << bit);
      int c = 0;
      for (int j = tid; j < n; j += 256) c += keys[j] >= cand;
      if (block_sum(c, red) >= k) T = cand;
    }
    // keys are distinct and the k-th largest is non-zero: exactly k pass
    for (int j = tid; j < n; j += 256)
      if (keys[j] >= T) tok[j] = a.x0[r0 + j];
  }
  if (a.n_unmasked && tid == 0) a.n_unmasked[b] = k_total;
}

// K9 for windows of at most 64 * KPL positions: one wavefront per sequence,
// KPL keys per lane in registers (position j = 64 i + lane).  The kernel is a
// chain of latencies (parameters, tokens and confidences, x0); the bitwise
// search's 32 counts were the longest part of it as workgroup sums (two
// barriers each), and are ballots and scalar bit counts here, with x0 loaded
// beside the confidences.  8 windows of 32 positions on an MI355X: 11.2 -> 3.3 us
// in a loop of this launch alone, 11.5 -> 3.9 traced inside a sampling step.
template <int KPL>
__global__ __launch_bounds__(64) void lowconf_unmask_wave_kernel(UnmaskArgs a) {
  const int b = blockIdx.x;
  const int32_t* p = a.params + 5 * (int64_t)b;
  const int64_t tok_off = p[0];
  const int n = min(min(p[1], a.max_win), 64 * KPL);
  const int64_t r0 = p[2];
  const int sr = p[3];
  const bool first_rule = p[4] != 0;
  const int lane = threadIdx.x;
  const bool valid = n > 0 && tok_off >= 0 && tok_off + n <= a.n_tokens && r0 >= 0 && r0 + n <= a.n_rows;
  if (!valid) {
    if (a.n_unmasked && lane == 0) a.n_unmasked[b] = 0;
    return;
  }
  int64_t* tok = a.tokens + tok_off;
  int64_t t[KPL], x0[KPL];
  uint32_t key[KPL];
#pragma unroll
  for (int i = 0; i < KPL; ++i) {
    const int j = min(64 * i + lane, n - 1);  // lanes past the window re-read its last position
    t[i] = tok[j];
    key[i] = a.conf[r0 + j];
    x0[i] = a.x0[r0 + j];
  }
  int nmask = 0;
#pragma unroll
  for (int i = 0; i < KPL; ++i) {
    const int j = 64 * i + lane;
    const bool masked = j < n && t[i] == a.mask_id;
    key[i] = masked ? ((conf_order(key[i]) << 16) | (0xffffu - (uint32_t)j)) : 0u;
    nmask += __builtin_popcountll(__builtin_amdgcn_ballot_w64(masked));
  }
  // steps_remain <= 0: nothing is unmasked (the reference divides by it)
  int k = sr > 0 ? min((nmask + sr - 1) / sr, nmask) : 0;
  const int k_total = k;
  const bool first = first_rule && k > 0 && __builtin_amdgcn_readfirstlane((int)key[0]) != 0;
  if (first) {  // position 0 goes first, the others share the rest
    if (lane == 0) {
      tok[0] = x0[0];
      key[0] = 0u;
    }
    --k;
  }
  if (k > 0) {
    uint32_t T = 0;
    for (int bit = 31; bit >= 0; --bit) {
      const uint32_t cand = T | (1u << bit);
      int c = 0;
#pragma unroll
      for (int i = 0; i < KPL; ++i) c += __builtin_popcountll(__builtin_amdgcn_ballot_w64(key[i] >= cand));
      if (c >= k) T = cand;
    }
    // keys are distinct and the k-th largest is non-zero: exactly k pass
#pragma unroll
    for (int i = 0; i < KPL; ++i)
      if (key[i] >= T) tok[64 * i + lane] = x0[i];
  }
  if (a.n_unmasked && lane == 0) a.n_unmasked[b] = k_total;
}

}  // namespace dllm

using namespace dllm;

extern "C" size_t dllm_softmax_max_workspace_size(int M, int V) {
  (void)M;
  (void)V;
  return 0;  // nothing is required
}

extern "C" size_t dllm_softmax_max_split_workspace_size(int M, int V) {
  // the noisy form's ranges are the most
  const int n = M > 0 && V > 0 ? max(smx_splits(M, V, true), smx_splits(M, V, false)) : 1;
  return n > 1 ? (size_t)M * n * 3 * sizeof(float) : 0;
}

static int softmax_max_launch(const char* name, const uint16_t* logits, int64_t ld, int M, int V,
                              const double* row_temperature, uint64_t seed, int64_t row_base, int64_t* x0,
                              uint16_t* x0_p, void* workspace, size_t workspace_bytes, void* stream) {
  if (M < 0 || V < 0) return fail(DLLM_ERR_INVALID_ARG, "%s: negative size", name);
  if (M == 0) return DLLM_OK;
  if (V == 0 || V % 8 != 0)
    return fail(DLLM_ERR_UNSUPPORTED, "%s: vocabulary size %d must be a positive multiple of 8", name, V);
  if (!logits || !x0 || !x0_p) return fail(DLLM_ERR_INVALID_ARG, "%s: null pointer", name);
  if (!aligned16(logits) || ld % 8 != 0 || ld < V)
    return fail(DLLM_ERR_INVALID_ARG, "%s: logits must be 16-byte aligned with a row stride >= V and a multiple of 8",
                name);
  SmxArgs a;
  a.logits = logits;
  a.ld = ld;
  a.M = M;
  a.V = V;
  a.chunks = V / 8;
  a.x0 = x0;
  a.x0p = x0_p;
  a.temp = row_temperature;
  a.seed = seed;
  a.row_base = row_base;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // without a workspace that holds the records every row is one workgroup's
  a.n_split = smx_splits(M, V, row_temperature != nullptr);
  a.rec = reinterpret_cast<float*>(workspace);
  if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 4 ||
      workspace_bytes < (size_t)M * a.n_split * 3 * sizeof(float) || (int64_t)M * a.n_split > INT32_MAX)
    a.n_split = 1;
  const dim3 grid((unsigned)(M * a.n_split));
  // Threads per row.  Measured in us, 1024 / 512 / 256 threads: 8 rows 13.3 /
  // 13.1 / 16.4, 256 rows 17.1 / 15.1 / 17.1, 384 rows 28.7 / 24.7 / 23.4, 1024
  // rows 59.2 / 47.0 / 45.8.  Noisy rows are bound by the hash: as many
  // wavefronts as the rows leave room for.
  if (row_temperature) {
    if (M <= 512)
      smx_row_kernel<true, 1024><<<grid, dim3(1024), 0, st>>>(a);
    else
      smx_row_kernel<true, 256><<<grid, dim3(256), 0, st>>>(a);
  } else {
    if (M <= 256)
      smx_row_kernel<false, 512><<<grid, dim3(512), 0, st>>>(a);
    else
      smx_row_kernel<false, 256><<<grid, dim3(256), 0, st>>>(a);
  }
  int rc = check_launch(name);
  if (rc == DLLM_OK && a.n_split > 1) {
    smx_merge_kernel<<<dim3((unsigned)((M + 3) / 4)), dim3(256), 0, st>>>(a);
    rc = check_launch(name);
  }
  return rc;
}

extern "C" int dllm_softmax_max(const uint16_t* logits, int64_t ld, int M, int V, int64_t* x0, uint16_t* x0_p,
                                void* workspace, size_t workspace_bytes, void* stream) {
  return softmax_max_launch("dllm_softmax_max", logits, ld, M, V, nullptr, 0, 0, x0, x0_p, workspace, workspace_bytes,
                            stream);
}

extern "C" int dllm_softmax_max_sample(const uint16_t* logits, int64_t ld, int M, int V,
                                       const double* row_temperature, uint64_t seed, int64_t row_base, int64_t* x0,
                                       uint16_t* x0_p, void* workspace, size_t workspace_bytes, void* stream) {
  if (row_base < 0) return fail(DLLM_ERR_INVALID_ARG, "dllm_softmax_max_sample: negative row_base");
  return softmax_max_launch("dllm_softmax_max_sample", logits, ld, M, V, row_temperature, seed, row_base, x0, x0_p,
                            workspace, workspace_bytes, stream);
}

extern "C" int dllm_lowconf_unmask(int64_t* tokens, int64_t n_tokens, const int32_t* seq_params, int n_seq,
                                   int max_win, const int64_t* x0, const uint16_t* conf, int64_t n_rows,
                                   int64_t mask_id, int32_t* n_unmasked, void* stream) {
  static const char* name = "dllm_lowconf_unmask";
  if (n_seq < 0 || max_win < 0 || n_tokens < 0 || n_rows < 0)
    return fail(DLLM_ERR_INVALID_ARG, "%s: negative size", name);
  if (n_seq == 0) return DLLM_OK;
  if (max_win > kUnmaskMaxWin)
    return fail(DLLM_ERR_UNSUPPORTED, "%s: window of %d positions exceeds %d", name, max_win, kUnmaskMaxWin);
  if (!tokens || !seq_params || (n_rows > 0 && (!x0 || !conf)))
    return fail(DLLM_ERR_INVALID_ARG, "%s: null pointer", name);
  UnmaskArgs a;
  a.tokens = tokens;
  a.n_tokens = n_tokens;
  a.params = seq_params;
  a.x0 = x0;
  a.conf = conf;
  a.n_rows = n_rows;
  a.mask_id = mask_id;
  a.max_win = max_win;
  a.n_unmasked = n_unmasked;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)n_seq);
  // One wavefront holds windows of up to 1024 positions in registers (16 keys
  // a lane); longer ones need the workgroup's LDS.
  if (max_win <= 64)
    lowconf_unmask_wave_kernel<1><<<grid, dim3(64), 0, st>>>(a);
  else if (max_win <= 256)
    lowconf_unmask_wave_kernel<4><<<grid, dim3(64), 0, st>>>(a);
  else if (max_win <= 1024)
    lowconf_unmask_wave_kernel<16><<<grid, dim3(64), 0, st>>>(a);
  else
    lowconf_unmask_kernel<<<grid, dim3(256), 0, st>>>(a);
  return check_launch(name);
}
