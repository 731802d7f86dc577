// Device-side KV precision admission for gfx950: the rate-distortion
// sensitivity proxy and the closed-form budget solver of
// shadowinfer/shadowkv/rd_allocator.py (kv_sensitivity :47-61,
// predict_codes_bytes :173-188, admit_codes :190-318).
//
// admit_codes ranks eligible token-heads by ascending score (importance x
// sensitivity, stable on the token-major index), walks the ranking with
// prefix sums of the bytes each entry saves, and cuts at the first prefix
// that covers the excess over the budget (a partial downgrade for the entry
// at the cut), then optionally evicts a second prefix. Only the cut entry
// matters, so the device never sorts: a weighted radix select over the
// score keys (digits of 11, 11 and 10 bits, most significant first) finds the
// key of the cut entry, a scan over the entries with that key (in index order, as
// a stable sort leaves them) finds the entry itself, and one pass rewrites the
// codes of everything ranked before it. Every step is an integer sum, so the
// cut is exact.
//
// One layer's 262144 entries are 1.5 MB: the time is launches, round trips and
// contended atomics, not bytes. So every block of a pass takes the step before
// it by itself (picks the digit from the histogram of the last pass, the entry
// from the chunk sums) instead of one block in a launch of its own, the first
// digit's histogram is part of the pass before it, threads load four entries at
// once, and at most kAdmBlocks blocks add to the same few counters: 10 launches
// for 30. (Handing over to the last block of a pass instead took as long as the
// 30 launches: its device-scope fences write back and drop the L2s, 20 us each.)
// The solver with eviction at 8192 x 32: 195 -> 55 us of kernels.
#include "si_common.h"

namespace si {
namespace {

constexpr int ADM_THREADS = 1024;
// A block per CU. The solver with eviction in us, by the most blocks that add to
// the counters (and with one launch per step and 2048 small blocks, before):
//   entries   64   128   256   512  before
//     1.0 M   82    70    71    72     295
//     4.2 M  250   154   121   133     341
//      17 M  951   540   344   299     602
constexpr int64_t kAdmBlocks = 256;
constexpr int TIE_CHUNK = 2 * ADM_THREADS;  // entries per block of the tie scan
constexpr int BINS = 2048;                  // of a digit's histogram
constexpr int MODE_DOWN = 0;     // ladder downgrade (fp32 -> fp16 -> int8 -> int4)
constexpr int MODE_EVICT = 1;    // eviction of the remaining bytes

struct AdmCosts {
  long long cost[5];   // bytes of one token-head per code (K + V with scales)
  long long delta[3];  // cost[c] - cost[c + 1]
};

// What a step of a selection leaves for the next pass.
struct Sel {
  unsigned long long R;  // weight the cut still has to cover
  unsigned int prefix;   // key bits fixed so far; the cut key after three digits
  int active;            // the selection runs
  int all;               // the whole ranking is inside the cut
};

struct AdmState {
  unsigned long long pred[2];  // total bytes after prep, downgrade
  unsigned long long ncand;    // eligible entries
  long long budget;            // bytes allowed (may be negative)
  int bad;                     // codes outside 0..4 were seen
  Sel sel[2][3];               // by mode, after each digit
};

// Bytes an entry of code c frees when taken down the ladder to int4.
__device__ __forceinline__ long long ladder_savings(const AdmCosts& cs, int c) {
  long long s = 0;
  for (int x = c; x < 3; ++x) s += cs.delta[x];
  return c >= 0 ? s : 0;
}

__device__ __forceinline__ unsigned long long weight(const AdmCosts& cs, int mode, int c) {
  if (c < 0 || c > 4) return 0;
  return (unsigned long long)(mode == MODE_DOWN ? ladder_savings(cs, c) : cs.cost[c]);
}

// Order-preserving key of an fp32 score: ascending keys = ascending scores,
// -0 == +0, NaN above +inf (torch.argsort puts NaN last).
__device__ __forceinline__ unsigned int score_key(float x) {
  if (x != x) return 0xffffffffu;
  if (x == 0.0f) x = 0.0f;
  const unsigned int u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

template <typename T>
__device__ __forceinline__ T block_sum(T v, T* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  const int wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  T s = 0;
  for (int w = 0; w < nw; ++w) s += red[w];
  return s;
}

// Inclusive scan of one value per thread over the block's 1024 threads.
__device__ __forceinline__ unsigned long long block_scan(unsigned long long v,
                                                         unsigned long long* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  __syncthreads();
  if (lane == 63) red[wave] = v;
  __syncthreads();
  for (int w = 0; w < wave; ++w) v += red[w];
  return v;
}

// Digit d of a key (0: bits 31..21, 1: 20..10, 2: 9..0) and the key bits above it.
__device__ __forceinline__ unsigned int digit_of(unsigned int k, int d) {
  return d == 0 ? k >> 21 : d == 1 ? (k >> 10) & 2047u : k & 1023u;
}
__device__ __forceinline__ unsigned int above_digit(unsigned int k, int d) {
  return d == 1 ? k >> 21 : k >> 10;  // d = 1 or 2
}

// Entries i .. i+3 of an array (zeros past n), in one load where p is aligned.
struct Four {
  unsigned int v[4];
};
template <typename T>
__device__ __forceinline__ Four load4(const T* p, int64_t i, int64_t n) {
  Four f;
  if (i + 4 <= n && (reinterpret_cast<uintptr_t>(p + i) & (4 * sizeof(T) - 1)) == 0) {
    if constexpr (sizeof(T) == 1) {
      const unsigned int w = *reinterpret_cast<const unsigned int*>(p + i);
#pragma unroll
      for (int e = 0; e < 4; ++e) f.v[e] = (unsigned int)(int)(T)(w >> (8 * e));
    } else {
      const uint4 w = *reinterpret_cast<const uint4*>(p + i);
      f.v[0] = w.x; f.v[1] = w.y; f.v[2] = w.z; f.v[3] = w.w;
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (sizeof(T) == 1) f.v[e] = i + e < n ? (unsigned int)(int)p[i + e] : 0u;
      else f.v[e] = i + e < n ? __builtin_bit_cast(unsigned int, p[i + e]) : 0u;
    }
  }
  return f;
}
__device__ __forceinline__ void store4(int8_t* p, int64_t i, int64_t n, const int (&c)[4]) {
  if (i + 4 <= n && (reinterpret_cast<uintptr_t>(p + i) & 3) == 0) {
    *reinterpret_cast<unsigned int*>(p + i) = (c[0] & 255) | (c[1] & 255) << 8 |
                                              (c[2] & 255) << 16 | (unsigned int)(c[3] & 255) << 24;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (i + e < n) p[i + e] = (int8_t)c[e];
  }
}

__global__ __launch_bounds__(ADM_THREADS) void adm_init(AdmState* st, unsigned long long* hist,
                                                        long long budget, int64_t* result) {
  for (int i = threadIdx.x; i < 6 * BINS; i += blockDim.x) hist[i] = 0;
  if (threadIdx.x == 0) {
    st->pred[0] = st->pred[1] = st->ncand = 0;
    st->budget = budget;
    st->bad = 0;
  }
  if (threadIdx.x < 3) result[threadIdx.x] = 0;
}

// The bin of a histogram that holds the cut: the first where the running weight
// reaches R (which then is what the cut still covers inside it). False in every
// thread when all bins together weigh less.
__device__ __forceinline__ bool pick_digit(const unsigned long long* __restrict__ hist,
                                           unsigned long long& R, unsigned int& bin,
                                           unsigned long long* red) {
  __shared__ unsigned long long left;
  __shared__ int hit;
  const int b = 2 * threadIdx.x;
  const unsigned long long w0 = hist[b], w1 = hist[b + 1];
  if (threadIdx.x == 0) hit = -1;
  const unsigned long long cum = block_scan(w0 + w1, red), before = cum - w0 - w1;
  if (before < R && cum >= R) {
    const bool second = before + w0 < R;
    hit = b + (second ? 1 : 0);
    left = R - before - (second ? w0 : 0);
  }
  __syncthreads();
  const bool found = hit >= 0;
  if (found) {
    bin = (unsigned int)hit;
    R = left;
  }
  return found;
}

// The selection after its digit d: the downgrade cuts the excess of the initial
// bytes over the budget, the eviction the excess left after the downgrade. The
// same in every block; the first leaves it for the next pass.
__device__ __forceinline__ Sel step_sel(AdmState* st, int mode, int d,
                                        const unsigned long long* __restrict__ hist,
                                        unsigned long long* red) {
  Sel s;
  if (d == 0) {
    const long long p = (long long)st->pred[mode], budget = st->budget;
    s.active = st->ncand > 0 && st->bad == 0 && p > budget;
    s.all = 0;
    s.prefix = 0;
    s.R = s.active ? (unsigned long long)p - (unsigned long long)budget : 0;
  } else {
    s = st->sel[mode][d - 1];
  }
  if (s.active && !s.all) {
    unsigned int bin = 0;
    if (pick_digit(hist + (3 * mode + d) * BINS, s.R, bin, red))
      s.prefix = (s.prefix << (d == 2 ? 10 : 11)) | bin;
    else
      s.all = 1;  // every candidate together saves less than the excess (d = 0)
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) st->sel[mode][d] = s;
  return s;
}

// Adds a block's LDS histogram to the global one.
__device__ __forceinline__ void flush_hist(const unsigned long long* lh, unsigned long long* hist) {
  __syncthreads();
  for (int b = threadIdx.x; b < BINS; b += ADM_THREADS)
    if (lh[b] != 0) atomicAdd(&hist[b], lh[b]);
}

// Sums the codes' bytes, and computes each entry's score key and eligibility
// (not a sink token, not protected) and the first digit's histogram of the
// downgrade's weights. out: where the call ends here (no budget), a copy of the
// codes.
__global__ __launch_bounds__(ADM_THREADS) void adm_prep(
    const int8_t* __restrict__ codes, int8_t* __restrict__ out, int64_t n, int64_t first,
    const float* __restrict__ imp, const float* __restrict__ sens,
    const uint8_t* __restrict__ prot, AdmCosts cs, unsigned int* __restrict__ key,
    uint8_t* __restrict__ cand, unsigned long long* __restrict__ hist, AdmState* st,
    int64_t* __restrict__ result) {
  __shared__ unsigned long long red[ADM_THREADS / 64];
  __shared__ unsigned long long lh[BINS];
  for (int b = threadIdx.x; b < BINS; b += ADM_THREADS) lh[b] = 0;
  __syncthreads();
  unsigned long long bytes = 0, nc = 0;
  int bad = 0;
  for (int64_t i = 4 * ((int64_t)blockIdx.x * ADM_THREADS + threadIdx.x); i < n;
       i += 4 * (int64_t)gridDim.x * ADM_THREADS) {
    const Four c4 = load4(codes, i, n), m4 = load4(imp, i, n);
    Four s4 = {}, p4 = {};
    if (sens != nullptr) s4 = load4(sens, i, n);
    if (prot != nullptr) p4 = load4(prot, i, n);
    int c[4];
    unsigned int k[4], el = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      c[e] = (int)c4.v[e];
      const float m = __uint_as_float(m4.v[e]);
      k[e] = score_key(sens != nullptr ? m * __uint_as_float(s4.v[e]) : m);
      if (i + e >= n) continue;
      if (c[e] < 0 || c[e] > 4) bad = 1;
      else bytes += (unsigned long long)cs.cost[c[e]];
      if (i + e < first || p4.v[e] != 0) continue;
      el |= 1u << (8 * e);
      ++nc;
      const unsigned long long w = weight(cs, MODE_DOWN, c[e]);
      if (w != 0) atomicAdd(&lh[digit_of(k[e], 0)], w);
    }
    if (out != nullptr) store4(out, i, n, c);
    // key and cand are padded to whole groups of four
    *reinterpret_cast<uint4*>(key + i) = make_uint4(k[0], k[1], k[2], k[3]);
    *reinterpret_cast<unsigned int*>(cand + i) = el;
  }
  flush_hist(lh, hist);
  bytes = block_sum(bytes, red);
  nc = block_sum(nc, red);
  const int any_bad = __syncthreads_or(bad);
  if (threadIdx.x == 0) {
    atomicAdd(&st->pred[0], bytes);
    atomicAdd(&st->ncand, nc);
    if (any_bad) {
      atomicOr(&st->bad, 1);
      atomicOr(reinterpret_cast<unsigned long long*>(result) + 2, 1ull);
    }
    if (out != nullptr) atomicAdd(reinterpret_cast<unsigned long long*>(result), bytes);
  }
}

// Picks digit d - 1, then makes the weight histogram of digit d (1 or 2) over the
// candidates whose higher digits equal the ones already fixed.
__global__ __launch_bounds__(ADM_THREADS) void adm_hist(
    int mode, int d, const unsigned int* __restrict__ key, const uint8_t* __restrict__ cand,
    const int8_t* __restrict__ codes, int64_t n, AdmCosts cs, unsigned long long* __restrict__ hist,
    AdmState* st) {
  __shared__ unsigned long long red[ADM_THREADS / 64];
  __shared__ unsigned long long lh[BINS];
  for (int b = threadIdx.x; b < BINS; b += ADM_THREADS) lh[b] = 0;
  const Sel s = step_sel(st, mode, d - 1, hist, red);
  if (!s.active || s.all) return;
  __syncthreads();
  for (int64_t i = 4 * ((int64_t)blockIdx.x * ADM_THREADS + threadIdx.x); i < n;
       i += 4 * (int64_t)gridDim.x * ADM_THREADS) {
    const Four k4 = load4(key, i, n), e4 = load4(cand, i, n), c4 = load4(codes, i, n);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (above_digit(k4.v[e], d) != s.prefix || e4.v[e] == 0) continue;
      const unsigned long long w = weight(cs, mode, (int)c4.v[e]);
      if (w != 0) atomicAdd(&lh[digit_of(k4.v[e], d)], w);
    }
  }
  flush_hist(lh, hist + (3 * mode + d) * BINS);
}

// Weight of the candidates with the cut key among entries i .. i+1.
__device__ __forceinline__ void tied_pair(int mode, unsigned int tau, int64_t i, int64_t n,
                                          const unsigned int* __restrict__ key,
                                          const uint8_t* __restrict__ cand,
                                          const int8_t* __restrict__ codes, const AdmCosts& cs,
                                          unsigned long long& w0, unsigned long long& w1) {
  w0 = w1 = 0;
  const bool a = i < n, b = i + 1 < n;
  const unsigned int k0 = a ? key[i] : 0, k1 = b ? key[i + 1] : 0;
  const int e0 = a ? cand[i] : 0, e1 = b ? cand[i + 1] : 0;
  const int c0 = a ? codes[i] : 0, c1 = b ? codes[i + 1] : 0;
  if (e0 && k0 == tau) w0 = weight(cs, mode, c0);
  if (e1 && k1 == tau) w1 = weight(cs, mode, c1);
}

// Picks the last digit, then sums per chunk the weight of the candidates whose
// key equals the cut key.
__global__ __launch_bounds__(ADM_THREADS) void adm_tie(
    int mode, const unsigned int* __restrict__ key, const uint8_t* __restrict__ cand,
    const int8_t* __restrict__ codes, int64_t n, AdmCosts cs,
    const unsigned long long* __restrict__ hist, unsigned long long* __restrict__ blk,
    AdmState* st) {
  __shared__ unsigned long long red[ADM_THREADS / 64];
  const Sel s = step_sel(st, mode, 2, hist, red);
  if (!s.active || s.all) return;
  unsigned long long w0, w1;
  tied_pair(mode, s.prefix, (int64_t)blockIdx.x * TIE_CHUNK + 2 * threadIdx.x, n, key, cand, codes,
            cs, w0, w1);
  const unsigned long long sum = block_sum(w0 + w1, red);
  if (threadIdx.x == 0) blk[blockIdx.x] = sum;
}

// The cut entry among the candidates with the cut key, in index order: the chunk
// whose running weight reaches R, then the entry inside it (two consecutive
// entries per thread); rem: the excess left when the ranking reaches it.
__device__ __forceinline__ void cut_entry(int mode, const Sel& s,
                                          const unsigned int* __restrict__ key,
                                          const uint8_t* __restrict__ cand,
                                          const int8_t* __restrict__ codes, int64_t n,
                                          const AdmCosts& cs,
                                          const unsigned long long* __restrict__ blk, int64_t nblk,
                                          unsigned long long* red, long long& b_idx,
                                          long long& rem) {
  __shared__ long long found, at;
  __shared__ unsigned long long left, so_far, excess;
  const int t = threadIdx.x;
  if (t == 0) found = at = -1;
  unsigned long long carry = 0;
  for (int64_t c0 = 0; c0 < nblk; c0 += ADM_THREADS) {
    const unsigned long long v = c0 + t < nblk ? blk[c0 + t] : 0;
    const unsigned long long inc = block_scan(v, red) + carry;
    if (inc >= s.R && inc - v < s.R) {
      found = c0 + t;
      left = s.R - (inc - v);  // weight left inside the chunk
    }
    if (t == ADM_THREADS - 1) so_far = inc;
    __syncthreads();
    if (found >= 0) break;
    carry = so_far;
    __syncthreads();
  }
  const long long chunk = found;
  if (chunk >= 0) {  // always: the digits guarantee enough weight
    const unsigned long long r = left;
    const int64_t i0 = chunk * TIE_CHUNK + 2 * t;
    unsigned long long w0, w1;
    tied_pair(mode, s.prefix, i0, n, key, cand, codes, cs, w0, w1);
    const unsigned long long inc = block_scan(w0 + w1, red), exc = inc - w0 - w1;
    if (exc < r && exc + w0 >= r) {
      at = i0;
      excess = r - exc;
    } else if (exc + w0 < r && inc >= r) {
      at = i0 + 1;
      excess = r - exc - w0;
    }
  }
  __syncthreads();
  b_idx = at;
  rem = at >= 0 ? (long long)excess : 0;
}

// Finds the cut entry, rewrites the codes of the candidates ranked before it
// (and its own) from `codes` to `out`, and sums the new total bytes. The
// downgrade before an eviction (result null) also makes the first digit's
// histogram of the eviction's weights.
__global__ __launch_bounds__(ADM_THREADS) void adm_apply(
    int mode, const unsigned int* __restrict__ key, const uint8_t* __restrict__ cand,
    const int8_t* __restrict__ codes, int8_t* __restrict__ out, int64_t n, AdmCosts cs,
    unsigned long long* __restrict__ hist, const unsigned long long* __restrict__ blk, int64_t nblk,
    AdmState* st, int64_t* __restrict__ result) {
  __shared__ unsigned long long red[ADM_THREADS / 64];
  __shared__ unsigned long long lh[BINS];
  const bool next = result == nullptr;
  if (next)
    for (int b = threadIdx.x; b < BINS; b += ADM_THREADS) lh[b] = 0;
  const Sel s = st->sel[mode][2];
  long long b_idx = -1, rem = 0;
  if (s.active && !s.all) cut_entry(mode, s, key, cand, codes, n, cs, blk, nblk, red, b_idx, rem);
  const int all = s.all;
  const unsigned int tau = s.prefix;
  __syncthreads();
  unsigned long long bytes = 0, ev = 0;
  for (int64_t i = 4 * ((int64_t)blockIdx.x * ADM_THREADS + threadIdx.x); i < n;
       i += 4 * (int64_t)gridDim.x * ADM_THREADS) {
    const Four k4 = load4(key, i, n), e4 = load4(cand, i, n), c4 = load4(codes, i, n);
    int o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int c = (int)c4.v[e];
      const unsigned int k = k4.v[e];
      const bool elig = e4.v[e] != 0;
      if (s.active && elig) {
        const bool before = all || k < tau || (k == tau && i + e < b_idx);
        const bool at = !all && i + e == b_idx;
        if (mode == MODE_DOWN) {
          if (before) {
            if (c != 4) c = 3;
          } else if (at && c != 4) {
            const long long s1 = c < 3 ? cs.delta[c] : 0;
            const int n1 = c < 3 ? c + 1 : c;
            const long long s2 = n1 < 3 ? cs.delta[n1] : 0;
            const int n2 = n1 < 3 ? n1 + 1 : n1;
            c = rem <= s1 ? n1 : rem <= s1 + s2 ? n2 : 3;
          }
        } else if (before || at) {
          if (c != 4) ++ev;
          c = 4;
        }
      }
      o[e] = c;
      if (i + e < n && c >= 0 && c <= 4) bytes += (unsigned long long)cs.cost[c];
      if (next && elig) {
        const unsigned long long w = weight(cs, MODE_EVICT, c);
        if (w != 0) atomicAdd(&lh[digit_of(k, 0)], w);
      }
    }
    store4(out, i, n, o);
  }
  if (next) flush_hist(lh, hist + 3 * MODE_EVICT * BINS);
  bytes = block_sum(bytes, red);
  ev = block_sum(ev, red);
  if (threadIdx.x == 0) {
    unsigned long long* r = reinterpret_cast<unsigned long long*>(result);
    atomicAdd(next ? &st->pred[1] : r, bytes);
    if (ev) atomicAdd(r + 1, ev);  // evictions only in the last pass
  }
}

// ---- kv_sensitivity ----------------------------------------------------------

template <int DT>
__device__ __forceinline__ float round_dt(float x) {
  if constexpr (DT == SI_DT_F32) return x;
  else if constexpr (DT == SI_DT_F16) return f16_bits_to_f32(f32_to_f16_bits(x));
  else return bf16_bits_to_f32(f32_to_bf16_bits(x));
}

template <int DT>
__device__ __forceinline__ float elem(const void* p, int64_t i) {
  if constexpr (DT == SI_DT_F32) return reinterpret_cast<const float*>(p)[i];
  else if constexpr (DT == SI_DT_F16) return f16_bits_to_f32(reinterpret_cast<const uint16_t*>(p)[i]);
  else return bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p)[i]);
}

// amax with NaN propagation (torch's max reduction); m holds |x| so far.
__device__ __forceinline__ float amax_nan(float m, float x) {
  const float a = fabsf(x);
  return (a != a || m != m) ? __int_as_float(0x7fc00000) : fmaxf(m, a);
}

// 16 lanes per token-head (b rows of D values); a block covers 16 tokens of
// one head. VEC: 16-byte loads (D * elem_size a multiple of 16, aligned rows).
template <int DT, bool VEC>
__global__ __launch_bounds__(256) void kv_sens_kernel(const void* __restrict__ k,
                                                      const void* __restrict__ v, int64_t B,
                                                      int64_t H, int64_t S, int64_t D,
                                                      void* __restrict__ out) {
  constexpr int ES = DT == SI_DT_F32 ? 4 : 2;
  constexpr int VE = 16 / ES;  // elements per 16-byte load
  const int lane = threadIdx.x & 15;
  const int64_t t = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
  const int64_t h = blockIdx.y;
  float ka = 0.0f, va = 0.0f;
  if (t < S) {
    for (int64_t b = 0; b < B; ++b) {
      const int64_t row = ((b * H + h) * S + t) * D;
      if constexpr (VEC) {
        for (int64_t d = (int64_t)lane * VE; d < D; d += 16 * VE) {
          const uint4 xk = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(k) + (row + d) * ES);
          const uint4 xv = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(v) + (row + d) * ES);
          const uint32_t wk[4] = {xk.x, xk.y, xk.z, xk.w};
          const uint32_t wv[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (DT == SI_DT_F32) {
              ka = amax_nan(ka, __uint_as_float(wk[e]));
              va = amax_nan(va, __uint_as_float(wv[e]));
            } else if constexpr (DT == SI_DT_F16) {
              ka = amax_nan(amax_nan(ka, f16_bits_to_f32(wk[e] & 0xffffu)), f16_bits_to_f32(wk[e] >> 16));
              va = amax_nan(amax_nan(va, f16_bits_to_f32(wv[e] & 0xffffu)), f16_bits_to_f32(wv[e] >> 16));
            } else {
              ka = amax_nan(amax_nan(ka, bf16_bits_to_f32(wk[e] & 0xffffu)), bf16_bits_to_f32(wk[e] >> 16));
              va = amax_nan(amax_nan(va, bf16_bits_to_f32(wv[e] & 0xffffu)), bf16_bits_to_f32(wv[e] >> 16));
            }
          }
        }
      } else {
        for (int64_t d = lane; d < D; d += 16) {
          ka = amax_nan(ka, elem<DT>(k, row + d));
          va = amax_nan(va, elem<DT>(v, row + d));
        }
      }
    }
  }
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) {
    ka = amax_nan(ka, __shfl_xor(ka, o, 16));
    va = amax_nan(va, __shfl_xor(va, o, 16));
  }
  if (lane != 0 || t >= S) return;
  const float s = round_dt<DT>(round_dt<DT>(ka * ka) + round_dt<DT>(va * va)) / 2.0f;
  store_any(out, DT, t * H + h, s);
}

}  // namespace
}  // namespace si

using namespace si;

namespace {

size_t adm_align(size_t x) { return (x + 255) & ~(size_t)255; }

struct AdmLayout {
  size_t key, cand, mid, hist, blk, state, total;
};

AdmLayout adm_layout(int64_t n) {
  AdmLayout l;
  const int64_t nblk = ceil_div(n, TIE_CHUNK);
  const size_t n4 = ((size_t)n + 3) & ~(size_t)3;
  l.key = 0;
  l.cand = adm_align(l.key + n4 * 4);
  l.mid = adm_align(l.cand + n4);  // the codes after the downgrade
  l.hist = adm_align(l.mid + (size_t)n);
  l.blk = adm_align(l.hist + 6 * BINS * 8);
  l.state = adm_align(l.blk + (size_t)(nblk > 0 ? nblk : 1) * 8);
  l.total = adm_align(l.state + sizeof(AdmState));
  return l;
}

unsigned adm_grid(int64_t n) {
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, 4 * ADM_THREADS), kAdmBlocks));
}

}  // namespace

extern "C" size_t si_admit_workspace_bytes(int64_t n_entries) {
  return n_entries < 0 ? 0 : adm_layout(n_entries).total;
}

extern "C" int si_admit_codes(const int8_t* codes, int8_t* out_codes, int64_t S, int64_t H,
                              const float* importance, const float* sensitivity,
                              const uint8_t* protected_mask, int64_t sink_tokens,
                              int64_t budget_bytes, int use_budget, int allow_eviction,
                              const int64_t* costs,
                              int64_t* result, void* workspace, size_t workspace_bytes,
                              si_stream_t stream) {
  clear_error();
  SI_CHECK_ARG(S >= 0 && H >= 0, "si_admit_codes: negative shape (%lld, %lld)", (long long)S,
               (long long)H);
  SI_CHECK_ARG(costs != nullptr && result != nullptr, "si_admit_codes: null costs or result");
  for (int c = 0; c < 5; ++c)
    SI_CHECK_ARG(costs[c] >= 0, "si_admit_codes: negative cost for code %d", c);
  const int64_t n = S * H;
  SI_CHECK_ARG(n == 0 || (codes && out_codes && importance),
               "si_admit_codes: null codes, out_codes or importance");
  const AdmLayout l = adm_layout(n);
  SI_CHECK_ARG(workspace != nullptr && workspace_bytes >= l.total &&
                   (reinterpret_cast<uintptr_t>(workspace) & 255) == 0,
               "si_admit_codes: workspace must be 256-byte aligned and hold %zu bytes", l.total);
  hipStream_t st = as_stream(stream);
  char* ws = static_cast<char*>(workspace);
  unsigned int* key = reinterpret_cast<unsigned int*>(ws + l.key);
  uint8_t* cand = reinterpret_cast<uint8_t*>(ws + l.cand);
  unsigned long long* hist = reinterpret_cast<unsigned long long*>(ws + l.hist);
  unsigned long long* blk = reinterpret_cast<unsigned long long*>(ws + l.blk);
  AdmState* state = reinterpret_cast<AdmState*>(ws + l.state);
  AdmCosts cs;
  for (int c = 0; c < 5; ++c) cs.cost[c] = costs[c];
  for (int c = 0; c < 3; ++c) cs.delta[c] = costs[c] - costs[c + 1];

  int8_t* mid = reinterpret_cast<int8_t*>(ws + l.mid);
  adm_init<<<1, ADM_THREADS, 0, st>>>(state, hist, budget_bytes, result);
  if (int rc = check_launch("si_admit_codes")) return rc;
  if (n == 0) return SI_OK;
  const unsigned grid = adm_grid(n);
  const int64_t nblk = ceil_div(n, TIE_CHUNK);
  SI_CHECK_ARG(nblk < ((int64_t)1 << 31), "si_admit_codes: too many entries (%lld)", (long long)n);
  // entries before `first` belong to sink tokens
  const int64_t first = std::max<int64_t>(0, std::min(sink_tokens, S)) * H;
  adm_prep<<<grid, ADM_THREADS, 0, st>>>(codes, use_budget ? nullptr : out_codes, n, first,
                                         importance, sensitivity, protected_mask, cs, key, cand,
                                         hist, state, result);
  if (int rc = check_launch("si_admit_codes")) return rc;
  if (!use_budget) return SI_OK;
  // Each pass reads one code array and writes another: every block of adm_apply
  // reads the cut entry's chunk, which others would be rewriting.
  for (int mode = MODE_DOWN; mode <= (allow_eviction ? MODE_EVICT : MODE_DOWN); ++mode) {
    const int8_t* from = mode == MODE_DOWN ? codes : mid;
    const bool last = mode == MODE_EVICT || !allow_eviction;
    for (int d = 1; d <= 2; ++d)
      adm_hist<<<grid, ADM_THREADS, 0, st>>>(mode, d, key, cand, from, n, cs, hist, state);
    adm_tie<<<(unsigned)nblk, ADM_THREADS, 0, st>>>(mode, key, cand, from, n, cs, hist, blk, state);
    adm_apply<<<grid, ADM_THREADS, 0, st>>>(mode, key, cand, from, last ? out_codes : mid, n, cs,
                                            hist, blk, nblk, state, last ? result : nullptr);
  }
  return check_launch("si_admit_codes");
}

extern "C" int si_kv_sensitivity(const void* k, const void* v, int dtype, int64_t B, int64_t H,
                                 int64_t S, int64_t D, void* out, si_stream_t stream) {
  clear_error();
  SI_CHECK_ARG(dtype_ok(dtype), "si_kv_sensitivity: unsupported dtype %d", dtype);
  SI_CHECK_ARG(B >= 0 && H >= 0 && S >= 0 && D >= 0, "si_kv_sensitivity: negative shape");
  if (S == 0 || H == 0) return SI_OK;
  SI_CHECK_ARG(out != nullptr && (B * D == 0 || (k != nullptr && v != nullptr)),
               "si_kv_sensitivity: null pointer");
  SI_CHECK_ARG(H < 65536, "si_kv_sensitivity: too many heads (%lld)", (long long)H);
  const int es = dtype_size(dtype);
  const bool vec = (D * es) % 16 == 0 && ((reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v)) & 15) == 0;
  const dim3 grid((unsigned)ceil_div(S, 16), (unsigned)H);
  hipStream_t st = as_stream(stream);
#define SI_SENS(DT_)                                                                  \
  do {                                                                                \
    if (vec) kv_sens_kernel<DT_, true><<<grid, 256, 0, st>>>(k, v, B, H, S, D, out);  \
    else kv_sens_kernel<DT_, false><<<grid, 256, 0, st>>>(k, v, B, H, S, D, out);     \
  } while (0)
  if (dtype == SI_DT_F32) SI_SENS(SI_DT_F32);
  else if (dtype == SI_DT_F16) SI_SENS(SI_DT_F16);
  else SI_SENS(SI_DT_BF16);
#undef SI_SENS
  return check_launch("si_kv_sensitivity");
}
