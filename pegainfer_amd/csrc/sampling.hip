// Sampling for gfx950: argmax, greedy top-1, temperature/top-k/top-p multinomial.
//
//   argmax_cuda            1 workgroup x 1024 lanes, 16-byte loads, lowest index wins ties
//                          (reference csrc/argmax.cu:18,29-31).
//   flashinfer_top1_cuda   64 workgroups; each folds its slice into a packed
//                          (orderable bf16 key << 32 | ~index) word and device-scope atomic-maxes it
//                          into the caller's row_states scratch; the last arriver (ticket counter,
//                          acq_rel) writes the token + top value and re-zeroes both words, so the
//                          scratch keeps the "zero-initialised once" contract of the reference
//                          (ops/sampling.rs:7).  Replaces FlashInfer TopKDispatch(k=1); ties ->
//                          lowest index.
//   pegainfer_sample       the draw below over many workgroups, from the vocabulary size on where that is faster
//   gpu_sample_flashinfer_cuda  softmax(logits*inv_T) -> fp32 probs (reference
//                          csrc/flashinfer_sampling.cu:13-70), then joint top-k / top-p filter on the
//                          original distribution (FlashInfer TopKTopPSamplingFromProb semantics,
//                          restated) by a 3-pass radix select over the fp32 bit patterns, then one
//                          inverse-CDF draw in index order.  RNG = splitmix64(seed); the reference's
//                          Philox stream lives in un-vendored FlashInfer -> distribution parity only.
#include <algorithm>

#include "common.h"
#include "pegainfer_kernels_blocks.h"
#include "pegainfer_kernels_ext.h"
#include "typed.h"

namespace pk {

__device__ __forceinline__ uint32_t bf16_order_key(uint16_t h) {
  if ((h & 0x7FFF) > 0x7F80) return 0;           // NaN never wins (reference: comparisons false)
  if (h == 0x8000) h = 0;                        // -0 == +0
  return (h & 0x8000) ? (uint32_t)(uint16_t)~h : (uint32_t)(h | 0x8000);
}
__device__ __forceinline__ unsigned long long pack_key(uint16_t h, int idx) {
  return ((unsigned long long)bf16_order_key(h) << 32) | (unsigned long long)(0xFFFFFFFFu - (uint32_t)idx);
}
__device__ __forceinline__ unsigned long long u64_max(unsigned long long a, unsigned long long b) {
  return a > b ? a : b;
}
__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    unsigned long long o = __shfl_xor(v, off, kWave);
    v = u64_max(v, o);
  }
  return v;
}

// local best over x[begin:end) strided by the whole grid of threads, 8 elements per 16-byte load
__device__ __forceinline__ unsigned long long scan_best(const Half* __restrict__ x, int n, int tid, int nthreads) {
  unsigned long long best = 0;
  if (aligned16(x)) {
    const int nvec = n >> 3;
    for (int i = tid; i < nvec; i += nthreads) {
      u32x4 v = reinterpret_cast<const u32x4*>(x)[i];
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        best = u64_max(best, pack_key((uint16_t)(w[j] & 0xFFFF), i * 8 + 2 * j));
        best = u64_max(best, pack_key((uint16_t)(w[j] >> 16), i * 8 + 2 * j + 1));
      }
    }
    for (int i = (nvec << 3) + tid; i < n; i += nthreads) best = u64_max(best, pack_key(x[i], i));
  } else {
    for (int i = tid; i < n; i += nthreads) best = u64_max(best, pack_key(x[i], i));
  }
  return best;
}

template <int WAVES>
__device__ __forceinline__ unsigned long long block_max_u64(unsigned long long v, unsigned long long* smem) {
  v = wave_max_u64(v);
  if ((threadIdx.x & 63) == 0) smem[threadIdx.x >> 6] = v;
  __syncthreads();
  unsigned long long r = smem[0];
#pragma unroll
  for (int i = 1; i < WAVES; ++i) r = u64_max(r, smem[i]);
  return r;
}

__global__ __launch_bounds__(1024) void argmax_kernel(const Half* __restrict__ x, int* __restrict__ out, int n) {
  __shared__ unsigned long long red[16];
  unsigned long long best = scan_best(x, n, threadIdx.x, 1024);
  best = block_max_u64<16>(best, red);
  if (threadIdx.x == 0) out[0] = n > 0 ? (int)(0xFFFFFFFFu - (uint32_t)(best & 0xFFFFFFFFu)) : 0;
}

constexpr int kTop1Blocks = 64;
// Workgroups that share a row.  Each costs two atomics in turn, and eight rows' state words share a cache line: with 64 whatever the row count 4
// rows of 151 936 took 8.6 us, 32 rows 16.9; so 6.1 and 7.4.
static inline int top1_blocks(int rows) { return std::min(kTop1Blocks, std::max(16, 128 / rows)); }
// Publish a workgroup's best key and draw its ticket.  Only atomics touch the two state words and agent-scope
// atomics are performed at the device coherence point, so no cache-wide release / acquire is needed (an ACQ_REL
// ticket cost an L2 write-back + invalidate per workgroup: 114 us for 64 rows x 64 workgroups).  What must hold is
// that this workgroup's max is performed before its ticket: the RETURNING fetch_max is waited for (vmcnt) first.
__device__ __forceinline__ unsigned long long top1_publish(unsigned long long* st, unsigned long long best) {
  const unsigned long long prev = __hip_atomic_fetch_max(&st[0], best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" :: "v"(prev) : "memory");   // uses prev: the returning form, completed
  return __hip_atomic_fetch_add(&st[1], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__global__ __launch_bounds__(256) void top1_kernel(const Half* __restrict__ logits, Half* __restrict__ top_value,
                                                   unsigned long long* __restrict__ state, int* __restrict__ out,
                                                   int n) {
  __shared__ unsigned long long red[4];
  unsigned long long best = scan_best(logits, n, blockIdx.x * 256 + threadIdx.x, kTop1Blocks * 256);
  best = block_max_u64<4>(best, red);
  if (threadIdx.x == 0) {
    const unsigned long long ticket = top1_publish(state, best);
    if (ticket == kTop1Blocks - 1) {
      const unsigned long long win = __hip_atomic_exchange(&state[0], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(&state[1], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int idx = (int)(0xFFFFFFFFu - (uint32_t)(win & 0xFFFFFFFFu));
      out[0] = idx;
      if (top_value) top_value[0] = logits[idx];
    }
  }
}

// The last workgroup of a row to arrive writes its token and leaves the row's two words zero.
__device__ __forceinline__ void top1_meet(unsigned long long* st, unsigned long long best, int* out) {
  if (top1_publish(st, best) != gridDim.x - 1) return;
  const unsigned long long win = __hip_atomic_exchange(&st[0], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&st[1], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // the token may go to pinned host memory
  __hip_atomic_store(out, (int)(0xFFFFFFFFu - (uint32_t)(win & 0xFFFFFFFFu)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// Batched greedy: grid (workgroups of a row, rows); row r uses state words [2r, 2r+1] (self-resetting).
__global__ __launch_bounds__(256) void batched_top1_kernel(const Half* __restrict__ logits, long row_stride,
                                                           unsigned long long* __restrict__ state,
                                                           int* __restrict__ out, int n) {
  __shared__ unsigned long long red[4];
  const int row = blockIdx.y;
  const Half* x = logits + (size_t)row * row_stride;
  unsigned long long best = scan_best(x, n, blockIdx.x * 256 + threadIdx.x, gridDim.x * 256);
  best = block_max_u64<4>(best, red);
  if (threadIdx.x == 0) top1_meet(state + 2 * (size_t)row, best, out + row);
}

// The end of a step's logits: what the output projection left (bf16, or fp32) becomes the fp32 logits and their bf16 image, and the greedy
// token of every row comes with them, eight values per thread and trip.  Grid (workgroups of a row, rows or as many as a grid takes), meeting as above.
// Launch-bound: 8 rows of 65 536 fp32 in 5.5 us where cast and greedy token took 4.7 + 8.4, with a factor before them 8 rows of 32 768 in 4.7
// (5.6 + 4.6 + 8.6), one bf16 row of 65 536 in 4.5 (cast, copy and greedy token 5.0 + 4.7 + 4.0).
template <typename T>
__global__ __launch_bounds__(256) void logits_finish_kernel(const T* src, float* out32, Half* out16, float scale, float cap, int n,
                                                            int rows, unsigned long long* __restrict__ state, int* __restrict__ out) {
  __shared__ unsigned long long red[4];
  const bool keep32 = reinterpret_cast<const void*>(src) == out32 && scale == 1.0f && !(cap > 0.f), keep16 = reinterpret_cast<const void*>(src) == out16;
  const bool vec = (n & 7) == 0 && aligned16(src) && aligned16(out32) && aligned16(out16);
  auto value = [&](float v) {
    if (scale != 1.0f) v *= scale;
    return cap > 0.f ? cap * tanhf(v / cap) : v;
  };
  for (int row = blockIdx.y; row < rows; row += gridDim.y) {
    const size_t at = (size_t)row * n;
    unsigned long long best = 0;
    if (vec) {
      for (int i = (blockIdx.x * 256 + threadIdx.x) * 8; i < n; i += gridDim.x * 256 * 8) {
        float v[8];
        Vec8<T>::load(src + at + i, v);
        uint32_t h[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          v[e] = value(v[e]);
          h[e] = f2bf(v[e]);
          best = u64_max(best, pack_key((uint16_t)h[e], i + e));
        }
        if (!keep32) { st4(out32 + at + i, v); st4(out32 + at + i + 4, v + 4); }
        if (!keep16) *reinterpret_cast<u32x4*>(out16 + at + i) = u32x4{h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16};
      }
    } else {
      for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const float v = value(ld(src + at + i));
        const uint16_t h = f2bf(v);
        best = u64_max(best, pack_key(h, i));
        if (!keep32) out32[at + i] = v;
        if (!keep16) out16[at + i] = h;
      }
    }
    if (!out) continue;
    best = block_max_u64<4>(best, red);
    if (threadIdx.x == 0) top1_meet(state + 2 * (size_t)row, best, out + row);
    __syncthreads();             // red is written again for the next row
  }
}

// ---------------------------------------------------------------- temperature / top-k / top-p
// One workgroup of 1024 lanes, 7 vectorised sweeps of the vocabulary (L2-resident after the first):
//   softmax: max, sum, write  |  3 radix passes that build the top-k COUNT and the top-p MASS histograms together
//   |  one sweep that folds the kept mass into 256-token chunk sums, then a block scan over the chunks and a wave
//   scan inside the chosen chunk give the inverse-CDF draw in index order.
// Histograms are integer (counts u32, masses as floor(p * 2^44) in u64): native LDS atomics, and an
// order-independent sum, so the thresholds - hence the support set - are reproducible run to run.  The bin that
// crosses the target is found with a block-wide suffix scan, not a serial walk.
constexpr int kSampleBlock = 1024;
constexpr int kSampleWaves = kSampleBlock / 64;
constexpr float kMassScale = 17592186044416.0f;  // 2^44

__device__ __forceinline__ float block_reduce_f(float v, bool is_max, float* smem16) {
  v = is_max ? wave_max(v) : wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) smem16[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = smem16[0];
  for (int i = 1; i < kSampleWaves; ++i) r = is_max ? fmaxf(r, smem16[i]) : r + smem16[i];
  return r;
}

// inclusive scan of one value per thread in thread order; *total = sum over the block
template <typename T, int WAVES = kSampleWaves>
__device__ __forceinline__ T block_scan_incl(T v, T* wave_tot /* WAVES */, T* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const T o = __shfl_up(v, off, kWave);
    if (lane >= off) v += o;
  }
  __syncthreads();
  if (lane == 63) wave_tot[w] = v;
  __syncthreads();
  T base = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) {
    const T x = wave_tot[i];
    if (i < w) base += x;
    tot += x;
  }
  *total = tot;
  return base + v;
}

// Walk the histogram from the top bin down: the bin b with  above + S(b+1) < target <= above + S(b)
// (S = suffix sum) is written to *chosen and *above += S(b+1).  Thread t owns NB / BLOCK bins from nb-1-t*per on (descending).
template <typename T, int NB, int BLOCK = kSampleBlock>
__device__ __forceinline__ void select_bin(const T* hist, T target_total, int* chosen, T* above, T* wave_tot) {
  constexpr int per = NB / BLOCK;
  const int t = threadIdx.x;
  const T prev = *above;
  const T target = target_total > prev ? target_total - prev : 0;
  T h[per], sum = 0;
#pragma unroll
  for (int k = 0; k < per; ++k) { h[k] = hist[NB - 1 - t * per - k]; sum += h[k]; }
  if (t == 0) *chosen = 0;  // target beyond the total (rounding): lowest bin, keeps everything below
  T total;
  T above_k = block_scan_incl<T, BLOCK / 64>(sum, wave_tot, &total) - sum;
  if (target == 0) {
    if (t == 0) *chosen = NB - 1;
  } else if (target > total) {
    if (t == 0) *above = prev + total - hist[0];
  } else {
#pragma unroll
    for (int k = 0; k < per; ++k) {
      if (above_k < target && target <= above_k + h[k]) {
        *chosen = NB - 1 - t * per - k;
        *above = prev + above_k;
      }
      above_k += h[k];
    }
  }
  __syncthreads();
}

__device__ __forceinline__ float uniform01(uint64_t seed) {
  uint64_t z = seed + 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (float)(z >> 40) * (1.0f / 16777216.0f);  // 24 random bits -> [0,1)
}

// f(value, index) over logits*inv_t, 8 per 16-byte load when aligned
template <typename F>
__device__ __forceinline__ void for_logits(const Half* __restrict__ logits, int n, float inv_t, F f) {
  const int tid = threadIdx.x;
  int done = 0;
  if (aligned16(logits)) {
    const int nvec = n >> 3;
    for (int i = tid; i < nvec; i += kSampleBlock) {
      const u32x4 v = reinterpret_cast<const u32x4*>(logits)[i];
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f(bf_lo(w[j]) * inv_t, i * 8 + 2 * j);
        f(bf_hi(w[j]) * inv_t, i * 8 + 2 * j + 1);
      }
    }
    done = nvec << 3;
  }
  for (int i = done + tid; i < n; i += kSampleBlock) f(bf2f(logits[i]) * inv_t, i);
}
// f(prob) over probs, 4 per 16-byte load when aligned (order of visits is irrelevant to the callers)
template <typename F>
__device__ __forceinline__ void for_probs(const float* __restrict__ probs, int n, F f) {
  const int tid = threadIdx.x;
  int done = 0;
  if (aligned16(probs)) {
    const int nvec = n >> 2;
    for (int i = tid; i < nvec; i += kSampleBlock) {
      const f32x4 v = reinterpret_cast<const f32x4*>(probs)[i];
      f(v[0]); f(v[1]); f(v[2]); f(v[3]);
    }
    done = nvec << 2;
  }
  for (int i = done + tid; i < n; i += kSampleBlock) f(probs[i]);
}

// ---- the draw: kept mass per chunk of cw consecutive tokens, then an inverse CDF in index order ----
__host__ __device__ inline int sample_chunk_width(int n) { return 256 * ((n + 256 * kSampleBlock - 1) / (256 * kSampleBlock)); }

// 4 consecutive kept-filtered probs of this lane
__device__ __forceinline__ int chunk_vals(const float* __restrict__ probs, int n, bool vec, float thr_f, int first, float (&a)[4]) {
  const int i0 = first + (threadIdx.x & 63) * 4;
  if (vec && i0 + 3 < n) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(probs + i0);
#pragma unroll
    for (int e = 0; e < 4; ++e) a[e] = v[e] >= thr_f ? v[e] : 0.f;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) a[e] = (i0 + e < n && probs[i0 + e] >= thr_f) ? probs[i0 + e] : 0.f;
  }
  return i0;
}

// kept mass of chunk c, one wave
__device__ __forceinline__ float chunk_mass(const float* __restrict__ probs, int n, bool vec, float thr_f, int c, int cw) {
  float t = 0.f;
  for (int j = 0; j < cw / 256; ++j) {
    float a[4];
    chunk_vals(probs, n, vec, thr_f, c * cw + j * 256, a);
    t += (a[0] + a[1]) + (a[2] + a[3]);
  }
  return wave_sum(t);
}

// one workgroup of kSampleBlock threads; `mine` = the kept mass of chunk threadIdx.x (0 past the last)
__device__ __forceinline__ void sample_draw(const float* __restrict__ probs, int n, bool vec, float thr_f, int cw, float mine, uint64_t seed,
                                            uint8_t* __restrict__ valid, int* __restrict__ out) {
  __shared__ float wtf[kSampleWaves], sh_rem;
  __shared__ int sh_chunk, sh_pick, sh_last;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid == 0) { sh_chunk = -1; sh_pick = 0x7FFFFFFF; sh_last = -1; }
  __syncthreads();
  float kept;
  const float incl = block_scan_incl<float>(mine, wtf, &kept);
  const float target = uniform01(seed) * kept;
  if (mine > 0.f) {
    if (incl > target && incl - mine <= target) { sh_chunk = tid; sh_rem = target - (incl - mine); }
    atomicMax(&sh_last, tid);  // last chunk holding kept mass (fallback when rounding leaves target >= kept)
  }
  __syncthreads();
  const bool fallback = sh_chunk < 0;
  const int c = fallback ? sh_last : sh_chunk;
  if (c >= 0 && wave == 0) {  // inverse CDF inside the chunk, index order
    const float rem = sh_rem;
    float run = 0.f;
    int last_kept = -1;
    for (int j = 0; j < cw / 256; ++j) {
      float a[4];
      const int i0 = chunk_vals(probs, n, vec, thr_f, c * cw + j * 256, a);
      const float lt = (a[0] + a[1]) + (a[2] + a[3]);
      float inc = lt;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const float o = __shfl_up(inc, off, kWave);
        if (lane >= off) inc += o;
      }
      float cum = run + inc - lt;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (a[e] > 0.f) {
          last_kept = i0 + e;
          if (!fallback && cum + a[e] > rem && cum <= rem) atomicMin(&sh_pick, i0 + e);
        }
        cum += a[e];
      }
      run += __shfl(inc, 63, kWave);
    }
    // not found inside the chunk (summation order differs from the chunk total by an ulp) or fallback: last kept
    int lk = last_kept;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) { const int o = __shfl_xor(lk, off, kWave); lk = lk > o ? lk : o; }
    if (lane == 0 && sh_pick == 0x7FFFFFFF) sh_pick = lk < 0 ? 0 : lk;
  }
  __syncthreads();
  if (tid == 0) {
    out[0] = sh_pick == 0x7FFFFFFF ? 0 : sh_pick;
    if (valid) valid[0] = 1;
  }
}

__global__ __launch_bounds__(kSampleBlock) void sample_kernel(const Half* __restrict__ logits,
                                                               float* __restrict__ probs,
                                                               uint8_t* __restrict__ valid, int* __restrict__ out,
                                                               int n, float inv_t, int top_k, float top_p,
                                                               uint64_t seed) {
  __shared__ float red[kSampleWaves];
  __shared__ uint32_t cnt[2048];
  __shared__ unsigned long long mass[2048];
  __shared__ uint32_t wt32[kSampleWaves];
  __shared__ unsigned long long wt64[kSampleWaves];
  __shared__ float chunk_sum[kSampleBlock];
  __shared__ uint32_t above_k;
  __shared__ unsigned long long above_p;
  __shared__ int chosen_k, chosen_p;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  // ---- softmax (reference logits_to_probs_kernel): p = expf(v - max) / sum ----
  float m = -INFINITY;
  for_logits(logits, n, inv_t, [&](float v, int) { m = fmaxf(m, v); });
  m = block_reduce_f(m, true, red);
  float s = 0.f;
  for_logits(logits, n, inv_t, [&](float v, int) { s += expf(v - m); });
  s = block_reduce_f(s, false, red);
  const float inv_sum = 1.0f / s;
  for_logits(logits, n, inv_t, [&](float v, int i) { probs[i] = expf(v - m) * inv_sum; });
  __syncthreads();

  // ---- joint filter thresholds on the ORIGINAL distribution: largest bit pattern v with count(p >= v) >= top_k,
  //      resp. mass(p >= v) >= top_p; 11 + 11 + 10 bit radix passes, both histograms per sweep ----
  const bool do_k = top_k > 0 && top_k < n, do_p = top_p < 1.0f;
  uint32_t pk = 0u, pp = 0u;
  if (do_k || do_p) {
    if (tid == 0) { above_k = 0u; above_p = 0ull; }
    const unsigned long long target_p = (unsigned long long)((double)top_p * (double)kMassScale);
    int shift = 32;
    for (int pass = 0; pass < 3; ++pass) {
      const int bits = pass < 2 ? 11 : 10, hi = shift, nb = 1 << bits;
      shift -= bits;
      for (int i = tid; i < nb; i += kSampleBlock) { cnt[i] = 0u; mass[i] = 0ull; }
      __syncthreads();
      for_probs(probs, n, [&](float p) {
        const uint32_t u = __builtin_bit_cast(uint32_t, p);
        const int bin = (u >> shift) & (nb - 1);
        if (do_k && (pass == 0 || (u >> hi) == (pk >> hi))) atomicAdd(&cnt[bin], 1u);
        if (do_p && (pass == 0 || (u >> hi) == (pp >> hi))) atomicAdd(&mass[bin], (unsigned long long)(p * kMassScale));
      });
      __syncthreads();
      if (do_k) {
        if (pass < 2) select_bin<uint32_t, 2048>(cnt, (uint32_t)top_k, &chosen_k, &above_k, wt32);
        else select_bin<uint32_t, 1024>(cnt, (uint32_t)top_k, &chosen_k, &above_k, wt32);
        pk |= (uint32_t)chosen_k << shift;
      }
      if (do_p) {
        if (pass < 2) select_bin<unsigned long long, 2048>(mass, target_p, &chosen_p, &above_p, wt64);
        else select_bin<unsigned long long, 1024>(mass, target_p, &chosen_p, &above_p, wt64);
        pp |= (uint32_t)chosen_p << shift;
      }
    }
  }
  const uint32_t thr = (do_k ? pk : 0u) > (do_p ? pp : 0u) ? (do_k ? pk : 0u) : (do_p ? pp : 0u);
  const float thr_f = __builtin_bit_cast(float, thr);

  const int cw = sample_chunk_width(n), nchunks = (n + cw - 1) / cw;
  const bool vec = aligned16(probs);
  for (int c = wave; c < nchunks; c += kSampleWaves) {   // wave w owns chunks w, w + 16, ...
    const float t = chunk_mass(probs, n, vec, thr_f, c, cw);
    if (lane == 0) chunk_sum[c] = t;
  }
  __syncthreads();
  sample_draw(probs, n, vec, thr_f, cw, tid < nchunks ? chunk_sum[tid] : 0.f, seed, valid, out);
}

// ---------------------------------------------------------------- the same draw over many workgroups
// The kernel above keeps one compute unit busy: at 151 936 logits 131 us, most of it 300 000 exponentials and the histograms' LDS
// atomics.  Here every sweep has a launch of its own over up to 128 workgroups, the histograms meet by global integer atomics, and each
// launch starts from what the one before left (the suffix scan that picks a radix digit runs in every workgroup).  The same token from
// the same bits: the maximum and the integer sums do not depend on their order, and the sum of the exponentials keeps the order
// it has above - value by value within each of 1024 threads, their partial sums by wave - with the exponentials themselves
// spread over four waves per 64 of those threads and passed through LDS.  151 936 logits: 131.6 -> 34.5 us with both filters,
// 56.2 -> 19.5 us without; bound by the chain of launches (4 us each).
struct SampleState {
  float wg_max[64], wave_sum[kSampleWaves], chunk_sum[kSampleBlock];
  float m, thr;
  struct Digits { uint32_t pk, above_k, pp; unsigned long long above_p; } digits[3];   // chosen before pass 0, 1, 2 and what lies above them
  uint32_t cnt[3][2048];
  unsigned long long mass[3][2048];
};
constexpr int kWideFrom = 24576;
constexpr int kWideBlock = 256, kSumRounds = 16;   // iterations of the 1024-thread walk whose exponentials wait in LDS at a time

__global__ __launch_bounds__(kWideBlock) void sample_max_kernel(const Half* __restrict__ logits, int n, float inv_t, SampleState* st) {
  __shared__ float red[4];
  const int g = blockIdx.x * kWideBlock + threadIdx.x, all = 64 * kWideBlock, nvec = n >> 3;
  for (int i = g; i < 3 * 2048; i += all) { st->cnt[0][i] = 0u; st->mass[0][i] = 0ull; }
  if (g == 0) st->digits[0] = {0u, 0u, 0u, 0ull};
  float m = -INFINITY;
  for (int i = g; i < nvec; i += all) {
    const u32x4 v = reinterpret_cast<const u32x4*>(logits)[i];
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) m = fmaxf(m, fmaxf(bf_lo(w[j]) * inv_t, bf_hi(w[j]) * inv_t));
  }
  if (g < n - (nvec << 3)) m = fmaxf(m, bf2f(logits[(nvec << 3) + g]) * inv_t);
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) st->wg_max[blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// workgroup w = wave w of the 1024-thread walk: threads 64 w .. 64 w + 63 take vectors tid, tid + 1024, ... and one of the last n % 8 values
__global__ __launch_bounds__(256) void sample_sum_kernel(const Half* __restrict__ logits, int n, float inv_t, SampleState* st) {
  __shared__ __attribute__((aligned(16))) float ex[kSumRounds][64][12];     // 8 values per thread, rows 48 bytes apart
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, tid = blockIdx.x * 64 + lane, nvec = n >> 3;
  const float m = wave_max(st->wg_max[lane]);
  float s = 0.f;
  const int iters = (nvec + kSampleBlock - 1) / kSampleBlock;
  for (int r0 = 0; r0 < iters; r0 += kSumRounds) {
    u32x4 v[kSumRounds / 4];
#pragma unroll
    for (int u = 0; u < kSumRounds / 4; ++u) {
      const int i = tid + (r0 + wave * (kSumRounds / 4) + u) * kSampleBlock;
      v[u] = reinterpret_cast<const u32x4*>(logits)[i < nvec ? i : 0];
    }
    __syncthreads();                                   // the round before is summed
#pragma unroll
    for (int u = 0; u < kSumRounds / 4; ++u) {
      const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
      float e[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) { e[2 * j] = expf(bf_lo(w[j]) * inv_t - m); e[2 * j + 1] = expf(bf_hi(w[j]) * inv_t - m); }
      float* d = ex[wave * (kSumRounds / 4) + u][lane];
      *reinterpret_cast<f32x4*>(d) = f32x4{e[0], e[1], e[2], e[3]};
      *reinterpret_cast<f32x4*>(d + 4) = f32x4{e[4], e[5], e[6], e[7]};
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll 4
      for (int k = 0; k < kSumRounds; ++k) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(ex[k][lane]), b = *reinterpret_cast<const f32x4*>(ex[k][lane] + 4);
        if (tid + (r0 + k) * kSampleBlock < nvec) {
          s += a.x; s += a.y; s += a.z; s += a.w;
          s += b.x; s += b.y; s += b.z; s += b.w;
        }
      }
    }
  }
  if (wave != 0) return;
  if (tid < n - (nvec << 3)) s += expf(bf2f(logits[(nvec << 3) + tid]) * inv_t - m);
  s = wave_sum(s);
  if (lane == 0) {
    st->wave_sum[blockIdx.x] = s;
    if (blockIdx.x == 0) st->m = m;
  }
}

// The digits after pass PASS - 1, from the digits before it and its histograms.  Every workgroup of the launch works them out.
template <int PASS>
__device__ __forceinline__ SampleState::Digits sample_digits(const SampleState* st, bool do_k, bool do_p, int top_k, float top_p) {
  __shared__ uint32_t wt32[kWideBlock / 64], above_k;
  __shared__ unsigned long long wt64[kWideBlock / 64], above_p;
  __shared__ int chosen_k, chosen_p;
  constexpr int nb = PASS == 3 ? 1024 : 2048, shift = PASS == 1 ? 21 : PASS == 2 ? 10 : 0;
  SampleState::Digits d = st->digits[PASS - 1];
  if (threadIdx.x == 0) { above_k = d.above_k; above_p = d.above_p; }
  __syncthreads();
  if (do_k) {
    select_bin<uint32_t, nb, kWideBlock>(st->cnt[PASS - 1], (uint32_t)top_k, &chosen_k, &above_k, wt32);
    d.pk |= (uint32_t)chosen_k << shift;
    d.above_k = above_k;
  }
  if (do_p) {
    select_bin<unsigned long long, nb, kWideBlock>(st->mass[PASS - 1], (unsigned long long)((double)top_p * (double)kMassScale), &chosen_p,
                                                   &above_p, wt64);
    d.pp |= (uint32_t)chosen_p << shift;
    d.above_p = above_p;
  }
  return d;
}

// One radix pass over all values; pass 0 also turns the logits into probabilities (and does nothing else without a filter).
template <int PASS>
__global__ __launch_bounds__(kWideBlock) void sample_hist_kernel(const Half* __restrict__ logits, float* __restrict__ probs, int n, float inv_t,
                                                                 int top_k, float top_p, SampleState* st) {
  __shared__ uint32_t cnt[2048];
  __shared__ unsigned long long mass[2048];
  constexpr int bits = PASS < 2 ? 11 : 10, hi = PASS == 0 ? 32 : PASS == 1 ? 21 : 10, shift = hi - bits, nb = 1 << bits;
  const bool do_k = top_k > 0 && top_k < n, do_p = top_p < 1.0f;
  const int g = blockIdx.x * kWideBlock + threadIdx.x, all = gridDim.x * kWideBlock, nvec = n >> 3;
  for (int i = threadIdx.x; i < nb; i += kWideBlock) { cnt[i] = 0u; mass[i] = 0ull; }
  SampleState::Digits d{};
  float m = 0.f, inv_sum = 0.f;
  if constexpr (PASS == 0) {
    m = st->m;
    float s = st->wave_sum[0];
    for (int i = 1; i < kSampleWaves; ++i) s += st->wave_sum[i];
    inv_sum = 1.0f / s;
  } else {
    d = sample_digits<PASS>(st, do_k, do_p, top_k, top_p);
    if (g == 0) st->digits[PASS] = d;
  }
  __syncthreads();
  auto take = [&](float p) {
    const uint32_t u = __builtin_bit_cast(uint32_t, p);
    const int bin = (u >> shift) & (nb - 1);
    bool in_k = do_k, in_p = do_p;
    if constexpr (PASS > 0) { in_k &= (u >> hi) == (d.pk >> hi); in_p &= (u >> hi) == (d.pp >> hi); }
    if (in_k) atomicAdd(&cnt[bin], 1u);
    if (in_p) atomicAdd(&mass[bin], (unsigned long long)(p * kMassScale));
  };
  for (int i = g; i < nvec; i += all) {
    float p[8];
    if constexpr (PASS == 0) {
      const u32x4 v = reinterpret_cast<const u32x4*>(logits)[i];
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        p[2 * j] = expf(bf_lo(w[j]) * inv_t - m) * inv_sum;
        p[2 * j + 1] = expf(bf_hi(w[j]) * inv_t - m) * inv_sum;
      }
      reinterpret_cast<f32x4*>(probs)[2 * i] = f32x4{p[0], p[1], p[2], p[3]};
      reinterpret_cast<f32x4*>(probs)[2 * i + 1] = f32x4{p[4], p[5], p[6], p[7]};
    } else {
      const f32x4 a = reinterpret_cast<const f32x4*>(probs)[2 * i], b = reinterpret_cast<const f32x4*>(probs)[2 * i + 1];
#pragma unroll
      for (int j = 0; j < 4; ++j) { p[j] = a[j]; p[4 + j] = b[j]; }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) take(p[j]);
  }
  if (g < n - (nvec << 3)) {
    const int i = (nvec << 3) + g;
    if constexpr (PASS == 0) probs[i] = expf(bf2f(logits[i]) * inv_t - m) * inv_sum;
    take(probs[i]);
  }
  if (!do_k && !do_p) return;
  __syncthreads();
  for (int i = threadIdx.x; i < nb; i += kWideBlock) {
    if (do_k && cnt[i]) atomicAdd(&st->cnt[PASS][i], cnt[i]);
    if (do_p && mass[i]) atomicAdd(&st->mass[PASS][i], mass[i]);
  }
}

// the kept mass of every chunk, a wave each
__global__ __launch_bounds__(kWideBlock) void sample_mass_kernel(const float* __restrict__ probs, int n, int top_k, float top_p,
                                                                 SampleState* st) {
  const bool do_k = top_k > 0 && top_k < n, do_p = top_p < 1.0f;
  uint32_t thr = 0u;
  if (do_k || do_p) {
    const SampleState::Digits d = sample_digits<3>(st, do_k, do_p, top_k, top_p);
    thr = d.pk > d.pp ? d.pk : d.pp;
  }
  const float thr_f = __builtin_bit_cast(float, thr);
  const int cw = sample_chunk_width(n), c = blockIdx.x * (kWideBlock / 64) + (threadIdx.x >> 6);
  if (blockIdx.x == 0 && threadIdx.x == 0) st->thr = thr_f;
  if (c * cw >= n) return;
  const float t = chunk_mass(probs, n, true, thr_f, c, cw);
  if ((threadIdx.x & 63) == 0) st->chunk_sum[c] = t;
}

__global__ __launch_bounds__(kSampleBlock) void sample_draw_kernel(const float* __restrict__ probs, uint8_t* __restrict__ valid,
                                                                   int* __restrict__ out, int n, uint64_t seed, const SampleState* st) {
  const int cw = sample_chunk_width(n), nchunks = (n + cw - 1) / cw;
  sample_draw(probs, n, true, st->thr, cw, threadIdx.x < nchunks ? st->chunk_sum[threadIdx.x] : 0.f, seed, valid, out);
}

static int64_t sample_probs_bytes(int n) { return ((int64_t)n * 4 + 15) & ~(int64_t)15; }

}  // namespace pk

using namespace pk;

extern "C" {

void argmax_cuda(const Half* x, int32_t* out, int32_t n, pegainfer_stream_t stream) {
  argmax_kernel<<<1, 1024, 0, as_stream(stream)>>>(x, out, n);
}

void flashinfer_top1_cuda(const Half* logits, Half* top1_value_scratch, uint8_t* row_states_scratch,
                          int32_t* output, int32_t vocab_size, pegainfer_stream_t stream) {
  top1_kernel<<<kTop1Blocks, 256, 0, as_stream(stream)>>>(
      logits, top1_value_scratch, reinterpret_cast<unsigned long long*>(row_states_scratch), output, vocab_size);
}

pegainfer_status_t pegainfer_batched_top1(const Half* logits, int32_t vocab_size, int32_t rows, int64_t row_stride,
                                          uint8_t* state_scratch, int32_t* out_tokens, pegainfer_stream_t stream) {
  if (rows <= 0) return 0;
  batched_top1_kernel<<<dim3(top1_blocks(rows), rows), 256, 0, as_stream(stream)>>>(
      logits, row_stride, reinterpret_cast<unsigned long long*>(state_scratch), out_tokens, vocab_size);
  return static_cast<pegainfer_status_t>(hipGetLastError());
}

pegainfer_status_t pegainfer_logits_finish(const void* src, int32_t src_dtype, float* out32, Half* out16, float scale, float cap,
                                           int32_t vocab_size, int32_t rows, uint8_t* state_scratch, int32_t* out_tokens,
                                           pegainfer_stream_t stream) {
  constexpr pegainfer_status_t bad = static_cast<pegainfer_status_t>(hipErrorInvalidValue);
  if (rows <= 0) return 0;
  if (!src || !out32 || !out16 || vocab_size <= 0 || (out_tokens && !state_scratch)) return bad;
  // in place: where type and values stay what they are, or in fp32
  if (out32 == static_cast<const void*>(out16) || (src == out32 && src_dtype != kDtF32) ||
      (src == out16 && (src_dtype != kDtBf16 || scale != 1.0f || cap > 0.f)))
    return bad;
  const int wgs = std::min(top1_blocks(rows), ceil_div(vocab_size, 8 * 256));
  if (!by_dtype(src_dtype, [&](auto* t) {
        using T = std::remove_pointer_t<decltype(t)>;
        logits_finish_kernel<T><<<dim3(wgs, std::min(rows, 65535)), 256, 0, as_stream(stream)>>>(static_cast<const T*>(src), out32, out16, scale, cap,
                                                                                                 vocab_size, rows, reinterpret_cast<unsigned long long*>(state_scratch), out_tokens);
      }))
    return bad;
  return static_cast<pegainfer_status_t>(hipGetLastError());
}

void gpu_sample_flashinfer_cuda(const Half* logits, float* probs_scratch, uint8_t* valid_scratch,
                                int32_t* output, int32_t vocab_size, float inv_temperature, int32_t top_k,
                                float top_p, uint64_t seed, pegainfer_stream_t stream) {
  sample_kernel<<<1, kSampleBlock, 0, as_stream(stream)>>>(logits, probs_scratch, valid_scratch, output,
                                                           vocab_size, inv_temperature, top_k, top_p, seed);
}

int64_t pegainfer_sample_scratch_bytes(int32_t vocab_size) { return sample_probs_bytes(vocab_size) + (int64_t)sizeof(SampleState); }

pegainfer_status_t pegainfer_sample(const Half* logits, void* scratch, uint8_t* valid_scratch, int32_t* output, int32_t vocab_size,
                                    float inv_temperature, int32_t top_k, float top_p, uint64_t seed, pegainfer_stream_t stream) {
  if (!logits || !scratch || !output || vocab_size <= 0) return static_cast<pegainfer_status_t>(hipErrorInvalidValue);
  hipStream_t s = as_stream(stream);
  float* probs = static_cast<float*>(scratch);
  const int n = vocab_size;
  // rows off 16 bytes (a row of an odd vocabulary) and small vocabularies, where the launches cost more than the sweeps: with both
  // filters 27.2 us alone against 30.2 at 16 384 logits, 39.6 against 29.8 at 32 768; without any 11.5 / 16.5 and 17.1 / 16.5
  if (n < kWideFrom || (reinterpret_cast<uintptr_t>(logits) & 15u) || (reinterpret_cast<uintptr_t>(scratch) & 15u)) {
    sample_kernel<<<1, kSampleBlock, 0, s>>>(logits, probs, valid_scratch, output, n, inv_temperature, top_k, top_p, seed);
    return static_cast<pegainfer_status_t>(hipGetLastError());
  }
  SampleState* st = reinterpret_cast<SampleState*>(static_cast<uint8_t*>(scratch) + sample_probs_bytes(n));
  const int wgs = std::min(128, ceil_div(n, 8 * kWideBlock));
  const bool filter = (top_k > 0 && top_k < n) || top_p < 1.0f;
  sample_max_kernel<<<64, kWideBlock, 0, s>>>(logits, n, inv_temperature, st);
  sample_sum_kernel<<<kSampleWaves, 256, 0, s>>>(logits, n, inv_temperature, st);
  sample_hist_kernel<0><<<wgs, kWideBlock, 0, s>>>(logits, probs, n, inv_temperature, top_k, top_p, st);
  if (filter) {
    sample_hist_kernel<1><<<wgs, kWideBlock, 0, s>>>(logits, probs, n, inv_temperature, top_k, top_p, st);
    sample_hist_kernel<2><<<wgs, kWideBlock, 0, s>>>(logits, probs, n, inv_temperature, top_k, top_p, st);
  }
  sample_mass_kernel<<<ceil_div(ceil_div(n, sample_chunk_width(n)), kWideBlock / 64), kWideBlock, 0, s>>>(probs, n, top_k, top_p, st);
  sample_draw_kernel<<<1, kSampleBlock, 0, s>>>(probs, valid_scratch, output, n, seed, st);
  return static_cast<pegainfer_status_t>(hipGetLastError());
}

}  // extern "C"
