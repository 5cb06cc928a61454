// Selection of a token row's experts, shared by the router's own kernels (moe_route.hip) and by the row kernels that close a sublayer in front of
// routed experts (row_step.hip, seq_blocks.hip, dyt_norm.hip).
#pragma once

#include <algorithm>

#include "common.h"
#include "typed.h"
#include "pegainfer_kernels_blocks.h"

namespace pk {

// Selection on one wave from per-expert values in LDS (s: sigmoid scores, or logits when score is softmax; ch: s + correction):
// softmax over ALL experts if asked, group scores, kept groups, then `top` wave-wide arg-max steps.  LDS accesses of one wave
// complete in order, so no barrier is needed between its steps.
template <typename A>
__device__ __forceinline__ void route_select_wave(float* s, float* ch, float* gs, const A* __restrict__ corr,
                                                  int32_t* __restrict__ out_e, float* __restrict__ out_w, int row, int lane, int E,
                                                  int G, int keep, int top, int score, int group_kind = 0, int renorm = 0,
                                                  float factor = 1.0f, int* pairs = nullptr) {
  if (score == PEGAINFER_SCORE_SOFTMAX) {            // s = exp(z - max) / sum over ALL experts, then the choice scores
    float mx = -INFINITY;
    for (int e = lane; e < E; e += 64) mx = fmaxf(mx, s[e]);
    mx = wave_max(mx);
    float sum = 0.f;
    for (int e = lane; e < E; e += 64) sum += expf(s[e] - mx);
    sum = wave_sum(sum);
    for (int e = lane; e < E; e += 64) {
      const float sc = expf(s[e] - mx) / sum;
      s[e] = sc;
      ch[e] = corr ? sc + ld(corr + e) : sc;
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (G > 1) {
    const int per = E / G;
    for (int g = lane; g < G; g += 64) {             // a lane scores a group: its two largest choices
      float b0 = -INFINITY, b1 = -INFINITY;
      for (int i = 0; i < per; ++i) {
        const float v = ch[g * per + i];
        if (v > b0) { b1 = b0; b0 = v; } else if (v > b1) b1 = v;
      }
      gs[g] = per >= 2 && group_kind == PEGAINFER_GROUP_TOP2_SUM ? b0 + b1 : b0;
    }
    __builtin_amdgcn_wave_barrier();
    for (int g = lane; g < G; g += 64) {             // kept = fewer than `keep` groups rank ahead (ties: the lower index)
      const float mine = gs[g];
      int ahead = 0;
      for (int o = 0; o < G; ++o) {
        const float v = gs[o];
        ahead += (v > mine || (v == mine && o < g)) ? 1 : 0;
      }
      if (ahead >= keep)
        for (int i = 0; i < per; ++i) ch[g * per + i] = -INFINITY;
    }
    __builtin_amdgcn_wave_barrier();
  }
  // The chosen experts with their weights, in choice order, go to out_e / out_w and, for whoever continues in this workgroup, to pairs.
  if (E <= 64) {
    // a lane per expert: its place is the number of eligible experts ahead of it (ties: the lower index)
    const float v = lane < E ? ch[lane] : -INFINITY, w = lane < E ? s[lane] : 0.f;
    // false for no number, which is never chosen (the compiler's ballot of `v > -INFINITY` counts it: an ordered "not equal" made unordered)
    const bool eligible = v >= -__FLT_MAX__;
    int ahead = 0;
    for (int o = 0; o < E; ++o) {
      const float ov = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), o));
      ahead += (ov > v || (ov == v && o < lane)) ? 1 : 0;
    }
    const int found = __popcll(__ballot(eligible));
    float scale = 1.0f;
    if (renorm || factor != 1.0f) {                  // the chosen weights divided by their sum (in choice order), times the factor
      if (eligible) ch[ahead] = w;                   // every lane holds its own value by now
      __builtin_amdgcn_wave_barrier();
      float sum = 0.f;
      for (int k = 0; k < min(top, found); ++k) sum += ch[k];
      scale = factor * (renorm ? 1.0f / (sum + 1e-20f) : 1.0f);
    }
    if (eligible && ahead < top) {
      out_e[(size_t)row * top + ahead] = lane;
      out_w[(size_t)row * top + ahead] = w * scale;
      if (pairs) pairs[row * top + ahead] = lane;
    }
    if (lane >= found && lane < top) {               // fewer eligible experts than choices
      out_e[(size_t)row * top + lane] = 0;
      out_w[(size_t)row * top + lane] = 0.f;
      if (pairs) pairs[row * top + lane] = 0;
    }
    return;
  }
  for (int k = 0; k < top; ++k) {
    float bv = -INFINITY;
    int be = 0x7FFFFFFF;
    for (int e = lane; e < E; e += 64) {             // ascending e per lane: the first maximum is the lowest index
      const float v = ch[e];
      if (v > bv) { bv = v; be = e; }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float ov = __shfl_xor(bv, off, kWave);
      const int oe = __shfl_xor(be, off, kWave);
      if (ov > bv || (ov == bv && oe < be)) { bv = ov; be = oe; }
    }
    const bool found = bv != -INFINITY;
    if (lane == 0) {
      out_e[(size_t)row * top + k] = found ? be : 0;
      out_w[(size_t)row * top + k] = found ? s[be] : 0.f;
      if (pairs) pairs[row * top + k] = found ? be : 0;
      if (found) ch[be] = -INFINITY;
    }
    __builtin_amdgcn_wave_barrier();
  }
  if ((renorm || factor != 1.0f) && lane == 0) {
    float sum = 0.f;
    for (int k = 0; k < top; ++k) sum += out_w[(size_t)row * top + k];
    const float inv = factor * (renorm ? 1.0f / (sum + 1e-20f) : 1.0f);
    for (int k = 0; k < top; ++k) out_w[(size_t)row * top + k] *= inv;
  }
}

// The same selection of one row with a lane per expert (E <= 64) and everything in registers; z: the lane's logit.  What follows a row in its own
// launch runs once per launch, so its instructions come from memory as its data does: this form is a fifth of the code of the one above, its
// wave-wide steps go through scalar registers, and it takes the choices one by one (`top` steps where the other one ranks E).
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ __forceinline__ float wave_max_uniform(float v) {
  v = row16_max(v);
  return fmaxf(fmaxf(lane_value(v, 0), lane_value(v, 16)), fmaxf(lane_value(v, 32), lane_value(v, 48)));
}
template <typename A>
__device__ __forceinline__ void route_select_lanes(float z, const A* __restrict__ corr, int32_t* __restrict__ out_e, float* __restrict__ out_w, int row,
                                                   int lane, int E, int G, int keep, int top, int score, int group_kind, int renorm, float factor) {
  const bool on = lane < E;
  const float add = corr && on ? ld(corr + lane) : 0.f;
  float w;
  if (score == PEGAINFER_SCORE_SOFTMAX) {
    const float mx = wave_max_uniform(on ? z : -INFINITY);
    w = on ? expf(z - mx) : 0.f;
    const float r = row16_sum(w);
    w /= (lane_value(r, 0) + lane_value(r, 16)) + (lane_value(r, 32) + lane_value(r, 48));
  } else {
    w = sigmoid_f(z);
  }
  float v = on ? (corr ? w + add : w) : -INFINITY;
  if (G > 1) {
    const int per = E / G, mine = lane / per;
    float b0 = -INFINITY, b1 = -INFINITY;
#pragma unroll 4
    for (int i = 0; i < per; ++i) {
      const float o = __shfl(v, min(mine * per + i, 63), kWave);
      if (o > b0) { b1 = b0; b0 = o; } else if (o > b1) b1 = o;
    }
    const float gs = per >= 2 && group_kind == PEGAINFER_GROUP_TOP2_SUM ? b0 + b1 : b0;
    int ahead = 0;
#pragma unroll 1
    for (int o = 0; o < G; ++o) {
      const float og = lane_value(gs, o * per);
      ahead += (og > gs || (og == gs && o < mine)) ? 1 : 0;
    }
    if (ahead >= keep) v = -INFINITY;
  }
  if (!(v >= -__FLT_MAX__)) v = -INFINITY;           // what is no number is never chosen
  float sum = 0.f, my_w = 0.f;
  int my_e = 0;
#pragma unroll 1
  for (int k = 0; k < top; ++k) {                    // the largest, of equal ones the first; none left: expert 0 with no weight
    const float best = wave_max_uniform(v);
    const unsigned long long held = __ballot(v == best && best > -INFINITY);
    if (!held) break;
    const int e = __ffsll(held) - 1;
    const float we = lane_value(w, e);
    sum += we;
    if (lane == k) { my_e = e; my_w = we; }
    if (lane == e) v = -INFINITY;
  }
  if (lane < top) {
    out_e[(size_t)row * top + lane] = my_e;
    out_w[(size_t)row * top + lane] = my_w * (factor * (renorm ? 1.0f / (sum + 1e-20f) : 1.0f));
  }
}

// The router behind a row that a workgroup has just made (decode steps): its logits, the choice and the shared expert's gate logit in the launch that
// leaves the row, so that neither a product nor a selection of their own follow.
// Bound by latency, and by what one compute unit takes in from memory (some 25 KB per us; the router of 33 x 2560 is 169 KB): the router's rows are
// asked for before the row's own sums begin, and meet the row (rounded as it is stored, through LDS) on the matrix cores: a wave
// takes 16 experts times every waves-th piece of 32 values, the row repeated over the columns.  Workgroups without a row, on the same XCDs,
// pull the router into the L2s meanwhile, a sixteenth of it or 8 KB each.
// Row, router product, selection and sort in three launches -> the row with its router in one (the experts' launches find their rows from the choices):
// 8 rows of 1024, 17 router rows 14.0 -> 7.3 us; 8 of 2048, 41: 17.0 -> 9.9; 4 of 2048, 32: 17.2 -> 10.5; one of 2560, 32: 16.5 -> 8.5.  Without the
// helping workgroups, and with conditional loads that kept 15 - 20 KB of instructions instead of 5: 10.8, 12.7, 13.3, 10.9.
// Only while three blocks of 16 hold the experts, and a row a workgroup (d <= 4096); and of those up to 240 KB of router: beyond that a compute unit's share of
// it costs more than the launches.
// The pieces of a wave in ascending order, then the waves in order: a logit's sum is fixed by the width alone.
constexpr int kTailBlocks = 3;                          // experts and gate row: at most three blocks of 16 (NB: blocks of a launch, two or three)
constexpr int kXcds = 8;
struct RouterTail {
  const uint16_t *w, *corr;                             // w NULL: no router follows
  int32_t* out_e;
  float *out_w, *gate;
  int64_t gate_stride;
  int E, extra, G, keep, top, score, group_kind, renorm;
  float factor;
  int rows;                                             // of the step: workgroups from there on have no row
};
template <int N, int NB>
struct RouteTail {
  static constexpr int kWaves = N / 64, P = N >= 1024 ? 4 : 8;      // pieces in flight per block; with 1024 threads a row has up to eight
  struct Shared {
    alignas(16) uint16_t row[N * 4];                    // both are read or written 16 bytes at a time
    alignas(16) float part[kWaves][NB * 16];
  };
  static_assert(alignof(Shared) % 16 == 0 && sizeof(Shared::row) % 16 == 0 && sizeof(Shared::part[0]) % 16 == 0, "16-byte accesses");
  u32x4 w[P][NB];
  // a workgroup without a row (the first few have none either: they fill the round of XCDs that the rows begin)
  static __device__ __forceinline__ bool helps(const RouterTail& t, int d) {
    const int b = blockIdx.x;
    if (b < t.rows) return false;
    const int first = (t.rows + kXcds - 1) & ~(kXcds - 1);
    if (b < first || (b & (kXcds - 1)) >= t.rows) return true;
    const int chunks = (t.E + t.extra) * d / 8, parts = (gridDim.x - first) / kXcds;
    const u32x4* src = reinterpret_cast<const u32x4*>(t.w);
    for (int i = (b - first) / kXcds * N + threadIdx.x; i < chunks; i += parts * N) {
      const u32x4 v = src[i];
      asm volatile("" ::"v"(v));
    }
    return true;
  }
  // pieces p0, p0 + 1, .. of this wave (its piece p covers the values from 32 (wave + kWaves p)); what lies past the row or the last expert
  // repeats the last, unused
  __device__ __forceinline__ void request(const RouterTail& t, int d, int p0 = 0) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const uint16_t* src = t.w + min(b * 16 + (lane & 15), t.E + t.extra - 1) * d + (lane >> 4) * 8;
#pragma unroll
      for (int p = 0; p < P; ++p) w[p][b] = *reinterpret_cast<const u32x4*>(src + min(32 * (wave + kWaves * (p0 + p)), d - 32));
    }
  }
  // a thread's chunk of four values of the row, as they are stored
  __device__ __forceinline__ void put(Shared& sh, int i, const float* v) const {
    *reinterpret_cast<u32x2*>(sh.row + i) = u32x2{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
  }
  __device__ __forceinline__ void finish(const RouterTail& t, Shared& sh, int d, int row) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    f32x4 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto products = [&](int p0) {
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int k = 32 * (wave + kWaves * (p0 + p));
        if (k >= d) break;
        const bf16x8_t x = *reinterpret_cast<const bf16x8_t*>(sh.row + k + (lane >> 4) * 8);
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w[p][b]), x, acc[b], 0, 0, 0);
      }
    };
    __syncthreads();
    products(0);
    if constexpr (P * kWaves * 32 < N * 4) {
      if (P * kWaves * 32 < d) {
        request(t, d, P);
        products(P);
      }
    }
    if ((lane & 15) == 0)                                // every column holds the same sums: expert 4 (lane >> 4) + i of the block
#pragma unroll
      for (int b = 0; b < NB; ++b) *reinterpret_cast<f32x4*>(&sh.part[wave][b * 16 + (lane >> 4) * 4]) = acc[b];
    __syncthreads();
    if (wave != 0) return;
    float z = 0.f;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) z += sh.part[v][min(lane, NB * 16 - 1)];
    if (t.gate && lane == t.E) t.gate[(int64_t)row * t.gate_stride] = z;
    route_select_lanes(z, t.corr, t.out_e, t.out_w, row, lane, t.E, t.G, t.keep, t.top, t.score, t.group_kind, t.renorm, t.factor);
  }
};
// what a kernel without a router behind it has in its place
struct NoTail {
  struct Shared {};
  static __device__ __forceinline__ bool helps(const RouterTail&, int) { return false; }
  __device__ __forceinline__ void request(const RouterTail&, int) {}
  __device__ __forceinline__ void put(Shared&, int, const float*) const {}
  __device__ __forceinline__ void finish(const RouterTail&, Shared&, int, int) {}
};

// workgroups of a launch with a router behind its rows
inline int tail_blocks(const RouterTail& t, int d) {
  const int kb8 = ((t.E + t.extra) * d * 2 + 8191) / 8192;
  return ((t.rows + kXcds - 1) & ~(kXcds - 1)) + kXcds * std::min(16, kb8);
}
inline bool router_tail_sizes(int experts, int has_gate, int d, int dtype) {
  return dtype == kDtBf16 && experts > 0 && experts + (has_gate ? 1 : 0) <= 16 * kTailBlocks && d > 0 && d % 32 == 0 && d <= 4096;
}
// ... and where it is the faster way: up to 240 KB of router.  The row's launch, both products of the experts and, without the tail, the router's product and the plan,
// cold weights, without / with (us): 48 rows of 2560 and 1 / 8 rows of a step 34.9 / 32.1, 67.4 / 68.8; 33 of 4096 41.7 / 39.1, 102.7 / 109.8; 48 of 4096
// 43.5 / 44.1, 4 rows 71.3 / 78.3.
inline bool router_tail_pays(int experts, int has_gate, int d, int dtype) {
  return router_tail_sizes(experts, has_gate, d, dtype) && (experts + (has_gate ? 1 : 0)) * d <= 120 * 1024;
}
// the descriptor's form of it; false: that router stays a launch of its own
inline bool router_tail(const pegainfer_router_tail_desc* q, int rows, int d, int dtype, RouterTail* t) {
  const int groups = std::max(1, q->n_groups);
  if (!router_tail_sizes(q->experts, q->gate_logit != nullptr, d, dtype) || !q->w || !q->out_expert || !q->out_weight || q->experts % groups ||
      q->top <= 0 || q->top > q->experts || q->keep_groups < 1 || q->keep_groups > groups || !host_aligned16(q->w) ||
      (q->score_kind != PEGAINFER_SCORE_SIGMOID && q->score_kind != PEGAINFER_SCORE_SOFTMAX) ||
      (q->group_kind != PEGAINFER_GROUP_TOP2_SUM && q->group_kind != PEGAINFER_GROUP_MAX))
    return false;
  *t = RouterTail{static_cast<const uint16_t*>(q->w), static_cast<const uint16_t*>(q->correction), q->out_expert, q->out_weight, q->gate_logit,
                  q->gate_stride, q->experts, q->gate_logit ? 1 : 0, groups, q->keep_groups, q->top, q->score_kind, q->group_kind, q->renorm, q->factor, rows};
  return true;
}

}  // namespace pk
