// Products of few rows (decode steps), as parts of a launch: the kernels of gemm_strided.hip and launches that do something else beside the product.
// The addressing is that of pegainfer_gemm_desc.
#pragma once

#include <type_traits>

#include "common.h"
#include "typed.h"
#include "pegainfer_kernels_blocks.h"

namespace pk {

// ------------------------------------------------------------------ up to four fp32 rows against fp32 weights (decode)
// No LDS and no barrier: a wave takes MB outputs (GLU: MB pairs of a gate row and its up row), lanes over k four values at a time, and fetches the rows
// it multiplies with beside the weights, pieces of 512 k two ahead of the products.  An output's k order is fixed by K alone.
// Bound by one memory latency behind the launch with few outputs and by the stream of weights with many.  With the rows in LDS first (a barrier
// before any product, 32-byte strides between lanes), 1 / 2 / 4 rows and cold weights: 1024 x 1024 3.4 / 4.2 / 5.5 -> 3.3 / 3.3 / 3.7 us, 1024 x 2048
// 4.2 / 5.4 / 7.4 -> 4.0 / 4.1 / 4.9, 3072 x 1024 5.1 / 6.3 / 8.3 -> 4.6 / 4.8 / 5.9, 6144 x 1024 7.3 / 8.2 / 10.3 -> 6.3 / 6.6 / 8.5,
// 32 768 x 1024 25.9 / 31.3 / 32.2 -> 21.0 / 21.2 / 24.6 (6.4 TB/s); on the fp32 matrix cores 2048 x 8192 took 28.2 with two rows, 14.1 here.  One fp32
// row against bf16 weights 65 536 x 2048: 54.9 -> 39.4.
// a lane's eight values of a piece of 512, in one or two loads that are whole lines over the wave
template <typename TW>
struct DirectPiece;
template <>
struct DirectPiece<float> {
  f32x4 v[2];
  static __device__ __forceinline__ int k_of(int p, int lane, int h) { return p * 512 + h * 256 + lane * 4; }
  static __device__ __forceinline__ int last(int K, int) { return K - 4; }
  __device__ __forceinline__ void load(const float* w, const int (&k)[2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) v[h] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(w + k[h]));
  }
  __device__ __forceinline__ f32x4 half(int h) const { return v[h]; }
};
template <>
struct DirectPiece<uint16_t> {
  u32x4 v;
  static __device__ __forceinline__ int k_of(int p, int lane, int h) { return p * 512 + lane * 8 + h * 4; }
  static __device__ __forceinline__ int last(int K, int h) { return K - 8 + 4 * h; }
  __device__ __forceinline__ void load(const uint16_t* w, const int (&k)[2]) { v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(w + k[0])); }
  __device__ __forceinline__ f32x4 half(int h) const {
    return h ? f32x4{bf_lo(v.z), bf_hi(v.z), bf_lo(v.w), bf_hi(v.w)} : f32x4{bf_lo(v.x), bf_hi(v.x), bf_lo(v.y), bf_hi(v.y)};
  }
};
// of 256 threads; bx, by, bz: the workgroup's place in a grid of (tiles of R rows, 4 MB outputs, groups)
template <typename TW, typename TY, typename TG, int R, int MB, bool GLU>
__device__ __forceinline__ void gemm_rows_direct_block(const pegainfer_gemm_desc& d, int act, int64_t up, int bx, int by, int bz) {
  constexpr int NW = GLU ? 2 : 1, CH = (MB == 4 ? 1 : 2) * (sizeof(TW) == 2 ? 2 : 1);      // pieces per register set
  typedef DirectPiece<TW> Piece;
  int g, row0, nrows;
  if (d.tile_group) {
    if (bx >= *d.n_tiles) return;
    g = d.tile_group[bx];
    row0 = d.tile_row0[bx];
    nrows = min(R, d.tile_rows[bx]);
  } else {
    g = bz;
    row0 = bx * R;
    nrows = min(R, d.rows - row0);
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, K = d.k;
  const int m0 = (by * 4 + wave) * MB;
  if (m0 >= d.m || nrows <= 0) return;
  auto x_row = [&](int r) {                                   // absent rows repeat the last one; they are never stored
    const int p = row0 + min(r, nrows - 1);
    return d.x_row_index ? d.x_row_index[p] : p;
  };
  const float* X = static_cast<const float*>(d.x) + (int64_t)g * d.x_group_stride;
  const TW* W = static_cast<const TW*>(d.w) + (int64_t)g * d.w_group_stride;
  const float* xp[R];
  const TW* wp[MB];
#pragma unroll
  for (int r = 0; r < R; ++r) xp[r] = X + (int64_t)x_row(r) * d.x_row_stride;
#pragma unroll
  for (int q = 0; q < MB; ++q) wp[q] = W + (int64_t)min(m0 + q, d.m - 1) * d.w_m_stride;      // a clamped row is loaded and dropped at the store
  struct Set { Piece w[CH][MB][NW]; f32x4 x[CH][R][2]; } A, B;
  auto issue = [&](int p0, Set& s) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      int k[2];                                               // a lane past the end repeats the last values, unused
#pragma unroll
      for (int h = 0; h < 2; ++h) k[h] = min(Piece::k_of(p0 + c, lane, h), Piece::last(K, h));
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int h = 0; h < 2; ++h) s.x[c][r][h] = *reinterpret_cast<const f32x4*>(xp[r] + k[h]);
#pragma unroll
      for (int q = 0; q < MB; ++q)
#pragma unroll
        for (int n = 0; n < NW; ++n) s.w[c][q][n].load(wp[q] + (n ? up : 0), k);
    }
  };
  float acc[MB][NW][R];
#pragma unroll
  for (int q = 0; q < MB; ++q)
#pragma unroll
    for (int n = 0; n < NW; ++n)
#pragma unroll
      for (int r = 0; r < R; ++r) acc[q][n][r] = 0.f;
  auto compute = [&](int p0, const Set& s) {
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (Piece::k_of(p0 + c, lane, h) >= K) continue;
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int q = 0; q < MB; ++q)
#pragma unroll
            for (int n = 0; n < NW; ++n) {
              const f32x4 w = s.w[c][q][n].half(h), x = s.x[c][r][h];
              float a = acc[q][n][r];
              a = fmaf(w.x, x.x, a); a = fmaf(w.y, x.y, a); a = fmaf(w.z, x.z, a); a = fmaf(w.w, x.w, a);
              acc[q][n][r] = a;
            }
      }
  };
  const int np = (K + 511) >> 9;
  issue(0, A);
  if (np > CH) issue(CH, B);
  for (int p = 0; p < np; p += 2 * CH) {
    compute(p, A);
    if (p + 2 * CH < np) issue(p + 2 * CH, A);
    if (p + CH >= np) break;
    compute(p + CH, B);
    if (p + 3 * CH < np) issue(p + 3 * CH, B);
  }
  // Sums over each 16 lanes, of which lane r MB + q keeps those of output q of row r: the way over the four runs of lanes, and what follows, is then one
  // for all (each sum by itself as in wave_sum, whose steps these are, and stored by one lane: four rows of 65 536 x 256 24.9 -> 19.3 us).
  static_assert(MB * R <= 16, "a lane of sixteen per sum");
  float v = 0.f, u = 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int q = 0; q < MB; ++q) {
      const bool mine = (lane & 15) == r * MB + q;
      const float t = row16_sum(acc[q][0][r]);
      v = mine ? t : v;
      if constexpr (GLU) {
        const float t2 = row16_sum(acc[q][1][r]);
        u = mine ? t2 : u;
      }
    }
  v += __shfl_xor(v, 16, kWave);
  v += __shfl_xor(v, 32, kWave);
  if constexpr (GLU) {
    u += __shfl_xor(u, 16, kWave);
    u += __shfl_xor(u, 32, kWave);
  }
  const int r = lane / MB, m = m0 + lane % MB;
  if (r >= nrows || m >= d.m) return;
  if constexpr (GLU) v = act_f(act, v) * u;
  else if (d.epilogue == PEGAINFER_EPI_RELU_SQ) { v = fmaxf(v, 0.f); v *= v; }
  else if (d.epilogue == PEGAINFER_EPI_GELU_ERF) v = gelu_erf_f(v);
  else if (d.epilogue == PEGAINFER_EPI_SIGMOID_GATE)
    v *= sigmoid_f(ld(static_cast<const TG*>(d.gate) + (int64_t)x_row(r) * d.gate_row_stride + g));
  const int yr = d.y_row_index ? d.y_row_index[row0 + r] : row0 + r;
  st(static_cast<TY*>(d.y) + (int64_t)g * d.y_group_stride + (int64_t)yr * d.y_row_stride + m, v);
}

// ------------------------------------------------------------------ few-rows form on the matrix cores (bf16 weights, decode)
// At most 16 rows per tile; bound by the stream of weights.  A wave takes OB blocks of 16 outputs, wk waves share a block's K (wave
// j the 64-wide pieces j, j + wk, ... of k; wk follows from K alone), their partial sums meet in LDS in wave order: an output's k order is
// fixed by K.  One load instruction covers 8 outputs x 128 bytes: lane = output (lane >> 1) & 7, 16-byte chunk 2 (lane >> 4) + (lane & 1).
// Taken unpermuted as an A operand, row 2 r + h holds output r's chunks of parity h, so the product with the x chunks of parity h is
// right in the rows of that parity and discarded in the others (the same layout as gemm_skinny.h).  x comes straight from memory - a tile's
// rows are few and stay in the caches - a chunk of pieces ahead, as the weights do: 16 KB of weights in flight per wave.
// fp32 rows enter as three bf16 parts of 8 bits each, cut off rather than rounded: their sum IS the value, every product is exact
// and the sums stay in fp32.
// Against the FMA form (eight rows in LDS, four weight loads in flight per wave): 17 experts of 2048 x 2048 with 24 pairs 51 -> 15.6 us
// (4.6 TB/s) up and, with the output matrix of 65 536 x 2048 and 8 rows among them, 79 -> 26 us on average; 32 768 x 1024 with 8 fp32
// rows 61 -> 18.7 us; 4 experts of 2048 x 2560 and one row each 15.1 -> 13.4 us.
__device__ __forceinline__ void split3(const f32x4& a, const f32x4& b, bf16x8_t (&o)[3]) {
  const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  uint32_t part[3][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t hi[2], mid[2], lo[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float x = v[2 * i + e];
      const uint32_t bits = __builtin_bit_cast(uint32_t, x);
      hi[e] = bits & 0xFFFF0000u;
      // an infinity has no remainder (x - x would be NaN); what is no number leaves one that is none, also where its cut-off part alone tells
      // it from an infinity
      const float r1 = (bits & 0x7FFFFFFFu) == 0x7F800000u ? 0.f : x - __builtin_bit_cast(float, hi[e]);
      mid[e] = __builtin_bit_cast(uint32_t, r1) & 0xFFFF0000u;
      lo[e] = __builtin_bit_cast(uint32_t, r1 - __builtin_bit_cast(float, mid[e]));
    }
    part[0][i] = (hi[0] >> 16) | hi[1];
    part[1][i] = (mid[0] >> 16) | mid[1];
    part[2][i] = (lo[0] >> 16) | (lo[1] & 0xFFFF0000u);
  }
#pragma unroll
  for (int s = 0; s < 3; ++s) o[s] = __builtin_bit_cast(bf16x8_t, u32x4{part[s][0], part[s][1], part[s][2], part[s][3]});
}

// 8 values of x as they are fetched, and as operands
template <typename TX>
struct RowPiece;
template <>
struct RowPiece<uint16_t> {
  static constexpr int kParts = 1;
  u32x4 v;
  __device__ __forceinline__ void load(const uint16_t* p) { v = *reinterpret_cast<const u32x4*>(p); }
  __device__ __forceinline__ void zero() { v = u32x4{0u, 0u, 0u, 0u}; }
  __device__ __forceinline__ void parts(bf16x8_t (&o)[1]) const { o[0] = __builtin_bit_cast(bf16x8_t, v); }
};
template <>
struct RowPiece<float> {
  static constexpr int kParts = 3;
  f32x4 a, b;
  __device__ __forceinline__ void load(const float* p) { a = *reinterpret_cast<const f32x4*>(p); b = *reinterpret_cast<const f32x4*>(p + 4); }
  __device__ __forceinline__ void zero() { a = f32x4{0.f, 0.f, 0.f, 0.f}; b = a; }
  __device__ __forceinline__ void parts(bf16x8_t (&o)[3]) const { split3(a, b, o); }
};

constexpr int kRowsMax = 16;   // token rows of a tile of the matrix-core few-rows form

// What the experts of few rows do beyond the grouped product (EX; pegainfer_expert_rows): a gated activation of two weight rows per output, and
// the slices of an expert that every row takes as further groups, behind the table's `slots` workgroup columns.
// In a decode step each launch costs some 4 us whatever it does: 8 rows, 16 experts of 2 x 512 x 1024 and a shared one of twice their size took
// 9.6 + 4.5 (activation) + 7.0 us and 5.0 + 4.2 for the shared one, here 9.6 + 6.4; 32 experts of 1024 x 2048 and a shared one of 2048
// 16.2 + 14.5 and 14.0 in three launches, here 16.9 + 15.4; one row, 4 of 32 experts of 2 x 1024 x 2560 13.2 + 4.6 + 8.4 and 15.4, here 14.4 + 9.0.
struct ExpertForm {
  int glu, slots, rows, pos0;
  float limit, alpha, shared_limit;
  const uint16_t* w;
  int64_t m_stride, group_stride, up;      // the shared expert's: of a weight row, of a slice, from a gate row to its up row
  // no table: the choices of the step's rows, one behind the other
  const int32_t* chosen;
  int32_t* tiles;                          // what the first product found for the second: per tile expert, pairs, their numbers
  int pairs, top, experts, by_pair;
};
// The tile'th run of at most 16 pairs of one expert, experts ascending and an expert's pairs as they lie, found by one wave from the choices (up to 256 of up
// to 64 experts): a load and some ballots where a launch would sort them into a table first (4.3 - 6.2 us).  By every wave for itself it
// takes 1.4 us longer: their instructions share the SIMDs.  A lane stands for an expert: its mask of 64 pairs is the conjunction of the
// number's bits over the lanes that hold them.  Returns the number of pairs, 0: no such tile.
constexpr int kChosenMost = 4, kTileWords = kRowsMax + 2;      // times 64 pairs
__device__ __forceinline__ int chosen_tile(const ExpertForm& ex, int tile, int lane, int* list, int* group) {
  auto expert_of = [&](int c) { return c + lane < ex.pairs ? ex.chosen[c + lane] : -1; };
  int e = 0, count = 0;
#pragma unroll 1
  for (int c = 0; c < ex.pairs; c += 64) {
    e = expert_of(c);
    unsigned long long m = __ballot((unsigned)e < (unsigned)ex.experts);
#pragma unroll
    for (int b = 0; b < 6; ++b) {
      const unsigned long long one = __ballot((e >> b) & 1);
      m &= (lane >> b) & 1 ? one : ~one;
    }
    count += __popcll(m);
  }
  const int tiles = (count + kRowsMax - 1) / kRowsMax;
  int before;                              // tiles of the experts ahead
  if (__ballot(tiles > 1)) {
    before = tiles;
#pragma unroll 1
    for (int x = 1; x < 64; x <<= 1) {
      const int o = __shfl_up(before, x, kWave);
      if (lane >= x) before += o;
    }
    before -= tiles;
  } else {
    before = __popcll(__ballot(tiles > 0) & ((1ull << lane) - 1));
  }
  const unsigned long long mine = __ballot(tile >= before && tile < before + tiles);
  if (!mine) return 0;
  const int g = __ffsll(mine) - 1;
  const int skip = (tile - __builtin_amdgcn_readlane(before, g)) * kRowsMax, left = __builtin_amdgcn_readlane(count, g) - skip;
  *group = g;
  int rank = -skip;
#pragma unroll 1
  for (int c = 0; c < ex.pairs; c += 64) {
    if (ex.pairs > 64) e = expert_of(c);
    const unsigned long long m = __ballot(e == g);
    const int at = rank + __popcll(m & ((1ull << lane) - 1));
    if (e == g && at >= 0 && at < kRowsMax) list[at] = c + lane;
    rank += __popcll(m);
  }
  return min(left, kRowsMax);
}
__device__ __forceinline__ float glu_f(const ExpertForm& ex, bool shared, float g, float u) {
  if (ex.glu == PEGAINFER_GLU_SILU) return g * sigmoid_f(g) * u;
  const float limit = shared ? ex.shared_limit : ex.limit;
  g = fminf(g, limit);
  return g * sigmoid_f(ex.alpha * g) * (fminf(fmaxf(u, -limit), limit) + 1.0f);
}

// of 256 threads; bx, by, bz: the workgroup's place in a grid of (tiles of rows, 4 / wk blocks of outputs, groups)
template <typename TX, typename TY, typename TG, int OB, bool EX = false>
__device__ __forceinline__ void gemm_rows_mfma_block(const pegainfer_gemm_desc& d, int wk, const ExpertForm& ex, int bx, int by, int bz) {
  constexpr int CH = OB == 1 && sizeof(TX) == 2 ? 4 : 2;      // 64-wide pieces per register set
  constexpr int NP = RowPiece<TX>::kParts;
  __shared__ f32x4 red[4][OB][64];
  __shared__ int list[EX ? kRowsMax : 1], found[2];          // of a tile without a table: its pairs; its expert, their number
  int g, row0, nrows, my_pair = 0;
  const bool shared = EX && bx >= ex.slots, chosen = EX && !shared && ex.chosen;
  if (shared) {
    g = bx - ex.slots;
    row0 = ex.pos0 + g * ex.rows;
    nrows = ex.rows;
  } else if (chosen) {
    if (bx >= d.max_tiles) return;               // (an odd number of columns may hold one more)
    row0 = 0;
    int32_t* t = ex.tiles ? ex.tiles + bx * kTileWords : nullptr;
    if (t && ex.by_pair) {                                    // found by the product before, asked for all at once
      g = t[0];
      nrows = t[1];
      my_pair = t[2 + (threadIdx.x & 15)];
      if (threadIdx.x < kRowsMax) list[threadIdx.x] = my_pair;
      const int first = __builtin_amdgcn_readfirstlane(my_pair);      // of all lanes, before any is left out
      if ((int)(threadIdx.x & 15) >= nrows) my_pair = first;
    } else {
      if (threadIdx.x < 64) {
        int e = 0;
        const int c = chosen_tile(ex, bx, threadIdx.x, list, &e);
        if (threadIdx.x == 0) { found[0] = e; found[1] = c; }
        __builtin_amdgcn_wave_barrier();                      // the list is read by other lanes of this wave
        if (t && by == 0 && threadIdx.x < kTileWords) {
          if (threadIdx.x == 0) t[0] = e;
          if (threadIdx.x == 1) t[1] = c;
          if (threadIdx.x >= 2 && (int)threadIdx.x < 2 + c) t[threadIdx.x] = list[threadIdx.x - 2];
        }
      }
      __syncthreads();
      g = found[0];
      nrows = found[1];
      if (nrows > 0) my_pair = list[min((int)threadIdx.x & 15, nrows - 1)];
    }
    g = __builtin_amdgcn_readfirstlane(g);
    nrows = __builtin_amdgcn_readfirstlane(nrows);
  } else if (d.tile_group) {
    if (bx >= *d.n_tiles) return;
    g = d.tile_group[bx];
    row0 = d.tile_row0[bx];
    nrows = min(kRowsMax, d.tile_rows[bx]);
  } else {
    g = bz;
    row0 = bx * kRowsMax;
    nrows = min(kRowsMax, d.rows - row0);
  }
  if (nrows <= 0) return;                                     // an empty tile of a table has no last row to repeat
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l15 = lane & 15, gq = lane >> 4;
  const bool glu = EX && OB == 2 && ex.glu;                   // block 0 holds gate rows, block 1 their up rows
  const int per_blk = glu ? 16 : OB * 16, per_wg = 4 / wk * per_blk;      // outputs of a wave's share, of a workgroup
  const int blk = wave / wk, ks = wave - blk * wk;
  const int m0 = by * per_wg + blk * per_blk;
  // rows of position p: a shared slice's positions are the step's rows in order
  auto x_row = [&](int p) {
    if (EX && ex.chosen) return shared ? (ex.by_pair ? p : p - row0) : ex.by_pair ? my_pair : my_pair / ex.top;      // a lane's own row
    return d.x_row_index ? (shared ? p - row0 : d.x_row_index[p]) : p;
  };
  auto y_row = [&](int p) { return chosen ? list[p] : d.y_row_index && !shared ? d.y_row_index[p] : p; };
  const TX* X = static_cast<const TX*>(d.x) + (shared ? 0 : (int64_t)g * d.x_group_stride);
  const uint16_t* W = shared ? ex.w + g * ex.group_stride : static_cast<const uint16_t*>(d.w) + (int64_t)g * d.w_group_stride;
  const int64_t wm = shared ? ex.m_stride : d.w_m_stride, up = shared ? ex.up : (int64_t)d.m * d.w_m_stride;
  const int tok = row0 + min(l15, nrows - 1);                 // absent rows repeat the last one; they are never stored
  const TX* xp = X + (int64_t)x_row(tok) * d.x_row_stride + gq * 16;
  const int pchunk = 2 * gq + (lane & 1);
  const uint16_t* wp[OB][2];
#pragma unroll
  for (int o = 0; o < OB; ++o)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      wp[o][h] = W + (int64_t)min(m0 + (glu ? 0 : o * 16) + h * 8 + ((lane >> 1) & 7), d.m - 1) * wm + (glu && o ? up : 0) + pchunk * 8;
  const int K = d.k, np = (K + 63) >> 6, mine = ks < np ? (np - ks + wk - 1) / wk : 0;   // pieces of k; those of this wave
  f32x4 acc[OB][2][2];
#pragma unroll
  for (int o = 0; o < OB; ++o)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[o][q >> 1][q & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Set { RowPiece<TX> x[CH][2]; u32x4 w[CH][OB][2]; } A, B;
  const u32x4 zero = {0u, 0u, 0u, 0u};
  auto issue = [&](int i0, Set& s) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (i0 + c >= mine) continue;
      const int k = (ks + (i0 + c) * wk) * 64;
      if (k + 64 <= K) {
#pragma unroll
        for (int h = 0; h < 2; ++h) s.x[c][h].load(xp + k + h * 8);
#pragma unroll
        for (int o = 0; o < OB; ++o)
#pragma unroll
          for (int h = 0; h < 2; ++h) s.w[c][o][h] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wp[o][h] + k));
      } else {                                                // the last piece of a K that is no multiple of 64 (it is one of 8)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (k + gq * 16 + h * 8 < K) s.x[c][h].load(xp + k + h * 8);
          else s.x[c][h].zero();
        }
#pragma unroll
        for (int o = 0; o < OB; ++o)
#pragma unroll
          for (int h = 0; h < 2; ++h) s.w[c][o][h] = k + pchunk * 8 < K ? *reinterpret_cast<const u32x4*>(wp[o][h] + k) : zero;
      }
    }
  };
  auto compute = [&](int i0, const Set& s) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (i0 + c >= mine) continue;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        bf16x8_t xf[NP];
        s.x[c][h].parts(xf);
#pragma unroll
        for (int q = NP - 1; q >= 0; --q)                     // the smallest part first
#pragma unroll
          for (int o = 0; o < OB; ++o)
#pragma unroll
            for (int rh = 0; rh < 2; ++rh)
              acc[o][rh][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, s.w[c][o][rh]), xf[q], acc[o][rh][h], 0, 0, 0);
      }
    }
  };
  issue(0, A);
  if (CH < mine) issue(CH, B);
  for (int i0 = 0; i0 < mine; i0 += 2 * CH) {
    compute(i0, A);
    if (i0 + 2 * CH < mine) issue(i0 + 2 * CH, A);
    if (i0 + CH >= mine) break;
    compute(i0 + CH, B);
    if (i0 + 3 * CH < mine) issue(i0 + 3 * CH, B);
  }
  // slot i of lane ln: output (i >> 1) * 8 + 2 (ln >> 4) + (i & 1) of the block, row ln & 15
#pragma unroll
  for (int o = 0; o < OB; ++o)
    red[wave][o][lane] = f32x4{acc[o][0][0][0] + acc[o][0][1][1], acc[o][0][0][2] + acc[o][0][1][3],
                               acc[o][1][0][0] + acc[o][1][1][1], acc[o][1][0][2] + acc[o][1][1][3]};
  __syncthreads();
  TY* Y = static_cast<TY*>(d.y) + (shared ? 0 : (int64_t)g * d.y_group_stride);
  const float* part = reinterpret_cast<const float*>(red);
  for (int e = tid; e < per_wg * 16; e += 256) {              // consecutive threads: consecutive outputs of one row
    const int out = e % per_wg, r = e / per_wg;
    const int m = by * per_wg + out;
    if (r >= nrows || m >= d.m) continue;
    const int b = out / per_blk, o = glu ? 0 : (out >> 4) % OB, j = out & 15;
    const int at = (o * 64 + ((j & 7) >> 1) * 16 + r) * 4 + (j >> 3) * 2 + (j & 1);
    float v = part[b * wk * OB * 256 + at];
    for (int w = 1; w < wk; ++w) v += part[(b * wk + w) * OB * 256 + at];
    const int p = row0 + r;
    if constexpr (NP > 1) {
      // a cut-off part of zero times an infinite weight is no number where the value's own product is an infinity: summed again from whole
      // values, up to the first that settles it
      if (v != v) {
        const TX* xr = X + (int64_t)x_row(p) * d.x_row_stride;
        const uint16_t* wr = W + (int64_t)m * d.w_m_stride;
        v = 0.f;
        for (int k = 0; k < K && v == v; ++k) v = fmaf(ld(xr + k), ld(wr + k), v);
      }
    }
    if (glu) {
      float u = part[b * wk * OB * 256 + at + 256];
      for (int w = 1; w < wk; ++w) u += part[(b * wk + w) * OB * 256 + at + 256];
      v = glu_f(ex, shared, v, u);
    } else if (d.epilogue == PEGAINFER_EPI_RELU_SQ) { v = fmaxf(v, 0.f); v *= v; }
    else if (d.epilogue == PEGAINFER_EPI_GELU_ERF) v = gelu_erf_f(v);
    else if (d.epilogue == PEGAINFER_EPI_SIGMOID_GATE)
      v *= sigmoid_f(ld(static_cast<const TG*>(d.gate) + (int64_t)x_row(p) * d.gate_row_stride + g));
    st(Y + (int64_t)y_row(p) * d.y_row_stride + m, v);
  }
}

// how the matrix-core form is launched: waves that share a block's K, blocks of outputs per wave, and the grid
struct RowsMfmaShape { int wk, ob; dim3 grid; };
inline RowsMfmaShape rows_mfma_shape(const pegainfer_gemm_desc& d) {
  const int np = ceil_div(d.k, 64), wk = np >= 8 ? 4 : np >= 4 ? 2 : 1;
  // the tiles that a table's bound allows for and that are empty come last: an even grid width would send the others' workgroups, in
  // their round robin over the XCDs, to some of the eight only
  const int row_tiles = d.tile_group ? d.max_tiles | 1 : ceil_div(d.rows, kRowsMax), groups = d.tile_group ? 1 : d.groups;
  const int blocks = ceil_div(d.m, 16 * (4 / wk));
  // two blocks of outputs per wave (each x piece used twice) where that still gives every compute unit two workgroups
  const bool two = (long)row_tiles * groups * blocks >= 4L * device_cus();
  return {wk, two ? 2 : 1, dim3(row_tiles, two ? ceil_div(blocks, 2) : blocks, groups)};
}
inline long rows_direct_all(const pegainfer_gemm_desc& d, int R) {
  return (long)(d.tile_group ? d.max_tiles | 1 : ceil_div(d.rows, R)) * (d.tile_group ? 1 : d.groups) * d.m;
}
// Outputs of a wave of the direct form: the more, the fewer workgroups come and go and the more often a row's values are used; the fewer, the more
// of a long row of weights is on its way.  So four from three outputs per wave of the chip on while a weight row is one piece (2 KB), for longer ones two, four
// where three or four rows and many outputs use them, and one where a single row needs nothing but weights.  One / two / four (us):
//   one row    16 384 x 256 9.9 / 7.0 / 5.3       16 384 x 1024 12.9 / 11.7 / 13.0   4096 x 8192 22.8 / 25.6 / 32.2
//   two rows   16 384 x 256 10.9 / 8.6 / 5.8      16 384 x 1024 13.8 / 12.3 / 13.8   4096 x 8192 26.6 / 25.8 / 32.7
//   four rows  16 384 x 256 15.4 / 12.7 / 7.5     16 384 x 1536 28.8 / 24.4 / 19.1   4096 x 8192 36.1 / 27.1 / 35.0
inline int rows_direct_outputs(const pegainfer_gemm_desc& d, int R, bool glu) {
  const long outputs = rows_direct_all(d, R), waves = 4L * device_cus();
  if (glu) return outputs >= 2 * waves ? 2 : 1;
  if (2 * outputs < 3 * waves) return 1;
  const bool f32 = d.w_dtype == kDtF32;
  const int words = f32 ? d.k : d.k / 2;                  // of a weight row
  if (words <= 512) return outputs >= 3 * waves ? 4 : 2;
  if (R == 1 && f32 && words >= 2048) return 1;
  return R > 2 && words <= 4096 && outputs >= 8 * waves ? 4 : 2;
}
// operands in 16-byte chunks
inline bool chunks_ok(const pegainfer_gemm_desc& d) {
  auto a16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  return d.w_k_stride == 1 && (d.k & 7) == 0 && (d.x_row_stride & 7) == 0 && (d.x_group_stride & 7) == 0 &&
         (d.w_m_stride & 7) == 0 && (d.w_group_stride & 7) == 0 && a16(d.x) && a16(d.w);
}

}  // namespace pk
