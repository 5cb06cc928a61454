// Attention over a paged LATENT cache (beside the paged K/V attention of attn_prefill.hip / attn_decode.hip).
//
// A token's cache entry in a layer is ONE vector shared by all heads: [c (rank) | kr (rot)] - the normalised compressed
// key/value latent and the rotated key part.  The per-head key up-projection is folded into the query
// (qc[t, h, :rank] = Wuk_h^T q_nope[t, h], the "absorb" GEMM) and the value up-projection is applied to the attention
// output (o[t, h] = Wuv_h o_lat[t, h]), so the kernel works on the cache as stored:
//     score_j = (qc[t, h, :] . entry_j) * scale,   o_lat[t, h, :] = sum_j softmax(score)_j entry_j[:rank].
// Every head of a token reads the same entries, and the rows of a step (prompt portions and single decoded tokens of
// several requests) differ only in (request, position): one kernel serves prefill, decode and mixed steps.
// Scores, softmax weights, running maxima / sums and the output accumulators are fp32; the fp32 instance reads an fp32
// cache, the bf16 instance widens bf16 entries exactly.
//
//   latent_prep_kernel        RMS-norm of the latent, rotation of the shared key part and of the query's rotated part (halves or
//                             neighbours), cache write; RMS-norm of a query latent (each part optional)
//   latent_attn_kernel        any sizes: one workgroup per (token, head, key split), 256 keys per round, scores by one thread per
//                             key, online softmax, value accumulation by one thread per latent dimension
//   latent_attn_mfma_kernel   bf16 cache, tiles of up to 64 (token, head) rows of one request: a wave per 16 rows
//   latent_attn_tile_kernel   the same tiles where the entry is whole blocks of 32 values of rank 256 or 512: eight waves share 64 rows and 64 keys
//   latent_attn_few_kernel    tiles of a few rows of a bf16 cache, any tile of an fp32 one: four waves per 16 or 32 rows
//   latent_attn_merge_kernel  combines the key splits of a row (log-sum-exp weights), fixed split order
// A row's result depends on its own query, position and cache entries only.  With contiguous splits the split count is a
// function of the row's key count alone; with dealt splits it also depends on the step's shape (rounding only).
#include <type_traits>

#include "gemm_rows.h"

namespace pk {

constexpr int kLatKeys = 256;        // keys per round = threads per workgroup
constexpr int kLatAcc = 4;           // latent dims per thread: rank <= 1024
constexpr int kLatSplitKeys = 1024;  // default keys per split of a row

__device__ __forceinline__ float block_max256(float v, float* red) {
  v = wave_max(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// How a row's keys are cut into splits.  Contiguous: split z holds keys z * grain .. (z + 1) * grain - 1, and the number of splits
// follows the context's length.  Dealt: runs of `grain` keys (one tile) go round the splits in turn - split z takes runs z,
// z + n, ... - so the launch's grid does not depend on the contexts' lengths and a recorded launch serves every later step.
struct LatentCut {
  int grain, dealt;
  __device__ __forceinline__ int splits_of(int n_keys, int max_splits) const { return min(max_splits, (n_keys + grain - 1) / grain); }
  __device__ __forceinline__ int end_of(int split, int n_keys) const { return dealt ? n_keys : min(n_keys, (split + 1) * grain); }
  __device__ __forceinline__ int step(int tile, int max_splits) const { return dealt ? tile * max_splits : tile; }
};

template <typename A>
__device__ __forceinline__ const A* latent_entry(const A* cache, int64_t page_stride, int64_t layer_off, int page_size,
                                                 const int32_t* pages, int j, int E) {
  return cache + (int64_t)pages[j / page_size] * page_stride + layer_off + (int64_t)(j % page_size) * E;
}

// What one prep launch does to a token row; every part is optional (its pointer NULL).
template <typename A>
struct LatentPrep {
  const A* dkv; int64_t dkv_stride; const A* c_norm;                      // [c: r | kr: dr] -> cache entry
  const A* ql; int64_t ql_stride; const A* ql_norm; A* ql_out; int q_rank;  // query latent, RMS-normed with a weight -> packed rows
  const A* q; int64_t q_stride; float* qc;                                // rotated parts of the heads' queries -> qc (fp32)
};

// the sizes and the cache of a prep launch
struct LatentPlace {
  float eps;
  const float* inv_freq;
  int rot_dims, pairs;
  const int32_t *positions, *token_req, *page_indptr, *page_ids;
  int64_t page_stride, layer_off;
  int page_size, H, dn, dr, r;
};

// of 256 threads: token row t, workgroup y of ny of the row
template <typename A>
__device__ __forceinline__ void latent_prep_block(int t, int y, int ny, const LatentPrep<A>& a, const LatentPlace& p, A* __restrict__ cache) {
  __shared__ float red[4];
  const int tid = threadIdx.x;
  const int pos = p.positions[t];
  const int r = p.r, E = r + p.dr;
  const A* dkv = a.dkv ? a.dkv + (int64_t)t * a.dkv_stride : nullptr;
  A* entry = nullptr;
  if (dkv) {
    const int req = p.token_req[t];
    entry = cache + (int64_t)p.page_ids[p.page_indptr[req] + pos / p.page_size] * p.page_stride + p.layer_off + (int64_t)(pos % p.page_size) * E;
  }
  // with several workgroups per row (few rows) the first norms the key latent, the last the query latent
  if (dkv && y == 0) {
    float ss = 0.f;
    for (int i = tid; i < r; i += 256) { const float v = ld(dkv + i); ss += v * v; }
    ss = block_sum<4>(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)r + p.eps);
    for (int i = tid; i < r; i += 256) st(entry + i, ld(dkv + i) * inv * ld(a.c_norm + i));
  }
  if (a.ql && y + 1 == ny) {
    const A* ql = a.ql + (int64_t)t * a.ql_stride;
    A* out = a.ql_out + (int64_t)t * a.q_rank;
    float ss = 0.f;
    for (int i = tid; i < a.q_rank; i += 256) { const float v = ld(ql + i); ss += v * v; }
    ss = block_sum<4>(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)a.q_rank + p.eps);
    for (int i = tid; i < a.q_rank; i += 256) st(out + i, ld(ql + i) * inv * ld(a.ql_norm + i));
  }
  const int half = p.rot_dims >> 1;
  const float fpos = (float)pos;
  // vector 0 = the shared key part (-> cache), vectors 1 .. p.H = the heads' rotated query parts (-> qc, fp32)
  const int w_end = (a.q ? p.H + 1 : 1) * p.dr;
  for (int w = (dkv ? 0 : p.dr) + y * 256 + tid; w < w_end; w += 256 * ny) {
    const int vec = w / p.dr, i = w % p.dr;
    const A* src = vec == 0 ? dkv + r : a.q + (int64_t)t * a.q_stride + (int64_t)(vec - 1) * (p.dn + p.dr) + p.dn;
    float out = ld(src + i);
    if (i < p.rot_dims) {
      float sn, cs;
      const int f = p.pairs ? i >> 1 : (i < half ? i : i - half);
      const bool second = p.pairs ? (i & 1) : i >= half;
      const float other = ld(src + (p.pairs ? i ^ 1 : second ? i - half : i + half));
      sincosf(fpos * p.inv_freq[f], &sn, &cs);
      out = second ? out * cs + other * sn : out * cs - other * sn;
    }
    if (vec == 0) st(entry + r + i, out);
    else a.qc[((int64_t)t * p.H + (vec - 1)) * E + r + i] = out;
  }
}
template <typename A>
__global__ __launch_bounds__(256) void latent_prep_kernel(LatentPrep<A> a, LatentPlace p, A* __restrict__ cache) {
  latent_prep_block<A>(blockIdx.x, blockIdx.y, gridDim.y, a, p, cache);
}

// Few rows (decoding): the prep and the product that carries the heads' queries into the latent space, which touch different values of qc and
// read the same rows, in one grid - two launches that wait on chains of their own and leave most of the chip idle.  The product's workgroups
// first.  4 rows, 16 heads, rank 512: 4.5 + 5.0 us one after the other, 5.2 in one (traced); 16 steps of four such layers and their prompts
// 8.70 -> 8.43 ms.
template <int OB>
__global__ __launch_bounds__(256) void latent_prep_absorb_kernel(LatentPrep<uint16_t> a, LatentPlace p, uint16_t* __restrict__ cache, int ny,
                                                                 pegainfer_gemm_desc d, int wk, int gx, int gy, int n_gemm) {
  const int b = blockIdx.x;
  if (b < n_gemm) {
    gemm_rows_mfma_block<uint16_t, float, uint16_t, OB, false>(d, wk, ExpertForm{}, b % gx, b / gx % gy, b / (gx * gy));
    return;
  }
  latent_prep_block<uint16_t>((b - n_gemm) / ny, (b - n_gemm) % ny, ny, a, p, cache);
}
template <int R, int MB>
__global__ __launch_bounds__(256) void latent_prep_absorb_f32_kernel(LatentPrep<float> a, LatentPlace p, float* __restrict__ cache, int ny,
                                                                     pegainfer_gemm_desc d, int gy, int n_gemm) {
  const int b = blockIdx.x;
  if (b < n_gemm) {
    gemm_rows_direct_block<float, float, uint16_t, R, MB, false>(d, 0, 0, 0, b % gy, b / gy);
    return;
  }
  latent_prep_block<float>((b - n_gemm) / ny, (b - n_gemm) % ny, ny, a, p, cache);
}

// What a split of a row leaves for the merge, all fp32: the rows' accumulators ([row][split][rank]; row = t * H + h), and behind
// them [row][split][maximum, sum], so that the accumulators of a rank that is a multiple of four lie on 16 bytes.
struct LatentPartial {
  float *acc, *max_sum;      // of one (row, split), or of a row's first split
  int r;
  __device__ __forceinline__ LatentPartial(float* base, int64_t slots, int rank, int64_t slot)
      : acc(base + slot * rank), max_sum(base + slots * rank + 2 * slot), r(rank) {}
  __device__ __forceinline__ LatentPartial(const float* base, int64_t slots, int rank, int64_t slot)
      : LatentPartial(const_cast<float*>(base), slots, rank, slot) {}
  __device__ __forceinline__ f32x4 load(int split, int d, bool vec) const {
    const float* p = acc + (int64_t)split * r + d;
    if (vec) return *reinterpret_cast<const f32x4*>(p);
    return f32x4{p[0], d + 1 < r ? p[1] : 0.f, d + 2 < r ? p[2] : 0.f, d + 3 < r ? p[3] : 0.f};
  }
};

template <typename A>
__global__ __launch_bounds__(256) void latent_attn_kernel(const float* __restrict__ qc, float* __restrict__ o_lat,
                                                          const A* __restrict__ cache, int64_t page_stride,
                                                          int64_t layer_off, int page_size,
                                                          const int32_t* __restrict__ positions,
                                                          const int32_t* __restrict__ token_req,
                                                          const int32_t* __restrict__ page_indptr,
                                                          const int32_t* __restrict__ page_ids, int H, int r, int dr,
                                                          float scale, float* __restrict__ partial, int max_splits, LatentCut cut) {
  extern __shared__ float smem[];
  __shared__ float red[4];
  const int t = blockIdx.x, h = blockIdx.y, split = blockIdx.z, tid = threadIdx.x;
  const int E = r + dr;
  const int n_keys = positions[t] + 1;
  const int n_splits = cut.splits_of(n_keys, max_splits);
  if (split >= n_splits) return;
  const int j_lo = split * cut.grain, j_hi = cut.end_of(split, n_keys), j_step = cut.step(kLatKeys, max_splits);
  float* q = smem;            // [E]
  float* p = smem + E;        // [kLatKeys]
  const float* qrow = qc + ((int64_t)t * H + h) * E;
  for (int i = tid; i < E; i += 256) q[i] = qrow[i];
  const int32_t* pages = page_ids + page_indptr[token_req[t]];
  float m = -INFINITY, l = 0.f, acc[kLatAcc] = {};
  __syncthreads();
  for (int j0 = j_lo; j0 < j_hi; j0 += j_step) {
    const int j = j0 + tid;
    float s = -INFINITY;
    if (j < j_hi) {
      const A* e = latent_entry(cache, page_stride, layer_off, page_size, pages, j, E);
      float a = 0.f;
      for (int i = 0; i < E; ++i) a = fmaf(q[i], ld(e + i), a);
      s = a * scale;
    }
    const float m_new = fmaxf(m, block_max256(s, red));
    const float corr = expf(m - m_new);      // m = -inf on the first round: exp(-inf) = 0
    const float pj = j < j_hi ? expf(s - m_new) : 0.f;
    p[tid] = pj;
    l = l * corr + block_sum<4>(pj, red);    // its barriers also publish p[]
    m = m_new;
    const int cnt = min(kLatKeys, j_hi - j0);
#pragma unroll
    for (int k = 0; k < kLatAcc; ++k) {
      const int d = tid + k * 256;
      if (d >= r) break;
      float a = acc[k] * corr;
      for (int i = 0; i < cnt; ++i)
        a = fmaf(p[i], ld(latent_entry(cache, page_stride, layer_off, page_size, pages, j0 + i, E) + d), a);
      acc[k] = a;
    }
    __syncthreads();
  }
  if (n_splits == 1) {
    const float inv = 1.0f / l;
#pragma unroll
    for (int k = 0; k < kLatAcc; ++k) {
      const int d = tid + k * 256;
      if (d < r) o_lat[((int64_t)t * H + h) * r + d] = acc[k] * inv;
    }
  } else {
    const LatentPartial part(partial, (int64_t)gridDim.x * H * max_splits, r, ((int64_t)t * H + h) * max_splits + split);
    if (tid == 0) { part.max_sum[0] = m; part.max_sum[1] = l; }
#pragma unroll
    for (int k = 0; k < kLatAcc; ++k) {
      const int d = tid + k * 256;
      if (d < r) part.acc[d] = acc[k];
    }
  }
}

// Latency-bound: a workgroup per row and 256 of its latent dims, four waves with every fourth split each, eight splits' values on their way
// together with the maxima and sums that weigh them; the waves' sums meet in LDS in wave order.  16 rows of 512 dims over 29 splits, 4 tokens: a thread per
// dim that walked the splits 9.1 us; a workgroup for all dims, values asked for behind the weights, four at a time 6.4; now 4.8 us.
__global__ __launch_bounds__(256) void latent_attn_merge_kernel(float* __restrict__ o_lat, const float* __restrict__ partial,
                                                                const int32_t* __restrict__ positions, int H, int r,
                                                                int max_splits, LatentCut cut) {
  extern __shared__ __attribute__((aligned(16))) float wsm[];   // [3][256] sums of waves 1 .. 3, then [n_splits] weights exp(m_s - m)
  const int t = blockIdx.x, h = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int d = blockIdx.z * 256 + lane * 4;
  const int n_splits = cut.splits_of(positions[t] + 1, max_splits);
  if (n_splits <= 1) return;
  const LatentPartial part(partial, (int64_t)gridDim.x * H * max_splits, r, ((int64_t)t * H + h) * max_splits);
  const bool vec = (r & 3) == 0, mine = d < r;
  constexpr int kAhead = 8;
  f32x4 v[kAhead];
  auto fetch = [&](int s0) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u) v[u] = mine && s0 + 4 * u < n_splits ? part.load(s0 + 4 * u, d, vec) : f32x4{0.f, 0.f, 0.f, 0.f};
  };
  // every wave reads the splits' maxima and sums itself
  const float m_own = lane < n_splits ? part.max_sum[2 * lane] : -INFINITY, l_own = lane < n_splits ? part.max_sum[2 * lane + 1] : 0.f;
  fetch(wave);
  float* weight = wsm + 3 * 256;
  float m = m_own;
  for (int s = lane + 64; s < n_splits; s += 64) m = fmaxf(m, part.max_sum[2 * s]);
  m = wave_max(m);
  float l = 0.f;
  if (lane < n_splits) {
    const float w = expf(m_own - m);
    l = l_own * w;
    if (wave == 0) weight[lane] = w;
  }
  for (int s = lane + 64; s < n_splits; s += 64) {
    const float w = expf(part.max_sum[2 * s] - m);
    l = fmaf(part.max_sum[2 * s + 1], w, l);
    if (wave == 0) weight[s] = w;
  }
  const float inv = 1.0f / wave_sum(l);
  __syncthreads();
  f32x4 a = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = wave; s0 < n_splits; s0 += 4 * kAhead) {
    if (s0 != wave) fetch(s0);
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      if (s0 + 4 * u < n_splits) a += v[u] * weight[s0 + 4 * u];
  }
  if (wave > 0) *reinterpret_cast<f32x4*>(wsm + (wave - 1) * 256 + lane * 4) = a;
  __syncthreads();
  if (wave == 0 && mine) {
#pragma unroll
    for (int w = 0; w < 3; ++w) a += *reinterpret_cast<const f32x4*>(wsm + w * 256 + lane * 4);
    float* o = o_lat + ((int64_t)t * H + h) * r + d;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (d + e < r) o[e] = a[e] * inv;
  }
}

// ------------------------------------------------------------------ MFMA form (bf16 cache)
// One workgroup = 64 consecutive (token, head) rows of ONE request (4 waves x 16 rows) against key tiles of 32 cache entries,
// v_mfma_f32_16x16x32_bf16 for both products:
//   scores^T [32 keys x 16 rows]  = entries [32 x E] . q^T          A = entry rows from LDS, B = the wave's q rows (bf16 in LDS)
//   out^T    [16 dims x 16 rows] += c^T [16 x 32 keys] . p^T        A = the SAME row-major tile read transposed, B = the lane's own p
// The score MFMA leaves lane (row l15, group g) with the scores of keys 4g..4g+3 and 16+4g..16+4g+3 of its row - exactly the
// eight values the second product wants from that lane as its B operand when the reduction index is numbered
// kidx = 8g + i  <->  key (i < 4 ? 4g + i : 16 + 4g + i - 4): the weights never move between lanes.  The matching A fragment
// (dim l15 of those eight keys) comes from two ds_read_b64_tr_b16: inside a 16-lane group lane 4j + c gives the address of
// dims 4c..4c+3 of key row j, and lane i receives dim i of the four rows - so the latent tile is staged once, row-major, and
// serves both products.  Every head of a token reads the same entries, so a tile of 64 rows (8 tokens x 8 heads, or one
// decoded token's heads) shares each staged key tile.  The next key tile's global loads are issued into registers before the
// current tile's products and written to LDS after them.  KH = 2: eight waves, the second four on keys 32 .. 63 of tiles of 64, with a
// softmax state of their own; the two meet in LDS at the end.  Softmax state (max, sum) and the output accumulators are fp32; q and
// the weights are rounded to bf16 where they enter the matrix cores.  Keys are split over blockIdx.y like the plain form.
constexpr int kTileRows = 64, kTileKeys = 32;
constexpr int kLatPrefetch = 10;     // 16-byte chunks per thread and key tile: 32 keys x (E / 8) <= 2560 chunks, E <= 640

// FULL: the rank is 16 ND, so no step over the latent dims asks whether it is there and the reads of several are on their way together: with
// the longer unroll of the scores 16 heads of 512 + 64, prompts of 300 - 900 tokens 225 -> 208 us, one of 1800 436 -> 387, 100 tokens behind 2000
// 317 -> 280.  A maximum that follows with a lag (no rescaling of most tiles) would take 194 us, but rounds the largest weight, which is
// exactly one here: 1.5 times the error on peaked rows.
template <int ND, bool FULL, int KH>
__global__ __launch_bounds__(256 * KH) void latent_attn_mfma_kernel(const float* __restrict__ qc, float* __restrict__ o_lat,
                                                               const uint16_t* __restrict__ cache, int64_t page_stride,
                                                               int64_t layer_off, int page_size,
                                                               const int32_t* __restrict__ positions,
                                                               const int32_t* __restrict__ token_req,
                                                               const int32_t* __restrict__ page_indptr,
                                                               const int32_t* __restrict__ page_ids,
                                                               const int32_t* __restrict__ tile_row0,
                                                               const int32_t* __restrict__ tile_rows, int H, int r, int dr,
                                                               float scale, float* __restrict__ partial, int n_tokens,
                                                               int max_splits, LatentCut cut) {
  extern __shared__ __align__(16) uint8_t lat_smem[];
  typedef short v4s_t __attribute__((ext_vector_type(4)));
  constexpr int N = 256 * KH, KEYS = kTileKeys * KH;
  const int E = r + dr, Epad = (E + 31) & ~31;
  const int qs = Epad + 8, cs = Epad + 8;                          // LDS row strides (bf16 elements), 16-byte multiples
  uint16_t* Qs = reinterpret_cast<uint16_t*>(lat_smem);            // [64][qs]
  uint16_t* Ck = Qs + kTileRows * qs;                              // [KEYS][cs]
  const int tid = threadIdx.x, wave = (tid >> 6) & 3, kh = tid >> 8, lane = tid & 63, l15 = lane & 15, g = lane >> 4;
  const int row0 = tile_row0[blockIdx.x], cnt = tile_rows[blockIdx.x], split = blockIdx.y;
  const int t_first = row0 / H, t_last = (row0 + cnt - 1) / H;
  const int pmax = positions[t_last];
  const int j_lo = split * cut.grain;
  if (j_lo > pmax) return;
  const int j_hi = cut.end_of(split, pmax + 1), j_step = cut.step(KEYS, max_splits);
  const int32_t* pages = page_ids + page_indptr[token_req[t_first]];
  const int nchunk = E >> 3, tile_chunks = KEYS * nchunk;
  // this thread's chunks of a key tile: key kk, element offset ch * 8 - fixed for the whole loop, so the integer divisions
  // happen once (a wave64 VALU instruction costs four cycles; an emulated division about forty of them)
  u32x4 pre[kLatPrefetch];
  int ck[kLatPrefetch];                                              // key << 16 | element
#pragma unroll
  for (int i = 0; i < kLatPrefetch; ++i) {
    const int c = tid + i * N;
    ck[i] = c < tile_chunks ? c / nchunk << 16 | c % nchunk * 8 : -1;
  }
  const int pshift = (page_size & (page_size - 1)) == 0 ? __ffs(page_size) - 1 : -1;
  auto fetch = [&](int j0) {
#pragma unroll
    for (int i = 0; i < kLatPrefetch; ++i) {
      if (ck[i] >= 0) {
        const int j = min(j0 + (ck[i] >> 16), j_hi - 1);
        const int pg = pshift >= 0 ? j >> pshift : j / page_size;
        const int slot = pshift >= 0 ? j & (page_size - 1) : j - pg * page_size;
        pre[i] = *reinterpret_cast<const u32x4*>(cache + (int64_t)pages[pg] * page_stride + layer_off + (int64_t)slot * E + (ck[i] & 0xFFFF));
      }
    }
  };
  fetch(j_lo);
  {  // q rows -> bf16 in LDS, eight values per step; only the 16-row blocks that hold rows are staged
    const int qchunks = Epad >> 3, rows_staged = min(kTileRows, (cnt + 15) & ~15);
    for (int c = tid; c < rows_staged * qchunks; c += N) {
      const int row = c / qchunks, k = (c - row * qchunks) * 8;
      u32x4 v = {0u, 0u, 0u, 0u};
      if (row < cnt && k < E) {
        const float* src = qc + (int64_t)(row0 + row) * E + k;
        const f32x4 a = *reinterpret_cast<const f32x4*>(src), b = *reinterpret_cast<const f32x4*>(src + 4);
        v = u32x4{pack_bf2(a.x, a.y), pack_bf2(a.z, a.w), pack_bf2(b.x, b.y), pack_bf2(b.z, b.w)};
      }
      *reinterpret_cast<u32x4*>(Qs + row * qs + k) = v;
    }
  }
  for (int i = tid; i < KEYS * (Epad - E); i += N) Ck[(i / (Epad - E)) * cs + E + i % (Epad - E)] = 0;
  const int my_row = wave * 16 + l15;
  const int pq = my_row < cnt ? positions[(row0 + my_row) / H] : -1;
  const bool wave_live = wave * 16 < cnt;                            // a wave without rows only helps staging
  f32x4 o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  // per-lane element offset of the transposed reads inside the key tile: key row 4g + (l15 >> 2), dims 4 (l15 & 3) ..
  const int tr_off = (kTileKeys * kh + 4 * g + (l15 >> 2)) * cs + 4 * (l15 & 3);
  for (int j0 = j_lo; j0 < j_hi; j0 += j_step) {
    __syncthreads();                                                 // the previous tile's reads are done
#pragma unroll
    for (int i = 0; i < kLatPrefetch; ++i)
      if (ck[i] >= 0) *reinterpret_cast<u32x4*>(Ck + (ck[i] >> 16) * cs + (ck[i] & 0xFFFF)) = pre[i];
    __syncthreads();
    if (j0 + j_step < j_hi) fetch(j0 + j_step);
    const int jw = j0 + kTileKeys * kh;                              // this wave's keys of the tile
    if (!wave_live || jw >= j_hi) continue;
    // two independent accumulator pairs over alternating k slices: with one wave per SIMD the LDS read -> MFMA -> MFMA chain
    // of a single pair would run at its latency
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f}, s2 = {0.f, 0.f, 0.f, 0.f}, s3 = {0.f, 0.f, 0.f, 0.f};
    const uint16_t* qp = Qs + my_row * qs + g * 8;
    const uint16_t* kp0 = Ck + (kTileKeys * kh + l15) * cs + g * 8;
    const uint16_t* kp1 = kp0 + 16 * cs;
    int kb = 0;
#pragma unroll 3
    for (; kb + 64 <= Epad; kb += 64) {
      const bf16x8_t qa = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(qp + kb));
      const bf16x8_t qb = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(qp + kb + 32));
      const bf16x8_t a0 = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(kp0 + kb));
      const bf16x8_t a1 = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(kp1 + kb));
      const bf16x8_t b0 = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(kp0 + kb + 32));
      const bf16x8_t b1 = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(kp1 + kb + 32));
      s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, qa, s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, qa, s1, 0, 0, 0);
      s2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0, qb, s2, 0, 0, 0);
      s3 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b1, qb, s3, 0, 0, 0);
    }
    if (kb < Epad) {
      const bf16x8_t qa = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(qp + kb));
      s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(kp0 + kb)), qa, s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(kp1 + kb)), qa, s1, 0, 0, 0);
    }
    s0 += s2;
    s1 += s3;
    float sc[8];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int j = jw + (i < 4 ? 4 * g + i : 16 + 4 * g + i - 4);
      const float v = (i < 4 ? s0[i] : s1[i - 4]) * scale;
      sc[i] = (j <= pq && j < j_hi) ? v : -INFINITY;
      mx = fmaxf(mx, sc[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    const float m_new = fmaxf(m, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float corr = __expf(m - m_use);
    float ps[8], lsum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      ps[i] = bf16_round_f(__expf(sc[i] - m_use));   // the sum uses the weights as the matrix core sees them
      lsum += ps[i];
    }
    lsum += __shfl_xor(lsum, 16, kWave);
    lsum += __shfl_xor(lsum, 32, kWave);
    l = l * corr + lsum;
    m = m_new;
    const u32x4 pw = {pack_bf2(ps[0], ps[1]), pack_bf2(ps[2], ps[3]), pack_bf2(ps[4], ps[5]), pack_bf2(ps[6], ps[7])};
    const bf16x8_t pv = __builtin_bit_cast(bf16x8_t, pw);
    const __attribute__((address_space(3))) uint16_t* ck3 =
        (const __attribute__((address_space(3))) uint16_t*)(Ck) + tr_off;
    // the running maximum of most rows stops moving after the first tiles: rescale only when some row of the wave needs it
    if (__any(corr != 1.0f)) {
#pragma unroll
      for (int d = 0; d < ND; ++d) o[d] *= corr;
    }
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      if (!FULL && d * 16 >= r) break;
      const v4s_t a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s_t __attribute__((address_space(3)))*)(ck3 + d * 16));
      const v4s_t a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s_t __attribute__((address_space(3)))*)(ck3 + d * 16 + 16 * cs));
      const u32x2 w0 = __builtin_bit_cast(u32x2, a0), w1 = __builtin_bit_cast(u32x2, a1);
      const bf16x8_t cv = __builtin_bit_cast(bf16x8_t, u32x4{w0.x, w0.y, w1.x, w1.y});
      o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cv, pv, o[d], 0, 0, 0);
    }
  }
  if constexpr (KH == 2) {                                           // the two halves of the keys meet in LDS
    __syncthreads();
    f32x4* fold = reinterpret_cast<f32x4*>(lat_smem);                // [4][ND][64], then [4][64][2]
    float* ml = reinterpret_cast<float*>(fold + 4 * ND * 64) + (wave * 64 + lane) * 2;
    if (kh == 1) {
#pragma unroll
      for (int d = 0; d < ND; ++d) fold[(wave * ND + d) * 64 + lane] = o[d];
      ml[0] = m;
      ml[1] = l;
    }
    __syncthreads();
    if (kh == 1) return;
    const float m1 = ml[0], m_all = fmaxf(m, m1), m_use = m_all == -INFINITY ? 0.f : m_all;
    const float w0 = __expf(m - m_use), w1 = __expf(m1 - m_use);
    l = l * w0 + ml[1] * w1;
    m = m_all;
#pragma unroll
    for (int d = 0; d < ND; ++d) o[d] = o[d] * w0 + fold[(wave * ND + d) * 64 + lane] * w1;
  }
  if (my_row >= cnt) return;
  const int own_splits = cut.splits_of(pq + 1, max_splits);
  const int64_t grow = row0 + my_row;
  if (own_splits == 1) {
    if (split != 0) return;
    const float inv = 1.0f / l;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      const int dd = d * 16 + 4 * g;
      if (dd < r) *reinterpret_cast<f32x4*>(o_lat + grow * r + dd) = o[d] * inv;
    }
  } else if (split < own_splits) {
    const LatentPartial part(partial, (int64_t)n_tokens * H * max_splits, r, grow * max_splits + split);
    if (g == 0) { part.max_sum[0] = m; part.max_sum[1] = l; }
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      const int dd = d * 16 + 4 * g;
      if (dd < r) *reinterpret_cast<f32x4*>(part.acc + dd) = o[d];
    }
  }
}

// ------------------------------------------------------------------ prompts' form (bf16 cache, whole blocks of 32 values)
// In the form above every wave reads all of a key tile twice from LDS for its sixteen rows, which is what it waits for: 92 KB per 16 rows and 32 keys.
// Here eight waves share the work on 64 rows and 64 keys so that little is read twice: for the scores a wave takes 16 keys and 32 rows, whose queries
// stay in its registers; the weights meet in LDS; for the values it takes an eighth of the latent dims for all 64 rows.  Key tiles come by
// LDS-DMA into two buffers, asked for a whole tile ahead, an instruction per key and part (latent, rotated) with the entry's place in scalar registers; a
// row's LDS stride of one 16-byte chunk more than its values keeps the reads off each other's banks.  Same products, roundings, masks and running maximum as above, one softmax state per row.
// 16 heads of 512 + 64, longest tiles first on both sides: prompts of 901, 701, 501 and 301 tokens 152 -> 100 us, one of 1800 226 -> 140, of 700 99 -> 63;
// 8 heads of 256 + 32 103 -> 65, 168 -> 104, 73 -> 49.  One prompt of 4096 tokens (512 + 64): matrix cores busy 20 % of the time, vector unit 24, LDS 31: the
// three take turns within a tile, with two waves per SIMD in step; registers (the queries' 144 and the values' 64 of 256) leave no room for more.
// Three barriers per tile: the tile has landed; the rows' maxima over each wave's keys; the weights and the rows' factors.
template <int ND, int EB>
struct LatentTileShape {              // rank 16 ND, entries of 32 EB values
  static constexpr int kKeys = 64, kR = 16 * ND, kE = 32 * EB, kChunks = kE / 8 + 1, kRow = kChunks * 8, kPStride = kKeys + 8;
  static constexpr size_t kLds = 2 * kKeys * kRow * 2 + kTileRows * kPStride * 2 + 6 * kTileRows * 4 + 2 * 64 * 16;
};
template <int ND, int EB>
__global__ __launch_bounds__(512) void latent_attn_tile_kernel(const float* __restrict__ qc, float* __restrict__ o_lat,
                                                               const uint16_t* __restrict__ cache, int64_t page_stride, int64_t layer_off, int page_size,
                                                               const int32_t* __restrict__ positions, const int32_t* __restrict__ token_req,
                                                               const int32_t* __restrict__ page_indptr, const int32_t* __restrict__ page_ids,
                                                               const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ tile_rows, int H, int r,
                                                               int dr, float scale, float* __restrict__ partial, int n_tokens, int max_splits, LatentCut cut) {
  typedef short v4s_t __attribute__((ext_vector_type(4)));
  typedef LatentTileShape<ND, EB> Sh;
  constexpr int KEYS = Sh::kKeys, E = Sh::kE, S = Sh::kChunks, R = Sh::kR, ROW = Sh::kRow, DB = ND / 8, PS = Sh::kPStride;
  extern __shared__ __align__(16) uint8_t lat_smem[];
  uint16_t* Ck = reinterpret_cast<uint16_t*>(lat_smem);              // [2][KEYS][ROW]
  uint16_t* P = Ck + 2 * KEYS * ROW;                                 // [64][PS] weights
  float* s_max = reinterpret_cast<float*>(P + kTileRows * PS);       // [4][64] maxima over 16 keys each
  float* s_corr = s_max + 4 * kTileRows;                             // [64]
  int* s_pos = reinterpret_cast<int*>(s_corr + kTileRows);           // [64] the rows' positions, -1: no row
  u32x4* s_q = reinterpret_cast<u32x4*>(s_pos + kTileRows);          // [2][64] the one block of the queries that finds no register
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l15 = lane & 15, g = lane >> 4;
  const int kb = wave & 3, half = wave >> 2;
  const int row0 = tile_row0[blockIdx.x], cnt = tile_rows[blockIdx.x], split = blockIdx.y;
  const int t_first = row0 / H, t_last = (row0 + cnt - 1) / H, pmax = positions[t_last];
  const int j_lo = split * cut.grain;
  if (j_lo > pmax) return;
  const int j_hi = cut.end_of(split, pmax + 1);
  const int32_t* pages = page_ids + page_indptr[token_req[t_first]];
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  const uint32_t ring = (uint32_t)(uintptr_t)(lds_ptr_t)lat_smem;
  // a wave fetches eight neighbouring keys, which lie on one page (page_size and the splits' grain are multiples of eight); keys past the end: the last
  auto page_of = [&](int j0) { return pages[min(j0 + wave * 8, j_hi - 1) / page_size]; };
  auto request = [&](int j0, int page, int buf) {
    const int first = min(j0 + wave * 8, j_hi - 1);
    const uint16_t* base = cache + (int64_t)page * page_stride + layer_off + (int64_t)(first % page_size) * E;
    const int last = j_hi - 1 - first;
    const uint32_t off = lane * 16;
    auto part = [&](int at) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t dst = ring + ((buf * KEYS + wave * 8 + i) * S + at / 8) * 16;
        const uint64_t src = reinterpret_cast<uint64_t>(base + min(i, last) * E + at);
        // (readfirstlane is an int: unsigned before it is widened)
        const uint64_t from = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(src >> 32)) << 32 |
                              (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)src);
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(from), "s"(__builtin_amdgcn_readfirstlane(dst)) : "memory", "m0");
      }
    };
    if (R == 512 || lane < R / 8) part(0);
    if (lane < (E - R) / 8) part(R);
  };
  request(j_lo, page_of(j_lo), 0);
  int page = page_of(j_lo + KEYS);
  // the rows go through the other buffer, as bf16, to the waves' registers: the scores' second operand
  if (tid < kTileRows) s_pos[tid] = tid < cnt ? positions[(row0 + tid) / H] : -1;
  {
    constexpr int ALL = kTileRows * (E / 8), N = (ALL + 511) / 512;
    u32x4 v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = min(i * 512 + tid, ALL - 1), row = c / (E / 8);
      const float* src = qc + (int64_t)(row0 + min(row, cnt - 1)) * E + (c - row * (E / 8)) * 8;
      const f32x4 a = *reinterpret_cast<const f32x4*>(src), b = *reinterpret_cast<const f32x4*>(src + 4);
      v[i] = u32x4{pack_bf2(a.x, a.y), pack_bf2(a.z, a.w), pack_bf2(b.x, b.y), pack_bf2(b.z, b.w)};
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = min(i * 512 + tid, ALL - 1), row = c / (E / 8);
      *reinterpret_cast<u32x4*>(Ck + (KEYS + row) * ROW + (c - row * (E / 8)) * 8) = v[i];
    }
  }
  auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };      // (not the tile on its way)
  barrier();
  bf16x8_t q[2][EB];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int k = 0; k < EB; ++k)
      q[rb][k] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(Ck + (KEYS + half * 32 + rb * 16 + l15) * ROW + 32 * k + 8 * g));
  if (kb == 0) s_q[half * 64 + lane] = __builtin_bit_cast(u32x4, q[1][EB - 1]);
  // the lane's number; what follows from it is worked out where it is needed and not kept over the loop, where there is no register for it
  auto here = [&] {
    int n = lane;
    asm volatile("" : "+v"(n));
    return n;
  };
  f32x4 o[4][DB];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int d = 0; d < DB; ++d) o[b][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};            // l: of this lane's keys alone
  int buf = 0;
  for (int j0 = j_lo; j0 < j_hi; j0 += KEYS, buf ^= 1) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (j0 + KEYS < j_hi) request(j0 + KEYS, page, buf ^ 1);
    page = page_of(j0 + 2 * KEYS);
    f32x4 s[2] = {};
    {
      const int ln = here();
      const uint16_t* kp = Ck + (buf * KEYS + kb * 16 + (ln & 15)) * ROW + 8 * (ln >> 4);
      constexpr int AHEAD = 2;                                       // reads on their way
      u32x4 a[AHEAD];
#pragma unroll
      for (int k = 0; k < AHEAD; ++k) a[k] = *reinterpret_cast<const u32x4*>(kp + 32 * k);
#pragma unroll
      for (int k = 0; k < EB; ++k) {
        const bf16x8_t now = __builtin_bit_cast(bf16x8_t, a[k % AHEAD]);
        s[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(now, q[0][k], s[0], 0, 0, 0);
        s[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(now, k < EB - 1 ? q[1][k] : __builtin_bit_cast(bf16x8_t, s_q[half * 64 + ln]), s[1], 0, 0, 0);
        if (k + AHEAD < EB) a[k % AHEAD] = *reinterpret_cast<const u32x4*>(kp + 32 * (k + AHEAD));
        __builtin_amdgcn_sched_barrier(0);                           // (and no more: there is no register for them)
      }
    }
    float sc[2][4];
    const int ln = here(), l15 = ln & 15, g = ln >> 4;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int pq = s_pos[half * 32 + rb * 16 + l15];
      float mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = j0 + kb * 16 + 4 * g + i;
        sc[rb][i] = (j <= pq && j < j_hi) ? s[rb][i] * scale : -INFINITY;
        mx = fmaxf(mx, sc[rb][i]);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
      mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
      if (g == 0) s_max[kb * kTileRows + half * 32 + rb * 16 + l15] = mx;
    }
    barrier();
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int row = half * 32 + rb * 16 + l15;
      const float m_new = fmaxf(m[rb], fmaxf(fmaxf(s_max[row], s_max[kTileRows + row]), fmaxf(s_max[2 * kTileRows + row], s_max[3 * kTileRows + row])));
      const float m_use = m_new == -INFINITY ? 0.f : m_new, corr = m_new == -INFINITY ? 1.f : __expf(m[rb] - m_use);
      float ps[4], sum = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ps[i] = bf16_round_f(__expf(sc[rb][i] - m_use));             // the sum uses the weights as the matrix core sees them
        sum += ps[i];
      }
      l[rb] = l[rb] * corr + sum;
      m[rb] = m_new;
      *reinterpret_cast<u32x2*>(P + row * PS + kb * 16 + 4 * g) = u32x2{pack_bf2(ps[0], ps[1]), pack_bf2(ps[2], ps[3])};
      if (kb == 0 && g == 0) s_corr[row] = corr;
    }
    barrier();
    {
      float c[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) c[b] = s_corr[b * 16 + l15];
      // the running maximum of most rows stops moving after the first tiles: rescale only when some row needs it
      if (__any(c[0] != 1.0f || c[1] != 1.0f || c[2] != 1.0f || c[3] != 1.0f)) {
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int d = 0; d < DB; ++d) o[b][d] *= c[b];
      }
    }
    const __attribute__((address_space(3))) uint16_t* ck3 = (const __attribute__((address_space(3))) uint16_t*)(Ck) +
        (buf * KEYS + 4 * g + (l15 >> 2)) * ROW + 4 * (l15 & 3) + wave * DB * 16;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      bf16x8_t w[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const uint16_t* pp = P + (b * 16 + l15) * PS + 32 * h + 4 * g;
        const u32x2 lo = *reinterpret_cast<const u32x2*>(pp), hi = *reinterpret_cast<const u32x2*>(pp + 16);
        w[b] = __builtin_bit_cast(bf16x8_t, u32x4{lo.x, lo.y, hi.x, hi.y});
      }
#pragma unroll
      for (int d = 0; d < DB; ++d) {
        const v4s_t a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s_t __attribute__((address_space(3)))*)(ck3 + 32 * h * ROW + d * 16));
        const v4s_t a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s_t __attribute__((address_space(3)))*)(ck3 + (32 * h + 16) * ROW + d * 16));
        const u32x2 w0 = __builtin_bit_cast(u32x2, a0), w1 = __builtin_bit_cast(u32x2, a1);
        const bf16x8_t cv = __builtin_bit_cast(bf16x8_t, u32x4{w0.x, w0.y, w1.x, w1.y});
#pragma unroll
        for (int b = 0; b < 4; ++b)
          o[b][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cv, w[b], o[b][d], 0, 0, 0);
      }
    }
  }
  barrier();
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const int row = half * 32 + rb * 16 + l15;
    l[rb] += __shfl_xor(l[rb], 16, kWave);
    l[rb] += __shfl_xor(l[rb], 32, kWave);
    if (g == 0) s_max[kb * kTileRows + row] = l[rb];
    if (kb == 0 && g == 0) s_corr[row] = m[rb];
  }
  barrier();
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int row = b * 16 + l15;
    if (row >= cnt) continue;
    const float sum = (s_max[row] + s_max[kTileRows + row]) + (s_max[2 * kTileRows + row] + s_max[3 * kTileRows + row]);
    const int own_splits = cut.splits_of(positions[(row0 + row) / H] + 1, max_splits);
    const int64_t grow = row0 + row;
    if (own_splits == 1 ? split != 0 : split >= own_splits) continue;
    const LatentPartial part(partial, (int64_t)n_tokens * H * max_splits, r, grow * max_splits + split);
    float* dst = own_splits == 1 ? o_lat + grow * r : part.acc;
    const float inv = own_splits == 1 ? 1.0f / sum : 1.0f;
    if (own_splits > 1 && wave == 0 && g == 0) { part.max_sum[0] = s_corr[row]; part.max_sum[1] = sum; }
#pragma unroll
    for (int d = 0; d < DB; ++d) *reinterpret_cast<f32x4*>(dst + (wave * DB + d) * 16 + 4 * g) = o[b][d] * inv;
  }
}

// ------------------------------------------------------------------ few-rows form (decoding, and every tile of an fp32 cache)
// The form above gives each wave sixteen rows of its own: a decoded token's sixteen heads then keep one wave of four busy, alone on its
// SIMD, with 2 x 18 dependent products for the scores and 64 transposed reads for the values of every key tile.  Here the four waves share
// the same 16 RB rows: wave w takes every fourth block of the entry for the scores (the four parts meet in LDS, added in wave order),
// eight threads per row take the softmax of the tile, and wave w takes every fourth block of latent dims of the values.  Queries
// stay in registers (a wave's own quarter of the entry), so LDS holds the key tile and the tile's scores alone.
// The fp32 instance works on v_mfma_f32_16x16x4_f32: lane (l15, g) fetches four neighbouring values at 4 g of a 16-wide block with one
// 16-byte read, and product e of the block takes value e of every lane - both operands numbered alike; its weights stay fp32.
// A key that a row does not see has weight zero in the products.  In bf16, as in the form above, an entry that is infinite or no number so reaches
// the rows of its request that share its key tile; in fp32 a tile with such an entry (all its scores are none) is summed key by key for the
// rows that see it, and the rows before it keep what the plain form gives them.
// Bound by the latency of one pass through scores, softmax and values (three barriers per tile of 32 keys), not by memory.
// With the merge, 16 heads of 512 + 64 and 4 requests of 500 to 900 keys in splits of 32: 17.1 (the form above) -> 15.9 us, 32 requests
// 53.6 -> 35.0 us.  In fp32, where a workgroup took one head and a thread one key: 8 heads of 256 + 64, two requests of up to 300 keys
// 54 -> 14 us, their 470 prompt tokens 228 -> 66 us.
template <typename A, int ND, int RB>
__global__ __launch_bounds__(256) void latent_attn_few_kernel(const float* __restrict__ qc, float* __restrict__ o_lat,
                                                              const A* __restrict__ cache, int64_t page_stride, int64_t layer_off,
                                                              int page_size, const int32_t* __restrict__ positions,
                                                              const int32_t* __restrict__ token_req,
                                                              const int32_t* __restrict__ page_indptr,
                                                              const int32_t* __restrict__ page_ids,
                                                              const int32_t* __restrict__ tile_row0,
                                                              const int32_t* __restrict__ tile_rows, int H, int r, int dr, float scale,
                                                              float* __restrict__ partial, int n_tokens, int max_splits, LatentCut cut) {
  typedef short v4s_t __attribute__((ext_vector_type(4)));
  constexpr bool F32 = std::is_same<A, float>::value;
  constexpr int kRows = 16 * RB;
  constexpr int kPer = 16 / (int)sizeof(A);               // values of a 16-byte chunk
  constexpr int KB = F32 ? 16 : 32;                       // width of a score block
  constexpr int kMaxE = ND <= 4 ? 384 : 640;              // widest entry of this instance (latent_few_shape)
  constexpr int NB = (kMaxE / KB + 3) / 4;                // blocks of a wave at most
  constexpr int NP = kTileKeys * kMaxE / kPer / 256;      // chunks of a key tile per thread
  constexpr int kSStride = kTileKeys + 4;
  extern __shared__ __align__(16) uint8_t lat_smem[];
  const int E = r + dr, Epad = (E + KB - 1) / KB * KB, cs = Epad + kPer;      // a row's LDS stride: 16 bytes past a multiple of 64
  A* Ck = reinterpret_cast<A*>(lat_smem);                                      // [32][cs]
  float* S = reinterpret_cast<float*>(Ck + kTileKeys * cs);                    // [4][kRows][kSStride] parts of the scores
  A* P = reinterpret_cast<A*>(S + 4 * kRows * kSStride);                       // [kRows][kSStride] weights
  float* s_row = reinterpret_cast<float*>(P + kRows * kSStride);               // [kRows] rescale of the tile, at the end 1 / sum
  __shared__ int s_spoilt[4];                              // per wave of the softmax: a score of the tile is no finite number
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l15 = lane & 15, g = lane >> 4;
  const int tile = blockIdx.x, sub = blockIdx.z, split = blockIdx.y;
  const int cnt = min(kRows, tile_rows[tile] - sub * kRows);
  if (cnt <= 0) return;
  const int row0 = tile_row0[tile] + sub * kRows;
  const int t_first = row0 / H, t_last = (row0 + cnt - 1) / H;
  const int pmax = positions[t_last];
  const int j_lo = split * cut.grain;
  if (j_lo > pmax) return;
  const int j_hi = cut.end_of(split, pmax + 1), j_step = cut.step(kTileKeys, max_splits);
  const int32_t* pages = page_ids + page_indptr[token_req[t_first]];
  const int nchunk = E / kPer, tile_chunks = kTileKeys * nchunk;
  u32x4 pre[NP];
  int ck_kk[NP], ck_el[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int c = tid + i * 256;
    ck_kk[i] = c < tile_chunks ? c / nchunk : -1;
    ck_el[i] = c < tile_chunks ? (c - ck_kk[i] * nchunk) * kPer : 0;
  }
  const int pshift = (page_size & (page_size - 1)) == 0 ? __ffs(page_size) - 1 : -1;
  auto fetch = [&](int j0) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if (ck_kk[i] >= 0) {
        const int j = min(j0 + ck_kk[i], j_hi - 1);
        const int pg = pshift >= 0 ? j >> pshift : j / page_size;
        const int slot = pshift >= 0 ? j & (page_size - 1) : j - pg * page_size;
        pre[i] = *reinterpret_cast<const u32x4*>(cache + (int64_t)pages[pg] * page_stride + layer_off + (int64_t)slot * E + ck_el[i]);
      }
    }
  };
  fetch(j_lo);
  // this wave's blocks of the queries: fp32 values 4 g .. of a block of 16, or bf16 values 8 g .. of a block of 32
  const int blocks = Epad / KB;
  u32x4 q[RB][NB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      q[rb][b] = u32x4{0u, 0u, 0u, 0u};
      const int k = (wave + 4 * b) * KB + g * kPer, row = rb * 16 + l15;
      if (row < cnt && k < E) {
        const float* src = qc + (int64_t)(row0 + row) * E + k;
        if constexpr (F32) q[rb][b] = *reinterpret_cast<const u32x4*>(src);
        else {
          const f32x4 a = *reinterpret_cast<const f32x4*>(src), c = *reinterpret_cast<const f32x4*>(src + 4);
          q[rb][b] = u32x4{pack_bf2(a.x, a.y), pack_bf2(a.z, a.w), pack_bf2(c.x, c.y), pack_bf2(c.z, c.w)};
        }
      }
    }
  for (int i = tid; i < kTileKeys * (Epad - E); i += 256) Ck[(i / (Epad - E)) * cs + E + i % (Epad - E)] = 0;
  // softmax: eight threads per row, four keys each
  const int my_row = tid >> 3, my_key = 4 * (tid & 7);
  const bool sm_live = my_row < cnt;                       // whole groups of eight lanes
  const int pq = sm_live ? positions[(row0 + my_row) / H] : -1;
  float m = -INFINITY, l = 0.f;
  f32x4 o[RB][ND];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int d = 0; d < ND; ++d) o[rb][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int j0 = j_lo; j0 < j_hi; j0 += j_step) {
    __syncthreads();                                       // the previous tile's values are read
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (ck_kk[i] >= 0) *reinterpret_cast<u32x4*>(Ck + ck_kk[i] * cs + ck_el[i]) = pre[i];
    __syncthreads();
    if (j0 + j_step < j_hi) fetch(j0 + j_step);
    {
      f32x4 s[RB][2];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) s[rb][0] = s[rb][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        if (wave + 4 * b >= blocks) break;
        const A* kp = Ck + l15 * cs + (wave + 4 * b) * KB + g * kPer;
        const u32x4 k0 = *reinterpret_cast<const u32x4*>(kp), k1 = *reinterpret_cast<const u32x4*>(kp + 16 * cs);
        if constexpr (F32) {
          const f32x4 f0 = __builtin_bit_cast(f32x4, k0), f1 = __builtin_bit_cast(f32x4, k1);
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
              const f32x4 qv = __builtin_bit_cast(f32x4, q[rb][b]);
              s[rb][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(f0[e], qv[e], s[rb][0], 0, 0, 0);
              s[rb][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(f1[e], qv[e], s[rb][1], 0, 0, 0);
            }
        } else {
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) {
            const bf16x8_t qv = __builtin_bit_cast(bf16x8_t, q[rb][b]);
            s[rb][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, k0), qv, s[rb][0], 0, 0, 0);
            s[rb][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, k1), qv, s[rb][1], 0, 0, 0);
          }
        }
      }
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
          *reinterpret_cast<f32x4*>(S + (wave * kRows + rb * 16 + l15) * kSStride + 16 * kb + 4 * g) = s[rb][kb];
    }
    __syncthreads();
    if (my_row < kRows) {                                  // whole waves
      f32x4 v = *reinterpret_cast<const f32x4*>(S + my_row * kSStride + my_key);
#pragma unroll
      for (int w = 1; w < 4; ++w) v += *reinterpret_cast<const f32x4*>(S + (w * kRows + my_row) * kSStride + my_key);
      if constexpr (F32) {
        bool spoilt = false;
#pragma unroll
        for (int e = 0; e < 4; ++e) spoilt |= !(fabsf(v[e]) <= __FLT_MAX__);
        if (const bool any = __any(spoilt); lane == 0) s_spoilt[wave] = any;
      }
      float mx = -INFINITY;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = j0 + my_key + e;
        v[e] = j <= pq && j < j_hi ? v[e] * scale : -INFINITY;
        mx = fmaxf(mx, v[e]);
      }
#pragma unroll
      for (int x = 1; x < 8; x <<= 1) mx = fmaxf(mx, __shfl_xor(mx, x, kWave));
      const float m_new = fmaxf(m, mx), m_use = m_new == -INFINITY ? 0.f : m_new;
      const float corr = F32 ? expf(m - m_use) : __expf(m - m_use);
      float sum = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = F32 ? expf(v[e] - m_use) : bf16_round_f(__expf(v[e] - m_use));   // the sum uses the weights as the matrix core sees them
        sum += v[e];
      }
#pragma unroll
      for (int x = 1; x < 8; x <<= 1) sum += __shfl_xor(sum, x, kWave);
      l = l * corr + sum;
      m = m_new;
      if constexpr (F32) *reinterpret_cast<f32x4*>(P + my_row * kSStride + my_key) = v;
      else *reinterpret_cast<u32x2*>(P + my_row * kSStride + my_key) = u32x2{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
      if ((tid & 7) == 0) s_row[my_row] = corr;
    }
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const float corr = s_row[rb * 16 + l15];
      if (__any(corr != 1.0f)) {
#pragma unroll
        for (int d = 0; d < ND; ++d) o[rb][d] *= corr;
      }
    }
    if constexpr (F32) {
      bool spoilt = false;
#pragma unroll
      for (int w = 0; w < 2 * RB; ++w) spoilt |= s_spoilt[w] != 0;
      if (spoilt) {                                        // uniform: each row takes the keys that it sees, one by one
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          const int row = rb * 16 + l15, seen = row < cnt ? min(positions[(row0 + row) / H] + 1, j_hi) - j0 : 0;
          for (int k = 0; k < min(seen, kTileKeys); ++k) {
            const float w = P[row * kSStride + k];
#pragma unroll
            for (int d = 0; d < ND; ++d) {
              const int dd = (wave + 4 * d) * 16;
              if (dd >= r) break;
              const f32x4 c = *reinterpret_cast<const f32x4*>(Ck + k * cs + dd + 4 * g);
#pragma unroll
              for (int e = 0; e < 4; ++e) o[rb][d][e] = fmaf(w, c[e], o[rb][d][e]);
            }
          }
        }
      } else {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          f32x4 p[RB];
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) p[rb] = *reinterpret_cast<const f32x4*>(P + (rb * 16 + l15) * kSStride + 16 * kb + 4 * g);
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int d = 0; d < ND; ++d) {
              const int dd = (wave + 4 * d) * 16;
              if (dd >= r) break;
              const float c = Ck[(16 * kb + 4 * g + e) * cs + dd + l15];
#pragma unroll
              for (int rb = 0; rb < RB; ++rb) o[rb][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(c, p[rb][e], o[rb][d], 0, 0, 0);
            }
        }
      }
    } else {
      bf16x8_t p[RB];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const A* pp = P + (rb * 16 + l15) * kSStride + 4 * g;
        const u32x2 a = *reinterpret_cast<const u32x2*>(pp), b = *reinterpret_cast<const u32x2*>(pp + 16);
        p[rb] = __builtin_bit_cast(bf16x8_t, u32x4{a.x, a.y, b.x, b.y});
      }
      const __attribute__((address_space(3))) uint16_t* ck3 =
          (const __attribute__((address_space(3))) uint16_t*)(Ck) + (4 * g + (l15 >> 2)) * cs + 4 * (l15 & 3);
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        const int dd = (wave + 4 * d) * 16;
        if (dd >= r) break;
        const v4s_t a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s_t __attribute__((address_space(3)))*)(ck3 + dd));
        const v4s_t a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s_t __attribute__((address_space(3)))*)(ck3 + dd + 16 * cs));
        const u32x2 w0 = __builtin_bit_cast(u32x2, a0), w1 = __builtin_bit_cast(u32x2, a1);
        const bf16x8_t cv = __builtin_bit_cast(bf16x8_t, u32x4{w0.x, w0.y, w1.x, w1.y});
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) o[rb][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cv, p[rb], o[rb][d], 0, 0, 0);
      }
    }
  }
  const int64_t slots = (int64_t)n_tokens * H * max_splits;
  __syncthreads();                                         // the last tile's rescales are read
  if (sm_live && (tid & 7) == 0) s_row[my_row] = 1.0f / l;
  __syncthreads();
  if (sm_live && (tid & 7) == 0 && cut.splits_of(pq + 1, max_splits) > max(1, split)) {
    const LatentPartial part(partial, slots, r, (int64_t)(row0 + my_row) * max_splits + split);
    part.max_sum[0] = m;
    part.max_sum[1] = l;
  }
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int row = rb * 16 + l15;
    if (row >= cnt) continue;
    const int own_splits = cut.splits_of(positions[(row0 + row) / H] + 1, max_splits);
    if (split >= own_splits) continue;
    const bool whole = own_splits == 1;
    const float inv = whole ? s_row[row] : 1.0f;
    float* dst = whole ? o_lat + (int64_t)(row0 + row) * r
                       : LatentPartial(partial, slots, r, (int64_t)(row0 + row) * max_splits + split).acc;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      const int dd = (wave + 4 * d) * 16 + 4 * g;
      if (dd < r) *reinterpret_cast<f32x4*>(dst + dd) = o[rb][d] * inv;
    }
  }
}

// One call's tiled form.  An fp32 cache always takes the few-rows form.  A bf16 cache takes it when the tiles hold no more than 16 rows
// on average, measured against the 64-row form (512 + 64, splits of 32, with the merge): 4 requests of 16 heads 15.9 / 17.1 us,
// 32 of them 35.0 / 53.6; at 32 rows per tile there is nothing between them (20.0 / 20.3, 37.8 / 37.5), at 64 the other is faster
// (35.7 / 30.0, a prompt of 1800 tokens 303 / 257).
struct LatentCall {
  const float* qc; float* o_lat;
  const void* cache; int64_t page_stride, layer_off; int page_size;
  const int32_t *positions, *token_req, *page_indptr, *page_ids, *tile_row0, *tile_rows;
  int n_tiles, H, r, dr; float scale; float* ws; int n_tokens, sp; LatentCut cut; hipStream_t s;

  // every instance may take what a compute unit has, asked for once
  template <typename K>
  static bool all_lds(K kern, size_t bytes = 159 * 1024) {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess;
  }
  template <typename A, typename K>
  void run(K kern, int subs, size_t lds, int threads = 256) const {
    kern<<<dim3(n_tiles, sp, subs), threads, lds, s>>>(qc, o_lat, static_cast<const A*>(cache), page_stride, layer_off, page_size, positions, token_req,
                                           page_indptr, page_ids, tile_row0, tile_rows, H, r, dr, scale, ws, n_tokens, sp, cut);
  }
  template <int ND, int EB>
  void tile_form() const {
    auto kern = &latent_attn_tile_kernel<ND, EB>;
    static_assert(LatentTileShape<ND, EB>::kLds <= kCuLds, "a compute unit's LDS");
    static const bool once = all_lds(kern, LatentTileShape<ND, EB>::kLds);
    (void)once;
    run<uint16_t>(kern, 1, LatentTileShape<ND, EB>::kLds, 512);
  }
  template <int ND>
  void wide() const {
    // The form that shares LDS reads, both sides measured at the kernel: ranks of 256 and 512 (its waves' eighths are two and four blocks of 16 dims), rotated
    // parts of one and two blocks of 32 values, eight neighbouring keys on one page.  Its queries and values lie in registers, so every size is a kernel of its own;
    // only these four are built and measured, any other size keeps the form below.
    if constexpr (ND >= 16) {
      if (r == ND * 16 && !(cut.dealt && sp > 1) && page_size % 8 == 0 && cut.grain % 8 == 0) {
        if (dr == 32) return tile_form<ND, ND / 2 + 1>();
        if (dr == 64) return tile_form<ND, ND / 2 + 2>();
      }
    }
    // A second set of waves, on the other half of tiles of 64 keys, where one workgroup's rows and keys fill a compute unit's LDS anyhow and both halves'
    // keys fit (entries of 417 to 608 values): each SIMD has two chains to work on.  16 heads of 512 + 64, four prompts of up to 900 tokens 214 -> 156 us
    // (longest tiles first: 179).  Keys dealt in runs of 32 stay with one set.
    const size_t one = tile_lds(1);
    if (2 * one > kCuLds && tile_lds(2) <= 159 * 1024 && !(cut.dealt && sp > 1)) {
      if (r == ND * 16) wide_form<ND, true, 2>();
      else wide_form<ND, false, 2>();
    } else if (r == ND * 16) wide_form<ND, true, 1>();
    else wide_form<ND, false, 1>();
  }
  static constexpr size_t kCuLds = 160 * 1024;
  size_t tile_lds(int kh) const { return (size_t)(kTileRows + kh * kTileKeys) * (((r + dr + 31) & ~31) + 8) * 2; }
  template <int ND, bool FULL, int KH>
  void wide_form() const {
    auto kern = &latent_attn_mfma_kernel<ND, FULL, KH>;
    static const bool once = all_lds(kern);
    (void)once;
    run<uint16_t>(kern, 1, std::max(tile_lds(KH), KH == 2 ? (size_t)4 * 64 * (ND * 16 + 8) : 0), 256 * KH);
  }
  template <typename A, int ND, int RB>
  void few_rows() const {
    auto kern = &latent_attn_few_kernel<A, ND, RB>;
    static const bool once = all_lds(kern);
    (void)once;
    constexpr int kRows = 16 * RB, KB = std::is_same<A, float>::value ? 16 : 32;
    const size_t cs = (r + dr + KB - 1) / KB * KB + 16 / sizeof(A);
    // the parts of a tile past its rows come last: between the others they would take those from some of the XCDs' turns
    run<A>(kern, kTileRows / kRows,
           (kTileKeys * cs + kRows * (kTileKeys + 4)) * sizeof(A) + (4 * kRows * (kTileKeys + 4) + kRows) * sizeof(float));
  }
  bool narrow() const { return (int64_t)n_tokens * H <= 16 * (int64_t)n_tiles; }
  template <typename A>
  void few() const {
    const bool small = r <= 256 && r + dr <= 384;
    if constexpr (std::is_same<A, float>::value) {
      if (!narrow()) return small ? few_rows<A, 4, 2>() : few_rows<A, 8, 2>();
    }
    small ? few_rows<A, 4, 1>() : few_rows<A, 8, 1>();
  }
};

static inline int latent_split_keys(int split_keys) { return split_keys > 0 ? split_keys : kLatSplitKeys; }
static inline int latent_max_splits(int max_kv_len, int split_keys) {
  const int sk = latent_split_keys(split_keys);
  return std::max(1, (max_kv_len + sk - 1) / sk);
}

static bool latent_prep_ok(const pegainfer_latent_prep_desc* d) {
  return !(d->rot_dims < 0 || d->rot_dims > d->rot || (d->rot_dims & 1) || d->rank <= 0 || d->page_size <= 0 || d->heads < 0 || d->nope < 0 ||
           (d->rot_dims > 0 && !d->inv_freq) || (d->rot_layout != PEGAINFER_ROT_PAIRS && d->rot_layout != PEGAINFER_ROT_HALVES) ||
           (!d->dkv && !d->q && !d->ql) || (d->dkv && (!d->c_norm_w || !d->cache)) || (d->q && !d->qc) ||
           (d->ql && (!d->ql_norm_w || !d->ql_out || d->q_rank <= 0)));
}
template <typename A>
static LatentPrep<A> latent_prep_parts(const pegainfer_latent_prep_desc* d) {
  return {static_cast<const A*>(d->dkv), d->dkv_stride, static_cast<const A*>(d->c_norm_w),
          static_cast<const A*>(d->ql), d->ql_stride, static_cast<const A*>(d->ql_norm_w), static_cast<A*>(d->ql_out), d->q_rank,
          static_cast<const A*>(d->q), d->q_stride, d->qc};
}
static LatentPlace latent_prep_place(const pegainfer_latent_prep_desc* d) {
  return {d->eps, d->inv_freq, d->rot_dims, d->rot_layout == PEGAINFER_ROT_PAIRS, d->positions, d->token_req, d->page_indptr, d->page_ids,
          d->page_stride, d->layer_off, d->page_size, d->heads, d->nope, d->rot, d->rank};
}
// few rows (decoding): a row's rotated parts spread over several workgroups; many rows fill the chip alone
static int latent_prep_per_row(const pegainfer_latent_prep_desc* d) {
  const int vals = (d->q ? d->heads + 1 : 1) * d->rot;
  return d->n_tokens >= 256 ? 1 : std::max(d->ql && d->dkv ? 2 : 1, std::min(8, (vals + 255) / 256));
}

}  // namespace pk

extern "C" {
using namespace pk;

pegainfer_status_t pegainfer_latent_prep(const void* proj, int64_t proj_row_stride, int64_t dkv_offset,
                                         const void* c_norm_w, float eps, const float* inv_freq, int32_t rot_dims,
                                         const int32_t* positions, const int32_t* token_req, const int32_t* page_indptr,
                                         const int32_t* page_ids, void* cache, int64_t page_stride, int64_t layer_off,
                                         int32_t page_size, float* qc, int32_t heads, int32_t nope, int32_t rot,
                                         int32_t rank, int32_t n_tokens, int32_t dtype, pegainfer_stream_t stream) {
  pegainfer_latent_prep_desc d{};
  const int64_t es = dtype == kDtF32 ? 4 : 2;
  d.dkv = static_cast<const uint8_t*>(proj) + dkv_offset * es; d.dkv_stride = proj_row_stride; d.c_norm_w = c_norm_w;
  d.q = proj; d.q_stride = proj_row_stride; d.qc = qc;
  d.eps = eps; d.inv_freq = inv_freq; d.rot_dims = rot_dims; d.rot_layout = PEGAINFER_ROT_HALVES;
  d.positions = positions; d.token_req = token_req; d.page_indptr = page_indptr; d.page_ids = page_ids;
  d.cache = cache; d.page_stride = page_stride; d.layer_off = layer_off; d.page_size = page_size;
  d.heads = heads; d.nope = nope; d.rot = rot; d.rank = rank; d.n_tokens = n_tokens; d.dtype = dtype;
  return pegainfer_latent_prep_form(&d, stream);
}

pegainfer_status_t pegainfer_latent_prep_form(const pegainfer_latent_prep_desc* d, pegainfer_stream_t stream) {
  if (!d) return (pegainfer_status_t)hipErrorInvalidValue;
  if (d->n_tokens <= 0) return 0;
  if (!latent_prep_ok(d)) return (pegainfer_status_t)hipErrorInvalidValue;
  if (!by_dtype(d->dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        latent_prep_kernel<A><<<dim3(d->n_tokens, latent_prep_per_row(d)), 256, 0, as_stream(stream)>>>(latent_prep_parts<A>(d), latent_prep_place(d),
                                                                                                       static_cast<A*>(d->cache));
      }))
    return (pegainfer_status_t)hipErrorInvalidValue;
  return (pegainfer_status_t)hipGetLastError();
}

int32_t pegainfer_latent_prep_absorb_ok(const pegainfer_latent_prep_desc* d, const pegainfer_gemm_desc* g) {
  if (!d || !g || d->n_tokens <= 0 || !latent_prep_ok(d) || g->plain || g->tile_group || g->x_row_index || g->y_row_index || g->m <= 0 || g->k <= 0 ||
      g->groups <= 0 || g->groups > 65535 || g->epilogue != PEGAINFER_EPI_NONE || g->rows != d->n_tokens || g->x_dtype != d->dtype || g->w_dtype != d->dtype ||
      g->y_dtype != kDtF32 || !chunks_ok(*g))
    return 0;
  // the forms that these rows take by themselves, so the same bits; of fp32 up to four outputs per wave of the chip (beyond, the product fills it by
  // itself)
  if (d->dtype == kDtBf16) return g->rows <= kRowsMax;
  return d->dtype == kDtF32 && g->rows <= 4 && rows_direct_all(*g, g->rows == 3 ? 4 : g->rows) < 16L * device_cus();
}

pegainfer_status_t pegainfer_latent_prep_absorb(const pegainfer_latent_prep_desc* d, const pegainfer_gemm_desc* g, pegainfer_stream_t stream) {
  if (!pegainfer_latent_prep_absorb_ok(d, g)) return (pegainfer_status_t)hipErrorInvalidValue;
  hipStream_t st = as_stream(stream);
  const int ny = latent_prep_per_row(d), n_prep = d->n_tokens * ny;
  const LatentPlace place = latent_prep_place(d);
  if (d->dtype == kDtBf16) {
    const RowsMfmaShape f = rows_mfma_shape(*g);
    const int gx = (int)f.grid.x, gy = (int)f.grid.y, n_gemm = gx * gy * (int)f.grid.z;
    auto go = [&](auto kern) {
      kern<<<n_gemm + n_prep, 256, 0, st>>>(latent_prep_parts<uint16_t>(d), place, static_cast<uint16_t*>(d->cache), ny, *g, f.wk, gx, gy, n_gemm);
    };
    if (f.ob == 2) go(latent_prep_absorb_kernel<2>);
    else go(latent_prep_absorb_kernel<1>);
  } else {
    const int R = g->rows == 3 ? 4 : g->rows, mb = std::min(2, rows_direct_outputs(*g, R, false));
    const int gy = ceil_div(g->m, 4 * mb), n_gemm = gy * g->groups;
    auto go = [&](auto kern) { kern<<<n_gemm + n_prep, 256, 0, st>>>(latent_prep_parts<float>(d), place, static_cast<float*>(d->cache), ny, *g, gy, n_gemm); };
    auto by_outputs = [&](auto r) {
      constexpr int RR = decltype(r)::value;
      if (mb == 2) go(latent_prep_absorb_f32_kernel<RR, 2>);
      else go(latent_prep_absorb_f32_kernel<RR, 1>);
    };
    if (R == 1) by_outputs(std::integral_constant<int, 1>());
    else if (R == 2) by_outputs(std::integral_constant<int, 2>());
    else by_outputs(std::integral_constant<int, 4>());
  }
  return (pegainfer_status_t)hipGetLastError();
}

int64_t pegainfer_latent_attention_workspace(int32_t n_tokens, int32_t heads, int32_t rank, int32_t max_kv_len,
                                             int32_t split_keys) {
  const int sp = latent_max_splits(max_kv_len, split_keys);
  return sp <= 1 ? 0 : (int64_t)n_tokens * heads * sp * (rank + 2);
}

int32_t pegainfer_latent_attention_tiled_ok(int32_t rank, int32_t rot, int64_t page_stride, int64_t layer_off, int32_t dtype) {
  // the entry's limit is the key tile's: 640 values (20 chunks of 16 bytes per thread in fp32, kLatPrefetch in bf16)
  const int chunk = dtype == kDtF32 ? 4 : 8;
  return (dtype == kDtBf16 || dtype == kDtF32) && rank % 16 == 0 && rank <= 512 && rot % chunk == 0 && rank + rot <= 640 &&
         page_stride % chunk == 0 && layer_off % chunk == 0;
}

// one launch (and its merge) with the keys cut as `cut` says into `sp` splits at most
static pegainfer_status_t latent_attention_launch(const float* qc, float* o_lat, const void* cache, int64_t page_stride,
                                                  int64_t layer_off, int32_t page_size, const int32_t* positions,
                                                  const int32_t* token_req, const int32_t* page_indptr, const int32_t* page_ids,
                                                  int32_t heads, int32_t rank, int32_t rot, float scale, int32_t n_tokens, int sp,
                                                  pk::LatentCut cut, float* workspace, const int32_t* tile_row0,
                                                  const int32_t* tile_rows, int32_t n_tiles, int32_t dtype, pegainfer_stream_t stream) {
  if (sp > 1 && !workspace) return (pegainfer_status_t)hipErrorInvalidValue;
  hipStream_t s = as_stream(stream);
  if (tile_row0) {
    if (!tile_rows || n_tiles <= 0 || !pegainfer_latent_attention_tiled_ok(rank, rot, page_stride, layer_off, dtype) ||
        (reinterpret_cast<uintptr_t>(cache) & 15u))
      return (pegainfer_status_t)hipErrorInvalidValue;
    const LatentCall c{qc, o_lat, cache, page_stride, layer_off, page_size, positions, token_req, page_indptr, page_ids, tile_row0, tile_rows,
                       n_tiles, heads, rank, rot, scale, workspace, n_tokens, sp, cut, s};
    if (dtype == kDtF32) c.few<float>();
    else if (c.narrow()) c.few<uint16_t>();
    else if (rank <= 64) c.wide<4>();
    else if (rank <= 128) c.wide<8>();
    else if (rank <= 256) c.wide<16>();
    else c.wide<32>();
  } else {
    if (rank > kLatAcc * 256) return (pegainfer_status_t)hipErrorInvalidValue;
    const size_t smem = (size_t)(rank + rot + kLatKeys) * sizeof(float);
    if (smem > 60000) return (pegainfer_status_t)hipErrorInvalidValue;
    dim3 grid(n_tokens, heads, sp);
    if (!by_dtype(dtype, [&](auto* t) {
          using A = std::remove_pointer_t<decltype(t)>;
          latent_attn_kernel<A><<<grid, 256, smem, s>>>(qc, o_lat, static_cast<const A*>(cache), page_stride, layer_off, page_size,
                                                        positions, token_req, page_indptr, page_ids, heads, rank, rot, scale,
                                                        workspace, sp, cut);
        }))
      return (pegainfer_status_t)hipErrorInvalidValue;
  }
  if (sp > 1) latent_attn_merge_kernel<<<dim3(n_tokens, heads, (rank + 255) / 256), 256, (3 * 256 + (size_t)sp) * sizeof(float), s>>>(o_lat, workspace, positions, heads, rank, sp, cut);
  return (pegainfer_status_t)hipGetLastError();
}

pegainfer_status_t pegainfer_latent_attention(const float* qc, float* o_lat, const void* cache, int64_t page_stride,
                                              int64_t layer_off, int32_t page_size, const int32_t* positions,
                                              const int32_t* token_req, const int32_t* page_indptr,
                                              const int32_t* page_ids, int32_t heads, int32_t rank, int32_t rot,
                                              float scale, int32_t n_tokens, int32_t max_kv_len, int32_t split_keys,
                                              float* workspace, const int32_t* tile_row0, const int32_t* tile_rows,
                                              int32_t n_tiles, int32_t dtype, pegainfer_stream_t stream) {
  if (n_tokens <= 0 || heads <= 0) return 0;
  const int sk = latent_split_keys(split_keys), sp = latent_max_splits(max_kv_len, split_keys);
  return latent_attention_launch(qc, o_lat, cache, page_stride, layer_off, page_size, positions, token_req, page_indptr, page_ids, heads,
                                 rank, rot, scale, n_tokens, sp, LatentCut{sk, 0}, workspace, tile_row0, tile_rows, n_tiles, dtype, stream);
}

int64_t pegainfer_latent_attention_dealt_workspace(int32_t n_tokens, int32_t heads, int32_t rank, int32_t n_split) {
  return n_split <= 1 ? 0 : (int64_t)n_tokens * heads * n_split * (rank + 2);
}

pegainfer_status_t pegainfer_latent_attention_dealt(const float* qc, float* o_lat, const void* cache, int64_t page_stride,
                                                    int64_t layer_off, int32_t page_size, const int32_t* positions,
                                                    const int32_t* token_req, const int32_t* page_indptr, const int32_t* page_ids,
                                                    int32_t heads, int32_t rank, int32_t rot, float scale, int32_t n_tokens,
                                                    int32_t n_split, float* workspace, const int32_t* tile_row0,
                                                    const int32_t* tile_rows, int32_t n_tiles, int32_t dtype,
                                                    pegainfer_stream_t stream) {
  if (n_tokens <= 0 || heads <= 0) return 0;
  if (n_split < 1 || n_split > 1024) return (pegainfer_status_t)hipErrorInvalidValue;
  return latent_attention_launch(qc, o_lat, cache, page_stride, layer_off, page_size, positions, token_req, page_indptr, page_ids, heads,
                                 rank, rot, scale, n_tokens, n_split, LatentCut{tile_row0 ? kTileKeys : kLatKeys, 1}, workspace, tile_row0,
                                 tile_rows, n_tiles, dtype, stream);
}

}  // extern "C"
