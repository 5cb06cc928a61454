// Strided / batched / grouped GEMM for the shapes the weight-streaming and 128/256-tile kernels of linear.hip do not take:
// per-head products over slices of a wider row (latent-attention absorb and value up-projection), expert-grouped rows
// gathered through an index (routed feed-forward), and every product of a model served in true fp32.
//
//   y[row, g, m] = sum_k x[row, g, k] * w[g, m, k]
//
// gemm_strided_kernel: any sizes and strides, and every product of a run that asks for plain kernels.  The forms below take operands
// in 16-byte chunks.
// 64 x 64 output tile per 256-thread workgroup, K in slices of 16 staged through LDS as fp32, each thread a 4 x 4 block
// of fp32 accumulators, k strictly ascending: an output's value depends on its own row and weights only (never on the
// tile it lands in, the batch or the group sizes).  Operand storage (bf16 or fp32) is a template parameter, so the bf16
// instance multiplies exact fp32 images of bf16 values and the fp32 instance is plain fp32 FMA - no reduced-precision
// matrix mode.
#include <type_traits>

#include "gemm_rows.h"

namespace pk {

constexpr int GT = 64, GM = 64, GK = 16;

template <typename TX, typename TW, typename TY, typename TG>
__global__ __launch_bounds__(256) void gemm_strided_kernel(pegainfer_gemm_desc d) {
  __shared__ float xs[GK][GT + 4];
  __shared__ float ws[GK][GM + 4];
  __shared__ int xrow[GT], yrow[GT];
  int g, row0, nrows;
  if (d.tile_group) {
    if ((int)blockIdx.x >= *d.n_tiles) return;
    g = d.tile_group[blockIdx.x];
    row0 = d.tile_row0[blockIdx.x];
    nrows = d.tile_rows[blockIdx.x];
  } else {
    g = blockIdx.z;
    row0 = blockIdx.x * GT;
    nrows = min(GT, d.rows - row0);
  }
  const int m0 = blockIdx.y * GM;
  const int tid = threadIdx.x;
  if (tid < GT) {
    const int p = row0 + tid;
    xrow[tid] = tid < nrows ? (d.x_row_index ? d.x_row_index[p] : p) : -1;
    yrow[tid] = tid < nrows ? (d.y_row_index ? d.y_row_index[p] : p) : -1;
  }
  __syncthreads();
  const TX* X = static_cast<const TX*>(d.x) + (int64_t)g * d.x_group_stride;
  const TW* W = static_cast<const TW*>(d.w) + (int64_t)g * d.w_group_stride;
  const int tr = (tid >> 4) * 4, tm = (tid & 15) * 4;   // this thread's 4 rows x 4 outputs
  float acc[4][4] = {};
  const bool w_k_fast = d.w_k_stride == 1;
  for (int k0 = 0; k0 < d.k; k0 += GK) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + i * 256;
      {
        const int r = idx >> 4, kk = idx & 15;
        const int src = xrow[r];
        xs[kk][r] = (src >= 0 && k0 + kk < d.k) ? ld(X + (int64_t)src * d.x_row_stride + k0 + kk) : 0.f;
      }
      {
        const int mm = w_k_fast ? idx >> 4 : idx & 63, kk = w_k_fast ? idx & 15 : idx >> 6;
        ws[kk][mm] = (m0 + mm < d.m && k0 + kk < d.k)
                         ? ld(W + (int64_t)(m0 + mm) * d.w_m_stride + (int64_t)(k0 + kk) * d.w_k_stride) : 0.f;
      }
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GK; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) { a[i] = xs[kk][tr + i]; b[i] = ws[kk][tm + i]; }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
  TY* Y = static_cast<TY*>(d.y) + (int64_t)g * d.y_group_stride;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int dst = yrow[tr + i];
    if (dst < 0) continue;
    float scale = 1.f;
    if (d.epilogue == PEGAINFER_EPI_SIGMOID_GATE)
      scale = sigmoid_f(ld(static_cast<const TG*>(d.gate) + (int64_t)xrow[tr + i] * d.gate_row_stride + g));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (m0 + tm + j >= d.m) continue;
      float v = acc[i][j];
      if (d.epilogue == PEGAINFER_EPI_RELU_SQ) { v = fmaxf(v, 0.f); v *= v; }
      else if (d.epilogue == PEGAINFER_EPI_GELU_ERF) v = gelu_erf_f(v);
      else if (d.epilogue == PEGAINFER_EPI_SIGMOID_GATE) v *= scale;
      st(Y + (int64_t)dst * d.y_row_stride + m0 + tm + j, v);
    }
  }
}


// ------------------------------------------------------------------ matrix-core form (bf16 weights, k contiguous)
// The same addressing (groups, gathered rows, tile table), output tiles of TR rows (64 or 128) x 128 outputs, four waves in a 2 x 2
// arrangement of v_mfma_f32_16x16x32_bf16 blocks, K in slices of MK (64 or 32).  Both operands travel by LDS-DMA into two slots, one slice ahead: a
// lane's source address carries the gather and the swizzle (swizzled()), so fragment reads meet no bank twice.  A wave's loads of a slice are
// waited for by count, the next slice's stay in flight under the products.
// fp32 x (the attention output in front of the value up-projection) is rounded to bf16 as it is read into fragments.  Rows and outputs past the
// tile's end load a valid row and are dropped at the store; the last slice's values past K are made zero in both operands.
// Needs 16-byte chunks: K % 8 == 0, strides % 8 == 0, aligned bases.
// Bound by what a compute unit takes in: 32 KB per slice and workgroup against 128 MFMAs, two workgroups per compute unit in turn.
// Work items go to the XCDs in eight contiguous runs (an XCD's L2 is where workgroups share an operand): with a tile table the outputs of a
// tile run fastest, so the neighbouring tiles of one expert read its weights together; without one the larger operand is read once.
// Before (slices staged through registers, fp32 chunks converted as they were fetched, so every load was waited for at once):
// 9600 pairs of 32 experts of 2048 x 2048 204 -> 134 us (600 TFLOP/s), of 2048 x 1024 into fp32 131 -> 75; 1024 fp32 rows x 2048 x 4096
// 127 -> 50; 2400 rows, 16 groups of 512 x 128 48 -> 21, fp32 rows of 128 x 512 34 -> 21.
constexpr int MM = 128;

// position of 16-byte chunk c of a row in LDS, CH chunks to a row: the rows a fragment read meets lie on different banks
template <int CH>
__device__ __forceinline__ int swizzled(int c, int row) { return c ^ (CH == 4 ? (row >> 1) & 3 : row & (CH - 1)); }

template <typename TX, int TR, int MK>
struct StridedMfmaShape {
  static constexpr int kXE = 16 / (int)sizeof(TX);                         // values of a chunk of x
  static constexpr int kXCh = MK / kXE, kWCh = MK / 8;                     // chunks of a row's slice
  static constexpr int kX = TR * kXCh * 16, kW = MM * kWCh * 16, kSlot = kX + kW;   // bytes of a slot
  static constexpr int kXLoads = kX / 4096, kWLoads = kW / 4096;           // DMA instructions per wave and slice
};

template <typename TX, typename TY, typename TG, int TR, int MK>
__global__ __launch_bounds__(256) void gemm_strided_mfma_kernel(pegainfer_gemm_desc d, int row_tiles, int rows_first) {
  typedef StridedMfmaShape<TX, TR, MK> Sh;
  extern __shared__ __attribute__((aligned(1024))) uint8_t mfma_lds[];
  __shared__ int xrow[TR], yrow[TR];
  const int mt = (d.m + MM - 1) / MM;
  int rt, m0, g;
  {
    const int tiles = d.tile_group ? *d.n_tiles : row_tiles, n = tiles * mt * (d.tile_group ? 1 : d.groups);
    const int xcd = blockIdx.x & 7, pos = blockIdx.x >> 3, q = n >> 3, rest = n & 7;
    if (pos >= q + (xcd < rest ? 1 : 0)) return;
    const int item = xcd * q + min(xcd, rest) + pos;
    g = item / (tiles * mt);
    const int i = item - g * (tiles * mt);
    rt = rows_first ? i % tiles : i / mt;
    m0 = (rows_first ? i / tiles : i % mt) * MM;
  }
  int row0 = rt * TR, nrows;
  if (d.tile_group) {
    g = d.tile_group[rt];
    row0 = d.tile_row0[rt];
    nrows = min(TR, d.tile_rows[rt]);
  } else {
    nrows = min(TR, d.rows - row0);
  }
  if (nrows <= 0) return;                            // a table may hold empty tiles; absent rows repeat the last one below
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l15 = lane & 15, gq = lane >> 4;
  if (tid < TR) {
    const int p = row0 + min(tid, nrows - 1);
    xrow[tid] = d.x_row_index ? d.x_row_index[p] : p;
    yrow[tid] = tid < nrows ? (d.y_row_index ? d.y_row_index[p] : p) : -1;
  }
  __syncthreads();
  const TX* X = static_cast<const TX*>(d.x) + (int64_t)g * d.x_group_stride;
  const uint16_t* W = static_cast<const uint16_t*>(d.w) + (int64_t)g * d.w_group_stride;
  constexpr int RJ = TR / 32;                       // 16-row blocks per wave
  const int wr = (wave & 1) * (TR / 2), wm = (wave >> 1) * 64;
  f32x4 acc[4][RJ];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < RJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const TX* xsrc[Sh::kXLoads];
  const uint16_t* wsrc[Sh::kWLoads];
  int xk[Sh::kXLoads], wk[Sh::kWLoads];             // first value of this lane's chunk in a slice
#pragma unroll
  for (int i = 0; i < Sh::kXLoads; ++i) {
    const int unit = (wave * Sh::kXLoads + i) * 64 + lane, row = unit / Sh::kXCh;
    xk[i] = swizzled<Sh::kXCh>(unit % Sh::kXCh, row) * Sh::kXE;
    xsrc[i] = X + (int64_t)xrow[row] * d.x_row_stride;
  }
#pragma unroll
  for (int i = 0; i < Sh::kWLoads; ++i) {
    const int unit = (wave * Sh::kWLoads + i) * 64 + lane, row = unit / Sh::kWCh;
    wk[i] = swizzled<Sh::kWCh>(unit % Sh::kWCh, row) * 8;
    wsrc[i] = W + (int64_t)min(m0 + row, d.m - 1) * d.w_m_stride;
  }
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  const uint32_t ring = (uint32_t)(uintptr_t)(lds_ptr_t)mfma_lds;
  auto dma = [&](const void* src, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                 :: "v"(src), "s"(__builtin_amdgcn_readfirstlane(dst)) : "memory", "m0");
  };
  auto issue = [&](int k0, int slot) {              // chunks past K load the row's last one: zeros in the products
    const uint32_t base = ring + slot * Sh::kSlot;
#pragma unroll
    for (int i = 0; i < Sh::kXLoads; ++i)
      dma(xsrc[i] + min(k0 + xk[i], d.k - Sh::kXE), base + (wave * Sh::kXLoads + i) * 1024);
#pragma unroll
    for (int i = 0; i < Sh::kWLoads; ++i) dma(wsrc[i] + min(k0 + wk[i], d.k - 8), base + Sh::kX + (wave * Sh::kWLoads + i) * 1024);
  };
  auto multiply = [&](int k0, int slot, auto tail) {
    const uint8_t *xs = mfma_lds + slot * Sh::kSlot, *ws = xs + Sh::kX;
#pragma unroll
    for (int ks = 0; ks < MK / 32; ++ks) {
      const int c = ks * 4 + gq;                    // this lane's eight values of k
      const bool past = tail.value && k0 + c * 8 >= d.k;
      bf16x8_t a[4], b[RJ];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        u32x4 v = *reinterpret_cast<const u32x4*>(ws + ((wm + i * 16 + l15) * Sh::kWCh + swizzled<Sh::kWCh>(c, l15)) * 16);
        if (past) v = u32x4{0u, 0u, 0u, 0u};
        a[i] = __builtin_bit_cast(bf16x8_t, v);
      }
#pragma unroll
      for (int j = 0; j < RJ; ++j) {
        const uint8_t* row = xs + (wr + j * 16 + l15) * Sh::kXCh * 16;
        u32x4 v;
        if constexpr (sizeof(TX) == 2) v = *reinterpret_cast<const u32x4*>(row + swizzled<Sh::kXCh>(c, l15) * 16);
        else {
          const f32x4 lo = *reinterpret_cast<const f32x4*>(row + swizzled<Sh::kXCh>(2 * c, l15) * 16),
                      hi = *reinterpret_cast<const f32x4*>(row + swizzled<Sh::kXCh>(2 * c + 1, l15) * 16);
          v = u32x4{pack_bf2(lo.x, lo.y), pack_bf2(lo.z, lo.w), pack_bf2(hi.x, hi.y), pack_bf2(hi.z, hi.w)};
        }
        if (past) v = u32x4{0u, 0u, 0u, 0u};
        b[j] = __builtin_bit_cast(bf16x8_t, v);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < RJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  };
  issue(0, 0);
  int slot = 0;
  for (int k0 = 0; k0 < d.k; k0 += MK, slot ^= 1) {
    if (k0 + MK < d.k) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");       // the slice before is multiplied: its slot is free
      issue(k0 + MK, slot ^ 1);
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(Sh::kXLoads + Sh::kWLoads) : "memory");   // this wave's part of slice k0 has landed
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    asm volatile("s_barrier" ::: "memory");          // everyone's part
    if (k0 + MK <= d.k) multiply(k0, slot, std::false_type{});
    else multiply(k0, slot, std::true_type{});
  }
  TY* Y = static_cast<TY*>(d.y) + (int64_t)g * d.y_group_stride;
  constexpr int kYBytes = 4 * (int)sizeof(TY);       // four neighbouring outputs of a row
  const bool vec = d.y_row_stride % 4 == 0 && d.y_group_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(d.y) & (kYBytes - 1)) == 0;
#pragma unroll
  for (int j = 0; j < RJ; ++j) {
    const int r = wr + j * 16 + l15;
    const int dst = yrow[r];
    if (dst < 0) continue;
    float scale = 1.f;
    if (d.epilogue == PEGAINFER_EPI_SIGMOID_GATE)
      scale = sigmoid_f(ld(static_cast<const TG*>(d.gate) + (int64_t)xrow[r] * d.gate_row_stride + g));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + wm + i * 16 + gq * 4;
      f32x4 v = acc[i][j];
      if (d.epilogue == PEGAINFER_EPI_RELU_SQ) {
#pragma unroll
        for (int e = 0; e < 4; ++e) { v[e] = fmaxf(v[e], 0.f); v[e] *= v[e]; }
      } else if (d.epilogue == PEGAINFER_EPI_GELU_ERF) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gelu_erf_f(v[e]);
      } else if (d.epilogue == PEGAINFER_EPI_SIGMOID_GATE) {
        v *= scale;
      }
      TY* out = Y + (int64_t)dst * d.y_row_stride + m;
      if (vec && m + 4 <= d.m) {
        if constexpr (sizeof(TY) == 4) *reinterpret_cast<f32x4*>(out) = v;
        else *reinterpret_cast<u32x2*>(out) = u32x2{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (m + e < d.m) st(out + e, v[e]);
      }
    }
  }
}

template <typename TX, typename TY, typename TG, int TR>
static void mfma_tiles_launch(const pegainfer_gemm_desc& d, hipStream_t s) {
  // fp32 rows of 128: slices of 32, so that more than one workgroup fits a compute unit's LDS (4096 x 4096 x 4096: 296 -> 279 us)
  constexpr int MK = sizeof(TX) == 4 && TR == 128 ? 32 : 64;
  auto kern = &gemm_strided_mfma_kernel<TX, TY, TG, TR, MK>;
  constexpr size_t lds = 2 * StridedMfmaShape<TX, TR, MK>::kSlot;
  static const bool once = (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), true);
  (void)once;
  const int tiles = d.tile_group ? d.max_tiles : ceil_div(d.rows, TR), mt = ceil_div(d.m, MM);
  const long items = (long)tiles * mt * (d.tile_group ? 1 : d.groups);
  const bool rows_first = !d.tile_group && (long)d.rows * sizeof(TX) < (long)d.m * 2;     // the weights are the larger operand: read once
  kern<<<dim3((unsigned)(8 * ceil_div(items, 8))), 256, lds, s>>>(d, tiles, rows_first ? 1 : 0);
}
template <typename TX, typename TY, typename TG>
static void mfma_form_launch(const pegainfer_gemm_desc& d, hipStream_t s) {
  // Tiles of 128 rows where they give two workgroups per compute unit, four for fp32 rows (128- / 64-row tiles): bf16 rows, 256 workgroups
  // (2048 x 2048 x 2048) 33 / 28 us, 320 (600 rows, 16 groups of 512 x 128) 10.9 / 9.4, 512 (4096 x 2048 x 2048) 45 / 53; fp32 rows, 304 (2400
  // x 2048 x 4096) 128 / 100 us, 1024 (4096 x 4096 x 4096) 279 / 302, (8192 rows, 16 groups of 128 x 512) 69 / 67.
  const long wide = (long)ceil_div(d.rows, 128) * ceil_div(d.m, MM) * d.groups;
  const bool big = d.tile_group ? d.tile_rows_cap >= 128 : wide >= (sizeof(TX) == 4 ? 4L : 2L) * device_cus();
  if (big) mfma_tiles_launch<TX, TY, TG, 128>(d, s);
  else mfma_tiles_launch<TX, TY, TG, 64>(d, s);
}

template <typename TW, typename TY, typename TG, int R, int MB, bool GLU>
__global__ __launch_bounds__(256) void gemm_rows_direct_kernel(pegainfer_gemm_desc d, int act, int64_t up) {
  gemm_rows_direct_block<TW, TY, TG, R, MB, GLU>(d, act, up, blockIdx.x, blockIdx.y, blockIdx.z);
}
template <typename TW, typename TY, typename TG, int R, bool GLU>
static void rows_direct_launch(const pegainfer_gemm_desc& d, int act, int64_t up, hipStream_t s) {
  const int row_tiles = d.tile_group ? d.max_tiles | 1 : ceil_div(d.rows, R), groups = d.tile_group ? 1 : d.groups;
  auto go = [&](auto mb) {
    constexpr int MB = decltype(mb)::value;
    gemm_rows_direct_kernel<TW, TY, TG, R, MB, GLU><<<dim3(row_tiles, ceil_div(d.m, 4 * MB), groups), 256, 0, s>>>(d, act, up);
  };
  const int mb = rows_direct_outputs(d, R, GLU);
  if constexpr (!GLU) {
    if (mb == 4) { go(std::integral_constant<int, 4>()); return; }
  }
  if (mb == 2) go(std::integral_constant<int, 2>());
  else go(std::integral_constant<int, 1>());
}

template <typename TX, typename TY, typename TG, int OB, bool EX = false>
__global__ __launch_bounds__(256) void gemm_rows_mfma_kernel(pegainfer_gemm_desc d, int wk, ExpertForm ex) {
  gemm_rows_mfma_block<TX, TY, TG, OB, EX>(d, wk, ex, blockIdx.x, blockIdx.y, blockIdx.z);
}
template <typename TX, typename TY, typename TG>
static void rows_mfma_launch(const pegainfer_gemm_desc& d, hipStream_t s) {
  const RowsMfmaShape f = rows_mfma_shape(d);
  if (f.ob == 2) gemm_rows_mfma_kernel<TX, TY, TG, 2><<<f.grid, 256, 0, s>>>(d, f.wk, ExpertForm{});
  else gemm_rows_mfma_kernel<TX, TY, TG, 1><<<f.grid, 256, 0, s>>>(d, f.wk, ExpertForm{});
}
template <typename TY>
static void expert_rows_launch(const pegainfer_gemm_desc& d, ExpertForm ex, int slices, hipStream_t s) {
  const int np = ceil_div(d.k, 64), wk = np >= 8 ? 4 : np >= 4 ? 2 : 1;
  const int columns = (d.max_tiles + slices) | 1;      // odd, as above; the shared slices last
  ex.slots = columns - slices;
  const int blocks = ceil_div(d.m, 16 * (4 / wk));
  if (ex.glu) gemm_rows_mfma_kernel<uint16_t, TY, uint16_t, 2, true><<<dim3(columns, blocks), 256, 0, s>>>(d, wk, ex);
  else if ((long)columns * blocks >= 4L * device_cus()) gemm_rows_mfma_kernel<uint16_t, TY, uint16_t, 2, true><<<dim3(columns, ceil_div(blocks, 2)), 256, 0, s>>>(d, wk, ex);
  else gemm_rows_mfma_kernel<uint16_t, TY, uint16_t, 1, true><<<dim3(columns, blocks), 256, 0, s>>>(d, wk, ex);
}

// ------------------------------------------------------------------ few-rows form on the matrix cores (fp32 weights, decode)
// At most 16 rows per tile, on v_mfma_f32_16x16x4_f32.  A wave takes OB blocks of 16 outputs, wk waves of the workgroup's eight share a
// block's K (wave j the 32-wide pieces j, j + wk, ...; wk follows from K alone), their sums meet in LDS in wave order: an output's k
// order is fixed by K.  Lane (l15, g) fetches the eight values from 8 g of a piece of output l15 and of row l15, whole lines of weights;
// product e of a piece takes value e of every lane, both operands numbered alike.  Four pieces of both operands are in flight per wave,
// nothing is staged and no barrier stands before the sums.
// Against FMA with eight rows in LDS: 32 768 x 1024 weights and 8 rows 54.9 -> 35.8 us, 1024 x 3072 19.2 -> 14.4; 16 rows (two passes over the
// weights there) 46.6 -> 16.3.
template <typename TY, typename TG, int OB>
__global__ __launch_bounds__(512) void gemm_rows_f32_kernel(pegainfer_gemm_desc d, int wk) {
  constexpr int NW = 8, CH = 2;                               // pieces per register set
  __shared__ f32x4 red[NW][OB][64];
  int g, row0, nrows;
  if (d.tile_group) {
    if ((int)blockIdx.x >= *d.n_tiles) return;
    g = d.tile_group[blockIdx.x];
    row0 = d.tile_row0[blockIdx.x];
    nrows = min(kRowsMax, d.tile_rows[blockIdx.x]);
  } else {
    g = blockIdx.z;
    row0 = blockIdx.x * kRowsMax;
    nrows = min(kRowsMax, d.rows - row0);
  }
  if (nrows <= 0) return;                                     // an empty tile of a table has no last row to repeat
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l15 = lane & 15, gq = lane >> 4;
  const int per_wg = NW / wk * OB * 16;                       // outputs of a workgroup
  const int blk = wave / wk, ks = wave - blk * wk;
  const int m0 = blockIdx.y * per_wg + blk * OB * 16;
  const int tok = row0 + min(l15, nrows - 1);                 // absent rows repeat the last one; they are never stored
  const float* xp = static_cast<const float*>(d.x) + (int64_t)g * d.x_group_stride +
                    (int64_t)(d.x_row_index ? d.x_row_index[tok] : tok) * d.x_row_stride;
  const float* wp[OB];
#pragma unroll
  for (int o = 0; o < OB; ++o)
    wp[o] = static_cast<const float*>(d.w) + (int64_t)g * d.w_group_stride + (int64_t)min(m0 + o * 16 + l15, d.m - 1) * d.w_m_stride;
  const int K = d.k, np = (K + 31) >> 5, mine = ks < np ? (np - ks + wk - 1) / wk : 0;   // pieces of k; those of this wave
  f32x4 acc[OB][2];
#pragma unroll
  for (int o = 0; o < OB; ++o) acc[o][0] = acc[o][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Set { f32x4 x[CH][2], w[CH][OB][2]; } A, B;
  auto issue = [&](int i0, Set& s) {                          // past the wave's pieces or K: a valid chunk, not multiplied
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int k = (ks + min(i0 + c, mine - 1) * wk) * 32 + gq * 8, kc = k < K ? k : 0;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        s.x[c][h] = *reinterpret_cast<const f32x4*>(xp + kc + 4 * h);
#pragma unroll
        for (int o = 0; o < OB; ++o) s.w[c][o][h] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(wp[o] + kc + 4 * h));
      }
    }
  };
  auto compute = [&](int i0, const Set& s) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (i0 + c >= mine) continue;
      const bool past = (ks + (i0 + c) * wk) * 32 + gq * 8 >= K;           // the last piece of a K that is no multiple of 32
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float xv = past ? 0.f : s.x[c][h][e];
#pragma unroll
          for (int o = 0; o < OB; ++o)
            acc[o][e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(past ? 0.f : s.w[c][o][h][e], xv, acc[o][e & 1], 0, 0, 0);
        }
    }
  };
  if (mine > 0) {
    issue(0, A);
    issue(CH, B);
    for (int i0 = 0; i0 < mine; i0 += 2 * CH) {
      compute(i0, A);
      if (i0 + 2 * CH < mine) issue(i0 + 2 * CH, A);
      if (i0 + CH >= mine) break;
      compute(i0 + CH, B);
      if (i0 + 3 * CH < mine) issue(i0 + 3 * CH, B);
    }
  }
#pragma unroll
  for (int o = 0; o < OB; ++o) red[wave][o][lane] = acc[o][0] + acc[o][1];   // outputs 4 (lane >> 4) .. of the block, row lane & 15
  __syncthreads();
  TY* Y = static_cast<TY*>(d.y) + (int64_t)g * d.y_group_stride;
  const float* part = reinterpret_cast<const float*>(red);
  for (int e = tid; e < per_wg * nrows; e += 512) {           // consecutive threads: consecutive outputs of one row
    const int out = e % per_wg, r = e / per_wg;
    const int m = blockIdx.y * per_wg + out;
    if (m >= d.m) continue;
    const int b = out / (OB * 16), o = (out >> 4) % OB, j = out & 15;
    const int at = (o * 64 + (j >> 2) * 16 + r) * 4 + (j & 3);
    float v = part[b * wk * OB * 256 + at];
    for (int w = 1; w < wk; ++w) v += part[(b * wk + w) * OB * 256 + at];
    const int p = row0 + r;
    if (d.epilogue == PEGAINFER_EPI_RELU_SQ) { v = fmaxf(v, 0.f); v *= v; }
    else if (d.epilogue == PEGAINFER_EPI_GELU_ERF) v = gelu_erf_f(v);
    else if (d.epilogue == PEGAINFER_EPI_SIGMOID_GATE)
      v *= sigmoid_f(ld(static_cast<const TG*>(d.gate) + (int64_t)(d.x_row_index ? d.x_row_index[p] : p) * d.gate_row_stride + g));
    st(Y + (int64_t)(d.y_row_index ? d.y_row_index[p] : p) * d.y_row_stride + m, v);
  }
}
template <typename TY, typename TG>
static void rows_f32_launch(const pegainfer_gemm_desc& d, hipStream_t s) {
  const int np = ceil_div(d.k, 32), wk = np >= 16 ? 8 : np >= 8 ? 4 : np >= 4 ? 2 : 1;
  const int row_tiles = d.tile_group ? d.max_tiles | 1 : ceil_div(d.rows, kRowsMax), groups = d.tile_group ? 1 : d.groups;   // | 1: as above
  const int blocks = ceil_div(d.m, 16 * (8 / wk));
  const bool two = (long)row_tiles * groups * blocks >= 4L * device_cus();
  if (two) gemm_rows_f32_kernel<TY, TG, 2><<<dim3(row_tiles, ceil_div(blocks, 2), groups), 512, 0, s>>>(d, wk);
  else gemm_rows_f32_kernel<TY, TG, 1><<<dim3(row_tiles, blocks, groups), 512, 0, s>>>(d, wk);
}

// ------------------------------------------------------------------ fp32 tiles on the fp32 matrix cores (fp32 operands, k contiguous)
// v_mfma_f32_16x16x4_f32 multiplies and adds in fp32 - the products of the FMA form, summed four k at a time - at the vector units' own peak,
// without their operand traffic: a lane's 16-byte LDS read feeds four instructions.  TR rows x 64 outputs per workgroup, wave w the
// outputs 16 w .. 16 w + 15 of all rows, K in slices of 64 through LDS with the next slice on its way in registers.  Lane (i, g) of a 16 x 16
// block holds k = 4 g + j of a 16-wide piece for instruction j, in both operands: an output's k order is fixed by K alone.
// Bound by the matrix cores where the tiles fill the chip; 32-row tiles where 64-row ones would give a compute unit fewer than two workgroups.
// The 26 projections of a prompt step of 466 rows (K 512 .. 3072, 832 .. 6144 outputs) took 4.9 ms on the FMA form - 64 x 64 tiles, 16 k per
// pair of barriers, nothing on its way - and take 0.92 ms: 25 us on 32-row tiles, 69 us (85 TFLOP/s) for 6144 outputs of 1024 k.
constexpr int FK = 64, FS = FK + 4, FM = 64;

template <typename TY, typename TG, int TR>
__global__ __launch_bounds__(256) void gemm_f32_mfma_kernel(pegainfer_gemm_desc d) {
  __shared__ __align__(16) float xs[TR * FS];
  __shared__ __align__(16) float ws[FM * FS];
  __shared__ int xrow[TR], yrow[TR];
  int g, row0, nrows;
  if (d.tile_group) {
    if ((int)blockIdx.x >= *d.n_tiles) return;
    g = d.tile_group[blockIdx.x];
    row0 = d.tile_row0[blockIdx.x];
    nrows = min(TR, d.tile_rows[blockIdx.x]);
  } else {
    g = blockIdx.z;
    row0 = blockIdx.x * TR;
    nrows = min(TR, d.rows - row0);
  }
  const int m0 = blockIdx.y * FM;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l15 = lane & 15, gq = lane >> 4;
  if (tid < TR) {
    const int p = row0 + tid;
    xrow[tid] = tid < nrows ? (d.x_row_index ? d.x_row_index[p] : p) : -1;
    yrow[tid] = tid < nrows ? (d.y_row_index ? d.y_row_index[p] : p) : -1;
  }
  __syncthreads();
  const float* X = static_cast<const float*>(d.x) + (int64_t)g * d.x_group_stride;
  const float* W = static_cast<const float*>(d.w) + (int64_t)g * d.w_group_stride;
  constexpr int RJ = TR / 16, XC = TR * (FK / 4) / 256, WC = FM * (FK / 4) / 256;   // row blocks; 16-byte chunks per thread and slice
  const float *xsrc[XC], *wsrc[WC];
#pragma unroll
  for (int i = 0; i < XC; ++i) {
    const int c = tid + i * 256, src = xrow[c >> 4];
    xsrc[i] = src >= 0 ? X + (int64_t)src * d.x_row_stride + (c & 15) * 4 : nullptr;
  }
#pragma unroll
  for (int i = 0; i < WC; ++i) {
    const int c = tid + i * 256, m = m0 + (c >> 4);
    wsrc[i] = m < d.m ? W + (int64_t)m * d.w_m_stride + (c & 15) * 4 : nullptr;
  }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[RJ], px[XC], pw[WC];
#pragma unroll
  for (int j = 0; j < RJ; ++j) acc[j] = zero;
  const int kc = (tid & 15) * 4;                 // this thread's k inside a slice
  auto fetch = [&](int k0) {
    const bool in = k0 + kc < d.k;
#pragma unroll
    for (int i = 0; i < XC; ++i) px[i] = xsrc[i] && in ? *reinterpret_cast<const f32x4*>(xsrc[i] + k0) : zero;
#pragma unroll
    for (int i = 0; i < WC; ++i) pw[i] = wsrc[i] && in ? *reinterpret_cast<const f32x4*>(wsrc[i] + k0) : zero;
  };
  fetch(0);
  for (int k0 = 0; k0 < d.k; k0 += FK) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < XC; ++i) *reinterpret_cast<f32x4*>(xs + ((tid + i * 256) >> 4) * FS + kc) = px[i];
#pragma unroll
    for (int i = 0; i < WC; ++i) *reinterpret_cast<f32x4*>(ws + ((tid + i * 256) >> 4) * FS + kc) = pw[i];
    __syncthreads();
    if (k0 + FK < d.k) fetch(k0 + FK);           // the next slice's loads fly while this one is multiplied
#pragma unroll
    for (int k = 0; k < FK; k += 16) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(ws + (wave * 16 + l15) * FS + k + gq * 4);
      f32x4 b[RJ];
#pragma unroll
      for (int j = 0; j < RJ; ++j) b[j] = *reinterpret_cast<const f32x4*>(xs + (j * 16 + l15) * FS + k + gq * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < RJ; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[j][e], acc[j], 0, 0, 0);
    }
  }
  TY* Y = static_cast<TY*>(d.y) + (int64_t)g * d.y_group_stride;
#pragma unroll
  for (int j = 0; j < RJ; ++j) {
    const int r = j * 16 + l15, dst = yrow[r];
    if (dst < 0) continue;
    float scale = 1.f;
    if (d.epilogue == PEGAINFER_EPI_SIGMOID_GATE)
      scale = sigmoid_f(ld(static_cast<const TG*>(d.gate) + (int64_t)xrow[r] * d.gate_row_stride + g));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = m0 + wave * 16 + gq * 4 + e;
      if (m >= d.m) continue;
      float v = acc[j][e];
      if (d.epilogue == PEGAINFER_EPI_RELU_SQ) { v = fmaxf(v, 0.f); v *= v; }
      else if (d.epilogue == PEGAINFER_EPI_GELU_ERF) v = gelu_erf_f(v);
      else if (d.epilogue == PEGAINFER_EPI_SIGMOID_GATE) v *= scale;
      st(Y + (int64_t)dst * d.y_row_stride + m, v);
    }
  }
}

template <typename TY, typename TG>
static void f32_tiles_launch(const pegainfer_gemm_desc& d, hipStream_t s) {
  const int groups = d.tile_group ? 1 : d.groups, mt = ceil_div(d.m, FM);
  const bool small = !d.tile_group && (long)ceil_div(d.rows, 64) * mt * groups < 2L * device_cus();
  const int TR = small ? 32 : 64;
  dim3 grid(d.tile_group ? d.max_tiles : ceil_div(d.rows, TR), mt, groups);
  if (small) gemm_f32_mfma_kernel<TY, TG, 32><<<grid, 256, 0, s>>>(d);
  else gemm_f32_mfma_kernel<TY, TG, 64><<<grid, 256, 0, s>>>(d);
}

template <typename TX, typename TW, typename TY>
static bool gemm_strided_launch(const pegainfer_gemm_desc& d, hipStream_t s) {
  dim3 grid(d.tile_group ? d.max_tiles : ceil_div(d.rows, GT), ceil_div(d.m, GM), d.tile_group ? 1 : d.groups);
  const bool gate32 = d.gate_dtype == kDtF32;
  if (!d.plain && chunks_ok(d)) {
    // few rows per tile: stream the weights once
    const int tr = d.tile_group ? (d.max_tile_rows > 0 ? d.max_tile_rows : (d.tile_rows_cap > 0 ? d.tile_rows_cap : GT)) : d.rows;
    if constexpr (std::is_same<TW, uint16_t>::value) {
      // one fp32 row stays on the FMA form: splitting it costs more than the matrix cores give (a 65 536 x 2048 matrix: 49 us against 57)
      if (tr <= kRowsMax && !(tr == 1 && std::is_same<TX, float>::value)) {
        if (gate32) rows_mfma_launch<TX, TY, float>(d, s);
        else rows_mfma_launch<TX, TY, uint16_t>(d, s);
        return true;
      }
    }
    if constexpr (std::is_same<TW, float>::value) {
      if (tr <= kRowsMax) {
        // Few rows by FMA, which needs no more than the rows' own products, while a grid's columns hold the outputs.
        const int R = d.m > 16 * 65535 ? 0 : tr <= 1 ? 1 : tr <= 2 ? 2 : tr <= 4 ? 4 : 0;
        auto run = [&](auto gate) {
          using TG = std::remove_pointer_t<decltype(gate)>;
          if (R == 1) rows_direct_launch<TW, TY, TG, 1, false>(d, 0, 0, s);
          else if (R == 2) rows_direct_launch<TW, TY, TG, 2, false>(d, 0, 0, s);
          else if (R == 4) rows_direct_launch<TW, TY, TG, 4, false>(d, 0, 0, s);
          else rows_f32_launch<TY, TG>(d, s);
        };
        if (gate32) run((float*)nullptr);
        else run((uint16_t*)nullptr);
        return true;
      }
    } else if constexpr (std::is_same<TX, float>::value) {
      if (tr <= 1 && d.m <= 16 * 65535) {
        if (gate32) rows_direct_launch<TW, TY, float, 1, false>(d, 0, 0, s);
        else rows_direct_launch<TW, TY, uint16_t, 1, false>(d, 0, 0, s);
        return true;
      }
    }
    if constexpr (std::is_same<TW, uint16_t>::value) {   // bf16 weights: the matrix cores
      if (gate32) mfma_form_launch<TX, TY, float>(d, s);
      else mfma_form_launch<TX, TY, uint16_t>(d, s);
      return true;
    } else if (!d.tile_group || d.tile_rows_cap <= GT) {
      if (gate32) f32_tiles_launch<TY, float>(d, s);
      else f32_tiles_launch<TY, uint16_t>(d, s);
      return true;
    }
  }
  if (d.tile_group && d.tile_rows_cap > GT) return false;   // a table cut for 128-row tiles cannot be walked by the 64-row form
  if (gate32) gemm_strided_kernel<TX, TW, TY, float><<<grid, 256, 0, s>>>(d);
  else gemm_strided_kernel<TX, TW, TY, uint16_t><<<grid, 256, 0, s>>>(d);
  return true;
}

}  // namespace pk

extern "C" pegainfer_status_t pegainfer_gemm_strided(const pegainfer_gemm_desc* dp, pegainfer_stream_t stream) {
  using namespace pk;
  const pegainfer_gemm_desc& d = *dp;
  if (d.m <= 0 || d.k <= 0) return 0;
  if (d.tile_group ? d.max_tiles <= 0 : (d.rows <= 0 || d.groups <= 0)) return 0;
  hipStream_t s = as_stream(stream);
  const int key = (d.x_dtype << 2) | (d.w_dtype << 1) | d.y_dtype;
  bool ok = false;
  switch (key) {
    case 0: ok = gemm_strided_launch<uint16_t, uint16_t, uint16_t>(d, s); break;
    case 1: ok = gemm_strided_launch<uint16_t, uint16_t, float>(d, s); break;
    case 4: ok = gemm_strided_launch<float, uint16_t, uint16_t>(d, s); break;
    case 5: ok = gemm_strided_launch<float, uint16_t, float>(d, s); break;
    case 7: ok = gemm_strided_launch<float, float, float>(d, s); break;
    default: break;
  }
  if (!ok) return (pegainfer_status_t)hipErrorInvalidValue;
  return (pegainfer_status_t)hipGetLastError();
}

static pegainfer_status_t expert_rows_impl(const pegainfer_expert_rows_desc* q, const pegainfer_chosen_desc* c, pegainfer_stream_t stream) {
  using namespace pk;
  constexpr pegainfer_status_t bad = (pegainfer_status_t)hipErrorInvalidValue;
  if (!q) return bad;
  pegainfer_gemm_desc d = q->g;
  if (c) {
    if (d.tile_group || d.x_row_index || d.y_row_index || !c->expert || !pegainfer_expert_rows_chosen_ok(c->rows, c->top, c->experts)) return bad;
    // no more tiles than pairs, and no more than one per expert and 16 pairs
    const int pairs = c->rows * c->top;
    d.max_tiles = std::min(pairs, c->experts + pairs / kRowsMax);
    d.tile_rows_cap = kRowsMax;
    d.max_tile_rows = 0;
  }
  const int slices = q->shared_w ? q->shared_groups : 0;
  if (d.m <= 0 || d.k <= 0 || d.max_tiles <= 0) return 0;
  const int rows = d.max_tile_rows > 0 ? d.max_tile_rows : d.tile_rows_cap;
  if ((!c && (!d.tile_group || !d.tile_row0 || !d.tile_rows || !d.n_tiles)) || d.plain || d.x_dtype != kDtBf16 || d.w_dtype != kDtBf16 ||
      (d.y_dtype != kDtBf16 && d.y_dtype != kDtF32) || rows < 1 || rows > kRowsMax || !chunks_ok(d) || d.epilogue == PEGAINFER_EPI_SIGMOID_GATE ||
      q->glu < PEGAINFER_GLU_NONE || q->glu > PEGAINFER_GLU_CLAMP || (q->glu && d.epilogue) || slices < 0 ||
      (slices && (q->shared_rows < 1 || q->shared_rows > kRowsMax || q->shared_pos0 < 0 || (q->shared_m_stride & 7) || (q->shared_group_stride & 7) ||
                  (q->shared_up & 7) || (reinterpret_cast<uintptr_t>(q->shared_w) & 15u))))
    return bad;
  const ExpertForm ex{q->glu, 0, q->shared_rows, q->shared_pos0, q->limit, q->alpha, q->shared_limit, static_cast<const uint16_t*>(q->shared_w),
                      q->shared_m_stride, q->shared_group_stride, q->shared_up, c ? c->expert : nullptr, c ? c->tiles : nullptr, c ? c->rows * c->top : 0, c ? c->top : 1,
                      c ? c->experts : 0, c ? c->x_by_pair : 0};
  if (d.y_dtype == kDtF32) expert_rows_launch<float>(d, ex, slices, as_stream(stream));
  else expert_rows_launch<uint16_t>(d, ex, slices, as_stream(stream));
  return (pegainfer_status_t)hipGetLastError();
}

extern "C" pegainfer_status_t pegainfer_expert_rows(const pegainfer_expert_rows_desc* q, pegainfer_stream_t stream) {
  return expert_rows_impl(q, nullptr, stream);
}

extern "C" int32_t pegainfer_expert_rows_chosen_ok(int32_t rows, int32_t top, int32_t experts) {
  return rows > 0 && rows <= pk::kRowsMax && top > 0 && (int64_t)rows * top <= 64 * pk::kChosenMost && experts > 0 && experts <= 64;
}
extern "C" pegainfer_status_t pegainfer_expert_rows_chosen(const pegainfer_expert_rows_desc* q, const pegainfer_chosen_desc* chosen, pegainfer_stream_t stream) {
  return chosen ? expert_rows_impl(q, chosen, stream) : (pegainfer_status_t)hipErrorInvalidValue;
}

extern "C" int32_t pegainfer_glu_gemm_ok(const pegainfer_glu_gemm_desc* q) {
  using namespace pk;
  if (!q) return 0;
  const pegainfer_gemm_desc& d = q->g;
  return d.x_dtype == kDtF32 && d.w_dtype == kDtF32 && d.y_dtype == kDtF32 && !d.plain && !d.tile_group && !d.epilogue && d.m > 0 && d.m <= 4 * 65535 &&
         d.k > 0 && d.rows > 0 && d.rows <= 4 && d.groups > 0 && d.groups <= 65535 && chunks_ok(d) && (q->up & 7) == 0 && q->act >= 0 &&
         q->act <= PEGAINFER_ACT_GELU_ERF;
}
extern "C" pegainfer_status_t pegainfer_glu_gemm(const pegainfer_glu_gemm_desc* q, pegainfer_stream_t stream) {
  using namespace pk;
  if (!pegainfer_glu_gemm_ok(q)) return (pegainfer_status_t)hipErrorInvalidValue;
  const int rows = q->g.rows;
  hipStream_t s = as_stream(stream);
  if (rows == 1) rows_direct_launch<float, float, float, 1, true>(q->g, q->act, q->up, s);
  else if (rows == 2) rows_direct_launch<float, float, float, 2, true>(q->g, q->act, q->up, s);
  else rows_direct_launch<float, float, float, 4, true>(q->g, q->act, q->up, s);
  return (pegainfer_status_t)hipGetLastError();
}
