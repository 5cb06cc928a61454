// Prefill GEMM, long prompts: 256 x 256 x 64 tiles, v_mfma_f32_16x16x32_bf16, 128 KiB of LDS.
//
//   Y[T, M] = X[T, K] . W[M, K]^T,  a workgroup owns 256 W rows x 256 token rows: four waves, one on each SIMD, wave (wr, wc) a
//   128 x 128 block of it as 8 x 8 MFMA tiles (256 accumulator registers).
//
// Bound by the matrix cores, which are busy 0.65 - 0.68 of all cycles of a launch (10 000 tokens, a last round that is not full among them), and by the power that
// they draw: the plain form takes the same cycles with random operands and with zeros, at 1.85 GHz and at 2.3 (profiles/cases_pmc_sq.csv: gemm-random, gemm-zeros).
// With eight waves of 128 x 64 (two a SIMD, one computing while the other reads, four phases a K tile) the bound was LDS: 28 ds_read_b128 a wave and K
// tile, 224 KB, and 64 KB that the DMA writes are 2250 of its cycles for 2048 of the matrix cores.  Waves of 128 x 128 read 128 KB, so that
//   * a wave has the matrix core of its SIMD to itself and everything else happens between two of its products (16 cycles each), a slot a product:
//     128 slots a K tile, in the program's order (sched_barrier);
//   * fragments are read one K step of 32 ahead, an instruction every second slot;
//   * a K tile's place in LDS is free once every wave has read its second step (slot 36: barrier); from there the tile after the next is fetched
//     into it by LDS-DMA (global_load_lds_dwordx4, XOR-swizzled through the SOURCE address), an instruction every eighth slot, as fast as
//     addresses are taken without holding a wave up (every second or fourth slot: 13 / 5 % slower), its M0 one slot before;
//   * the next tile has to be there at slot 96 (counted vmcnt: what the tile after it has been asked for stays in flight; barrier): its last piece is asked for
//     at slot 29;
//   * results leave through LDS as whole lines: 8 bytes a lane in runs of 32, as the products leave them, took 8 us a tile, whole rows of 256 bytes 4;
//   * a workgroup takes one tile.  It has all of its compute unit's LDS and registers: what it does not give up nobody else gets.  Workgroups that stayed
//     for every 256th tile hid 2 us of fetching and up to 4 of stores a tile, which made a launch alone 1 % faster (plain form; none the SwiGLU form), but one
//     that found its unit held began only as the others were through: 10 000 tokens, 19 456 x 2560 beside 8 held units 1221 us of 802 (822 of 796 a tile a
//     workgroup, 951 of 907 with eight waves), and another stream's launch waited 578 us for a unit (49, 61).
// Measured against the eight waves, same bits, random operands, cold weights (us): 10 000 tokens: 19 456 x 2560 907 -> 796, 2560 x 9728 407 -> 371, 6144 x 2560
// 268 -> 230; 5362 tokens: 2560 x 9728 217 -> 188, 2560 x 4096 96 -> 84.  The SwiGLU form, whose 128 gated units a lane are as long as eight K tiles'
// products: 10 000 tokens, 9728 x 2560 800 -> 736, 2048 tokens, 12 288 x 4096 321 -> 290, 1024 tokens, 9728 x 2560 104 -> 99.
// Per-element K order (K tile by K tile, k-step 0 then 1) is that of the other tiled kernels: same bits.
#pragma once

#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.h"

namespace pk {

constexpr int G256_BM = 256, G256_BT = 256, G256_BK = 64;
constexpr int kG256HalfBytes = 128 * 128;            // 128 rows x 128 B
constexpr int kG256LdsBytes = 8 * kG256HalfBytes;    // 2 parities x {A_lo, A_hi, B_lo, B_hi}
constexpr int kG256TurnBytes = 4 * 8192;             // where the waves turn their results
enum { kHalfAlo = 0, kHalfAhi = 1, kHalfBlo = 2, kHalfBhi = 3 };

template <int... I, typename F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, F&& f) { (f(std::integral_constant<int, I>()), ...); }
// f(0), f(1), .. f(N - 1), the numbers as types
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) { each_of(std::make_integer_sequence<int, N>(), f); }

// PART: a K slice's fp32 partials (the split-K launch).  NT: a single tile of tokens, so that this workgroup is the only reader of its W rows (SplitOut::w_nt); an
// instance of its own, as a fetch has a slot.  256 tokens (us): 32 768 x 2560 63.1 -> 58.2, 65 536 x 4096 155 -> 126, SwiGLU of 16 384 x 2560 68.8 -> 62.4.
template <bool SILU, bool PART = false, bool NT = false>
__global__ __launch_bounds__(256, 1) void mfma_gemm256_kernel(const Half* __restrict__ W, const Half* __restrict__ X,
                                                           Half* __restrict__ Y, int M, int T, int K, int m_tiles,
                                                           int t_tiles, SplitOut so, float* __restrict__ part = nullptr,
                                                           int nk_slice = 0) {
  extern __shared__ __attribute__((aligned(16))) u32x4 g256_smem[];
  const int ntiles = m_tiles * t_tiles;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wr = wave >> 1, wc = wave & 1;
  const int l15 = lane & 15, g = lane >> 4;
  // the value as one that nothing before knows: what follows from it is computed where it is used, not kept across the products
  auto again = [](int v) {
    asm volatile("" : "+v"(v));
    return v;
  };
  int zslice = (int)blockIdx.y;
  // t_major: row tile fastest inside an XCD's run - for T > M (o_proj / down_proj / qkv at 10 k tokens) an XCD then pulls
  // 1/8 of X and all of W through its L2 instead of all of X and 1/8 of W
  // chunk: the slow dimension of the order is walked in chunks of `chunk` tiles, so the ~32 workgroups an XCD runs at a time
  // are a (32 / chunk) x chunk block of tiles sharing 32 / chunk + chunk operand panels through its L2 instead of 1 + 32: gate_up at
  // 10 k tokens (76 x 40 tiles, token tile fastest) fetched 4.2 GB from the memory side per launch for 151 MB of operands - every X
  // panel once per row tile (FETCH_SIZE, profiles/r6c_ctx10000_pmc_fetch.csv)
  int mt, tt;
  {
    int tile = (int)blockIdx.x;
    if (PART && so.xcd_slices) {
      // K-split launches: one contiguous run of (slice, tile) work items per XCD in SLICE-major order, so an XCD pulls
      // one K slice of X through its L2 instead of all of X (see mfma_gemm128x256_kernel); same work items, same bits
      const int nitems = ntiles * (int)gridDim.y, id = (int)blockIdx.x + (int)gridDim.x * (int)blockIdx.y;
      const int q = nitems / 8, r = nitems % 8, xcd = id % 8, idx = id / 8;
      const int at = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
      zslice = at / ntiles;
      tile = at - zslice * ntiles;
    } else {  // XCD-aware order (block b runs on XCD b % 8): every XCD walks a contiguous run of tiles, token tile fastest
      const int q = ntiles / 8, r = ntiles % 8, xcd = tile % 8, idx = tile / 8;
      tile = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
    }
    if (so.chunk > 0) {
      const int fast_n = so.t_major ? m_tiles : t_tiles, slow_n = so.t_major ? t_tiles : m_tiles;   // fast = the inner dimension of the plain order
      const int per_chunk = slow_n * so.chunk;                  // tiles of one full chunk of the FAST dimension
      const int c = tile / per_chunk, rem = tile - c * per_chunk;
      const int cw = fast_n - c * so.chunk < so.chunk ? fast_n - c * so.chunk : so.chunk;
      const int slow = rem / cw, fast = c * so.chunk + rem - slow * cw;
      mt = so.t_major ? fast : slow;
      tt = so.t_major ? slow : fast;
    } else {
      mt = so.t_major ? tile % m_tiles : tile / t_tiles;
      tt = so.t_major ? tile / m_tiles : tile - mt * t_tiles;
    }
  }

  // ---- DMA sources: piece p of an operand = its rows p * 32 + wave * 8 + (lane >> 3), LDS slot lane & 7: the lane fetches global slot
  //      (lane & 7) ^ (row & 7) so that readers use lds_slot().  The last tile of a direction begins
  //      256 before the end (the kernel is taken from 256 rows and tokens on): what it shares with the tile before it, both leave with the same bits ----
  // SILU: m0 = the first of 128 activation columns
  const int m0 = SILU ? std::min(so.silu_c0 + mt * 128, silu_cols_end(so) - 128) : std::min(mt * G256_BM, M - G256_BM);
  const int t0 = std::min(tt * G256_BT, T - G256_BT);
  // PART: a K slice of nk_slice K tiles (even and at least four, like the last, shorter one: the tiles are walked in pairs); the workgroup's fp32 tile goes to
  // part[z][T][M] and a slice-sum launch adds the slices in z order (down_proj at 1-2 k tokens: 40-80 tiles of 256 x 256 for 256 CUs)
  const int kt_begin = PART ? zslice * nk_slice : 0, nk = PART ? std::min(K / G256_BK - kt_begin, nk_slice) : K / G256_BK;
  const char* a_at = reinterpret_cast<const char*>(W + (size_t)m0 * K + (size_t)kt_begin * G256_BK);
  const char* b_at = reinterpret_cast<const char*>(X + (size_t)t0 * K + (size_t)kt_begin * G256_BK);
  uint32_t piece_at[8];
#pragma unroll
  for (int p = 0; p < 8; ++p) piece_at[p] = (uint32_t)(p * 32 + wave * 8 + (lane >> 3)) * (uint32_t)(K * 2) + (uint32_t)((lane & 7) ^ (lane >> 3)) * 16u;
  const int64_t up_rows = SILU ? (int64_t)so.silu_I * K * 2 : 0;
  typedef __attribute__((address_space(3))) void* lptr_t;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lptr_t)&g256_smem[0] + wave * 1024u);
  // piece q of a K tile (0-7: W, 8-15: X) in the place of parity par, `at` bytes behind the tile that a_at, b_at point to: M0, then the load
  auto aim = [&](auto q, auto par) {
    const uint32_t to = lds0 + (uint32_t)(decltype(par)::value * 65536 + decltype(q)::value * 4096);
    asm volatile("s_mov_b32 m0, %0" ::"s"(to) : "m0");
  };
  struct From { const char *a, *up, *b; };         // where a K tile lies in W (SILU: and the up rows) and in X
  auto from = [&](int at) { return From{a_at + at, a_at + up_rows + at, b_at + at}; };
  auto fetch = [&](auto qc, const From& f) {
    constexpr int q = decltype(qc)::value;
    // SILU: a tile is 128 gate rows and their 128 up rows, a wave's m-tiles 0-3 gate rows, 4-7 the same up rows
    const char* base = q >= 8 ? f.b : SILU && (q & 2) ? f.up : f.a;
    const uint32_t v = piece_at[q >= 8 || !SILU ? q & 7 : (q >> 2) * 2 + (q & 1)];
    if constexpr (NT && q < 8) asm volatile("global_load_lds_dwordx4 %0, %1 nt" ::"v"(v), "s"(base) : "memory");
    else asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(v), "s"(base) : "memory");
  };

  f32x4 acc[8][8];
  bf16x8_t fa[2][8], fb[2][8];
  // fragments of K step `ks` in the order of their first use: a0, b0 .. b7, a1 .. a7
  auto read = [&](auto qc, auto ksc, auto parc) {
    constexpr int q = decltype(qc)::value, ks = decltype(ksc)::value;
    const u32x4* at = g256_smem + decltype(parc)::value * 4096;
    if constexpr (q == 0 || q >= 9) {
      constexpr int i = q == 0 ? 0 : q - 8;
      fa[ks][i] = __builtin_bit_cast(bf16x8_t, at[lds_slot(wr * 128 + i * 16 + l15, ks * 4 + g)]);
    } else {
      fb[ks][q - 1] = __builtin_bit_cast(bf16x8_t, at[2048 + lds_slot(wc * 128 + (q - 1) * 16 + l15, ks * 4 + g)]);
    }
  };
  typedef std::integral_constant<int, 0> P0;
  typedef std::integral_constant<int, 1> P1;
  // the slots of a K tile (see above); a piece whose slot lies behind the last one is fetched by the next K tile
  constexpr int kFree = 36, kLanded = 96, kEvery = 8, kReadEvery = 2;
  // one K tile in the place of parity par.  MORE: there is a tile after the next to fetch; NEXT: there is a next one
  auto ktile = [&](auto parc, auto morec, auto nextc) {
    constexpr int par = decltype(parc)::value;
    constexpr bool MORE = decltype(morec)::value, NEXT = decltype(nextc)::value;
    typedef std::integral_constant<int, par ^ 1> Other;
    const From next = from(128), after = from(256);
    __builtin_amdgcn_sched_barrier(0);
    static_for<128>([&](auto nc) {
      constexpr int n = decltype(nc)::value, ks = n >> 6;
      if constexpr (n % kReadEvery == 0 && n / kReadEvery < 16) read(std::integral_constant<int, n / kReadEvery>(), P1(), parc);
      if constexpr (MORE && n == kFree) {        // every wave has its fragments of this tile
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (NEXT && n == kLanded) {      // the next tile is there; of the one after it, what has been asked for may be on its way
        constexpr int asked = MORE ? (kLanded - 2 - kFree) / kEvery + 1 : 0;
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"(asked) : "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (NEXT && n >= kLanded && (n - kLanded) % kReadEvery == 0 && (n - kLanded) / kReadEvery < 16)
        read(std::integral_constant<int, (n - kLanded) / kReadEvery>(), P0(), Other());
      constexpr int own = n - kFree, late = n + 128 - kFree;
      if constexpr (MORE && own >= 0 && own % kEvery == 0 && own / kEvery < 16) aim(std::integral_constant<int, own / kEvery>(), parc);
      if constexpr (MORE && own >= 0 && own % kEvery == 1 && own / kEvery < 16) fetch(std::integral_constant<int, own / kEvery>(), after);
      if constexpr (NEXT && n < kFree && late % kEvery == 0 && late / kEvery < 16) aim(std::integral_constant<int, late / kEvery>(), Other());
      if constexpr (NEXT && n < kFree && late % kEvery == 1 && late / kEvery < 16) fetch(std::integral_constant<int, late / kEvery>(), next);
      __builtin_amdgcn_sched_barrier(0);         // a product lies between M0 and the load that reads it
      constexpr int i = (n & 63) >> 3, j = i & 1 ? 7 - (n & 7) : n & 7;
      // as text, so that the sums stay in the accumulator registers between the products, which what reads them at a tile's end pulls them out of
      // otherwise.  Operands come from LDS or from a product 64 slots before, so that no wait belongs between them and this one
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fa[ks][i]), "v"(fb[ks][j]));
      __builtin_amdgcn_sched_barrier(0);
    });
    a_at += 128;
    b_at += 128;
  };
  static_assert(kFree % kEvery != 127 % kEvery, "an aim and its load lie in one iteration");

  // K tiles 0 and 1 (the first iteration fetches the last pieces of K tile 1 again)
  {
    auto fetch_now = [&](auto q, auto par, const From& f) {
      aim(q, par);
      asm volatile("s_nop 0");
      fetch(q, f);
    };
    const From first = from(0), second = from(128);
    static_for<16>([&](auto q) { fetch_now(q, P0(), first); });
    static_for<16>([&](auto q) { fetch_now(q, P1(), second); });
  }
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[i][j]));
    }
  asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
  __builtin_amdgcn_s_barrier();                    // K tile 0 is there
  static_for<16>([&](auto q) { read(q, P0(), P0()); });
  asm volatile("s_nop 7" ::: "memory");            // (a product's text tells nobody that a register just written must rest before it)
  __builtin_amdgcn_sched_barrier(0);
  int kt = 0;
  do {
    ktile(P0(), std::true_type(), std::true_type());
    ktile(P1(), std::true_type(), std::true_type());
    kt += 2;
  } while (kt + 2 < nk);
  ktile(P0(), std::false_type(), std::true_type());
  ktile(P1(), std::false_type(), std::false_type());
  // The last products' way to their registers.  Nothing may read a sum before, and the compiler, which does not see that a product's text takes its time, is free
  // to copy one right behind its last product: all of them pass through here as accumulator registers
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < 8; ++i)
    asm volatile("" : "+a"(acc[i][0]), "+a"(acc[i][1]), "+a"(acc[i][2]), "+a"(acc[i][3]), "+a"(acc[i][4]), "+a"(acc[i][5]), "+a"(acc[i][6]), "+a"(acc[i][7]));
  __builtin_amdgcn_sched_barrier(0);

  const int mw = SILU ? m0 + wr * 64 : m0 + wr * 128, tw = t0 + wc * 128;      // the wave's block
  // ---- epilogue.  A lane holds rows m = .. + g*4 + e (4 consecutive) of token t = .. + l15; the wave turns its block in its own 8 KB of LDS (chunks
  //      of 16 bytes, XOR-swizzled by the token), 32 tokens at a time, and stores whole rows of a token.  `wide`: every row that is written begins on
  //      16 bytes and the segments are whole chunks of eight values; else a chunk leaves in halves of four values, which no boundary cuts: rows of
  //      outputs, segments and gated columns are multiples of four and begin on 8 bytes (glds_gemm_ok, pegainfer_gemm_split, gemm_silu_impl).  Value
  //      by value such segments took 1.5 to 2.5 times as long (M 6144 in 4100 + 1020 + 1024, K 2560, 2048 tokens: 91 us, 56 in halves; 8192
  //      in 4096 + 2052 + 2044, K 256, 4096 tokens: 89, 26) ----
  const int ln = again(lane), e15 = ln & 15, eg = ln >> 4;
  char* own = reinterpret_cast<char*>(g256_smem) + kG256LdsBytes + wave * 8192;
  if constexpr (PART) {                          // 16 tokens of 512 bytes at a time
    float* pz = part + (size_t)zslice * T * M;    // the workspace's own start, rows of fours: on 16 bytes
    static_for<8>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < 8; ++i) *reinterpret_cast<f32x4*>(own + e15 * 512 + (((i * 4 + eg) ^ e15) << 4)) = acc[i][j];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int tl = q * 2 + (ln >> 5);
        const f32x4 v = *reinterpret_cast<const f32x4*>(own + tl * 512 + (((ln & 31) ^ tl) << 4));
        *reinterpret_cast<f32x4*>(pz + (size_t)(tw + j * 16 + tl) * M + mw + (ln & 31) * 4) = v;
      }
    });
  } else {
    auto chunk_of = [&](int tl, int c) { return reinterpret_cast<u32x4*>(own + tl * 256 + ((c ^ (tl & 15)) << 4)); };
    auto turn = [&](auto pc) {                   // tokens 32 p .. of the wave's block, rows of 256 bytes
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const f32x4& a = acc[i][decltype(pc)::value * 2 + h];
          *reinterpret_cast<u32x2*>(own + (h * 16 + e15) * 256 + (((i * 2 + (eg >> 1)) ^ e15) << 4) + (eg & 1) * 8) =
              u32x2{pack_bf2(a[0], a[1]), pack_bf2(a[2], a[3])};
        }
      __builtin_amdgcn_wave_barrier();
    };
    if constexpr (SILU) {                        // 64 gate values and their 64 up values, bf16 as the GEMM's output is before SwiGLU (fused_proj.cu:57-62)
      const bool wide = aligned16(Y) && ((so.silu_I | m0 | so.silu_c0 | silu_cols_end(so)) & 7) == 0;
      auto rows = [&](auto roundc) {
        auto unit = [&](float sg, float up) { return (decltype(roundc)::value ? bf16_round_f(sg) : sg) * up; };
        Half* to = Y + (size_t)(tw + (ln >> 3)) * so.silu_I + mw + (ln & 7) * 8;
        u32x4 o[2][4];                           // a pass's results wait while the next one's are made
        auto leave = [&](auto p) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            Half* at = to + (size_t)(decltype(p)::value * 32 + q * 8) * so.silu_I;
            const u32x4 v = o[decltype(p)::value & 1][q];
            if (wide) {
              *reinterpret_cast<u32x4*>(at) = v;
            } else {
              *reinterpret_cast<u32x2*>(at) = u32x2{v[0], v[1]};
              *reinterpret_cast<u32x2*>(at + 4) = u32x2{v[2], v[3]};
            }
          }
        };
        static_for<4>([&](auto p) {
          turn(p);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int tl = q * 8 + (ln >> 3);
            const u32x4 ga = *chunk_of(tl, ln & 7), up = *chunk_of(tl, 8 + (ln & 7));
            u32x4& r = o[decltype(p)::value & 1][q];
            if (__all(silu_mid_ok(ga))) {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                r[e] = pack_bf2(unit(silu_mid_f(bf_lo(ga[e])), bf_lo(up[e])), unit(silu_mid_f(bf_hi(ga[e])), bf_hi(up[e])));
            } else {                             // rare: value by value, in place
              Half *at = reinterpret_cast<Half*>(chunk_of(tl, ln & 7)), *ua = reinterpret_cast<Half*>(chunk_of(tl, 8 + (ln & 7)));
#pragma unroll 1
              for (int e = 0; e < 8; ++e) at[e] = f2bf(unit(silu_f(bf2f(at[e])), bf2f(ua[e])));
              r = *chunk_of(tl, ln & 7);
            }
          }
          if constexpr (decltype(p)::value >= 1) leave(std::integral_constant<int, decltype(p)::value - 1>());
        });
        leave(std::integral_constant<int, 3>());
      };
      if (so.silu_round) rows(std::true_type());
      else rows(std::false_type());
    } else {
      const bool wide = aligned16(Y) && (M & 7) == 0 &&
                        (!so.Y1 || (aligned16(so.Y1) && aligned16(so.Y2) && aligned16(so.Y3) && ((so.M0 | so.M1 | so.M2) & 7) == 0));
      struct Segment { Half* at; int ld, m; };
      auto segment = [&](int r) {                // where row r goes
        if (!so.Y1) return Segment{Y, M, r};
        const int b1 = so.M0 + so.M1, b2 = b1 + so.M2;
        if (r < so.M0) return Segment{Y, so.M0, r};
        if (r < b1) return Segment{so.Y1, so.M1, r - so.M0};
        if (r < b2) return Segment{so.Y2, so.M2, r - b1};
        return Segment{so.Y3, M - b2, r - b2};
      };
      if (wide) {
        const Segment sg = segment(mw + e15 * 8);
        u32x4 v[32];
        static_for<4>([&](auto p) {
          turn(p);
#pragma unroll
          for (int q = 0; q < 8; ++q) v[decltype(p)::value * 8 + q] = *chunk_of(q * 4 + eg, e15);
        });
#pragma unroll
        for (int q = 0; q < 32; ++q) *reinterpret_cast<u32x4*>(sg.at + (size_t)(tw + q * 4 + eg) * sg.ld + sg.m) = v[q];
      } else {
        const Segment half = segment(mw + (ln & 31) * 4);
        static_for<4>([&](auto p) {
          turn(p);
          const int tp = tw + decltype(p)::value * 32;
#pragma unroll 4
          for (int q = 0; q < 16; ++q) {
            const int tl = q * 2 + (ln >> 5);
            *reinterpret_cast<u32x2*>(half.at + (size_t)(tp + tl) * half.ld + half.m) = reinterpret_cast<const u32x2*>(chunk_of(tl, (ln & 31) >> 1))[ln & 1];
          }
        });
      }
    }
  }
}

// K must be a multiple of 128 (K tiles are processed in pairs, two pairs at least); same alignment rules as the other LDS-DMA kernels
inline bool gemm256_ok(int M, int T, int K) { return (K % 128) == 0 && K >= 256 && M >= 256 && T >= 256; }

inline bool gemm_t_major(int M, int T, const SplitOut& so) {   // PEGAINFER_GEMM_T_MAJOR=0: always row-tile-major runs (A/B)
  static const bool on = [] { const char* e = getenv("PEGAINFER_GEMM_T_MAJOR"); return !(e && e[0] == '0'); }();
  return on && so.silu_I == 0 && T > M;
}
// m_head > 0: that many tiles of rows, what follows is another launch's (plain form)
inline void gemm256_launch(const Half* W, const Half* X, Half* Y, int M, int T, int K, SplitOut so, hipStream_t s, int m_head = 0) {
  const bool silu = so.silu_I > 0;
  const int m_tiles = silu ? ceil_div(silu_cols_end(so) - so.silu_c0, 128) : m_head ? m_head : ceil_div(M, G256_BM), t_tiles = ceil_div(T, G256_BT);
  so.t_major = gemm_t_major(M, T, so);
  {  // PEGAINFER_GEMM_CHUNK=0: the plain order (A/B); N: chunks of N tiles
    static const int chunk = [] { const char* e = getenv("PEGAINFER_GEMM_CHUNK"); return e && *e ? atoi(e) : 8; }();
    // chunks of equal width (17 tiles: 6 + 6 + 5, not 8 + 8 + 1); only for launches of more than one round of tiles.  4 / 6 / 8 measure
    // the same (TTFT(10 000) 94.9-95.4 ms against 98.4 plain, 12: 96.0, 16: 96.8 - profiles/r6_gemm_chunk_sweep.txt)
    const int fast_n = so.t_major ? m_tiles : t_tiles;
    const int nch = chunk > 0 ? ceil_div(fast_n, chunk) : 0;
    so.chunk = nch > 1 && (long)m_tiles * t_tiles > 256 ? ceil_div(fast_n, nch) : 0;
  }
  const bool nt = t_tiles == 1 && weights_nt_on();
  auto launch = [&](auto silu_form, auto nt_form) {
    constexpr bool SILU = decltype(silu_form)::value, NT = decltype(nt_form)::value;
    static const bool once = [] {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&mfma_gemm256_kernel<SILU, false, NT>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, kG256LdsBytes + kG256TurnBytes);
      return true;
    }();
    (void)once;
    mfma_gemm256_kernel<SILU, false, NT><<<m_tiles * t_tiles, 256, kG256LdsBytes + kG256TurnBytes, s>>>(W, X, Y, M, T, K, m_tiles, t_tiles, so);
  };
  if (silu && nt) launch(std::true_type(), std::true_type());
  else if (silu) launch(std::true_type(), std::false_type());
  else if (nt) launch(std::false_type(), std::true_type());
  else launch(std::false_type(), std::false_type());
}

// split-K launch of the plain form: fp32 partials into `part` ([ksplit][T][M]); the caller sums the slices
inline bool splitk_xcd_on() {   // PEGAINFER_SPLITK_XCD=0: the slices of a tile on one XCD (A/B)
  static const bool v = [] { const char* e = getenv("PEGAINFER_SPLITK_XCD"); return !(e && e[0] == '0'); }();
  return v;
}
inline void gemm256_splitk_launch(const Half* W, const Half* X, int M, int T, int K, float* part, int ksplit, int nk_slice,
                                  hipStream_t s) {
  const int m_tiles = ceil_div(M, G256_BM), t_tiles = ceil_div(T, G256_BT);
  static const bool once = [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&mfma_gemm256_kernel<false, true>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, kG256LdsBytes + kG256TurnBytes);
    return true;
  }();
  (void)once;
  mfma_gemm256_kernel<false, true><<<dim3(m_tiles * t_tiles, ksplit), 256, kG256LdsBytes + kG256TurnBytes, s>>>(
      W, X, nullptr, M, T, K, m_tiles, t_tiles,
      SplitOut{nullptr, nullptr, nullptr, 0, 0, 0, 0, 0, 0, 0, 0, ksplit > 1 && splitk_xcd_on(), 0}, part, nk_slice);
}

// ---- stream-K form of the 256 x 256 kernel, on the schedule of eight waves (2 x 4, blocks of 128 x 64) --------------------------------------------------------------------
// The data-parallel launch above pays for tile quantisation: 304 tiles (gate_up at 1024 tokens) are one full round of the
// 256 CUs plus 48 tiles that cost a second full tile time; 152 tiles (512 tokens) leave 104 CUs idle.  Here the launch is
// PERSISTENT - one workgroup per CU - and the work is the linear sequence of (tile, K-tile pair) units, tile-major, dealt in
// equal contiguous ranges: workgroup position p owns units [U p / G, U (p + 1) / G).  A range is cut at tile boundaries into
// segments; each segment runs a main loop of eight phases per pair of K tiles - a K tile is four half-tiles (A_lo / A_hi: the rows of a wave's m-tiles 0-3 /
// 4-7, B_lo / B_hi: the tokens of its n-tiles 0-1 / 2-3), a phase one quadrant of products and the DMA of one half-tile, the second wave row a barrier
// behind the first - over its K range and then
//   * covers the whole tile            -> the ordinary epilogue;
//   * starts inside a tile             -> (only ever a workgroup's FIRST segment) the fp32 accumulators go to the workgroup's
//                                         256 KiB slot of the split-K workspace, lane-contiguous, write-through (sc1) stores,
//                                         drained, then flag[p] = 1: published EARLY in the workgroup's timeline, no waiting;
//   * starts a tile but ends inside it -> (only ever its LAST segment) the workgroup OWNS the tile: it takes the partials of
//                                         positions p + 1, p + 2, ... up to the one that holds the tile's last unit, in that
//                                         order (= ascending K), adds them to its accumulators, clears their flags, and runs
//                                         the epilogue.  Those partials were published a whole range ago.
// So the sum over K is taken in a FIXED order that depends on (M, T, K, G) only: deterministic, rerun- and graph-stable, but
// not the K order of the data-parallel kernels - the bit identity across routes is given up for prefill GEMMs at
// these sizes; the oracle comparison under the derived bar referees.  No deadlock: a publisher never waits,
// an owner waits only for publishers, and all G <= CU-count workgroups are co-resident (one per CU by LDS).  Positions follow
// the XCD-aware order of the other kernels (block b runs on XCD b % 8): neighbours in the unit order share an XCD's L2 except
// at seven seams, so most partials are re-read from the L2 they were written through.
constexpr int kG256SlotFloats = 256 * 256;   // one workgroup's accumulators: 8 x 4 f32x4 per thread x 512 threads
template <bool SILU>
__global__ __launch_bounds__(512) void mfma_gemm256_streamk_kernel(const Half* __restrict__ W, const Half* __restrict__ X,
                                                                   Half* __restrict__ Y, int M, int T, int K, int m_tiles,
                                                                   int t_tiles, SplitOut so, float* __restrict__ part,
                                                                   uint32_t* __restrict__ flags) {
  extern __shared__ __attribute__((aligned(16))) u32x4 g256_smem[];
  const int G = gridDim.x;
  int pos = blockIdx.x;
  {  // XCD-aware position: the workgroups of one XCD are neighbours in the unit order
    const int q = G / 8, r = G % 8, xcd = pos % 8, idx = pos / 8;
    pos = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
  }
  const int KP = K / (2 * G256_BK);                       // K-tile pairs per tile
  // TEAMS (second form, same round): the first form dealt the (tile, K pair) units tile-major to single workgroups and LOST
  // (gate_up at 1024 tokens 154 us against 136-140 data-parallel, profiles/r6_streamk_gemm_ab.txt): neighbours in the unit
  // order then sit at K offsets a third of a tile apart, no two workgroups ever want the same W K-tile at the same time, and
  // the 4-fold W re-use the data-parallel order gets from an XCD's L2 (the t_tiles token tiles of one row tile run side by
  // side) is gone.  So the unit is a ROW tile's K pair, dealt to TEAMS of t_tiles workgroups - consecutive positions, one
  // XCD - whose member tt computes token tile tt of every unit of the team's range: the members walk the same W K-tiles in
  // step, exactly the sharing pattern of the data-parallel launch.  A member's partner for the hand-off is the same member
  // of the next team (position + t_tiles).
  const int nteams = G / t_tiles;
  if (pos >= nteams * t_tiles) return;                    // G % t_tiles left-over workgroups
  const int team = pos / t_tiles, tt = pos - team * t_tiles;
  const long U = (long)m_tiles * KP;
  auto range_begin = [&](int tm) { return U * tm / nteams; };
  const long u_begin = range_begin(team), u_end = range_begin(team + 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wr = wave >> 2, wc = wave & 3;
  const int l15 = lane & 15, g = lane >> 4;
  typedef __attribute__((address_space(3))) void* lptr_t;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lptr_t)&g256_smem[0];
  auto half_ptr = [&](int par, int which) { return g256_smem + (size_t)(par * 4 + which) * (kG256HalfBytes / 16); };

  f32x4 acc[8][4];
  bf16x8_t a[4][2], b[2][2];
  auto read_a = [&](int par, int which) {
    const u32x4* h = half_ptr(par, which);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        a[i][ks] = __builtin_bit_cast(bf16x8_t, h[lds_slot(wr * 64 + i * 16 + l15, ks * 4 + g)]);
  };
  auto read_b = [&](int par, int which) {
    const u32x4* h = half_ptr(par, which);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        b[j][ks] = __builtin_bit_cast(bf16x8_t, h[lds_slot(wc * 32 + j * 16 + l15, ks * 4 + g)]);
  };
  auto quad = [&](int ih, int jh) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[ih * 4 + i][jh * 2 + j] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][ks], b[j][ks], acc[ih * 4 + i][jh * 2 + j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
  };

  long u = u_begin;
  while (u < u_end) {
    const int mt = (int)(u / KP), kp0 = (int)(u - (long)mt * KP);
    const int kp1 = (long)(KP - kp0) < u_end - u ? KP : kp0 + (int)(u_end - u);
    const int m0 = mt * G256_BM, t0 = tt * G256_BT;
    const int nk = 2 * (kp1 - kp0);
    // ---- DMA sources of this tile (as in the data-parallel kernel), advanced to the segment's first K tile ----
    const Half* src[4][2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int p = (j * 8 + wave) * 64 + lane, hrow = p >> 3, cs = (p & 7) ^ (hrow & 7);
      {
        const int wr_ = hrow >> 6, r = hrow & 63;
#pragma unroll
        for (int hi = 0; hi < 2; ++hi) {
          int row;
          if (SILU) {
            int gr = so.silu_c0 + mt * 128 + wr_ * 64 + r;
            gr = gr < silu_cols_end(so) ? gr : silu_cols_end(so) - 1;
            row = gr + (hi ? so.silu_I : 0);
          } else {
            row = m0 + wr_ * 128 + hi * 64 + r;
            row = row < M ? row : M - 1;
          }
          src[hi ? kHalfAhi : kHalfAlo][j] = W + (size_t)row * K + cs * 8 + (size_t)kp0 * 2 * G256_BK;
        }
      }
      {
        const int wc_ = hrow >> 5, r = hrow & 31;
#pragma unroll
        for (int hi = 0; hi < 2; ++hi) {
          int tr = t0 + wc_ * 64 + hi * 32 + r;
          tr = tr < T ? tr : T - 1;
          src[hi ? kHalfBhi : kHalfBlo][j] = X + (size_t)tr * K + cs * 8 + (size_t)kp0 * 2 * G256_BK;
        }
      }
    }
    auto stage = [&](int which, int kt) {
      const int ktc = kt < nk ? kt : nk - 1;
      const uint32_t slot = lds0 + (uint32_t)(((kt & 1) * 4 + which) * kG256HalfBytes);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint32_t dst = __builtin_amdgcn_readfirstlane(slot + (uint32_t)(j * 8 + wave) * 1024u);
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                     :: "v"(src[which][j] + (size_t)ktc * G256_BK), "s"(dst) : "memory", "m0");
      }
    };
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // ---- the 8-phase main loop over K tiles [2 kp0, 2 kp1) ----
    stage(kHalfAlo, 0); stage(kHalfBlo, 0); stage(kHalfBhi, 0); stage(kHalfAhi, 0);
    stage(kHalfAlo, 1); stage(kHalfBhi, 1);
    asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (wr == 1) __builtin_amdgcn_s_barrier();
    auto ktile = [&](int kt, int par) {
      read_b(par, kHalfBlo);
      __builtin_amdgcn_sched_barrier(0);
      read_a(par, kHalfAlo);
      stage(kHalfAhi, kt + 1);
      __builtin_amdgcn_s_barrier();
      quad(0, 0);
      __builtin_amdgcn_s_barrier();
      read_b(par, kHalfBhi);
      stage(kHalfBlo, kt + 1);
      __builtin_amdgcn_s_barrier();
      quad(0, 1);
      __builtin_amdgcn_s_barrier();
      read_a(par, kHalfAhi);
      stage(kHalfAlo, kt + 2);
      __builtin_amdgcn_s_barrier();
      quad(1, 1);
      __builtin_amdgcn_s_barrier();
      read_b(par, kHalfBlo);
      stage(kHalfBhi, kt + 2);
      asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      quad(1, 0);
      __builtin_amdgcn_s_barrier();
    };
    for (int kt = 0; kt < nk; kt += 2) {
      ktile(kt, 0);
      ktile(kt + 1, 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (wr == 0) __builtin_amdgcn_s_barrier();   // both wave rows are level again: the LDS may be re-staged

    if (kp0 != 0) {
      // ---- publish: lane-contiguous write-through stores (one 1 KiB line per wave and instruction), drain, flag ----
      float* slot = part + (size_t)pos * kG256SlotFloats + (size_t)threadIdx.x * 4;
      asm volatile("" : "+v"(slot));   // opaque: keeps the 32 loop-invariant store addresses from being hoisted (and spilled)
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          asm volatile("global_store_dwordx4 %0, %1, off sc1" :: "v"(slot + (size_t)(i * 4 + j) * 2048), "v"(acc[i][j]) : "memory");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (threadIdx.x == 0) __hip_atomic_store(flags + pos, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      if (kp1 != KP) {
        // ---- own the tile: add the later K ranges in ascending order ----
        const long need = (long)(mt + 1) * KP;
        long covered = u_end;
        int tm = team;
        for (int p = pos + t_tiles; covered < need; p += t_tiles) {
          if (threadIdx.x == 0)
            while (__hip_atomic_load(flags + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u) __builtin_amdgcn_s_sleep(2);
          __syncthreads();
          const float* slot = part + (size_t)p * kG256SlotFloats + (size_t)threadIdx.x * 4;
          asm volatile("" : "+v"(slot));
#pragma unroll
          for (int qt = 0; qt < 4; ++qt) {   // four batches of eight 16-byte loads: 32 registers next to the 128 accumulators
            f32x4 tmp[8];
#pragma unroll
            for (int q = 0; q < 8; ++q)
              asm volatile("global_load_dwordx4 %0, %1, off sc1" : "=v"(tmp[q]) : "v"(slot + (size_t)(qt * 8 + q) * 2048) : "memory");
            // the waitcnt is tied to the loaded registers so that no use can be scheduled in front of it
            asm volatile("s_waitcnt vmcnt(0)"
                         : "+v"(tmp[0]), "+v"(tmp[1]), "+v"(tmp[2]), "+v"(tmp[3]), "+v"(tmp[4]), "+v"(tmp[5]), "+v"(tmp[6]), "+v"(tmp[7])
                         :: "memory");
#pragma unroll
            for (int q = 0; q < 8; ++q) acc[(qt * 8 + q) >> 2][(qt * 8 + q) & 3] += tmp[q];
          }
          __syncthreads();   // every wave has taken its part of the slot
          if (threadIdx.x == 0) __hip_atomic_store(flags + p, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          tm += 1;
          covered = range_begin(tm + 1);
        }
      }
      // ---- epilogue (the data-parallel kernel's): lane holds rows m = .. + g*4 + e of token t = .. + l15 ----
      if (SILU) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int t = t0 + wc * 64 + j * 16 + l15;
          if (t >= T) continue;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int m = so.silu_c0 + mt * 128 + wr * 64 + i * 16 + g * 4;
            float r[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float sg = silu_f(bf16_round_f(acc[i][j][e]));
              r[e] = (so.silu_round ? bf16_round_f(sg) : sg) * bf16_round_f(acc[i + 4][j][e]);
            }
            if (m + 3 < silu_cols_end(so)) {
              u32x2 o;
              o.x = pack_bf2(r[0], r[1]);
              o.y = pack_bf2(r[2], r[3]);
              *reinterpret_cast<u32x2*>(Y + (size_t)t * so.silu_I + m) = o;
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (m + e < silu_cols_end(so)) Y[(size_t)t * so.silu_I + m + e] = f2bf(r[e]);
            }
          }
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int t = t0 + wc * 64 + j * 16 + l15;
          if (t >= T) continue;
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int m = m0 + wr * 128 + i * 16 + g * 4;
            Half* dst = Y;
            int ld = M, mm = m, mlim = M;
            if (so.Y1) {
              const int b1 = so.M0 + so.M1, b2 = b1 + so.M2;
              if (m < so.M0) { ld = mlim = so.M0; }
              else if (m < b1) { dst = so.Y1; ld = mlim = so.M1; mm = m - so.M0; }
              else if (m < b2) { dst = so.Y2; ld = mlim = so.M2; mm = m - b1; }
              else { dst = so.Y3; ld = mlim = M - b2; mm = m - b2; }
            }
            if (mm + 3 < mlim) {
              u32x2 o;
              o.x = pack_bf2(acc[i][j][0], acc[i][j][1]);
              o.y = pack_bf2(acc[i][j][2], acc[i][j][3]);
              *reinterpret_cast<u32x2*>(dst + (size_t)t * ld + mm) = o;
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (mm + e < mlim) dst[(size_t)t * ld + mm + e] = f2bf(acc[i][j][e]);
            }
          }
        }
      }
    }
    u += kp1 - kp0;
  }
}

// Stream-K plan, by shape and CU count only (the launcher and pegainfer_debug_gemm_route share it): taken - when switched
// on - where a round of 256 x 256 tiles would leave more than `min_waste_pct` % of the CU-rounds idle and the K range of a
// team is long enough to amortise a pipeline fill (>= 4 K-tile pairs).
// OFF by default: measured SLOWER than the data-parallel launch + tail at every shape it applies to (profiles/r6_streamk_*:
// gate_up 512 / 1024 / 2048 tokens 91 / 151 / 265 us against 71 / 137 / 230; TTFT(1024) 11.7 against 10.9 ms) - every
// workgroup publishes and re-reads a 256 KiB fp32 tile at the same moment, 64 MB each way through the fabric with nothing
// to overlap it, which costs more than the idle CU-rounds it removes.  PEGAINFER_STREAMK=1 / pegainfer_debug_streamk(1)
// switch it on (the GPU tests do: the kernel stays correct and deterministic).
extern int g_streamk_override;   // linear.hip: pegainfer_debug_streamk; -1 = the environment decides
inline bool gemm256_streamk_on() {
  static const bool v = [] { const char* e = getenv("PEGAINFER_STREAMK"); return e && e[0] == '1'; }();
  return g_streamk_override >= 0 ? g_streamk_override != 0 : v;
}
inline bool gemm256_streamk_plan(long tiles256, int K, int cus, int t_tiles) {
  static const int min_waste = [] { const char* e = getenv("PEGAINFER_STREAMK_MIN_WASTE"); return e && *e ? atoi(e) : 8; }();
  if (!gemm256_streamk_on() || cus < 8 || tiles256 <= 0 || t_tiles < 1 || t_tiles > cus / 8) return false;   // a team fits an XCD
  const long rounds = (tiles256 + cus - 1) / cus;
  const long waste_pct = 100 - 100 * tiles256 / (rounds * cus);
  const long nteams = cus / t_tiles, row_units = tiles256 / t_tiles * (K / (2 * G256_BK));
  const long idle_pct = 100 - 100 * nteams * t_tiles / cus;             // workgroups that fit no team
  return waste_pct >= min_waste + idle_pct && row_units / nteams >= 4;
}

inline void gemm256_streamk_launch(const Half* W, const Half* X, Half* Y, int M, int T, int K, SplitOut so, float* part,
                                   uint32_t* flags, int cus, hipStream_t s) {
  const bool silu = so.silu_I > 0;
  const int m_tiles = silu ? ceil_div(silu_cols_end(so) - so.silu_c0, 128) : ceil_div(M, G256_BM), t_tiles = ceil_div(T, G256_BT);
  so.w_nt = 0;
  if (silu) {
    static const bool once = [] {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&mfma_gemm256_streamk_kernel<true>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, kG256LdsBytes);
      return true;
    }();
    (void)once;
    mfma_gemm256_streamk_kernel<true><<<cus, 512, kG256LdsBytes, s>>>(W, X, Y, M, T, K, m_tiles, t_tiles, so, part, flags);
  } else {
    static const bool once = [] {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&mfma_gemm256_streamk_kernel<false>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, kG256LdsBytes);
      return true;
    }();
    (void)once;
    mfma_gemm256_streamk_kernel<false><<<cus, 512, kG256LdsBytes, s>>>(W, X, Y, M, T, K, m_tiles, t_tiles, so, part, flags);
  }
}

// ---- 128 x 256 tiles: the same machinery for matrices with too few 256-row tiles to fill the chip (qkv / o_proj /
// down_proj at ~0.5-2 k tokens: 2560 rows are 10 tiles of 256 but 20 of 128).  8 waves as 2 x 4, wave (wr, wc) owns
// 64 W rows x 64 token rows = 4 x 4 MFMA tiles (64 accumulator VGPRs).  A K tile is THREE 16 KiB half-tiles - A (all 128
// rows), B_lo / B_hi (token rows of n-tiles 0-1 / 2-3 of every wave column) - and two phases:
//     phase 1: read A + B_lo, quadrant lo (16 MFMAs)        phase 2: read B_hi, quadrant hi (16 MFMAs)
// LDS holds a ring of three K tiles (144 KiB): the three half-tiles of K tile kt + 2 are staged during K tile kt into the
// slots K tile kt - 1 was read from, one counted vmcnt(6) per K tile (tile kt + 2 stays in flight across the barrier,
// tile kt + 1 has landed), wave row 1 runs one barrier behind wave row 0 as above.  Per-element K order unchanged: same
// bits as the other tiled kernels.
// Measured (profiles/r3_gemm128x256_ab.txt, 1024 tokens, cold weights): qkv 57 -> 43 us, down_proj 84 -> 67 us, o_proj
// 45 -> 41 us; per-CU efficiency ~40-45 % (the 256 x 256 kernel: 57 %): a 128 x 256 tile moves 48 KiB into LDS per 32
// MFMAs per wave, ~3/4 of a CU's L1 fill rate at the MFMA-bound pace.  A variant with double-buffered fragment registers
// and ONE barrier per K tile (every read a quadrant ahead of its MFMAs, no wave-row skew) was 25 % SLOWER (qkv 55 us):
// without the skew both waves of a SIMD sit in the same segment and nothing feeds the matrix pipe across the barrier.
constexpr int G128_BM = 128;
constexpr int kG128LdsBytes = 9 * kG256HalfBytes;
enum { kG128A = 0, kG128Blo = 1, kG128Bhi = 2 };

// NF = 4: four more waves that do nothing but issue the DMAs (12 per K tile each), in the barrier rhythm of a
// wave-row-0 wave; the eight compute waves issue none.  A DMA instruction costs its wave ~133 cycles of issue slot
// (tools/probes/ingest_probe) - six per wave and K tile were 800 cycles next to 32 MFMAs = 512.  159 VGPRs: three waves
// per SIMD fit.  NF = 0: the form in which every wave stages its share, kept for the A/B (PEGAINFER_GEMM128X256_FEED=0).
// MT = 16-row MFMA tiles per wave row: 4 = the 128-row tile; 3 = a 96-row tile (plain NF = 4 form only) for
// matrices whose 128-row tiling leaves CUs idle - the stacked qkv at 768 / 1024 tokens: 144 / 192 tiles of 128 rows, 192 / 256
// of 96.  Same per-element K order: same bits.
template <bool SILU, int NF, int MT = 4>
__global__ __launch_bounds__(512 + NF * 64) void mfma_gemm128x256_kernel(const Half* __restrict__ W, const Half* __restrict__ X,
                                                               Half* __restrict__ Y, int M, int T, int K, int m_tiles,
                                                               int t_tiles, SplitOut so, float* __restrict__ part,
                                                               int nk_slice) {
  extern __shared__ __attribute__((aligned(16))) u32x4 g256_smem[];
  const int ntiles = m_tiles * t_tiles;
  int tile = blockIdx.x, zslice = (int)blockIdx.y;
  if (part && so.xcd_slices) {
    // K-split launches: the hardware deals workgroups to XCDs by their linear id; give every XCD one contiguous run of
    // (slice, tile) work items in SLICE-major order, so an XCD works on (mostly) one K slice of a few row tiles.  With the slices
    // of a tile on one XCD (the 2-D grid's natural order: gridDim.x is a multiple of 8) every XCD pulled the WHOLE of X through
    // its L2 - down_proj at 1024 tokens fetched 209 MB from the memory side for 70 MB of operands (FETCH_SIZE, profiles/
    // r6b_ctx1024_pmc_fetch.csv).  Same work items, same arithmetic: same bits.
    const int nitems = ntiles * (int)gridDim.y, id = (int)blockIdx.x + (int)gridDim.x * (int)blockIdx.y;
    const int q = nitems / 8, r = nitems % 8, xcd = id % 8, idx = id / 8;
    const int item = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
    zslice = item / ntiles;
    tile = item - zslice * ntiles;
  } else {
    const int q = ntiles / 8, r = ntiles % 8, xcd = tile % 8, idx = tile / 8;
    tile = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
  }
  const int mt = so.t_major ? tile % m_tiles : tile / t_tiles, tt = so.t_major ? tile / m_tiles : tile - mt * t_tiles;   // see mfma_gemm256_kernel
  constexpr int BMT = 32 * MT;            // W rows per tile
  const int m0 = so.m_first + mt * BMT, t0 = tt * G256_BT;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wr = wave >> 2, wc = wave & 3;
  const int l15 = lane & 15, g = lane >> 4;

  constexpr int NI = NF ? NF : 8;           // waves that issue DMAs
  constexpr int PPW = 16 / NI;              // 1 KiB pieces per issuing wave and half-tile
  constexpr int PPA = 4 * MT / NI;          // ... of the A half-tile (32 * MT rows = 4 * MT pieces)
  constexpr int HT = MT / 2;                // SwiGLU form: gate m-tiles per wave row (their up rows are the wave row's other half)
  static_assert((4 * MT) % NI == 0 && (MT % 2 == 0 || !SILU), "the SwiGLU form pairs m-tiles: an even count per wave row");
  const bool feeder = NF && wave >= 8;
  const int wi = NF ? wave - 8 : wave;      // index among the issuing waves (compute waves of the NF form: negative, unused)
  const Half* src[3][PPW];
#pragma unroll
  for (int j = 0; j < PPW; ++j) {
    const int p = (j * NI + (wi < 0 ? 0 : wi)) * 64 + lane, hrow = p >> 3, cs = (p & 7) ^ (hrow & 7);
    int row;
    if (SILU) {   // a wave row's m-tiles 0 .. HT-1 are 16 * HT gate rows, HT .. MT-1 their up rows: gate and up of an element meet in one lane
      const int hr = hrow < BMT ? hrow : BMT - 1, wrow = hr / (16 * MT), ti = (hr >> 4) - wrow * MT, up = ti >= HT;
      int gr = so.silu_c0 + mt * (16 * MT) + wrow * (16 * HT) + (ti - (up ? HT : 0)) * 16 + (hr & 15);
      gr = gr < silu_cols_end(so) ? gr : silu_cols_end(so) - 1;
      row = gr + (up ? so.silu_I : 0);
    } else {
      row = m0 + (hrow < BMT ? hrow : BMT - 1);
      row = row < M ? row : M - 1;
    }
    src[kG128A][j] = W + (size_t)row * K + cs * 8;
    const int wc_ = hrow >> 5, r = hrow & 31;
#pragma unroll
    for (int hi = 0; hi < 2; ++hi) {
      int tr = t0 + wc_ * 64 + hi * 32 + r;
      tr = tr < T ? tr : T - 1;
      src[hi ? kG128Bhi : kG128Blo][j] = X + (size_t)tr * K + cs * 8;
    }
  }
  typedef __attribute__((address_space(3))) void* lptr_t;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lptr_t)&g256_smem[0];
  const int kt_begin = part ? zslice * nk_slice : 0;
  const int nk_total = K / G256_BK;
  const int nk = part ? (nk_total - kt_begin < nk_slice ? nk_total - kt_begin : nk_slice) : nk_total;
#pragma unroll
  for (int w = 0; w < 3; ++w)
#pragma unroll
    for (int j = 0; j < PPW; ++j) src[w][j] += (size_t)kt_begin * G256_BK;
  // stage half-tile `which` of K tile kt into ring slot `ring` (clamped past the end: a dead slot, the load only keeps
  // vmcnt uniform)
  auto stage = [&](int which, int kt, int ring) {
    const int ktc = kt < nk ? kt : nk - 1;
    const uint32_t slot = lds0 + (uint32_t)((ring * 3 + which) * kG256HalfBytes);
#pragma unroll
    for (int j = 0; j < PPW; ++j) {
      if (which == kG128A && j >= PPA) break;
      const uint32_t dst = __builtin_amdgcn_readfirstlane(slot + (uint32_t)(j * NI + wi) * 1024u);
      if (which == kG128A && so.w_nt)   // a single token tile: W bytes have one reader (SplitOut::w_nt)
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt"
                     :: "v"(src[which][j] + (size_t)ktc * G256_BK), "s"(dst) : "memory", "m0");
      else
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                     :: "v"(src[which][j] + (size_t)ktc * G256_BK), "s"(dst) : "memory", "m0");
    }
  };
  auto half_ptr = [&](int ring, int which) { return g256_smem + (size_t)(ring * 3 + which) * (kG256HalfBytes / 16); };

  f32x4 acc[MT][4];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8_t a[MT][2], b[2][2];
  auto read_a = [&](int ring) {
    const u32x4* h = half_ptr(ring, kG128A);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        a[i][ks] = __builtin_bit_cast(bf16x8_t, h[lds_slot(wr * (16 * MT) + i * 16 + l15, ks * 4 + g)]);
  };
  auto read_b = [&](int ring, int which) {
    const u32x4* h = half_ptr(ring, which);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        b[j][ks] = __builtin_bit_cast(bf16x8_t, h[lds_slot(wc * 32 + j * 16 + l15, ks * 4 + g)]);
  };
  auto quad = [&](int jh) {   // 16 MFMAs: all 4 m-tiles, n-tiles jh*2..
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][jh * 2 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][ks], b[j][ks], acc[i][jh * 2 + j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
  };

  constexpr int kTileDmas = PPA + 2 * PPW;  // DMAs per issuing wave and K tile: the counted wait leaves one tile in flight
  if (feeder) {
    // the whole staging side, in the barrier rhythm of a wave-row-0 wave (the EARLIEST any wave of the NF = 0 form touched
    // a ring slot, so the hazards are the ones argued above): A + B_lo of tile kt + 2 in phase 1, B_hi in phase 2
    stage(kG128A, 0, 0); stage(kG128Blo, 0, 0); stage(kG128Bhi, 0, 0);
    stage(kG128A, 1, 1); stage(kG128Blo, 1, 1); stage(kG128Bhi, 1, 1);
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kTileDmas) : "memory");
    __builtin_amdgcn_s_barrier();
    int ring = 0;
    for (int kt = 0; kt < nk; ++kt) {
      const int ring2 = ring + 2 >= 3 ? ring - 1 : ring + 2;
      stage(kG128A, kt + 2, ring2);
      stage(kG128Blo, kt + 2, ring2);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_s_barrier();
      stage(kG128Bhi, kt + 2, ring2);
      asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kTileDmas) : "memory");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_s_barrier();
      ring = ring + 1 == 3 ? 0 : ring + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the clamped tail loads must not outlive the workgroup's LDS
    __builtin_amdgcn_s_barrier();
    return;
  }
  // ---- prologue: K tiles 0 and 1 requested, tile 0 landed ----
  if constexpr (NF == 0) {
    stage(kG128A, 0, 0); stage(kG128Blo, 0, 0); stage(kG128Bhi, 0, 0);
    stage(kG128A, 1, 1); stage(kG128Blo, 1, 1); stage(kG128Bhi, 1, 1);
    asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
  }
  __builtin_amdgcn_s_barrier();
  if (wr == 1) __builtin_amdgcn_s_barrier();   // the second wave row runs one barrier behind the first

  // one K tile = two phases (fragment reads + DMA issue | barrier | 16 MFMAs | barrier); the counted wait sits in front
  // of the first barrier of the last phase, so it covers both wave rows (see the 256 x 256 kernel)
  auto ktile = [&](int kt, int ring) {
    const int ring2 = (ring + 2) % 3;
    read_b(ring, kG128Blo);
    __builtin_amdgcn_sched_barrier(0);
    read_a(ring);
    if constexpr (NF == 0) {
      stage(kG128A, kt + 2, ring2);
      stage(kG128Blo, kt + 2, ring2);
    }
    __builtin_amdgcn_s_barrier();
    quad(0);
    __builtin_amdgcn_s_barrier();
    read_b(ring, kG128Bhi);
    if constexpr (NF == 0) {
      stage(kG128Bhi, kt + 2, ring2);
      asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
    }
    __builtin_amdgcn_s_barrier();
    quad(1);
    __builtin_amdgcn_s_barrier();
  };
  for (int kt = 0; kt < nk; kt += 3) {
    ktile(kt, 0);
    if (kt + 1 < nk) ktile(kt + 1, 1);
    if (kt + 2 < nk) ktile(kt + 2, 2);
  }
  if constexpr (NF == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the clamped tail loads must not outlive the workgroup's LDS
  if (wr == 0) __builtin_amdgcn_s_barrier();

  if constexpr (SILU) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = t0 + wc * 64 + j * 16 + l15;
      if (t >= T) continue;
#pragma unroll
      for (int i = 0; i < HT; ++i) {
        const int m = so.silu_c0 + mt * (16 * MT) + wr * (16 * HT) + i * 16 + g * 4;
        float r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {  // the GEMM output is bf16 before SwiGLU (fused_proj.cu:57-62)
          const float sg = silu_f(bf16_round_f(acc[i][j][e]));
          r[e] = (so.silu_round ? bf16_round_f(sg) : sg) * bf16_round_f(acc[i + HT][j][e]);
        }
        if (m + 3 < silu_cols_end(so)) {
          u32x2 o;
          o.x = pack_bf2(r[0], r[1]);
          o.y = pack_bf2(r[2], r[3]);
          *reinterpret_cast<u32x2*>(Y + (size_t)t * so.silu_I + m) = o;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (m + e < silu_cols_end(so)) Y[(size_t)t * so.silu_I + m + e] = f2bf(r[e]);
        }
      }
    }
    return;
  }
  if (part) {
    float* pz = part + (size_t)zslice * T * M;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = t0 + wc * 64 + j * 16 + l15;
      if (t >= T) continue;
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int m = m0 + wr * (16 * MT) + i * 16 + g * 4;
        if (m + 3 < M) {
          *reinterpret_cast<f32x4*>(pz + (size_t)t * M + m) = acc[i][j];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (m + e < M) pz[(size_t)t * M + m + e] = acc[i][j][e];
        }
      }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int t = t0 + wc * 64 + j * 16 + l15;
    if (t >= T) continue;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m = m0 + wr * (16 * MT) + i * 16 + g * 4;
      Half* dst = Y;
      int ld = M, mm = m, mlim = M;
      if (so.Y1) {
        const int b1 = so.M0 + so.M1, b2 = b1 + so.M2;
        if (m < so.M0) { ld = mlim = so.M0; }
        else if (m < b1) { dst = so.Y1; ld = mlim = so.M1; mm = m - so.M0; }
        else if (m < b2) { dst = so.Y2; ld = mlim = so.M2; mm = m - b1; }
        else { dst = so.Y3; ld = mlim = M - b2; mm = m - b2; }
      }
      if (mm + 3 < mlim) {
        u32x2 o;
        o.x = pack_bf2(acc[i][j][0], acc[i][j][1]);
        o.y = pack_bf2(acc[i][j][2], acc[i][j][3]);
        *reinterpret_cast<u32x2*>(dst + (size_t)t * ld + mm) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (mm + e < mlim) dst[(size_t)t * ld + mm + e] = f2bf(acc[i][j][e]);
      }
    }
  }
}

inline bool gemm128x256_ok(int M, int T, int K) { return (K % G256_BK) == 0 && K >= 128 && M >= 128 && T > 64; }

// plain (part == nullptr, ksplit == 1) or split-K (fp32 partials into part[ksplit][T][M]; the caller sums the slices)
inline bool gemm128x256_feed_on() {
  static const bool v = [] { const char* e = getenv("PEGAINFER_GEMM128X256_FEED"); return !(e && e[0] == '0'); }();
  return v;
}
template <bool SILU, int NF, int MT = 4>
inline void gemm128x256_launch_nf(const Half* W, const Half* X, Half* Y, int M, int T, int K, const SplitOut& so, float* part,
                                  int ksplit, int nk_slice, int m_tiles, int t_tiles, hipStream_t s) {
  static const bool once = [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&mfma_gemm128x256_kernel<SILU, NF, MT>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, kG128LdsBytes);
    return true;
  }();
  (void)once;
  mfma_gemm128x256_kernel<SILU, NF, MT><<<dim3(m_tiles * t_tiles, part ? ksplit : 1), 512 + NF * 64, kG128LdsBytes, s>>>(
      W, X, Y, M, T, K, m_tiles, t_tiles, so, part, nk_slice);
}
// 96-row tiles (MT = 3), plain un-split feeder form: see the kernel's header
inline void gemm96x256_launch(const Half* W, const Half* X, Half* Y, int M, int T, int K, SplitOut so, hipStream_t s) {
  const int t_tiles = ceil_div(T, G256_BT);
  so.w_nt = t_tiles == 1 && weights_nt_on();
  gemm128x256_launch_nf<false, 4, 3>(W, X, Y, M, T, K, so, nullptr, 1, 0, ceil_div(M - so.m_first, 96), t_tiles, s);
}
// SwiGLU form on 64-row tiles (MT = 2: 16 gate rows + their 16 up rows per wave row): the thin tail behind the 256 x 256 round
inline void gemm64x256_silu_launch(const Half* W, const Half* X, Half* Y, int M, int T, int K, SplitOut so, hipStream_t s) {
  const int t_tiles = ceil_div(T, G256_BT);
  so.w_nt = t_tiles == 1 && weights_nt_on();
  gemm128x256_launch_nf<true, 4, 2>(W, X, Y, M, T, K, so, nullptr, 1, 0, ceil_div(silu_cols_end(so) - so.silu_c0, 32), t_tiles, s);
}
inline void gemm128x256_launch(const Half* W, const Half* X, Half* Y, int M, int T, int K, SplitOut so, float* part,
                               int ksplit, int nk_slice, hipStream_t s) {
  const int t_tiles = ceil_div(T, G256_BT);
  so.w_nt = t_tiles == 1 && weights_nt_on();
  so.t_major = gemm_t_major(M, T, so);
  so.xcd_slices = part && ksplit > 1 && splitk_xcd_on();
  const bool feed = gemm128x256_feed_on();
  if (so.silu_I > 0) {   // SwiGLU form (un-split only): a tile = 64 gate rows + their 64 up rows
    const int m_tiles = ceil_div(silu_cols_end(so) - so.silu_c0, 64);
    if (feed) gemm128x256_launch_nf<true, 4>(W, X, Y, M, T, K, so, nullptr, 1, 0, m_tiles, t_tiles, s);
    else gemm128x256_launch_nf<true, 0>(W, X, Y, M, T, K, so, nullptr, 1, 0, m_tiles, t_tiles, s);
    return;
  }
  const int m_tiles = ceil_div(M - so.m_first, G128_BM);
  if (feed) gemm128x256_launch_nf<false, 4>(W, X, Y, M, T, K, so, part, ksplit, nk_slice, m_tiles, t_tiles, s);
  else gemm128x256_launch_nf<false, 0>(W, X, Y, M, T, K, so, part, ksplit, nk_slice, m_tiles, t_tiles, s);
}

}  // namespace pk
