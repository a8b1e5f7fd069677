// The W4A16 product for many batch rows (prefill, large serving batches):
//
//   y[b, m] = sum_g s[m, g] * (sum_{k in g} q[m, k] x[b, k]),
//
// q exact in fp16, every group's inner sum on the matrix cores in fp32, the
// scale applied to that sum in fp32 (folding it into fp16 weights would round
// every weight), one rounding to fp16 at the end. With kGateUp a wave's tile
// is 32 rows of Wg and the same 32 rows of Wu, and h = fp16(silu(g) * u).
//
// What bounds it. A SIMD issues one vector instruction in about 5 cycles,
// MFMAs among them, and a 32x32x16 MFMA keeps the matrix core for 32: up to
// six other instructions per MFMA go out in its shadow (two waves per SIMD:
// 34.4 cycles per MFMA with six, 32.3 with none; for 16x16x32, 17.4 with two
// and 26.2 with four, so the larger shape). A group of a 64 x 128 tile takes
// 64 MFMAs, 192 instructions to decode the weights, 128 to scale the sums and
// about 60 for LDS, loads and addresses: 6.05 per MFMA by the counters. So:
//   * a wave decodes its weights once for up to 128 batch rows, into 64
//     registers that serve all of them as MFMA operands, and shares x with
//     the waves beside it through LDS; the weights go through LDS only for
//     the transpose, private to the wave;
//   * the weights are the MFMA's columns, so a lane's 16 sums share a row of
//     W and one scale register;
//   * x and W reach LDS by buffer loads to LDS, three units of x in a ring,
//     the next group's weights during the current one, so no register waits
//     on memory;
//   * two waves per SIMD, out of phase, fill each other's decode. Two
//     workgroups of four waves per CU fall out of phase by themselves (28672 x
//     8192, B = 2048: 811 us against 870 for one workgroup of eight waves);
//     where a workgroup has eight waves, its second four lag by half a group.
// What is left is idle MFMA slots, not the clock: 28672 x 8192, B = 2048 takes
// 1.57 million cycles, of which the MFMAs fill 58% (a run with counters, 956 us:
// 1.65 GHz, 1010 TFLOP/s; without them 820-860 us, 1120-1170). A fp16 library
// product of that shape reaches 1270-1390 at 1.6 GHz, 76-83% of the slots.
//
// Measured (us, cold weights; before: the 16-row tiles of gemv_reuse_pfb or
// gemv_reuse_lds, and for gate/up those of gate_up_silu_tiles_lds):
//   M = 28672, K = 8192:  B = 2048 820 (1970)   B = 1000 466 (1002)  B = 128 70 (143)
//   M = K = 4096:         B = 1000 38 (82)      B = 256 16.2 (20.5)
//   M = 11008, K = 4096:  B = 512 60 (124)      B = 128 22.8 (37.7)  B = 32 13.5 (14.1)
//   M = 5000, K = 4224:   B = 512 36 (110)      B = 128 16.6 (33.1)  B = 17 8.6 (11.7)
//   gate/up, I = 11008, H = 4096: B = 512 113 (365)  B = 64 22.5 (46.8)
//   gate/up, I = 28672, H = 8192: B = 256 240 (1012) B = 32 71 (130)
#pragma once

#include "dk_mlp.hpp"

namespace dk {

typedef float f16_t __attribute__((ext_vector_type(16)));

// The 8 nibbles of a word as fp16 in their natural order: byte j holds
// weights 2j (low nibble) and 2j + 1 (high). The byte goes to both halves
// (v_perm), the low half keeps its low nibble and the high half its high
// one, XORed into 1024 + u and 1024 + 16 u (one v_bitop3), and one packed
// fma with a factor and an addend per half makes both exact: 12 operations
// for 8 weights, where unpack_word takes 9 but leaves the pairs 16 bits apart
// (0,4)(1,5)(2,6)(3,7), which x would have to be shuffled to match.
__device__ __forceinline__ h8_t unpack_word_natural(uint32_t w) {
  const h2_t mul = {(_Float16)1.0f, (_Float16)0.0625f};
  const h2_t add = {(_Float16)-1032.0f, (_Float16)-72.0f};
  h8_t r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t sel = 0x0c000c00u + 0x00010001u * j;
    asm("" : "+s"(sel));  // the selectors stay in SGPRs: vector registers are short
    const uint32_t p = __builtin_amdgcn_perm(0u, w, sel);
    const h2_t q = as_h2((p & 0x00F0000Fu) ^ 0x64806408u) * mul + add;
    r[2 * j] = q[0];
    r[2 * j + 1] = q[1];
  }
  return r;
}

typedef const __attribute__((address_space(3))) h8_t* lds_h8_ptr;
typedef const __attribute__((address_space(3))) uint32_t* lds_u32_ptr;
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(3))) u32x4_t* lds_u4_ptr;

__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(uintptr_t)(lds_void_ptr)p;
}

// Raw buffer descriptor of `bytes` bytes at `base`, in SGPRs.
__device__ __forceinline__ u32x4_t gemm_rsrc(const char* base, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  u32x4_t r;
  r[0] = (uint32_t)a;
  r[1] = (uint32_t)(a >> 32) & 0xffffu;
  r[2] = bytes;
  r[3] = 0x00020000u;
  return r;
}

// Buffer loads to LDS as single asm blocks: the compiler then counts neither
// them in vmcnt nor their LDS writes, and the kernel's own waits (exact
// counts) and "memory" clobbers order them; nothing is loaded into a
// register. m0 holds the wave's LDS byte address; lane l's 16 bytes land at
// 16 l past it, a zero-extended halfword at 4 l. The five wait states cover
// an SGPR of the descriptor that a vector instruction wrote just before (the
// compiler does not look into the block). m0 is a clobber: without it the
// compiler keeps an address that it has in m0 for a builtin load past the
// block. It warns that m0 is a reserved register, one that it does not save.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <int kOffset>
__device__ __forceinline__ void dma16(uint32_t lds, uint32_t voff, u32x4_t r) {
  asm volatile(
      "s_add_u32 m0, %0, %3\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds),
      "v"(voff), "s"(r), "i"(kOffset)
      : "memory", "scc", "m0");
}
template <int kOffset>
__device__ __forceinline__ void dma2(uint32_t lds, uint32_t voff, u32x4_t r) {
  asm volatile(
      "s_add_u32 m0, %0, %3\n\ts_nop 3\n\tbuffer_load_ushort %1, %2, 0 offen lds" ::"s"(lds),
      "v"(voff), "s"(r), "i"(kOffset)
      : "memory", "scc", "m0");
}
#pragma clang diagnostic pop

// Waits until at most N of the wave's loads are in flight and its LDS reads
// are done, and, where waves share the staged x, for the others: every wave's
// part of the unit has then arrived, and the unit before it has been read.
template <int N, bool kBarrier>
__device__ __forceinline__ void gemm_wait() {
  if constexpr (kBarrier)
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"(N) : "memory");
  else
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(N) : "memory");
}

// A stream is the WMN waves that share x: the same batch rows and groups.
// kGroups: weights are loaded so many groups ahead.
template <int kWaves, int WMN, int MT>
struct GemmLds {
  static constexpr int kStreams = kWaves / WMN;
  static constexpr int kUnit = WMN * 256;  // uint4 of a stream's unit of x
  static constexpr int kRing = 3;          // units staged
  uint4 x[kRing][kStreams * kUnit];
  static constexpr int kGroups = MT == 1 ? 2 : 1;
  uint4 w[kGroups][kWaves][MT * 128];  // a wave's rows of one group
  uint32_t s[kGroups][kWaves][MT][64];
};

// WMN waves side by side (MT row tiles of 32 each; for gate/up one of Wg and
// one of Wu) by WKN waves that take every WKN-th group of K; each wave 32 NBT
// batch rows. With MT = 1, for batches whose grid would leave CUs idle or a
// step waiting for HBM, the weights are half as many, so two groups of them
// are staged (5000 x 4224, B = 17: 8.6 us against 11.8 for MT = 2). x is
// staged in units: with WMN > 1 of 16 WMN batch rows by a group, with WMN = 1,
// where no other wave reads them and no barrier is needed, of 32 rows by half
// a group. P units make a group; unit u + 2 is issued during unit u.
template <int WMN, int WKN, int NBT, int MT, bool kGateUp>
__global__ __launch_bounds__(WMN * WKN * 64, 2) void gemm_w4(
    const uint4* __restrict__ w0p, const uint16_t* __restrict__ s0p, const uint4* __restrict__ w1p,
    const uint16_t* __restrict__ s1p, const uint4* __restrict__ x4, uint16_t* __restrict__ y, int M,
    int K, int B) {
  constexpr int kWaves = WMN * WKN;
  using Lds = GemmLds<kWaves, WMN, MT>;
  constexpr bool kShared = WMN > 1;
  constexpr int kHalves = kShared ? 1 : 2;       // units per b tile
  constexpr int kTiles = kShared ? WMN / 2 : 1;  // 32-row b tiles per unit
  constexpr int kSteps = 8 / kHalves;            // MFMA steps of a tile in a unit
  constexpr int P = NBT * kHalves / kTiles;      // units per group
  constexpr int kNx = 4;                         // x loads per wave and unit
  constexpr int kAhead = Lds::kRing - 1;         // units issued ahead
  constexpr int kNw = 3 * MT;                    // weight and scale loads per wave and group
  constexpr int kRows = kGateUp ? 32 : 32 * MT;  // output rows per wave
  static_assert(MT == 2 || (!kShared && !kGateUp), "one m tile: private x, one matrix");
  static_assert(kAhead <= P && kNx * WMN * kHalves == 8 * kTiles, "load counts");
  using std::integral_constant;
  __shared__ Lds lds;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % WMN;
  const int kk = wave / WMN;  // the stream: one part of K
  const int lag = kShared && kWaves == 8 ? (wave >> 2) * (P / 2) : 0;

  // Batch tiles fastest: workgroups side by side on an XCD share weights.
  const int tb = (B + 32 * NBT - 1) / (32 * NBT);
  const int id = xcd_contiguous_block(blockIdx.x, gridDim.x);
  const int mtile = __builtin_amdgcn_readfirstlane(id / tb);
  const int m0 = mtile * (WMN * kRows) + wm * kRows;
  const int b0 = (id - mtile * tb) * (32 * NBT);
  const int G = K >> 7;
  const int its = (G - kk + WKN - 1) / WKN;  // groups kk, kk + WKN, ...

  // x: load i covers 4 rows of the unit (8 half rows), the stream's waves one
  // after the other; lane l the slot l % 16 of row l / 16 (l % 8 of l / 8),
  // which holds the chunk that the swizzle of frag() below puts there.
  const uint32_t xl = lds_address(&lds.x[0][kk * Lds::kUnit + wm * kNx * 64]);
  constexpr uint32_t kSlot = Lds::kStreams * Lds::kUnit * 16;
  const uint32_t xrow = 2u * (uint32_t)K;
  constexpr int kLoadRows = 4 * kHalves;
  const uint32_t xoff = kHalves == 1
                            ? (lane >> 4) * xrow + (((lane & 15) ^ (lane >> 4)) << 4)
                            : (lane >> 3) * xrow + (((lane & 7) ^ (lane >> 4)) << 4);
  const int xrow0 = b0 + wm * kNx * kLoadRows;
  const int xleft = __builtin_amdgcn_readfirstlane(B - xrow0);
  const int gfirst = min(kk, G - 1);
  const char* xg = reinterpret_cast<const char*>(x4) + (size_t)xrow0 * xrow + (size_t)gfirst * 256;
  auto x_rsrc = [&](const char* base, int p) {
    const int row = p / kHalves * 32 * kTiles;
    return gemm_rsrc(base + (size_t)row * xrow + p % kHalves * 128, max(0, xleft - row) * xrow);
  };
  auto issue_x = [&](u32x4_t r, uint32_t lds0, auto iv) {
    constexpr int i = decltype(iv)::value;
    uint32_t xo = xoff;
    asm volatile("" : "+v"(xo));  // the offsets are recomputed: registers are short
    dma16<i * 1024>(lds0, (xo ^ (64u * (kHalves == 1 ? i : i % 2))) + i * kLoadRows * xrow, r);
  };
  auto issue_x_all = [&](u32x4_t r, uint32_t lds0) {
    issue_x(r, lds0, integral_constant<int, 0>());
    issue_x(r, lds0, integral_constant<int, 1>());
    issue_x(r, lds0, integral_constant<int, 2>());
    issue_x(r, lds0, integral_constant<int, 3>());
  };
  // Weights: load i covers rows 16 i .. + 15 of the wave's, lane l the
  // slot l % 4 of row l / 4, which holds chunk (l % 4) ^ (row / 4 % 4).
  const uint32_t wl = lds_address(&lds.w[0][wave][0]);
  const uint32_t sl = lds_address(&lds.s[0][wave][0][0]);
  constexpr uint32_t kWSlot = kWaves * MT * 2048, kSSlot = kWaves * MT * 256;
  const uint32_t wrow = (uint32_t)K / 2;
  const uint32_t woff = (lane >> 2) * wrow + (((lane & 3) ^ ((lane >> 4) & 3)) << 4);
  const int wleft = __builtin_amdgcn_readfirstlane(min(kRows, M - m0));
  const int row1 = kGateUp ? 0 : 32;
  const uint32_t left0 = max(0, wleft), left1 = max(0, wleft - row1);
  const char* wg0 = reinterpret_cast<const char*>(w0p) + (size_t)m0 * wrow + (size_t)gfirst * 64;
  const char* wg1 = reinterpret_cast<const char*>(kGateUp ? w1p : w0p) +
                    (size_t)(m0 + row1) * wrow + (size_t)gfirst * 64;
  const char* sg0 = reinterpret_cast<const char*>(s0p) + ((size_t)m0 * G + gfirst) * 2;
  const char* sg1 = reinterpret_cast<const char*>(kGateUp ? s1p : s0p) +
                    ((size_t)(m0 + row1) * G + gfirst) * 2;
  uint32_t wbuf = 0;  // the buffer of the group at hand (two with one m tile)
  auto issue_w = [&](auto iv) {  // i < 2 MT: weights, else scales
    constexpr int i = decltype(iv)::value;
    constexpr int t = i < 2 * MT ? i / 2 : i - 2 * MT;
    if constexpr (i < 2 * MT) {
      uint32_t wo = woff;
      asm volatile("" : "+v"(wo));
      dma16<i * 1024>(wl + wbuf * kWSlot, i % 2 ? wo + 16 * wrow : wo,
                      gemm_rsrc(t ? wg1 : wg0, (t ? left1 : left0) * wrow));
    } else {
      uint32_t r = threadIdx.x;
      asm volatile("" : "+v"(r));
      dma2<t * 256>(sl + wbuf * kSSlot, (r & 31) * (uint32_t)G * 2,
                    gemm_rsrc(t ? sg1 : sg0, (t ? left1 : left0) * (2 * G)));
    }
  };

  // tot[i][j]: the sums of the wave's m tile i and b tile j (32 x 32), this
  // lane's column lane % 32 and rows 8 (v / 4) + 4 (lane / 32) + v % 4.
  f16_t tot[MT][NBT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NBT; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) tot[i][j][v] = 0.0f;

  const int r32 = lane & 31;
  const int half = lane >> 5;
  // A row's 16 chunks (words) of a group: whole rows, half h of the wave takes
  // 8 h + t, t = 0..7, one per MFMA, and chunk c of row r sits in slot
  // c ^ (r % 16); half rows, 2 t + h, in slot c ^ (r / 2 % 8).
  const uint32_t xread =
      lds_address(&lds.x[0][kk * Lds::kUnit]) +
      (kHalves == 1 ? r32 * 256 + (((8 * half) ^ (r32 & 15)) << 4)
                    : r32 * 128 + ((half ^ ((r32 >> 1) & 7)) << 4));
  const uint32_t wread =
      wl + r32 * 64 +
      (kHalves == 1 ? ((2 * half) ^ ((r32 >> 2) & 3)) * 16 : ((r32 >> 2) & 3) * 16 + half * 4);
  // Words t = 4 n .. 4 n + 3 of the wave's tile i.
  auto read_words = [&](uint32_t (&a)[8], int i, int n) {
    if constexpr (kHalves == 1) {
      const u32x4_t v =
          *(lds_u4_ptr)(uintptr_t)((wread ^ (16u * n)) + wbuf * kWSlot + i * 2048);
      a[4 * n] = v.x, a[4 * n + 1] = v.y, a[4 * n + 2] = v.z, a[4 * n + 3] = v.w;
    } else {
#pragma unroll
      for (int t = 4 * n; t < 4 * n + 4; ++t)
        a[t] = *(lds_u32_ptr)(uintptr_t)((wread ^ (16u * (t / 2))) + wbuf * kWSlot + i * 2048 +
                                         t % 2 * 8);
    }
  };

  // Past a row's end the last group's loads are repeated and not used.
  auto next_w = [&](bool more) {
    wg0 += more ? WKN * 64 : 0;
    wg1 += more ? WKN * 64 : 0;
    sg0 += more ? WKN * 2 : 0;
    sg1 += more ? WKN * 2 : 0;
  };
  auto issue_w_all = [&] {
    issue_w(integral_constant<int, 0>());
    issue_w(integral_constant<int, 1>());
    issue_w(integral_constant<int, 2>());
    if constexpr (MT == 2) {
      issue_w(integral_constant<int, 3>());
      issue_w(integral_constant<int, 4>());
      issue_w(integral_constant<int, 5>());
    }
  };
  issue_w_all();
  if constexpr (Lds::kGroups == 2) {
    next_w(1 < its);
    wbuf = 1;
    issue_w_all();
    wbuf = 0;
  }
#pragma unroll
  for (int u = 0; u < kAhead; ++u) issue_x_all(x_rsrc(xg, u), xl + u * kSlot);
  for (int d = 0; d < lag; ++d) asm volatile("s_barrier" ::: "memory");
  // A tile's sums of the group wait in acc for the next tile's loads: they
  // are scaled and added to tot while those arrive.
  f16_t acc[MT] = {};
  float sc[MT] = {};
  auto add_scaled = [&](f16_t& sum, int i) {
#pragma unroll
    for (int v = 0; v < 16; ++v) sum[v] = __builtin_fmaf(acc[i][v], sc[i], sum[v]);
    asm volatile("" : "+v"(sum));  // pins the order of the steps
  };
  uint32_t slot = 0;  // byte offset of the unit's slot
  for (int it = 0; it < its; ++it) {
    next_w(it + Lds::kGroups < its);
    const char* xnext = xg + (it + 1 < its ? WKN * 256 : 0);
    h8_t wq[MT][8];
    uint32_t a[MT][8];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      // In flight beyond this unit's x: that of the next units, and the next
      // group's weights if they were issued after it.
      if (p >= 1 && p < kAhead)
        gemm_wait<(kAhead - 1) * kNx + kNw, kShared>();
      else
        gemm_wait<(kAhead - 1) * kNx, kShared>();
      constexpr int kRing = 3;  // x fragments in flight
      uint32_t xa0 = xread + slot;
      asm volatile("" : "+v"(xa0));
      auto frag = [&](int s) {
        return *(lds_h8_ptr)(uintptr_t)((xa0 ^ (16u * kHalves * (s % kSteps))) +
                                        8192u * (s / kSteps));
      };
      h8_t xf[kRing];
#pragma unroll
      for (int s = 0; s < kRing - 1; ++s) xf[s] = frag(s);
      float next_sc[MT];
      if (p == 0) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          read_words(a[i], i, 0);
          uint32_t r = threadIdx.x;
          asm volatile("" : "+v"(r));
          next_sc[i] = h2f((uint16_t) * (lds_u32_ptr)(uintptr_t)(sl + wbuf * kSSlot + i * 256 +
                                                                 (r & 31) * 4));
        }
      }
      if (p % kHalves == 0) {
        const int prev = ((p + P - 1) % P / kHalves + 1) * kTiles - 1;
#pragma unroll
        for (int i = 0; i < MT; ++i) add_scaled(tot[i][prev], i);
      }
      if (p == 0) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          wq[i][0] = unpack_word_natural(a[i][0]);
          sc[i] = next_sc[i];
        }
      }
      const uint32_t ahead = xl + (slot == 0 ? kAhead * kSlot : slot - kSlot);
      const u32x4_t xr = x_rsrc(p + kAhead < P ? xg : xnext, (p + kAhead) % P);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < kSteps * kTiles; ++s) {
        const int t = s % kSteps + p % kHalves * kSteps;  // of the tile's eight
        if (s + kRing - 1 < kSteps * kTiles) xf[(s + kRing - 1) % kRing] = frag(s + kRing - 1);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          if (t == 0 && s > 0) add_scaled(tot[i][p * kTiles + s / kSteps - 1], i);
          const f16_t zero = {};
          acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[s % kRing], wq[i][t],
                                                          t ? acc[i] : zero, 0, 0, 0);
          asm volatile("" : "+v"(acc[i]));
          // The loads and the rest of the decode go out between the MFMAs.
          if (p < kHalves && s < kSteps && t < 7) wq[i][t + 1] = unpack_word_natural(a[i][t + 1]);
          if (p == 0 && s == 0) read_words(a[i], i, 1);
          // Slots of the first loads; two loads to a slot with one m tile.
          const int n = (s * MT + i) * (3 - MT);
          constexpr int kW = kHalves == 1 ? 6 : 2;
          const int kX = kHalves == 1 ? 12 : p == 0 ? 4 : MT == 2 ? 1 : 0;
#define DK_AT(first, i) (n <= (first) + (i) && (first) + (i) < n + 3 - MT)
          if (p == 0) {
            // The group's words have left the buffer that these loads take.
            if (n == kW) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (DK_AT(kW, 0)) issue_w(integral_constant<int, 0>());
            if (DK_AT(kW, 1)) issue_w(integral_constant<int, 1>());
            if (DK_AT(kW, 2)) issue_w(integral_constant<int, 2>());
            if constexpr (MT == 2) {
              if (DK_AT(kW, 3)) issue_w(integral_constant<int, 3>());
              if (DK_AT(kW, 4)) issue_w(integral_constant<int, 4>());
              if (DK_AT(kW, 5)) issue_w(integral_constant<int, 5>());
            }
          }
          if (DK_AT(kX, 0)) issue_x(xr, ahead, integral_constant<int, 0>());
          if (DK_AT(kX, 1)) issue_x(xr, ahead, integral_constant<int, 1>());
          if (DK_AT(kX, 2)) issue_x(xr, ahead, integral_constant<int, 2>());
          if (DK_AT(kX, 3)) issue_x(xr, ahead, integral_constant<int, 3>());
#undef DK_AT
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      slot = slot == kAhead * kSlot ? 0 : slot + kSlot;
    }
    xg = xnext;
    if constexpr (Lds::kGroups == 2) wbuf ^= 1;
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) add_scaled(tot[i][NBT - 1], i);
  if constexpr (kShared) {
    // Every wave meets the same barriers: those of a group it has not, and the
    // half group by which the other waves lag.
    const int rest = ((G + WKN - 1) / WKN - its) * P + (kWaves == 8 ? P / 2 - lag : 0);
    for (int d = 0; d < rest; ++d) asm volatile("s_barrier" ::: "memory");
  }
  gemm_wait<0, true>();

  // The sums go through LDS, as many batch rows at a time as fit, where the K
  // parts meet (added in order) and from where rows leave 8 columns to a lane.
  // In every other four rows the halves of the columns (with one m tile, the
  // rows of a pair) are swapped, so that the two halves of a wave's store take
  // different banks. A wave without other K
  // parts reads only its own, with no barrier.
  float* red = reinterpret_cast<float*>(&lds);
  constexpr int kAtOnce = WKN > 1 && NBT == 4 ? 2 : 1;  // 32-row b tiles
  constexpr int kCols = 32 * MT, kTile = 32 * kCols;
  static_assert(kWaves * kAtOnce * kTile * 4 <= sizeof(Lds), "room for the sums");
  constexpr int kPerRow = kRows / 8;  // 8-column pieces of an output row
  constexpr int kPieces = 32 * kAtOnce * kPerRow / WKN;
  const bool wide = M % 8 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
#pragma unroll
  for (int j = 0; j < NBT; j += kAtOnce) {
    float* mine = red + wave * kAtOnce * kTile + r32 + half * (4 * kCols);
    float* const put[2] = {mine + half * 32, mine - half * 32 + (MT == 2 ? 32 : 0)};
    if (WKN > 1 && j > 0) __syncthreads();
#pragma unroll
    for (int d = 0; d < kAtOnce; ++d)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          put[MT == 2 ? i : v % 2][d * kTile + (8 * (v / 4) + v % 4) * kCols] = tot[i][j + d][v];
    if constexpr (WKN > 1)
      __syncthreads();
    else
      wave_lds_sync();
#pragma unroll
    for (int u = 0; u < (kPieces + 63) / 64; ++u) {
      const int piece = kk * kPieces + u * 64 + lane;
      const int row = piece / kPerRow, c8 = piece % kPerRow;
      const int b = b0 + 32 * j + row, m = m0 + 8 * c8;
      const int swap = row & 4;
      const int at = MT == 2 ? row * kCols : (row ^ (swap >> 2)) * kCols;
      if ((kPieces < 64 && lane >= kPieces) || b >= B) continue;
      const float* from = red + wm * kAtOnce * kTile + at;
      auto sum = [&](int c, float (&out)[8]) {
#pragma unroll
        for (int q = 0; q < WKN; ++q) {
          const float4* f = reinterpret_cast<const float4*>(from + q * (WMN * kAtOnce * kTile) +
                                                            8 * (MT == 2 ? c ^ swap : c));
          const float part[8] = {f[0].x, f[0].y, f[0].z, f[0].w, f[1].x, f[1].y, f[1].z, f[1].w};
#pragma unroll
          for (int e = 0; e < 8; ++e) out[e] = q ? out[e] + part[e] : part[e];
        }
      };
      float a[8];
      sum(c8, a);
      if constexpr (kGateUp) {
        float up[8];
        sum(c8 + 4, up);
#pragma unroll
        for (int e = 0; e < 8; ++e) a[e] = silu_f32(a[e]) * up[e];
      }
      uint16_t* to = y + (size_t)b * M + m;
      if (wide) {
        if (m < M) {
          h8_t o;
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = (_Float16)a[e];
          *reinterpret_cast<h8_t*>(to) = o;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (m + e < M) to[e] = f2h(a[e]);
      }
    }
    if constexpr (WKN == 1) wave_lds_sync();
  }
}

}  // namespace dk
