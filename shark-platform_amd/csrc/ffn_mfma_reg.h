// Projection for some dozen token rows per expert: weights go from memory through registers into the matrix cores, token rows through LDS.
//
// The streaming kernel (ffn_skinny.hip) reads the token rows from L2 once per 16 or 32 weight rows and has few wavefronts in flight
// where a down projection has few items; the prefill kernel (ffn_mfma_ws.hip) passes every weight through LDS behind one barrier per 64
// reduction elements, whose loaders set the pace of a unit whatever its rows.  Here a workgroup of eight wavefronts (one per CU) takes
// 256 weight rows x up to 64 token rows: a wavefront owns two 16-row weight tiles (GATEUP: gate and up of the same features), converts
// them in its own registers into MFMA operands and multiplies them with all token rows, which it reads from LDS.  No weight passes
// through LDS and no weight is converted twice.
//
//   chunk     256 reduction elements.  Weights: three register sets, requested three chunks ahead piece by piece as a set's registers
//             come free; token rows: four LDS stages, filled three chunks ahead by direct loads, one barrier per chunk.  At a barrier
//             the loads of two chunks could be in flight; the compiler's wait for the weights, which does not count the token loads,
//             leaves 2 NTJ fewer (of 16 + 8 in a Q4_1 unit of two tiles and 64 rows, of 8 + 8 in a half unit).
//   step      32 elements: the MFMAs of step s, the conversion of the weights of step s + 1 and the LDS reads of its token fragments
//             are interleaved (the next chunk's first step included, so the barrier does not empty the matrix pipe).
//   wide unit the same with up to 96 token rows (template argument MT, 16-row token tiles): two register sets and three LDS stages of 48 KB.
//             An expert with 65 to 96 rows converts its weights once instead of twice (60 rows per expert, 8 x 4096 x 14336, Q4_1 bf16:
//             gate/up 259 -> 218 us, down 137 -> 110; 300 rows of [14336, 4096] in four tiles of 75: 61 -> 53 us).  112 rows spill; units
//             of 128 weight rows x 160 token rows (half as many conversions, twice the operand reads) gave 49 and 46 us for those 300
//             rows in Q4_1 bf16 and Q8_0 fp16, where this one takes 53 and 48, and lost elsewhere.
//             A launch of several experts takes units of up to 64 rows here instead where they need no more rounds (fewer_rows).
//   half unit the units after the last whole round over the workgroups are cut into two of 128 weight rows if the halves fit one round
//             (a tile per wavefront): 8 experts of [4096, 14336] are 128 units, 256 halves.
//
// What bounds it: at 25 rows per expert HBM (gate/up of 8 x 4096 x 14336, Q8_0 fp16 169 us = 5.9 TB/s, Q4_1 fp16 124 us = 4.7 TB/s), in
// bf16 the vector instructions of the exact fp16 -> bf16 conversion (161 us); with more rows the issue slots of a SIMD, which its two
// wavefronts' conversions and MFMAs share (51 rows 191, 163 and 190 us): a vector instruction takes 4 cycles of a SIMD (and a wavefront
// issues one every 8), a 16 x 16 x 32 MFMA 8 beside the 16 of the matrix pipe, an operand read 8, which for a Q4_1 bf16 chunk with 64 rows
// is 5100 of the 5500 to 5900 cycles measured; and the requests of the CU's vector-memory path: leaving out the
// scale loads, 256 bytes each, gave 7-10 %.  Tried without gain: workgroups of four wavefronts, two per
// CU (token rows cross L2 twice: down 58 -> 80 us); sixteen wavefronts of one tile (128 registers: spills); the loads of a unit running
// ahead into the next one (5-10 % for units of 8 chunks, 0-15 % slower for longer ones: the registers it needs are the third weight set).
#pragma once
#include "ffn_mfma_common.h"

namespace stmoe {

template <int V> struct RgInt { static constexpr int value = V; };

struct RegArgs {
  GemmParams p;
  int n_tiles;      // units per token tile: 256 weight rows each
  int wgs_per_xcd;  // grid size / 8
  int tile_rows;    // most token rows of a unit, at most 16 MT
  int fewer_rows;   // wide kernel: most token rows of a unit where the launch takes no more rounds with so many (0: always tile_rows)
};

// Register sets of weights, LDS stages of token rows in a kernel whose units have up to `mt` 16-row token tiles.
static constexpr int reg_sets(int mt) { return mt <= 4 ? 3 : 2; }
static constexpr int reg_stages(int mt) { return mt <= 4 ? 4 : 3; }
// Whether the refills of a register set in the chunks after the last whole round over the sets, which nobody reads, are kept.
static constexpr bool reg_keeps_refills(int mt) { return mt > 4; }

// Vector-memory instructions that may be in flight when the token rows of the next chunk have to be there: what a wavefront issues after
// them, `x` token loads and `w` weight loads a chunk.
static constexpr int reg_wait(int mt, int x, int w) { return (reg_stages(mt) - 2) * x + (reg_sets(mt) - 1) * w; }
// Whether every chunk's token rows have landed where they are read, for reductions of 1 to 9 chunks, in the order in which the kernel
// issues its loads.  Loads return in the order of their issue.  At a barrier all but reg_wait() of those issued have landed, and the
// weights of the chunk, which the compiler waits for at touch().  Refills that nobody reads the compiler may drop, unless they are kept:
// they don't count as issued.
static constexpr bool reg_tokens_landed(int mt, int x, int w) {
  const int S = reg_sets(mt), D = reg_stages(mt);
  for (int chunks = 1; chunks <= 9; ++chunks) {
    int issued = 0, x_end[16] = {}, w_end[16] = {};
    w_end[0] = issued += w;
    for (int c = 0; c < D - 1; ++c) x_end[c] = issued += x;
    for (int c = 1; c < S; ++c) w_end[c] = issued += w;
    for (int c = 0; c <= chunks; ++c) {  // the barrier in front of chunk c, then what chunk c issues up to the next one
      const int landed = issued - reg_wait(mt, x, w) > w_end[c] ? issued - reg_wait(mt, x, w) : w_end[c];
      if (landed < x_end[c]) return false;
      x_end[c + D - 1] = issued += x;
      if (reg_keeps_refills(mt) || c < chunks / S * S) w_end[c + S] = issued += w;
    }
  }
  return true;
}

// A 16-row weight tile in the packed streaming order.  LOADS: load instructions per chunk.
template <int WF> struct RegTile;
template <> struct RegTile<WF_Q8_0_P> {
  static constexpr int LOADS = 5;
  const uint8_t *q, *d;
  __device__ __forceinline__ void init(const WeightView& w, int64_t row0, int64_t, int64_t kred) {
    q = w.qs + (row0 >> 4) * (kred >> 6) * 1024;
    d = w.d + (row0 >> 4) * (kred >> 8) * 256;
  }
};
template <> struct RegTile<WF_FP8_F32D_P> {
  static constexpr int LOADS = 4;
  const uint8_t* q;
  float dv;
  __device__ __forceinline__ void init(const WeightView& w, int64_t row0, int64_t e, int64_t kred) {
    q = w.qs + (row0 >> 4) * (kred >> 6) * 1024;
    dv = reinterpret_cast<const float*>(w.d)[w.d_count > 1 ? e : 0];
  }
};
template <> struct RegTile<WF_Q4_1_P> {
  static constexpr int LOADS = 4;
  const uint8_t *q, *d, *m;
  __device__ __forceinline__ void init(const WeightView& w, int64_t row0, int64_t, int64_t kred) {
    q = w.qs + (row0 >> 4) * (kred >> 7) * 1024;
    d = w.d + (row0 >> 4) * (kred >> 8) * 256;
    m = w.m + (row0 >> 4) * (kred >> 8) * 256;
  }
};

// A chunk of a weight tile as lane (n = lane % 16, g = lane / 16) holds it: row n, the elements given at `frag`.
template <int WF> struct RegData;
template <> struct RegData<WF_Q8_0_P> {
  u32x4_t q[4], d;
  // the part of chunk c that can be requested during MFMA step s, when the weights of step s + 1 are being converted
  __device__ __forceinline__ void load(const RegTile<WF_Q8_0_P>& t, int c, int lane, int s) {
    if (s & 1) q[s >> 1] = ld_stream16(t.q + (int64_t)c * 4096 + (s >> 1) * 1024 + lane * 16);
    if (s == 7) d = ld_stream16(t.d + (int64_t)c * 256 + (lane & 15) * 16);
  }
  __device__ __forceinline__ void touch() { asm volatile("" : "+v"(q[0]), "+v"(q[1]), "+v"(q[2]), "+v"(q[3]), "+v"(d)); }
  // MFMA step s covers elements 64 (s / 2) + 16 g + 8 (s % 2) .. + 7
  template <typename T> __device__ __forceinline__ u32x4_t frag(const RegTile<WF_Q8_0_P>&, int s, int g) const {
    const int i = s >> 1, h = s & 1;
    const half2_t dd = as_half2(__builtin_amdgcn_perm(d[i], d[i], (g & 2) ? 0x03020302u : 0x01000100u));
    const half2_t bias = {(f16_t)1152.0f, (f16_t)1152.0f};
    u32x4_t out;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint32_t u = q[i][2 * h + j] ^ 0x80808080u;
      const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);
      const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
      out[2 * j] = h2_to_T<T>(as_u32((as_half2(lo) - bias) * dd));
      out[2 * j + 1] = h2_to_T<T>(as_u32((as_half2(hi) - bias) * dd));
    }
    return out;
  }
};
template <> struct RegData<WF_FP8_F32D_P> {
  u32x4_t q[4];
  __device__ __forceinline__ void load(const RegTile<WF_FP8_F32D_P>& t, int c, int lane, int s) {
    if (s & 1) q[s >> 1] = ld_stream16(t.q + (int64_t)c * 4096 + (s >> 1) * 1024 + lane * 16);
  }
  __device__ __forceinline__ void touch() { asm volatile("" : "+v"(q[0]), "+v"(q[1]), "+v"(q[2]), "+v"(q[3])); }
  template <typename T> __device__ __forceinline__ u32x4_t frag(const RegTile<WF_FP8_F32D_P>& t, int s, int) const {
    const int i = s >> 1, h = s & 1;
    float f[8], f2[4];
    fp8x4_to_f32(q[i][2 * h], f2);
#pragma unroll
    for (int b = 0; b < 4; ++b) f[b] = f2[b];
    fp8x4_to_f32(q[i][2 * h + 1], f2);
#pragma unroll
    for (int b = 0; b < 4; ++b) f[4 + b] = f2[b];
    uint32_t o[4];
    scale8_pack<T>(f, t.dv, o);
    return (u32x4_t){o[0], o[1], o[2], o[3]};
  }
};
template <> struct RegData<WF_Q4_1_P> {
  u32x4_t q[2], d, m;
  __device__ __forceinline__ void load(const RegTile<WF_Q4_1_P>& t, int c, int lane, int s) {
    if ((s & 3) == 3) q[s >> 2] = ld_stream16(t.q + (int64_t)c * 2048 + (s >> 2) * 1024 + lane * 16);
    if (s == 7) {
      d = ld_stream16(t.d + (int64_t)c * 256 + (lane & 15) * 16);
      m = ld_stream16(t.m + (int64_t)c * 256 + (lane & 15) * 16);
    }
  }
  __device__ __forceinline__ void touch() { asm volatile("" : "+v"(q[0]), "+v"(q[1]), "+v"(d), "+v"(m)); }
  // MFMA step s covers elements 128 (s / 4) + 32 g + 8 (s % 4) .. + 7 (block 4 (s / 4) + g)
  template <typename T> __device__ __forceinline__ u32x4_t frag(const RegTile<WF_Q4_1_P>&, int s, int g) const {
    const int i = s >> 2, j = s & 3;
    const uint32_t sel = (g & 1) ? 0x03020302u : 0x01000100u;
    const uint32_t d0 = d[2 * i], d1 = d[2 * i + 1], m0 = m[2 * i], m1 = m[2 * i + 1];  // (values: a select of elements went through memory)
    const uint32_t dw = (g & 2) ? d1 : d0, mw = (g & 2) ? m1 : m0;
    Q4Scale sc;
    sc.dd = as_half2(__builtin_amdgcn_perm(dw, dw, sel));
    sc.mm = as_half2(__builtin_amdgcn_perm(mw, mw, sel));
    const half2_t n1024 = {(f16_t)-1024.0f, (f16_t)-1024.0f}, n64 = {(f16_t)-64.0f, (f16_t)-64.0f};
    sc.c1024 = sc.dd * n1024;
    sc.c64 = sc.dd * n64;
    uint32_t h[4];
    q4_dword_dequant_packed(q[i][j], sc, h);
    u32x4_t out;
#pragma unroll
    for (int b = 0; b < 4; ++b) out[b] = h2_to_T<T>(h[b]);
    return out;
  }
};
// 16-byte unit of a token row that lane group g needs for MFMA step s (rows of 256 elements = 32 units)
template <int WF> __device__ __forceinline__ int reg_x_unit(int s, int g) {
  return IsQ4<WF>::value ? 16 * (s >> 2) + 4 * g + (s & 3) : 8 * (s >> 1) + 2 * g + (s & 1);
}

// Unit u of LDS row r lives at unit u ^ reg_x_swizzle(r).  ds_read_b128 serves 16 lanes per cycle: four rows 4 q .. 4 q + 3 of each
// lane group g, with q = g ^ t in cycle t.  The units of the lane groups differ by 2 (1-byte formats: the row itself spreads them) or
// by 4 (nibbles: q must move to a value h(q) for which g ^ h(g ^ t) runs through all four values).
template <int WF> __device__ __forceinline__ int reg_x_swizzle(int r) {
  return IsQ4<WF>::value ? (r & 3) | ((r >> 1) & 4) | (((r << 1) ^ r) & 8) : r & 15;
}

template <typename T, int WF, int MODE, int MT>
__global__ void __launch_bounds__(512, 2)
grouped_mfma_reg_kernel(RegArgs args) {
  constexpr int BN = 256;
  extern __shared__ __align__(16) uint8_t lds_reg[];
  const GemmParams& p = args.p;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n_in = lane & 15, g = lane >> 4;
  const int xcd = blockIdx.x & 7, wg = blockIdx.x >> 3, wgs = args.wgs_per_xcd, n_tiles = args.n_tiles;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
      (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)lds_reg));
  const int nch = (int)(p.kred >> 8), last = nch - 1;

  // ---- the XCD's list: experts' token tiles (equal sizes, at most tile_rows rows) x feature tiles, an expert's token tiles of one
  // feature tile side by side
  int begin, rows;
  {
    const int off = big_lane_offsets(p);
    int end = __builtin_amdgcn_ds_bpermute(4 * (lane + 1), off);
    if (p.offsets && p.E == 64) end = lane == 63 ? p.offsets[64] : end;
    begin = off;
    rows = lane < p.E ? end - off : 0;
    if (!p.offsets) { begin = 0; rows = lane == 0 ? (int)p.fixed_rows : 0; }
  }
  int main = (rows + args.tile_rows - 1) / args.tile_rows;
  int main_end = wave_inclusive_sum(main);
  if constexpr (MT > 4) {
    if (args.fewer_rows > 0) {
      const int main2 = (rows + args.fewer_rows - 1) / args.fewer_rows, end2 = wave_inclusive_sum(main2);
      if (reg_half_rounds(__builtin_amdgcn_readlane(end2, 63) * n_tiles) <= reg_half_rounds(__builtin_amdgcn_readlane(main_end, 63) * n_tiles)) {
        main = main2;
        main_end = end2;
      }
    }
  }
  const int U = __builtin_amdgcn_readlane(main_end, 63) * n_tiles;
  const int f0 = (int)((int64_t)U * xcd / 8), f1 = (int)((int64_t)U * (xcd + 1) / 8), n_units = f1 - f0;
  const int rest = n_units % wgs;
  const int whole = 2 * rest <= wgs ? n_units - rest : n_units;  // the units after these are cut into two of 128 weight rows
  const int n_items = whole + 2 * (n_units - whole);

  for (int item = wg; item < n_items; item += wgs) {
    int u, half;
    if (item < whole) { u = f0 + item; half = -1; }
    else { u = f0 + whole + (item - whole) / 2; half = (item - whole) & 1; }
    const int e = __builtin_ctzll(__ballot(main_end * n_tiles > u));
    const int b = __builtin_amdgcn_readlane(begin, e), rws = __builtin_amdgcn_readlane(rows, e), m = __builtin_amdgcn_readlane(main, e);
    u -= (__builtin_amdgcn_readlane(main_end, e) - m) * n_tiles;
    const int ntile = u / m, s_tile = u - ntile * m;
    const int row_begin = b + (int)((int64_t)rws * s_tile / m), row_end = b + (int)((int64_t)rws * (s_tile + 1) / m);

    auto unit = [&](auto nt_tag, auto ntj_tag) {
      constexpr int NT = decltype(nt_tag)::value, NTJ = decltype(ntj_tag)::value;
      constexpr int S = reg_sets(MT), D = reg_stages(MT), WL = RegTile<WF>::LOADS * NT;
      constexpr int STAGE = 16 * NTJ * 512;
      static_assert(reg_tokens_landed(MT, NTJ, WL), "a chunk's token rows may be read before they have landed");
      // vector instructions that convert one weight fragment, for the issue order of a step
      constexpr int VALU_STEP = (WF == WF_FP8_F32D_P ? 14 : IsQ4<WF>::value ? 17 : 16) + (__is_same(T, f16_t) || WF == WF_FP8_F32D_P ? 0 : 12);
      // weight tiles of this wavefront
      RegTile<WF> wt[NT];
      int col[NT];  // first output feature of each tile
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if (MODE == MODE_GATEUP) {
          const bool up = NT == 2 ? t == 1 : wave >= 4;
          col[t] = ntile * (BN / 2) + (NT == 2 ? wave * 16 : half * 64 + (wave & 3) * 16);
          const WeightView& wv = up ? p.w1 : p.w0;
          wt[t].init(wv, (int64_t)e * wv.rows + col[t], e, p.kred);
        } else {
          col[t] = ntile * BN + (NT == 2 ? wave * 32 + t * 16 : half * 128 + wave * 16);
          wt[t].init(p.w0, (int64_t)e * p.w0.rows + col[t], e, p.kred);
        }
      }
      RegData<WF> w[S][NT];
      auto load_w = [&](RegData<WF>(&d)[NT], int c) {
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
          for (int t = 0; t < NT; ++t) d[t].load(wt[t], c, lane, s);
      };
      int pair[NTJ];  // sorted position, then the pair there
#pragma unroll
      for (int j = 0; j < NTJ; ++j) pair[j] = min(row_begin + 16 * j + 2 * wave + (lane >> 5), row_end - 1);
      if (p.perm) {
#pragma unroll
        for (int j = 0; j < NTJ; ++j) pair[j] = p.perm[pair[j]];
      }
      __builtin_amdgcn_sched_barrier(0);
      load_w(w[0], 0);
      __builtin_amdgcn_sched_barrier(0);
      uint32_t xoff[NTJ];
#pragma unroll
      for (int j = 0; j < NTJ; ++j) {
        const int lr = 16 * j + 2 * wave + (lane >> 5);
        const int64_t src = p.perm ? pair[j] / p.k_top : pair[j];
        xoff[j] = (uint32_t)((src * p.lda + (((lane & 31) ^ reg_x_swizzle<WF>(lr)) << 3)) * 2);
      }
      auto load_x = [&](int slot, int c) {
        const void* src = uniform_ptr(reinterpret_cast<const uint8_t*>(p.a) + (uint32_t)c * 512u);
#pragma unroll
        for (int j = 0; j < NTJ; ++j) vm_load16_to_lds<kBaseFromVector>(src, xoff[j], lds0 + slot * STAGE + (16 * j + 2 * wave) * 512);
      };
#pragma unroll
      for (int c = 0; c < D - 1; ++c) load_x(c, min(c, last));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 1; i < S; ++i) load_w(w[i], min(i, last));
      __builtin_amdgcn_sched_barrier(0);
      uint32_t xr[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) xr[q] = n_in * 512 + (((reg_x_unit<WF>(q, g) & 15) ^ reg_x_swizzle<WF>(n_in)) << 4);
      floatx4_t acc[NT][NTJ];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < NTJ; ++j) acc[t][j] = (floatx4_t){0.f, 0.f, 0.f, 0.f};
      int slot = 0, c = 0;
      u32x4_t af[2][NT], bf[NTJ];
      auto read_x = [&](int at_slot, int s, int j) __attribute__((always_inline)) {
        bf[j] = *reinterpret_cast<const u32x4_t*>(lds_reg + at_slot * STAGE + xr[s & 3] + (s >> 2) * 256 + j * 8192);
      };
      auto convert = [&](int set, const RegData<WF>(&wc)[NT], int s) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; ++t) af[set][t] = wc[t].template frag<T>(wt[t], s, g);
      };
      // The weights of chunk c + 1 and this wavefront's share of its token rows have landed, then everybody's.  The compiler adds its own
      // wait for the weights at touch(), which counts weight loads only: it lets (S - 1) WL be in flight, (D - 2) NTJ fewer than would do.
      auto arrive = [&](RegData<WF>(&wn)[NT]) __attribute__((always_inline)) {
        vm_wait<reg_wait(MT, NTJ, WL)>();
#pragma unroll
        for (int t = 0; t < NT; ++t) wn[t].touch();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      };
      auto chunk = [&](RegData<WF>(&wc)[NT], RegData<WF>(&wn)[NT]) __attribute__((always_inline)) {
        const int next = slot == D - 1 ? 0 : slot + 1, c_load = min(c + S, last);
        // A SIMD serves its older wavefront first: that one went through a chunk at its own pace (3500 cycles of 5900, Q4_1 bf16, 64 rows)
        // and waited, while the younger one finished alone, at half the rate at which a SIMD issues.  In bf16, where issue slots are what
        // runs out, the younger one goes first for half a chunk: 1 to 4 % (8 experts of 4096 x 14336 at 203 tokens 297 -> 292 us, 64 rows of
        // [14336, 4096] 28.7 -> 27.5).  In fp16 nothing (-1 to 1 %).  (Gate/up of Q8_0 in
        // the wide kernel has no register left for it: one would go to scratch memory, whose accesses the counted waits do not know.)
        constexpr bool HAND_OVER = !__is_same(T, f16_t) && !(MT > 4 && WF == WF_Q8_0_P && MODE == MODE_GATEUP);
        const bool hand_over = HAND_OVER && wave >= 4;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          if (s == 0 && hand_over) __builtin_amdgcn_s_setprio(1);
          if (s == 4 && hand_over) __builtin_amdgcn_s_setprio(0);
#pragma unroll
          for (int t = 0; t < NT; ++t) wc[t].load(wt[t], c_load, lane, s);
          if (s == 7) {
            __builtin_amdgcn_sched_barrier(0);
            arrive(wn);
            load_x(slot, min(c + D, last));
            __builtin_amdgcn_sched_barrier(0);
          }
          convert((s + 1) & 1, s == 7 ? wn : wc, (s + 1) & 7);
          // A token fragment's register is read again as soon as its MFMAs are issued, so that LDS has the other fragments'
          // MFMAs to answer in; the conversion of the next step's weights fills the gaps between them.
#pragma unroll
          for (int j = 0; j < NTJ; ++j) {
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t][j] = mfma16b<T>(af[s & 1][t], bf[j], acc[t][j]);
            read_x(s == 7 ? next : slot, (s + 1) & 7, j);
          }
#pragma unroll
          for (int j = 0; j < NTJ; ++j) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
              __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
              __builtin_amdgcn_sched_group_barrier(0x002, (VALU_STEP + NTJ - 1) / NTJ, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        slot = next;
        ++c;
      };
      arrive(w[0]);
      load_x(D - 1, min(D - 1, last));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NTJ; ++j) read_x(0, 0, j);
      convert(0, w[0], 0);
      __builtin_amdgcn_sched_barrier(0);
      // whole rounds over the register sets, then what is left: one loop without exits in its body, so that the compiler knows at
      // every wait how many weight loads are in flight
      for (int r = nch / S; r > 0; --r) {
#pragma unroll
        for (int i = 0; i < S; ++i) chunk(w[i], w[(i + 1) % S]);
      }
      const int left = nch % S;
      if (left > 0) chunk(w[0], w[1]);
      if constexpr (S > 2) {
        if (left > 1) chunk(w[1], w[2]);
      }
      vm_wait<0>();
      if constexpr (reg_keeps_refills(MT)) {
#pragma unroll
        for (int i = 0; i < S; ++i)
#pragma unroll
          for (int t = 0; t < NT; ++t) w[i][t].touch();
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // LDS is free for the next unit (and the exchange below)
      // (Q8_0 in bf16 has the longest conversion and two registers too few for the epilogue's addresses through the K loop: there the
      // lane's number is computed again.  The other instances have them to spare, and Q4_1 in fp16 would be 1 % slower for it.  The wide
      // kernel has none to spare at all: there the kernel's arguments are read again as well)
      const int out_lane = MT > 4 || (WF == WF_Q8_0_P && !__is_same(T, f16_t)) ? lane_again() : lane;
      auto kernarg = __builtin_amdgcn_kernarg_segment_ptr();
      if (MT > 4) asm volatile("" : "+s"(kernarg));
      const GemmParams& p = MT > 4 ? reinterpret_cast<const RegArgs*>((const void*)kernarg)->p : args.p;
      const int r0 = row_begin + (out_lane & 15), c0 = 4 * (out_lane >> 4);
      if constexpr (MODE == MODE_GATEUP) {
        if constexpr (NT == 1) {  // the up sums travel to the wavefront that has the gate sums
          if (wave >= 4) {
#pragma unroll
            for (int j = 0; j < NTJ; ++j)
              *reinterpret_cast<floatx4_t*>(lds_reg + (((wave & 3) * NTJ + j) * 64 + lane) * 16) = acc[0][j];
          }
          __syncthreads();
        }
        if (NT == 2 || wave < 4) {
          const FakeQuant fq = fq_scale(p);
          auto store = [&](auto act_tag) __attribute__((always_inline)) {
            constexpr int ACT = decltype(act_tag)::value;
#pragma unroll
            for (int j = 0; j < NTJ; ++j) {
              floatx4_t up;
              if constexpr (NT == 2) up = acc[1][j];
              else up = *reinterpret_cast<const floatx4_t*>(lds_reg + (((wave & 3) * NTJ + j) * 64 + lane) * 16);
              const int r = r0 + 16 * j;
              __builtin_amdgcn_sched_barrier(0);  // (one tile at a time: the accumulators leave no room for more)
              if (r < row_end) {
                const float gq[4] = {acc[0][j][0], acc[0][j][1], acc[0][j][2], acc[0][j][3]}, uq[4] = {up[0], up[1], up[2], up[3]};
                *reinterpret_cast<uint2*>(reinterpret_cast<T*>(p.out) + out_row(p, r) * p.ldo + col[0] + c0) = gateup_quad<T, ACT>(gq, uq, fq);
              }
            }
          };
          if (p.act == STMOE_ACT_SILU) store(EpiAct<STMOE_ACT_SILU>{});
          else store(EpiAct<STMOE_ACT_GELU_ERF>{});
        }
        if constexpr (NT == 1) __syncthreads();
      } else {
#pragma unroll
        for (int j = 0; j < NTJ; ++j) {
          const int r = r0 + 16 * j;
          if (r < row_end) {
            T* orow = reinterpret_cast<T*>(p.out) + out_row(p, r) * p.ldo + c0;
#pragma unroll
            for (int t = 0; t < NT; ++t)
              *reinterpret_cast<uint2*>(orow + col[t]) =
                  make_uint2(pack2<T>(acc[t][j][0], acc[t][j][1]), pack2<T>(acc[t][j][2], acc[t][j][3]));
          }
        }
      }
    };
    auto sized = [&](auto nt_tag) {
      const int tiles = (row_end - row_begin + 15) >> 4;
      if constexpr (MT > 4) {  // (units of up to 64 rows where they take no more rounds: 0.99 of the time of the narrow kernel's, with their three sets)
        if (tiles <= 4) unit(nt_tag, RgInt<4>{});
        else if (tiles == 5) unit(nt_tag, RgInt<5>{});
        else unit(nt_tag, RgInt<6>{});
      } else {
        if (tiles <= 1) unit(nt_tag, RgInt<1>{});
        else if (tiles == 2) unit(nt_tag, RgInt<2>{});
        else if (tiles == 3) unit(nt_tag, RgInt<3>{});
        else unit(nt_tag, RgInt<4>{});
      }
    };
    if (half < 0) sized(RgInt<2>{});
    else sized(RgInt<1>{});
  }
}

// `tile_rows`: most token rows of a unit.
template <typename T, int WF, int MODE, int MT>
static int launch_reg_m(const GemmParams& p, int tile_rows, int fewer_rows, hipStream_t st) {
  constexpr size_t lds_bytes = (size_t)reg_stages(MT) * 16 * MT * 512;
  static std::atomic<uint64_t> lds_ready{0};
  auto kern = grouped_mfma_reg_kernel<T, WF, MODE, MT>;
  if (int rc = reserve_lds(reinterpret_cast<const void*>(kern), lds_bytes, lds_ready, "mfma reg kernel")) return rc;
  const int n_tiles = (int)(MODE == MODE_GATEUP ? p.n_out / 128 : p.n_out / 256);
  kern<<<dim3(8 * kRegWgsPerXcd), 512, lds_bytes, st>>>(RegArgs{p, n_tiles, kRegWgsPerXcd, tile_rows, fewer_rows});
  return check_launch("grouped_mfma_reg");
}
template <int MT> static int launch_reg_mt(int act_dtype, int wtag, int mode, const GemmParams& p, int tile_rows, int fewer_rows, hipStream_t st) {
#define STMOE_REG(T, WF) (mode == MODE_GATEUP ? launch_reg_m<T, WF, MODE_GATEUP, MT>(p, tile_rows, fewer_rows, st) : launch_reg_m<T, WF, MODE_DOWN, MT>(p, tile_rows, fewer_rows, st))
  if (act_dtype == STMOE_F16) {
    if (wtag == WF_Q8_0_P) return STMOE_REG(f16_t, WF_Q8_0_P);
    if (wtag == WF_Q4_1_P) return STMOE_REG(f16_t, WF_Q4_1_P);
    return STMOE_REG(f16_t, WF_FP8_F32D_P);
  }
  if (wtag == WF_Q8_0_P) return STMOE_REG(bf16_t, WF_Q8_0_P);
  if (wtag == WF_Q4_1_P) return STMOE_REG(bf16_t, WF_Q4_1_P);
  return STMOE_REG(bf16_t, WF_FP8_F32D_P);
#undef STMOE_REG
}

}  // namespace stmoe
