// Prefill kernel for fp8 (e4m3fn) activations and packed fp8 tensor-scaled weights on the fp8 matrix cores.
//
// Neither operand needs a conversion on its way to the matrix cores, so no byte passes through a register before the
// MFMA reads it: every wavefront sends its share of a later stage global -> LDS directly (global_load_lds_dwordx4) and
// then only reads LDS operands and issues MFMAs.
//
//   256 x 256 workgroup tile (GATEUP: 128 gate + the same 128 up rows), 8 wavefronts of 128 weight rows x 64 token
//   rows, K stage 64 (one v_mfma_scale_f32_32x32x64_f8f6f4 deep), four stages of 16 KB weights + 16 KB tokens + 2 KB
//   ride-along tokens = 136 KB, loads issued three stages ahead (more stages do not fit), one barrier per stage.
//   order:   the two wavefronts of a SIMD take the halves of a stage in opposite orders.  Behind the barrier of stage s wavefronts 4-7
//            multiply stage s - 1, whose operands they have in registers, and then read those of stage s; wavefronts 0-3 first read
//            stage s and then multiply it.  So one of the two always has MFMAs to issue and the other one's LDS latency and load
//            issue (about 300 cycles each) pass beside the 512 cycles of MFMAs.  All of a stage's operands are in registers
//            before its first MFMA.
//   ride-along rows: an expert with a few rows more than c full tiles would need a partial tile for them, whose units load all
//            256 rows and leave most matrix cores idle; each full tile takes up to 32 of them along instead (tail_rows).
//   weights: a packed 1 KB piece (16 rows x 64 k; lane 16 g + n holds row n, k = 16 g .. + 15) lands in LDS as it is;
//            MFMA lane (r, h) supplies row r, samples 32 h .. 32 h + 31: pieces' units 2 h and 2 h + 1 of row r % 16,
//            16 consecutive lanes read 256 consecutive bytes.
//   tokens:  quantised rows, 64 bytes per stage; lane l of a load fetches the 16 bytes that belong at LDS position l
//            (row l / 4 of the load's 16 rows, the unit that x_unit maps to position l % 4), so that the gather and the
//            bank swizzle cost nothing; rows of a partial token tile are spread over the four token-row groups.  (A swizzle
//            under which two rows of a cycle shared their banks: 4 to 5 % more for the launches below.)
//   results: D[8 (i / 4) + 4 h + i % 4][r] (probed on the hardware: rows are the weight rows, columns the token rows);
//            both token blocks' operands (16 registers) and the four weight blocks' (32) are read once per wavefront and stage.
//   epilogue: the fp32 dot products of the quantised samples are scaled once by scale_x * d_w; the gate/up epilogue can
//            quantise the gated intermediate to e4m3fn for the down projection.
//   What bounds it: power.  4096 tokens, 8 experts of 4096 x 14336, gate/up + down, both sides traced on one box: both wavefronts of a SIMD in the
//            same order 1032 + 496 us of 1608 for the layer, in opposite orders 820 + 394 of 1301 (without the profiler 1499 and 1205; the rest
//            are router, dispatch, the rows' quantizer and combine).  Counters: 1.96 + 0.95 M cycles at 1.98 GHz, the matrix cores busy
//            0.48 of them; 1.35 + 0.66 M at 1.73 and 1.69, busy 0.69 and 0.71.  Over 1800 layers of 1 to 32 experts, 1024 to 6144 x 1024 to 16384,
//            8 % less time on average (nine took 2 to 10 % more in that run; 24 layers around the worst of them, 12 to 20 experts with one tile each, 5 to 10 % less).
//            An early build of it without any barrier took 16 % fewer
//            cycles at a clock 9 % lower.  A launch with nothing but the loads takes 590 + 300 us, 13 TB/s of the 34 that
//            these loads reach from L2 without a barrier per stage: one stage in flight is as fast as two, so not latency.
//            Tried and slower, because something other than MFMAs comes between a wavefront's MFMAs: the loads between them
//            (+15 %), a load's operands read as soon as the last MFMA has used the register (+15 %), both wavefronts late
//            (+15 %); loads issued in front of the LDS reads (+20 %) or while the early wavefronts' reads are under way (+7 %):
//            both go through the CU's one vector-memory path.
#include "ffn_mfma_common.h"

namespace stmoe {

typedef int intx8_t __attribute__((ext_vector_type(8)));
typedef float floatx16_t __attribute__((ext_vector_type(16)));
template <int V> struct F8Int { static constexpr int value = V; };

__device__ __forceinline__ intx8_t join8(const u32x4_t& lo, const u32x4_t& hi) {
  return (intx8_t){(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
}

// LDS unit (16 bytes) of a token row's unit u in a 64-byte stage row.  ds_read_b128 serves sixteen lanes a cycle, of lanes 0 .. 31 first the
// quads of lanes 0, 3, 5 and 6, then 1, 2, 4 and 7 (lanes 32 .. 63 likewise), and four rows cover all banks: rows of the four quads that
// read the same logical unit must find it at four different positions, which the lower two bits of the quad give.
__device__ __forceinline__ int x_unit(int row, int u) { return u ^ ((row >> 2) & 3); }

// vm_load16_to_lds for the first 16 lanes only (256 bytes), without a branch around it.  Every lane of the wavefront must be active.
__device__ __forceinline__ void f8_load16_to_lds_16_lanes(const void* base, uint32_t byte_off, uint32_t lds_addr) {
  lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);
  asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 exec, 0xffff\n\ts_nop %3\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(byte_off), "s"(base), "s"(lds_addr),
               "n"(kBaseFromVector)
               : "memory", "m0");
}

// A wavefront's share of a stage, four loads of a kilobyte: two weight pieces (w + w0, w + w1) and twice 16 token rows (x + x0, x + x1) to
// LDS address `lds_addr` and the kilobytes after it.  The n-th load's immediate offset of 1024 n counts for the LDS and for the global address.
__device__ __forceinline__ void f8_load_share(const void* w, uint32_t w0, uint32_t w1, const void* x, uint32_t x0, uint32_t x1, uint32_t lds_addr) {
  lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);
  asm volatile(
      "s_mov_b32 m0, %6\n\t"
      "s_nop %7\n\tglobal_load_lds_dwordx4 %0, %4\n\t"
      "s_nop %7\n\tglobal_load_lds_dwordx4 %1, %4 offset:1024\n\t"
      "s_nop %7\n\tglobal_load_lds_dwordx4 %2, %5 offset:2048\n\t"
      "s_nop %7\n\tglobal_load_lds_dwordx4 %3, %5 offset:3072" ::"v"(w0), "v"(w1), "v"(x0), "v"(x1), "s"(w), "s"(x), "s"(lds_addr), "n"(kBaseFromVector)
      : "memory", "m0");
}

struct F8Args {
  GemmParams p;
  int n_tiles;
  int wgs_per_xcd;  // grid size / 8
};

// One entry of a workgroup's unit table: what lane r of the table holds for the workgroup's r-th unit.
struct F8Unit {
  int e, ntile, row_begin, row_end;
  int tail_begin, tail_rows;  // rows of the expert that ride along with this full tile (0: none)
};
// Rows that a full token tile takes along: one MFMA column block.
static constexpr int kF8TailRows = 32;

// The launch's units in the order of big_unit (ffn_mfma_common.h: an XCD takes an eighth of the main list, expert by
// expert and feature tile by feature tile with an expert's token tiles of one feature tile next to each other, then an
// eighth of the partial token tiles), looked up for a different item in every lane: the loop over the experts is the
// same for all lanes (row counts come from readlane), each lane keeps what matches its own item.  `lane_off`: lane l holds
// the first row of expert l (lane E: the row total).  Returns whether the lane's item exists.
__device__ __forceinline__ bool f8_unit_of_lane(int lane_off, int E, int BM, int n_tiles, int xcd, int item, int balance, bool absorb, F8Unit& out) {
  int F = 0, R = 0;
  for (int e = 0; e < E; ++e) {
    const int rows = __builtin_amdgcn_readlane(lane_off, e + 1) - __builtin_amdgcn_readlane(lane_off, e);
    const BigExpertTiles x = big_expert_tiles(rows, BM, absorb, balance, kF8TailRows);
    F += x.main;
    R += x.partial;
  }
  const int UF = F * n_tiles, UR = R * n_tiles;
  const int f0 = (int)((int64_t)UF * xcd / 8), f1 = (int)((int64_t)UF * (xcd + 1) / 8);
  const int r0 = (int)((int64_t)UR * xcd / 8), r1 = (int)((int64_t)UR * (xcd + 1) / 8);
  const bool in_main = item < f1 - f0;
  const bool in_partial = !in_main && item - (f1 - f0) < r1 - r0;
  int u = in_main ? f0 + item : r0 + item - (f1 - f0);
  // partial list: feature tile by feature tile, one unit per expert that has a partial token tile
  const int p_ntile = R > 0 ? u / max(R, 1) : 0;
  int p_s = u - p_ntile * R;
  bool found = false;
  out.e = 0; out.ntile = 0; out.row_begin = 0; out.row_end = 0; out.tail_begin = 0; out.tail_rows = 0;
  for (int e = 0; e < E; ++e) {
    const int b = __builtin_amdgcn_readlane(lane_off, e), rows = __builtin_amdgcn_readlane(lane_off, e + 1) - b;
    const BigExpertTiles x = big_expert_tiles(rows, BM, absorb, balance, kF8TailRows);
    if (in_main) {
      const int units = x.main * n_tiles;
      if (!found && u < units) {
        const int ntile = u / max(x.main, 1), s = u - ntile * x.main;
        out.e = e;
        out.ntile = ntile;
        if (x.even) {
          out.row_begin = b + (int)((int64_t)rows * s / x.main);
          out.row_end = b + (int)((int64_t)rows * (s + 1) / x.main);
        } else {
          out.row_begin = b + s * BM;
          out.row_end = out.row_begin + BM;
          const int first = rows / BM * BM + kF8TailRows * s;
          if (big_tail_absorbed(rows, BM, absorb, kF8TailRows) && first < rows) {
            out.tail_begin = b + first;
            out.tail_rows = min(kF8TailRows, rows - first);
          }
        }
        found = true;
      }
      if (!found) u -= units;
    } else if (in_partial && x.partial) {
      if (!found && p_s == 0) {
        out.e = e;
        out.ntile = p_ntile;
        out.row_begin = b + rows / BM * BM;
        out.row_end = b + rows;
        found = true;
      }
      --p_s;
    }
  }
  return found;
}

// One workgroup per CU walks its XCD's unit list as one uninterrupted stream of K stages: the loads run D - 1 stages
// ahead of the MFMAs across unit boundaries, so a new unit's first operands are already in LDS when the previous unit's
// results are being written, and the pipeline is filled once per launch instead of once per unit (a workgroup per unit
// spent a fifth of its time on its own start: launch, tile lookup, first loads).  Token rows are read in sorted order
// without a gather (p.perm must be NULL: the quantising pass in front of the gate/up launch writes the rows grouped by
// expert), so that a unit's operand addresses are arithmetic on its table entry and nothing has to be fetched to start it.
template <typename T, int MODE>
__global__ void __launch_bounds__(512, 1)
grouped_fp8_ws_kernel(F8Args args) {
  constexpr int BN = 256, BM = 256, KS = 64;      // K samples (= bytes per row) per stage
  // A stage: eight shares of two weight pieces (32 weight rows) and 32 token rows, 2 KB each, then the ride-along rows.
  constexpr int SHARE = 32 * KS + 32 * KS, XSTAGE = 8 * SHARE;
  constexpr int STAGE = XSTAGE + kF8TailRows * KS, D = 4;  // stages in LDS
  constexpr int kBalance = 1;
  extern __shared__ __align__(16) uint8_t lds8[];
  const GemmParams& p = args.p;
  const int n_tiles = args.n_tiles;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int xcd = blockIdx.x & 7, wg = blockIdx.x >> 3, wgs = args.wgs_per_xcd;
  const int E = p.offsets ? p.E : 1;
  const int lane_off = p.offsets ? big_lane_offsets(p) : (lane == 1 ? (int)p.fixed_rows : 0);
  const int nst = (int)(p.kred >> 6);
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)lds8));
  const uint32_t w_lds = lds0 + wave * SHARE, t_lds = lds0 + XSTAGE + 4 * wave * KS;
  const uint32_t lane16 = lane * 16;
  // bytes from one K stage of a token row to the next: 64 in a plain row, a whole block of rows in the blocked layout
  const uint32_t x_row_bytes = p.a_block_rows ? (uint32_t)KS : (uint32_t)p.lda;
  const uint32_t x_stage_bytes = p.a_block_rows ? (uint32_t)(p.a_block_rows * KS) : (uint32_t)KS;

  // This wavefront's two row tiles of 16 weight rows: neighbours in one matrix (GATEUP: wavefronts 0-3 gate, 4-7 up).
  const WeightView& w_mine = MODE == MODE_GATEUP && wave >= 4 ? p.w1 : p.w0;
  const uint32_t tile_bytes = (uint32_t)(p.kred * 16);
  const int64_t w_expert_tiles = w_mine.rows >> 4;
  const uint8_t* const w_first = reinterpret_cast<const uint8_t*>(uniform_ptr(w_mine.qs + (int64_t)(2 * wave % (MODE == MODE_GATEUP ? BN / 32 : BN / 16)) * tile_bytes));

  // Launches without ride-along rows walk their units with an instance that knows nothing of them: their loads and the branches around
  // them cost 4 % (2048 rows of one expert, gate/up 239 -> 249 us).
  auto walk = [&](auto tails_tag) __attribute__((always_inline)) {
    constexpr bool TAILS = decltype(tails_tag)::value != 0;
    // LDS-direct loads per wavefront and stage: 2 weight pieces, 2 x 16 token rows and 4 ride-along rows
    constexpr int LOADS = TAILS ? 5 : 4;

    // ---- operands: lane (r, h) supplies row r, samples 32 h .. 32 h + 31 ------------------------------------
    const int wn = wave & 1, wm = wave >> 1;
    const bool late = wave >= 4;
    const int r32 = lane & 31, h32 = lane >> 5;
    // weight row r of a 32-row block: piece r / 16, lane position 16 g + r % 16 for g = 2 h, 2 h + 1
    const uint8_t* const a_rd = lds8 + (MODE == MODE_GATEUP ? wn * 2 : wn * 4) * SHARE + (r32 >> 4) * 1024 + ((32 * h32 + (r32 & 15)) << 4);
    const int xrow = wm * 64 + r32;
    const uint8_t* const b_rd = lds8 + wm * 2 * SHARE + 2048 + r32 * KS;
    const int bu0 = x_unit(xrow, 2 * h32) << 4, bu1 = x_unit(xrow, 2 * h32 + 1) << 4;  // rows xrow and xrow + 32 swizzle alike
    floatx16_t acc[4][2];
    // Ride-along rows.  The four wavefronts that share a weight half (128 rows) take 32 of its rows each against all of the unit's ride-along
    // rows: one MFMA per stage, GATEUP 16 gate rows and the same 16 up rows, so that both sums of a feature meet in one lane.
    floatx16_t tacc;
    // A stage's operands, all of them in registers before its first MFMA.
    u32x4_t a_op[4][2], b_op[2][2], ta_op[2], tb_op[2];
    auto read_operands = [&](auto both_tag, auto tail_tag, int slot) __attribute__((always_inline)) {
      constexpr bool BOTH = decltype(both_tag)::value;  // rows in both 32-row token blocks
      const uint8_t* bp = b_rd + slot * STAGE;
#pragma unroll
      for (int q = 0; q < (BOTH ? 2 : 1); ++q) {
        b_op[q][0] = *reinterpret_cast<const u32x4_t*>(bp + q * SHARE + bu0);
        b_op[q][1] = *reinterpret_cast<const u32x4_t*>(bp + q * SHARE + bu1);
      }
#pragma unroll
      for (int ti = 0; ti < 4; ++ti) {
        // 32-row block ti of the wavefront: GATEUP blocks 0, 1 are gate rows, 2, 3 the matching up rows (pieces 8 ..)
        const uint8_t* ap = a_rd + slot * STAGE + (MODE == MODE_GATEUP ? (ti < 2 ? 0 : 4) + (ti & 1) : ti) * SHARE;
        a_op[ti][0] = *reinterpret_cast<const u32x4_t*>(ap);
        a_op[ti][1] = *reinterpret_cast<const u32x4_t*>(ap + 256);
      }
      if constexpr (decltype(tail_tag)::value != 0) {
        // GATEUP: lanes r < 16 take piece wm of the wavefront's four gate pieces, the others of its up pieces; DOWN: its 32-row block wm
        const uint8_t* ap = a_rd + slot * STAGE + (MODE == MODE_GATEUP ? (wm >> 1) * SHARE + (wm & 1) * 1024 + (r32 >> 4) * (4 * SHARE - 1024) : wm * SHARE);
        const uint8_t* tp = lds8 + slot * STAGE + XSTAGE + r32 * KS;  // (swizzled like xrow)
        ta_op[0] = *reinterpret_cast<const u32x4_t*>(ap);
        ta_op[1] = *reinterpret_cast<const u32x4_t*>(ap + 256);
        tb_op[0] = *reinterpret_cast<const u32x4_t*>(tp + bu0);
        tb_op[1] = *reinterpret_cast<const u32x4_t*>(tp + bu1);
      }
    };
    auto multiply = [&](auto both_tag, auto tail_tag) __attribute__((always_inline)) {
      constexpr bool BOTH = decltype(both_tag)::value;
#pragma unroll
      for (int ti = 0; ti < 4; ++ti)
#pragma unroll
        for (int q = 0; q < (BOTH ? 2 : 1); ++q)
          acc[ti][q] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(join8(a_op[ti][0], a_op[ti][1]), join8(b_op[q][0], b_op[q][1]), acc[ti][q], 0, 0, 0, 127, 0, 127);
      if constexpr (decltype(tail_tag)::value != 0)
        tacc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(join8(ta_op[0], ta_op[1]), join8(tb_op[0], tb_op[1]), tacc, 0, 0, 0, 127, 0, 127);
      // (issued here, not behind the barrier that follows)
#pragma unroll
      for (int ti = 0; ti < 4; ++ti)
#pragma unroll
        for (int q = 0; q < (BOTH ? 2 : 1); ++q) asm volatile("" : "+v"(acc[ti][q]));
      if constexpr (decltype(tail_tag)::value != 0) asm volatile("" : "+v"(tacc));
    };

    // ---- epilogue: scale by the activations' reciprocal scale times the weights' scale ---------------------
    // What it needs, the kernel's arguments and the lane's place, is derived here from values that the compiler cannot see through:
    // in front of the K loops it would hold registers that they don't have to spare.
    auto epilogues = [&](auto both_tag, auto tail_tag, const F8Unit& un, int rpg, int my_rows) __attribute__((always_inline)) {
      constexpr bool BOTH = decltype(both_tag)::value;
      auto kernarg = __builtin_amdgcn_kernarg_segment_ptr();
      asm volatile("" : "+s"(kernarg));
      const GemmParams& q = reinterpret_cast<const F8Args*>((const void*)kernarg)->p;
      const int l = lane_again(), r32 = l & 31, h32 = l >> 5;
      const float xsc = q.x_scale[0];
      const float out_rs = q.out_scale ? q.out_scale[0] : 0.0f;
      // 1 / out_rs once; per element v * inv refined by one residual step (fma(-q0, rs, v) * inv + q0), which is the
      // correctly rounded quotient except in rare last-bit cases that the following rounding to T absorbs
      const float out_inv = q.out_scale ? __builtin_amdgcn_rcpf(out_rs) : 0.0f;
      const float s0 = xsc * reinterpret_cast<const float*>(q.w0.d)[q.w0.d_count > 1 ? un.e : 0];
      const float s1 = MODE == MODE_GATEUP ? xsc * reinterpret_cast<const float*>(q.w1.d)[q.w1.d_count > 1 ? un.e : 0] : 0.0f;
      // four consecutive features `col`.. of output row `orow_i`: gate and up sums (GATEUP), or the sums `g` (DOWN)
      auto store_quad = [&](auto act_tag, int64_t orow_i, int64_t col, const float(&g)[4], const float(&u)[4]) __attribute__((always_inline)) {
        constexpr int ACT = decltype(act_tag)::value;
        const int64_t orow = orow_i * q.ldo;
        if (MODE == MODE_GATEUP) {
          float gq[4], uq[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            gq[i] = g[i] * s0;
            uq[i] = u[i] * s1;
          }
          if (q.out_scale) {  // e4m3fn(clamp(T(v / rscale))) for the next fp8 projection
            float t[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float a = round_to<T>(act_fast<ACT>(round_to<T>(gq[i])));
              const float v = round_to<T>(__fmul_rn(a, round_to<T>(uq[i])));
              const float q0 = v * out_inv;
              const float q1 = __builtin_fmaf(__builtin_fmaf(-q0, out_rs, v), out_inv, q0);
              t[i] = fminf(fmaxf(round_to<T>(q1), -448.0f), 448.0f);
            }
            int qv = __builtin_amdgcn_cvt_pk_fp8_f32(t[0], t[1], 0, false);  // hardware OCP e4m3fn, round to nearest even
            qv = __builtin_amdgcn_cvt_pk_fp8_f32(t[2], t[3], qv, true);
            const int64_t at = q.out_block_rows ? ((col >> 6) * q.out_block_rows + orow_i) * KS + (col & 63) : orow + col;
            *reinterpret_cast<int*>(reinterpret_cast<uint8_t*>(q.out) + at) = qv;
          } else {
            *reinterpret_cast<uint2*>(reinterpret_cast<T*>(q.out) + orow + col) = gateup_quad<T, ACT>(gq, uq);
          }
        } else {
          *reinterpret_cast<uint2*>(reinterpret_cast<T*>(q.out) + orow + col) =
              make_uint2(pack2<T>(g[0] * s0, g[1] * s0), pack2<T>(g[2] * s0, g[3] * s0));
        }
      };
      auto block = [&](auto tj_tag, auto act_tag) __attribute__((always_inline)) {
        constexpr int tj = decltype(tj_tag)::value;
        if (tj * 32 + r32 < my_rows) {
          const int64_t orow_i = out_row(q, un.row_begin + wm * rpg + tj * 32 + r32);
#pragma unroll
          for (int ti = 0; ti < (MODE == MODE_GATEUP ? 2 : 4); ++ti)
#pragma unroll
            for (int b = 0; b < 4; ++b) {  // four consecutive features per 8-row band of the 32 x 32 result
              const int64_t col = (int64_t)un.ntile * (MODE == MODE_GATEUP ? BN / 2 : BN) + wn * (MODE == MODE_GATEUP ? 64 : 128) + ti * 32 + 8 * b + 4 * h32;
              const floatx16_t &c = acc[ti][tj], &d = acc[MODE == MODE_GATEUP ? ti + 2 : ti][tj];
              const float g[4] = {c[4 * b], c[4 * b + 1], c[4 * b + 2], c[4 * b + 3]}, u[4] = {d[4 * b], d[4 * b + 1], d[4 * b + 2], d[4 * b + 3]};
              store_quad(act_tag, orow_i, col, g, u);
              __builtin_amdgcn_sched_barrier(0);  // one quad at a time: the accumulators leave no room for more
            }
        }
      };
      auto tail = [&](auto act_tag) __attribute__((always_inline)) {
        if (r32 < un.tail_rows) {
          const int64_t orow_i = out_row(q, un.tail_begin + r32);
#pragma unroll
          for (int b = 0; b < (MODE == MODE_GATEUP ? 2 : 4); ++b) {
            const int64_t col = MODE == MODE_GATEUP ? (int64_t)un.ntile * (BN / 2) + wn * 64 + wm * 16 + 8 * b + 4 * h32
                                                    : (int64_t)un.ntile * BN + wn * 128 + wm * 32 + 8 * b + 4 * h32;
            constexpr int UP = MODE == MODE_GATEUP ? 8 : 0;
            const float g[4] = {tacc[4 * b], tacc[4 * b + 1], tacc[4 * b + 2], tacc[4 * b + 3]};
            const float u[4] = {tacc[UP + 4 * b], tacc[UP + 4 * b + 1], tacc[UP + 4 * b + 2], tacc[UP + 4 * b + 3]};
            store_quad(act_tag, orow_i, col, g, u);
          }
        }
      };
      auto all = [&](auto act_tag) __attribute__((always_inline)) {
        block(F8Int<0>{}, act_tag);
        if constexpr (BOTH) block(F8Int<1>{}, act_tag);
        if constexpr (decltype(tail_tag)::value != 0) tail(act_tag);
      };
      if (MODE == MODE_DOWN || q.act == STMOE_ACT_SILU) all(EpiAct<STMOE_ACT_SILU>{});
      else all(EpiAct<STMOE_ACT_GELU_ERF>{});
    };
    // Rows per token-row group of 64 LDS rows: the rows of a partial tile are spread over the four groups in multiples of 16.
    auto rows_per_group = [](int rows_here) { return min(64, ((rows_here + 3) / 4 + 15) / 16 * 16); };

    // ---- the workgroup's units, up to 64 at a time -----------------------------------------------------------
    // Round r of the walk takes the item of the XCD's list at place (wg + r (wgs / 2 + 1)) mod wgs of that round (see
    // grouped_mfma_ws_kernel: neighbouring items differ systematically in cost and a workgroup that kept its place in every
    // round would collect one kind).  Lane r of the table holds round r's unit.
    for (int round0 = 0;; round0 += 64) {
      F8Unit mine;
      const int round = round0 + lane;
      const int place = (wg + round * ((wgs >> 1) + 1)) % wgs;
      const bool have = f8_unit_of_lane(lane_off, E, BM, n_tiles, xcd, round * wgs + place, kBalance, TAILS, mine);
      // (the items of later rounds come later in the list: the lanes that hold a unit are lanes 0 .. n_units - 1)
      const int n_units = __builtin_popcountll(__ballot(have));
      if (n_units == 0) return;
      // (the table lies behind the stages; every wavefront writes the same values and reads back its own)
      int* const table = reinterpret_cast<int*>(lds8 + D * STAGE);
      *reinterpret_cast<int4*>(table + lane * 8) = make_int4(mine.e | (mine.ntile << 8), mine.row_begin, mine.row_end, mine.tail_begin);
      table[lane * 8 + 4] = mine.tail_rows;
      auto unit_at = [&](int i) {
        F8Unit un;
        const int4 t = *reinterpret_cast<const int4*>(table + i * 8);
        const int en = __builtin_amdgcn_readfirstlane(t.x);
        un.e = en & 0xff;
        un.ntile = en >> 8;
        un.row_begin = __builtin_amdgcn_readfirstlane(t.y);
        un.row_end = __builtin_amdgcn_readfirstlane(t.z);
        un.tail_begin = __builtin_amdgcn_readfirstlane(t.w);
        un.tail_rows = __builtin_amdgcn_readfirstlane(table[i * 8 + 4]);
        return un;
      };

      // ---- the load side: stage `gl` of the batch = stage `sl` of unit `ul` ------------------------------------
      // One M0 value serves the share's four loads: an instruction's immediate offset counts for both addresses, which the global
      // ones below make up for.
      const uint8_t *wq = nullptr, *xq = nullptr;  // at the stage that is loaded next
      uint32_t xoff[2] = {0, 0}, toff = 0, load_slot = 0;
      int ul = -1, left = 0;  // unit, stages of it still to load
      auto next_unit = [&]() __attribute__((always_inline)) {
        if (ul + 1 == n_units) {  // past the batch's last stage: that one again, into slots that nobody reads
          left = 1;
          wq -= 1024;
          xq -= x_stage_bytes;
          return;
        }
        ++ul;
        left = nst;
        const F8Unit un = unit_at(ul);
        const int rows_here = un.row_end - un.row_begin, rpg = rows_per_group(rows_here);
        wq = w_first + ((int64_t)un.e * w_expert_tiles + (int64_t)un.ntile * (MODE == MODE_GATEUP ? BN / 32 : BN / 16)) * tile_bytes;
        xq = reinterpret_cast<const uint8_t*>(p.a) + (int64_t)un.row_begin * x_row_bytes - 3072;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          // token rows: lane l fills LDS row 32 wave + 16 j + l / 4 with the 16 bytes that belong at position l % 4
          // (x_unit is an involution: position -> logical unit); LDS rows without a tile row re-read a valid one
          const int lr = 32 * wave + 16 * j + (lane >> 2);
          const int r = min((lr >> 6) * rpg + min(lr & 63, rpg - 1), rows_here - 1);
          xoff[j] = (uint32_t)r * x_row_bytes + (x_unit(lr, lane & 3) << 4) + (j == 0 ? 1024 : 0);
        }
        if constexpr (TAILS) {  // (a unit without ride-along rows: its own rows again, never used)
          const int tr = 4 * wave + ((lane & 15) >> 2);
          const int i = un.tail_rows > 0 ? un.tail_begin - un.row_begin + min(tr, un.tail_rows - 1) : min(tr, rows_here - 1);
          toff = (uint32_t)i * x_row_bytes + (x_unit(tr, lane & 3) << 4);
        }
      };
      auto issue_next = [&]() __attribute__((always_inline)) {
        if (left == 0) next_unit();
        f8_load_share(wq, lane16, lane16 + tile_bytes - 1024, xq, xoff[0], xoff[1], w_lds + load_slot);
        if constexpr (TAILS) f8_load16_to_lds_16_lanes(xq + 3072, toff, t_lds + load_slot);
        wq += 1024;
        xq += x_stage_bytes;
        --left;
        load_slot = load_slot == (D - 1) * STAGE ? 0 : load_slot + STAGE;
      };

      // every wavefront loads its share of every stage and meets every barrier, with or without token rows of its own
#pragma unroll 1
      for (int st = 0; st < D - 1; ++st) issue_next();
      int slot = 0;
#pragma unroll 1
      for (int u = 0; u < n_units; ++u) {
        const F8Unit un = unit_at(u);
        const int rows_here = un.row_end - un.row_begin, rpg = rows_per_group(rows_here);
        const int my_rows = min(rpg, rows_here - wm * rpg);
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[a][b][q] = 0.0f;
#pragma unroll
        for (int q = 0; q < 16; ++q) tacc[q] = 0.0f;
        // Interval st: everybody's share of stage st has landed, everybody has read the stage before, whose slot is filled again.
        auto meet = [&]() __attribute__((always_inline)) {
          vm_wait<(D - 2) * LOADS>();  // the loads of the D - 2 stages after this one may still be in flight
          asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
        };
        auto stages_early = [&](auto both_tag, auto tail_tag) __attribute__((always_inline)) {
#pragma unroll 1
          for (int st = 0; st < nst; ++st) {
            meet();
            if constexpr (decltype(both_tag)::value >= 0) read_operands(both_tag, tail_tag, slot);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            issue_next();
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (decltype(both_tag)::value >= 0) multiply(both_tag, tail_tag);
            slot = slot == D - 1 ? 0 : slot + 1;
          }
        };
        auto stages_late = [&](auto both_tag, auto tail_tag) __attribute__((always_inline)) {
          meet();
          issue_next();
          if constexpr (decltype(both_tag)::value >= 0) read_operands(both_tag, tail_tag, slot);
          slot = slot == D - 1 ? 0 : slot + 1;
#pragma unroll 1
          for (int st = 1; st < nst; ++st) {
            meet();
            if constexpr (decltype(both_tag)::value >= 0) multiply(both_tag, tail_tag);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (decltype(both_tag)::value >= 0) read_operands(both_tag, tail_tag, slot);
            __builtin_amdgcn_sched_barrier(0);
            issue_next();
            slot = slot == D - 1 ? 0 : slot + 1;
          }
          if constexpr (decltype(both_tag)::value >= 0) multiply(both_tag, tail_tag);
        };
        auto stages = [&](auto both_tag, auto tail_tag) __attribute__((always_inline)) {
          if (late) stages_late(both_tag, tail_tag);
          else stages_early(both_tag, tail_tag);
        };
        if (TAILS && un.tail_rows > 0) {
          if constexpr (TAILS) {
            stages(F8Int<1>{}, F8Int<1>{});
            epilogues(F8Int<1>{}, F8Int<1>{}, un, rpg, my_rows);
          }
        } else if (my_rows > 32) {
          stages(F8Int<1>{}, F8Int<0>{});
          epilogues(F8Int<1>{}, F8Int<0>{}, un, rpg, my_rows);
        } else if (my_rows > 0) {
          stages(F8Int<0>{}, F8Int<0>{});
          epilogues(F8Int<0>{}, F8Int<0>{}, un, rpg, my_rows);
        } else {
          stages(F8Int<-1>{}, F8Int<0>{});
        }
      }
      // (a further batch, if the workgroup has more than 64 units, starts with empty LDS stages: the loads past this one's end have
      // landed and the last stage has been read by everybody)
      vm_wait<0>();
      __syncthreads();
    }
  };
  // Ride-along rows save their expert's partial tile and cost the full tiles an MFMA per nine and their loads: a unit that carries them
  // takes 10-15 % longer, every other one of the launch some 4 %.  They are taken along where that saves an eighth of the rounds over the
  // CUs or more.  44 layers of 4 to 16 experts with 1 to 40 rows more than whole tiles, 1024 to 6144 x 1024 to 16384: 5 % less time than
  // without them (-1 to 14 %), and the same within 0.1 % as where any round saved decides (single layers 3 % less to 1 % more).
  const int lane_end = __builtin_amdgcn_ds_bpermute(4 * (lane + 1), lane_off);
  const int lane_rows = lane < E ? lane_end - lane_off : 0;
  auto rounds = [&](bool absorb) {
    const BigExpertTiles x = big_expert_tiles(lane_rows, BM, absorb, kBalance, kF8TailRows);
    const int units = __builtin_amdgcn_readlane(wave_inclusive_sum(x.main + x.partial), 63) * n_tiles;
    return (units + 8 * wgs - 1) / (8 * wgs);
  };
  // (a scalar branch: as a vector one the comparison cost the kernel four registers and the layer above 0.7 %)
  if (__builtin_amdgcn_readfirstlane(8 * rounds(true) <= 7 * rounds(false))) walk(F8Int<1>{});
  else walk(F8Int<0>{});
}

template <typename T, int MODE>
static int launch_fp8_ws_m(const GemmParams& p, int64_t max_rows, hipStream_t st) {
  constexpr int BN = 256, BM = 256;
  constexpr size_t lds_bytes = (size_t)4 * (BN + BM + kF8TailRows) * 64 + 64 * 32;  // four stages and the unit table
  static std::atomic<uint64_t> lds_ready{0};
  auto kern = grouped_fp8_ws_kernel<T, MODE>;
  if (int rc = reserve_lds(reinterpret_cast<const void*>(kern), lds_bytes, lds_ready, "fp8 ws kernel")) return rc;
  const int n_tiles = (int)(MODE == MODE_GATEUP ? p.n_out / (BN / 2) : p.n_out / BN);
  const int experts = p.offsets ? p.E : 1;
  const int m_slots = (int)((max_rows + BM - 1) / BM) + experts;
  // one workgroup per CU (it takes all of the CU's LDS), fewer when an XCD's list cannot be longer than that
  const int per_xcd = std::min(kBigCusPerXcd, big_grid(n_tiles, m_slots, false) / 8);
  kern<<<dim3((unsigned)(8 * per_xcd)), 512, lds_bytes, st>>>(F8Args{p, n_tiles, per_xcd});
  return check_launch("grouped_fp8_ws");
}

// act_dtype: dtype of the results; activations are e4m3fn bytes (p.a, p.lda in bytes), weights packed fp8.
int launch_fp8_ws(int act_dtype, int wtag, int mode, const GemmParams& p, int64_t max_rows, hipStream_t st) {
  if (max_rows == 0) return STMOE_OK;
  if (!p.x_scale) return set_error(STMOE_ERR_NULL, "fp8 ws kernel: activation scale is NULL");
  if (wtag != WF_FP8_F32D_P) return set_error(STMOE_ERR_UNSUPPORTED, "fp8 ws kernel: needs packed fp8 weights with fp32 scale(s)");
  if (p.offsets && p.E >= 64) return set_error(STMOE_ERR_UNSUPPORTED, "fp8 ws kernel: at most 63 experts");
  if (p.perm) return set_error(STMOE_ERR_UNSUPPORTED, "fp8 ws kernel: token rows must be grouped by expert already (no gather)");
  if (p.kred % 256 != 0 || p.lda % 16 != 0 || p.ldo % 4 != 0 || p.n_out % (mode == MODE_GATEUP ? 128 : 256) != 0)
    return set_error(STMOE_ERR_UNSUPPORTED, "fp8 ws kernel: needs K %% 256 == 0 and output features in whole tiles");
  if (std::max(max_rows, (int64_t)p.a_block_rows) * p.kred >= (int64_t)1 << 32)
    return set_error(STMOE_ERR_UNSUPPORTED, "fp8 ws kernel: activations span 4 GB or more");
  if (act_dtype == STMOE_F16)
    return mode == MODE_GATEUP ? launch_fp8_ws_m<f16_t, MODE_GATEUP>(p, max_rows, st) : launch_fp8_ws_m<f16_t, MODE_DOWN>(p, max_rows, st);
  if (act_dtype == STMOE_BF16)
    return mode == MODE_GATEUP ? launch_fp8_ws_m<bf16_t, MODE_GATEUP>(p, max_rows, st) : launch_fp8_ws_m<bf16_t, MODE_DOWN>(p, max_rows, st);
  return set_error(STMOE_ERR_DTYPE, "fp8 ws kernel: result dtype %d", act_dtype);
}

}  // namespace stmoe
