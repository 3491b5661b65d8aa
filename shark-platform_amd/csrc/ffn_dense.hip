// Prefill kernel for unquantized 16-bit expert weights of the activations' type: 256 (or 128) weight rows x up to 256 token
// rows per workgroup, K step 64, both operands straight from global memory into LDS.
//
// What bounds it: up to some 200 rows per expert the weight stream (a layer of 8 x 3 x 14336 x 4096 in bf16 is 2.8 GB, 430 us
// at the rate of a large copy), beyond that the matrix pipe.  Nothing has to be converted, so there are no loader wavefronts:
// all eight issue their share of the direct loads of a later K step and multiply the current one.
//
//   LDS: as many stages of either operand as 160 KB hold, four at most (three are the least that give a load two K steps to arrive;
//     64 KB in flight per CU cover the memory latency; over 41 layers eight at most are 0.7 % slower than four: short reductions start
//     later).  256 weight rows and 192 or 256 token rows leave room for three and two.  Rows of 128 bytes, XOR-swizzled in 16-byte units
//     (see ffn_mfma_common.h): the direct load puts lane l's 16 bytes at its base + 16 l, so the lanes fetch the units of a row in
//     swizzled order.
//   units: LDS and loads for 32, 128, 192 or 256 token rows.  With 192 a quarter of the loads from L2 goes (and of 128 weight rows a token row
//     has as many steps to arrive as the weights): gate/up of 515 tokens (129 rows per expert) 416 us with 256 only, 398 so.
//   last round: units left over after the last whole round over an XCD's CUs are cut into two of 128 weight rows if the halves fit one
//     round (with whole units / halves, us: gate/up of 515 tokens, three rounds and 16 units, 387 / 371; to 6144 features, one and 16, 187 / 169;
//     down of 2048 tokens, two and 16, 510 / 456).  The halves of less than a round take what units of 128 weight rows take: [4096, 8192] at 400
//     tokens, 16 units, 133 and 133 (whole 162).
//   wavefronts: 4 x 2 (64 x 64 of BN = 256) up to 128 rows, 2 x 4 (128 x 48 or 64) above; the rows of a unit are spread evenly
//     over the token groups in multiples of 16 and only the column blocks that hold rows are multiplied.
//   The reduction runs in the order of the 128 x 128 kernel: the sums are the same bits.
// Measured (8 experts of 4096 x 14336, top-2, bf16; gate/up + down, us; 128 x 128 kernel / this one): 100 tokens 425 + 272 /
// 331 + 170, 515 tokens 675 + 317 / 371 to 398 + 200 (4.8 to 5.1 TB/s of weights; where the pages lie moves it), 2048 tokens 1936 + 835 /
// 1004 + 456 (0.96 PFLOP/s; SiLU by expf and a division, as the 128 x 128 kernel computes it, is some 20 us of the gate/up launch).
// Slower at 515 tokens, gate/up: weights and tokens sent by different wavefronts 442, both loads behind the first half's products 465,
// after the step's products 488.
#include "ffn_mfma_common.h"

namespace stmoe {

template <int V> struct DenseInt { static constexpr int value = V; };

// Stages in LDS of a unit of `bn` weight rows and `lds_rows` token rows.  A CU's loads return in the order of their issue, token rows that
// hit in L2 behind the weights in front of them: one operand further ahead than the other is of no use, so both get as many stages as fit,
// except that three weight stages are worth two token stages.
struct DenseStages {
  int w, x;
};
static constexpr int kDenseLds = 160 * 1024;
static constexpr DenseStages dense_stages(int bn, int lds_rows) {
  const int both = kDenseLds / ((bn + lds_rows) * 128);
  return both >= 3 ? DenseStages{both < 4 ? both : 4, both < 4 ? both : 4} : DenseStages{3, 2};
}

template <typename T, int MODE, int BN_LAUNCH>
__global__ void __launch_bounds__(512, 1)
grouped_dense_kernel(GemmParams p, int n_tiles) {
  constexpr int BM = 256;
  extern __shared__ __align__(16) uint16_t lds[];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, n_in = lane & 15;
  // The XCD's units; those after the last whole round over its CUs are cut into two of half the weight rows if the halves fit one round.
  BigTile tile;
  int half = -1;
  {
    const int xcd = blockIdx.x & 7;
    int item = blockIdx.x >> 3;
    const BigLanes lanes = big_lanes(p, big_lane_offsets(p), lane, BM, false, 2);
    const BigPlan plan = big_plan(lanes, n_tiles, xcd, false);
    if constexpr (BN_LAUNCH == 256) {
      const int units = plan.whole, rest = units % kBigCusPerXcd, whole = 2 * rest <= kBigCusPerXcd ? units - rest : units;
      if (item >= whole) {
        half = (item - whole) & 1;
        item = whole + (item - whole) / 2;
        if (item >= units) return;
      }
    }
    if (!big_unit(lanes, BM, n_tiles, plan, item, tile, false)) return;
  }
  const int row_begin = tile.row_begin, rows_here = tile.row_end - tile.row_begin;
  const int nkt = (int)(p.kred >> 6), last = nkt - 1;

  auto unit = [&](auto bn_tag, auto groups_tag, auto blocks_tag) {
    constexpr int BN = decltype(bn_tag)::value, WSTAGE = BN * BIG_LS;
    constexpr int GROUPS = decltype(groups_tag)::value;           // token-row groups
    constexpr int BLOCKS = decltype(blocks_tag)::value;           // 16-row column blocks of a group
    constexpr int RPG = 16 * BLOCKS, XROWS = GROUPS * RPG;        // LDS rows of a group, of a token stage
    constexpr int WN = 8 / GROUPS, TI = BN / 16 / WN;             // wavefronts along the features, 16-feature blocks of each
    constexpr int XSTAGE = XROWS * BIG_LS;
    constexpr DenseStages ST = dense_stages(BN, XROWS);
    constexpr int WA = ST.w - 1, XA = ST.x - 1;                   // K steps ahead
    constexpr int WLOADS = BN / 64, XLOADS = (XROWS + 63) / 64;   // direct loads of 8 rows per wavefront and K step
    static_assert((ST.w * BN + ST.x * XROWS) * 128 <= kDenseLds && WA >= 2 && (XA == WA || XA == 1) && WA * (WLOADS + XLOADS) <= 63, "stages and waits");
    const int ntile = BN == BN_LAUNCH ? tile.ntile : 2 * tile.ntile + half;
    const int rpg = min(RPG, ((rows_here + GROUPS - 1) / GROUPS + 15) / 16 * 16);  // tile row grp * rpg + i <-> LDS row grp * RPG + i
    uint16_t* const Wbase = lds;                  // [ST.w][BN][64]
    uint16_t* const Xbase = lds + ST.w * WSTAGE;  // [ST.x][XROWS][64]

    // ---- loads: this wavefront's rows are 64 j + 8 wave .. + 7 of either operand's tile
    const int unit_off = ((lane & 7) ^ (lane >> 3)) << 4;  // LDS unit lane % 8 of row lane / 8 holds this unit of the row
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint16_t*)lds);
    const uint32_t w_lds = __builtin_amdgcn_readfirstlane(lds0 + wave * 8 * BIG_LS * 2);
    const uint32_t x_lds = __builtin_amdgcn_readfirstlane(lds0 + (ST.w * WSTAGE + (XROWS < 64 ? wave & 3 : wave) * 8 * BIG_LS) * 2);
    const char* wsrc[WLOADS];
#pragma unroll
    for (int j = 0; j < WLOADS; ++j) {
      const int r = 64 * j;  // (a block of 64 rows is all gate or all up)
      const bool up = MODE == MODE_GATEUP && r >= BN / 2;
      const WeightView& wv = up ? p.w1 : p.w0;
      const int64_t row = (int64_t)tile.e * wv.rows + (MODE == MODE_GATEUP ? (int64_t)ntile * (BN / 2) + (up ? r - BN / 2 : r)
                                                                           : (int64_t)ntile * BN + r) + wave * 8;
      wsrc[j] = reinterpret_cast<const char*>(wv.qs) + row * p.kred * 2;
    }
    const uint32_t woff = (uint32_t)((lane >> 3) * (int)p.kred * 2 + unit_off);
    uint32_t xoff[XLOADS];
#pragma unroll
    for (int j = 0; j < XLOADS; ++j) {
      // LDS rows that hold no tile row re-read a valid one (their outputs are never stored); of 32 rows wavefronts 4-7 send the same again
      const int lr = (64 * j + 8 * wave + (lane >> 3)) % XROWS, grp = lr / RPG, in = lr - grp * RPG;
      const int i = row_begin + min(grp * rpg + min(in, rpg - 1), rows_here - 1);
      const int64_t src = p.perm ? (int64_t)(p.perm[i] / p.k_top) : (int64_t)i;
      xoff[j] = (uint32_t)(src * p.lda * 2 + unit_off);
    }
    // Requests past the last step read the last step again (into a stage that nobody reads), so that the number of loads in
    // flight is the same at every wait.
    auto load_w = [&](int kt, int stage) {
      const int64_t off = (int64_t)min(kt, last) * (BIG_BK * 2);
#pragma unroll
      for (int j = 0; j < WLOADS; ++j) vm_load16_to_lds(wsrc[j] + off, woff, w_lds + (uint32_t)((stage * WSTAGE + 64 * j * BIG_LS) * 2));
    };
    auto load_x = [&](int kt, int stage) {
      const char* src = reinterpret_cast<const char*>(p.a) + (int64_t)min(kt, last) * (BIG_BK * 2);
#pragma unroll
      for (int j = 0; j < XLOADS; ++j) vm_load16_to_lds(src, xoff[j], x_lds + (uint32_t)((stage * XSTAGE + 64 * j * BIG_LS) * 2));
    };
    // Order of the loads, and what the waits (at most N of a wavefront's loads still in flight, the N youngest) leave:
    //   as many stages of both: W0 X0 .. | step kt: W, X(kt + WA); behind its wait W, X(kt + 1) have landed: N = (WA - 1) (WLOADS + XLOADS)
    //   else:                   W0 X0 W1 | step kt: X(kt + 1) W(kt + 2); behind its wait W, X(kt + 1) have landed: N = WLOADS
    constexpr bool XEARLY = XA == WA;
    constexpr int INFLIGHT = XEARLY ? (WA - 1) * (WLOADS + XLOADS) : WLOADS;
    // ---- operands
    const int wn = wave % WN, wm = wave / WN;
    const int my_rows = min(rpg, rows_here - wm * rpg);  // rows of this wavefront's group (<= 0: none)
    const int ntj = my_rows > 0 ? (my_rows + 15) >> 4 : 0;
    const uint16_t* a_rd[2];  // K half ks: unit ks * 4 + g of the wavefront's first weight row + n_in, and of its token row
    const uint16_t* b_rd[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int u = ((ks * 4 + g) ^ (n_in & 7)) << 3;
      a_rd[ks] = Wbase + ((MODE == MODE_GATEUP ? wn * (BN / 2 / WN) : wn * (BN / WN)) + n_in) * BIG_LS + u;
      b_rd[ks] = Xbase + (wm * RPG + n_in) * BIG_LS + u;
    }
    auto block_row = [](int ti) { return MODE == MODE_GATEUP ? (ti < TI / 2 ? ti * 16 : BN / 2 + (ti - TI / 2) * 16) : ti * 16; };
    floatx4_t acc[TI][BLOCKS];
#pragma unroll
    for (int a = 0; a < TI; ++a)
#pragma unroll
      for (int b = 0; b < BLOCKS; ++b) acc[a][b] = (floatx4_t){0.f, 0.f, 0.f, 0.f};

    auto compute = [&](auto ntj_tag, int ws, int xs, int ks) {
      constexpr int NTJ = decltype(ntj_tag)::value;
      if constexpr (NTJ > 0) {
        const uint16_t* ap = a_rd[ks] + ws * WSTAGE;
        const uint16_t* bp = b_rd[ks] + xs * XSTAGE;
        u32x4_t bf[NTJ];
#pragma unroll
        for (int tj = 0; tj < NTJ; ++tj) bf[tj] = *reinterpret_cast<const u32x4_t*>(bp + tj * 16 * BIG_LS);
#pragma unroll
        for (int ti = 0; ti < TI; ++ti) {
          const u32x4_t af = *reinterpret_cast<const u32x4_t*>(ap + block_row(ti) * BIG_LS);
          // (alternating direction: one operand changes per instruction, which saves power at the power limit)
#pragma unroll
          for (int tj = 0; tj < NTJ; ++tj) {
            const int t = (ti & 1) ? NTJ - 1 - tj : tj;
            acc[ti][t] = mfma16b<T>(af, bf[t], acc[ti][t]);
          }
        }
        // two weight fragments ahead of the multiplications, then one read per fragment's MFMAs
        __builtin_amdgcn_sched_group_barrier(0x100, NTJ + 2, 0);
#pragma unroll
        for (int i = 0; i < TI - 2; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, NTJ, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2 * NTJ, 0);
      }
    };
    // Step kt overwrites the stages that step kt - 1 read; the barrier at its end lies between.
    auto k_loop = [&](auto ntj_tag) {
      int ws = 0, xs = 0;
      for (int kt = 0; kt < nkt; ++kt) {
        const int wl = ws == 0 ? ST.w - 1 : ws - 1, xl = xs == 0 ? ST.x - 1 : xs - 1;
        if constexpr (XEARLY) load_w(kt + WA, wl);
        else load_x(kt + 1, xl);
        compute(ntj_tag, ws, xs, 0);
        if constexpr (XEARLY) load_x(kt + XA, xl);
        else load_w(kt + WA, wl);
        compute(ntj_tag, ws, xs, 1);
        vm_wait<INFLIGHT>();
        __syncthreads();
        ws = ws == ST.w - 1 ? 0 : ws + 1;
        xs = xs == ST.x - 1 ? 0 : xs + 1;
      }
    };
#pragma unroll
    for (int i = 0; i < WA; ++i) {
      load_w(i, i);
      if (i < XA) load_x(i, i);
    }
    vm_wait<INFLIGHT>();
    __syncthreads();
    if (BLOCKS > 3 && ntj == 4) k_loop(DenseInt<BLOCKS < 4 ? 0 : 4>{});
    else if (BLOCKS > 2 && ntj == 3) k_loop(DenseInt<BLOCKS < 3 ? 0 : 3>{});
    else if (BLOCKS > 1 && ntj == 2) k_loop(DenseInt<BLOCKS < 2 ? 0 : 2>{});
    else if (ntj == 1) k_loop(DenseInt<1>{});
    else k_loop(DenseInt<0>{});
    vm_wait<0>();  // the requests past the last step: nothing may land in LDS after the workgroup is done

    // ---- results: lane (n_in, g) holds features 4 g .. 4 g + 3 of each block for token row n_in of each column block
    const FakeQuant fq = fq_scale(p);
#pragma unroll
    for (int tj = 0; tj < BLOCKS; ++tj) {
      if (tj * 16 + n_in >= my_rows) continue;
      T* orow = reinterpret_cast<T*>(p.out) + out_row(p, row_begin + wm * rpg + tj * 16 + n_in) * p.ldo + 4 * g;
      if constexpr (MODE == MODE_GATEUP) {
        orow += (int64_t)ntile * (BN / 2) + wn * (BN / 2 / WN);
#pragma unroll
        for (int ti = 0; ti < TI / 2; ++ti) {
          const floatx4_t ga = acc[ti][tj], ua = acc[ti + TI / 2][tj];
          const float gq[4] = {ga[0], ga[1], ga[2], ga[3]}, uq[4] = {ua[0], ua[1], ua[2], ua[3]};
          uint2* dst = reinterpret_cast<uint2*>(orow + ti * 16);
          if (p.act == STMOE_ACT_SILU) *dst = gateup_quad<T, ACT_SILU_IEEE>(gq, uq, fq);
          else *dst = gateup_quad<T, STMOE_ACT_GELU_ERF>(gq, uq, fq);
        }
      } else {
        orow += (int64_t)ntile * BN + wn * (BN / WN);
#pragma unroll
        for (int ti = 0; ti < TI; ++ti) {
          const floatx4_t v = acc[ti][tj];
          *reinterpret_cast<uint2*>(orow + ti * 16) = make_uint2(pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]));
        }
      }
    }
  };
  auto sized = [&](auto bn_tag) {
    if (rows_here <= 32) unit(bn_tag, DenseInt<2>{}, DenseInt<1>{});
    else if (rows_here <= 128) unit(bn_tag, DenseInt<2>{}, DenseInt<4>{});
    else if (rows_here <= 192) unit(bn_tag, DenseInt<4>{}, DenseInt<3>{});
    else unit(bn_tag, DenseInt<4>{}, DenseInt<4>{});
  };
  if (BN_LAUNCH == 256 && half < 0) sized(DenseInt<BN_LAUNCH>{});
  else sized(DenseInt<128>{});
}

template <typename T, int MODE, int BN>
static int launch_dense_m(const GemmParams& p, int64_t max_rows, hipStream_t st) {
  constexpr size_t lds_bytes = kDenseLds;
  static std::atomic<uint64_t> lds_ready{0};
  auto kern = grouped_dense_kernel<T, MODE, BN>;
  if (int rc = reserve_lds(reinterpret_cast<const void*>(kern), lds_bytes, lds_ready, "dense kernel")) return rc;
  const int n_tiles = (int)(p.n_out / (MODE == MODE_GATEUP ? BN / 2 : BN));
  const int experts = p.offsets ? p.E : 1;
  const int m_slots = (int)((max_rows + 255) / 256) + experts;
  kern<<<dim3((unsigned)(big_grid(n_tiles, m_slots, false) + (BN == 256 ? 8 * kBigCusPerXcd / 2 : 0))), 512, lds_bytes, st>>>(p, n_tiles);
  return check_launch("grouped_dense");
}
// 128 weight rows per unit instead of 256 while 256 would leave CUs without a unit (a unit per 256 features and expert, and half
// a unit more per 256 rows).  Measured (8 experts, top-2, bf16, us, 256 / 128): gate/up of 1024 features from 1024, 300 tokens 12.6 / 12.5, 2048
// tokens 35 / 30; of 6144 from 4096, 515 tokens 169 / 177; of 14336 515 tokens 371 / 403.  Down to 4096 features from 14336: 515 tokens
// 198 / 200, 1024 tokens 334 / 421; to 2048 from 4096, 1500 tokens 58 / 59.  Over 12900 launches of 1 to 64 experts, 512 to 14336 x 512 to
// 14336, 2 to 2500 rows per expert, by this measure of units: up to 96 the same (halves), 96 to 128 256 rows take 0.99 of the time, 128 to 192 0.92 (up to
// 1.49: launches of just over half a round), beyond 0.9 to 0.95 (up to 1.4, from 512 on 1.2).  On the line at 192 a launch takes 1.02 of the
// better choice, at 128 1.01.
template <typename T>
static int launch_dense_t(int mode, const GemmParams& p, int64_t max_rows, hipStream_t st) {
  const int64_t wide = mode == MODE_GATEUP ? 128 : 256, experts = p.offsets ? std::min<int64_t>(p.E, max_rows) : 1;
  const bool narrow = p.n_out % wide != 0 || p.n_out / wide * (experts + max_rows / 512) < 192;
  if (mode == MODE_GATEUP) return narrow ? launch_dense_m<T, MODE_GATEUP, 128>(p, max_rows, st) : launch_dense_m<T, MODE_GATEUP, 256>(p, max_rows, st);
  return narrow ? launch_dense_m<T, MODE_DOWN, 128>(p, max_rows, st) : launch_dense_m<T, MODE_DOWN, 256>(p, max_rows, st);
}

// Whether launch_dense has a kernel for the launch.
bool dense_takes(int act_dtype, int wtag, int mode, const GemmParams& p, int64_t max_rows) {
  if (!(act_dtype == STMOE_F16 && wtag == WF_DENSE_F16) && !(act_dtype == STMOE_BF16 && wtag == WF_DENSE_BF16)) return false;
  if (p.choices || p.x_scale || (p.offsets ? p.E > 64 : p.fixed_rows >= ((int64_t)1 << 31))) return false;
  if (p.kred % 64 != 0 || p.kred >= (1 << 24) || p.lda % 8 != 0 || p.ldo % 4 != 0 || !aligned16(p.a)) return false;
  if (p.n_out % (mode == MODE_GATEUP ? 64 : 128) != 0) return false;
  // token rows are addressed with 32-bit byte offsets from the activation base
  const int64_t src_rows = p.perm ? (max_rows + p.k_top - 1) / p.k_top : max_rows;
  return src_rows * p.lda * 2 < ((int64_t)1 << 32);
}

int launch_dense(int act_dtype, int wtag, int mode, const GemmParams& p, int64_t max_rows, hipStream_t st) {
  if (max_rows == 0 || p.n_out == 0) return STMOE_OK;
  if (!dense_takes(act_dtype, wtag, mode, p, max_rows))
    return set_error(STMOE_ERR_UNSUPPORTED, "dense kernel: needs 16-bit weights of the activations' type, K %% 64 == 0, output features in "
                     "whole tiles and at most 64 experts");
  return act_dtype == STMOE_F16 ? launch_dense_t<f16_t>(mode, p, max_rows, st) : launch_dense_t<bf16_t>(mode, p, max_rows, st);
}

}  // namespace stmoe
