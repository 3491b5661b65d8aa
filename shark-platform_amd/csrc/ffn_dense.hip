// Prefill kernel for unquantized 16-bit expert weights of the activations' type: 256 (or 128) weight rows x up to 256 token
// rows per workgroup, K step 64, both operands straight from global memory into LDS.
//
// What bounds it: up to some 200 rows per expert the weight stream (a layer of 8 x 3 x 14336 x 4096 in bf16 is 2.8 GB, 430 us
// at the rate of a large copy), beyond that the matrix pipe.  Nothing has to be converted, so there are no loader wavefronts:
// all eight issue their share of the direct loads of a later K step and multiply the current one.
//
//   LDS: three weight stages (32 KB each with BN = 256), so that a stage has two K steps to arrive (64 KB in flight per CU cover
//     the memory latency), and three token stages of 128 or 256 rows; 256 weight rows and 256 token rows leave room for two of
//     them, whose rows come from L2 and have one K step.  (BN = 128 with two token stages of 256 rows: down projection of 515
//     tokens 259 us, with three 197.)  Rows of 128 bytes, XOR-swizzled in 16-byte
//     units (see ffn_mfma_common.h): the direct load puts lane l's 16 bytes at its base + 16 l, so the lanes fetch the units
//     of a row in swizzled order.
//   wavefronts: 4 x 2 (64 x 64 of BN = 256) up to 128 rows, 2 x 4 (128 x 64) above; the rows of a unit are spread evenly over
//     the token groups in multiples of 16 and only the column blocks that hold rows are multiplied.
//   The reduction runs in the order of the 128 x 128 kernel: the sums are the same bits.
// Measured (8 experts of 4096 x 14336, top-2, bf16; gate/up + down, us; 128 x 128 kernel / this one): 100 tokens 421 + 279 /
// 329 + 195, 515 tokens 640 + 313 / 376 + 212 (5 TB/s of weights), 2048 tokens 1916 + 823 / 1025 + 537 (0.92 PFLOP/s; SiLU
// by expf and a division, as the 128 x 128 kernel computes it, is 20 us of the 1025: on the hardware exp2 and reciprocal 1002).
#include "ffn_mfma_common.h"

namespace stmoe {

template <int V> struct DenseInt { static constexpr int value = V; };

template <typename T, int MODE, int BN>
__global__ void __launch_bounds__(512, 1)
grouped_dense_kernel(GemmParams p, int n_tiles) {
  constexpr int BM = 256;
  constexpr int WSTAGE = BN * BIG_LS;  // elements
  extern __shared__ __align__(16) uint16_t lds[];
  BigTile tile;
  if (!big_tile_id(p, BM, n_tiles, false, tile, false, 2)) return;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, n_in = lane & 15;
  const int row_begin = tile.row_begin, rows_here = tile.row_end - tile.row_begin;
  const int nkt = (int)(p.kred >> 6), last = nkt - 1;

  auto unit = [&](auto groups_tag) {
    constexpr int GROUPS = decltype(groups_tag)::value;  // token-row groups of 64 LDS rows
    constexpr int WN = 8 / GROUPS, TI = BN / 16 / WN;    // wavefronts along the features, 16-feature blocks of each
    constexpr int XSTAGE = GROUPS * 64 * BIG_LS;
    constexpr bool XEARLY = GROUPS == 2 || BN == 128;    // token rows two K steps ahead (three stages), else one (two stages)
    constexpr int XSTAGES = XEARLY ? 3 : 2;
    constexpr int WLOADS = BN / 64, XLOADS = GROUPS;     // direct loads of 8 rows per wavefront and K step
    const int rpg = min(64, ((rows_here + GROUPS - 1) / GROUPS + 15) / 16 * 16);  // tile row grp * rpg + i <-> LDS row grp * 64 + i
    uint16_t* const Wbase = lds;               // [3][BN][64]
    uint16_t* const Xbase = lds + 3 * WSTAGE;  // [XSTAGES][64 GROUPS][64]

    // ---- loads: this wavefront's rows are 64 j + 8 wave .. + 7 of either operand's tile
    const char* wsrc[WLOADS];
#pragma unroll
    for (int j = 0; j < WLOADS; ++j) {
      const int r = 64 * j;  // (a block of 64 rows is all gate or all up)
      const bool up = MODE == MODE_GATEUP && r >= BN / 2;
      const WeightView& wv = up ? p.w1 : p.w0;
      const int64_t row = (int64_t)tile.e * wv.rows + (MODE == MODE_GATEUP ? (int64_t)tile.ntile * (BN / 2) + (up ? r - BN / 2 : r)
                                                                           : (int64_t)tile.ntile * BN + r) + wave * 8;
      wsrc[j] = reinterpret_cast<const char*>(wv.qs) + row * p.kred * 2;
    }
    const int unit_off = ((lane & 7) ^ (lane >> 3)) << 4;  // LDS unit lane % 8 of row lane / 8 holds this unit of the row
    const uint32_t woff = (uint32_t)((lane >> 3) * (int)p.kred * 2 + unit_off);
    uint32_t xoff[XLOADS];
#pragma unroll
    for (int j = 0; j < XLOADS; ++j) {
      // LDS rows that hold no tile row re-read a valid one (their outputs are never stored)
      const int i = row_begin + min(j * rpg + min(wave * 8 + (lane >> 3), rpg - 1), rows_here - 1);
      const int64_t src = p.perm ? (int64_t)(p.perm[i] / p.k_top) : (int64_t)i;
      xoff[j] = (uint32_t)(src * p.lda * 2 + unit_off);
    }
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint16_t*)lds);
    const uint32_t w_lds = __builtin_amdgcn_readfirstlane(lds0 + wave * 8 * BIG_LS * 2);
    const uint32_t x_lds = __builtin_amdgcn_readfirstlane(lds0 + (3 * WSTAGE + wave * 8 * BIG_LS) * 2);
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
      b_rd[ks] = Xbase + (wm * 64 + n_in) * BIG_LS + u;
    }
    auto block_row = [](int ti) { return MODE == MODE_GATEUP ? (ti < TI / 2 ? ti * 16 : BN / 2 + (ti - TI / 2) * 16) : ti * 16; };
    floatx4_t acc[TI][4];
#pragma unroll
    for (int a = 0; a < TI; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = (floatx4_t){0.f, 0.f, 0.f, 0.f};

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
    // Order of the loads, and what the waits (at most N of a wavefront's loads still in flight, the N youngest) leave:
    //   XEARLY: W0 X0 W1 X1 | step kt: W(kt+2) X(kt+2); behind its wait W, X(kt+1) have landed: N = WLOADS + XLOADS
    //   else:   W0 X0 W1    | step kt: X(kt+1) W(kt+2); behind its wait W, X(kt+1) have landed: N = WLOADS
    // Step kt overwrites the stages that step kt - 1 read; the barrier at its end lies between.
    constexpr int INFLIGHT = XEARLY ? WLOADS + XLOADS : WLOADS;
    auto k_loop = [&](auto ntj_tag) {
      int ws = 0, xs = 0;
      for (int kt = 0; kt < nkt; ++kt) {
        const int ws2 = ws == 0 ? 2 : ws - 1;  // stage of step kt + 2
        if constexpr (XEARLY) load_w(kt + 2, ws2);
        else load_x(kt + 1, xs ^ 1);
        compute(ntj_tag, ws, xs, 0);
        if constexpr (XEARLY) load_x(kt + 2, ws2);
        else load_w(kt + 2, ws2);
        compute(ntj_tag, ws, xs, 1);
        vm_wait<INFLIGHT>();
        __syncthreads();
        ws = ws == 2 ? 0 : ws + 1;
        xs = xs == XSTAGES - 1 ? 0 : xs + 1;
      }
    };
    load_w(0, 0);
    load_x(0, 0);
    load_w(1, 1);
    if constexpr (XEARLY) load_x(1, 1);
    vm_wait<INFLIGHT>();
    __syncthreads();
    if (ntj == 4) k_loop(DenseInt<4>{});
    else if (ntj == 3) k_loop(DenseInt<3>{});
    else if (ntj == 2) k_loop(DenseInt<2>{});
    else if (ntj == 1) k_loop(DenseInt<1>{});
    else k_loop(DenseInt<0>{});
    vm_wait<0>();  // the requests past the last step: nothing may land in LDS after the workgroup is done

    // ---- results: lane (n_in, g) holds features 4 g .. 4 g + 3 of each block for token row n_in of each column block
    const FakeQuant fq = fq_scale(p);
#pragma unroll
    for (int tj = 0; tj < 4; ++tj) {
      if (tj * 16 + n_in >= my_rows) continue;
      T* orow = reinterpret_cast<T*>(p.out) + out_row(p, row_begin + wm * rpg + tj * 16 + n_in) * p.ldo + 4 * g;
      if constexpr (MODE == MODE_GATEUP) {
        orow += (int64_t)tile.ntile * (BN / 2) + wn * (BN / 2 / WN);
#pragma unroll
        for (int ti = 0; ti < TI / 2; ++ti) {
          const floatx4_t ga = acc[ti][tj], ua = acc[ti + TI / 2][tj];
          const float gq[4] = {ga[0], ga[1], ga[2], ga[3]}, uq[4] = {ua[0], ua[1], ua[2], ua[3]};
          uint2* dst = reinterpret_cast<uint2*>(orow + ti * 16);
          if (p.act == STMOE_ACT_SILU) *dst = gateup_quad<T, ACT_SILU_IEEE>(gq, uq, fq);
          else *dst = gateup_quad<T, STMOE_ACT_GELU_ERF>(gq, uq, fq);
        }
      } else {
        orow += (int64_t)tile.ntile * BN + wn * (BN / WN);
#pragma unroll
        for (int ti = 0; ti < TI; ++ti) {
          const floatx4_t v = acc[ti][tj];
          *reinterpret_cast<uint2*>(orow + ti * 16) = make_uint2(pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]));
        }
      }
    }
  };
  if (rows_here <= BM / 2) unit(DenseInt<2>{});
  else unit(DenseInt<4>{});
}

template <typename T, int MODE, int BN>
static int launch_dense_m(const GemmParams& p, int64_t max_rows, hipStream_t st) {
  // three weight stages and the larger of three token stages of 128 rows and two (BN = 128: three) of 256
  constexpr size_t lds_bytes = (size_t)(3 * BN + (BN == 128 ? 3 : 2) * 256) * BIG_LS * 2;
  static_assert(lds_bytes <= 160 * 1024 && 3 * 128 <= 2 * 256, "stages fit a CU's LDS");
  static std::atomic<uint64_t> lds_ready{0};
  auto kern = grouped_dense_kernel<T, MODE, BN>;
  if (int rc = reserve_lds(reinterpret_cast<const void*>(kern), lds_bytes, lds_ready, "dense kernel")) return rc;
  const int n_tiles = (int)(p.n_out / (MODE == MODE_GATEUP ? BN / 2 : BN));
  const int experts = p.offsets ? p.E : 1;
  const int m_slots = (int)((max_rows + 255) / 256) + experts;
  kern<<<dim3((unsigned)big_grid(n_tiles, m_slots, false)), 512, lds_bytes, st>>>(p, n_tiles);
  return check_launch("grouped_dense");
}
// 128 weight rows per unit instead of 256 while 256 would leave CUs without a unit (a unit per 256 features and expert, and half
// a unit more per 256 rows).  Measured (8 experts, top-2, bf16, us, 256 / 128): gate/up of 1024 features 300 tokens 17 / 12, 2048
// tokens 36 / 32; of 4096 features 80 tokens 43 / 46; of 14336 515 tokens 374 / 406.  Down to 4096 features from 14336: 515 tokens
// 267 / 197, 1024 tokens 346 / 422; to 2048 from 4096, 1500 tokens 98 / 58.
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
