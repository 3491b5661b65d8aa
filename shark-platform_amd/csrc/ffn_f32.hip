// Grouped projection with fp32 activations on the matrix cores (v_mfma_f32_16x16x4_f32: products and sums in fp32).
//
// What bounds it: the layers that run in fp32 are small (8 experts of a few hundred by a thousand), every expert has a few
// rows, and a launch is one sweep over the expert weights.  With one wavefront per output value, as the general kernel
// computes, every weight is read once per row of its expert and a wavefront lives for a handful of loads; here 16 weight rows
// meet 16, 32 or 64 token rows per sweep.  A workgroup takes one expert and 16 output features (GATEUP: of gate and up; DOWN:
// 32 features where they divide), its four wavefronts a quarter of the reduction each: a layer of 8 x 1024 x 512 has 512 such
// items, 2048 wavefronts, whose loads are all in flight after two steps.  The quarters are added through LDS in a fixed order.
// Order of the loads: they return in the order of their issue, so the tokens of an item's rows are requested first, then its weights, then
// the token rows; two chunks of both are in flight up to 32 rows, of the weights alone from 33 rows on, every load unconditional (a row's
// ragged end re-reads its last piece and drops it in registers: an instance of its own, TAIL).  With one chunk ahead, each load under its own condition, and the wavefront's number in a vector
// register, every wait was for all loads in flight: 64 tokens of 512 x 1024 16.8 + 12.0 us; now 12.6 + 8.3.  Layer (8 experts, top-2, us,
// before / now): 64 tokens of 512 x 1024 37.0 / 29.5, 109 tokens of 896 x 1280 74 / 66, 128 tokens of 1024 x
// 1536 85 / 75; Q8_0 weights of 1024 x 1024, 2000 tokens 432 / 342; one Q8_0 matrix of [2048, 2048], 60 rows 28.7 / 19.0.  (On the general
// kernel the first took 110.)  Weights requested in front of the tokens: 3 us more.
// Registers: all 256 are in use, and a register in scratch memory comes back through the same in-order path as the loads ahead of it.  So
// a weight row is converted and multiplied with all token rows before the next one is (with both in any order ten of 54 instances
// kept 12 to 44 bytes a lane in scratch memory: 3000 launches of 1 to 16 experts, 256 to 2048 x 128 to 2048, 1 to 100 rows per expert, plain
// and quantized weights, take 0.872 of the time of the first order of loads with it and 0.843 without, slower by more than 3 % 1.8 and 0.3 %).
// Order of the sums: the matrix instruction rounds after every product, so one running sum per quarter was up to 3.6 times as far
// from fp64 as the general kernel, whose 64 lanes hold short sums (K = 4096: rms error 9.6 / 2.7 times 2^-24 of the result's rms;
// K = 512: 3.5 / 1.6).  A chunk of 64 elements is eight sums of 8 products, added in pairs: 1.9 and 1.4, below the general kernel at
// every K from 64 to 4096.  The additions run beside the other wavefront's products: layers of the sizes above 0 to 4 % slower, a
// product of 2000 x 1024 x 1024 6 % faster.
//
// Operands: weight rows are the MFMA "A" rows, token rows the "B" columns; one step multiplies 4 reduction elements, one per
// lane group.  The operands only have to agree on which element a lane holds, so a lane loads what is contiguous for it:
//   plain fp32 weights: 16 bytes, elements 16 i + 4 g .. + 3 of a chunk of 64 (a load instruction reads 64 bytes of a row)
//   the other formats:  the 16 elements 16 g .. 16 g + 15 of the chunk (Chunk16), widened to fp32
// and the token operand follows.
#include "ffn_kernels.h"

namespace stmoe {

typedef float floatx4_t __attribute__((ext_vector_type(4)));

// One chunk of 64 reduction elements of one row: value(4 i + r) is the lane's element of MFMA step 4 i + r.  `TAIL`:
// a row's last chunk may have `blocks` < 4 pieces of 16 elements: the loads read the last one again, drop() puts zeros there.
template <int WF, bool TAIL> struct F32Weight {
  static constexpr bool kRowContiguous = false;
  Chunk16<WF> c;
  __device__ __forceinline__ void load(const WeightView& w, int64_t e, int64_t n, int64_t k, int g, int blocks) {
    c.load(w, e, n, k + 16 * (TAIL ? min(g, blocks - 1) : g));
  }
  __device__ __forceinline__ void drop(int g, int blocks) {
    if (g >= blocks) c.zero();
  }
  __device__ __forceinline__ void values(float (&v)[16]) const { c.to_f32(v); }
};
template <bool TAIL> struct F32Weight<WF_DENSE_F32, TAIL> {
  static constexpr bool kRowContiguous = true;
  floatx4_t q[4];
  __device__ __forceinline__ void load(const WeightView& w, int64_t e, int64_t n, int64_t k, int g, int blocks) {
    const float* p = reinterpret_cast<const float*>(w.qs) + (e * w.rows + n) * w.cols + k + 4 * g;
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = *reinterpret_cast<const floatx4_t*>(p + 16 * (TAIL ? min(i, blocks - 1) : i));
  }
  __device__ __forceinline__ void drop(int, int blocks) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i >= blocks) q[i] = (floatx4_t){0.f, 0.f, 0.f, 0.f};
  }
  __device__ __forceinline__ void values(float (&v)[16]) const {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = q[i >> 2][i & 3];
  }
};

// A wavefront's quarter of the reduction, [begin, end) in chunks, and its weight rows.
template <int WF, int MODE, int NT, bool TAIL> struct F32Quarter {
  int begin, end;
  int64_t wrow[NT];
  F32Weight<WF, TAIL> w[2][NT];
  // (the reduction length is a multiple of 16: a chunk's 16-element pieces are whole)
  static __device__ __forceinline__ int blocks_of(const GemmParams& p, int c) { return (int)min((int64_t)4, (p.kred - (int64_t)c * 64) >> 4); }
  __device__ __forceinline__ void load(const GemmParams& p, int e, int g, int slot, int c) {
    const int blocks = blocks_of(p, c);
#pragma unroll
    for (int t = 0; t < NT; ++t) w[slot][t].load(MODE == MODE_GATEUP && t == 1 ? p.w1 : p.w0, e, wrow[t], (int64_t)c * 64, g, blocks);
  }
  __device__ __forceinline__ void load_first(const GemmParams& p, int e, int g) {
#pragma unroll
    for (int j = 0; j < 2; ++j) load(p, e, g, j, max(min(begin + j, end - 1), 0));
  }
};

template <int WF, int MODE, int NT, bool TAIL, int MT>
__device__ __forceinline__ void f32_pass(const GemmParams& p, int e, F32Quarter<WF, MODE, NT, TAIL>& quarter, int tile, int r0, int re, int lane, int wave,
                                         floatx4_t (*red)[64]) {
  constexpr bool ROWC = F32Weight<WF, TAIL>::kRowContiguous;
  // (plain fp32 weights: the lane's addresses are computed in each pass; kept for all three, seven registers went to scratch memory)
  if (ROWC) asm volatile("" : "+v"(lane));
  const int g = lane >> 4, n_in = lane & 15;
  const int c_begin = quarter.begin, c_end = quarter.end;
  const float* xrow[MT];
  int src[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) src[mt] = min(r0 + mt * 16 + n_in, re - 1);  // rows past the end re-read the last one (never stored)
  if (p.perm) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) src[mt] = p.perm[src[mt]];
  }
  // The weights are on their way while the tokens of the rows and then the token rows are fetched.  (Behind the tokens: loads return in order.)
  __builtin_amdgcn_sched_barrier(0);
  quarter.load_first(p, e, g);
  __builtin_amdgcn_sched_barrier(0);
  if (p.perm) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) src[mt] /= p.k_top;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) xrow[mt] = reinterpret_cast<const float*>(p.a) + (int64_t)src[mt] * p.lda;
  floatx4_t acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[mt][t] = (floatx4_t){0.f, 0.f, 0.f, 0.f};

  auto load_x = [&](floatx4_t (&x)[MT][4], int c) {
    const int blocks = quarter.blocks_of(p, c);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        x[mt][i] = *reinterpret_cast<const floatx4_t*>(xrow[mt] + (int64_t)c * 64 + (ROWC ? 16 * (TAIL ? min(i, blocks - 1) : i) + 4 * g : 16 * (TAIL ? min(g, blocks - 1) : g) + 4 * i));
  };
  auto multiply = [&](F32Weight<WF, TAIL> (&w)[NT], floatx4_t (&x)[MT][4], int c) {
    const int blocks = quarter.blocks_of(p, c);
    if (TAIL && blocks < 4) {
#pragma unroll
      for (int t = 0; t < NT; ++t) w[t].drop(g, blocks);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if ((ROWC ? i : g) >= blocks) x[mt][i] = (floatx4_t){0.f, 0.f, 0.f, 0.f};
    }
    // A chunk's sixteen instructions are eight chains of two, which start at zero and are added in pairs; the chunk's sum then
    // goes to the running one.
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      float v[16];
      w[t].values(v);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        floatx4_t half[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          floatx4_t c[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[8 * h + 2 * i], x[mt][2 * h + (i >> 1)][(2 * i) & 3], (floatx4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[8 * h + 2 * i + 1], x[mt][2 * h + (i >> 1)][(2 * i + 1) & 3], c[i], 0, 0, 0);
          half[h] = (c[0] + c[1]) + (c[2] + c[3]);
        }
        acc[mt][t] += half[0] + half[1];
        // (finished here: sunk behind the next chunk's loads, the adds would keep the chains of all tiles in registers)
        asm volatile("" : "+v"(acc[mt][t]));
        if (mt == MT - 1) __builtin_amdgcn_sched_barrier(0);  // (see the head: no register may go to scratch memory)
      }
    }
  };
  // No request is under a condition of its own: such loads were waited for one by one.
  if (MT > 2 && c_begin < c_end) {
    // The weights two chunks ahead (for more token rows there are no registers).  One copy of the 128 to 256 multiplications: two
    // alternating buffers doubled the code and measured up to a fifth slower.
    floatx4_t x[MT][4];
#pragma unroll 1
    for (int c = c_begin; c < c_end; ++c) {
      load_x(x, c);
      multiply(quarter.w[0], x, c);
#pragma unroll
      for (int t = 0; t < NT; ++t) quarter.w[0][t] = quarter.w[1][t];
      quarter.load(p, e, g, 1, min(c + 2, c_end - 1));
    }
  }
  if (MT <= 2 && c_begin < c_end) {
    // Both operands two chunks ahead; none is requested that nobody reads, except that an odd last chunk is requested twice.
    floatx4_t x[2][MT][4];
    load_x(x[0], c_begin);
    load_x(x[1], min(c_begin + 1, c_end - 1));
    int c = c_begin;
#pragma unroll 1
    for (; c + 2 < c_end; c += 2) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        multiply(quarter.w[j], x[j], c + j);
        const int ahead = min(c + j + 2, c_end - 1);
        quarter.load(p, e, g, j, ahead);
        load_x(x[j], ahead);
      }
    }
    multiply(quarter.w[0], x[0], c);
    if (c + 1 < c_end) multiply(quarter.w[1], x[1], c + 1);
  }

  // the four quarters, ((0 + 1) + (2 + 3)); wavefront w finishes token tile w
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < NT; ++t) red[(mt * NT + t) * 4 + wave][lane] = acc[mt][t];
  __syncthreads();
  if (wave < MT) {
    const int mt = wave, i = r0 + mt * 16 + n_in;
    floatx4_t sum[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const floatx4_t(*q)[64] = red + (mt * NT + t) * 4;
      sum[t] = (q[0][lane] + q[1][lane]) + (q[2][lane] + q[3][lane]);
    }
    if (i < re) {
      const float scale = p.x_scale ? *p.x_scale : 1.0f;
      float* orow = reinterpret_cast<float*>(p.out) + out_row(p, i) * p.ldo;
      auto store = [&](int64_t n, const floatx4_t& v) {  // features n .. n + 3
        if (n + 3 < p.n_out && (p.ldo & 3) == 0) {
          *reinterpret_cast<floatx4_t*>(orow + n) = v;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < p.n_out) orow[n + r] = v[r];
        }
      };
      if constexpr (MODE == MODE_GATEUP) {
        const FakeQuant fq = fq_scale(p);
        floatx4_t v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = gateup_epilogue<float>(p.act, sum[0][r], sum[1][r], scale, fq);
        store((int64_t)tile * 16 + 4 * g, v);
      } else {
#pragma unroll
        for (int t = 0; t < NT; ++t) store((int64_t)tile * 16 * NT + 16 * t + 4 * g, sum[t] * scale);
      }
    }
  }
  __syncthreads();  // the buffer is reused by the next pass
}

// grid: (feature tiles, experts, passes in flight)
template <int WF, int MODE, int NT, bool TAIL>
__global__ void __launch_bounds__(256, 2) grouped_f32_kernel(GemmParams p) {
  __shared__ floatx4_t red[4 * NT * 4][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int e = blockIdx.y, tile = blockIdx.x;
  const int nch = (int)((p.kred + 63) >> 6);
  F32Quarter<WF, MODE, NT, TAIL> quarter;
  quarter.begin = nch * wave / 4;
  quarter.end = nch * (wave + 1) / 4;
#pragma unroll
  for (int t = 0; t < NT; ++t)
    // Features past the end re-read the last one (never stored).  A quarter without a chunk (fewer than 256 elements) requests one all the
    // same, and all its lanes the same row's: down projection of 64 elements, 87 tokens of 6 of 56 experts, 4064 features 67 -> 43 us.
    quarter.wrow[t] = min((int64_t)tile * (MODE == MODE_GATEUP ? 16 : 16 * NT) + (MODE == MODE_GATEUP ? 0 : 16 * t) + (quarter.begin < quarter.end ? lane & 15 : 0), p.n_out - 1);
  int rb, re;
  expert_range(p, e, rb, re);
  for (int r0 = rb + 64 * (int)blockIdx.z; r0 < re; r0 += 64 * (int)gridDim.z) {
    const int left = re - r0;
    if (left <= 16) f32_pass<WF, MODE, NT, TAIL, 1>(p, e, quarter, tile, r0, re, lane, wave, red);
    else if (left <= 32) f32_pass<WF, MODE, NT, TAIL, 2>(p, e, quarter, tile, r0, re, lane, wave, red);
    else f32_pass<WF, MODE, NT, TAIL, 4>(p, e, quarter, tile, r0, min(re, r0 + 64), lane, wave, red);
  }
}

template <int WF, int MODE, int NT>
static int launch_f32_nt(const GemmParams& p, int64_t max_rows, hipStream_t st) {
  const int64_t tiles = (p.n_out + (MODE == MODE_GATEUP ? 15 : 16 * NT - 1)) / (MODE == MODE_GATEUP ? 16 : 16 * NT);
  const int64_t experts = p.offsets ? p.E : 1;
  // passes of 64 rows side by side, as many as one expert can have and as keep the grid within some thousand workgroups
  const int64_t rows = p.expert_rows_bound > 0 && p.expert_rows_bound < max_rows ? p.expert_rows_bound : max_rows;
  const int64_t passes = std::min<int64_t>((rows + 63) / 64, std::max<int64_t>(1, 8192 / (tiles * experts)));
  if (experts > 65535 || tiles >= ((int64_t)1 << 31)) return set_error(STMOE_ERR_UNSUPPORTED, "f32 kernel: %lld experts exceed its grid", (long long)experts);
  const dim3 grid((unsigned)tiles, (unsigned)experts, (unsigned)passes);
  if (p.kred % 64 == 0) grouped_f32_kernel<WF, MODE, NT, false><<<grid, 256, 0, st>>>(p);
  else grouped_f32_kernel<WF, MODE, NT, true><<<grid, 256, 0, st>>>(p);
  return check_launch("grouped_f32");
}
template <int WF>
static int launch_f32_t(int mode, const GemmParams& p, int64_t max_rows, hipStream_t st) {
  if (mode == MODE_GATEUP) return launch_f32_nt<WF, MODE_GATEUP, 2>(p, max_rows, st);
  // DOWN: 16 features per item while 32 would leave CUs without one
  const int64_t experts = p.offsets ? std::min<int64_t>(p.E, max_rows) : 1;
  return (p.n_out + 31) / 32 * experts >= 512 ? launch_f32_nt<WF, MODE_DOWN, 2>(p, max_rows, st) : launch_f32_nt<WF, MODE_DOWN, 1>(p, max_rows, st);
}

int launch_f32(int wtag, int mode, const GemmParams& p, int64_t max_rows, hipStream_t st) {
  if (max_rows == 0 || p.n_out == 0) return STMOE_OK;
  if (p.kred % 16 != 0 || p.lda % 4 != 0)
    return set_error(STMOE_ERR_UNSUPPORTED, "f32 kernel: needs K %% 16 == 0 and 16-byte aligned rows");
  switch (wtag) {
    case WF_Q8_0: return launch_f32_t<WF_Q8_0>(mode, p, max_rows, st);
    case WF_Q4_1: return launch_f32_t<WF_Q4_1>(mode, p, max_rows, st);
    case WF_FP8_F32D: return launch_f32_t<WF_FP8_F32D>(mode, p, max_rows, st);
    case WF_DENSE_F32: return launch_f32_t<WF_DENSE_F32>(mode, p, max_rows, st);
    case WF_DENSE_F16: return launch_f32_t<WF_DENSE_F16>(mode, p, max_rows, st);
    case WF_DENSE_BF16: return launch_f32_t<WF_DENSE_BF16>(mode, p, max_rows, st);
    case WF_Q8_0_P: return launch_f32_t<WF_Q8_0_P>(mode, p, max_rows, st);
    case WF_Q4_1_P: return launch_f32_t<WF_Q4_1_P>(mode, p, max_rows, st);
    case WF_FP8_F32D_P: return launch_f32_t<WF_FP8_F32D_P>(mode, p, max_rows, st);
    default: return set_error(STMOE_ERR_UNSUPPORTED, "f32 kernel: no instantiation for weight tag %d", wtag);
  }
}

}  // namespace stmoe
