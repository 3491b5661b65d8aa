// Grouped projection with fp32 activations on the matrix cores (v_mfma_f32_16x16x4_f32: products and sums in fp32).
//
// What bounds it: the layers that run in fp32 are small (8 experts of a few hundred by a thousand), every expert has a few
// rows, and a launch is one sweep over the expert weights.  With one wavefront per output value, as the general kernel
// computes, every weight is read once per row of its expert and a wavefront lives for a handful of loads; here 16 weight rows
// meet 16, 32 or 64 token rows per sweep.  A workgroup takes one expert and 16 output features (GATEUP: of gate and up; DOWN:
// 32 features where they divide), its four wavefronts a quarter of the reduction each: a layer of 8 x 1024 x 512 has 512 such
// items, 2048 wavefronts, whose loads are all in flight after two steps.  The quarters are added through LDS in a fixed order.
// Measured (8 experts, top-2, gate/up + down, us; general kernel / this one): 64 tokens of 512 x 1024 71 + 33 / 17 + 11; the
// whole layer 110 / 38 us, of which the host takes 31.  109 tokens of 896 x 1280: layer 325 / 69 us; 101 tokens of 256 x 1152
// 154 / 47.  At 10 tokens of 768 x 1536 the gate/up launch reads 3.3 TB/s; with 25 rows per expert and more the time goes into the
// multiplications (32 cycles each for 16 x 16 x 4).  Eight wavefronts per item instead of four: no change.
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

// One chunk of 64 reduction elements of one row: value(4 i + r) is the lane's element of MFMA step 4 i + r.
template <int WF> struct F32Weight {
  static constexpr bool kRowContiguous = false;
  Chunk16<WF> c;
  __device__ __forceinline__ void load(const WeightView& w, int64_t e, int64_t n, int64_t k, int g, bool ok) {
    if (ok) c.load(w, e, n, k + 16 * g);
    else c.zero();
  }
  __device__ __forceinline__ void values(float (&v)[16]) const { c.to_f32(v); }
};
template <> struct F32Weight<WF_DENSE_F32> {
  static constexpr bool kRowContiguous = true;
  floatx4_t q[4];
  __device__ __forceinline__ void load(const WeightView& w, int64_t e, int64_t n, int64_t k, int g, int blocks) {
    const float* p = reinterpret_cast<const float*>(w.qs) + (e * w.rows + n) * w.cols + k + 4 * g;
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = i < blocks ? *reinterpret_cast<const floatx4_t*>(p + 16 * i) : (floatx4_t){0.f, 0.f, 0.f, 0.f};
  }
  __device__ __forceinline__ void values(float (&v)[16]) const {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = q[i >> 2][i & 3];
  }
};

template <int WF, int MODE, int NT, int MT>
__device__ __forceinline__ void f32_pass(const GemmParams& p, int e, const int64_t (&wrow)[NT], int tile, int r0, int re, int lane, int wave,
                                         floatx4_t (*red)[64]) {
  constexpr bool ROWC = F32Weight<WF>::kRowContiguous;
  const int g = lane >> 4, n_in = lane & 15;
  const int nch = (int)((p.kred + 63) >> 6), c_begin = nch * wave / 4, c_end = nch * (wave + 1) / 4;
  const float* xrow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int i = min(r0 + mt * 16 + n_in, re - 1);  // rows past the end re-read the last one (never stored)
    const int64_t src = p.perm ? (int64_t)(p.perm[i] / p.k_top) : (int64_t)i;
    xrow[mt] = reinterpret_cast<const float*>(p.a) + src * p.lda;
  }
  floatx4_t acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[mt][t] = (floatx4_t){0.f, 0.f, 0.f, 0.f};

  // (the reduction length is a multiple of 16: a chunk's 16-element pieces are whole, those past the end read as zeros)
  auto blocks_of = [&](int c) { return (int)min((int64_t)4, (p.kred - (int64_t)c * 64) >> 4); };
  auto load_w = [&](F32Weight<WF> (&w)[NT], int c) {
    const int blocks = blocks_of(c);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const WeightView& wv = MODE == MODE_GATEUP && t == 1 ? p.w1 : p.w0;
      if constexpr (ROWC) w[t].load(wv, e, wrow[t], (int64_t)c * 64, g, blocks);
      else w[t].load(wv, e, wrow[t], (int64_t)c * 64, g, g < blocks);
    }
  };
  auto load_x = [&](floatx4_t (&x)[MT][4], int c) {
    const int blocks = blocks_of(c);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool ok = ROWC ? i < blocks : g < blocks;
        x[mt][i] = ok ? *reinterpret_cast<const floatx4_t*>(xrow[mt] + (int64_t)c * 64 + (ROWC ? 16 * i + 4 * g : 16 * g + 4 * i)) : (floatx4_t){0.f, 0.f, 0.f, 0.f};
      }
  };
  auto multiply = [&](const F32Weight<WF> (&w)[NT], const floatx4_t (&x)[MT][4]) {
    float v[NT][16];
#pragma unroll
    for (int t = 0; t < NT; ++t) w[t].values(v[t]);
    // A chunk's sixteen instructions are eight chains of two, which start at zero and are added in pairs; the chunk's sum then
    // goes to the running one.
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        floatx4_t half[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          floatx4_t c[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t][8 * h + 2 * i], x[mt][2 * h + (i >> 1)][(2 * i) & 3], (floatx4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t][8 * h + 2 * i + 1], x[mt][2 * h + (i >> 1)][(2 * i + 1) & 3], c[i], 0, 0, 0);
          half[h] = (c[0] + c[1]) + (c[2] + c[3]);
        }
        acc[mt][t] += half[0] + half[1];
        // (finished here: sunk behind the next chunk's loads, the adds would keep the chains of all tiles in registers)
        asm volatile("" : "+v"(acc[mt][t]));
      }
  };
  if (c_begin < c_end) {
    // Both operands one chunk ahead while the registers allow it (four token tiles: the weights only).  Requests are
    // unconditional (past the end the last chunk again), so that no wait covers a younger one.
    F32Weight<WF> w0[NT], w1[NT];
    floatx4_t x0[MT][4], x1[MT <= 2 ? MT : 1][4];
    load_w(w0, c_begin);
    load_x(x0, c_begin);
    // (one copy of the 64 to 256 multiplications: two alternating buffers doubled the code and measured up to a fifth slower)
#pragma unroll 1
    for (int c = c_begin; c < c_end; ++c) {
      const int c1 = min(c + 1, c_end - 1);
      load_w(w1, c1);
      if constexpr (MT <= 2) load_x(x1, c1);
      multiply(w0, x0);
      if constexpr (MT > 2) load_x(x0, c1);
#pragma unroll
      for (int t = 0; t < NT; ++t) w0[t] = w1[t];
      if constexpr (MT <= 2) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int i = 0; i < 4; ++i) x0[mt][i] = x1[mt][i];
      }
    }
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
template <int WF, int MODE, int NT>
__global__ void __launch_bounds__(256, 2) grouped_f32_kernel(GemmParams p) {
  __shared__ floatx4_t red[4 * NT * 4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int e = blockIdx.y, tile = blockIdx.x;
  int rb, re;
  expert_range(p, e, rb, re);
  int64_t wrow[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)  // features past the end re-read the last one (never stored)
    wrow[t] = min((int64_t)tile * (MODE == MODE_GATEUP ? 16 : 16 * NT) + (MODE == MODE_GATEUP ? 0 : 16 * t) + (lane & 15), p.n_out - 1);
  for (int r0 = rb + 64 * (int)blockIdx.z; r0 < re; r0 += 64 * (int)gridDim.z) {
    const int left = re - r0;
    if (left <= 16) f32_pass<WF, MODE, NT, 1>(p, e, wrow, tile, r0, re, lane, wave, red);
    else if (left <= 32) f32_pass<WF, MODE, NT, 2>(p, e, wrow, tile, r0, re, lane, wave, red);
    else f32_pass<WF, MODE, NT, 4>(p, e, wrow, tile, r0, min(re, r0 + 64), lane, wave, red);
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
  grouped_f32_kernel<WF, MODE, NT><<<dim3((unsigned)tiles, (unsigned)experts, (unsigned)passes), 256, 0, st>>>(p);
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
