// RMSNorm kernels (bf16, fp32 accumulation) for CDNA4.
//
// Capability parity: the fused rmsnorm+residual epilogue the reference
// delegates to its vLLM containers.
//
// One 256-thread workgroup per token row; bf16x8 vector loads (16 B/lane);
// row held in registers between the sum-of-squares pass and the scale pass
// (template ITERS gives compile-time register indexing).
//
// Few rows (a decode step) take the time of one chain of loads, sums and
// stores: the weight is requested with the row (AHEAD), the new residual is
// written behind the sums. Many rows are bound by memory, and what the weight
// takes of the registers costs workgroups in flight. us a call, the weight and
// the residual in the plain order and this (residual added, bf16 out): 4096
// wide, 1 row 2.6 and 2.3, 64 rows 2.9 and 2.5, 1024 7.2 and 7.1, 4099 22.2
// and 22.1; 16384 wide, 1 row 5.2 and 3.9, 64 rows 6.6 and 5.3. A step of eight
// layers, with sums by exchanges among registers and rope's cache slot requested
// early: 897 and 890 us at one row, 1723 and 1708 at six with long contexts.

#include "common.h"

namespace fi {

// ITERS = ceil(hidden / (256 threads * 8 elems)); supports hidden <= ITERS*2048.
// FP8_OUT: `out` is u8 (OCP e4m3) and a per-row dynamic scale is written to
// `out_scales` — the fused epilogue for the fp8 serving mode (the normalized
// row only feeds a fp8 GEMM there, so the bf16 intermediate is never
// materialized).
// AHEAD: the weight is requested with the row, not behind the sums.
// F32_IN: the rows of `in` are fp32.
template <int ITERS, bool FUSED_ADD, bool FP8_OUT, bool AHEAD,
          bool F32_IN = false>
__global__ __launch_bounds__(256) void rms_norm_kernel(
    void* __restrict__ out_p,       // [T, H] bf16 (FP8_OUT: u8 e4m3)
    float* __restrict__ out_scales, // [T] (FP8_OUT only; else nullptr)
    const void* __restrict__ in_p,  // [T, H]  (FUSED_ADD: the just-computed layer output x)
    u16* __restrict__ residual,     // [T, H]  in/out (FUSED_ADD only; else nullptr)
    const u16* __restrict__ weight, // [H]
    const float eps,
    const int hidden) {
  const int row = blockIdx.x;
  const int tid = threadIdx.x;
  const int64_t base = static_cast<int64_t>(row) * hidden;

  const u16* in = static_cast<const u16*>(in_p);
  constexpr int kRowsAtOnce = 2048;       // eight workgroups a CU
  constexpr int kSecondFirst = ITERS > 1;
  float vals[ITERS][8];
  bf16x8 wt[ITERS];
  float sumsq = 0.f;
  // the new residual is written behind the sums, whose barriers would wait
  // for it; with more rows than the chip holds at once it goes out before,
  // beside other rows' loads
  const bool late = AHEAD && gridDim.x <= kRowsAtOnce;
  auto keep = [&](int it) {
    const int col = (it * blockDim.x + tid) * 8;
    bf16x8 nr;
#pragma unroll
    for (int j = 0; j < 8; ++j) nr.h[j] = f32_to_bf16(vals[it][j]);
    *reinterpret_cast<bf16x8*>(residual + base + col) = nr;
  };

#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int col = (it * blockDim.x + tid) * 8;
    if (col < hidden) {
      typedef __attribute__((ext_vector_type(8))) float floatx8;
      bf16x8 v;
      floatx8 vf;
      if (F32_IN)
        vf = *reinterpret_cast<const floatx8*>(
            static_cast<const float*>(in_p) + base + col);
      else
        v = *reinterpret_cast<const bf16x8*>(in + base + col);
      if (AHEAD) wt[it] = *reinterpret_cast<const bf16x8*>(weight + col);
      if (FUSED_ADD) {
        bf16x8 r = *reinterpret_cast<const bf16x8*>(residual + base + col);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          vals[it][j] = bf16_to_f32(v.h[j]) + bf16_to_f32(r.h[j]);
        if (!late) keep(it);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          vals[it][j] = F32_IN ? vf[j] : bf16_to_f32(v.h[j]);
      }
      // in an order that is written out: left to the compiler, which of the
      // first two squares is rounded before it is added changes with what
      // surrounds the loop, and outputs with it
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x = vals[it][it == 0 && j < 2 ? j ^ kSecondFirst : j];
        sumsq = fmaf(x, x, sumsq);
      }
    }
  }

  __shared__ float scratch[4];
  sumsq = wave_reduce_sum(sumsq);
  sumsq = block_reduce_sum<4>(sumsq, scratch);
  const float inv_rms = rsqrtf(sumsq / hidden + eps);
  auto weight_of = [&](int it) {
    return AHEAD ? wt[it]
                 : *reinterpret_cast<const bf16x8*>(
                       weight + (it * blockDim.x + tid) * 8);
  };

  if (FP8_OUT) {
    // a second block reduce for the row absmax of the normalized values ->
    // per-row scale -> pack via v_cvt_pk_fp8_f32
    float amax = 0.f;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int col = (it * blockDim.x + tid) * 8;
      if (col < hidden) {
        const bf16x8 w = weight_of(it);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float y = vals[it][j] * inv_rms * bf16_to_f32(w.h[j]);
          amax = fmaxf(amax, fabsf(y));
          if (!AHEAD) vals[it][j] = y;
        }
      }
    }
    __shared__ float scratch_max[4];
    amax = wave_reduce_max(amax);
    amax = block_reduce_max<4>(amax, scratch_max);
    const float scale = fmaxf(amax, 1e-8f) / 448.0f;
    const float inv_scale = 1.f / scale;
    if (tid == 0) out_scales[blockIdx.x] = scale;
    unsigned char* out8 = static_cast<unsigned char*>(out_p);
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int col = (it * blockDim.x + tid) * 8;
      if (col < hidden) {
        float sv[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float y = AHEAD ? vals[it][j] * inv_rms *
                                      bf16_to_f32(wt[it].h[j])
                                : vals[it][j];
          sv[j] = y * inv_scale;
        }
        u32 packed[2];
        pack_fp8x8(sv, packed);
        *reinterpret_cast<u32*>(out8 + base + col) = packed[0];
        *reinterpret_cast<u32*>(out8 + base + col + 4) = packed[1];
        if (FUSED_ADD && late) keep(it);
      }
    }
  } else {
    u16* out = static_cast<u16*>(out_p);
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int col = (it * blockDim.x + tid) * 8;
      if (col < hidden) {
        const bf16x8 w = weight_of(it);
        bf16x8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          o.h[j] = f32_to_bf16(vals[it][j] * inv_rms * bf16_to_f32(w.h[j]));
        *reinterpret_cast<bf16x8*>(out + base + col) = o;
        if (FUSED_ADD && late) keep(it);
      }
    }
  }
}

template <bool FUSED_ADD, bool FP8_OUT, bool F32_IN = false>
void launch_norm(void* out, float* out_scales, const void* in,
                     u16* residual, const u16* weight, float eps, int tokens,
                     int hidden, hipStream_t stream) {
  dim3 grid(tokens), block(256);
  const int iters = ceil_div(hidden, 256 * 8);
  // With the weight ahead of the sums rows of more than 12288 values take 126
  // to 169 registers instead of 70 to 96: half the workgroups in flight. 1024
  // rows of 16384, residual added, e4m3 out: 28.9 us, and 20.2 behind them;
  // 14336 18.9 and 17.4. Up to 12288 the two differ by 2 % either way.
  constexpr int kAlwaysAhead = 6;
#define FI_LAUNCH(N, AHEAD)                                                  \
  hipLaunchKernelGGL(                                                        \
      (rms_norm_kernel<N, FUSED_ADD, FP8_OUT, AHEAD, F32_IN>), grid, block,  \
      0, stream, out, out_scales, in, residual, weight, eps, hidden)
#define FI_CASE(N)                                                           \
  case N:                                                                    \
    if (N <= kAlwaysAhead || tokens <= 256)                                  \
      FI_LAUNCH(N, true);                                                    \
    else                                                                     \
      FI_LAUNCH(N, N <= kAlwaysAhead);                                       \
    break;
  switch (iters) {
    FI_CASE(1)
    FI_CASE(2)
    FI_CASE(3)
    FI_CASE(4)
    FI_CASE(5)
    FI_CASE(6)
    FI_CASE(7)
    FI_CASE(8)
    default:
      // hidden > 16384 unsupported by this kernel family
      abort();
  }
#undef FI_CASE
#undef FI_LAUNCH
}

template <bool FUSED_ADD, bool FP8_OUT>
void launch_rms_norm(void* out, float* out_scales, const u16* in,
                     u16* residual, const u16* weight, float eps, int tokens,
                     int hidden, hipStream_t stream) {
  launch_norm<FUSED_ADD, FP8_OUT>(out, out_scales, in, residual, weight, eps,
                                  tokens, hidden, stream);
}

void launch_stream_norm(u16* out, const float* in, const u16* weight,
                        float eps, int tokens, int hidden,
                        hipStream_t stream) {
  launch_norm<false, false, true>(out, nullptr, in, nullptr, weight, eps,
                                  tokens, hidden, stream);
}

template void launch_rms_norm<true, false>(void*, float*, const u16*, u16*,
                                           const u16*, float, int, int,
                                           hipStream_t);
template void launch_rms_norm<false, false>(void*, float*, const u16*, u16*,
                                            const u16*, float, int, int,
                                            hipStream_t);
template void launch_rms_norm<true, true>(void*, float*, const u16*, u16*,
                                          const u16*, float, int, int,
                                          hipStream_t);
template void launch_rms_norm<false, true>(void*, float*, const u16*, u16*,
                                           const u16*, float, int, int,
                                           hipStream_t);

// stream = x in fp32, scaled = x times weight, squares[row] = their sum
template <class X>
__global__ __launch_bounds__(256) void stream_begin_kernel(
    float* __restrict__ stream, u16* __restrict__ scaled,
    float* __restrict__ squares, const X* __restrict__ x,
    const u16* __restrict__ weight, const int hidden) {
  typedef __attribute__((ext_vector_type(8))) float floatx8;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * hidden;
  float sum = 0.f;
  for (int col = threadIdx.x * 8; col < hidden; col += 256 * 8) {
    floatx8 v;
    if constexpr (sizeof(X) == 4) {
      v = *reinterpret_cast<const floatx8*>(x + base + col);
    } else {
      const bf16x8 h = *reinterpret_cast<const bf16x8*>(x + base + col);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = bf16_to_f32(h.h[j]);
    }
    bf16x8 g;
    __builtin_memcpy(&g, weight + col, sizeof(g));   // on any grid
    bf16x8 y;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      y.h[j] = f32_to_bf16(v[j] * bf16_to_f32(g.h[j]));
      sum = fmaf(v[j], v[j], sum);
    }
    *reinterpret_cast<floatx8*>(stream + base + col) = v;
    *reinterpret_cast<bf16x8*>(scaled + base + col) = y;
  }
  __shared__ float scratch[4];
  sum = block_reduce_sum<4>(wave_reduce_sum(sum), scratch);
  if (threadIdx.x == 0) squares[blockIdx.x] = sum;
}

template <class X>
void launch_stream_begin(float* stream, u16* scaled, float* squares,
                         const X* x, const u16* weight, int rows, int hidden,
                         hipStream_t s) {
  hipLaunchKernelGGL(stream_begin_kernel<X>, dim3(rows), dim3(256), 0, s,
                     stream, scaled, squares, x, weight, hidden);
}

template void launch_stream_begin<u16>(float*, u16*, float*, const u16*,
                                       const u16*, int, int, hipStream_t);
template void launch_stream_begin<float>(float*, u16*, float*, const float*,
                                         const u16*, int, int, hipStream_t);

}  // namespace fi
