// FP8 (OCP e4m3) fused activation-quantization kernels for CDNA4.
//
// The fp8 serving mode needs per-token-quantized activations for
// torch._scaled_mm; a standalone eager quant pass measured MORE expensive
// than the fp8 GEMM savings, so quantization is fused into the producers:
//  * silu_and_mul_fp8: SwiGLU epilogue emitting fp8 + per-row scale
//    (feeds down_proj).
//  * quant_fp8_rows: bf16 -> fp8 row quant (feeds o_proj from the
//    attention output).
// The RMSNorm fp8 variants live in norm.hip (feed qkv/gate_up).
// Native v_cvt_pk_fp8_f32 packs 2 f32 -> 2 fp8 bytes per instruction.

#include "common.h"

namespace fi {

constexpr float kFp8Max = 448.0f;

template <bool ONCE>
FI_DEV bf16x8 load8(const u16* p) {
  const u32x4* from = reinterpret_cast<const u32x4*>(p);
  return __builtin_bit_cast(
      bf16x8, ONCE ? __builtin_nontemporal_load(from) : *from);
}

// One workgroup per row, which it holds in registers between the absmax pass and
// the convert pass, eight columns a thread at a time. THREADS 256, or 0: of the
// launch, up to 1024. Few rows take the time of one chain from load to store,
// which is the shorter the more threads share it; many are bound by memory, and
// more of them are in flight the smaller they are. ONCE: what is read and
// written goes past the caches, for more than the memory-side one holds. us,
// 12288 columns of silu(gate) * up, 256 threads of six vectors each, and up to
// 1024: 1 row 4.3 and 3.2, 64 rows 4.8 and 3.6, 1000 11.6 and 11.6, 8000 95 and 87,
// with ONCE 74 (6.6 TB/s; at 2000 rows, 98 MB, 20 either way). 5120 columns as
// they are: 16 rows 2.5 and 2.4, 1000 3.5 and 4.5, 8000 19 and 22.4.
template <int THREADS, int ITERS, bool SILU_MUL, bool ONCE>
__global__ __launch_bounds__(THREADS ? THREADS : 1024)
void row_quant_fp8_kernel(
    unsigned char* __restrict__ out,   // [T, cols] fp8
    float* __restrict__ out_scales,    // [T]
    const u16* __restrict__ in,        // [T, cols] bf16 (SILU_MUL: [T, 2*cols])
    const int cols) {
  const int row = blockIdx.x;
  const int tid = threadIdx.x;
  const int threads = THREADS ? THREADS : static_cast<int>(blockDim.x);
  const int64_t in_row = static_cast<int64_t>(row) * (SILU_MUL ? 2 * cols : cols);

  float vals[ITERS][8];
  float amax = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int col = (it * threads + tid) * 8;
    if (col < cols) {
      if (SILU_MUL) {
        const bf16x8 g = load8<ONCE>(in + in_row + col);
        const bf16x8 u = load8<ONCE>(in + in_row + cols + col);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float gf = bf16_to_f32(g.h[j]);
          vals[it][j] = silu(gf) * bf16_to_f32(u.h[j]);
        }
      } else {
        const bf16x8 v = load8<ONCE>(in + in_row + col);
#pragma unroll
        for (int j = 0; j < 8; ++j) vals[it][j] = bf16_to_f32(v.h[j]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(vals[it][j]));
    }
  }

  __shared__ float scratch[16];
  amax = wave_reduce_max(amax);
  if (THREADS) {
    amax = block_reduce_max<THREADS / kWaveSize>(amax, scratch);
  } else {
    if (tid % kWaveSize == 0) scratch[tid / kWaveSize] = amax;
    __syncthreads();
    for (int i = 0; i < threads / kWaveSize; ++i)
      amax = fmaxf(amax, scratch[i]);
  }
  const float scale = fmaxf(amax, 1e-8f) / kFp8Max;
  const float inv_scale = 1.f / scale;
  if (tid == 0) out_scales[row] = scale;

#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int col = (it * threads + tid) * 8;
    if (col < cols) {
      float sv[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) sv[j] = vals[it][j] * inv_scale;
      u32 packed[2];
      pack_fp8x8(sv, packed);
      auto* to = reinterpret_cast<uint64_t*>(
          out + static_cast<int64_t>(row) * cols + col);
      const uint64_t both = static_cast<uint64_t>(packed[1]) << 32 | packed[0];
      if (ONCE) __builtin_nontemporal_store(both, to);
      else *to = both;
    }
  }
}

template <bool SILU_MUL>
void launch_row_quant_fp8(unsigned char* out, float* scales, const u16* in,
                          int rows, int cols, hipStream_t stream) {
  if (cols > 16384) abort();     // more than two vectors of 1024 threads
  const bool wide = cols > (SILU_MUL ? 6144 : 10240) ||
                    (cols > 4096 && rows <= (SILU_MUL ? 512 : 256));
  const int iters = ceil_div(cols, wide ? 8192 : 2048);
  const int threads =
      wide ? ceil_div(ceil_div(ceil_div(cols, 8), iters), kWaveSize) * kWaveSize
           : 256;
  const bool once = beyond_caches(static_cast<int64_t>(rows) * cols *
                                  (SILU_MUL ? 4 : 2));
#define FI_QUANT(THREADS, N)                                                  \
  do {                                                                        \
    auto kernel = once ? &row_quant_fp8_kernel<THREADS, N, SILU_MUL, true>    \
                       : &row_quant_fp8_kernel<THREADS, N, SILU_MUL, false>;  \
    hipLaunchKernelGGL(kernel, dim3(rows), dim3(threads), 0, stream, out,     \
                       scales, in, cols);                                     \
  } while (0)
  if (wide) {
    if (iters == 1) FI_QUANT(0, 1);
    else FI_QUANT(0, 2);
  } else if (iters <= 1) {
    FI_QUANT(256, 1);
  } else if (iters == 2) {
    FI_QUANT(256, 2);
  } else if (iters == 3) {
    FI_QUANT(256, 3);
  } else if constexpr (!SILU_MUL) {
    if (iters == 4) FI_QUANT(256, 4);
    else FI_QUANT(256, 5);
  }
#undef FI_QUANT
}

template void launch_row_quant_fp8<true>(unsigned char*, float*, const u16*,
                                         int, int, hipStream_t);
template void launch_row_quant_fp8<false>(unsigned char*, float*, const u16*,
                                          int, int, hipStream_t);

}  // namespace fi
