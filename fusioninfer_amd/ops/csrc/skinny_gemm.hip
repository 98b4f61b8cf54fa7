// y = x W^T for a few rows of x (decode steps, the head of a prompt step):
// bf16 operands, fp32 accumulation, W [N, K] row-major as checkpoints have
// it. Bound by reading W once.
//
// A workgroup takes 16 * RF rows of W at a time; its NW waves split K. Each
// wave streams its part through a private ring in LDS: DMA, 128 values of K
// of every row per stage, up to R - 1 stages ahead, no barrier but one per
// finished tile (the sum over the waves). About 64-96 KB are in flight per
// CU, which is what hides the memory latency; registers or a shared
// double buffer do not hold that much. The ring runs on over tile borders.
// Rows are stored as 16 chunks of 16 bytes, chunk c of row r at c ^ r, so
// the fragment reads (16 rows, one chunk each) are free of bank conflicts
// while a DMA still reads whole 256-byte pieces of rows. W is read with the
// non-temporal hint: nothing reads it again before the next step (a plain
// read of 200 MB runs at 6.0 TB/s here, with the hint at 6.5).
//
// MFMA 16x16x32 with A = W, B = x: a lane ends with four neighbouring
// outputs of one row of x.
//
// Measured against the library's GEMM at M = 1 / 16, us (GB/s of W): N 24576,
// K 4096: 44.6 / 45.1 -> 32.0 / 33.4 (6290 / 6020); 4096, 12288: 22.3 / 23.0
// -> 17.8 / 21.3; 6144, 4096: 15.1 / 15.6 -> 9.6 / 12.1; 4096, 4096: 15.0 /
// 15.1 -> 7.7 / 9.3; 151936, 4096: 250 / 260 -> 187 / 203; 512, 2048: 8.0 /
// 8.1 -> 3.7 / 4.5. SILU_MUL: the second half of W's rows are the
// "up" rows of the first half's "gate" rows; a tile is 16 of each and
// leaves silu(gate) * up, without a pass over the [M, N] product.

#include "common.h"

namespace fi {

namespace {

typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) float floatx4;

constexpr int kStageK = 128;          // values of K per stage
constexpr int kFragB = 16 * kStageK * 2;  // 16 rows of a stage

template <int N>
FI_DEV void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// XR: DMAs for the rows of x per stage, four rows each
template <int NW, int RF, int XR, int R, bool SILU_MUL>
__global__ __launch_bounds__(NW * kWaveSize)
void skinny_gemm_kernel(u16* __restrict__ out, const u16* __restrict__ x,
                        const u16* __restrict__ w,
                        const u16* __restrict__ bias, const int M,
                        const int N, const int K, const int64_t x_stride,
                        const int64_t out_stride) {
  static_assert(!SILU_MUL || RF == 2, "gate rows and up rows");
  constexpr int kStageB = RF * kFragB + XR * 1024;
  constexpr int kLoads = RF * 4 + XR;       // DMAs of a stage
  constexpr int kScratch = NW * RF * kWaveSize;  // float4
  static_assert(NW * R * kStageB + 2 * kScratch * 16 <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(1024)))
  unsigned char smem[NW * R * kStageB + 2 * kScratch * 16];

  const int lane = threadIdx.x % kWaveSize;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  const int tiles = (SILU_MUL ? N / 2 : N) / (SILU_MUL ? 16 : 16 * RF);
  const int stages = K / kStageK;
  const int s_lo = wave * stages / NW, s_hi = (wave + 1) * stages / NW;

  unsigned char* ring = smem + wave * (R * kStageB);
  const u32 ring_lds = static_cast<u32>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) unsigned char*)ring));
  floatx4* scratch = reinterpret_cast<floatx4*>(smem + NW * R * kStageB);

  // per-lane source offsets: DMA j copies rows 4j..4j+3, lane l chunk
  // (l & 15) ^ row of row 4j + (l >> 4) to its place l & 15
  u32 w_off[4], x_off[XR];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = 4 * j + (lane >> 4);
    w_off[j] = static_cast<u32>(row * K + ((lane & 15) ^ row) * 8) * 2;
  }
#pragma unroll
  for (int j = 0; j < XR; ++j) {
    const int row = 4 * j + (lane >> 4);
    x_off[j] = static_cast<u32>(min(row, M - 1) * x_stride +
                                ((lane & 15) ^ row) * 8) * 2;
  }
  // fragment reads: row lane & 15 (of x: rows past the staged ones repeat),
  // chunk 4 kk + (lane >> 4)
  const int row = lane & 15, xrow = row & (4 * XR - 1);
  int wr[4], xr[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const int c = kk * 4 + (lane >> 4);
    wr[kk] = row * 256 + ((c ^ row) & 15) * 16;
    xr[kk] = RF * kFragB + xrow * 256 + ((c ^ xrow) & 15) * 16;
  }

  const int mine = tiles > static_cast<int>(blockIdx.x)
      ? (tiles - 1 - static_cast<int>(blockIdx.x)) /
                static_cast<int>(gridDim.x) + 1
      : 0;
  const int total = mine * (s_hi - s_lo);

  // stages requested so far: tile, stage, ring slot
  int it = blockIdx.x, is = s_lo, islot = 0, issued = 0;
  auto request = [&] {
    const u32 dst = ring_lds + islot * kStageB;
#pragma unroll
    for (int f = 0; f < RF; ++f) {
      const int64_t r0 = SILU_MUL ? it * 16 + f * (N / 2)
                                  : (it * RF + f) * 16;
      const u16* src = w + r0 * K + is * kStageK;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        dma_to_lds16_nt(dst + f * kFragB + j * 1024, src, w_off[j]);
    }
#pragma unroll
    for (int j = 0; j < XR; ++j)
      dma_to_lds16(dst + RF * kFragB + j * 1024, x + is * kStageK, x_off[j]);
    ++issued;
    if (++islot == R) islot = 0;
    if (++is == s_hi) {
      is = s_lo;
      it += gridDim.x;
    }
  };
  for (int i = 0; i < R - 1; ++i)
    if (i < total) request();

  int slot = 0, done = 0;
  for (int t = 0; t < mine; ++t) {
    const int tile = blockIdx.x + t * gridDim.x;
    floatx4 acc[RF];
#pragma unroll
    for (int f = 0; f < RF; ++f) acc[f] = {0.f, 0.f, 0.f, 0.f};
    for (int s = s_lo; s < s_hi; ++s, ++done) {
      // all but the stages behind this one have landed
      if (issued - done >= R - 1) {
        wait_vm<(R - 2) * kLoads>();
      } else if (R > 3 && issued - done == 2) {
        wait_vm<kLoads>();
      } else {
        wait_vm<0>();
      }
      // the slot read in the previous step is free again
      if (issued < total) request();
      const unsigned char* st = ring + slot * kStageB;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const short8 b = *reinterpret_cast<const short8*>(st + xr[kk]);
#pragma unroll
        for (int f = 0; f < RF; ++f) {
          const short8 a =
              *reinterpret_cast<const short8*>(st + f * kFragB + wr[kk]);
          acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[f], 0, 0,
                                                           0);
        }
      }
      if (++slot == R) slot = 0;
    }
    // sum over the waves; two scratch areas in turn, so that the next tile's
    // sums never meet this tile's reads
    floatx4* sc = scratch + (t & 1) * kScratch;
#pragma unroll
    for (int f = 0; f < RF; ++f)
      sc[(wave * RF + f) * kWaveSize + lane] = acc[f];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int m = lane & 15, n4 = (lane >> 4) * 4;
    if (wave < (SILU_MUL ? 1 : RF) && m < M) {
      floatx4 sum[2];
#pragma unroll
      for (int f = 0; f < (SILU_MUL ? 2 : 1); ++f) {
        sum[f] = sc[(SILU_MUL ? f : wave) * kWaveSize + lane];
#pragma unroll
        for (int i = 1; i < NW; ++i)
          sum[f] += sc[(i * RF + (SILU_MUL ? f : wave)) * kWaveSize + lane];
      }
      const int n = (SILU_MUL ? tile : tile * RF + wave) * 16 + n4;
      bf16x4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = sum[0][r];
        if (SILU_MUL)
          v = v / (1.f + __expf(-v)) * sum[1][r];
        else if (bias)
          v += bf16_to_f32(bias[n + r]);
        o.h[r] = f32_to_bf16(v);
      }
      *reinterpret_cast<bf16x4*>(out + m * out_stride + n) = o;
    }
  }
}

}  // namespace

// M <= 16, K a multiple of 128, N of 16 (32 with silu_mul).
void launch_skinny_gemm(u16* out, const u16* x, const u16* w,
                        const u16* bias, int M, int N, int K,
                        int64_t x_stride, int64_t out_stride, bool silu_mul,
                        hipStream_t stream) {
#define FI_SK(NW, RF, XR, R, S)                                               \
  hipLaunchKernelGGL((skinny_gemm_kernel<NW, RF, XR, R, S>), dim3(grid),      \
                     dim3(NW * kWaveSize), 0, stream, out, x, w, bias, M, N,  \
                     K, x_stride, out_stride)
  // 32 rows and four waves per tile read x half as often and keep longer
  // runs per wave; with fewer than 192 such tiles the chip is filled better
  // by 16 rows and eight waves. Measured wide / not (M = 1, us): N 24576, K
  // 4096 32.0 / 31.6; 6144, 4096 9.6 / 11.2; 4096, 4096 9.3 / 7.7; 4096,
  // 12288 23.3 / 17.8; at M = 16 33.4 / 37.9, 12.1 / 14.2, 11.3 / 9.3.
  const bool wide = silu_mul || (N % 32 == 0 && N >= 6144);
  const int tiles = silu_mul ? N / 32 : (wide ? N / 32 : N / 16);
  const int grid = std::min(tiles, 256);
  if (wide) {
    if (silu_mul) {
      if (M <= 4) FI_SK(4, 2, 1, 4, true);
      else if (M <= 8) FI_SK(4, 2, 2, 3, true);
      else FI_SK(4, 2, 4, 3, true);
    } else {
      if (M <= 4) FI_SK(4, 2, 1, 4, false);
      else if (M <= 8) FI_SK(4, 2, 2, 3, false);
      else FI_SK(4, 2, 4, 3, false);
    }
  } else {
    if (M <= 4) FI_SK(8, 1, 1, 3, false);
    else if (M <= 8) FI_SK(8, 1, 2, 3, false);
    else FI_SK(8, 1, 4, 2, false);
  }
#undef FI_SK
}

}  // namespace fi
