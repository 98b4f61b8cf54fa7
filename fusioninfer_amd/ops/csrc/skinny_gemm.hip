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
//
// A norm between two layers is not a launch of its own (2 to 2.7 us in a
// graph, as long as a tenth of a layer's products): ADD, the layer in front,
// adds its product to the residual stream, fp32, and leaves the sums times the
// norm's weight and the squares of each 16 columns; SCALED, the one behind,
// reads these as x and divides its products by the root mean square, which a
// wave of its own sums up while the others read W. us at M = 1 / 16, a norm
// and the product, then SCALED: N 6144, K 4096 12.7 / 14.7 -> 9.9 / 12.3;
// 24576, 4096 with SILU_MUL 34.8 / 35.7 -> 32.7 / 33.4; PLAIN and ADD: 4096,
// 4096 7.7 / 9.2 -> 8.0 / 9.4; 4096, 12288 18.1 / 21.4 -> 18.4 / 21.9. (With
// the norm inside, on fp32 rows that a workgroup stages and multiplies by the
// weight itself: 6144, 4096 at 6 rows 13.0, and no room for more than 8.)
// A step of eight layers: 885 -> 850 us at one row, 1062 -> 1024 at 13.

#include <type_traits>

#include "common.h"

namespace fi {

namespace {

typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) float floatx4;

constexpr int kStageK = 128;          // values of K per stage

template <int N>
FI_DEV void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// what becomes of the product
enum { PLAIN, SCALED, ADD, GELU };

FI_DEV void sync_waves() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// sum over the lanes l, l ^ 16, l ^ 32, l ^ 48
FI_DEV float sum_of_quarters(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  const auto h = __builtin_amdgcn_permlane32_swap(
      __float_as_int(v), __float_as_int(v), false, false);
  v = __int_as_float(h[0]) + __int_as_float(h[1]);
  const auto r = __builtin_amdgcn_permlane16_swap(
      __float_as_int(v), __float_as_int(v), false, false);
  v = __int_as_float(r[0]) + __int_as_float(r[1]);
#endif
  return v;
}

// By one wave, from squares [parts][16]: lane l < 4 ends with the sums of rows
// 4 l to 4 l + 3.
FI_DEV floatx4 sum_of_parts(const float* squares, int parts, int lane) {
  floatx4 sum = {0.f, 0.f, 0.f, 0.f};
  const floatx4* from = reinterpret_cast<const floatx4*>(squares) + lane;
  constexpr int kAtOnce = 8;    // loads on their way, 16 parts each
  for (int p0 = 0; p0 < parts; p0 += kAtOnce * 16) {
    floatx4 v[kAtOnce];
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i) {
      const int p = p0 + i * 16 + (lane >> 2);
      const floatx4 got = from[(min(p, parts - 1) - (lane >> 2)) * 4];
      v[i] = p < parts ? got : floatx4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i) sum += v[i];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float v = sum[i];
    v += dpp_move<0x128>(v);   // row_ror:8
    v += dpp_move<0x124>(v);   // row_ror:4
    sum[i] = sum_of_quarters(v);
  }
  return sum;
}

// XR: DMAs for the rows of x per stage, four rows each. WR: rows of W of a
// fragment; eight leave half of a product unused.
template <int NW, int RF, int XR, int R, bool SILU_MUL, int MODE, int WR = 16>
__global__ __launch_bounds__((NW + (MODE == SCALED)) * kWaveSize)
void skinny_gemm_kernel(void* __restrict__ out_p, const u16* __restrict__ x,
                        const u16* __restrict__ w,
                        const u16* __restrict__ bias,
                        float* __restrict__ squares, const int parts,
                        const float eps, const u16* __restrict__ norm,
                        u16* __restrict__ scaled,
                        const int M, const int N, const int K,
                        const int64_t x_stride, const int64_t out_stride) {
  static_assert(!SILU_MUL || RF == 2, "gate rows and up rows");
  static_assert(MODE != ADD || !SILU_MUL);
  using Out = std::conditional_t<MODE == ADD, float, u16>;
  Out* out = static_cast<Out*>(out_p);
  static_assert(WR == 16 || (WR == 8 && RF == 1 && MODE == PLAIN));
  constexpr int kFragB = WR * kStageK * 2;       // rows of W of a stage
  constexpr int kStageB = RF * kFragB + XR * 1024;
  constexpr int kLoads = RF * (WR / 4) + XR;     // DMAs of a stage
  constexpr int kScratch = NW * RF * kWaveSize;  // float4
  constexpr int kRingB = NW * R * kStageB;
  constexpr int kSquaresB = MODE == SCALED ? 64 : 0;
  // two scratch areas in turn, so that the next tile's sums never meet this
  // tile's reads; or one, and a barrier more for each tile but the first
  constexpr int kAreas =
      kRingB + 2 * kScratch * 16 + kSquaresB <= 160 * 1024 ? 2 : 1;
  constexpr int kScratchB = kAreas * kScratch * 16;
  static_assert(kRingB + kScratchB + kSquaresB <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(1024)))
  unsigned char smem[kRingB + kScratchB + kSquaresB];

  const int lane = threadIdx.x % kWaveSize;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  const int tiles = (SILU_MUL ? N / 2 : N) / (SILU_MUL ? 16 : WR * RF);
  const int stages = K / kStageK;
  const int s_lo = wave * stages / NW, s_hi = (wave + 1) * stages / NW;

  unsigned char* ring = smem + wave * (R * kStageB);
  const u32 ring_lds = static_cast<u32>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) unsigned char*)ring));
  floatx4* scratch = reinterpret_cast<floatx4*>(smem + kRingB);
  float* sq = reinterpret_cast<float*>(smem + kRingB + kScratchB);

  // per-lane source offsets: DMA j copies rows 4j..4j+3, lane l chunk
  // (l & 15) ^ row of row 4j + (l >> 4) to its place l & 15
  u32 w_off[WR / 4], x_off[XR];
#pragma unroll
  for (int j = 0; j < WR / 4; ++j) {
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
    wr[kk] = (row & (WR - 1)) * 256 + ((c ^ (row & (WR - 1))) & 15) * 16;
    xr[kk] = RF * kFragB + xrow * 256 + ((c ^ xrow) & 15) * 16;
  }

  const int mine = tiles > static_cast<int>(blockIdx.x)
      ? (tiles - 1 - static_cast<int>(blockIdx.x)) /
                static_cast<int>(gridDim.x) + 1
      : 0;
  const int total = mine * (s_hi - s_lo);

  // The rows' squares are one more wave's: the others' waits count their DMAs.
  if (MODE == SCALED && wave == NW) {
    const floatx4 sum = sum_of_parts(squares, parts, lane);
    if (lane < 4)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        sq[lane * 4 + i] = rsqrtf(sum[i] / K + eps);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    for (int t = 0; t < mine; ++t) {
      if (kAreas == 1 && t > 0) sync_waves();
      sync_waves();
    }
    return;
  }

  // stages requested so far: tile, stage, ring slot
  int it = blockIdx.x, is = s_lo, islot = 0, issued = 0;
  auto request = [&] {
    const u32 dst = ring_lds + islot * kStageB;
#pragma unroll
    for (int f = 0; f < RF; ++f) {
      const int64_t r0 = SILU_MUL ? it * 16 + f * (N / 2)
                                  : (it * RF + f) * WR;
      const u16* src = w + r0 * K + is * kStageK;
#pragma unroll
      for (int j = 0; j < WR / 4; ++j)
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
    const int m = lane & 15, n4 = (lane >> 4) * 4;
    const bool mine_to_store =
        wave < (SILU_MUL ? 1 : RF) && m < M && (WR == 16 || n4 < WR);
    const int n = (SILU_MUL ? tile : tile * RF + wave) * WR + n4;
    // (requested here: at its use nothing else would be on its way)
    floatx4 old;
    bf16x4 g;
    if (MODE == ADD && mine_to_store) {
      old = *reinterpret_cast<const floatx4*>(out + m * out_stride + n);
      if (norm != nullptr)
        __builtin_memcpy(&g, norm + n, sizeof(g));   // on any grid
    }
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
    // sum over the waves
    if (kAreas == 1 && t > 0) sync_waves();   // the area has been read
    floatx4* sc = scratch + (kAreas == 2 ? (t & 1) * kScratch : 0);
#pragma unroll
    for (int f = 0; f < RF; ++f)
      sc[(wave * RF + f) * kWaveSize + lane] = acc[f];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    sync_waves();
    float part = 0.f;
    if (mine_to_store) {
      floatx4 sum[2];
#pragma unroll
      for (int f = 0; f < (SILU_MUL ? 2 : 1); ++f) {
        sum[f] = sc[(SILU_MUL ? f : wave) * kWaveSize + lane];
#pragma unroll
        for (int i = 1; i < NW; ++i)
          sum[f] += sc[(i * RF + (SILU_MUL ? f : wave)) * kWaveSize + lane];
        if (MODE == SCALED) sum[f] *= sq[m];
      }
      if constexpr (MODE == ADD) {
        const floatx4 v = old + sum[0];
        *reinterpret_cast<floatx4*>(out + m * out_stride + n) = v;
        if (norm != nullptr) {
          bf16x4 o;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            o.h[r] = f32_to_bf16(v[r] * bf16_to_f32(g.h[r]));
            part = fmaf(v[r], v[r], part);
          }
          *reinterpret_cast<bf16x4*>(scaled + static_cast<int64_t>(m) * N +
                                     n) = o;
        }
      } else {
        bf16x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = sum[0][r];
          if (SILU_MUL)
            v = v / (1.f + __expf(-v)) * sum[1][r];
          else if (MODE == GELU)
            v = gelu(v);
          else if (bias)
            v += bf16_to_f32(bias[n + r]);
          o.h[r] = f32_to_bf16(v);
        }
        *reinterpret_cast<bf16x4*>(out + m * out_stride + n) = o;
      }
    }
    if (MODE == ADD && norm != nullptr && wave < RF) {
      part = sum_of_quarters(part);
      if (lane < M) squares[(tile * RF + wave) * 16 + lane] = part;
    }
  }
}

}  // namespace

// M <= 16, K a multiple of 128, N of 16 (32 with silu_mul)
void launch_skinny_gemm(u16* out, const u16* x, const u16* w, const u16* bias,
                        const SkinnyExtra& extra, int M, int N, int K,
                        int64_t x_stride, int64_t out_stride, bool silu_mul,
                        hipStream_t stream) {
#define FI_SK(NW, RF, XR, R, S, MODE, ...)                                    \
  hipLaunchKernelGGL((skinny_gemm_kernel<NW, RF, XR, R, S, MODE, ##__VA_ARGS__>), \
                     dim3(grid), dim3((NW + (MODE == SCALED)) * kWaveSize),   \
                     0, stream,                                               \
                     MODE == ADD ? static_cast<void*>(extra.add) : out, x, w, \
                     bias,                                                    \
                     MODE == ADD ? extra.squares_out                          \
                                 : const_cast<float*>(extra.squares_in),      \
                     extra.parts, extra.eps, extra.norm, extra.scaled, M, N,  \
                     K, x_stride, out_stride)
  // 32 rows and four waves per tile read x half as often and keep longer
  // runs per wave; with fewer than 192 such tiles the chip is filled better
  // by 16 rows and eight waves. Measured wide / not (M = 1, us): N 24576, K
  // 4096 32.0 / 31.6; 6144, 4096 9.6 / 11.2; 4096, 4096 9.3 / 7.7; 4096,
  // 12288 23.3 / 17.8; at M = 16 33.4 / 37.9, 12.1 / 14.2, 11.3 / 9.3.
  const bool wide = silu_mul || (N % 32 == 0 && N >= 6144);
  // where tiles of 16 rows fill half of the chip at most, twice as many of eight
  // have two thirds of the bytes each on their way for half as long. us at M = 1
  // / 4 / 16: 2048, 6144 8.2 / 9.0 / 10.9 and 6.7 / 6.9 / 9.5; 2048, 2048 4.0 /
  // 4.2 / 4.7 and 3.7 / 3.8 / 4.2; 256, 4096 4.5 / 4.8 / 6.2 and 3.7 / 3.9 / 5.2
  const bool plain = extra.squares_in == nullptr && extra.add == nullptr &&
                     !extra.gelu && !silu_mul;
  const bool few = plain && N <= 2048;
  const int tiles = silu_mul || wide ? N / 32 : few ? N / 8 : N / 16;
  const int grid = std::min(tiles, 256);
#define FI_SK_WIDE(S, MODE)                                                   \
  do {                                                                        \
    if (M <= 4) FI_SK(4, 2, 1, 4, S, MODE);                                   \
    else if (M <= 8) FI_SK(4, 2, 2, 3, S, MODE);                              \
    else FI_SK(4, 2, 4, 3, S, MODE);                                          \
  } while (0)
#define FI_SK_NARROW(MODE)                                                    \
  do {                                                                        \
    if (M <= 4) FI_SK(8, 1, 1, 3, false, MODE);                               \
    else if (M <= 8) FI_SK(8, 1, 2, 3, false, MODE);                          \
    else FI_SK(8, 1, 4, 2, false, MODE);                                      \
  } while (0)
  if (extra.squares_in != nullptr) {
    if (silu_mul) FI_SK_WIDE(true, SCALED);
    else if (wide) FI_SK_WIDE(false, SCALED);
    else FI_SK_NARROW(SCALED);
  } else if (extra.add != nullptr) {
    if (wide) FI_SK_WIDE(false, ADD);
    else FI_SK_NARROW(ADD);
  } else if (extra.gelu) {
    if (wide) FI_SK_WIDE(false, GELU);
    else FI_SK_NARROW(GELU);
  } else {
    if (silu_mul) FI_SK_WIDE(true, PLAIN);
    else if (wide) FI_SK_WIDE(false, PLAIN);
    else if (!few) FI_SK_NARROW(PLAIN);
    else if (M <= 4) FI_SK(8, 1, 1, 4, false, PLAIN, 8);
    else if (M <= 8) FI_SK(8, 1, 2, 4, false, PLAIN, 8);
    else FI_SK(8, 1, 4, 3, false, PLAIN, 8);
  }
#undef FI_SK_NARROW
#undef FI_SK_WIDE
#undef FI_SK
}

}  // namespace fi
