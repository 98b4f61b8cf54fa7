// y = x W^T for 17 to 256 rows of x (a decode batch, a short prompt): bf16
// operands, fp32 accumulation, W [N, K] row-major. Bound by reading W once up
// to about 200 rows; there the matrix cores catch up.
//
// The product is cut into tiles of TN rows of W by all of x, the tiles into
// stages of KS values of K, and the row of all stages of all tiles into one
// equal part per workgroup (256 of them), so that every CU streams the same
// amount of W whatever N and K are. A part that holds a whole tile writes its
// result; pieces of a tile go to scratch in fp32 and a second kernel sums
// them. Within a workgroup all waves share the stages: DMA into a ring in
// LDS, R - 1 stages ahead, one barrier per stage, running on over the borders
// of tiles. x comes from L2, MB / TN times the traffic of W.
//
// Rows lie in LDS as chunks of 16 bytes, chunk c of row r at c ^ r, so the
// fragment reads are free of bank conflicts while a DMA reads whole pieces of
// rows. MFMA 16x16x32 with A = W, B = x: a lane ends with four neighbouring
// outputs of one row of x. SILU_MUL: the first half of a tile's rows are gate
// rows and the second the up rows that go with them; a wave holds both.
//
// What L2 delivers to the CUs, W and x together, ends at about 10 TB/s (x
// requests of 16 KB per CU in flight or 64 made no difference, nor did other
// row strides of x); hence tiles at least as tall as x has rows, taller where
// N allows. The second kernel of a cut product costs 4.7 us at the least.
// Measured, us (GB/s of W) at 32 / 64 / 128 / 256 rows: N 24576, K 4096 with
// silu 31.4 (6410) / 34.5 / 44.6 / 64, the library's GEMM and the pass
// behind it 48 / 51 / 55 / 67; 4096, 12288 21 (4700) / 26 / 33 / 45 against
// 26 / 37 / 66 / 53; 151936, 4096 211 (5880) / 238 / 266 / 391 against 264 /
// 262 / 279 / 350.
//
// FP8: the same kernel on e4m3 rows, 1 to 128 of them. 24576 x 4096 at 1 / 32
// / 64 rows 20.0 (5040) / 19.3 / 24.3 us, the library's GEMM 30.8 / 24.4 /
// 25.9; 4096 x 12288 14.2 (3550) / 14.5 / 19.4 against 21.1 / 20.5 / 24.1.

#include "common.h"

namespace fi {

namespace {

typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) float floatx4;

template <int N>
FI_DEV void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// parts of `total` units of `unit` stages over `n` workgroups
struct Cut {
  int per, rem, unit;
  FI_DEV Cut(int total, int n, int unit)
      : per(total / n), rem(total % n), unit(unit) {}
  FI_DEV int start(int i) const { return (i * per + min(i, rem)) * unit; }
  // the part that holds a stage (unit 1)
  FI_DEV int holder(int stage) const {
    const int wide = rem * (per + 1);
    return stage < wide ? stage / (per + 1) : rem + (stage - wide) / per;
  }
};

// at most `stages` stages of L DMAs each of this wave are still on the way
template <int L, int MAX>
FI_DEV void wait_stages(int stages) {
  if (MAX >= 5 && stages >= 5) return wait_vm<5 * L>();
  if (MAX >= 4 && stages == 4) return wait_vm<4 * L>();
  if (MAX >= 3 && stages == 3) return wait_vm<3 * L>();
  if (MAX >= 2 && stages == 2) return wait_vm<2 * L>();
  if (MAX >= 1 && stages == 1) return wait_vm<L>();
  wait_vm<0>();
}

// WN x WM waves; a wave holds RF fragments of 16 rows of W by CF of x; the
// ring has RW stages of W, which LWAVES of the waves load, and RX of x
template <int WN_, int RF_, int WM_, int CF_, int KS_, int RW_, int RX_,
          int LWAVES>
struct PartShape {
  static constexpr int WN = WN_, RF = RF_, WM = WM_, CF = CF_, KS = KS_,
                       RW = RW_, RX = RX_;
  static constexpr int kWaves = WN * WM;
  static constexpr int kWLoaders = LWAVES, kXLoaders = kWaves - LWAVES;
  static constexpr int TN = WN * RF * 16, MB = WM * CF * 16;
  static constexpr int kRowB = KS * 2, kChunks = kRowB / 16;
  static constexpr int kWB = TN * kRowB, kXB = MB * kRowB;  // of a stage
  static constexpr int kRowsPerDma = 1024 / kRowB;
  static constexpr int LW = TN / kRowsPerDma / kWLoaders;
  static constexpr int LX = MB / kRowsPerDma / kXLoaders;
  static constexpr int kPiece = TN * MB / 4;  // float4
  static_assert(RF % 2 == 0 && TN / 2 % kRowsPerDma == 0);
  static_assert(LW * kRowsPerDma * kWLoaders == TN &&
                LX * kRowsPerDma * kXLoaders == MB);
  static_assert(RW * kWB + RX * kXB <= 160 * 1024 && RW >= 2 && RW <= 7 &&
                RX >= 2 && RX <= 7);
};

// fragment of W rows (of the tile) that wave column wn holds as its rf-th
template <class S, bool SILU_MUL>
FI_DEV int w_fragment(int wn, int rf) {
  if (!SILU_MUL) return wn * S::RF + rf;
  constexpr int h = S::RF / 2;
  return rf < h ? wn * h + rf : S::TN / 32 + wn * h + rf - h;
}

// FP8: the scales of the rows of x and of W
struct Scales {
  const float* x;
  const float* w;
};

// results n4 .. n4+3 of row m; SILU_MUL: of gate values g and up values u
template <bool SILU_MUL, bool FP8>
FI_DEV void store4(u16* out, const u16* bias, const Scales& scales,
                   const floatx4& g, const floatx4& u, int m, int n,
                   int64_t out_stride) {
  bf16x4 o;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float v = g[r];
    if (FP8) v *= scales.x[m] * scales.w[n + r];
    if (SILU_MUL)
      v = v / (1.f + __expf(-v)) * u[r];
    else if (bias)
      v += bf16_to_f32(bias[n + r]);
    o.h[r] = f32_to_bf16(v);
  }
  *reinterpret_cast<bf16x4*>(out + m * out_stride + n) = o;
}

// FP8: e4m3 values, two to a u16 everywhere (K and strides too); a chunk of 16
// goes through two products, in the same order for W and x
template <class S, bool SILU_MUL, bool FP8>
__global__ __launch_bounds__(S::kWaves * kWaveSize)
void part_gemm_kernel(u16* __restrict__ out, floatx4* __restrict__ pieces,
                      const u16* __restrict__ x, const u16* __restrict__ w,
                      const u16* __restrict__ bias, const Scales scales,
                      const int M, const int N, const int K,
                      const int64_t x_stride,
                      const int64_t out_stride, const int tiles,
                      const int unit) {
  constexpr int LW = S::LW, LX = S::LX, RF = S::RF, CF = S::CF;
  __shared__ __attribute__((aligned(1024)))
  unsigned char smem[S::RW * S::kWB + S::RX * S::kXB];

  const int lane = threadIdx.x % kWaveSize;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  const int wn = wave / S::WM, wm = wave % S::WM;
  const int SK = K / S::KS;
  const Cut cut(tiles * SK / unit, gridDim.x, unit);
  const int lo = cut.start(blockIdx.x), hi = cut.start(blockIdx.x + 1);

  // Some waves load W, the others x: a wave's DMAs land in order, and x,
  // which comes from L2, shall not wait for the W requested before it.
  const bool loads_w = wave < S::kWLoaders;
  const int lwave = loads_w ? wave : wave - S::kWLoaders;
  const int loaders = loads_w ? S::kWLoaders : S::kXLoaders;
  const u32 ring_lds =
      static_cast<u32>(reinterpret_cast<uintptr_t>(
          (__attribute__((address_space(3))) unsigned char*)smem)) +
      (loads_w ? 0 : S::RW * S::kWB) + lwave * 1024;
  // DMA j copies rows (loaders j + lwave) * kRowsPerDma on; lane l brings chunk
  // (l % kChunks) ^ row of one of them to its place
  constexpr int kMax = LW > LX ? LW : LX;
  const u16* base[kMax];
  u32 off[kMax];
  auto chunk = [&](int j) {
    const int r = (j * loaders + lwave) * S::kRowsPerDma + lane / S::kChunks;
    return static_cast<u32>(((lane % S::kChunks) ^ r) & (S::kChunks - 1)) *
           16;
  };
  auto aim = [&](int tile) {      // at the W rows of a tile
#pragma unroll
    for (int j = 0; j < LW; ++j) {
      const int r0 = (j * S::kWLoaders + lwave) * S::kRowsPerDma;
      int first, last;            // of the matrix, for this DMA
      if (SILU_MUL) {
        const bool up = r0 >= S::TN / 2;
        first = tile * (S::TN / 2) + (up ? N / 2 + r0 - S::TN / 2 : r0);
        last = up ? N - 1 : N / 2 - 1;
      } else {
        first = tile * S::TN + r0;
        last = N - 1;
      }
      first = min(first, last);   // rows past the end repeat the last
      base[j] = w + static_cast<int64_t>(first) * K;
      off[j] = static_cast<u32>(min(lane / S::kChunks, last - first)) * K * 2 +
               chunk(j);
    }
  };
  // Every part walks through its stages of a tile from another one on, and
  // around: parts in step would all read the same few channels, rows being a
  // multiple of their interleave apart.
  int rt = lo / SK, rslot = 0, issued = lo;
  int ra, rb, rs;                 // stages of the tile that are this part's
  auto enter = [&] {
    ra = max(lo - rt * SK, 0);
    rb = max(min(hi - rt * SK, SK), ra + 1);
    rs = ra + static_cast<int>(blockIdx.x / 8) % (rb - ra);
  };
  enter();
  int left = rb - ra;
  if (loads_w) {
    aim(rt);
  } else {
#pragma unroll
    for (int j = 0; j < LX; ++j) {
      const int r = (j * S::kXLoaders + lwave) * S::kRowsPerDma +
                    lane / S::kChunks;
      base[j] = x;
      off[j] = static_cast<u32>(min(r, M - 1) * x_stride * 2) + chunk(j);
    }
  }
  auto request = [&] {
    if (issued >= hi) return;
    if (loads_w) {
      const u32 dst = ring_lds + rslot * S::kWB;
#pragma unroll
      for (int j = 0; j < LW; ++j)
        dma_to_lds16_nt(dst + j * S::kWLoaders * 1024, base[j] + rs * S::KS,
                        off[j]);
      if (++rslot == S::RW) rslot = 0;
    } else {
      const u32 dst = ring_lds + rslot * S::kXB;
#pragma unroll
      for (int j = 0; j < LX; ++j)
        dma_to_lds16(dst + j * S::kXLoaders * 1024, x + rs * S::KS, off[j]);
      if (++rslot == S::RX) rslot = 0;
    }
    ++issued;
    if (++rs == rb) rs = ra;
    if (--left == 0) {
      ++rt;
      enter();
      left = rb - ra;
      if (loads_w) aim(rt);
    }
  };
  for (int i = 0; i < (loads_w ? S::RW : S::RX) - 1; ++i) request();

  // fragment reads: row lane & 15 of a fragment, chunk 4 kk + (lane >> 4);
  // fragments are 16 rows apart, which the swizzle does not see
  const int frow = lane & 15;
  int fr[S::KS / 32];
#pragma unroll
  for (int kk = 0; kk < S::KS / 32; ++kk)
    fr[kk] = frow * S::kRowB +
             (((kk * 4 + (lane >> 4)) ^ frow) & (S::kChunks - 1)) * 16;

  int wslot = 0, xslot = 0, pos = lo;
  while (pos < hi) {
    const int tile = pos / SK;
    const int begin = tile * SK, end = begin + SK;
    const bool from_start = pos == begin;
    const int stop = min(hi, end);
    floatx4 acc[RF][CF];
#pragma unroll
    for (int f = 0; f < RF; ++f)
#pragma unroll
      for (int c = 0; c < CF; ++c) acc[f][c] = {0.f, 0.f, 0.f, 0.f};
    for (; pos < stop; ++pos) {
      // this wave's share of the stage has landed; after the barrier all
      // shares have, and every wave is done with the slot read last
      if (loads_w)
        wait_stages<LW, S::RW - 2>(issued - pos - 1);
      else
        wait_stages<LX, S::RX - 2>(issued - pos - 1);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      request();
      const unsigned char* st = smem + wslot * S::kWB;
      const unsigned char* sx = smem + S::RW * S::kWB + xslot * S::kXB +
                                wm * CF * 16 * S::kRowB;
#pragma unroll
      for (int kk = 0; kk < S::KS / 32; ++kk) {
        short8 a[RF], b[CF];
#pragma unroll
        for (int f = 0; f < RF; ++f)
          a[f] = *reinterpret_cast<const short8*>(
              st + w_fragment<S, SILU_MUL>(wn, f) * 16 * S::kRowB + fr[kk]);
#pragma unroll
        for (int c = 0; c < CF; ++c)
          b[c] = *reinterpret_cast<const short8*>(sx + c * 16 * S::kRowB +
                                                  fr[kk]);
#pragma unroll
        for (int f = 0; f < RF; ++f)
#pragma unroll
          for (int c = 0; c < CF; ++c) {
            if constexpr (FP8) {
              typedef __attribute__((ext_vector_type(2))) long long i64x2;
              const i64x2 a8 = __builtin_bit_cast(i64x2, a[f]);
              const i64x2 b8 = __builtin_bit_cast(i64x2, b[c]);
#pragma unroll
              for (int i = 0; i < 2; ++i)
                acc[f][c] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
                    a8[i], b8[i], acc[f][c], 0, 0, 0);
            } else {
              acc[f][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  a[f], b[c], acc[f][c], 0, 0, 0);
            }
          }
      }
      if (++wslot == S::RW) wslot = 0;
      if (++xslot == S::RX) xslot = 0;
    }
    if (from_start && stop == end) {
#pragma unroll
      for (int f = 0; f < (SILU_MUL ? RF / 2 : RF); ++f) {
        const int n = tile * (SILU_MUL ? S::TN / 2 : S::TN) +
                      w_fragment<S, SILU_MUL>(wn, f) * 16 + (lane >> 4) * 4;
#pragma unroll
        for (int c = 0; c < CF; ++c) {
          const int m = (wm * CF + c) * 16 + (lane & 15);
          if (m < M && n < (SILU_MUL ? N / 2 : N))
            store4<SILU_MUL, FP8>(out, bias, scales, acc[f][c],
                                  acc[SILU_MUL ? f + RF / 2 : f][c], m, n,
                                  out_stride);
        }
      }
    } else {
      // a part holds at most two pieces: the end of a tile that an earlier
      // part began (0) and the start of one that goes on (1)
      floatx4* p = pieces + (static_cast<int64_t>(blockIdx.x) * 2 +
                             (from_start ? 1 : 0)) * S::kPiece +
                   wave * RF * CF * kWaveSize + lane;
#pragma unroll
      for (int f = 0; f < RF; ++f)
#pragma unroll
        for (int c = 0; c < CF; ++c)
          p[(f * CF + c) * kWaveSize] = acc[f][c];
    }
  }
}

// One row of workgroups per border between parts; the first border inside a
// tile sums its pieces.
template <class S, bool SILU_MUL, bool FP8>
__global__ __launch_bounds__(256)
void part_gemm_join_kernel(u16* __restrict__ out,
                           const floatx4* __restrict__ pieces,
                           const u16* __restrict__ bias, const Scales scales,
                           const int M, const int N, const int K,
                           const int64_t out_stride, const int tiles,
                           const int parts) {
  constexpr int RF = S::RF, CF = S::CF;
  constexpr int kUse = SILU_MUL ? RF / 2 : RF;   // fragments with results
  const int SK = K / S::KS;
  const Cut cut(tiles * SK, parts, 1);
  const int part = blockIdx.x + 1;
  const int border = cut.start(part);
  const int tile = border / SK;
  const int begin = tile * SK, end = begin + SK;
  if (border == begin || cut.start(part - 1) > begin) return;
  const int i = blockIdx.y * 256 + threadIdx.x;  // of a wave's kept results
  const int lane = i % kWaveSize;
  const int c = i / kWaveSize % CF, f = i / kWaveSize / CF % kUse;
  const int wave = i / kWaveSize / CF / kUse;
  if (wave >= S::kWaves) return;                 // the last block's rest
  const int wn = wave / S::WM, wm = wave % S::WM;
  const int m = (wm * CF + c) * 16 + (lane & 15);
  const int n = tile * (SILU_MUL ? S::TN / 2 : S::TN) +
                w_fragment<S, SILU_MUL>(wn, f) * 16 + (lane >> 4) * 4;
  if (m >= M || n >= (SILU_MUL ? N / 2 : N)) return;
  const int at = ((wave * RF + f) * CF + c) * kWaveSize + lane;
  constexpr int kUp = S::RF / 2 * CF * kWaveSize;
  const floatx4* p =
      pieces + (static_cast<int64_t>(part - 1) * 2 + 1) * S::kPiece + at;
  floatx4 g = p[0], u = {0.f, 0.f, 0.f, 0.f};
  if (SILU_MUL) u = p[kUp];
  const int last = cut.holder(end - 1);
  for (int q = part; q <= last; q += 4) {
    floatx4 gs[4], us[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p = pieces + static_cast<int64_t>(min(q + i, last)) * 2 * S::kPiece +
          at;
      gs[i] = p[0];
      if (SILU_MUL) us[i] = p[kUp];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (q + i <= last) {
        g += gs[i];
        if (SILU_MUL) u += us[i];
      }
  }
  store4<SILU_MUL, FP8>(out, bias, scales, g, u, m, n, out_stride);
}

// How a shape cuts [N, K] up and what that takes by what limits it here: a
// CU's share of HBM (25 GB/s), its share of what L2 delivers (39 GB/s, W and
// x together), and, where tiles are cut, 5 us for the second kernel and the
// way of the pieces through memory. Whole tiles on an uneven number of CUs
// against even parts with a join comes out of the same sum, and so does the
// caller's choice between this kernel and the library: up to 128 rows nine
// in ten sizes take 0.9 to 1.25 times the estimate (e4m3 1.0 to 1.6), above
// them 0.75 to 0.9.
struct Plan {
  int tiles = 0, parts = 0;
  bool split = false;
  double us = 0;
};

template <class S>
Plan plan_of(int N, int K, bool split) {
  constexpr int kChip = 256;
  Plan p;
  p.tiles = ceil_div(N, S::TN);
  const int64_t stages = static_cast<int64_t>(p.tiles) * (K / S::KS);
  p.split = split;
  // two stages at least, so that the ring has something to run ahead on
  p.parts = static_cast<int>(
      std::min<int64_t>(kChip, split ? (stages + 1) / 2 : p.tiles));
  const int64_t most = split
      ? (stages + p.parts - 1) / p.parts
      : static_cast<int64_t>(ceil_div(p.tiles, p.parts)) * (K / S::KS);
  p.us = most * std::max(S::kWB / 25e3, (S::kWB + S::kXB) / 39e3);
  if (split) p.us += 5 + p.parts * (S::kPiece * 16 * 2 / 4e6);
  return p;
}

template <class S>
Plan plan_of(int N, int K) {
  const Plan a = plan_of<S>(N, K, false), b = plan_of<S>(N, K, true);
  return a.us <= b.us ? a : b;
}

template <class S, bool SILU_MUL, bool FP8>
void launch_part(const Plan& pl, u16* out, float* pieces, const u16* x,
                 const u16* w, const u16* bias, const Scales& scales, int M,
                 int N, int K, int64_t x_stride, int64_t out_stride,
                 hipStream_t stream) {
  auto* p = reinterpret_cast<floatx4*>(pieces);
  hipLaunchKernelGGL((part_gemm_kernel<S, SILU_MUL, FP8>), dim3(pl.parts),
                     dim3(S::kWaves * kWaveSize), 0, stream, out, p, x, w,
                     bias, scales, M, N, K, x_stride, out_stride, pl.tiles,
                     pl.split ? 1 : K / S::KS);
  if (!pl.split || pl.parts == 1) return;
  hipLaunchKernelGGL((part_gemm_join_kernel<S, SILU_MUL, FP8>),
                     dim3(pl.parts - 1,
                          ceil_div(S::kPiece / (SILU_MUL ? 2 : 1), 256)),
                     dim3(256), 0, stream, out, p, bias, scales, M, N, K,
                     out_stride, pl.tiles, pl.parts);
}

// Row classes and their shapes: tiles of 96 rows where the chip takes them
// whole, 64 or 32 where N is small and K is cut, 128 or more where N is
// large and x would be read too often.
using A32 = PartShape<3, 2, 2, 1, 128, 5, 4, 4>;
using B32 = PartShape<2, 2, 2, 1, 64, 7, 7, 2>;
using A64 = PartShape<3, 2, 2, 2, 64, 7, 6, 4>;
using B64 = PartShape<2, 2, 4, 1, 64, 7, 7, 4>;
using C64 = PartShape<4, 2, 2, 2, 64, 6, 6, 4>;
using A128 = PartShape<3, 2, 4, 2, 64, 7, 4, 4>;
using B128 = PartShape<2, 2, 4, 2, 64, 7, 5, 4>;
using C128 = PartShape<4, 4, 2, 4, 64, 3, 4, 4>;
using A256 = PartShape<3, 2, 4, 4, 64, 5, 3, 4>;
using B256 = PartShape<2, 2, 8, 2, 64, 6, 3, 8>;

// calls f(shape, plan) for the shape that takes least
template <class F, class... Shapes>
void with_best(int N, int K, const F& f, Shapes...) {
  const Plan plans[] = {plan_of<Shapes>(N, K)...};
  const Plan* best = plans;
  for (const Plan& p : plans)
    if (p.us < best->us) best = &p;
  int i = 0;
  ((best == plans + i++ ? f(Shapes{}, *best) : void()), ...);
}

template <class F>
void with_shape(int M, int N, int K, const F& f) {
  if (M <= 32) with_best(N, K, f, A32{}, B32{});
  else if (M <= 64) with_best(N, K, f, A64{}, B64{}, C64{});
  else if (M <= 128) with_best(N, K, f, A128{}, B128{}, C128{});
  else with_best(N, K, f, A256{}, B256{});
}

}  // namespace

// what the chosen plan takes by its own estimate, in us
double part_gemm_us(int M, int N, int K) {
  double us = 0;
  with_shape(M, N, K, [&](auto, const Plan& pl) { us = pl.us; });
  return us;
}

// floats of scratch that launch_part_gemm needs
int64_t part_gemm_floats(int M, int N, int K) {
  int64_t n = 0;
  with_shape(M, N, K, [&](auto shape, const Plan& pl) {
    n = pl.split ? static_cast<int64_t>(pl.parts) * 2 * shape.kPiece * 4 : 0;
  });
  return n;
}

// 1 <= M <= 256, K a multiple of 128, N of 16 (32 with silu_mul)
void launch_part_gemm(u16* out, float* pieces, const u16* x, const u16* w,
                      const u16* bias, int M, int N, int K, int64_t x_stride,
                      int64_t out_stride, bool silu_mul,
                      hipStream_t stream) {
  with_shape(M, N, K, [&](auto shape, const Plan& pl) {
    using S = decltype(shape);
    if (silu_mul)
      launch_part<S, true, false>(pl, out, pieces, x, w, bias, Scales{}, M, N,
                                  K, x_stride, out_stride, stream);
    else
      launch_part<S, false, false>(pl, out, pieces, x, w, bias, Scales{}, M,
                                   N, K, x_stride, out_stride, stream);
  });
}

// e4m3 x and W with a scale per row each; K a multiple of 256
void launch_part_gemm_fp8(u16* out, float* pieces, const unsigned char* x,
                          const float* x_scales, const unsigned char* w,
                          const float* w_scales, int M, int N, int K,
                          int64_t x_stride, int64_t out_stride,
                          hipStream_t stream) {
  with_shape(M, N, K / 2, [&](auto shape, const Plan& pl) {
    launch_part<decltype(shape), false, true>(
        pl, out, pieces, reinterpret_cast<const u16*>(x),
        reinterpret_cast<const u16*>(w), nullptr, Scales{x_scales, w_scales},
        M, N, K / 2, x_stride / 2, out_stride, stream);
  });
}

}  // namespace fi
