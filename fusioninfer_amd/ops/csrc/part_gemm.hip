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
// What bounds it, from DMAs alone without products: a CU has at most some 41
// KB on the way and gets its data in the order asked for, so x, which comes
// from L2, waits behind W, which comes from HBM; both together arrive at 55 to
// 60 KB/us per CU (x alone at 130, W alone at 26, which is what HBM gives to 256
// CUs), whatever the depth of the rings. Hence tiles at least as tall as x has
// rows, taller where N allows. The second kernel of a cut product costs 4.7 us
// at the least, and results leave by stores that the next stages' waits count
// (8192 to 12288 x 1024 to 2048 at 17 to 128 rows 0.5 to 1.5 % less; where HBM is
// the bound nothing, 151936 x 4096 at 64 rows 249 us in whole tiles, 236 cut).
//
// From 129 rows on, and below where tiles have 128 rows, the fragment reads
// would be the bound, a wave of 32 x 64 results reading as much as it
// multiplies: there four waves hold a tile's rows of W by a quarter of x
// (part_gemm_ahead_kernel), read the fragments of half a stage during the
// products of the other half, and cross one barrier a stage.
// Before and now at 192 rows: 24576 x 4096 with silu 57 and 50 us, 4096 x 12288
// 43 and 38, 8192 x 8192 55 and 42; at 256 63 and 59, 45 and 43.5, 56 and 49;
// 151936 x 4096 at 256 446 and 345, the library 358.
//
// Measured, us (GB/s of W) at 32 / 64 / 128 / 256 rows: N 24576, K 4096 with
// silu 33.4 (6030) / 33.9 / 44.3 / 58, the library's GEMM and the pass behind it
// 48 / 49 / 53 / 70; 4096, 12288 21 (4780) / 26 / 33 / 42 against 26 / 37 / 66 /
// 55; 151936, 2048 109 (5690) / 129 / 151 / 192 against 146 / 153 / 168 / 212 (at
// 256 rows 176 by tiles of 256 x 256).
//
// Where a norm follows, the second kernel does the sum with the residual and
// the norm too (part_gemm_norm_kernel): a launch of 3 to 5 us less, and the
// product is not rounded before the sum. us in a graph, product and norm / both
// in one, at 43 / 64 / 128 / 256 rows: 4096 x 4096 16.3, 17.0, 21.8, 28.5 / 14.6,
// 15.1, 19.7, 27.1; 4096 x 12288 27.5, 28.8, 35.5, 45.7 / 25.9, 27.7, 33.9, 43.9;
// e4m3 at 64 rows 16.4 / 14.2 and 23.6 / 21.5. (At 256 rows the library takes
// 4096 x 4096 and its norm in 26.4.)
//
// FP8: the same kernel on e4m3 rows, 1 to 128 of them. 24576 x 4096 at 16 / 32
// / 64 rows 19.3 (5210) / 19.9 / 22.7 us, the library's GEMM 30.0 / 25.3 /
// 26.4; 4096 x 12288 13.9 (3630) / 14.5 / 18.0 against 19.2 / 20.3 / 24.2.

#include <cmath>
#include <type_traits>

#include "pieces.h"
#include "tile_engine.h"

namespace fi {

void launch_rope_of_pieces(u16*, const PieceRows&, const RopeArgs&, int,
                           hipStream_t);

namespace {

template <int N>
FI_DEV void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

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
  static constexpr bool kAhead = false, kCuts = true, kColumns = false;
  static_assert(RF % 2 == 0 && TN / 2 % kRowsPerDma == 0);
  static_assert(LW * kRowsPerDma * kWLoaders == TN &&
                LX * kRowsPerDma * kXLoaders == MB);
  static_assert(RW * kWB + RX * kXB <= 160 * 1024 && RW >= 2 && RW <= 7 &&
                RX >= 2 && RX <= 7);
};

// the same for part_gemm_ahead_kernel: four waves of RF x CF fragments
template <int RF, int CF, int RW, int RX>
struct AheadShape : PartShape<1, RF, 4, CF, 64, RW, RX, 2> {
  static constexpr bool kAhead = true, kColumns = 4 * CF * 16 > 128;
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

// Where a piece has a lane's results of a fragment: fragment by fragment of a
// wave, or, with ROWS, for a kernel that sums whole rows. There rows of the tile
// follow one another; in shapes for more than 128 rows of x, where that kernel
// has workgroups enough and the product is held up by its stores, 16 columns of
// all rows do (kColumns): a wave's store is 1 KB in one, not 16 times 64 bytes.
// (Both kernels with rows / columns: 4096 x 4096 at 43 rows 15.7 / 16.4 us, at 192
// 25.3 / 24.4, at 256 30.0 / 27.7; 4096 x 12288 at 65 and 128 rows, waves that
// read ahead too, 30.4 and 33.8 / 31.2 and 34.2.)
template <class S, bool ROWS>
FI_DEV int in_piece(int wave, int wn, int wm, int f, int c, int lane) {
  if (!ROWS) return ((wave * S::RF + f) * S::CF + c) * kWaveSize + lane;
  const int m = (wm * S::CF + c) * 16 + (lane & 15), nf = wn * S::RF + f;
  return S::kColumns ? (nf * S::MB + m) * 4 + (lane >> 4)
                   : m * (S::TN / 4) + nf * 4 + (lane >> 4);
}

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
template <class S, bool SILU_MUL, bool FP8, bool ROWS>
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

  // results on their way out are behind the DMAs that the next stages wait for
  constexpr int kStores = (SILU_MUL ? RF / 2 : RF) * CF;
  int wslot = 0, xslot = 0, pos = lo, behind = 0;
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
    // two loops, so that the one that all stages but a few go through does not
    // ask each time (4096 x 12288 at 17 / 64 / 128 rows in one loop 22.3 / 27.4 /
    // 35.1 us, in two 20.4 / 26.0 / 33.9)
    auto run = [&](auto behind_stores, const int to) {
      for (; pos < to; ++pos) {
        // this wave's share of the stage has landed; after the barrier all
        // shares have, and every wave is done with the slot read last
        constexpr bool kBehind = decltype(behind_stores)::value;
        if (loads_w) {
          if (kBehind && issued - pos > S::RW - 2)
            wait_vm<(S::RW - 2) * LW + kStores>();
          else
            wait_stages<LW, S::RW - 2>(issued - pos - 1);
        } else {
          if (kBehind && issued - pos > S::RX - 2)
            wait_vm<(S::RX - 2) * LX + kStores>();
          else
            wait_stages<LX, S::RX - 2>(issued - pos - 1);
        }
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
    };
    if (behind > 0) run(std::true_type{}, min(stop, pos + behind));
    run(std::false_type{}, stop);
    if (!ROWS && from_start && stop == end) {
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
      // stage pos + RW - 2 has been requested before the stores
      behind = 0;
      if ((wm * CF + CF - 1) * 16 < M &&
          (tile + 1) * (SILU_MUL ? S::TN / 2 : S::TN) <=
              (SILU_MUL ? N / 2 : N))
        behind = (loads_w ? S::RW : S::RX) - 1;
    } else {
      // a part holds at most two pieces: the end of a tile that an earlier
      // part began (0) and the start of one that goes on (1)
      floatx4* p = pieces + (static_cast<int64_t>(blockIdx.x) * 2 +
                             (from_start ? 1 : 0)) * S::kPiece;
#pragma unroll
      for (int f = 0; f < RF; ++f)
#pragma unroll
        for (int c = 0; c < CF; ++c)
          p[in_piece<S, ROWS>(wave, wn, wm, f, c, lane)] = acc[f][c];
      behind = (loads_w ? S::RW : S::RX) - 1;
    }
  }
}

// Four waves that read ahead, each a tile's rows of W by a quarter of x; two
// load W, two x (LOADS_W). Each MFMA is followed by at most one read or DMA, in
// an order that is pinned: one wave per SIMD hides nothing by itself. While the
// first half of a stage (32 of K) is multiplied the fragments of the second are
// read; with them in registers, and the next stage landed, the barrier frees the
// stage's place, and the second half's products cover the reads of the next
// stage's first half and half of the DMAs into the free place.
template <class S, bool SILU_MUL, bool ROWS, bool LOADS_W>
FI_DEV void run_ahead(u16* __restrict__ out, floatx4* __restrict__ pieces,
                      const u16* __restrict__ x, const u16* __restrict__ w,
                      const u16* __restrict__ bias, const int M, const int N,
                      const int K, const int64_t x_stride,
                      const int64_t out_stride, const int tiles,
                      const int unit, unsigned char* smem, const int wave,
                      const int lane) {
  constexpr int RF = S::RF, CF = S::CF;
  constexpr int R = LOADS_W ? S::RW : S::RX, L = LOADS_W ? S::LW : S::LX;
  constexpr int kLoaders = LOADS_W ? S::kWLoaders : S::kXLoaders;
  constexpr int kSlotB = LOADS_W ? S::kWB : S::kXB;
  const int SK = K / S::KS;
  const Cut cut(tiles * SK / unit, gridDim.x, unit);
  const int lo = cut.start(blockIdx.x), hi = cut.start(blockIdx.x + 1);
  const int lwave = LOADS_W ? wave : wave - S::kWLoaders;

  // ---- requests: DMA j of a wave brings eight rows, group kLoaders j + lwave;
  // lane l chunk (l % 8) ^ key of one of them. The row is in the vector
  // offset, the place along K in the scalar one; rows past the descriptor's
  // end come as zeros.
  const u32 ring = static_cast<u32>(reinterpret_cast<uintptr_t>(
                       (__attribute__((address_space(3))) unsigned char*)
                           smem)) +
                   (LOADS_W ? 0 : S::RW * S::kWB) + lwave * 1024;
  const u32 row_b = LOADS_W ? K * 2 : static_cast<u32>(x_stride) * 2;
  u32 voff[L];
#pragma unroll
  for (int j = 0; j < L; ++j) {
    const int half = LOADS_W && SILU_MUL ? L / 2 : L;
    const int g = j * kLoaders + lwave;
    const int r = (j % half * kLoaders + lwave) * 8 + (lane >> 3);
    voff[j] = (LOADS_W ? r : min(r, M - 1)) * row_b +
              (((lane & 7) ^ ((lane >> 4) | ((g & 1) << 2))) << 4);
  }
  u32x4 d0{}, d1{};
  u32 soff = 0;
  int rt = lo / SK, issued = lo, rs = 0, ra = 0, rb = 0, left = 0;
  constexpr int kPast = 1 << 30;
  auto seek = [&] { soff = left > kPast / 2 ? 0 : rs * S::kRowB; };
  auto enter = [&] {
    if (issued >= hi) {           // past the end nothing is read
      d0[2] = d1[2] = 0;
      left = kPast;
      return;
    }
    ra = max(lo - rt * SK, 0);
    rb = max(min(hi - rt * SK, SK), ra + 1);
    rs = ra + static_cast<int>(blockIdx.x / 8) % (rb - ra);
    left = rb - ra;
    if (LOADS_W) {
      const int n0 = rt * (SILU_MUL ? S::TN / 2 : S::TN);
      const int cols = SILU_MUL ? N / 2 : N;
      const u32 bytes = min(SILU_MUL ? S::TN / 2 : S::TN, cols - n0) * row_b;
      d0 = uniform_descriptor(w + static_cast<int64_t>(n0) * K, bytes);
      if (SILU_MUL)
        d1 = uniform_descriptor(w + static_cast<int64_t>(cols + n0) * K,
                                bytes);
    }
  };
  if (!LOADS_W) d0 = uniform_descriptor(x, (M - 1) * row_b + K * 2);
  enter();
  seek();
  u32 rdst = ring;
  int rslot = 0;
  auto m0_of = [&](int j) { set_m0(rdst + j * kLoaders * 1024); };
  auto load_of = [&](int j) {
    if (!LOADS_W)
      load_lds(d0, voff[j], soff);
    else
      load_lds_nt(SILU_MUL && j >= L / 2 ? d1 : d0, voff[j], soff);
  };
  auto requested = [&] {
    rdst += kSlotB;
    if (++rslot == R) {
      rslot = 0;
      rdst = ring;
    }
    ++issued;
    if (++rs == rb) rs = ra;
    if (--left == 0) {
      ++rt;
      enter();
    }
    seek();
  };

  // ---- fragment reads
  const int ir = lane & 15, q = lane >> 4;
  const int rd = ir * S::kRowB + ((q ^ (ir >> 1 & 7)) << 4);
  short8 a0[CF], b0[RF], a1[CF], b1[RF];
  floatx4 acc[RF][CF];
  int wat = 0, xat = S::RW * S::kWB + wave * CF * 16 * S::kRowB;
  auto read = [&](short8 (&a)[CF], short8 (&b)[RF], int half, int i) {
    const int at = rd ^ (half * 64);
    if (i < CF)
      a[i] = *reinterpret_cast<const short8*>(smem + xat + at +
                                              i * 16 * S::kRowB);
    else
      b[i - CF] = *reinterpret_cast<const short8*>(
          smem + wat + at + (i - CF) * 16 * S::kRowB);
  };
  constexpr int kReads = RF + CF, kMfmas = RF * CF;
  constexpr int kEvery = 2 * kReads <= kMfmas + 1 ? 2 : 1;  // products a read
  // DMAs go out at even distances over both halves: kSoon of a stage's L in the
  // second half, the rest in the first half of the next stage
  constexpr int kSoon = L / 2, kApart = kMfmas / (L - kSoon);
  static_assert(kReads <= kMfmas && L % 2 == 0 && kApart >= 2);
  constexpr int kStores = (SILU_MUL ? RF / 2 : RF) * CF;
  auto product = [&](int i, const short8 (&a)[CF], const short8 (&b)[RF],
                     bool first) {
    const int c = i / RF, f = i % RF;
    if (first) mfma_first(acc[f][c], b[f], a[c]);
    else mfma(acc[f][c], b[f], a[c]);
    __builtin_amdgcn_sched_barrier(0);
  };

  for (int k = 0; k < R; ++k) {
#pragma unroll
    for (int j = 0; j < L; ++j) {
      if (k == R - 1 && j >= kSoon) break;
      m0_of(j);
      asm volatile("s_nop 4");
      load_of(j);
    }
    if (k < R - 1) requested();
  }
  wait_vm<(R - 2) * L + kSoon>();
  sync_waves();
#pragma unroll
  for (int i = 0; i < kReads; ++i) read(a0, b0, 0, i);
  int wslot = 0, xslot = 0;
  auto stage = [&](auto first, bool behind) {
#pragma unroll
    for (int i = 0; i < kMfmas; ++i) {
      product(i, a0, b0, first);
      if (i % kEvery == 0 && i / kEvery < kReads)
        read(a1, b1, 1, i / kEvery);
      if (i / kApart < L - kSoon) {
        if (i % kApart == 0) m0_of(kSoon + i / kApart);
        if (i % kApart == 1) load_of(kSoon + i / kApart);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    requested();
    // the stage is in registers, this wave's share of the next has landed;
    // after the barrier that is so for all waves
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (behind) wait_vm<(R - 2) * L + kStores>();
    else wait_vm<(R - 2) * L>();
    sync_waves();
    wat += S::kWB;
    if (++wslot == S::RW) wslot = wat = 0;
    xat += S::kXB;
    if (++xslot == S::RX) {
      xslot = 0;
      xat -= S::RX * S::kXB;
    }
#pragma unroll
    for (int i = 0; i < kMfmas; ++i) {
      product(i, a1, b1, false);
      if (i % kEvery == 0 && i / kEvery < kReads)
        read(a0, b0, 0, i / kEvery);
      if (i / kApart < kSoon) {
        if (i % kApart == 0) m0_of(i / kApart);
        if (i % kApart == 1) load_of(i / kApart);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  int pos = lo, behind = 0;
  while (pos < hi) {
    const int tile = pos / SK;
    const int begin = tile * SK, end = begin + SK;
    const bool from_start = pos == begin;
    const int stop = min(hi, end);
    stage(std::true_type{}, behind > 0);
    --behind;
    for (++pos; pos < stop; ++pos, --behind)
      stage(std::false_type{}, behind > 0);
    settle();
    int l = lane;
    asm volatile("" : "+v"(l));
    if (!ROWS && from_start && stop == end) {
#pragma unroll
      for (int f = 0; f < (SILU_MUL ? RF / 2 : RF); ++f) {
        const int n = tile * (SILU_MUL ? S::TN / 2 : S::TN) + f * 16 +
                      (l >> 4) * 4;
#pragma unroll
        for (int c = 0; c < CF; ++c) {
          const int m = (wave * CF + c) * 16 + (l & 15);
          if (m < M && n < (SILU_MUL ? N / 2 : N))
            store4<SILU_MUL, false>(
                out, bias, Scales{}, acc_of(acc[f][c]),
                acc_of(acc[SILU_MUL ? f + RF / 2 : f][c]), m, n, out_stride);
        }
      }
      behind = 0;
      if ((wave * CF + CF - 1) * 16 < M &&
          (tile + 1) * (SILU_MUL ? S::TN / 2 : S::TN) <=
              (SILU_MUL ? N / 2 : N))
        behind = R - 2;
    } else {
      floatx4* p = pieces + (static_cast<int64_t>(blockIdx.x) * 2 +
                             (from_start ? 1 : 0)) * S::kPiece;
#pragma unroll
      for (int f = 0; f < RF; ++f)
#pragma unroll
        for (int c = 0; c < CF; ++c)
          p[in_piece<S, ROWS>(wave, 0, wave, f, c, l)] = acc_of(acc[f][c]);
      behind = R - 2;
    }
  }
  // no DMA may land in LDS that is no longer this workgroup's
  wait_vm<0>();
}

template <class S, bool SILU_MUL, bool ROWS>
__global__ __launch_bounds__(256, 1)
void part_gemm_ahead_kernel(u16* __restrict__ out,
                            floatx4* __restrict__ pieces,
                            const u16* __restrict__ x,
                            const u16* __restrict__ w,
                            const u16* __restrict__ bias, const int M,
                            const int N, const int K, const int64_t x_stride,
                            const int64_t out_stride, const int tiles,
                            const int unit) {
  __shared__ __attribute__((aligned(1024)))
  unsigned char smem[S::RW * S::kWB + S::RX * S::kXB];
  const int lane = threadIdx.x % kWaveSize;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  if (wave < S::kWLoaders)
    run_ahead<S, SILU_MUL, ROWS, true>(out, pieces, x, w, bias, M, N, K,
                                       x_stride, out_stride, tiles, unit, smem,
                                       wave, lane);
  else
    run_ahead<S, SILU_MUL, ROWS, false>(out, pieces, x, w, bias, M, N, K,
                                        x_stride, out_stride, tiles, unit,
                                        smem, wave, lane);
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

// The second kernel where a norm follows: a workgroup sums a row's pieces, adds
// the residual, writes it back and leaves the normed row, as bf16 or (FP8) as
// e4m3 with the row's scale. Bound by the way of the pieces through memory,
// all of a thread's on their way at once; 256 rows of 4096 take 7.8 us,
// the sum of pieces alone 6.8 and the norm 4.4.
template <bool FP8, int THREADS, int ITERS>
__global__ __launch_bounds__(THREADS)
void part_gemm_norm_kernel(void* __restrict__ out, float* __restrict__ out_scales,
                           const PieceRows pieces, u16* __restrict__ residual,
                           const u16* __restrict__ norm, const float eps,
                           const Scales scales, const int M, const int N) {
  const int m = piece_row(pieces.columns);
  if (m >= M) return;
  const int64_t row = static_cast<int64_t>(m) * N;
  floatx4 v[ITERS];
  bf16x4 weight[ITERS];
  float squares = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int n = (it * THREADS + static_cast<int>(threadIdx.x)) * 4;
    v[it] = {0.f, 0.f, 0.f, 0.f};
    if (n < N) {
      weight[it] = *reinterpret_cast<const bf16x4*>(norm + n);
      const bf16x4 r = *reinterpret_cast<const bf16x4*>(residual + row + n);
      constexpr int kAtOnce = 8;
      for (PieceReader p(pieces, m, n); p.next <= p.last; p.next += kAtOnce) {
        floatx4 got[kAtOnce];
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i)
          got[i] = __builtin_bit_cast(floatx4, p.get(i, 0));
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i) v[it] += got[i];
      }
      bf16x4 sum;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (FP8) v[it][j] *= scales.x[m] * scales.w[n + j];
        v[it][j] += bf16_to_f32(r.h[j]);
        sum.h[j] = f32_to_bf16(v[it][j]);
        squares = fmaf(v[it][j], v[it][j], squares);
      }
      *reinterpret_cast<bf16x4*>(residual + row + n) = sum;
    }
  }
  __shared__ float scratch[2][THREADS / kWaveSize];
  squares = block_reduce_sum<THREADS / kWaveSize>(wave_reduce_sum(squares),
                                                  scratch[0]);
  const float inv_rms = rsqrtf(squares / N + eps);
  float most = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int n = (it * THREADS + static_cast<int>(threadIdx.x)) * 4;
    if (n >= N) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[it][j] *= inv_rms * bf16_to_f32(weight[it].h[j]);
      most = fmaxf(most, fabsf(v[it][j]));
    }
    if (!FP8) {
      bf16x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o.h[j] = f32_to_bf16(v[it][j]);
      *reinterpret_cast<bf16x4*>(static_cast<u16*>(out) + row + n) = o;
    }
  }
  if (!FP8) return;
  most = block_reduce_max<THREADS / kWaveSize>(wave_reduce_max(most),
                                               scratch[1]);
  const float scale = fmaxf(most, 1e-8f) / 448.0f, inv = 1.f / scale;
  if (threadIdx.x == 0) out_scales[m] = scale;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int n = (it * THREADS + static_cast<int>(threadIdx.x)) * 4;
    if (n >= N) continue;
    float o[8] = {v[it][0] * inv, v[it][1] * inv, v[it][2] * inv,
                  v[it][3] * inv};
    u32 packed[2];
    pack_fp8x8(o, packed);
    *reinterpret_cast<u32*>(static_cast<unsigned char*>(out) + row + n) =
        packed[0];
  }
}

// us of a shape: a stage while few CUs stream and while all do, where HBM has its
// say; what whole tiles take beside their stages; what cut ones do beside those
// and 3 us, the second kernel and the way of the pieces through memory.
struct Times {
  double whole, cut, lone, full;
};

// How a shape cuts [N, K] up and what that takes by its times, which are
// measured (20 N by eleven K, weights that no cache holds, plain, with silu and
// e4m3, 10000 runs). Whole tiles on an uneven number of CUs against even parts
// with a join comes out of the same sum, and so does the caller's choice between
// this kernel and the library. Of what the best shape takes the one taken takes
// 0.5 to 0.6 % more on average, 20 at most (65536 x 2048 with silu at 17 rows), and
// the sum is 7 % off (one rate of a stage, whether few CUs stream or all: 1.3 %
// more, 27 at most, and 13 % off).
struct Plan {
  int tiles = 0, parts = 0;
  bool split = false;
  double us = 0;
};

// stage: by how much this kind of operands makes a stage longer
template <class S>
Plan plan_of(int N, int K, bool split, double stage) {
  constexpr int kChip = 256;
  constexpr Times us = S::kUs;
  Plan p;
  p.tiles = ceil_div(N, S::TN);
  p.split = split;
  const int64_t of_tile = K / S::KS, stages = p.tiles * of_tile;
  // two stages at least, so that the ring has something to run ahead on
  p.parts = static_cast<int>(
      std::min<int64_t>(kChip, split ? (stages + 1) / 2 : p.tiles));
  // rounds that all CUs take part in, and the last one
  const int rounds = split ? 1 : ceil_div(p.tiles, kChip);
  const int64_t most = split ? (stages + p.parts - 1) / p.parts : of_tile;
  const double busy =
      (split ? p.parts : p.tiles - (rounds - 1) * kChip) / double{kChip};
  const double shared = us.full * busy;
  const double last = std::sqrt(std::sqrt(
      us.lone * us.lone * us.lone * us.lone + shared * shared * shared * shared));
  p.us = stage * ((rounds - 1) * most * us.full + most * last) +
         (split ? 3 + us.cut * busy : us.whole);
  return p;
}

template <class S>
Plan plan_of(int N, int K, double stage) {
  const Plan whole = plan_of<S>(N, K, false, stage);
  if (!S::kCuts) return whole;
  const Plan cut = plan_of<S>(N, K, true, stage);
  return whole.us <= cut.us ? whole : cut;
}

template <class S, bool SILU_MUL, bool FP8, bool ROWS>
void launch_products(const Plan& pl, u16* out, float* pieces, const u16* x,
                     const u16* w, const u16* bias, const Scales& scales,
                     int M, int N, int K, int64_t x_stride, int64_t out_stride,
                     hipStream_t stream) {
  auto* p = reinterpret_cast<floatx4*>(pieces);
  const int unit = pl.split ? 1 : K / S::KS;
  if constexpr (S::kAhead) {
    static_assert(!FP8);
    hipLaunchKernelGGL((part_gemm_ahead_kernel<S, SILU_MUL, ROWS>),
                       dim3(pl.parts), dim3(256), 0, stream, out, p, x, w,
                       bias, M, N, K, x_stride, out_stride, pl.tiles, unit);
  } else {
    hipLaunchKernelGGL((part_gemm_kernel<S, SILU_MUL, FP8, ROWS>),
                       dim3(pl.parts), dim3(S::kWaves * kWaveSize), 0, stream,
                       out, p, x, w, bias, scales, M, N, K, x_stride,
                       out_stride, pl.tiles, unit);
  }
}

template <class S, bool SILU_MUL, bool FP8>
void launch_part(const Plan& pl, u16* out, float* pieces, const u16* x,
                 const u16* w, const u16* bias, const Scales& scales, int M,
                 int N, int K, int64_t x_stride, int64_t out_stride,
                 hipStream_t stream) {
  launch_products<S, SILU_MUL, FP8, false>(pl, out, pieces, x, w, bias, scales,
                                           M, N, K, x_stride, out_stride,
                                           stream);
  if constexpr (S::kCuts) {
    if (!pl.split || pl.parts == 1) return;
    auto* p = reinterpret_cast<const floatx4*>(pieces);
    hipLaunchKernelGGL((part_gemm_join_kernel<S, SILU_MUL, FP8>),
                       dim3(pl.parts - 1,
                            ceil_div(S::kPiece / (SILU_MUL ? 2 : 1), 256)),
                       dim3(256), 0, stream, out, p, bias, scales, M, N, K,
                       out_stride, pl.tiles, pl.parts);
  }
}

// Row classes and their shapes: tiles of 96 rows where the chip takes them
// whole, 64 where N is small and K is cut, 128 or more where N is large and x
// would be read too often. Waves that read ahead are ahead of the others from
// 129 rows on, and at 65 to 128 where tiles of 128 rows are.
struct B32 : PartShape<2, 2, 2, 1, 64, 7, 7, 2> {
  static constexpr Times kUs{4.7, 3.7, 0.242, 0.303};
};
// (cut, these two are next to never the best, and far off where parts begin in
// step: 10240 x 12288 at 17 rows 44 us with tiles of 64 rows, 56 with 128)
struct A32 : PartShape<3, 2, 2, 1, 128, 5, 4, 4> {
  static constexpr Times kUs{4.8, 0, 0.555, 0.929};
  static constexpr bool kCuts = false;
};
struct C32 : PartShape<4, 2, 2, 1, 128, 4, 4, 4> {
  static constexpr Times kUs{4.6, 0, 0.652, 1.21};
  static constexpr bool kCuts = false;
};
struct B64 : PartShape<2, 2, 4, 1, 64, 7, 7, 4> {
  static constexpr Times kUs{5.8, 5.9, 0.277, 0.361};
};
struct A64 : PartShape<3, 2, 2, 2, 128, 4, 4, 4> {
  static constexpr Times kUs{6.3, 7.3, 0.617, 1.009};
};
struct C64 : PartShape<4, 2, 2, 2, 64, 6, 6, 4> {
  static constexpr Times kUs{6.2, 7.7, 0.412, 0.669};
};
struct D64 : PartShape<4, 4, 2, 2, 64, 4, 4, 4> {
  static constexpr Times kUs{5.3, 12, 0.812, 1.239};
};
struct B128 : PartShape<2, 2, 4, 2, 64, 7, 5, 4> {
  static constexpr Times kUs{7.2, 8.3, 0.367, 0.448};
};
struct A128 : PartShape<3, 2, 4, 2, 64, 7, 4, 4> {
  static constexpr Times kUs{7.7, 10.8, 0.461, 0.584};
};
struct C128 : AheadShape<8, 2, 6, 4> {
  static constexpr Times kUs{7.9, 10.7, 0.483, 0.759};
};
struct D128 : PartShape<4, 4, 2, 4, 64, 3, 4, 4> {
  static constexpr Times kUs{8.9, 16.6, 1.04, 1.348};
};
struct A192 : AheadShape<6, 3, 5, 4> {
  static constexpr Times kUs{6.3, 11.3, 0.563, 0.701};
};
struct C192 : AheadShape<8, 3, 4, 4> {
  static constexpr Times kUs{6, 13.1, 0.668, 0.911};
};
struct A256 : AheadShape<6, 4, 5, 3> {
  static constexpr Times kUs{7.1, 12.4, 0.665, 0.839};
};
struct C256 : AheadShape<8, 4, 4, 3> {
  static constexpr Times kUs{6.8, 14.6, 0.778, 1.075};
};
// for few tiles with few stages each (10240 x 2048 with silu at 256 rows 25 us, by
// waves that read ahead 29), and rows of W too long for the others' offsets
// within a tile
struct B256 : PartShape<2, 2, 8, 2, 64, 6, 3, 8> {
  static constexpr Times kUs{6.3, 11, 0.576, 0.672};
};

// calls f(shape, plan) for the shape that takes least
template <class F, class... Shapes>
void with_best(int N, int K, double stage, const F& f, Shapes...) {
  const Plan plans[] = {plan_of<Shapes>(N, K, stage)...};
  const Plan* best = plans;
  for (const Plan& p : plans)
    if (p.us < best->us) best = &p;
  int i = 0;
  ((best == plans + i++ ? f(Shapes{}, *best) : void()), ...);
}

// A stage of e4m3 has twice the products on the same bytes: the longer the more
// rows of x there are.
template <bool FP8, class F>
void with_shape(int M, int N, int K, const F& f) {
  // the waves that read ahead are bf16 ones with 32-bit offsets in a tile of W
  const bool ahead = !FP8 && K <= 1 << 22;
  const double stage = !FP8 ? 1 : M <= 32 ? 1.03 : M <= 64 ? 1.08 : 1.24;
  if (M <= 32) {
    with_best(N, K, stage, f, A32{}, B32{}, C32{});
  } else if (M <= 64) {
    with_best(N, K, stage, f, A64{}, B64{}, C64{}, D64{});
  } else if (!ahead) {
    if (M <= 128) with_best(N, K, stage, f, A128{}, B128{}, D128{});
    else with_best(N, K, stage, f, B256{});
  } else if constexpr (!FP8) {
    if (M <= 128) with_best(N, K, stage, f, A128{}, B128{}, C128{}, D128{});
    else if (M <= 192) with_best(N, K, stage, f, A192{}, C192{});
    else with_best(N, K, stage, f, A256{}, B256{}, C256{});
  }
}

}  // namespace

// what the chosen plan takes by its own estimate, in us
double part_gemm_us(int M, int N, int K, bool fp8) {
  double us = 0;
  auto take = [&](auto, const Plan& pl) { us = pl.us; };
  if (fp8) with_shape<true>(M, N, K / 2, take);
  else with_shape<false>(M, N, K, take);
  return us;
}

// floats of scratch that launch_part_gemm (fp8: launch_part_gemm_fp8 with twice
// the K) needs
int64_t part_gemm_floats(int M, int N, int K, bool fp8) {
  int64_t n = 0;
  auto count = [&](auto shape, const Plan& pl) {
    n = pl.split ? static_cast<int64_t>(pl.parts) * 2 * shape.kPiece * 4 : 0;
  };
  if (fp8) with_shape<true>(M, N, K, count);
  else with_shape<false>(M, N, K, count);
  return n;
}

// 1 <= M <= 256, K a multiple of 128, N of 16 (32 with silu_mul)
void launch_part_gemm(u16* out, float* pieces, const u16* x, const u16* w,
                      const u16* bias, int M, int N, int K, int64_t x_stride,
                      int64_t out_stride, bool silu_mul,
                      hipStream_t stream) {
  with_shape<false>(M, N, K, [&](auto shape, const Plan& pl) {
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
  with_shape<true>(M, N, K / 2, [&](auto shape, const Plan& pl) {
    launch_part<decltype(shape), false, true>(
        pl, out, pieces, reinterpret_cast<const u16*>(x),
        reinterpret_cast<const u16*>(w), nullptr, Scales{x_scales, w_scales},
        M, N, K / 2, x_stride / 2, out_stride, stream);
  });
}

// The products of 17 to 256 rows (e4m3: 1 to 128) in pieces, and then sum(where
// they are). Whether that is done, which it is where the pieces are summed by a
// second kernel anyway and no part holds more than a tile; if not, or without
// scratch, nothing is. x_scales: e4m3 operands, sizes in pairs of values.
template <class F>
bool in_pieces(float* pieces, const u16* x, const float* x_scales,
               const u16* w, const float* w_scales, const u16* bias, int M,
               int N, int K, int64_t x_stride, hipStream_t stream,
               const F& sum) {
  bool done = false;
  auto run = [&](auto shape, const Plan& pl, auto fp8) {
    using S = decltype(shape);
    constexpr bool kFp8 = decltype(fp8)::value;
    if constexpr (S::kCuts) {
      if (!pl.split || pl.tiles >= pl.parts) return;
      done = true;
      if (pieces == nullptr) return;
      launch_products<S, false, kFp8, true>(
          pl, nullptr, pieces, x, w, nullptr, Scales{x_scales, w_scales}, M, N,
          K, x_stride, 0, stream);
      sum(PieceRows{pieces, bias, S::TN, K / S::KS, pl.tiles, pl.parts, S::MB,
                    S::kColumns});
    }
  };
  if (x_scales != nullptr)
    with_shape<true>(M, N, K, [&](auto shape, const Plan& pl) {
      run(shape, pl, std::true_type{});
    });
  else
    with_shape<false>(M, N, K, [&](auto shape, const Plan& pl) {
      run(shape, pl, std::false_type{});
    });
  return done;
}

// residual += x W^T and the norm behind, N up to 16384
bool launch_part_gemm_norm(void* out, float* out_scales, u16* residual,
                           const u16* norm, float eps, float* pieces,
                           const u16* x, const float* x_scales, const u16* w,
                           const float* w_scales, int M, int N, int K,
                           int64_t x_stride, hipStream_t stream) {
  if (N > 16384) return false;
  return in_pieces(
      pieces, x, x_scales, w, w_scales, nullptr, M, N, K, x_stride, stream,
      [&](const PieceRows& rows) {
        const dim3 grid(ceil_div(M, 16) * 16);
#define FI_NORM(FP8, THREADS, ITERS)                                          \
  hipLaunchKernelGGL((part_gemm_norm_kernel<FP8, THREADS, ITERS>), grid,      \
                     dim3(THREADS), 0, stream, out, out_scales, rows,         \
                     residual, norm, eps, Scales{x_scales, w_scales}, M, N)
#define FI_NORM_N(FP8)                                                        \
  if (N <= 2048) FI_NORM(FP8, 512, 1);                                        \
  else if (N <= 4096) FI_NORM(FP8, 1024, 1);                                  \
  else if (N <= 8192) FI_NORM(FP8, 1024, 2);                                  \
  else FI_NORM(FP8, 1024, 4)
        if (x_scales != nullptr) {
          FI_NORM_N(true);
        } else {
          FI_NORM_N(false);
        }
#undef FI_NORM_N
#undef FI_NORM
      });
}

// x W^T + bias as heads of 64 or 128: queries normed and rotated to q, K and V
// rows to the paged cache
bool launch_part_gemm_rope(u16* q, const RopeArgs& rope, const u16* bias,
                           float* pieces, const u16* x, const u16* w, int M,
                           int N, int K, int64_t x_stride,
                           hipStream_t stream) {
  return in_pieces(pieces, x, nullptr, w, nullptr, bias, M, N, K, x_stride,
                   stream, [&](const PieceRows& rows) {
                     launch_rope_of_pieces(q, rows, rope, M, stream);
                   });
}

}  // namespace fi
