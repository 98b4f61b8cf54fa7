// y = x W^T for more than 256 rows of x (prompts): bf16 operands, or e4m3
// with a scale per row of either, fp32 accumulation, W [N, K] row-major.
// Bound by the matrix cores.
//
// 256 persistent workgroups, one per CU, take tiles of 256 rows of x by 256
// rows of W. Four waves hold 128 x 128 results each (256 registers), which
// is what keeps LDS out of the way: every fragment read feeds eight MFMAs, so
// a stage of 64 of K costs LDS 1024 cycles of reads and 512 of writes beside
// the 2048 that the matrix cores need. (Eight waves of 128 x 64 read half as
// much again and reach 1.42 PFLOP/s at most.)
//
// A stage is 64 KB, 256 rows of 128 bytes from either operand; two of them
// are kept. A stage is used in two halves of 32 of K. While the first half is
// multiplied the fragments of the second are read; with them in registers the
// stage's place is free (a barrier), three quarters of the way through the
// first half, and the stage after the next is requested into it from there
// on: it has five quarters of a stage's time to arrive. The second half's
// products cover the reads of the next stage's first half. Every MFMA is
// followed by at most one other instruction, in an order that is pinned: one
// wave per SIMD hides nothing by itself. The DMAs run on over the borders of
// tiles, so a tile's results are written while the next one's stages arrive;
// its first stage does not wait for them, and no accumulators are cleared
// (0.3 % of 24576 x 4096 at 8192 rows, e4m3 0.7 %).
//
// Rows lie in LDS as eight chunks of 16 bytes, chunk c of row r at c ^ key(r):
// the 16 lanes that LDS serves together then touch all its banks (no
// conflicts counted), and a DMA still reads whole lines of eight rows.
//
// MFMA with A = x, B = W, 16x16x32 in bf16. A wave's 128 columns are dealt to the
// places of its fragments so that lane i of 16 has columns 8 i to 8 i + 7 of a
// row, 16 bytes beside the next lane's: a CU takes stores 64 bytes of neighbouring
// lanes at a time, a tile's 128 KB in 0.9 us so, in 3.5 with A = W, where
// neighbouring lanes have neighbouring rows. (Once all CUs write at the same time
// memory takes as long.) us, the latter and this: 8000 x 2048, N 5120 142.9 and
// 139.4; e4m3, 8 bytes a lane, 8100 x 4096, N 6144, 4096, 24576 166, 106, 603 and
// 161, 101, 585; 4099 x 4096, N 6144 102 and 98.
//
// What whole rounds of 256 tiles leave over is cut along K into equal pieces
// (tile_plan), which a second kernel sums in a fixed order.
//
// Where rows are a multiple of 4 KB, reads of the same K by all CUs meet on few
// memory channels. With rows longer than 16 KB every other column tile starts
// half way along K: bf16, 4096 x 12288 at 4099, 6000 and 7600 rows 294, 437 and
// 540 us, so 285, 428 and 526 (at 1024 rows 90 and 91); K 10240 the same either
// way; e4m3, 8192 x 32768 at 2700 rows 569 and 542, K 20480 the same. Where x is
// one or two tiles tall no two CUs (or only two) read the same of W, and
// columns start at 32 places: 151936 x 4096 at 256 rows 320 and 296, 65536 x 4096
// 151 and 122, 24576 x 4096 with silu at 300 98 and 88. (The same at 1024 rows
// 177 and 174, 4096 x 12288 at 4099 300 and 317.)
//
// e4m3: the same bytes in the same places, so a stage is 128 of K. MFMA
// 32x32x64 (four times a bf16 product's time, eight times its work), a lane
// has two chunks of a row; scales are applied in the epilogue. 8192 rows, us
// (PFLOP/s), the library's GEMM and this: 4096 x 12288 281 (2.93) and 265
// (3.12), 24576 x 4096 633 (2.60) and 574 (2.87); where the library's tiles
// leave the chip idle, 4099 rows, 4096 x 12288: 270 (1.53) and 151 (2.73).
//
// SILU_MUL: the first half of a tile's W rows are gate rows and the second
// the up rows that go with them; a wave holds both. GELU: of the fp32 sums; a
// pass over 7100 rows of 6144 that took 33 us beside a product of 150.

#include <type_traits>

#include "tile_engine.h"

namespace fi {

namespace {

constexpr int kTile = 256, kChip = 256;
constexpr int kRowB = 128;                // of a row in a stage
constexpr int kHalfB = kTile * kRowB;     // one operand's part of a stage
constexpr int kStageB = 2 * kHalfB;
constexpr int kPiece = kTile * kTile / 4;  // float4

// How [mt, nt] tiles are dealt: `whole` to every workgroup, then `rest` in
// `cut` pieces each, one per workgroup.
struct TilePlan {
  int mt, nt, whole, rest, cut;
  double us;
};

// Tile `at` of the order in which they are dealt: runs of four row tiles by
// all column tiles. The 32 that an XCD works on share 4 + 8 panels in its L2.
// (8 or 16 row tiles a run, or rounds of 16 x 16 tiles over all XCDs, lose 1
// to 5 %.)
struct Tile {
  int m, n;
};
FI_DEV Tile tile_at(const TilePlan& p, int at) {
  constexpr int kRun = 4;
  const int run = at / (kRun * p.nt);
  at -= run * kRun * p.nt;
  const int rows = min(kRun, p.mt - run * kRun);
  const int n = at / rows;
  return Tile{run * kRun + at - n * rows, n};
}

// What the operands' type decides. A fragment is kRows rows of either operand
// by half a stage of K; a lane has kChunks chunks of a row of it and, of a
// product, results in one column, four neighbouring rows of x at a time.
template <bool FP8>
struct Kind {
  using Elem = u16;
  using Frag = short8;
  using Acc = floatx4;
  static constexpr int kRows = 16, kChunks = 1;
  FI_DEV static void put(Frag& f, int, const short8& v) { f = v; }
};
template <>
struct Kind<true> {
  using Elem = unsigned char;
  using Frag = intx8;
  using Acc = floatx16;
  static constexpr int kRows = 32, kChunks = 2;
  FI_DEV static void put(Frag& f, int chunk, const short8& v) {
    const intx4 q = __builtin_bit_cast(intx4, v);
#pragma unroll
    for (int i = 0; i < 4; ++i) f[chunk * 4 + i] = q[i];
  }
};

// what becomes of the products: nothing, + bias, silu(gate) * up, gelu
enum { PLAIN, BIAS, SILU, GELU };

// C neighbouring outputs of a row of x, from its sums and (SILU) the up values
// that go with them. FP8: times xs, the row's scale, and ws, those of W's rows.
template <int MODE, bool FP8, int C>
FI_DEV void store_row(u16* to, const u16* bias, const float (&sum)[C],
                      const float (&up)[C], float xs, const float* ws) {
  struct alignas(2 * C) Outputs {
    u16 h[C];
  } o, add;
  if (MODE == BIAS) add = *reinterpret_cast<const Outputs*>(bias);
#pragma unroll
  for (int c = 0; c < C; ++c) {
    float y = sum[c];
    if (FP8) y *= xs * ws[c];
    if (MODE == SILU) y = silu(y) * up[c];
    if (MODE == GELU) y = gelu(y);
    if (MODE == BIAS) y += bf16_to_f32(add.h[c]);
    o.h[c] = f32_to_bf16(y);
  }
  store_global(to, o);
}

// Where a lane's results lie. Slot i of fragment f holds column i * kLaneCols +
// f % kLaneCols of the wave's, so a lane has the kLaneCols neighbouring columns
// of its kLaneRows rows of a fragment of x.
template <bool FP8, bool SILU_MUL>
struct Lanes {
  static constexpr int kRows = Kind<FP8>::kRows, kFrags = 128 / kRows;
  static constexpr int kLaneRows = kRows * kRows / kWaveSize;
  static constexpr int kLaneCols = SILU_MUL ? kFrags / 2 : kFrags;
  static_assert(!FP8 || !SILU_MUL);
  // row of a fragment that a lane's result r of it belongs to
  FI_DEV static int row(int lane, int r) {
    return (r >> 2) * 8 + lane / kRows * 4 + (r & 3);
  }
};

template <int MODE, bool FP8>
__global__ __launch_bounds__(256, 1)
void tile_gemm_kernel(u16* __restrict__ out, floatx4* __restrict__ pieces,
                      const typename Kind<FP8>::Elem* __restrict__ x,
                      const typename Kind<FP8>::Elem* __restrict__ w,
                      const u16* __restrict__ bias,
                      const float* __restrict__ x_scales,
                      const float* __restrict__ w_scales, const int M,
                      const int N, const int K, const int64_t x_stride,
                      const int64_t out_stride, const TilePlan plan,
                      const int turn) {
  using T = Kind<FP8>;
  constexpr bool SILU_MUL = MODE == SILU;
  constexpr int kElemB = sizeof(typename T::Elem);
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * kStageB];
  const u32 lds0 = static_cast<u32>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) unsigned char*)smem));
  const int lane = threadIdx.x % kWaveSize;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  const int wm = wave >> 1, wn = wave & 1;
  const int SK = K * kElemB / kRowB;
  // out columns of a tile, and all of them
  constexpr int kCols = SILU_MUL ? kTile / 2 : kTile;
  const int cols = SILU_MUL ? N / 2 : N;

  // neighbours on one XCD (every eighth workgroup) take neighbouring tiles
  const int place = (blockIdx.x & 7) * (kChip / 8) + (blockIdx.x >> 3);
  const int units = plan.whole + (place < plan.rest * plan.cut ? 1 : 0);
  if (units == 0) return;
  struct Unit {
    int m, n, lo, count, rot;   // tile, first stage and stages, where to begin
  };
  auto unit = [&](int i) {
    Unit t;
    int at;
    if (i < plan.whole) {
      at = ((blockIdx.x & 7) * plan.whole + i) * (kChip / 8) +
           (blockIdx.x >> 3);
      t.lo = 0;
      t.count = SK;
    } else {
      const int p = place / plan.rest;
      at = plan.whole * kChip + place - p * plan.rest;
      t.lo = p * SK / plan.cut;
      t.count = (p + 1) * SK / plan.cut - t.lo;
    }
    const Tile tile = tile_at(plan, at);
    t.m = tile.m;
    t.n = tile.n;
    t.rot = t.n % turn * t.count / turn;
    return t;
  };

  // ---- requests: DMA j of a wave brings eight rows, group wave + 4 j of the
  // tile; lane l chunk (l % 8) ^ key of one of them. The row is in the vector
  // offset and the place along K in the scalar one, which so never reaches
  // past a descriptor's end: rows past it are cut off by the vector offset
  // alone (the bound that it is held against is the size less the scalar
  // offset, and need not be right where that is negative).
  const u32 ab = static_cast<u32>(x_stride) * kElemB, wb = K * kElemB;
  u32 a_voff[8], b_voff[4];
  using L = Lanes<FP8, SILU_MUL>;
  // the W row of the half tile that lies in its slot s
  auto column_at = [](int s) {
    constexpr int kWave = L::kRows * L::kLaneCols;
    return s / kWave * kWave + s % L::kRows * L::kLaneCols +
           s % kWave / L::kRows;
  };
#pragma unroll
  for (int j = 0; j < 8; ++j)
    a_voff[j] = ((wave + 4 * j) * 8 + (lane >> 3)) * ab +
                (((lane & 7) ^ ((lane >> 4) | ((wave & 1) << 2))) << 4);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    b_voff[j] = column_at((wave + 4 * j) * 8 + (lane >> 3)) * wb +
                (((lane & 7) ^ ((lane >> 4) | ((wave & 1) << 2))) << 4);
  u32x4 da, db, dc;             // x rows, first and second half of W's rows
  constexpr int kPast = 1 << 30;
  int ru = 0, rs = 0, rend = 0, rlo = 0, left = 0;
  auto aim = [&] {
    if (ru == units) {          // past the end nothing is read
      da[2] = db[2] = dc[2] = 0;
      left = kPast;
      return;
    }
    const Unit t = unit(ru++);
    const int rows = min(kTile, M - t.m * kTile);
    da = uniform_descriptor(x + static_cast<int64_t>(t.m) * kTile * x_stride,
                       (rows - 1) * ab + wb);
    const int n0 = t.n * kCols;
    const int n1 = SILU_MUL ? cols + n0 : n0 + kTile / 2;
    const int end1 = SILU_MUL ? N : cols;
    db = uniform_descriptor(w + static_cast<int64_t>(n0) * K,
                       min(kTile / 2, cols - n0) * wb);
    if (n1 < end1)
      dc = uniform_descriptor(w + static_cast<int64_t>(n1) * K,
                              min(kTile / 2, end1 - n1) * wb);
    else
      dc = db;                  // nobody uses these columns
    rlo = t.lo;
    rend = t.lo + t.count;
    rs = t.lo + t.rot;
    left = t.count;
  };
  aim();
  u32 rdst = lds0 + wave * 1024;
  u32 soff = 0;
  auto seek = [&] { soff = left > kPast / 2 ? 0 : rs * kRowB; };
  seek();
  auto m0_of = [&](int j) {
    set_m0(rdst + j * 4096);
    if (FP8) asm volatile("s_nop 0");   // no product lies in between
  };
  auto load_of = [&](int j) {
    if (j < 8) load_lds(da, a_voff[j], soff);
    else if (j < 12) load_lds(db, b_voff[j - 8], soff);
    else load_lds(dc, b_voff[j - 12], soff);
  };
  auto requested = [&] {
    rdst ^= kStageB;
    if (++rs == rend) rs = rlo;
    if (--left == 0) aim();
    seek();
  };

  // ---- fragment reads: row lane % kRows, from chunk 4 half + q on; the i-th
  // of eight
  constexpr int kRows = T::kRows, kChunks = T::kChunks, kFrags = 8 / kChunks;
  const int ir = lane % kRows, q = lane / kRows * kChunks;
  const u32 a_rd = (wm * 128 + ir) * kRowB + ((q ^ (ir >> 1 & 7)) << 4);
  const u32 b_rd = kHalfB + (wn * (SILU_MUL ? 64 : 128) + ir) * kRowB +
                   ((q ^ (ir >> 1 & 7)) << 4);
  using Frag = typename T::Frag;
  auto rda = [&](Frag (&to)[kFrags], int buf, int half, int i) {
    const int mi = i / kChunks, c = i % kChunks;
    T::put(to[mi], c, *reinterpret_cast<const short8*>(
        smem + buf * kStageB + (a_rd ^ (half * 64 + c * 16)) +
        mi * kRows * kRowB));
  };
  auto rdb = [&](Frag (&to)[kFrags], int buf, int half, int i) {
    const int f = i / kChunks, c = i % kChunks;
    T::put(to[f], c, *reinterpret_cast<const short8*>(
        smem + buf * kStageB + (b_rd ^ (half * 64 + c * 16)) +
        (SILU_MUL ? (f >> 2) * 128 + (f & 3) * 16 : f * kRows) * kRowB));
  };
  Frag a0[kFrags], b0[kFrags], a1[kFrags], b1[kFrags];
  typename T::Acc acc[kFrags][kFrags];
  // place i of 64 in a half stage: a product, in e4m3 every fourth time (it
  // takes as long as four)
  auto product = [&](int i, const Frag (&b)[kFrags], const Frag (&a)[kFrags],
                     bool first) {
    constexpr int kEach = 64 / (kFrags * kFrags);
    const int mi = i / kEach / kFrags, f = i / kEach % kFrags;
    if (i % kEach == 0) {
      if (first) mfma_first(acc[mi][f], a[mi], b[f]);
      else mfma(acc[mi][f], a[mi], b[f]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  for (int k = 0; k < 2; ++k) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      m0_of(j);
      asm volatile("s_nop 4");
      load_of(j);
    }
    requested();
  }
  asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
  sync_waves();
#pragma unroll
  for (int f = 0; f < 8; ++f) {
    rdb(b0, 0, 0, f);
    rda(a0, 0, 0, f);
  }
  int buf = 0;
  constexpr int kFree = 40, kEarly = 6;  // MFMAs up to the first barrier, DMAs
                                         // between the two
  // of a whole tile, at least (a row's outputs are one instruction or more, and a
  // wait that counts too few is only longer), as far as the counter goes
  constexpr int kStores = FP8 ? 63 - kEarly : 32;
  // `behind`: that many follow the DMAs that are waited for
  auto stage = [&](auto first, bool behind) {
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      product(i, b0, a0, first);
      if (i < 16 && i % 2 == 0) rdb(b1, buf, 1, i / 2);
      if (i >= 16 && i < 32 && i % 2 == 0) rda(a1, buf, 1, i / 2 - 8);
      if (i == kFree) {
        // all waves hold the stage in registers
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        sync_waves();
      }
      const int j = i - kFree - 1;
      if (j >= 0 && j < 2 * kEarly) {
        if (j % 2 == 0) m0_of(j / 2);
        else load_of(j / 2);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // the next stage has landed: this wave's DMAs but the youngest, and
    // after the barrier all waves'
    if (first && behind)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kEarly + kStores) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kEarly) : "memory");
    sync_waves();
    buf ^= 1;
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      product(i, b1, a1, false);
      // (e4m3: the last a few of its longer products before they are used)
      constexpr int kGap = FP8 ? 3 : 4;
      if (i % kGap == 0 && i < 8 * kGap) rdb(b0, buf, 0, i / kGap);
      if (i % kGap == 0 && i >= 8 * kGap && i < 16 * kGap)
        rda(a0, buf, 0, i / kGap - 8);
      if (i / 4 < 16 - kEarly) {
        if (i % 4 == 1) m0_of(kEarly + i / 4);
        if (i % 4 == 2) load_of(kEarly + i / 4);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    requested();
  };

  bool behind = false;
  for (int u = 0; u < units; ++u) {
    const Unit t = unit(u);
    stage(std::true_type{}, behind);
    for (int s = 1; s < t.count; ++s) stage(std::false_type{}, false);
    settle();
    behind = false;
    // (from a fresh copy of the lane, or the addresses would be kept in
    // registers that the loop needs)
    int l = lane;
    asm volatile("" : "+v"(l));
    const int row0 = t.m * kTile + wm * 128;
    if (t.count == SK) {
      constexpr int kLaneCols = L::kLaneCols;
      const int row1 = row0 + L::row(l, 0);
      const int col1 = t.n * kCols + wn * (kCols / 2) + l % kRows * kLaneCols;
      // scales, all of them before the first store and waited for on every
      // path: a load behind a store waits for it too, and one that may still
      // be under way at the next stage would make that wait for all DMAs
      floatx4 xs[16] = {}, ws = {};
      if (FP8) {
        if (row0 + 128 <= M) {
#pragma unroll
          for (int i = 0; i < 16; ++i)
            __builtin_memcpy(&xs[i], x_scales + row1 + i * 8, 16);
        } else {
#pragma unroll
          for (int i = 0; i < 16; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              xs[i][r] = x_scales[min(row1 + i * 8 + r, M - 1)];
        }
        ws = *reinterpret_cast<const floatx4*>(w_scales + min(col1, cols - 4));
#pragma unroll
        for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(xs[i]));
        asm volatile("" : "+v"(ws));
      }
      auto store = [&](bool inside) {
        if (!inside && col1 >= cols) return;
        const u16* add = MODE == BIAS ? bias + col1 : nullptr;
        constexpr int kGroups = L::kLaneRows / 4, kGap = kRows / kGroups;
        u16* to = out + row1 * out_stride + col1;
        int row = row1;
#pragma unroll
        for (int g = 0; g < kFrags * kGroups; ++g) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const auto& of = acc[g / kGroups];
            const int at = g % kGroups * 4 + r;
            if (inside || row < M) {
              float sum[kLaneCols], up[kLaneCols];
#pragma unroll
              for (int c = 0; c < kLaneCols; ++c) {
                sum[c] = acc_of(of[c][at]);
                up[c] = SILU_MUL ? acc_of(of[c + kFrags - kLaneCols][at]) : 0.f;
              }
              store_row<MODE, FP8, kLaneCols>(
                  to, add, sum, up, xs[FP8 ? g : 0][r],
                  reinterpret_cast<const float*>(&ws));
            }
            // (a step at a time, or all rows' places would be kept)
            const int step = r < 3 ? 1 : kGap - 3;
            to += step * out_stride;
            row += step;
            asm volatile("" : "+v"(to), "+v"(row));
          }
        }
      };
      behind = t.m * kTile + kTile <= M && t.n * kCols + kCols <= cols;
      if (behind)
        store(true);
      else
        store(false);
    } else {
      // four columns (of a lane's) of a row at a time
      floatx4* p = pieces + static_cast<int64_t>(place) * kPiece +
                   wave * 64 * kWaveSize + l;
#pragma unroll
      for (int mi = 0; mi < kFrags; ++mi) {
        if (row0 + mi * kRows < M) {
#pragma unroll
          for (int r = 0; r < L::kLaneRows; ++r)
#pragma unroll
            for (int f = 0; f < kFrags; f += 4)
              p[(r * kFrags + f) / 4 * kWaveSize] =
                  floatx4{acc_of(acc[mi][f][r]), acc_of(acc[mi][f + 1][r]),
                          acc_of(acc[mi][f + 2][r]),
                          acc_of(acc[mi][f + 3][r])};
        }
        p += L::kLaneRows * kFrags / 4 * kWaveSize;
      }
    }
  }
  // no DMA may land in LDS that is no longer this workgroup's
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Sums the pieces of the cut tiles: blockIdx.y is the tile, a thread takes a
// lane's columns of one row, in kOps quads.
//
// Which parts of a piece a workgroup reads, and so which XCD, decides how fast the
// next launch writes its pieces: with 32 workgroups of 256 threads a tile the
// products in front of a join take 2 to 4 us longer than with 16 of 512 (joined gate
// and up, M x K x N, us: 257 x 1024 x 4096 26.4 and 23.4, 511 x 1408 x 2048 30.4 and
// 27.2, 257 x 2048 x 2816 29.2 and 25.5; plain 26.6 and 23.4, 30.7 and 27.8, 29.2 and
// 25.7). e4m3: 64 of 256, 257 x 2048 x 4096 23.8 and 26.6, 511 x 4096 x 2560 31.7 and
// 34.7.
template <bool FP8>
constexpr int kJoinThreads = FP8 ? 256 : 512;

template <int MODE, bool FP8>
__global__ __launch_bounds__(kJoinThreads<FP8>)
void tile_gemm_join_kernel(u16* __restrict__ out,
                           const floatx4* __restrict__ pieces,
                           const u16* __restrict__ bias,
                           const float* __restrict__ x_scales,
                           const float* __restrict__ w_scales, const int M,
                           const int N, const int64_t out_stride,
                           const TilePlan plan) {
  constexpr bool SILU_MUL = MODE == SILU;
  using L = Lanes<FP8, SILU_MUL>;
  constexpr int kCols = SILU_MUL ? kTile / 2 : kTile, kRows = L::kRows;
  const int cols = SILU_MUL ? N / 2 : N;
  constexpr int kOps = L::kFrags / 4, kLaneCols = L::kLaneCols;
  const int i = blockIdx.x * kJoinThreads<FP8> + threadIdx.x;
  const int lane = i % kWaveSize, r = i / kWaveSize % L::kLaneRows;
  const int mi = i / kWaveSize / L::kLaneRows % L::kFrags;
  const int wave = i / kWaveSize / L::kLaneRows / L::kFrags;
  const Tile tile = tile_at(plan, plan.whole * kChip + blockIdx.y);
  const int row = tile.m * kTile + (wave >> 1) * 128 + mi * kRows +
                  L::row(lane, r);
  const int col = tile.n * kCols + (wave & 1) * (kCols / 2) +
                  lane % kRows * kLaneCols;
  if (row >= M || col >= cols) return;
  floatx4 s[kOps];
  const floatx4* p = pieces + static_cast<int64_t>(blockIdx.y) * kPiece +
                     i / kWaveSize * kOps * kWaveSize + lane;
  const int64_t next = static_cast<int64_t>(plan.rest) * kPiece;
  for (int c = 0; c < plan.cut; c += 4) {
    floatx4 v[4][kOps];
#pragma unroll
    for (int k = 0; k < 4; ++k)   // pieces past the last repeat it
#pragma unroll
      for (int o = 0; o < kOps; ++o)
        v[k][o] = p[min(c + k, plan.cut - 1) * next + o * kWaveSize];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (c + k < plan.cut)
#pragma unroll
        for (int o = 0; o < kOps; ++o) s[o] = c + k ? s[o] + v[k][o] : v[k][o];
  }
  float sum[kLaneCols], up[kLaneCols];
#pragma unroll
  for (int c = 0; c < kLaneCols; ++c) {
    sum[c] = s[c / 4][c % 4];
    up[c] = SILU_MUL ? s[kOps - 1][c % 4] : 0.f;
  }
  store_row<MODE, FP8, kLaneCols>(out + row * out_stride + col,
                                  MODE == BIAS ? bias + col : nullptr, sum, up,
                                  FP8 ? x_scales[row] : 0.f, w_scales + col);
}

// A stage takes 1.42 us (e4m3 too); a piece costs 0.06 us of the way through
// memory and all of them 4 us for the second kernel. (504 sizes of 512 to 8192 rows and
// 14 N and K: 0.98 of what is measured on average, 0.7 to 1.13.)
// KB: bytes of a row
TilePlan tile_plan(int M, int N, int KB) {
  constexpr double kStage = 1.42;
  TilePlan p;
  p.mt = ceil_div(M, kTile);
  p.nt = ceil_div(N, kTile);
  const int64_t tiles = static_cast<int64_t>(p.mt) * p.nt;
  p.whole = static_cast<int>(tiles / kChip);
  p.rest = static_cast<int>(tiles % kChip);
  const int SK = KB / kRowB;
  p.cut = 1;
  double least = p.rest ? SK * kStage : 0;
  // two stages a piece at least: that many are requested ahead
  for (int c = 2; p.rest && c * p.rest <= kChip && 2 * c <= SK && c <= 16;
       ++c) {
    const double us = ceil_div(SK, c) * kStage + 4 + c * p.rest * 0.06;
    if (us < least) {
      least = us;
      p.cut = c;
    }
  }
  p.us = 5 + p.whole * SK * kStage + least;
  return p;
}

template <int MODE, bool FP8>
void launch(u16* out, float* pieces, const typename Kind<FP8>::Elem* x,
            const typename Kind<FP8>::Elem* w, const u16* bias,
            const float* x_scales, const float* w_scales, int M, int N, int K,
            int64_t x_stride, int64_t out_stride, hipStream_t stream) {
  const int KB = K * static_cast<int>(sizeof(typename Kind<FP8>::Elem));
  const TilePlan p = tile_plan(M, N, KB);
  auto* pc = reinterpret_cast<floatx4*>(pieces);
  // the places along K that column tiles start at
  const int turn = p.mt <= 2 ? 32 : KB > 16384 && KB % 4096 == 0 ? 2 : 1;
  hipLaunchKernelGGL((tile_gemm_kernel<MODE, FP8>), dim3(kChip), dim3(256), 0,
                     stream, out, pc, x, w, bias, x_scales, w_scales, M, N, K,
                     x_stride, out_stride, p, turn);
  if (p.cut > 1)
    hipLaunchKernelGGL((tile_gemm_join_kernel<MODE, FP8>),
                       dim3(FP8 ? 64 : 16, p.rest), dim3(kJoinThreads<FP8>), 0,
                       stream, out, pc, bias, x_scales, w_scales, M, N,
                       out_stride, p);
}

}  // namespace

// by its own estimate, in us
double tile_gemm_us(int M, int N, int KB) { return tile_plan(M, N, KB).us; }

// floats of scratch that launch_tile_gemm needs
int64_t tile_gemm_floats(int M, int N, int KB) {
  const TilePlan p = tile_plan(M, N, KB);
  return p.cut > 1 ? static_cast<int64_t>(p.rest) * p.cut * kPiece * 4 : 0;
}

// K a multiple of 64 and 128 at least, N of 16 (32 with silu_mul)
void launch_tile_gemm(u16* out, float* pieces, const u16* x, const u16* w,
                      const u16* bias, int M, int N, int K, int64_t x_stride,
                      int64_t out_stride, bool silu_mul, bool gelu,
                      hipStream_t stream) {
  if (gelu)
    launch<GELU, false>(out, pieces, x, w, bias, nullptr, nullptr, M, N, K,
                        x_stride, out_stride, stream);
  else if (silu_mul)
    launch<SILU, false>(out, pieces, x, w, bias, nullptr, nullptr, M, N, K,
                        x_stride, out_stride, stream);
  else if (bias)
    launch<BIAS, false>(out, pieces, x, w, bias, nullptr, nullptr, M, N, K,
                        x_stride, out_stride, stream);
  else
    launch<PLAIN, false>(out, pieces, x, w, bias, nullptr, nullptr, M, N, K,
                         x_stride, out_stride, stream);
}

// e4m3: K a multiple of 128 and 256 at least
void launch_tile_gemm_fp8(u16* out, float* pieces, const unsigned char* x,
                          const float* x_scales, const unsigned char* w,
                          const float* w_scales, int M, int N, int K,
                          int64_t x_stride, int64_t out_stride,
                          hipStream_t stream) {
  launch<PLAIN, true>(out, pieces, x, w, nullptr, x_scales, w_scales, M, N, K,
                      x_stride, out_stride, stream);
}

}  // namespace fi
