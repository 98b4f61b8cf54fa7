// y = x W^T for more than 256 rows of x (prompts): bf16 operands, fp32
// accumulation, W [N, K] row-major. Bound by the matrix cores.
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
// tiles, so a tile's results are written while the next one's stages arrive.
//
// Rows lie in LDS as eight chunks of 16 bytes, chunk c of row r at c ^ key(r):
// the 16 lanes that LDS serves together then touch all its banks (no
// conflicts counted), and a DMA still reads whole lines of eight rows.
// MFMA 16x16x32 with A = W, B = x; the W rows of a fragment pair are dealt so
// that a lane ends with eight neighbouring outputs of one row of x.
//
// What whole rounds of 256 tiles leave over is cut along K into equal pieces
// (tile_plan), which a second kernel sums in a fixed order.
//
// Where both operands are larger than the 256 MB memory-side cache and rows
// are a multiple of 4 KB and longer than 16 KB, reads of the same K by all
// CUs meet on few memory channels (8192 x 4096 x 12288: 1.28 PFLOP/s, with K
// of 12160 or 12416 1.49); there every other column tile starts half way
// along K (1.41).
//
// SILU_MUL: the first half of a tile's W rows are gate rows and the second
// the up rows that go with them; a wave holds both.

#include "common.h"

namespace fi {

namespace {

typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) float floatx4;

constexpr int kTile = 256, kChip = 256, kKS = 64;
constexpr int kHalfB = kTile * kKS * 2;   // one operand's part of a stage
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

FI_DEV void set_m0(u32 lds) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0" ::"s"(lds) : "memory");
#endif
}
// 16 bytes per lane to LDS at m0 + 16 lane; set_m0 lies at least one
// instruction ahead
FI_DEV void load_lds(u32x4 desc, u32 voff, u32 soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds"
               :
               : "v"(voff), "s"(desc), "s"(soff)
               : "memory");
#endif
}
// in scalar registers, as the loads want it
FI_DEV u32x4 uniform_descriptor(const void* p, u32 bytes) {
  u32x4 d = descriptor_of(p, bytes);
#pragma unroll
  for (int i = 0; i < 4; ++i) d[i] = __builtin_amdgcn_readfirstlane(d[i]);
  return d;
}
// acc += w x^T. In asm, so that the accumulators have one place, the
// accumulation registers: from the builtin the compiler keeps some of them
// elsewhere and copies them in and out of every stage. What it does not see
// are the wait states between other writers or readers of an accumulator and
// the product; settle() is put there. (Products of a stage do not wait for
// each other: an accumulator comes round after 64.)
FI_DEV void mfma(floatx4& acc, const short8& w, const short8& x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
               : "+a"(acc)
               : "v"(w), "v"(x));
#endif
}
FI_DEV float acc_of(float a) {
  float v = a;
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
#endif
  return v;
}
FI_DEV floatx4 acc_of(const floatx4& a) {
  return floatx4{acc_of(a[0]), acc_of(a[1]), acc_of(a[2]), acc_of(a[3])};
}
FI_DEV void settle() {
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
FI_DEV void sync_waves() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// W row (of the tile) of fragment f's row 0 in wave column wn; row i of the
// fragment lies (i >> 2) * 8 + (i & 3) further on
template <bool SILU_MUL>
FI_DEV constexpr int w_row(int f) {
  return SILU_MUL ? (f >> 2) * 128 + (f >> 1 & 1) * 32 + (f & 1) * 4
                  : (f >> 1) * 32 + (f & 1) * 4;
}

// what becomes of the products: nothing, + bias, silu(gate) * up
enum { PLAIN, BIAS, SILU };

// eight outputs of a row of x: fragments a, b; SILU: of gate values, the up
// values that go with them in u, v
template <int MODE>
FI_DEV void store8(u16* to, const u16* bias, const floatx4& a,
                   const floatx4& b, const floatx4& u, const floatx4& v) {
  bf16x8 o, add;
  if (MODE == BIAS) add = *reinterpret_cast<const bf16x8*>(bias);
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    float y = r < 4 ? a[r] : b[r - 4];
    if (MODE == SILU)
      y = y / (1.f + __expf(-y)) * (r < 4 ? u[r] : v[r - 4]);
    if (MODE == BIAS) y += bf16_to_f32(add.h[r]);
    o.h[r] = f32_to_bf16(y);
  }
  *reinterpret_cast<bf16x8*>(to) = o;
}

template <int MODE>
__global__ __launch_bounds__(256, 1)
void tile_gemm_kernel(u16* __restrict__ out, floatx4* __restrict__ pieces,
                      const u16* __restrict__ x, const u16* __restrict__ w,
                      const u16* __restrict__ bias, const int M, const int N,
                      const int K, const int64_t x_stride,
                      const int64_t out_stride, const TilePlan plan,
                      const int turn) {
  constexpr bool SILU_MUL = MODE == SILU;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * kStageB];
  const u32 lds0 = static_cast<u32>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) unsigned char*)smem));
  const int lane = threadIdx.x % kWaveSize;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  const int wm = wave >> 1, wn = wave & 1;
  const int SK = K / kKS;
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
    t.rot = (t.n & 1) * turn * t.count / 2;
    return t;
  };

  // ---- requests: DMA j of a wave brings eight rows, group wave + 4 j of the
  // tile; lane l chunk (l % 8) ^ key of one of them
  const u32 ab = static_cast<u32>(x_stride) * 2, wb = K * 2;
  const u32 a_voff = (lane >> 3) * ab +
                     (((lane & 7) ^ ((lane >> 4) | ((wave & 1) << 2))) << 4);
  const u32 b_voff = (lane >> 3) * wb +
                     (((lane & 7) ^ (((lane >> 4) & 1) | (wave << 1))) << 4);
  u32x4 da, db, dc;             // x rows, first and second half of W's rows
  int ru = 0, rs = 0, rend = 0, rlo = 0, left = 0;
  auto aim = [&] {
    if (ru == units) {          // past the end nothing is read
      da[2] = db[2] = dc[2] = 0;
      left = 1 << 30;
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
    dc = uniform_descriptor(w + static_cast<int64_t>(min(n1, end1)) * K,
                       max(0, min(kTile / 2, end1 - n1)) * wb);
    rlo = t.lo;
    rend = t.lo + t.count;
    rs = t.lo + t.rot;
    left = t.count;
  };
  aim();
  const u32 a_step = 32 * ab, b_step = 32 * wb;   // four groups of eight rows
  u32 rdst = lds0 + wave * 1024;
  u32 a_soff = 0, b_soff = 0;
  auto seek = [&] {
    a_soff = wave * 8 * ab + rs * 128;
    b_soff = wave * 8 * wb + rs * 128;
  };
  seek();
  auto m0_of = [&](int j) { set_m0(rdst + j * 4096); };
  auto load_of = [&](int j) {
    if (j < 8) load_lds(da, a_voff, a_soff + j * a_step);
    else if (j < 12) load_lds(db, b_voff, b_soff + (j - 8) * b_step);
    else load_lds(dc, b_voff, b_soff + (j - 12) * b_step);
  };
  auto requested = [&] {
    rdst ^= kStageB;
    if (++rs == rend) rs = rlo;
    if (--left == 0) aim();
    seek();
  };

  // ---- fragment reads: row lane & 15, chunk 4 half + (lane >> 4)
  const int i16 = lane & 15, q = lane >> 4;
  const u32 a_rd = (wm * 128 + i16) * 128 + ((q ^ (i16 >> 1)) << 4);
  const u32 b_rd = kHalfB +
      (wn * (SILU_MUL ? 64 : 128) + (i16 >> 2) * 8 + (i16 & 3)) * 128 +
      ((q ^ ((i16 >> 1 & 1) | (i16 >> 2) << 1)) << 4);
  auto rda = [&](int buf, int half, int mi) {
    return *reinterpret_cast<const short8*>(
        smem + buf * kStageB + (a_rd ^ (half * 64)) + mi * 2048);
  };
  auto rdb = [&](int buf, int half, int f) {
    return *reinterpret_cast<const short8*>(
        smem + buf * kStageB + (b_rd ^ (half * 64)) + w_row<SILU_MUL>(f) * 128);
  };
  short8 a0[8], b0[8], a1[8], b1[8];
  floatx4 acc[8][8];

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
    b0[f] = rdb(0, 0, f);
    a0[f] = rda(0, 0, f);
  }
  int buf = 0;
  constexpr int kFree = 40, kEarly = 6;  // MFMAs up to the first barrier, DMAs
                                         // between the two
  auto stage = [&] {
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      const int mi = i >> 3, f = i & 7;
      mfma(acc[mi][f], b0[f], a0[mi]);
      __builtin_amdgcn_sched_barrier(0);
      if (i < 16 && i % 2 == 0) b1[i / 2] = rdb(buf, 1, i / 2);
      if (i >= 16 && i < 32 && i % 2 == 0) a1[i / 2 - 8] = rda(buf, 1, i / 2 - 8);
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
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kEarly) : "memory");
    sync_waves();
    buf ^= 1;
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      const int mi = i >> 3, f = i & 7;
      mfma(acc[mi][f], b1[f], a1[mi]);
      __builtin_amdgcn_sched_barrier(0);
      if (i % 4 == 0 && i < 32) b0[i / 4] = rdb(buf, 0, i / 4);
      if (i % 4 == 0 && i >= 32) a0[i / 4 - 8] = rda(buf, 0, i / 4 - 8);
      if (i / 4 < 16 - kEarly) {
        if (i % 4 == 1) m0_of(kEarly + i / 4);
        if (i % 4 == 2) load_of(kEarly + i / 4);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    requested();
  };

  for (int u = 0; u < units; ++u) {
#pragma unroll
    for (int mi = 0; mi < 8; ++mi)
#pragma unroll
      for (int f = 0; f < 8; ++f) acc[mi][f] = {0.f, 0.f, 0.f, 0.f};
    settle();
    const Unit t = unit(u);
    for (int s = 0; s < t.count; ++s) stage();
    settle();
    // (from a fresh copy of the lane, or the addresses would be kept in
    // registers that the loop needs)
    int l = lane;
    asm volatile("" : "+v"(l));
    const int row0 = t.m * kTile + wm * 128;
    if (t.count == SK) {
      const int row1 = row0 + (l & 15);
      const int col1 = t.n * kCols + wn * (kCols / 2) + (l >> 4) * 8;
      u16* to = out + row1 * out_stride + col1;
      const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
      auto store = [&](bool inside) {
#pragma unroll
        for (int mi = 0; mi < 8; ++mi) {
          if (inside || row1 + mi * 16 < M) {
#pragma unroll
            for (int f = 0; f < (SILU_MUL ? 4 : 8); f += 2)
              if (inside || col1 + f * 16 < cols)
                store8<MODE>(to + f * 16,
                             MODE == BIAS ? bias + col1 + f * 16 : nullptr,
                             acc_of(acc[mi][f]), acc_of(acc[mi][f + 1]),
                             SILU_MUL ? acc_of(acc[mi][(f + 4) % 8]) : zero,
                             SILU_MUL ? acc_of(acc[mi][(f + 5) % 8]) : zero);
          }
          to += 16 * out_stride;
        }
      };
      if (t.m * kTile + kTile <= M && t.n * kCols + kCols <= cols)
        store(true);
      else
        store(false);
    } else {
      floatx4* p = pieces + static_cast<int64_t>(place) * kPiece +
                   wave * 64 * kWaveSize + l;
#pragma unroll
      for (int mi = 0; mi < 8; ++mi) {
        if (row0 + mi * 16 < M) {
#pragma unroll
          for (int f = 0; f < 8; ++f) p[f * kWaveSize] = acc_of(acc[mi][f]);
        }
        p += 8 * kWaveSize;
      }
    }
  }
  // no DMA may land in LDS that is no longer this workgroup's
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Sums the pieces of the cut tiles: blockIdx.y is the tile, a thread takes
// eight outputs.
template <int MODE>
__global__ __launch_bounds__(256)
void tile_gemm_join_kernel(u16* __restrict__ out,
                           const floatx4* __restrict__ pieces,
                           const u16* __restrict__ bias, const int M,
                           const int N, const int64_t out_stride,
                           const TilePlan plan) {
  constexpr bool SILU_MUL = MODE == SILU;
  constexpr int kCols = SILU_MUL ? kTile / 2 : kTile;
  const int cols = SILU_MUL ? N / 2 : N;
  constexpr int kPairs = SILU_MUL ? 2 : 4;
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int lane = i % kWaveSize, f = i / kWaveSize % kPairs * 2;
  const int mi = i / kWaveSize / kPairs % 8, wave = i / kWaveSize / kPairs / 8;
  const Tile tile = tile_at(plan, plan.whole * kChip + blockIdx.y);
  const int m = tile.m, n = tile.n;
  const int row = m * kTile + (wave >> 1) * 128 + mi * 16 + (lane & 15);
  const int col = n * kCols + (wave & 1) * (kCols / 2) + f * 16 +
                  (lane >> 4) * 8;
  if (row >= M || col >= cols) return;
  constexpr int kOps = SILU_MUL ? 4 : 2;
  floatx4 s[4];
  const floatx4* p = pieces + static_cast<int64_t>(blockIdx.y) * kPiece +
                     ((wave * 8 + mi) * 8 + f) * kWaveSize + lane;
  const int64_t next = static_cast<int64_t>(plan.rest) * kPiece;
  for (int c = 0; c < plan.cut; c += 4) {
    floatx4 v[4][kOps];
#pragma unroll
    for (int k = 0; k < 4; ++k)   // pieces past the last repeat it
#pragma unroll
      for (int o = 0; o < kOps; ++o)
        v[k][o] = p[min(c + k, plan.cut - 1) * next +
                    ((o & 1) + (o >> 1) * 4) * kWaveSize];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (c + k < plan.cut)
#pragma unroll
        for (int o = 0; o < kOps; ++o) s[o] = c + k ? s[o] + v[k][o] : v[k][o];
  }
  store8<MODE>(out + row * out_stride + col,
               MODE == BIAS ? bias + col : nullptr, s[0], s[1],
               s[SILU_MUL ? 2 : 0], s[SILU_MUL ? 3 : 1]);
}

// A stage takes 1.42 us; a piece costs 0.06 us of the way through memory and
// all of them 4 us for the second kernel. (504 sizes of 512 to 8192 rows and
// 14 N and K: 0.98 of what is measured on average, 0.7 to 1.13.)
TilePlan tile_plan(int M, int N, int K) {
  constexpr double kStage = 1.42;
  TilePlan p;
  p.mt = ceil_div(M, kTile);
  p.nt = ceil_div(N, kTile);
  const int64_t tiles = static_cast<int64_t>(p.mt) * p.nt;
  p.whole = static_cast<int>(tiles / kChip);
  p.rest = static_cast<int>(tiles % kChip);
  const int SK = K / kKS;
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

}  // namespace

// by its own estimate, in us
double tile_gemm_us(int M, int N, int K) { return tile_plan(M, N, K).us; }

// floats of scratch that launch_tile_gemm needs
int64_t tile_gemm_floats(int M, int N, int K) {
  const TilePlan p = tile_plan(M, N, K);
  return p.cut > 1 ? static_cast<int64_t>(p.rest) * p.cut * kPiece * 4 : 0;
}

// K a multiple of 64 and 128 at least, N of 16 (32 with silu_mul)
void launch_tile_gemm(u16* out, float* pieces, const u16* x, const u16* w,
                      const u16* bias, int M, int N, int K, int64_t x_stride,
                      int64_t out_stride, bool silu_mul, hipStream_t stream) {
  const TilePlan p = tile_plan(M, N, K);
  auto* pc = reinterpret_cast<floatx4*>(pieces);
  const int turn = K > 8192 && K % 2048 == 0 ? 1 : 0;
  auto launch = [&](auto mode) {
    constexpr int MODE = decltype(mode)::value;
    hipLaunchKernelGGL((tile_gemm_kernel<MODE>), dim3(kChip), dim3(256), 0,
                       stream, out, pc, x, w, bias, M, N, K, x_stride,
                       out_stride, p, turn);
    if (p.cut > 1)
      hipLaunchKernelGGL((tile_gemm_join_kernel<MODE>),
                         dim3(MODE == SILU ? 16 : 32, p.rest), dim3(256), 0,
                         stream, out, pc, bias, M, N, out_stride, p);
  };
  if (silu_mul) launch(std::integral_constant<int, SILU>{});
  else if (bias) launch(std::integral_constant<int, BIAS>{});
  else launch(std::integral_constant<int, PLAIN>{});
}

}  // namespace fi
