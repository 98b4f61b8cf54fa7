// Grouped MFMA GEMM for long expert segments (128-row blocks, prompts) whose K
// is a multiple of 64. Bound by the matrix cores.
//
// 256 persistent workgroups, one per CU, take tiles of 128 rows by 512 columns
// of the expert's B (256 gate and the same 256 up columns where the epilogue
// joins them). Four waves side by side hold 128 x 128 results each, so a
// fragment read from LDS feeds eight MFMAs; the form with 128 x 256 tiles, two
// workgroups per CU and B in registers loads half as much again per product
// (48 bytes a cycle and CU, of 64 that the first-level cache delivers; here
// 40).
//
// Two neighbouring blocks of an expert take tiles of 256 rows by 256 columns
// instead (PAIRS), waves two by two: 64 KB a stage, not 80, and every fragment of B
// once for both. (All that differs is where a wave's requests go and what it reads;
// a wave's products are the same.) us, blocks apart and in pairs: down, 128 experts,
// top 8, 2048 x 768, 8100 rows 242 and 227, 4000 146 and 139; 64 experts, 2048 x
// 1408, top 6, 8192 rows 281 and 278; 8 experts, 4096 x 6144, top 2, 8192 rows 767
// and 743. Rows that are gathered gain where experts have few blocks
// (launch_moe_wide).
//
// A stage is 64 of K: 128 gathered rows of 128 bytes, and 64 of B's packed
// fragments (1 KB each), 80 KB in all; two of them are kept, all of a CU's
// LDS. As in the dense kernel of 256 x 256 tiles a stage is used in two halves:
// the second half's fragments are read while the first is multiplied, then
// the stage's place is free and the stage after the next is requested into
// it. Every MFMA is followed by at most one other step, in an order that is
// pinned; with PAIRS eight of the requests ask for the tile's shape first. (A body
// per shape does not fit the registers; requests that ask nothing, with the four
// that a square tile has no use for out of range: gate|up the same, down 225 and
// 239 us at 8100 rows.) The DMAs run on over the borders of tiles; the rows' ids
// come through the scalar cache, since a vector load would wait for all DMAs
// in front of it.
//
// LDS: 16-byte chunk c of row r sits at c ^ (r >> 1 & 7); B's fragments lie as
// they are packed, in the f-th columns c at c ^ f. MFMA operands are A, B; B is
// read so that lane i of 16 has column 8 i + f of a wave's in product f: eight
// neighbouring columns of a row (of each four rows; joined ones four), beside
// those of the next lane.
//
// Workgroups of one XCD take a contiguous run of tiles, eight row blocks by
// all column tiles at a time.
//
// Results leave in that order because a CU takes stores 64 bytes of neighbouring
// lanes at a time: 128 KB in 0.9 us so (8 bytes a lane 1.7), in 3.5 where a lane's
// 16 bytes are another row than the next one's (all CUs at once: 5.7 either way).
// 8100 rows, 128 experts, top 8, 2048 x 768: down 251 and 240 us, gate|up 414 and
// 416; 4000 rows 152 and 146.
//
// A stage takes 1.4 to 1.7 us; a tile's end 5 to 7, most of it until its results
// have left (the stages after the first wait for them). Tiles of 128 x 256, two to
// a CU, and these, us (TFLOP/s of the real rows, now): 8765 rows, 128 experts, top
// 8, 2048 x 768: gate|up 467 and 466 (946), down 308 and 254 (869); 8192 rows, 64
// experts, top 6, 2048 x 1408: 544 and 555 (1022), down 324 and 278 (1020); 8192
// rows, 8 experts, top 2, 4096 x 6144: gate|up 1385 and 1335 (1235).

#include <hip/hip_runtime.h>

#include <type_traits>

#include "tile_engine.h"

namespace fi {

namespace {

constexpr int kWideM = 128, kChip = 256;
constexpr int kRowsB = kWideM * 128, kWaveB = 16 * 1024;  // A's, a wave's B
constexpr int kWideStageB = kRowsB + 4 * kWaveB;
constexpr int kRunRows = 8;                               // row blocks of a run

// Which blocks are the second of a pair: lane l of `lo` and `hi` has those of
// blocks 64 l to 64 l + 63, of the first 4096; others go alone.
struct Pairs {
  u32 lo = 0, hi = 0;
  FI_DEV bool second(int m) const {
    const u32 l = __builtin_amdgcn_readlane(lo, m / 64 & 63);
    const u32 h = __builtin_amdgcn_readlane(hi, m / 64 & 63);
    return m < 64 * kWaveSize && ((m & 32 ? h : l) >> (m & 31) & 1);
  }
};

// From one pass over the ids. (Looked up for every place, back to the beginning
// of its expert's blocks, it costs more the more of them there are: 8 experts,
// 2048 x 1408, 32768 rows with half of them on one, down 381 and 337 us so.)
FI_DEV Pairs pairs_of(const int* __restrict__ expert_ids, int nv, int lane) {
  Pairs p;
  const int words = min((nv + 63) / 64, kWaveSize);
  int last = 0, last_id = -1;    // beginning, id of the word before
  constexpr int kAtOnce = 16;
  for (int w0 = 0; w0 < words; w0 += kAtOnce) {
    int id[kAtOnce];
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i)
      id[i] = expert_ids[min((w0 + i) * 64 + lane, nv - 1)];
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i) {
      if (w0 + i >= words) break;
      const int base = (w0 + i) * 64, m = base + lane;
      const int up = __shfl_up(id[i], 1, kWaveSize);
      const int before = lane == 0 ? last_id : up;
      const unsigned long long begins =
          __ballot(m < nv && (m == 0 || id[i] != before));
      const unsigned long long up_to = begins & (~0ull >> (63 - lane));
      const int of = m - (up_to ? base + 63 - __builtin_clzll(up_to) : last);
      const unsigned long long seconds = __ballot(m < nv && (of & 1));
      if (begins) last = base + 63 - __builtin_clzll(begins);
      last_id = __builtin_amdgcn_readlane(id[i], kWaveSize - 1);
      p.lo = lane == w0 + i ? static_cast<u32>(seconds) : p.lo;
      p.hi = lane == w0 + i ? static_cast<u32>(seconds >> 32) : p.hi;
    }
  }
  return p;
}

template <int MODE, bool PAIRS>
__global__ __launch_bounds__(256, 1) void moe_wide_kernel(
    u16* __restrict__ out,              // [PM, N]
    const u16* __restrict__ a,          // gathered x [T, K]; MODE 0 [PM, K]
    const u16* __restrict__ b,          // [E][K/32][NB/16][64][8]
    const int* __restrict__ sorted_ids, // [PM]
    const int* __restrict__ expert_ids, // [PM/128]
    const int* __restrict__ n_valid, const int K, const int N, const int NT,
    const u32 a_bytes, const float limit) {
  constexpr bool GATE_UP = MODE == 1 || MODE == 3;
  __shared__ __attribute__((aligned(1024))) unsigned char
      smem[2 * kWideStageB];
  const u32 lds0 = static_cast<u32>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) unsigned char*)smem));
  const int lane = threadIdx.x % kWaveSize;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  const int SK = K / 64;

  // tiles of this workgroup: `first`, and every 32nd after it
  const int nv = const_ints(n_valid)[0];
  const int total = nv * NT, per = (total + 7) / 8;
  const int run0 = (blockIdx.x & 7) * per;
  const int first = run0 + (blockIdx.x >> 3);
  const int end = min(run0 + per, total);
  if (first >= end) return;
  constexpr int kNext = kChip / 8;
  // A place in the order is a block's n-th wide tile. Where it and a neighbour
  // are a pair, the places of both are the pair's square tiles, of half as many
  // columns; there may be one fewer.
  struct Place {
    int m, n;      // first block, columns
    int square, none;
  };
  const ConstInts experts = const_ints(expert_ids);
  Pairs pairs;
  if (PAIRS) pairs = pairs_of(expert_ids, nv, lane);
  auto place_of = [&](int at) __attribute__((always_inline)) {
    const int m0 = at / (kRunRows * NT) * kRunRows;
    const int rows = min(kRunRows, nv - m0);
    const int in = at - m0 * NT;
    const int n = in / rows, m = m0 + in - n * rows;
    const bool second = PAIRS && pairs.second(m);
    if (!PAIRS || !(second || (m + 1 < nv && pairs.second(m + 1))))
      return Place{m, n, 0, 0};
    const int column = (second ? NT : 0) + n;
    return Place{m - second, column, 1, column * (GATE_UP ? 128 : 256) >= N};
  };

  // ---- requests. Of a wide tile DMAs 0 to 3 bring eight rows of A each and 4 to
  // 19 a fragment of this wave's B; of a square one 0 to 7 rows and 8 to 15 the
  // fragments of half a stage of two waves' B.
  const int NB16 = (GATE_UP ? 2 * N : N) / 16;
  const u32 b_step = static_cast<u32>(NB16) * 1024;   // 32 of K
  constexpr int kOwn = GATE_UP ? 4 : 8;   // fragments apart from up's
  const u32 up = N / 16 * 1024u;
  u32 a_voff[8] = {};
  u32x4 da, db;
  int rat = first, left = 0;
  u32 a_soff = 0, b_soff[2] = {}, b_col[kOwn];
  // where DMAs 0 to 3, 4 to 7, 8 to 11 and the others go in a stage, less 1 KB
  // each for those before
  u32 to_lds[4];
  int rsquare = 0;
  Place next{}, after{}, third{};   // tiles that are requested, not yet done
  int waiting = 0;
  auto put = [&](Place& at, const Place& t, int turn) {
    at.m = waiting == turn ? t.m : at.m;
    at.n = waiting == turn ? t.n : at.n;
    at.square = waiting == turn ? t.square : at.square;
  };
  // (out of line captures would be in memory, and no value uniform)
  auto aim = [&]() __attribute__((always_inline)) {
    Place t{0, 0, 0, 1};
    for (; rat < end && t.none; rat += kNext) t = place_of(rat);
    a_soff = 0;
    if (t.none) {               // past the end the last tile's beginning again
      b_soff[0] = rsquare ? (wave & 1) * b_step : 0;
      b_soff[1] = rsquare ? b_soff[0] : b_step;
      left = 1 << 30;
      return;
    }
    put(next, t, 0);
    put(after, t, 1);
    put(third, t, 2);
    ++waiting;
    rsquare = t.square;
    b_soff[0] = rsquare ? (wave & 1) * b_step : 0;
    b_soff[1] = rsquare ? b_soff[0] : b_step;
    to_lds[0] = wave * (rsquare ? 8192 : 4096);
    to_lds[1] = rsquare ? to_lds[0] : kRowsB + wave * kWaveB - 4096;
    to_lds[2] = rsquare ? 2 * kRowsB + wave * 8192 - 4096 : to_lds[1];
    to_lds[3] = rsquare ? to_lds[2] - 8192 : to_lds[1];
#pragma unroll
    for (int h = 0; h < (PAIRS ? 2 : 1); ++h) {
      // (a wide tile's a second time: around a branch they would be vector loads)
      const int row0 = wave * (rsquare ? 64 : 32) + (rsquare ? h * 32 : 0);
      int ids[32];
      if (MODE != 0) {
        const auto from =
            const_ints(sorted_ids + t.m * kWideM + row0);
#pragma unroll
        for (int i = 0; i < 32; ++i) ids[i] = from[i];
        // in scalar registers, or the choice by lane becomes a vector load
#pragma unroll
        for (int i = 0; i < 32; ++i) asm volatile("" : "+s"(ids[i]));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int row = row0 + i * 8 + (lane >> 3);
        if (MODE != 0) {
          row = ids[i * 8];
#pragma unroll
          for (int r = 1; r < 8; ++r)
            row = (lane >> 3) == r ? ids[i * 8 + r] : row;
        }
        a_voff[h * 4 + i] = static_cast<u32>(row) * (K * 2) +
                            (((lane & 7) ^ (lane >> 4 | (i & 1) << 2)) << 4);
      }
    }
    da = MODE != 0 ? uniform_descriptor(a, a_bytes)
                   : uniform_descriptor(
                         a + static_cast<int64_t>(t.m) * kWideM * K,
                         kWideM * K * (rsquare ? 4 : 2));
    db = uniform_descriptor(
        b + static_cast<int64_t>(experts[t.m]) * (K / 32) * NB16 * 512,
        K / 32 * b_step);
    const int group = rsquare ? t.n * 2 + (wave >> 1) : t.n * 4 + wave;
#pragma unroll
    for (int f = 0; f < kOwn; ++f)
      b_col[f] = min(group * kOwn + f, N / 16 - 1) * 1024;
    left = SK;
  };
  aim();
  if (waiting == 0) return;
  u32 rbuf = lds0;
  auto m0_of = [&](int j) { set_m0(rbuf + to_lds[min(j / 4, 3)] + j * 1024); };
  auto load_of = [&](int j, int square) __attribute__((always_inline)) {
    if (j >= 16 && square) return;
    if (j < 4 || (j < 8 && square)) {
      load_lds(da, a_voff[j % 8], a_soff);
    } else {
      const int f = (j - 4) % 8, half = (j - 4) / 8;
      load_lds(db, (lane ^ f) * 16u,
               b_soff[half] + b_col[f % kOwn] + (f >= kOwn ? up : 0));
    }
  };
  auto requested = [&]() __attribute__((always_inline)) {
    rbuf = 2 * lds0 + kWideStageB - rbuf;
    a_soff += 128;
    b_soff[0] += 2 * b_step;
    b_soff[1] += 2 * b_step;
    if (--left == 0) aim();
  };

  // ---- fragment reads: A row lane & 15, chunk 4 half + (lane >> 4)
  const int i16 = lane & 15, q = lane >> 4;
  const u32 a_rd = i16 * 128 + ((q ^ (i16 >> 1)) << 4);
  constexpr int kEach = GATE_UP ? 4 : 8;   // of a lane's columns in a row
  const u32 b_rd = i16 * kEach / 16 * 1024 +
                   (q * 16 + ((i16 * kEach & 15) | i16 * kEach / 16)) * 16;
  u32 a_at, b_at;                // of this wave in a stage
  auto read_at = [&](int square) {
    a_at = square ? (wave >> 1) * kRowsB : 0;
    b_at = square ? 2 * kRowsB + (wave & 1) * kWaveB : kRowsB + wave * kWaveB;
  };
  read_at(next.square);
  auto rda = [&](u32 buf, int half, int mi) {
    return *reinterpret_cast<const short8*>(
        smem + (buf + a_at) + (a_rd ^ (half * 64)) + mi * 2048);
  };
  auto rdb = [&](u32 buf, int half, int f) {
    return *reinterpret_cast<const short8*>(
        smem + (buf + b_at) + (b_rd ^ (f * 16)) + half * 8192 +
        f / kEach * 4096);
  };
  short8 a0[8], b0[8], a1[8], b1[8];
  floatx4 acc[8][8];

  for (int k = 0; k < 2; ++k) {
#pragma unroll
    for (int j = 0; j < 20; ++j) {
      m0_of(j);
      asm volatile("s_nop 4");
      load_of(j, rsquare);
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
  u32 buf = 0;
  constexpr int kCols = GATE_UP ? 64 : 128;   // of a wave
  // of a tile, at least: a lane's part of a row is one instruction or more, and a
  // wait that counts too few is only longer
  constexpr int kStores = 32;
  constexpr int kFree = 40, kEarly = 6;  // MFMAs up to the first barrier, DMAs
                                         // between the two
  // `behind`: stores that follow the DMAs that are waited for; `last`: of the tile
  auto stage = [&](auto first, bool behind,
                   bool last) __attribute__((always_inline)) {
    const int square = rsquare;  // of the tile that is requested
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      const int mi = i >> 3, f = i & 7;
      if (first) mfma_first(acc[mi][f], a0[mi], b0[f]);
      else mfma(acc[mi][f], a0[mi], b0[f]);
      __builtin_amdgcn_sched_barrier(0);
      if (i < 16 && i % 2 == 0) b1[i / 2] = rdb(buf, 1, i / 2);
      if (i >= 16 && i < 32 && i % 2 == 0)
        a1[i / 2 - 8] = rda(buf, 1, i / 2 - 8);
      if (i == kFree) {
        // all waves hold the stage in registers
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        sync_waves();
      }
      const int j = i - kFree - 1;
      if (j >= 0 && j < 2 * kEarly) {
        if (j % 2 == 0) m0_of(j / 2);
        else load_of(j / 2, square);
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
    buf = kWideStageB - buf;
    if (last) read_at(after.square);
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      const int mi = i >> 3, f = i & 7;
      mfma(acc[mi][f], a1[mi], b1[f]);
      __builtin_amdgcn_sched_barrier(0);
      if (i % 4 == 0 && i < 32) b0[i / 4] = rdb(buf, 0, i / 4);
      if (i % 4 == 0 && i >= 32) a0[i / 4 - 8] = rda(buf, 0, i / 4 - 8);
      if (i / 4 < 20 - kEarly) {
        if (i % 4 == 1) m0_of(kEarly + i / 4);
        if (i % 4 == 2) load_of(kEarly + i / 4, square);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    requested();
  };

  bool behind = false;
  while (waiting > 0) {
    stage(std::true_type{}, behind, false);
    for (int s = 1; s < SK; ++s) stage(std::false_type{}, false, s == SK - 1);
    settle();
    const Place t = next;
    next = after;
    after = third;
    --waiting;
    const int group = t.square ? t.n * 2 + (wave & 1) : t.n * 4 + wave;
    const int block = t.square ? t.m + (wave >> 1) : t.m;
    // (from a fresh copy of the lane, or the addresses would be kept in
    // registers that the loop needs)
    int l = lane;
    asm volatile("" : "+v"(l));
    const int col = group * kCols + (l & 15) * kEach;
    auto store = [&](bool inside) {
      if (!inside && col >= N) return;
      u16* to = out +
                static_cast<int64_t>(block * kWideM + (l >> 4) * 4) * N + col;
#pragma unroll
      for (int mi = 0; mi < 8; ++mi) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          struct alignas(2 * kEach) {
            u16 h[kEach];
          } o;
#pragma unroll
          for (int c = 0; c < kEach; ++c) {
            float v = acc_of(acc[mi][c][r]);
            if (GATE_UP) {
              const float u = acc_of(acc[mi][(c + 4) % 8][r]);
              if (MODE == 3) {
                const float gt = fminf(v, limit);
                const float up1 = fminf(fmaxf(u, -limit), limit);
                v = (gt / (1.f + __expf(-1.702f * gt))) * (up1 + 1.f);
              } else {
                v = silu(v) * u;
              }
            } else if (MODE == 2) {
              v = fmaxf(v, 0.f);
              v *= v;
            }
            o.h[c] = f32_to_bf16(v);
          }
          store_global(to, o);
          // (a step at a time, or all rows' places would be kept)
          to += static_cast<int64_t>(r < 3 ? 1 : 13) * N;
          asm volatile("" : "+v"(to));
        }
      }
    };
    behind = (group + 1) * kCols <= N;
    if (behind) store(true);
    else store(false);
  }
  // no DMA may land in LDS that is no longer this workgroup's
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

}  // namespace

// Gathered rows go in pairs unless experts have about 16 blocks or more (every one
// is taken to leave half a block empty): the ids of a pair's rows, and the questions
// of its shape, cost a tile 2 to 4 us, which pays while few blocks share the
// weights. us, both products, gate|up apart and in pairs: 128 experts, 2048 x 768, 2
// blocks each 331 and 315, 2.3 each 396 and 388, 4.4 each 632 and 621, 8.5 each 1165
// and 1140; 64 of 2048 x 1408, 6.5 each, 848 and 824, 12.5 each 1531 and 1513; 8 of
// 4096 x 6144, 16 each, 2083 and 2090, 33 each, one of them 129, 3941 and 3960. (With
// a lower clock, as after long steps: 4.4 each 650 and 651, 6.5 each 871 and 863. In
// whole steps of four layers, one after the other, pairs are ahead, 4.4 each 5113
// and 5068, 8.5 9378 and 9252; behind a pause of 0.1 s they lose 1 to 1.5 %, 6320 and
// 6421, 11532 and 11644.)
// Where few experts have all rows the host does not see it, and pairs lose: 8100 rows
// for 16 of 128 545 and 554; gate|up alone, 8 of 128 with 24 blocks each, 136 and 146
// (130 by tiles of 128 x 256), 16 with 32 each 306 and 316. Uneven rows as such do
// not: 128 experts of 58 to 2 blocks 364 and 369, of 17 to 3 389 and 384, 64 of 72 to
// 2 672 and 666. (Asking in the kernel how many experts there are, and taking blocks
// alone then, gives nothing back: 316 and 322, 64 experts 440 and 466.)
void launch_moe_wide(u16* out, const u16* a, const u16* b,
                     const int* sorted_ids, const int* expert_ids,
                     const int* n_valid, int max_mtiles, int experts,
                     int rows, int K, int N, int mode, float limit,
                     hipStream_t stream) {
  const int nt = ceil_div(N, mode == 1 || mode == 3 ? 256 : 512);
#define FI_WIDE(M, P)                                                        \
  hipLaunchKernelGGL((moe_wide_kernel<M, P>), dim3(kChip), dim3(256), 0,     \
                     stream, out, a, b, sorted_ids, expert_ids, n_valid, K,  \
                     N, nt, static_cast<u32>(rows) * (K * 2), limit)
  if (mode == 0) {
    FI_WIDE(0, true);
  } else if (max_mtiles <= 16 * experts) {
    if (mode == 1) FI_WIDE(1, true);
    else if (mode == 2) FI_WIDE(2, true);
    else FI_WIDE(3, true);
  } else {
    if (mode == 1) FI_WIDE(1, false);
    else if (mode == 2) FI_WIDE(2, false);
    else FI_WIDE(3, false);
  }
#undef FI_WIDE
}

}  // namespace fi
