// Prefill attention by whole query tiles: workgroups of four waves, two of them
// on a CU (three or four for heads of 64), each with one query tile, or with a
// list of them that it goes through without a pause (LISTS).
//
// One workgroup per query tile, as many as there are tiles, spends 7 to 10 us
// of each on other things than products: its start, the tile table and what
// that leads to one after the other, the first keys' and the queries' way, the
// results' way out; a prompt of a thousand tokens has 8 key tiles of 2 us for
// a query tile on average. By lists only as many workgroups run as fit on the
// chip (rows_grid; more where a list would be longer than kRowsList), and the
// next query tile's first keys are requested while the last ones of this tile
// are worked on, its queries while those are weighed.
//
// Who takes which tile is settled in advance: query tiles in order of their
// work (key tiles), the longest first, dealt to the workgroups of an XCD to and
// fro. Every workgroup counts the tiles of each work into LDS and finds its own
// from that (the order of equal ones is their order in the table), so that no
// counter outlives the launch. Of more than kRowsSort query tiles the order is
// the table's from its end. A query tile's products and their order are the
// same whoever takes it.
//
// One workgroup per query tile as it was, without rows stored whole and fragments
// read ahead, and this, us on one card, 32 query heads, 8 K/V heads of 128
// (TFLOP/s of the visible pairs): 8 x 1024 rows 115 and 94 (730), 8 of 1376 to 553
// rows 141 and 114 (750), 4 x 2048 183 and 163, 64 x 128 50 and 37, 200 x 100 145
// and 105, one of 8192 574 and 536 (1026); e4m3 8 x 1024 129 and 105; 16 query heads
// 71 and 52. A prompt of 1024 alone 30 and 27. Heads of 64: 8 x 1024 66 and 59, 16
// on 16 46 and 35, one of 8192 334 and 312. Of the mixers, 4 x 1800 rows, 16 heads
// of 128 on 16: 96 and 75, of 64 64 and 50; 8 x 1024, 32 on 8, behind a window of
// 512 99 and 92. Matrix cores are busy 40 to 52 % of the time, vector
// instructions issue for 50, LDS reads for 25.
//
// No form keeps registers in scratch memory: a value read back from there waits
// for the stores and for the next tile's keys in front of it (us with and without:
// 8 of 1376 to 553 rows, e4m3, 136 and 131; heads of 64, 64 x 128 rows, 33 and 23).
//
// EXT (bf16): positions instead of context lengths, cache blocks of any size, a
// sink, a gate, a sliding window that keeps the first keys. Tiles that no row
// of the workgroup sees are left out.
#pragma once

#include <algorithm>

#include "prefill_kernel.h"

namespace fi {

constexpr int kRowsWaves = attn_waves(false);
// workgroups of a CU, by their registers, and in all
constexpr int rows_each(int head_dim, bool lists) {
  return head_dim == 64 ? (lists ? 3 : 4) : 2;
}
constexpr int rows_groups(int head_dim) {
  return 256 * rows_each(head_dim, true);
}
constexpr int kRowsList = kWaveSize;   // query tiles of one, at most
constexpr int kRowsSort = 8192;        // query tiles that are put in order

// Whether a launch goes by lists. A list's start takes 4 to 6 us more (every
// query tile's lengths, their order), and at its end some CUs have nothing left
// while others still go through theirs, up to a tenth of the work of two or
// three rounds; what it saves is a start and an end per further query tile.
//  * One round: there is nothing to save.
//  * A window: tiles are short and alike, and CUs that take them as they come
//    end together (us, lists and one each: 2 x 4000, 32 heads of 128 on 8, 123 and
//    111, 16 on 4 66 and 61; 8 x 1024 95 and 95).
//  * Heads of 64, where a tile takes half as long and more of them run at once:
//    for up to three rounds of contexts that are neither short nor long (8 x 1024,
//    16 heads on 16, 35 and 42, 32 on 8 59 and 60, 64 on 8 114 and 101; 24 x 256 25
//    and 23; one of 8192 340 and 308; 4 x 1800, mixers, 50 and 61).
//  * Otherwise always (8 x 1024 94 and 102, 400 x 40 98 and 164, one of 8192 530
//    and 535), but for short contexts of one query tile per entry of the tile
//    table, where there are no empty ones to skip (mixers, 16 heads on 16: 60 x 64
//    22 and 20, 40 x 128 27 and 23, 16 x 512 41 and 47).
// sub: query tiles per entry; longest: no context is longer.
inline bool rows_by_lists(int64_t items, int head_dim, int sub, int window,
                          int64_t longest) {
  const int groups = rows_groups(head_dim);
  if (items <= groups || window > 0) return false;
  if (head_dim == 64)
    return items <= 3 * groups && longest >= 512 && longest <= 4096;
  return sub > 1 || longest >= 512;
}

// workgroups of a launch by lists with `items` query tiles of all head groups
inline int rows_grid(int64_t items, int head_dim) {
  constexpr int64_t kRound = 8 * kRowsList;
  return static_cast<int>(std::max<int64_t>(
      rows_groups(head_dim), (items + kRound - 1) / kRound * 8));
}

template <int D, bool PAGED, bool FP8, bool EXT, bool LISTS>
__global__ __launch_bounds__(kRowsWaves * kWaveSize, rows_each(D, LISTS))
void prefill_rows_kernel(const PrefillArgs p) {
  static_assert(!EXT || (PAGED && !FP8));
  constexpr bool kWindow = EXT && !LISTS;   // launches with one
  using R = RowSoftmax<D>;
  constexpr int kWaves = kRowsWaves, kBufs = 2;
  constexpr int KF = R::KF, kRowB = R::kRowB, kChunk = R::kChunk;
  constexpr int kTileB = R::kTileB, kRowsPerDma = R::kRowsPerDma;
  constexpr int kWRows = kKVTile / kWaves;   // rows a wave copies
  constexpr int kDma = kWRows / kRowsPerDma;  // DMAs per wave and matrix
  constexpr int kStores = 32 / kRowsPerDma;   // of a wave's whole rows
  static_assert(kWRows == 16, "a cache block per wave");

  __shared__ __attribute__((aligned(1024)))
  unsigned char smem[2 * kBufs * kTileB];
  const u32 lds0 = static_cast<u32>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) unsigned char*)smem));

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWaveSize);
  const int lane = tid % kWaveSize;
  const int col = lane & 31;           // this lane's query vector
  const int hi1 = lane >> 5;
  const int wph = kWaves / p.hpb;      // waves per query head
  const int groups = p.num_q_heads / p.hpb;

  // ---- this workgroup's query tiles: its r-th is place place_of(r) in the
  // order, head groups side by side (neighbouring workgroups go to different
  // XCDs), the longest first
  auto place_of = [&](int r) {
    const int b = blockIdx.x, j = b / 8, per = gridDim.x / 8;
    return LISTS ? 8 * (r * per + (r & 1 ? per - 1 - j : j)) + (b & 7) : b;
  };
  QTile mine = {};                     // lane r: of the r-th
  unsigned long long to_do = 1;
  if (!LISTS) {
    mine = uniform_tile(q_tile<PAGED, EXT>(p, p.nq - 1 - place_of(0) / groups));
    if (mine.work == 0) return;
  } else {
    int my_qt = -1;
    if (p.nq > kRowsSort) {
      const int place = place_of(lane);
      if (place < p.nq * groups) my_qt = p.nq - 1 - place / groups;
    } else {
      // bucket b of works at (b % 32) * 64 + b / 32, so that lane b / 32 reads
      // its 32 without conflicts; the last bucket has all longer ones too
      constexpr int kBuckets = 2048;
      int* count = reinterpret_cast<int*>(smem);
      u16* works = reinterpret_cast<u16*>(smem + kBuckets * 4);
      int* found = reinterpret_cast<int*>(smem + kBuckets * 4 + kRowsSort * 2);
      static_assert(kBuckets * 4 + kRowsSort * 2 + kRowsList * 4 <=
                    2 * kBufs * kTileB);
      constexpr int kThreads = kWaves * kWaveSize;
      for (int i = tid; i < kBuckets; i += kThreads) count[i] = 0;
      __syncthreads();
      for (int i = tid; i < p.nq; i += kThreads) {
        const int b = min(q_tile<PAGED, EXT>(p, i).work, kBuckets - 1);
        works[i] = b;
        if (b > 0) atomicAdd(&count[b % 32 * 64 + b / 32], 1);
      }
      __syncthreads();
      // lane l: buckets 2047 - 32 l down to 2016 - 32 l
      const int line = 63 - lane;
      int own = 0;
      for (int k = 0; k < 32; ++k) own += count[k * 64 + line];
      int incl = own;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
      }
      const int all = __shfl(incl, 63, 64);
      if (tid < kRowsList) found[tid] = -1;
      __syncthreads();
      for (int r = wave; r < kRowsList; r += kWaves) {
        int rank = place_of(r) / groups;
        if (rank >= all) break;          // places ascend
        const int l = __builtin_ctzll(__ballot(incl > rank));
        rank -= __shfl(incl, l, 64) - __shfl(own, l, 64);
        // the bucket: lane k has the k-th from the line's top
        int in = lane < 32 ? count[(31 - lane) * 64 + 63 - l] : 0;
        const int here = in;
#pragma unroll
        for (int off = 1; off < 32; off <<= 1) {
          const int o = __shfl_up(in, off, 64);
          if (lane >= off) in += o;
        }
        const int k =
            __builtin_ctzll(__ballot(lane < 32 && in > rank));
        rank -= __shfl(in, k, 64) - __shfl(here, k, 64);
        const int work = (63 - l) * 32 + 31 - k;
        // its rank-th query tile
        for (int i0 = 0; i0 < p.nq; i0 += kWaveSize) {
          const int i = i0 + lane;
          const unsigned long long same =
              __ballot(i < p.nq && works[min(i, p.nq - 1)] == work);
          const int n = __builtin_popcountll(same);
          if (rank < n) {
            const int before = __builtin_popcountll(
                same & ((1ull << lane) - 1));
            if ((same >> lane & 1) && before == rank) found[r] = i;
            break;
          }
          rank -= n;
        }
      }
      __syncthreads();
      my_qt = found[lane];
    }
    if (my_qt >= 0) mine = q_tile<PAGED, EXT>(p, my_qt);
    to_do = __ballot(my_qt >= 0 && mine.work > 0);
    if (to_do == 0) return;
    __syncthreads();                   // the lists' LDS is free
  }

  // the first of `of`, uniform
  struct Item {
    QTile t;
    int hg, first, skip_lo, skip_hi;   // first and skipped key tiles
  };
  auto item_of = [&](unsigned long long of) {
    const int r = LISTS ? __builtin_ctzll(of) : 0;
    Item it;
    it.t = mine;
    if (LISTS) {
      it.t.seq = __builtin_amdgcn_readlane(mine.seq, r);
      it.t.row0 = __builtin_amdgcn_readlane(mine.row0, r);
      it.t.seq_start = __builtin_amdgcn_readlane(mine.seq_start, r);
      it.t.seq_len = __builtin_amdgcn_readlane(mine.seq_len, r);
      it.t.k_len = __builtin_amdgcn_readlane(mine.k_len, r);
      it.t.work = __builtin_amdgcn_readlane(mine.work, r);
    }
    it.hg = place_of(r) % groups;
    // tiles between the kept first keys and the window of the first row
    it.skip_lo = kWindow ? ceil_div(p.keep_first, kKVTile) : 0;
    it.skip_hi = kWindow && p.window > 0
        ? max(it.t.k_len - it.t.seq_len + it.t.row0 - p.window + 1, 0) /
              kKVTile
        : 0;
    it.first = kWindow && it.skip_lo == 0 ? it.skip_hi : 0;
    return it;
  };
  auto after = [&](const Item& it, int tile) {
    const int n = tile + 1;
    return kWindow && n >= it.skip_lo && n < it.skip_hi ? it.skip_hi : n;
  };

  // ---- staging: the next key tile to request, of this query tile or a later
  // one. Wave w copies rows 16w..16w+15 of it, one cache block. Rows past
  // the end repeat the last one (finite values; their scores are masked).
  unsigned long long to_request = LISTS ? to_do & (to_do - 1) : 0;
  Item ahead = item_of(to_do);
  int atile = ahead.first;
  bool more = true;                    // there is such a tile
  int blk = 0;
  // EXT, blocks of other sizes than 16: this lane's rows of a tile
  const bool by_row = EXT && p.block_size != 16;
  int64_t row_at[EXT ? kDma : 1];
  auto kv_head_of = [&](const Item& it) {
    return it.hg * p.hpb / (p.num_q_heads / p.num_kv_heads);
  };
  auto look_up = [&] {                 // where the tile's rows are
    if (EXT && by_row) {
      const int* bt = p.block_tables + static_cast<int64_t>(ahead.t.seq) *
                                           p.max_blocks;
      int r0 = lane / kChunk;
      if (R::kFew) asm volatile("" : "+v"(r0));
#pragma unroll
      for (int i = 0; i < kDma; ++i) {
        const int key = min(atile * kKVTile + wave * kWRows +
                                i * kRowsPerDma + r0,
                            ahead.t.k_len - 1);
        row_at[i] = (static_cast<int64_t>(bt[key / p.block_size]) *
                         p.num_kv_heads + kv_head_of(ahead)) * p.block_size +
                    key % p.block_size;
      }
    } else if (PAGED && !FP8) {
      blk = const_ints(p.block_tables + static_cast<int64_t>(ahead.t.seq) *
                                            p.max_blocks)
          [min(atile * 4 + wave, (ahead.t.k_len - 1) >> 4)];
    }
  };
  // where this lane's first DMAs of a cache block begin; those of the i-th
  // rows lie at ^ 1024 i, their chunks of K at ^ 64 i
  const u32 k_from = lane / kChunk * kRowB +
                     ((lane % kChunk) ^ R::k_swz(lane / kChunk)) * 16;
  const u32 v_from = lane / kChunk * kRowB +
                     ((lane % kChunk) ^ R::v_swz(lane / kChunk)) * 16;
  auto stage = [&](int buf) {
    const u32 kdst = lds0 + buf * kTileB + wave * kWRows * kRowB;
    const u32 vdst = kdst + kBufs * kTileB;
    // of a row, where rows are not side by side
    u32 k_in = k_from, v_in = v_from;
    int r0 = lane / kChunk;
    if (R::kFew) asm volatile("" : "+v"(k_in), "+v"(v_in), "+v"(r0));
    if (EXT && by_row) {
#pragma unroll
      for (int i = 0; i < kDma; ++i) {
        const int64_t at = row_at[i] * kRowB;
        dma_to_lds16_at(kdst + i * 1024,
                        static_cast<const unsigned char*>(p.k) + at +
                            ((k_in ^ (i * 64)) & (kRowB - 1)));
        dma_to_lds16_at(vdst + i * 1024,
                        static_cast<const unsigned char*>(p.v) + at +
                            (v_in & (kRowB - 1)));
      }
      return;
    }
    const u16* kb;
    const u16* vb;
    int first, limit;                  // row of the wave, last valid row
    int64_t ks, vs;
    if (PAGED) {
      const int64_t base = (static_cast<int64_t>(blk) * p.num_kv_heads +
                            kv_head_of(ahead)) * 16 * D;
      kb = static_cast<const u16*>(p.k) + base;
      vb = static_cast<const u16*>(p.v) + base;
      first = 0;
      limit = ahead.t.k_len - 1 -
              min(atile * 4 + wave, (ahead.t.k_len - 1) >> 4) * 16;
      ks = vs = D;
    } else {
      const int row = min(atile * kKVTile, ahead.t.k_len - 1);
      kb = static_cast<const u16*>(p.k) +
           (ahead.t.seq_start + row) * p.k_stride +
           int64_t(kv_head_of(ahead)) * D;
      vb = static_cast<const u16*>(p.v) +
           (ahead.t.seq_start + row) * p.v_stride +
           int64_t(kv_head_of(ahead)) * D;
      first = wave * kWRows;
      limit = ahead.t.k_len - 1 - row;
      ks = p.k_stride;
      vs = p.v_stride;
    }
    if (PAGED && limit >= kWRows - 1) {  // no row lies past the end
#pragma unroll
      for (int i = 0; i < kDma; ++i) {
        dma_to_lds16(kdst + i * 1024, kb, k_from ^ (i * (1024 + 64)));
        dma_to_lds16(vdst + i * 1024, vb, v_from ^ (i * 1024));
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < kDma; ++i) {
      const int src = min(first + i * kRowsPerDma + r0, limit);
      dma_to_lds16(kdst + i * 1024, kb,
                   src * static_cast<int>(ks) * 2 +
                       ((k_in ^ (i * 64)) & (kRowB - 1)));
      dma_to_lds16(vdst + i * 1024, vb,
                   src * static_cast<int>(vs) * 2 + (v_in & (kRowB - 1)));
    }
  };
  // fp8: a thread owns 16 dims of one row of K and of V
  constexpr int kParts = D / 16;
  constexpr int kStep = kWaves * kWaveSize / kParts;  // rows per step
  constexpr int kSteps = kKVTile / kStep;
  static_assert(kSteps * kStep == kKVTile);
  const int f_row0 = tid / kParts, f_part = tid % kParts;
  uint4 k_raw[kSteps], v_raw[kSteps];
  auto load_fp8 = [&] {
    const ConstInts bt = const_ints(
        p.block_tables + static_cast<int64_t>(ahead.t.seq) * p.max_blocks);
#pragma unroll
    for (int i = 0; i < kSteps; ++i) {
      const int src = min(atile * kKVTile + f_row0 + i * kStep,
                          ahead.t.k_len - 1);
      const int64_t off =
          ((static_cast<int64_t>(bt[src >> 4]) * p.num_kv_heads +
            kv_head_of(ahead)) * 16 + (src & 15)) * D + f_part * 16;
      k_raw[i] = *reinterpret_cast<const uint4*>(
          static_cast<const unsigned char*>(p.k) + off);
      v_raw[i] = *reinterpret_cast<const uint4*>(
          static_cast<const unsigned char*>(p.v) + off);
    }
  };
  auto write_fp8 = [&](int buf) {
    auto put = [&](unsigned char* dst, const uint4& raw, int f_row, int swz) {
      const u32 w[4] = {raw.x, raw.y, raw.z, raw.w};
      float f[16];
#pragma unroll
      for (int i = 0; i < 4; ++i) unpack_fp8x4(w[i], &f[i * 4]);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        bf16x8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o.h[j] = f32_to_bf16(f[h * 8 + j]);
        *reinterpret_cast<bf16x8*>(
            dst + f_row * kRowB + (((f_part * 2 + h) ^ swz) * 16)) = o;
      }
    };
#pragma unroll
    for (int i = 0; i < kSteps; ++i) {
      const int r = f_row0 + i * kStep;
      put(smem + buf * kTileB, k_raw[i], r, R::k_swz(r));
      put(smem + (kBufs + buf) * kTileB, v_raw[i], r, R::v_swz(r));
    }
  };
  auto step_ahead = [&] {
    atile = after(ahead, atile);
    if (atile < ahead.t.work) return;
    if (!LISTS || to_request == 0) {
      more = false;
      return;
    }
    ahead = item_of(to_request);
    to_request &= to_request - 1;
    atile = ahead.first;
  };
  look_up();
  if (FP8) {
    load_fp8();
    write_fp8(0);
  } else {
    stage(0);
  }
  step_ahead();
  bool loaded = more;                  // fp8: the next tile is in registers
  if (more) {
    if (FP8) {
      load_fp8();
      step_ahead();
    } else {
      look_up();
    }
  }

  // ---- query fragments (B operand of S^T): lane holds
  // Q[row0+col][f*16 + hi1*8 .. +8]
  short8 b_q[KF];
  auto head_of = [&](const Item& it) { return it.hg * p.hpb + wave / wph; };
  auto row0_of = [&](const Item& it) {
    return it.t.row0 + (wave % wph) * 32;
  };
  auto load_q = [&](const Item& it) {
    const int qr = min(row0_of(it) + col, it.t.seq_len - 1);
    const u16* qrow = p.q + (it.t.seq_start + qr) * p.q_stride +
                      static_cast<int64_t>(head_of(it)) * D;
#pragma unroll
    for (int f = 0; f < KF; ++f)
      b_q[f] = *reinterpret_cast<const short8*>(qrow + f * 16 + hi1 * 8);
  };
  Item it = item_of(to_do);
  load_q(it);

  RowSoftmax<D> row(lane, p.scale);
  const float sgn = sign_of(p.scale);
  int buf = 0;
  bool behind = false;                 // this wave's last kStores vector
                                       // memory instructions are stores
  while (true) {
    turn_queries(b_q, sgn);
    // arrived here, not at their first use: that is inside the loop,
    // where the wait would take in the DMAs of every tile
#pragma unroll
    for (int f = 0; f < KF; ++f) asm volatile("" : "+v"(b_q[f]));
    row.clear();
    const int head = head_of(it), row0 = row0_of(it);
    const bool active = row0 < it.t.seq_len;
    const int ctx_start = it.t.k_len - it.t.seq_len;
    const int my_q_max = ctx_start + min(row0 + 32, it.t.seq_len) - 1;
    // of this lane's query vector, less what its keys lie further on than crow's
    const int q_at = ctx_start + row0 + col - 4 * hi1;
    floatx16 s_acc[2];
    bool seen = false;
    int tile = it.first;
    auto weigh = [&] {                 // the scores of `tile`
      if (!seen) return;
      const int kv0 = tile * kKVTile;
      // only tiles at the diagonal or the end mask
      if (kv0 + kKVTile - 1 > ctx_start + row0) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (kv0 + 32 * b + crow(r, 0) > q_at)
              s_acc[b][r] = -INFINITY;
      }
      if (kWindow && p.window > 0 && kv0 + kKVTile > p.keep_first &&
          my_q_max - kv0 >= p.window) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = kv0 + 32 * b + crow(r, 0);
            if (q_at - key >= p.window && key + 4 * hi1 >= p.keep_first)
              s_acc[b][r] = -INFINITY;
          }
      }
      row.add(smem, (kBufs + buf) * kTileB, s_acc);
    };
    while (true) {
      // this tile has landed (this wave's part; the barrier covers the
      // others'), and nobody reads the buffer that is filled next
      if (!FP8) {
        if (behind)
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kStores) : "memory");
        else
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        behind = false;
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (FP8) {
        if (loaded) write_fp8(buf ^ 1);
        loaded = more;
        if (more) {
          load_fp8();
          step_ahead();
        }
      } else if (more) {
        stage(buf ^ 1);
        step_ahead();
        if (more) look_up();
      }
      const int kv0 = tile * kKVTile;
      // (or outside the window of every row of the wave)
      seen = active && kv0 <= my_q_max &&
             !(kWindow && p.window > 0 && kv0 >= p.keep_first &&
               kv0 + kKVTile <= ctx_start + row0 - p.window + 1);
      if (seen)
        row.scores(smem, buf * kTileB, (kBufs + buf) * kTileB, b_q, s_acc);
      const int n = after(it, tile);
      if (LISTS && n >= it.t.work) break;
      weigh();
      if (!LISTS && n >= it.t.work) break;
      tile = n;
      buf ^= 1;
    }
    // the next query tile's queries, while the last keys are weighed
    to_do &= to_do - 1;
    const Item now = it;
    if (LISTS && to_do != 0) {
      it = item_of(to_do);
      load_q(it);
    }
    if (LISTS) weigh();

    // ---- epilogue: every wave is done with the tile, whose place the
    // results are turned over in
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (active) {
      // (made again, not kept)
      const int lane = __builtin_amdgcn_mbcnt_hi(
          ~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0));
      const int col = lane & 31, hi1 = lane >> 5;
      row.l_row += half_swap(row.l_row);
      float inv = row.l_row > 0.f ? 1.f / row.l_row : 0.f;
      const u16* gp = nullptr;
      if (EXT && row0 + col < now.t.seq_len) {
        if (p.sink != nullptr) {
          // in the domain of whichever is larger
          const float sk = p.sink[head] * 1.4426950408889634f;
          const float mc = row.m_row * row.c, top = fmaxf(mc, sk);
          const float a = __builtin_amdgcn_exp2f(mc - top);
          inv = a / (row.l_row * a + __builtin_amdgcn_exp2f(sk - top));
        }
        if (p.gate != nullptr) {
          gp = p.gate + (now.t.seq_start + row0 + col) *
                            static_cast<int64_t>(p.g_stride);
          if (p.gate_elem) {
            gp += static_cast<int64_t>(head) * D;
          } else {
            inv *= 1.f / (1.f + expf(-bf16_to_f32(gp[head])));
            gp = nullptr;
          }
        }
      }
      const int rows = now.t.seq_len - row0;
      u16* out = p.out + (static_cast<int64_t>(now.t.seq_start + row0) *
                              p.num_q_heads + head) * D;
      put_rows<D>(
          smem, (wave / 2 * kBufs + buf) * kTileB + wave % 2 * 32 * kRowB, out,
          static_cast<int64_t>(p.num_q_heads) * D, rows, lane,
          [&](int cb, int r) {
            bf16x4 w;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              float v = row.o_acc[cb][r + j] * inv;
              if (EXT && gp != nullptr)
                v *= 1.f / (1.f + expf(-bf16_to_f32(
                                      gp[cb * 32 + crow(r, hi1) + j])));
              w.h[j] = f32_to_bf16(v);
            }
            return w;
          });
      behind = rows >= 32 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
    }
    if (!LISTS || to_do == 0) return;
    buf ^= 1;
  }
}

// `longest`: no key lies further on in its context
template <int D, bool PAGED, bool FP8, bool EXT>
void launch_rows(const PrefillArgs& a, int64_t longest, hipStream_t stream) {
  const int64_t items = static_cast<int64_t>(a.num_q_heads / a.hpb) * a.nq;
  const dim3 block(kRowsWaves * kWaveSize);
  if (rows_by_lists(items, D, a.sub, a.window, longest))
    hipLaunchKernelGGL((prefill_rows_kernel<D, PAGED, FP8, EXT, true>),
                       dim3(rows_grid(items, D)), block, 0, stream, a);
  else
    hipLaunchKernelGGL((prefill_rows_kernel<D, PAGED, FP8, EXT, false>),
                       dim3(static_cast<unsigned>(items)), block, 0, stream, a);
}

}  // namespace fi
