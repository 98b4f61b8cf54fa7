// Varlen causal prefill / context attention (flash-style, MFMA).
//
// out[t, h, :] = softmax(Q K^T * scale, causal) V, GQA, bf16 in / fp32
// accumulate. PAGED variant reads K/V from the paged cache via block tables
// (q rows are only each sequence's NEW tokens — prefix-cache hits and
// chunked prefill skip cached tokens).
//
// A workgroup holds 32 query vectors per wave of one K/V head: R rows times
// HPB query heads that share it (HPB = the largest of 4, 2, 1 that divides
// the group). Rows of one workgroup lie close together, so causal raggedness
// costs at most one K/V tile per wave.
//
// Per K/V tile of 64 tokens:
//  * K and V rows go from global memory to LDS by DMA, one or two tiles
//    ahead, ONE barrier per tile. The DMA is written in asm: the compiler
//    orders every LDS read after every DMA builtin it can see (it emitted
//    vmcnt(0) in front of each tile's reads, which waited for the tile just
//    requested); the waits here are the real ones.
//  * S^T = K Q^T (mfma_32x32x16, A = K): a query's scores sit in one lane
//    (and its half-wave partner), the softmax is in-register.
//  * O^T += V^T P^T (A = V^T read from the row-major tile with the LDS
//    transpose read, B = P^T): the order of the keys within a 16-deep step
//    is the one in which the score registers already hold them, so P needs
//    a pack and no lane exchange, and the running maximum, the sum and the
//    final division stay lane-local too. V staged through registers and
//    written transposed in 2-byte pieces was the largest part of the tile
//    before.
//  * Rows are stored swizzled in 16-byte chunks so that both read patterns
//    touch every bank evenly.
// Bound by the vector ALU beside the matrix cores: a tile costs a wave 1024
// cycles of MFMA and more of exponentials (512), scaling, sums, maxima, packs and
// addresses, which two waves per SIMD overlap in part.
//
// Here: what the forms share, and the split form. Whole query tiles:
// prefill_rows.h; 64 query vectors per wave: prefill_pair.h.
//
// SPLIT: when whole query tiles would leave the chip idle, the K/V tiles of
// all query tiles form one line that up to 256 workgroups cut into equal
// parts; a query tile that is cut leaves unnormalised fp32 pieces behind and
// a second kernel adds them up.
//
// C-fragment row map (32x32): row = (r&3) + 8*(r>>2) + 4*(lane>>5),
// col = lane&31.
//
// Capability parity: the paged-attention prefill the reference delegates
// to vLLM.
#pragma once

#include "common.h"

namespace fi {

typedef __attribute__((ext_vector_type(4))) short short4v;
typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(16))) float floatx16;

constexpr int kKVTile = 64;                   // kv tokens per LDS tile
constexpr float kPNegInf = -1e30f;
// keep the running maximum while a tile's exceeds it by no more than this
// (base-2 units, e^8): P is then bounded by e^8, which f32 accumulation
// absorbs, and the accumulators are rescaled only where it matters
constexpr float kDeferThr = 11.5416f;

FI_DEV constexpr int crow(int r, int hi1) {
  return (r & 3) + 8 * (r >> 2) + 4 * hi1;
}

// the other half-wave's value of the same lane & 31
FI_DEV float half_swap(float v) {
  const auto s = __builtin_amdgcn_permlane32_swap(
      __float_as_int(v), __float_as_int(v), false, false);
  return __int_as_float((threadIdx.x & 32) ? s[0] : s[1]);
}

struct PrefillArgs {
  u16* out;               // [T, Hq, D]
  const u16* q;           // [T] rows, stride q_stride
  const void* k;          // dense rows OR k_cache when PAGED
  const void* v;
  const int* tile_seq;    // [ntiles] sequence index
  const int* tile_row0;   // [ntiles] first NEW q row
  const int* cu_seqlens;  // [nseqs+1] over NEW tokens
  const int* block_tables;  // [S, max_blocks] (PAGED)
  const int* seq_lens_k;    // [S] total ctx len (PAGED)
  float* piece_o;           // [slots][2][256 * D]  (SPLIT)
  float* piece_ml;          // [slots][2][waves][64][2] (SPLIT)
  int4* cut;                // [slots] what a part's end cuts (SPLIT)
  int64_t q_stride, k_stride, v_stride;
  int max_blocks, num_q_heads, num_kv_heads;
  int hpb;                  // query heads per workgroup
  int rows;                 // rows per workgroup
  int slots;                // workgroups of the SPLIT form
  int sub;                  // query tiles per entry of the tile table
  int nq;                   // query tiles in all
  float scale;
  // EXT
  const int* positions;     // [T] context position of every new row
  const float* sink;        // [Hq] or nullptr: joins the denominator
  const u16* gate;          // sigmoid gate per (row, head) or entry, or nullptr
  int64_t g_stride;
  bool gate_elem;
  int block_size;           // rows of a cache block
  int window, keep_first;   // window > 0: key j for p - j < window or
                            // j < keep_first
};

// one query tile: rows [row0, ..) of a sequence and its K/V tiles
struct QTile {
  int seq, row0, seq_start, seq_len, k_len, work;
};

template <bool PAGED, bool EXT = false>
FI_DEV QTile q_tile(const PrefillArgs& p, int qt) {
  QTile t;
  const int rows = p.rows;
  const int tile = qt / p.sub;
  t.seq = p.tile_seq[tile];
  t.row0 = p.tile_row0[tile] + (qt - tile * p.sub) * rows;
  t.seq_start = p.cu_seqlens[t.seq];
  t.seq_len = p.cu_seqlens[t.seq + 1] - t.seq_start;
  if (EXT)  // a portion's positions ascend by one
    t.k_len = t.seq_len > 0 ? p.positions[t.seq_start] + t.seq_len : 0;
  else
    t.k_len = PAGED ? p.seq_lens_k[t.seq] : t.seq_len;
  t.work = 0;
  if (t.row0 < t.seq_len)
    t.work = (t.k_len - t.seq_len + min(t.row0 + rows, t.seq_len) - 1) /
                 kKVTile + 1;
  return t;
}

FI_DEV QTile uniform_tile(QTile t) {
  t.seq = __builtin_amdgcn_readfirstlane(t.seq);
  t.row0 = __builtin_amdgcn_readfirstlane(t.row0);
  t.seq_start = __builtin_amdgcn_readfirstlane(t.seq_start);
  t.seq_len = __builtin_amdgcn_readfirstlane(t.seq_len);
  t.k_len = __builtin_amdgcn_readfirstlane(t.k_len);
  t.work = __builtin_amdgcn_readfirstlane(t.work);
  return t;
}

// the K/V tiles of all query tiles of one head group, by one wave
template <bool PAGED>
FI_DEV int total_work(const PrefillArgs& p, int lane) {
  int sum = 0;
  for (int i = lane; i < p.nq; i += kWaveSize) sum += q_tile<PAGED>(p, i).work;
#pragma unroll
  for (int off = 32; off; off >>= 1) sum += __shfl_xor(sum, off, 64);
  return __builtin_amdgcn_readfirstlane(sum);
}

// query tile that holds place `at` of a head group's line, and the place
// within it; every wave of the launch computes the same
template <bool PAGED>
FI_DEV int find_tile(const PrefillArgs& p, int lane, int at, int* within) {
  int before = 0;
  for (int i0 = 0; i0 < p.nq; i0 += kWaveSize) {
    const int i = i0 + lane;
    const int w = i < p.nq ? q_tile<PAGED>(p, i).work : 0;
    int incl = w;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(incl, off, 64);
      if (lane >= off) incl += o;
    }
    const unsigned long long hit = __ballot(before + incl > at);
    if (hit) {
      const int l = __builtin_ctzll(hit);
      *within = __builtin_amdgcn_readfirstlane(
          at - before - (__shfl(incl, l, 64) - __shfl(w, l, 64)));
      return i0 + l;
    }
    before += __builtin_amdgcn_readfirstlane(__shfl(incl, 63, 64));
  }
  *within = 0;
  return p.nq;
}

// place of a workgroup's part in the whole line: neighbours on one XCD
// (every eighth workgroup) take neighbouring parts and share K/V in its L2
FI_DEV int split_slot(int b, int slots) {
  return (b & 7) * (slots / 8) + (b >> 3);
}
struct Parts {
  int64_t each;  // tiles of a part; the first `more` parts have one more
  int more;
  FI_DEV Parts(int64_t total, int slots)
      : each(total / slots), more(static_cast<int>(total % slots)) {}
  FI_DEV int64_t begin(int slot) const {
    return slot * each + min(slot, more);
  }
};

// FP8 (PAGED only): the cache holds OCP e4m3. LDS tiles stay bf16, so K and
// V pass through registers with an exact conversion (half the bytes from
// memory), one tile ahead.
//
// The split form runs one workgroup of 8 waves per CU, which reads K/V half as
// often, with three buffers; the other form two workgroups of 4 waves with two,
// so that one computes while the other is between two query tiles.
constexpr int attn_waves(bool split) { return split ? 8 : 4; }

// (in asm, or each operand that comes from a product is made canonical first)
FI_DEV float largest(float a, float b, float c) {
  float v = a;
#if defined(__HIP_DEVICE_COMPILE__)
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(v) : "v"(a), "v"(b), "v"(c));
#endif
  return v;
}

// What a wave does with a tile in LDS: 32 query vectors, one per lane and its
// half-wave partner.
//
// The order is pinned: fragments are read four products ahead of their use (two
// for heads of 64), V's first ones before the softmax, and a 16-deep step's
// products go between the exponentials and sums of the next one. (Left to the
// compiler, each product of V waits for its own read just issued, which two waves
// per SIMD hide in part: 8 x 1024 rows 104 us and 94 so, one of 8192 569 and 536.)
template <int D>
struct RowSoftmax {
  static constexpr int KF = D / 16;      // QK^T 16-deep steps over head dim
  static constexpr int CB = D / 32;      // 32-dim blocks of the output
  static constexpr int kRowB = D * 2;    // bytes of a K or V row
  static constexpr int kChunk = D / 8;   // 16-byte chunks of a row
  static constexpr int kTileB = kKVTile * kRowB;
  static constexpr int kRowsPerDma = 1024 / kRowB;
  static constexpr int kAhead = D == 64 ? 2 : 4;   // fragments
  // places that each tile or query tile needs again are made again, not kept:
  // three or four workgroups share a CU's registers
  static constexpr bool kFew = D == 64;
  static_assert(D == 128 || D == 64, "swizzles are for these row sizes");

  int k_off, v_off;                      // of fragment 0
  float c;                               // scale * log2(e)
  float m_row, l_row;                    // l of this half-wave's keys
  floatx16 o_acc[CB];
  short8 v_frag[kAhead];

  // swizzled chunk of a row: K rows are read one chunk per lane over 32
  // rows, V rows four lanes to 32 bytes over 8 rows
  FI_DEV static int k_swz(int row) {
    return D == 128 ? row & 15 : (row >> 1) & 7;
  }
  FI_DEV static int v_swz(int row) {
    return D == 128 ? (row & 3) << 2 : ((row >> 1) & 1) << 2;
  }
  FI_DEV RowSoftmax(int lane, float scale) {
    const int col = lane & 31, hi1 = lane >> 5;
    k_off = col * kRowB + ((hi1 ^ k_swz(col)) * 16);
    const int row = 4 * hi1 + ((lane & 15) >> 2);
    v_off = row * kRowB +
            (((((lane >> 4) & 1) * 2 + ((lane & 3) >> 1)) ^ v_swz(row)) * 16) +
            (lane & 1) * 8;
    // (uniform: in a scalar register)
    c = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(
        scale == 0.f ? 1.f : fabsf(scale) * 1.4426950408889634f)));
  }
  FI_DEV void clear() {
    m_row = kPNegInf;
    l_row = 0.f;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int r = 0; r < 16; ++r) o_acc[cb][r] = 0.f;
  }
  FI_DEV static void pin() { __builtin_amdgcn_sched_barrier(0); }
  // fragment n of K: step n / 2, keys 32 (n & 1) on
  FI_DEV short8 read_k(const unsigned char* smem, int at, int n) const {
    return *reinterpret_cast<const short8*>(
        smem + ((at + k_off) ^ ((n >> 1) * 32)) + (n & 1) * 32 * kRowB);
  }
  // of V: step n / CB, dims 32 (n % CB) on
  FI_DEV short8 read_v(const unsigned char* smem, int at, int n) const {
    const unsigned char* a =
        smem + ((at + v_off) ^ (n % CB * 64)) + n / CB * 16 * kRowB;
    const short4v lo = lds_read_tr4(a), hi = lds_read_tr4(a + 8 * kRowB);
    return short8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  }
  // S^T[kv 64 x q 32] of the tile whose K and V begin at k_at and v_at
  FI_DEV void scores(const unsigned char* smem, int k_at, int v_at,
                     const short8 (&b_q)[KF], floatx16 (&s_acc)[2]) {
    short8 k_frag[kAhead];
#pragma unroll
    for (int n = 0; n < kAhead; ++n) k_frag[n] = read_k(smem, k_at, n);
    __builtin_amdgcn_s_setprio(1);
    pin();
#pragma unroll
    for (int n = 0; n < 2 * KF; ++n) {
      const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f,
                             0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      s_acc[n & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          k_frag[n % kAhead], b_q[n >> 1], n < 2 ? zero : s_acc[n & 1], 0, 0,
          0);
      pin();
      if (n + kAhead < 2 * KF)
        k_frag[n % kAhead] = read_k(smem, k_at, n + kAhead);
      else
        v_frag[n + kAhead - 2 * KF] =
            read_v(smem, v_at, n + kAhead - 2 * KF);
      pin();
    }
    __builtin_amdgcn_s_setprio(0);
  }
  // the online softmax, and O^T[D x q 32] += V^T[D x 64] P^T[64 x 32]
  FI_DEV void add(const unsigned char* smem, int v_at,
                  const floatx16 (&s_acc)[2]) {
    // (the products' results are not waited for in front of asm)
    asm volatile("s_nop 15" ::: "memory");
    pin();
    float rm = s_acc[0][0];
#pragma unroll
    for (int r = 0; r < 16; ++r) rm = largest(rm, s_acc[0][r], s_acc[1][r]);
    rm = fmaxf(rm, half_swap(rm));
    if (!__all((rm - m_row) * c <= kDeferThr)) {
      const float m_new = fmaxf(m_row, rm);
      const float alpha = __builtin_amdgcn_exp2f((m_row - m_new) * c);
      m_row = m_new;
      l_row *= alpha;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[cb][r] *= alpha;
    }
    const float mc = m_row * c;
    float rs[4] = {0.f, 0.f, 0.f, 0.f};
    bf16x8 w[2];                         // this step's weights and the next's
    auto weights = [&](int kc, int from, int to) {
#pragma unroll
      for (int j = from; j < to; ++j) {
        const float pv = __builtin_amdgcn_exp2f(
            fmaf(s_acc[kc >> 1][8 * (kc & 1) + j], c, -mc));
        rs[j & 3] += pv;
        w[kc & 1].h[j] = f32_to_bf16(pv);
      }
      // (here, or all weights would be kept for sums at the tile's end)
#pragma unroll
      for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(rs[i]));
    };
    weights(0, 0, 8);
    // (a wave with products in front of one without; us without and with, 32
    // heads of 128 on 8, e4m3: 4099 rows behind 16384 1281 and 1265, 8 of 1376 to
    // 553 131 and 126; heads of 64, one of 8192: 312 and 330)
    if (!kFew) __builtin_amdgcn_s_setprio(1);
    pin();
#pragma unroll
    for (int n = 0; n < 4 * CB; ++n) {
      const int kc = n / CB, cb = n % CB;
      o_acc[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          v_frag[n % kAhead], __builtin_bit_cast(short8, w[kc & 1]),
          o_acc[cb], 0, 0, 0);
      pin();
      if (n + kAhead < 4 * CB)
        v_frag[n % kAhead] = read_v(smem, v_at, n + kAhead);
      if (kc < 3) weights(kc + 1, cb * 8 / CB, (cb + 1) * 8 / CB);
      pin();
    }
    if (!kFew) __builtin_amdgcn_s_setprio(0);
    l_row += (rs[0] + rs[1]) + (rs[2] + rs[3]);
  }
};

// the other sign's queries, or none for a scale of zero, so that the maximum
// can be taken over unscaled scores
FI_DEV float sign_of(float scale) {
  return scale > 0.f ? 1.f : (scale < 0.f ? -1.f : 0.f);
}
template <int KF>
FI_DEV void turn_queries(short8 (&b_q)[KF], float sgn) {
  if (sgn == 1.f) return;
#pragma unroll
  for (int f = 0; f < KF; ++f) {
    bf16x8 h = __builtin_bit_cast(bf16x8, b_q[f]);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      h.h[j] = f32_to_bf16(bf16_to_f32(h.h[j]) * sgn);
    b_q[f] = __builtin_bit_cast(short8, h);
  }
}

// A wave's 32 rows of results leave through LDS (32 rows from `at` on that nobody
// else uses), neighbouring lanes neighbouring dims: from the lanes' own places
// a store would be 64 pieces of 8 bytes (8 x 1024 rows, 32 heads, 67 MB: 113.0
// and 110.4 us, 8 of 1376 to 553 rows 144.4 and 134.3). w(cb, r) are dims
// cb * 32 + crow(r, hi1) on of this lane's row; `rows` of the 32 are there.
template <int D, class W>
FI_DEV void put_rows(unsigned char* smem, int at, u16* out, int64_t stride,
                     int rows, int lane, const W& w) {
  using R = RowSoftmax<D>;
  if (R::kFew) asm volatile("" : "+v"(lane));
  const int col = lane & 31, hi1 = lane >> 5;
  // 16-byte chunk c of row r sits at c ^ r
  const int put = at + col * R::kRowB + (col & (R::kChunk - 1)) * 16 + hi1 * 8;
#pragma unroll
  for (int cb = 0; cb < R::CB; ++cb)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<bf16x4*>(smem + (put ^ ((cb * 4 + r / 4) * 16))) =
          w(cb, r);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  const bool wide = reinterpret_cast<uintptr_t>(out) % 16 == 0;
  const int r0 = lane / R::kChunk, ch = lane % R::kChunk;
  const int get = at + r0 * R::kRowB + (ch ^ r0) * 16;
  u16* to = out + r0 * stride + ch * 8;
  auto store = [&](bool all) {
#pragma unroll
    for (int i = 0; i < 32 / R::kRowsPerDma; ++i) {
      const int r = i * R::kRowsPerDma;
      if (all || r + r0 < rows) {
        const uint4 v = *reinterpret_cast<const uint4*>(
            smem + (get ^ (r & (R::kChunk - 1)) * 16) + r * R::kRowB);
        if (all || wide) {
          store_global(to, v);
        } else {                       // rows off the 16-byte grid
          store_global(to, make_uint2(v.x, v.y));
          store_global(to + 4, make_uint2(v.z, v.w));
        }
      }
      to += R::kRowsPerDma * stride;
      if (R::kFew) asm volatile("" : "+v"(to));
    }
  };
  if (wide && rows >= 32) store(true);
  else store(false);
}

// The split form.
template <int D, bool PAGED, bool FP8>
__global__ __launch_bounds__(attn_waves(true) * kWaveSize, 2)
void prefill_attn_kernel(const PrefillArgs p) {
  using R = RowSoftmax<D>;
  constexpr int kWaves = attn_waves(true), kBufs = 3;
  constexpr int KF = R::KF, CB = R::CB, kRowB = R::kRowB, kChunk = R::kChunk;
  constexpr int kTileB = R::kTileB, kRowsPerDma = R::kRowsPerDma;
  constexpr int kWRows = kKVTile / kWaves;   // rows a wave copies
  constexpr int kDma = kWRows / kRowsPerDma;  // DMAs per wave and matrix

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

  RowSoftmax<D> row(lane, p.scale);
  const float sgn = sign_of(p.scale);

  int hg = 0, qt = 0, from = 0;
  // (head group, query tile, slot behind the last piece's, 0) of the
  // tile that begins in this part and is cut by its end; -1: none
  int4 cut = make_int4(0, -1, 0, 0);
  const int u = total_work<PAGED>(p, lane);
  const int64_t total = static_cast<int64_t>(u) * (p.num_q_heads / p.hpb);
  const int slot = split_slot(blockIdx.x, p.slots);
  const Parts parts(total, p.slots);
  int64_t pos = parts.begin(slot);
  const int64_t pos_end = parts.begin(slot + 1);
  if (pos < pos_end) {
    hg = static_cast<int>(pos / u);
    qt = find_tile<PAGED>(p, lane, static_cast<int>(pos - int64_t(hg) * u),
                          &from);
  }
  // the tile at the end: the part itself or a later one finishes it
  if (pos < pos_end && pos_end < total) {
    const int h = static_cast<int>(pos_end / u);
    int within;
    const int i = find_tile<PAGED>(
        p, lane, static_cast<int>(pos_end - int64_t(h) * u), &within);
    if (within > 0 && pos_end - within >= pos) {
      const int64_t end = pos_end - within + q_tile<PAGED>(p, i).work;
      cut = make_int4(h, i, slot + 1, 0);
      while (cut.z < p.slots && parts.begin(cut.z) < end) ++cut.z;
    }
  }
  if (tid == 0) p.cut[slot] = cut;

  while (pos < pos_end) {
    const QTile t = uniform_tile(q_tile<PAGED>(p, qt));
    if (t.work == 0) {                 // rows past the sequence's end
      if (++qt == p.nq) { qt = 0; ++hg; }
      continue;
    }
    const int ta = from;
    const int tb = static_cast<int>(
        min(static_cast<int64_t>(t.work), from + (pos_end - pos)));
    const int head = hg * p.hpb + wave / wph;
    const int kv_head = hg * p.hpb / (p.num_q_heads / p.num_kv_heads);
    const int ctx_start = t.k_len - t.seq_len;
    const int row0 = t.row0 + (wave % wph) * 32;
    const bool active = row0 < t.seq_len;
    const int last_blk = (t.k_len - 1) >> 4;
    const ConstInts bt_row = const_ints(
        PAGED ? p.block_tables + static_cast<int64_t>(t.seq) * p.max_blocks
              : nullptr);

    // ---- staging ---------------------------------------------------------
    // wave w copies rows 8w..8w+7 of a tile: half a cache block. Rows past
    // the end repeat the last one (finite values; their scores are masked).
    auto block_of = [&](int tile) {
      return bt_row[min(tile * 4 + wave * kWRows / 16, last_blk)];
    };
    auto stage_dma = [&](int tile, int blk, int buf) {
      const u32 kdst = lds0 + buf * kTileB + wave * kWRows * kRowB;
      const u32 vdst = kdst + kBufs * kTileB;
      const u16* kb;
      const u16* vb;
      int first, limit;                // row of the wave, last valid row
      int64_t ks, vs;
      if (PAGED) {
        const int64_t base =
            (static_cast<int64_t>(blk) * p.num_kv_heads + kv_head) * 16 * D;
        kb = static_cast<const u16*>(p.k) + base;
        vb = static_cast<const u16*>(p.v) + base;
        const int b = min(tile * 4 + wave * kWRows / 16, last_blk);
        first = wave * kWRows & 15;
        limit = t.k_len - 1 - b * 16;
        ks = vs = D;
      } else {
        const int r0 = min(tile * kKVTile, t.k_len - 1);
        kb = static_cast<const u16*>(p.k) +
             (t.seq_start + r0) * p.k_stride + int64_t(kv_head) * D;
        vb = static_cast<const u16*>(p.v) +
             (t.seq_start + r0) * p.v_stride + int64_t(kv_head) * D;
        first = wave * kWRows;
        limit = t.k_len - 1 - r0;
        ks = p.k_stride;
        vs = p.v_stride;
      }
      if (PAGED && limit >= first + kWRows - 1) {  // no row past the end
        const int r0 = first + lane / kChunk;
        const u32 ko = r0 * kRowB + ((lane % kChunk) ^ R::k_swz(r0)) * 16;
        const u32 vo = r0 * kRowB + ((lane % kChunk) ^ R::v_swz(r0)) * 16;
#pragma unroll
        for (int i = 0; i < kDma; ++i) {
          dma_to_lds16(kdst + i * 1024, kb, ko ^ (i * (1024 + 64)));
          dma_to_lds16(vdst + i * 1024, vb, vo ^ (i * 1024));
        }
        return;
      }
#pragma unroll
      for (int i = 0; i < kDma; ++i) {
        const int r = i * kRowsPerDma + lane / kChunk;  // row of the wave
        const int tr = wave * kWRows + r;                    // row of the tile
        const int src = min(first + r, limit);
        const u32 ko = static_cast<u32>(
            src * static_cast<int>(ks) * 2 +
            (((lane % kChunk) ^ R::k_swz(tr)) * 16));
        const u32 vo = static_cast<u32>(
            src * static_cast<int>(vs) * 2 +
            (((lane % kChunk) ^ R::v_swz(tr)) * 16));
        dma_to_lds16(kdst + i * 1024, kb, ko);
        dma_to_lds16(vdst + i * 1024, vb, vo);
      }
    };
    // fp8: a thread owns 16 dims of one row of K and of V
    constexpr int kParts = D / 16;
    constexpr int kStep = kWaves * kWaveSize / kParts;  // rows per step
    constexpr int kSteps = ceil_div(kKVTile, kStep);
    const int f_row0 = tid / kParts, f_part = tid % kParts;
    const bool f_own = kStep <= kKVTile || f_row0 < kKVTile;
    uint4 k_raw[kSteps], v_raw[kSteps];
    auto load_fp8 = [&](int tile) {
      if (!f_own) return;
#pragma unroll
      for (int i = 0; i < kSteps; ++i) {
        const int src = min(tile * kKVTile + f_row0 + i * kStep, t.k_len - 1);
        const int64_t off =
            ((static_cast<int64_t>(bt_row[src >> 4]) * p.num_kv_heads +
              kv_head) * 16 + (src & 15)) * D + f_part * 16;
        k_raw[i] = *reinterpret_cast<const uint4*>(
            static_cast<const unsigned char*>(p.k) + off);
        v_raw[i] = *reinterpret_cast<const uint4*>(
            static_cast<const unsigned char*>(p.v) + off);
      }
    };
    auto write_fp8 = [&](int buf) {
      if (!f_own) return;
      auto put = [&](unsigned char* dst, const uint4& raw, int f_row,
                     int swz) {
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

    // the previous query tile's LDS reads are over in every wave
    __builtin_amdgcn_s_barrier();
    int blk = 0;
    if (FP8) {
      load_fp8(ta);
      write_fp8(0);
      if (ta + 1 < tb) load_fp8(ta + 1);
    } else {
      stage_dma(ta, PAGED ? block_of(ta) : 0, 0);
      if (ta + 1 < tb) stage_dma(ta + 1, PAGED ? block_of(ta + 1) : 0, 1);
      if (PAGED) blk = block_of(ta + kBufs - 1);
    }

    // ---- query fragments (B operand of S^T): lane holds
    // Q[row0+col][f*16 + hi1*8 .. +8]
    short8 b_q[KF];
    if (active) {
      const int qr = min(row0 + col, t.seq_len - 1);
      const u16* qrow = p.q + (t.seq_start + qr) * p.q_stride +
                        static_cast<int64_t>(head) * D;
#pragma unroll
      for (int f = 0; f < KF; ++f)
        b_q[f] = *reinterpret_cast<const short8*>(qrow + f * 16 + hi1 * 8);
      turn_queries(b_q, sgn);
      // arrived here, not at their first use: that is inside the loop,
      // where the wait would take in the DMAs of every tile
#pragma unroll
      for (int f = 0; f < KF; ++f) asm volatile("" : "+v"(b_q[f]));
    }

    row.clear();
    const int my_q_max = ctx_start + min(row0 + 32, t.seq_len) - 1;
    const int q_pos = ctx_start + row0 + col;
    int buf = 0;
    for (int tile = ta; tile < tb; ++tile) {
      const int kv0 = tile * kKVTile;
      // this tile has landed (this wave's part; the barrier covers the
      // others'), and nobody reads the buffer that is filled next
      if (!FP8) {
        if (tile + 1 < tb)
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kDma) : "memory");
        else
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      const int buf1 = buf == kBufs - 1 ? 0 : buf + 1;
      if (FP8) {
        if (tile + 1 < tb) write_fp8(buf1);
        if (tile + 2 < tb) load_fp8(tile + 2);
      } else if (tile + kBufs - 1 < tb) {
        stage_dma(tile + kBufs - 1, blk, buf1 == kBufs - 1 ? 0 : buf1 + 1);
        if (PAGED) blk = block_of(tile + kBufs);
      }

      if (active && kv0 <= my_q_max) {
        floatx16 s_acc[2];
        row.scores(smem, buf * kTileB, (kBufs + buf) * kTileB, b_q, s_acc);
        // only tiles at the diagonal or the end mask
        if (kv0 + kKVTile - 1 > ctx_start + row0) {
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r)
              if (kv0 + 32 * b + crow(r, hi1) > q_pos)
                s_acc[b][r] = -INFINITY;
        }
        row.add(smem, (kBufs + buf) * kTileB, s_acc);
      }
      buf = buf1;
    }

    // ---- epilogue ----
    row.l_row += half_swap(row.l_row);
    if (ta == 0 && tb == t.work) {
      // turned over in the buffers that nobody reads or fills any more
      constexpr int kHalves = kTileB / (32 * kRowB);   // waves per buffer
      const int free_buf = (buf + wave / kHalves % (kBufs - 1)) % kBufs;
      const int mine =
          (wave / kHalves / (kBufs - 1) * kBufs + free_buf) * kTileB +
          wave % kHalves * 32 * kRowB;
      const float inv = row.l_row > 0.f ? 1.f / row.l_row : 0.f;
      if (active)
        put_rows<D>(smem, mine,
                    p.out + (static_cast<int64_t>(t.seq_start + row0) *
                                 p.num_q_heads + head) * D,
                    static_cast<int64_t>(p.num_q_heads) * D,
                    t.seq_len - row0, lane, [&](int cb, int r) {
                      bf16x4 w;
#pragma unroll
                      for (int j = 0; j < 4; ++j)
                        w.h[j] = f32_to_bf16(row.o_acc[cb][r + j] * inv);
                      return w;
                    });
    } else {
      const int piece = slot * 2 + (ta > 0 ? 0 : 1);
      float* o = p.piece_o + (static_cast<int64_t>(piece) * kWaves + wave) *
                                 32 * D + lane;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[(cb * 16 + r) * 64] = row.o_acc[cb][r];
      float2* ml = reinterpret_cast<float2*>(p.piece_ml) +
                   (static_cast<int64_t>(piece) * kWaves + wave) * 64 + lane;
      *ml = make_float2(row.m_row, row.l_row);
    }
    pos += tb - ta;
    from = 0;
    if (++qt == p.nq) { qt = 0; ++hg; }
  }
}

}  // namespace fi
