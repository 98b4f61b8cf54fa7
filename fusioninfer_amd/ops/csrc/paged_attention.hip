// Paged-attention DECODE for CDNA4 (gfx950): one query row per sequence
// against the paged KV cache ([num_blocks, Hk, 16, D], bf16 or e4m3).
// Memory-bound: every sequence's K and V are read once, each read serves the
// G query heads of a K/V head.
//
// All (sequence, K/V head) contexts form one line of steps (16 * PP tokens);
// up to 1024 waves, four per CU, take equal parts of it, so ragged and few
// long contexts load the chip as evenly as many equal ones, and the launch
// shape does not depend on the lengths (hipGraph replay). A wave streams its
// part through a private ring in LDS by DMA, three steps ahead: 96 KB in
// flight per CU, no barrier anywhere. The next context's queries arrive
// through the same queue, so the ring runs on over the borders of contexts.
// A context that is cut leaves unnormalised fp32 pieces; a second kernel
// adds them up.
//
// Per step, with heads as MFMA columns (16, of which G count):
//   S[token, head] = K Q^T            mfma 16x16x32, A = K rows from LDS
//   O^T[dim, head] += V^T P^T         A = V through the transposing LDS
//                                     read, B = P as the scores' registers
//                                     already hold it (the order of the
//                                     tokens within a step is theirs), in
//                                     three bf16 terms that are the fp32 P
// A lane keeps one head's statistics; e4m3 rows are converted exactly after
// the LDS read. 96 KB in flight and some hundred cycles of work per 8 KB
// step leave memory as the bound of long contexts. P in one bf16 term is 0.4
// us less for one of 301 tokens, 1 to 2 % of the bf16 contexts below and 2 us
// of the e4m3 ones; its weights have 8 bits where the sum they are divided by
// has 24.
// Where a context is cut depends on the lengths of all contexts of the
// launch, and so do the last bits of the fp32 sums: a row of one batch can
// differ by a bf16 rounding from the same row among other neighbours.
//
// Measured at 32 query heads, D 128, both kernels, us (TB/s of K/V), before
// -> now: 256 contexts of 1024-1279 tokens, 8 K/V heads 278 (4.3) -> 212
// (5.7); 6 of 20-32 thousand 168 (3.9) -> 110 (6.0); 13 of 70-4100 42 -> 26;
// 64 of 512-2048 e4m3 101 (1.6) -> 36 (4.4), with 4 K/V heads bf16 58 (2.7)
// -> 36 (4.4); one of 301 12.0 -> 10.5, one of 8000 19.5 -> 15.4.
//
// Capability parity: the paged-attention decode the reference delegates to
// its vLLM containers.

#include "common.h"

#include <type_traits>

namespace fi {

namespace {

typedef __attribute__((ext_vector_type(4))) short short4v;
typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) float floatx4;

constexpr int kPage = 16;        // tokens of a cache block
constexpr int kDecWaves = 4;     // waves of a workgroup
constexpr int kDecSlots = 1024;  // parts of the line
constexpr int kRing = 4;         // steps of a wave's ring
constexpr int kMaxGroup = 8;
constexpr int kMinPages = 4;     // a part is no shorter than this
constexpr float kNegInf = -1e30f;
// see the prefill kernel: rescale only when the maximum grows by more than
// this (base-2 units)
constexpr float kDeferThr = 11.5416f;

struct DecodeArgs {
  u16* out;                 // [S, Hq, D]
  const u16* q;             // [S] rows, stride q_stride, Hq * D values
  const unsigned char* k;   // cache bytes
  const unsigned char* v;
  const int* block_tables;  // [S, max_blocks]
  const int* seq_lens;      // [S]
  float* piece_o;           // [slots][2][G][D]
  float* piece_ml;          // [slots][2][G][2]
  int2* cut;                // [S][Hk] parts [first, behind) of a cut
                            // context; first -1: it was not cut
  int64_t q_stride;
  int num_seqs, max_blocks, num_kv_heads, group;
  float scale;
};

template <int PP>
FI_DEV int steps_of(int ctx) {
  return (max(ctx, 1) + kPage * PP - 1) / (kPage * PP);
}

struct Place {
  int seq, head, step;
};

// The line: sequences in order, of each its K/V heads, of each its steps.
// The first 64 sequences' steps and their running sum stay in the lanes.
template <int PP>
struct Line {
  int n, incl, lane;
  int64_t total;  // steps of all

  FI_DEV void chunk(const DecodeArgs& p, int i0, int* n_, int* incl_) const {
    const int i = i0 + lane;
    int x = i < p.num_seqs ? steps_of<PP>(p.seq_lens[i]) : 0;
    *n_ = x;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(x, off, 64);
      if (lane >= off) x += o;
    }
    *incl_ = x;
  }

  FI_DEV Line(const DecodeArgs& p, int lane_) : lane(lane_) {
    chunk(p, 0, &n, &incl);
    int sum = 0;
#pragma unroll 4
    for (int i = kWaveSize + lane; i < p.num_seqs; i += kWaveSize)
      sum += steps_of<PP>(p.seq_lens[i]);
    if (p.num_seqs > kWaveSize) {
#pragma unroll
      for (int off = 32; off; off >>= 1) sum += __shfl_xor(sum, off, 64);
    }
    total = static_cast<int64_t>(__builtin_amdgcn_readfirstlane(
                sum + __shfl(incl, 63, 64))) * p.num_kv_heads;
  }

  FI_DEV Place find(const DecodeArgs& p, int64_t at) const {
    const int hk = p.num_kv_heads;
    int64_t before = 0;
    int cn = n, ci = incl;
    for (int i0 = 0;;) {
      const unsigned long long hit =
          __ballot(before + static_cast<int64_t>(ci) * hk > at);
      if (hit) {
        const int l = __builtin_ctzll(hit);
        const int nl = __builtin_amdgcn_readfirstlane(__shfl(cn, l, 64));
        const int in =
            static_cast<int>(at - before) -
            (__builtin_amdgcn_readfirstlane(__shfl(ci, l, 64)) - nl) * hk;
        return {i0 + l, in / nl, in % nl};
      }
      before += static_cast<int64_t>(
          __builtin_amdgcn_readfirstlane(__shfl(ci, 63, 64))) * hk;
      i0 += kWaveSize;
      if (i0 >= p.num_seqs) return {p.num_seqs - 1, hk - 1, 0};  // not reached
      chunk(p, i0, &cn, &ci);
    }
  }
};

// part s of the line is [begin(s), begin(s + 1))
struct Parts {
  int64_t each, total;
  FI_DEV Parts(int64_t t, int min_each)
      : each(max((t + kDecSlots - 1) / kDecSlots,
                 static_cast<int64_t>(min_each))),
        total(t) {}
  FI_DEV int64_t begin(int s) const { return min(s * each, total); }
};

// value of the lane with the other 16 (32) bit
FI_DEV float swap16(float x) {
  const auto s = __builtin_amdgcn_permlane16_swap(
      __float_as_int(x), __float_as_int(x), false, false);
  return __int_as_float((threadIdx.x & 16) ? s[0] : s[1]);
}
FI_DEV float swap32(float x) {
  const auto s = __builtin_amdgcn_permlane32_swap(
      __float_as_int(x), __float_as_int(x), false, false);
  return __int_as_float((threadIdx.x & 32) ? s[0] : s[1]);
}

// eight e4m3 bytes to bf16, exact
FI_DEV short8 fp8_to_bf16(uint2 w) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((ext_vector_type(2))) __bf16 bf2;
  typedef __attribute__((ext_vector_type(4))) u32 u4;
  u4 o;
  o.x = __builtin_bit_cast(
      u32, bf2(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.x, 1.f, false)));
  o.y = __builtin_bit_cast(
      u32, bf2(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.x, 1.f, true)));
  o.z = __builtin_bit_cast(
      u32, bf2(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.y, 1.f, false)));
  o.w = __builtin_bit_cast(
      u32, bf2(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w.y, 1.f, true)));
  return __builtin_bit_cast(short8, o);
#else
  return short8{};
#endif
}

// Transposing LDS read of bytes: within 16 lanes, lane 2i+j points at
// entries 8j..8j+7 of row i of an 8 x 16 block and receives the eight rows'
// entries of column (lane & 15).
FI_DEV uint2 lds_read_tr8(const unsigned char* p) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((ext_vector_type(2))) int i2;
  const i2 r = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
      (__attribute__((address_space(3))) i2*)(p));
  return make_uint2(r.x, r.y);
#else
  return make_uint2(0, 0);
#endif
}

template <int D, bool FP8>
struct DecShape {
  static constexpr int kRowB = D * (FP8 ? 1 : 2);
  // pages of a step: 8 KB of K and V together (4 KB for the smallest rows)
  static constexpr int PP = kRowB == 256 ? 1 : 2;
  static_assert(!FP8 || PP == 2, "byte transposes take two pages");
};

template <int D, bool FP8>
__global__ __launch_bounds__(kDecWaves * kWaveSize)
void paged_attn_decode_kernel(const DecodeArgs p) {
  constexpr int kRowB = DecShape<D, FP8>::kRowB, PP = DecShape<D, FP8>::PP;
  constexpr int KK = D / 32, DT = D / 16;
  constexpr int kChunk = kRowB / 16;           // 16-byte chunks of a row
  constexpr int kRowsDma = 1024 / kRowB;       // rows of a DMA
  constexpr int kPageDma = kPage / kRowsDma;   // DMAs of a page
  constexpr int kMatB = PP * kPage * kRowB;    // K (or V) bytes of a step
  constexpr int kLoads = 2 * PP * kPageDma;    // DMAs of a step
  constexpr int kQB = kMaxGroup * D * 2;       // a context's queries
  constexpr int kWaveB = kRing * (2 * kMatB + kQB);
  static_assert(kDecWaves * kWaveB <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(1024)))
  unsigned char smem[kDecWaves * kWaveB];

  const int lane = threadIdx.x % kWaveSize;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  const int slot = blockIdx.x * kDecWaves + wave;
  unsigned char* ring = smem + wave * kWaveB;
  unsigned char* qring = ring + kRing * 2 * kMatB;
  const u32 ring_lds = static_cast<u32>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) unsigned char*)ring));
  const u32 q_lds = ring_lds + kRing * 2 * kMatB;
  const int G = p.group, hk = p.num_kv_heads;

  const Line<PP> line(p, lane);
  const Parts parts(line.total, kMinPages / PP);
  const int64_t lo = parts.begin(slot), hi = parts.begin(slot + 1);
  if (lo >= hi) return;

  // ---- producer ----
  auto k_swz = [](int row) {
    return kRowB == 256 ? row & 15
                        : (kRowB == 128 ? (row >> 1) & 7 : (row >> 2) & 3);
  };
  auto v_swz = [](int row) {
    return FP8 ? (kRowB == 128 ? (row >> 1) & 7 : (row >> 2) & 3)
               : (kRowB == 256 ? (row & 7) << 1 : ((row >> 1) & 3) << 1);
  };
  const ConstInts lens = const_ints(p.seq_lens);
  const ConstInts tables = const_ints(p.block_tables);
  const Place first = line.find(p, lo);
  const int total = static_cast<int>(hi - lo);
  struct Cursor {
    int seq, head, step, ctx, steps;
  };
  auto at_seq = [&](int seq, int head, int step) {
    Cursor c;
    c.seq = __builtin_amdgcn_readfirstlane(seq);
    c.head = __builtin_amdgcn_readfirstlane(head);
    c.step = __builtin_amdgcn_readfirstlane(step);
    c.ctx = max(lens[c.seq], 1);
    c.steps = steps_of<PP>(c.ctx);
    return c;
  };
  auto next_context = [&](const Cursor& c) {
    if (c.head + 1 < hk) {
      Cursor n = c;
      n.head = c.head + 1;
      n.step = 0;
      return n;
    }
    return at_seq(c.seq + 1, 0, 0);
  };
  Cursor in = at_seq(first.seq, first.head, first.step);
  int page[PP], in_slot = 0, in_q = 0, issued = 0;
  auto load_pages = [&] {
#pragma unroll
    for (int i = 0; i < PP; ++i)
      page[i] = tables[static_cast<int64_t>(in.seq) * p.max_blocks +
                       min(in.step * PP + i, (in.ctx - 1) / kPage)];
  };
  auto request_q = [&] {
    const u16* src = p.q + in.seq * p.q_stride +
                     static_cast<int64_t>(in.head) * G * D;
    for (int b = 0; b < G * D * 2; b += 1024)
      dma_to_lds16(q_lds + in_q * kQB + b, src,
                   min(b + lane * 16, G * D * 2 - 16));
  };
  auto request = [&] {
    const u32 dst = ring_lds + in_slot * 2 * kMatB;
#pragma unroll
    for (int i = 0; i < PP; ++i) {
      const int64_t base =
          (static_cast<int64_t>(page[i]) * hk + in.head) * (kPage * kRowB);
      // rows behind the context's end repeat its last one (finite values,
      // masked scores)
      const int limit =
          in.ctx - 1 - min(in.step * PP + i, (in.ctx - 1) / kPage) * kPage;
#pragma unroll
      for (int j = 0; j < kPageDma; ++j) {
        const int r = j * kRowsDma + lane / kChunk;  // of the page
        const int sr = i * kPage + r;                // of the step
        const u32 row = min(r, limit) * kRowB;
        const u32 at = (i * kPage + j * kRowsDma) * kRowB;
        dma_to_lds16_nt(dst + at, p.k + base,
                        row + ((lane % kChunk) ^ k_swz(sr)) * 16);
        dma_to_lds16_nt(dst + kMatB + at, p.v + base,
                        row + ((lane % kChunk) ^ v_swz(sr)) * 16);
      }
    }
    ++issued;
    if (++in_slot == kRing) in_slot = 0;
    if (issued == total) return;
    if (++in.step == in.steps) {
      in = next_context(in);
      if (++in_q == kRing) in_q = 0;
      load_pages();
      request_q();
    } else {
      load_pages();
    }
  };
  load_pages();
  request_q();
  for (int i = 0; i < kRing - 1; ++i)
    if (issued < total) request();

  // ---- consumer ----
  const int tok = lane & 15, g = lane >> 4;  // also: head column, quarter
  int k_off[KK], v_off[DT];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk)
    k_off[kk] = FP8
        ? tok * kRowB + (((kk * 2 + (g >> 1)) ^ k_swz(tok)) * 16) +
              (g & 1) * 8
        : tok * kRowB + (((kk * 4 + g) ^ k_swz(tok)) * 16);
  {
    // row this lane points at: tokens 4g.. of a page; bytes: of both pages
    const int r = FP8 ? (tok >> 1) : (tok >> 2);
    const int row = FP8 ? (r >> 2) * kPage + 4 * g + (r & 3) : 4 * g + r;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      v_off[dt] = FP8
          ? row * kRowB + ((dt ^ v_swz(row)) * 16) + (tok & 1) * 8
          : row * kRowB + (((dt * 2 + ((tok & 3) >> 1)) ^ v_swz(row)) * 16) +
                (tok & 1) * 8;
  }
  const float sgn = p.scale > 0.f ? 1.f : (p.scale < 0.f ? -1.f : 0.f);
  const float c = p.scale == 0.f
      ? 1.f : fabsf(p.scale) * 1.4426950408889634f;  // log2(e)

  Cursor at = at_seq(first.seq, first.head, first.step);
  int ring_slot = 0, q_slot = 0, done = 0;
  while (done < total) {
    const int n = min(at.steps - at.step, total - done);
    const bool begins = at.step == 0, ends = at.step + n == at.steps;
    short8 b_q[KK];
    float m_row = kNegInf, l_row = 0.f;
    floatx4 o_acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o_acc[dt] = {0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < n; ++i, ++done) {
      // everything up to this step has landed, queries included: newer
      // requests are at most those of the steps behind it
      if (issued - done >= kRing - 1)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kRing - 2) * kLoads)
                     : "memory");
      else if (issued - done == 2)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (i == 0) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          b_q[kk] = *reinterpret_cast<const short8*>(
              qring + q_slot * kQB + min(tok, G - 1) * (D * 2) +
              (kk * 4 + g) * 16);
          if (sgn != 1.f) {
            bf16x8 h = __builtin_bit_cast(bf16x8, b_q[kk]);
#pragma unroll
            for (int j = 0; j < 8; ++j)
              h.h[j] = f32_to_bf16(bf16_to_f32(h.h[j]) * sgn);
            b_q[kk] = __builtin_bit_cast(short8, h);
          }
        }
        // read before the slot is requested again
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
      if (issued < total) request();

      const unsigned char* kb = ring + ring_slot * 2 * kMatB;
      const unsigned char* vb = kb + kMatB;
      floatx4 s[PP];
#pragma unroll
      for (int pg = 0; pg < PP; ++pg) {
        s[pg] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          const unsigned char* a = kb + pg * kPage * kRowB + k_off[kk];
          const short8 a_k = FP8
              ? fp8_to_bf16(*reinterpret_cast<const uint2*>(a))
              : *reinterpret_cast<const short8*>(a);
          s[pg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_k, b_q[kk],
                                                          s[pg], 0, 0, 0);
        }
      }
      if (at.step == at.steps - 1) {
        const int t0 = at.step * PP * kPage + 4 * g;
#pragma unroll
        for (int pg = 0; pg < PP; ++pg)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (t0 + pg * kPage + r >= at.ctx) s[pg][r] = -INFINITY;
      }
      float rm = s[0][0];
#pragma unroll
      for (int pg = 0; pg < PP; ++pg)
#pragma unroll
        for (int r = 0; r < 4; ++r) rm = fmaxf(rm, s[pg][r]);
      rm = fmaxf(rm, swap16(rm));
      rm = fmaxf(rm, swap32(rm));
      if (!__all((rm - m_row) * c <= kDeferThr)) {
        const float m_new = fmaxf(m_row, rm);
        const float alpha = __builtin_amdgcn_exp2f((m_row - m_new) * c);
        m_row = m_new;
        l_row *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int r = 0; r < 4; ++r) o_acc[dt][r] *= alpha;
      }
      const float mc = m_row * c;
      short4v pb[3][PP];       // the weights' terms, per page
#pragma unroll
      for (int pg = 0; pg < PP; ++pg)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float e =
              __builtin_amdgcn_exp2f(fmaf(s[pg][r], c, -mc));
          l_row += e;
          u16 terms[3];
          split_weight(e, terms);
#pragma unroll
          for (int x = 0; x < 3; ++x)
            pb[x][pg][r] = static_cast<short>(terms[x]);
        }
      // term by term over all columns, so that no product waits for the one
      // before it; a single page's first two terms share a 32-deep product
      short8 a_v[DT];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        if constexpr (FP8) {
          a_v[dt] = fp8_to_bf16(lds_read_tr8(vb + v_off[dt]));
        } else {
          const short4v x = lds_read_tr4(vb + v_off[dt]);
          const short4v y = PP == 1
              ? x : lds_read_tr4(vb + v_off[dt] + kPage * kRowB);
          a_v[dt] = short8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
        }
      }
#pragma unroll
      for (int x = 0; x < (PP == 1 ? 1 : 3); ++x) {
        const short4v u = pb[x][0], v = PP == 1 ? pb[1][0] : pb[x][PP - 1];
        const short8 b = {u[0], u[1], u[2], u[3], v[0], v[1], v[2], v[3]};
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          o_acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a_v[dt], b, o_acc[dt], 0, 0, 0);
      }
      if (PP == 1) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          o_acc[dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
              short4v{a_v[dt][0], a_v[dt][1], a_v[dt][2], a_v[dt][3]},
              pb[2][0], o_acc[dt], 0, 0, 0);
      }
      if (++ring_slot == kRing) ring_slot = 0;
      ++at.step;
    }

    // ---- this context (or this part of it) is done; column = head,
    // register r of tile dt = dim 16 dt + 4 g + r
    l_row += swap16(l_row);
    l_row += swap32(l_row);
    if (begins && lane == 0) {
      const int64_t end = lo + done - n + at.steps;
      p.cut[at.seq * hk + at.head] = ends
          ? make_int2(-1, 0)
          : make_int2(slot, static_cast<int>((end + parts.each - 1) /
                                             parts.each));
    }
    if (tok < G) {
      if (begins && ends) {
        const float inv = 1.f / l_row;
        u16* o = p.out +
                 (static_cast<int64_t>(at.seq) * hk * G + at.head * G + tok) *
                     D + 4 * g;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          bf16x4 w;
#pragma unroll
          for (int r = 0; r < 4; ++r) w.h[r] = f32_to_bf16(o_acc[dt][r] * inv);
          *reinterpret_cast<bf16x4*>(o + dt * 16) = w;
        }
      } else {
        const int64_t piece =
            static_cast<int64_t>(slot * 2 + (begins ? 1 : 0)) * G + tok;
        float* o = p.piece_o + piece * D + 4 * g;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          *reinterpret_cast<floatx4*>(o + dt * 16) = o_acc[dt];
        if (g == 0) {
          p.piece_ml[piece * 2] = m_row;
          p.piece_ml[piece * 2 + 1] = l_row;
        }
      }
    }
    if (done < total) {
      at = next_context(at);
      if (++q_slot == kRing) q_slot = 0;
    }
  }
}

// Adds up a cut context's pieces. A block takes a context, or, where there
// are few, one query head of it; its waves share the pieces, a long
// context's are loaded sixteen at a time.
constexpr int kJoinWaves = 8;

template <int D>
__global__ __launch_bounds__(kJoinWaves * kWaveSize)
void paged_attn_join_kernel(const DecodeArgs p, const int heads) {
  constexpr int V = D / 64;
  __shared__ float part[kJoinWaves][D + 2];
  const int blocks = p.group / heads;   // of a context
  const int context = blockIdx.x / blocks;
  const int2 cut = p.cut[context];
  if (cut.x < 0) return;
  const int lane = threadIdx.x % kWaveSize, G = p.group;
  const int wave = threadIdx.x / kWaveSize;
  const int sub = wave / heads, subs = kJoinWaves / heads;
  const int h = (blockIdx.x % blocks) * heads + wave % heads;
  const int first = cut.x;
  const float c = p.scale == 0.f
      ? 1.f : fabsf(p.scale) * 1.4426950408889634f;
  float m = kNegInf, l = 0.f, o[V];
#pragma unroll
  for (int j = 0; j < V; ++j) o[j] = 0.f;
  // `count` pieces from s0 on, loads first; where there are fewer the first
  // again, as zeros (it may hold infinities) of weight 0
  auto add = [&](int s0, auto count) {
    constexpr int N = decltype(count)::value;
    float pm[N], pl[N], x[N][V];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int s = s0 + i * subs;
      const bool there = s < cut.y;
      const int64_t piece = static_cast<int64_t>(
          s == first || !there ? first * 2 + 1 : s * 2) * G + h;
      pm[i] = p.piece_ml[piece * 2];
      pl[i] = p.piece_ml[piece * 2 + 1];
      if (!there) {
        pm[i] = kNegInf;
        pl[i] = 0.f;
      }
#pragma unroll
      for (int j = 0; j < V; ++j) {
        x[i][j] = p.piece_o[piece * D + lane * V + j];
        if (!there) x[i][j] = 0.f;
      }
    }
    float mx = m;
#pragma unroll
    for (int i = 0; i < N; ++i) mx = fmaxf(mx, pm[i]);
    const float a = __builtin_amdgcn_exp2f((m - mx) * c);
    m = mx;
    l *= a;
#pragma unroll
    for (int j = 0; j < V; ++j) o[j] *= a;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float b = __builtin_amdgcn_exp2f((pm[i] - mx) * c);
      l = fmaf(pl[i], b, l);
#pragma unroll
      for (int j = 0; j < V; ++j) o[j] = fmaf(x[i][j], b, o[j]);
    }
  };
  int s0 = first + sub;
  for (; s0 + 3 * subs < cut.y; s0 += 16 * subs)
    add(s0, std::integral_constant<int, 16>());
  for (; s0 < cut.y; s0 += 2 * subs)
    add(s0, std::integral_constant<int, 2>());
  if (lane == 0) {
    part[wave][D] = m;
    part[wave][D + 1] = l;
  }
#pragma unroll
  for (int j = 0; j < V; ++j) part[wave][lane * V + j] = o[j];
  __syncthreads();
  if (sub) return;
  float mx = kNegInf;
  for (int i = 0; i < subs; ++i) mx = fmaxf(mx, part[i * heads + wave % heads][D]);
  l = 0.f;
#pragma unroll
  for (int j = 0; j < V; ++j) o[j] = 0.f;
  for (int i = 0; i < subs; ++i) {
    const float b = __builtin_amdgcn_exp2f((part[i * heads + wave % heads][D] - mx) * c);
    l = fmaf(part[i * heads + wave % heads][D + 1], b, l);
#pragma unroll
    for (int j = 0; j < V; ++j)
      o[j] = fmaf(part[i * heads + wave % heads][lane * V + j], b, o[j]);
  }
  const float inv = 1.f / l;
  u16* row = p.out + (static_cast<int64_t>(context) * G + h) * D + lane * V;
#pragma unroll
  for (int j = 0; j < V; ++j) row[j] = f32_to_bf16(o[j] * inv);
}

}  // namespace

bool decode_attn_supported(int head_dim, int group) {
  return (head_dim == 128 || head_dim == 64) &&
         (group == 1 || group == 2 || group == 4 || group == 8);
}

int64_t decode_piece_floats(int num_seqs, int num_kv_heads, int head_dim,
                            int group) {
  return static_cast<int64_t>(kDecSlots) * 2 * group * (head_dim + 2) +
         2 * static_cast<int64_t>(num_seqs) * num_kv_heads;
}

void launch_paged_attn_decode(u16* out, const u16* q, const void* k_cache,
                              const void* v_cache, const int* block_tables,
                              const int* seq_lens, int num_seqs,
                              int64_t q_stride, int max_blocks,
                              int num_kv_heads, int head_dim, int group,
                              float scale, bool fp8, float* pieces,
                              hipStream_t stream) {
  DecodeArgs a;
  a.out = out;
  a.q = q;
  a.k = static_cast<const unsigned char*>(k_cache);
  a.v = static_cast<const unsigned char*>(v_cache);
  a.block_tables = block_tables;
  a.seq_lens = seq_lens;
  a.piece_o = pieces;
  a.piece_ml = pieces + static_cast<int64_t>(kDecSlots) * 2 * group * head_dim;
  a.cut = reinterpret_cast<int2*>(
      a.piece_ml + static_cast<int64_t>(kDecSlots) * 2 * group * 2);
  a.q_stride = q_stride;
  a.num_seqs = num_seqs;
  a.max_blocks = max_blocks;
  a.num_kv_heads = num_kv_heads;
  a.group = group;
  a.scale = scale;
  const dim3 block(kDecWaves * kWaveSize);
  // one context of 8000 tokens leaves 125 pieces: a block per query head
  // takes 5 us where a block per context takes 11
  const int contexts = num_seqs * num_kv_heads;
  const int heads = contexts < 256 ? 1 : group;
#define FI_DEC(DD, F8)                                                        \
  do {                                                                        \
    hipLaunchKernelGGL((paged_attn_decode_kernel<DD, F8>),                    \
                       dim3(kDecSlots / kDecWaves), block, 0, stream, a);     \
    hipLaunchKernelGGL((paged_attn_join_kernel<DD>),                          \
                       dim3(contexts * (group / heads)),                      \
                       dim3(kJoinWaves * kWaveSize), 0, stream, a, heads);    \
  } while (0)
  if (head_dim == 128) {
    if (fp8) FI_DEC(128, true);
    else FI_DEC(128, false);
  } else {
    if (fp8) FI_DEC(64, true);
    else FI_DEC(64, false);
  }
#undef FI_DEC
}

}  // namespace fi
