// The split form of the prefill kernel over the paged cache for bf16 rows of
// 128: 64 query vectors per wave.
//
// Four waves, one per SIMD, hold two groups of 32 query vectors each, so that
// a fragment of K or V read from LDS feeds two products: with one group per
// wave (eight waves) LDS delivered 256 KB per tile, as many cycles as the
// matrix cores need. Nothing hides a lone wave's softmax, so it is spread by
// hand: while a tile's scores are in work, the next tile's are multiplied.
//
// A tile is 64 places, each one MFMA (32x32x16, 32 cycles) and about as many
// cycles of something else, in an order that is pinned:
//   0..31   S of the next tile       0..54   exponentials of this one, those
//   32..63  O += V^T P of this one           of a 16-deep step before its
//                                            product
//                                    32..63  maxima of the next tile
// Fragments are read four ahead. At place 48 the tile after the next has
// landed in every wave, and nobody reads the tile before this one any more:
// the fifth tile from there is requested into its place (five are kept, all
// of a CU's LDS).
//
// Tiles at the diagonal, those whose maximum makes a rescaling necessary, the
// last one of a part and every 64th go step by step, without the overlap.
// Scores, maxima, sums and the order of the keys are those of
// prefill_attn_kernel, bit for bit.
//
// Measured, us, eight waves of one group and this (32 query heads, 8 K/V
// heads), repeated alone: 4099 rows behind 16384 1231 -> 1132 (1.09 PFLOP/s),
// 6000 behind 14000 1651 -> 1534, 1000 behind 30000 520 -> 484; behind an idle
// card, or between the linear layers of a step, at a lower clock, 4099 rows take
// 1210 to 1320. Matrix cores busy 56 % of the time at 2.05 GHz; vector
// instructions issue for 53 %, waits take 19 %. (Twelve registers are spilled,
// outside the overlapped form.)

#pragma once

#include <type_traits>
#include <utility>

#include "prefill_kernel.h"
#include "tile_engine.h"

namespace fi {

// f(0), f(1), ... f(N - 1) with the number in its type
template <class F, int... I>
FI_DEV void each_place(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

// 16 bytes per lane to LDS at m0 + 16 lane; set_m0 lies at least one
// instruction ahead
FI_DEV void pair_load(const void* base, u32 offset) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("global_load_lds_dwordx4 %0, %1"
               :
               : "v"(offset), "s"(base)
               : "memory");
#endif
}
// S = K Q^T (+ S): scores in vector registers, queries in accumulation
// registers; O += V^T P: results in accumulation registers. In asm, so that
// each has one place (from the builtins the compiler moves a third of them
// back and forth). The wait states between a product and other instructions
// on its registers are kept by distance, or by settle().
FI_DEV void qk_first(floatx16& s, const short8& k, const short8& q) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0"
               : "=&v"(s)
               : "v"(k), "a"(q));
#endif
}
FI_DEV void qk(floatx16& s, const short8& k, const short8& q) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0"
               : "+v"(s)
               : "v"(k), "a"(q));
#endif
}
FI_DEV void pv(floatx16& o, const short8& v, const short8& w) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0"
               : "+a"(o)
               : "v"(v), "v"(w));
#endif
}
FI_DEV void clear_result(float& a) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_accvgpr_write_b32 %0, 0" : "=a"(a));
#endif
}
// (in asm, or each operand that comes from asm is made canonical first)
FI_DEV float max3(float a, float b, float c) {
  float v = a;
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_max3_f32 %0, %1, %2, %3" : "=v"(v) : "v"(a), "v"(b), "v"(c));
#endif
  return v;
}
typedef __attribute__((ext_vector_type(2))) float floatx2;
FI_DEV floatx2 move(floatx2 from) {
  floatx2 to = from;
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mov_b64 %0, %1" : "=v"(to) : "v"(from));
#endif
  return to;
}
FI_DEV void pin() { __builtin_amdgcn_sched_barrier(0); }

// A template only so that it may lie in a header.
template <int kWaves>
__global__ __launch_bounds__(kWaves * kWaveSize, 1)
void prefill_pair_kernel(const PrefillArgs p) {
  static_assert(kWaves == 4);
  constexpr int D = 128, kGroups = 2, kBufs = 5;
  constexpr int KF = D / 16, CB = D / 32, kRowB = D * 2, kChunk = D / 8;
  constexpr int kTileB = kKVTile * kRowB;
  constexpr int kWRows = kKVTile / kWaves, kDma = 4;  // per wave and matrix
  constexpr int kAll = kWaves * kGroups;              // groups of a workgroup

  __shared__ __attribute__((aligned(1024)))
  unsigned char smem[2 * kBufs * kTileB];
  const u32 lds0 = static_cast<u32>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) unsigned char*)smem));

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWaveSize);
  const int lane = tid % kWaveSize;
  const int col = lane & 31;           // this lane's query vector of a group
  const int hi1 = lane >> 5;
  const int wph = kAll / p.hpb;        // groups per query head, even

  auto k_swz = [](int row) { return row & 15; };
  auto v_swz = [](int row) { return (row & 3) << 2; };
  // fragment f of K at k_off ^ 32 f, cb of V at v_off ^ 64 cb
  const int k_off = col * kRowB + ((hi1 ^ k_swz(col)) * 16);
  const int v_row = 4 * hi1 + ((lane & 15) >> 2);
  const int v_off = kBufs * kTileB + v_row * kRowB +
                    (((((lane >> 4) & 1) * 2 + ((lane & 3) >> 1)) ^
                      v_swz(v_row)) * 16) + (lane & 1) * 8;

  // where this lane's DMAs of the first four rows begin
  const u32 k_from = lane / kChunk * kRowB +
                     ((lane % kChunk) ^ (lane / kChunk)) * 16;
  const u32 v_from = lane / kChunk * kRowB +
                     ((lane % kChunk) ^ v_swz(lane / kChunk)) * 16;

  const float sgn = p.scale > 0.f ? 1.f : (p.scale < 0.f ? -1.f : 0.f);
  const float c = p.scale == 0.f
      ? 1.f : fabsf(p.scale) * 1.4426950408889634f;  // log2(e)

  int64_t pos = 0, pos_end = 1;
  int hg = 0, qt = 0, from = 0;
  int4 cut = make_int4(0, -1, 0, 0);
  const int u = total_work<true>(p, lane);
  const int64_t total = static_cast<int64_t>(u) * (p.num_q_heads / p.hpb);
  const int slot = split_slot(blockIdx.x, p.slots);
  const Parts parts(total, p.slots);
  pos = parts.begin(slot);
  pos_end = parts.begin(slot + 1);
  if (pos < pos_end) {
    hg = static_cast<int>(pos / u);
    qt = find_tile<true>(p, lane, static_cast<int>(pos - int64_t(hg) * u),
                          &from);
  }
  // the tile at the end: the part itself or a later one finishes it
  if (pos < pos_end && pos_end < total) {
    const int h = static_cast<int>(pos_end / u);
    int within;
    const int i = find_tile<true>(
        p, lane, static_cast<int>(pos_end - int64_t(h) * u), &within);
    if (within > 0 && pos_end - within >= pos) {
      const int64_t end = pos_end - within + q_tile<true>(p, i).work;
      cut = make_int4(h, i, slot + 1, 0);
      while (cut.z < p.slots && parts.begin(cut.z) < end) ++cut.z;
    }
  }
  if (tid == 0) p.cut[slot] = cut;

  while (pos < pos_end) {
    const QTile t = uniform_tile(q_tile<true>(p, qt));
    if (t.work == 0) {                 // rows past the sequence's end
      if (++qt == p.nq) { qt = 0; ++hg; }
      continue;
    }
    const int ta = from;
    const int tb = static_cast<int>(
        min(static_cast<int64_t>(t.work), from + (pos_end - pos)));
    const int head = hg * p.hpb + wave * kGroups / wph;
    const int kv_head = hg * p.hpb / (p.num_q_heads / p.num_kv_heads);
    const int ctx_start = t.k_len - t.seq_len;
    const int row0 = t.row0 + (wave * kGroups % wph) * 32;  // of group 0
    const bool active = row0 < t.seq_len;
    const int last_blk = (t.k_len - 1) >> 4;
    const ConstInts bt_row = const_ints(
        p.block_tables + static_cast<int64_t>(t.seq) * p.max_blocks);

    // ---- staging: wave w copies rows 16w..16w+15 of a tile, one cache
    // block. Rows past the end repeat the last one, tiles past the part's
    // last one repeat that (nobody reads them).
    auto block_of = [&](int tile) {
      return bt_row[min(min(tile, tb - 1) * 4 + wave, last_blk)];
    };
    const u16 *kb = nullptr, *vb = nullptr;
    int limit = 0;
    u32 dst = 0;
    auto aim = [&](int tile, int blk, int buf) {
      dst = lds0 + buf * kTileB + wave * kWRows * kRowB;
      const int64_t base =
          (static_cast<int64_t>(blk) * p.num_kv_heads + kv_head) * 16 * D;
      kb = static_cast<const u16*>(p.k) + base;
      vb = static_cast<const u16*>(p.v) + base;
      limit = t.k_len - 1 - min(min(tile, tb - 1) * 4 + wave, last_blk) * 16;
    };
    auto m0_of = [&](int i) {
      set_m0(dst + (i & 1) * kBufs * kTileB + (i >> 1) * 1024);
    };
    auto load_of = [&](int i) {
      const int r = (i >> 1) * 4 + lane / kChunk;  // row of the wave
      const int src = min(r, limit);
      if (i & 1)
        pair_load(vb, src * kRowB + ((lane % kChunk) ^ v_swz(r)) * 16);
      else
        pair_load(kb, src * kRowB + ((lane % kChunk) ^ k_swz(r)) * 16);
    };
    // the same where no row lies past the end
    auto load_whole = [&](auto place) {
      constexpr int i = place, r = (i >> 1) * 4;
      if constexpr (i & 1)
        pair_load(vb, v_from ^ (r * kRowB));
      else
        pair_load(kb, k_from ^ (r * kRowB + r * 16));
    };
    auto stage_all = [&] {
#pragma unroll
      for (int i = 0; i < 2 * kDma; ++i) {
        m0_of(i);
        asm volatile("s_nop 4");
        load_of(i);
      }
    };

    // the previous query tile's LDS reads and DMAs are over in every wave
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    for (int i = 0; i < kBufs - 1; ++i) {
      aim(ta + i, block_of(ta + i), i);
      stage_all();
    }
    // cache blocks of the 64 tiles from ids_from on, one per lane (a scalar
    // load would make every wait for LDS wait for it too)
    int ids = 0, ids_from = 0;

    // ---- query fragments
    short8 b_q[kGroups][KF];
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      const int qr = min(row0 + g * 32 + col, t.seq_len - 1);
      const u16* qrow = p.q + (t.seq_start + qr) * p.q_stride +
                        static_cast<int64_t>(head) * D;
#pragma unroll
      for (int f = 0; f < KF; ++f) {
        b_q[g][f] = *reinterpret_cast<const short8*>(qrow + f * 16 + hi1 * 8);
        if (sgn != 1.f) {
          bf16x8 h = __builtin_bit_cast(bf16x8, b_q[g][f]);
#pragma unroll
          for (int j = 0; j < 8; ++j)
            h.h[j] = f32_to_bf16(bf16_to_f32(h.h[j]) * sgn);
          b_q[g][f] = __builtin_bit_cast(short8, h);
        }
      }
    }
    // arrived here, not at their first use inside the loop, and in the
    // registers that the products take them from
#pragma unroll
    for (int g = 0; g < kGroups; ++g)
#pragma unroll
      for (int f = 0; f < KF; ++f) {
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" : "+a"(b_q[g][f]));
#endif
      }

    float m_row[kGroups] = {kPNegInf, kPNegInf}, l_row[kGroups] = {0.f, 0.f};
    floatx16 o_acc[kGroups][CB];
#pragma unroll
    for (int g = 0; g < kGroups; ++g)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float o;
          clear_result(o);
          o_acc[g][cb][r] = o;
        }

    // ---- pieces of a tile's work
    using Scores = floatx16[kGroups][2];
    int vbuf = 0, kbuf = 1, sbuf = kBufs - 1;  // this tile's V, the next
                                               // one's K, where to request to
    short8 kf[4], vf[4];
    auto read_k = [&](int buf, int n) {       // fragment n: f = n / 2, b
      return *reinterpret_cast<const short8*>(
          smem + ((buf * kTileB + k_off) ^ ((n >> 1) * 32)) +
          (n & 1) * 32 * kRowB);
    };
    auto read_v = [&](int buf, int n) {       // kc = n / 4, cb
      const unsigned char* a =
          smem + ((buf * kTileB + v_off) ^ ((n & 3) * 64)) +
          (n >> 2) * 16 * kRowB;
      const short4v lo = lds_read_tr4(a), hi = lds_read_tr4(a + 8 * kRowB);
      return short8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    auto score = [&](floatx16& s, const short8& k, int g, int f) {
      if (f == 0) qk_first(s, k, b_q[g][f]);
      else qk(s, k, b_q[g][f]);
    };
    auto largest = [&](const floatx16 (&s)[2]) {
      float rm = fmaxf(s[0][0], s[1][0]);
#pragma unroll
      for (int r = 1; r < 16; ++r) rm = fmaxf(rm, fmaxf(s[0][r], s[1][r]));
      return rm;
    };
    bool calm = false;   // the next tile's maxima need no rescaling
    auto still = [&](float r0, float r1) {
      const bool a = (fmaxf(r0, half_swap(r0)) - m_row[0]) * c <= kDeferThr;
      const bool b = (fmaxf(r1, half_swap(r1)) - m_row[1]) * c <= kDeferThr ||
                     row0 + 32 >= t.seq_len;
      return static_cast<bool>(__all(static_cast<int>(a) & b));
    };
    // a new maximum: sums and results are rescaled where it matters
    auto raise = [&](int g, float rm) {
      rm = fmaxf(rm, half_swap(rm));
      if (!__all((rm - m_row[g]) * c <= kDeferThr)) {
        const float m_new = fmaxf(m_row[g], rm);
        const float alpha = __builtin_amdgcn_exp2f((m_row[g] - m_new) * c);
        m_row[g] = m_new;
        l_row[g] *= alpha;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
          for (int r = 0; r < 16; ++r) o_acc[g][cb][r] *= alpha;
      }
    };
    auto advance = [&] {
      vbuf = kbuf;
      kbuf = kbuf == kBufs - 1 ? 0 : kbuf + 1;
      sbuf = sbuf == kBufs - 1 ? 0 : sbuf + 1;
    };
    const int q_max = ctx_start + min(row0 + kGroups * 32, t.seq_len) - 1;

    // a tile wholly visible to both groups, with another one behind it
    auto overlapped = [&](int tile, Scores& cur, Scores& nxt) {
      float rm[kGroups], rs[kGroups][4] = {};
      const float mc[kGroups] = {m_row[0] * c, m_row[1] * c};
      bf16x8 w[kGroups][4];
      float last = 0.f;
      auto take = [&](auto place) {
        constexpr int v = place, kc = v >> 4, g = v >> 3 & 1, j = v & 7;
        rs[g][j & 3] += last;
        asm volatile("" : "+v"(rs[g][j & 3]));   // here, not after the loop
        w[g][kc].h[j] = f32_to_bf16(last);
      };
      auto exponential = [&](auto place) {
        constexpr int v = place, kc = v >> 4, g = v >> 3 & 1, j = v & 7;
        const float e = __builtin_amdgcn_exp2f(
            fmaf(cur[g][kc >> 1][(kc & 1) * 8 + j], c, -mc[g]));
        // (the one before: an exponential cannot be used at once)
        if constexpr (v > 0) take(std::integral_constant<int, v - 1>{});
        last = e;
      };
      each_place([&](auto place) {
        constexpr int s = place, n = s >> 1 & 15, g = s & 1;
        if constexpr (s < 32)
          score(nxt[g][n & 1], kf[n & 3], g, n >> 1);
        else
          pv(o_acc[g][n & 3], vf[n & 3],
             __builtin_bit_cast(short8, w[g][n >> 2]));
        pin();
        // fragments four ahead, behind the second product of the one whose
        // registers they take
        if constexpr (g == 1) {
          constexpr int ahead = (s >> 1) + 4;
          if constexpr (ahead < 16)
            kf[ahead & 3] = read_k(kbuf, ahead);
          else if constexpr (ahead < 32)
            vf[ahead & 3] = read_v(vbuf, ahead - 16);
          else
            kf[ahead & 3] = read_k(kbuf == kBufs - 1 ? 0 : kbuf + 1,
                                   ahead - 32);
        }
        if constexpr (s < 55) {
          constexpr int from = s * 64 / 55, to = (s + 1) * 64 / 55;
          exponential(std::integral_constant<int, from>{});
          if constexpr (to - from == 2)
            exponential(std::integral_constant<int, from + 1>{});
        }
        if constexpr (s == 55) take(std::integral_constant<int, 63>{});
        if constexpr (s >= 32) {
          // two of the next tile's scores: the maximum, and into the place
          // of those whose exponentials are done
          constexpr int m = s - 32, h = m >> 2 & 1, b = m >> 4;
          constexpr int r = (m >> 3 & 1) * 8 + (m & 3) * 2;
          floatx2 two = {nxt[h][b][r], nxt[h][b][r + 1]};
          rm[h] = max3(m == h * 4 ? two[0] : rm[h], two[0], two[1]);
          two = move(two);
          cur[h][b][r] = two[0];
          cur[h][b][r + 1] = two[1];
        }
        if constexpr (s == 48) {
          // (this wave's DMAs but the youngest tile's)
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kDma) : "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
          aim(tile + kBufs - 1,
              __builtin_amdgcn_readlane(ids, tile + kBufs - 1 - ids_from),
              sbuf);
        }
        if constexpr (s >= 48 && g == 0) m0_of((s - 48) >> 1);
        if constexpr (s >= 48 && g == 1)
          load_whole(std::integral_constant<int, (s - 48) / 2>{});
        pin();
      }, std::make_integer_sequence<int, 64>{});
#pragma unroll
      for (int g = 0; g < kGroups; ++g)
        l_row[g] += (rs[g][0] + rs[g][1]) + (rs[g][2] + rs[g][3]);
      calm = still(rm[0], rm[1]);
      advance();
    };

    // any tile, step by step
    auto plain = [&](int tile, Scores& cur, Scores& nxt) {
      const int kv0 = tile * kKVTile;
      if (tile + 1 < tb && active)
#pragma unroll
        for (int n = 0; n < 16; ++n) {
          const short8 k = read_k(kbuf, n);
#pragma unroll
          for (int g = 0; g < kGroups; ++g) score(nxt[g][n & 1], k, g, n >> 1);
        }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      ids_from = tile + kBufs - 1;
      const int at = min(min(ids_from + lane, tb - 1) * 4 + wave, last_blk);
      ids = p.block_tables[static_cast<int64_t>(t.seq) * p.max_blocks + at];
      asm volatile("" : "+v"(ids));          // waited for here
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kDma) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      aim(tile + kBufs - 1, __builtin_amdgcn_readfirstlane(ids), sbuf);
      stage_all();
      settle();
#pragma unroll
      for (int g = 0; g < kGroups; ++g) {
        const int r0 = row0 + g * 32;
        if (r0 >= t.seq_len ||
            kv0 > ctx_start + min(r0 + 32, t.seq_len) - 1) continue;
        if (kv0 + kKVTile - 1 > ctx_start + r0) {
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r)
              if (kv0 + 32 * b + crow(r, hi1) > ctx_start + r0 + col)
                cur[g][b][r] = -INFINITY;
        }
        raise(g, largest(cur[g]));
        const float mc = m_row[g] * c;
        float rs[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) {
          bf16x8 w;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float e = __builtin_amdgcn_exp2f(
                fmaf(cur[g][kc >> 1][(kc & 1) * 8 + j], c, -mc));
            rs[j & 3] += e;
            w.h[j] = f32_to_bf16(e);
          }
          const short8 wk = __builtin_bit_cast(short8, w);
          settle();
#pragma unroll
          for (int cb = 0; cb < CB; ++cb)
            pv(o_acc[g][cb], read_v(vbuf, kc * 4 + cb), wk);
        }
        l_row[g] += (rs[0] + rs[1]) + (rs[2] + rs[3]);
      }
      if (tile + 1 < tb && active)
        calm = still(largest(nxt[0]), largest(nxt[1]));
      advance();
      // as the overlapped form leaves them
#pragma unroll
      for (int n = 0; n < 4; ++n) kf[n] = read_k(kbuf, n);
    };

    // the first tiles have landed
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    Scores s0, s1;
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      const short8 k = read_k(0, n);
#pragma unroll
      for (int g = 0; g < kGroups; ++g) score(s0[g][n & 1], k, g, n >> 1);
    }
#pragma unroll
    for (int n = 0; n < 4; ++n) kf[n] = read_k(kbuf, n);
    auto smooth = [&](int tile) {
      return tile + 1 < tb && active && calm &&
             tile + kBufs - 1 - ids_from < kWaveSize &&
             min(tile + kBufs, tb) * kKVTile <= t.k_len &&
             tile * kKVTile + kKVTile - 1 <= ctx_start + row0;
    };
    for (int tile = ta; tile < tb; ++tile) {
      while (smooth(tile)) overlapped(tile++, s0, s1);
      plain(tile, s0, s1);
#pragma unroll
      for (int g = 0; g < kGroups; ++g)
#pragma unroll
        for (int b = 0; b < 2; ++b) s0[g][b] = s1[g][b];
    }

    // ---- epilogue ----
    settle();
    const bool whole = ta == 0 && tb == t.work;
    const int piece = slot * 2 + (ta > 0 ? 0 : 1);
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      const int row = row0 + g * 32 + col;
      l_row[g] += half_swap(l_row[g]);
      if (whole) {
        if (row < t.seq_len) {
          const float inv = l_row[g] > 0.f ? 1.f / l_row[g] : 0.f;
          u16* orow = p.out + (static_cast<int64_t>(t.seq_start + row) *
                                   p.num_q_heads + head) * D;
#pragma unroll
          for (int cb = 0; cb < CB; ++cb)
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
              bf16x4 w;
#pragma unroll
              for (int j = 0; j < 4; ++j)
                w.h[j] = f32_to_bf16(acc_of(o_acc[g][cb][r + j]) * inv);
              *reinterpret_cast<bf16x4*>(orow + cb * 32 + crow(r, hi1)) = w;
            }
        }
      } else {
        const int64_t at = static_cast<int64_t>(piece) * kAll +
                           wave * kGroups + g;
        float* o = p.piece_o + at * 32 * D + lane;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            o[(cb * 16 + r) * 64] = acc_of(o_acc[g][cb][r]);
        reinterpret_cast<float2*>(p.piece_ml)[at * 64 + lane] =
            make_float2(m_row[g], l_row[g]);
      }
    }
    pos += tb - ta;
    from = 0;
    if (++qt == p.nq) { qt = 0; ++hg; }
  }
  // no DMA may land in LDS that is no longer this workgroup's
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

}  // namespace fi
