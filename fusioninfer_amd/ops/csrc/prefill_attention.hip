// Prefill attention: the join of cut query tiles, the plan of a launch and
// the launch itself.

#include "prefill_pair.h"
#include "prefill_rows.h"

#include <cmath>

namespace fi {

// Adds up the pieces of the query tile that a part's end cuts, in the block
// of the part in which the tile begins. blockIdx.y: 32 query vectors (a wave
// of the attention kernel); a wave here takes eight accumulator registers of
// every lane, of up to eight pieces at once so that their loads overlap.
template <int D, bool PAGED>
__global__ __launch_bounds__(D / 16 * kWaveSize)
void prefill_attn_join_kernel(const PrefillArgs p) {
  constexpr int kRegs = 8, kGroup = 8;
  const int slot = blockIdx.x, qwave = blockIdx.y, kWaves = gridDim.y;
  const int part = threadIdx.x / kWaveSize, lane = threadIdx.x % kWaveSize;
  const int4 cut = p.cut[slot];
  if (cut.y < 0) return;
  const int hg = cut.x;
  const QTile t = q_tile<PAGED>(p, cut.y);
  const int wph = kWaves / p.hpb;
  const int row0 = t.row0 + (qwave % wph) * 32;
  if (row0 >= t.seq_len) return;
  const float c = p.scale == 0.f
      ? 1.f : fabsf(p.scale) * 1.4426950408889634f;

  float m = kPNegInf, l = 0.f, o[kRegs];
#pragma unroll
  for (int r = 0; r < kRegs; ++r) o[r] = 0.f;
  for (int s0 = slot; s0 < cut.z; s0 += kGroup) {
    float2 ml[kGroup];
    float x[kGroup][kRegs];
#pragma unroll
    for (int g = 0; g < kGroup; ++g) {
      const int s = s0 + g;
      const bool there = s < cut.z;  // otherwise the first again, as zeros
      const int64_t piece =
          static_cast<int64_t>(there ? s * 2 + (s == slot ? 1 : 0)
                                     : slot * 2 + 1) * kWaves + qwave;
      ml[g] = reinterpret_cast<const float2*>(p.piece_ml)[piece * 64 + lane];
      if (!there) ml[g] = make_float2(kPNegInf, 0.f);
      const float* src = p.piece_o + piece * 32 * D + part * kRegs * 64 + lane;
#pragma unroll
      for (int r = 0; r < kRegs; ++r) {
        x[g][r] = src[r * 64];
        if (!there) x[g][r] = 0.f;     // it may hold infinities
      }
    }
    float mx = m;
#pragma unroll
    for (int g = 0; g < kGroup; ++g) mx = fmaxf(mx, ml[g].x);
    const float a = __builtin_amdgcn_exp2f((m - mx) * c);
    m = mx;
    l *= a;
#pragma unroll
    for (int r = 0; r < kRegs; ++r) o[r] *= a;
#pragma unroll
    for (int g = 0; g < kGroup; ++g) {
      const float b = __builtin_amdgcn_exp2f((ml[g].x - mx) * c);
      l += ml[g].y * b;
#pragma unroll
      for (int r = 0; r < kRegs; ++r) o[r] = fmaf(x[g][r], b, o[r]);
    }
  }
  const int col = lane & 31, hi1 = lane >> 5;
  if (row0 + col >= t.seq_len) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  u16* orow = p.out + (static_cast<int64_t>(t.seq_start + row0 + col) *
                           p.num_q_heads + hg * p.hpb + qwave / wph) * D;
#pragma unroll
  for (int r = 0; r < kRegs; r += 4) {
    bf16x4 w;
#pragma unroll
    for (int j = 0; j < 4; ++j) w.h[j] = f32_to_bf16(o[r + j] * inv);
    const int reg = part * kRegs + r;  // of the tile kernel's accumulators
    *reinterpret_cast<bf16x4*>(orow + reg / 16 * 32 + crow(reg % 16, hi1)) = w;
  }
}

// Heads of a workgroup and query tiles of a launch, and whether to split.
//
// The host knows bounds: query tiles (nq), the longest K/V range and the
// number of new rows. Whole query tiles take ceil(fill) rounds of the chip,
// fill = workgroups / 256 (below one round a lone workgroup runs about 1.4
// times as fast); the split form takes `fill` of them and about 35 us more
// for its schedule, the pieces and the second launch, which is what 26 tiles
// take. Where the new rows are most of the context, tiles differ in length
// and longest-first already evens them out. Measured, whole / split in us, 32
// query heads, 8 K/V heads of 128: 16 rows behind 2000 42 / 33; 512 behind 2048
// 52 / 50; 1024 behind 1024 44 / 59; 1024 behind 8192 184 / 170; 4099 behind 16384
// 1443 / 1201; 4096 behind 16384 (exactly two rounds) 1125 / 1127; 2048 from the
// start 52 / 88. Of 22 portions of 16 to 4099 rows behind 1024 to 16384 the choice
// is the faster one or within 4 %; with an e4m3 cache, whose whole tiles take a
// tenth longer, within 14, with heads of 64 within 17. Of several contexts it
// takes all for the longest, and can miss: 16 heads, four of 300 rows behind 1200
// to 4000 87 / 61, whole; 32 heads, 700, 33 and 1200 behind 6000 212 / 234, split.
//
// The split form with 64 query vectors per wave (`pair`) takes 0.92 of the
// time per tile, but 15 us more for its longer pipeline and the tiles that go
// step by step: it is ahead from parts of 128 tiles on (8 query heads, 4 K/V
// heads, 1024 rows behind 8192, parts of 17: 82 us, 96 with pairs; 32 and 8,
// 700 + 33 + 1200 behind 6000, parts of 120: 239 and 255; 1000 behind 30000,
// parts of 242: 509 and 484; 4099 behind 16384 1285 and 1188). `pairs`: whether that kernel takes the operands,
// bf16 rows of 128 in a paged cache.
PrefillPlan plan_prefill_attn(int ntiles, int tile_rows, int num_q_heads,
                              int num_kv_heads, int new_rows, int max_k_len,
                              bool pairs) {
  const int group = num_q_heads / num_kv_heads;
  auto layout = [&](bool split) {
    PrefillPlan pl;
    pl.split = split;
    pl.pair = false;
    pl.waves = attn_waves(split);
    pl.hpb = group % 4 == 0 ? 4 : (group % 2 == 0 ? 2 : 1);
    pl.rows = pl.waves * 32 / pl.hpb;
    pl.sub = ceil_div(tile_rows, pl.rows);
    pl.nq = ntiles * pl.sub;
    pl.slots = 0;
    pl.longest = max_k_len;
    return pl;
  };
  PrefillPlan pl = layout(true);
  const int64_t blocks = static_cast<int64_t>(pl.nq) *
                         (num_q_heads / pl.hpb);
  const int64_t tiles = ceil_div(max_k_len, kKVTile);
  const double fill = blocks / 256.0;
  pl.pair = pairs && fill * tiles >= 128;
  const double idle = fill < 1.0 ? 1.0 - std::min(1.0, 1.4 * fill)
                                 : std::ceil(fill) -
                                       (pl.pair ? 0.96 : 1.04) * fill;
  // A workgroup's rows lie within one entry of the tile table: the split
  // form's 256 (one head per workgroup) do not fit into entries of 128.
  if (pl.rows > tile_rows ||
      2 * static_cast<int64_t>(new_rows) > max_k_len || idle * tiles <= 26)
    return layout(false);
  // parts of at least eight tiles, in whole rounds over the XCDs
  pl.slots = static_cast<int>(std::min<int64_t>(
      256, std::max<int64_t>(8, blocks * tiles / 8 / 8 * 8)));
  return pl;
}

int64_t prefill_piece_floats(const PrefillPlan& pl, int head_dim) {
  return static_cast<int64_t>(pl.slots) *
         (2 * pl.waves * (32 * head_dim + kWaveSize * 2) + 4);
}

void launch_prefill_attn(u16* out, const u16* q, const void* k, const void* v,
                         const int* tile_seq, const int* tile_row0,
                         const int* cu_seqlens, const int* block_tables,
                         const int* seq_lens_k, int max_blocks,
                         int64_t q_stride, int64_t k_stride, int64_t v_stride,
                         int num_q_heads, int num_kv_heads, int head_dim,
                         float scale, bool fp8, const PrefillPlan& pl,
                         float* pieces, hipStream_t stream) {
  const bool paged = block_tables != nullptr;
  PrefillArgs a = {};
  a.out = out;
  a.q = q;
  a.k = k;
  a.v = v;
  a.tile_seq = tile_seq;
  a.tile_row0 = tile_row0;
  a.cu_seqlens = cu_seqlens;
  a.block_tables = block_tables;
  a.seq_lens_k = seq_lens_k;
  a.piece_o = pieces;
  a.piece_ml = pieces ? pieces + static_cast<int64_t>(pl.slots) * 2 *
                                     pl.waves * 32 * head_dim
                      : nullptr;
  a.cut = reinterpret_cast<int4*>(
      pieces ? a.piece_ml + static_cast<int64_t>(pl.slots) * 2 * pl.waves *
                                kWaveSize * 2
             : nullptr);
  a.q_stride = q_stride;
  a.k_stride = k_stride;
  a.v_stride = v_stride;
  a.max_blocks = max_blocks;
  a.num_q_heads = num_q_heads;
  a.num_kv_heads = num_kv_heads;
  a.hpb = pl.hpb;
  a.rows = pl.rows;
  a.slots = pl.slots;
  a.sub = pl.sub;
  a.nq = pl.nq;
  a.scale = scale;
  const dim3 block(pl.waves * kWaveSize);
#define FI_PF_LAUNCH(DD, PP, F8)                                              \
  do {                                                                        \
    if (pl.split) {                                                           \
      if (DD == 128 && PP && !F8 && pl.pair)                                  \
        hipLaunchKernelGGL((prefill_pair_kernel<4>), dim3(pl.slots),          \
                           dim3(4 * kWaveSize), 0, stream, a);                \
      else                                                                    \
        hipLaunchKernelGGL((prefill_attn_kernel<DD, PP, F8>),                 \
                           dim3(pl.slots), block, 0, stream, a);              \
      hipLaunchKernelGGL((prefill_attn_join_kernel<DD, PP>),                  \
                         dim3(pl.slots, pl.waves),                            \
                         dim3(DD / 16 * kWaveSize), 0, stream, a);            \
    } else {                                                                  \
      launch_rows<DD, PP, F8, false>(a, pl.longest, stream);                  \
    }                                                                         \
  } while (0)
  if (fp8 && !paged) abort();  // fp8 KV is a cache format; dense is bf16
  if (head_dim == 128) {
    if (paged) {
      if (fp8) FI_PF_LAUNCH(128, true, true);
      else FI_PF_LAUNCH(128, true, false);
    } else {
      FI_PF_LAUNCH(128, false, false);
    }
  } else if (head_dim == 64) {
    if (paged) {
      if (fp8) FI_PF_LAUNCH(64, true, true);
      else FI_PF_LAUNCH(64, true, false);
    } else {
      FI_PF_LAUNCH(64, false, false);
    }
  } else {
    abort();
  }
#undef FI_PF_LAUNCH
}

}  // namespace fi
