// Fused per-head RMSNorm (Qwen3 qk-norm) + NeoX rotary embedding of Q and K
// rows, in place, or (CACHE) with the K rows and the untouched V rows going
// straight into the paged cache [num_blocks, Hk, block_size, D].
//
// Bound by memory: every row is read and written once. A lane holds eight
// elements, so D / 8 lanes hold a head and a wave four heads (D = 128) or
// eight (64) of one token; the rotate-half partner is D / 16 lanes away in
// the same row of 16 lanes, and the norm's sum is three or four exchanges
// within it. A workgroup is one token, or four waves of one where there are
// few; every load is requested before anything waits for one. cos/sin come from
// a table (f32 [P, D], cos | sin): sines computed here would make it bound by
// the VALU. us at 32 + 2 * 8 heads of 128, loads as they are needed and a
// rolled loop for the sum, and this: 64 tokens 2.9 and 2.5, 1024 7.7 and 6.0,
// 4099 19.7 and 16.0 (6.3 TB/s), 8765 44.6 and 37.7; e4m3 cache, 8765 43.8 and
// 37.9.
//
// Capability parity: RoPE / qk-norm epilogue and cache write the reference
// delegates to vLLM.

#include "pieces.h"

namespace fi {

namespace {

// rows are slices of the projections' output: no alignment is assumed
typedef u32 u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kRopeWaves = 16;      // of a workgroup, at most

FI_DEV u32x4_any load8(const u16* p) {
  return *reinterpret_cast<const u32x4_any*>(p);
}
FI_DEV void unpack8(const u32x4_any& w, float v[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = bf16_to_f32(static_cast<u16>(w[i] & 0xffff));
    v[2 * i + 1] = bf16_to_f32(static_cast<u16>(w[i] >> 16));
  }
}

// sum over the L lanes of a head, by exchanges with the lane 8 (L = 16), 4, 2
// and 1 away
template <int L>
FI_DEV float head_sum(float s) {
  if constexpr (L == 16) {
    s += dpp_move<0x128>(s);         // row_ror:8
    s += dpp_move<0x124>(s);         // row_ror:4
  } else {
    s += __shfl_xor(s, 4);
  }
  s += dpp_move<0x4E>(s);            // quad_perm [2,3,0,1]
  s += dpp_move<0xB1>(s);            // quad_perm [1,0,3,2]
  return s;
}

struct CacheRows {
  void* k;           // [num_blocks, Hk, block_size, D] bf16 or e4m3
  void* v;
  const int* slots;  // [T], negative: the row is not kept
  int block_size;
  float k_inv_scale, v_inv_scale;  // fp8 only
};

// UNITS: times four heads (D = 128) or eight (64) that a wave takes of a token
// PIECES: the rows are sums of pieces (+ bias) of a product that is cut, a
// launch and a pass over them less; results of q go to q. Bound by the way of
// the pieces through memory as their sum alone is: 64 rows, 32 + 2 * 8 heads of
// 128, 5.8 us with 16 waves a workgroup, 1.1 less with four; the sum alone 4.6
// and the rest 4.0 (256 rows 9.4, 6.7 and 4.2).
// NORM: there is a weight for q or k. (Without one a sum that nobody reads
// costs a launch for few tokens 0.2 to 0.5 us of 2.3.)
template <int D, bool CACHE, bool FP8, int UNITS, bool PIECES, bool NORM>
__global__ __launch_bounds__(kRopeWaves * kWaveSize) void rope_qk_norm_kernel(
    u16* __restrict__ q,             // [T, Hq*D] rows, stride q_stride
    u16* __restrict__ k,             // [T, Hk*D] rows, stride k_stride
    const u16* __restrict__ v,       // CACHE: [T, Hk*D] rows
    const int64_t q_stride, const int64_t k_stride, const int64_t v_stride,
    const u16* __restrict__ q_weight,  // [D] or nullptr
    const u16* __restrict__ k_weight,  // [D] or nullptr
    const float* __restrict__ cos_sin,  // [P, D]
    const int* __restrict__ positions,  // [T]
    const int num_q_heads, const int num_kv_heads,
    const float eps, const CacheRows cache, const PieceRows pieces,
    const int tokens) {
  static_assert(!PIECES || (CACHE && UNITS == 1));
  constexpr int L = D / 8;           // lanes per head
  constexpr int H = kWaveSize / L;   // heads at a time
  const int lane = threadIdx.x % kWaveSize;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  const int token = PIECES ? piece_row(pieces.columns)
                           : static_cast<int>(blockIdx.x);
  if (PIECES && token >= tokens) return;
  const int heads = num_q_heads + (CACHE ? 2 : 1) * num_kv_heads;
  const int waves = blockDim.x / kWaveSize;
  const int head0 = (blockIdx.y * waves + wave) * (H * UNITS) + lane / L;
  const int e = (lane % L) * 8;      // first element of this lane

  // all loads are requested before anything waits for one of them
  const int slot = CACHE ? cache.slots[token] : 0;
  const int position = positions[token];
  u32x4_any raw[UNITS], wr[UNITS];
  f32x4_any c[2], s[2];
  auto row_of = [&](int head) {
    const int kv = head - num_q_heads;           // K heads, then V heads
    return head < num_q_heads ? q + token * q_stride + head * D
        : CACHE && kv >= num_kv_heads
            ? v + token * v_stride + (kv - num_kv_heads) * D
            : k + token * k_stride + kv * D;
  };
  constexpr int kAtOnce = 6;         // pieces
  const int column = min(head0, heads - 1) * D + e;
  PieceReader reader(pieces, PIECES ? token : 0, PIECES ? column : 0);
  u32x4 got[PIECES ? kAtOnce : 1][2];
  u32x4_any add{};
  if constexpr (PIECES) {
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) got[i][h] = reader.get(i, h * 16);
    if (pieces.bias != nullptr) add = load8(pieces.bias + column);
  } else {
#pragma unroll
    for (int u = 0; u < UNITS; ++u)
      // heads past the last one repeat it
      raw[u] = load8(row_of(min(head0 + u * H, heads - 1)) + e);
  }
  auto weight_of = [&](int head) {
    return head < num_q_heads ? q_weight : k_weight;
  };
  if constexpr (NORM) {
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const u16* w = weight_of(head0 + u * H);
      wr[u] =
          load8((w != nullptr ? w : reinterpret_cast<const u16*>(cos_sin)) + e);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  const int pair = e % (D / 2);      // rotary pair of the first element
  const float* cs = cos_sin + static_cast<int64_t>(position) * D + pair;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    c[i] = *reinterpret_cast<const f32x4_any*>(cs + 4 * i);
    s[i] = *reinterpret_cast<const f32x4_any*>(cs + D / 2 + 4 * i);
  }
  __builtin_amdgcn_sched_barrier(0);
  const float sign = e < D / 2 ? -1.f : 1.f;

  // (no branch around what a load feeds: the compiler would move the load into
  // it, behind the waits for the others)
#pragma unroll
  for (int u = 0; u < UNITS; ++u) {
    const int head = head0 + u * H;
    const bool is_q = head < num_q_heads;
    const int kv = head - num_q_heads;
    const bool is_v = CACHE && kv >= num_kv_heads;
    float x[8];
    if constexpr (PIECES) {
      unpack8(add, x);
      for (;;) {
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i)
#pragma unroll
          for (int j = 0; j < 8; ++j)
            x[j] += __uint_as_float(got[i][j / 4][j % 4]);
        reader.next += kAtOnce;
        if (reader.next > reader.last) break;
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i)
#pragma unroll
          for (int h = 0; h < 2; ++h) got[i][h] = reader.get(i, h * 16);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        raw[u][i] = static_cast<u32>(f32_to_bf16(x[2 * i])) |
                    (static_cast<u32>(f32_to_bf16(x[2 * i + 1])) << 16);
    } else {
      unpack8(raw[u], x);
    }
    if constexpr (NORM) {
      const bool normed = weight_of(head) != nullptr;
      float wf[8], sum = 0.f;
      unpack8(wr[u], wf);
#pragma unroll
      for (int i = 0; i < 8; ++i) sum += x[i] * x[i];
      sum = head_sum<L>(sum);
      const float inv_rms = rsqrtf(sum / D + eps);
#pragma unroll
      for (int i = 0; i < 8; ++i)
        x[i] = normed ? x[i] * (inv_rms * wf[i]) : x[i];
    }
    // x1' = x1 cos - x2 sin in the first half, x2' = x2 cos + x1 sin
    u32x4_any bits;
    u16 y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float other = L == 16 ? dpp_move<0x128>(x[i])
                                  : __shfl_xor(x[i], L / 2);
      y[i] = f32_to_bf16(x[i] * c[i / 4][i % 4] +
                         sign * other * s[i / 4][i % 4]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      bits[i] = is_v ? raw[u][i]
                     : static_cast<u32>(y[2 * i]) |
                           (static_cast<u32>(y[2 * i + 1]) << 16);
    if (head >= heads) continue;
    if (!CACHE || is_q) {
      *reinterpret_cast<u32x4_any*>(const_cast<u16*>(row_of(head)) + e) = bits;
      continue;
    }
    if (slot < 0) continue;          // padding
    const int h = is_v ? kv - num_kv_heads : kv;
    const int64_t dst =
        ((static_cast<int64_t>(slot / cache.block_size) * num_kv_heads + h) *
             cache.block_size + slot % cache.block_size) * D + e;
    void* to = is_v ? cache.v : cache.k;
    if (FP8) {
      // the row as bf16 holds it, clamped to e4m3's largest value: the
      // conversion makes NaN of what lies beyond
      const float inv = is_v ? cache.v_inv_scale : cache.k_inv_scale;
      float f[8];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        f[i] = fminf(fmaxf(bf16_to_f32(static_cast<u16>(
                               bits[i / 2] >> (16 * (i % 2)))) * inv,
                           -448.f), 448.f);
      u32 packed[2];
      pack_fp8x8(f, packed);
      *reinterpret_cast<uint2*>(static_cast<unsigned char*>(to) + dst) =
          make_uint2(packed[0], packed[1]);
    } else {
      *reinterpret_cast<u32x4_any*>(static_cast<u16*>(to) + dst) = bits;
    }
  }
}

// of a workgroup, for so many of a token: few tokens are spread over more CUs
// (us with 16 waves and with four, 32 + 2 * 8 heads of 128: 64 tokens 2.8 and
// 2.5, 128 2.95 and 2.66, 256 3.15 and 3.05; of pieces, product and all, 6144 x
// 4096: 17 rows 17.0 and 15.5, 128 26.3 and 25.6)
int waves_of(int waves, int tokens) {
  return std::min(waves, tokens <= 256 ? 4 : kRopeWaves);
}

template <int D, int UNITS, bool NORM>
void launch_rope(u16* q, u16* k, const u16* v, int64_t q_stride,
                 int64_t k_stride, int64_t v_stride, const u16* q_weight,
                 const u16* k_weight, const float* cos_sin,
                 const int* positions, int tokens, int hq, int hk, float eps,
                 const CacheRows& cache, bool fp8, hipStream_t stream) {
  if (tokens == 0) return;
  const int waves = ceil_div(hq + (v ? 2 : 1) * hk,
                             kWaveSize / (D / 8) * UNITS);
  auto kernel = !v ? &rope_qk_norm_kernel<D, false, false, UNITS, false, NORM>
      : fp8 ? &rope_qk_norm_kernel<D, true, true, UNITS, false, NORM>
            : &rope_qk_norm_kernel<D, true, false, UNITS, false, NORM>;
  const int at_once = waves_of(waves, tokens);
  hipLaunchKernelGGL(kernel, dim3(tokens, ceil_div(waves, at_once)),
                     dim3(at_once * kWaveSize), 0, stream, q, k, v, q_stride,
                     k_stride, v_stride, q_weight, k_weight, cos_sin,
                     positions, hq, hk, eps, cache, PieceRows{}, tokens);
}

template <int D, bool NORM>
void launch_of_pieces(u16* q, const PieceRows& pieces, const RopeArgs& a,
                      int tokens, hipStream_t stream) {
  const CacheRows cache{a.k_cache, a.v_cache, a.slots, a.block_size,
                        a.k_inv_scale, a.v_inv_scale};
  const int waves = ceil_div(a.num_q_heads + 2 * a.num_kv_heads,
                             kWaveSize / (D / 8));
  auto kernel = a.fp8 ? &rope_qk_norm_kernel<D, true, true, 1, true, NORM>
                      : &rope_qk_norm_kernel<D, true, false, 1, true, NORM>;
  const int at_once = waves_of(waves, tokens);
  hipLaunchKernelGGL(
      kernel, dim3(ceil_div(tokens, 16) * 16, ceil_div(waves, at_once)),
      dim3(at_once * kWaveSize), 0, stream, q, nullptr,
      nullptr, static_cast<int64_t>(a.num_q_heads) * D, 0, 0, a.q_weight,
      a.k_weight, a.cos_sin, a.positions, a.num_q_heads, a.num_kv_heads,
      a.eps, cache, pieces, tokens);
}

}  // namespace

// head_dim 64 or 128; without v the K rows stay in place
void launch_rope_qk_norm(u16* q, u16* k, const u16* v, int64_t q_stride,
                         int64_t k_stride, int64_t v_stride,
                         const u16* q_weight, const u16* k_weight,
                         const float* cos_sin, const int* positions,
                         int tokens, int num_q_heads, int num_kv_heads,
                         int head_dim, float eps, void* k_cache,
                         void* v_cache, const int* slots, int block_size,
                         bool fp8, float k_inv_scale, float v_inv_scale,
                         hipStream_t stream) {
  const CacheRows cache{k_cache, v_cache, slots, block_size, k_inv_scale,
                        v_inv_scale};
  // from 2^22 values on a wave takes twice the heads: cos, sin and weights
  // once, twice the loads on the way (8765 tokens, 32 + 2 * 8 heads of 128: 48
  // us with one unit, 38 with two; 512 tokens 4.1 and 4.5; 1000 tokens of 64 + 2
  // * 8 heads without a norm 9.8 and 8.9)
  const bool many = static_cast<int64_t>(tokens) * head_dim *
                        (num_q_heads + (v ? 2 : 1) * num_kv_heads) >= 1 << 22;
  const bool norm = q_weight != nullptr || k_weight != nullptr;
#define FI_ROPE(D, U, NORM)                                                    \
  launch_rope<D, U, NORM>(q, k, v, q_stride, k_stride, v_stride, q_weight,     \
                          k_weight, cos_sin, positions, tokens, num_q_heads,   \
                          num_kv_heads, eps, cache, fp8, stream)
#define FI_ROPE_N(D, U)                                                        \
  do {                                                                         \
    if (norm) FI_ROPE(D, U, true);                                             \
    else FI_ROPE(D, U, false);                                                 \
  } while (0)
  if (head_dim == 128) {
    if (many) FI_ROPE_N(128, 2);
    else FI_ROPE_N(128, 1);
  } else {
    if (many) FI_ROPE_N(64, 2);
    else FI_ROPE_N(64, 1);
  }
#undef FI_ROPE_N
#undef FI_ROPE
}

// q [tokens, num_q_heads * head_dim] and the cache's rows, from a product in
// pieces; head_dim 64 or 128
void launch_rope_of_pieces(u16* q, const PieceRows& pieces, const RopeArgs& a,
                           int tokens, hipStream_t stream) {
  const bool norm = a.q_weight != nullptr || a.k_weight != nullptr;
  auto launch = a.head_dim == 128
      ? (norm ? &launch_of_pieces<128, true> : &launch_of_pieces<128, false>)
      : (norm ? &launch_of_pieces<64, true> : &launch_of_pieces<64, false>);
  launch(q, pieces, a, tokens, stream);
}

}  // namespace fi
