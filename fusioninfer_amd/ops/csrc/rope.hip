// Fused per-head RMSNorm (Qwen3 qk-norm) + NeoX rotary embedding of Q and K
// rows, in place, or (CACHE) with the K rows and the untouched V rows going
// straight into the paged cache [num_blocks, Hk, block_size, D].
//
// Bound by memory: every row is read and written once. A lane holds eight
// elements, so D / 8 lanes hold a head and a wave four heads (D = 128) or
// eight (64) of one token; the rotate-half partner is D / 16 lanes away in
// the same row of 16 lanes, and the norm's sum is three or four exchanges
// within it. One wave per (token, head) with two elements per lane and a
// second kernel for the cache took 87 + 9 us at 8765 tokens, 32 + 2 * 4
// heads of 128; this takes 41 us (4.4 TB/s). cos/sin come from a table (f32
// [P, D], cos | sin): sines computed here would make it bound by the VALU.
//
// Capability parity: RoPE / qk-norm epilogue and cache write the reference
// delegates to vLLM.

#include "common.h"

namespace fi {

namespace {

// rows are slices of the projections' output: no alignment is assumed
typedef u32 u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kRopeWaves = 4;

FI_DEV void load8(const u16* p, float v[8]) {
  const u32x4_any w = *reinterpret_cast<const u32x4_any*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = bf16_to_f32(static_cast<u16>(w[i] & 0xffff));
    v[2 * i + 1] = bf16_to_f32(static_cast<u16>(w[i] >> 16));
  }
}

struct CacheRows {
  void* k;           // [num_blocks, Hk, block_size, D] bf16 or e4m3
  void* v;
  const int* slots;  // [T], negative: the row is not kept
  int block_size;
  float k_inv_scale, v_inv_scale;  // fp8 only
};

template <int D, bool CACHE, bool FP8>
__global__ __launch_bounds__(kRopeWaves * kWaveSize) void rope_qk_norm_kernel(
    u16* __restrict__ q,             // [T, Hq*D] rows, stride q_stride
    u16* __restrict__ k,             // [T, Hk*D] rows, stride k_stride
    const u16* __restrict__ v,       // CACHE: [T, Hk*D] rows
    const int64_t q_stride, const int64_t k_stride, const int64_t v_stride,
    const u16* __restrict__ q_weight,  // [D] or nullptr
    const u16* __restrict__ k_weight,  // [D] or nullptr
    const float* __restrict__ cos_sin,  // [P, D]
    const int* __restrict__ positions,  // [T]
    const int tokens, const int num_q_heads, const int num_kv_heads,
    const int groups,                // waves per token
    const float eps, const CacheRows cache) {
  constexpr int L = D / 8;           // lanes per head
  const int lane = threadIdx.x % kWaveSize;
  const u32 unit = __builtin_amdgcn_readfirstlane(
      blockIdx.x * kRopeWaves + threadIdx.x / kWaveSize);
  const int token = unit / groups;
  if (token >= tokens) return;
  const int head = (unit - token * groups) * (kWaveSize / L) + lane / L;
  if (head >= num_q_heads + (CACHE ? 2 : 1) * num_kv_heads) return;
  const int e = (lane % L) * 8;      // first element of this lane
  const bool is_q = head < num_q_heads;
  const int kv = head - num_q_heads;             // K heads, then V heads
  const bool is_v = CACHE && kv >= num_kv_heads;

  // (requested here, not at its use behind the sums)
  const int slot = CACHE ? cache.slots[token] : 0;
  const u16* row = is_q ? q + token * q_stride + head * D
      : is_v ? v + token * v_stride + (kv - num_kv_heads) * D
             : k + token * k_stride + kv * D;
  float x[8];
  load8(row + e, x);

  if (!is_v) {
    const int pair = e % (D / 2);    // rotary pair of the first element
    const float* cs = cos_sin + static_cast<int64_t>(positions[token]) * D +
                      pair;
    f32x4_any c[2], s[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      c[i] = *reinterpret_cast<const f32x4_any*>(cs + 4 * i);
      s[i] = *reinterpret_cast<const f32x4_any*>(cs + D / 2 + 4 * i);
    }
    const u16* w = is_q ? q_weight : k_weight;
    if (w != nullptr) {
      float wf[8];
      load8(w + e, wf);
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) sum += x[i] * x[i];
#pragma unroll
      for (int off = L / 2; off > 0; off >>= 1) {
        if (off == 8) sum += dpp_move<0x128>(sum);       // row_ror:8
        else if (off == 4 && L == 16) sum += dpp_move<0x124>(sum);  // :4
        else if (off == 2) sum += dpp_move<0x4E>(sum);
        else if (off == 1) sum += dpp_move<0xB1>(sum);
        else sum += __shfl_xor(sum, off);
      }
      const float inv_rms = rsqrtf(sum / D + eps);
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] *= inv_rms * wf[i];
    }
    // x1' = x1 cos - x2 sin in the first half, x2' = x2 cos + x1 sin
    const float sign = e < D / 2 ? -1.f : 1.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float other = L == 16 ? dpp_move<0x128>(x[i])
                                  : __shfl_xor(x[i], L / 2);
      x[i] = x[i] * c[i / 4][i % 4] + sign * other * s[i / 4][i % 4];
    }
  }

  u32x4_any bits;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    bits[i] = static_cast<u32>(f32_to_bf16(x[2 * i])) |
              (static_cast<u32>(f32_to_bf16(x[2 * i + 1])) << 16);
  if (!CACHE || is_q) {
    *reinterpret_cast<u32x4_any*>(const_cast<u16*>(row) + e) = bits;
    return;
  }
  if (slot < 0) return;              // padding
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

template <int D>
void launch_rope(u16* q, u16* k, const u16* v, int64_t q_stride,
                 int64_t k_stride, int64_t v_stride, const u16* q_weight,
                 const u16* k_weight, const float* cos_sin,
                 const int* positions, int tokens, int hq, int hk, float eps,
                 const CacheRows& cache, bool fp8, hipStream_t stream) {
  const int groups = ceil_div(hq + (v ? 2 : 1) * hk, kWaveSize / (D / 8));
  const int64_t units = static_cast<int64_t>(tokens) * groups;
  if (units == 0) return;
  auto kernel = !v ? &rope_qk_norm_kernel<D, false, false>
      : fp8 ? &rope_qk_norm_kernel<D, true, true>
            : &rope_qk_norm_kernel<D, true, false>;
  hipLaunchKernelGGL(kernel, dim3((units + kRopeWaves - 1) / kRopeWaves),
                     dim3(kRopeWaves * kWaveSize), 0, stream, q, k, v,
                     q_stride, k_stride, v_stride, q_weight, k_weight,
                     cos_sin, positions, tokens, hq, hk, groups, eps, cache);
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
  if (head_dim == 128)
    launch_rope<128>(q, k, v, q_stride, k_stride, v_stride, q_weight,
                     k_weight, cos_sin, positions, tokens, num_q_heads,
                     num_kv_heads, eps, cache, fp8, stream);
  else
    launch_rope<64>(q, k, v, q_stride, k_stride, v_stride, q_weight,
                    k_weight, cos_sin, positions, tokens, num_q_heads,
                    num_kv_heads, eps, cache, fp8, stream);
}

}  // namespace fi
