// Common device helpers for FusionInfer-AMD CDNA4 (gfx950) kernels.
//
// Design notes:
//  * wave64 everywhere; block sizes are multiples of 64.
//  * bf16 loads are ALWAYS vectorized (short4/short8 reinterpret).
//  * bf16<->f32 via bit ops (RNE) — matches hardware v_cvt rounding.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>

#define FI_DEV __device__ __forceinline__

namespace fi {

constexpr int kWaveSize = 64;

using u16 = unsigned short;
using u32 = unsigned int;

// 16-byte vector of 8 bf16 values (raw bits).
struct alignas(16) bf16x8 {
  u16 h[8];
};
// 8-byte vector of 4 bf16 values.
struct alignas(8) bf16x4 {
  u16 h[4];
};

FI_DEV float bf16_to_f32(u16 h) {
  union {
    u32 u;
    float f;
  } x;
  x.u = static_cast<u32>(h) << 16;
  return x.f;
}

FI_DEV u16 f32_to_bf16(float f) {
  // native cast -> ONE v_cvt_pk_bf16_f32 (RNE, NaN-safe); the manual
  // bit-twiddled RNE this replaces cost ~6 VALU ops per element
  union {
    u16 u;
    __bf16 h;
  } c;
  c.h = static_cast<__bf16>(f);
  return c.u;
}

template <int CTRL>
FI_DEV float dpp_move(float x) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL,
                                         0xF, 0xF, true));
}

// Wave-wide reductions (64 lanes, all of them active), by exchanges with the
// lane 32, 16, 8, 4, 2 and 1 away. They stay among the registers: six of them
// through LDS, as __shfl_xor has them, take 700 cycles. Swapping a register
// with itself leaves either half's (row's) value in one of two; after the
// exchange over 8 lanes a row has period 8, so a rotation by 4 reaches the
// lane 4 away.
template <class Op>
FI_DEV float wave_reduce(float v, Op op) {
#if defined(__HIP_DEVICE_COMPILE__)
  const auto h = __builtin_amdgcn_permlane32_swap(
      __float_as_int(v), __float_as_int(v), false, false);
  v = op(__int_as_float(h[0]), __int_as_float(h[1]));
  const auto r = __builtin_amdgcn_permlane16_swap(
      __float_as_int(v), __float_as_int(v), false, false);
  v = op(__int_as_float(r[0]), __int_as_float(r[1]));
  v = op(v, dpp_move<0x128>(v));   // row_ror:8
  v = op(v, dpp_move<0x124>(v));   // row_ror:4
  v = op(v, dpp_move<0x4E>(v));    // quad_perm [2,3,0,1]
  v = op(v, dpp_move<0xB1>(v));    // quad_perm [1,0,3,2]
#endif
  return v;
}

FI_DEV float wave_reduce_sum(float v) {
  return wave_reduce(v, [](float a, float b) { return a + b; });
}

FI_DEV float wave_reduce_max(float v) {
  return wave_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}

// Block-wide sum over NWAVES waves (each wave passes its wave-reduced value
// with lane 0 valid). `scratch` must hold NWAVES floats.
template <int NWAVES>
FI_DEV float block_reduce_sum(float wave_val, float* scratch) {
  const int wave = threadIdx.x / kWaveSize;
  const int lane = threadIdx.x % kWaveSize;
  if (lane == 0) scratch[wave] = wave_val;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int i = 0; i < NWAVES; ++i) total += scratch[i];
  return total;
}

// 8 or 16 bytes to global memory. Where a pointer has been through asm the
// compiler no longer sees that it is one to there; its store is then a flat one,
// which LDS waits wait for too and which a counted wait must not rely on the
// order of.
template <class T>
FI_DEV void store_global(u16* to, const T& value) {
  typedef __attribute__((ext_vector_type(sizeof(T) / 4))) u32 Words;
  *(__attribute__((address_space(1))) Words*)to =
      __builtin_bit_cast(Words, value);
}

// more than the memory-side cache holds: what is read once better goes past it
inline bool beyond_caches(int64_t bytes) { return bytes > int64_t{256} << 20; }

__host__ __device__ __forceinline__ constexpr int ceil_div(int a, int b) {
  return (a + b - 1) / b;
}

// How a launch of the prefill attention kernel is laid out: query heads and
// rows of a workgroup, workgroup row blocks per tile-table entry and in all,
// whether K/V ranges are cut into equal parts, and the longest context's bound.
struct PrefillPlan {
  int waves, hpb, rows, sub, nq, slots, longest;
  bool split, pair;
};

// Heads of a projection's rows that are normed per head, rotated and kept in the
// paged cache [num_blocks, Hk, block_size, head_dim].
struct RopeArgs {
  const u16* q_weight;    // [head_dim] or nullptr
  const u16* k_weight;
  const float* cos_sin;   // [P, head_dim], cos | sin
  const int* positions;   // [T]
  int num_q_heads, num_kv_heads, head_dim;
  float eps;
  void* k_cache;
  void* v_cache;
  const int* slots;       // [T], negative: the row is not kept
  int block_size;
  bool fp8;
  float k_inv_scale, v_inv_scale;
};

// What the kernel for few rows does beside out = x W^T, by what is not null.
// squares_in [parts][16]: rows of x are divided by the root mean square that
// these have as sums of squares of K values. add: the product is added to it,
// fp32, in place of out; with norm scaled [M, N] gets the sums times norm, and
// squares_out [N / 16][16] their squares. gelu: of the product.
struct SkinnyExtra {
  const float* squares_in = nullptr;
  int parts = 0;
  float eps = 0.f;
  float* add = nullptr;
  const u16* norm = nullptr;
  u16* scaled = nullptr;
  float* squares_out = nullptr;
  bool gelu = false;
};

// v / (1 + e), the bits of the division (all 2^32 values of silu compared) in
// half its instructions: with one wave per SIMD an epilogue hides none of
// them. A reciprocal (of a quarter of the divisor, since those below the normal
// range come out as zero), the quotient, its remainder times the reciprocal
// added, infinities and NaN put right. (The reciprocal alone, a unit off in
// the last place, saves 1 % of a GEMM: 24576 x 4096 at 8192 rows 1084 us, and
// 1095.)
FI_DEV float over_one_plus(float v, float e) {
#if defined(__HIP_DEVICE_COMPILE__)
  const float d = 1.f + e;
  const float r = __builtin_amdgcn_rcpf(fmaf(e, 0.25f, 0.25f)) * 0.25f;
  const float q = v * r;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, v), r, q), d, v);
#else
  return 0.f;
#endif
}
FI_DEV float silu(float v) { return over_one_plus(v, __expf(-v)); }
// the tanh form: 0.5 (1 + tanh(a)) is 1 / (1 + exp(-2 a))
FI_DEV float gelu(float v) {
  return over_one_plus(
      v, __expf(-1.5957691216057308f * (v + 0.044715f * v * v * v)));
}

// pack 8 f32 into 8 OCP-e4m3 bytes (two u32 words) via v_cvt_pk_fp8_f32
FI_DEV void pack_fp8x8(const float* v, unsigned int out[2]) {
#if defined(__HIP_DEVICE_COMPILE__)
  unsigned int w0 = 0, w1 = 0;
  w0 = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], w0, false);
  w0 = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], w0, true);
  w1 = __builtin_amdgcn_cvt_pk_fp8_f32(v[4], v[5], w1, false);
  w1 = __builtin_amdgcn_cvt_pk_fp8_f32(v[6], v[7], w1, true);
  out[0] = w0;
  out[1] = w1;
#else
  out[0] = out[1] = 0;  // host pass never executes device code
#endif
}

// unpack 4 OCP-e4m3 bytes (one u32) -> 4 f32 via v_cvt_pk_f32_fp8
FI_DEV void unpack_fp8x4(u32 w, float out[4]) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(w, false);
  const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(w, true);
  out[0] = lo[0];
  out[1] = lo[1];
  out[2] = hi[0];
  out[3] = hi[1];
#else
  out[0] = out[1] = out[2] = out[3] = 0.f;
#endif
}

// 16 bytes per lane from global memory straight to LDS: lane l's land at
// lds + 16 l. Base and LDS address are wave-uniform, the byte offset is per
// lane. In asm because the compiler makes every LDS read wait for all DMAs
// it knows of; whoever reads the data waits with s_waitcnt vmcnt (DMAs of a
// wave complete in order) and, for other waves' data, a barrier. The wait
// states are those of an m0 write and of a base that the vector unit wrote.
FI_DEV void dma_to_lds16(u32 lds, const void* base, u32 offset) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 4\n\t"
      "global_load_lds_dwordx4 %1, %2"
      :
      : "s"(lds), "v"(offset), "s"(base)
      : "memory");  // m0: reserved, set in front of every use
#endif
}

// the same with an address of its own per lane
FI_DEV void dma_to_lds16_at(u32 lds, const void* from) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 4\n\t"
      "global_load_lds_dwordx4 %1, off"
      :
      : "s"(lds), "v"(from)
      : "memory");
#endif
}

// the same for data that is read once: it leaves the caches first
FI_DEV void dma_to_lds16_nt(u32 lds, const void* base, u32 offset) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 4\n\t"
      "global_load_lds_dwordx4 %1, %2 nt"
      :
      : "s"(lds), "v"(offset), "s"(base)
      : "memory");
#endif
}

// the same through a buffer descriptor (base, 0, bytes, format): scalar
// base + vector offset + scalar offset; what lies behind the end reads as 0
typedef __attribute__((ext_vector_type(4))) u32 u32x4;
FI_DEV u32x4 descriptor_of(const void* p, u32 bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  return u32x4{static_cast<u32>(a), static_cast<u32>(a >> 32), bytes,
               0x00020000u};
}
FI_DEV void buffer_to_lds16(u32 lds, u32x4 desc, u32 voff, u32 soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 4\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen lds"
      :
      : "s"(lds), "v"(voff), "s"(desc), "s"(soff)
      : "memory");
#endif
}

// 16-byte loads at scalar base + vector offset + scalar offset (bytes)
#if defined(__HIP_DEVICE_COMPILE__)
typedef __amdgpu_buffer_rsrc_t BufferRsrc;
FI_DEV BufferRsrc buffer_of(const void* p, u32 bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes,
                                           0x00020000);
}
FI_DEV u32x4 buffer_load16(BufferRsrc r, u32 voff, u32 soff) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
}
#else
struct BufferRsrc {};
FI_DEV BufferRsrc buffer_of(const void*, u32) { return {}; }
FI_DEV u32x4 buffer_load16(BufferRsrc, u32, u32) { return {}; }
#endif

// Integers that no kernel of the launch writes, read through the scalar
// cache (at a wave-uniform index they return on lgkmcnt, not behind the
// DMAs).
typedef const __attribute__((address_space(4))) int* ConstInts;
FI_DEV ConstInts const_ints(const int* p) {
  return (ConstInts)(reinterpret_cast<uintptr_t>(p));
}

// Transposing LDS read of 16-bit values: within 16 lanes, lane 4i+j points
// at entries 4j..4j+3 of row i of a 4 x 16 block and receives the four rows'
// entries of column (lane & 15).
FI_DEV __attribute__((ext_vector_type(4))) short lds_read_tr4(
    const unsigned char* p) {
  typedef __attribute__((ext_vector_type(4))) short v4;
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) v4*)(p));
#else
  return v4{0, 0, 0, 0};
#endif
}

// A softmax weight for the bf16 matrix cores without loss: three terms of
// eight bits each, by truncation, add up to the fp32 value. No term is 0, so
// that an infinite operand stays what it is; 2^-126 of a finite one is nothing.
FI_DEV void split_weight(float p, u16 (&terms)[3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    p = fmaxf(p, 0x1p-126f);
    const u32 top = __float_as_uint(p) & 0xffff0000u;
    terms[i] = static_cast<u16>(top >> 16);
    p -= __uint_as_float(top);
  }
}

template <int NWAVES>
FI_DEV float block_reduce_max(float wave_val, float* scratch) {
  const int wave = threadIdx.x / kWaveSize;
  const int lane = threadIdx.x % kWaveSize;
  if (lane == 0) scratch[wave] = wave_val;
  __syncthreads();
  float m = scratch[0];
#pragma unroll
  for (int i = 1; i < NWAVES; ++i) m = fmaxf(m, scratch[i]);
  return m;
}

}  // namespace fi
