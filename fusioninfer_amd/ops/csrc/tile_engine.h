// Pieces of the kernels in which one wave per SIMD holds 128 x 128 results:
// DMAs to LDS whose base register is set apart from the load, matrix products
// on accumulation registers, waits that the compiler does not see.

#pragma once

#include "common.h"

namespace fi {

typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) float floatx4;
typedef __attribute__((ext_vector_type(16))) float floatx16;
typedef __attribute__((ext_vector_type(4))) int intx4;
typedef __attribute__((ext_vector_type(8))) int intx8;

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
// the same for data that is read once: it leaves the caches first
FI_DEV void load_lds_nt(u32x4 desc, u32 voff, u32 soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("buffer_load_dwordx4 %0, %1, %2 offen nt lds"
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
FI_DEV void mfma(floatx16& acc, const intx8& w, const intx8& x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_32x32x64_f8f6f4 %0, %1, %2, %0"
               : "+a"(acc)
               : "v"(w), "v"(x));
#endif
}
// acc = w x^T: a tile's first products
FI_DEV void mfma_first(floatx4& acc, const short8& w, const short8& x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0"
               : "=a"(acc)
               : "v"(w), "v"(x));
#endif
}
FI_DEV void mfma_first(floatx16& acc, const intx8& w, const intx8& x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("v_mfma_f32_32x32x64_f8f6f4 %0, %1, %2, 0"
               : "=a"(acc)
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

}  // namespace fi
