// Grouped MFMA GEMM for long expert segments (128-row blocks, prompts).
//
// A workgroup computes 128 rows by 256 columns (128 gate and the same 128 up
// columns where the epilogue joins them) with four waves side by side in N:
//  * the A tile is shared: 64 values of K of 128 gathered rows per stage go
//    to LDS by DMA, two stages ahead, three buffers, one barrier a stage;
//  * every wave owns 64 columns of B, so its packed fragments go straight
//    from global memory to registers, two 32-deep steps ahead (a third step
//    ahead spills), and no byte of B passes through LDS or is loaded twice
//    in a workgroup.
// Per 32 of K a wave issues 32 MFMAs (512 cycles) against 8 LDS reads and 4
// loads; two waves per SIMD. The form before (64/128 columns, two waves per
// column, a full wait and barrier every 32 of K) spent its time in those
// waits and in loading B twice.
// MFMA operands are B, A: a lane ends with four neighbouring columns of a
// row and stores 8 bytes.
// Workgroups of one XCD take a contiguous run of tiles, eight row blocks by
// all column tiles at a time, so an expert's B is read into one L2 and A
// rows stay there over the column tiles.
//
// Measured, us (TFLOP/s of the real rows), before -> now: 8765 rows, 128
// experts, top 8, width 2048, 768 per expert: gate|up 993 (444) -> 546
// (808), down 766 (288) -> 323 (682; an eighth of the tiles is padding);
// 8192 rows, 8 experts, top 2, 2048 x 3072: 571 -> 370 (1114), 427 -> 209
// (986); 4096 x 6144: 2774 -> 1429 (1154), 2087 -> 773 (1067).

#include <hip/hip_runtime.h>

#include "common.h"

namespace fi {

namespace {

typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) float floatx4;

constexpr int kTileM = 128, kStageB = kTileM * 128;  // 64 bf16 per row
constexpr int kRowGroup = 8;                         // row blocks of a group

template <int MODE>
__global__ __launch_bounds__(256, 2) void moe_tile_kernel(
    u16* __restrict__ out,              // [PM, N]
    const u16* __restrict__ a,          // gathered x [T, K]; MODE 0 [PM, K]
    const u16* __restrict__ b,          // [E][K/32][NB/16][64][8]
    const int* __restrict__ sorted_ids, // [PM]
    const int* __restrict__ expert_ids, // [PM/128]
    const int* __restrict__ n_valid, const int K, const int N, const int NT,
    const u32 a_bytes, const float limit) {
  constexpr bool GATE_UP = MODE == 1 || MODE == 3;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[3 * kStageB];
  const u32 lds0 = static_cast<u32>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) unsigned char*)smem));

  // tile of this workgroup
  const int nv = const_ints(n_valid)[0];
  const int total = nv * NT, per = (total + 7) / 8;
  const int j8 = blockIdx.x >> 3;
  const int at = (blockIdx.x & 7) * per + j8;
  if (j8 >= per || at >= total) return;
  const int m_lo = at / (kRowGroup * NT) * kRowGroup;
  const int m_n = min(kRowGroup, nv - m_lo);
  const int in = at - m_lo * NT;
  const int ntile = in / m_n, mtile = m_lo + in % m_n;

  const int lane = threadIdx.x % kWaveSize;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  const int e = const_ints(expert_ids)[mtile];
  const int ksteps = K / 32;
  // the main loop takes 128 of K at a time; what is left over goes first
  const int head = ksteps % 4, stages = (ksteps - head) / 2;

  // ---- A: wave w copies rows 32w..32w+31, eight per DMA; 16-byte chunk c
  // of row r sits at c ^ (r >> 1 & 7)
  u32 a_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = wave * 32 + i * 8 + (lane >> 3);
    const int row = MODE != 0 ? sorted_ids[mtile * kTileM + r] : r;
    a_off[i] = static_cast<u32>(row) * (K * 2) +
               ((lane & 7) ^ ((r >> 1) & 7)) * 16;
  }
  const u32x4 a_desc = descriptor_of(
      MODE != 0 ? a : a + static_cast<int64_t>(mtile) * kTileM * K,
      MODE != 0 ? a_bytes : kTileM * K * 2);
  auto stage_a = [&](int s, int buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      buffer_to_lds16(lds0 + buf * kStageB + (wave * 32 + i * 8) * 128,
                      a_desc, a_off[i], head * 64 + s * 128);
  };

  // ---- B fragments of this wave: two gate and two up, or four
  const int NB16 = (GATE_UP ? 2 * N : N) / 16;
  const int n16 = GATE_UP ? ntile * 8 + wave * 2 : ntile * 16 + wave * 4;
  // scalar base and step offsets, one vector offset for all of them
  const u32 b_step = static_cast<u32>(NB16) * 1024;
  const auto b_rsrc = buffer_of(
      b + static_cast<int64_t>(e) * ksteps * NB16 * 512, ksteps * b_step);
  u32 b_f[4];
#pragma unroll
  for (int f = 0; f < 4; ++f)
    b_f[f] = (min(n16 + (GATE_UP ? f & 1 : f), N / 16 - 1) +
              (GATE_UP && f >= 2 ? N / 16 : 0)) * 1024;
  short8 bw[4][4];
  auto load_b = [&](int kt, short8 (&dst)[4]) {
    const u32 off = min(kt, ksteps - 1) * b_step;
#pragma unroll
    for (int f = 0; f < 4; ++f)
      dst[f] = __builtin_bit_cast(
          short8, buffer_load16(b_rsrc, lane * 16, b_f[f] + off));
  };

  // fragment reads: row lane & 15, chunk 4 (k step & 1) + (lane >> 4)
  int f_off[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    f_off[h] = (lane & 15) * 128 +
               (((h * 4 + (lane >> 4)) ^ ((lane & 15) >> 1)) * 16);

  floatx4 acc[8][4];
#pragma unroll
  for (int mi = 0; mi < 8; ++mi)
#pragma unroll
    for (int f = 0; f < 4; ++f) acc[mi][f] = {0.f, 0.f, 0.f, 0.f};

  if (stages) {
    stage_a(0, 0);
    stage_a(1, 1);
  }
  for (int kt = 0; kt < head; ++kt) {
    load_b(kt, bw[0]);
#pragma unroll
    for (int mi = 0; mi < 8; ++mi) {
      const int r = mi * 16 + (lane & 15);
      const int row = MODE != 0 ? sorted_ids[mtile * kTileM + r] : r;
      const short8 av = *reinterpret_cast<const short8*>(
          (MODE != 0 ? a : a + static_cast<int64_t>(mtile) * kTileM * K) +
          static_cast<int64_t>(row) * K + kt * 32 + (lane >> 4) * 8);
#pragma unroll
      for (int f = 0; f < 4; ++f)
        acc[mi][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            bw[0][f], av, acc[mi][f], 0, 0, 0);
    }
  }
  load_b(head, bw[0]);
  load_b(head + 1, bw[1]);
  int buf = 2;
  auto next_stage = [&](int stage) {
    // This stage's rows were requested two stages ago; at least 12 of this
    // wave's loads are younger (B of the steps since). Then all waves have
    // theirs, and nobody reads the buffer filled next.
    asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    buf = buf == 2 ? 0 : buf + 1;
    if (stage + 2 < stages) stage_a(stage + 2, buf == 0 ? 2 : buf - 1);
  };
  auto step = [&](int kt, int half, short8 (&use)[4], short8 (&fill)[4]) {
    load_b(kt + 2, fill);
    // requested here, not where the scheduler finds a free register
    __builtin_amdgcn_sched_barrier(0);
    const unsigned char* as = smem + buf * kStageB + f_off[half];
#pragma unroll
    for (int mi = 0; mi < 8; ++mi) {
      const short8 av = *reinterpret_cast<const short8*>(as + mi * 16 * 128);
#pragma unroll
      for (int f = 0; f < 4; ++f)
        acc[mi][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            use[f], av, acc[mi][f], 0, 0, 0);
    }
  };
  for (int s = 0; s < stages; s += 2) {
    const int kt = head + s * 2;
    next_stage(s);
    step(kt, 0, bw[0], bw[2]);
    step(kt + 1, 1, bw[1], bw[3]);
    next_stage(s + 1);
    step(kt + 2, 0, bw[2], bw[0]);
    step(kt + 3, 1, bw[3], bw[1]);
  }

#pragma unroll
  for (int mi = 0; mi < 8; ++mi) {
    u16* row = out + static_cast<int64_t>(mtile * kTileM + mi * 16 +
                                          (lane & 15)) * N + (lane >> 4) * 4;
#pragma unroll
    for (int f = 0; f < (GATE_UP ? 2 : 4); ++f) {
      if (n16 + f >= N / 16) continue;
      bf16x4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = acc[mi][f][r];
        if (MODE == 3) {
          const float gt = fminf(v, limit);
          const float up =
              fminf(fmaxf(acc[mi][f + 2][r], -limit), limit);
          v = (gt / (1.f + __expf(-1.702f * gt))) * (up + 1.f);
        } else if (MODE == 1) {
          v = (v / (1.f + __expf(-v))) * acc[mi][f + 2][r];
        } else if (MODE == 2) {
          v = fmaxf(v, 0.f);
          v *= v;
        }
        o.h[r] = f32_to_bf16(v);
      }
      *reinterpret_cast<bf16x4*>(row + (n16 + f) * 16) = o;
    }
  }
}

}  // namespace

void launch_moe_tile(u16* out, const u16* a, const u16* b,
                     const int* sorted_ids, const int* expert_ids,
                     const int* n_valid, int max_mtiles, int rows, int K,
                     int N, int mode, float limit, hipStream_t stream) {
  const int nt = ceil_div(N, mode == 1 || mode == 3 ? 128 : 256);
  const dim3 grid(ceil_div(max_mtiles * nt, 8) * 8);
#define FI_TILE(M)                                                            \
  hipLaunchKernelGGL((moe_tile_kernel<M>), grid, dim3(256), 0, stream, out,   \
                     a, b, sorted_ids, expert_ids, n_valid, K, N, nt,        \
                     static_cast<u32>(rows) * (K * 2), limit)
  if (mode == 1) FI_TILE(1);
  else if (mode == 2) FI_TILE(2);
  else if (mode == 3) FI_TILE(3);
  else FI_TILE(0);
#undef FI_TILE
}

}  // namespace fi
