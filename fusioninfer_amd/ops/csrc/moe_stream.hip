// Grouped expert GEMM for blocks of 16 rows, the few rows per expert of a
// decode step: bound by reading the weights of the experts in use once.
//
// A unit is a block of 16 rows by 16 * COLS output columns. The units of all
// blocks in use form one row, cut into 256 equal parts, one workgroup of
// eight waves each: no wave of workgroups is nearly empty, whatever the
// routing. The waves split K. Weights are packed in fragment order, so a wave
// reads them straight into registers, a kilobyte per load, the loads of the
// next stretch in flight while this one is multiplied (128 KB per CU); they
// are read once and marked so. A wave keeps its slice of the rows in
// registers from one unit to the next (KEEP) where the slice fits: rows read
// again for every 16 columns cost half the weights' traffic between L2 and
// the CUs, which ends at about 10 TB/s. The waves' sums meet in LDS, one
// barrier per unit, one wave after the other writing the result. All rows and
// weights are addressed in 64 bits: blocks of 128 rows whose operands are too
// large for the tiles' 32-bit offsets come here as eight of 16.
//
// The fragments of the weights are the first operand, so a lane ends with
// four neighbouring columns of one row.
//
// 128 experts, K 2048, gate and up of 768, then K 768, N 2048, us (GB/s of
// the weights in use) at 1 / 8 / 64 tokens of 8 experts each: 10.4 + 7.0 / 52
// (6430) + 31 / 132 (5990) + 72 (5500); one wave per 16 columns with all of K
// and the rows read again for each: 26 + 17 / 82 + 37 / 148 (5340) + 86
// (4580).

#include <hip/hip_runtime.h>

#include "common.h"

namespace fi {

namespace {

typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) float floatx4;

constexpr int kStreamWaves = 8;

FI_DEV short8 load_once(const u16* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const short8*>(p));
}

// MODE 0: plain GEMM over act rows; 1: gathered x rows, gate | up columns,
// silu(gate) * up; 2: gathered x rows, up alone, relu(up)^2; 3: as 1 with the
// clamped unit g' sigmoid(1.702 g') (u' + 1), g' = min(g, limit), u' =
// clamp(u, -limit, limit). C: steps of 32 of K that a wave requests together.
template <int MODE, int C, int COLS, bool KEEP>
__global__ __launch_bounds__(kStreamWaves * kWaveSize)
void moe_stream_kernel(
    u16* __restrict__ out,              // [PM, N] bf16
    const u16* __restrict__ a,          // MODE 0: act [PM, K]; else x [T, K]
    const u16* __restrict__ b,          // [E][K/32][NB/16][64][8] bf16
    const int* __restrict__ sorted_ids, // [PM] token row per padded slot
    const int* __restrict__ expert_ids, // local expert of 16 << per rows
    const int* __restrict__ n_valid,    // device scalar: those in use
    const int per, const int K, const int N, const float limit) {
  constexpr bool GATE_UP = MODE == 1 || MODE == 3;
  constexpr int NF = GATE_UP ? 2 * COLS : COLS;   // fragments per step
  __shared__ floatx4 sums[2][kStreamWaves][NF][kWaveSize];

  const int lane = threadIdx.x % kWaveSize;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  const int per_block = N / (16 * COLS);          // units of a row block
  const int units = (*n_valid << per) * per_block;
  const int each = units / gridDim.x, rem = units % gridDim.x;
  const int part = blockIdx.x;
  const int lo = part * each + min(part, rem);
  const int hi = lo + each + (part < rem ? 1 : 0);
  if (lo >= hi) return;

  const int NB16 = (GATE_UP ? 2 * N : N) / 16;
  const int steps = K / 32;
  const int s_lo = wave * steps / kStreamWaves;
  const int s_hi = (wave + 1) * steps / kStreamWaves;
  const int s_end = max(s_hi - 1, s_lo);          // last step to read
  const int chunks = KEEP ? 1
                          : ((steps + kStreamWaves - 1) / kStreamWaves +
                             C - 1) / C;

  struct Stretch {
    short8 b[C * NF];
    short8 a[KEEP ? 1 : C];
  };
  // rows of the block whose loads are being requested
  int block = -1;
  const u16* a_row = nullptr;
  const u16* b_e = nullptr;
  short8 kept[KEEP ? C : 1];
  auto enter = [&](int m) {
    block = m;
    const int slot = m * 16 + (lane & 15);
    const int row = MODE != 0 ? sorted_ids[slot] : slot;
    a_row = a + static_cast<int64_t>(row) * K + (lane >> 4) * 8;
    b_e = b + static_cast<int64_t>(expert_ids[m >> per]) * steps * NB16 * 512 +
          lane * 8;
  };
  auto load_rows = [&](short8* v, int s0) {
#pragma unroll
    for (int i = 0; i < C; ++i)
      v[i] = *reinterpret_cast<const short8*>(a_row +
                                              min(s0 + i, s_end) * 32);
  };
  auto request = [&](Stretch& d, int u, int c) {
    const int m = u / per_block, col = u - m * per_block;
    if (m != block) enter(m);
    const int s0 = s_lo + c * C;
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const u16* p = b_e + static_cast<int64_t>(
          min(s0 + i, s_end) * NB16 + col * COLS) * 512;
#pragma unroll
      for (int f = 0; f < NF; ++f)
        d.b[i * NF + f] = load_once(
            p + (f % COLS + (f >= COLS ? N / 16 : 0)) * 512);
    }
    if (!KEEP) load_rows(d.a, s0);
    __builtin_amdgcn_sched_barrier(0);
  };

  floatx4 acc[NF];
  auto clear = [&] {
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[f] = {0.f, 0.f, 0.f, 0.f};
  };
  auto multiply = [&](const Stretch& d, int c) {
    const int s0 = s_lo + c * C;
#pragma unroll
    for (int i = 0; i < C; ++i)
      if (s0 + i < s_hi)
#pragma unroll
        for (int f = 0; f < NF; ++f)
          acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              d.b[i * NF + f], KEEP ? kept[i] : d.a[i], acc[f], 0, 0, 0);
  };
  auto finish = [&](int u) {
    const int m = u / per_block, col = u - m * per_block;
    auto& s = sums[u & 1];
#pragma unroll
    for (int f = 0; f < NF; ++f) s[wave][f][lane] = acc[f];
    // also ends this wave's reads of the other buffer
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    clear();
    if (wave != u % kStreamWaves) return;
    floatx4 v[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      v[f] = s[0][f][lane];
#pragma unroll
      for (int i = 1; i < kStreamWaves; ++i) v[f] += s[i][f][lane];
    }
    u16* o = out + static_cast<int64_t>(m * 16 + (lane & 15)) * N +
             col * COLS * 16 + (lane >> 4) * 4;
#pragma unroll
    for (int f = 0; f < COLS; ++f) {
      bf16x4 r4;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float g = v[f][r];
        if (GATE_UP) {
          float up = v[COLS + f < NF ? COLS + f : f][r];
          if (MODE == 3) {
            g = fminf(g, limit);
            up = fminf(fmaxf(up, -limit), limit);
            g = (g / (1.f + __expf(-1.702f * g))) * (up + 1.f);
          } else {
            g = (g / (1.f + __expf(-g))) * up;
          }
        } else if (MODE == 2) {
          g = fmaxf(g, 0.f);
          g *= g;
        }
        r4.h[r] = f32_to_bf16(g);
      }
      *reinterpret_cast<bf16x4*>(o + f * 16) = r4;
    }
  };

  // stretches of all units in a row, two at a time
  int u = lo, c = 0;              // being multiplied
  int ru = lo, rc = 0;            // being requested
  int kept_block = -1;
  auto step = [&](Stretch& now, Stretch& next) {
    if (ru < hi) {
      if (++rc == chunks) {
        rc = 0;
        ++ru;
      }
      if (ru < hi) request(next, ru, rc);
    }
    if (KEEP) {
      const int m = u / per_block;
      if (m != kept_block) {
        // the request above may have gone on to the next block
        const int ahead = block;
        if (ahead != m) enter(m);
        load_rows(kept, s_lo);
        if (ahead != m) enter(ahead);
        kept_block = m;
      }
    }
    multiply(now, c);
    if (++c == chunks) {
      finish(u);
      c = 0;
      ++u;
    }
  };
  clear();
  Stretch d0, d1;
  request(d0, ru, rc);
  while (true) {
    step(d0, d1);
    if (u >= hi) break;
    step(d1, d0);
    if (u >= hi) break;
  }
}

template <int MODE>
void launch_stream(u16* out, const u16* a, const u16* b,
                   const int* sorted_ids, const int* expert_ids,
                   const int* n_valid, int blocks, int per, int K, int N,
                   float limit, hipStream_t stream) {
  constexpr bool gate = MODE == 1 || MODE == 3;
  const int span = ceil_div(K / 32, kStreamWaves);   // steps per wave
  const int units = (blocks << per) * (N / 16);      // at the most
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(std::min(units, 256)),
                       dim3(kStreamWaves * kWaveSize), 0, stream, out, a, b,
                       sorted_ids, expert_ids, n_valid, per, K, N, limit);
  };
  // sixteen loads together, fewer where K gives a wave only two or three
  // steps (K = 512, 16 experts of 1536 columns: 2 steps by 32 columns 7.0 us
  // at 64 tokens, 3 by 64 9.5)
  if (span <= 2)
    run(&moe_stream_kernel<MODE, 2, gate ? 1 : 2, true>);
  else if (span <= 3)
    run(&moe_stream_kernel<MODE, 3, gate ? 2 : 4, true>);
  else if (span <= 4)
    run(&moe_stream_kernel<MODE, 4, gate ? 2 : 4, true>);
  else if (span <= 8)
    run(&moe_stream_kernel<MODE, 8, gate ? 1 : 2, true>);
  else
    run(&moe_stream_kernel<MODE, 6, gate ? 1 : 2, false>);
}

}  // namespace

// row blocks of 16 << per rows, K a multiple of 32, N of 64
void launch_moe_stream(u16* out, const u16* a, const u16* b,
                       const int* sorted_ids, const int* expert_ids,
                       const int* n_valid, int blocks, int per, int K, int N,
                       int mode, float limit, hipStream_t stream) {
  auto* f = mode == 0 ? &launch_stream<0> : mode == 1 ? &launch_stream<1>
      : mode == 2 ? &launch_stream<2> : &launch_stream<3>;
  f(out, a, b, sorted_ids, expert_ids, n_valid, blocks, per, K, N, limit,
    stream);
}

}  // namespace fi
