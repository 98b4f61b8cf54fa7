// Grouped MFMA GEMM for MoE expert compute (gfx950).
//
// Replaces capacity-padded torch.bmm experts (and their
// per-layer `counts.max()` host sync) with a vLLM-style block-aligned
// grouped GEMM: token assignments are sorted by expert and each expert's
// segment is padded to a multiple of BLOCK_M on the DEVICE, so every
// m-tile belongs to exactly one expert and all launch shapes are static
// — the whole MoE decode step becomes hipGraph-capturable.
// (Capability parity: expert serving the reference invokes via vLLM
// images; it publishes no kernels of its own.)
//
// Expert weights are packed offline into MFMA B-fragment order
// [E][K/32][N/16][64][8], so a wave reads a fragment as one run of memory.
// Blocks beyond the real (data-dependent) count read a device scalar and
// exit: the grid is static, the work is dynamic. The bf16 kernels are
// elsewhere, by rows per block; here are their dispatch and the fp8 kernel.
//
// C-fragment map (16x16): row = (lane>>4)*4 + r, col = lane&15.
// A-fragment: lane holds A[row = lane&15][k = (lane>>4)*8 + e], e<8.
// B-fragment: lane holds B[k = (lane>>4)*8 + e][col = lane&15].

#include <hip/hip_runtime.h>

#include <cmath>

#include "common.h"

namespace fi {

void launch_moe_tile(u16*, const u16*, const u16*, const int*, const int*,
                     const int*, int, int, int, int, int, float, hipStream_t);
void launch_moe_wide(u16*, const u16*, const u16*, const int*, const int*,
                     const int*, int, int, int, int, int, int, float,
                     hipStream_t);
void launch_moe_stream(u16*, const u16*, const u16*, const int*, const int*,
                       const int*, int, int, int, int, int, float,
                       hipStream_t);

namespace {

typedef __attribute__((ext_vector_type(4))) float floatx4;

// fp8 grouped GEMM: A (e4m3, per-row scales from the fused-norm / row
// quant) x B (e4m3, per-expert per-out-channel scales) on
// mfma_f32_16x16x32_fp8_fp8 — HALF the weight bytes of bf16 in the
// weight-bandwidth-bound decode regime, and no per-expert host loops:
// the fp8 MoE path becomes hipGraph-capturable (the first version ran per-expert
// torch._scaled_mm with .nonzero() syncs). Dequant happens in the
// epilogue: v = acc * a_scale[row] * b_scale[col].
//
// WM x WN waves (4 total), MITER 16-row fragments per wave, NITER 16-col
// fragments per wave. Block tile: rows BM = 16*WM*MITER, cols BN =
// 16*WN*NITER of the OUTPUT space. GATE_UP: B is packed over 2N columns
// (gate at n, up at n + N); the epilogue writes silu(gate)*up.
typedef long long i64;

template <int WM, int WN, int MITER, int NITER, bool GATE_UP,
          bool STAGE_A = false>
__global__ __launch_bounds__(256) void moe_gemm_fp8_kernel(
    u16* __restrict__ out,               // [PM, N] bf16
    const unsigned char* __restrict__ a, // e4m3 [T, K] or act8 [PM, K]
    const float* __restrict__ a_scales,  // [T] / [PM] per-row
    const unsigned char* __restrict__ b, // [E][K/32][NB/16][64][8] e4m3
    const float* __restrict__ b_scales,  // [E][NB] per out channel
    const int* __restrict__ sorted_ids,
    const int* __restrict__ expert_ids,
    const int* __restrict__ n_valid,
    const int K, const int N) {
  constexpr int BM = 16 * WM * MITER;
  static_assert(!STAGE_A || BM == 128, "STAGE_A is tuned for BM=128");
  const int mtile = blockIdx.x;
  if (mtile >= *n_valid) return;

  const int lane = threadIdx.x % kWaveSize;
  const int wave = threadIdx.x / kWaveSize;
  const int wm = wave / WN;
  const int wn = wave % WN;
  const int nt0 = (blockIdx.y * WN + wn) * NITER;
  const int e = expert_ids[mtile];
  const int row0 = mtile * BM + wm * (16 * MITER);

  const int NB16 = (GATE_UP ? 2 * N : N) / 16;
  const unsigned char* b_e =
      b + static_cast<int64_t>(e) * (K / 32) * NB16 * (64 * 8);
  const float* bs_e = b_scales + static_cast<int64_t>(e) * NB16 * 16;
  const unsigned char* bg_p[NITER];
  const unsigned char* bu_p[NITER];
#pragma unroll
  for (int ni = 0; ni < NITER; ++ni) {
    bg_p[ni] = b_e + (static_cast<int64_t>(nt0 + ni) * 64 + lane) * 8;
    bu_p[ni] = GATE_UP
        ? b_e + ((static_cast<int64_t>(nt0 + ni) + N / 16) * 64 + lane) * 8
        : nullptr;
  }
  const int64_t b_step = static_cast<int64_t>(NB16) * 64 * 8;

  const unsigned char* a_p[MITER];
  int a_row[MITER];
#pragma unroll
  for (int mi = 0; mi < MITER; ++mi) {
    const int slot = row0 + mi * 16 + (lane & 15);
    a_row[mi] = GATE_UP ? sorted_ids[slot] : slot;
    a_p[mi] = a + static_cast<int64_t>(a_row[mi]) * K + (lane >> 4) * 8;
  }

  // STAGE_A (BM=128): [128 rows][32 B] e4m3 tile through LDS via glds
  // (2-phase; swizzle byte^=(row&1)<<4 on the SOURCE — rule 21)
  constexpr int kARowB = 32;                    // 32 e4m3 per row
  constexpr int kATileB = 128 * kARowB;         // 4 KiB
  __shared__ unsigned char a8_lds[STAGE_A ? 2 * kATileB : 1];
  const int tid = threadIdx.x;
  int64_t stage_row_off = 0;
  int stage_src_off = 0, stage_dst = 0;
  if (STAGE_A) {
    const int X = tid * 16;                     // one 16-B piece per thread
    const int srow = X / kARowB;
    const int sbyte = (X % kARowB) ^ ((srow & 1) << 4);
    const int gr = GATE_UP ? sorted_ids[mtile * BM + srow]
                           : mtile * BM + srow;
    stage_row_off = static_cast<int64_t>(gr) * K;
    stage_src_off = sbyte;
    stage_dst = X;
  }
  auto stage_a = [&](int kt, int buf) {
    if (!STAGE_A) return;
    const unsigned char* src = a + stage_row_off + kt * 32 + stage_src_off;
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) void*)src,
        (__attribute__((address_space(3))) void*)(
            a8_lds + buf * kATileB + stage_dst),
        16, 0, 0);
  };
  int a_lds_off[MITER];
  if (STAGE_A) {
#pragma unroll
    for (int mi = 0; mi < MITER; ++mi) {
      const int srow = wm * (16 * MITER) + mi * 16 + (lane & 15);
      const int byte = ((lane >> 4) * 8) ^ ((srow & 1) << 4);
      a_lds_off[mi] = srow * kARowB + byte;
    }
    stage_a(0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }

  floatx4 acc_g[MITER][NITER];
  floatx4 acc_u[GATE_UP ? MITER : 1][NITER];
#pragma unroll
  for (int mi = 0; mi < MITER; ++mi)
#pragma unroll
    for (int ni = 0; ni < NITER; ++ni) {
      acc_g[mi][ni] = {0.f, 0.f, 0.f, 0.f};
      if (GATE_UP) acc_u[mi][ni] = {0.f, 0.f, 0.f, 0.f};
    }

  const int ksteps = K / 32;
  if (STAGE_A) {
    for (int kt = 0; kt < ksteps; ++kt) {
      if (kt + 1 < ksteps) stage_a(kt + 1, (kt + 1) & 1);
      const unsigned char* abuf = a8_lds + (kt & 1) * kATileB;
      i64 av[MITER];
#pragma unroll
      for (int mi = 0; mi < MITER; ++mi)
        av[mi] = *reinterpret_cast<const i64*>(abuf + a_lds_off[mi]);
#pragma unroll
      for (int ni = 0; ni < NITER; ++ni) {
        const i64 bg = *reinterpret_cast<const i64*>(bg_p[ni] + kt * b_step);
        i64 bu = 0;
        if (GATE_UP)
          bu = *reinterpret_cast<const i64*>(bu_p[ni] + kt * b_step);
#pragma unroll
        for (int mi = 0; mi < MITER; ++mi) {
          acc_g[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
              av[mi], bg, acc_g[mi][ni], 0, 0, 0);
          if (GATE_UP)
            acc_u[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
                av[mi], bu, acc_u[mi][ni], 0, 0, 0);
        }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
  } else {
    // register double-buffered pipeline (see the bf16 kernel: the
    // BM=16 decode variants are latency-bound without it; unroll-by-2
    // keeps buffer indices compile-time — rule 20)
    constexpr int NU = GATE_UP ? NITER : 1;
    i64 av0[MITER], av1[MITER], bg0[NITER], bg1[NITER], bu0[NU], bu1[NU];
    auto issue = [&](i64 (&avd)[MITER], i64 (&bgd)[NITER],
                     i64 (&bud)[NU], int kt) {
#pragma unroll
      for (int mi = 0; mi < MITER; ++mi)
        avd[mi] = *reinterpret_cast<const i64*>(a_p[mi] + kt * 32);
#pragma unroll
      for (int ni = 0; ni < NITER; ++ni) {
        bgd[ni] = *reinterpret_cast<const i64*>(bg_p[ni] + kt * b_step);
        if (GATE_UP)
          bud[ni] = *reinterpret_cast<const i64*>(bu_p[ni] + kt * b_step);
      }
    };
    auto consume = [&](i64 (&avv)[MITER], i64 (&bgv)[NITER],
                       i64 (&buv)[NU]) {
#pragma unroll
      for (int ni = 0; ni < NITER; ++ni)
#pragma unroll
        for (int mi = 0; mi < MITER; ++mi) {
          acc_g[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
              avv[mi], bgv[ni], acc_g[mi][ni], 0, 0, 0);
          if (GATE_UP)
            acc_u[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
                avv[mi], buv[ni % NU], acc_u[mi][ni], 0, 0, 0);
        }
    };
    issue(av0, bg0, bu0, 0);
    for (int kt = 0; kt < ksteps; kt += 2) {
      if (kt + 1 < ksteps) issue(av1, bg1, bu1, kt + 1);
      consume(av0, bg0, bu0);
      if (kt + 1 < ksteps) {
        if (kt + 2 < ksteps) issue(av0, bg0, bu0, kt + 2);
        consume(av1, bg1, bu1);
      }
    }
  }

#pragma unroll
  for (int ni = 0; ni < NITER; ++ni) {
    const int col = (nt0 + ni) * 16 + (lane & 15);
    const float bs_g = bs_e[col];
    const float bs_u = GATE_UP ? bs_e[N + col] : 0.f;
#pragma unroll
    for (int mi = 0; mi < MITER; ++mi) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int oslot = row0 + mi * 16 + (lane >> 4) * 4 + r;
        const int arow = GATE_UP ? sorted_ids[oslot] : oslot;
        const float as = a_scales[arow];
        float v;
        if (GATE_UP) {
          const float g = acc_g[mi][ni][r] * as * bs_g;
          const float u = acc_u[mi][ni][r] * as * bs_u;
          v = (g / (1.f + __expf(-g))) * u;
        } else {
          v = acc_g[mi][ni][r] * as * bs_g;
        }
        out[static_cast<int64_t>(oslot) * N + col] = f32_to_bf16(v);
      }
    }
  }
}

}  // namespace

// Whether blocks of 128 rows go by tiles of 512 columns, one per CU (256 of two
// blocks), or by those of 256, two per CU. A round of the wide ones takes 0.82
// (gathered rows: 0.88) of the time that the others need for as many products,
// but a round that is begun takes all of it; the others lose a quarter of a
// round. How many blocks there are only the GPU knows: every expert is taken to
// leave half a block empty. Where most experts have one block, gate and up are
// bound by the weights and the wide tiles, with fewer loads in flight, lose 6 %;
// where most have two, whose weights a CU then loads once for both, they gain 15
// (128 experts, 2048 x 768, top 8, us, narrow and wide: 1024 rows 161 and 171,
// 2048 203 and 216, 2500 230 and 196, 3000 215 and 193; 64 experts, 2048 x 1408,
// top 6: 1024 rows 153 and 169, 1500 216 and 203). Over 54 products of three
// shapes of experts (600 to 8100 rows) this choice takes 0.9 % longer than the
// better of the two, the narrow tiles alone 11.
bool wide_tiles(int max_mtiles, int experts, int K, int N, int mode) {
  if (K % 64 != 0 || K < 128) return false;
  const int cols = mode == 1 || mode == 3 ? 256 : 512;
  if (mode != 0 && 10 * max_mtiles < 21 * experts) return false;
  const double blocks = max_mtiles - 0.5 * experts;
  const double rounds = std::ceil(blocks * ceil_div(N, cols) / 256);
  return (mode == 0 ? 0.82 : 0.88) * rounds < blocks * N / cols / 256 + 0.25;
}

// block_m 16: few rows per expert, bound by the weights; 128: many.
void launch_moe_gemm(u16* out, const u16* a, const u16* b,
                     const int* sorted_ids, const int* expert_ids,
                     const int* n_valid, int max_mtiles, int experts, int rows,
                     int K, int N, int block_m, int mode, float limit,
                     hipStream_t stream) {
  // The tiles read gathered rows and one expert's weights at 32-bit byte
  // offsets; operands beyond those go through the streaming kernel, which
  // takes a block of 128 rows as eight of 16.
  const int64_t limit32 = int64_t(1) << 31;      // bf16 values in 4 GB
  const int NB = mode == 1 || mode == 3 ? 2 * N : N;
  if (block_m == 16 || static_cast<int64_t>(K) * NB >= limit32 ||
      (mode != 0 && static_cast<int64_t>(rows) * K >= limit32))
    launch_moe_stream(out, a, b, sorted_ids, expert_ids, n_valid, max_mtiles,
                      block_m == 16 ? 0 : 3, K, N, mode, limit, stream);
  else if (wide_tiles(max_mtiles, experts, K, N, mode) &&
           reinterpret_cast<uintptr_t>(b) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(out) % 16 == 0)
    launch_moe_wide(out, a, b, sorted_ids, expert_ids, n_valid, max_mtiles,
                    experts, rows, K, N, mode, limit, stream);
  else
    launch_moe_tile(out, a, b, sorted_ids, expert_ids, n_valid, max_mtiles,
                    rows, K, N, mode, limit, stream);
}

void launch_moe_gemm_fp8(u16* out, const unsigned char* a,
                         const float* a_scales, const unsigned char* b,
                         const float* b_scales, const int* sorted_ids,
                         const int* expert_ids, const int* n_valid,
                         int max_mtiles, int K, int N, int block_m,
                         bool gate_up, hipStream_t stream) {
  if (block_m == 16) {
    const dim3 grid(max_mtiles, N / 64);
    if (gate_up)
      hipLaunchKernelGGL((moe_gemm_fp8_kernel<1, 4, 1, 1, true>), grid,
                         dim3(256), 0, stream, out, a, a_scales, b, b_scales,
                         sorted_ids, expert_ids, n_valid, K, N);
    else
      hipLaunchKernelGGL((moe_gemm_fp8_kernel<1, 4, 1, 1, false>), grid,
                         dim3(256), 0, stream, out, a, a_scales, b, b_scales,
                         sorted_ids, expert_ids, n_valid, K, N);
  } else {
    static const bool stage_a8 = [] {
      const char* e = getenv("FI_MOE_STAGE_A");
      return !(e && e[0] == '0');
    }();
    if (gate_up) {
      const dim3 grid(max_mtiles, N / 64);
      if (stage_a8)
        hipLaunchKernelGGL((moe_gemm_fp8_kernel<2, 2, 4, 2, true, true>),
                           grid, dim3(256), 0, stream, out, a, a_scales, b,
                           b_scales, sorted_ids, expert_ids, n_valid, K, N);
      else
        hipLaunchKernelGGL((moe_gemm_fp8_kernel<2, 2, 4, 2, true, false>),
                           grid, dim3(256), 0, stream, out, a, a_scales, b,
                           b_scales, sorted_ids, expert_ids, n_valid, K, N);
    } else {
      const dim3 grid(max_mtiles, N / 128);
      if (stage_a8)
        hipLaunchKernelGGL((moe_gemm_fp8_kernel<2, 2, 4, 4, false, true>),
                           grid, dim3(256), 0, stream, out, a, a_scales, b,
                           b_scales, sorted_ids, expert_ids, n_valid, K, N);
      else
        hipLaunchKernelGGL((moe_gemm_fp8_kernel<2, 2, 4, 4, false, false>),
                           grid, dim3(256), 0, stream, out, a, a_scales, b,
                           b_scales, sorted_ids, expert_ids, n_valid, K, N);
    }
  }
}

}  // namespace fi
