// Router of the softmax-top-k experts and the block alignment of its
// choices (gfx950, wave64).
//
//  * moe_router_logits: x W^T in fp32 for the few tokens of a decode step;
//    bf16 operands, exact products, fp32 sums, as with both converted to
//    fp32 first. 16 tokens by 16 experts per workgroup, four waves split K:
//    one CU reading all of W (512 KB at 128 x 2048) in fragment order alone
//    took 35 us with its launch, 32 workgroups take 6. Many tokens are a
//    library GEMM.
//  * moe_router_topk: softmax, top-k and optional renormalisation, one wave
//    per token. A round of the choice is a register-to-register maximum and
//    two ballots (the value's and the index's maximum through twelve LDS
//    lane exchanges took 8.5 us for eight of 128 experts, now 4.6; both with
//    the launch).
//  * moe_align: token assignments sorted by expert, every expert's segment
//    padded to block_m rows, without host synchronisation and with static
//    shapes. The order within an expert is that in which its atomic
//    counter was reached, different from run to run: the grouped GEMM
//    computes each row the same wherever it sits and the combine gathers by
//    pos. Up to kAlignOne assignments one workgroup does it all in LDS;
//    more are counted and placed by up to 64 workgroups in two launches
//    (70 thousand: 61 us by one workgroup, 5 + 7 by two launches). vLLM
//    parity: moe_align_block_size (csrc/moe/moe_align_sum_kernels.cu).

#include <hip/hip_runtime.h>

#include "common.h"

namespace fi {

namespace {

typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) float floatx4;

// maximum over the wave, in every lane: four rotations within 16 lanes, then
// the swaps across them
template <int CTRL>
FI_DEV float max_rotated(float v) {
  return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(
                      0, __float_as_int(v), CTRL, 0xf, 0xf, true)));
}
FI_DEV float wave_max(float v) {
  v = max_rotated<0x121>(v);  // row_ror:1
  v = max_rotated<0x122>(v);
  v = max_rotated<0x124>(v);
  v = max_rotated<0x128>(v);
  const auto a = __builtin_amdgcn_permlane16_swap(
      __float_as_int(v), __float_as_int(v), false, false);
  v = fmaxf(__int_as_float(a[0]), __int_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(
      __float_as_int(v), __float_as_int(v), false, false);
  return fmaxf(__int_as_float(b[0]), __int_as_float(b[1]));
}

__global__ void moe_router_topk_kernel(
    const float* __restrict__ logits,  // [T, E] fp32
    float* __restrict__ topv,          // [T, k]
    int* __restrict__ topi,            // [T, k]
    const int T, const int E, const int k, const bool renorm) {
  const int t = blockIdx.x * (blockDim.x / kWaveSize)
      + threadIdx.x / kWaveSize;
  if (t >= T) return;
  const int lane = threadIdx.x % kWaveSize;
  const float* row = logits + static_cast<int64_t>(t) * E;
  // two logit slots per lane (E <= 128). With renorm, weights = softmax over
  // the top-k LOGITS (the partition cancels); without it, over all. Ties
  // pick the smaller expert index.
  const float l0 = lane < E ? row[lane] : -INFINITY;
  const float l1 = lane + 64 < E ? row[lane + 64] : -INFINITY;
  const float m = wave_max(fmaxf(l0, l1));
  float s = 0.f;
  if (!renorm) {
    s = (lane < E ? __expf(l0 - m) : 0.f) +
        (lane + 64 < E ? __expf(l1 - m) : 0.f);
#pragma unroll
    for (int off = 32; off; off >>= 1) s += __shfl_xor(s, off);
  }
  bool free0 = lane < E, free1 = lane + 64 < E;  // remaining candidates
  float ksum = 0.f, mine = 0.f;                  // mine: of choice `lane`
  int index = 0;
  for (int it = 0; it < k; ++it) {
    const float v = wave_max(fmaxf(free0 ? l0 : -INFINITY,
                                   free1 ? l1 : -INFINITY));
    unsigned long long hit = __ballot(free0 && l0 == v);
    int idx = 0;
    if (hit) {
      idx = __builtin_ctzll(hit);
    } else if ((hit = __ballot(free1 && l1 == v))) {
      idx = 64 + __builtin_ctzll(hit);
    } else {  // only NaN left: the first candidates in order
      hit = __ballot(free0);
      idx = hit ? __builtin_ctzll(hit)
                : 64 + __builtin_ctzll(__ballot(free1) | (1ull << 63));
    }
    if (idx == lane) free0 = false;
    if (idx == lane + 64) free1 = false;
    const float e = __expf(v - m);
    ksum += e;
    if (lane == (it & 63)) {
      mine = e;
      index = idx;
    }
    if ((it & 63) == 63 || it == k - 1) {
      const int at = (it & ~63) + lane;
      if (at <= it) {
        topi[static_cast<int64_t>(t) * k + at] = index;
        topv[static_cast<int64_t>(t) * k + at] = renorm ? mine : mine / s;
      }
    }
  }
  if (renorm) {
    // the first 64 weights are still in the lanes where k fits
    for (int at = lane; at < k; at += kWaveSize) {
      const float e = k <= kWaveSize ? mine
                                     : topv[static_cast<int64_t>(t) * k + at];
      topv[static_cast<int64_t>(t) * k + at] = e / ksum;
    }
  }
}

constexpr int kLogitWaves = 4;

__global__ __launch_bounds__(kLogitWaves * kWaveSize)
void moe_router_logits_kernel(const u16* __restrict__ x,
                              const u16* __restrict__ w,
                              float* __restrict__ logits, const int T,
                              const int E, const int K) {
  __shared__ floatx4 part[kLogitWaves][kWaveSize];
  const int lane = threadIdx.x % kWaveSize;
  const int wave = threadIdx.x / kWaveSize;
  const int t0 = blockIdx.x * 16, e0 = blockIdx.y * 16;
  const int steps = K / 32;
  const int lo = wave * steps / kLogitWaves;
  const int hi = (wave + 1) * steps / kLogitWaves;
  const int64_t in = (lane >> 4) * 8;
  const u16* xr = x + static_cast<int64_t>(min(t0 + (lane & 15), T - 1)) * K +
                  in;
  const u16* wr = w + static_cast<int64_t>(e0 + (lane & 15)) * K + in;
  constexpr int kAhead = 8;   // steps requested together
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = lo; s0 < hi; s0 += kAhead) {
    short8 a[kAhead], b[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int s = min(s0 + i, hi - 1);
      a[i] = *reinterpret_cast<const short8*>(wr + s * 32);
      b[i] = *reinterpret_cast<const short8*>(xr + s * 32);
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
      if (s0 + i < hi)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[i], acc, 0, 0,
                                                      0);
  }
  part[wave][lane] = acc;
  __syncthreads();
  const int t = t0 + (lane & 15);
  if (wave != 0 || t >= T) return;
  floatx4 sum = part[0][lane];
#pragma unroll
  for (int i = 1; i < kLogitWaves; ++i) sum += part[i][lane];
  *reinterpret_cast<floatx4*>(logits + static_cast<int64_t>(t) * E + e0 +
                              (lane >> 4) * 4) = sum;
}

// ---------------------------------------------------------------- alignment

constexpr int kAlignThreads = 1024, kMaxExperts = 1024;
constexpr int kAlignOne = 4096;   // assignments of the one-workgroup form
constexpr int kAlignBlocks = 64;

struct AlignLds {
  int pad0[kMaxExperts + 1];  // first slot of an expert's segment
  int tcum[kMaxExperts + 1];  // row blocks up to and with the expert
  int waves[kAlignThreads / kWaveSize];
};

// segment starts from one count per thread (thread e holds expert e's);
// returns the number of row blocks
FI_DEV int segment_starts(AlignLds& s, int count, int E, int block_m) {
  const int tid = threadIdx.x, lane = tid % kWaveSize, wave = tid / kWaveSize;
  const int tiles = tid < E ? (count + block_m - 1) / block_m : 0;
  int incl = tiles;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(incl, off, 64);
    if (lane >= off) incl += o;
  }
  if (lane == 63) s.waves[wave] = incl;
  __syncthreads();
  int before = 0, all = 0;
  for (int i = 0; i < kAlignThreads / kWaveSize; ++i) {
    if (i < wave) before += s.waves[i];
    all += s.waves[i];
  }
  if (tid < E) {
    s.pad0[tid] = (before + incl - tiles) * block_m;
    s.tcum[tid] = before + incl;
  }
  __syncthreads();
  return all;
}

// expert of row block t: the first with tcum > t (the padded tail: the last)
FI_DEV int block_expert(const AlignLds& s, int E, int t) {
  int lo = 0, hi = E - 1, ans = E - 1;
  while (lo <= hi) {
    const int mid = (lo + hi) >> 1;
    if (s.tcum[mid] > t) { ans = mid; hi = mid - 1; }
    else lo = mid + 1;
  }
  return ans;
}

__global__ __launch_bounds__(kAlignThreads) void moe_align_kernel(
    const int* __restrict__ topi,  // [n] = T*topk flattened GLOBAL ids
    int* __restrict__ sorted_ids,  // [PM]   (zeroed here; pad rows -> 0)
    int* __restrict__ expert_ids,  // [PM / block_m]
    int* __restrict__ n_valid,     // [1] real m-tile count
    int* __restrict__ pos,         // [n]  padded slot (-1 = non-local)
    const int n, const int topk, const int e_start, const int e_end,
    const int block_m, const int PM) {
  const int E = e_end - e_start;
  __shared__ AlignLds s;
  __shared__ int cnt[kMaxExperts + 1];
  const int tid = threadIdx.x;
  for (int i = tid; i <= E; i += kAlignThreads) cnt[i] = 0;
  for (int i = tid; i < PM; i += kAlignThreads) sorted_ids[i] = 0;
  __syncthreads();
  for (int i = tid; i < n; i += kAlignThreads) {
    const int e = topi[i] - e_start;
    if (e >= 0 && e < E) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  const int tiles = segment_starts(s, tid < E ? cnt[tid] : 0, E, block_m);
  if (tid == 0) n_valid[0] = tiles;
  for (int t = tid; t < PM / block_m; t += kAlignThreads)
    expert_ids[t] = block_expert(s, E, t);
  for (int i = tid; i < E; i += kAlignThreads) cnt[i] = 0;
  __syncthreads();
  for (int i = tid; i < n; i += kAlignThreads) {
    const int e = topi[i] - e_start;
    if (e < 0 || e >= E) { pos[i] = -1; continue; }
    const int p = s.pad0[e] + atomicAdd(&cnt[e], 1);
    pos[i] = p;
    sorted_ids[p] = i / topk;
  }
}

// counts of one workgroup's share, and its share of the cleared slots
__global__ __launch_bounds__(kAlignThreads) void moe_align_count_kernel(
    const int* __restrict__ topi, int* __restrict__ counts,  // [blocks, E]
    int* __restrict__ sorted_ids, const int n, const int e_start, const int E,
    const int PM) {
  __shared__ int cnt[kMaxExperts];
  const int tid = threadIdx.x;
  for (int i = tid; i < E; i += kAlignThreads) cnt[i] = 0;
  const int stride = gridDim.x * kAlignThreads;
  for (int i = blockIdx.x * kAlignThreads + tid; i < PM; i += stride)
    sorted_ids[i] = 0;
  __syncthreads();
  const int each = (n + gridDim.x - 1) / gridDim.x;
  const int lo = blockIdx.x * each, hi = min(n, lo + each);
  for (int i = lo + tid; i < hi; i += kAlignThreads) {
    const int e = topi[i] - e_start;
    if (e >= 0 && e < E) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  for (int i = tid; i < E; i += kAlignThreads)
    counts[blockIdx.x * E + i] = cnt[i];
}

__global__ __launch_bounds__(kAlignThreads) void moe_align_place_kernel(
    const int* __restrict__ topi, const int* __restrict__ counts,
    int* __restrict__ sorted_ids, int* __restrict__ expert_ids,
    int* __restrict__ n_valid, int* __restrict__ pos, const int n,
    const int topk, const int e_start, const int E, const int block_m,
    const int PM) {
  __shared__ AlignLds s;
  __shared__ int next[kMaxExperts];
  const int tid = threadIdx.x;
  int all = 0, before = 0;
  if (tid < E) {
#pragma unroll 8
    for (int b = 0; b < static_cast<int>(gridDim.x); ++b) {
      const int c = counts[b * E + tid];
      if (b < static_cast<int>(blockIdx.x)) before += c;
      all += c;
    }
  }
  const int tiles = segment_starts(s, all, E, block_m);
  if (tid < E) next[tid] = s.pad0[tid] + before;
  if (tid == 0 && blockIdx.x == 0) n_valid[0] = tiles;
  const int stride = gridDim.x * kAlignThreads;
  for (int t = blockIdx.x * kAlignThreads + tid; t < PM / block_m; t += stride)
    expert_ids[t] = block_expert(s, E, t);
  __syncthreads();
  const int each = (n + gridDim.x - 1) / gridDim.x;
  const int lo = blockIdx.x * each, hi = min(n, lo + each);
  for (int i = lo + tid; i < hi; i += kAlignThreads) {
    const int e = topi[i] - e_start;
    if (e < 0 || e >= E) { pos[i] = -1; continue; }
    const int p = atomicAdd(&next[e], 1);
    pos[i] = p;
    sorted_ids[p] = i / topk;
  }
}

}  // namespace

void launch_moe_router_topk(const float* logits, float* topv, int* topi,
                            int T, int E, int k, bool renorm,
                            hipStream_t stream) {
  const int waves = 4;  // 4 tokens per 256-thread block
  hipLaunchKernelGGL(moe_router_topk_kernel,
                     dim3(ceil_div(T, waves)), dim3(waves * kWaveSize), 0,
                     stream, logits, topv, topi, T, E, k, renorm);
}

// E a multiple of 16, K of 32
void launch_moe_router_logits(const u16* x, const u16* w, float* logits,
                              int T, int E, int K, hipStream_t stream) {
  hipLaunchKernelGGL(moe_router_logits_kernel,
                     dim3(ceil_div(T, 16), E / 16),
                     dim3(kLogitWaves * kWaveSize), 0, stream, x, w, logits,
                     T, E, K);
}

// ints of scratch that an alignment of n assignments needs
int64_t moe_align_scratch(int n, int experts) {
  return n > kAlignOne ? static_cast<int64_t>(kAlignBlocks) * experts : 0;
}

void launch_moe_align(const int* topi, int* sorted_ids, int* expert_ids,
                      int* n_valid, int* pos, int* scratch, int n, int topk,
                      int e_start, int e_end, int block_m, int PM,
                      hipStream_t stream) {
  if (n <= kAlignOne) {
    hipLaunchKernelGGL(moe_align_kernel, dim3(1), dim3(kAlignThreads), 0,
                       stream, topi, sorted_ids, expert_ids, n_valid, pos, n,
                       topk, e_start, e_end, block_m, PM);
    return;
  }
  const int E = e_end - e_start;
  const int blocks = std::min(kAlignBlocks, ceil_div(n, kAlignThreads));
  hipLaunchKernelGGL(moe_align_count_kernel, dim3(blocks),
                     dim3(kAlignThreads), 0, stream, topi, scratch,
                     sorted_ids, n, e_start, E, PM);
  hipLaunchKernelGGL(moe_align_place_kernel, dim3(blocks),
                     dim3(kAlignThreads), 0, stream, topi, scratch,
                     sorted_ids, expert_ids, n_valid, pos, n, topk, e_start,
                     E, block_m, PM);
}

}  // namespace fi
