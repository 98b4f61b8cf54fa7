// PyTorch bindings for the FusionInfer-AMD CDNA4 kernel library.

#include <torch/extension.h>

#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include "common.h"

namespace fi {

template <bool FUSED_ADD, bool FP8_OUT>
void launch_rms_norm(void*, float*, const u16*, u16*, const u16*, float, int,
                     int, hipStream_t);
void launch_silu_and_mul(u16*, const u16*, int64_t, int, hipStream_t);
template <bool SILU_MUL>
void launch_row_quant_fp8(unsigned char*, float*, const u16*, int, int,
                          hipStream_t);
void launch_rope_qk_norm(u16*, u16*, const u16*, int64_t, int64_t, int64_t,
                         const u16*, const u16*, const float*, const int*, int,
                         int, int, int, float, void*, void*, const int*, int,
                         bool, float, float, hipStream_t);
void launch_reshape_and_cache(const u16*, const u16*, void*, void*,
                              const int*, int64_t, int64_t, int, int, int,
                              int, bool, float, float, hipStream_t);
template <bool GATHER>
void launch_kv_block_copy(u16*, u16*, u16*, const int*, int, int64_t,
                          hipStream_t);
bool decode_attn_supported(int, int);
int64_t decode_piece_floats(int, int, int, int);
void launch_paged_attn_decode(u16*, const u16*, const void*, const void*,
                              const int*, const int*, int, int64_t, int, int,
                              int, int, float, bool, float*, hipStream_t);
PrefillPlan plan_prefill_attn(int, int, int, int, int, int, bool);
int64_t prefill_piece_floats(const PrefillPlan&, int);
void launch_prefill_attn(u16*, const u16*, const void*, const void*,
                         const int*, const int*, const int*, const int*,
                         const int*, int, int64_t, int64_t, int64_t, int, int,
                         int, float, bool, const PrefillPlan&, float*,
                         hipStream_t);
void launch_skinny_gemm(u16*, const u16*, const u16*, const u16*,
                        const SkinnyExtra&, int, int, int, int64_t, int64_t,
                        bool, hipStream_t);
void launch_stream_norm(u16*, const float*, const u16*, float, int, int,
                        hipStream_t);
template <class X>
void launch_stream_begin(float*, u16*, float*, const X*, const u16*, int, int,
                         hipStream_t);
int64_t part_gemm_floats(int, int, int, bool);
double part_gemm_us(int, int, int, bool);
bool launch_part_gemm_norm(void*, float*, u16*, const u16*, float, float*,
                           const u16*, const float*, const u16*, const float*,
                           int, int, int, int64_t, hipStream_t);
bool launch_part_gemm_rope(u16*, const RopeArgs&, const u16*, float*,
                           const u16*, const u16*, int, int, int, int64_t,
                           hipStream_t);
void launch_part_gemm(u16*, float*, const u16*, const u16*, const u16*, int,
                      int, int, int64_t, int64_t, bool, hipStream_t);
void launch_part_gemm_fp8(u16*, float*, const unsigned char*, const float*,
                          const unsigned char*, const float*, int, int, int,
                          int64_t, int64_t, hipStream_t);
int64_t tile_gemm_floats(int, int, int);
double tile_gemm_us(int, int, int);
void launch_tile_gemm(u16*, float*, const u16*, const u16*, const u16*, int,
                      int, int, int64_t, int64_t, bool, bool, hipStream_t);
void launch_tile_gemm_fp8(u16*, float*, const unsigned char*, const float*,
                          const unsigned char*, const float*, int, int, int,
                          int64_t, int64_t, hipStream_t);

}  // namespace fi

namespace {

using fi::u16;

#define CHECK_BF16_CUDA(t)                                     \
  TORCH_CHECK((t).is_cuda(), #t " must be on GPU");            \
  TORCH_CHECK((t).scalar_type() == at::kBFloat16, #t " must be bf16")

u16* bf16_ptr(at::Tensor& t) { return reinterpret_cast<u16*>(t.data_ptr()); }
const u16* bf16_cptr(const at::Tensor& t) {
  return reinterpret_cast<const u16*>(t.data_ptr());
}

hipStream_t current_stream() {
  return c10::hip::getCurrentHIPStream().stream();
}

// KV caches are bf16 or fp8 (OCP e4m3, scale 1.0)
bool cache_is_fp8(const at::Tensor& t) {
  TORCH_CHECK(
      t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat8_e4m3fn,
      "kv cache must be bf16 or float8_e4m3fn");
  return t.scalar_type() == at::kFloat8_e4m3fn;
}

void rms_norm(at::Tensor out, at::Tensor input, at::Tensor weight, double eps) {
  CHECK_BF16_CUDA(out);
  CHECK_BF16_CUDA(input);
  TORCH_CHECK(input.is_contiguous() && out.is_contiguous());
  const int hidden = input.size(-1);
  const int tokens = input.numel() / hidden;
  fi::launch_rms_norm<false, false>(bf16_ptr(out), nullptr, bf16_cptr(input),
                                    nullptr, bf16_cptr(weight),
                                    static_cast<float>(eps), tokens, hidden,
                                    current_stream());
}

// of fp32 rows
void stream_norm(at::Tensor out, at::Tensor input, at::Tensor weight,
                 double eps) {
  CHECK_BF16_CUDA(out);
  CHECK_BF16_CUDA(weight);
  TORCH_CHECK(input.is_cuda() && input.scalar_type() == at::kFloat &&
              input.is_contiguous() && out.is_contiguous() &&
              weight.is_contiguous() && input.dim() == 2 &&
              out.sizes() == input.sizes());
  const int hidden = input.size(1);
  TORCH_CHECK(hidden > 0 && hidden % 8 == 0 && hidden <= 16384 &&
                  weight.numel() == hidden,
              "stream_norm: unsupported sizes");
  // (weight on any grid, as in the other norms)
  TORCH_CHECK(reinterpret_cast<uintptr_t>(out.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(input.data_ptr()) % 16 == 0);
  if (input.numel() == 0) return;
  fi::launch_stream_norm(bf16_ptr(out), input.data_ptr<float>(),
                         bf16_cptr(weight), static_cast<float>(eps),
                         input.size(0), hidden, current_stream());
}

void fused_add_rms_norm(at::Tensor input, at::Tensor residual,
                        at::Tensor weight, double eps) {
  CHECK_BF16_CUDA(input);
  CHECK_BF16_CUDA(residual);
  TORCH_CHECK(input.is_contiguous() && residual.is_contiguous());
  const int hidden = input.size(-1);
  const int tokens = input.numel() / hidden;
  // in-place: residual += input; input = rmsnorm(residual)
  fi::launch_rms_norm<true, false>(bf16_ptr(input), nullptr, bf16_cptr(input),
                                   bf16_ptr(residual), bf16_cptr(weight),
                                   static_cast<float>(eps), tokens, hidden,
                                   current_stream());
}

#define CHECK_FP8_OUT(o, s)                                                  \
  TORCH_CHECK((o).scalar_type() == at::kFloat8_e4m3fn && (o).is_cuda() &&    \
              (o).is_contiguous());                                          \
  TORCH_CHECK((s).scalar_type() == at::kFloat && (s).is_cuda())

void rms_norm_fp8(at::Tensor out, at::Tensor out_scales, at::Tensor input,
                  at::Tensor weight, double eps) {
  CHECK_BF16_CUDA(input);
  CHECK_FP8_OUT(out, out_scales);
  TORCH_CHECK(input.is_contiguous());
  const int hidden = input.size(-1);
  const int tokens = input.numel() / hidden;
  fi::launch_rms_norm<false, true>(
      out.data_ptr(), out_scales.data_ptr<float>(), bf16_cptr(input), nullptr,
      bf16_cptr(weight), static_cast<float>(eps), tokens, hidden,
      current_stream());
}

void fused_add_rms_norm_fp8(at::Tensor out, at::Tensor out_scales,
                            at::Tensor input, at::Tensor residual,
                            at::Tensor weight, double eps) {
  CHECK_BF16_CUDA(input);
  CHECK_BF16_CUDA(residual);
  CHECK_FP8_OUT(out, out_scales);
  TORCH_CHECK(input.is_contiguous() && residual.is_contiguous());
  const int hidden = input.size(-1);
  const int tokens = input.numel() / hidden;
  // residual += input (in place); out = fp8(rmsnorm(residual))
  fi::launch_rms_norm<true, true>(
      out.data_ptr(), out_scales.data_ptr<float>(), bf16_cptr(input),
      bf16_ptr(residual), bf16_cptr(weight), static_cast<float>(eps), tokens,
      hidden, current_stream());
}

void silu_and_mul_fp8(at::Tensor out, at::Tensor out_scales, at::Tensor input) {
  CHECK_BF16_CUDA(input);
  CHECK_FP8_OUT(out, out_scales);
  TORCH_CHECK(input.is_contiguous());
  const int inter = out.size(-1);
  TORCH_CHECK(input.size(-1) == 2 * inter);
  TORCH_CHECK(inter % 8 == 0);
  fi::launch_row_quant_fp8<true>(
      static_cast<unsigned char*>(out.data_ptr()),
      out_scales.data_ptr<float>(), bf16_cptr(input),
      input.numel() / (2 * inter), inter, current_stream());
}

void quant_fp8_rows(at::Tensor out, at::Tensor out_scales, at::Tensor input) {
  CHECK_BF16_CUDA(input);
  CHECK_FP8_OUT(out, out_scales);
  TORCH_CHECK(input.is_contiguous());
  const int cols = input.size(-1);
  TORCH_CHECK(cols % 8 == 0);
  fi::launch_row_quant_fp8<false>(
      static_cast<unsigned char*>(out.data_ptr()),
      out_scales.data_ptr<float>(), bf16_cptr(input), input.numel() / cols,
      cols, current_stream());
}

void silu_and_mul(at::Tensor out, at::Tensor input) {
  CHECK_BF16_CUDA(out);
  CHECK_BF16_CUDA(input);
  TORCH_CHECK(input.is_contiguous() && out.is_contiguous());
  const int inter = out.size(-1);
  TORCH_CHECK(input.size(-1) == 2 * inter);
  TORCH_CHECK(inter % 8 == 0);
  fi::launch_silu_and_mul(bf16_ptr(out), bf16_cptr(input),
                          input.numel() / (2 * inter), inter,
                          current_stream());
}

void rope_qk_norm(at::Tensor q, at::Tensor k,
                  c10::optional<at::Tensor> q_weight,
                  c10::optional<at::Tensor> k_weight, at::Tensor cos_sin,
                  at::Tensor positions, int64_t num_q_heads,
                  int64_t num_kv_heads, int64_t head_dim, double eps) {
  CHECK_BF16_CUDA(q);
  CHECK_BF16_CUDA(k);
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat && cos_sin.is_cuda());
  TORCH_CHECK(positions.scalar_type() == at::kInt && positions.is_cuda());
  // q/k may be row-strided slices of the fused qkv projection output
  TORCH_CHECK(q.dim() == 2 && k.dim() == 2);
  TORCH_CHECK(q.stride(1) == 1 && k.stride(1) == 1);
  TORCH_CHECK(head_dim == 64 || head_dim == 128,
              "rope: heads of 64 or 128 values");
  const int tokens = q.size(0);
  fi::launch_rope_qk_norm(
      bf16_ptr(q), bf16_ptr(k), nullptr, q.stride(0), k.stride(0), 0,
      q_weight ? bf16_cptr(*q_weight) : nullptr,
      k_weight ? bf16_cptr(*k_weight) : nullptr, cos_sin.data_ptr<float>(),
      positions.data_ptr<int>(), tokens, num_q_heads, num_kv_heads, head_dim,
      static_cast<float>(eps), nullptr, nullptr, nullptr, 1, false, 1.f, 1.f,
      current_stream());
}

// rope_qk_norm of q in place; k's result and v go to the paged cache alone
void rope_qk_norm_cache(at::Tensor q, at::Tensor k, at::Tensor v,
                        c10::optional<at::Tensor> q_weight,
                        c10::optional<at::Tensor> k_weight,
                        at::Tensor cos_sin, at::Tensor positions,
                        at::Tensor k_cache, at::Tensor v_cache,
                        at::Tensor slot_mapping, int64_t num_q_heads,
                        double eps, double k_inv_scale, double v_inv_scale) {
  CHECK_BF16_CUDA(q);
  CHECK_BF16_CUDA(k);
  CHECK_BF16_CUDA(v);
  const bool fp8 = cache_is_fp8(k_cache);
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat && cos_sin.is_cuda());
  TORCH_CHECK(positions.scalar_type() == at::kInt && positions.is_cuda());
  TORCH_CHECK(slot_mapping.scalar_type() == at::kInt &&
              slot_mapping.is_cuda());
  TORCH_CHECK(q.dim() == 2 && k.dim() == 2 && v.dim() == 2);
  TORCH_CHECK(q.stride(1) == 1 && k.stride(1) == 1 && v.stride(1) == 1);
  const int tokens = q.size(0);
  const int kv_heads = k_cache.size(1), head_dim = k_cache.size(3);
  TORCH_CHECK(head_dim == 64 || head_dim == 128,
              "rope: heads of 64 or 128 values");
  TORCH_CHECK(q.size(1) == num_q_heads * head_dim &&
              k.size(1) == kv_heads * head_dim && v.size(1) == k.size(1) &&
              k.size(0) == tokens && v.size(0) == tokens &&
              positions.numel() >= tokens && slot_mapping.numel() >= tokens &&
              cos_sin.size(-1) == head_dim);
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous() &&
              v_cache.sizes() == k_cache.sizes() &&
              v_cache.scalar_type() == k_cache.scalar_type());
  fi::launch_rope_qk_norm(
      bf16_ptr(q), bf16_ptr(k), bf16_cptr(v), q.stride(0), k.stride(0),
      v.stride(0), q_weight ? bf16_cptr(*q_weight) : nullptr,
      k_weight ? bf16_cptr(*k_weight) : nullptr, cos_sin.data_ptr<float>(),
      positions.data_ptr<int>(), tokens, num_q_heads, kv_heads, head_dim,
      static_cast<float>(eps), k_cache.data_ptr(), v_cache.data_ptr(),
      slot_mapping.data_ptr<int>(), k_cache.size(2), fp8,
      static_cast<float>(k_inv_scale), static_cast<float>(v_inv_scale),
      current_stream());
}

void reshape_and_cache(at::Tensor k, at::Tensor v, at::Tensor k_cache,
                       at::Tensor v_cache, at::Tensor slot_mapping,
                       double k_inv_scale, double v_inv_scale) {
  CHECK_BF16_CUDA(k);
  CHECK_BF16_CUDA(v);
  const bool fp8 = cache_is_fp8(k_cache);
  TORCH_CHECK(slot_mapping.scalar_type() == at::kInt);
  TORCH_CHECK(k.dim() == 2 && v.dim() == 2);  // [T, Hk*D] (maybe strided rows)
  TORCH_CHECK(k.stride(1) == 1 && v.stride(1) == 1);
  const int kv_heads = k_cache.size(1);
  const int block_size = k_cache.size(2);
  const int head_dim = k_cache.size(3);
  fi::launch_reshape_and_cache(
      bf16_cptr(k), bf16_cptr(v), k_cache.data_ptr(), v_cache.data_ptr(),
      slot_mapping.data_ptr<int>(), k.stride(0), v.stride(0), k.size(0),
      kv_heads, block_size, head_dim, fp8,
      static_cast<float>(k_inv_scale), static_cast<float>(v_inv_scale),
      current_stream());
}

void gather_kv_blocks(at::Tensor staging, at::Tensor k_cache,
                      at::Tensor v_cache, at::Tensor block_ids) {
  TORCH_CHECK(staging.is_cuda() &&
              staging.scalar_type() == k_cache.scalar_type());
  TORCH_CHECK(block_ids.scalar_type() == at::kInt);
  const int n = block_ids.size(0);
  // raw byte mover in u16 units (fp8 blocks are half the bytes)
  const int64_t block_elems = k_cache.size(1) * k_cache.size(2) *
      k_cache.size(3) * k_cache.element_size() / 2;
  fi::launch_kv_block_copy<true>(
      static_cast<fi::u16*>(staging.data_ptr()),
      static_cast<fi::u16*>(k_cache.data_ptr()),
      static_cast<fi::u16*>(v_cache.data_ptr()), block_ids.data_ptr<int>(), n,
      block_elems, current_stream());
}

void scatter_kv_blocks(at::Tensor staging, at::Tensor k_cache,
                       at::Tensor v_cache, at::Tensor block_ids) {
  TORCH_CHECK(staging.is_cuda() &&
              staging.scalar_type() == k_cache.scalar_type());
  TORCH_CHECK(block_ids.scalar_type() == at::kInt);
  const int n = block_ids.size(0);
  const int64_t block_elems = k_cache.size(1) * k_cache.size(2) *
      k_cache.size(3) * k_cache.element_size() / 2;
  fi::launch_kv_block_copy<false>(
      static_cast<fi::u16*>(staging.data_ptr()),
      static_cast<fi::u16*>(k_cache.data_ptr()),
      static_cast<fi::u16*>(v_cache.data_ptr()), block_ids.data_ptr<int>(), n,
      block_elems, current_stream());
}

// What 16-byte pieces are copied from straight to LDS starts on their grid:
// the tensor itself or a copy.
at::Tensor dma_whole(const at::Tensor& t) {
  if (reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0) return t;
  return t.clone(at::MemoryFormat::Contiguous);
}

// and so does every row, at 32-bit byte offsets within a tile of 64
at::Tensor dma_rows(const at::Tensor& t) {
  if (t.stride(0) % 8 == 0 && t.stride(0) <= (1 << 24)) return dma_whole(t);
  return t.clone(at::MemoryFormat::Contiguous);
}

void paged_attention_decode(at::Tensor out, at::Tensor q, at::Tensor k_cache,
                            at::Tensor v_cache, at::Tensor block_tables,
                            at::Tensor seq_lens, double scale) {
  CHECK_BF16_CUDA(out);
  CHECK_BF16_CUDA(q);
  const bool fp8 = cache_is_fp8(k_cache);
  TORCH_CHECK(block_tables.scalar_type() == at::kInt &&
              block_tables.is_contiguous());
  TORCH_CHECK(seq_lens.scalar_type() == at::kInt);
  seq_lens = seq_lens.contiguous();
  TORCH_CHECK(q.dim() == 3);  // [S, Hq, D], rows may be strided
  TORCH_CHECK(out.is_contiguous() && out.sizes() == q.sizes());
  const int num_seqs = q.size(0);
  const int num_heads = q.size(1);
  const int head_dim = q.size(2);
  const int num_kv_heads = k_cache.size(1);
  TORCH_CHECK(k_cache.size(2) == 16, "cache block_size must be 16");
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == head_dim);
  TORCH_CHECK(fi::decode_attn_supported(head_dim, num_heads / num_kv_heads) &&
                  num_heads % num_kv_heads == 0,
              "decode attention takes head sizes 64 and 128 and 1, 2, 4 or 8 "
              "query heads per K/V head");
  if (num_seqs == 0) return;
  q = dma_rows(q);
  k_cache = dma_whole(k_cache);
  v_cache = dma_whole(v_cache);
  at::Tensor pieces = at::empty(
      {fi::decode_piece_floats(num_seqs, num_kv_heads, head_dim,
                               num_heads / num_kv_heads)},
      q.options().dtype(at::kFloat));
  fi::launch_paged_attn_decode(
      bf16_ptr(out), bf16_cptr(q), k_cache.data_ptr(), v_cache.data_ptr(),
      block_tables.data_ptr<int>(), seq_lens.data_ptr<int>(), num_seqs,
      q.stride(0), block_tables.size(1), num_kv_heads, head_dim,
      num_heads / num_kv_heads, static_cast<float>(scale), fp8,
      pieces.data_ptr<float>(), current_stream());
}

// whether the kernel with two groups of queries per wave takes the operands
bool prefill_pairs(int head_dim, bool paged, bool fp8) {
  return paged && head_dim == 128 && !fp8;
}

// a call's choice: cut K/V ranges, two groups of queries per wave, parts
std::tuple<bool, bool, int> prefill_plan(int tiles, int tile_rows,
                                         int num_q_heads, int num_kv_heads,
                                         int new_rows, int max_k_len,
                                         int head_dim, bool paged, bool fp8) {
  const fi::PrefillPlan pl = fi::plan_prefill_attn(
      tiles, tile_rows, num_q_heads, num_kv_heads, new_rows, max_k_len,
      prefill_pairs(head_dim, paged, fp8));
  return {pl.split, pl.pair, pl.slots};
}

// room for the pieces of cut query tiles
at::Tensor prefill_pieces(const fi::PrefillPlan& pl, const at::Tensor& q) {
  if (!pl.split) return at::Tensor();
  return at::empty({fi::prefill_piece_floats(pl, q.size(2))},
                   q.options().dtype(at::kFloat));
}

void prefill_attention(at::Tensor out, at::Tensor q, at::Tensor k,
                       at::Tensor v, at::Tensor tile_seq, at::Tensor tile_row0,
                       at::Tensor cu_seqlens, double scale,
                       int64_t tile_rows) {
  TORCH_CHECK(tile_rows == 128 || tile_rows == 256,
              "tile_rows must be 128 or 256");
  CHECK_BF16_CUDA(out);
  CHECK_BF16_CUDA(q);
  TORCH_CHECK(tile_seq.scalar_type() == at::kInt &&
              tile_row0.scalar_type() == at::kInt &&
              cu_seqlens.scalar_type() == at::kInt);
  TORCH_CHECK(q.dim() == 3 && k.dim() == 3 && v.dim() == 3);
  const int num_q_heads = q.size(1);
  const int head_dim = q.size(2);
  const int num_kv_heads = k.size(1);
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == head_dim);
  TORCH_CHECK(k.stride(2) == 1 && k.stride(1) == head_dim);
  TORCH_CHECK(v.stride(2) == 1 && v.stride(1) == head_dim);
  k = dma_rows(k);
  v = dma_rows(v);
  const fi::PrefillPlan pl = fi::plan_prefill_attn(
      tile_seq.size(0), tile_rows, num_q_heads, num_kv_heads, q.size(0),
      k.size(0), prefill_pairs(head_dim, false, false));
  at::Tensor pieces = prefill_pieces(pl, q);
  fi::launch_prefill_attn(
      bf16_ptr(out), bf16_cptr(q), bf16_cptr(k), bf16_cptr(v),
      tile_seq.data_ptr<int>(), tile_row0.data_ptr<int>(),
      cu_seqlens.data_ptr<int>(), nullptr, nullptr, 0,
      q.stride(0), k.stride(0), v.stride(0), num_q_heads, num_kv_heads,
      head_dim, static_cast<float>(scale), false, pl,
      pl.split ? pieces.data_ptr<float>() : nullptr, current_stream());
}

void prefill_attention_paged(at::Tensor out, at::Tensor q, at::Tensor k_cache,
                             at::Tensor v_cache, at::Tensor tile_seq,
                             at::Tensor tile_row0, at::Tensor cu_seqlens,
                             at::Tensor block_tables, at::Tensor seq_lens_k,
                             double scale, int64_t tile_rows, bool pairs) {
  TORCH_CHECK(tile_rows == 128 || tile_rows == 256,
              "tile_rows must be 128 or 256");
  CHECK_BF16_CUDA(out);
  CHECK_BF16_CUDA(q);
  const bool fp8 = cache_is_fp8(k_cache);
  TORCH_CHECK(tile_seq.scalar_type() == at::kInt &&
              tile_row0.scalar_type() == at::kInt &&
              cu_seqlens.scalar_type() == at::kInt &&
              block_tables.scalar_type() == at::kInt &&
              seq_lens_k.scalar_type() == at::kInt);
  TORCH_CHECK(block_tables.is_contiguous());
  TORCH_CHECK(q.dim() == 3);
  TORCH_CHECK(out.is_contiguous() && out.sizes() == q.sizes());
  const int num_q_heads = q.size(1);
  const int head_dim = q.size(2);
  const int num_kv_heads = k_cache.size(1);
  TORCH_CHECK(k_cache.size(2) == 16, "cache block_size must be 16");
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == head_dim);
  k_cache = dma_whole(k_cache);
  v_cache = dma_whole(v_cache);
  const fi::PrefillPlan pl = fi::plan_prefill_attn(
      tile_seq.size(0), tile_rows, num_q_heads, num_kv_heads, q.size(0),
      block_tables.size(1) * 16, pairs && prefill_pairs(head_dim, true, fp8));
  at::Tensor pieces = prefill_pieces(pl, q);
  fi::launch_prefill_attn(
      bf16_ptr(out), bf16_cptr(q), k_cache.data_ptr(), v_cache.data_ptr(),
      tile_seq.data_ptr<int>(), tile_row0.data_ptr<int>(),
      cu_seqlens.data_ptr<int>(), block_tables.data_ptr<int>(),
      seq_lens_k.data_ptr<int>(), block_tables.size(1),
      q.stride(0), 0, 0, num_q_heads, num_kv_heads, head_dim,
      static_cast<float>(scale), fp8, pl,
      pl.split ? pieces.data_ptr<float>() : nullptr, current_stream());
}

void check_few_rows(const at::Tensor& out, const at::Tensor& x,
                    const at::Tensor& w, bool silu_mul, int64_t most,
                    at::ScalarType out_type = at::kBFloat16,
                    at::ScalarType x_type = at::kBFloat16) {
  TORCH_CHECK(out.is_cuda() && out.scalar_type() == out_type &&
              x.is_cuda() && x.scalar_type() == x_type);
  CHECK_BF16_CUDA(w);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && out.dim() == 2);
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(M >= 1 && M <= most && w.size(1) == K && K % 128 == 0 &&
                  K > 0 && N > 0 && N % (silu_mul ? 32 : 16) == 0 &&
                  K <= (1 << 24) && N <= (1 << 24),
              "few_rows_gemm: unsupported sizes");
  TORCH_CHECK(out.size(0) == M && out.size(1) == (silu_mul ? N / 2 : N));
  TORCH_CHECK(x.stride(1) == 1 && x.stride(0) % 8 == 0 &&
              x.stride(0) <= (1 << (M <= 16 ? 24 : 22)) && w.is_contiguous() &&
              out.stride(1) == 1 && out.stride(0) % 4 == 0);
  TORCH_CHECK(reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(out.data_ptr()) %
                      (4 * out.element_size()) == 0);
}

const u16* check_bias(const c10::optional<at::Tensor>& bias, int64_t N,
                      bool silu_mul) {
  if (!bias.has_value()) return nullptr;
  TORCH_CHECK(!silu_mul && bias->is_cuda() &&
              bias->scalar_type() == at::kBFloat16 && bias->is_contiguous() &&
              bias->numel() == N);
  return bf16_cptr(*bias);
}

// out [M, N] (silu_mul: [M, N / 2]) = x [M, K] @ w [N, K]^T (+ bias); of up to
// 16 rows its gelu
void few_rows_gemm(at::Tensor out, at::Tensor x, at::Tensor w,
                   c10::optional<at::Tensor> bias, bool silu_mul, bool gelu) {
  check_few_rows(out, x, w, silu_mul, gelu ? 16 : 256);
  TORCH_CHECK(!gelu || !(silu_mul || bias.has_value()));
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  const u16* b = check_bias(bias, N, silu_mul);
  if (M <= 16) {
    fi::SkinnyExtra extra;
    extra.gelu = gelu;
    fi::launch_skinny_gemm(bf16_ptr(out), bf16_cptr(x), bf16_cptr(w), b, extra,
                           M, N, K, x.stride(0), out.stride(0), silu_mul,
                           current_stream());
    return;
  }
  at::Tensor pieces = at::empty({fi::part_gemm_floats(M, N, K, false)},
                                x.options().dtype(at::kFloat));
  fi::launch_part_gemm(bf16_ptr(out), pieces.data_ptr<float>(), bf16_cptr(x),
                       bf16_cptr(w), b, M, N, K, x.stride(0), out.stride(0),
                       silu_mul, current_stream());
}

// the same of up to 16 rows of x, divided by the root mean square that squares
// [parts, 16] are the sums of
void few_rows_scaled_gemm(at::Tensor out, at::Tensor x, at::Tensor squares,
                          double eps, at::Tensor w,
                          c10::optional<at::Tensor> bias, bool silu_mul) {
  check_few_rows(out, x, w, silu_mul, 16);
  TORCH_CHECK(squares.is_cuda() && squares.scalar_type() == at::kFloat &&
              squares.dim() == 2 && squares.size(0) >= 1 &&
              squares.size(0) <= (1 << 20) && squares.size(1) == 16 &&
              squares.is_contiguous() &&
              reinterpret_cast<uintptr_t>(squares.data_ptr()) % 16 == 0);
  fi::SkinnyExtra extra;
  extra.squares_in = squares.data_ptr<float>();
  extra.parts = squares.size(0);
  extra.eps = static_cast<float>(eps);
  fi::launch_skinny_gemm(bf16_ptr(out), bf16_cptr(x), bf16_cptr(w),
                         check_bias(bias, w.size(0), silu_mul), extra,
                         x.size(0), w.size(0), x.size(1), x.stride(0),
                         out.stride(0), silu_mul, current_stream());
}

void check_stream(const at::Tensor& stream, const at::Tensor& norm,
                  const at::Tensor& scaled, const at::Tensor& squares,
                  int64_t parts) {
  const int64_t M = stream.size(0), N = stream.size(1);
  CHECK_BF16_CUDA(norm);
  CHECK_BF16_CUDA(scaled);
  TORCH_CHECK(M <= 16 && N % 16 == 0 && norm.is_contiguous() &&
              norm.numel() == N && scaled.is_contiguous() &&
              scaled.sizes() == stream.sizes() && squares.is_cuda() &&
              squares.scalar_type() == at::kFloat && squares.is_contiguous() &&
              squares.dim() == 2 && squares.size(0) == parts &&
              squares.size(1) == 16);
  // (norm on any grid, as in the norms that are kernels of their own)
  TORCH_CHECK(reinterpret_cast<uintptr_t>(scaled.data_ptr()) % 16 == 0);
}

// stream [M, N] fp32 += x [M, K] @ w [N, K]^T, up to 16 rows; with norm also
// scaled [M, N] = stream times norm, squares [N / 16, 16] of the rows
void few_rows_gemm_add(at::Tensor stream, at::Tensor x, at::Tensor w,
                       c10::optional<at::Tensor> norm,
                       c10::optional<at::Tensor> scaled,
                       c10::optional<at::Tensor> squares) {
  check_few_rows(stream, x, w, false, 16, at::kFloat);
  fi::SkinnyExtra extra;
  extra.add = stream.data_ptr<float>();
  TORCH_CHECK(norm.has_value() == scaled.has_value() &&
              norm.has_value() == squares.has_value());
  if (norm.has_value()) {
    check_stream(stream, *norm, *scaled, *squares, w.size(0) / 16);
    extra.norm = bf16_cptr(*norm);
    extra.scaled = bf16_ptr(*scaled);
    extra.squares_out = squares->data_ptr<float>();
  }
  fi::launch_skinny_gemm(nullptr, bf16_cptr(x), bf16_cptr(w), nullptr, extra,
                         x.size(0), w.size(0), x.size(1), x.stride(0),
                         stream.stride(0), false, current_stream());
}

// stream [M, N] = rows (bf16 or fp32), scaled and squares [1, 16] as above
void stream_begin(at::Tensor stream, at::Tensor scaled, at::Tensor squares,
                  at::Tensor rows, at::Tensor norm) {
  TORCH_CHECK(stream.is_cuda() && stream.scalar_type() == at::kFloat &&
              stream.dim() == 2 && stream.size(0) >= 1 &&
              stream.is_contiguous() && rows.is_cuda() &&
              rows.is_contiguous() && rows.sizes() == stream.sizes() &&
              stream.size(1) > 0 && stream.size(1) <= (1 << 24) &&
              reinterpret_cast<uintptr_t>(stream.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(rows.data_ptr()) % 16 == 0);
  check_stream(stream, norm, scaled, squares, 1);
  const int M = stream.size(0), N = stream.size(1);
  if (rows.scalar_type() == at::kFloat) {
    fi::launch_stream_begin(stream.data_ptr<float>(), bf16_ptr(scaled),
                            squares.data_ptr<float>(),
                            static_cast<const float*>(rows.data_ptr()), bf16_cptr(norm), M, N,
                            current_stream());
  } else {
    CHECK_BF16_CUDA(rows);
    fi::launch_stream_begin(stream.data_ptr<float>(), bf16_ptr(scaled),
                            squares.data_ptr<float>(), bf16_cptr(rows),
                            bf16_cptr(norm), M, N, current_stream());
  }
}

// the same for more rows, by tiles of 256 x 256
void many_rows_gemm(at::Tensor out, at::Tensor x, at::Tensor w,
                    c10::optional<at::Tensor> bias, bool silu_mul, bool gelu) {
  TORCH_CHECK(!gelu || !(silu_mul || bias.has_value()));
  CHECK_BF16_CUDA(out);
  CHECK_BF16_CUDA(x);
  CHECK_BF16_CUDA(w);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && out.dim() == 2);
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(M >= 1 && M <= (1 << 24) && w.size(1) == K && K % 64 == 0 &&
                  K >= 128 && N > 0 && N % (silu_mul ? 32 : 16) == 0 &&
                  K <= (1 << 22) && N <= (1 << 24) &&
                  (M + 255) / 256 * ((N + 255) / 256) <= (1 << 24),
              "many_rows_gemm: unsupported sizes");
  TORCH_CHECK(out.size(0) == M && out.size(1) == (silu_mul ? N / 2 : N));
  TORCH_CHECK(x.stride(1) == 1 && x.stride(0) % 8 == 0 && x.stride(0) >= K &&
              x.stride(0) <= (1 << 22) && w.is_contiguous() &&
              out.stride(1) == 1 && out.stride(0) % 8 == 0);
  TORCH_CHECK(reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(out.data_ptr()) % 16 == 0);
  const u16* b = nullptr;
  if (bias.has_value()) {
    TORCH_CHECK(!silu_mul && bias->is_cuda() &&
                bias->scalar_type() == at::kBFloat16 &&
                bias->is_contiguous() && bias->numel() == N &&
                reinterpret_cast<uintptr_t>(bias->data_ptr()) % 16 == 0);
    b = bf16_cptr(*bias);
  }
  at::Tensor pieces = at::empty({fi::tile_gemm_floats(M, N, 2 * K)},
                                x.options().dtype(at::kFloat));
  fi::launch_tile_gemm(bf16_ptr(out), pieces.data_ptr<float>(), bf16_cptr(x),
                       bf16_cptr(w), b, M, N, K, x.stride(0), out.stride(0),
                       silu_mul, gelu, current_stream());
}

void check_few_rows_fp8(const at::Tensor& x, const at::Tensor& x_scales,
                        const at::Tensor& w, const at::Tensor& w_scales,
                        int64_t most) {
  TORCH_CHECK(x.is_cuda() && w.is_cuda() &&
              x.scalar_type() == at::kFloat8_e4m3fn &&
              w.scalar_type() == at::kFloat8_e4m3fn);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2);
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(M >= 1 && M <= most && w.size(1) == K && K % 256 == 0 && K > 0 &&
                  N > 0 && N % 16 == 0 && K <= (1 << 24) && N <= (1 << 24),
              "few_rows_gemm_fp8: unsupported sizes");
  TORCH_CHECK(x.stride(1) == 1 && x.stride(0) % 16 == 0 &&
              x.stride(0) <= (1 << 22) && w.is_contiguous());
  TORCH_CHECK(reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0);
  TORCH_CHECK(x_scales.is_cuda() && x_scales.scalar_type() == at::kFloat &&
              x_scales.is_contiguous() && x_scales.numel() == M &&
              w_scales.is_cuda() && w_scales.scalar_type() == at::kFloat &&
              w_scales.is_contiguous() && w_scales.numel() == N);
}

// out [M, N] bf16 = (x [M, K] * x_scales) @ (w [N, K] * w_scales)^T, e4m3
void few_rows_gemm_fp8(at::Tensor out, at::Tensor x, at::Tensor x_scales,
                       at::Tensor w, at::Tensor w_scales) {
  check_few_rows_fp8(x, x_scales, w, w_scales, 256);
  CHECK_BF16_CUDA(out);
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(out.dim() == 2 && out.size(0) == M && out.size(1) == N &&
              out.stride(1) == 1 && out.stride(0) % 4 == 0 &&
              reinterpret_cast<uintptr_t>(out.data_ptr()) % 8 == 0);
  at::Tensor pieces = at::empty({fi::part_gemm_floats(M, N, K / 2, true)},
                                x.options().dtype(at::kFloat));
  fi::launch_part_gemm_fp8(
      bf16_ptr(out), pieces.data_ptr<float>(),
      static_cast<const unsigned char*>(x.data_ptr()),
      x_scales.data_ptr<float>(),
      static_cast<const unsigned char*>(w.data_ptr()),
      w_scales.data_ptr<float>(), M, N, K, x.stride(0), out.stride(0),
      current_stream());
}

// (x [M, K] @ w [N, K]^T + bias) as heads: queries normed and rotated to q [M,
// num_q_heads * D], K and V rows to the cache; false, with nothing done, where
// the kernels for that are not chosen
bool few_rows_gemm_rope(at::Tensor q, at::Tensor x, at::Tensor w,
                        c10::optional<at::Tensor> bias,
                        c10::optional<at::Tensor> q_weight,
                        c10::optional<at::Tensor> k_weight,
                        at::Tensor cos_sin, at::Tensor positions,
                        at::Tensor k_cache, at::Tensor v_cache,
                        at::Tensor slot_mapping, int64_t num_q_heads,
                        double eps, double k_inv_scale, double v_inv_scale) {
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  const int64_t Hk = k_cache.size(1), D = k_cache.size(3);
  CHECK_BF16_CUDA(q);
  CHECK_BF16_CUDA(x);
  CHECK_BF16_CUDA(w);
  const bool fp8 = cache_is_fp8(k_cache);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && M >= 1 && M <= 256 &&
              w.size(1) == K && K > 0 && K % 128 == 0 && K <= (1 << 24) &&
              N > 0 && N % 16 == 0 && N <= (1 << 24) && x.stride(1) == 1 &&
              x.stride(0) % 8 == 0 && x.stride(0) <= (1 << 22) &&
              w.is_contiguous() &&
              reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0);
  TORCH_CHECK((D == 64 || D == 128) && num_q_heads >= 1 &&
              N == (num_q_heads + 2 * Hk) * D && q.dim() == 2 &&
              q.size(0) == M && q.size(1) == num_q_heads * D &&
              q.is_contiguous());
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat && cos_sin.is_cuda() &&
              cos_sin.size(-1) == D && positions.is_cuda() &&
              positions.scalar_type() == at::kInt && positions.numel() >= M &&
              slot_mapping.is_cuda() &&
              slot_mapping.scalar_type() == at::kInt &&
              slot_mapping.numel() >= M);
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous() &&
              v_cache.sizes() == k_cache.sizes() &&
              v_cache.scalar_type() == k_cache.scalar_type());
  for (const auto& t : {q_weight, k_weight})
    TORCH_CHECK(!t || (t->is_cuda() && t->scalar_type() == at::kBFloat16 &&
                       t->is_contiguous() && t->numel() == D));
  fi::RopeArgs rope{
      q_weight ? bf16_cptr(*q_weight) : nullptr,
      k_weight ? bf16_cptr(*k_weight) : nullptr,
      cos_sin.data_ptr<float>(), positions.data_ptr<int>(),
      static_cast<int>(num_q_heads), static_cast<int>(Hk),
      static_cast<int>(D), static_cast<float>(eps), k_cache.data_ptr(),
      v_cache.data_ptr(), slot_mapping.data_ptr<int>(),
      static_cast<int>(k_cache.size(2)), fp8,
      static_cast<float>(k_inv_scale), static_cast<float>(v_inv_scale)};
  const u16* b = check_bias(bias, N, false);
  const auto run = [&](float* pieces) {
    return M > 16 && fi::launch_part_gemm_rope(
                         bf16_ptr(q), rope, b, pieces, bf16_cptr(x),
                         bf16_cptr(w), M, N, K, x.stride(0), current_stream());
  };
  if (!run(nullptr)) return false;
  at::Tensor pieces = at::empty({fi::part_gemm_floats(M, N, K, false)},
                                x.options().dtype(at::kFloat));
  return run(pieces.data_ptr<float>());
}

void check_norm(const at::Tensor& out, const at::Tensor& residual,
                const at::Tensor& norm, int64_t M, int64_t N) {
  CHECK_BF16_CUDA(residual);
  CHECK_BF16_CUDA(norm);
  TORCH_CHECK(out.dim() == 2 && out.size(0) == M && out.size(1) == N &&
              out.is_contiguous() && residual.sizes() == out.sizes() &&
              residual.is_contiguous() && norm.is_contiguous() &&
              norm.numel() == N);
  TORCH_CHECK(reinterpret_cast<uintptr_t>(out.data_ptr()) % 8 == 0 &&
              reinterpret_cast<uintptr_t>(residual.data_ptr()) % 8 == 0 &&
              reinterpret_cast<uintptr_t>(norm.data_ptr()) % 8 == 0);
}

// residual [M, N] += x [M, K] @ w [N, K]^T, out [M, N] = its rms norm times
// norm; false, with nothing done, where the kernels for that are not chosen
bool few_rows_gemm_norm(at::Tensor out, at::Tensor x, at::Tensor w,
                        at::Tensor residual, at::Tensor norm, double eps) {
  check_few_rows(out, x, w, false, 256);
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  check_norm(out, residual, norm, M, N);
  const auto run = [&](float* pieces) {
    return M > 16 &&
           fi::launch_part_gemm_norm(
               out.data_ptr(), nullptr, bf16_ptr(residual), bf16_cptr(norm),
               static_cast<float>(eps), pieces, bf16_cptr(x), nullptr,
               bf16_cptr(w), nullptr, M, N, K, x.stride(0), current_stream());
  };
  if (!run(nullptr)) return false;
  at::Tensor pieces = at::empty({fi::part_gemm_floats(M, N, K, false)},
                                x.options().dtype(at::kFloat));
  return run(pieces.data_ptr<float>());
}

// the same with e4m3 operands and rows out, a scale per row each
bool few_rows_gemm_norm_fp8(at::Tensor out, at::Tensor out_scales,
                            at::Tensor x, at::Tensor x_scales, at::Tensor w,
                            at::Tensor w_scales, at::Tensor residual,
                            at::Tensor norm, double eps) {
  check_few_rows_fp8(x, x_scales, w, w_scales, 128);
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(out.is_cuda() && out.scalar_type() == at::kFloat8_e4m3fn &&
              out_scales.is_cuda() &&
              out_scales.scalar_type() == at::kFloat &&
              out_scales.is_contiguous() && out_scales.numel() == M);
  check_norm(out, residual, norm, M, N);
  const auto run = [&](float* pieces) {
    return fi::launch_part_gemm_norm(
        out.data_ptr(), out_scales.data_ptr<float>(), bf16_ptr(residual),
        bf16_cptr(norm), static_cast<float>(eps), pieces,
        static_cast<const u16*>(x.data_ptr()), x_scales.data_ptr<float>(),
        static_cast<const u16*>(w.data_ptr()), w_scales.data_ptr<float>(), M,
        N, K / 2, x.stride(0) / 2, current_stream());
  };
  if (!run(nullptr)) return false;
  at::Tensor pieces = at::empty({fi::part_gemm_floats(M, N, K / 2, true)},
                                x.options().dtype(at::kFloat));
  return run(pieces.data_ptr<float>());
}

// the same for more rows, by tiles of 256 x 256
void many_rows_gemm_fp8(at::Tensor out, at::Tensor x, at::Tensor x_scales,
                        at::Tensor w, at::Tensor w_scales) {
  CHECK_BF16_CUDA(out);
  TORCH_CHECK(x.is_cuda() && w.is_cuda() &&
              x.scalar_type() == at::kFloat8_e4m3fn &&
              w.scalar_type() == at::kFloat8_e4m3fn);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && out.dim() == 2);
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(M >= 1 && M <= (1 << 24) && w.size(1) == K && K % 128 == 0 &&
                  K >= 256 && N > 0 && N % 16 == 0 && K <= (1 << 22) &&
                  N <= (1 << 24) &&
                  (M + 255) / 256 * ((N + 255) / 256) <= (1 << 24),
              "many_rows_gemm_fp8: unsupported sizes");
  TORCH_CHECK(out.size(0) == M && out.size(1) == N);
  TORCH_CHECK(x.stride(1) == 1 && x.stride(0) % 16 == 0 && x.stride(0) >= K &&
              x.stride(0) <= (1 << 22) && w.is_contiguous() &&
              out.stride(1) == 1 && out.stride(0) % 8 == 0);
  TORCH_CHECK(reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(out.data_ptr()) % 16 == 0);
  TORCH_CHECK(x_scales.is_cuda() && x_scales.scalar_type() == at::kFloat &&
              x_scales.is_contiguous() && x_scales.numel() == M &&
              w_scales.is_cuda() && w_scales.scalar_type() == at::kFloat &&
              w_scales.is_contiguous() && w_scales.numel() == N &&
              reinterpret_cast<uintptr_t>(w_scales.data_ptr()) % 16 == 0);
  at::Tensor pieces = at::empty({fi::tile_gemm_floats(M, N, K)},
                                x.options().dtype(at::kFloat));
  fi::launch_tile_gemm_fp8(
      bf16_ptr(out), pieces.data_ptr<float>(),
      static_cast<const unsigned char*>(x.data_ptr()),
      x_scales.data_ptr<float>(),
      static_cast<const unsigned char*>(w.data_ptr()),
      w_scales.data_ptr<float>(), M, N, K, x.stride(0), out.stride(0),
      current_stream());
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rms_norm", &rms_norm, "RMSNorm (bf16, fp32 accum)");
  m.def("stream_norm", &stream_norm, "RMSNorm (fp32 to bf16)");
  m.def("fused_add_rms_norm", &fused_add_rms_norm,
        "in-place residual add + RMSNorm");
  m.def("silu_and_mul", &silu_and_mul, "fused SiLU-mul");
  m.def("rms_norm_fp8", &rms_norm_fp8, "RMSNorm with fused fp8 row quant");
  m.def("fused_add_rms_norm_fp8", &fused_add_rms_norm_fp8,
        "residual add + RMSNorm with fused fp8 row quant");
  m.def("silu_and_mul_fp8", &silu_and_mul_fp8,
        "fused SiLU-mul with fp8 row quant");
  m.def("quant_fp8_rows", &quant_fp8_rows, "per-row dynamic fp8 quant");
  m.def("rope_qk_norm", &rope_qk_norm,
        "fused per-head qk RMSNorm + NeoX RoPE (in-place)");
  m.def("rope_qk_norm_cache", &rope_qk_norm_cache,
        "rope_qk_norm with K and V scattered into the paged cache");
  m.def("reshape_and_cache", &reshape_and_cache, "scatter K/V into paged cache");
  m.def("gather_kv_blocks", &gather_kv_blocks, "pack KV blocks for PD send");
  m.def("scatter_kv_blocks", &scatter_kv_blocks, "unpack KV blocks from PD recv");
  m.def("few_rows_gemm", &few_rows_gemm, "x W^T for up to 256 rows of x",
        py::arg("out"), py::arg("x"), py::arg("w"), py::arg("bias"),
        py::arg("silu_mul"), py::arg("gelu") = false);
  m.def("few_rows_scaled_gemm", &few_rows_scaled_gemm,
        "linear layer of up to 16 rows over their root mean square");
  m.def("few_rows_gemm_add", &few_rows_gemm_add,
        "fp32 stream += linear layer of up to 16 rows, and the next norm");
  m.def("stream_begin", &stream_begin, "fp32 stream of rows, the next norm");
  m.def("few_rows_gemm_us", &fi::part_gemm_us,
        "estimate for M of 17 to 256 rows (e4m3: 1 to 128), N, K", py::arg("M"),
        py::arg("N"), py::arg("K"), py::arg("fp8") = false);
  m.def("many_rows_gemm", &many_rows_gemm, "x W^T by tiles of 256 x 256",
        py::arg("out"), py::arg("x"), py::arg("w"), py::arg("bias"),
        py::arg("silu_mul"), py::arg("gelu") = false);
  m.def("many_rows_gemm_us", &fi::tile_gemm_us,
        "estimate for M, N, bytes of a row of K");
  m.def("many_rows_gemm_fp8", &many_rows_gemm_fp8,
        "x W^T by tiles of 256 x 256, e4m3 with scales per row");
  m.def("few_rows_gemm_rope", &few_rows_gemm_rope,
        "heads of x W^T to q and the cache, or false");
  m.def("few_rows_gemm_norm", &few_rows_gemm_norm,
        "residual += x W^T and its norm, or false");
  m.def("few_rows_gemm_norm_fp8", &few_rows_gemm_norm_fp8,
        "the same with e4m3 operands and rows out");
  m.def("few_rows_gemm_fp8", &few_rows_gemm_fp8,
        "x W^T for up to 256 rows of e4m3 x with scales per row");
  m.def("paged_attention_decode", &paged_attention_decode,
        "paged decode attention");
  m.def("prefill_attention", &prefill_attention, "varlen causal MFMA prefill");
  m.def("prefill_attention_paged", &prefill_attention_paged,
        "varlen causal MFMA prefill over the paged cache (context attention)",
        py::arg("out"), py::arg("q"), py::arg("k_cache"), py::arg("v_cache"),
        py::arg("tile_seq"), py::arg("tile_row0"), py::arg("cu_seqlens"),
        py::arg("block_tables"), py::arg("seq_lens_k"), py::arg("scale"),
        py::arg("tile_rows"), py::arg("pairs") = true);
  m.def("prefill_plan", &prefill_plan,
        "(split, two groups of queries per wave, parts) for tiles, tile_rows, "
        "query heads, K/V heads, new rows, longest K/V range, head_dim, paged, "
        "fp8");
}
