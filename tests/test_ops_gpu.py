"""GPU numerics tests: every HIP kernel vs the PyTorch fp32 reference.

Mirrors the reference's test strategy tier 1 (table-driven unit tests)
applied to the data plane: each op is compared against
ops/reference.py on random inputs.
"""

import math
import random

import pytest
import torch

import fusioninfer_amd.ops as ops
from fusioninfer_amd.ops import reference as ref

pytestmark = pytest.mark.gpu

DEV = "cuda"


def setup_module():
    assert ops.has_native(), "HIP extension must be present on a GPU box"
    torch.manual_seed(0)


def assert_close_bf16(actual, expected_f32, atol=2e-2, rtol=2e-2):
    torch.testing.assert_close(
        actual.float(), expected_f32.float(), atol=atol, rtol=rtol
    )


@pytest.mark.parametrize("tokens,hidden", [(1, 1024), (17, 4096), (256, 4096), (33, 8192)])
def test_rms_norm(tokens, hidden):
    x = torch.randn(tokens, hidden, dtype=torch.bfloat16, device=DEV)
    w = torch.randn(hidden, dtype=torch.bfloat16, device=DEV)
    out = ops.rms_norm(x, w, 1e-6)
    expected = ref.rms_norm(x.cpu(), w.cpu(), 1e-6)
    assert_close_bf16(out.cpu(), expected)


@pytest.mark.parametrize("tokens,hidden", [(16, 4096), (130, 4096)])
def test_fused_add_rms_norm(tokens, hidden):
    x = torch.randn(tokens, hidden, dtype=torch.bfloat16, device=DEV)
    res = torch.randn(tokens, hidden, dtype=torch.bfloat16, device=DEV)
    w = torch.randn(hidden, dtype=torch.bfloat16, device=DEV)
    x_ref, res_ref = ref.fused_add_rms_norm(x.cpu(), res.cpu(), w.cpu(), 1e-6)
    out, new_res = ops.fused_add_rms_norm(x, res, w, 1e-6)
    assert_close_bf16(new_res.cpu(), res_ref)
    assert_close_bf16(out.cpu(), x_ref)


@pytest.mark.parametrize("hidden", [12288, 12296, 14344, 16384])
@pytest.mark.parametrize("tokens", [1, 256, 257, 2048, 2049])
def test_norms_of_wide_rows(tokens, hidden):
    """Where the weight is requested and the residual is written changes at
    257 and 2049 rows and above 12288 values."""
    g = torch.Generator(DEV).manual_seed(tokens + hidden)
    x, res = (torch.randn(tokens, hidden, dtype=torch.bfloat16, device=DEV,
                          generator=g) for _ in range(2))
    w = torch.randn(hidden, dtype=torch.bfloat16, device=DEV, generator=g)

    def normed(rows):
        rows = rows.float()
        return rows * torch.rsqrt(rows.square().mean(-1, keepdim=True)
                                  + 1e-6) * w.float()

    def near_fp8(f8, scales, exact):
        # half a step of e4m3 is 2^-4 of a value, and 2^-10 of the scale
        # where values are small
        err = (f8.float() * scales[:, None] - exact).abs()
        assert (err <= exact.abs() / 16 + scales[:, None] / 512).all()

    exact = normed(x)
    assert_close_bf16(ops.rms_norm(x, w, 1e-6), exact)
    near_fp8(*ops.rms_norm_fp8(x, w, 1e-6), exact)
    total = x.float() + res.float()
    exact = normed(total)
    f8, scales, new = ops.fused_add_rms_norm_fp8(x, res.clone(), w, 1e-6)
    assert torch.equal(new, total.bfloat16())
    near_fp8(f8, scales, exact)
    out, new = ops.fused_add_rms_norm(x, res, w, 1e-6)
    assert torch.equal(new, total.bfloat16())
    assert_close_bf16(out, exact)


@pytest.mark.parametrize("hidden", [1024, 2048, 2056, 4096, 16384])
def test_norm_order_of_the_first_squares(hidden):
    """A thread adds its squares by fma, of the first two the second comes
    first (the first in rows of up to 2048 values): the same two values
    further on, in that order, give the same bits, and in the other order
    they do not always."""
    rows = 4096
    g = torch.Generator(DEV).manual_seed(hidden)
    x, res = (torch.randn(rows, 2, dtype=torch.bfloat16, device=DEV,
                          generator=g) for _ in range(2))
    w = torch.ones(hidden, dtype=torch.bfloat16, device=DEV)

    def scales_and_rows(*at):
        a, b = (torch.zeros(rows, hidden, dtype=torch.bfloat16, device=DEV)
                for _ in range(2))
        a[:, list(at)], b[:, list(at)] = x, res
        scales = ops.fused_add_rms_norm_fp8(a, b.clone(), w, 0.0)[1]
        return scales, ops.fused_add_rms_norm(a, b, w, 0.0)[0][:, list(at)]

    first, first_rows = scales_and_rows(0, 1)
    same, same_rows = scales_and_rows(*((2, 3) if hidden <= 2048 else (3, 2)))
    other, _ = scales_and_rows(*((3, 2) if hidden <= 2048 else (2, 3)))
    assert torch.equal(first, same) and torch.equal(first_rows, same_rows)
    assert not torch.equal(first, other)


@pytest.mark.parametrize("tokens,inter", [(7, 12288), (64, 512)])
def test_silu_and_mul(tokens, inter):
    x = torch.randn(tokens, 2 * inter, dtype=torch.bfloat16, device=DEV)
    out = ops.silu_and_mul(x)
    expected = ref.silu_and_mul(x.cpu())
    assert_close_bf16(out.cpu(), expected)


def _assert_fp8_close(got_f8, got_sc, exp_f8, exp_sc, exact=None):
    """fp8 kernel vs CPU reference. The kernel quantizes from unrounded
    f32 registers while the reference quantizes the bf16-rounded op
    output, so scales agree only to bf16 precision and elements may land
    one e4m3 quantum apart — compare dequantized values against the
    reference DEQUANTIZED output within fp8 quantization error (e4m3: 3
    mantissa bits, max rel step 2^-4; two independent quantizations of
    near-identical data differ by <~1 quantum RMS)."""
    torch.testing.assert_close(got_sc.cpu(), exp_sc, atol=1e-5, rtol=2e-2)
    got = got_f8.float().cpu() * got_sc.cpu().unsqueeze(-1)
    exp = exp_f8.float() * exp_sc.unsqueeze(-1)
    rel = (got - exp).norm() / exp.norm().clamp(min=1e-6)
    assert rel.item() < 0.05, rel.item()
    if exact is not None:  # anchor to the unquantized fp32 op output
        rel = (got - exact.float()).norm() / exact.float().norm().clamp(min=1e-6)
        assert rel.item() < 0.06, rel.item()


@pytest.mark.parametrize("tokens,hidden", [(1, 1024), (17, 4096), (64, 8192)])
def test_rms_norm_fp8(tokens, hidden):
    x = torch.randn(tokens, hidden, dtype=torch.bfloat16, device=DEV)
    w = torch.randn(hidden, dtype=torch.bfloat16, device=DEV)
    f8, sc = ops.rms_norm_fp8(x, w, 1e-6)
    ef8, esc = ref.rms_norm_fp8(x.cpu(), w.cpu(), 1e-6)
    _assert_fp8_close(f8, sc, ef8, esc, exact=ref.rms_norm(x.cpu(), w.cpu(), 1e-6))


@pytest.mark.parametrize("tokens,hidden", [(16, 4096), (130, 4096)])
def test_fused_add_rms_norm_fp8(tokens, hidden):
    x = torch.randn(tokens, hidden, dtype=torch.bfloat16, device=DEV)
    res = torch.randn(tokens, hidden, dtype=torch.bfloat16, device=DEV)
    w = torch.randn(hidden, dtype=torch.bfloat16, device=DEV)
    exact, _ = ref.fused_add_rms_norm(x.cpu(), res.cpu(), w.cpu(), 1e-6)
    ef8, esc, eres = ref.fused_add_rms_norm_fp8(x.cpu(), res.cpu(), w.cpu(), 1e-6)
    f8, sc, new_res = ops.fused_add_rms_norm_fp8(x, res, w, 1e-6)
    assert_close_bf16(new_res.cpu(), eres)
    _assert_fp8_close(f8, sc, ef8, esc, exact=exact)


@pytest.mark.parametrize("tokens,inter", [(7, 12288), (64, 512)])
def test_silu_and_mul_fp8(tokens, inter):
    x = torch.randn(tokens, 2 * inter, dtype=torch.bfloat16, device=DEV)
    f8, sc = ops.silu_and_mul_fp8(x)
    ef8, esc = ref.silu_and_mul_fp8(x.cpu())
    _assert_fp8_close(f8, sc, ef8, esc, exact=ref.silu_and_mul(x.cpu()))


@pytest.mark.parametrize("tokens,cols", [(1, 4096), (33, 2048), (256, 4096)])
def test_quant_fp8_rows(tokens, cols):
    x = torch.randn(tokens, cols, dtype=torch.bfloat16, device=DEV)
    f8, sc = ops.quant_fp8_rows(x)
    ef8, esc = ref.quant_fp8_rows(x.cpu())
    _assert_fp8_close(f8, sc, ef8, esc, exact=x.cpu())


@pytest.mark.parametrize("cols", [2056, 4096, 4104, 6144, 6152, 8192, 8200, 10240,
                                  10248, 12288, 16384])
@pytest.mark.parametrize("silu_mul", [False, True])
def test_quant_fp8_of_rows_of_all_lengths(cols, silu_mul):
    """One to five vectors a thread, workgroups of all sizes, and the loads and
    stores for more than the caches hold give the bits of short calls; those
    are within half a step of e4m3 (2^-4 relative, 2^-10 of the scale) and fp32
    roundings of silu of the exact rows, the largest of which is 448."""
    width = cols * (2 if silu_mul else 1)
    call = ops.silu_and_mul_fp8 if silu_mul else ops.quant_fp8_rows
    rows = (1 << 27) // width + 3        # of 2 bytes: more than 256 MB
    x = torch.randn(rows, width, device=DEV, dtype=torch.bfloat16)
    f8, sc = call(x)
    for part in (slice(0, 1), slice(1, 34), slice(34, 634),
                 slice(rows - 40, rows)):
        g8, gs = call(x[part])
        assert torch.equal(g8.view(torch.uint8), f8[part].view(torch.uint8))
        assert torch.equal(gs, sc[part])
    want = x[-40:].double()
    if silu_mul:
        want = torch.nn.functional.silu(want[:, :cols]) * want[:, cols:]
    scale = want.abs().amax(1) / 448
    torch.testing.assert_close(sc[-40:].double(), scale, rtol=2 ** -18, atol=0)
    got = f8[-40:].double() * sc[-40:].double()[:, None]
    assert ((got - want).abs() <= want.abs() * (2 ** -4 + 2 ** -18)
            + scale[:, None] * 2 ** -10).all()



@pytest.mark.parametrize("qk_norm", [True, False])
@pytest.mark.parametrize("head_dim", [64, 128])
def test_rope_qk_norm(qk_norm, head_dim):
    T, Hq, Hk = 33, 8, 2
    torch.manual_seed(1)
    # row-strided slices of a fused qkv buffer, like the real model
    qkv = torch.randn(T, (Hq + 2 * Hk) * head_dim, dtype=torch.bfloat16, device=DEV)
    q = qkv[:, : Hq * head_dim]
    k = qkv[:, Hq * head_dim : (Hq + Hk) * head_dim]
    positions = torch.randint(0, 500, (T,), dtype=torch.int32, device=DEV)
    cos_sin = ops.compute_cos_sin_cache(head_dim, 512, 10000.0).to(DEV)
    qw = torch.randn(head_dim, dtype=torch.bfloat16, device=DEV) if qk_norm else None
    kw = torch.randn(head_dim, dtype=torch.bfloat16, device=DEV) if qk_norm else None

    q_ref, k_ref = ref.rope_qk_norm(
        q.cpu().view(T, Hq, head_dim),
        k.cpu().view(T, Hk, head_dim),
        positions.cpu().long(),
        cos_sin.cpu(),
        qw.cpu() if qw is not None else None,
        kw.cpu() if kw is not None else None,
        1e-6,
    )
    ops.rope_qk_norm_(q, k, positions, cos_sin, Hq, Hk, head_dim, qw, kw, 1e-6)
    assert_close_bf16(q.cpu().view(T, Hq, head_dim), q_ref)
    assert_close_bf16(k.cpu().view(T, Hk, head_dim), k_ref)


def test_reshape_and_cache():
    T, Hk, D, bs, nblocks = 37, 4, 128, 16, 12
    k = torch.randn(T, Hk * D, dtype=torch.bfloat16, device=DEV)
    v = torch.randn(T, Hk * D, dtype=torch.bfloat16, device=DEV)
    k_cache = torch.zeros(nblocks, Hk, bs, D, dtype=torch.bfloat16, device=DEV)
    v_cache = torch.zeros_like(k_cache)
    slots = torch.randperm(nblocks * bs, device=DEV)[:T].to(torch.int32)
    k_ref = k_cache.cpu().clone()
    v_ref = v_cache.cpu().clone()
    ref.reshape_and_cache(
        k.cpu().view(T, Hk, D), v.cpu().view(T, Hk, D), k_ref, v_ref, slots.cpu().long()
    )
    ops.reshape_and_cache(k, v, k_cache, v_cache, slots)
    torch.testing.assert_close(k_cache.cpu(), k_ref)
    torch.testing.assert_close(v_cache.cpu(), v_ref)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("T,Hq,Hk,D,pad", [
    (1, 16, 8, 128, 0),
    (33, 8, 2, 64, 8),    # a wave's last heads are missing
    (130, 5, 1, 128, 1),  # odd heads; rows at any address
    (7, 1, 1, 64, 3),
])
def test_rope_qk_norm_cache(T, Hq, Hk, D, pad, fp8):
    """One kernel against the two it stands for: q, both caches, bit for bit
    what rope_qk_norm_ and reshape_and_cache leave, rows of negative slots
    left out. And against the fp32 oracle: one bf16 rounding each (2^-9, 2^-8
    of an ulp that falls the other way) and 1e-5 for fp32 sums; a cached row
    as bf16 rounds it, in e4m3 with its scale at most one step (2^-3) off."""
    torch.manual_seed(2)
    qkv = torch.randn(T, (Hq + 2 * Hk) * D + pad, device=DEV,
                      dtype=torch.bfloat16)[:, pad:]
    cos_sin = ops.compute_cos_sin_cache(D, 512, 10000.0).to(DEV)
    positions = torch.randint(0, 512, (T,), dtype=torch.int32, device=DEV)
    qw = torch.randn(D, dtype=torch.bfloat16, device=DEV)
    slots = torch.randperm(160, device=DEV)[:T].to(torch.int32)
    if T > 2:
        slots[1] = -1
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    caches = [torch.zeros(10, Hk, 16, D, device=DEV).to(dt)
              for _ in range(4)]
    cut = lambda t: (t[:, :Hq * D], t[:, Hq * D:(Hq + Hk) * D],
                     t[:, (Hq + Hk) * D:])
    want_q, want_k = ref.rope_qk_norm(
        *(t.cpu().float().view(T, -1, D) for t in cut(qkv)[:2]),
        positions.cpu().long(), cos_sin.cpu(), qw.cpu().float(), None)
    want_v = cut(qkv)[2].cpu().float().view(T, Hk, D)
    q, k, v = cut(qkv.clone())
    ops.rope_qk_norm_(q, k, positions, cos_sin, Hq, Hk, D, qw, None)
    ops.reshape_and_cache(k.contiguous(), v.contiguous(), *caches[:2], slots,
                          1 / 3., 1 / 4.)
    got, k0, v0 = cut(qkv)
    ops.rope_qk_norm_cache_(got, k0, v0, positions, cos_sin, *caches[2:],
                            slots, Hq, qw, None, 1e-6, 1 / 3., 1 / 4.)
    assert torch.equal(got, q)
    for a, b in zip(caches[:2], caches[2:]):
        assert a.float().abs().sum() > 0
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    assert_close_bf16(got.cpu().view(T, Hq, D), want_q, atol=1e-5,
                      rtol=2 ** -8)
    kept = (slots >= 0).cpu()
    at = slots[slots >= 0].cpu().long()
    for cache, want, inv in ((caches[2], want_k, 1 / 3.),
                             (caches[3], want_v, 1 / 4.)):
        row = cache.cpu().float()[at // 16, :, at % 16]
        want = want[kept] * (inv if fp8 else 1.0)
        assert_close_bf16(row, want, atol=2 ** -9 if fp8 else 1e-5,
                          rtol=2 ** -3 if fp8 else 2 ** -8)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("Hq,Hk,D", [
    (5, 1, 128),     # a wave's second unit is partly, or not at all, there
    (72, 4, 128),    # more heads than a workgroup's waves take
    (33, 3, 64),
])
def test_rope_qk_norm_cache_of_many_tokens(Hq, Hk, D, norm, fp8):
    """Many tokens, from 2^22 values on two units of heads per wave, are bit
    for bit what the same tokens in shorter calls are, of up to 256 of them
    with four waves a workgroup; q against the fp32 oracle, one bf16 rounding
    (2^-8: of an ulp that falls the other way) and 1e-5 for fp32 sums."""
    torch.manual_seed(3)
    T = -(-2 ** 22 // ((Hq + 2 * Hk) * D))
    qkv = torch.randn(T, (Hq + 2 * Hk) * D, device=DEV, dtype=torch.bfloat16)
    cos_sin = ops.compute_cos_sin_cache(D, 512, 10000.0).to(DEV)
    positions = torch.randint(0, 512, (T,), dtype=torch.int32, device=DEV)
    qw, kw = torch.randn(2, D, device=DEV).to(torch.bfloat16) if norm \
        else (None, None)
    blocks = T // 16 + 2
    slots = torch.randperm(blocks * 16, device=DEV)[:T].to(torch.int32)
    slots[300] = -1
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    caches = [torch.zeros(blocks, Hk, 16, D, device=DEV).to(dt) for _ in range(4)]

    def run(x, rows, k_cache, v_cache):
        q, k, v = x[rows].split([Hq * D, Hk * D, Hk * D], dim=1)
        ops.rope_qk_norm_cache_(q, k, v, positions[rows], cos_sin, k_cache,
                                v_cache, slots[rows], Hq, qw, kw, 1e-6,
                                1 / 3., 1 / 4.)

    whole, parts = qkv.clone(), qkv.clone()
    run(whole, slice(0, T), *caches[:2])
    run(parts, slice(0, 256), *caches[2:])
    run(parts, slice(256, T), *caches[2:])
    assert torch.equal(whole, parts)
    for a, b in zip(caches[:2], caches[2:]):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    want, _ = ref.rope_qk_norm(
        qkv[:, :Hq * D].cpu().float().view(T, Hq, D),
        qkv[:, Hq * D:(Hq + Hk) * D].cpu().float().view(T, Hk, D),
        positions.cpu().long(), cos_sin.cpu(),
        *(w.cpu().float() if norm else None for w in (qw, kw)))
    assert_close_bf16(whole[:, :Hq * D].cpu().view(T, Hq, D), want,
                      atol=1e-5, rtol=2 ** -8)


def test_kv_block_gather_scatter_roundtrip():
    Hk, D, bs, nblocks = 2, 128, 16, 20
    k_cache = torch.randn(nblocks, Hk, bs, D, dtype=torch.bfloat16, device=DEV)
    v_cache = torch.randn_like(k_cache)
    ids = torch.tensor([3, 7, 1, 19], dtype=torch.int32, device=DEV)
    staging = ops.gather_kv_blocks(k_cache, v_cache, ids)
    expected = ref.gather_kv_blocks(k_cache.cpu(), v_cache.cpu(), ids.cpu().long())
    torch.testing.assert_close(staging.cpu(), expected)

    # scatter into a fresh cache at different ids
    k2 = torch.zeros_like(k_cache)
    v2 = torch.zeros_like(v_cache)
    ids2 = torch.tensor([0, 2, 4, 6], dtype=torch.int32, device=DEV)
    ops.scatter_kv_blocks(staging, k2, v2, ids2)
    torch.testing.assert_close(k2[ids2.long()].cpu(), k_cache[ids.long()].cpu())
    torch.testing.assert_close(v2[ids2.long()].cpu(), v_cache[ids.long()].cpu())


@pytest.mark.parametrize("group", [1, 4, 8])
@pytest.mark.parametrize(
    "seq_lens", [[1], [16], [1, 5, 16, 17, 255, 1023]]
)
def test_paged_attention_decode(group, seq_lens):
    torch.manual_seed(2)
    Hk, D, bs = 2, 128, 16
    Hq = Hk * group
    S = len(seq_lens)
    max_blocks = (max(seq_lens) + bs - 1) // bs
    total_blocks = sum((L + bs - 1) // bs for L in seq_lens) + 2
    q = torch.randn(S, Hq, D, dtype=torch.bfloat16, device=DEV)
    k_cache = torch.randn(total_blocks, Hk, bs, D, dtype=torch.bfloat16, device=DEV)
    v_cache = torch.randn_like(k_cache)
    # assign blocks sequentially
    bt = torch.zeros(S, max_blocks, dtype=torch.int32, device=DEV)
    nxt = 1
    for s, L in enumerate(seq_lens):
        n = (L + bs - 1) // bs
        bt[s, :n] = torch.arange(nxt, nxt + n, dtype=torch.int32)
        nxt += n
    lens = torch.tensor(seq_lens, dtype=torch.int32, device=DEV)
    scale = 1.0 / math.sqrt(D)
    out = ops.paged_attention_decode(q, k_cache, v_cache, bt, lens, scale)
    expected = ref.paged_attention_decode(
        q.cpu(), k_cache.cpu(), v_cache.cpu(), bt.cpu(), lens.cpu(), scale
    )
    assert_close_bf16(out.cpu(), expected, atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize(
    "seq_lens,hq,hk",
    [([64], 4, 4), ([128], 8, 2), ([1, 33, 64, 100, 257], 8, 2)],
)
def test_prefill_attention(head_dim, seq_lens, hq, hk):
    torch.manual_seed(3)
    T = sum(seq_lens)
    q = torch.randn(T, hq, head_dim, dtype=torch.bfloat16, device=DEV)
    k = torch.randn(T, hk, head_dim, dtype=torch.bfloat16, device=DEV)
    v = torch.randn(T, hk, head_dim, dtype=torch.bfloat16, device=DEV)
    cu = torch.tensor(
        [0] + list(torch.tensor(seq_lens).cumsum(0)), dtype=torch.int32, device=DEV
    )
    scale = 1.0 / math.sqrt(head_dim)
    out = ops.prefill_attention(q, k, v, cu, scale)
    expected = ref.prefill_attention(q.cpu(), k.cpu(), v.cpu(), cu.cpu(), scale)
    assert_close_bf16(out.cpu(), expected, atol=3e-2, rtol=3e-2)


def _shifted(t, by):
    """t's values in a tensor that starts `by` elements off the grid."""
    flat = torch.empty(t.numel() + by, dtype=t.dtype, device=t.device)
    return flat[by:].view(t.shape).copy_(t)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("pad,by", [(4, 0), (8, 1), (1, 3)])
def test_attention_rows_off_the_16_byte_grid(head_dim, pad, by):
    """K, V and caches whose rows or start lie off the grid of the 16-byte
    copies give the bits that the same values on the grid give."""
    g = torch.Generator().manual_seed(head_dim + pad)

    def rnd(*shape):
        return torch.randn(*shape, generator=g).to(torch.bfloat16).to(DEV)

    T, hk, w = 130, 2, 2 * head_dim
    q, k, v = rnd(T, 4, head_dim), rnd(T, hk, head_dim), rnd(T, hk, head_dim)
    cu = torch.tensor([0, 33, T], dtype=torch.int32, device=DEV)
    wide = _shifted(torch.cat([k.view(T, w), v.view(T, w), rnd(T, pad)], 1),
                    by)
    scale = head_dim ** -0.5
    assert torch.equal(
        ops.prefill_attention(q, k, v, cu, scale),
        ops.prefill_attention(q, wide[:, :w].view(T, hk, head_dim),
                              wide[:, w:2 * w].view(T, hk, head_dim), cu,
                              scale))
    kc, vc = rnd(9, hk, 16, head_dim), rnd(9, hk, 16, head_dim)
    off = _shifted(kc, by), _shifted(vc, by)
    bt = torch.randperm(9, generator=g).int()[None].to(DEV)
    lens = torch.tensor([140], dtype=torch.int32, device=DEV)
    one = torch.tensor([0, 1], dtype=torch.int32, device=DEV)
    assert torch.equal(
        ops.paged_attention_decode(q[:1], kc, vc, bt, lens, scale),
        ops.paged_attention_decode(q[:1], *off, bt, lens, scale))
    assert torch.equal(
        ops.prefill_attention_paged(q[:1], kc, vc, bt, one, lens, scale),
        ops.prefill_attention_paged(q[:1], *off, bt, one, lens, scale))


def test_prefill_attention_spiked_scores():
    """Force large per-tile max jumps so online-softmax rescale paths fire
    (bounded random data never exercises them)."""
    torch.manual_seed(4)
    L, hq, hk, D = 256, 2, 2, 128
    q = torch.randn(L, hq, D, dtype=torch.bfloat16, device=DEV)
    k = torch.randn(L, hk, D, dtype=torch.bfloat16, device=DEV) * 0.1
    # spike some K rows late in the sequence: max jumps at a late tile
    k[200] = q[250, 0].sign() * 3.0
    k[77] = q[100, 1].sign() * 2.0
    v = torch.randn(L, hk, D, dtype=torch.bfloat16, device=DEV)
    cu = torch.tensor([0, L], dtype=torch.int32, device=DEV)
    out = ops.prefill_attention(q, k, v, cu)
    expected = ref.prefill_attention(q.cpu(), k.cpu(), v.cpu(), cu.cpu(), 1.0 / math.sqrt(D))
    assert_close_bf16(out.cpu(), expected, atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize(
    "ctx_lens,new_lens",
    [([48], [48]), ([128], [32]), ([64, 100, 300], [64, 36, 44])],
)
def test_prefill_attention_paged(ctx_lens, new_lens):
    """Context attention over the paged cache vs the fp32 reference."""
    torch.manual_seed(5)
    Hq, Hk, D, bs = 8, 2, 128, 16
    S = len(ctx_lens)
    Tn = sum(new_lens)
    max_blocks = max((c + bs - 1) // bs for c in ctx_lens)
    total_blocks = sum((c + bs - 1) // bs for c in ctx_lens) + 1
    q = torch.randn(Tn, Hq, D, dtype=torch.bfloat16, device=DEV)
    k_cache = torch.randn(total_blocks, Hk, bs, D, dtype=torch.bfloat16, device=DEV)
    v_cache = torch.randn_like(k_cache)
    bt = torch.zeros(S, max_blocks, dtype=torch.int32, device=DEV)
    nxt = 1
    for s, c in enumerate(ctx_lens):
        n = (c + bs - 1) // bs
        bt[s, :n] = torch.arange(nxt, nxt + n, dtype=torch.int32)
        nxt += n
    cu_q = torch.tensor(
        [0] + list(torch.tensor(new_lens).cumsum(0)), dtype=torch.int32, device=DEV
    )
    lens_k = torch.tensor(ctx_lens, dtype=torch.int32, device=DEV)
    scale = 1.0 / math.sqrt(D)
    out = ops.prefill_attention_paged(q, k_cache, v_cache, bt, cu_q, lens_k, scale)
    expected = ref.prefill_attention_paged(
        q.cpu(), k_cache.cpu(), v_cache.cpu(), bt.cpu(), cu_q.cpu(),
        lens_k.cpu(), scale,
    )
    assert_close_bf16(out.cpu(), expected, atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize(
    "hq,hk,ctx_lens,new_lens,scale_by",
    [
        # whole row blocks: ends on, before and behind K/V tiles (64) and
        # row blocks (128 / heads per workgroup), groups of 1, 2, 3, 8
        (4, 4, [129, 64, 1], [129, 1, 1], 1.0),
        (4, 2, [65, 200], [65, 63], -1.0),
        (6, 2, [300], [257], 0.0),
        (16, 2, [97, 31], [33, 31], 1.0),
        # cut K/V ranges: one row, a row block and one row, several requests
        # whose row blocks share parts, parts that end on a row block
        (8, 2, [2100], [1], 1.0),
        (8, 2, [4400, 2049], [65, 3], 1.0),
        (3, 3, [3000, 40, 2500], [130, 40, 2], -1.0),
        (16, 2, [2560, 2560], [64, 64], 1.0),
    ],
)
def test_prefill_attention_row_blocks_and_parts(hq, hk, ctx_lens, new_lens,
                                                scale_by, head_dim, fp8):
    """Edges of row blocks, K/V tiles and equal parts against the fp32
    reference. Bound: P and the output are rounded to bf16 (2^-9 each) and
    |v| stays below 5, hence 2e-2."""
    g = torch.Generator().manual_seed(11)

    def rnd(*shape):
        return torch.randn(*shape, generator=g).to(torch.bfloat16).to(DEV)

    bs = 16
    need = [(c + bs - 1) // bs for c in ctx_lens]
    perm = (torch.randperm(sum(need), generator=g) + 1).int()
    bt = torch.zeros(len(need), max(need), dtype=torch.int32)
    for s, row in enumerate(perm.split(need)):
        bt[s, :need[s]] = row
    q = rnd(sum(new_lens), hq, head_dim)
    k_cache = rnd(sum(need) + 1, hk, bs, head_dim)
    v_cache = rnd(sum(need) + 1, hk, bs, head_dim)
    if fp8:
        k_cache, v_cache = _fp8_cache(k_cache), _fp8_cache(v_cache)
    else:
        # rows behind a context's end are never read
        for s, c in enumerate(ctx_lens):
            if c % bs:
                v_cache[int(bt[s, need[s] - 1]), :, c % bs:] = float("nan")
                k_cache[int(bt[s, need[s] - 1]), :, c % bs:] = float("nan")
    cu = torch.tensor([0] + list(torch.tensor(new_lens).cumsum(0)),
                      dtype=torch.int32)
    lens = torch.tensor(ctx_lens, dtype=torch.int32)
    scale = scale_by / math.sqrt(head_dim)
    out = ops.prefill_attention_paged(q, k_cache, v_cache, bt.to(DEV),
                                      cu.to(DEV), lens.to(DEV), scale)
    want = ref.prefill_attention_paged(q.cpu(), k_cache.cpu(), v_cache.cpu(),
                                       bt, cu, lens, scale)
    assert_close_bf16(out.cpu(), want, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("scale_by", [1.0, -1.0, 8.0])
@pytest.mark.parametrize("hq,hk", [
    (64, 16),    # four heads per workgroup
    (64, 32),    # two
    (64, 64),    # one
])
def test_prefill_attention_long_parts(hq, hk, scale_by):
    """Parts of more than 128 K/V tiles (two groups of queries per wave):
    odd rows, a portion of 33 and one whose end lies within a tile, maxima
    that jump late, against float64. Bound: P and the output are rounded to
    bf16 (2^-9 each) and |v| stays below 6, hence 2.4e-2. One group per wave
    over the same parts gives the same bits."""
    g = torch.Generator().manual_seed(hq + hk)
    new_lens, ctx_lens, D = [901, 33], [9001, 8064], 128
    need = [-(-c // 16) for c in ctx_lens]
    perm = (torch.randperm(sum(need), generator=g) + 1).int()
    bt = torch.zeros(len(need), max(need), dtype=torch.int32)
    for i, row in enumerate(perm.split(need)):
        bt[i, :need[i]] = row

    def rnd(*shape):
        return torch.randn(*shape, generator=g).to(torch.bfloat16).to(DEV)

    q = rnd(sum(new_lens), hq, D)
    kc, vc = rnd(sum(need) + 1, hk, 16, D), rnd(sum(need) + 1, hk, 16, D)
    kc[int(bt[0, 300]), :, 5] *= 3.0     # a key that outweighs those before
    for c in (kc, vc):                   # behind the end: never read
        c[int(bt[0, need[0] - 1]), :, ctx_lens[0] % 16:] = float("nan")
    cu = torch.tensor([0, 901, 934], dtype=torch.int32, device=DEV)
    lens = torch.tensor(ctx_lens, dtype=torch.int32, device=DEV)
    scale = scale_by / math.sqrt(D)
    out = ops.prefill_attention_paged(q, kc, vc, bt.to(DEV), cu, lens, scale)
    tile_rows = ops.prefill_tile_rows(new_lens)
    tiles = ops.build_prefill_tiles(new_lens, device=DEV, rows=tile_rows)
    plan = (tiles[0].shape[0], tile_rows, hq, hk, len(q), bt.shape[1] * 16, D,
            True)
    assert ops._C.prefill_plan(*plan, False)[:2] == (True, True)
    assert ops._C.prefill_plan(*plan, True)[:2] == (True, False)
    alone = torch.empty_like(out)
    ops._C.prefill_attention_paged(alone, q, kc, vc, *tiles, cu, bt.to(DEV),
                                   lens, scale, tile_rows, pairs=False)
    assert torch.equal(out, alone)
    at = 0
    for i, (n, c) in enumerate(zip(new_lens, ctx_lens)):
        rows = bt[i, :need[i]].long().to(DEV)
        hide = torch.arange(c, device=DEV) > torch.arange(
            c - n, c, device=DEV)[:, None]
        for h in range(0, hq, 7):
            k = kc[rows, h * hk // hq].reshape(-1, D)[:c].double()
            v = vc[rows, h * hk // hq].reshape(-1, D)[:c].double()
            s = (q[at:at + n, h].double() @ k.T) * scale
            s = s.masked_fill(hide, -math.inf)
            want = torch.softmax(s, 1) @ v
            err = (out[at:at + n, h].double() - want).abs()
            assert (err <= 2.4e-2).all(), (i, h, err.max())
        at += n


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hq,hk,head_dim,seqs,longest", [
    (32, 8, 128, 9, 700),     # a few query tiles each, of very uneven work
    (8, 2, 128, 60, 150),     # lists that end with none
    (64, 64, 128, 420, 3),    # more than a list holds: more workgroups
    (8, 2, 64, 60, 150),      # heads of 64: one each, whatever their number
    (24, 8, 128, 150, 70),    # three heads a group: one per workgroup
    (32, 8, 128, 1040, 9),    # more query tiles than are put in order
    (64, 64, 64, 420, 3),
])
def test_prefill_attention_lists_of_query_tiles(hq, hk, head_dim, seqs,
                                                longest, fp8):
    """Workgroups that take several query tiles one after the other, against
    launches so small that each takes one: the same bits for every row, rows of
    other requests and behind a context's end never read."""
    rng = random.Random(seqs)
    g = torch.Generator().manual_seed(seqs)
    new = [rng.randint(1, longest) for _ in range(seqs)]
    past = [rng.choice([0, 0, 5, 40]) for _ in range(seqs)]
    ctx = [a + b for a, b in zip(new, past)]
    need = [-(-c // 16) for c in ctx]
    perm = (torch.randperm(sum(need), generator=g) + 1).int()
    bt = torch.zeros(seqs, max(need), dtype=torch.int32)
    for i, row in enumerate(perm.split(need)):
        bt[i, :need[i]] = row
    q = torch.randn(sum(new), hq, head_dim, generator=g).bfloat16().to(DEV)
    kc, vc = (torch.randn(sum(need) + 1, hk, 16, head_dim,
                          generator=g).bfloat16().to(DEV) for _ in range(2))
    if fp8:
        kc, vc = _fp8_cache(kc), _fp8_cache(vc)
    else:
        for i, c in enumerate(ctx):
            if c % 16:
                for t in (kc, vc):
                    t[int(bt[i, need[i] - 1]), :, c % 16:] = float("nan")
    bt = bt.to(DEV)

    def run(i, j):
        first = sum(new[:i])
        rows = q[first:first + sum(new[i:j])]
        cu = torch.tensor([0] + list(torch.tensor(new[i:j]).cumsum(0)),
                          dtype=torch.int32, device=DEV)
        lens = torch.tensor(ctx[i:j], dtype=torch.int32, device=DEV)
        table = ops.build_prefill_tiles(new[i:j], device=DEV, rows=256)
        plan = ops._C.prefill_plan(table[0].shape[0], 256, hq, hk, len(rows),
                                   max(need) * 16, head_dim, True, fp8)
        if plan[0]:                      # parts round elsewhere
            return None
        return ops.prefill_attention_paged(rows, kc, vc, bt[i:j], cu, lens,
                                           head_dim ** -0.5, *table, 256)

    out = run(0, seqs)
    assert out is not None and torch.isfinite(out).all()
    # 256 rows of a group of one head are two query tiles or more, and 512
    # query tiles over all heads go one to a workgroup
    per = 256 * hq // 128
    step = max(1, 512 // per) if longest <= 256 else 1
    picks = range(0, seqs, step) if seqs <= 150 else \
        rng.sample(range(seqs - step), 40)
    tested = 0
    for i in picks:
        want = run(i, min(i + step, seqs))
        if want is not None:
            at = sum(new[:i])
            assert torch.equal(out[at:at + len(want)], want), i
            tested += 1
    assert tested > 0
    i = max(range(seqs), key=lambda n: new[n])
    at = sum(new[:i])
    b = bt[i, :need[i]].long()
    k, v = (t[b].float().permute(1, 0, 2, 3).reshape(hk, -1, head_dim)
            [:, :ctx[i]].repeat_interleave(hq // hk, 0).cpu() for t in (kc, vc))
    s = q[at:at + new[i]].float().cpu().transpose(0, 1) @ k.transpose(1, 2)
    hide = torch.arange(ctx[i]) > torch.arange(past[i], ctx[i])[:, None]
    want = torch.softmax((s * head_dim ** -0.5).masked_fill(hide, -math.inf),
                         -1) @ v
    # P and the output are rounded to bf16 (2^-9 each), |v| stays below 5
    assert_close_bf16(out[at:at + new[i]].cpu(),
                      want.transpose(0, 1).bfloat16(), atol=2e-2, rtol=2e-2)


LIST_LENS = [700, 1, 130, 513, 64, 900, 300]   # new rows of the requests


@pytest.mark.parametrize("hq,hk,head_dim", [
    (32, 8, 128),     # a group's heads side by side in a workgroup
    (40, 8, 128),     # one head a workgroup
    (32, 8, 64), (32, 32, 64)])
def test_prefill_attention_dense_lists_of_query_tiles(hq, hk, head_dim):
    """Dense rows, more query tiles than workgroups: the bits of each request
    alone; rows of the next request are never read for this one's."""
    g = torch.Generator().manual_seed(hq + head_dim)
    lens = LIST_LENS
    q, k, v = (torch.randn(sum(lens), h, head_dim, generator=g).bfloat16()
               .to(DEV) for h in (hq, hk, hk))
    at = [0, *torch.tensor(lens).cumsum(0).tolist()]

    def run(i, j):
        cu = torch.tensor([n - at[i] for n in at[i:j + 1]], dtype=torch.int32,
                          device=DEV)
        rows = slice(at[i], at[j])
        return ops.prefill_attention(q[rows], k[rows], v[rows], cu)

    out = run(0, len(lens))
    for i in range(len(lens)):
        assert torch.equal(out[at[i]:at[i + 1]], run(i, i + 1)), i


@pytest.mark.parametrize("hq,hk,fp8", [(32, 8, False), (32, 8, True),
                                       (32, 32, False), (32, 32, True)])
def test_prefill_attention_lists_of_query_tiles_heads_of_64(hq, hk, fp8):
    """Heads of 64 go by lists between one round of workgroups and three, of
    contexts of 512 to 4096 (here 960 query tiles; contexts of 944 and fewer):
    the bits of each request alone. And rows off the 16-byte grid."""
    g = torch.Generator().manual_seed(hk)
    new, past = LIST_LENS, [40, 0, 0, 5, 0, 40, 0]
    ctx = [a + b for a, b in zip(new, past)]
    need = [-(-c // 16) for c in ctx]
    bt = torch.zeros(len(new), max(need), dtype=torch.int32)
    for i, row in enumerate((torch.randperm(sum(need), generator=g) + 1)
                            .int().split(need)):
        bt[i, :need[i]] = row
    q = torch.randn(sum(new), hq, 64, generator=g).bfloat16().to(DEV)
    kc, vc = (torch.randn(sum(need) + 1, hk, 16, 64, generator=g).bfloat16()
              .to(DEV) for _ in range(2))
    if fp8:
        kc, vc = _fp8_cache(kc), _fp8_cache(vc)
    bt = bt.to(DEV)
    at = [0, *torch.tensor(new).cumsum(0).tolist()]

    def run(i, j, out=None):
        cu = torch.tensor([n - at[i] for n in at[i:j + 1]], dtype=torch.int32,
                          device=DEV)
        lens = torch.tensor(ctx[i:j], dtype=torch.int32, device=DEV)
        return ops.prefill_attention_paged(q[at[i]:at[j]], kc, vc, bt[i:j], cu,
                                           lens, out=out)

    out = run(0, len(new))
    for i in range(len(new)):
        assert torch.equal(out[at[i]:at[i + 1]], run(i, i + 1)), i
    off = torch.full((out.numel() + 8,), 7.0, dtype=out.dtype, device=DEV)
    run(0, len(new), off[4:-4].view(out.shape))
    assert torch.equal(off[4:-4].view(out.shape), out)
    assert (off[:4] == 7).all() and (off[-4:] == 7).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("heads,groups,block,window,keep,gate", [
    (32, 8, 16, 0, 0, None), (32, 8, 1, 0, 0, "entry"),
    (32, 32, 8, 0, 0, "head"),     # one head a workgroup
    (32, 8, 16, 200, 70, "entry"),  # a window: one query tile a workgroup
    (40, 8, 1, 33, 0, "head")])
def test_sink_attention_many_row_tiles(D, heads, groups, block, window, keep,
                                       gate):
    """More query tiles than workgroups (832 and more), the next one's keys of
    another portion: the bits of each portion alone, also off the 16-byte grid."""
    from fusioninfer_amd.ops import seqmix

    g = torch.Generator().manual_seed(D + heads + window)
    new, past = LIST_LENS, [40, 0, 277, 5, 0, 64, 0]
    ctx = [a + b for a, b in zip(new, past)]
    need = [-(-c // block) for c in ctx]
    order = torch.randperm(sum(need) + 2, generator=g)
    table = torch.zeros(len(new), max(need), dtype=torch.int32)
    for i, row in enumerate(order[:sum(need)].int().split(need)):
        table[i, :need[i]] = row
    T = sum(new)
    q = torch.randn(T, heads, D, generator=g).bfloat16().to(DEV)
    k, v = (torch.randn(len(order), groups, block, D, generator=g).bfloat16()
            .to(DEV) for _ in range(2))
    sink = (torch.randn(heads, generator=g) * 3).to(DEV)
    og = {"head": torch.randn(T, heads, generator=g),
          "entry": torch.randn(T, heads * D, generator=g)}.get(gate)
    og = None if og is None else og.bfloat16().to(DEV)
    at = [0, *torch.tensor(new).cumsum(0).tolist()]

    def run(i, j, out=None):
        rows = slice(at[i], at[j])
        return seqmix.sink_paged_attention(
            q[rows], k, v, table[i:j].to(DEV),
            torch.cat([torch.full((n,), m) for m, n in enumerate(new[i:j])])
            .int().to(DEV),
            torch.cat([torch.arange(p, p + n) for n, p in
                       zip(new[i:j], past[i:j])]).int().to(DEV), D ** -0.5,
            sink=sink, out_gate=None if og is None else og[rows],
            seq_cu=torch.tensor([n - at[i] for n in at[i:j + 1]],
                                dtype=torch.int32, device=DEV),
            tiles=seqmix.build_attention_tiles(new[i:j], device=DEV),
            window=window, keep_first=keep, out=out)

    out = run(0, len(new))
    assert torch.isfinite(out).all()
    for i in range(len(new)):
        assert torch.equal(out[at[i]:at[i + 1]], run(i, i + 1)), i
    off = torch.full((out.numel() + 8,), 7.0, dtype=out.dtype, device=DEV)
    run(0, len(new), off[4:-4].view(out.shape))
    assert torch.equal(off[4:-4].view(out.shape), out)
    assert (off[:4] == 7).all() and (off[-4:] == 7).all()


@pytest.mark.parametrize("hq,hk", [(2, 2), (3, 1)])
def test_prefill_attention_one_head_per_workgroup_small_entries(hq, hk):
    """4099 new rows make the tile table's entries 128 rows; with one head
    per workgroup a row still belongs to one workgroup: the same bits every
    time. Bound as above."""
    g = torch.Generator().manual_seed(8)
    D, new, past = 64, 4099, 8205
    blocks = -(-(new + past) // 16)
    assert ops.prefill_tile_rows([new]) == 128
    q = torch.randn(new, hq, D, generator=g).bfloat16().to(DEV)
    k = torch.randn(blocks, hk, 16, D, generator=g).bfloat16().to(DEV)
    v = torch.randn(blocks, hk, 16, D, generator=g).bfloat16().to(DEV)
    bt = torch.randperm(blocks, generator=g).int()[None].to(DEV)
    cu = torch.tensor([0, new], dtype=torch.int32, device=DEV)
    lens = torch.tensor([new + past], dtype=torch.int32, device=DEV)
    outs = [ops.prefill_attention_paged(q, k, v, bt, cu, lens, D ** -0.5)
            for _ in range(3)]
    want = ref.prefill_attention_paged(q, k, v, bt, cu, lens, D ** -0.5)
    assert_close_bf16(outs[0], want, atol=2e-2, rtol=2e-2)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize(
    "group,hk,lens,scale_by",
    [
        # ends around pages (16) and two-page steps
        (4, 2, [1, 15, 16, 17, 31, 32, 33], 1.0),
        # contexts shorter than a part, more of them than lanes, several
        # borders inside one part
        (2, 3, [1 + (7 * i) % 50 for i in range(150)], -1.0),
        # one context over many parts; parts that cut it unevenly
        (8, 1, [5000], 1.0),
        (1, 4, [3, 2500, 16, 900], 1.0),
        # long and short in turn: whole contexts between cut ones
        (4, 8, [1200, 5, 1201, 64, 3000, 1] * 6, 0.0),
    ],
)
def test_paged_attention_decode_parts(group, hk, lens, scale_by, head_dim,
                                      fp8):
    """Borders of pages, contexts and parts against the fp32 reference (same
    bound as above); what lies behind a context's end is never read."""
    g = torch.Generator().manual_seed(13)
    bs, S = 16, len(lens)

    def rnd(*shape):
        return torch.randn(*shape, generator=g).to(torch.bfloat16).to(DEV)

    need = [(c + bs - 1) // bs for c in lens]
    perm = (torch.randperm(sum(need), generator=g) + 1).int()
    bt = torch.zeros(S, max(need) + 3, dtype=torch.int32)
    for s, row in enumerate(perm.split(need)):
        bt[s, :need[s]] = row
    # the query part of a merged projection
    q = rnd(S, 2 * group * hk * head_dim)[:, : group * hk * head_dim]
    q = q.view(S, group * hk, head_dim)
    k_cache = rnd(sum(need) + 1, hk, bs, head_dim)
    v_cache = rnd(sum(need) + 1, hk, bs, head_dim)
    if fp8:
        k_cache, v_cache = _fp8_cache(k_cache), _fp8_cache(v_cache)
    else:
        for s, c in enumerate(lens):
            if c % bs:
                v_cache[int(bt[s, need[s] - 1]), :, c % bs:] = float("nan")
                k_cache[int(bt[s, need[s] - 1]), :, c % bs:] = float("nan")
    scale = scale_by / math.sqrt(head_dim)
    sl = torch.tensor(lens, dtype=torch.int32)
    out = ops.paged_attention_decode(q, k_cache, v_cache, bt.to(DEV),
                                     sl.to(DEV), scale)
    want = ref.paged_attention_decode(q.cpu(), k_cache.cpu(), v_cache.cpu(),
                                      bt, sl, scale)
    assert_close_bf16(out.cpu(), want, atol=2e-2, rtol=2e-2)
    # rows off the 16-byte grid give the same
    off = torch.empty(S, q[0].numel() + 1, dtype=q.dtype, device=DEV)[:, 1:]
    off = off.view(S, group * hk, head_dim).copy_(q)
    assert torch.equal(out, ops.paged_attention_decode(
        off, k_cache, v_cache, bt.to(DEV), sl.to(DEV), scale))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("group", [1, 4, 8])
def test_paged_attention_decode_weights_are_fp32(group, head_dim, fp8):
    """The last value row takes back what the others add up to, so that the
    sum is far smaller than its terms: a weight of eight bits is off by 2^-9
    of a term. Bound: the bf16 result's 2^-8 of itself, and 1e-5 of the terms
    for fp32 scores of 128 products (2^-24 of their 80 or so each) and exp2."""
    g = torch.Generator().manual_seed(17)
    bs, hk, lens = 16, 2, [2, 3, 7, 16, 17, 33]
    cache = torch.float8_e4m3fn if fp8 else torch.bfloat16
    S, blocks = len(lens), -(-max(lens) // bs)
    scale = 1.0 / math.sqrt(head_dim)

    def rnd(*shape):
        return torch.randn(*shape, generator=g).to(cache).double()

    q = torch.randn(S, hk, 1, head_dim, generator=g).to(torch.bfloat16)
    q = q.expand(-1, -1, group, -1).reshape(S, hk * group, head_dim)
    k_cache = rnd(S * blocks, hk, bs, head_dim)
    v_cache = rnd(S * blocks, hk, bs, head_dim)
    bt = torch.arange(S * blocks, dtype=torch.int32).view(S, blocks)
    want = torch.empty(S, hk * group, head_dim, dtype=torch.float64)
    size = torch.empty_like(want)
    for i, n in enumerate(lens):
        rows = slice(i * blocks, (i + 1) * blocks)
        for h in range(hk):
            k = k_cache[rows, h].reshape(-1, head_dim)[:n]
            v = v_cache[rows, h].reshape(-1, head_dim)[:n].clone()
            p = torch.softmax(k @ q[i, h * group].double() * scale, 0)
            v[-1] = (-(p[:-1] @ v[:-1]) / p[-1]).clamp(-400, 400).to(
                cache).double()
            v_cache[i * blocks + (n - 1) // bs, h, (n - 1) % bs] = v[-1]
            want[i, h * group:(h + 1) * group] = p @ v
            size[i, h * group:(h + 1) * group] = p @ v.abs()
    out = ops.paged_attention_decode(
        q.to(DEV), k_cache.to(cache).to(DEV), v_cache.to(cache).to(DEV),
        bt.to(DEV), torch.tensor(lens, dtype=torch.int32, device=DEV), scale)
    err = (out.cpu().double() - want).abs()
    assert (err <= 2 ** -8 * want.abs() + 1e-5 * size).all(), \
        (err / size).max()


@pytest.mark.parametrize("head_dim", [64, 128])
def test_paged_attention_decode_infinite_values(head_dim):
    """An infinite value makes its column infinite and no other, also where
    it stands in the context's last row."""
    bs, lens = 16, [1, 5, 16, 40]
    S, blocks = len(lens), 3
    g = torch.Generator().manual_seed(3)
    q = torch.randn(S, 4, head_dim, generator=g).to(torch.bfloat16)
    k_cache = torch.randn(S * blocks, 1, bs, head_dim, generator=g).to(q.dtype)
    v_cache = torch.randn(S * blocks, 1, bs, head_dim, generator=g).to(q.dtype)
    for i, n in enumerate(lens):
        v_cache[i * blocks + (n - 1) // bs, 0, (n - 1) % bs, 7] = math.inf
        v_cache[i * blocks, 0, 0, 9] = -math.inf
    bt = torch.arange(S * blocks, dtype=torch.int32).view(S, blocks)
    sl = torch.tensor(lens, dtype=torch.int32)
    scale = 1.0 / math.sqrt(head_dim)
    out = ops.paged_attention_decode(q.to(DEV), k_cache.to(DEV),
                                     v_cache.to(DEV), bt.to(DEV), sl.to(DEV),
                                     scale).cpu()
    want = ref.paged_attention_decode(q, k_cache, v_cache, bt, sl, scale)
    assert (out[..., 7] == math.inf).all() and (out[..., 9] == -math.inf).all()
    rest = torch.ones(head_dim, dtype=torch.bool)
    rest[[7, 9]] = False
    assert_close_bf16(out[..., rest], want[..., rest])


# ------------------------------------------------------------ fp8 KV cache

def _fp8_cache(t):
    return t.to(torch.float8_e4m3fn)


def test_reshape_and_cache_fp8():
    T, Hk, D, bs, nblocks = 37, 4, 128, 16, 12
    k = torch.randn(T, Hk * D, dtype=torch.bfloat16, device=DEV)
    v = torch.randn(T, Hk * D, dtype=torch.bfloat16, device=DEV)
    k_cache = torch.zeros(nblocks, Hk, bs, D, dtype=torch.float8_e4m3fn,
                          device=DEV)
    v_cache = torch.zeros_like(k_cache)
    slots = torch.randperm(nblocks * bs, device=DEV)[:T].to(torch.int32)
    k_ref = torch.zeros(nblocks, Hk, bs, D, dtype=torch.float8_e4m3fn)
    v_ref = torch.zeros_like(k_ref)
    ref.reshape_and_cache(
        k.cpu().view(T, Hk, D), v.cpu().view(T, Hk, D), k_ref, v_ref,
        slots.cpu().long()
    )
    ops.reshape_and_cache(k, v, k_cache, v_cache, slots)
    # hardware cvt vs torch cast can differ 1 ulp on RNE ties -> compare
    # dequantized with one-quantum tolerance
    torch.testing.assert_close(
        k_cache.float().cpu(), k_ref.float(), atol=0.07, rtol=0.07
    )
    torch.testing.assert_close(
        v_cache.float().cpu(), v_ref.float(), atol=0.07, rtol=0.07
    )


def test_reshape_and_cache_fp8_inv_scale():
    """Per-layer static KV scales: the write multiplies by the inverse
    scale before e4m3 conversion; out-of-range inputs saturate (matching
    the reference's clamp) instead of NaN-ing."""
    T, Hk, D, bs, nblocks = 9, 2, 64, 16, 4
    k = torch.randn(T, Hk * D, dtype=torch.bfloat16, device=DEV) * 3.0
    v = torch.randn(T, Hk * D, dtype=torch.bfloat16, device=DEV) * 600.0
    k_cache = torch.zeros(nblocks, Hk, bs, D, dtype=torch.float8_e4m3fn,
                          device=DEV)
    v_cache = torch.zeros_like(k_cache)
    slots = torch.arange(T, device=DEV, dtype=torch.int32)
    k_ref = torch.zeros(nblocks, Hk, bs, D, dtype=torch.float8_e4m3fn)
    v_ref = torch.zeros_like(k_ref)
    ref.reshape_and_cache(
        k.cpu().view(T, Hk, D), v.cpu().view(T, Hk, D), k_ref, v_ref,
        slots.cpu().long(), 1.0 / 3.0, 1.0 / 4.0
    )
    ops.reshape_and_cache(k, v, k_cache, v_cache, slots, 1.0 / 3.0, 1.0 / 4.0)
    assert torch.isfinite(v_cache.float()).all()
    torch.testing.assert_close(
        k_cache.float().cpu(), k_ref.float(), atol=0.07, rtol=0.07
    )
    torch.testing.assert_close(
        v_cache.float().cpu(), v_ref.float(), atol=12.0, rtol=0.07
    )


@pytest.mark.parametrize("group", [1, 4, 8])
@pytest.mark.parametrize("seq_lens", [[1], [1, 5, 16, 17, 255, 1023]])
def test_paged_attention_decode_fp8kv(group, seq_lens):
    """Decode over an fp8 (e4m3, scale-1) cache: the kernel and the fp32
    reference read the SAME quantized cache, so tolerances stay tight."""
    torch.manual_seed(6)
    Hk, D, bs = 2, 128, 16
    Hq = Hk * group
    S = len(seq_lens)
    max_blocks = (max(seq_lens) + bs - 1) // bs
    total_blocks = sum((L + bs - 1) // bs for L in seq_lens) + 2
    q = torch.randn(S, Hq, D, dtype=torch.bfloat16, device=DEV)
    k_cache = _fp8_cache(
        torch.randn(total_blocks, Hk, bs, D, dtype=torch.bfloat16, device=DEV))
    v_cache = _fp8_cache(
        torch.randn(total_blocks, Hk, bs, D, dtype=torch.bfloat16, device=DEV))
    bt = torch.zeros(S, max_blocks, dtype=torch.int32, device=DEV)
    nxt = 1
    for s, L in enumerate(seq_lens):
        n = (L + bs - 1) // bs
        bt[s, :n] = torch.arange(nxt, nxt + n, dtype=torch.int32)
        nxt += n
    lens = torch.tensor(seq_lens, dtype=torch.int32, device=DEV)
    scale = 1.0 / math.sqrt(D)
    out = ops.paged_attention_decode(q, k_cache, v_cache, bt, lens, scale)
    expected = ref.paged_attention_decode(
        q.cpu(), k_cache.cpu(), v_cache.cpu(), bt.cpu(), lens.cpu(), scale
    )
    # G=8 dispatches the fp8 MFA variant, which quantizes Q to e4m3
    # per head (the reference keeps fp32 Q) — one extra quantization
    # step of score error
    tol = 6e-2 if group == 8 else 3e-2
    assert_close_bf16(out.cpu(), expected, atol=tol, rtol=tol)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize(
    "ctx_lens,new_lens",
    [([48], [48]), ([64, 100, 300], [64, 36, 44])],
)
def test_prefill_attention_paged_fp8kv(head_dim, ctx_lens, new_lens):
    torch.manual_seed(7)
    Hq, Hk, bs, D = 8, 2, 16, head_dim
    S = len(ctx_lens)
    Tn = sum(new_lens)
    max_blocks = max((c + bs - 1) // bs for c in ctx_lens)
    total_blocks = sum((c + bs - 1) // bs for c in ctx_lens) + 1
    q = torch.randn(Tn, Hq, D, dtype=torch.bfloat16, device=DEV)
    k_cache = _fp8_cache(
        torch.randn(total_blocks, Hk, bs, D, dtype=torch.bfloat16, device=DEV))
    v_cache = _fp8_cache(
        torch.randn(total_blocks, Hk, bs, D, dtype=torch.bfloat16, device=DEV))
    bt = torch.zeros(S, max_blocks, dtype=torch.int32, device=DEV)
    nxt = 1
    for s, c in enumerate(ctx_lens):
        n = (c + bs - 1) // bs
        bt[s, :n] = torch.arange(nxt, nxt + n, dtype=torch.int32)
        nxt += n
    cu_q = torch.tensor(
        [0] + list(torch.tensor(new_lens).cumsum(0)), dtype=torch.int32,
        device=DEV
    )
    lens_k = torch.tensor(ctx_lens, dtype=torch.int32, device=DEV)
    scale = 1.0 / math.sqrt(D)
    out = ops.prefill_attention_paged(q, k_cache, v_cache, bt, cu_q, lens_k,
                                      scale)
    expected = ref.prefill_attention_paged(
        q.cpu(), k_cache.cpu(), v_cache.cpu(), bt.cpu(), cu_q.cpu(),
        lens_k.cpu(), scale
    )
    assert_close_bf16(out.cpu(), expected, atol=3e-2, rtol=3e-2)


def test_kv_block_copy_fp8_roundtrip():
    Hk, D, bs, nblocks = 2, 128, 16, 20
    k_cache = _fp8_cache(
        torch.randn(nblocks, Hk, bs, D, dtype=torch.bfloat16, device=DEV))
    v_cache = _fp8_cache(
        torch.randn(nblocks, Hk, bs, D, dtype=torch.bfloat16, device=DEV))
    ids = torch.tensor([3, 7, 1, 19], dtype=torch.int32, device=DEV)
    staging = ops.gather_kv_blocks(k_cache, v_cache, ids)
    assert staging.dtype == torch.float8_e4m3fn
    k2 = torch.zeros_like(k_cache)
    v2 = torch.zeros_like(v_cache)
    ids2 = torch.tensor([0, 2, 4, 6], dtype=torch.int32, device=DEV)
    ops.scatter_kv_blocks(staging, k2, v2, ids2)
    torch.testing.assert_close(
        k2[ids2.long()].float().cpu(), k_cache[ids.long()].float().cpu())
    torch.testing.assert_close(
        v2[ids2.long()].float().cpu(), v_cache[ids.long()].float().cpu())


# ---------------------------------------------------------------- MoE


@pytest.mark.parametrize("block_m", [16, 128])
@pytest.mark.parametrize("gate_up", [True, False])
def test_moe_gemm_vs_reference(block_m, gate_up):
    """Grouped MFMA GEMM vs the CPU fp32 reference (same align inputs)."""
    torch.manual_seed(block_m + int(gate_up))
    E, K, N = 5, 256, 128
    T = 300
    w = torch.randn(E, K, (2 * N) if gate_up else N,
                    dtype=torch.bfloat16, device=DEV) * 0.05
    b_packed = ops.pack_moe_weights(w)
    # synthetic block-aligned assignment: uneven expert loads
    counts = [0, 7, block_m, 2 * block_m + 3, 1]
    tiles = [-(-c // block_m) for c in counts if c > 0]
    n_tiles = sum(tiles)
    PM = (n_tiles + 2) * block_m  # slack tiles past n_valid stay untouched
    sorted_ids = torch.zeros(PM, dtype=torch.int32, device=DEV)
    expert_ids = torch.zeros(PM // block_m, dtype=torch.int32, device=DEV)
    p = 0
    t = 0
    for e, c in enumerate(counts):
        if c == 0:
            continue
        nt = -(-c // block_m)
        for i in range(c):
            sorted_ids[p + i] = t % T
            t += 3
        expert_ids[p // block_m : p // block_m + nt] = e
        p += nt * block_m
    n_valid = torch.tensor([n_tiles], dtype=torch.int32, device=DEV)
    a = torch.randn(max(T, PM), K, dtype=torch.bfloat16, device=DEV)
    out = torch.full((PM, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.moe_gemm(out, a, b_packed, sorted_ids, expert_ids, n_valid,
                 block_m, gate_up)
    want = torch.full((PM, N), float("nan"), dtype=torch.bfloat16)
    from fusioninfer_amd.ops import reference as _r

    _r.moe_gemm(want, a.cpu(), b_packed.cpu(), sorted_ids.cpu(),
                expert_ids.cpu(), n_valid.cpu(), block_m, gate_up)
    rows = n_tiles * block_m
    torch.testing.assert_close(
        out[:rows].float().cpu(), want[:rows].float(), atol=3e-2, rtol=3e-2
    )
    # tiles past n_valid untouched on both
    assert out[rows:].isnan().all()


def test_moe_combine_vs_reference():
    torch.manual_seed(3)
    T, topk, H, PM = 23, 4, 256, 128
    y = torch.randn(PM, H, dtype=torch.bfloat16, device=DEV)
    pos = torch.randint(-1, PM, (T * topk,), dtype=torch.int32, device=DEV)
    w = torch.rand(T * topk, dtype=torch.float32, device=DEV)
    out = torch.empty(T, H, dtype=torch.bfloat16, device=DEV)
    ops.moe_combine(out, y, pos, w)
    want = torch.empty(T, H, dtype=torch.bfloat16)
    from fusioninfer_amd.ops import reference as _r

    _r.moe_combine(want, y.cpu(), pos.cpu(), w.cpu())
    torch.testing.assert_close(out.float().cpu(), want.float(),
                               atol=2e-2, rtol=2e-2)


def test_moe_grouped_forward_matches_manual():
    """Full MoEMLP grouped path on GPU vs a per-token manual reference."""
    import torch.nn.functional as F

    from fusioninfer_amd.models.model import MoEMLP
    from fusioninfer_amd.models.registry import get_model_config

    torch.manual_seed(11)
    cfg = get_model_config("tiny-qwen3-moe")
    with torch.device(DEV):
        mlp = MoEMLP(cfg, layer_idx=0)
    for T in (1, 9, 300):
        x = torch.randn(T, cfg.hidden_size, dtype=torch.bfloat16,
                        device=DEV) * 0.5
        got = mlp(x).float()
        logits = x.float() @ mlp.router_weight.float().T
        topv, topi = torch.softmax(logits, -1).topk(mlp.top_k, -1)
        topv = topv / topv.sum(-1, keepdim=True)
        exp = torch.zeros_like(got)
        for t in range(T):
            for k in range(mlp.top_k):
                e = int(topi[t, k])
                gu = x[t].float() @ mlp.gate_up_t[e].float()
                g, u = gu.chunk(2)
                y = (F.silu(g) * u) @ mlp.down_t[e].float()
                exp[t] += float(topv[t, k]) * y
        rel = (got - exp).norm() / exp.norm()
        assert rel.item() < 0.05, (T, rel.item())


def test_moe_gemm_fp8_vs_reference():
    """Grouped fp8 GEMM (dequant epilogue) vs the CPU fp32 reference."""
    torch.manual_seed(9)
    E, K, N, T = 4, 128, 128, 200
    for gate_up in (True, False):
        w = (torch.randn(E, K, (2 * N) if gate_up else N) * 0.1).to(
            torch.float8_e4m3fn).cuda()
        ws = torch.rand(E, (2 * N) if gate_up else N,
                        dtype=torch.float32, device=DEV) * 0.2 + 0.01
        b_packed = ops.pack_moe_weights(w.view(torch.int8)).view(
            torch.float8_e4m3fn)
        block_m = 16
        counts = [5, 0, 2 * block_m, 9]
        tiles = [-(-c // block_m) for c in counts if c > 0]
        n_tiles = sum(tiles)
        PM = (n_tiles + 1) * block_m
        sorted_ids = torch.zeros(PM, dtype=torch.int32, device=DEV)
        expert_ids = torch.zeros(PM // block_m, dtype=torch.int32, device=DEV)
        p = t = 0
        for e, c in enumerate(counts):
            if c == 0:
                continue
            nt = -(-c // block_m)
            for i in range(c):
                sorted_ids[p + i] = t % T
                t += 7
            expert_ids[p // block_m: p // block_m + nt] = e
            p += nt * block_m
        n_valid = torch.tensor([n_tiles], dtype=torch.int32, device=DEV)
        a = (torch.randn(max(T, PM), K) * 0.3).to(torch.float8_e4m3fn).cuda()
        a_s = torch.rand(max(T, PM), dtype=torch.float32, device=DEV) + 0.1
        out = torch.zeros(PM, N, dtype=torch.bfloat16, device=DEV)
        ops.moe_gemm_fp8(out, a, a_s, b_packed, ws, sorted_ids, expert_ids,
                         n_valid, block_m, gate_up)
        want = torch.zeros(PM, N, dtype=torch.bfloat16)
        from fusioninfer_amd.ops import reference as _r

        _r.moe_gemm_fp8(want, a.cpu(), a_s.cpu(), b_packed.cpu(), ws.cpu(),
                        sorted_ids.cpu(), expert_ids.cpu(), n_valid.cpu(),
                        block_m, gate_up)
        rows = n_tiles * block_m
        torch.testing.assert_close(out[:rows].float().cpu(),
                                   want[:rows].float(),
                                   atol=5e-2, rtol=5e-2)


def test_moe_align_kernel_matches_python():
    """The fused alignment kernel vs the torch composition (the CPU/
    semantic oracle, which also runs on GPU tensors): tile counts and
    expert_ids must be EQUAL; slot assignments may permute within an
    expert's segment (arrival vs stable order) but must satisfy the
    same invariants."""
    import types

    from fusioninfer_amd.models.model import MoEMLP

    torch.manual_seed(5)
    cases = [
        (13, 2, 8, 0, 8, 16),     # small, all local
        (300, 8, 16, 4, 12, 16),  # EP slice: half the experts non-local
        (256, 8, 8, 0, 8, 128),   # prefill block_m
        (1, 8, 128, 0, 128, 16),  # decode single token, many experts
        (512, 8, 128, 0, 128, 16),   # the most of the one-workgroup form
        (4097, 1, 3, 0, 3, 128),     # one more: two launches, odd shares
        (3000, 8, 128, 32, 96, 128),
        (1100, 4, 1000, 0, 1000, 16),
    ]
    for T, k, E, e0, e1, bm in cases:
        topi = torch.randint(0, E, (T, k), device=DEV)
        fake = types.SimpleNamespace(e_start=e0, e_end=e1)
        p_sid, p_eid, p_nv, p_pos, p_PM = MoEMLP._moe_align(fake, topi, bm)
        sid, eid, nv, pos, PM = ops.moe_align(topi, e0, e1, bm)
        assert PM == p_PM
        assert int(nv.item()) == int(p_nv.item())
        assert torch.equal(eid, p_eid)
        flat = topi.reshape(-1).cpu()
        pos_c, sid_c = pos.cpu(), sid.cpu()
        local = [(int(e) >= e0) and (int(e) < e1) for e in flat]
        seen = set()
        for i, e in enumerate(flat.tolist()):
            p = int(pos_c[i])
            if not local[i]:
                assert p == -1
                continue
            assert 0 <= p < PM and p not in seen
            seen.add(p)
            assert int(sid_c[p]) == i // k          # row gather correct
            assert int(eid[p // bm]) == e - e0      # right expert tile
        # padding rows are zeroed (the GEMM's dummy-row contract)
        pad = [i for i in range(PM) if i not in seen]
        assert all(int(sid_c[i]) == 0 for i in pad)


def test_moe_router_topk_matches_torch():
    """Fused router tail vs the torch composition: same experts, same
    weights, same (descending) order. Random fp32 logits are distinct
    almost surely, so exact order comparison is stable."""
    torch.manual_seed(9)
    for T, E, k, renorm in [(7, 8, 2, True), (256, 128, 8, True),
                            (33, 64, 4, False), (1, 128, 8, True)]:
        logits = torch.randn(T, E, device=DEV, dtype=torch.float32)
        tv, ti = ops.moe_router_topk(logits, k, renorm)
        probs = torch.softmax(logits, -1)
        etv, eti = probs.topk(k, -1)
        if renorm:
            etv = etv / etv.sum(-1, keepdim=True)
        assert torch.equal(ti.long(), eti), (T, E, k)
        torch.testing.assert_close(tv, etv, atol=2e-6, rtol=2e-6)


@pytest.mark.parametrize("T,E,K,k,renorm", [
    (1, 128, 2048, 8, True),
    (17, 16, 32, 16, False),    # one step: three waves hold nothing
    (64, 48, 288, 3, True),     # odd share of K, part of a batch of loads
    (512, 128, 2048, 128, True),  # every expert chosen
    (513, 112, 1024, 8, False),   # the library's product
    (5, 40, 256, 2, True),
])
def test_moe_router(T, E, K, k, renorm):
    """Router against a float64 product: the same experts
    where their gap exceeds what fp32 sums of K products can move, weights
    to that accuracy."""
    g = torch.Generator().manual_seed(T + E)
    x = torch.randn(T, K, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(E, K, generator=g) * 0.05).to(torch.bfloat16).to(DEV)
    tv, ti = ops.moe_router(x, w, k, renorm)
    logits = x.double() @ w.double().T
    probs = torch.softmax(logits, -1)
    ev, ei = probs.topk(k, -1)
    gap = -torch.diff(logits.sort(-1, descending=True).values[:, :k + 1])
    sure = (gap > 1e-4).all(-1) if gap.numel() else torch.ones(T, dtype=bool)
    assert torch.equal(ti.long()[sure], ei[sure])
    if renorm:
        ev = ev / ev.sum(-1, keepdim=True)
    torch.testing.assert_close(tv.double(), ev, atol=1e-5, rtol=1e-4)


def test_moe_router_topk_ties():
    """Equal logits: the smaller index first; every expert once."""
    for E, k in [(128, 8), (128, 128), (70, 70), (5, 5)]:
        logits = torch.zeros(3, E, device=DEV)
        logits[1, E // 2:] = 1.0
        logits[2, ::2] = -float("inf")
        tv, ti = ops.moe_router_topk(logits, k, False)
        half = [*range(E // 2, E), *range(E // 2)]
        odd = [*range(1, E, 2), *range(0, E, 2)]
        assert ti[0].tolist() == list(range(k))
        assert ti[1].tolist() == half[:k]
        assert ti[2].tolist() == odd[:k]
        torch.testing.assert_close(tv[0], torch.full_like(tv[0], 1 / E))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,top,H", [(3, 1, 8), (7, 9, 2056), (5, 8, 4096),
                                     (4, 2, 30)])
def test_moe_combine_widths(T, top, H, dtype):
    """Whole vectors and ragged widths, more experts than one batch of
    loads, absent rows (whose memory may hold anything)."""
    g = torch.Generator().manual_seed(H)
    y = torch.randn(T * top + 1, H, generator=g).to(dtype).to(DEV)
    y[T * top] = float("nan")
    pos = torch.randperm(T * top, generator=g).int()
    pos[1::3] = -1
    w = torch.rand(T * top, generator=g)
    out = torch.empty(T, H, dtype=dtype, device=DEV)
    ops.moe_combine(out, y, pos.to(DEV), w.to(DEV))
    rows = y.double()[pos.clamp(min=0).long().to(DEV)]
    rows[(pos < 0).to(DEV)] = 0.0
    want = (rows * w.double().to(DEV)[:, None]).view(T, top, H).sum(1)
    # half a unit of the result's type, and fp32 sums
    half = 2 ** -8 if dtype == torch.bfloat16 else 0.0
    err = (out.double() - want).abs()
    assert (err <= want.abs() * half + 1e-5).all()


@pytest.mark.parametrize("T,top,H", [(1, 1, 8), (3, 8, 2048), (64, 9, 2056),
                                     (5, 4, 4096), (5, 4, 4104), (2, 16, 8192),
                                     (300, 8, 264), (4, 2, 8200)])
def test_moe_combine_norm(T, top, H):
    """The combined rows, the residual and the norm behind: fp32 sums of top
    products and one rounding to bf16 each (2^-9 relative)."""
    g = torch.Generator().manual_seed(T + top + H)
    y = torch.randn(T * top + 5, H, generator=g).to(torch.bfloat16)
    pos = torch.randperm(T * top + 5, generator=g)[: T * top].int()
    pos[::7] = -1
    w = torch.rand(T * top, generator=g)
    old = torch.randn(T, H, generator=g).to(torch.bfloat16)
    norm = torch.randn(H, generator=g).to(torch.bfloat16)
    rows = y.double()[pos.clamp(min=0).long()] * (pos >= 0).double()[:, None]
    combined = (rows * w.double()[:, None]).view(T, top, H).sum(1)
    want = combined + old.double()
    out, res = ops.moe_combine_norm(y.to(DEV), pos.to(DEV), w.to(DEV),
                                    old.to(DEV), norm.to(DEV), 1e-6)
    # wider rows go through two kernels: the combined ones are rounded
    # between, by 2^-9 of themselves, which the sum with the residual keeps
    err = (top + 1) * 2 ** -21 + (0 if H <= 8192
                                  else combined.abs() * 2 ** -9)
    assert ((res.cpu().double() - want).abs()
            <= want.abs() * 2 ** -8 + 2 * err).all()
    inv = (want.square().mean(1, keepdim=True) + 1e-6).rsqrt()
    want = want * inv * norm.double()
    assert ((out.cpu().double() - want).abs()
            <= want.abs() * 2 ** -8 + 2 * err * inv * norm.double().abs()
            ).all()


def test_moe_combine_norm_of_no_rows():
    """No expert has a row for any token: the residual alone, and its norm."""
    g = torch.Generator().manual_seed(5)
    old = torch.randn(3, 64, generator=g).bfloat16().to(DEV)
    norm = torch.randn(64, generator=g).bfloat16().to(DEV)
    out, res = ops.moe_combine_norm(
        old[:0], torch.full((3, 2), -1, dtype=torch.int32, device=DEV),
        torch.ones(6, device=DEV), old.clone(), norm, 1e-6)
    assert torch.equal(res, old)
    assert torch.equal(out, ops.rms_norm(old, norm, 1e-6))


def test_moe_combine_past_the_caches():
    """More rows than the memory-side cache holds give the bits of the same
    tokens in shorter calls; what rows that nobody has hold does not matter."""
    T, top, H = 8200, 8, 2048
    y = torch.randn(T * top, H, device=DEV, dtype=torch.bfloat16)
    y[0] = float("nan")
    pos = torch.randperm(T * top, device=DEV).int()
    pos[pos == 0] = -1
    pos[::11] = -1
    w = torch.rand(T * top, device=DEV)
    old, norm = (torch.randn(n, H, device=DEV, dtype=torch.bfloat16)
                 for n in (T, 1))
    out, res = ops.moe_combine_norm(y, pos, w, old.clone(), norm[0], 1e-6)
    plain = ops.moe_combine(torch.empty_like(old), y, pos, w)
    assert out.isfinite().all() and plain.isfinite().all()
    for a in (0, 4000, T - 7):
        b = min(a + 500, T)
        cut = slice(a * top, b * top)
        o, r = ops.moe_combine_norm(y, pos[cut], w[cut], old[a:b].clone(),
                                    norm[0], 1e-6)
        assert torch.equal(o, out[a:b]) and torch.equal(r, res[a:b])
        assert torch.equal(ops.moe_combine(torch.empty_like(o), y, pos[cut],
                                           w[cut]), plain[a:b])




# ------------------------------------------------------------ skinny GEMM


@pytest.mark.parametrize("rows", [1, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("n,k,bias", [
    (16, 128, False),      # one tile, one stage: most waves hold nothing
    (48, 384, True),       # fewer stages than waves
    (4112, 1024, True),    # more tiles than workgroups, 16 rows each
    (6144, 640, False),    # 32-row tiles, uneven split of K
    (16448, 2048, True),   # 32-row tiles in several rounds
])
def test_skinny_linear(rows, n, k, bias):
    """Few rows against a float64 product; one bf16 rounding of the result
    (2^-9 relative) and fp32 sums of k products."""
    g = torch.Generator().manual_seed(n + k + rows)
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    b = torch.randn(n, generator=g).to(torch.bfloat16).to(DEV) if bias \
        else None
    # rows of a wider tensor, as a split projection hands out
    x = torch.randn(rows, 2 * k, generator=g).to(torch.bfloat16).to(DEV)[:, k:]
    assert ops._skinny_ok(x, w, 16)
    out = ops.linear(x, w, b)
    want = x.double() @ w.double().T + (0.0 if b is None else b.double())
    err = (out.double() - want).abs()
    assert (err <= want.abs() * 2 ** -8 + 1e-4 * k ** 0.5).all()
    if n % 32 == 0 and not bias:
        out = ops.linear_silu_mul(x, w)
        prod = x.double() @ w.double().T
        want = torch.nn.functional.silu(prod[:, : n // 2]) * prod[:, n // 2:]
        err = (out.double() - want).abs()
        assert (err <= want.abs() * 2 ** -8 + 1e-3 * k ** 0.5).all()


@pytest.mark.parametrize("rows", [17, 32, 33, 64, 65, 128, 129, 256])
@pytest.mark.parametrize("n,k,bias", [
    (16, 128, True),        # one ragged tile, one or two stages
    (224, 384, False),      # fewer stages than workgroups; odd tiles
    (4128, 2560, True),     # cut tiles, a ragged last one, several pieces
    (288, 16384, False),    # a tile in many pieces
    (24608, 256, False),    # whole tiles and one more
])
def test_linear_in_parts(rows, n, k, bias):
    """17 to 256 rows against a float64 product; one bf16 rounding of the
    result (2^-9 relative) and fp32 sums of k products."""
    g = torch.Generator().manual_seed(n + k + rows)
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    b = torch.randn(n, generator=g).to(torch.bfloat16).to(DEV) if bias \
        else None
    x = torch.randn(rows, 2 * k, generator=g).to(torch.bfloat16).to(DEV)[:, k:]
    out = torch.empty(rows, n, dtype=torch.bfloat16, device=DEV)
    ops._C.few_rows_gemm(out, x, w, b, False)
    prod = x.double() @ w.double().T
    want = prod + (0.0 if b is None else b.double())
    assert ((out.double() - want).abs()
            <= want.abs() * 2 ** -8 + 1e-4 * k ** 0.5).all()
    if n % 32 == 0 and not bias:
        out = torch.empty(rows, n // 2, dtype=torch.bfloat16, device=DEV)
        ops._C.few_rows_gemm(out, x, w, None, True)
        want = torch.nn.functional.silu(prod[:, : n // 2]) * prod[:, n // 2:]
        assert ((out.double() - want).abs()
                <= want.abs() * 2 ** -8 + 1e-3 * k ** 0.5).all()


@pytest.mark.parametrize("rows", [31, 64, 100, 128, 192, 193, 255])
@pytest.mark.parametrize("n,k,bias", [
    (65552, 128, True),     # results on their way behind stages of next tiles
    (65568, 256, False),
    (24624, 384, False),    # a tile of 96 rows for every workgroup, and a rest
    (12320, 1024, False),   # fewer whole tiles than workgroups
])
def test_linear_in_parts_of_several_tiles(rows, n, k, bias):
    """Parts that hold several tiles, whole or cut, against a float64 product;
    one bf16 rounding of the result (2^-9 relative) and fp32 sums of k
    products. What lies behind the last row of either operand has no part in
    the result, and rows that are not of the result stay as they were."""
    g = torch.Generator().manual_seed(n + k + rows)
    w, x = (torch.full((m + 256, k), float("nan"), dtype=torch.bfloat16,
                       device=DEV) for m in (n, rows))
    w[:n] = torch.randn(n, k, generator=g)
    x[:rows] = torch.randn(rows, k, generator=g)
    w, x = w[:n], x[:rows]
    b = torch.randn(n, generator=g).to(torch.bfloat16).to(DEV) if bias \
        else None
    prod = x.double() @ w.double().T
    out = torch.full((rows + 1, n), 7.0, dtype=torch.bfloat16, device=DEV)
    ops._C.few_rows_gemm(out[:rows], x, w, b, False)
    want = prod + (0.0 if b is None else b.double())
    assert ((out[:rows].double() - want).abs()
            <= want.abs() * 2 ** -8 + 1e-4 * k ** 0.5).all()
    assert (out[rows] == 7.0).all()
    if n % 32 == 0 and not bias:
        out = torch.full((rows + 1, n // 2), 7.0, dtype=torch.bfloat16,
                         device=DEV)
        ops._C.few_rows_gemm(out[:rows], x, w, None, True)
        want = torch.nn.functional.silu(prod[:, : n // 2]) * prod[:, n // 2:]
        assert ((out[:rows].double() - want).abs()
                <= want.abs() * 2 ** -8 + 1e-3 * k ** 0.5).all()
        assert (out[rows] == 7.0).all()


@pytest.mark.parametrize("rows", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("n,k,bias", [
    (16, 128, False), (16, 1152, True), (2032, 256, True), (2048, 6144, False),
    (2064, 384, True),      # the first that goes by tiles of 16 rows again
])
def test_linear_by_tiles_of_eight_rows(rows, n, k, bias):
    """Against float64: fp32 sums of k products, one bf16 rounding (2^-9
    relative). What lies behind the last row of either operand has no part."""
    g = torch.Generator().manual_seed(n + k + rows)
    w, x = (torch.full((m + 32, k), float("nan"), dtype=torch.bfloat16,
                       device=DEV) for m in (n, rows))
    w[:n] = torch.randn(n, k, generator=g)
    x[:rows] = torch.randn(rows, k, generator=g)
    w, x = w[:n], x[:rows]
    b = torch.randn(n, generator=g).to(torch.bfloat16).to(DEV) if bias \
        else None
    out = torch.full((rows + 1, n), 7.0, dtype=torch.bfloat16, device=DEV)
    ops._C.few_rows_gemm(out[:rows], x, w, b, False)
    want = x.double() @ w.double().T + (0.0 if b is None else b.double())
    assert ((out[:rows].double() - want).abs()
            <= want.abs() * 2 ** -8 + 1e-4 * k ** 0.5).all()
    assert (out[rows] == 7.0).all()


@pytest.mark.parametrize("rows", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("n,k,parts,bias", [
    (16, 128, 1, True),        # one tile; most waves without a stage
    (2576, 1152, 127, False),  # tiles of 16 rows, parts short of a round
    (6176, 384, 129, True),    # of 32, and one over
    (24640, 512, 32, False),   # several tiles for some workgroups
    (12320, 2048, 300, False),
])
def test_linear_of_stream_rows(rows, n, k, parts, bias):
    """Rows divided by the root mean square that parts add up to, against
    float64; the result is rounded to bf16 once (2^-9 relative) and the sums
    of k products are fp32. What the parts hold for rows beyond x, and what
    lies behind any operand's last row, has no part in the result."""
    g = torch.Generator().manual_seed(n + k + rows)
    w, x = (torch.full((m + 32, k), float("nan"), dtype=torch.bfloat16,
                       device=DEV) for m in (n, rows))
    w[:n] = torch.randn(n, k, generator=g)
    x[:rows] = torch.randn(rows, k, generator=g)
    w, x = w[:n], x[:rows]
    sq = torch.full((parts + 16, 16), float("nan"), device=DEV)
    sq[:parts, :rows] = torch.rand(parts, rows, generator=g).to(DEV) * k / parts
    sq = sq[:parts]
    b = torch.randn(n, generator=g).to(torch.bfloat16).to(DEV) if bias \
        else None
    inv = (sq[:, :rows].double().sum(0) / k + 0.5).rsqrt()[:, None]
    prod = x.double() @ w.double().T * inv
    out = torch.full((rows + 1, n), 7.0, dtype=torch.bfloat16, device=DEV)
    ops._C.few_rows_scaled_gemm(out[:rows], x, sq, 0.5, w, b, False)
    want = prod + (0.0 if b is None else b.double())
    assert ((out[:rows].double() - want).abs()
            <= want.abs() * 2 ** -8 + 1e-4 * k ** 0.5).all()
    assert (out[rows] == 7.0).all()
    if n % 32 == 0 and not bias:
        out = torch.full((rows + 1, n // 2), 7.0, dtype=torch.bfloat16,
                         device=DEV)
        ops._C.few_rows_scaled_gemm(out[:rows], x, sq, 0.5, w, None, True)
        want = torch.nn.functional.silu(prod[:, : n // 2]) * prod[:, n // 2:]
        assert ((out[:rows].double() - want).abs()
                <= want.abs() * 2 ** -8 + 1e-3 * k ** 0.5).all()
        assert (out[rows] == 7.0).all()


@pytest.mark.parametrize("rows", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("n,k", [(128, 128), (2560, 1152), (4224, 256),
                                 (6272, 384), (16384, 128)])
def test_stream_add(rows, n, k):
    """The sums keep fp32: off by the sums of k products alone; the rows for
    the norm are theirs, bit by bit, and the squares add up in any order (n
    roundings at most). Its norm, in one pass, has one rounding to bf16."""
    g = torch.Generator().manual_seed(n + k + rows)
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16).to(DEV)
    norm = torch.randn(n, generator=g).to(torch.bfloat16).to(DEV)
    begun = torch.randn(rows, n, generator=g).to(torch.bfloat16).to(DEV)
    first = ops.stream_begin(begun, norm, 1e-6)
    stream = first.stream
    for r in (first, ops.stream_begin(stream, norm, 1e-6)):
        assert torch.equal(r.stream, begun.float())
        assert torch.equal(r.scaled, begun * norm)
        torch.testing.assert_close(
            r.squares.sum(0)[:rows].double(),
            begun.double().square().sum(1), rtol=n * 2.0 ** -24, atol=0)
    want = stream.double() + x.double() @ w.double().T
    without = stream.clone()
    assert ops.stream_add_(without, x, w) is None
    r = ops.stream_add_(stream, x, w, norm, 1e-6)
    assert r.stream is stream and torch.equal(stream, without)
    assert ((stream.double() - want).abs()
            <= want.abs() * 2 ** -23 + 1e-4 * k ** 0.5).all()
    assert torch.equal(r.scaled, (stream * norm.float()).to(torch.bfloat16))
    assert r.squares.shape == (n // 16, 16)
    torch.testing.assert_close(
        r.squares.sum(0)[:rows].double(), stream.double().square().sum(1),
        rtol=n * 2.0 ** -24, atol=0)
    want = (stream.double() * norm.double()
            * (stream.double().square().mean(1, keepdim=True) + 1e-6).rsqrt())
    assert ((ops.stream_norm(stream, norm, 1e-6).double() - want).abs()
            <= want.abs() * 2 ** -8).all()


@pytest.mark.parametrize("offset", [1, 2, 4, 7])
def test_stream_norms_weight_on_any_grid(offset):
    """A norm's weight may begin anywhere, as in rms_norm: the bits are those
    of a weight on the 16-byte grid."""
    g = torch.Generator().manual_seed(offset)
    n, k, rows = 2576, 256, 5
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16).to(DEV)
    begun = torch.randn(rows, n, generator=g).to(torch.bfloat16).to(DEV)
    flat = torch.randn(n + 8, generator=g).to(torch.bfloat16).to(DEV)
    norm = flat[offset:offset + n]

    def run(weight):
        first = ops.stream_begin(begun, weight, 1e-6)
        got = [first.scaled.clone(), first.squares[:, :rows].clone()]
        then = ops.stream_add_(first.stream, x, w, weight, 1e-6)
        return [*got, then.scaled, then.squares[:, :rows], then.stream,
                ops.stream_norm(then.stream, weight, 1e-6)]

    assert norm.data_ptr() % 16 != 0
    for a, b in zip(run(norm), run(norm.clone())):
        assert torch.equal(a, b)
    assert torch.equal(ops.rms_norm(begun, norm, 1e-6),
                       ops.rms_norm(begun, norm.clone(), 1e-6))


@pytest.mark.parametrize("fp8,rows", [
    (fp8, rows) for rows in (1, 16, 17, 32, 33, 64, 65, 128, 129, 192, 193,
                             256) for fp8 in (False, True)
    if rows <= 128 or not fp8])
@pytest.mark.parametrize("n,k,cut,cut_fp8", [
    (4096, 4096, 17, 1),
    (2064, 4608, 17, 1),      # a tile that is not full
    (1040, 512, 17, 1),       # few parts, fewer stages in each
    (5136, 5120, 17, 1),      # two turns of a workgroup along a row
    (8208, 8192, 17, 1), (12304, 12288, 17, 1),   # four
    (16384, 16384, 33, 33),   # the longest row
    (16400, 16384, 257, 129),  # longer than the kernel takes, if cut
    (8208, 1024, 257, 129),   # whole tiles
])
def test_linear_in_parts_and_norm(rows, n, k, cut, cut_fp8, fp8):
    """The sum of a residual and a product in parts, and its norm, against
    float64: fp32 sums of k products; the sum and the normed row are rounded to
    bf16 once (2^-9 relative), or the row to e4m3 (2^-4, 2^-10 of the scale
    where it is smallest). Nothing is written behind the last row, nor anything
    at all where another way is taken: of fewer rows than those from which on
    the product is cut and summed so."""
    g = torch.Generator(device=DEV).manual_seed(n + k + rows)

    def randn(*shape):
        return torch.randn(*shape, generator=g, device=DEV)

    x = randn(rows, k).to(torch.bfloat16)
    w = randn(n, k).to(torch.bfloat16)
    norm = randn(n).to(torch.bfloat16)
    old = (randn(rows + 1, n) * k ** 0.5).to(torch.bfloat16)
    residual = old.clone()
    if fp8:
        x, xs = ops.quant_fp8_rows(x)
        w, ws = w.to(torch.float8_e4m3fn), torch.rand(n, generator=g,
                                                      device=DEV)
        prod = (x.double() * xs.double()[:, None]) @ (
            w.double() * ws.double()[:, None]).T
        out = torch.ones(rows + 1, n, device=DEV).to(x.dtype)
        scales = torch.full((rows + 1,), 7.0, device=DEV)
        done = ops._C.few_rows_gemm_norm_fp8(
            out[:rows], scales[:rows], x, xs, w, ws, residual[:rows], norm,
            1e-6)
        got = out[:rows].double() * scales[:rows].double()[:, None]
        assert scales[rows] == 7.0 and (out[rows].float() == 1.0).all()
    else:
        prod = x.double() @ w.double().T
        out = torch.full((rows + 1, n), 7.0, dtype=torch.bfloat16, device=DEV)
        done = ops._C.few_rows_gemm_norm(out[:rows], x, w, residual[:rows],
                                         norm, 1e-6)
        got = out[:rows].double()
        assert (out[rows] == 7.0).all()
    assert done == (rows >= (cut_fp8 if fp8 else cut))
    if not done:
        assert torch.equal(residual, old)
        return
    assert torch.equal(residual[rows], old[rows])
    want = prod + old[:rows].double()
    err = 1e-4 * k ** 0.5
    assert ((residual[:rows].double() - want).abs()
            <= want.abs() * 2 ** -8 + err).all()
    inv = (want.square().mean(1, keepdim=True) + 1e-6).rsqrt()
    want = want * inv * norm.double()
    err = err * inv * norm.double().abs()
    if fp8:
        bound = want.abs() * (2 ** -4 + 2 ** -8) + err + (
            scales[:rows].double()[:, None] * 2 ** -10)
    else:
        bound = want.abs() * 2 ** -8 + err
    assert ((got - want).abs() <= bound).all()


@pytest.mark.parametrize("rows,n,k", [
    (1, 6144, 2048), (4, 16, 128), (5, 2064, 384), (8, 6176, 384),
    (9, 24640, 256), (16, 1040, 1152),
    (257, 528, 256),       # a tile and a row, the last columns of a tile
    (300, 4096, 2048),     # tiles in pieces
    (2304, 8192, 320),     # whole rounds and a rest
])
def test_linear_gelu(rows, n, k):
    """The tanh form of gelu of a product against float64: its slope is below
    1.13, the product's sums are fp32, the result has one rounding to bf16."""
    g = torch.Generator().manual_seed(n + k + rows)
    w, x = (torch.full((m + 256, k), float("nan"), dtype=torch.bfloat16,
                       device=DEV) for m in (n, rows))
    w[:n] = torch.randn(n, k, generator=g) * k ** -0.5 * 3
    x[:rows] = torch.randn(rows, k, generator=g)
    w, x = w[:n], x[:rows]
    out = torch.full((rows + 1, n), 7.0, dtype=torch.bfloat16, device=DEV)
    kernel = ops._C.few_rows_gemm if rows <= 16 else ops._C.many_rows_gemm
    kernel(out[:rows], x, w, None, False, True)
    want = torch.nn.functional.gelu(x.double() @ w.double().T,
                                    approximate="tanh")
    assert ((out[:rows].double() - want).abs()
            <= want.abs() * 2 ** -8 + 1e-4).all()
    assert (out[rows] == 7.0).all()
    taken = ops.linear_gelu(x, w)
    assert taken is None or torch.equal(taken, out[:rows])
    assert taken is not None or rows > 16


@pytest.mark.parametrize("rows", [16, 17, 43, 64, 65, 129, 193, 256])
@pytest.mark.parametrize("hq,hk,d,k,bias,norm,fp8,cut", [
    (32, 8, 128, 4096, False, True, False, True),
    (32, 4, 128, 2048, True, False, True, True),
    (14, 2, 64, 3584, True, True, False, True),
    (9, 1, 64, 512, False, False, True, True),     # heads that fill no wave
    (70, 5, 128, 8192, False, True, False, True),  # two workgroups a token
    (70, 5, 128, 8192, True, True, True, True),
    (70, 5, 128, 1024, False, True, False, False),   # whole tiles
])
def test_linear_in_parts_to_heads(rows, hq, hk, d, k, bias, norm, fp8, cut):
    """Queries, keys and values of a product in parts, normed, rotated and in
    the cache, against float64: fp32 sums of k products, which the norm scales,
    each result rounded to bf16 once (2^-9 relative), to e4m3 once more (2^-4,
    2^-10 where it is smallest). Rows without a slot are not kept. Of up to 16
    rows, or where the product is not cut, nothing is done."""
    g = torch.Generator().manual_seed(rows + hq + d + k)
    n, bs = (hq + 2 * hk) * d, 16
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(n, k, device=DEV, generator=torch.Generator(
        device=DEV).manual_seed(k)) * k ** -0.5).to(torch.bfloat16)
    b = torch.randn(n, generator=g).to(torch.bfloat16).to(DEV) if bias \
        else None
    qw, kw = (torch.rand(2, d, generator=g) + 0.5).to(torch.bfloat16).to(DEV) \
        if norm else (None, None)
    pos = torch.randint(0, 500, (rows,), generator=g).int().to(DEV)
    cs = ops.compute_cos_sin_cache(d, 512, 1e4).to(DEV)
    blocks = rows // bs + 3
    slots = torch.randperm(blocks * bs, generator=g)[:rows].int()
    slots[::9] = -1
    kc, vc = (torch.zeros(blocks, hk, bs, d, device=DEV).to(
        torch.float8_e4m3fn if fp8 else torch.bfloat16) for _ in range(2))
    q = torch.full((rows + 1, hq * d), 7.0, dtype=torch.bfloat16, device=DEV)
    done = ops._C.few_rows_gemm_rope(
        q[:rows], x, w, b, qw, kw, cs, pos, kc, vc, slots.to(DEV), hq, 1e-6,
        0.5, 2.0)
    assert (q[rows] == 7.0).all()
    assert done == (cut and rows > 16)
    if not done:
        assert not kc.float().any() and not vc.float().any()
        assert (q == 7.0).all()
        return
    heads = x.double() @ w.double().T + (0.0 if b is None else b.double())
    heads = heads.view(rows, hq + 2 * hk, d)
    err = torch.full_like(heads, 1e-5)
    if norm:
        inv = (heads.square().mean(-1, keepdim=True) + 1e-6).rsqrt()
        wt = torch.cat([qw.expand(hq, d), kw.expand(hk, d),
                        torch.ones_like(kw).expand(hk, d)]).double()
        inv[:, hq + hk:] = 1.0
        heads, err = heads * inv * wt, 4 * err * inv * wt
    c, s = (t.double()[:, None] for t in cs[pos.long()].chunk(2, dim=-1))
    x1, x2 = heads.chunk(2, dim=-1)
    turned = torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], -1)
    err = 2 * err.amax(-1, keepdim=True).expand_as(err)
    got, want = q[:rows].view(rows, hq, d).double(), turned[:, :hq]
    assert ((got - want).abs() <= want.abs() * 2 ** -8 + err[:, :hq]).all()
    kept = (slots >= 0).nonzero()[:, 0].to(DEV)
    at = slots.to(DEV)[kept].long()
    for cache, want, e, scale in (
            (kc, turned[:, hq:hq + hk], err[:, hq:hq + hk], 0.5),
            (vc, heads[:, hq + hk:], err[:, hq + hk:], 2.0)):
        got = cache[at // bs, :, at % bs].double()
        want, e = want[kept], e[kept]
        bound = want.abs() * 2 ** -8 + e
        if fp8:
            want, bound = want * scale, bound * scale
            bound = bound + want.abs() * 2 ** -4 + 2.0 ** -10
        assert ((got - want).abs() <= bound).all()
        rest = torch.ones(blocks * bs, dtype=torch.bool, device=DEV)
        rest[at] = False
        rest = rest.nonzero()[:, 0]
        assert not cache[rest // bs, :, rest % bs].float().any()


@pytest.mark.parametrize("rows", [128, 129])
def test_linear_in_parts_of_long_rows(rows):
    """Rows of W too long for 32-bit offsets within a tile (x one row, given
    that often). x is scaled so that the products are of size one: a bf16
    rounding of the result and fp32 sums (2^17 additions in a lane's turn,
    2^-24 of their size each, errors of either sign)."""
    g = torch.Generator(device=DEV).manual_seed(rows)
    n, k = 16, (1 << 22) + 128
    w = torch.randn(n, k, generator=g, device=DEV).to(torch.bfloat16)
    x = (torch.randn(1, k, generator=g, device=DEV) / 2048).to(
        torch.bfloat16).expand(rows, k)
    out = torch.empty(rows, n, dtype=torch.bfloat16, device=DEV)
    ops._C.few_rows_gemm(out, x, w, None, False)
    want = x[:1].double() @ w.double().T
    assert ((out.double() - want).abs()
            <= want.abs() * 2 ** -8 + 1e-4).all()


@pytest.mark.parametrize("rows", [1, 255, 257, 1029])
@pytest.mark.parametrize("n,k,bias", [
    (16, 128, True),        # one ragged tile, two stages, whole
    (288, 192, False),      # three stages: not to be cut
    (4128, 1024, True),     # cut tiles, a ragged last one
    (288, 16384, False),    # 16 pieces, every other tile begins half way
    (65568, 128, False),    # whole rounds of tiles and a rest
    (65568, 128, True),
    (33056, 1024, False),   # whole rounds, the rest cut (257, 1029 rows)
    (33056, 1024, True),
])
def test_linear_by_tiles(rows, n, k, bias):
    """Tiles of 256 x 256 against a float64 product; one bf16 rounding of the
    result (2^-9 relative) and fp32 sums of k products. Rows that are not of
    the result stay as they were."""
    g = torch.Generator().manual_seed(n + k + rows)
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    b = torch.randn(n, generator=g).to(torch.bfloat16).to(DEV) if bias \
        else None
    x = torch.randn(rows, 2 * k, generator=g).to(torch.bfloat16).to(DEV)[:, k:]
    out = torch.full((rows + 1, n), 7.0, dtype=torch.bfloat16, device=DEV)
    ops._C.many_rows_gemm(out[:rows], x, w, b, False)
    prod = x.double() @ w.double().T
    want = prod + (0.0 if b is None else b.double())
    assert ((out[:rows].double() - want).abs()
            <= want.abs() * 2 ** -8 + 1e-4 * k ** 0.5).all()
    assert (out[rows] == 7.0).all()
    if n % 32 == 0 and not bias:
        out = torch.full((rows + 1, n // 2), 7.0, dtype=torch.bfloat16,
                         device=DEV)
        ops._C.many_rows_gemm(out[:rows], x, w, None, True)
        want = torch.nn.functional.silu(prod[:, : n // 2]) * prod[:, n // 2:]
        assert ((out[:rows].double() - want).abs()
                <= want.abs() * 2 ** -8 + 1e-3 * k ** 0.5).all()
        assert (out[rows] == 7.0).all()


@pytest.mark.parametrize("rows,n,k", [
    (257, 144, 128),      # one row and 16 columns over; two stages
    (264, 16, 1024),      # eight rows over, half a tile of W without a row
    (513, 272, 4096),     # cut tiles, one row and 16 columns over
])
def test_linear_by_tiles_reads_its_operands_alone(rows, n, k):
    """What lies behind the last row of either operand has no part in the
    result."""
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, k, generator=g).bfloat16().to(DEV)
    w = torch.randn(n, k, generator=g).bfloat16().to(DEV)
    xn, wn = (torch.full((512 + t.shape[0], k), float("nan"),
                         dtype=torch.bfloat16, device=DEV) for t in (x, w))
    xn[:rows], wn[:n] = x, w
    out, same = (torch.empty(rows, n, dtype=torch.bfloat16, device=DEV)
                 for _ in range(2))
    ops._C.many_rows_gemm(out, x, w, None, False)
    ops._C.many_rows_gemm(same, xn[:rows], wn[:n], None, False)
    assert torch.equal(out, same)
    want = x.double() @ w.double().T
    assert ((out.double() - want).abs()
            <= want.abs() * 2 ** -8 + 1e-4 * k ** 0.5).all()


@pytest.mark.parametrize("fp8", [False, True])
def test_linear_by_tiles_carries_what_is_not_finite(fp8):
    """An infinity or NaN reaches its row or column as in float64, and no
    other; across a tile's border too."""
    rows, n, k = 300, 528, 512
    g = torch.Generator().manual_seed(k)
    x = torch.randn(rows, k, generator=g)
    w = torch.randn(n, k, generator=g)
    x[7, 3], x[299, 511] = float("nan"), float("nan")
    w[255, 5], w[520, 0] = float("nan"), float("nan")
    if fp8:
        f8 = torch.float8_e4m3fn
        x, w = x.to(f8).to(DEV), w.to(f8).to(DEV)
        xs, ws = torch.ones(rows, device=DEV), torch.ones(n, device=DEV)
        xs[100], ws[300] = float("inf"), float("inf")
        out = torch.empty(rows, n, dtype=torch.bfloat16, device=DEV)
        ops._C.many_rows_gemm_fp8(out, x, xs, w, ws)
        want = (x.double() @ w.double().T) * xs.double()[:, None] * ws.double()
    else:
        x[100, 0], w[300, 7] = float("inf"), float("-inf")
        x, w = x.bfloat16().to(DEV), w.bfloat16().to(DEV)
        out = torch.empty(rows, n, dtype=torch.bfloat16, device=DEV)
        ops._C.many_rows_gemm(out, x, w, None, False)
        want = x.double() @ w.double().T
    assert torch.equal(out.isnan(), want.isnan())
    assert torch.equal(out.isposinf(), want.isposinf())
    assert torch.equal(out.isneginf(), want.isneginf())
    err = (out.double() - want).abs()[want.isfinite()]
    assert (err <= want[want.isfinite()].abs() * 2 ** -8
            + 3e-4 * k ** 0.5).all()


def test_silu_by_tiles_of_far_gates():
    """Gates down to where 1 + exp(-gate) leaves fp32, infinite ones and NaN,
    against float64: exp of fp32 is off by |gate| 2^-23, the result has one
    bf16 rounding. (A product with a zero carries a row's infinity into all
    of its sums, so each kind has a column of x to itself.)"""
    n, k = 512, 128
    gates = torch.linspace(-88.5, 88.5, n // 2 - 4).bfloat16()
    gates = torch.cat([gates, torch.tensor([-1e30, -200.0, 0.0, 1e38])
                       .bfloat16()])
    w = torch.zeros(n, k, dtype=torch.bfloat16)
    w[: n // 2, 0] = gates
    w[n // 2:, 0] = 2.0 ** 100
    w[: n // 2, 1] = w[n // 2:, 2] = 1.0
    x = torch.zeros(300, k, dtype=torch.bfloat16)
    x[:290, 0] = 1.0
    x[290:292, 1], x[292:294, 1] = float("inf"), float("-inf")
    x[294:296, 1] = float("nan")
    x[290:296, 2] = 1.0
    out = torch.empty(300, n // 2, dtype=torch.bfloat16, device=DEV)
    ops._C.many_rows_gemm(out, x.to(DEV), w.to(DEV), None, True)
    got = out.double().cpu()
    g = gates.double()
    want = g / (1 + torch.exp(-g)) * 2.0 ** 100
    err = (got[:290, :-4] - want[:-4]).abs()
    assert (err <= want[:-4].abs() * (2 ** -8 + 89 * 2 ** -23)).all()
    assert (got[:290, -4:-1] == 0).all() and got[:290, -1].isinf().all()
    assert got[290:296].isnan().all()


def test_linear_takes_tiles():
    """Whole rounds with every other tile begun half way and a cut rest, as
    ops.linear chooses it; what it refuses goes to the library."""
    g = torch.Generator().manual_seed(3)
    x = torch.randn(4099, 12288, generator=g).to(torch.bfloat16).to(DEV)
    w = torch.randn(4096, 12288, generator=g).to(torch.bfloat16).to(DEV)
    assert ops._tiles_ok(x, w, 16)
    want = x.double() @ w.double().T
    assert ((ops.linear(x, w).double() - want).abs()
            <= want.abs() * 2 ** -8 + 1e-4 * 12288 ** 0.5).all()
    x, w = x[:, :4096], w[:, :4096].contiguous()
    for other in (x[:, 1:129], x.float(), x[:256]):
        assert not ops._tiles_ok(other, w[:, :other.shape[1]].contiguous(), 16)
    assert ops._tiles_ok(x, w, 16) and not ops._tiles_ok(x, w.T, 16)
    square = x[:4096].contiguous()
    assert ops._tiles_ok(square, w, 16) and not ops._tiles_ok(square.T, w, 16)
    with torch.enable_grad():
        assert not ops._tiles_ok(x, w.clone().requires_grad_(), 16)


@pytest.mark.parametrize("rows", [129, 192, 255, 256, 511])
@pytest.mark.parametrize("n,k,bias", [(49184, 2048, True), (151936, 192, False),
                                      (66560, 1344, False)])
def test_linear_by_one_or_two_rows_of_tiles(rows, n, k, bias):
    """Tiles that begin at 32 places along K, fewer stages than places among
    them, against a float64 product; one bf16 rounding and fp32 sums."""
    g = torch.Generator().manual_seed(n + k + rows)
    w, x = (torch.full((m + 256, k), float("nan"), dtype=torch.bfloat16,
                       device=DEV) for m in (n, rows))
    w[:n] = torch.randn(n, k, generator=g)
    x[:rows] = torch.randn(rows, k, generator=g)
    w, x = w[:n], x[:rows]
    b = torch.randn(n, generator=g).to(torch.bfloat16).to(DEV) if bias \
        else None
    prod = x.double() @ w.double().T
    out = torch.full((rows + 1, n), 7.0, dtype=torch.bfloat16, device=DEV)
    ops._C.many_rows_gemm(out[:rows], x, w, b, False)
    want = prod + (0.0 if b is None else b.double())
    assert ((out[:rows].double() - want).abs()
            <= want.abs() * 2 ** -8 + 1e-4 * k ** 0.5).all()
    assert (out[rows] == 7.0).all()
    if rows <= 256 and k == 2048:
        assert ops._one_row_of_tiles(x, w, b)
        assert torch.equal(ops.linear(x, w, b), out[:rows])
        assert not ops._one_row_of_tiles(x[:128], w, b)
        assert not ops._one_row_of_tiles(x[:1].expand(rows, k), w, b)
        assert not ops._one_row_of_tiles(x, w[:4096], None)
    if n % 32 == 0 and not bias:
        out = torch.full((rows + 1, n // 2), 7.0, dtype=torch.bfloat16,
                         device=DEV)
        ops._C.many_rows_gemm(out[:rows], x, w, None, True)
        want = torch.nn.functional.silu(prod[:, : n // 2]) * prod[:, n // 2:]
        assert ((out[:rows].double() - want).abs()
                <= want.abs() * 2 ** -8 + 1e-3 * k ** 0.5).all()
        assert (out[rows] == 7.0).all()


@pytest.mark.parametrize("rows", [17, 32])
def test_linear_silu_mul_in_parts_of_96_rows(rows):
    """One tile of 96 rows in many pieces, whose kept third of a wave's
    results fills one and a half blocks of the join. x is scaled so that the
    products are of size one: a bf16 rounding of the result (2^-9 relative)
    and fp32 sums (16 and 256 additions of 2^-24 each, a few of that)."""
    g = torch.Generator().manual_seed(rows)
    n, k = 96, 1 << 17
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).to(DEV)
    x = (torch.randn(rows, k, generator=g) / 256).to(torch.bfloat16).to(DEV)
    assert ops._skinny_ok(x, w, 32, True)
    prod = x.double() @ w.double().T
    want = torch.nn.functional.silu(prod[:, : n // 2]) * prod[:, n // 2:]
    err = (ops.linear_silu_mul(x, w).double() - want).abs()
    assert (err <= want.abs() * 2 ** -8 + 1e-4).all()


@pytest.mark.parametrize("rows", [1, 32, 33, 64, 65, 128, 129, 256])
@pytest.mark.parametrize("n,k", [
    (16, 256),           # one ragged tile, one or two stages
    (4128, 2560),        # cut tiles, a ragged last one
    (288, 16384),        # a tile in many pieces
    (24608, 512),        # whole tiles and one more
])
def test_linear_fp8_in_parts(rows, n, k):
    """e4m3 rows with scales against a float64 product; one bf16 rounding of
    the result (2^-9 relative), fp32 sums and two scale products."""
    g = torch.Generator().manual_seed(n + k + rows)
    f8 = torch.float8_e4m3fn
    w = torch.randn(n, k, generator=g).to(f8).to(DEV)
    x = torch.randn(rows, 2 * k, generator=g).to(f8).to(DEV)[:, k:]
    ws = torch.rand(n, generator=g).to(DEV) + 0.5
    xs = torch.rand(rows, generator=g).to(DEV) + 0.5
    out = torch.empty(rows, n, dtype=torch.bfloat16, device=DEV)
    ops._C.few_rows_gemm_fp8(out, x, xs, w, ws)
    want = (x.double() @ w.double().T) * xs.double()[:, None] * ws.double()
    assert ((out.double() - want).abs()
            <= want.abs() * 2 ** -8 + 3e-4 * k ** 0.5).all()


@pytest.mark.parametrize("rows", [1, 31, 255, 257, 1029])
@pytest.mark.parametrize("n,k", [
    (16, 256),           # one ragged tile, two stages, whole
    (288, 384),          # three stages: not to be cut
    (4128, 2048),        # cut tiles, a ragged last one
    (288, 32768),        # 16 pieces, every other tile begins half way
    (65568, 256),        # whole rounds of tiles and a rest
    (33056, 2048),       # whole rounds, the rest cut (257, 1029 rows)
])
def test_linear_fp8_by_tiles(rows, n, k):
    """e4m3 tiles of 256 x 256 against a float64 product: one bf16 rounding of
    the result (2^-9 relative), fp32 sums and two scale products. Rows that
    are not of the result stay as they were."""
    g = torch.Generator().manual_seed(n + k + rows)
    f8 = torch.float8_e4m3fn
    w = torch.randn(n, k, generator=g).to(f8).to(DEV)
    x = torch.randn(rows, 2 * k, generator=g).to(f8).to(DEV)[:, k:]
    ws = torch.rand(n, generator=g).to(DEV) + 0.5
    xs = torch.rand(rows, generator=g).to(DEV) + 0.5
    out = torch.full((rows + 1, n), 7.0, dtype=torch.bfloat16, device=DEV)
    ops._C.many_rows_gemm_fp8(out[:rows], x, xs, w, ws)
    want = (x.double() @ w.double().T) * xs.double()[:, None] * ws.double()
    assert ((out[:rows].double() - want).abs()
            <= want.abs() * 2 ** -8 + 3e-4 * k ** 0.5).all()
    assert (out[rows] == 7.0).all()


def test_linear_fp8_takes_tiles():
    """What the tiles take and what they leave to the library."""
    f8 = torch.float8_e4m3fn
    x = torch.randn(4099, 4096, device=DEV).to(f8)
    w = torch.randn(4096, 4096, device=DEV).to(f8)
    xs = torch.rand(4099, device=DEV) + 0.5
    ws = torch.rand(4097, device=DEV) + 0.5
    assert ops._tiles_fp8_ok(x, xs, w, ws[:4096])
    for refused in ((x[:256], xs[:256], w, ws[:4096]),
                    (x[:1024], xs[:1024], w, ws[:4096]),
                    (x, xs, w, ws[1:]), (x, xs[:, None], w, ws[:4096]),
                    (x[:, 8:4040], xs, w[:, 8:4040], ws[:4096]),
                    (x.cpu(), xs.cpu(), w.cpu(), ws[:4096].cpu())):
        assert not ops._tiles_fp8_ok(*refused)
    want = (x.double() @ w.double().T) * xs.double()[:, None]
    for s in (ws[:4096], ws[1:]):
        err = (ops.linear_fp8(x, xs, w, s).double() - want * s.double()).abs()
        assert (err <= (want * s.double()).abs() * 2 ** -8 + 0.02).all()


def test_linear_fp8_takes_parts_by_size():
    """The sizes that stream and those of the library give the same."""
    f8 = torch.float8_e4m3fn
    for rows, n, k, streams in [(1, 4096, 4096, True), (64, 4096, 4096, False),
                                (64, 2048, 8192, True), (3, 64, 256, False),
                                (200, 4096, 8192, False)]:
        assert ops._streams_fp8(rows, n, k) == streams
        x = torch.randn(rows, k, device=DEV).to(f8)
        w = torch.randn(n, k, device=DEV).to(f8)
        xs = torch.rand(rows, device=DEV) + 0.5
        ws = torch.rand(n, device=DEV) + 0.5
        want = (x.double() @ w.double().T) * xs.double()[:, None] * ws.double()
        err = (ops.linear_fp8(x, xs, w, ws).double() - want).abs()
        assert (err <= want.abs() * 2 ** -8 + 3e-4 * k ** 0.5).all()


def test_linear_takes_parts_by_size():
    """The sizes that stream and those that stay with the library give the
    same product."""
    for rows, n, k, streams in [(48, 4096, 4096, True), (48, 64, 256, False),
                                (48, 8192, 1024, False),
                                (200, 5120, 4096, True),
                                (200, 2048, 4096, False)]:
        x = torch.randn(rows, k, device=DEV).to(torch.bfloat16)
        w = torch.randn(n, k, device=DEV).to(torch.bfloat16)
        assert ops._skinny_ok(x, w, 16) == streams
        want = x.double() @ w.double().T
        assert ((ops.linear(x, w).double() - want).abs()
                <= want.abs() * 2 ** -8 + 1e-4 * k ** 0.5).all()


def test_skinny_linear_leaves_other_calls_to_the_library():
    """Row counts, types, strides and sizes that the kernel does not take
    give what torch gives; gradients still flow."""
    F = torch.nn.functional

    def rnd(*shape, dtype=torch.bfloat16):
        return torch.randn(*shape, device=DEV).to(dtype)

    w = rnd(64, 256)
    cases = [
        (rnd(17, 256), w), (rnd(0, 256), w), (rnd(2, 3, 256), w),
        (rnd(4, 256, dtype=torch.float32), w.float()),
        (rnd(256, 4).T, w), (rnd(4, 264)[:, 4:260], w),
        (rnd(4, 192), rnd(64, 192)), (rnd(4, 256), rnd(40, 256)),
        (rnd(4, 256), rnd(256, 64).T),
    ]
    for x, m in cases:
        assert not ops._skinny_ok(x, m, 16)
        torch.testing.assert_close(ops.linear(x, m), F.linear(x, m))
    x = rnd(4, 256).requires_grad_()
    ops.linear(x, w).sum().backward()
    assert x.grad is not None


def test_linear_elsewhere_than_on_the_current_gpu(monkeypatch):
    """Operands of another GPU than the current one, or of two places, are
    torch's to follow or refuse."""
    f8 = torch.float8_e4m3fn
    x = torch.randn(4, 4096, device=DEV).to(torch.bfloat16)
    w = torch.randn(4096, 4096, device=DEV).to(torch.bfloat16)
    b = torch.zeros(4096, dtype=torch.bfloat16)
    assert ops._skinny_ok(x, w, 16)
    with pytest.raises(RuntimeError, match="same device"):
        ops.linear(x, w.cpu())
    with pytest.raises(RuntimeError, match="same device"):
        ops.linear(x, w, b)
    calls = []
    for name in ("few_rows_gemm", "few_rows_gemm_fp8"):
        monkeypatch.setattr(ops._C, name, lambda *a: calls.append(a))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    assert torch.equal(ops.linear(x, w), torch.nn.functional.linear(x, w))
    ops.linear_silu_mul(x, w)
    ops.linear_fp8(x.to(f8), torch.ones(4, device=DEV), w.to(f8),
                   torch.ones(4096, device=DEV))
    assert not calls


@pytest.mark.parametrize("rows", [4, 64])
def test_linear_under_transforms_and_modes(rows):
    """Batching, tangents, traces, operator modes and autocast reach the
    product of a linear layer as they reach torch's."""
    from torch.autograd import forward_ad
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils.flop_counter import FlopCounterMode

    F = torch.nn.functional

    def rnd(*shape):
        return torch.randn(shape, device=DEV).to(torch.bfloat16)

    x, t, w, b = rnd(rows, 256), rnd(rows, 256), rnd(64, 256), rnd(64)
    batch = rnd(3, rows, 256)

    def tangent(linear):
        with forward_ad.dual_level():
            out = linear(forward_ad.make_dual(x, t), w, b)
            return forward_ad.unpack_dual(out).tangent

    def flops(linear):
        with FlopCounterMode(display=False) as count:
            linear(x, w, b)
        return torch.tensor(count.get_total_flops())

    def autocast(linear):
        with torch.autocast("cuda", torch.float16):
            return linear(x, w, b)

    for way in (
        lambda f: torch.vmap(lambda v: f(v, w, b))(batch),
        lambda f: torch.func.jvp(lambda v: f(v, w, b), (x,), (t,))[1],
        lambda f: torch.func.grad(lambda v: f(v, w, b).sum())(x),
        lambda f: make_fx(lambda v: f(v, w, b))(x)(t),
        lambda f: torch.jit.trace(lambda v: f(v, w, b), x)(t),
        tangent, flops, autocast,
    ):
        torch.testing.assert_close(way(ops.linear), way(F.linear))

    class Named(torch.Tensor):
        pass

    assert type(ops.linear(x.as_subclass(Named), w)) is Named
    x.requires_grad_()
    ops.linear(x, w).sum().backward()
    assert x.grad is not None


@pytest.mark.parametrize("rows", [4, 64])
@pytest.mark.parametrize("shape", [(1,), (), ("rows", 1), (1, 64),
                                   ("rows", 64)])
def test_linear_bias_that_broadcasts(rows, shape):
    """A bias of another shape than [N] gives what torch gives."""
    def rnd(*shape):
        return torch.randn(shape, device=DEV).to(torch.bfloat16)

    x, w = rnd(rows, 256), rnd(64, 256)
    b = rnd(*[rows if d == "rows" else d for d in shape])
    torch.testing.assert_close(ops.linear(x, w, b),
                               torch.nn.functional.linear(x, w, b))


# ------------------------------------------------- grouped GEMM, 128 rows


@pytest.mark.parametrize("k", [32, 96, 128, 224, 768])
@pytest.mark.parametrize("n,gate_up,act", [
    (64, True, None),          # less than one column tile
    (320, True, None),         # ragged last tile, ragged wave
    (192, True, "clamped_glu"),
    (64, False, "relu_sq"),
    (128, False, None),
    (640, False, None),        # two and a half column tiles
])
def test_moe_gemm_row_blocks_of_128(k, n, gate_up, act):
    check_moe_gemm(k, n, gate_up, act, 128)


@pytest.mark.parametrize("k", [128, 192, 1088])
@pytest.mark.parametrize("n,gate_up,act", [
    (2880, True, None),         # ragged last tile and wave, one round
    (7744, True, "clamped_glu"),  # two rounds
    (5760, False, "relu_sq"),
    (5760, False, None),
    (7744, True, None),
    (15488, False, "relu_sq"),
    (15488, False, None),
])
def test_moe_gemm_wide_tiles(k, n, gate_up, act):
    mode = 3 if act == "clamped_glu" else 1 if gate_up else 2 if act else 0
    # as many blocks and experts as the check has
    assert ops._moe_native().moe_gemm_wide(18, 7, k, n, mode)
    assert not ops._moe_native().moe_gemm_wide(18, 7, k + 32, n, mode)
    check_moe_gemm(k, n, gate_up, act, 128)


@pytest.mark.parametrize("n,gate_up,act", [
    (2880, True, None), (5760, False, "relu_sq"), (5760, False, None)])
def test_moe_gemm_wide_tiles_carry_what_is_not_finite(n, gate_up, act):
    """A row's infinity or NaN stays in the row, an expert's in the expert's
    column."""
    g = torch.Generator().manual_seed(n)
    experts, k, T = 7, 128, 2000
    mode = 1 if gate_up else 2 if act else 0
    x = torch.randn(T, k, generator=g)
    w = torch.randn(experts, k, 2 * n if gate_up else n, generator=g)
    x[5, 1], x[700, 0], x[1999, 127] = (float(v) for v in ("nan", "inf",
                                                           "-inf"))
    w[2, 9, n - 1] = float("nan")
    topi = (torch.arange(T) % experts).int()[:, None].to(DEV)
    sid, eid, nv, pos, PM = ops.moe_align(topi, 0, experts, 128)
    assert ops._moe_native().moe_gemm_wide(PM // 128, experts, k, n, mode)
    x, w = x.bfloat16().to(DEV), w.bfloat16().to(DEV)
    ids = sid.long()
    gathered = torch.where((ids < T)[:, None], x[ids.clamp(max=T - 1)], 0)
    out = torch.empty(PM, n, dtype=torch.bfloat16, device=DEV)
    ops.moe_gemm(out, x if mode else gathered, ops.pack_moe_weights(w), sid,
                 eid, nv, 128, gate_up, act, 3.0)
    for m in range(int(nv)):
        at = slice(m * 128, (m + 1) * 128)
        live = ids[at] < T
        y = gathered[at][live].double() @ w[int(eid[m])].double()
        if gate_up:
            y = torch.nn.functional.silu(y[:, :n]) * y[:, n:]
        elif act:
            # (the kernel's maximum takes the number that is none for zero)
            y = torch.where(y.isnan(), 0, y).clamp(min=0).square()
        got = out[at][live].double()
        assert torch.equal(got.isnan(), y.isnan()), m
        assert torch.equal(got.isinf(), y.isinf()), m


def test_moe_gemm_wide_tiles_are_the_narrow_ones():
    """Blocks of 128 rows have the same bits whether there are enough of them
    for wide tiles or not; gates reach to where 1 + exp(-gate) leaves fp32."""
    g = torch.Generator().manual_seed(11)
    experts, k, n, T = 4, 128, 2880, 2000
    x = torch.randn(T, k, generator=g).bfloat16()
    x[::3] *= 8
    w = torch.randn(experts, k, 2 * n, generator=g).bfloat16()
    topi = torch.randint(0, experts, (T, 1), generator=g).int().to(DEV)
    sid, eid, nv, pos, PM = ops.moe_align(topi, 0, experts, 128)
    x, b = x.to(DEV), ops.pack_moe_weights(w.to(DEV))
    out = torch.zeros(PM, n, dtype=torch.bfloat16, device=DEV)
    blocks = int(nv)
    wide = ops._moe_native().moe_gemm_wide
    assert wide(PM // 128, experts, k, n, 1) and not wide(4, experts, k, n, 1)
    ops.moe_gemm(out, x, b, sid, eid, nv, 128, True, None, 3.0)
    few = torch.zeros_like(out)
    for m in range(0, blocks, 4):
        count = min(4, blocks - m)
        rows = slice(m * 128, (m + count) * 128)
        ops.moe_gemm(few[rows], x, b, sid[rows], eid[m:m + count],
                     torch.full_like(nv, count), 128, True, None, 3.0)
    assert torch.equal(out, few)


@pytest.mark.parametrize("n,gate_up", [
    (896, True), (1792, False),     # one square tile fewer than places
    (1024, True), (2048, False)])
def test_moe_gemm_pairs_of_blocks(n, gate_up):
    """Experts of one block, whole pairs and pairs and one, and of more blocks
    than are looked at together, have the bits of blocks taken alone."""
    counts = [1, 2, 8, 9, 3, 16, 1, 16]
    g = torch.Generator().manual_seed(n)
    k, T, experts = 192, 700, len(counts)
    eid = torch.tensor(sum(([e] * c for e, c in enumerate(counts)), []),
                       dtype=torch.int32, device=DEV)
    blocks = len(eid)
    nv = torch.tensor([blocks], dtype=torch.int32, device=DEV)
    sid = torch.randint(0, T, (blocks * 128,), generator=g).int().to(DEV)
    x = torch.randn(T if gate_up else blocks * 128, k, generator=g)
    w = torch.randn(experts, k, n * (2 if gate_up else 1), generator=g)
    x, b = x.bfloat16().to(DEV), ops.pack_moe_weights(w.bfloat16().to(DEV))
    wide, mode = ops._moe_native().moe_gemm_wide, 1 if gate_up else 0
    assert wide(blocks, experts, k, n, mode)
    assert not wide(8, experts, k, n, mode)
    out = torch.zeros(blocks * 128, n, dtype=torch.bfloat16, device=DEV)
    few = torch.zeros_like(out)
    ops.moe_gemm(out, x, b, sid, eid, nv, 128, gate_up)
    for m in range(0, blocks, 8):
        rows = slice(m * 128, (m + 8) * 128)
        ops.moe_gemm(few[rows], x if gate_up else x[rows], b, sid[rows],
                     eid[m:m + 8], torch.full_like(nv, 8), 128, gate_up)
    assert torch.equal(out, few)


@pytest.mark.parametrize("gate_up", [True, False])
@pytest.mark.parametrize("counts", [
    [1, 2, 8, 9, 3, 16, 1, 16] + [1] * 8 + [2] * 4,
    [1] * 60 + [43, 1, 70, 3, 64],   # pairs over the ends of 64 blocks
    [1, 62, 3, 70, 130],   # many blocks an expert: gathered rows go alone
])
def test_moe_gemm_pairs_of_many_blocks(counts, gate_up):
    """Few and many blocks an expert, more than a word of the pairs' bits holds: the
    bits of blocks taken alone."""
    g = torch.Generator().manual_seed(len(counts))
    k, T, experts = 128, 700, len(counts)
    eid = torch.tensor(sum(([e] * c for e, c in enumerate(counts)), []),
                       dtype=torch.int32, device=DEV)
    blocks = len(eid)
    wide, mode = ops._moe_native().moe_gemm_wide, 1 if gate_up else 0
    n = next(n for n in range(640, 4096, 128)
             if wide(blocks, experts, k, n, mode))
    few_blocks = next(m for m in range(8, 64, 8)
                      if not wide(m, experts, k, n, mode))
    nv = torch.tensor([blocks], dtype=torch.int32, device=DEV)
    sid = torch.randint(0, T, (blocks * 128,), generator=g).int().to(DEV)
    x = torch.randn(T if gate_up else blocks * 128, k, generator=g)
    w = torch.randn(experts, k, n * (2 if gate_up else 1), generator=g)
    x, b = x.bfloat16().to(DEV), ops.pack_moe_weights(w.bfloat16().to(DEV))
    out = torch.zeros(blocks * 128, n, dtype=torch.bfloat16, device=DEV)
    few = torch.zeros_like(out)
    ops.moe_gemm(out, x, b, sid, eid, nv, 128, gate_up)
    for m in range(0, blocks, few_blocks):
        rows = slice(m * 128, min(m + few_blocks, blocks) * 128)
        ids = torch.zeros(few_blocks, dtype=torch.int32, device=DEV)
        ids[:len(eid[m:m + few_blocks])] = eid[m:m + few_blocks]
        ops.moe_gemm(few[rows], x if gate_up else x[rows], b, sid[rows], ids,
                     torch.full_like(nv, len(eid[m:m + few_blocks])), 128,
                     gate_up)
    assert torch.equal(out, few)


@pytest.mark.parametrize("k", [32, 224, 512, 768, 1024, 2080, 2624])
@pytest.mark.parametrize("n,gate_up,act", [
    (64, True, None), (320, True, "clamped_glu"), (192, False, "relu_sq"),
    (128, False, None),
])
def test_moe_gemm_row_blocks_of_16(k, n, gate_up, act):
    """Waves with no step, two, three, four and eight steps of K, more than
    one stretch with a remainder."""
    check_moe_gemm(k, n, gate_up, act, 16)


def test_moe_block_rows():
    """Small blocks where 128 rows have no kernel; as before from 64 rows
    per expert on."""
    assert ops.moe_block_rows(63 * 8, 8, 96, 2048) == 16
    assert ops.moe_block_rows(63 * 8, 8, 128, 64) == 16
    assert ops.moe_block_rows(64 * 8, 8, 96, 64) == 128
    assert ops.moe_block_rows(512, 128, 768, 2048) == 16
    assert ops.moe_block_rows(4096, 128, 768, 2048) == 128


def check_moe_gemm(k, n, gate_up, act, bm):
    """Experts with no row, one row, a whole block, a block and one row and
    many, against float64 products; one bf16 rounding of the result (2^-9)
    and fp32 sums of k products of unit variance."""
    g = torch.Generator().manual_seed(k + n)
    T, top = 700, 2
    sizes = [0, 1, 128, 129, 300, 0, 842]   # assignments, 2 T in all
    experts = torch.cat([torch.full((c,), e) for e, c in enumerate(sizes)])
    topi = experts[torch.randperm(T * top, generator=g)].view(T, top)
    topi = topi.int().to(DEV)
    gather = gate_up or act is not None
    nb = 2 * n if gate_up else n
    w = torch.randn(len(sizes), k, nb, generator=g).to(torch.bfloat16).to(DEV)
    sid, eid, nv, pos, PM = ops.moe_align(topi, 0, len(sizes), bm)
    rows = torch.randn(T if gather else PM, k, generator=g)
    rows = rows.to(torch.bfloat16).to(DEV)
    out = torch.empty(PM, n, dtype=torch.bfloat16, device=DEV)
    ops.moe_gemm(out, rows, ops.pack_moe_weights(w), sid, eid, nv, bm,
                 gate_up, act, 3.0)
    assert int(nv) == sum(-(-c // bm) for c in sizes)
    for m in range(int(nv)):
        at = slice(m * bm, (m + 1) * bm)
        a = rows[sid[at].long()] if gather else rows[at]
        y = a.double() @ w[int(eid[m])].double()
        slack = 1e-5 * k ** 0.5
        if act == "clamped_glu":
            gt, up = y[:, :n].clamp(max=3.0), y[:, n:].clamp(-3.0, 3.0)
            y = gt * torch.sigmoid(1.702 * gt) * (up + 1.0)
            slack *= 20
        elif gate_up:
            y = torch.nn.functional.silu(y[:, :n]) * y[:, n:]
            slack *= 20 * k ** 0.5
        elif act == "relu_sq":
            y = y.clamp(min=0).square()
            slack *= 20 * k ** 0.5
        err = (out[at].double() - y).abs()
        assert (err <= y.abs() * 2 ** -8 + slack).all(), m


@pytest.mark.parametrize("bm", [16, 128])
@pytest.mark.parametrize("act,gate_up", [(None, True), ("relu_sq", False)])
def test_moe_gemm_rows_over_4_gb(bm, act, gate_up):
    """Gathered rows at both ends of 2^31 values and more; bound as above."""
    g = torch.Generator().manual_seed(bm)
    T, k, n = (1 << 20) + 64, 2048, 64
    x = torch.empty(T, k, dtype=torch.bfloat16, device=DEV)
    ids = torch.cat([torch.arange(64), torch.arange(T - 64, T)])
    ids = ids[torch.randperm(128, generator=g)].int().to(DEV)
    x[:64] = torch.randn(64, k, generator=g).to(x.dtype).to(DEV)
    x[-64:] = torch.randn(64, k, generator=g).to(x.dtype).to(DEV)
    w = torch.randn(1, k, 2 * n if gate_up else n, generator=g)
    w = (w / 32).to(x.dtype).to(DEV)
    out = torch.empty(128, n, dtype=x.dtype, device=DEV)
    ops.moe_gemm(out, x, ops.pack_moe_weights(w), ids,
                 torch.zeros(128 // bm, dtype=torch.int32, device=DEV),
                 torch.tensor([128 // bm], dtype=torch.int32, device=DEV), bm,
                 gate_up, act, 0.0)
    y = x[ids.long()].double() @ w[0].double()
    y = torch.nn.functional.silu(y[:, :n]) * y[:, n:] if gate_up \
        else y.clamp(min=0).square()
    assert ((out.double() - y).abs() <= y.abs() * 2 ** -8 + 1e-4).all()


@pytest.mark.parametrize("bm", [16, 128])
def test_moe_gemm_expert_of_4_gb(bm):
    """An expert of 2^31 values: its first and last fragments are found."""
    g = torch.Generator().manual_seed(bm)
    k, n = 1 << 15, 1 << 16
    part = torch.randn(2, 32, 16, generator=g).bfloat16().to(DEV)
    b = torch.zeros(1, k // 32, n // 16, 64, 8, dtype=torch.bfloat16,
                    device=DEV)
    b[0, 0, 0], b[0, -1, -1] = ops.pack_moe_weights(part)[:, 0, 0]
    a = torch.randn(128, k, generator=g).bfloat16().to(DEV)
    out = torch.empty(128, n, dtype=torch.bfloat16, device=DEV)
    ops.moe_gemm(out, a, b, torch.zeros(128, dtype=torch.int32, device=DEV),
                 torch.zeros(128 // bm, dtype=torch.int32, device=DEV),
                 torch.tensor([128 // bm], dtype=torch.int32, device=DEV), bm,
                 False, None, 0.0)
    for got, y in ((out[:, :16], a[:, :32].double() @ part[0].double()),
                   (out[:, -16:], a[:, -32:].double() @ part[1].double())):
        assert ((got.double() - y).abs() <= y.abs() * 2 ** -8 + 1e-4).all()
    assert not out[:, 16:-16].any()


@pytest.mark.parametrize("bm", [16, 128])
@pytest.mark.parametrize("gate_up", [True, False])
def test_moe_gemm_rows_off_the_16_byte_grid(bm, gate_up):
    """Rows that start off the grid give the bits of rows on it."""
    g = torch.Generator().manual_seed(bm)
    x = torch.randn(128, 256, generator=g).bfloat16().to(DEV)
    w = ops.pack_moe_weights(
        torch.randn(1, 256, 256, generator=g).bfloat16().to(DEV))
    ids = torch.randperm(128, generator=g).int().to(DEV)
    outs = []
    for a in (x, _shifted(x, 3)):
        outs.append(torch.empty(128, 128 if gate_up else 256, dtype=x.dtype,
                                device=DEV))
        ops.moe_gemm(outs[-1], a, w, ids,
                     torch.zeros(128 // bm, dtype=torch.int32, device=DEV),
                     torch.tensor([128 // bm], dtype=torch.int32, device=DEV),
                     bm, gate_up)
    assert torch.equal(*outs)


# --------------------------- attention with sink, gate and window, bf16 rows


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("heads,groups,block,window,keep,gate", [
    (4, 1, 16, 0, 0, None),
    (8, 1, 1, 0, 0, "head"),       # rows of their own blocks
    (6, 3, 16, 64, 0, "entry"),    # window of a tile: nothing kept
    (3, 3, 8, 100, 70, "head"),    # kept keys beyond the first tile
    (2, 2, 1, 33, 5, "entry"),
    (5, 1, 16, 300, 1, None),      # window wider than some contexts
])
def test_sink_attention_row_tiles(D, heads, groups, block, window, keep,
                                  gate):
    """Portions of 1, 32, 129 and 300 rows, some behind cached keys, against
    the fp32 reference on the same bf16 values. Weights and results are
    rounded once to bf16 each: at most 2^-8 of the largest value."""
    from fusioninfer_amd.ops import seqmix

    g = torch.Generator().manual_seed(D + heads + window)
    new, past = [1, 32, 129, 300], [40, 0, 277, 64]
    ctx = [a + b for a, b in zip(new, past)]
    need = [-(-c // block) for c in ctx]
    order = torch.randperm(sum(need) + 2, generator=g)
    table = torch.zeros(len(new), max(need), dtype=torch.int32)
    for i, n in enumerate(need):
        table[i, :n] = order[sum(need[:i]):sum(need[:i + 1])]
    T = sum(new)
    q = torch.randn(T, heads, D, generator=g).bfloat16()
    k = torch.randn(len(order), groups, block, D, generator=g).bfloat16()
    v = torch.randn(len(order), groups, block, D, generator=g).bfloat16()
    sink = torch.randn(heads, generator=g) * 3
    og = {"head": torch.randn(T, heads, generator=g).bfloat16(),
          "entry": torch.randn(T, heads * D, generator=g).bfloat16()}.get(gate)
    cu = torch.tensor([0, *torch.tensor(new).cumsum(0)], dtype=torch.int32)
    rows = torch.cat([torch.full((n,), i) for i, n in enumerate(new)]).int()
    pos = torch.cat([torch.arange(p, p + n) for n, p in zip(new, past)]).int()
    want = seqmix.sink_paged_attention(
        q.float(), k.float(), v.float(), table, rows, pos, D ** -0.5,
        sink=sink, out_gate=None if og is None else og.float(), seq_cu=cu,
        window=window, keep_first=keep)
    dev = lambda t: None if t is None else t.to(DEV)
    got = seqmix.sink_paged_attention(
        dev(q), dev(k), dev(v), dev(table), dev(rows), dev(pos), D ** -0.5,
        sink=dev(sink), out_gate=dev(og), seq_cu=dev(cu),
        tiles=seqmix.build_attention_tiles(new, device=DEV), window=window,
        keep_first=keep)
    err = (got.cpu().float() - want.view(got.shape)).abs().max()
    assert err <= 2 ** -8 * v.float().abs().max()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("off", ["q", "k", "v"])
def test_sink_attention_row_tiles_off_the_16_byte_grid(D, off):
    """Tensors that start 8 bytes off the grid take the tiles that stage
    through registers; bound as above, against the rows on the grid: both
    round weights and results to bf16 once."""
    from fusioninfer_amd.ops import seqmix

    g = torch.Generator().manual_seed(D)
    new, past, block = [1, 70, 200], [40, 0, 61], 16
    need = [-(-(a + b) // block) for a, b in zip(new, past)]
    table = torch.zeros(3, max(need), dtype=torch.int32)
    for i, n in enumerate(need):
        table[i, :n] = torch.arange(n) + sum(need[:i])
    T = sum(new)
    x = {n: torch.randn(*shape, generator=g).bfloat16().to(DEV) for n, shape in
         (("q", (T, 4, D)), ("k", (sum(need), 2, block, D)),
          ("v", (sum(need), 2, block, D)))}
    cu = torch.tensor([0, *torch.tensor(new).cumsum(0)], dtype=torch.int32)
    rows = torch.cat([torch.full((n,), i) for i, n in enumerate(new)]).int()
    pos = torch.cat([torch.arange(p, p + n) for n, p in zip(new, past)]).int()
    outs = [seqmix.sink_paged_attention(
        t["q"], t["k"], t["v"], table.to(DEV), rows.to(DEV), pos.to(DEV),
        D ** -0.5, seq_cu=cu.to(DEV),
        tiles=seqmix.build_attention_tiles(new, device=DEV))
        for t in (x, dict(x, **{off: _shifted(x[off], 4)}))]
    err = (outs[0].float() - outs[1].float()).abs().max()
    assert err <= 2 * 2 ** -8 * x["v"].float().abs().max()


@pytest.mark.parametrize("DK,DV", [(64, 64), (128, 128), (192, 128),
                                   (288, 256)])
@pytest.mark.parametrize("heads,groups,block,window,keep,gate", [
    (1, 1, 16, 0, 0, None),
    (16, 1, 16, 0, 0, "head"),
    (20, 1, 1, 300, 260, "entry"),   # two batches of heads; kept span
    (12, 3, 8, 40, 0, "head"),
])
def test_sink_attention_spans(DK, DV, heads, groups, block, window, keep,
                              gate):
    """Single rows at the edges of waves and spans of keys, values a slice of
    the key rows where they are smaller, against float64. The weights are not
    rounded: one bf16 rounding of the result, 2^-8 of it, and fp32 sums."""
    from fusioninfer_amd.ops import seqmix

    g = torch.Generator().manual_seed(DK + heads + window)
    ctx = [1, 16, 64, 65, 256, 257, 1000, 64 * 256 + 3]
    need = [-(-c // block) for c in ctx]
    order = torch.randperm(sum(need) + 2, generator=g)
    table = torch.zeros(len(ctx), max(need), dtype=torch.int32)
    for i, n in enumerate(need):
        table[i, :n] = order[sum(need[:i]):sum(need[:i + 1])]
    T, own = len(ctx), DK == DV
    q = torch.randn(T, heads, DK, generator=g).bfloat16()
    k = torch.randn(len(order), groups, block, DK, generator=g).bfloat16()
    v = torch.randn(len(order), groups, block, DV, generator=g).bfloat16() \
        if own else k[..., :DV]
    sink = torch.randn(heads, generator=g) * 3
    og = {"head": torch.randn(T, heads, generator=g).bfloat16(),
          "entry": torch.randn(T, heads * DV, generator=g).bfloat16()
          }.get(gate)
    rows = torch.arange(T).int()
    pos = torch.tensor(ctx).int() - 1
    dev = lambda t: None if t is None else t.to(DEV)
    got = seqmix.sink_paged_attention(
        dev(q), dev(k), dev(v) if own else None, dev(table), dev(rows),
        dev(pos), DK ** -0.5, sink=dev(sink), value_dims=DV,
        out_gate=dev(og), window=window, keep_first=keep)
    rep = heads // groups
    for i, c in enumerate(ctx):
        j = torch.arange(c)
        at = (table[i, j // block].long(), j % block)
        see = j >= c - window if window else j >= 0
        see |= j < keep
        for h in range(heads):
            kk = k[at[0], h // rep, at[1]].double()
            s = kk @ q[i, h].double() * DK ** -0.5
            s[~see] = -float("inf")
            w = torch.softmax(torch.cat([s, sink[h:h + 1].double()]), 0)[:-1]
            want = w @ v[at[0], h // rep, at[1]].double()
            if gate == "head":
                want = want * torch.sigmoid(og[i, h].double())
            elif gate == "entry":
                want = want * torch.sigmoid(
                    og[i, h * DV:(h + 1) * DV].double())
            err = (got[i, h].cpu().double() - want).abs()
            assert (err <= want.abs() * 2 ** -8 + 2e-5).all(), (i, h)


@pytest.mark.parametrize("DK,DV", [(128, 128), (288, 256)])
def test_sink_attention_spans_infinite_values(DK, DV):
    """An infinite value makes its column infinite and no other."""
    from fusioninfer_amd.ops import seqmix

    g = torch.Generator().manual_seed(DK)
    ctx, block = [1, 17, 300], 16
    need = [-(-c // block) for c in ctx]
    table = torch.zeros(len(ctx), max(need), dtype=torch.int32)
    for i, n in enumerate(need):
        table[i, :n] = torch.arange(n) + sum(need[:i])
    q = torch.randn(len(ctx), 4, DK, generator=g).bfloat16()
    k = torch.randn(sum(need), 1, block, DK, generator=g).bfloat16()
    v = torch.randn(sum(need), 1, block, DV, generator=g).bfloat16()
    for i, c in enumerate(ctx):
        v[table[i, (c - 1) // block], 0, (c - 1) % block, 7] = math.inf
        v[table[i, 0], 0, 0, 9] = -math.inf
    got = seqmix.sink_paged_attention(
        q.to(DEV), k.to(DEV), v.to(DEV), table.to(DEV),
        torch.arange(len(ctx), dtype=torch.int32, device=DEV),
        torch.tensor(ctx, dtype=torch.int32, device=DEV) - 1,
        DK ** -0.5).view(len(ctx), 4, DV).cpu()
    assert (got[..., 7] == math.inf).all()
    assert (got[..., 9] == -math.inf).all()
    rest = torch.ones(DV, dtype=torch.bool)
    rest[[7, 9]] = False
    assert got[..., rest].isfinite().all()


@pytest.mark.parametrize("head_dim", [64, 128])
def test_prefill_attention_parts_infinite_values(head_dim):
    """Cut K/V ranges: an infinite value makes its column infinite and no
    other, whichever piece it is in."""
    bs, ctx, n = 16, 2100, 3
    g = torch.Generator().manual_seed(4)
    blocks = -(-ctx // bs)
    q = torch.randn(n, 8, head_dim, generator=g).bfloat16()
    k = torch.randn(blocks, 2, bs, head_dim, generator=g).bfloat16()
    v = torch.randn(blocks, 2, bs, head_dim, generator=g).bfloat16()
    v[0, :, 3, 5] = math.inf
    v[70, :, 0, 6] = -math.inf
    out = ops.prefill_attention_paged(
        q.to(DEV), k.to(DEV), v.to(DEV),
        torch.arange(blocks, dtype=torch.int32, device=DEV)[None],
        torch.tensor([0, n], dtype=torch.int32, device=DEV),
        torch.tensor([ctx], dtype=torch.int32, device=DEV),
        head_dim ** -0.5).cpu()
    assert (out[..., 5] == math.inf).all()
    assert (out[..., 6] == -math.inf).all()
    rest = torch.ones(head_dim, dtype=torch.bool)
    rest[[5, 6]] = False
    assert out[..., rest].isfinite().all()
