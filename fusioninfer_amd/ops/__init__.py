"""Op dispatch: CDNA4 HIP kernels on GPU, PyTorch fp32 reference on CPU.

Policy (required by the build contract): on a GPU box the HIP extension is
the ONLY execution path — if ``_C.so`` is missing or fails to import, any
GPU-tensor call raises immediately instead of silently falling back to
eager PyTorch. CPU tensors (CI containers without a GPU) use the reference
implementations from ``fusioninfer_amd.ops.reference``.
"""

from __future__ import annotations

import math
from typing import NamedTuple, Optional

import torch
from torch.autograd import forward_ad

from fusioninfer_amd.ops import reference as ref

_C = None
_C_IMPORT_ERROR: Optional[BaseException] = None
try:
    import importlib

    _C = importlib.import_module("fusioninfer_amd.ops._C")
except Exception as e:  # pragma: no cover - exercised only when build broken
    _C_IMPORT_ERROR = e


def has_native() -> bool:
    return _C is not None


def _require_native():
    if _C is None:
        raise RuntimeError(
            "fusioninfer_amd HIP extension (_C.so) is not available but a GPU "
            "tensor was passed — refusing to fall back to eager PyTorch on "
            "the GPU path. Build it with `python -m fusioninfer_amd.ops.build`."
        ) from _C_IMPORT_ERROR


# ---------------------------------------------------------------- norm ops

def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    if x.is_cuda:
        _require_native()
        out = torch.empty_like(x)
        _C.rms_norm(out, x, weight, eps)
        return out
    return ref.rms_norm(x, weight, eps)


def fused_add_rms_norm(x, residual, weight, eps: float):
    """In-place on GPU: residual += x; x = rmsnorm(residual). Returns (x, residual)."""
    if x.is_cuda:
        _require_native()
        _C.fused_add_rms_norm(x, residual, weight, eps)
        return x, residual
    return ref.fused_add_rms_norm(x, residual, weight, eps)


def silu_and_mul(x: torch.Tensor) -> torch.Tensor:
    if x.is_cuda:
        _require_native()
        out = torch.empty(
            (*x.shape[:-1], x.shape[-1] // 2), dtype=x.dtype, device=x.device
        )
        _C.silu_and_mul(out, x)
        return out
    return ref.silu_and_mul(x)


# ---------------------------------------------------------------- linear

SKINNY_ROWS = 16  # rows of x up to which a GEMM always streams W
PART_ROWS = 256   # and up to which it does for the sizes below
_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _streams(M: int, N: int, K: int, silu_mul: bool = False) -> bool:
    """Whether the streaming kernels beat the library's GEMM for x [M, K],
    W [N, K]. Up to 16 rows they always do; matrices of less than 2^23
    values, and K below 2048 up to N 8192, take a few us either way and stay
    with the library.

    Up to 128 rows the kernel's own estimate (tiles, parts, joins) is held
    against what the library is seen to take: up to 64 rows W at 3.2 TB/s or
    4.2 us per 1000 of K, and 4.4 us, above them 3.6 TB/s or 3.8 us, and 8;
    with silu_mul 3 us or 1.2 more for the pass over the product. (Where that
    errs most: 12288 x 2560 at 128 rows streams in 26.4 us, the library takes
    23.2.)

    Weights that no cache holds, launched from a graph, 20 N of 1024 to
    151936, eleven K of 1024 to 14336: with _streams_many this choice takes
    0.7 to 1.7 % longer than the best of the library, parts in any shape and
    tiles up to 128 rows, 1.7 to 2.0 % at 144 to 192 and 3.4 to 3.8 at 224
    and 256; the library alone 13 to 22. With silu_mul 0.8 to 1.0 % and 2.3
    to 3.9, the library alone 18 to 32."""
    if M <= SKINNY_ROWS:
        return True
    if M > PART_ROWS or N * K < 1 << 23 or K < 2048 and N <= 8192:
        return False
    if M > 128:
        return _streams_many(M, N, K, silu_mul)
    if M <= 64:
        library = 4.4 + max(2 * N * K / 3.2e6, 4.2e-3 * K) + 3 * silu_mul
    else:
        library = 8 + max(2 * N * K / 3.6e6, 3.8e-3 * K) + 1.2 * silu_mul
    return _C.few_rows_gemm_us(M, N, K) < library


def _streams_many(M: int, N: int, K: int, silu_mul: bool) -> bool:
    """_streams from 129 rows on. There both compute more than they read, and
    the library's choice of tiles jumps with M, N and K, so the lines are where
    one of the two is ahead for good (us, the library and here). N above 2^15:
    the library, but for one row of tiles where _one_row says so and W beyond
    2^16 (57344 x 8192 at 160 and 256 rows 183 and 226, 217 and 260; 40960 x
    4096 at 256 93 and 108; 151936 x 4096 at 256 361 and 303). Few values of W,
    short rows and N 12289 to 16384: the library (2048 x 4096 at 192 16.0 and
    21.0, 4096 x 2048 at 256 13.7 and 20.2, 16384 x 2560 at 144 28.6 and 32.9);
    what it has tiles for at few rows too: up to 144 (8192 x 2048 15.7 and
    21.1, 6144 x 4096 39.6 and 24.4), up to 160 (3072 x 4096 16.6 and 21.2, 4096
    x 4096 27.2 and 21.6). With silu_mul here: the pass over the product costs
    the library 3 to 10."""
    if K < 2048 and (N > 96 * 256 or not silu_mul):
        return False
    if N > 1 << 15:
        return not (N <= 1 << 16 and K >= 8192) and (
            silu_mul or N > 1 << 16 or _one_row(M, N, K, silu_mul))
    if silu_mul:
        return True
    if N * K < 3 << 22 or 12288 < N <= 1 << 14 and N * K <= 3 << 24:
        return False
    if M > 192:
        return N * K >= 5 << 22 and K > 2048
    if M > 160 or K >= 6144:
        return True
    if M > 144:
        return N > 1 << 14 or K >= 2560 and N * K >= 1 << 24
    return N >= 12288 or N <= 6144 and N * K >= 1 << 24


def _one_row(M: int, N: int, K: int, silu_mul: bool) -> bool:
    """Of 129 to 256 rows, whether one row of 256 x 256 tiles is ahead of
    parts, by the two kernels' own estimates: wide W, where the chip has whole
    rounds of tiles (151936 x 4096 at 160 and 256 rows 306 and 343 us in parts,
    273 and 300 so). Up to 2^16 long K is the library's: 57344 x 4096 at 256
    rows 117 us here, 116 there, 57344 x 5120 at 160 139 and 126; with silu_mul
    40960 x 2048 at 256 52, the library 61, in parts 59."""
    if N <= 1 << 16:
        ok = N >= (40960 if silu_mul else 49152) and (
            K <= 4096 or silu_mul and N >= 57344 and K < 8192)
    else:
        ok = N <= 1 << 20 and K < 8192
    return ok and (_C.many_rows_gemm_us(M, N, 2 * K)
                   < _C.few_rows_gemm_us(M, N, K))


def _memory_alone(x, w, bias) -> bool:
    """Whether a call is about its operands' memory and nothing else. The
    kernels see no compilation, functional transform, operator or autocast
    mode, tensor subclass, gradient or tangent (nor a trace); torch's own
    operations carry all of them. A microsecond: it runs at every call."""
    return (
        type(x) in _PLAIN and type(w) in _PLAIN
        and (bias is None or type(bias) in _PLAIN)
        and not (torch.is_grad_enabled() and (
            x.requires_grad or w.requires_grad
            or bias is not None and bias.requires_grad))
        and forward_ad._current_level < 0
        and torch._C._functorch.maybe_current_level() is None
        and torch._C._len_torch_dispatch_stack() == 0
        and torch._C._len_torch_function_stack() == 0
        and not torch.is_autocast_enabled("cuda")
        and not torch.compiler.is_compiling()
    )


def _on_current_gpu(x, w, *others) -> bool:
    """Whether all lie on the GPU that a launch goes to; torch's operations
    follow their operands or refuse a mixture."""
    d = x.get_device()
    return (0 <= d == w.get_device() and all(t.get_device() == d
                                             for t in others)
            and d == torch.cuda.current_device())


def _skinny_ok(x, w, unit: int, silu_mul: bool = False, bias=None) -> bool:
    """Whether x W^T (+ bias) can run on the streaming kernels: few bf16
    rows, whole 128-value stages of K, whole tiles of N, 16-byte aligned
    rows, a bias of [N], an eager call without gradients. A family that
    builds only its own extension keeps the library's GEMM."""
    return (
        _C is not None and not torch._C._is_tracing()
        and x.dim() == 2 and w.dim() == 2 and 1 <= x.shape[0] <= PART_ROWS
        and _memory_alone(x, w, bias)
        and (_on_current_gpu(x, w) if bias is None
             else _on_current_gpu(x, w, bias))
        and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
        and x.shape[1] == w.shape[1] and 0 < x.shape[1] <= 1 << 24
        and x.shape[1] % 128 == 0
        and 0 < w.shape[0] <= 1 << 24 and w.shape[0] % unit == 0
        and x.stride(1) == 1 and x.stride(0) % 8 == 0
        and x.stride(0) <= 1 << (24 if x.shape[0] <= SKINNY_ROWS else 22)
        and _streams(x.shape[0], w.shape[0], x.shape[1], silu_mul)
        and w.is_contiguous()
        and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
        and (bias is None or (
            bias.dtype == torch.bfloat16 and bias.is_contiguous()
            and bias.shape == w.shape[:1]))
    )


def _tiles(M: int, N: int, K: int, silu_mul: bool = False) -> bool:
    """Whether the kernel of 256 x 256 tiles beats the library's GEMM for
    more than 256 rows. On whole rounds of tiles both reach 1.4 to 1.55
    PFLOP/s; the kernel cuts what is left over into even pieces, where the
    library's choice of tiles takes up to twice as long (4099 rows, 4096 x
    12288: 281 us here, 614; 24576 x 4096 572 and 695; 2700 rows 380 and
    471). The kernel's own estimate is held against 8 us and 1.2 PFLOP/s, or
    the chain of 7 us per 1000 of K; with silu_mul the pass over the product
    is added, which the kernel has in its epilogue (7600 rows, 24576 x 4096
    1020 us here, 1127). Over 504 sizes this took 2.6 % longer than the better
    of the two, the library alone 4.8 (up to 98), the kernel alone 11 (before
    rows of x and W went by the vector offset, which made the kernel up to an
    eighth faster where K is long).

    Where both operands together outgrow the memory-side cache and rows are
    longer than 16 KB the two are even or the library is ahead (4096 x 12288
    at 7600 rows 519 us, 525 here, at 8192 530 and 528; 8192 x 14336 at 6000
    900 and 1008)."""
    if K > 8192 and (M + N) * K > 1 << 27:
        return False
    library = max(8 + 2 * M * N * K / 1.2e9, 7e-3 * K)
    if silu_mul:
        library += 3 * M * N / 5e6
    return _C.many_rows_gemm_us(M, N, 2 * K) < library


def _tiles_ok(x, w, unit: int, silu_mul: bool = False, bias=None) -> bool:
    """As _skinny_ok, for the rows above: whole 64-value stages of K."""
    return (
        _C is not None and not torch._C._is_tracing()
        and x.dim() == 2 and w.dim() == 2 and x.shape[0] > PART_ROWS
        and _memory_alone(x, w, bias)
        and (_on_current_gpu(x, w) if bias is None
             else _on_current_gpu(x, w, bias))
        and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
        and x.shape[1] == w.shape[1] and 128 <= x.shape[1] <= 1 << 22
        and x.shape[1] % 64 == 0 and x.shape[0] <= 1 << 20
        and 0 < w.shape[0] <= 1 << 20 and w.shape[0] % unit == 0
        and x.stride(1) == 1 and x.stride(0) % 8 == 0
        and x.shape[1] <= x.stride(0) <= 1 << 22
        and _tiles(x.shape[0], w.shape[0], x.shape[1], silu_mul)
        and w.is_contiguous()
        and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
        and (bias is None or (
            bias.dtype == torch.bfloat16 and bias.is_contiguous()
            and bias.shape == w.shape[:1] and bias.data_ptr() % 16 == 0))
    )


def _one_row_of_tiles(x, w, bias=None, silu_mul: bool = False) -> bool:
    """Whether 129 to 256 rows that stream go by tiles of 256 x 256 for it."""
    M, N, K = x.shape[0], w.shape[0], w.shape[1]
    return (
        M > 128 and x.stride(0) >= K
        and (bias is None or bias.data_ptr() % 16 == 0)
        and _one_row(M, N, K, silu_mul)
    )


def linear(x: torch.Tensor, w: torch.Tensor,
           bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x W^T (+ bias): a few bf16 rows stream W once through the kernels for
    that, many rows go by tiles where the library's GEMM leaves the chip
    idle, anything else is the library's."""
    if _skinny_ok(x, w, 16, bias=bias):
        out = torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype,
                          device=x.device)
        if _one_row_of_tiles(x, w, bias):
            _C.many_rows_gemm(out, x, w, bias, False)
        else:
            _C.few_rows_gemm(out, x, w, bias, False)
        return out
    if _tiles_ok(x, w, 16, bias=bias):
        out = torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype,
                          device=x.device)
        _C.many_rows_gemm(out, x, w, bias, False)
        return out
    return torch.nn.functional.linear(x, w, bias)


def _streams_fp8(M: int, N: int, K: int) -> bool:
    """As _streams, for e4m3 operands with scales per row. Up to 16 rows the
    library is behind at nearly all sizes (24576 x 4096 at 16 rows 30 us, 19
    here); up to 64 rows it takes W at 4.7 TB/s and 7.8 us or 2.2 us per 1000
    of K (6144 x 4096 at 64 13.5 and 14.8, 4096 x 12288 24.2 and 18.0), and
    less for few values of W (2560 x 4096 9.4 and 11.7). From 65 rows on it
    is ahead but for long K and few tiles (4096 x 12288 at 96 and 128 rows 30
    and 36, here 24 and 25). Twelve N and eleven K, launched from a graph:
    this choice takes 0.3 to 1.7 % longer than the best of the two up to 96
    rows (the library alone 10 to 48), 2.0 at 128."""
    if M > 128 or N * K < 1 << 23:
        return False
    if M <= SKINNY_ROWS:
        return True
    if M > 64:
        return M >= 96 and K >= 2 * N and N >= 3072
    if M > 32 and N * K < 3 << 22:
        return False
    return _C.few_rows_gemm_us(M, N, K, True) < max(7.8 + N * K / 4.7e6,
                                                    0.6 + 2.2e-3 * K)


def _tiles_fp8(M: int, N: int, K: int) -> bool:
    """As _tiles, for e4m3 operands: the kernel's own estimate against 6 us
    and 2.2 PFLOP/s, or 18 us and 2 us per 1000 of K above 8192 (4096 x 4096
    at 1024 rows 38 us here, the library 28; at 8192 100 and 111; 4096 x
    12288 at 4099 151 and 270). Over twelve N and K and up to 17 M of
    257 to 8192 this takes 2.4 % longer than the better of the two, the
    library alone 8.9 (up to 75), the kernel alone 8.7."""
    return _C.many_rows_gemm_us(M, N, K) < max(
        6 + 2 * M * N * K / 2.2e9, 18 + 2e-3 * max(0, K - 8192))


def _tiles_fp8_ok(x, x_scales, w, w_scales) -> bool:
    """As _tiles_ok, for e4m3 operands with a scale per row each."""
    return (
        _C is not None and not torch._C._is_tracing()
        and x.dim() == 2 and w.dim() == 2 and x.shape[0] > PART_ROWS
        and _memory_alone(x, w, x_scales) and type(w_scales) in _PLAIN
        and _on_current_gpu(x, w, x_scales, w_scales)
        and x.dtype == w.dtype == torch.float8_e4m3fn
        and x.shape[1] == w.shape[1] and 256 <= x.shape[1] <= 1 << 22
        and x.shape[1] % 128 == 0 and x.shape[0] <= 1 << 20
        and 0 < w.shape[0] <= 1 << 20 and w.shape[0] % 16 == 0
        and x.stride(1) == 1 and x.stride(0) % 16 == 0
        and x.shape[1] <= x.stride(0) <= 1 << 22
        and _tiles_fp8(x.shape[0], w.shape[0], x.shape[1])
        and w.is_contiguous()
        and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
        and x_scales.dtype == w_scales.dtype == torch.float32
        and x_scales.is_contiguous() and w_scales.is_contiguous()
        and x_scales.shape == x.shape[:1] and w_scales.shape == w.shape[:1]
        and w_scales.data_ptr() % 16 == 0
    )


def _few_rows_fp8_ok(x, x_scales, w, w_scales) -> bool:
    """As _skinny_ok, for e4m3 operands with a scale per row each: whole
    256-value stages of K."""
    return (
        _C is not None and x.dim() == 2 and w.dim() == 2
        and 1 <= x.shape[0] <= 128 and x.shape[1] == w.shape[1]
        and _on_current_gpu(x, w, x_scales, w_scales)
        and x.dtype == w.dtype == torch.float8_e4m3fn
        and x.shape[1] % 256 == 0 and w.shape[0] % 16 == 0
        and 0 < x.shape[1] <= 1 << 24 and 0 < w.shape[0] <= 1 << 24
        and _streams_fp8(x.shape[0], w.shape[0], x.shape[1])
        and x.stride(1) == 1 and x.stride(0) % 16 == 0
        and x.stride(0) <= 1 << 22 and w.is_contiguous()
        and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
        and x_scales.dtype == w_scales.dtype == torch.float32
        and x_scales.is_contiguous() and w_scales.is_contiguous()
        and x_scales.shape == x.shape[:1]
        and w_scales.shape == w.shape[:1]
    )


def linear_fp8(x: torch.Tensor, x_scales: torch.Tensor, w: torch.Tensor,
               w_scales: torch.Tensor) -> torch.Tensor:
    """(x * x_scales) (w * w_scales)^T in bf16 on the GPU: x [M, K] and w
    [N, K] e4m3, a scale per row each."""
    if _few_rows_fp8_ok(x, x_scales, w, w_scales):
        out = torch.empty((x.shape[0], w.shape[0]), dtype=torch.bfloat16,
                          device=x.device)
        _C.few_rows_gemm_fp8(out, x, x_scales, w, w_scales)
        return out
    if _tiles_fp8_ok(x, x_scales, w, w_scales):
        out = torch.empty((x.shape[0], w.shape[0]), dtype=torch.bfloat16,
                          device=x.device)
        _C.many_rows_gemm_fp8(out, x, x_scales, w, w_scales)
        return out
    return torch._scaled_mm(
        x, w.t(),  # column-major view of the row-major weight
        scale_a=x_scales.unsqueeze(1), scale_b=w_scales.unsqueeze(0),
        out_dtype=torch.bfloat16)


def linear_silu_mul(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """silu(x G^T) * (x U^T) with w = [G; U]; in one kernel where linear has
    one, whose gate and up values are not rounded in between."""
    if _skinny_ok(x, w, 32, True):
        out = torch.empty((x.shape[0], w.shape[0] // 2), dtype=x.dtype,
                          device=x.device)
        if _one_row_of_tiles(x, w, silu_mul=True):
            _C.many_rows_gemm(out, x, w, None, True)
        else:
            _C.few_rows_gemm(out, x, w, None, True)
        return out
    if _tiles_ok(x, w, 32, True):
        out = torch.empty((x.shape[0], w.shape[0] // 2), dtype=x.dtype,
                          device=x.device)
        _C.many_rows_gemm(out, x, w, None, True)
        return out
    return silu_and_mul(linear(x, w))


def linear_gelu(x: torch.Tensor, w: torch.Tensor) -> Optional[torch.Tensor]:
    """gelu(x W^T), the tanh form, where a kernel for few rows or many has it
    in its epilogue; else None. (A pass of its own is a launch of 2.5 us for few
    rows and 33 us for 7100 of 6144. Four layers with four prompts of 1.8
    thousand tokens and eight tokens each: 5540 us, and 5410.)"""
    few = x.dim() == 2 and x.shape[0] <= SKINNY_ROWS
    if not (_skinny_ok(x, w, 16) if few else _tiles_ok(x, w, 16)):
        return None
    out = torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype, device=x.device)
    (_C.few_rows_gemm if few else _C.many_rows_gemm)(out, x, w, None, False,
                                                     True)
    return out


class StreamRows(NamedTuple):
    """Rows of a residual stream on their way into its norm. scaled [M, K] is
    stream times weight, the columns of squares [parts, 16] add up to the sums
    of the rows' squares."""

    stream: torch.Tensor   # [M, K] fp32
    weight: torch.Tensor   # [K] bf16
    eps: float
    scaled: torch.Tensor
    squares: torch.Tensor


def stream_rows_ok(rows: int, columns: int) -> bool:
    """Whether a residual stream [rows, columns] goes as StreamRows: up to 16
    rows always, since a norm then costs next to nothing. us, a norm's launch
    and the product / the product of StreamRows, at 1 and 16 rows: 6144 x 4096
    12.7, 14.7 / 9.9, 12.3; 24576 x 4096 with SiLU 34.8, 35.7 / 32.7, 33.4;
    5120 x 2048 8.4, 10.1 / 6.8, 8.2; 4096 x 1024 5.2, 6.0 / 4.0, 4.2. What
    the layer in front takes for the sum and the rows: 0.2 to 0.5 more."""
    return 0 < rows <= SKINNY_ROWS and columns % 128 == 0


def _stream_rows(stream, weight, eps: float, parts: int) -> StreamRows:
    return StreamRows(
        stream, weight, eps,
        torch.empty(stream.shape, dtype=weight.dtype, device=stream.device),
        torch.empty((parts, 16), dtype=torch.float32, device=stream.device))


def stream_begin(x: torch.Tensor, weight: torch.Tensor,
                 eps: float) -> StreamRows:
    """A stream that is a copy of up to 16 rows x, before the norm of
    weight."""
    _require_native()
    rows = _stream_rows(
        torch.empty(x.shape, dtype=torch.float32, device=x.device), weight,
        eps, 1)
    _C.stream_begin(rows.stream, rows.scaled, rows.squares, x, weight)
    return rows


def stream_norm(stream: torch.Tensor, weight: torch.Tensor,
                eps: float) -> torch.Tensor:
    """rms_norm of fp32 rows, in weight's type."""
    _require_native()
    out = torch.empty(stream.shape, dtype=weight.dtype, device=stream.device)
    _C.stream_norm(out, stream, weight, eps)
    return out


def stream_linear(rows: StreamRows, w: torch.Tensor,
                  bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """linear of the normed rows: the product is divided by the root mean
    squares."""
    x = rows.scaled
    if _skinny_ok(x, w, 16, bias=bias):
        out = torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype,
                          device=x.device)
        _C.few_rows_scaled_gemm(out, x, rows.squares, rows.eps, w, bias, False)
        return out
    return linear(stream_norm(*rows[:3]), w, bias)


def stream_linear_silu_mul(rows: StreamRows, w: torch.Tensor) -> torch.Tensor:
    """linear_silu_mul of the normed rows."""
    x = rows.scaled
    if _skinny_ok(x, w, 32, True):
        out = torch.empty((x.shape[0], w.shape[0] // 2), dtype=x.dtype,
                          device=x.device)
        _C.few_rows_scaled_gemm(out, x, rows.squares, rows.eps, w, None, True)
        return out
    return linear_silu_mul(stream_norm(*rows[:3]), w)


def stream_add_(stream: torch.Tensor, x: torch.Tensor, w: torch.Tensor,
                weight: Optional[torch.Tensor] = None,
                eps: float = 0.0) -> Optional[StreamRows]:
    """stream += linear(x, w), the product unrounded where the kernel for few
    rows runs; with the weight of the norm behind it its rows."""
    if not _skinny_ok(x, w, 16):
        stream.add_(linear(x, w))
        return None if weight is None else stream_begin(stream, weight, eps)
    if weight is None:
        _C.few_rows_gemm_add(stream, x, w, None, None, None)
        return None
    rows = _stream_rows(stream, weight, eps, w.shape[0] // 16)
    _C.few_rows_gemm_add(stream, x, w, weight, rows.scaled, rows.squares)
    return rows


class NormedRows(NamedTuple):
    """Rows behind their norm; of the fp8 mode with a scale each."""

    x: object


def _norm_ok(residual, weight, rows: int, columns: int) -> bool:
    return (
        type(residual) in _PLAIN and type(weight) in _PLAIN
        and residual.dtype == weight.dtype == torch.bfloat16
        and residual.get_device() == weight.get_device()
        == torch.cuda.current_device()
        and residual.shape == (rows, columns) and weight.shape == (columns,)
        and residual.is_contiguous() and weight.is_contiguous()
        and residual.data_ptr() % 8 == 0 and weight.data_ptr() % 8 == 0
    )


def linear_add_rms_norm(x: torch.Tensor, w: torch.Tensor,
                        residual: torch.Tensor, weight: torch.Tensor,
                        eps: float):
    """fused_add_rms_norm(linear(x, w), residual, weight, eps); 17 to 256 rows,
    where pieces of the product are summed by a second kernel, leave that one
    added and normed."""
    if (SKINNY_ROWS < x.shape[0] <= PART_ROWS and _skinny_ok(x, w, 16)
            and _norm_ok(residual, weight, x.shape[0], w.shape[0])):
        out = torch.empty_like(residual)
        if _C.few_rows_gemm_norm(out, x, w, residual, weight, eps):
            return out, residual
    return fused_add_rms_norm(linear(x, w), residual, weight, eps)


# ------------------------------------------------------- fp8 fused epilogues
#
# The fp8 serving mode quantizes activations per-token for torch._scaled_mm;
# done eagerly that costs more than the fp8 GEMM saves, so quantization is
# fused into the producing kernel (norm / SwiGLU) or done in one pass
# (quant_fp8_rows for the attention output).

def rms_norm_fp8(x: torch.Tensor, weight: torch.Tensor, eps: float):
    """Returns (x_fp8 [T, H] e4m3, scales [T] fp32)."""
    if x.is_cuda:
        _require_native()
        out = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=x.device)
        scales = torch.empty(x.shape[0], dtype=torch.float32, device=x.device)
        _C.rms_norm_fp8(out, scales, x, weight, eps)
        return out, scales
    return ref.rms_norm_fp8(x, weight, eps)


def fused_add_rms_norm_fp8(x, residual, weight, eps: float):
    """residual += x in place; returns (x_fp8, scales, residual)."""
    if x.is_cuda:
        _require_native()
        out = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=x.device)
        scales = torch.empty(x.shape[0], dtype=torch.float32, device=x.device)
        _C.fused_add_rms_norm_fp8(out, scales, x, residual, weight, eps)
        return out, scales, residual
    return ref.fused_add_rms_norm_fp8(x, residual, weight, eps)


def linear_fp8_add_rms_norm(x: torch.Tensor, x_scales: torch.Tensor,
                            w: torch.Tensor, w_scales: torch.Tensor,
                            residual: torch.Tensor, weight: torch.Tensor,
                            eps: float):
    """As linear_add_rms_norm, in e4m3: ((rows, scales), residual)."""
    if (_few_rows_fp8_ok(x, x_scales, w, w_scales)
            and _norm_ok(residual, weight, x.shape[0], w.shape[0])):
        out = torch.empty(residual.shape, dtype=x.dtype, device=x.device)
        scales = torch.empty_like(x_scales)
        if _C.few_rows_gemm_norm_fp8(out, scales, x, x_scales, w, w_scales,
                                     residual, weight, eps):
            return (out, scales), residual
    out, scales, residual = fused_add_rms_norm_fp8(
        linear_fp8(x, x_scales, w, w_scales), residual, weight, eps)
    return (out, scales), residual


def silu_and_mul_fp8(x: torch.Tensor):
    """x: [T, 2*I] -> (act_fp8 [T, I] e4m3, scales [T] fp32)."""
    if x.is_cuda:
        _require_native()
        inter = x.shape[-1] // 2
        out = torch.empty(
            (*x.shape[:-1], inter), dtype=torch.float8_e4m3fn, device=x.device
        )
        scales = torch.empty(x.shape[0], dtype=torch.float32, device=x.device)
        _C.silu_and_mul_fp8(out, scales, x)
        return out, scales
    return ref.silu_and_mul_fp8(x)


def quant_fp8_rows(x: torch.Tensor):
    """Per-row dynamic fp8 quant: (x_fp8, scales [T] fp32)."""
    if x.is_cuda:
        _require_native()
        out = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=x.device)
        scales = torch.empty(x.shape[0], dtype=torch.float32, device=x.device)
        _C.quant_fp8_rows(out, scales, x)
        return out, scales
    return ref.quant_fp8_rows(x)


# ---------------------------------------------------------------- rope

def rope_qk_norm_(
    q: torch.Tensor,          # [T, Hq*D] (row-strided slice OK)
    k: torch.Tensor,          # [T, Hk*D]
    positions: torch.Tensor,  # [T] int32
    cos_sin: torch.Tensor,    # [P, D] fp32
    num_q_heads: int,
    num_kv_heads: int,
    head_dim: int,
    q_weight: Optional[torch.Tensor] = None,
    k_weight: Optional[torch.Tensor] = None,
    eps: float = 1e-6,
):
    """Fused optional per-head RMSNorm + NeoX RoPE, in-place. Returns (q, k).
    The models here call rope_qk_norm_cache_, which on the CPU comes back to
    this; on the GPU this form is there for callers without a paged cache."""
    if q.is_cuda:
        _require_native()
        _C.rope_qk_norm(
            q, k, q_weight, k_weight, cos_sin, positions,
            num_q_heads, num_kv_heads, head_dim, eps,
        )
        return q, k
    qv = q.view(-1, num_q_heads, head_dim)
    kv = k.view(-1, num_kv_heads, head_dim)
    qo, ko = ref.rope_qk_norm(qv, kv, positions.long(), cos_sin, q_weight, k_weight, eps)
    q.copy_(qo.reshape(q.shape))
    k.copy_(ko.reshape(k.shape))
    return q, k


def rope_qk_norm_cache_(q, k, v, positions, cos_sin, k_cache, v_cache,
                        slot_mapping, num_q_heads: int,
                        q_weight: Optional[torch.Tensor] = None,
                        k_weight: Optional[torch.Tensor] = None,
                        eps: float = 1e-6, k_inv_scale: float = 1.0,
                        v_inv_scale: float = 1.0):
    """rope_qk_norm_ followed by reshape_and_cache, in one kernel on the
    GPU, where K's result is then in the cache alone (k is left as it is).
    Returns q."""
    if q.is_cuda:
        _require_native()
        _C.rope_qk_norm_cache(q, k, v, q_weight, k_weight, cos_sin, positions,
                              k_cache, v_cache, slot_mapping, num_q_heads,
                              eps, k_inv_scale, v_inv_scale)
        return q
    rope_qk_norm_(q, k, positions, cos_sin, num_q_heads, k_cache.shape[1],
                  k_cache.shape[3], q_weight, k_weight, eps)
    reshape_and_cache(k, v, k_cache, v_cache, slot_mapping, k_inv_scale,
                      v_inv_scale)
    return q


def _rope_in_one(M: int, N: int, K: int) -> bool:
    """Whether the kernel that sums the pieces of a product and goes on with
    its heads is ahead of two. Its reads of pieces wait for one another where a
    tile has many pieces, or many rows many heads. (us, product and rope apart
    and so: 6144 x 4096 at 43, 64 and 128 rows 19.4, 20.2, 26.5 and 18.5, 19.7,
    25.6, 10240 x 4096 at 64 27.5 and 27.0, at 65 29.1 and 31.4; 5120 x 8192 at
    64 27.1 and 26.1, at 65 29.3 and 31.2; 8192 x 4096 at 128 28.3 and 29.1; 256
    rows of 6144 x 4096, with 16 waves a workgroup, 33.1 and 33.6. Eleven kinds
    of heads, seven K, eight numbers of rows: 3.3 % less than two kernels with
    this rule, 3.5 % always in one, with 10 % more at worst.)"""
    return K <= 8192 if M <= 64 else N <= 6144 and K <= 6144


def linear_rope_qk_norm_cache(x, w, bias, positions, cos_sin, k_cache, v_cache,
                              slot_mapping, num_q_heads: int,
                              q_weight: Optional[torch.Tensor] = None,
                              k_weight: Optional[torch.Tensor] = None,
                              eps: float = 1e-6, k_inv_scale: float = 1.0,
                              v_inv_scale: float = 1.0):
    """rope_qk_norm_cache_ of linear(x, w, bias)'s queries, keys and values
    [T, (Hq | Hk | Hk) * D], where one kernel sums the pieces of 17 to 128 rows'
    product and goes on; else None. Returns q."""
    if not (SKINNY_ROWS < x.shape[0] <= 128
            and _rope_in_one(x.shape[0], w.shape[0], x.shape[1])
            and _skinny_ok(x, w, 16, bias=bias)
            and k_cache.shape[3] in (64, 128)
            and w.shape[0] == (num_q_heads + 2 * k_cache.shape[1])
            * k_cache.shape[3]):
        return None
    q = torch.empty((x.shape[0], num_q_heads * k_cache.shape[3]),
                    dtype=x.dtype, device=x.device)
    return q if _C.few_rows_gemm_rope(
        q, x, w, bias, q_weight, k_weight, cos_sin, positions, k_cache,
        v_cache, slot_mapping, num_q_heads, eps, k_inv_scale, v_inv_scale,
    ) else None


# ---------------------------------------------------------------- kv cache

def reshape_and_cache(k, v, k_cache, v_cache, slot_mapping,
                      k_inv_scale: float = 1.0, v_inv_scale: float = 1.0):
    """Scatter K/V rows into the paged cache. For fp8 caches the rows are
    multiplied by the INVERSE per-layer static scales before e4m3
    conversion (vLLM k_scale/v_scale); bf16 caches ignore the scales
    (the read side compensates only on the fp8 path)."""
    if k.is_cuda:
        _require_native()
        _C.reshape_and_cache(k, v, k_cache, v_cache, slot_mapping,
                             k_inv_scale, v_inv_scale)
        return
    H, D = k_cache.shape[1], k_cache.shape[3]
    ref.reshape_and_cache(
        k.view(-1, H, D), v.view(-1, H, D), k_cache, v_cache,
        slot_mapping.long(), k_inv_scale, v_inv_scale,
    )


def gather_kv_blocks(k_cache, v_cache, block_ids) -> torch.Tensor:
    if k_cache.is_cuda:
        _require_native()
        n = int(block_ids.numel())
        staging = torch.empty(
            (2, n, *k_cache.shape[1:]), dtype=k_cache.dtype, device=k_cache.device
        )
        _C.gather_kv_blocks(staging, k_cache, v_cache, block_ids)
        return staging
    return ref.gather_kv_blocks(k_cache, v_cache, block_ids.long())


def scatter_kv_blocks(staging, k_cache, v_cache, block_ids):
    if k_cache.is_cuda:
        _require_native()
        _C.scatter_kv_blocks(staging, k_cache, v_cache, block_ids)
        return
    ref.scatter_kv_blocks(staging, k_cache, v_cache, block_ids.long())


# ---------------------------------------------------------------- attention

def paged_attention_decode(
    q: torch.Tensor,            # [S, Hq, D]
    k_cache: torch.Tensor,      # [B, Hk, bs, D]
    v_cache: torch.Tensor,
    block_tables: torch.Tensor,  # [S, max_blocks] int32
    seq_lens: torch.Tensor,      # [S] int32
    scale: Optional[float] = None,
    out: Optional[torch.Tensor] = None,  # [S, Hq, D] contiguous
) -> torch.Tensor:
    if scale is None:
        scale = 1.0 / math.sqrt(q.shape[-1])
    if q.is_cuda:
        _require_native()
        if out is None:
            out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        _C.paged_attention_decode(out, q, k_cache, v_cache, block_tables,
                                  seq_lens, scale)
        return out
    o = ref.paged_attention_decode(q, k_cache, v_cache, block_tables, seq_lens, scale)
    return o if out is None else out.copy_(o)


# rows per entry of the prefill tile table (128 or 256); the kernel cuts
# entries into the row blocks of its workgroups itself
import os as _os

PREFILL_TILE_ROWS = (4 if _os.environ.get("FI_PF_NW", "8").startswith("4")
                     else 8) * 32


def prefill_tile_rows(seq_lens) -> int:
    """Rows per tile-table entry of a batch: 128 once any sequence has 4096
    new tokens, so that a ragged end leaves fewer empty row blocks."""
    if seq_lens and max(seq_lens) >= 4096:
        return 128
    return PREFILL_TILE_ROWS


def build_prefill_tiles(seq_lens, device=None, rows=None):
    """Host-side tile table for the prefill kernel: one entry per `rows`
    q-rows of each sequence (rows must be 128 or 256 and MATCH the
    tile_rows passed to the kernel).

    seq_lens: list[int]. Returns (tile_seq, tile_row0) int32 tensors.
    """
    rows = rows or PREFILL_TILE_ROWS
    tile_seq, tile_row0 = [], []
    for s, L in enumerate(seq_lens):
        for r0 in range(0, L, rows):
            tile_seq.append(s)
            tile_row0.append(r0)
    return (
        torch.tensor(tile_seq, dtype=torch.int32, device=device),
        torch.tensor(tile_row0, dtype=torch.int32, device=device),
    )


def prefill_attention(
    q: torch.Tensor,           # [T, Hq, D]
    k: torch.Tensor,           # [T, Hk, D]
    v: torch.Tensor,           # [T, Hk, D]
    cu_seqlens: torch.Tensor,  # [S+1] int32
    scale: Optional[float] = None,
    tile_seq: Optional[torch.Tensor] = None,
    tile_row0: Optional[torch.Tensor] = None,
    tile_rows: Optional[int] = None,
) -> torch.Tensor:
    if scale is None:
        scale = 1.0 / math.sqrt(q.shape[-1])
    if q.is_cuda:
        _require_native()
        if tile_seq is None:
            lens = (cu_seqlens[1:] - cu_seqlens[:-1]).tolist()
            tile_rows = tile_rows or prefill_tile_rows(lens)
            tile_seq, tile_row0 = build_prefill_tiles(
                lens, device=q.device, rows=tile_rows
            )
        out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        _C.prefill_attention(out, q, k, v, tile_seq, tile_row0, cu_seqlens,
                             scale, tile_rows or PREFILL_TILE_ROWS)
        return out
    return ref.prefill_attention(q, k, v, cu_seqlens, scale, causal=True)


def prefill_attention_paged(
    q: torch.Tensor,             # [Tnew, Hq, D] new tokens only
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_tables: torch.Tensor,  # [S, max_blocks] int32
    cu_seqlens_q: torch.Tensor,  # [S+1] int32 over new tokens
    seq_lens_k: torch.Tensor,    # [S] int32 total context length
    scale: Optional[float] = None,
    tile_seq: Optional[torch.Tensor] = None,
    tile_row0: Optional[torch.Tensor] = None,
    tile_rows: Optional[int] = None,
    out: Optional[torch.Tensor] = None,  # [Tnew, Hq, D] contiguous
) -> torch.Tensor:
    """Context attention: new tokens attend over the paged cache (their own
    K/V must already be written via reshape_and_cache)."""
    if scale is None:
        scale = 1.0 / math.sqrt(q.shape[-1])
    if q.is_cuda:
        _require_native()
        if tile_seq is None:
            lens = (cu_seqlens_q[1:] - cu_seqlens_q[:-1]).tolist()
            tile_rows = tile_rows or prefill_tile_rows(lens)
            tile_seq, tile_row0 = build_prefill_tiles(
                lens, device=q.device, rows=tile_rows
            )
        if out is None:
            out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        _C.prefill_attention_paged(
            out, q, k_cache, v_cache, tile_seq, tile_row0, cu_seqlens_q,
            block_tables, seq_lens_k, scale,
            tile_rows or PREFILL_TILE_ROWS,
        )
        return out
    o = ref.prefill_attention_paged(
        q, k_cache, v_cache, block_tables, cu_seqlens_q, seq_lens_k, scale
    )
    return o if out is None else out.copy_(o)


# ---------------------------------------------------------------- MoE

def pack_moe_weights(w: torch.Tensor) -> torch.Tensor:
    """Pack per-expert weights [E, K, N] into MFMA B-fragment order
    [E, K/32, N/16, 64, 8] for the grouped GEMM: lane l of a wave reads
    its 8 contiguous bf16 B elements (B[k=(l>>4)*8+e][n=l&15] within a
    32x16 k-by-n subtile) with one 16 B load — one fully-coalesced 1 KiB
    transaction per wave per K-step."""
    E, K, N = w.shape
    assert K % 32 == 0 and N % 16 == 0, (K, N)
    return (
        w.view(E, K // 32, 4, 8, N // 16, 16)
        .permute(0, 1, 4, 2, 5, 3)
        .reshape(E, K // 32, N // 16, 64, 8)
        .contiguous()
    )


_C_MOE = None
_C_MOE_ERR: Optional[BaseException] = None


def _moe_native():
    """The expert-routing kernels live in their own extension
    (``_C_moe.so``) so that any model family with routed experts compiles
    only them, not the transformer kernels."""
    global _C_MOE, _C_MOE_ERR
    if _C_MOE is None:
        try:
            import importlib

            _C_MOE = importlib.import_module("fusioninfer_amd.ops._C_moe")
        except Exception as e:  # noqa: BLE001
            _C_MOE_ERR = e
            raise RuntimeError(
                "fusioninfer_amd expert-routing extension (_C_moe.so) is "
                "not available but a GPU tensor was passed; build it with "
                "`python -m fusioninfer_amd.ops.build moe`."
            ) from e
    return _C_MOE


def has_moe_native() -> bool:
    try:
        return _moe_native() is not None
    except RuntimeError:
        return False


def _moe_gemm_mode(gate_up: bool, up_act) -> int:
    """0: plain GEMM over act rows; 1: gathered x rows, gate|up columns,
    silu(gate) * up; 2: gathered x rows, up columns alone, relu(up)^2;
    3: gathered x rows, gate|up columns, clamped gated unit
    g' sigmoid(1.702 g') (u' + 1) with g' = min(g, limit),
    u' = clamp(u, -limit, limit)."""
    if up_act is None:
        return 1 if gate_up else 0
    if up_act == "clamped_glu" and gate_up:
        return 3
    if up_act != "relu_sq" or gate_up:
        raise ValueError(f"unsupported expert activation {up_act!r}")
    return 2


def moe_gemm(out, a, b_packed, sorted_ids, expert_ids, n_valid,
             block_m: int, gate_up: bool, up_act=None, limit: float = 0.0):
    """Grouped GEMM over block-aligned expert segments.

    out [PM, N] bf16; a = x [T, K] (gate_up, rows gathered via sorted_ids)
    or act [PM, K]; b_packed from pack_moe_weights ([E, K/32, NB/16, 64, 8]
    with NB = 2N when gate_up). n_valid: device int32 scalar tensor with
    the real m-tile count (static grid, dynamic work — hipGraph-safe).
    gate_up=True fuses the SwiGLU epilogue: out = silu(gate) * up.
    up_act="relu_sq" (with gate_up=False): a = x gathered like gate_up,
    b holds the up matrix alone and out = relu(a @ up)^2.
    up_act="clamped_glu" (with gate_up=True): the gated unit clamps gate
    from above and up on both sides at ``limit`` (see _moe_gemm_mode)."""
    mode = _moe_gemm_mode(gate_up, up_act)
    if out.is_cuda:
        _moe_native().moe_gemm(out, a, b_packed, sorted_ids, expert_ids,
                               n_valid, block_m, mode, float(limit))
        return out
    return ref.moe_gemm(out, a, b_packed, sorted_ids, expert_ids, n_valid,
                        block_m, gate_up, up_act, limit)


def moe_gemm_plain(out, a, w, sorted_ids, expert_ids, n_valid, block_m: int,
                   gate_up: bool, up_act=None, limit: float = 0.0):
    """Grouped GEMM of the same block-aligned layout for ANY sizes and for
    fp32 or bf16 operands (fp32 accumulation): w is the experts' natural
    [E, out, in] weight ([E, 2N, K] with gate rows first when gate_up,
    which also applies out = silu(gate) * up; up_act="relu_sq": [E, N, K]
    up rows alone on gathered x rows, out = relu(.)^2). GPU only."""
    _moe_native().moe_gemm_plain(out, a, w, sorted_ids, expert_ids, n_valid,
                                 block_m, _moe_gemm_mode(gate_up, up_act),
                                 float(limit))
    return out


def moe_gemm_fp8(out, a, a_scales, b_packed, b_scales, sorted_ids,
                 expert_ids, n_valid, block_m: int, gate_up: bool):
    """Grouped fp8 (e4m3) GEMM with dequant epilogue: out[bf16] =
    (A_fp8 @ B_fp8) * a_scale[row] * b_scale[expert, col]; gate_up fuses
    SwiGLU. Same block-aligned layout as moe_gemm; b_packed from
    pack_moe_weights over the [E, K, N] e4m3 weights."""
    if out.is_cuda:
        _moe_native().moe_gemm_fp8(out, a, a_scales, b_packed, b_scales,
                                   sorted_ids, expert_ids, n_valid, block_m,
                                   gate_up)
        return out
    return ref.moe_gemm_fp8(out, a, a_scales, b_packed, b_scales,
                            sorted_ids, expert_ids, n_valid, block_m,
                            gate_up)


def moe_block_rows(assignments: int, experts: int, ff: int,
                   width: int) -> int:
    """Rows per block of the grouped bf16 GEMMs. Blocks of 16 stream the
    weights once per block, blocks of 128 are bound by the matrix cores at
    several times the work: they win as soon as experts take up two small
    blocks, if there are column tiles of 128 enough for every CU. gate_up +
    down with 16 / 128 rows, us: 128 experts of 2048 x 768, 8, 16, 24, 62
    rows each on average 200 / 268, 281 / 266, 405 / 266, 870 / 267; 8
    experts of 2048 x 3072, 16 and 32 rows 77 / 91, 120 / 92; 16 of 1536 x
    512, 16 and 32 rows 26 / 41, 40 / 41."""
    if assignments >= 64 * experts:
        return 128
    if width % 128 or ff % 64:
        return 16
    if experts * -(-ff // 128) >= 256:
        return 128 if assignments > 16 * experts else 16
    return 128 if assignments >= 32 * experts else 16


def moe_align(topi: torch.Tensor, e_start: int, e_end: int, block_m: int):
    """Device-side block alignment of expert assignments (GPU only;
    MoEMLP._moe_align's torch composition is the CPU reference and the
    semantic oracle): one launch up to 4096 assignments, two with scratch
    counts above. The order of the slots within an expert is unspecified and
    may differ from run to run; results do not depend on it (a row's K loop
    is the same in every slot, the combine gathers by pos). Returns
    (sorted_ids [PM], expert_ids [PM/bm], n_valid [1], pos [T*k], PM)."""
    C = _moe_native()
    T, k = topi.shape
    n = T * k
    E_local = e_end - e_start
    PM = ((n + block_m - 1) // block_m + E_local) * block_m
    dev = topi.device
    sorted_ids = torch.empty(PM, dtype=torch.int32, device=dev)
    expert_ids = torch.empty(PM // block_m, dtype=torch.int32, device=dev)
    n_valid = torch.empty(1, dtype=torch.int32, device=dev)
    pos = torch.empty(n, dtype=torch.int32, device=dev)
    C.moe_align(topi.reshape(-1).int().contiguous(), sorted_ids,
                expert_ids, n_valid, pos, k, e_start, e_end, block_m)
    return sorted_ids, expert_ids, n_valid, pos, PM


def moe_router_topk(logits: torch.Tensor, k: int, renorm: bool):
    """Fused router tail (GPU): softmax + top-k + optional top-k
    renormalization in one wave-per-token kernel. logits [T, E] fp32;
    returns (topv [T,k] fp32 weights, topi [T,k] int32 expert ids,
    descending; ties pick the smaller index)."""
    C = _moe_native()
    T, E = logits.shape
    topv = torch.empty(T, k, dtype=torch.float32, device=logits.device)
    topi = torch.empty(T, k, dtype=torch.int32, device=logits.device)
    C.moe_router_topk(logits.contiguous(), topv, topi, k, renorm)
    return topv, topi


ROUTER_ROWS = 512  # tokens up to which the router kernel forms the logits


def moe_router(x: torch.Tensor, w: torch.Tensor, k: int, renorm: bool):
    """Router on the GPU: softmax over x W^T (bf16 operands, fp32 sums),
    top-k, optional renormalization; results as moe_router_topk's. The
    product of two bf16 values is exact in fp32, so neither form converts
    its operands first. Up to ROUTER_ROWS tokens a small kernel forms the
    logits, above them the library's bf16 GEMM with fp32 results. Logits
    and choice of 8 of 128 experts, width 2048, with the kernel / the GEMM /
    the fp32 product with its conversions: 1 token 7.5 / 8.6 / 15 us, 64:
    9.4 / 9.0 / 16, 512: 9.6 / 9.0 / 19, 4096: 35 / 16 / 54 (every sixteen
    tokens read all of W through the caches). Where the two tie, a decode
    step's graph holds no GEMM that may clear its output first."""
    T, K = x.shape
    E = w.shape[0]
    if x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16 or T == 0:
        return moe_router_topk(x.float() @ w.float().T, k, renorm)
    if (T <= ROUTER_ROWS and E % 16 == 0 and K % 32 == 0
            and x.is_contiguous() and w.is_contiguous()
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0):
        logits = torch.empty(T, E, dtype=torch.float32, device=x.device)
        _moe_native().moe_router_logits(x, w, logits)
    else:
        logits = torch.mm(x, w.T, out_dtype=torch.float32)
    return moe_router_topk(logits, k, renorm)


def moe_route(logits: torch.Tensor, k: int, score: str = "softmax",
              renorm: bool = True, scale: float = 1.0):
    """Router tail for any expert count: scores = softmax(logits) or
    sigmoid(logits) in fp32, the k largest chosen (ties: smaller index),
    weights = chosen scores, divided by their sum + 1e-20 when ``renorm``,
    times ``scale``. Returns (weights [T,k] fp32, ids [T,k] int32)."""
    if score not in ("softmax", "sigmoid"):
        raise ValueError(f"unknown router score {score!r}")
    if logits.is_cuda:
        T, E = logits.shape
        topv = torch.empty(T, k, dtype=torch.float32, device=logits.device)
        topi = torch.empty(T, k, dtype=torch.int32, device=logits.device)
        _moe_native().moe_route(logits.contiguous(), topv, topi, k,
                                score == "sigmoid", renorm, float(scale))
        return topv, topi
    return ref.moe_route(logits, k, score, renorm, scale)


def moe_route_grouped(logits: torch.Tensor, correction: torch.Tensor,
                      k: int, groups: int = 1, keep: int = 1):
    """Group-limited router tail: s = sigmoid(logits) in fp32; the choice
    runs on s + correction, restricted to the experts of the ``keep`` best
    of ``groups`` equal groups of neighbouring experts (group score = sum
    of its two largest choice scores); weights = the chosen s, not
    renormalised. Returns (weights [T,k] fp32, ids [T,k] int32)."""
    E = logits.shape[1]
    if groups < 1 or E % groups or not 1 <= keep <= groups:
        raise ValueError("experts must split into equal groups, "
                         "1 <= keep <= groups")
    if k > keep * (E // groups):
        raise ValueError("top exceeds the experts of the kept groups")
    if logits.is_cuda:
        T = logits.shape[0]
        topv = torch.empty(T, k, dtype=torch.float32, device=logits.device)
        topi = torch.empty(T, k, dtype=torch.int32, device=logits.device)
        _moe_native().moe_route_grouped(logits.contiguous(), correction,
                                        topv, topi, k, groups, keep)
        return topv, topi
    return ref.moe_route_grouped(logits, correction, k, groups, keep)


def moe_route_corrected(logits: torch.Tensor, correction: torch.Tensor,
                        k: int, experts: int):
    """Router tail with a choice correction and identity experts: s =
    softmax(logits) in fp32 over all columns (``logits`` may be the leading
    columns of a wider row), the k largest s + correction chosen (ties:
    smaller index), weights = the chosen s, not renormalised. Ids from
    ``experts`` on are identity experts; their weights are summed per row.
    Returns (weights [T,k] fp32, ids [T,k] int32, identity weight [T])."""
    E = logits.shape[1]
    if not 1 <= k <= E or not 1 <= experts <= E:
        raise ValueError("top and experts must be within the router's rows")
    if logits.is_cuda:
        T = logits.shape[0]
        dev = logits.device
        topv = torch.empty(T, k, dtype=torch.float32, device=dev)
        topi = torch.empty(T, k, dtype=torch.int32, device=dev)
        idw = torch.empty(T, dtype=torch.float32, device=dev)
        _moe_native().moe_route_corrected(logits, correction, topv, topi,
                                          idw, k, experts)
        return topv, topi, idw
    return ref.moe_route_corrected(logits, correction, k, experts)


def moe_combine(out, y, pos, w):
    """out[t] = sum_k w[t,k] * y[pos[t,k]] (pos < 0 skipped). Deterministic
    (no atomics) so token-exact tests stay reproducible. bf16 or fp32
    rows of any width."""
    if out.is_cuda:
        _moe_native().moe_combine(out, y, pos, w)
        return out
    return ref.moe_combine(out, y, pos, w)


def moe_combine_norm(y, pos, w, residual, weight, eps: float):
    """residual += the rows of moe_combine and the norm behind that, in one
    pass: (rows, residual)."""
    T, H = residual.shape
    if (residual.dtype == y.dtype == weight.dtype == torch.bfloat16
            and H % 8 == 0 and H <= 8192 and len(y) > 0 and y.is_contiguous()
            and residual.is_contiguous() and weight.is_contiguous()
            and residual.is_cuda
            and (residual.data_ptr() | weight.data_ptr() | y.data_ptr()) % 16
            == 0):
        out = torch.empty_like(residual)
        _moe_native().moe_combine_norm(out, residual, weight, eps, y, pos, w)
        return out, residual
    out = torch.empty((T, H), dtype=y.dtype, device=y.device)
    return fused_add_rms_norm(moe_combine(out, y, pos, w), residual, weight,
                              eps)


compute_cos_sin_cache = ref.compute_cos_sin_cache
