"""Dense decoder-layer ops through the HIP library: projections at decode
batch sizes, RMSNorm with the residual sum, and the SwiGLU gate.

The reference runs these as torch in Python: ``FuseLayerNorm``
(microinfer/layer/norm.py:20-35; ``_compiled_add_rms_norm`` :13-16 when its
ops are compiled), the FFN's SwiGLU (``_compiled_swiglu``,
microinfer/layer/transformer.py:12-15, ``FFN.forward`` :82-88) and every
projection as ``F.linear``. Each function here is one HIP launch with the
same result up to float32 summation order; ``supported_*`` tell the caller
when a request is outside what the kernels take (32-bit tensors, unaligned
rows, more than 64 rows, or 4096 for ``hip_linear_fused`` without a norm) and
``prefer_*`` when the HIP projection is measured faster than torch's, so the
caller keeps torch for the rest.
"""

from __future__ import annotations

import torch

from microinfer_amd import _lib

_HALF = (torch.bfloat16, torch.float16)
LINEAR_MAX_ROWS = 64
FUSED_MAX_ROWS = 4096  # hip_linear_fused without a norm


def _rows_aligned(t: torch.Tensor) -> bool:
    es = t.element_size()
    return (t.dim() == 2 and t.stride(1) == 1 and t.data_ptr() % 16 == 0
            and (t.stride(0) * es) % 16 == 0)


def supported_linear(x: torch.Tensor, weight: torch.Tensor,
                     max_rows: int = LINEAR_MAX_ROWS) -> bool:
    return (x.is_cuda and x.dtype in _HALF and weight.dtype == x.dtype and x.dim() == 2
            and weight.dim() == 2 and 0 < x.shape[0] <= max_rows
            and x.shape[1] == weight.shape[1] and weight.shape[0] % 16 == 0
            and x.shape[1] % 32 == 0 and _rows_aligned(x) and _rows_aligned(weight))


def prefer_hip_linear(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether ``hip_linear`` beats torch's product for this request.

    Measured on MI355X (hipGraph-replayed, the Qwen3-0.6B projections, us per
    launch, HIP against hipBLASLt): at 64 rows QKV 4.5 / 8.5, output 4.3 /
    8.0, gate/up 8.0 / 11.9, down 4.7 / 9.7; at 8 rows 3.7 / 5.9, 3.8 /
    8.1, 5.3 / 8.0, 4.4 / 9.1. A vocabulary projection (more than 32768
    columns) goes to hipBLASLt past 32 rows, 40 where k is at most 2048
    (151936 x 1024 at 1 / 32 / 40 / 48 / 64 rows 52 / 72 / 78.5 / 80 / 107
    against 62 / 75 / 78.7 / 79 / 83; x 2048 at 32 / 40 / 48 rows 137 / 147 /
    151 against 149 / 152 / 146; x 4096 at 24 / 32 / 33 / 48 rows 243 / 258 /
    267 / 281 against 268 / 272 / 258 / 257)."""
    return supported_linear(x, weight) and _measured_faster(x.shape[0], weight)


def _measured_faster(rows: int, weight: torch.Tensor) -> bool:
    n, k = weight.shape
    return rows <= (40 if k <= 2048 else 32) or n <= 32768


def prefer_hip_rows(rows: int, weight: torch.Tensor) -> bool:
    """``prefer_hip_linear`` for aligned x of ``rows`` rows of weight's dtype."""
    return (0 < rows <= LINEAR_MAX_ROWS and weight.is_cuda and weight.dtype in _HALF
            and weight.dim() == 2 and weight.shape[0] % 16 == 0 and weight.shape[1] % 32 == 0
            and _rows_aligned(weight) and _measured_faster(rows, weight))


def prefer_hip_prefill(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether ``hip_linear_fused`` (no norm) beats torch's product past 64 rows.

    Prefill steps are launched eagerly, and a call takes half the host time of
    torch's (9 against 18 us), so the line follows whole steps of the engine
    (four chunks, us a step, HIP against hipBLASLt): 1024-wide layers, 28 of
    them on prefixes of 700, at 128 / 512 / 566 / 640 rows 2964 / 2970 / 3174 /
    3220 against 4320 / 4340 / 4379 / 4590, 8 of them on prefixes of 4000, where
    the device bounds the step, 1002 / 1197 / 1344 / 1372 against 1407 / 1413 /
    1435 / 1466, at 1024 rows 1552 against 1479; 2048-wide layers at 400 / 640
    rows without a prefix 2023 / 2110 against 2223 / 2188, on prefixes of 2000
    2137 / 2563 against 2107 / 2469.
    On the device alone the tiles of up to 512 rows win, the library's past
    that: 4096 x 1024 at 128 / 333 / 512 / 520 / 640 rows 6.1 / 10.1 / 10.6 /
    15.5 / 16.1 against 9.6 / 10.2 / 11.0 / 13.4 / 12.0, 1024 x 3072 6.6 / 10.5 /
    11.7 / 14.9 / 15.6 against 8.2 / 12.0 / 12.3 / 13.9 / 13.9, 6144 x 1024 with
    the gate 9.3 / 16.8 / 16.9 / 18.8 / 19.0 against 12.7 / 17.9 / 18.8 / 19.2 /
    19.8; weights of 2^23 elements from about 256 rows on (4096 x 2048 at 192 /
    333 / 640 rows 12.4 / 15.5 / 25.7 against 16.4 / 13.8 / 21.7). Larger ones
    are the library's: 6144 x 2048 at 128 / 333 / 640 rows 15.8 / 28.7 / 36.5
    against 15.6 / 24.9 / 25.8."""
    return (x.shape[0] <= 640 and weight.shape[0] * weight.shape[1] <= 1 << 23
            and supported_linear(x, weight, FUSED_MAX_ROWS))


def prefer_fused_norm(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether the norm in front of a preferred projection is better done
    inside it: every workgroup then scales the x rows it reads again, which
    past 16 rows and 2048 elements costs more than the norm's own launch (one
    launch against two, us: 24576 x 4096 at 33 rows 67 / 53, at 64 69 / 70;
    12288 x 2048 at 64 rows 23.4 / 26.3, 4096 x 1024 6.7 / 8.3), and with 33
    to 48 rows where the columns make more workgroups of 32 than there are CUs
    (at 33 / 48 rows 12288 x 1024 16.1 / 16.6 against 13.3 / 14.2, 16384 x
    2048 28 / 29 against 24 / 26; 8192 x 2048 15.4 / 15.9 against 18.4 / 19.2).
    float16 rows are normalised before they are scaled, a pass more: worth it
    up to 16 rows (4096 x 1024 at 1 / 16 / 17 / 64 rows 4.2 / 6.1 / 7.8 / 8.6
    against 6.1 / 6.9 / 7.3 / 7.7; 24576 x 4096 at 16 rows 43 against 44)."""
    rows, k = x.shape
    one = (rows <= 16 or (k <= 2048 and x.dtype != torch.float16
                          and not (32 < rows <= 48 and weight.shape[0] > 8192)))
    return one and prefer_hip_linear(x, weight)


def hip_linear(x: torch.Tensor, weight: torch.Tensor, *,
               out: torch.Tensor | None = None) -> torch.Tensor:
    """``F.linear(x, weight)`` for ``x [m <= 64, k]``, ``weight [n, k]``."""
    _lib.require_device(x, weight, out, what="dense projection")
    if not supported_linear(x, weight):
        raise ValueError("hip_linear: x [m <= 64, k] and weight [n % 16 == 0, k % 32 == 0] "
                         "of one 16-bit dtype with 16-byte aligned rows are required")
    m, k = x.shape
    n = weight.shape[0]
    if out is None:
        out = torch.empty((m, n), dtype=x.dtype, device=x.device)
    elif out.shape != (m, n) or out.dtype != x.dtype or not _rows_aligned(out):
        raise ValueError("hip_linear: out must be [m, n] of x's dtype with aligned rows")
    _lib.check(_lib.load().mi_linear(
        x.data_ptr(), x.stride(0), weight.data_ptr(), weight.stride(0), out.data_ptr(),
        out.stride(0), m, n, k, _lib.dtype_code(x.dtype), _lib.stream_handle(x.device)),
        "mi_linear")
    return out


def hip_linear_swiglu(x: torch.Tensor, gate_up: torch.Tensor, *,
                      out: torch.Tensor | None = None) -> torch.Tensor:
    """``F.silu(gate) * up`` of ``gate, up = F.linear(x, gate_up).chunk(2, -1)``
    (``FFN.forward``, transformer.py:82-88) in one launch: ``gate_up [2 I, k]``
    holds the gate's rows then the up projection's; the result ``[m, I]`` is
    ``hip_silu_mul(hip_linear(x, gate_up))`` bit for bit."""
    _lib.require_device(x, gate_up, out, what="gate/up projection")
    if not supported_linear(x, gate_up) or gate_up.shape[0] % 32:
        raise ValueError("hip_linear_swiglu: x [m <= 64, k] and gate_up [2 I, k] (I % 16 == 0, "
                         "k % 32 == 0) of one 16-bit dtype with 16-byte aligned rows are "
                         "required")
    m, k = x.shape
    inter = gate_up.shape[0] // 2
    if out is None:
        out = torch.empty((m, inter), dtype=x.dtype, device=x.device)
    elif out.shape != (m, inter) or out.dtype != x.dtype or not _rows_aligned(out):
        raise ValueError("hip_linear_swiglu: out must be [m, I] of x's dtype with aligned rows")
    _lib.check(_lib.load().mi_linear_swiglu(
        x.data_ptr(), x.stride(0), gate_up.data_ptr(), gate_up.stride(0), out.data_ptr(),
        out.stride(0), m, inter, k, _lib.dtype_code(x.dtype), _lib.stream_handle(x.device)),
        "mi_linear_swiglu")
    return out


def hip_linear_fused(x: torch.Tensor, weight: torch.Tensor, *,
                     norm_weight: torch.Tensor | None = None, eps: float = 0.0,
                     residual: torch.Tensor | None = None, swiglu: bool = False) -> torch.Tensor:
    """``residual + F.linear(rms_norm(x) * norm_weight, weight)`` in one launch,
    or with ``swiglu`` the gate ``silu(gate) * up`` of a ``[2 I, k]`` weight;
    ``norm_weight`` and ``residual`` are optional (``FuseLayerNorm.forward``,
    norm.py:26-35, around the projections of ``TransformerLayer.forward``,
    transformer.py:245-252). The roundings are those of the separate calls,
    except that with bf16 the norm's product is rounded once and its scale
    applied to the float32 sum."""
    _lib.require_device(x, weight, norm_weight, residual, what="fused projection")
    limit = FUSED_MAX_ROWS if norm_weight is None else LINEAR_MAX_ROWS
    if not supported_linear(x, weight, limit) or (swiglu and weight.shape[0] % 32):
        raise ValueError("hip_linear_fused: x [m <= 4096 (64 with a norm), k] and weight "
                         "[n % 16 == 0, k % 32 == 0] (gate/up: n % 32 == 0) of one 16-bit dtype "
                         "with 16-byte aligned rows are required")
    m, k = x.shape
    n = weight.shape[0]
    width = n // 2 if swiglu else n
    if norm_weight is not None and (norm_weight.shape != (k,) or norm_weight.dtype != x.dtype
                                    or not norm_weight.is_contiguous()
                                    or norm_weight.data_ptr() % 16):
        raise ValueError("hip_linear_fused: norm_weight must be an aligned [k] of x's dtype")
    if residual is not None and (residual.shape != (m, width) or residual.dtype != x.dtype
                                 or not _rows_aligned(residual)):
        raise ValueError("hip_linear_fused: residual must be [m, width] of x's dtype with "
                         "aligned rows")
    out = torch.empty((m, width), dtype=x.dtype, device=x.device)
    _lib.check(_lib.load().mi_linear_fused(
        x.data_ptr(), x.stride(0), 0 if norm_weight is None else norm_weight.data_ptr(),
        float(eps), weight.data_ptr(), weight.stride(0),
        0 if residual is None else residual.data_ptr(),
        0 if residual is None else residual.stride(0), out.data_ptr(), out.stride(0), m, n, k,
        int(swiglu), _lib.dtype_code(x.dtype), _lib.stream_handle(x.device)), "mi_linear_fused")
    return out


def supported_rows(*tensors: torch.Tensor) -> bool:
    """Whether the norm / SwiGLU kernels take these ``[rows, dim]`` tensors."""
    first = tensors[0]
    return all(t is None or (t.is_cuda and t.dtype == first.dtype and t.dtype in _HALF
                             and _rows_aligned(t)) for t in tensors)


def hip_rms_norm_residual(x: torch.Tensor, residual: torch.Tensor | None, weight: torch.Tensor,
                          eps: float) -> tuple[torch.Tensor, torch.Tensor]:
    """``FuseLayerNorm.forward`` (norm.py:26-35): returns
    ``(rms_norm(x + residual) * weight, x + residual)``; with no residual the
    sum is ``x`` itself (returned, not copied)."""
    _lib.require_device(x, residual, weight, what="RMSNorm")
    rows, dim = x.shape
    if not supported_rows(x, residual) or weight.dtype != x.dtype or weight.shape != (dim,) \
            or dim % 8 or dim > 8192 or weight.data_ptr() % 16:
        raise ValueError("hip_rms_norm_residual: 16-bit [rows, dim % 8 == 0] tensors with "
                         "aligned rows and a matching [dim] weight are required")
    out = torch.empty_like(x)
    combined = x if residual is None else torch.empty_like(x)
    _lib.check(_lib.load().mi_rms_norm_residual(
        x.data_ptr(), x.stride(0), 0 if residual is None else residual.data_ptr(),
        0 if residual is None else residual.stride(0), weight.data_ptr(), float(eps),
        out.data_ptr(), out.stride(0), 0 if residual is None else combined.data_ptr(),
        combined.stride(0), rows, dim, _lib.dtype_code(x.dtype),
        _lib.stream_handle(x.device)), "mi_rms_norm_residual")
    return out, combined


def hip_silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    """``F.silu(gate) * up`` with ``gate, up = gate_up.chunk(2, dim=-1)``
    (transformer.py:12-15)."""
    _lib.require_device(gate_up, what="SwiGLU")
    rows, width = gate_up.shape
    if not supported_rows(gate_up) or width % 16:
        raise ValueError("hip_silu_mul: a 16-bit [rows, 2 * inter] tensor with inter % 8 == 0 "
                         "and aligned rows is required")
    inter = width // 2
    out = torch.empty((rows, inter), dtype=gate_up.dtype, device=gate_up.device)
    _lib.check(_lib.load().mi_silu_mul(
        gate_up.data_ptr(), gate_up.stride(0), out.data_ptr(), out.stride(0), rows, inter,
        _lib.dtype_code(gate_up.dtype), _lib.stream_handle(gate_up.device)), "mi_silu_mul")
    return out
