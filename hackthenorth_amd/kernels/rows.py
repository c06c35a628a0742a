"""Projections of two or more rows that read each weight once (MFMA tiles).

The speculative verify pass scores k + 1 tokens in one forward; the reference
runs its multi-row projections as Triton GEMM tiles (dryft/engine/
projections.py:168-183, kernels/gateup.py:40-58, kernels/split_down.py:85-101).
Here few rows (strip_rows) are one htn_gemm_rows launch (16-column strips, the
RMSNorm inside, plus a K-split reduction when the strips alone cannot fill the
GPU) and more rows one htn_gemm_tiles launch (LDS-staged output tiles, plus the
finish of its k split), with the batch-one GEMVs' bf16 rounding boundaries.
In a prompt's prefill the plain product of the gate/up projection from
TILE_ROWS rows on, of a plain store from LIBRARY_ROWS rows on and of a residual
projection with the next norm past them runs through hipBLASLt
(htn_gemm_library) with the epilogues as row-wise launches, where the library
has an algorithm. 8-bit weights (QuantizedWeight) take htn_gemm_tiles_w8 at
every row count.
"""
import torch

from .. import _lib
from ..quant import QuantizedWeight
from .greedy import greedy_head

MAX_ROWS = 128    # rows per htn_gemm_rows launch
# Bytes from which a bf16 vocabulary is streamed past the caches, one row of it
# as the batch-one head. 33 MB from HBM, a row without the norm: 12.1 us on the
# strips, 10.2 on the head (8.7 / 10.6 where the last pass left all of it cached,
# which a whole model's other weights do not).
STREAM_HEAD_BYTES = 16 << 20
ARGMAX_ROWS = 32  # rows per 8-bit head launch (HTN_GEMM_TILES_ARGMAX_ROWS)
TILE_ROWS = 256
# A plain store (QKV) of LIBRARY_ROWS rows goes to the library, a residual
# projection with the next norm past them, or past WIDE_ROWS where it is wider
# than deep; a residual projection alone stays on the tiles at any count. 8B at
# 300 rows QKV 32 us on the tiles and 30 through the library, O with its norm 29
# and 35, down 59 and 78; at 512 rows 44 / 38, 35 / 39, 79 / 90; at 2048 the
# library wins throughout (QKV 85 us against 137). A short k leaves the tiles'
# finish a larger share: [5120, 1024] 300 rows 23.4 / 23.2, 512 33.1 / 26.6;
# [4096, 2048] 24.5 / 24.6 and 30.1 / 27.0; but the 0.6B with its O ([1024,
# 2048]) on the tiles 259 us of 512 rows for three layers, through the library 264.
LIBRARY_ROWS, WIDE_ROWS = 512, 320
# Plain products of TILE_ROWS rows or more through hipBLASLt (False: this
# library's tiled kernel for every prompt projection, e.g. to measure it).
LIBRARY = True


def _normed(x, gain, eps):
    """The rows' RMSNorm with `gain` (one row-norm launch), or x without one."""
    if gain is None:
        return x
    rows, k = x.shape
    xn = torch.empty((rows, k), dtype=x.dtype, device=x.device)
    _lib.call("htn_rms_norm", _lib.ptr(x), x.stride(0), _lib.ptr(gain), _lib.ptr(xn), rows, k,
              float(eps), _lib.stream(x.device))
    return xn


def _library(x, weight, width):
    """bf16(x W^T) for every row through hipBLASLt (htn_gemm_library), or
    None when the library has no algorithm for the shape."""
    if not LIBRARY:
        return None
    rows, k = x.shape
    lib = _lib.load()
    out = torch.empty((rows, width), dtype=x.dtype, device=x.device)
    workspace = torch.empty(lib.htn_gemm_library_workspace_bytes() // 16, 4, dtype=torch.float32,
                            device=x.device)
    rc = lib.htn_gemm_library(_lib.ptr(x), x.stride(0), _lib.ptr(weight), width, k, rows,
                              _lib.ptr(out), out.stride(0), _lib.ptr(workspace),
                              _lib.stream(x.device))
    if rc == _lib.HTN_EUNSUPPORTED:
        return None
    _lib.check(rc, "htn_gemm_library")
    return out


def _prefill(x, weight, n, epilogue, gain=None, eps=1e-6):
    """Store or SwiGLU epilogue over every row of a prompt: the plain product
    through the library, SwiGLU as a row-wise launch; the tiled kernel below
    LIBRARY_ROWS rows of a store and when the library declines the shape."""
    xn = _normed(x, gain, eps)
    width = 2 * n if epilogue == _lib.EPI_SWIGLU else n
    y = _library(xn, weight, width) \
        if epilogue != _lib.EPI_STORE or x.shape[0] >= LIBRARY_ROWS else None
    if y is None:
        return _tiles(xn, weight, n, epilogue)
    if epilogue == _lib.EPI_STORE:
        return y
    rows = x.shape[0]
    out = torch.empty((rows, n), dtype=x.dtype, device=x.device)
    _lib.call("htn_swiglu", _lib.ptr(y), y.stride(0), _lib.ptr(y[:, n:]), y.stride(0),
              _lib.ptr(out), rows, n, _lib.stream(x.device))
    return out


def _weight(weight):
    """(bytes, row scales or None, format code) of a bf16 or 8-bit weight."""
    if isinstance(weight, QuantizedWeight):
        return weight.data, weight.scale, weight.code
    return weight, None, 0


def prompt(x, weight):
    """Whether the library may take part: bf16 projections of TILE_ROWS rows or more."""
    return x.shape[0] >= TILE_ROWS and not isinstance(weight, QuantizedWeight)


def _tiles_scratch(device, rows, n, k, epilogue, fmt):
    nbytes = _lib.load().htn_gemm_tiles_w8_scratch_bytes(rows, n, k, epilogue, fmt)
    return torch.empty((nbytes + 15) // 16, 4, dtype=torch.float32, device=device) \
        if nbytes > 0 else None


def _tiles(x, weight, n, epilogue, residual=None, gain=None, eps=1e-6):
    """One tiled launch over every row of x (after the rows' RMSNorm with
    `gain`, when given); returns the [M, n] output."""
    rows, k = x.shape
    x = _normed(x, gain, eps)
    data, scale, fmt = _weight(weight)
    out = torch.empty((rows, n), dtype=x.dtype, device=x.device)
    scratch = _tiles_scratch(x.device, rows, n, k, epilogue, fmt)
    tail = (n, k, rows, epilogue, _lib.ptr(residual),
            residual.stride(0) if residual is not None else 0, _lib.ptr(out), out.stride(0))
    if fmt:
        _lib.call("htn_gemm_tiles_w8", _lib.ptr(x), x.stride(0), _lib.ptr(data), _lib.ptr(scale),
                  fmt, *tail, None, _lib.ptr(scratch), _lib.stream(x.device))
    else:
        _lib.call("htn_gemm_tiles", _lib.ptr(x), x.stride(0), _lib.ptr(data), *tail,
                  _lib.ptr(scratch), _lib.stream(x.device))
    return out


def _tiles_residual_norm(x, weight, residual, gain, eps):
    """(out, normed) of a residual projection and the next RMSNorm: one launch
    and, when the tiles split k, its finish, which writes both."""
    rows, k = x.shape
    n = weight.shape[0]
    data, scale, fmt = _weight(weight)
    out = torch.empty((rows, n), dtype=x.dtype, device=x.device)
    normed = torch.empty_like(out)
    scratch = _tiles_scratch(x.device, rows, n, k, _lib.EPI_RESIDUAL, fmt)
    _lib.call("htn_gemm_tiles_residual_norm", _lib.ptr(x), x.stride(0), _lib.ptr(data),
              _lib.ptr(scale), fmt, n, k, rows, _lib.ptr(residual), residual.stride(0),
              _lib.ptr(out), out.stride(0), _lib.ptr(gain), float(eps), _lib.ptr(normed),
              _lib.ptr(scratch), _lib.stream(x.device))
    return out, normed


def strip_rows(n, k, swiglu=False, norm=False):
    """Rows up to which a bf16 [n, k] projection takes the strips (swiglu: n
    counts the gate and up rows; norm: with the input rows' RMSNorm).

    A strip re-reads its rows' x per 16 columns, so its time grows with rows and
    k (17, 33 and 65 rows begin another row tile), while the tiles pay a second
    launch for their k split and one for a norm first. Strips / tiles in us,
    weights from HBM:
    [4096, 1024] 64 rows 7.3 / 8.1; [2048, 2048] 32 rows 7.6 / 9.0, 48 9.8 / 9.1;
    [4096, 2048] 32 rows 8.0 / 9.3; [6144, 2560] 16 rows 11.7 / 11.8, 24 13.8 /
    12.2; [24576, 4096] 16 rows 32.8 / 32.5, 17 39.0 / 33.0. SwiGLU of few
    columns: [6144, 2048] 24 rows 12.0 / 14.8. Past k = 4096 they cross by 12
    rows ([2560, 9728] 8 rows 13.7 / 15.2, 12 15.8 / 15.3; [5120, 5120] 8 rows 15
    / 14), but not where whole rounds of strips fill the CUs ([4096, 12288] 16
    rows 23.8 / 28.1) nor with a norm in the strips' launch ([2048, 6144] 16
    rows 16.8 / 18.6)."""
    if k <= 1024 and n * k <= 5 << 20:
        return 64
    if k <= 3072 and n * k < 12 << 20 or swiglu and n <= 8192 and k <= 5120:
        return 32
    if k <= 4096 or n % 4096 == 0 or norm and n * k < 20 << 20:
        return 16
    return 12 if k <= 8192 else 8


def norm_strip_rows(n, k):
    """strip_rows of a residual projection whose rows the next projection
    normalises: on the strips in that one's launch, at its expense, on the tiles
    in this one's finish. Both together, strips / tiles, 12 rows: 4B O and gate/up
    33.5 / 31.9, down and QKV 29.3 / 27.0, 8 rows 31.2 / 31.3 and 25.6 / 25.2; 8B
    44.3 / 45.5 and 39.8 / 43.5, 16 rows 47.1 / 46.7 and 44.3 / 44.1; a 2048-wide
    model's down and QKV 19.1 / 19.6."""
    return 8 if n * k >= 10 << 20 and n > 2048 and n % 4096 else strip_rows(n, k)


def _tileable(x, weight):
    """Rows and output widths that the tiles' 8-byte stores and 32-bit offsets
    cover; not rows that overlap (an expanded row, sliding windows), which the
    strips read."""
    return weight.shape[0] % 8 == 0 and x.shape[1] <= x.stride(0) < 1 << 22


def tiled(x, weight, swiglu=False, norm=False):
    """Whether a projection of these rows (strip_rows) takes the tiles: 8-bit weights always,
    bf16 ones past the strips' rows; TILE_ROWS rows or more have no other kernel."""
    if isinstance(weight, QuantizedWeight) or x.shape[0] >= TILE_ROWS:
        return True
    return x.shape[0] > strip_rows(*weight.shape, swiglu, norm) and _tileable(x, weight)


def norm_tiled(x, weight, residual):
    """Whether a residual projection with the next RMSNorm takes the tiles: of
    a prompt's rows up to LIBRARY_ROWS (WIDE_ROWS where n > k), and there not
    those of which the library's product and the row-wise residual add take more: widths off the
    64-wide k steps, residual rows that overlap, far strides."""
    if isinstance(weight, QuantizedWeight):
        return True
    n, k = weight.shape
    if not prompt(x, weight):
        return x.shape[0] > norm_strip_rows(n, k) and _tileable(x, weight)
    return x.shape[0] <= (LIBRARY_ROWS if k >= n else WIDE_ROWS) and k % 64 == 0 \
        and residual.stride(0) >= n and x.stride(0) < 1 << 22


def writes_norm(x, weight, residual):
    """Whether a layer's residual projection is to write the next RMSNorm too
    (residual_norm_rows): on the tiles and after the library's product."""
    return prompt(x, weight) or norm_tiled(x, weight, residual)


def _scratch(device, rows, n, k, epilogue, norm):
    nbytes = _lib.load().htn_gemm_rows_scratch_bytes(rows, n, k, epilogue, int(norm))
    if nbytes <= 0:
        return None
    return torch.empty((nbytes + 7) // 8, dtype=torch.int64, device=device)


def _check(x, weight):
    if x.dim() != 2 or x.dtype != torch.bfloat16 or x.stride(1) != 1:
        raise ValueError("rows must be a bf16 [M, K] matrix with unit column stride")
    if isinstance(weight, QuantizedWeight):
        if weight.shape[1] != x.shape[1]:
            raise ValueError("weight must be an 8-bit [N, K] matrix matching x")
        return
    if weight.dim() != 2 or weight.dtype != torch.bfloat16 or not weight.is_contiguous() \
            or weight.shape[1] != x.shape[1]:
        raise ValueError("weight must be a contiguous bf16 [N, K] matrix matching x")


def _launch(x, weight, n, epilogue, gain=None, eps=1e-6, residual=None, out=None, tokens=None):
    rows, k = x.shape
    scratch = _scratch(x.device, rows, n, k, epilogue, gain is not None)
    _lib.call("htn_gemm_rows", _lib.ptr(x), x.stride(0), _lib.ptr(gain), float(eps),
              _lib.ptr(weight), n, k, rows, epilogue, _lib.ptr(residual),
              residual.stride(0) if residual is not None else 0, _lib.ptr(out),
              out.stride(0) if out is not None else 0, _lib.ptr(tokens), _lib.ptr(scratch),
              _lib.stream(x.device))


def _chunks(rows):
    return [(s, min(rows, s + MAX_ROWS)) for s in range(0, rows, MAX_ROWS)]


def projection_rows(x, weight, gain=None, eps=1e-6):
    """bf16(W x_m) for every row m of x [M, K]; gain applies RMSNorm first."""
    _check(x, weight)
    _lib.require_gpu(x, _weight(weight)[0], gain)
    if tiled(x, weight, norm=gain is not None):
        run = _prefill if prompt(x, weight) else _tiles
        return run(x, weight, weight.shape[0], _lib.EPI_STORE, gain=gain, eps=eps)
    out = torch.empty((x.shape[0], weight.shape[0]), dtype=x.dtype, device=x.device)
    for s, e in _chunks(x.shape[0]):
        _launch(x[s:e], weight, weight.shape[0], _lib.EPI_STORE, gain, eps, out=out[s:e])
    return out


def residual_rows(x, weight, residual):
    """bf16(bf16(W x_m) + residual_m) for every row (O and down projections)."""
    _check(x, weight)
    if residual.shape != (x.shape[0], weight.shape[0]) or residual.dtype != torch.bfloat16 \
            or residual.stride(1) != 1:
        raise ValueError("residual must be bf16 [M, N] with unit column stride")
    _lib.require_gpu(x, _weight(weight)[0], residual)
    if tiled(x, weight):
        return _tiles(x, weight, weight.shape[0], _lib.EPI_RESIDUAL, residual=residual)
    out = torch.empty((x.shape[0], weight.shape[0]), dtype=x.dtype, device=x.device)
    for s, e in _chunks(x.shape[0]):
        _launch(x[s:e], weight, weight.shape[0], _lib.EPI_RESIDUAL, residual=residual[s:e],
                out=out[s:e])
    return out


def residual_norm_rows(x, weight, residual, gain, eps=1e-6):
    """(out, normed): out = residual_rows(x, weight, residual) and normed its
    RMSNorm with `gain` (the next layer's input), written by the finish of a
    projection that splits K, by the residual add of the library's, else by a
    launch of its own."""
    _check(x, weight)
    n = weight.shape[0]
    if residual.shape != (x.shape[0], n) or residual.dtype != torch.bfloat16 \
            or residual.stride(1) != 1:
        raise ValueError("residual must be bf16 [M, N] with unit column stride")
    if gain is None or gain.shape != (n,) or gain.dtype != torch.bfloat16 \
            or not gain.is_contiguous():
        raise ValueError("gain must be a contiguous bf16 [N] vector")
    _lib.require_gpu(x, _weight(weight)[0], residual, gain)
    if norm_tiled(x, weight, residual):
        return _tiles_residual_norm(x, weight, residual, gain, eps)
    if x.shape[0] >= TILE_ROWS:
        rows = x.shape[0]
        y = _library(x, weight, n)
        if y is None:
            out = _tiles(x, weight, n, _lib.EPI_RESIDUAL, residual=residual)
            normed = torch.empty_like(out)
            _lib.call("htn_rms_norm", _lib.ptr(out), out.stride(0), _lib.ptr(gain),
                      _lib.ptr(normed), rows, n, float(eps), _lib.stream(x.device))
            return out, normed
        # bf16(bf16(y) + residual) and its RMSNorm in one row-wise launch.
        if not residual.is_contiguous():
            residual = residual.contiguous()
        out = torch.empty((rows, n), dtype=x.dtype, device=x.device)
        normed = torch.empty_like(out)
        _lib.call("htn_add_rms_norm", _lib.ptr(y), _lib.ptr(residual), _lib.ptr(gain),
                  _lib.ptr(out), _lib.ptr(normed), rows, n, float(eps), _lib.stream(x.device))
        return out, normed
    out = torch.empty((x.shape[0], n), dtype=x.dtype, device=x.device)
    normed = torch.empty_like(out)
    for s, e in _chunks(x.shape[0]):
        rows, k = x[s:e].shape
        scratch = _scratch(x.device, rows, n, k, _lib.EPI_RESIDUAL_NORM, False)
        _lib.call("htn_gemm_rows_residual_norm", _lib.ptr(x[s:e]), x.stride(0),
                  _lib.ptr(weight), n, k, rows, _lib.ptr(residual[s:e]), residual.stride(0),
                  _lib.ptr(out[s:e]), out.stride(0), _lib.ptr(gain), float(eps),
                  _lib.ptr(normed[s:e]), _lib.ptr(scratch), _lib.stream(x.device))
    return out, normed


def swiglu_rows(x, gate_up_weight, gain=None, eps=1e-6):
    """SwiGLU of the packed gate/up projection ([2I, K]: gate rows, then up rows)."""
    _check(x, gate_up_weight)
    if gate_up_weight.shape[0] % 2:
        raise ValueError("packed gate/up width must be even")
    _lib.require_gpu(x, _weight(gate_up_weight)[0], gain)
    n = gate_up_weight.shape[0] // 2
    if tiled(x, gate_up_weight, True, gain is not None):
        run = _prefill if prompt(x, gate_up_weight) else _tiles
        return run(x, gate_up_weight, n, _lib.EPI_SWIGLU, gain=gain, eps=eps)
    out = torch.empty((x.shape[0], n), dtype=x.dtype, device=x.device)
    for s, e in _chunks(x.shape[0]):
        _launch(x[s:e], gate_up_weight, n, _lib.EPI_SWIGLU, gain, eps, out=out[s:e])
    return out


def streams_head(weight):
    """Whether one row against this vocabulary takes the batch-one head without
    a norm to share its launch: 8-bit ones and bf16 ones of STREAM_HEAD_BYTES."""
    return isinstance(weight, QuantizedWeight) or 2 * weight.numel() >= STREAM_HEAD_BYTES


def greedy_rows(x, weight, gain=None, eps=1e-6):
    """argmax_n bf16(W x_m) per row (lowest id on ties); gain applies RMSNorm first."""
    _check(x, weight)
    _lib.require_gpu(x, _weight(weight)[0], gain)
    tokens = torch.empty((x.shape[0],), dtype=torch.int64, device=x.device)
    if x.shape[0] == 1 and x.is_contiguous() and (gain is not None or streams_head(weight)):
        # The batch-one head normalises in its launch and streams the weight
        # with nothing else to do (8B: 182 us against 220).
        return greedy_head(x, gain, eps, weight, tokens)
    if isinstance(weight, QuantizedWeight):
        xn = _normed(x, gain, eps)
        n, k = weight.shape
        for s in range(0, x.shape[0], ARGMAX_ROWS):
            part = xn[s:s + ARGMAX_ROWS]
            rows = part.shape[0]
            scratch = _tiles_scratch(x.device, rows, n, k, _lib.EPI_ARGMAX, weight.code)
            _lib.call("htn_gemm_tiles_w8", _lib.ptr(part), part.stride(0), _lib.ptr(weight.data),
                      _lib.ptr(weight.scale), weight.code, n, k, rows, _lib.EPI_ARGMAX, None, 0,
                      None, 0, _lib.ptr(tokens[s:]), _lib.ptr(scratch), _lib.stream(x.device))
        return tokens
    for s, e in _chunks(x.shape[0]):
        _launch(x[s:e], weight, weight.shape[0], _lib.EPI_ARGMAX, gain, eps,
                tokens=tokens[s:e])
    return tokens
