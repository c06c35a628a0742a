"""The tiled multi-row GEMM at every tile shape its plan can pick, bf16 and 8-bit.

Bars: a store within one bf16 ulp of the float64 product (the fp32 sum of k
products carries at most k * 2^-24 relative to the sum of their magnitudes, far
below half an ulp of outputs of that size, except near zero, where the bound
is that sum); residual and SwiGLU outputs within the general bf16 bar; the
fused norm bit-identical to the row norm of the stored rows; argmax ids whose
logit lies within one bf16 ulp of the best.
"""
import pytest
import torch

from hackthenorth_amd.kernels import rows as RW
from hackthenorth_amd.kernels.rmsnorm import rms_norm
from hackthenorth_amd.quant import QuantizedWeight

pytestmark = pytest.mark.gpu
FORMATS = ["bf16", "int8", "fp8_e4m3"]
# Rows around the tiles' edges (16 to 256 rows), widths off the 128- and
# 256-row weight tiles and off the eight XCD columns, k of one step, of fewer
# steps than the staging ring and of several splits; the last seven take the
# 128- and 160-row tiles and the eight-wave ones of 128 to 256 rows.
CASES = [(2, 40, 64), (16, 136, 192), (17, 1000, 2560), (33, 136, 512), (48, 264, 1024),
         (49, 2568, 576), (65, 1032, 4096), (97, 520, 2048), (129, 2560, 1088),
         (160, 264, 9728), (201, 1544, 1024), (225, 5128, 640), (300, 6144, 1024),
         (513, 2560, 2048), (160, 12296, 512), (225, 12296, 640), (300, 12296, 640),
         (450, 8200, 1024), (500, 12288, 512), (700, 6152, 640), (1000, 6152, 640)]
# With these, every tile that the plan picks for bf16 and for 8-bit weights in
# each epilogue, with its k split and whole, its weights cached and streamed
# (tests/test_rows_routes.py looks them up).
COVER = [(523, 528, 64), (1353, 16, 1792), (2, 13688, 768), (2, 1992, 5312), (18, 5168, 2048),
         (34, 6848, 2112), (1227, 1032, 3840), (198, 14112, 6976), (1337, 5632, 64),
         (42, 22944, 704), (293, 1416, 8256), (1839, 1096, 9472), (17, 17000, 640),
         (653, 13320, 64), (696, 16504, 64), (67, 568, 3584), (397, 320, 6784), (884, 552, 7360),
         (1375, 4240, 64), (196, 2944, 3328), (17, 12296, 448), (235, 5448, 6784), (33, 11600, 64)]


def bf16(seed, *shape, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * std).to(torch.bfloat16)


def weight(fmt, n, k, seed):
    """(device weight, float64 values) of a random [n, k] projection."""
    w = bf16(seed, n, k, std=0.02)
    if fmt == "bf16":
        return w.cuda(), w.double()
    q = QuantizedWeight.quantize(w, fmt)
    codes = q.data.view(torch.int8 if fmt == "int8" else torch.float8_e4m3fn)
    values = codes.float().double() * q.scale.double()[:, None]
    return QuantizedWeight(q.data.cuda(), q.scale.cuda(), fmt), values


def gpu_operands(fmt, m, n, k, seed=20):
    """x [m, k] and a [2n, k] weight, made on the GPU: (x, weight, its first n
    rows, float64 values)."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    x = normal(m, k)
    if fmt == "bf16":
        w = normal(2 * n, k) * 0.02
        return x, w, w[:n], w.double()
    scale = torch.empty(2 * n, device="cuda").uniform_(0.8, 1.2, generator=g) * 0.02 / 30
    codes = normal(2 * n, k).float() * 30
    codes = codes.round().clamp(-127, 127).to(torch.int8) if fmt == "int8" \
        else codes.to(torch.float8_e4m3fn)
    data = codes.view(torch.uint8)
    return x, QuantizedWeight(data, scale, fmt), QuantizedWeight(data[:n], scale[:n], fmt), \
        codes.double() * scale.double()[:, None]


def check_store(got, x, values):
    x, values = x.double().cuda(), values.cuda()
    exact = x @ values.T
    slack = x.shape[1] * 2.0 ** -24 * (x.abs() @ values.abs().T)
    ulp = torch.pow(2.0, torch.floor(torch.log2(exact.abs().clamp_min(1e-30))) - 7)
    assert bool(((got.double() - exact).abs() <= ulp + slack).all())


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k", CASES)
def test_tiles_match_the_exact_product(fmt, m, n, k):
    x = bf16(1, m, k)
    xd, (w, values) = x.cuda(), weight(fmt, 2 * n, k, 2)
    half = QuantizedWeight(w.data[:n].contiguous(), w.scale[:n].contiguous(), fmt) \
        if fmt != "bf16" else w[:n].contiguous()
    check_store(RW._tiles(xd, half, n, RW._lib.EPI_STORE), x, values[:n])
    res, gain = bf16(3, m, n), bf16(4, n)
    out, normed = RW._tiles_residual_norm(xd, half, res.cuda(), gain.cuda(), 1e-6)
    y = (x.double().cuda() @ values.cuda().T).to(torch.bfloat16).cpu()
    torch.testing.assert_close(out.cpu().float(), (y[:, :n].float() + res.float()),
                               atol=2e-2, rtol=2e-2)
    if n <= 8192:  # the standalone norm takes rows of up to 8192 columns
        assert torch.equal(normed, rms_norm(out, gain.cuda(), 1e-6))
    gu = y.float()
    torch.testing.assert_close(RW._tiles(xd, w, n, RW._lib.EPI_SWIGLU).cpu().float(),
                               torch.nn.functional.silu(gu[:, :n]) * gu[:, n:],
                               atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k", COVER)
def test_every_tile_of_the_plan(fmt, m, n, k):
    x, w, half, values = gpu_operands(fmt, m, n, k)
    check_store(RW._tiles(x, half, n, RW._lib.EPI_STORE), x, values[:n])
    y = (x.double() @ values.T).to(torch.bfloat16).float()
    res, gain = bf16(21, m, n).cuda(), bf16(22, n).cuda()
    if n > 16384:  # past the row-wise norm's widest rows
        out = RW._tiles(x, half, n, RW._lib.EPI_RESIDUAL, residual=res)
    else:
        out, normed = RW._tiles_residual_norm(x, half, res, gain, 1e-6)
        if n <= 8192:
            assert torch.equal(normed, rms_norm(out, gain, 1e-6))
    torch.testing.assert_close(out.float(), y[:, :n] + res.float(), atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(RW._tiles(x, w, n, RW._lib.EPI_SWIGLU).float(),
                               torch.nn.functional.silu(y[:, :n]) * y[:, n:],
                               atol=2e-2, rtol=2e-2)


# Rows and widths on tiles of 16, 32, 48, 64, 96, 128, 160, 224 and 256 rows.
FORM_CASES = [(3, 137, 1088), (20, 1001, 4096), (40, 1003, 4096), (70, 2050, 2560), (97, 522, 2048),
              (129, 2563, 1088), (201, 1541, 1024), (198, 14113, 512), (653, 13321, 64),
              (696, 16505, 64), (235, 5449, 6784), (884, 553, 7360)]


def tiles_abi(fmt, x, w, n, epilogue, residual=None, y_stride=None, y_offset=0, split=True):
    """The C entry on rows of any stride; y [m, n] of stride `y_stride` from
    `y_offset` elements into a NaN buffer, of which nothing else may change."""
    lib, (m, k) = RW._lib, x.shape
    data, scale, code = RW._weight(w)
    nbytes = lib.load().htn_gemm_tiles_w8_scratch_bytes(m, n, k, epilogue, code) if split else 0
    scratch = torch.full((nbytes // 4 + 4,), float("nan"), device="cuda") if nbytes else None
    stride = n if y_stride is None else y_stride
    buffer = torch.full((m * stride + y_offset + 8,), float("nan"), dtype=torch.bfloat16,
                        device="cuda")
    y = buffer[y_offset:y_offset + m * stride].view(m, stride)
    head = (lib.ptr(x), x.stride(0), lib.ptr(data))
    tail = (n, k, m, epilogue, lib.ptr(residual), residual.stride(0) if residual is not None else 0,
            lib.ptr(y), stride)
    if code:
        lib.call("htn_gemm_tiles_w8", *head, lib.ptr(scale), code, *tail, None, lib.ptr(scratch),
                 lib.stream(x.device))
    else:
        lib.call("htn_gemm_tiles", *head, *tail, lib.ptr(scratch), lib.stream(x.device))
    assert bool(buffer[:y_offset].isnan().all()) and bool(y[:, n:].isnan().all()) \
        and bool(buffer[y_offset + m * stride:].isnan().all())
    return y[:, :n]


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("m,n,k", FORM_CASES)
def test_tiles_take_any_row_stride_and_odd_widths(fmt, split, m, n, k):
    """Padded input rows, residual rows and outputs; widths off the four columns
    of a lane; for 8-bit weights outputs of odd strides at odd addresses; with
    scratch and without (each tile's k range whole)."""
    x, w, half, values = gpu_operands(fmt, m, n, k)
    wide = torch.full((m, k + 8), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide[:, :k] = x
    padded = torch.zeros(m, n + 3, dtype=torch.bfloat16, device="cuda")
    padded[:, :n] = bf16(23, m, n).cuda()
    res = padded[:, :n]
    stride, offset = (n + (-n) % 4, 0) if fmt == "bf16" else (n + 2 + n % 2, 1)
    y = (x.double() @ values.T).to(torch.bfloat16).float()
    form = dict(y_stride=stride, y_offset=offset, split=split)
    check_store(tiles_abi(fmt, wide[:, :k], half, n, RW._lib.EPI_STORE, **form), x, values[:n])
    torch.testing.assert_close(
        tiles_abi(fmt, wide[:, :k], half, n, RW._lib.EPI_RESIDUAL, res, **form).float(),
        y[:, :n] + res.float(), atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(
        tiles_abi(fmt, wide[:, :k], w, n, RW._lib.EPI_SWIGLU, **form).float(),
        torch.nn.functional.silu(y[:, :n]) * y[:, n:], atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k", [(5, 264, 2048), (40, 1000, 512), (129, 520, 2048), (201, 14112, 512),
                                   (300, 12296, 640)])
def test_tiles_keep_nonfinite_values_to_their_rows_and_columns(fmt, m, n, k):
    """Rows of x with an infinity or a NaN and weight rows with one (8-bit: an
    fp8 NaN code, an infinite scale) give what the product gives, and every
    other output stays finite."""
    x, _, half, values = gpu_operands(fmt, m, n, k)
    values = values[:n].clone()
    x[1, k // 2], x[m - 1, 3] = float("inf"), float("nan")
    if fmt == "bf16":
        half[n // 2, 7] = float("-inf")
        values[n // 2, 7] = float("-inf")
    elif fmt == "fp8_e4m3":
        half.data[n // 2, 7] = 0x7F
        values[n // 2, 7] = float("nan")
    exact = x.double() @ values.T
    if fmt == "int8":
        half.scale[n // 2] = float("inf")
        exact[:, n // 2] *= float("inf")
    got = RW._tiles(x, half, n, RW._lib.EPI_STORE).double()
    assert torch.equal(got.isnan(), exact.isnan()) and torch.equal(got.isposinf(), exact.isposinf())
    assert torch.equal(got.isneginf(), exact.isneginf())
    finite = exact.isfinite()
    assert int((~finite).sum()) <= 2 * n + m
    torch.testing.assert_close(got[finite], exact[finite], atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("fmt", FORMATS[1:])
@pytest.mark.parametrize("m,n,k", [(2, 136, 256), (16, 40, 64), (17, 3000, 1024), (32, 520, 512),
                                   (70, 1000, 256)])
def test_argmax_tiles_pick_the_best_row(fmt, m, n, k):
    x = bf16(5, m, k)
    w, values = weight(fmt, n, k, 6)
    got = RW.greedy_rows(x.cuda(), w).cpu()
    logits = x.double() @ values.T
    best = logits.max(dim=1).values
    ulp = torch.pow(2.0, torch.floor(torch.log2(best.abs().clamp_min(1e-30))) - 7)
    assert bool((best - logits.gather(1, got[:, None])[:, 0] <= ulp).all())


@pytest.mark.parametrize("fmt", FORMATS[1:])
def test_argmax_tiles_ties_choose_the_lowest_id(fmt):
    w = torch.zeros(500, 128)
    w[[7, 130, 499]] = 1.0
    q = QuantizedWeight.quantize(w, fmt)
    q = QuantizedWeight(q.data.cuda(), torch.ones(500, device="cuda"), fmt)
    assert RW.greedy_rows(torch.ones(3, 128, dtype=torch.bfloat16, device="cuda"), q).tolist() \
        == [7, 7, 7]


@pytest.mark.parametrize("fmt", FORMATS)
def test_tiles_replay_in_a_graph(fmt):
    """A captured split launch and its finish replay to the eager bits."""
    m, n, k = 40, 512, 4096
    x, (w, _) = bf16(7, m, k).cuda(), weight(fmt, n, k, 8)
    res, gain = bf16(9, m, n).cuda(), bf16(10, n).cuda()
    with torch.inference_mode():
        eager = RW._tiles_residual_norm(x, w, res, gain, 1e-6)
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = RW._tiles_residual_norm(x, w, res, gain, 1e-6)
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out[0], eager[0]) and torch.equal(out[1], eager[1])
            RW._tiles_residual_norm(x, w, res, gain, 1e-6)


@pytest.mark.parametrize("m,v", [(2, 16), (3, 2000), (5, 16400), (8, 150000)])
def test_strip_argmax_over_few_and_many_strips(m, v):
    """The strips' per-row finish: one strip, under and over 1024 strips (one
    key per thread), over 8192 (a thread's second round)."""
    x, w = bf16(11, m, 64).cuda(), bf16(12, v, 64).cuda()
    got = RW.greedy_rows(x, w)
    logits = x.double() @ w.double().T
    best = logits.max(dim=1).values
    ulp = torch.pow(2.0, torch.floor(torch.log2(best.abs())) - 7)
    assert bool((best - logits.gather(1, got[:, None])[:, 0] <= ulp).all())
