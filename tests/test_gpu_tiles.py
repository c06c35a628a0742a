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
