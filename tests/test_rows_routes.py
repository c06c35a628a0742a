"""Which kernel the multi-row projections take for rows of unusual strides and
widths: what the strips and the library accept is not sent to the tiles, which
refuse it. The routes are looked up on the CPU, the results compared on the GPU."""
import ctypes
import random

import pytest
import torch

from hackthenorth_amd import _lib
from hackthenorth_amd.kernels import rows as RW
from hackthenorth_amd.kernels.rmsnorm import rms_norm
from test_gpu_tiles import CASES, COVER


def matrix(rows, cols, layout, device="cpu", seed=0):
    """bf16 [rows, cols]: contiguous, padded rows, one row expanded, or windows
    that slide by eight elements."""
    g = torch.Generator().manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g).to(torch.bfloat16).to(device)
    if layout == "expanded":
        return normal(1, cols).expand(rows, cols)
    if layout == "windows":
        return normal(8 * rows + cols).as_strided((rows, cols), (8, 1))
    if layout == "padded":
        return normal(rows, cols + 24)[:, :cols]
    return normal(rows, cols)


# The projections of models 1024, 2048, 2560, 4096 and 5120 wide: the last row
# count on the strips, without and with an input norm, and for residual
# projections with the next norm.
@pytest.mark.parametrize("n,k,swiglu,plain,with_input_norm,with_next_norm", [
    (4096, 1024, False, 64, 64, None), (1024, 2048, False, 32, 32, 32),
    (6144, 1024, True, 32, 32, None), (1024, 3072, False, 32, 32, 32),
    (4096, 2048, False, 32, 32, None), (2048, 2048, False, 32, 32, 32),
    (12288, 2048, True, 16, 16, None), (2048, 6144, False, 12, 16, 12),
    (6144, 2560, False, 16, 16, None), (2560, 4096, False, 16, 16, 8),
    (19456, 2560, True, 16, 16, None), (2560, 9728, False, 8, 8, 8),
    (6144, 4096, False, 16, 16, None), (4096, 4096, False, 16, 16, 16),
    (24576, 4096, True, 16, 16, None), (4096, 12288, False, 16, 16, 16),
    (7168, 5120, False, 12, 12, None), (5120, 5120, False, 12, 12, 8),
    (5120, 17408, False, 8, 8, 8), (6144, 2048, True, 32, 32, None)])
def test_strips_end_by_weight_size(n, k, swiglu, plain, with_input_norm, with_next_norm):
    w = torch.empty(n, k, dtype=torch.bfloat16, device="meta")
    for last, norm in ((plain, False), (with_input_norm, True)):
        for rows in (last, last + 1):
            x = torch.empty(rows, k, device="meta")
            assert RW.tiled(x, w, swiglu, norm) == (rows > last)
    for rows in (with_next_norm, with_next_norm + 1) if with_next_norm else ():
        x, res = torch.empty(rows, k, device="meta"), torch.empty(rows, n, device="meta")
        assert RW.norm_tiled(x, w, res) == RW.writes_norm(x, w, res) == (rows > with_next_norm)


@pytest.mark.parametrize("n,k,last", [(4096, 4096, 512), (1024, 2048, 512), (2048, 1024, 320)])
def test_residual_norm_goes_to_the_library_by_rows_and_shape(n, k, last):
    w = torch.empty(n, k, dtype=torch.bfloat16, device="meta")
    for rows in (256, last, last + 1):
        x, res = torch.empty(rows, k, device="meta"), torch.empty(rows, n, device="meta")
        assert RW.norm_tiled(x, w, res) == (rows <= last) and RW.writes_norm(x, w, res)


@pytest.mark.parametrize("rows,n,k", [(17, 4096, 4096), (65, 512, 1024), (100, 512, 1024),
                                      (255, 4096, 4096)])
def test_overlapping_rows_stay_on_the_strips(rows, n, k):
    w = torch.empty(n, k, dtype=torch.bfloat16)
    assert not RW.tiled(matrix(rows, k, "expanded"), w)
    assert not RW.tiled(matrix(rows, k, "windows"), w)
    assert RW.tiled(matrix(rows, k, "padded"), w) == RW.tiled(matrix(rows, k, "plain"), w)


@pytest.mark.parametrize("rows", [256, 300, 320])
def test_residual_norm_of_a_prompt_leaves_what_the_tiles_refuse_to_the_library(rows):
    n, k = 512, 1024
    w, res = torch.empty(n, k, dtype=torch.bfloat16), matrix(rows, n, "plain")
    x = matrix(rows, k, "plain")
    assert RW.norm_tiled(x, w, res) and RW.norm_tiled(matrix(rows, k, "padded"), w, res)
    assert not RW.norm_tiled(x, w, matrix(rows, n, "expanded"))
    for off in (8, 40):  # the library takes every multiple of eight
        assert not RW.norm_tiled(matrix(rows, k + off, "plain"),
                                 torch.empty(n, k + off, dtype=torch.bfloat16), res)


def test_tile_cases_cover_the_plan():
    """Every launch the plan picks over sizes drawn from 2 to 2000 rows, widths
    from 16 to 23000 and k to 12000 (256 CUs, as on the device): tile, k split or
    whole, cached or streamed weights, per epilogue, bf16 and 8-bit."""
    lib, out = _lib.load(), (ctypes.c_int32 * 4)()

    def launches(rows, n, k):
        found = set()
        for epilogue in (_lib.EPI_STORE, _lib.EPI_RESIDUAL, _lib.EPI_SWIGLU):
            for fmt in (0, 1):
                assert lib.htn_gemm_tiles_plan(rows, n, k, epilogue, fmt, out) == _lib.HTN_OK
                assert (out[2] > 1) == (lib.htn_gemm_tiles_w8_scratch_bytes(
                    rows, n, k, epilogue, fmt) > 0)
                found.add((epilogue, fmt, out[0], out[1], out[2] > 1, out[3]))
        return found
    covered = set().union(*(launches(*c) for c in CASES + COVER))
    rng, drawn = random.Random(1), set()
    for _ in range(20000):
        drawn |= launches(int(2 ** rng.uniform(1, 11)), 8 * int(2 ** rng.uniform(1, 11.5)),
                          64 * int(2 ** rng.uniform(0, 7.6)))
    assert drawn <= covered, sorted(drawn - covered)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["expanded", "windows", "padded"])
@pytest.mark.parametrize("rows,n,k", [(9, 4096, 2048), (20, 4096, 2048), (40, 264, 1024),
                                      (129, 512, 9728), (255, 1000, 512)])
def test_rows_of_any_stride_give_the_contiguous_rows_results(rows, n, k, layout):
    x = matrix(rows, k, layout, "cuda")
    w = 0.02 * matrix(2 * n, k, "plain", "cuda", 1)
    top, res = w[:n].contiguous(), matrix(rows, n, "plain", "cuda", 2)
    gain = matrix(1, n, "plain", "cuda", 3)[0]
    xg = matrix(1, k, "plain", "cuda", 4)[0]
    y = x.float() @ top.float().T
    kw = dict(atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(RW.projection_rows(x, top).float(), y, **kw)
    if rows <= 32 or layout == "padded":  # the row-wise norm reads no overlapping rows
        torch.testing.assert_close(RW.projection_rows(x, top, xg).float(),
                                   RW.projection_rows(x.contiguous(), top, xg).float(), **kw)
    out, normed = RW.residual_norm_rows(x, top, res, gain)
    torch.testing.assert_close(out.float(), y.bfloat16().float() + res.float(), **kw)
    torch.testing.assert_close(RW.residual_rows(x, top, res).float(), out.float(), **kw)
    torch.testing.assert_close(normed.float(), torch.nn.functional.rms_norm(
        out.float(), (n,), gain.float(), 1e-6), **kw)
    gu = (x.float() @ w.float().T).bfloat16().float()
    torch.testing.assert_close(RW.swiglu_rows(x, w).float(),
                               torch.nn.functional.silu(gu[:, :n]) * gu[:, n:], **kw)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,k,layout", [(256, 512, 1032, "plain"), (512, 264, 520, "plain"),
                                             (300, 512, 1024, "expanded")])
def test_residual_norm_rows_off_the_tiles(rows, n, k, layout):
    x, w = matrix(rows, k, "plain", "cuda"), 0.02 * matrix(n, k, "plain", "cuda", 1)
    res, gain = matrix(rows, n, layout, "cuda", 2), matrix(1, n, "plain", "cuda", 3)[0]
    out, normed = RW.residual_norm_rows(x, w, res, gain)
    torch.testing.assert_close(out.float(), (x.float() @ w.float().T).bfloat16().float() + res.float(),
                               atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(normed.float(), torch.nn.functional.rms_norm(
        out.float(), (n,), gain.float(), 1e-6), atol=2e-2, rtol=2e-2)


def test_small_vocabularies_stay_on_the_strips():
    def vocabulary(v, k):
        return torch.empty(v, k, dtype=torch.bfloat16, device="meta")
    assert not RW.streams_head(vocabulary(8191, 1024)) and RW.streams_head(vocabulary(8192, 1024))
    codes, scale = torch.empty(16, 64, dtype=torch.uint8), torch.empty(16)
    assert RW.streams_head(RW.QuantizedWeight(codes, scale, "int8"))


@pytest.mark.gpu
@pytest.mark.parametrize("vocab", [8191, 8192])  # either side of the streamed size
@pytest.mark.parametrize("rows", [1, 3, 15, 16, 17, 40])
def test_greedy_rows_around_the_streamed_size(vocab, rows):
    x, w = matrix(rows, 1024, "plain", "cuda"), matrix(vocab, 1024, "plain", "cuda", 1)
    gain = matrix(1, 1024, "plain", "cuda", 2)[0]
    for g in (None, gain):
        xn = x if g is None else rms_norm(x, g, 1e-6)
        logits = xn.double() @ w.double().T
        got, best = RW.greedy_rows(x, w, g), logits.max(dim=1).values
        ulp = torch.pow(2.0, torch.floor(torch.log2(best)) - 7)
        # In the head's launch, the norm's sum of squares in another order may round
        # an element of a row the other way: four of the largest at most.
        slack = 0 if g is None else 4 * 2.0 ** -8 * float(xn.abs().max()) * float(w.abs().max())
        assert bool((best - logits.gather(1, got[:, None])[:, 0] <= ulp + slack).all())
