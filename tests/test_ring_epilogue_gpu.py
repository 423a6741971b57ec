"""The LDS-ring tiles' straight epilogue (outputs without raw accumulators, through range-checked 32-bit offsets) and the
deep tiles: edges of tiles in both directions, every output type, residual and SiLU, against the oracle bit for bit (the
epilogue's SiLU to its tolerance), with the memory around the output untouched."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from kea_kernels import lowbit
from kea_kernels.binary import kernels
from oracle import oracle as O
from test_gemm_gpu import Case, _bits, _gpu_bits

pytestmark = pytest.mark.gpu
DEV = "cuda"
RING = [t for t in range(1, 40) if kernels.config_name(t) and " k/" not in kernels.config_name(t)]


def _run(case, tile, dtype, m=None, silu=False, residual=False, pad=4):
    """The output columns with everything around them poisoned: `pad` columns and two rows past the end."""
    m = case.m if m is None else m
    y = torch.full((m + 2, case.n + pad), float("nan"), device=DEV, dtype=dtype)
    res = None
    if residual:
        y[:m, :case.n] = torch.randn(m, case.n, generator=torch.Generator().manual_seed(m)).to(DEV)
        res = y
    r0 = y[:m, :case.n].float().cpu().numpy().copy()
    try:
        lowbit.gemm(case.wbits, case.dq, case.dqs, case.words, case.n, case.k, case.dalpha, case.dbias, y, None, m=m,
                    silu=silu, residual=res, residual_factor=0.5, config=kernels.GemmConfig(tile, 1))
    except ValueError as e:
        assert "does not fit" in str(e)
        return None
    torch.cuda.synchronize()
    assert torch.isnan(y[m:].float()).all() and torch.isnan(y[:, case.n:].float()).all(), kernels.config_name(tile)
    return y[:m, :case.n].cpu().contiguous(), r0


@pytest.mark.parametrize("wbits,parts,m,n,k", [
    (1, 1, 130, 260, 640),     # two columns and a row block past every tile's edge
    (2, 3, 65, 516, 272),      # K one unit past a 256-k stage
    (1, 2, 257, 128, 400),
    (2, 1, 17, 1030, 1040),    # N % 4 != 0: whole tiles straight, the last column tile general
    (1, 3, 1, 4, 16),
])
@torch.inference_mode()
def test_straight_epilogue_on_every_ring_tile(wbits, parts, m, n, k):
    case = Case(wbits, parts, m, n, k, seed=m + n, bias=True)
    acc = case.oracle_acc()
    ref = case.oracle_y(acc)
    for tile in RING:
        for dtype in (torch.float16, torch.bfloat16, torch.float32):
            got = _run(case, tile, dtype)
            if got is not None:
                assert np.array_equal(_gpu_bits(got[0], dtype), _bits(ref, dtype)), (kernels.config_name(tile), dtype)
        got = _run(case, tile, torch.float32, residual=True)
        if got is not None:  # y = residual + value * factor, two roundings
            want = got[1] + ref * np.float32(0.5)
            assert np.array_equal(_gpu_bits(got[0], torch.float32), want.view(np.uint32)), kernels.config_name(tile)
        got = _run(case, tile, torch.float32, silu=True)
        if got is not None:
            np.testing.assert_allclose(got[0].numpy(), case.oracle_y(acc, silu=True), rtol=2e-6, atol=2e-6)


@pytest.mark.parametrize("tile", [24, 25, 26])
@pytest.mark.parametrize("k", [128, 512, 2048, 2192])
@torch.inference_mode()
def test_deep_tiles_ring_and_tile_order(tile, k):
    """One to many stages of 128 k, and from K = 2048 the tile order by XCD: nine to seventeen row tiles (eight and the
    rest in the plain order), leading rows of a taller q, a last column tile of 4 columns."""
    case = Case(1, 1, 1090, 516, k, seed=k)
    ref = case.oracle_y(case.oracle_acc())
    for m in (1090, 1025, 900):
        got = _run(case, tile, torch.float16, m=m)[0]
        assert np.array_equal(_gpu_bits(got, torch.float16), _bits(ref[:m], torch.float16)), m


@torch.inference_mode()
def test_wide_output_rows_take_the_general_epilogue():
    """A row stride past the 32-bit offsets' range (2^20 elements) gives the same bits."""
    case = Case(1, 1, 20, 96, 256, seed=3)
    ref = case.oracle_y(case.oracle_acc())
    y = torch.zeros(20, 1 << 20, device=DEV, dtype=torch.float16)[:, :96]
    for tile in (4, 24):
        y.zero_()
        lowbit.gemm(1, case.dq, case.dqs, case.words, 96, 256, case.dalpha, None, y, None,
                    config=kernels.GemmConfig(tile, 1))
        assert np.array_equal(_gpu_bits(y.cpu().contiguous(), torch.float16), O.to_f16_bits(ref))
