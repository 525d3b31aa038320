"""The K loops of the large-tile kernels at their shortest lengths: 256x256 and 128x128
tiles (rings of five and nine panels) and 192x192 wave pairs (two and three slots) over 1
to 6 K-steps, every K mask and both forms.  The panel rings accumulate in the 64x64
kernels' order: the same bits.  Wave pairs sum two K chains: exact-sum inputs, bitwise against the 64x64 kernels."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import polar_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
C0 = O.COEFFICIENTS[0]
EXACT_COEFFS = (2.0, -1.0, 1.0)
# gram's K is the long side, poly's and apply's the short one; widths of whole 64-element
# blocks, of 16-byte chunks, even and odd; the last two run the right-Gram form
SHAPES = [(1, 40, 64), (2, 130, 192), (1, 200, 250), (1, 300, 328), (1, 270, 271), (1, 383, 384),
          (2, 330, 200), (1, 500, 256)]


def _step(monkeypatch, x, coeffs, env):
    with monkeypatch.context() as mp:
        mp.setenv("MUON_POLAR_STREAM_K", "0")
        for k, v in env.items():
            mp.setenv(k, v)
        op = (torch.ops.muon_ascend950.polar_step_tall if x.shape[1] > x.shape[2]
              else torch.ops.muon_ascend950.polar_step)
        y = op(x, *coeffs)
        torch.cuda.synchronize()
    return y


SMALL = {"MUON_POLAR_GRAM_TILE": "64", "MUON_POLAR_POLY_TILE": "64", "MUON_POLAR_APPLY_TILE_M": "64",
         "MUON_POLAR_DIAG_PAIRS": "0"}


@pytest.mark.parametrize("tile,depth", [("256", "2"), ("128", "2"), ("128", "4")])
@pytest.mark.parametrize("shape", SHAPES)
def test_panel_rings_equal_64_tiles(monkeypatch, shape, tile, depth):
    import muon_ascend950  # noqa: F401

    x = O.make_input(shape, seed=51).to(DEV)
    big = {f"MUON_POLAR_{s}_DEPTH": depth for s in ("GRAM", "POLY", "APPLY")}
    big.update({"MUON_POLAR_GRAM_TILE": tile, "MUON_POLAR_POLY_TILE": tile,
                "MUON_POLAR_APPLY_TILE_M": tile})
    assert torch.equal(_step(monkeypatch, x, C0, big), _step(monkeypatch, x, C0, SMALL))


@pytest.mark.parametrize("depth", ["2", "3"])
@pytest.mark.parametrize("shape", SHAPES)
def test_wave_pairs_sum_exactly(monkeypatch, shape, depth):
    import muon_ascend950  # noqa: F401

    tall = shape[1] > shape[2]
    mats = O.sparse_sign_input(shape, 8, seed=52)
    x = torch.from_numpy(np.stack([m.toarray() for m in mats]).astype(np.float32))
    x = x.to(torch.bfloat16).to(DEV)
    pairs = {"MUON_POLAR_GRAM_TILE": "192", "MUON_POLAR_POLY_TILE": "192",
             "MUON_POLAR_GRAM_DEPTH": depth, "MUON_POLAR_POLY_DEPTH": depth}
    y = _step(monkeypatch, x, EXACT_COEFFS, pairs)
    assert torch.equal(y, _step(monkeypatch, x, EXACT_COEFFS, SMALL))
    for i, m in enumerate(mats):
        want, max_sum = O.polar_step_fused_sparse(m.T.tocsr() if tall else m, *EXACT_COEFFS)
        assert max_sum < 2**24  # every fp32 sum is exact in any order
        want = torch.from_numpy((want.T if tall else want).astype(np.float32))
        assert torch.equal(y[i].float().cpu(), want.to(torch.bfloat16).float())
