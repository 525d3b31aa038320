"""Whole steps of small matrices in one workgroup (polar_resident.hip): the stage kernels'
bits (unsplit, single diagonal tiles) at every number of 32-row blocks, at the edges of
16-row and 32-column blocks, at widths of whole vectors, even, odd and under 8, tall, in
batches whose matrices start off 16-byte boundaries, with the normalisation and in place of
a chain of any length."""

from __future__ import annotations

import os

import pytest
import torch

from oracle import polar_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
SHAPES = [(1, 1, 1), (3, 3, 5), (2, 7, 7), (1, 16, 17), (2, 31, 33), (1, 32, 2048), (2, 40, 24),
          (3, 64, 65), (1, 65, 90), (5, 96, 96), (2, 97, 130), (1, 128, 384), (3, 129, 257),
          (1, 160, 256), (2, 192, 128), (300, 9, 40), (256, 161, 192), (257, 15, 16)]


@pytest.fixture
def mf(monkeypatch):
    import muon_fusion_ascend950_amd as module

    # (any variable that tunes the stages turns the resident kernel off)
    for k in [k for k in os.environ if k.startswith("MUON_POLAR_") and k != "MUON_POLAR_CAPI_LIBRARY"]:
        monkeypatch.delenv(k)
    return module


def route(shape):
    """1: single steps resident, 2: chains (tall odd widths run transposed)."""
    from muon_fusion_ascend950_amd import capi

    batch, m, n = shape
    if m > n and n % 8:
        m, n = n, m
    return capi.check_plan(batch, m, n, cus=256, blocks_per_cu=(2, 2, 2)).resident


def _stages(monkeypatch, f):
    with monkeypatch.context() as mp:
        mp.setenv("MUON_POLAR_RESIDENT", "0")
        mp.setenv("MUON_POLAR_STREAM_K", "0")
        mp.setenv("MUON_POLAR_DIAG_PAIRS", "0")
        y = f()
        torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("shape", SHAPES)
def test_steps_and_chains_have_the_stage_kernels_bits(monkeypatch, mf, shape):
    x = O.make_input(shape, seed=61).to(DEV)
    raw = (x.float() * 37.0).to(torch.bfloat16)
    calls = [lambda: mf.polar_step(x, *O.COEFFICIENTS[0]),
             lambda: mf.polar_express(raw),
             lambda: mf.polar_express(x, O.COEFFICIENTS[:2], normalize=False),
             # more steps than one launch takes
             lambda: mf.polar_express(raw, O.COEFFICIENTS + O.COEFFICIENTS[4:] * 4)]
    assert route(shape) == 3
    for f in calls:
        y = f()
        torch.cuda.synchronize()
        assert torch.isfinite(y).all()
        want = _stages(monkeypatch, f)
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("offset", [1, 2, 8])
@pytest.mark.parametrize("shape", [(2, 20, 33), (1, 64, 64), (1, 5, 7)])
def test_addresses_off_16_bytes_and_nothing_written_outside(mf, shape, offset):
    from muon_fusion_ascend950_amd import capi

    batch, m, n = shape
    x0 = O.make_input(shape, seed=62).to(DEV)
    buf = torch.zeros(x0.numel() + 16, dtype=torch.bfloat16, device=DEV)
    x = buf[offset:offset + x0.numel()].view(shape)
    x.copy_(x0)
    out = torch.full((x0.numel() + 32,), 7.0, dtype=torch.bfloat16, device=DEV)
    y = out[16 + offset:16 + offset + x0.numel()].view(shape)
    ws, _ = capi.alloc_workspace(*shape)
    capi.step(x, y, ws, *O.COEFFICIENTS[0])
    torch.cuda.synchronize()
    assert torch.equal(y, mf.polar_step(x0, *O.COEFFICIENTS[0]))
    assert (out[:16 + offset] == 7.0).all() and (out[16 + offset + x0.numel():] == 7.0).all()


def test_infinities_and_nans_stay_in_their_matrix(mf):
    x = O.make_input((3, 40, 50), seed=63).to(DEV)
    clean = mf.polar_step(x, *O.COEFFICIENTS[0])
    bad = x.clone()
    bad[1, 3, 4] = float("inf")
    bad[1, 7, 9] = float("nan")
    y = mf.polar_step(bad, *O.COEFFICIENTS[0])
    assert torch.equal(y[0], clean[0]) and torch.equal(y[2], clean[2])
    assert not torch.isfinite(y[1].float()).any()


@pytest.mark.parametrize("shape", [(64, 384, 128), (85, 352, 120)])
def test_a_chain_is_its_steps_where_only_the_chain_is_resident(mf, shape):
    assert route(shape) == 2
    x = O.make_input(shape, seed=64).to(DEV)
    want = x
    for c in O.COEFFICIENTS:
        want = mf.polar_step(want, *c)
    assert torch.equal(mf.polar_express(x, O.COEFFICIENTS, normalize=False), want)


@pytest.mark.parametrize("steps", [8, 9, 16, 17])
# the stages cut [2,31,1501]'s gram; tall; whole vectors; even
@pytest.mark.parametrize("shape", [(2, 31, 1501), (3, 129, 257), (1, 257, 64), (2, 64, 96), (1, 95, 130)])
def test_chains_of_any_length_are_their_steps(mf, shape, steps):
    assert route(shape) == 3
    x = (O.make_input(shape, seed=65).float() * 11.0).to(torch.bfloat16).to(DEV)
    coeffs = (O.COEFFICIENTS + O.COEFFICIENTS[4:] * 12)[:steps]
    want = mf.polar_express(x, (), normalize=True)
    for c in coeffs:
        want = mf.polar_step(want, *c)
    assert torch.isfinite(want).all() and torch.equal(mf.polar_express(x, coeffs), want)


@pytest.mark.parametrize("steps", [1, 4, 5, 9])
@pytest.mark.parametrize("shape", [(3, 40, 64), (2, 33, 130), (1, 31, 57), (2, 72, 40), (2, 57, 31)])
def test_muon_updates_have_the_stage_kernels_bits(monkeypatch, mf, shape, steps):
    assert route(shape) & 2
    gen = torch.Generator(device=DEV).manual_seed(66)
    p, g, b = (torch.randn(shape, generator=gen, device=DEV) for _ in range(3))
    coeffs = O.COEFFICIENTS + O.COEFFICIENTS[4:] * 4

    def update():
        q, buf = p.clone(), b.clone()
        mf.muon_update(q, g, buf, lr=0.1, ns_steps=steps, coefficients=coeffs)
        return torch.stack([q, buf])

    y = update()
    assert torch.isfinite(y).all() and torch.equal(y, _stages(monkeypatch, update))
