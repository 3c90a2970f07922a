"""The row form of the linear mix (csrc/mix_rows.hip) against float64: every number of channels it is built for and the first it
is not, tree counts around its chunk of 64, row counts around its tiles and shares, and both sides of its rule on rows."""
import ctypes

import pytest
import torch

from hingetreefortorch_amd import _lib

pytestmark = pytest.mark.gpu


def _mix(dev, B, T, O, bias=True, seed=0):
    lib = _lib.load()
    gen = torch.Generator().manual_seed(seed)
    f, lin, g = (torch.randn(s, generator=gen) for s in ((B, T), (O, T), (B, O)))
    bv = torch.randn(O, generator=gen) if bias else None
    df, dl, dg = f.to(dev), lin.to(dev), g.to(dev)
    db = bv.to(dev) if bias else None
    p = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    out = torch.full((B, O), float("nan"), device=dev)
    assert lib.ht_tree_mix_forward(B, T, O, 1, p(df), p(dl), p(db), p(out), stream) == 0
    want = f.double() @ lin.double().T + (bv.double() if bias else 0)
    # sums of T rounded products of unit normals: sqrt(T) 2^-24 of the result's scale sqrt(T), a factor ten for the extremes
    assert (out.cpu().double() - want).abs().max() <= 1e-5 * T ** 0.5 + 1e-6
    for want_h, want_l in ((True, True), (True, False), (False, True)):
        h = torch.full((B, T), float("nan"), device=dev) if want_h else None
        dlin = torch.full((O, T), float("nan"), device=dev) if want_l else None
        assert lib.ht_tree_mix_backward(B, T, O, 1, p(df), p(dl), p(dg), p(h), p(dlin), 0, stream) == 0
        if want_h:
            assert (h.cpu().double() - g.double() @ lin.double()).abs().max() <= 1e-5 * O ** 0.5 + 1e-6
        if want_l:
            assert (dlin.cpu().double() - g.double().T @ f.double()).abs().max() <= 1e-5 * B ** 0.5 + 1e-6


@pytest.mark.parametrize("O", list(range(1, 34)))
def test_channels(dev, O):
    _mix(dev, 333, 77, O, bias=O % 2 == 0, seed=O)


@pytest.mark.parametrize("B,T", [(1, 1), (31, 63), (32, 64), (33, 65), (2, 1000), (1000, 1), (4099, 7), (16384, 130), (16385, 129),
                                 (70001, 3)])
@pytest.mark.parametrize("O", [3, 16, 17])
def test_rows_and_trees(dev, B, T, O):
    _mix(dev, B, T, O, seed=B + T)


def test_infinite_row_stays_in_its_row(dev):
    lib = _lib.load()
    B, T, O = 40, 70, 5
    f, lin = torch.ones(B, T, device=dev), torch.ones(O, T, device=dev)
    f[3, 69] = float("inf")
    out = torch.empty(B, O, device=dev)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    assert lib.ht_tree_mix_forward(B, T, O, 1, p(f), p(lin), None, p(out), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    want = torch.full((B, O), float(T))
    want[3] = float("inf")
    assert torch.equal(out.cpu(), want)
