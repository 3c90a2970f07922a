"""The walk records' layout and the loops that read four samples of a tree at once: sample counts around the line pitch, every
remainder modulo four, shares of the samples that end inside a superblock, and both sides of the row kernel's tile rule."""
import pytest
import torch

from conftest import make_forest
from oracle import hinge_oracle as ho
import hingetree_cpp as ops
from test_gpu_pairs import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fern", [False, True], ids=["tree", "fern"])
@pytest.mark.parametrize("M,dtype", [(1, torch.float32), (10, torch.float32), (26, torch.float32), (2, torch.float64)])
@pytest.mark.parametrize("B", [1021, 1022, 1023, 1024, 1025, 1055, 1057])
def test_pitch_edges(dev, B, M, dtype, fern):
    _check(dev, B, 24, [], 300, 4, [M] if M > 1 else [], fern, dtype, B)


@pytest.mark.parametrize("B", [3, 4, 5, 6, 7, 9])
def test_few_samples_of_many_trees(dev, B):
    _check(dev, B, 24, [], 100000, 2, [], False, torch.float32, B)


@pytest.mark.parametrize("M", [1, 4, 10, 26, 64])
@pytest.mark.parametrize("B", [9001, 9002, 9003, 12544])
def test_shares_of_samples(dev, B, M):
    _check(dev, B, 24, [], 130, 4, [M] if M > 1 else [], False, torch.float32, B + M)


# rows of whole and of broken 64-byte sectors, tree counts around 200, the widest feature count two 16-sample tiles share a
# CU with (872) and its neighbours
@pytest.mark.parametrize("fern", [False, True], ids=["tree", "fern"])
@pytest.mark.parametrize("F,T,M", [(100, 300, 4), (511, 144, 12), (600, 300, 4), (617, 201, 6), (617, 199, 6), (872, 201, 10),
                                   (873, 201, 10), (300, 205, 20), (30, 250, 8), (300, 203, 1), (30, 202, 9)])
def test_row_tiles(dev, F, T, M, fern):
    x, thr, ordn, w, _ = make_forest(1337, F, [], T, 5, [M] if M > 1 else [], fern, torch.float32, seed=F + T)
    ref = ho.forward(x, thr, ordn, w, fern)
    args = [t.to(dev) for t in (x, thr, ordn, w)]
    pre = "fern_" if fern else "tree_"
    assert torch.equal(getattr(ops, pre + "forward")(*args).cpu(), ref)
    assert torch.equal(getattr(ops, pre + "forward_records")(*args)[0].cpu(), ref)
