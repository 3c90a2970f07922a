"""Both sides of the rule that sends problems of few (sample, tree) pairs to kernels of their own (csrc/forest_pairs.hip):
shapes just inside it, with the remainders its lanes, batches and shares can meet, and shapes just beyond it for the tile
and tree kernels, at the row widths and tiles these are instantiated for."""
import pytest
import torch

from conftest import make_forest, rel_err
from oracle import hinge_oracle as ho
import hingetree_cpp as ops

pytestmark = pytest.mark.gpu


def _check(dev, B, F, Kd, T, D, Md, fern, dtype, seed):
    x, thr, ordn, w, gout = make_forest(B, F, Kd, T, D, Md, fern, dtype, seed=seed)
    # on a grid on which every margin is exact, so that the float64 evaluation walks like the float32 one even where two
    # margins of a path tie
    x, thr = torch.round(x * 1024) / 1024, torch.round(thr * 1024) / 1024
    ref = ho.forward(x, thr, ordn, w, fern)
    exact = ho.backward(x.double(), thr.double(), ordn, w.double(), gout.double(), fern=fern)
    gx, gthr, gord, gw, gg = [t.to(dev) for t in (x, thr, ordn, w, gout)]
    pre = "fern_" if fern else "tree_"
    assert torch.equal(getattr(ops, pre + "forward")(gx, gthr, gord, gw).cpu(), ref)
    out, rec = getattr(ops, pre + "forward_records")(gx, gthr, gord, gw)
    assert torch.equal(out.cpu(), ref) and rec is not None
    # float32: sums of up to S or T * M rounded terms, accumulated in float64 or in a float32 tree
    tol = 1e-5 if dtype == torch.float32 else 1e-12
    for det in (False, True):
        got = getattr(ops, pre + "backward_records")(rec, det, gx, True, gthr, True, gord, False, gw, True, gg)
        for a, b in zip((got[0], got[1], got[3]), exact):
            assert rel_err(a.cpu().double(), b) <= tol, (det, a.shape)
    only = getattr(ops, pre + "backward_records")(rec, False, gx, False, gthr, True, gord, False, gw, False, gg)
    assert only[0] is None and only[3] is None and rel_err(only[1].cpu().double(), exact[1]) <= tol
    only = getattr(ops, pre + "backward_records")(rec, False, gx, True, gthr, False, gord, False, gw, False, gg)
    assert only[1] is None and only[3] is None and rel_err(only[0].cpu().double(), exact[0]) <= tol


@pytest.mark.parametrize("fern", [False, True], ids=["tree", "fern"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("case", [
    (1, 1, [], 1, 1, []), (1, 5, [], 65, 3, [2]), (63, 7, [], 1, 12, [1]), (65, 9, [], 3, 5, [3]), (300, 33, [], 7, 1, [4]),
    (5, 20000, [], 3, 4, [5]), (33, 16, [], 100, 7, [26]), (17, 8, [3, 5], 6, 4, [4, 4]), (700, 10, [], 5, 6, [17]),
    (9000, 6, [], 4, 3, [65]), (20000, 12, [], 3, 5, [1]), (2, 70000, [], 2, 17, [1]), (65536, 4, [], 1, 4, [2])],
    ids=lambda c: "x".join(str(v) for v in c).replace(" ", ""))
def test_few_pairs(dev, case, dtype, fern):
    _check(dev, *case, fern, dtype, 1)


@pytest.mark.parametrize("fern", [False, True], ids=["tree", "fern"])
@pytest.mark.parametrize("B", [4100, 4099], ids=["aligned", "ragged"])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 20, 64])
def test_row_widths_beyond(dev, M, B, fern):
    _check(dev, B, 24, [], 130, 5, [M] if M > 1 else [], fern, torch.float32, M)


@pytest.mark.parametrize("fern", [False, True], ids=["tree", "fern"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("F", [96, 1024, 1500, 4000])
@pytest.mark.parametrize("M", [1, 3, 10, 33])
@pytest.mark.parametrize("T", [133, 140])
def test_tiles_beyond(dev, T, M, F, dtype, fern):
    _check(dev, 4003, F, [], T, 4, [M] if M > 1 else [], fern, dtype, M + F)


@pytest.mark.parametrize("fern", [False, True], ids=["tree", "fern"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("Kd,Md", [([10, 10], [4, 4]), ([7], [3]), ([200], [])], ids=["image", "short", "long"])
def test_inner_positions_beyond(dev, Kd, Md, dtype, fern):
    K = 1
    for k in Kd:
        K *= k
    _check(dev, 4003 // K + 1, 24, Kd, 140, 4, Md, fern, dtype, K)


def _cancelling(S, F, T, D, M, fern):
    """Inputs of which every term of every gradient is a small multiple of 1/2, so that float64 sums are exact, while the
    second half of the samples takes back what the first half adds, but for a remainder of a few units: a sum that is
    rounded to float32 on the way (past 2^24) does not come back to it."""
    gen = torch.Generator().manual_seed(S + T + D + M)
    draw = lambda lo, hi, *shape: torch.randint(lo, hi, shape, generator=gen)
    V, half = (D if fern else 2 ** D - 1), S // 2
    x = draw(-4, 5, S, F).float()
    x[half:2 * half] = x[:half]
    thr, ordn = draw(-3, 3, T, V).float() + 0.5, draw(0, F, T, V)
    w = 2.0 * draw(0, 2, T, 2 ** D, M).float() - 1.0
    g = draw(0, 2 ** 20 if M <= 4 else 2 ** 18, S, T, M).float()  # (times 15/2 at most, or summed over M, below 2^24)
    g[half:2 * half] = draw(-1, 2, half, T, M).float() - g[:half]
    g[2 * half:] = 1.0
    return x, thr, ordn, w, g


SHARED_OUT = [(25600, 16, 4, 7, 64), (20001, 5, 3, 5, 1), (60000, 4, 1, 1, 2), (9000, 6, 4, 3, 65), (100000, 8, 1, 6, 26)]


@pytest.mark.parametrize("fern", [False, True], ids=["tree", "fern"])
@pytest.mark.parametrize("case", SHARED_OUT, ids=lambda c: "x".join(map(str, c)))
def test_shares_meet_in_float64(dev, case, fern):
    x, thr, ordn, w, g = _cancelling(*case, fern)
    exact = ho.backward(x.double(), thr.double(), ordn, w.double(), g.double(), fern=fern)
    gx, gthr, gord, gw, gg = [t.to(dev) for t in (x, thr, ordn, w, g)]
    pre = "fern_" if fern else "tree_"
    rec = getattr(ops, pre + "forward_records")(gx, gthr, gord, gw)[1]
    for need in ((True, True, True), (False, True, False), (False, False, True)):
        got = getattr(ops, pre + "backward_records")(rec, False, gx, need[0], gthr, need[1], gord, False, gw, need[2], gg)
        for a, b, n in zip((got[0], got[1], got[3]), exact, need):
            assert torch.equal(a.cpu(), b.float()) if n else a is None


@pytest.mark.parametrize("S", [3, 5000])
def test_products_of_a_row_round_once(dev, S):
    """c = sum_m w g in fused multiply-adds, as the tree kernels form it: what a rounded product leaves of its own exact
    value is seen."""
    a, b = torch.tensor(1.0 + 2.0 ** -12), torch.tensor(1.0 - 3 * 2.0 ** -13)
    x, thr, ordn = torch.ones(S, 2), torch.zeros(1, 1), torch.zeros(1, 1, dtype=torch.int64)
    w = torch.stack([torch.ones(()), a]).expand(1, 2, 2).contiguous()
    g = torch.stack([-(a * b), b]).expand(S, 1, 2).contiguous()
    left = float(a.double() * b.double() - (a * b).double())
    assert left != 0.0
    gx, gthr, gord, gw, gg = [t.to(dev) for t in (x, thr, ordn, w, g)]
    rec = ops.tree_forward_records(gx, gthr, gord, gw)[1]
    dx, dthr, _, _ = ops.tree_backward_records(rec, False, gx, True, gthr, True, gord, False, gw, False, gg)
    assert (dx[:, 0] == left).all() and float(dthr) == -S * left


@pytest.mark.parametrize("fern", [False, True], ids=["tree", "fern"])
@pytest.mark.parametrize("case", SHARED_OUT + [(19200, 5, 1, 1, 12), (4000, 8, 60, 4, 3)], ids=lambda c: "x".join(map(str, c)))
def test_stateless_sums_in_float64(dev, case, fern):
    x, thr, ordn, w, g = _cancelling(*case, fern)
    exact = ho.backward(x.double(), thr.double(), ordn, w.double(), g.double(), fern=fern)
    gx, gthr, gord, gw, gg = [t.to(dev) for t in (x, thr, ordn, w, g)]
    for need in ((True, True, True), (False, True, False), (True, False, False)):
        got = getattr(ops, ("fern_" if fern else "tree_") + "backward")(gx, need[0], gthr, need[1], gord, False, gw, need[2], gg)
        for a, b, n in zip((got[0], got[1], got[3]), exact, need):
            assert torch.equal(a.cpu(), b.float()) if n else a is None


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("case", [(1, 4, [], 1, 1, [1]), (4096, 8, [], 3, 12, [9]), (4097, 8, [], 3, 12, [9]), (40, 21000, [], 2, 3, [2]),
                                  (4100, 20600, [], 1, 2, [1]), (7, 70000, [], 2, 17, [1]), (90, 5, [11, 3], 40, 5, [4, 4])],
                         ids=lambda c: "x".join(str(v) for v in c).replace(" ", ""))
def test_stateless_few_pairs(dev, case, dtype):
    """Small stateless calls on either side of the rules: the few-pairs kernel, leaf tables and features that it does not
    take, few and many samples of those."""
    for fern in (False, True):
        x, thr, ordn, w, gout = make_forest(*case, fern, dtype, seed=5)
        x, thr = torch.round(x * 1024) / 1024, torch.round(thr * 1024) / 1024
        exact = ho.backward(x.double(), thr.double(), ordn, w.double(), gout.double(), fern=fern)
        args = [t.to(dev) for t in (x, thr, ordn, w, gout)]
        got = getattr(ops, ("fern_" if fern else "tree_") + "backward")(args[0], True, args[1], True, args[2], False, args[3],
                                                                       True, args[4])
        for a, b in zip((got[0], got[1], got[3]), exact):
            assert rel_err(a.cpu().double(), b) <= (1e-5 if dtype == torch.float32 else 1e-12), (fern, a.shape)


@pytest.mark.parametrize("fern", [False, True], ids=["tree", "fern"])
@pytest.mark.parametrize("case", [(16384, 5, [], 32, 3, [6]), (16383, 5, [], 32, 3, [6]), (16390, 9, [], 23, 4, [13]),
                                  (16400, 100, [], 63, 2, [11]), (16384, 12, [], 48, 5, [4]), (16385, 12, [], 33, 5, [3]),
                                  (3001, 20, [], 301, 3, [3]), (4096, 20, [], 301, 3, [3]), (16400, 30, [], 64, 9, [4]),
                                  (8193, 30, [], 256, 11, [4]), (16384, 300, [], 31, 2, [5]), (16384, 300, [], 65, 2, [5]),
                                  (8192, 40, [], 40, 4, []), (8193, 40, [], 40, 4, []), (8193, 300, [], 63, 3, [26]),
                                  (17000, 200, [], 31, 3, [26]), (17000, 200, [], 32, 3, [5])],
                         ids=lambda c: "x".join(str(v) for v in c).replace(" ", ""))
def test_tile_rule(dev, case, fern):
    """The sample tiles that the row kernel's rule picks, on both sides of its lines."""
    _check(dev, *case, fern, torch.float32, 3)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("case", [(700, 20, [], 64, 9, [20]), (700, 20, [], 65, 9, [20]), (500, 20, [], 191, 9, [20]),
                                  (500, 20, [], 192, 9, [20]), (900, 20, [], 200, 9, [16]), (900, 20, [], 201, 9, [16]),
                                  (900, 20, [], 201, 8, [16])], ids=lambda c: "x".join(str(v) for v in c).replace(" ", ""))
def test_leaf_tables_on_the_rule(dev, case, dtype):
    """Large leaf tables on both sides of the lines between the few-pairs kernel and the tree kernels."""
    _check(dev, *case, False, dtype, 4)
