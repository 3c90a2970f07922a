"""The product on split operands (csrc/split_gemm.hip) and the sums over vertex-ordered samples behind it, at the edges of
their tiles, steps, chunks and blocks, on either side of the size from which the projection takes them."""
import pytest
import torch

from conftest import rel_err
import hingetree_cpp as ops
from hingetreefortorch_amd import LinearHingeForest

pytestmark = pytest.mark.gpu


# the rule: B * K * N >= 2^30 multiply-adds
SIZES = [(2048, 512, 1024), (2047, 512, 1024), (257, 16400, 260), (4097, 1030, 255), (70000, 17, 1024), (513, 4099, 513),
         (1 << 15, 1, 1 << 15), (300, 13, 40)]


@pytest.mark.parametrize("B,K,N", SIZES, ids=[f"{b}x{k}x{n}" for b, k, n in SIZES])
def test_projection_product(dev, B, K, N):
    g = torch.Generator().manual_seed(B + K + N)
    x = torch.randn(B, K, generator=g).to(dev)
    lin = (torch.randn(N, K, generator=g) * 2.0 ** torch.randint(-20, 20, (N, 1), generator=g)).to(dev)
    zhat, mean, rstd, var = ops.linear_bn_forward(x, lin, 0.0)
    xd, ld = x.double(), lin.double()
    cols = torch.arange(0, N, max(1, N // 256), device=dev)
    z = xd @ ld[cols].t()
    # every product exact to 2^-26, every addition rounded to 2^-24 of what it has summed so far
    bound = (K + 8) * 2.0 ** -24 * (xd.abs() @ ld[cols].abs().t())
    got = zhat[:, cols].double() / rstd[cols].double() + mean[cols].double()
    # (and the normalisation's own three roundings, of numbers up to |z - mean| and |mean|)
    bound += 4 * 2.0 ** -24 * (z.abs() + z.abs().max(0).values)
    assert ((got - z).abs() <= bound).all()
    scale = z.abs().max(0).values
    assert ((mean[cols].double() - z.mean(0)).abs() <= bound.max(0).values + 2.0 ** -24 * scale).all()
    assert rel_err(var[cols].double() / scale ** 2, z.var(0, unbiased=False) / scale ** 2) <= 1e-4


def test_projection_product_non_finite(dev):
    """An infinity or NaN reaches exactly the columns it enters (their statistics are then NaN, as in the plain product)."""
    g = torch.Generator().manual_seed(4)
    B, K, N = 2048, 512, 1100
    x, lin = torch.randn(B, K, generator=g), torch.randn(N, K, generator=g)
    lin[7, 3] = float("inf")
    lin[900, 500] = float("nan")
    lin[11, 0] = 3.4e38  # (the largest numbers are cut, not rounded to infinity)
    x[:, 0] *= 1e-3
    zhat = ops.linear_bn_forward(x.to(dev), lin.to(dev), 1e-5)[0].cpu()
    bad = torch.isnan(zhat).any(0)
    assert bad[7] and bad[900] and not bad[[i for i in range(N) if i not in (7, 900, 11)]].any()


@pytest.mark.parametrize("B,K,T,D,shared", [(8192, 64, 3, 4, False), (8193, 65, 3, 4, True), (16500, 63, 2, 7, False),
                                            (700, 130, 9, 3, True), (515, 1, 70, 5, False), (9000, 7, 4, 6, True)])
def test_records_backward_blocks(dev, B, K, T, D, shared):
    """dLin from the walk records against the dense route: samples in one, two and three blocks, one ragged; columns in
    one chunk, a sliver of a second, and fewer than a lane's four; features shared between vertices or private."""
    g = torch.Generator().manual_seed(B + K)
    V, N = 2 ** D - 1, (40 if shared else T * (2 ** D - 1))
    x, lin = torch.rand(B, K, generator=g).to(dev), (torch.randn(N, K, generator=g) / K ** 0.5).to(dev)
    thr = (3.0 * torch.rand(T, V, generator=g) - 1.5).to(dev)
    ordn = (torch.randint(0, N, (T, V), generator=g) if shared else torch.arange(T * V).reshape(T, V)).to(dev)
    w, up = torch.randn(T, 2 ** D, 2, generator=g).to(dev), torch.randn(B, T, 2, generator=g).to(dev)
    out, rec, z, mean, rstd, var = ops.tree_linear_bn_forward_records(x, lin, 1e-5, thr, ordn, w)
    got = ops.tree_linear_bn_backward_records(rec, x, lin, True, z, rstd, thr, True, ordn, w, True, up, mean=mean)
    assert got is not None
    zhat = (z - mean) * rstd
    dz, dthr, _, dw = ops.tree_backward_records(rec, True, zhat, True, thr, True, ordn, False, w, True, up)
    gd, rz = dz.double(), zhat.double()
    want = (rstd.double() * (gd - gd.mean(0) - rz * (gd * rz).mean(0))).t() @ x.double()
    scale = max(float(rstd.abs().max()), 1.0)
    assert rel_err(got[0].double(), want) <= 2e-5 * scale
    assert rel_err(got[1], dthr) <= 1e-5 and rel_err(got[2], dw) <= 1e-5


def test_running_statistics(dev):
    torch.manual_seed(2)
    model = LinearHingeForest(20, 6, 3, extra_outputs=2, momentum=0.3).to(dev)
    plain = torch.nn.BatchNorm1d(42, momentum=0.3, affine=False).to(dev)
    for _ in range(3):
        x = torch.randn(50, 20, device=dev)
        before = model.bn.running_mean._version
        model(x)
        plain(model.fc(x))
        assert model.bn.running_mean._version > before
        assert rel_err(model.bn.running_mean, plain.running_mean) <= 1e-5
        assert rel_err(model.bn.running_var, plain.running_var) <= 1e-5
    assert int(model.bn.num_batches_tracked) == 3


def test_records_backward_deepest(dev):
    """16383 vertices: those of the last level have their sums of c * zhat in memory, in part."""
    test_records_backward_blocks(dev, 9000, 8, 1, 14, False)


def test_records_backward_in_two_launches(dev):
    """More units of work (a tree, a block of samples, 64 columns) than one launch of the sums over segments takes."""
    test_records_backward_blocks(dev, 20, 64 * 64 + 1, (1 << 14) + 9, 1, False)


def test_projection_product_infinite_inputs(dev):
    """An infinite input makes its row of the product infinite, with the weights' signs, and so the columns' means; NaN only
    where a plain product is NaN (infinity times zero, infinities of both signs)."""
    g = torch.Generator().manual_seed(6)
    B, K, N = 2048, 512, 1100  # 1.15e9 multiply-adds: the split product; a ragged tile of columns
    x, lin = torch.randn(B, K, generator=g), torch.randn(N, K, generator=g)
    x[5, 3], x[1999, 511] = float("inf"), float("-inf")
    lin[4, 3] = 0.0
    thr, w = torch.zeros(2, 7), torch.randn(2, 8, 2, generator=g)
    ordn = torch.randint(0, N, (2, 7), generator=g)
    got = ops.tree_linear_bn_forward_records(*[t.to(dev) for t in (x, lin)], 1e-5, *[t.to(dev) for t in (thr, ordn, w)])
    z, mean = got[2].cpu(), got[3].cpu()
    want = x.double() @ lin.double().t()
    bad = [5, 1999]
    assert torch.isnan(want[5, 4]) and torch.equal(torch.isnan(z), torch.isnan(want))
    assert torch.isinf(want[bad]).sum() == 2 * N - 1
    clean = [b for b in range(B) if b not in bad]
    assert torch.equal(torch.nan_to_num(z[bad].double()), torch.nan_to_num(want[bad].float().double()))
    # (every addition rounded to 2^-24 of what it has summed so far)
    bound = (K + 8) * 2.0 ** -24 * (x[clean].double().abs() @ lin.double().abs().t())
    assert ((z[clean] - want[clean]).abs() <= bound).all()
    assert torch.equal(torch.isnan(mean), torch.isnan(want.mean(0)))
    infinite = torch.isinf(want.mean(0))
    assert infinite.any() and torch.equal(mean[infinite].double(), want.mean(0)[infinite])


@pytest.mark.parametrize("exponent", [-100, -109, -118, -126])
def test_projection_product_of_tiny_inputs(dev, exponent):
    """Inputs of 2^-109 and more lose nothing in the split, smaller ones up to 2^-134 each."""
    g = torch.Generator().manual_seed(7)
    B, K, N = 2048, 512, 1100
    x = torch.ldexp((1.0 + torch.rand(B, K, generator=g)) * (2.0 * torch.randint(0, 2, (B, K), generator=g) - 1.0),
                    torch.tensor(exponent))
    lin = torch.ldexp(torch.randn(N, K, generator=g), torch.tensor(90))
    thr, w = torch.zeros(2, 7), torch.randn(2, 8, 2, generator=g)
    ordn = torch.randint(0, N, (2, 7), generator=g)
    z = ops.tree_linear_bn_forward_records(x.to(dev), lin.to(dev), 1e-5, *[t.to(dev) for t in (thr, ordn, w)])[2].cpu()
    sizes = lin.double().abs()
    bound = (K + 8) * 2.0 ** -24 * (x.double().abs() @ sizes.t())
    if exponent < -109:
        bound += 2.0 ** -134 * sizes.sum(1)
    assert ((z - x.double() @ lin.double().t()).abs() <= bound).all()
    # ... which is well inside what these inputs would lose if their second parts were dropped
    assert float((z - x.double() @ lin.double().t()).norm() / z.double().norm()) <= 2.0 ** (-20 if exponent >= -109 else -9)


def test_records_backward_sums_in_blocks(dev):
    """8192 samples that all select one vertex: its sum of c * xc is formed in blocks of 16, runs of 512 and an atomic per run.
    With float32 additions, each off by at most 2^-24 (rms 2^-24 / sqrt(3)) of what it has summed, and terms of random sign,
    these three leave 264, 368 and 264 of a term's rms times that, together 2.0e-7 of the sum's sqrt(8192); one serial
    sum of 512 would leave 1450."""
    g = torch.Generator().manual_seed(8)
    B, K, T = 8192, 64, 16
    x, lin = torch.rand(B, K, generator=g).to(dev), torch.randn(T, K, generator=g).to(dev)
    thr, ordn = torch.zeros(T, 1, device=dev), torch.arange(T, device=dev).reshape(T, 1)
    w, up = torch.randn(T, 2, 1, generator=g).to(dev), torch.randn(B, T, 1, generator=g).to(dev)
    out, rec, z, mean, rstd, var = ops.tree_linear_bn_forward_records(x, lin, 1e-5, thr, ordn, w)
    got = ops.tree_linear_bn_backward_records(rec, x, lin, True, z, rstd, thr, True, ordn, w, True, up, mean=mean)[0]
    zhat = (z - mean) * rstd
    dz = ops.tree_backward_records(rec, True, zhat, True, thr, False, ordn, False, w, False, up)[0].double()
    zhat = zhat.double()
    want = (rstd.double() * (dz - dz.mean(0) - zhat * (dz * zhat).mean(0))).t() @ x.double()
    assert float((got.double() - want).norm() / want.norm()) <= 2.0e-7


def test_projection_product_has_no_bias(dev):
    """The column means of the product against float64. Its entries are off by some 4e-7 of their rms in either direction, so
    the average over 16384 rows and 256 columns is good to a few 1e-10 and the bound leaves a factor of ten, unless the
    rounding favours a direction (matrix instructions that round down leave 4e-8)."""
    g = torch.Generator(device=dev).manual_seed(9)
    B, K, N = 16384, 784, 256
    x, lin = torch.randn(B, K, generator=g, device=dev), torch.randn(N, K, generator=g, device=dev)
    mean = ops.linear_bn_forward(x, lin, 1e-5)[1]
    z = x.double() @ lin.double().t()
    assert abs(float((mean.double() - z.mean(0)).mean() / z.std())) <= 5e-9
