"""The native graph nodes (csrc_host/hingetree_autograd.cpp) against the Python autograd functions they stand in for:
same outputs, same gradients for every subset of wanted ones, same refusals."""
import pytest
import torch

from conftest import make_conv, make_forest, rel_err
import hingetree_cpp as ops
from hingetreefortorch_amd import functions as fn

pytestmark = pytest.mark.gpu


def _case(name, fern):
    """(function, arguments, positions of the differentiable ones)"""
    if name == "forest":
        x, thr, ordn, w, _ = make_forest(70, 20, [], 12, 4, [3], fern, torch.float32)
        return (fn.HingeFern if fern else fn.HingeTree), [x, thr, ordn, w], [0, 1, 3]
    if name == "expanded":
        x, thr, ordn, w, _ = make_forest(2, 9, [6, 5], 5, 3, [4, 4], fern, torch.float32)
        return (fn.HingeFernExpanded if fern else fn.HingeTreeExpanded), [x, thr, ordn, w, 2], [0, 1, 3]
    if name == "mix":
        x, thr, ordn, w, _ = make_forest(40, 20, [], 12, 4, [2], fern, torch.float32)
        g = torch.Generator().manual_seed(3)
        return ((fn.HingeFernFusedLinear if fern else fn.HingeTreeFusedLinear),
                [x, thr, ordn, w, torch.randn(5, 12, generator=g), torch.randn(5, generator=g)], [0, 1, 3, 4, 5])
    if name == "conv":
        x, thr, ordn, w = make_conv(2, 3, 4, [9, 8], 3, [], (3, 3), fern, torch.float32)
        return (fn.HingeFernConv2d if fern else fn.HingeTreeConv2d), [x, thr, ordn, w, (3, 3), (1, 1), (1, 1), (1, 1)], [0, 1, 3]
    g = torch.Generator().manual_seed(5)
    if name == "linear_bn":
        return fn.LinearBatchNorm, [torch.randn(64, 12, generator=g), torch.randn(20, 12, generator=g), 1e-5], [0, 1]
    x, thr, ordn, w, _ = make_forest(64, 6 * 7, [], 6, 3, [2], False, torch.float32)
    return (fn.LinearBatchNormForest, [torch.randn(64, 12, generator=g), torch.randn(42, 12, generator=g), 1e-5, thr, ordn, w, fern],
            [0, 1, 3, 5]) if not fern else None


def _run(host, function, args, wanted):
    before = ops.host
    ops.use_host(host)
    try:
        args = [a.detach().clone() if isinstance(a, torch.Tensor) else a for a in args]
        for i in wanted:
            args[i].requires_grad_(True)
        out = function.apply(*args)
        first = out[0] if isinstance(out, tuple) else out
        g = torch.randn(first.shape, generator=torch.Generator().manual_seed(9)).to(first.device)
        grads = torch.autograd.grad(first, [args[i] for i in wanted], g, retain_graph=True) if wanted else ()
        assert first.requires_grad == bool(wanted)
        if wanted:
            torch.autograd.grad(first, [args[wanted[0]]], g)
            with pytest.raises(RuntimeError, match="second time"):
                torch.autograd.grad(first, [args[wanted[0]]], g)
        return out if isinstance(out, tuple) else (out,), grads
    finally:
        ops.use_host(before)


@pytest.mark.parametrize("fern", [False, True], ids=["tree", "fern"])
@pytest.mark.parametrize("name", ["forest", "expanded", "mix", "conv", "linear_bn", "linear_forest"])
def test_native_nodes_match_python_functions(dev, name, fern):
    case = _case(name, fern)
    if case is None:
        pytest.skip("one private feature per vertex: trees only")
    function, args, diff = case
    args = [a.to(dev) if isinstance(a, torch.Tensor) else a for a in args]
    for wanted in [[], diff] + [[i] for i in diff]:
        out_n, grad_n = _run("native", function, args, wanted)
        out_p, grad_p = _run("python", function, args, wanted)
        assert len(out_n) == len(out_p)
        for a, b in zip(out_n, out_p):
            assert torch.equal(a, b)
        for a, b in zip(grad_n, grad_p):
            assert a.shape == b.shape and rel_err(a, b) <= 1e-5


def test_saved_tensors_are_guarded(dev):
    """A tensor the backward pass needs, changed in place after the forward pass, is refused."""
    x, thr, ordn, w, gout = [t.to(dev) for t in make_forest(30, 8, [], 4, 3, [2], False, torch.float32)]
    w.requires_grad_(True)
    out = fn.HingeTree.apply(x, thr, ordn, w)
    x.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward(gout)


@pytest.mark.parametrize("train", [False, True], ids=["eval", "train"])
@pytest.mark.parametrize("kind", ["forest", "expanded", "mix", "conv", "linear"])
def test_traced_module_follows_its_input(dev, kind, train):
    import hingetreefortorch_amd as ht
    torch.manual_seed(1)
    make, shape = {"forest": (lambda: ht.RandomHingeForest(12, 5, 3), (30, 12)),
                   "expanded": (lambda: ht.RandomHingeForestExpanded(6, 4, 3, extra_outputs=[4, 4]), (2, 6, 5, 5)),
                   "mix": (lambda: ht.RandomHingeForestFusedLinear(12, 6, 3, 3), (30, 12)),
                   "conv": (lambda: ht.HingeTreeConv2d(3, 4, 3, 3, padding=1), (2, 3, 7, 7)),
                   "linear": (lambda: ht.LinearHingeForest(10, 4, 3), (30, 10))}[kind]
    module = make().to(dev).train(train)
    with torch.no_grad():
        traced = torch.jit.trace(module, (torch.randn(shape, device=dev),), check_trace=False)
        for seed in (2, 3):
            x = torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dev)
            before = module.bn.running_mean.clone() if kind == "linear" else None
            got = traced(x)
            if before is not None:
                assert train != torch.equal(module.bn.running_mean, before)
            # (two routes of the projection: their products round alike)
            assert rel_err(got, module(x)) <= 1e-5
