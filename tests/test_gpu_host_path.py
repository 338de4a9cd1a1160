"""The calls that run through the extension module of the host path (csrc/host.cpp): the same outputs and gradients, to the last
bit, as the functions of the Python layer that they stand for, at first and second order, and what has to stay Python's."""
import pytest
import torch

from e3nn_amd import _lib, nn, o3
from e3nn_amd.nn.message import message_tensor_product
from tests import kernel_sets as ks

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ENTRIES = ("harmonics", "dense", "message", "fc_forward", "fc_layer", "mix", "lin2_alpha")


def _rand(gen, *shape, grad=True, dtype=torch.float32):
    return torch.randn(*shape, device=DEV, generator=gen).to(dtype).requires_grad_(grad)


def _graph(gen, nodes=30, edges=400):
    src, dst = (torch.randint(0, nodes, (edges,), device=DEV, generator=gen) for _ in range(2))
    return src, dst, nn.DstSortedEdges(src, dst, nodes)


def _harmonics(gen):
    return o3.SphericalHarmonics([0, 1, 2], True, "component"), [_rand(gen, 501, 3)]


def _dense(dtype, grads):
    def make(gen):
        tp = ks.mfma_small().to(DEV)
        shapes = [(70, tp.irreps_in1.dim), (70, tp.irreps_in2.dim), (tp.weight_numel,)]
        return lambda a, b, w: tp(a, b, w), [_rand(gen, *s, grad=g, dtype=dtype) for s, g in zip(shapes, grads)]

    return make


def _message(dtype, grads, harmonics=False):
    def make(gen):
        feats = "16x0e+16x1o+16x2e"
        tp = message_tensor_product(feats, o3.Irreps.spherical_harmonics(2), irreps_out=feats)
        _, _, edges = _graph(gen)
        x, attr, w = (_rand(gen, *s, grad=g, dtype=dtype) for s, g in zip([(30, 144), (400, 3 if harmonics else 9), (400, tp.weight_numel)], grads))
        if harmonics:
            return lambda a, b, c: tp.forward_gather_scatter_sh(a, b, c, edges), [x, attr, w]
        return lambda a, b, c: tp.forward_gather_scatter(a, b, c, edges=edges), [x, attr, w]

    return make


def _block(gen):
    feats = "32x0e+32x1o+32x2e"
    conv = nn.Convolution(feats, "4x0e", o3.Irreps.spherical_harmonics(2), feats, [8, 64], 20.0).to(DEV)
    src, dst, edges = _graph(gen)
    names = [n for n, _ in conv.named_parameters()]
    attr, edge_attr, scalars = _rand(gen, 30, 4, grad=False), _rand(gen, 400, 9, grad=False), _rand(gen, 400, 8, grad=False)
    call = lambda x, *ps: torch.func.functional_call(conv, dict(zip(names, ps)), (x, attr, src, dst, edge_attr, scalars), {"edges": edges})  # noqa: E731
    return call, [_rand(gen, 30, 288), *(_rand(gen, *p.shape) for p in conv.parameters())]


CASES = {
    "harmonics": _harmonics, "dense": _dense(torch.float32, (True, True, True)), "dense, x2 alone": _dense(torch.float32, (False, True, False)),
    "dense bf16": _dense(torch.bfloat16, (True, True, True)), "message": _message(torch.float32, (True, True, True)),
    "message, weights alone": _message(torch.float32, (False, False, True)), "message bf16": _message(torch.bfloat16, (True, True, True)),
    "message of vectors": _message(torch.float32, (True, True, True), True), "block": _block,
}  # fmt: skip


def _everything(f, inputs):
    """Output, first gradients (from the pass that can be differentiated and from the one that cannot), second ones."""
    inputs = [t.detach().clone().requires_grad_(t.requires_grad) for t in inputs]
    need = [t for t in inputs if t.requires_grad]
    out = f(*inputs)
    cot = torch.linspace(-1, 1, out.numel(), device=DEV).reshape(out.shape).to(out.dtype)
    first = torch.autograd.grad(out, need, cot, create_graph=True)
    energy = sum(t.double().square().sum() for t in first)
    second = torch.autograd.grad(energy, need, allow_unused=True) if energy.requires_grad else ()
    return [out, *first, *(t for t in second if t is not None), *torch.autograd.grad(f(*inputs), need, cot), f(*(t.detach() for t in inputs))]


@pytest.mark.parametrize("case", CASES)
def test_host_path_and_python_functions_give_the_same_bits(case, monkeypatch):
    f, inputs = CASES[case](torch.Generator(DEV).manual_seed(0))
    got = _everything(f, inputs)
    calls = []
    for name in ENTRIES:
        monkeypatch.setattr(_lib.native(), name, lambda *args, name=name: calls.append(name))
    ref = _everything(f, inputs)
    assert calls and len(got) == len(ref)
    # (weight gradients summed by atomics meet in any order)
    for a, b in zip(got, ref):
        assert torch.equal(a, b) or float((a - b).norm()) < 1e-6 * float(b.norm())


def test_host_path_saves_through_hooks_and_checks_versions():
    sh, (v,) = _harmonics(torch.Generator(DEV).manual_seed(1))
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.cpu())[1], lambda t: t.to(DEV)):
        out = sh(v)
    assert packed == [v.shape] and torch.equal(torch.autograd.grad(out.sum(), v)[0], torch.autograd.grad(sh(v).sum(), v)[0])
    moved = v * 1.0
    out = sh(moved)
    with torch.no_grad():
        moved.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()
    with pytest.raises(RuntimeError, match="functorch"):  # transforms are the Python function's, which says that it has none
        torch.func.vmap(sh)(v.detach().reshape(3, 167, 3))
