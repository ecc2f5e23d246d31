"""CPU tests of the C++ autograd nodes: what they do when a backward pass is itself differentiated, with forward-mode tangents and under
function transforms.  The products and the embedding run
through torch on host tensors, the operators on meta tensors (shapes only): no kernel is launched."""
import pytest
import torch
import torch.nn.functional as F

from maltos_amd import ops  # noqa: F401  (registers the operators)
from maltos_amd._native import native


def _second(f, leaves):
    """Gradient of a penalty on the first derivatives."""
    first = torch.autograd.grad((f(*leaves) ** 3).sum(), leaves, create_graph=True)
    return torch.autograd.grad(sum((g ** 2).sum() for g in first), leaves)


@pytest.mark.parametrize("into_grad", [False, True])
@pytest.mark.parametrize("shape", [(5, 6), (2, 3, 6), (6,)])
def test_second_derivative_of_the_linear_layer(shape, into_grad):
    gen = torch.Generator().manual_seed(1)
    x, w = torch.randn(shape, generator=gen, dtype=torch.double), torch.randn(4, 6, generator=gen, dtype=torch.double)
    leaves = x.requires_grad_(True), w.requires_grad_(True)
    if into_grad:
        w.grad = torch.zeros_like(w)
    dx, dw = _second(lambda x, w: native().linear(x, w, into_grad), leaves)
    if into_grad:   # the last pass, which is not recorded, adds its own part to the buffer
        dw = dw + w.grad
    for got, want in zip((dx, dw), _second(F.linear, leaves)):
        assert torch.allclose(got, want, rtol=1e-12)
    if into_grad:   # a recorded pass adds to .grad with history, as torch does
        (native().linear(x, w, True) ** 2).sum().backward(create_graph=True)
        assert w.grad.grad_fn is not None


def test_second_derivative_of_the_embedding():
    gen = torch.Generator().manual_seed(2)
    w = torch.randn(7, 4, generator=gen, dtype=torch.double).requires_grad_(True)
    ids = torch.tensor([[1, 2, 2], [0, 6, 1]])
    (got,), (want,) = (_second(f, (w,)) for f in (lambda w: native().embedding(w, ids, False), lambda w: F.embedding(ids, w)))
    assert torch.allclose(got, want, rtol=1e-12)


def _meta(*shape):
    return torch.empty(shape, device="meta", requires_grad=True)


_OPS = {
    "attn_fwd": lambda: (lambda q, k, v: torch.ops.maltos.attn_fwd(q, k, v, 1, 0.5, None, None, None, None)[0], [_meta(1, 2, 4, 8) for _ in range(3)]),
    "rmsnorm_fwd": lambda: (lambda x, w: torch.ops.maltos.rmsnorm_fwd(x, w, 1e-5)[0], [_meta(3, 8), _meta(8)]),
    "add_rmsnorm_fwd": lambda: (lambda x, r, w: sum(torch.ops.maltos.add_rmsnorm_fwd(x, r, w, 1e-5)[:2]), [_meta(3, 8), _meta(3, 8), _meta(8)]),
    "swiglu_fwd": lambda: (torch.ops.maltos.swiglu_fwd, [_meta(3, 8), _meta(3, 8)]),
    "ce_fwd_bwd": lambda: (lambda x: torch.ops.maltos.ce_fwd_bwd(x, torch.zeros(3, dtype=torch.long, device="meta"), -100)[0], [_meta(3, 8)]),
}


@pytest.mark.parametrize("name", _OPS)
def test_a_second_derivative_without_a_formula_raises(name):
    f, leaves = _OPS[name]()
    for wanted in range(len(leaves)):
        first = torch.autograd.grad(f(*leaves).sum() ** 2, leaves, create_graph=True)   # (recording alone is fine)
        with pytest.raises(RuntimeError, match="no second derivative"):
            torch.autograd.grad(sum(g.sum() ** 2 for g in first), leaves[wanted], allow_unused=True)
    with pytest.raises(RuntimeError, match="no second derivative"):
        first = torch.autograd.grad(f(*leaves).sum() ** 2, leaves, create_graph=True)
        sum(g.sum() ** 2 for g in first).backward()


def test_rotations_are_differentiable_twice():
    cos, sin = torch.empty(4, 4, device="meta"), torch.empty(4, 4, device="meta")
    for f, leaves in ((lambda x: torch.ops.maltos.rope(x, cos, sin, None, 0, False), [_meta(1, 2, 4, 8)]),
                      (lambda a, b: sum(torch.ops.maltos.rope_pair(a, b, cos, sin, None, 0, False)), [_meta(1, 2, 4, 8), _meta(1, 2, 4, 8)])):
        first = torch.autograd.grad((f(*leaves) ** 2).sum(), leaves, create_graph=True)
        second = torch.autograd.grad(sum((g ** 2).sum() for g in first), leaves)
        assert [g.shape for g in second] == [t.shape for t in leaves]


@pytest.mark.parametrize("f,shapes", [(lambda x, w: native().linear(x, w, False), [(5, 6), (4, 6)]),
                                      (lambda w: native().embedding(w, torch.tensor([[1, 2, 2], [0, 6, 1]]), False), [(7, 4)])], ids=["linear", "embedding"])
def test_tangents_and_transforms_of_the_linear_layer_and_the_embedding(f, shapes):
    plain = {2: lambda x, w: F.linear(x, w), 1: lambda w: F.embedding(torch.tensor([[1, 2, 2], [0, 6, 1]]), w)}[len(shapes)]
    gen = torch.Generator().manual_seed(3)
    values, tangents = ([torch.randn(s, generator=gen, dtype=torch.double) for s in shapes] for _ in range(2))
    for requires_grad in (False, True):
        leaves = [v.clone().requires_grad_(requires_grad) for v in values]
        with torch.autograd.forward_ad.dual_level():
            for only in range(len(shapes)):   # one tangent at a time
                args = [torch.autograd.forward_ad.make_dual(v, t) if i == only else v for i, (v, t) in enumerate(zip(leaves, tangents))]
                got, want = (torch.autograd.forward_ad.unpack_dual(g(*args)).tangent for g in (f, plain))
                assert torch.allclose(got, want)
    for got, want in ((torch.func.jvp(g, tuple(values), tuple(tangents))[1] for g in (f, plain)),
                      (torch.func.grad(lambda *a: (g(*a) ** 2).sum())(*values) for g in (f, plain)),
                      (torch.func.vmap(g, in_dims=(0, *[None] * (len(shapes) - 1)))(torch.stack([values[0]] * 2), *values[1:]) for g in (f, plain))):
        assert torch.allclose(got, want)


@pytest.mark.parametrize("requires_grad", [False, True])
@pytest.mark.parametrize("name", _OPS)
def test_a_tangent_without_a_formula_raises(name, requires_grad):
    f, leaves = _OPS[name]()
    leaves = [t.detach().requires_grad_(requires_grad) for t in leaves]
    with torch.autograd.forward_ad.dual_level():
        for only in range(len(leaves)):
            args = [torch.autograd.forward_ad.make_dual(t, torch.empty_like(t)) if i == only else t for i, t in enumerate(leaves)]
            with pytest.raises(NotImplementedError, match="forward-mode"):
                f(*args)


def test_tangents_through_rotations_and_joint_projections_raise():
    cos, sin = torch.empty(4, 4, device="meta"), torch.empty(4, 4, device="meta")
    x = torch.empty(1, 2, 4, 8, device="meta")
    group = native().Adjacent([torch.empty(4, 6)])
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.empty_like(x))
        rows = torch.autograd.forward_ad.make_dual(torch.empty(3, 6), torch.empty(3, 6))
        for call in (lambda: torch.ops.maltos.rope(dual, cos, sin, None, 0, False), lambda: torch.ops.maltos.rope_pair(x, dual, cos, sin, None, 0, False),
                     lambda: native().rope_attention(x, x, dual, cos, sin, None, 0, None, None), lambda: native().cross_entropy_over_logits(rows, rows, 0),
                     lambda: native().adjacent_linears(rows, group, [torch.empty(4, 6)], False), lambda: native().gate_up(rows, group, [torch.empty(4, 6)], False)):
            with pytest.raises(NotImplementedError, match="forward-mode"):
                call()


def test_kept_rows_belong_to_parameters_of_one_shape_and_type():
    """What a module keeps about its projections is made anew when another parameter lies at the address of an old one."""
    memory = torch.zeros(64)
    group = native().Adjacent([memory.view(8, 8)])
    assert group.made_for([memory.view(8, 8)])
    for other in (memory.view(4, 16), memory.view(16, 4), memory[:32].view(4, 8), memory.view(torch.int32).view(8, 8), memory.view(8, 8).requires_grad_(True)):
        assert not group.made_for([other])


@pytest.mark.parametrize("name", _OPS)
def test_nested_function_transforms_raise_where_a_second_derivative_is_missing(name):
    f, leaves = _OPS[name]()
    values, total = [t.detach() for t in leaves], lambda *a: f(*a).sum()
    every = tuple(range(len(values)))
    first = torch.func.grad(total, argnums=every)
    assert [g.shape for g in first(*values)] == [v.shape for v in values]
    penalty = lambda *a: sum((g ** 2).sum() for g in first(*a))
    with pytest.raises(RuntimeError, match="no second derivative"):
        torch.func.grad(penalty, argnums=every)(*values)
    with pytest.raises(RuntimeError, match="no second derivative"):
        penalty(*leaves)   # (the leaves require gradients: torch's autograd around the transform)
