"""How the autograd nodes of the model and the operators behave beside the plain backward pass: saved-tensor hooks, frozen and
shared parameters, second derivatives, tangents."""
import pytest
import torch

from maltos_amd.llama import LlamaConfig, LlamaForCausalLM, set_grad_accumulation_into_buffers

pytestmark = pytest.mark.gpu


def _model(dev, dtype=torch.bfloat16, **config):
    cfg = dict(vocab_size=512, hidden_size=256, intermediate_size=688, num_hidden_layers=2, num_attention_heads=4,
               num_key_value_heads=2, max_position_embeddings=128, rms_norm_eps=1e-5) | config
    torch.manual_seed(5)
    return LlamaForCausalLM(LlamaConfig(**cfg)).to(dev).to(dtype)


def _batch(dev):
    ids = torch.randint(0, 512, (2, 101), generator=torch.Generator().manual_seed(1)).to(dev)
    return {"input_ids": ids, "labels": ids.clone()}


def _contiguous(t):
    return torch.empty(t.shape, dtype=t.dtype, device=t.device).copy_(t)


def _transposed(t):   # the same values, memory order of the dimensions reversed except for the last
    if t.dim() < 3:
        return _contiguous(t)
    order = [*reversed(range(t.dim() - 1)), t.dim() - 1]
    return _contiguous(t.permute(order)).permute([order.index(d) for d in range(t.dim())])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("pack", ["host", "contiguous", "transposed"])
@pytest.mark.parametrize("seq", [101, 1])
def test_saved_tensors_may_come_back_in_another_layout(dev, dtype, pack, seq):
    model, batch = _model(dev, dtype), _batch(dev)
    batch = {k: v[:, :seq].contiguous() for k, v in batch.items()}
    model(batch).backward()
    want = [p.grad.clone() for p in model.parameters()]
    model.zero_grad()
    if pack == "host":
        hooks = torch.autograd.graph.save_on_cpu(pin_memory=True)
    else:
        hooks = torch.autograd.graph.saved_tensors_hooks(_contiguous if pack == "contiguous" else _transposed, lambda t: t)
    with hooks:
        loss = model(batch)
    loss.backward()
    for (name, p), w in zip(model.named_parameters(), want):
        # the same kernels on the same values, the products' operands copied at most
        assert torch.equal(p.grad, w), name


def test_gradient_penalty_through_the_model_raises(dev):
    """No term of a second derivative is dropped without a word: the nodes of the layers have no second derivative."""
    model, batch = _model(dev), _batch(dev)
    weights = [p for p in model.parameters()]
    loss = model(batch)
    first = torch.autograd.grad(loss, weights, create_graph=True)
    model.zero_grad()
    model(batch).backward()
    for g, p in zip(first, weights):   # (recording alone changes nothing; sums of products in another order)
        assert (g.detach().float() - p.grad.float()).norm() <= 1e-2 * p.grad.float().norm()
    for g in (first[0], first[3], first[-1]):   # embedding, a projection, the head
        with pytest.raises(RuntimeError, match="no second derivative"):
            torch.autograd.grad(g.float().square().sum(), weights, allow_unused=True, retain_graph=True)


@pytest.mark.parametrize("name", ["layers.1.self_attn.q_proj.weight", "layers.0.mlp.down_proj.weight", "layers.1.input_layernorm.weight", "embed_tokens.weight"])
def test_tangent_of_a_weight_is_not_dropped_by_the_model(dev, name):
    model, batch = _model(dev), _batch(dev)
    weights = dict(model.named_parameters())
    with torch.autograd.forward_ad.dual_level(), pytest.raises(NotImplementedError, match="forward-mode"):
        dual = torch.autograd.forward_ad.make_dual(weights[name].detach(), torch.ones_like(weights[name]))
        torch.func.functional_call(model, {name: dual}, (batch,))


@pytest.mark.parametrize("pairs", [(("k_proj", "v_proj"),), (("q_proj", "k_proj"), ("k_proj", "v_proj")), (("gate_proj", "up_proj"),)])
def test_projections_that_share_a_weight_add_both_gradients_into_its_buffer(dev, pairs):
    def shared_model():
        model = _model(dev, torch.float32, num_key_value_heads=4)
        for layer in model.layers:
            for a, b in pairs:
                holder = layer.mlp if a == "gate_proj" else layer.self_attn
                getattr(holder, b).weight = getattr(holder, a).weight
        return model

    plain, buffers, batch = shared_model(), shared_model(), _batch(dev)
    set_grad_accumulation_into_buffers(buffers)
    for model in (plain, buffers):
        for p in model.parameters():
            p.grad = torch.zeros_like(p)
        for _ in range(2):
            model(batch).backward()
    for (name, p), q in zip(buffers.named_parameters(), plain.parameters()):
        assert (p.grad - q.grad).norm() <= 1e-5 * q.grad.norm(), name   # fp32 sums in another order


_FROZEN = {"all": lambda n: True, "projections": lambda n: "_proj" in n, "some": lambda n: "k_proj" in n or "up_proj" in n or "layers.0" in n,
           "all-but-o": lambda n: "o_proj" not in n and "down_proj" not in n, "all-but-v": lambda n: "layers.1.self_attn.v_proj" not in n}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form", ["layers-at-once", "modules", "into-buffers"])
@pytest.mark.parametrize("frozen", _FROZEN)
def test_frozen_weights_get_no_gradient_and_the_others_theirs(dev, dtype, form, frozen):
    def gradients(model, x):
        if form == "modules":
            model.layers[0].register_forward_hook(lambda *a: None)
        model({"hidden_states": x, "labels": _batch(dev)["labels"]}).backward()
        return x.grad

    trained, partly = _model(dev, dtype), _model(dev, dtype)
    for name, p in partly.named_parameters():
        p.requires_grad_(not _FROZEN[frozen](name))
    if form == "into-buffers":   # a frozen weight's buffer is left alone
        for model in (trained, partly):
            set_grad_accumulation_into_buffers(model)
            for name, p in model.named_parameters():
                p.grad = torch.zeros_like(p)
    hidden = torch.randn(2, 101, 256, generator=torch.Generator().manual_seed(2)).to(dev, dtype)
    dx, want = (gradients(m, hidden.clone().requires_grad_(True)) for m in (partly, trained))
    rel = 1e-2 if dtype == torch.bfloat16 else 1e-5   # (other launches add up in another order)
    assert (dx.double() - want.double()).norm() <= rel * want.double().norm()
    for (name, p), q in zip(partly.named_parameters(), trained.parameters()):
        if not p.requires_grad:
            assert p.grad is None or (p.grad == 0).all(), name
        elif q.grad is not None:
            assert (p.grad.double() - q.grad.double()).norm() <= rel * q.grad.double().norm(), name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hook", [False, True], ids=["layers-at-once", "modules"])
def test_frozen_weights_cost_no_products(dev, dtype, hook):
    """Their gradients are not formed: the backward pass asks for at least their bytes less."""
    taken = {}
    for frozen in (False, True):
        model = _model(dev, dtype)
        model.layers.requires_grad_(not frozen)
        if hook:
            model.layers[0].register_forward_hook(lambda *a: None)
        hidden = torch.randn(2, 101, 256, generator=torch.Generator().manual_seed(2)).to(dev, dtype).requires_grad_(True)
        loss = model({"hidden_states": hidden, "labels": _batch(dev)["labels"]})
        before = torch.cuda.memory_stats()["requested_bytes.all.allocated"]
        loss.backward()
        taken[frozen] = torch.cuda.memory_stats()["requested_bytes.all.allocated"] - before
    size = sum(p.numel() * p.element_size() for p in model.layers.parameters() if p.dim() == 2)
    assert taken[False] - taken[True] >= size, (taken, size)


def test_gradients_of_some_weights_alone(dev):
    """autograd.grad for one of several projections with adjacent weights: the others' buffers are not written."""
    from maltos_amd.optim import FusedAdamW, MasterWeightsOptimizer

    model, batch = _model(dev), _batch(dev)
    opt = MasterWeightsOptimizer(model.parameters(), optimizer_factory=lambda ps: FusedAdamW(ps, lr=1e-3), flat=True)
    model(batch).backward()
    names = ["layers.0.self_attn.k_proj.weight", "layers.1.mlp.up_proj.weight", "layers.1.self_attn.o_proj.weight"]
    weights = dict(model.named_parameters())
    want = [weights[n].grad.clone() for n in names]
    opt.zero_grad()
    got = torch.autograd.grad(model(batch), [weights[n] for n in names])
    assert (opt.flat_model_grad == 0).all()
    for name, g, w in zip(names, got, want):
        assert (g.double() - w.double()).norm() <= 1e-2 * w.double().norm(), name
    set_grad_accumulation_into_buffers(model)
    model(batch).backward(inputs=[weights[n] for n in names])
    for name, p in weights.items():
        if name in names:
            w = want[names.index(name)]
            assert (p.grad.double() - w.double()).norm() <= 1e-2 * w.double().norm(), name
        else:
            assert (p.grad == 0).all(), name


@pytest.mark.parametrize("form", ["layers-at-once", "modules"])
@pytest.mark.parametrize("name", ["self_attn.q_proj", "self_attn.o_proj", "mlp.up_proj", "mlp.down_proj", "input_layernorm"])
def test_weights_modified_between_forward_and_backward_are_noticed(dev, form, name):
    model, batch = _model(dev), _batch(dev)
    if form == "modules":
        model.layers[0].register_forward_hook(lambda *a: None)
    loss = model(batch)
    with torch.no_grad():
        model.get_submodule("layers.1." + name).weight.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()


@pytest.mark.parametrize("cls", ["LlamaMLP", "LlamaDecoderLayer", "LlamaRMSNorm", "HipLinear", "HipAttentionCore", "LlamaAttention"])
def test_a_replaced_forward_of_a_class_is_called(dev, cls, monkeypatch):
    import maltos_amd.llama as llama

    model, batch, calls = _model(dev), _batch(dev), []
    original = getattr(llama, cls).forward
    if cls == "HipAttentionCore":   # (only asked when rotation and attention are separate)
        monkeypatch.setattr(llama.LlamaAttention, "fuse_rope_attention", False)
    want = model(batch)
    monkeypatch.setattr(getattr(llama, cls), "forward", lambda self, *a, **kw: (calls.append(1), original(self, *a, **kw))[1])
    got = model(batch)
    assert calls and torch.allclose(got, want, rtol=1e-3)


def test_a_replaced_forward_of_a_projection_is_called(dev):
    model, batch, calls = _model(dev), _batch(dev), []
    projection = model.layers[0].self_attn.k_proj
    original = projection.forward
    projection.forward = lambda x: (calls.append(1), original(x))[1]
    model(batch)
    assert len(calls) == 1


def test_second_derivative_of_a_rotation(dev):
    """|R x|^2 has the gradient 2 x, and |2 x|^2 the gradient 8 x: by recorded passes and by nested function transforms."""
    from maltos_amd import ops

    gen = torch.Generator().manual_seed(6)
    x = torch.randn(1, 2, 5, 8, generator=gen).to(dev)
    angles = torch.rand(5, 4, generator=gen).to(dev)
    cos, sin = angles.cos(), angles.sin()
    for rotate in (lambda t: ops.rope(t, cos, sin), lambda t: ops.rope_pair(t, t, cos, sin)[1]):
        first = torch.func.grad(lambda t: rotate(t).square().sum())
        assert torch.allclose(torch.func.grad(lambda t: first(t).square().sum())(x), 8 * x, atol=1e-5)
        leaf = x.clone().requires_grad_(True)
        (g,) = torch.autograd.grad(rotate(leaf).square().sum(), leaf, create_graph=True)
        (second,) = torch.autograd.grad(g.square().sum(), leaf)
        assert torch.allclose(g.detach(), 2 * x, atol=1e-5) and torch.allclose(second, 8 * x, atol=1e-5)
