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
