"""The work that a user of this package has it do on one GPU, as cases that can be timed and compared.

    listed()            named cases: training steps, evaluation, attention alone, the ring of a context-parallel rank,
                        the layer kernels and the optimizer, from the smallest calls to the benchmark configurations
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program holds before the call: model, optimizer, batch, tensors (on the GPU)
    run(state)          one pass through the public entry points, and everything it computes
    work(case)          bytes and floating-point operations one pass cannot do without
    tolerance(case)     how far two correct implementations at the same precision may differ

Head dimensions 64 and 128 are those of the configurations (LLaMA-50M and the long-context ones); 32 and 96 stand for
smaller and odd models.  Sizes are those of the configurations, of their micro-batches and shards, and ragged ones.
"""
from __future__ import annotations

import math

import torch

from maltos_amd import ops
from maltos_amd.gemm_tuning import tuned_gemms_off, use_tuned_gemms
from maltos_amd.grad_clip import clip_grad_norm_, clip_grad_norm_fused_
from maltos_amd.graph_step import CapturedForwardBackward
from maltos_amd.llama import LlamaConfig, LlamaForCausalLM, set_grad_accumulation_into_buffers
from maltos_amd.optim import FusedAdamW, MasterWeightsOptimizer
from maltos_amd.ring_attention import zigzag_ring_attention

DEV = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
LLAMA_50M = dict(vocab=32000, hidden=512, inter=1376, layers=8, heads=8, kv_heads=8)
LLAMA_TINY = dict(vocab=8192, hidden=256, inter=688, layers=4, heads=4, kv_heads=4)


def listed() -> list[dict]:
    return [
        # the LLaMA-50M training step of the benchmark: eager, gradients in flat buffers, clip on the device
        dict(name="train_50m", kind="train", dtype="bf16", batch=8, seq=2048, packed=False, form="eager", **LLAMA_50M),
        # the same step with forward and backward replayed from a graph, the form for launch-bound loops
        dict(name="train_50m_graph", kind="train", dtype="bf16", batch=8, seq=2048, packed=False, form="graph", **LLAMA_50M),
        # one micro-batch of packed documents, as gradient accumulation feeds them to a rank (one row of about 1024 tokens)
        dict(name="train_50m_packed_row", kind="train", dtype="bf16", batch=1, seq=1023, packed=True, form="eager", **LLAMA_50M),
        # the tiny fp32 model that recipes are checked with; the clip reads the norm on the host, as the step runner does
        dict(name="train_tiny_fp32", kind="train", dtype="fp32", batch=8, seq=256, packed=False, form="eager", **LLAMA_TINY),
        # evaluation: logits of a ragged batch, no gradients
        dict(name="eval_50m_ragged", kind="eval", dtype="bf16", batch=3, seq=777, packed=False, **LLAMA_50M),
        # the largest single attention: the headline configuration, forward and backward
        dict(name="attn_causal_4096", kind="attention", dtype="bf16", batch=4, heads=16, kv_heads=16, q_len=4096, k_len=4096,
             head_dim=128, causal=True),
        # a short unaligned sequence: the smallest call, all latency
        dict(name="attn_short", kind="attention", dtype="bf16", batch=2, heads=4, kv_heads=4, q_len=200, k_len=200, head_dim=64,
             causal=True),
        # fp32 attention of a checked recipe with grouped heads and an odd length
        dict(name="attn_fp32_odd", kind="attention", dtype="fp32", batch=2, heads=8, kv_heads=4, q_len=777, k_len=777, head_dim=64,
             causal=True),
        # packed documents with grouped-query heads: one attention layer over 8192-token rows
        dict(name="attn_packed_gqa", kind="packed", dtype="bf16", batch=2, heads=32, kv_heads=8, seq=8192, head_dim=128, doc=1056),
        # one rank of zigzag ring attention over 32768 tokens
        dict(name="ring_rank", kind="ring", dtype="bf16", heads=16, local=8192, head_dim=128, world=4, rank=1),
        # the layer kernels alone on a ragged number of rows and a vocabulary that no vector width divides
        dict(name="layers_ragged", kind="layers", dtype="bf16", rows=1021, hidden=768, inter=2056, heads=12, head_dim=64, vocab=50257),
        # norm, clip and AdamW over the flat buffers of the 50M model, as the sharded optimizer layouts call them
        dict(name="optim_flat_50m", kind="optim", dtype="bf16", params=58_073_600),
    ]


# ---- drawn cases --------------------------------------------------------------------------------------------------
def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_model(rng, dtype: str) -> dict:
    head_dim = rng.choice([64, 64, 64, 128])
    hidden = head_dim * rng.choice([2, 4, 6, 8] if head_dim == 64 else [2, 4])
    heads = hidden // head_dim
    return dict(vocab=rng.choice([8192, 16001, 32000]) if dtype == "bf16" else 8192, hidden=hidden, inter=8 * (hidden // 3),
                layers=rng.randint(2, 8 if dtype == "bf16" else 4), heads=heads,
                kv_heads=rng.choice([k for k in (heads, heads // 2, heads // 4) if k and heads % k == 0]))


def draw(rng) -> dict:
    kind = rng.choice(["train", "train", "train", "eval", "attention", "attention", "attention", "packed", "ring", "layers", "optim"])
    if kind in ("train", "eval"):
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        case = dict(kind=kind, dtype=dtype, batch=0, seq=_log_int(rng, 96, 2048), packed=rng.random() < 0.4, **_draw_model(rng, dtype))
        most = 16384 if dtype == "bf16" else 2048
        case["seq"] = min(case["seq"], most)
        case["batch"] = max(1, min(16, _log_int(rng, 1, max(2, most // case["seq"]))))
        while case["batch"] > 1 and case["batch"] * case["seq"] > most:
            case["batch"] -= 1
        if kind == "train":
            case["form"] = rng.choice(["eager", "eager", "graph"]) if dtype == "bf16" else "eager"
        return case
    if kind == "attention":
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        head_dim = rng.choice([64, 64, 64, 128, 128, 128, 32, 96])
        group = rng.choice([1, 1, 2, 4])
        q_len = _log_int(rng, 64, 8192 if dtype == "bf16" and head_dim in (64, 128) else 1024)
        kv_heads = rng.randint(1, 8)
        case = dict(kind=kind, dtype=dtype, batch=rng.randint(1, 8), heads=group * kv_heads, kv_heads=kv_heads, q_len=q_len,
                    k_len=q_len * rng.choice([1, 1, 1, 2]), head_dim=head_dim, causal=rng.random() < 0.7)
        most = 9.6e11 if dtype == "bf16" and head_dim in (64, 128) else 3e10
        while work(case)["flops"] > most:
            if case["batch"] > 1:
                case["batch"] -= 1
            else:
                case["q_len"], case["k_len"] = max(64, case["q_len"] * 3 // 4), max(64, case["k_len"] * 3 // 4)
        return case
    if kind == "packed":
        group = rng.choice([1, 2, 4])
        seq = _log_int(rng, 500, 8192)
        kv_heads = rng.randint(2, 8)
        return dict(kind=kind, dtype="bf16", batch=rng.randint(1, 2 if seq > 4096 else 4), heads=group * kv_heads, kv_heads=kv_heads, seq=seq,
                    head_dim=rng.choice([64, 128]), doc=_log_int(rng, 64, 2048))
    if kind == "ring":
        world = rng.choice([2, 3, 4])
        return dict(kind=kind, dtype="bf16", heads=rng.randint(2, 16), local=2 * _log_int(rng, 256, 3584), head_dim=rng.choice([64, 128]),
                    world=world, rank=rng.randrange(world))
    if kind == "layers":
        heads, head_dim = rng.randint(2, 16), rng.choice([64, 128])
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        return dict(kind=kind, dtype=dtype, rows=_log_int(rng, 64, 6000 if dtype == "bf16" else 2048), hidden=8 * rng.randint(32, 256),
                    inter=8 * rng.randint(64, 512), heads=heads, head_dim=head_dim,
                    vocab=rng.choice([8192, 32000, 50257, rng.randint(1000, 60000)]))
    return dict(kind="optim", dtype="bf16", params=_log_int(rng, 100_000, 58_000_000))


# ---- what a program holds before the call -------------------------------------------------------------------------
def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(gen, *shape, dtype=torch.bfloat16) -> torch.Tensor:
    return torch.randn(*shape, generator=gen, device=DEV).to(dtype)


def _documents(batch: int, seq: int, mean: int, seed: int):
    """int64 positions and sequence ids of packed rows: documents of 64 .. 2 * mean - 64 tokens (at least 16), the last
    one of a row cut off."""
    gen = torch.Generator().manual_seed(seed)
    lo, hi = max(16, min(64, mean // 2)), max(32, 2 * mean - 64)
    count = -(-seq // lo) + 1
    lengths = torch.randint(lo, hi + 1, (batch, count), generator=gen)
    ends = lengths.cumsum(1)
    index = torch.arange(seq).expand(batch, seq).contiguous()
    doc = torch.searchsorted(ends, index, right=True)
    starts = torch.cat([torch.zeros(batch, 1, dtype=torch.long), ends], dim=1)
    return index - starts.gather(1, doc), doc


def _batch(case: dict, seed: int) -> dict:
    gen = _generator(seed)
    ids = torch.randint(0, case["vocab"], (case["batch"], case["seq"] + 1), generator=gen, device=DEV)
    batch = {"input_ids": ids[:, :-1].clone(), "labels": ids[:, 1:].clone()}
    if case["packed"]:
        pos, doc = _documents(case["batch"], case["seq"], max(32, case["seq"] // 4), seed)
        last = torch.ones_like(pos, dtype=torch.bool)
        last[:, :-1] = doc[:, 1:] != doc[:, :-1]
        batch["labels"][last.to(DEV)] = -100   # the last token of a document has no target
        batch["position_ids"], batch["sequence_ids"] = pos.to(DEV), doc.to(DEV)
    return batch


def _model(case: dict, seed: int) -> LlamaForCausalLM:
    config = LlamaConfig(vocab_size=case["vocab"], hidden_size=case["hidden"], intermediate_size=case["inter"], num_hidden_layers=case["layers"],
                         num_attention_heads=case["heads"], num_key_value_heads=case["kv_heads"], max_position_embeddings=2048, rms_norm_eps=1e-5)
    with torch.device(DEV):
        model = LlamaForCausalLM(config)
    gen = _generator(seed)
    with torch.no_grad():
        for p in model.parameters():
            if p.dim() >= 2:
                p.normal_(0.0, 0.02, generator=gen)
    return model.to(DTYPES[case["dtype"]])


def _prepare_train(case: dict, seed: int) -> dict:
    # as the benchmark and the step runner: the shipped GEMM selection, weight gradients added into bound buffers
    use_tuned_gemms()
    model = _model(case, seed)
    set_grad_accumulation_into_buffers(model)
    adamw = lambda params: FusedAdamW(params, lr=3e-4, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1)
    params = list(model.parameters())
    opt = MasterWeightsOptimizer(params, optimizer_factory=adamw) if case["dtype"] == "bf16" else adamw(params)
    batch = _batch(case, seed + 1)
    state = {"model": model, "opt": opt, "batch": batch}
    if case["form"] == "graph":
        state["captured"] = CapturedForwardBackward(model, batch, embed=model.embed_tokens, clear_grads=lambda: opt.zero_grad(set_to_none=True))
    return state


def _prepare_eval(case: dict, seed: int) -> dict:
    use_tuned_gemms()
    batch = _batch(case, seed + 1)
    del batch["labels"]
    return {"model": _model(case, seed), "batch": batch}


def _prepare_attention(case: dict, seed: int) -> dict:
    # [B, S, H, D] storage seen as [B, H, S, D]: what the projections of a layer hand over
    gen, dtype = _generator(seed), DTYPES[case["dtype"]]
    B, H, Hkv, D = case["batch"], case["heads"], case["kv_heads"], case["head_dim"]
    rows = lambda S, heads: _normal(gen, B, S, heads, D, dtype=dtype).transpose(1, 2)
    return {"q": rows(case["q_len"], H).requires_grad_(True), "k": rows(case["k_len"], Hkv).requires_grad_(True),
            "v": rows(case["k_len"], Hkv).requires_grad_(True), "dout": rows(case["q_len"], H),
            "mask": ops.MASK_CAUSAL if case["causal"] else ops.MASK_NONE}


def _prepare_packed(case: dict, seed: int) -> dict:
    gen = _generator(seed)
    B, S, H, D = case["batch"], case["seq"], case["heads"], case["head_dim"]
    rows, Hkv = lambda heads: _normal(gen, B, S, heads, D).transpose(1, 2), case["kv_heads"]
    pos, doc = (t.to(DEV, torch.int32) for t in _documents(B, S, case["doc"], seed))
    return {"q": rows(H).requires_grad_(True), "k": rows(Hkv).requires_grad_(True), "v": rows(Hkv).requires_grad_(True), "dout": rows(H),
            "pos": pos, "doc": doc}


def _prepare_ring(case: dict, seed: int) -> dict:
    gen = _generator(seed)
    rows = lambda: _normal(gen, 1, case["heads"], case["local"], case["head_dim"])
    chunks = [(rows().requires_grad_(True), rows().requires_grad_(True)) for _ in range(case["world"])]
    return {"q": rows().requires_grad_(True), "dout": rows(), "chunks": chunks, "rank": case["rank"], "world": case["world"]}


def _prepare_layers(case: dict, seed: int) -> dict:
    gen, dtype = _generator(seed), DTYPES[case["dtype"]]
    N, h, I, H, D, V = (case[k] for k in ("rows", "hidden", "inter", "heads", "head_dim", "vocab"))
    rnd = lambda *shape: _normal(gen, *shape, dtype=dtype)
    angles = torch.arange(N, device=DEV)[:, None] * (10000.0 ** (-torch.arange(0, D, 2, device=DEV) / D))[None, :]
    labels = torch.randint(0, V, (N,), generator=gen, device=DEV)
    labels[::17] = -100   # rows without a target: document ends, padding
    leaf = lambda t: t.requires_grad_(True)
    return {"x": leaf(rnd(N, h)), "res": leaf(rnd(N, h)), "w": leaf(1 + 0.1 * rnd(h)), "dh": rnd(N, h), "dy": rnd(N, h),
            "q": leaf(rnd(1, N, H, D).transpose(1, 2)), "k": leaf(rnd(1, N, H, D).transpose(1, 2)), "dq": rnd(1, N, H, D).transpose(1, 2),
            "dk": rnd(1, N, H, D).transpose(1, 2), "cos": angles.cos().to(dtype), "sin": angles.sin().to(dtype), "gate": leaf(rnd(N, I)),
            "up": leaf(rnd(N, I)), "dact": rnd(N, I), "logits": leaf(rnd(N, V)), "labels": labels}


def _prepare_optim(case: dict, seed: int) -> dict:
    gen, n = _generator(seed), case["params"]
    f32 = lambda scale: torch.randn(n, generator=gen, device=DEV) * scale
    return {"p": f32(0.02), "m": f32(1e-3), "v": f32(1e-3).square_(), "grad": f32(1e-3).bfloat16(), "grad32": torch.empty(n, device=DEV),
            "model": torch.empty(n, device=DEV, dtype=torch.bfloat16), "step": 100}


_PREPARE = {"train": _prepare_train, "eval": _prepare_eval, "attention": _prepare_attention, "packed": _prepare_packed,
            "ring": _prepare_ring, "layers": _prepare_layers, "optim": _prepare_optim}


def prepare(case: dict, seed: int) -> dict:
    tuned_gemms_off()
    return _PREPARE[case["kind"]](case, seed) | {"kind": case["kind"]}


# ---- one pass -----------------------------------------------------------------------------------------------------
def _run_train(s: dict) -> dict:
    model, opt, batch = s["model"], s["opt"], s["batch"]
    if "captured" in s:
        loss = s["captured"](batch)
    else:
        loss = model(batch)
        loss.backward()
    if isinstance(opt, MasterWeightsOptimizer):
        norm = clip_grad_norm_fused_(opt, 1.0)
        opt.step()
        opt.zero_grad(set_to_none=True)
        first = opt.state[opt.master_params[0]]   # every parameter's moments are views of one flat buffer each
        return {"loss": loss.detach(), "sq_norm": norm, "grads": opt.flat_master_grad, "master": opt.flat_master, "model": opt.flat_model,
                "exp_avg": first["exp_avg"]._base, "exp_avg_sq": first["exp_avg_sq"]._base}
    params = [p for group in opt.param_groups for p in group["params"]]
    norm = clip_grad_norm_(opt, 1.0)
    opt.step()
    grads = [p.grad for p in params]
    opt.zero_grad(set_to_none=True)
    # weights and moments of the matrices of the first layer, the embedding and the head stand beside every parameter's gradient
    return {"loss": loss.detach(), "norm": norm, "grads": grads, "embed": params[0].detach(), "exp_avg": opt.state[params[0]]["exp_avg"],
            "exp_avg_sq": opt.state[params[0]]["exp_avg_sq"], "layer": [p.detach() for p in params[1:10]], "head": params[-1].detach()}


def _run_eval(s: dict) -> torch.Tensor:
    with torch.no_grad():
        return s["model"](s["batch"])


def _run_attention(s: dict) -> tuple:
    out, lse = ops.attention(s["q"], s["k"], s["v"], mask_mode=s["mask"], return_lse=True)
    return (out.detach(), lse.detach(), *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"]))


def _run_packed(s: dict) -> tuple:
    ops.clear_doc_plan_cache()   # a new batch brings new ids: one layer pays for its own mask plan
    out, lse = ops.attention(s["q"], s["k"], s["v"], mask_mode=ops.MASK_DOC, q_pos=s["pos"], k_pos=s["pos"], q_seq=s["doc"], k_seq=s["doc"],
                             return_lse=True)
    return (out.detach(), lse.detach(), *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"]))


def _run_ring(s: dict) -> tuple:
    out, lse = zigzag_ring_attention(s["q"], s["chunks"], rank=s["rank"], world_size=s["world"], return_lse=True)
    return (out.detach(), lse, *torch.autograd.grad(out, (s["q"], *(t for chunk in s["chunks"] for t in chunk)), s["dout"]))


def _run_layers(s: dict) -> dict:
    h, y = ops.add_rms_norm(s["x"], s["res"], s["w"], 1e-5)
    norm = torch.autograd.grad((h, y), (s["x"], s["res"], s["w"]), (s["dh"], s["dy"]))
    qr, kr = ops.rope_pair(s["q"], s["k"], s["cos"], s["sin"])
    rope = torch.autograd.grad((qr, kr), (s["q"], s["k"]), (s["dq"], s["dk"]))
    act = ops.swiglu(s["gate"], s["up"])
    swiglu = torch.autograd.grad(act, (s["gate"], s["up"]), s["dact"])
    loss = ops.cross_entropy(s["logits"], s["labels"])
    (dlogits,) = torch.autograd.grad(loss, s["logits"])
    return {"norm": (h.detach(), y.detach(), *norm), "rope": (qr.detach(), kr.detach(), *rope), "swiglu": (act.detach(), *swiglu),
            "loss": loss.detach(), "dlogits": dlogits}


def _run_optim(s: dict) -> dict:
    sq = torch.empty((), dtype=torch.float64, device=DEV)
    ops.grad_to_f32_(s["grad32"], s["grad"], sq_out=sq)
    s["step"] += 1
    ops.adamw_step_(s["p"], s["grad32"], s["m"], s["v"], lr=3e-4, beta1=0.9, beta2=0.95, eps=1e-8, weight_decay=0.1, step=s["step"],
                    p_lowp=s["model"], sq_norm=sq, max_norm=1.0)
    return {k: s[k] for k in ("grad32", "p", "m", "v", "model")} | {"sq": sq}


_RUN = {"train": _run_train, "eval": _run_eval, "attention": _run_attention, "packed": _run_packed, "ring": _run_ring,
        "layers": _run_layers, "optim": _run_optim}


def run(state: dict):
    return _RUN[state["kind"]](state)


# ---- what a pass cannot do without --------------------------------------------------------------------------------
def _pairs(case: dict) -> float:
    """Visible (query, key) pairs of one head and row."""
    if case["kind"] == "packed" or case.get("packed"):
        mean = case["doc"] if case["kind"] == "packed" else max(32, case["seq"] // 4)
        return case["seq"] * min(mean, case["seq"]) * 0.66   # sum of L^2 / 2 for lengths spread evenly around the mean
    if case["kind"] == "ring":
        return case["world"] * case["local"] ** 2 / 2.0
    if case["kind"] in ("train", "eval"):
        return case["seq"] ** 2 / 2.0
    q, k = case["q_len"], case["k_len"]
    return q * k - q * q / 2.0 if case["causal"] else float(q * k)


def _params(case: dict) -> int:
    h = case["hidden"]
    kv = h * case["kv_heads"] // case["heads"]
    return case["layers"] * (2 * h * h + 2 * h * kv + 3 * h * case["inter"] + 2 * h) + 2 * case["vocab"] * h + h


def work(case: dict) -> dict:
    kind, e = case["kind"], 2 if case["dtype"] == "bf16" else 4
    if kind in ("train", "eval"):
        tokens, n = case["batch"] * case["seq"], _params(case)
        passes = 3 if kind == "train" else 1
        flops = passes * 2.0 * tokens * (n - case["vocab"] * case["hidden"])
        flops += (3.5 if kind == "train" else 1.0) * 4.0 * case["batch"] * case["layers"] * case["hidden"] * _pairs(case)
        # training: weights read, gradient written, master weight and two moments read and written
        return {"flops": flops, "bytes": n * (24.0 + 3 * e if kind == "train" else e) + (0 if kind == "train" else e * tokens * case["vocab"])}
    if kind in ("attention", "packed"):
        Sq, Sk = (case["q_len"], case["k_len"]) if kind == "attention" else (case["seq"], case["seq"])
        B, H, D = case["batch"], case["heads"], case["head_dim"]
        rows = 4 * H * Sq + 4 * case["kv_heads"] * Sk   # q, out, dout, dq and k, v, dk, dv
        return {"flops": 3.5 * 4.0 * B * H * D * _pairs(case), "bytes": float(B * (rows * D * e + 4 * H * Sq))}
    if kind == "ring":
        H, S, D = case["heads"], case["local"], case["head_dim"]
        return {"flops": 3.5 * 4.0 * H * D * _pairs(case), "bytes": float(H * S * (D * e * (4 + 4 * case["world"]) + 4))}
    if kind == "layers":
        N, h, I, H, D, V = (case[k] for k in ("rows", "hidden", "inter", "heads", "head_dim", "vocab"))
        return {"flops": 0.0, "bytes": float(N * e * (4 * h + 4 * h + 8 * H * D + 3 * I + 5 * I + 2 * V))}
    return {"flops": 0.0, "bytes": case["params"] * (2 + 4 + 12 + 12 + 2.0)}


def tolerance(case: dict) -> dict:
    if case["kind"] == "train":   # gradients through every layer, and the moments made of them
        return {"rel": 2e-2} if case["dtype"] == "bf16" else {"rel": 1e-4, "max": 0.05}
    if case["kind"] == "optim":
        return {"rel": 1e-5, "max": 1e-2}   # the bf16 copy of a weight may round the other way
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 1e-5, "max": 1e-2}
