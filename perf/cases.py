"""The work that performance is measured on: training steps, served requests and the standalone attention ops, each through the
entry point that a user's program calls, over the range of sizes that it is used at.

* "train": one step (forward, backward, AdamW) of the Llama decoder through `initialize`, ZeRO-3, bf16
* "serve": requests through the ragged inference engine: all prompts in one `put`, `steps` decode steps for all of them, `flush`.
  Model "llama" is the uniform decoder, "lefisun" the hybrid one of the serving benchmark (rotary attention with a sink beside a
  matrix memory, retention, routed experts)
* "evoformer": forward and backward of the attention with a per-key and a pair bias
* "sparse": forward and backward of block-sparse attention

`exact` states the same functions in 64 bits in plain torch."""
import math

import numpy as np
import torch

BF16, F64 = torch.bfloat16, torch.float64
EPS, THETA = 1e-5, 10000.0


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    def train(name, **kw):
        return dict(name=name, kind="train", **kw)

    def serve(name, **kw):
        return dict(name=name, kind="serve", **kw)

    return [
        # the benchmark's "tiny" model on a short batch, as in a debugging run or a small model's fine-tuning: launches count
        train("train_tiny_1x128", width=1024, layers=2, heads=8, kv_heads=8, ff=2816, vocab=8000, batch=1, seq=128),
        # grouped keys, a sequence length that fills no tile
        train("train_2048_gqa_3x1000", width=2048, layers=2, heads=16, kv_heads=4, ff=5632, vocab=32000, batch=3, seq=1000),
        # Llama-2-7B's layers at its training length (two of the 32)
        train("train_4096_2x4096", width=4096, layers=2, heads=32, kv_heads=32, ff=11008, vocab=32000, batch=2, seq=4096),
        # a long document is read: attention and large products
        serve("prefill_4096_1x8192", model="llama", width=4096, layers=2, prompts=1, length=8192, ragged=False, steps=0),
        # many short requests of unequal length arrive at once
        serve("prefill_2048_21x300", model="llama", width=2048, layers=4, prompts=21, length=300, ragged=True, steps=0),
        # one interactive user: weights are streamed for one token at a time
        serve("decode_4096_b1", model="llama", width=4096, layers=4, prompts=1, length=100, ragged=False, steps=32),
        # a server under load, prompts of some length and answers to all of them together
        serve("decode_4096_b48", model="llama", width=4096, layers=2, prompts=48, length=160, ragged=True, steps=24),
        # the small width, a moderate batch over longer contexts
        serve("decode_2048_b12", model="llama", width=2048, layers=4, prompts=12, length=640, ragged=True, steps=32),
        # the hybrid decoder with routed experts: prompts, and a batch of answers
        serve("lefisun_prefill_4096_4x2048", model="lefisun", width=4096, layers=2, prompts=4, length=2048, ragged=False, steps=0),
        serve("lefisun_decode_2048_b16", model="lefisun", width=2048, layers=2, prompts=16, length=200, ragged=True, steps=24),
        # the Evoformer benchmark's shape
        dict(name="evoformer_256x256", kind="evoformer", batch=1, rows=256, seq=256, heads=4, dim=32),
        # BigBird over a long document with padding at its end
        dict(name="bigbird_2x16384", kind="sparse", layout="bigbird", batch=2, heads=8, seq=16384, dim=128, block=64, padding=True),
    ]


def _log(rng, lo, hi):
    """A whole number, even over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("train", "train", "prefill", "prefill", "decode", "decode", "lefisun", "lefisun", "evoformer", "sparse"))
    if kind == "train":
        width = rng.choice((1024, 2048, 4096))
        heads = width // 128
        seq = _log(rng, 100, 4096)
        return dict(kind="train", width=width, layers=2, heads=heads, kv_heads=heads // rng.choice((1, 2, 4)),
                    ff=rng.choice((2816, 5632, 8192)), vocab=rng.choice((8000, 32000)), batch=_log(rng, 1, max(1, 8192 // seq)), seq=seq)
    if kind in ("prefill", "decode", "lefisun"):
        steps = 0 if kind == "prefill" or (kind == "lefisun" and rng.random() < 0.5) else rng.randint(8, 32)
        prompts = _log(rng, 1, 48)
        length = _log(rng, 20, min(8192 // prompts, 8192 if steps == 0 else 1024))
        width = rng.choice((2048, 4096))
        return dict(kind="serve", model="lefisun" if kind == "lefisun" else "llama", width=width, layers=2, prompts=prompts,
                    length=length, ragged=rng.random() < 0.7, steps=steps)
    if kind == "evoformer":
        return dict(kind="evoformer", batch=1, rows=_log(rng, 24, 256), seq=rng.randint(40, 256), heads=rng.choice((4, 8)),
                    dim=32)
    return dict(kind="sparse", layout=rng.choice(("bigbird", "fixed")), batch=rng.randint(1, 2), heads=rng.choice((4, 8)),
                seq=128 * _log(rng, 8, 128), dim=rng.choice((64, 128)), block=rng.choice((32, 64)), padding=rng.random() < 0.5)


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(int(seed) % (1 << 62))


def _normal(g, shape, std=1.0, mean=0.0, dtype=BF16):
    return torch.empty(shape, device="cuda", dtype=torch.float32).normal_(mean, std, generator=g).to(dtype)


def _train_weights(c, seed):
    """{parameter name: bf16 tensor} in the model's layout: q, k and v rows, gate and up rows together."""
    g, W, D = _gen(seed), c["width"], c["width"] // c["heads"]
    out_std = 0.02 / math.sqrt(2 * c["layers"])   # (projections back into the residual, scaled down by its depth)
    w = {"model.embed_tokens.weight": _normal(g, (c["vocab"], W), 0.1)}
    for i in range(c["layers"]):
        p = f"model.layers.{i}."
        w[p + "input_layernorm.weight"] = _normal(g, (W, ), 0.1, 1.0)
        w[p + "self_attn.qkv_proj.weight"] = _normal(g, ((c["heads"] + 2 * c["kv_heads"]) * D, W), 0.02)
        w[p + "self_attn.o_proj.weight"] = _normal(g, (W, W), out_std)
        w[p + "post_attention_layernorm.weight"] = _normal(g, (W, ), 0.1, 1.0)
        w[p + "mlp.gate_up_proj.weight"] = _normal(g, (2 * c["ff"], W), 0.02)
        w[p + "mlp.down_proj.weight"] = _normal(g, (W, c["ff"]), out_std)
    w["model.norm.weight"] = _normal(g, (W, ), 0.1, 1.0)
    w["lm_head.weight"] = _normal(g, (c["vocab"], W), 0.02)
    return w


def _train_tokens(c, seed):
    return torch.randint(0, c["vocab"], (c["batch"], c["seq"]), device="cuda", generator=_gen(seed + 1))


ADAM = dict(lr=1e-4, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1)
CLIP = 1.0

SERVE_VOCAB = 32000
EXPERTS, TOP, GROUPS, KEEP, CHUNK, GATE_CAP = 32, 4, 4, 2, 2048, 15.0
LEFT, RIGHT, EMBED_SCALE, CODE = 0.8, 0.6, 50.0, 8


def _sizes(c):
    """Heads of 128, grouped keys and the feed-forward of the serving benchmark."""
    h = c["width"] // 128
    return dict(heads=h, kv=8 if h > 8 else h, ff={2048: 5632, 4096: 14336}[c["width"]])


def _requests(c, seed):
    """(prompts, tokens of every decode step), on the host as a server receives them."""
    rng = np.random.default_rng(seed + 2)
    lens = [int(rng.integers(max(1, c["length"] // 2), c["length"] + 1)) if c["ragged"] else c["length"] for _ in range(c["prompts"])]
    new = lambda n: torch.from_numpy(rng.integers(0, SERVE_VOCAB, n))  # noqa: E731
    return [new(n) for n in lens], [[new(1) for _ in lens] for _ in range(c["steps"])]


def _serve_weights(c, seed):
    """{parameter name: tensor} in the model's layout. Projections back into the residual are scaled down by its depth. The routers
    go by the token: they read the last columns of the residual, which the embedding alone writes, with values that leave no
    token near a tie, so that rounding in the layers changes no expert."""
    g, s, W, D, V = _gen(seed), _sizes(c), c["width"], 128, SERVE_VOCAB
    out_std = 0.02 / math.sqrt(2 * c["layers"])
    w = {"embed": _normal(g, (V, W), 0.02 if c["model"] == "lefisun" else 0.25)}
    f32 = dict(dtype=torch.float32)
    for i in range(c["layers"]):
        p = f"layers.{i}."
        if c["model"] == "llama":
            w[p + "ln1_w"], w[p + "ln2_w"] = _normal(g, (W, ), 0.1, 1.0), _normal(g, (W, ), 0.1, 1.0)
            w[p + "qkv_w"] = _normal(g, ((s["heads"] + 2 * s["kv"]) * D, W), 0.02)
            w[p + "o_w"] = _normal(g, (W, s["heads"] * D), out_std)
            w[p + "fc1_w"], w[p + "fc2_w"] = _normal(g, (2 * s["ff"], W), 0.02), _normal(g, (W, s["ff"]), out_std)
            continue
        H, R, ff = s["heads"], s["heads"] // 2, s["ff"] // TOP
        w[p + "res1.norm_w"], w[p + "res2.norm_w"] = _normal(g, (W, ), 0.1, 1.0, **f32), _normal(g, (W, ), 0.1, 1.0, **f32)
        if i % 2 == 0:
            left = (H + 2 * s["kv"]) * D
            w[p + "qkv_w"] = _normal(g, (left + 4 * R * D + 2 * R, W), 0.02)
            w[p + "o_w"] = _normal(g, (W, (H + R) * D), out_std)
            w[p + "left_bias"] = _normal(g, (left, ), 0.1, **f32)
            w[p + "left_q_norm"], w[p + "left_k_norm"] = _normal(g, (H * D, ), 0.1, 1.0, **f32), _normal(g, (s["kv"] * D, ), 0.1, 1.0, **f32)
            w[p + "right_i_b"], w[p + "right_f_b"] = _normal(g, (R, ), 0.5, **f32), _normal(g, (R, ), 1.0, 3.0, **f32)
            w[p + "right_head_norm"] = _normal(g, (R * D, ), 0.06, RIGHT, **f32)  # (carries the side's factor)
        else:
            w[p + "qkv_w"] = _normal(g, (4 * H * D, W), 0.02)
            w[p + "o_w"] = _normal(g, (W, H * D), out_std)
        w[p + "router_w"] = _normal(g, (EXPERTS, W), 0.5)
        w[p + "router_w"][:, :-CODE] = 0
        w[p + "res2.norm_w"][-CODE:] = 1
        w[p + "fc1_w"], w[p + "fc2_w"] = _normal(g, (EXPERTS, 2 * ff, W), 0.02), _normal(g, (EXPERTS, W, ff), out_std)
        w[p + "o_w"][-CODE:] = 0
        w[p + "fc2_w"][:, -CODE:] = 0
    if c["model"] == "lefisun":
        _part_routes(w, g, c["layers"])
    w["norm_w"] = _normal(g, (W, ), 0.1, 1.0, dtype=torch.float32 if c["model"] == "lefisun" else BF16)
    w["lm_head"] = w["embed"] if c["model"] == "lefisun" else _normal(g, (V, W), 0.02)
    return w


def _part_routes(w, g, layers):
    """Draws the router's columns of the embedding anew for every token that has a near tie in some layer."""
    todo = torch.arange(SERVE_VOCAB, device="cuda")
    while todo.numel():
        code = _normal(g, (todo.numel(), CODE), 0.02)
        w["embed"][todo, -CODE:] = code
        near = torch.zeros(todo.numel(), dtype=torch.bool, device="cuda")
        for i in range(layers):
            z = code.float() @ w[f"layers.{i}.router_w"][:, -CODE:].float().t()
            least = 0.04 * z.std(-1)
            best = z.view(-1, GROUPS, EXPERTS // GROUPS).max(-1).values
            top = best.topk(KEEP + 1, -1).values
            inside = z.masked_fill((best < top[:, KEEP - 1:KEEP]).repeat_interleave(EXPERTS // GROUPS, 1), -math.inf)
            scores = inside.topk(TOP + 1, -1).values
            near |= (top[:, KEEP - 1] - top[:, KEEP] < least) | (scores[:, TOP - 1] - scores[:, TOP] < least)
        todo = todo[near]


def _decays(heads):
    return [1 - 2**(-5 - 3 * i / heads) for i in range(heads)]


def _spec(c):
    from deepspeedsyclsupport_amd.inference.model_implementations.transformer import DSModelSpec
    s, D = _sizes(c), 128
    common = dict(vocab_size=SERVE_VOCAB, hidden_size=c["width"], num_layers=c["layers"], num_heads=s["heads"], num_kv_heads=s["kv"],
                  intermediate_size=s["ff"], head_dim=D, norm="rms", norm_eps=EPS)
    if c["model"] == "llama":
        return DSModelSpec(arch="llama", pos="rope", rope_theta=THETA, max_positions=16384, **common)
    h = s["heads"]
    mixers = ({"left": {"heads": h, "kv_heads": s["kv"], "dim": D, "vdim": D, "scale": D**-0.5, "mask": {"size": CHUNK},
                        "rot": {"base": 5e5, "dims": D // 2, "scaling": {"factor": 4.0}}},
               "right": {"heads": h // 2, "dim": D, "vdim": D, "gate_cap": GATE_CAP}, "left_scale": LEFT, "right_scale": RIGHT},
              {"heads": h, "dim": D, "vdim": D, "rot": {"base": 1e4, "dims": D}, "decay": _decays(h)})
    mlp = {"kind": "routed", "expert": {"ff": s["ff"] // TOP},
           "router": {"experts": EXPERTS, "top": TOP, "groups": {"count": GROUPS, "keep": KEEP}}}
    layers = tuple({"type": ("parallel", "retention")[i % 2], "mixer": mixers[i % 2], "mlp": mlp} for i in range(c["layers"]))
    return DSModelSpec(arch="lefisun", pos="none", residual="pre_norm", tie_embeddings=True, embed_scale=EMBED_SCALE,
                       layer_specs=layers, **common)


def _evoformer_inputs(c, seed):
    """Activations, a mask of some masked residues per row, pair biases, an output gradient."""
    g = _gen(seed)
    B, N, S, H, D = c["batch"], c["rows"], c["seq"], c["heads"], c["dim"]
    q, k, v = (_normal(g, (B, N, S, H, D)) for _ in range(3))
    gone = torch.rand((B, N, 1, 1, S), device="cuda", generator=g) < 0.1
    return q, k, v, torch.zeros_like(gone, dtype=BF16).masked_fill_(gone, -1e4), _normal(g, (B, 1, H, S, S)), _normal(g, (B, N, S, H, D))


def _sparse_layout(c, seed):
    """[blocks, blocks], for all heads: windows, global blocks and (BigBird) random ones."""
    n, rng = c["seq"] // c["block"], np.random.default_rng(seed + 3)
    i, j = np.arange(n)[:, None], np.arange(n)[None]
    if c["layout"] == "bigbird":
        lay = (abs(i - j) <= 1) | (i == 0) | (j == 0)
        lay[np.arange(n), rng.integers(0, n, n)] = True
    else:
        lay = (i // 4 == j // 4) | (j % 4 == 3)
    return torch.from_numpy(lay)


def _sparse_inputs(c, seed):
    g, shape = _gen(seed), (c["batch"], c["heads"], c["seq"], c["dim"])
    q, k, v, do = (_normal(g, shape) for _ in range(4))
    mask = None
    if c["padding"]:
        ends = torch.randint(c["seq"] - c["seq"] // 4, c["seq"] + 1, (c["batch"], 1), device="cuda", generator=g)
        mask = torch.zeros(c["batch"], c["seq"], device="cuda").masked_fill_(torch.arange(c["seq"], device="cuda")[None] >= ends, -1e4)
    return q, k, v, do, mask


# ------------------------------------------------------------------------------------------------ preparation
def _prepare_train(c, seed):
    import deepspeedsyclsupport_amd as ds
    from deepspeedsyclsupport_amd.models.llama import LlamaConfig, LlamaForCausalLM
    cfg = LlamaConfig(vocab_size=c["vocab"], hidden_size=c["width"], intermediate_size=c["ff"], num_hidden_layers=c["layers"],
                      num_attention_heads=c["heads"], num_key_value_heads=c["kv_heads"], max_position_embeddings=c["seq"],
                      rms_norm_eps=EPS, rope_theta=THETA)
    was = torch.get_default_dtype()
    torch.set_default_dtype(BF16)
    try:
        with torch.device("cuda"):
            model = LlamaForCausalLM(cfg)
    finally:
        torch.set_default_dtype(was)
    weights = _train_weights(c, seed)
    with torch.no_grad():
        for name, p in model.named_parameters():
            p.copy_(weights[name])
    config = {"train_micro_batch_size_per_gpu": c["batch"], "gradient_accumulation_steps": 1, "steps_per_print": 10**9,
              "bf16": {"enabled": True}, "gradient_clipping": CLIP,
              "optimizer": {"type": "AdamW", "params": {**ADAM, "betas": list(ADAM["betas"])}},
              "zero_optimization": {"stage": 3, "overlap_comm": True, "contiguous_gradients": True}}
    engine, _, _, _ = ds.initialize(model=model, config=config)
    return dict(case=c, engine=engine, params=list(engine.module.parameters()), ids=_train_tokens(c, seed))


def _prepare_serve(c, seed):
    from deepspeedsyclsupport_amd.inference.model_implementations.hybrid import model_class
    from deepspeedsyclsupport_amd.inference.v2 import AllocationMode, InferenceEngineV2, RaggedInferenceEngineConfig
    spec = _spec(c)
    model = model_class(spec)(spec, dtype=BF16, device="cuda")
    weights = _serve_weights(c, seed)
    with torch.no_grad():
        for name, p in model.named_parameters():
            p.copy_(weights[name])
    model.add_decode_layout()   # (what the engine factories do by default where memory allows it)
    prompts, steps = _requests(c, seed)
    block = 64
    blocks = sum(-(-(p.numel() + len(steps)) // block) + 1 for p in prompts)
    config = RaggedInferenceEngineConfig(
        state_manager={"memory_config": {"mode": AllocationMode.ALLOCATE, "size": blocks}, "max_ragged_batch_size": 8192,
                       "max_ragged_sequence_count": 64, "max_tracked_sequences": 64, "max_context": 16384},
        kv_cache={"block_size": block})
    return dict(case=c, engine=InferenceEngineV2(model, config), prompts=prompts, steps=steps)


def prepare(case, seed):
    if case["kind"] == "train":
        return _prepare_train(case, seed)
    if case["kind"] == "serve":
        return _prepare_serve(case, seed)
    if case["kind"] == "evoformer":
        q, k, v, mask, pair, do = _evoformer_inputs(case, seed)
        return dict(case=case, inputs=[t.requires_grad_() for t in (q, k, v, pair)], mask=mask, do=do)
    from deepspeedsyclsupport_amd.ops.sparse_attention import SparseSelfAttention, SparsityConfig
    lay = _sparse_layout(case, seed).long()

    class Given(SparsityConfig):   # (a layout of the user's own, as any of the configurations makes one)

        def make_layout(self, seq_len):
            return lay[None].expand(self.num_heads, -1, -1).contiguous()

    q, k, v, do, mask = _sparse_inputs(case, seed)
    attend = SparseSelfAttention(Given(num_heads=case["heads"], block=case["block"]), key_padding_mask_mode="add",
                                 max_seq_length=case["seq"])
    return dict(case=case, attend=attend, inputs=[t.requires_grad_() for t in (q, k, v)], mask=mask, do=do)


# ------------------------------------------------------------------------------------------------ one pass
def run(state):
    kind = state["case"]["kind"]
    if kind == "train":
        engine = state["engine"]
        loss = engine(state["ids"], labels=state["ids"])
        engine.backward(loss)
        grads = [p.grad for p in state["params"]]
        engine.step()
        return {"loss": loss.detach(), "grads": grads, "weights": [p.detach() for p in state["params"]]}
    if kind == "serve":
        engine, uids = state["engine"], list(range(len(state["prompts"])))
        logits = [engine.put(uids, state["prompts"])]
        for tokens in state["steps"]:
            logits.append(engine.put(uids, tokens))
        for u in uids:
            engine.flush(u)
        return logits
    if kind == "evoformer":
        from deepspeedsyclsupport_amd.ops.deepspeed4science import DS4Sci_EvoformerAttention
        q, k, v, pair = state["inputs"]
        out = DS4Sci_EvoformerAttention(q, k, v, [state["mask"], pair])
    else:
        out = state["attend"](*state["inputs"], key_padding_mask=state["mask"])
    return [out.detach(), *torch.autograd.grad(out, state["inputs"], state["do"])]


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _serve_work(c):
    """Mean prompt lengths stand for ragged ones. Every put reads the weights that its tokens use once, and the keys, values and
    states of its sequences; the logits are written."""
    s, W, D, L, V = _sizes(c), c["width"], 128, c["layers"], SERVE_VOCAB
    n, mean = c["prompts"], c["length"] * (0.75 if c["ragged"] else 1.0)
    puts = [(n * mean, 0.0, mean)] + [(n, mean + i, 1.0) for i in range(c["steps"])]   # (tokens, context before, new per sequence)
    nbytes = flops = 0.0
    for tokens, before, new in puts:
        per_token, matrices = V * W * n / tokens, V * W
        for i in range(L):
            if c["model"] == "llama":
                dense = W * (s["heads"] + 2 * s["kv"]) * D + W * s["heads"] * D + 3 * W * s["ff"]
                per_token, matrices = per_token + dense, matrices + dense
                att, span, kv = s["heads"], before + new / 2, s["kv"]
            else:
                H, R = s["heads"], s["heads"] // 2
                mix = W * ((H + 2 * s["kv"]) * D + 4 * R * D + 2 * R + (H + R) * D) if i % 2 == 0 else 5 * W * H * D
                expert = 3 * W * (s["ff"] // TOP)
                per_token += mix + W * EXPERTS + TOP * expert
                matrices += mix + W * EXPERTS + expert * EXPERTS * (1 - (1 - TOP / EXPERTS)**tokens)
                state = (R if i % 2 == 0 else H) * D * D
                nbytes += n * state * 4 * (2 if before else 1)
                flops += 4 * tokens * state
                if i % 2:
                    continue
                att, span, kv = H, min(before + new / 2, CHUNK), s["kv"]
            flops += 4 * tokens * att * D * span
            nbytes += 2 * 2 * kv * D * n * (min(before, CHUNK if c["model"] == "lefisun" else before) + new)
        flops += 2 * tokens * per_token
        nbytes += 2 * matrices + 2 * W * tokens + 2 * n * V
    return {"bytes": nbytes, "flops": flops}


def work(case):
    c = case
    if c["kind"] == "serve":
        return _serve_work(c)
    if c["kind"] == "train":
        W, L, T, D = c["width"], c["layers"], c["batch"] * c["seq"], c["width"] // c["heads"]
        layer = W * (c["heads"] + 2 * c["kv_heads"]) * D + W * W + 3 * W * c["ff"]
        dense = L * layer + c["vocab"] * W
        params = dense + c["vocab"] * W
        # weights read in both directions, gradients written and read, master and moments read and written, weights written
        nbytes = params * (2 + 2 + 2 + 2 + 24 + 2) + 8 * T
        # a layer's activations: its inputs kept for the backward pass, once written and once read
        nbytes += L * T * 2 * 2 * (4 * W + (c["heads"] + 2 * c["kv_heads"]) * D + 3 * c["ff"])
        return {"bytes": nbytes, "flops": 6 * dense * T + 3.5 * 4 * L * c["batch"] * c["heads"] * D * c["seq"]**2 / 2}
    if c["kind"] == "evoformer":
        z, S, H, D = c["batch"] * c["rows"], c["seq"], c["heads"], c["dim"]
        return {"bytes": 2 * (8 * z * S * H * D + z * S + 2 * c["batch"] * H * S * S), "flops": 14 * z * H * S * S * D}
    n = c["seq"] // c["block"]
    pairs = 5 * n + n if c["layout"] == "bigbird" else n * (4 + 0.75 * n / 4)
    return {"bytes": 2 * 8 * c["batch"] * c["heads"] * c["seq"] * c["dim"],
            "flops": 14 * c["batch"] * c["heads"] * pairs * c["block"]**2 * c["dim"]}


def tolerance(case):
    # bf16 operands, products and stored activations. Measured against `exact`: training gradients 0.005 to 0.018, the uniform
    # decoder with its bf16 residual 0.006 to 0.017, the hybrid one with its fp32 residual 0.003 to 0.004, attention 0.002 to 0.0025
    if case["kind"] == "train" or case.get("model") == "llama":
        return {"rel": 0.03}
    return {"rel": 0.015 if case["kind"] == "serve" else 0.01}


# ------------------------------------------------------------------------------------------------ the same in 64 bits
def _rms(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _turn(x, dims, base, factor=1.0):
    """x [..., n, d]: pairs (j, j + dims / 2) turn by position * base^(-2 j / dims) / factor."""
    n, half = x.shape[-2], dims // 2
    a = torch.arange(n, device=x.device, dtype=F64)[:, None] * base**(-2 * torch.arange(half, device=x.device, dtype=F64) / dims) / factor
    u, v = x[..., :half], x[..., half:dims]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin(), x[..., dims:]], -1)


def _attend(q, k, v, scale, chunk=0, sink=False):
    """q [H, n, d], k, v [G, n, d], causal; `chunk`: keys of the query's own chunk only; `sink`: a score of zero without a value."""
    n, rep, out = q.shape[1], q.shape[0] // k.shape[0], []
    i = torch.arange(n, device=q.device)
    hidden = i[None] > i[:, None]
    if chunk:
        hidden |= i[None] // chunk != i[:, None] // chunk
    for h in range(q.shape[0]):
        s = (q[h] @ k[h // rep].t() * scale).masked_fill_(hidden, -math.inf)
        if sink:
            s = torch.cat([s, s.new_zeros(n, 1)], 1)
        out.append(torch.softmax(s, -1)[:, :n] @ v[h // rep])
    return torch.stack(out)


def _heads(x, n):
    return x.reshape(x.shape[0], n, -1).transpose(0, 1)


def _joined(x):
    return x.transpose(0, 1).reshape(x.shape[1], -1)


def _train_exact(c, seed):
    w = {k: v.to(F64).requires_grad_() for k, v in _train_weights(c, seed).items()}
    ids, H, G = _train_tokens(c, seed), c["heads"], c["kv_heads"]
    D, losses = c["width"] // H, []
    for b in range(c["batch"]):
        x = w["model.embed_tokens.weight"][ids[b]]
        for i in range(c["layers"]):
            p = f"model.layers.{i}."
            qkv = (_rms(x) * w[p + "input_layernorm.weight"]) @ w[p + "self_attn.qkv_proj.weight"].t()
            q, k, v = (_heads(t, n) for t, n in zip(qkv.split([H * D, G * D, G * D], 1), (H, G, G)))
            x = x + _joined(_attend(_turn(q, D, THETA), _turn(k, D, THETA), v, D**-0.5)) @ w[p + "self_attn.o_proj.weight"].t()
            gate, up = ((_rms(x) * w[p + "post_attention_layernorm.weight"]) @ w[p + "mlp.gate_up_proj.weight"].t()).chunk(2, 1)
            x = x + (torch.nn.functional.silu(gate) * up) @ w[p + "mlp.down_proj.weight"].t()
        logits = (_rms(x) * w["model.norm.weight"])[:-1] @ w["lm_head.weight"].t()
        loss = torch.nn.functional.cross_entropy(logits, ids[b, 1:], reduction="sum") / (c["batch"] * (c["seq"] - 1))
        loss.backward()
        losses.append(loss.detach())
    grads = [t.grad for t in w.values()]
    norm = math.sqrt(sum(float((t * t).sum()) for t in grads))
    clip = CLIP / (norm + 1e-6) if norm > CLIP else 1.0
    lr, eps, wd = ADAM["lr"], ADAM["eps"], ADAM["weight_decay"]
    new = [t.detach() * (1 - lr * wd) - lr * (t.grad * clip) / ((t.grad * clip).abs() + eps) for t in w.values()]
    return {"loss": sum(losses), "grads": grads, "weights": new}


def _memory(q, k, v, log_in, log_forget):
    """Matrix memory, all weights of one head at once: the state is kept relative to a running maximum that starts at zero."""
    F = log_forget.cumsum(-1)
    z = (F[:, :, None] - F[:, None, :] + log_in[:, None, :]).masked_fill_(
        torch.ones(q.shape[1], q.shape[1], device=q.device, dtype=torch.bool).triu_(1), -math.inf)
    m = torch.maximum(z.max(-1).values, F)
    a = torch.exp(z - m[..., None]) * (q @ k.transpose(1, 2))
    return (a @ v) / (torch.maximum(a.sum(-1).abs(), torch.exp(-m)) + 1e-6)[..., None]


def _experts(w, p, h):
    z = torch.softmax(h @ w[p + "router_w"].t(), -1)
    best = z.view(-1, GROUPS, EXPERTS // GROUPS).max(-1).values
    allowed = torch.zeros_like(best, dtype=torch.bool).scatter_(1, best.topk(KEEP, -1).indices, True)
    wt, e = z.masked_fill(~allowed.repeat_interleave(EXPERTS // GROUPS, 1), -1.0).topk(TOP, -1)
    wt = wt / (wt.sum(-1, keepdim=True) + 1e-20)
    out = torch.zeros_like(h)
    for x in range(EXPERTS):
        t, j = (e == x).nonzero(as_tuple=True)
        gate, up = (h[t] @ w[p + "fc1_w"][x].t()).chunk(2, 1)
        out.index_add_(0, t, (torch.nn.functional.silu(gate) * up) @ w[p + "fc2_w"][x].t() * wt[t, j, None])
    return out


def _lefisun_layer(w, p, c, i, x):
    s, D = _sizes(c), 128
    H, G, R, silu = s["heads"], s["kv"], s["heads"] // 2, torch.nn.functional.silu
    qkv = (_rms(x) * w[p + "res1.norm_w"]) @ w[p + "qkv_w"].t()
    if i % 2 == 0:
        left = (H + 2 * G) * D
        q, k, v = (qkv[:, :left] + w[p + "left_bias"]).split([H * D, G * D, G * D], 1)
        q, k = _heads(_rms(q) * w[p + "left_q_norm"], H), _heads(_rms(k) * w[p + "left_k_norm"], G)
        q, k = (_turn(t, D // 2, 5e5, 4.0) for t in (q, k))
        one = _joined(_attend(q, k, _heads(v, G), D**-0.5, CHUNK, True)) * LEFT
        q, k, v, g, gi, gf = qkv[:, left:].split([R * D] * 4 + [R, R], 1)
        cap = lambda t: GATE_CAP * torch.tanh(t / GATE_CAP)  # noqa: E731
        mem = _memory(_heads(q, R) * D**-0.5, _heads(k, R), _heads(v, R), cap(gi + w[p + "right_i_b"]).t(),
                      torch.nn.functional.logsigmoid(cap(gf + w[p + "right_f_b"])).t())
        y = torch.cat([one, _joined(_rms(mem)) * w[p + "right_head_norm"] * torch.sigmoid(g)], 1)
    else:
        q, k, v, g = qkv.chunk(4, 1)
        q, k = (_turn(_heads(t, H), D, 1e4) for t in (q, k))
        n = torch.arange(x.shape[0], device=x.device)
        gap = (n[:, None] - n[None]).to(F64)
        v, out = _heads(v, H), []
        for h, a in enumerate(_decays(H)):
            out.append((q[h] @ k[h].t() * D**-0.5 * torch.pow(a, gap.clamp(min=0)) * (gap >= 0)) @ v[h])
        y = _joined(_rms(torch.stack(out))) * silu(g)
    x = x + y @ w[p + "o_w"].t()
    return x + _experts(w, p, _rms(x) * w[p + "res2.norm_w"])


def _serve_exact(c, seed):
    w = {k: v.to(F64) for k, v in _serve_weights(c, seed).items()}
    s, D, (prompts, steps) = _sizes(c), 128, _requests(c, seed)
    H, G, rows = s["heads"], s["kv"], []
    for b, prompt in enumerate(prompts):
        ids = torch.cat([prompt] + [t[b] for t in steps]).cuda()
        x = w["embed"][ids] * (EMBED_SCALE if c["model"] == "lefisun" else 1.0)
        for i in range(c["layers"]):
            p = f"layers.{i}."
            if c["model"] == "lefisun":
                x = _lefisun_layer(w, p, c, i, x)
                continue
            qkv = (_rms(x) * w[p + "ln1_w"]) @ w[p + "qkv_w"].t()
            q, k, v = (_heads(t, n) for t, n in zip(qkv.split([H * D, G * D, G * D], 1), (H, G, G)))
            x = x + _joined(_attend(_turn(q, D, THETA), _turn(k, D, THETA), v, D**-0.5)) @ w[p + "o_w"].t()
            gate, up = ((_rms(x) * w[p + "ln2_w"]) @ w[p + "fc1_w"].t()).chunk(2, 1)
            x = x + (torch.nn.functional.silu(gate) * up) @ w[p + "fc2_w"].t()
        rows.append((_rms(x[prompt.numel() - 1:]) * w["norm_w"]) @ w["lm_head"].t())
    return [torch.stack([r[j] for r in rows]) for j in range(c["steps"] + 1)]


def _evoformer_exact(c, seed):
    q, k, v, mask, pair, do = (t.to(F64) for t in _evoformer_inputs(c, seed))
    for t in (q, k, v, pair):
        t.requires_grad_()
    outs, D = [], c["dim"]
    for n in range(0, c["rows"], 32):
        a, b, d = (t[:, n:n + 32].transpose(2, 3) for t in (q, k, v))
        s = a @ b.transpose(-1, -2) * D**-0.5 + mask[:, n:n + 32] + pair
        o = (torch.softmax(s, -1) @ d).transpose(2, 3)
        o.backward(do[:, n:n + 32])
        outs.append(o.detach())
    return [torch.cat(outs, 1), q.grad, k.grad, v.grad, pair.grad]


def _sparse_exact(c, seed):
    q, k, v, do, mask = _sparse_inputs(c, seed)
    lay = _sparse_layout(c, seed).cuda()
    hidden = ~lay.repeat_interleave(c["block"], 0).repeat_interleave(c["block"], 1)
    out = [torch.empty(q.shape, dtype=F64, device="cuda") for _ in range(4)]
    for b in range(c["batch"]):
        for h in range(c["heads"]):
            one = [t[b, h].to(F64).requires_grad_() for t in (q, k, v)]
            s = one[0] @ one[1].t() * c["dim"]**-0.5
            if mask is not None:
                s = s + mask[b].to(F64)
            o = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ one[2]
            for t, g in zip(out, (o.detach(), *torch.autograd.grad(o, one, do[b, h].to(F64)))):
                t[b, h] = g
    return out


def exact(case, seed):
    return {"train": _train_exact, "serve": _serve_exact, "evoformer": _evoformer_exact, "sparse": _sparse_exact}[case["kind"]](case, seed)
