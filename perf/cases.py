"""What is measured: the framework's work through its public entry points, at sizes of its own models and tests.

Whole steps go through ``ModelRunner`` and its executor, as a server drives them (random weights of a seed, a page pool, block tables
in no order); the parts that only some designs have go through their layers and ``hip_ops``, as a model's glue calls them.

    decode    one step of running requests: every layer, the head, the greedy token of each row (graph replay)
    prefill   one batch of prompts: every layer, the head for the last tokens, the page pool filled
    delta     gated delta rule between its projections: prompts (convolution, recurrence, norm and gate) or a step
    scan      selective state space between its projections: prompts or a step
    latent    attention over cached latents: a step (with the value projection behind it) or prompts
    experts   a token's experts: stream started from the embedding, router, products, weighted sum into the stream
    sample    tokens drawn from logits, each row with parameters of its own
"""
from __future__ import annotations

import json
import math
import os
import random
import tempfile

import numpy as np
import torch

DEV = "cuda:0"
BLOCK = 64
BF16, F16, F32, F64 = torch.bfloat16, torch.float16, torch.float32, torch.float64
DTYPES = {"bf16": BF16, "f16": F16, "f32": F32}

_QWEN = dict(max_position_embeddings=32768, rms_norm_eps=1e-6, rope_theta=1000000.0, hidden_act="silu", torch_dtype="bfloat16")
MODELS = {
    "qwen3-0.6b": dict(_QWEN, model_type="qwen3", architectures=["Qwen3ForCausalLM"], hidden_size=1024, num_hidden_layers=28,
                       num_attention_heads=16, num_key_value_heads=8, head_dim=128, intermediate_size=3072, vocab_size=151936,
                       tie_word_embeddings=True, attention_bias=False),
    "qwen3-1.7b": dict(_QWEN, model_type="qwen3", architectures=["Qwen3ForCausalLM"], hidden_size=2048, num_hidden_layers=28,
                       num_attention_heads=16, num_key_value_heads=8, head_dim=128, intermediate_size=6144, vocab_size=151936,
                       tie_word_embeddings=True, attention_bias=False),
    "qwen2-7b": dict(_QWEN, model_type="qwen2", architectures=["Qwen2ForCausalLM"], hidden_size=3584, num_hidden_layers=28,
                     num_attention_heads=28, num_key_value_heads=4, intermediate_size=18944, vocab_size=152064,
                     tie_word_embeddings=False),
    "opt-125m": dict(model_type="opt", architectures=["OPTForCausalLM"], hidden_size=768, num_hidden_layers=12, num_attention_heads=12,
                     ffn_dim=3072, vocab_size=50272, max_position_embeddings=2048, word_embed_proj_dim=768, do_layer_norm_before=True,
                     activation_function="relu", enable_bias=True, layer_norm_elementwise_affine=True, tie_word_embeddings=True,
                     torch_dtype="float16", eos_token_id=2, bos_token_id=2, pad_token_id=1),
}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one user waiting for a chat answer: launches and dependent latencies
        dict(name="decode_one", kind="decode", model="qwen3-0.6b", rows=1, longest=777),
        # a server at its full batch (the headline workload), contexts around 1024
        dict(name="decode_full", kind="decode", model="qwen3-1.7b", rows=256, longest=1100),
        # a batch of unlike prompts at the largest dense layers; four layers stand for 28 that are the same
        dict(name="prefill_wide", kind="prefill", model="qwen2-7b", layers=4, dtype="bf16", prompts=12, longest=2731),
        # a small model in the precision that results are checked in
        dict(name="prefill_f32", kind="prefill", model="opt-125m", layers=12, dtype="f32", prompts=8, longest=1021),
        # recurrent layers of a mixed design: many prompts, one decay per head
        dict(name="delta_prompts", kind="delta", step=False, channel=False, heads=16, kv_heads=8, dim=128, rows=16, longest=1490, dtype="bf16"),
        # few long prompts, a decay per key channel
        dict(name="delta_long", kind="delta", step=False, channel=True, heads=8, kv_heads=8, dim=128, rows=3, longest=4011, dtype="bf16"),
        # a step of running requests: the states stream through
        dict(name="delta_step", kind="delta", step=True, channel=False, heads=16, kv_heads=8, dim=128, rows=48, longest=2000, dtype="bf16"),
        # state space layers of the other mixed design: few long prompts
        dict(name="scan_prompts", kind="scan", step=False, heads=64, groups=1, dim=64, state=128, rows=4, longest=3900, dtype="bf16"),
        # latent attention of running requests
        dict(name="latent_step", kind="latent", step=True, heads=16, kv_rank=512, rot=64, dim=128, window=2048, rows=64, longest=3000, dtype="bf16"),
        # experts: a batch of prompts
        dict(name="experts_prompts", kind="experts", width=2048, ff=768, experts=32, top=4, sigmoid=False, rows=9001, dtype="bf16"),
        # experts: a step of running requests
        dict(name="experts_step", kind="experts", width=2048, ff=768, experts=32, top=4, sigmoid=False, rows=24, dtype="bf16"),
        # tokens of a full batch, mixed parameters
        dict(name="sample_mixed", kind="sample", rows=256, vocab=151936, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["decode", "prefill", "delta", "delta", "scan", "latent", "experts", "experts", "sample"])
    half = rng.choice(["bf16", "bf16", "bf16", "f16"])
    if kind == "decode":
        return dict(kind=kind, model=rng.choice(["qwen3-0.6b", "qwen3-1.7b"]), rows=_log(rng, 1, 200), longest=_log(rng, 64, 1024))
    if kind == "prefill":
        if rng.random() < 0.5:
            return dict(kind=kind, model="opt-125m", layers=12, dtype=rng.choice(["f32", "bf16", "f16"]), prompts=_log(rng, 1, 8),
                        longest=_log(rng, 16, 1000))
        return dict(kind=kind, model=rng.choice(["qwen3-0.6b", "qwen3-1.7b", "qwen2-7b"]), layers=4, dtype=half, prompts=_log(rng, 1, 12),
                    longest=_log(rng, 32, 2700))
    if kind == "delta":
        step, channel = rng.random() < 0.4, rng.random() < 0.5
        heads = rng.choice([8, 16]) if not channel else rng.choice([4, 8])
        return dict(kind=kind, step=step, channel=channel, heads=heads, kv_heads=heads // 2 if not channel else heads,
                    dim=rng.choice([64, 128, 128]), rows=_log(rng, 1, 128) if step else _log(rng, 1, 16),
                    longest=_log(rng, 64, 1490 if not channel else 750), dtype=half if step else "bf16")
    if kind == "scan":
        step = rng.random() < 0.3
        return dict(kind=kind, step=step, heads=rng.choice([32, 64]), groups=rng.choice([1, 2]), dim=64, state=rng.choice([64, 128]),
                    rows=_log(rng, 1, 128) if step else _log(rng, 1, 8), longest=_log(rng, 64, 1900), dtype=half)
    if kind == "latent":
        step = rng.random() < 0.6
        return dict(kind=kind, step=step, heads=16, kv_rank=512, rot=64, dim=128, window=rng.choice([0, 2048]),
                    rows=_log(rng, 1, 64) if step else _log(rng, 1, 8), longest=_log(rng, 64, 3000 if step else 1900), dtype=half)
    if kind == "experts":
        width, ff = rng.choice([(1024, 384), (2048, 768)])
        return dict(kind=kind, width=width, ff=ff, experts=32, top=rng.choice([4, 8]), sigmoid=rng.random() < 0.4, rows=_log(rng, 1, 4500),
                    dtype=half)
    return dict(kind=kind, rows=_log(rng, 1, 256), vocab=rng.choice([50272, 151936]), dtype=half)


def _lengths(case):
    """Lengths of a case's sequences, from a half of the longest on, the longest among them."""
    n = case.get("rows") or case.get("prompts")
    rng = random.Random(7919 * n + case["longest"])
    out = [rng.randint(-(-case["longest"] // 2), case["longest"]) for _ in range(n)]
    out[rng.randrange(n)] = case["longest"]
    return out


def _mean_lengths(case):
    n = case.get("rows") or case.get("prompts")
    return n, (n - 1) * 0.75 * case["longest"] + case["longest"]


def _generator(seed, part=0):
    return torch.Generator(device=DEV).manual_seed(seed * 1000003 + part)


def _normal(gen, *shape, dtype=F32, std=1.0):
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=gen)


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _cu(lengths):
    return _i32([0, *np.cumsum(lengths).tolist()])


def _tables(lengths, seed):
    """A pool's pages dealt to the sequences in no order."""
    pages = [-(-n // BLOCK) for n in lengths]
    order = list(range(sum(pages)))
    random.Random(seed + 1).shuffle(order)
    out = []
    for n in pages:
        out.append(order[:n])
        del order[:n]
    return out


def _padded(tables):
    width = max(map(len, tables))
    return _i32([t + [-1] * (width - len(t)) for t in tables])


# ---------------------------------------------------------------- whole steps
def _tokens(case, lengths, seed):
    rng = np.random.default_rng(seed + 2)
    vocab = MODELS[case["model"]]["vocab_size"]
    return [rng.integers(3, vocab, n).tolist() for n in lengths]


def _prepare_model(case, seed):
    from minivllm_amd import Config
    from minivllm_amd.engine.model_runner import ModelRunner
    from minivllm_amd.engine.sequence import Sequence
    from minivllm_amd.sampling_params import SamplingParams

    decode = case["kind"] == "decode"
    lengths = _lengths(case)
    tables = _tables(lengths, seed)
    config = dict(MODELS[case["model"]])
    if not decode:
        config["num_hidden_layers"] = case["layers"]
    longest = -(-case["longest"] // BLOCK) * BLOCK
    with tempfile.TemporaryDirectory() as folder:
        with open(os.path.join(folder, "config.json"), "w") as f:
            json.dump(config, f)
        cfg = Config(folder, dtype={"bf16": "bfloat16", "f16": "float16", "f32": "float32"}[case.get("dtype", "bf16")],
                     kvcache_block_size=BLOCK, max_num_seqs=len(lengths), max_model_len=longest,
                     max_num_batched_tokens=max(longest, longest if decode else sum(lengths)), num_kvcache_blocks=sum(map(len, tables)),
                     enforce_eager=not decode, load_format="dummy", seed=seed)
        runner = ModelRunner(cfg, 0)
    executor = runner.inference_executor
    if decode:      # what earlier steps left in the pool
        executor.kv_cache.normal_(0.0, 1.0, generator=_generator(seed))
    else:
        executor.kv_cache.zero_()
    sequences = []
    for ids, pages in zip(_tokens(case, lengths, seed), tables):
        s = Sequence(ids, SamplingParams(temperature=0.0, max_tokens=64, ignore_eos=True), block_size=BLOCK)
        s.block_table = pages
        sequences.append(s)
    return dict(case=case, runner=runner, executor=executor, sequences=sequences)


def _run_model(state):
    prefill = state["case"]["kind"] == "prefill"
    logits, tokens = state["executor"].execute_batch(state["sequences"], prefill)
    out = {"logits": logits, "tokens": np.asarray(tokens)}
    if prefill:
        out["cache"] = state["executor"].kv_cache
    return out


def _weights(case, seed):
    """The model's random weights, in the order in which they are drawn (normal, 0.02; norms 1, biases 0)."""
    c, dtype = MODELS[case["model"]], DTYPES[case.get("dtype", "bf16")]
    gen, h = torch.Generator(device=DEV).manual_seed(seed), c["hidden_size"]
    def mat(*shape):
        return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, 0.02, generator=gen)

    opt = c["model_type"] == "opt"
    yield mat(c["vocab_size"], h)
    if opt:
        yield mat(c["max_position_embeddings"] + 2, h)
    for _ in range(case.get("layers", c["num_hidden_layers"])):
        if opt:
            yield mat(3 * h, h), mat(h, h), mat(c["ffn_dim"], h), mat(h, c["ffn_dim"])
        else:
            d = c.get("head_dim") or h // c["num_attention_heads"]
            heads, kv, ff = c["num_attention_heads"], c["num_key_value_heads"], c["intermediate_size"]
            yield mat((heads + 2 * kv) * d, h), mat(h, heads * d), mat(2 * ff, h), mat(h, ff)
    if not c["tie_word_embeddings"]:
        yield mat(c["vocab_size"], h)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _exact_model(case, seed):
    """The model in 64 bits.  (Angles' cosines and sines are rounded to the model's dtype: a convention of these models.)"""
    c, dtype, decode = MODELS[case["model"]], DTYPES[case.get("dtype", "bf16")], case["kind"] == "decode"
    opt, h, heads = c["model_type"] == "opt", c["hidden_size"], c["num_attention_heads"]
    kv = c.get("num_key_value_heads", heads)
    d = c.get("head_dim") or h // heads
    lengths = _lengths(case)
    tables, tokens = _tables(lengths, seed), _tokens(case, lengths, seed)
    layers, pages = case.get("layers", c["num_hidden_layers"]), sum(map(len, tables))
    weights = _weights(case, seed)
    table = next(weights)
    where = [torch.arange(n, device=DEV) for n in lengths]
    slots = [torch.tensor(t, device=DEV)[w // BLOCK] * BLOCK + w % BLOCK for t, w in zip(tables, where)]
    if decode:
        cache = torch.empty((2, layers, pages * BLOCK, kv, d), dtype=dtype, device=DEV).normal_(0.0, 1.0, generator=_generator(seed))
        ids, pos = torch.tensor([t[-1] for t in tokens], device=DEV), torch.tensor([n - 1 for n in lengths], device=DEV)
        cut = list(range(len(lengths) + 1))
    else:
        cache = torch.zeros((2, layers, pages * BLOCK, kv, d), dtype=F64, device=DEV)
        ids, pos = torch.tensor(sum(tokens, []), device=DEV), torch.cat(where)
        cut = [0, *np.cumsum(lengths).tolist()]
    x = table[ids].double()
    if opt:
        x = x + next(weights)[pos + 2].double()
    else:
        freq = 1.0 / c["rope_theta"] ** (torch.arange(0, d, 2, dtype=F64, device=DEV) / d)
        angle = pos.double()[:, None] * freq
        cos, sin = (f(angle).to(dtype).double()[:, None] for f in (torch.cos, torch.sin))
    for layer in range(layers):
        wqkv, wo, w1, w2 = (w.double() for w in next(weights))
        u = torch.nn.functional.layer_norm(x, (h,)) if opt else _rms(x, 1e-6)
        q, k, v = (u @ wqkv.T).split([heads * d, kv * d, kv * d], 1)
        q, k, v = q.unflatten(1, (heads, d)), k.unflatten(1, (kv, d)), v.unflatten(1, (kv, d))
        if c["model_type"] == "qwen3":
            q, k = _rms(q, 1e-6), _rms(k, 1e-6)
        if not opt:
            q, k = (torch.cat([a * cos - b * sin, b * cos + a * sin], -1) for a, b in (t.chunk(2, -1) for t in (q, k)))
        out = torch.empty_like(q)
        for i, n in enumerate(lengths):
            lo, hi = cut[i], cut[i + 1]
            if decode:
                ks, vs = (torch.cat([cache[j, layer, slots[i][:-1]].double(), t[lo:hi]]) for j, t in ((0, k), (1, v)))
            else:
                ks, vs = k[lo:hi], v[lo:hi]
                cache[0, layer, slots[i]], cache[1, layer, slots[i]] = ks, vs
            qs = q[lo:hi].unflatten(1, (kv, heads // kv)).permute(1, 2, 0, 3).flatten(1, 2)     # [kv, heads / kv * rows, d]
            score = torch.bmm(qs, ks.permute(1, 2, 0).contiguous()) * d ** -0.5
            if not decode:
                late = torch.arange(n, device=DEV)[None, :] > torch.arange(n, device=DEV)[:, None]
                score.unflatten(1, (heads // kv, n)).masked_fill_(late, -math.inf)
            o = torch.bmm(score.softmax(-1), vs.transpose(0, 1).contiguous())
            out[lo:hi] = o.unflatten(1, (heads // kv, hi - lo)).permute(2, 0, 1, 3).flatten(1, 2)
            del score, o
        x = x + out.flatten(1) @ wo.T
        u = torch.nn.functional.layer_norm(x, (h,)) if opt else _rms(x, 1e-6)
        u = u @ w1.T
        x = x + (torch.relu(u) if opt else torch.nn.functional.silu(u[:, :u.shape[1] // 2]) * u[:, u.shape[1] // 2:]) @ w2.T
    x = torch.nn.functional.layer_norm(x, (h,)) if opt else _rms(x, 1e-6)
    if not decode:
        x = x[torch.tensor(cut[1:], device=DEV) - 1]
    head = table if c["tie_word_embeddings"] else next(weights)
    logits = x @ head.double().T
    out = {"logits": logits, "tokens": None}
    if not decode:
        out["cache"] = cache.view(2, layers, pages, BLOCK, kv, d)
    return out


def _work_model(case):
    c, size = MODELS[case["model"]], DTYPES[case.get("dtype", "bf16")].itemsize
    h, heads, opt = c["hidden_size"], c["num_attention_heads"], c["model_type"] == "opt"
    kv = c.get("num_key_value_heads", heads)
    d = c.get("head_dim") or h // heads
    layers = case.get("layers", c["num_hidden_layers"])
    layer = (heads + 2 * kv) * d * h + heads * d * h + (2 * h * c["ffn_dim"] if opt else 3 * h * c["intermediate_size"])
    n, total = _mean_lengths(case)
    head = c["vocab_size"] * h
    if case["kind"] == "decode":
        return {"bytes": size * (layers * (layer + 2 * kv * d * total) + head + n * c["vocab_size"]),
                "flops": 2.0 * n * (layers * layer + head) + layers * 4.0 * heads * d * total}
    pairs = total * (total / n) / 2 * 1.03
    return {"bytes": size * (layers * (layer + 2 * kv * d * total) + head + total * h + n * c["vocab_size"]),
            "flops": 2.0 * (total * layers * layer + n * head) + layers * 4.0 * heads * d * pairs}


# ---------------------------------------------------------------- recurrences
TAPS = 4


def _context(case, lengths):
    from minivllm_amd.utils.context import set_context

    slots = _i32(list(range(len(lengths)))[::-1])
    if case["step"]:
        lens = _i32(lengths)
        return lambda: set_context(False, context_lens=lens, state_slots=slots)
    cu = _cu(lengths)
    return lambda: set_context(True, max(lengths), max(lengths), cu, cu, state_slots=slots)


def _conv_rows(case, lengths, x, w, b, kept, slots):
    """silu of the causal convolution in 64 bits, and what is kept of the inputs; kept [2, slots, taps - 1, channels]."""
    x, w, kept, out = x.double(), w.double(), kept.clone().double(), torch.empty(x.shape, dtype=F64, device=DEV)
    at = 0
    for i, n in enumerate(lengths):
        m = 1 if case["step"] else n
        before = kept[(n - 1) & 1, slots[i]] if case["step"] else torch.zeros_like(kept[0, 0])
        rows = torch.cat([before, x[at:at + m]])
        out[at:at + m] = sum(rows[j:j + m] * w[j] for j in range(TAPS))
        kept[n & 1, slots[i]] = rows[m:]
        at += m
    return torch.nn.functional.silu(out if b is None else out + b.double()), kept


def _by_sequence(rows, lengths):
    """[T, ...] -> [sequences, longest, ...], zeros behind the ends."""
    out = torch.zeros((len(lengths), max(lengths)) + rows.shape[1:], dtype=rows.dtype, device=DEV)
    at = 0
    for i, n in enumerate(lengths):
        out[i, :n] = rows[at:at + n]
        at += n
    return out


def _speeds(gen, n, dtype):
    """Raw biases of step sizes between 0.001 and 0.1, log-uniform."""
    dt = torch.exp(torch.rand(n, generator=gen, device=DEV, dtype=F32) * math.log(100.0) + math.log(0.001))
    return (dt + torch.log(-torch.expm1(-dt))).to(dtype)


def _rates(gen, n, dtype):
    return torch.log(1 + 15 * torch.rand(n, generator=gen, device=DEV, dtype=F32)).to(dtype)


def _delta_inputs(case, seed):
    gen, dtype = _generator(seed), DTYPES[case["dtype"]]
    heads, kv, d = case["heads"], case["kv_heads"], case["dim"]
    lengths = _lengths(case)
    t = len(lengths) if case["step"] else sum(lengths)
    channels = (heads + 2 * kv) * d
    w = dict(conv=_normal(gen, TAPS, channels, dtype=dtype, std=0.5), A_log=_rates(gen, heads, dtype),
             dt_bias=_speeds(gen, heads * (d if case["channel"] else 1), dtype), norm=(1 + _normal(gen, d, std=0.1)).to(dtype))
    x, beta = _normal(gen, t, channels, dtype=dtype), _normal(gen, t, heads, dtype=dtype)
    if case["channel"]:     # both through projections of a low rank
        a, gate = _normal(gen, t, 128, dtype=dtype), _normal(gen, t, 128, dtype=dtype)
        w["a2"], w["g2"] = (_normal(gen, heads * d, 128, dtype=dtype, std=128 ** -0.5) for _ in range(2))
    else:
        a, gate = _normal(gen, t, heads, dtype=dtype), _normal(gen, t, heads * d, dtype=dtype)
    slots = len(lengths)
    state, kept = torch.zeros((2, slots, heads, d, d), device=DEV), torch.zeros((2, slots, TAPS - 1, channels), dtype=dtype, device=DEV)
    if case["step"]:
        state.copy_(_normal(gen, slots, heads, d, d, std=0.1)[None])
        kept.copy_(_normal(gen, slots, TAPS - 1, channels, dtype=dtype)[None])
    return lengths, w, x, beta, a, gate, state, kept


def _prepare_delta(case, seed):
    from minivllm_amd.layers import GatedDeltaRule

    lengths, w, x, beta, a, gate, state, kept = _delta_inputs(case, seed)
    dtype, heads, d = x.dtype, case["heads"], case["dim"]
    before = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
        with torch.device(DEV):
            rule = GatedDeltaRule(heads, case["kv_heads"], d, d, TAPS, 1e-6, "sigmoid" if case["channel"] else "silu",
                                  (128, 128) if case["channel"] else None)
    finally:
        torch.set_default_dtype(before)
    rule.requires_grad_(False)
    for name in ("conv", "A_log", "dt_bias", "norm"):
        getattr(rule, name).copy_(w[name])
    if case["channel"]:
        for name in ("a2", "g2"):
            rule.lift.weight_loader(rule.lift.weight, w[name], name)
        rule.lift.pack_for_decode()
    rule.state, rule.conv_state = state, kept
    z = torch.zeros((x.shape[0], rule.columns), dtype=dtype, device=DEV)      # the projection's rows
    for name, rows in (("v", x), ("b", beta), *((("a1", a), ("g1", gate)) if case["channel"] else (("a", a), ("g", gate)))):
        z[:, rule.at[name]:rule.at[name] + rows.shape[1]] = rows
    return dict(case=case, rule=rule, z=z, context=_context(case, lengths))


def _run_delta(state):
    rule, z = state["rule"], state["z"]
    state["context"]()
    out = torch.empty((z.shape[0], rule.shape.heads * rule.shape.p), dtype=z.dtype, device=z.device)
    with torch.inference_mode():
        rule(z, out)
    return {"out": out, "state": rule.state, "kept": rule.conv_state}


def _exact_delta(case, seed):
    lengths, w, x, beta, a, gate, state, kept = _delta_inputs(case, seed)
    heads, kv, d, step = case["heads"], case["kv_heads"], case["dim"], case["step"]
    slots = list(range(len(lengths)))[::-1]
    rows, kept = _conv_rows(case, lengths, x, w["conv"], None, kept, slots)
    v, k, q = rows.split([heads * d, kv * d, kv * d], 1)
    v, k, q = v.unflatten(1, (heads, d)), k.unflatten(1, (kv, d)), q.unflatten(1, (kv, d))
    k, q = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (k, q))
    k, q = (t.repeat_interleave(heads // kv, 1) for t in (k, q * d ** -0.5))
    a, gate = a.double(), gate.double()
    if case["channel"]:
        a, gate = a @ w["a2"].double().T, gate @ w["g2"].double().T
    a = (a + w["dt_bias"].double()).unflatten(1, (heads, -1))                 # [T, heads, d or 1]
    decay = torch.exp(-torch.exp(w["A_log"].double())[:, None] * torch.nn.functional.softplus(a, threshold=60.0))
    beta = torch.sigmoid(beta.double())[..., None]
    many = [1] * len(lengths) if step else lengths
    v, k, q, decay, beta = (_by_sequence(t, many) for t in (v, k, q, decay, beta))
    state = state.double()
    s = torch.stack([state[(n - 1) & 1, slots[i]] if step else torch.zeros_like(state[0, 0]) for i, n in enumerate(lengths)])
    o = torch.zeros((len(lengths), max(many), heads, d), dtype=F64, device=DEV)
    ends = torch.tensor(many, device=DEV)
    for t in range(max(many)):
        live = (ends > t)[:, None, None, None]
        new = s * decay[:, t, :, :, None]
        u = beta[:, t] * (v[:, t] - (k[:, t, :, None] @ new)[:, :, 0])
        new = new + k[:, t, :, :, None] * u[:, :, None]
        o[:, t] = (q[:, t, :, None] @ new)[:, :, 0]
        s = torch.where(live, new, s)
    for i, n in enumerate(lengths):
        state[n & 1, slots[i]] = s[i]
    o = torch.cat([o[i, :n] for i, n in enumerate(many)])
    gate = gate.unflatten(1, (heads, d))
    o = _rms(o, 1e-6) * w["norm"].double() * (torch.sigmoid(gate) if case["channel"] else torch.nn.functional.silu(gate))
    return {"out": o.flatten(1), "state": state, "kept": kept}


def _work_delta(case):
    n, total = _mean_lengths(case)
    t = n if case["step"] else total
    heads, kv, d, size = case["heads"], case["kv_heads"], case["dim"], DTYPES[case["dtype"]].itemsize
    row = (2 * heads + 2 * kv) * d + heads + (256 if case["channel"] else heads * (d + 1))
    states = n * heads * d * d * 4.0 * (2 if case["step"] else 1)
    # (token by token: decay, k S, k u, q S)
    return {"bytes": t * row * size + states, "flops": t * heads * d * d * 7.0}


def _scan_inputs(case, seed):
    gen, dtype = _generator(seed), DTYPES[case["dtype"]]
    heads, groups, d, n = case["heads"], case["groups"], case["dim"], case["state"]
    lengths = _lengths(case)
    t = len(lengths) if case["step"] else sum(lengths)
    channels = heads * d + 2 * groups * n
    w = dict(conv=_normal(gen, TAPS, channels, dtype=dtype, std=0.5), conv_b=_normal(gen, channels, dtype=dtype, std=0.1),
             a_log=_rates(gen, heads, dtype), dt_bias=_speeds(gen, heads, dtype), d=_normal(gen, heads, dtype=dtype),
             norm=(1 + _normal(gen, heads * d, std=0.1)).to(dtype))
    z = _normal(gen, t, heads * d + channels + heads, dtype=dtype)       # the projection's rows: gate | x | b | c | step sizes
    slots = len(lengths)
    state, kept = torch.zeros((2, slots, heads, n, d), device=DEV), torch.zeros((2, slots, TAPS - 1, channels), dtype=dtype, device=DEV)
    if case["step"]:
        state.copy_(_normal(gen, slots, heads, n, d, std=0.1)[None])
        kept.copy_(_normal(gen, slots, TAPS - 1, channels, dtype=dtype)[None])
    return lengths, w, z, state, kept


def _prepare_scan(case, seed):
    lengths, w, z, state, kept = _scan_inputs(case, seed)
    heads, groups, d, n = case["heads"], case["groups"], case["dim"], case["state"]
    return dict(case=case, w=w, z=z, ssm=state, kept=kept, shape=(heads, groups, d, n, heads * d, heads * d + groups * n),
                slots=_i32(list(range(len(lengths)))[::-1]), lens=_i32(lengths), cu=_cu(lengths), longest=max(lengths))


def _run_scan(s):
    from minivllm_amd import hip_ops as H

    w, z, shape, case = s["w"], s["z"], s["shape"], s["case"]
    heads, groups, p = shape[:3]
    wide, channels = heads * p, w["conv"].shape[1]
    x, dt = z[:, wide:wide + channels], z[:, wide + channels:]
    if case["step"]:
        y = H.ssm_step(x, dt, w["conv"], w["conv_b"], w["dt_bias"], w["a_log"], w["d"], shape, s["kept"], s["ssm"], s["slots"], s["lens"])
    else:
        xc = H.causal_conv(x, w["conv"], w["conv_b"], shape, s["kept"], s["slots"], s["cu"], s["cu"], s["longest"])
        y = H.ssm_prefill(xc, dt, w["dt_bias"], w["a_log"], w["d"], shape, s["ssm"], s["slots"], s["cu"], s["cu"], s["longest"])
    out = H.gated_group_norm(y, z[:, :wide], w["norm"], heads, p, p, groups, 1e-6)
    return {"out": out, "state": s["ssm"], "kept": s["kept"]}


def _exact_scan(case, seed):
    lengths, w, z, state, kept = _scan_inputs(case, seed)
    heads, groups, d, n, step = case["heads"], case["groups"], case["dim"], case["state"], case["step"]
    slots, wide = list(range(len(lengths)))[::-1], heads * d
    rows, kept = _conv_rows(case, lengths, z[:, wide:-heads], w["conv"], w["conv_b"], kept, slots)
    x, b, c = rows.split([wide, groups * n, groups * n], 1)
    x, b, c = x.unflatten(1, (heads, d)), *(t.unflatten(1, (groups, n)).repeat_interleave(heads // groups, 1) for t in (b, c))
    dt = torch.nn.functional.softplus(z[:, -heads:].double() + w["dt_bias"].double(), threshold=60.0)
    decay = torch.exp(-torch.exp(w["a_log"].double()) * dt)
    many = [1] * len(lengths) if step else lengths
    xs, b, c, dt, decay = (_by_sequence(t, many) for t in (x, b, c, dt, decay))
    state = state.double()
    s = torch.stack([state[(m - 1) & 1, slots[i]] if step else torch.zeros_like(state[0, 0]) for i, m in enumerate(lengths)])
    y = torch.zeros((len(lengths), max(many), heads, d), dtype=F64, device=DEV)
    ends = torch.tensor(many, device=DEV)
    for t in range(max(many)):
        new = s * decay[:, t, :, None, None] + (b[:, t] * dt[:, t, :, None])[..., None] * xs[:, t, :, None]
        y[:, t] = (c[:, t, :, None] @ new)[:, :, 0]
        s = torch.where((ends > t)[:, None, None, None], new, s)
    for i, m in enumerate(lengths):
        state[m & 1, slots[i]] = s[i]
    y = torch.cat([y[i, :m] for i, m in enumerate(many)]) + w["d"].double()[:, None] * x
    y = y.flatten(1) * torch.nn.functional.silu(z[:, :wide].double())
    y = _rms(y.unflatten(1, (groups, -1)), 1e-6).flatten(1) * w["norm"].double()
    return {"out": y, "state": state, "kept": kept}


def _work_scan(case):
    n, total = _mean_lengths(case)
    t, size = n if case["step"] else total, DTYPES[case["dtype"]].itemsize
    wide, cells = case["heads"] * case["dim"], case["heads"] * case["dim"] * case["state"]
    return {"bytes": t * size * (3 * wide + 2 * case["groups"] * case["state"] + case["heads"]) + n * cells * 4.0 * (2 if case["step"] else 1),
            "flops": t * cells * 5.0}


# ---------------------------------------------------------------- latent attention
def _latent_inputs(case, seed):
    gen, dtype = _generator(seed), DTYPES[case["dtype"]]
    heads, kv, rot, d = case["heads"], case["kv_rank"], case["rot"], case["dim"]
    lengths = _lengths(case)
    if case["step"]:
        tables = _tables(lengths, seed)
        plane = _normal(gen, sum(map(len, tables)), BLOCK, kv + rot, dtype=dtype)
        q = _normal(gen, len(lengths), heads, kv + rot, dtype=dtype, std=0.6)
        return lengths, tables, plane, q, _normal(gen, heads, d, kv, dtype=dtype, std=kv ** -0.5)
    t = sum(lengths)
    q, kvx = _normal(gen, t, heads, d + rot, dtype=dtype), _normal(gen, t, 2 * heads * d, dtype=dtype)
    rows = _normal(gen, t, rot, dtype=dtype)
    return lengths, q, kvx, rows


def _angles(case, positions):
    freq = 1e4 ** (-2.0 * torch.arange(case["rot"] // 2, dtype=F64, device=DEV) / case["rot"])
    angle = positions.double()[:, None] * freq
    return angle.cos(), angle.sin()


def _prepare_latent(case, seed):
    lengths, *rest = _latent_inputs(case, seed)
    if case["step"]:
        tables, plane, q, w = rest
        return dict(case=case, tables=_padded(tables), plane=plane, q=q, w=w, lens=_i32(lengths))
    q, kvx, rows = rest
    cos, sin = (t.float() for t in _angles(case, torch.arange(case["longest"], device=DEV)))
    return dict(case=case, q=q, kvx=kvx, rows=rows, cu=_cu(lengths), longest=max(lengths), cos=cos, sin=sin,
                positions=torch.cat([torch.arange(n, device=DEV) for n in lengths]))


def _run_latent(s):
    from minivllm_amd import hip_ops as H

    case = s["case"]
    heads, d = case["heads"], case["dim"]
    scale = (d + case["rot"]) ** -0.5
    if case["step"]:
        lat = H.latent_decode(s["q"], s["plane"], s["tables"], s["lens"], case["kv_rank"], scale, case["window"])
        out = torch.empty((lat.shape[0], heads, d), dtype=lat.dtype, device=lat.device)
        H.head_linear(lat, s["w"], out)
        return out
    k, v = (s["kvx"][:, i * heads * d:(i + 1) * heads * d].unflatten(1, (heads, d)) for i in range(2))
    return H.latent_prefill(s["q"], k, v, s["rows"], s["cu"], s["cu"], s["longest"], s["longest"], s["positions"], s["cos"], s["sin"],
                            case["rot"], scale, case["window"])


def _exact_latent(case, seed):
    lengths, *rest = _latent_inputs(case, seed)
    heads, kv, d, window = case["heads"], case["kv_rank"], case["dim"], case["window"] or 1 << 30
    scale, out, at = (d + case["rot"]) ** -0.5, [], 0
    if case["step"]:
        tables, plane, q, w = rest
        for i, n in enumerate(lengths):
            rows = plane[torch.tensor(tables[i], device=DEV)].flatten(0, 1)[max(0, n - window):n].double()
            p = (q[i].double() @ rows.T * scale).softmax(-1)
            out.append(torch.bmm(w.double(), (p @ rows[:, :kv])[:, :, None])[:, :, 0])
        return torch.stack(out)
    q, kvx, rows = rest
    for n in lengths:
        pos = torch.arange(n, device=DEV)
        cos, sin = (t[:, None] for t in _angles(case, pos))
        qs, r = q[at:at + n].double(), rows[at:at + n].double()
        a, b = qs[..., d::2], qs[..., d + 1::2]
        rotated = torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)
        k, v = kvx[at:at + n].double().unflatten(1, (2, heads, d)).unbind(1)
        score = torch.bmm(qs[..., :d].transpose(0, 1).contiguous(), k.permute(1, 2, 0).contiguous()) + rotated.transpose(0, 1) @ r.T
        ahead = pos[:, None] - pos[None, :]
        p = (score * scale).masked_fill((ahead < 0) | (ahead >= window), -math.inf).softmax(-1)
        out.append(torch.bmm(p, v.transpose(0, 1).contiguous()).transpose(0, 1))
        at += n
    return torch.cat(out)


def _work_latent(case):
    n, total = _mean_lengths(case)
    heads, kv, rot, d, size = case["heads"], case["kv_rank"], case["rot"], case["dim"], DTYPES[case["dtype"]].itemsize
    window = case["window"] or 1 << 30
    if case["step"]:
        keys = n * min(window, total / n)
        return {"bytes": size * (keys * (kv + rot) + n * heads * (kv + rot + d) + heads * d * kv),
                "flops": 2.0 * heads * keys * (2 * kv + rot) + 2.0 * n * heads * d * kv}
    long = total / n
    pairs = total * (min(long, window) - min(long, window) ** 2 / (2 * long)) * 1.03
    return {"bytes": size * total * (heads * (4 * d + rot) + rot), "flops": 2.0 * heads * pairs * (2 * d + rot)}


# ---------------------------------------------------------------- experts
VOCAB = 32000


def _expert_inputs(case, seed):
    gen, dtype = _generator(seed), DTYPES[case["dtype"]]
    width, ff, experts = case["width"], case["ff"], case["experts"]
    extra = 0 if case["sigmoid"] else 2       # (the softmax router has two experts that hand the token through)
    w = dict(embed=_normal(gen, VOCAB, width, dtype=dtype), router=_normal(gen, experts + extra, width, dtype=dtype, std=width ** -0.5),
             correction=_normal(gen, experts + extra, dtype=dtype, std=0.01),
             gate_up=_normal(gen, experts, 2, ff, width, dtype=dtype, std=width ** -0.5),
             down=_normal(gen, experts, width, ff, dtype=dtype, std=ff ** -0.5))
    ids = torch.randint(0, VOCAB, (case["rows"],), generator=gen, device=DEV)
    return extra, w, ids


def _prepare_experts(case, seed):
    from minivllm_amd.layers import ExpertMLP

    extra, w, ids = _expert_inputs(case, seed)
    before = torch.get_default_dtype()
    torch.set_default_dtype(w["embed"].dtype)
    try:
        with torch.device(DEV):
            mlp = ExpertMLP(case["width"], case["experts"], extra, case["top"], 1 if case["sigmoid"] else 2, 1, 2.5, case["ff"],
                            sigmoid=case["sigmoid"], raw_weights=case["sigmoid"])
    finally:
        torch.set_default_dtype(before)
    mlp.requires_grad_(False)
    for name in ("router", "correction", "gate_up", "down"):
        getattr(mlp, name).copy_(w[name])
    mlp.finish_weights()
    return dict(mlp=mlp, embed=w["embed"], ids=ids)


def _run_experts(s):
    from minivllm_amd import hip_ops as H

    ids, embed = s["ids"], s["embed"]
    with torch.inference_mode():
        x = torch.empty((ids.shape[0], embed.shape[1]), dtype=F32, device=ids.device)
        h = H.residual_update(x, embed=embed, ids=ids, start=True)
        y, chosen = s["mlp"](h)
        h = H.residual_update(x, y=y, dtype=embed.dtype, experts=chosen)
    return {"stream": x, "next": h}


def _exact_experts(case, seed):
    extra, w, ids = _expert_inputs(case, seed)
    h, top, experts = w["embed"][ids].double(), case["top"], case["experts"]
    logits = h @ w["router"].double().T
    score = torch.sigmoid(logits) if case["sigmoid"] else logits.softmax(-1)
    choice = score + w["correction"].double()
    if not case["sigmoid"]:       # the better of two groups
        groups = choice.unflatten(1, (2, -1))
        worse = groups.amax(-1, keepdim=True) < choice.amax(-1)[:, None, None]
        choice = groups.masked_fill(worse, -math.inf).flatten(1)
    ids = choice.topk(top, -1).indices
    weight = score.gather(1, ids)
    weight = (weight if case["sigmoid"] else weight / (weight.sum(-1, keepdim=True) + 1e-20)) * 2.5
    x = h.clone()
    for e in range(experts + extra):
        rows, at = (ids == e).nonzero(as_tuple=True)
        y = h[rows]
        if e < experts:
            gate, up = (y @ w["gate_up"][e, i].double().T for i in range(2))
            y = (torch.nn.functional.silu(gate) * up) @ w["down"][e].double().T
        x.index_add_(0, rows, y * weight[rows, at][:, None])
    return {"stream": x, "next": x}


def _work_experts(case):
    t, width, ff, size = case["rows"], case["width"], case["ff"], DTYPES[case["dtype"]].itemsize
    used = case["experts"] * (1 - (1 - case["top"] / case["experts"]) ** t)
    return {"bytes": size * (used * 3 * width * ff + t * 2 * width + 34 * width) + 4 * t * width,
            "flops": 2.0 * t * (case["top"] * 3 * width * ff + 34 * width)}


# ---------------------------------------------------------------- sampling
def _prepare_sample(case, seed):
    gen, rng = _generator(seed), random.Random(seed)
    logits = _normal(gen, case["rows"], case["vocab"], dtype=DTYPES[case["dtype"]], std=2.5)
    rows = []
    for _ in range(case["rows"]):      # greedy, the default, the examples' preset, a nucleus, a floor
        rows.append(rng.choice([(0.0, -1, 1.0, 0.0), (1.0, -1, 1.0, 0.0), (0.6, 40, 0.95, 0.0), (0.8, -1, 0.9, 0.0), (0.7, -1, 1.0, 0.05)]))
    t, k, p, m = zip(*rows)
    return dict(logits=logits, seed=seed, temperatures=torch.tensor(t, device=DEV), top_ks=torch.tensor(k, device=DEV),
                top_ps=torch.tensor(p, device=DEV), min_ps=torch.tensor(m, device=DEV))


def _run_sample(s):
    from minivllm_amd import hip_ops as H

    return H.sample(s["logits"], s["temperatures"], s["top_ks"], s["top_ps"], s["min_ps"], seed=s["seed"], offset=1)


def _work_sample(case):
    n = case["rows"] * case["vocab"]
    return {"bytes": n * DTYPES[case["dtype"]].itemsize, "flops": 2.0 * n}


# ---------------------------------------------------------------- by kind
_KINDS = {
    "decode": (_prepare_model, _run_model, _exact_model, _work_model),
    "prefill": (_prepare_model, _run_model, _exact_model, _work_model),
    "delta": (_prepare_delta, _run_delta, _exact_delta, _work_delta),
    "scan": (_prepare_scan, _run_scan, _exact_scan, _work_scan),
    "latent": (_prepare_latent, _run_latent, _exact_latent, _work_latent),
    "experts": (_prepare_experts, _run_experts, _exact_experts, _work_experts),
    "sample": (_prepare_sample, _run_sample, None, _work_sample),
}


def prepare(case, seed):
    state = _KINDS[case["kind"]][0](case, seed)
    return dict(state, kind=case["kind"])


def run(state):
    return _KINDS[state["kind"]][1](state)


def work(case):
    return _KINDS[case["kind"]][3](case)


def exact(case, seed):
    fn = _KINDS[case["kind"]][2]
    return None if fn is None else fn(case, seed)


def tolerance(case):
    """About four times what a path was seen to be off its 64-bit value (in brackets)."""
    kind, f32, f16 = case["kind"], case.get("dtype") == "f32", case.get("dtype") == "f16"
    if kind == "decode":        # 28 layers of 16-bit rounding (4e-2), the largest of as many logits as there are words (0.24)
        return {"rel": 0.16, "max": 0.9, "differ": 0.25}
    if kind == "prefill":       # four or twelve layers (bf16 2e-2, f16 2e-3, f32 1.4e-6)
        if f32:
            return {"rel": 6e-6, "max": 4e-5, "differ": 0.0}
        return {"rel": 0.01, "max": 0.1, "differ": 0.1} if f16 else {"rel": 0.08, "max": 0.6, "differ": 0.25}
    if kind == "sample":        # a draw that falls on the other side of an edge between two words
        return {"rel": 0.0, "differ": 0.02}
    # (bf16 3e-3, rows that a norm makes large again 0.15; f16 an eighth of it)
    return {"rel": 2e-3, "max": 0.1} if f16 else {"rel": 1.2e-2, "max": 0.6}
