"""What this package's speed is measured on: the calls a user's program makes, over the sizes it makes them with.

Four kinds of case:

    gpt         one forward of the FP8 GPT with a KV cache (`GPT.forward_last`): a decode step of a batch, or a prompt
    stack       the same of a layer stack (Palilix, Zodirax), in bfloat16 or true 32-bit
    linear      a `Float8Linear`, inference or one training pass (output and both gradients)
    attention   the attention seam (`flash_attn_with_kvcache`) with rows of unequal length

`exact` states each of them once more in plain torch: float64 throughout, with the e4m3 / e5m2 roundings that define a tensorwise FP8
product, and nothing of this package but the inputs that `prepare` makes.
"""
import math

import torch
import torch.nn.functional as F

from nanochat_amd.engine import KVCache
from nanochat_amd.flash_attention import flash_attn
from nanochat_amd.fp8 import convert_to_float8_training
from nanochat_amd.gpt import compute_window_sizes
from nanochat_amd.palilix import Palilix
from nanochat_amd.synthetic import config_for_depth, palilix_config, random_init_model, random_stack_model, zodirax_config
from nanochat_amd.zodirax import Zodirax

DEVICE = "cuda"
HEAD = 128                                  # dimensions of a head, everywhere
DESIGNS = {"palilix": Palilix, "zodirax": Zodirax}
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}


def listed():
    return [
        # a chat with the smallest model, one sequence: nothing but launches and latency
        dict(name="gpt_step_d4_b1", kind="gpt", depth=4, kv_heads=0, batch=1, context=63, tokens=1, vocab=32768),
        # a few sampled continuations of a medium model
        dict(name="gpt_step_d20_b8", kind="gpt", depth=20, kv_heads=0, batch=8, context=640, tokens=1, vocab=32768),
        # the decode benchmark: d26, 64 sequences, a full context
        dict(name="gpt_step_d26_b64", kind="gpt", depth=26, kv_heads=0, batch=64, context=2047, tokens=1, vocab=32768),
        # the prompt in front of it
        dict(name="gpt_prompt_d26_1792", kind="gpt", depth=26, kv_heads=0, batch=1, context=0, tokens=1792, vocab=32768),
        # the linears by themselves, a batch of training tokens: evaluation, and a training pass
        dict(name="linear_8192_1664_6656", kind="linear", rows=8192, k=1664, n=6656, train=False),
        dict(name="train_8192_6656_1664", kind="linear", rows=8192, k=6656, n=1664, train=True),
        # grouped-query attention over 128 conversations of different lengths
        dict(name="attention_ragged_b128", kind="attention", batch=128, heads=16, kv_heads=4, tokens=1, context=2040, ragged=True, window=-1),
        # serving a layer stack: a full batch with experts and a small batch of the other design, and their prompts
        dict(name="palilix_step_b64", kind="stack", design="palilix", dtype="bfloat16", heads=16, groups=2, batch=64, context=2047, tokens=1, vocab=32768,
             dense=False, rank=512, experts=64, expert_ff=1024, window=0),
        dict(name="palilix_prompt_1792", kind="stack", design="palilix", dtype="bfloat16", heads=16, groups=2, batch=1, context=0, tokens=1792, vocab=32768,
             dense=False, rank=512, experts=64, expert_ff=1024, window=0),
        dict(name="zodirax_step_b16", kind="stack", design="zodirax", dtype="bfloat16", heads=16, groups=2, batch=16, context=2047, tokens=1, vocab=32768,
             dense=True, rank=0, experts=0, expert_ff=0, window=1024),
        dict(name="zodirax_prompt_w4096_1792", kind="stack", design="zodirax", dtype="bfloat16", heads=32, groups=1, batch=1, context=0, tokens=1792,
             vocab=32768, dense=True, rank=0, experts=0, expert_ff=0, window=1024),
        # true 32-bit, an odd prompt (checking a checkpoint, replaying a trace)
        dict(name="palilix_f32_prompt_333", kind="stack", design="palilix", dtype="float32", heads=8, groups=1, batch=1, context=0, tokens=333, vocab=32768,
             dense=False, rank=512, experts=64, expert_ff=512, window=0),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """Another case of the same ranges, odd sizes among them, none larger than the largest listed one of its kind."""
    kind = rng.choice(["gpt", "gpt", "stack", "stack", "stack", "linear", "linear", "attention"])
    if kind == "linear":
        train = rng.random() < 0.5
        rows = _log(rng, 1, 8192)
        # (a training pass takes rows in sixteens: the gradient's product sums over them)
        return dict(kind=kind, rows=16 * -(-rows // 16) if train else rows, k=16 * _log(rng, 16, 416), n=16 * _log(rng, 16, 416), train=train)
    if kind == "attention":
        kv = rng.choice([1, 2, 4, 5, 8])
        tokens = rng.choice([1, 1, 1, 2, 7, 40])
        return dict(kind=kind, batch=_log(rng, 1, 128 if tokens == 1 else 16), heads=kv * rng.choice([1, 2, 4]), kv_heads=kv, tokens=tokens, context=_log(rng, 64, 2000),
                    ragged=rng.random() < 0.5, window=rng.choice([-1, 511]))
    prompt = rng.random() < 0.45
    batch, context, tokens = (_log(rng, 1, 4), 0, _log(rng, 17, 1792)) if prompt else (_log(rng, 1, 64), _log(rng, 16, 2046), 1)
    if prompt:
        tokens = min(tokens, 1792 // batch)
        if rng.random() < 0.25:                     # a further portion of a longer prompt
            tokens = max(2, min(tokens, 500))
            context = _log(rng, 64, 1000)
    vocab = rng.choice([32768, 32768, _log(rng, 1000, 32000)])
    if kind == "gpt":
        depth = 2 * rng.randint(2, 13)
        heads = depth // 2
        return dict(kind=kind, depth=depth, kv_heads=heads // 2 if heads % 2 == 0 and rng.random() < 0.4 else 0, batch=batch, context=context, tokens=tokens, vocab=vocab)
    design = rng.choice(["palilix", "zodirax"])
    if rng.random() < 0.25:
        dtype, heads, groups, batch, tokens, context = "float32", rng.randint(3, 7), 1, min(batch, 16), min(tokens, 400 // batch or 1), min(context, 500)
    else:
        dtype, heads, groups = "bfloat16", rng.choice([4, 6, 7, 8, 12, 16]), rng.choice([1, 2])
    case = dict(kind=kind, design=design, dtype=dtype, heads=heads, groups=groups, batch=batch, context=context, tokens=max(1, tokens), vocab=vocab)
    if design == "palilix":
        return case | dict(dense=rng.random() < 0.3, rank=rng.choice([256, 512]), experts=rng.choice([16, 48, 64]), expert_ff=rng.choice([320, 512, 1024]), window=0)
    return case | dict(dense=True, rank=0, experts=0, expert_ff=0, window=rng.choice([100, 512, 1024]))


# ------------------------------------------------------------------------------------------------ inputs
def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _ids(g, batch, tokens, vocab):
    return torch.randint(0, vocab, (batch, tokens), generator=g, device=DEVICE)


def _gpt_config(case):
    return config_for_depth(case["depth"], vocab_size=case["vocab"], n_kv_head=case["kv_heads"] or None)


def _stack_config(case):
    width = case["heads"] * HEAD
    if case["design"] == "palilix":
        return palilix_config(width, case["heads"], rank=case["rank"], experts=case["experts"], expert_ff=case["expert_ff"], vocab=case["vocab"], groups=case["groups"],
                              dense=case["dense"])
    return zodirax_config(width, case["heads"], window=case["window"], vocab=case["vocab"], groups=case["groups"])


def _prepare_gpt(case, seed):
    """The model with its quantized weights, and a cache whose rows hold `context` tokens each (normed keys of length 1.2 sqrt(128))."""
    g = _generator(seed)
    cfg = _gpt_config(case)
    model = random_init_model(cfg, DEVICE, seed=seed)
    with torch.no_grad():
        # the sublayers write a part of the residual stream, not most of it.  (At full size a chain of FP8 layers multiplies a last-bit
        # difference up to 4 % of the logits, whatever computes it: two correct implementations could not be told from a wrong one.)
        for block in model.transformer.h:
            block.attn.c_proj.weight.mul_(GPT_PROJECTIONS)
            block.mlp.c_proj.weight.mul_(GPT_PROJECTIONS)
    B, n, T = case["batch"], case["context"], case["tokens"]
    cache = KVCache(B, cfg.n_kv_head, n + T, HEAD, cfg.n_layer, DEVICE, torch.bfloat16)
    if n:
        for k, v in zip(cache.k_cache, cache.v_cache):
            k[:, :n].normal_(0.0, 1.2, generator=g)
            v[:, :n].normal_(0.0, 1.0, generator=g)
        cache.advance(n)
        cache.prev_embedding = F.rms_norm(torch.randn(B, 1, cfg.n_embd, generator=g, device=DEVICE), (cfg.n_embd,)).bfloat16()
    state = dict(kind="gpt", model=model, cache=cache, ids=_ids(g, B, T, case["vocab"]))
    model._ensure_plan()
    return state


GPT_PROJECTIONS = 0.1


def _prepare_stack(case, seed):
    """The model, a cache with `context` tokens (one prompt, copied into every row as the Engine does), and the next tokens of every row."""
    g = _generator(seed)
    model = random_stack_model(DESIGNS[case["design"]], _stack_config(case), DEVICE, DTYPES[case["dtype"]], seed=seed)
    with torch.no_grad():
        for name, t in model.held_tensors().items():
            if name.endswith("router"):
                t.mul_(6.0)             # scores apart, as trained ones are: where all experts score alike, a last bit swaps two that weigh the same
    B, n, T = case["batch"], case["context"], case["tokens"]
    prompt, ids = _ids(g, 1, max(n, 1), case["vocab"]), _ids(g, B, T, case["vocab"])
    one = None
    if n:
        one = model.new_cache(1, n)
        model.forward_last(prompt, kv_cache=one)
    cache = model.new_cache(B, n + T, prefill_from=one)
    model._ensure_plan(n + T)
    return dict(kind="stack", model=model, cache=cache, ids=ids, prompt=prompt)


def _prepare_linear(case, seed):
    g = _generator(seed)
    rows, k, n = case["rows"], case["k"], case["n"]
    s = 3 ** 0.5 * k ** -0.5
    holder = torch.nn.Sequential(torch.nn.Linear(k, n, bias=False, device=DEVICE, dtype=torch.bfloat16))
    with torch.no_grad():
        holder[0].weight.uniform_(-s, s, generator=g)
    convert_to_float8_training(holder)
    x = torch.randn(rows, k, generator=g, device=DEVICE).bfloat16().requires_grad_(case["train"])
    grad = (1e-3 * torch.randn(rows, n, generator=g, device=DEVICE)).bfloat16()
    return dict(kind="linear", linear=holder[0].requires_grad_(case["train"]), x=x, grad=grad if case["train"] else None)


def _prepare_attention(case, seed):
    g = _generator(seed)
    B, T, H, G, n = (case[k] for k in ("batch", "tokens", "heads", "kv_heads", "context"))

    def normal(scale, *shape):
        return torch.empty(*shape, device=DEVICE, dtype=torch.bfloat16).normal_(0.0, scale, generator=g)
    lengths = torch.randint(max(1, n // 32), n + 1, (B,), generator=g, device=DEVICE, dtype=torch.int32) if case["ragged"] else torch.full((B,), n, device=DEVICE, dtype=torch.int32)
    return dict(kind="attention", q=normal(1.2, B, T, H, HEAD), k=normal(1.2, B, T, G, HEAD), v=normal(1.0, B, T, G, HEAD), k_cache=normal(1.2, B, n + T, G, HEAD),
                v_cache=normal(1.0, B, n + T, G, HEAD), lengths=lengths, window=(case["window"], 0))


def prepare(case, seed):
    return {"gpt": _prepare_gpt, "stack": _prepare_stack, "linear": _prepare_linear, "attention": _prepare_attention}[case["kind"]](case, seed)


# ------------------------------------------------------------------------------------------------ a pass
def run(state):
    if state["kind"] == "attention":
        y = flash_attn.flash_attn_with_kvcache(state["q"], state["k_cache"], state["v_cache"], k=state["k"], v=state["v"], cache_seqlens=state["lengths"], causal=True,
                                               window_size=state["window"])
        return y, state["k_cache"], state["v_cache"]
    if state["kind"] == "linear":
        linear, x, grad = state["linear"], state["x"], state["grad"]
        if grad is None:
            with torch.no_grad():
                return linear(x)
        out = linear(x)
        return (out, *torch.autograd.grad(out, (x, linear.weight), grad))
    # a forward, then one token position back: the next pass finds the cache as this one did
    model, cache, ids = state["model"], state["cache"], state["ids"]
    pos, tokens, before = cache.get_pos(), ids.shape[1], cache.mark()
    out = {"logits": model.forward_last(ids, kv_cache=cache)}
    if state["kind"] == "gpt":
        out |= {"k": cache.k_cache[:, :, pos:], "v": cache.v_cache[:, :, pos:], "embedding": cache.prev_embedding}
    else:
        out |= {"rows": [r[:, pos:] for r in cache.rows], "states": list(cache.state_buffers()[0])}
    cache.rewind(tokens, before)
    return out


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _pairs(context, tokens, window):
    """(query, key) pairs of a causal window of `window` keys, and the keys that are read."""
    return sum(min(context + t + 1, window) for t in range(tokens)), min(context + tokens, window + tokens - 1)


def work(case):
    if case["kind"] == "linear":
        rows, k, n = case["rows"], case["k"], case["n"]
        if case["train"]:
            return {"bytes": 2 * rows * k * 2 + n * k * 3 + rows * n * 2 * 2, "flops": 6 * rows * k * n}
        return {"bytes": rows * k * 2 + n * k + rows * n * 2, "flops": 2 * rows * k * n}
    B, n, T = case["batch"], case["context"], case["tokens"]
    if case["kind"] == "attention":
        window = case["window"] + 1 if case["window"] >= 0 else 1 << 30
        pairs, keys = _pairs(n // 2 if case["ragged"] else n, T, window)
        return {"bytes": B * 2 * HEAD * (2 * case["heads"] * T + 2 * case["kv_heads"] * (keys + T)), "flops": B * 4 * HEAD * case["heads"] * pairs}
    V = case["vocab"]
    if case["kind"] == "gpt":
        cfg = _gpt_config(case)
        kv = cfg.n_kv_head * HEAD
        params = cfg.n_layer * cfg.n_embd * (2 * cfg.n_embd + 2 * kv + 8 * cfg.n_embd)
        each = [_pairs(n, T, w + 1) for w, _ in compute_window_sizes(cfg)]
        return {"bytes": params + V * cfg.n_embd + B * (sum(k for _, k in each) * 4 * kv + 4 * V + T * (cfg.n_layer * 4 * kv + 2 * cfg.n_embd)),
                "flops": B * (2 * params * T + 2 * V * cfg.n_embd + sum(p for p, _ in each) * 4 * cfg.n_embd)}
    return _stack_work(_stack_config(case), B, n, T, 2 if case["dtype"] == "bfloat16" else 4)


def _stack_work(cfg, B, n, T, size):
    """Weights once (of the experts, those that B * T tokens are expected to choose), cached rows and states in and out, the tokens' products."""
    W, V = cfg["width"], cfg["vocab"]
    weights, flops, cache = V * W, B * 2 * V * W, 4 * B * V
    for layer in cfg["layers"]:
        m, f = layer["mixer"], layer["mlp"]
        dense = 0
        for part in ([m["left"], m["right"]] if layer["type"] == "parallel" else [m]):
            if layer["type"] == "latent_attention":
                H, d, r, e, rank = part["heads"], part["dim"], part["rot_dim"], part["vdim"], part["kv_rank"]
                dense += W * (H * (d + r) + rank + r + H * e) + rank * H * (d + e)
                pairs, keys = _pairs(n, T, 1 << 30)
                # per pair the fewer of the two forms: heads expanded, or in the latent space (one token)
                flops += B * 2 * H * pairs * (min(d + e, 2 * rank) + r if T > 1 else 2 * rank + r)
                cache += B * size * (keys + T) * (rank + r)
            elif "kv_heads" in part:
                H, G, d = part["heads"], part["kv_heads"], part["dim"]
                dense += W * d * (2 * H + 2 * G)
                pairs, keys = _pairs(n, T, part["mask"]["size"] + part["mask"]["keep_first"])
                flops += B * 4 * H * d * pairs
                cache += B * size * (keys + T) * 2 * G * d
            elif "decay" in part:
                H, d, e = part["heads"], part["dim"], part["vdim"]
                dense += W * H * (2 * d + 3 * e)
                flops += B * T * 4 * H * d * e
                cache += B * 4 * H * d * e * (2 if n else 1)
            else:
                inner, s, rank = part["inner"], part["state"], part["dt_rank"]
                dense += inner * (3 * W + 2 * rank + 2 * s)
                flops += B * T * 6 * inner * s
                cache += B * 4 * inner * (s + part["conv"] - 1) * (2 if n else 1)
        if f and f["kind"] == "moe":
            E, top, ff, shared = f["router"]["experts"], f["router"]["top"], f["expert"]["ff"], f["shared"]["ff"]
            dense += W * (E + 3 * shared)
            weights += 3 * W * ff * E * (1 - (1 - top / E) ** (B * T))
            flops += B * T * 6 * W * ff * top
        elif f:
            dense += W * f["ff"] * (2 if cfg["architecture"] == "Palilix" else 3)
        weights, flops = weights + dense, flops + B * T * 2 * dense
    return {"bytes": size * (weights + B * T * W) + cache, "flops": flops}


# ------------------------------------------------------------------------------------------------ tolerances
def tolerance(case):
    """Relative error (2-norm) of an output, about four times what the path shows against float64 (linear, attention, 32-bit: 1.7e-3, 1.7e-3,
    2e-6) or, where layers of rounded operands follow each other, against itself with the cached positions summed in another order
    (GPT and Palilix 1e-2, Zodirax 4e-3)."""
    if case["kind"] == "linear":
        return {"rel": 8e-3, "max": 0.05}
    if case["kind"] == "attention":
        return {"rel": 1e-2, "max": 0.1}
    if case["kind"] == "stack" and case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 2e-3}
    return {"rel": 1.5e-2 if case.get("design") == "zodirax" else 3e-2, "max": 0.9}


# ------------------------------------------------------------------------------------------------ the same in 64 bits
def _to_fp8(x, dtype=torch.float8_e4m3fn):
    """What a tensorwise FP8 product sees of x: x times (largest value of the format / largest magnitude), rounded, and back."""
    scale = (torch.finfo(dtype).max / x.abs().max().double().clamp(min=1e-12)).float()
    return (x.float() * scale).clamp(-torch.finfo(dtype).max, torch.finfo(dtype).max).to(dtype).double() / scale.double()


def _rms(x, eps, weight=1.0):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight


def _turn(x, angle, sign=1):
    """Pairs (i, i + r) of the last axis by `angle` [..., r] (its table of cosines and sines may have been rounded); the rest passes."""
    cos, sin = angle
    r = cos.shape[-1]
    a, b = x[..., :r], x[..., r:2 * r]
    return torch.cat([a * cos - sign * b * sin, b * cos + sign * a * sin, x[..., 2 * r:]], dim=-1)


def _attend(q, k, v, seen, scale, sink=None):
    """q [B,T,H,d], k [B,n,G,d], v [B,n,G,e], seen [1 or B,T,n] -> [B,T,H,e]; head h reads key head h // (H / G)."""
    B, T, H, d = q.shape
    G, R, n = k.shape[2], H // k.shape[2], k.shape[1]
    q = q.view(B, T, G, R, d).permute(0, 2, 3, 1, 4).reshape(B * G, R * T, d)
    s = torch.bmm(q, k.permute(0, 2, 3, 1).reshape(B * G, d, n)).mul_(scale).view(B, G, R, T, n)
    s.masked_fill_(~seen[:, None, None], -math.inf)
    if sink is None:
        p = s.softmax(-1)
    else:
        s0 = sink.view(1, G, R, 1, 1)
        top = torch.maximum(s.amax(-1, keepdim=True), s0)
        p = (s - top).exp_()
        p /= p.sum(-1, keepdim=True) + (s0 - top).exp()
    y = torch.bmm(p.view(B * G, R * T, n), v.permute(0, 2, 1, 3).reshape(B * G, n, -1))
    return y.view(B, G, R, T, -1).permute(0, 3, 1, 2, 4).reshape(B, T, H, -1)


def _seen(context, tokens, window, keep_first=0):
    i = context + torch.arange(tokens, device=DEVICE)[:, None]
    j = torch.arange(context + tokens, device=DEVICE)[None, :]
    return ((j <= i) & ((i - j < window) | (j < keep_first)))[None]


def _exact_linear(case, seed):
    s = prepare(case, seed)
    x, w = _to_fp8(s["x"].detach()), _to_fp8(s["linear"].weight.detach())
    if not case["train"]:
        return x @ w.T
    g = _to_fp8(s["grad"], torch.float8_e5m2)
    return (x @ w.T, g @ w, g.T @ x)


def _exact_attention(case, seed):
    s = prepare(case, seed)
    out = []
    for b, n in enumerate(s["lengths"].tolist()):
        for c in ("k", "v"):
            s[c + "_cache"][b, n:n + case["tokens"]] = s[c][b]
        k, v = (s[c + "_cache"][b:b + 1, :n + case["tokens"]].double() for c in ("k", "v"))
        window = case["window"] + 1 if case["window"] >= 0 else 1 << 30
        out.append(_attend(s["q"][b:b + 1].double(), k, v, _seen(n, case["tokens"], window), HEAD ** -0.5))
    return torch.cat(out), s["k_cache"].double(), s["v_cache"].double()


def _exact_gpt(case, seed):
    s = prepare(case, seed)
    cfg, cache, ids = _gpt_config(case), s["cache"], s["ids"]
    p = {k: v for k, v in s["model"].state_dict().items()}
    B, T, n, H, G, E = *ids.shape, case["context"], cfg.n_head, cfg.n_kv_head, cfg.n_embd
    eps = torch.finfo(torch.float32).eps

    def d(name):
        return p[name].double()

    def linear(x8, name):
        return x8 @ _to_fp8(p[name]).T
    # (the model's table: fp32 angles, rounded to bfloat16)
    freq = 1.0 / (100000 ** (torch.arange(0, HEAD, 2, dtype=torch.float32, device=DEVICE) / HEAD))
    angles = torch.outer(torch.arange(n, n + T, dtype=torch.float32, device=DEVICE), freq)[None, :, None]
    angle = (angles.cos().bfloat16().double(), angles.sin().bfloat16().double())
    x = _rms(d("transformer.wte.weight")[ids], eps)
    embedding = x[:, -1:]
    before = torch.cat([torch.zeros_like(x[:, :1]), x[:, :-1]], dim=1) if T > 1 else cache.prev_embedding.double() if cache.prev_embedding is not None else torch.zeros_like(x)
    x = x + d("smear_lambda") * torch.sigmoid(x[..., :24] @ d("smear_gate.weight").T) * before
    x0, back, ks, vs = x, None, [], []
    for i, (window, _) in enumerate(compute_window_sizes(cfg)):
        at = f"transformer.h.{i}."
        x = d("resid_lambdas")[i] * x + d("x0_lambdas")[i] * x0
        h = _rms(x, eps)
        h8 = _to_fp8(h)
        q, k, v = (linear(h8, f"{at}attn.c_{c}.weight").view(B, T, -1, HEAD) for c in "qkv")
        if f"value_embeds.{i}.weight" in p:
            gate = 3 * torch.sigmoid(h[..., :12] @ d(at + "attn.ve_gate.weight").T)
            v = v + gate[..., None] * p[f"value_embeds.{i}.weight"][ids].double().view(B, T, G, HEAD)
        q, k = (1.2 * _rms(_turn(t, angle, -1), eps) for t in (q, k))
        ks.append(k.bfloat16())
        vs.append(v.bfloat16())
        lo = max(0, n - window)
        keys, values = (torch.cat([c[i][:, lo:n].double(), t], dim=1) for c, t in ((cache.k_cache, k), (cache.v_cache, v)))
        y = _attend(q, keys, values, _seen(n, T, window + 1)[..., lo:], HEAD ** -0.5)
        x = x + linear(_to_fp8(y.reshape(B, T, E)), at + "attn.c_proj.weight")
        h = linear(_to_fp8(_rms(x, eps)), at + "mlp.c_fc.weight").relu().square()
        x = x + linear(_to_fp8(h), at + "mlp.c_proj.weight")
        if i == cfg.n_layer // 2:
            back = x
    x = _rms(x - d("backout_lambda") * back, eps)[:, -1:] if T == 1 else _rms(x - d("backout_lambda") * back, eps)
    logits = linear(_to_fp8(x)[:, -1], "lm_head.weight")[:, :cfg.vocab_size]
    return {"logits": 15 * torch.tanh(logits / 15), "k": torch.stack(ks).double(), "v": torch.stack(vs).double(), "embedding": embedding}


def _frequencies(rot):
    f = torch.tensor([float(rot["base"]) ** (-2.0 * i / rot["dims"]) for i in range(rot["dims"] // 2)], dtype=torch.float64, device=DEVICE)
    if "scaling" not in rot:
        return f
    s = rot["scaling"]
    mix = ((s["original"] * f / (2 * math.pi) - s["low"]) / (s["high"] - s["low"])).clamp(0.0, 1.0)
    return (1 - mix) * f / s["factor"] + mix * f


def _angle(rot, n, T):
    a = torch.outer(torch.arange(n, n + T, dtype=torch.float64, device=DEVICE), _frequencies(rot))[None, :, None]
    return a.cos(), a.sin()


class _Stack:
    """A layer stack over float64 weights, a sequence of portions: `memory[layer]` keeps what the mixers remember."""

    def __init__(self, case, model):
        self.cfg = _stack_config(case)
        self.w = {k: v.detach() for k, v in model.named_tensors().items()}
        self.eps = self.cfg["norm"]["eps"]
        self.memory = {}
        self.n = 0

    def d(self, name):
        return self.w[name].double()

    def forward(self, ids):
        cfg, eps, palilix = self.cfg, self.eps, self.cfg["architecture"] == "Palilix"
        x = self.d("embed")[ids] * cfg["embedding"]["scale"]
        norm = self.layer_norm if palilix else lambda v, name: _rms(v, eps, 1 + self.d(name))
        rows, states = [], []
        for i, layer in enumerate(cfg["layers"]):
            h = norm(x, f"l{i}.norm1") if palilix else x
            at, m = f"l{i}.mix.", layer["mixer"]
            if layer["type"] == "parallel":
                left, kv = self.window_attention(h, at + "left.", m["left"])
                right, state = self.retention(h, at + "right.", m["right"])
                y = m["left_scale"] * left + m["right_scale"] * right
                rows.append(kv)
                states.append(state)
            elif layer["type"] == "latent_attention":
                y, row = self.latent_attention(h, at, m)
                rows.append(row)
            else:
                y, state = self.retention(h, at, m) if layer["type"] == "retention" else self.scan(h, at, m)
                states.append(state)
            if palilix:
                x = x + y + self.feed_forward(h, f"l{i}.mlp.", layer["mlp"])
            else:
                x = x + norm(y, f"l{i}.norm1")
                f = f"l{i}.mlp."
                x = x + norm((F.silu(x @ self.d(f + "gate").T) * (x @ self.d(f + "up").T)) @ self.d(f + "down").T, f"l{i}.norm2")
        self.n += ids.shape[1]
        last = norm(x[:, -1], "final.norm") @ self.d("head" if palilix else "embed").T
        if palilix:
            cap = cfg["logit_softcap"]
            last = cap * torch.tanh(last * cfg["logit_scale"] / cap)
        return {"logits": last, "rows": rows, "states": states}

    def layer_norm(self, x, name):
        x = x - x.mean(-1, keepdim=True)
        return _rms(x, self.eps, self.d(name))

    def keep(self, name, new):
        """`new` [B,T,...] behind what is kept under the name (one row's memory serves every row of a batch)."""
        old = self.memory.get(name)
        both = new if old is None else torch.cat([old.expand(new.shape[0], *old.shape[1:]), new], dim=1)
        self.memory[name] = both
        return both

    def latent_attention(self, h, at, m):
        B, T, _ = h.shape
        H, dn, r, rank = m["heads"], m["dim"], m["rot_dim"], m["kv_rank"]
        angle = _angle(m["rot"], self.n, T)
        q = (h @ self.d(at + "q").T).view(B, T, H, -1)
        low = h @ self.d(at + "dkv").T
        new = torch.cat([_rms(low[..., :rank], self.eps, self.d(at + "dkv.norm")), _turn(low[..., None, rank:], angle)[:, :, 0]], dim=-1)
        rows = self.keep(at, new)
        k = torch.cat([(rows[..., :rank] @ self.d(at + "uk").T).view(B, -1, H, dn), rows[:, :, None, rank:].expand(-1, -1, H, -1)], dim=-1)
        v = (rows[..., :rank] @ self.d(at + "uv").T).view(B, -1, H, m["vdim"])
        y = _attend(torch.cat([q[..., :dn], _turn(q[..., dn:], angle)], dim=-1), k, v, _seen(self.n, T, 1 << 30), m["scale"])
        return y.reshape(B, T, -1) @ self.d(at + "o").T, new

    def window_attention(self, h, at, m):
        B, T, _ = h.shape
        angle = _angle(m["rot"], self.n, T)
        q, k, v = (h @ self.d(at + c).T + self.d(f"{at}{c}.b") for c in "qkv")
        q, k = (_turn(_rms(t, self.eps, self.d(f"{at}{c}.norm")).view(B, T, -1, m["dim"]), angle) for t, c in ((q, "q"), (k, "k")))
        G = m["kv_heads"]
        new = torch.cat([k, v.view(B, T, G, -1)], dim=-1).view(B, T, -1)               # a cached row: every head's key and value
        k, v = self.keep(at, new).view(B, self.n + T, G, m["dim"] + m["vdim"]).split([m["dim"], m["vdim"]], dim=-1)
        seen = _seen(self.n, T, m["mask"]["size"], m["mask"]["keep_first"])
        y = _attend(q, k, v, seen, m["scale"], self.d(at + "sink"))
        return y.reshape(B, T, -1) @ self.d(at + "o").T, new

    def retention(self, h, at, m):
        """Over a portion: o_i = decay^(i+1) q_i S + sum over j <= i of decay^(i-j) (q_i . k_j) v_j."""
        B, T, _ = h.shape
        joint = "rot" not in m                                  # lightning attention: silu on q, k, v; one norm over all heads, sigmoid gate
        q, k, v = ((h @ self.d(at + c).T).view(B, T, m["heads"], -1) for c in "qkv")
        if joint:
            q, k, v = F.silu(q), F.silu(k), F.silu(v)
        else:
            angle = _angle(m["rot"], self.n, T)
            q, k = _turn(q, angle), _turn(k, angle) * m["dim"] ** -0.5
        q, k, v = (t.permute(0, 2, 1, 3).contiguous() for t in (q, k, v))
        # (the model holds its decays in 32 bits)
        log = torch.tensor(m["decay"], dtype=torch.float32, device=DEVICE).double().log()[:, None, None]
        t = torch.arange(T, dtype=torch.float64, device=DEVICE)
        apart = t[:, None] - t[None, :]
        old = self.memory.get(at)
        old = torch.zeros(1, *q.shape[1:2], q.shape[3], v.shape[3], dtype=q.dtype, device=DEVICE) if old is None else old
        fade = torch.where(apart >= 0, torch.exp(log * apart.clamp(min=0)), 0.0)
        o = torch.matmul(torch.matmul(q, k.transpose(2, 3).contiguous()) * fade, v) + torch.matmul(q * torch.exp(log * (t + 1)[:, None]), old)
        state = old * torch.exp(log * T) + torch.matmul((k * torch.exp(log * (T - 1 - t)[:, None])).transpose(2, 3).contiguous(), v)
        self.memory[at] = state
        o = o.permute(0, 2, 1, 3)
        g = h @ self.d(at + "g").T
        if joint:
            o = _rms(o.reshape(B, T, -1), self.eps, self.d(at + "norm")) * torch.sigmoid(g)
        else:
            o = _rms(o, self.eps).reshape(B, T, -1) * F.silu(g)
        return o @ self.d(at + "o").T, state

    def scan(self, h, at, m):
        B, T, _ = h.shape
        inner, taps = m["inner"], m["conv"]
        x, z = (h @ self.d(at + "in").T).split([inner, inner], dim=-1)
        old, S = self.memory.get(at, (torch.zeros(1, taps - 1, inner, dtype=h.dtype, device=DEVICE), torch.zeros(1, inner, m["state"], dtype=h.dtype, device=DEVICE)))
        padded = torch.cat([old.expand(B, -1, -1), x], dim=1)
        u = F.silu(sum(padded[:, i:i + T] * self.d(at + "conv")[:, i] for i in range(taps)) + self.d(at + "conv.b"))
        step, b, c = (u @ self.d(at + "x").T).split([m["dt_rank"], m["state"], m["state"]], dim=-1)
        dt = F.softplus(step @ self.d(at + "dt").T + self.d(at + "dt.b"))
        A = -self.d(at + "A_log").exp()
        S, y = S.expand(B, -1, -1), []
        for t in range(T):
            S = torch.exp(dt[:, t, :, None] * A) * S + (dt[:, t] * u[:, t])[..., None] * b[:, t, None, :]
            y.append((S * c[:, t, None, :]).sum(-1))
        self.memory[at] = (padded[:, T:], S)
        y = torch.stack(y, dim=1) + self.d(at + "D") * u
        return (y * F.silu(z)) @ self.d(at + "o").T, torch.cat([S.transpose(1, 2), padded[:, T:]], dim=1)

    def feed_forward(self, h, at, m):
        if m["kind"] == "dense":
            return F.gelu(h @ self.d(at + "up").T, approximate="tanh") @ self.d(at + "down").T

        def glu(x, name, limit):
            gate, up = (x @ self.d(f"{name}.gate").T).clamp(max=limit), (x @ self.d(f"{name}.up").T).clamp(-limit, limit)
            return (gate * torch.sigmoid(1.702 * gate) * (up + 1)) @ self.d(f"{name}.down").T
        flat = h.reshape(-1, h.shape[-1])
        score, chosen = (flat @ self.d(at + "router").T).softmax(-1).topk(m["router"]["top"], dim=-1)
        score = score / score.sum(-1, keepdim=True)
        y = glu(flat, at + "shared", m["shared"]["limit"])
        for e in range(m["router"]["experts"]):
            row, place = (chosen == e).nonzero(as_tuple=True)
            if len(row):
                y.index_add_(0, row, score[row, place, None] * glu(flat[row], f"{at}e{e}", m["expert"]["limit"]))
        return y.view_as(h)


def _exact_stack(case, seed):
    s = prepare(case, seed)
    stack = _Stack(case, s["model"])
    if case["context"]:
        stack.forward(s["prompt"])
    return stack.forward(s["ids"])


@torch.no_grad()
def exact(case, seed):
    return {"gpt": _exact_gpt, "stack": _exact_stack, "linear": _exact_linear, "attention": _exact_attention}[case["kind"]](case, seed)
