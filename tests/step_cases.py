"""Decode steps of few rows whose outcome hangs on each stretch of keys: what tests/test_gpu_gpt.py compares and how far it may be off, and (tests/test_step_cases.py, on the CPU) that
a lost or an extra stretch is further off than that."""
import torch
import torch.nn.functional as F

from nanochat_amd.gpt import GPTConfig, compute_window_sizes
from nanochat_amd.synthetic import random_init_model

# the edges of the launch's forms: 512, 1024, 1536 and 1792 columns, one and two query heads to a key head, one row and eight, rows that are empty, of one batch of keys
# and one more, at the border of a workgroup's share of keys (128), past a window, and of unequal length: layers, heads, key heads, rows, windows
STEP_CASES = [(3, 2, 2, [0], "SSL"), (4, 2, 2, [63, 1], "SSL"), (3, 4, 4, [127, 128, 129], "SL"), (5, 4, 2, [300], "LS"), (3, 5, 5, [5] * 8, "SSL"),
              (4, 8, 4, [0, 31, 32, 33, 256, 257, 500, 511], "SL"), (3, 9, 9, [700, 2], "LS"), (3, 12, 6, [40] * 7, "SSL"), (4, 13, 13, [1000], "LS"), (3, 13, 13, [600] * 8, "SL"),
              (3, 14, 7, [513, 512, 511], "SL"), (3, 14, 14, [130] * 4, "LS")]
# A wave's run of keys is a batch of its loads at least, 24 or 32 of them: with a key that stands out every 24 each run has one
APART = 24
# Relative, per row: of a layer's appended keys or values, and of the logits.  The forms that are compared round in the same places and sum in another order, so most values have the same bits;
# where a sum rounds the other way a bf16 value moves by 2^-8 of itself and an e4m3 value by 2^-3, one of the 256 or more terms of the next product: 2^-3 / sqrt(256) = 0.8 % of its row.
KV_BAR, LOGIT_BAR = 1e-2, 2e-2


def step_model(layers, heads, kv_heads, pattern, device, seed=5):
    """Random weights, with attention a large part of the residual stream (of the last layer, which only logits show, the largest) and the MLP a small one."""
    cfg = GPTConfig(sequence_len=512, vocab_size=1024, n_layer=layers, n_head=heads, n_kv_head=kv_heads, n_embd=128 * heads, window_pattern=pattern)
    model = random_init_model(cfg, device, seed=seed)
    with torch.no_grad():
        for block in model.transformer.h:
            block.mlp.c_proj.weight.mul_(0.1)
        model.transformer.h[-1].attn.c_proj.weight.mul_(4.0)
    return model


def first_seen(window, n):
    """The first of n cached keys that the next token sees."""
    return 0 if window < 0 else max(0, n - window)


def fill(cache, cfg, lengths, seed=6):
    """Rows that hold `lengths` tokens each, and the embedding of the last one.  Values of every 24th key that is seen, of the first and of the last, and of all that are not to be seen, stand out
    by so much that attention is about them: each of the first counts as many times as there are others between them."""
    device = cache.k_cache.device
    g = torch.Generator(device=device).manual_seed(seed)
    cache.k_cache.normal_(0.0, 1.2, generator=g)
    cache.v_cache.normal_(0.0, 1.0, generator=g)
    for i, (window, _) in enumerate(compute_window_sizes(cfg)):
        for b, n in enumerate(lengths):
            lo = first_seen(window, n)
            marks = sorted({*range(lo, n, APART), *([n - 1] if n else [])})
            scale = torch.full((cache.v_cache.shape[2],), max(1.0, (n - lo) / max(1, len(marks))), device=device)
            loud = scale[0].item()
            scale[lo:n] = 0.3
            scale[marks] = loud
            cache.v_cache[i, b] *= scale[:, None, None].to(cache.v_cache.dtype)
    cache.prev_embedding = F.rms_norm(torch.randn(len(lengths), 1, cfg.n_embd, generator=g, device=device), (cfg.n_embd,)).bfloat16()
    return cache


def appended(cache, lengths, step):
    """Keys and values of the token that was appended `step` tokens ago counted from the first: [2, layers, rows, kv heads * 128]."""
    return torch.stack([torch.stack([c[:, b, n + step] for b, n in enumerate(lengths)], dim=1) for c in (cache.k_cache, cache.v_cache)]).flatten(3).float()


def apart(got, want):
    """Relative difference of every row (over the last axis)."""
    got, want = got.float(), want.float()
    return (got - want).norm(dim=-1) / want.norm(dim=-1).clamp_min(1e-30)
