"""Decode steps of few rows whose outcome hangs on each stretch of keys: what tests/test_gpu_gpt.py compares and how far it may be off, and (tests/test_step_cases.py, on the CPU) that
a lost or an extra stretch is further off than that."""
from typing import NamedTuple

import torch
import torch.nn.functional as F

from nanochat_amd.gpt import GPTConfig, compute_window_sizes
from nanochat_amd.synthetic import random_init_model



class Case(NamedTuple):
    layers: int
    heads: int
    kv_heads: int
    lengths: list
    pattern: str
    sequence_len: int = 512
    apart: int = 24                   # one key of so many stands out: a wave's run of keys is a batch of its loads at least, 24 or 32 of them, so each run has one


# the edges of the launch's forms: 512, 1024, 1536 and 1792 columns, one and two query heads to a key head, one row and eight, rows that are empty, of one batch of keys
# and one more, at the border of a workgroup's share of keys (128), past a window, and of unequal length; then rows of more keys than 12 workgroups share, up to what 13 and 24 of them do, and
# so many keys that a narrow model takes all units
STEP_CASES = [Case(3, 2, 2, [0], "SSL"), Case(4, 2, 2, [63, 1], "SSL"), Case(3, 4, 4, [127, 128, 129], "SL"), Case(5, 4, 2, [300], "LS"), Case(3, 5, 5, [5] * 8, "SSL"),
              Case(4, 8, 4, [0, 31, 32, 33, 256, 257, 500, 511], "SL"), Case(3, 9, 9, [700, 2], "LS"), Case(3, 12, 6, [40] * 7, "SSL"), Case(4, 13, 13, [1000], "LS"),
              Case(3, 13, 13, [600] * 8, "SL"), Case(3, 14, 7, [513, 512, 511], "SL"), Case(3, 14, 14, [130] * 4, "LS"),
              Case(3, 1, 1, [13311, 30, 13312], "L", 32768, 100), Case(3, 2, 1, [30000], "L", 32768, 150), Case(3, 2, 2, [26000, 9, 25000], "LS", 32768, 120),
              Case(3, 4, 4, [8000, 700, 8001, 6000], "L", 8192, 72)]
# Relative, per row: of a layer's appended keys or values, and of the logits.  The forms that are compared round in the same places and sum in another order, so most values have the same bits;
# where a sum rounds the other way a bf16 value moves by 2^-8 of itself and an e4m3 value by 2^-3, one of the 256 or more terms of the next product: 2^-3 / sqrt(256) = 0.8 % of its row.
KV_BAR, LOGIT_BAR = 1e-2, 2e-2


def step_model(case, device, seed=5):
    """Random weights, with attention a large part of the residual stream (of the last layer, which only logits show, the largest) and the MLP a small one."""
    cfg = GPTConfig(sequence_len=case.sequence_len, vocab_size=1024, n_layer=case.layers, n_head=case.heads, n_kv_head=case.kv_heads, n_embd=128 * case.heads,
                    window_pattern=case.pattern)
    model = random_init_model(cfg, device, seed=seed)
    with torch.no_grad():
        for block in model.transformer.h:
            block.mlp.c_proj.weight.mul_(0.1)
        model.transformer.h[-1].attn.c_proj.weight.mul_(4.0)
    return model


def first_seen(window, n):
    """The first of n cached keys that the next token sees."""
    return 0 if window < 0 else max(0, n - window)


def fill(cache, cfg, case, seed=6):
    """Rows that hold the case's tokens, and the embedding of the last one.  Values of every `apart`th key that is seen, of the first and of the last, and of all that are not to be seen, stand out
    by so much that attention is about them: each of the first counts as many times as there are others between them (of more than 16 more, as their
    sum's length goes with the root of their number)."""
    device = cache.k_cache.device
    g = torch.Generator(device=device).manual_seed(seed)
    cache.k_cache.normal_(0.0, 1.2, generator=g)
    cache.v_cache.normal_(0.0, 1.0, generator=g)
    for i, (window, _) in enumerate(compute_window_sizes(cfg)):
        for b, n in enumerate(case.lengths):
            lo = first_seen(window, n)
            marks = sorted({*range(lo, n, case.apart), *([n - 1] if n else [])})
            scale = torch.full((cache.v_cache.shape[2],), max(1.0, (n - lo) / max(1.0, len(marks) * min(len(marks), 16)) ** 0.5), device=device)
            loud = scale[0].item()
            scale[lo:n] = 0.3
            scale[marks] = loud
            cache.v_cache[i, b] *= scale[:, None, None].to(cache.v_cache.dtype)
    cache.prev_embedding = F.rms_norm(torch.randn(len(case.lengths), 1, cfg.n_embd, generator=g, device=device), (cfg.n_embd,)).bfloat16()
    return cache


def appended(cache, lengths, step):
    """Keys and values of the token that step 0, 1, .. appended: [2, layers, rows, kv heads * 128]."""
    return torch.stack([torch.stack([c[:, b, n + step] for b, n in enumerate(lengths)], dim=1) for c in (cache.k_cache, cache.v_cache)]).flatten(3).float()


def apart(got, want):
    """Relative difference of every row (over the last axis)."""
    got, want = got.float(), want.float()
    return (got - want).norm(dim=-1) / want.norm(dim=-1).clamp_min(1e-30)
