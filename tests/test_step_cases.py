"""The bars of the step in one launch (tests/step_cases.py) would show a mistake: the oracle, on the CPU, with a stretch of keys lost or one key too many or too few."""
import pytest
import torch

from oracle import decode_ref, gpt_ref
from step_cases import KV_BAR, LOGIT_BAR, STEP_CASES, appended, apart, fill, first_seen, step_model


def oracle_step(rt, cfg, case, spoil=None):
    cache = fill(decode_ref.new_cache(cfg, len(case.lengths), max(case.lengths) + 2, torch.bfloat16), cfg, case)
    cache.cache_seqlens.copy_(torch.tensor(case.lengths, dtype=torch.int32))
    if spoil:
        spoil(cache)
    toks = torch.randint(0, 1024, (len(case.lengths), 1), generator=torch.Generator().manual_seed(7))
    logits = gpt_ref.forward(rt, toks, cache)[:, -1]
    return logits, appended(cache, case.lengths, 0)


@pytest.mark.parametrize("case", [c for c in STEP_CASES if c.heads <= 9 and 0 < max(c.lengths) and c.kv_heads * sum(c.lengths) <= 30000], ids=str)
def test_bars_of_a_step_would_show_a_lost_stretch_of_keys(case):
    """Each layer's first, last and middle run of keys (24, or of long rows what one of 24 workgroups reads), its first key and its last one (of rows up to 1000), of all rows; and a window that is
    one key too wide or too narrow: the next layer's keys or values of each row, or its logits behind the last layer, are further off than twice what the comparison on the GPU allows."""
    lengths, long = case.lengths, max(case.lengths) > 1000
    model = step_model(case, "cpu")
    cfg = model.config
    params = {k: v.detach() for k, v in model.state_dict().items()}
    rt = gpt_ref.Runtime(gpt_ref.GPTConfig(**{k: getattr(cfg, k) for k in ("sequence_len", "vocab_size", "n_layer", "n_head", "n_kv_head", "n_embd", "window_pattern")}), params,
                         compute_dtype=torch.bfloat16, fp8=True, uniform_sdpa=False)
    logits, kv = oracle_step(rt, cfg, case)
    windows = list(rt.windows)

    def shown(i, rows, spoiled, what):
        off = apart(spoiled[1][:, i + 1], kv[:, i + 1]).amax(0) / KV_BAR if i + 1 < case.layers else apart(spoiled[0], logits) / LOGIT_BAR
        for b in rows:
            assert off[b] > 2, f"layer {i}, row {b} of {lengths[b]}, {what}: {off[b]:.2f} times the bar"
    holding = [b for b, n in enumerate(lengths) if n > 0]
    for i in range(case.layers):
        def runs(n):
            lo = first_seen(windows[i][0], n)
            mid, run = lo + (n - lo) // 2, max(case.apart, n // 24 if long else 0)
            found = {"first run": (lo, lo + run), "middle run": (mid, mid + run), "last run": (max(lo, n - run), n)}
            return found if long else found | {"first key": (lo, lo + 1), "last key": (n - 1, n)}
        for what in runs(1):
            def lose(cache):
                for b in holding:
                    first, end = runs(lengths[b])[what]
                    cache.v_cache[i, b, first:min(end, lengths[b])] = 0
            shown(i, holding, oracle_step(rt, cfg, case, lose), what)
        past = [b for b, n in enumerate(lengths) if 0 <= windows[i][0] < n and not long]
        for more in (1, -1):
            rt.windows[i] = (windows[i][0] + more, windows[i][1])
            if past:
                shown(i, past, oracle_step(rt, cfg, case), f"window {more:+d}")
            rt.windows[i] = windows[i]
