"""Palilix on the GPU against the plain restatement in oracle/palilix_ref.py (float64): whole prompts, decoding, portions, batches of
unequal sequences, slots that are used again, generation through the Engine; both storage types."""
import ctypes
import functools
import json
import math

import pytest
import torch

from nanochat_amd import ops
from nanochat_amd.engine import Engine
from nanochat_amd.palilix import Palilix
from nanochat_amd.registry import load_model
from nanochat_amd.synthetic import SyntheticTokenizer
from oracle import palilix_ref as ref
from palilix_cases import CASES, config, dense, latent, moe, retention, variant, weights
from stack_helpers import BAR, DEV, DTYPES, build_model, check, ids, judge, rel_rms, run, say, tokens, trace_runner, write_model

pytestmark = pytest.mark.gpu


@functools.lru_cache(maxsize=None)
def case_weights(name):
    return weights(CASES[name], seed=len(name))


@functools.lru_cache(maxsize=None)
def oracle_logits(name, n):
    cfg = CASES[name]
    return ref.forward(cfg, {k: v.double() for k, v in case_weights(name).items()}, tokens(cfg, n))


@functools.lru_cache(maxsize=None)
def case_model(name, dtype):
    return build(CASES[name], case_weights(name), dtype)


def build(cfg, w, dtype):
    return build_model(Palilix, cfg, w, dtype)


# ------------------------------------------------------------------------------------------------ linears
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind", [0, 1, 2, 3, 6, 7])
def test_linear_kernels(dtype, kind):
    say(f"linears, kind {kind}, {dtype}")
    g = torch.Generator().manual_seed(kind)
    for M, N, K in [(1, 16, 64), (3, 48, 128), (16, 1040, 192), (17, 96, 64), (33, 144, 448), (64, 80, 704), (65, 256, 64), (129, 144, 320), (300, 1072, 128)]:
        a, w = torch.randn(M, K, generator=g).to(dtype), (torch.randn(N, K, generator=g) / K ** 0.5).to(dtype)
        want = a.double() @ w.double().T
        if kind == 1:
            want = ref.gelu_tanh(want)
        elif kind == 2:
            want = ref.clamped_glu(want[:, 0::2], want[:, 1::2], 0.6)
        elif kind == 6:
            want = ref.silu(want)
        elif kind == 7:
            want = ref.silu(want[:, 0::2]) * want[:, 1::2]
        for kernel in (1, 2, 3, 4):
            got = ops.stack_linear(a.to(DEV), w.to(DEV), kind=kind, limit=0.6, kernel=kernel).cpu()
            tol = 1e-2 if got.dtype == torch.bfloat16 else 2e-5
            assert torch.allclose(got.double(), want, rtol=tol, atol=tol), (M, N, K, kernel, (got.double() - want).abs().max().item())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kernel", (3, 4, 5, 6, 7, 8))
def test_tiles_at_their_edges(kernel, dtype):
    """One row and column group less than a tile, a tile, one more; sums of one, two and three K-steps and more than the ring of stages holds."""
    say(f"tile edges, kernel {kernel}, {dtype}")
    g = torch.Generator().manual_seed(5)
    steps = 64 if dtype == torch.bfloat16 else 32
    for M, N, K in [(1, 16, 1), (31, 48, 2), (33, 80, 9), (63, 112, 1), (64, 128, 2), (65, 144, 3), (127, 240, 4), (128, 256, 5), (129, 272, 7), (257, 528, 4)]:
        K = -(-K * steps // 64) * 64
        a, w = torch.randn(M, K, generator=g).to(dtype), (torch.randn(N, K, generator=g) / K ** 0.5).to(dtype)
        got = ops.stack_linear(a.to(DEV), w.to(DEV), kernel=kernel).cpu()
        tol = 1e-2 if dtype == torch.bfloat16 else 2e-5       # one rounding to bf16 is 2^-9 of values up to about 4; fp32 sums of up to 320 terms
        assert torch.allclose(got.double(), a.double() @ w.double().T, rtol=tol, atol=tol), (M, N, K)


@pytest.mark.parametrize("kind", [0, 1, 2, 3, 6, 7])
def test_wide_tiles_have_the_sums_of_the_others(kind):
    """Tiles of 256 x 256 and halves of them (the last but one: 256 whole and 90 half ones, the last row of halves ending behind the last column), to the bit."""
    say(f"256 x 256 tiles, kind {kind}")
    g = torch.Generator(device=DEV).manual_seed(9)
    for M, N, K in [(1, 16, 64), (255, 144, 128), (256, 256, 192), (257, 528, 320), (300, 1072, 448), (1700, 10912, 192), (1792, 4096, 64)]:
        a, w = torch.randn(M, K, generator=g, device=DEV).bfloat16(), (torch.randn(N, K, generator=g, device=DEV) / K ** 0.5).bfloat16()
        want = ops.stack_linear(a, w, kind=kind, limit=0.6, kernel=4)
        assert torch.equal(ops.stack_linear(a, w, kind=kind, limit=0.6, kernel=9), want), (M, N, K)


# columns and kind of each run; the ends lie inside tiles of 256, inside halves of them, on a tile's border, and the last one inside a group of eight columns
WIDE_RUNS = {"mixers, router, GLU": [(208, 0), (64, 3), (432, 2)], "residual": [(560, 4)], "residual behind a border": [(256, 0), (304, 4)], "logits": [(1003, 5)],
             "four": [(16, 6), (240, 7), (144, 1), (201, 5)]}


@pytest.mark.parametrize("M", [130, 257, 1700])
@pytest.mark.parametrize("runs", WIDE_RUNS)
def test_wide_tiles_of_stacked_weights(runs, M):
    """What a forward sends through the 256 x 256 tiles: several runs of columns, sums added to the residual stream, logits; whole tiles and, for 1700 rows, halves
    behind 256 of them.  To the bit those of the 64 x 64 tiles, also where the kernel is chosen; the rows of A lie apart, and nothing else is
    written."""
    say(f"256 x 256 tiles, {runs}, {M} rows")
    g = torch.Generator(device=DEV).manual_seed(M)
    parts = WIDE_RUNS[runs]
    if M == 1700 and len(parts) < 4:
        parts = [(9472, 0)] + parts                  # (280 tiles and more; those behind the 256th are cut into halves)
    N, K = sum(cols for cols, _ in parts), 192
    a, w = torch.randn(M, K + 64, generator=g, device=DEV).bfloat16()[:, :K], (torch.randn(N, K, generator=g, device=DEV) / K ** 0.5).bfloat16()
    stream = torch.randn(M, 1024, generator=g, device=DEV)
    got = []
    for kernel in (4, 9, 0):
        # (rows longer than their columns, and a row behind the last)
        room = [torch.full((M + 1, (cols // 2 if kind in (2, 7) else cols) + 8), 7.0, dtype=torch.float32 if kind in (3, 4, 5) else torch.bfloat16, device=DEV) for cols, kind in parts]
        views = [t[:M, :-8] for t in room]
        for (cols, kind), v in zip(parts, views):
            if kind == 4:
                v.copy_(stream[:, :cols])
        ops.stack_linear_runs(a, w, [(cols, kind, v) for (cols, kind), v in zip(parts, views)], limit=0.6, kernel=kernel)
        assert all((t[M] == 7).all() and (t[:, -8:] == 7).all() for t in room)
        got.append([v.clone() for v in views])
    assert all(torch.equal(x, y) for other in got[1:] for x, y in zip(got[0], other))


@pytest.mark.parametrize("dtype", DTYPES)
def test_few_rows_have_the_same_sums_in_every_kernel(dtype):
    """Up to 64 rows a result does not depend on the kernel or the tile: the same additions in the same order, to the bit (sums of one K-step, of
    steps that do not divide by four, and of chains that begin in the middle of one)."""
    say(f"same sums, {dtype}")
    g = torch.Generator().manual_seed(6)
    for M, N, K in [(1, 16, 64), (5, 80, 192), (16, 144, 320), (17, 64, 704), (33, 208, 1088), (64, 320, 1792)]:
        a, w = torch.randn(M, K, generator=g).to(DEV, dtype), torch.randn(N, K, generator=g).to(DEV, dtype)
        want = ops.stack_linear(a, w, kind=3, kernel=1)
        for kernel in (6, 7, 8):
            assert torch.equal(ops.stack_linear(a, w, kind=3, kernel=kernel), want), (M, N, K, kernel)


@pytest.mark.parametrize("dtype", DTYPES)
def test_whatever_kernel_is_chosen_for_few_rows_has_the_same_sums(dtype):
    """The choice, on both sides of its borders (rows, columns, length of the sum), against a tile; sums whose quarters are 8, 12, 14 and 23 steps
    of 64 bytes, that is whole and broken batches of the few-rows kernel."""
    say(f"chosen kernel, {dtype}")
    g = torch.Generator().manual_seed(7)
    for M, N, K in [(1, 48, 1024), (16, 80, 1536), (4, 4112, 1792), (5, 4112, 1024), (4, 8208, 1024), (16, 8208, 512), (17, 8192, 512), (32, 8208, 512), (33, 64, 512), (2, 12304, 2944)]:
        a, w = torch.randn(M, K, generator=g).to(DEV, dtype), torch.randn(N, K, generator=g).to(DEV, dtype)
        want = ops.stack_linear(a, w, kind=3, kernel=6)
        for kernel in (0, 1):
            assert torch.equal(ops.stack_linear(a, w, kind=3, kernel=kernel), want), (M, N, K, kernel)


@pytest.mark.parametrize("M,K", [(1, (1 << 20) + 64), (20, (1 << 20) + 64), (64, (1 << 23) + 64)])
def test_long_sums_of_few_rows(M, K):
    """Sums of more than 2^20 terms, and 64 rows of them that make an operand of more than 2 GiB."""
    say(f"long sums, {M} rows of {K}")
    g = torch.Generator(device=DEV).manual_seed(8)
    a, w = torch.randn(M, K, generator=g, device=DEV), torch.randn(48, K, generator=g, device=DEV) / K ** 0.5
    want = sum(p.double() @ q.double().T for p, q in zip(a.split(1 << 20, 1), w.split(1 << 20, 1)))
    got = ops.stack_linear(a, w)
    # Four chains of K / 4 terms of size K^-1/2: after t terms a chain is t^1/2 K^-1/2, and adding a term rounds that by 2^-24 of it at most.  The squares
    # add up to (K / 4)^2 / (2 K) 2^-48 a chain, K / 8 2^-48 for the four; five standard deviations of that for the largest of 3072 results.
    bound = 5 * 2.0 ** -24 * (K / 8) ** 0.5
    assert (got.double() - want).abs().max().item() < bound


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", [31, 100])
def test_bytes_that_the_profile_states_for_the_recurrence(n, dtype):
    """Projections in and outputs out in the storage type; the states (fp32) once in and out token by token, four times per chunk in chunks."""
    say(f"profile of the recurrence, {n} tokens, {dtype}")
    heads, dim = 2, 64
    cfg = config([(retention(heads=heads, dim=dim, vdim=dim, rot_dims=32), None)], vocab=50)
    model, lib = build(cfg, weights(cfg, seed=2), dtype), ops._lib.stack_lib()
    lib.nc_profile_enable(1)
    try:
        run(model, tokens(cfg, n), [n])
        torch.cuda.synchronize()
        ms, units, launches = ops.C.c_double(), ops.C.c_double(), ops.C.c_int64()
        assert lib.nc_profile_read(2, ops.C.byref(ms), ops.C.byref(units), ops.C.byref(launches)) == 0
    finally:
        lib.nc_profile_enable(0)
    size, chunk = (4, 32) if dtype == torch.float32 else (2, 64)
    states = 2 if n < 32 else 4 * -(-n // chunk)
    assert launches.value == 1 and units.value == heads * (n * 5 * dim * size + states * 4 * dim * dim)


# ------------------------------------------------------------------------------------------------ whole prompts
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", list(CASES))
def test_whole_prompt(name, dtype):
    say(f"whole prompt, {name}, {dtype}")
    for n in (1, 2, 45, 150):
        toks = tokens(CASES[name], n)
        check(run(case_model(name, dtype), toks, [n]), oracle_logits(name, n), dtype, f"{name}, {n} tokens")


@pytest.mark.parametrize("name", ["odd", "wide"])
def test_32_bit_portions_at_the_edges_of_their_kernels(name):
    """32 tokens to a chunk of the recurrence, 16 query rows and 64 keys to a block of the latent attention: one less, as many, one more, alone and
    behind other portions."""
    say(f"32-bit portions, {name}")
    for cuts in ([31], [32], [33], [64], [65], [7, 32, 33], [64, 8, 63]):
        n = sum(cuts)
        check(run(case_model(name, torch.float32), tokens(CASES[name], n), cuts), oracle_logits(name, n), torch.float32, f"{name}, portions {cuts}")


@pytest.mark.parametrize("name", ["odd", "wide"])
def test_32_bit_portions_of_more_query_rows_than_compute_units(name):
    """3 or 4 heads: from 86 or 65 tokens on 16 query rows share a block of keys; a last block of rows and of keys that is full, short by one or
    has one, alone and behind other portions."""
    say(f"32-bit portions of many rows, {name}")
    for cuts in ([85], [86], [96], [97], [64, 128], [7, 121], [100, 91], [257]):
        n = sum(cuts)
        check(run(case_model(name, torch.float32), tokens(CASES[name], n), cuts), oracle_logits(name, n), torch.float32, f"{name}, portions {cuts}")


@pytest.mark.parametrize("name", ["odd", "wide"])
def test_32_bit_portions_of_unequal_sequences(name):
    """24 tokens to each of five sequences of different lengths: their query rows together are more than the compute units, none shares another's keys."""
    say(f"32-bit portions of unequal sequences, {name}")
    cfg, model = CASES[name], case_model(name, torch.float32)
    w64, lengths, new = {k: v.double() for k, v in case_weights(name).items()}, [3, 70, 33, 1, 104], 24
    seqs = [tokens(cfg, n + new, seed=40 + n) for n in lengths]
    cache = model.new_cache(len(seqs), 128)
    for r, (s, n) in enumerate(zip(seqs, lengths)):
        alone = model.new_cache(1, 128)
        model.forward_last(ids(s[:n]), kv_cache=alone)
        cache.load_row(r, alone)
    got = model.forward(torch.tensor([s[n:] for s, n in zip(seqs, lengths)], device=DEV), kv_cache=cache)
    for r, (s, n) in enumerate(zip(seqs, lengths)):
        check(got[r], ref.forward(cfg, w64, s)[n:], torch.float32, f"{name}, row {r}")


def test_32_bit_scores_of_many_rows_are_as_exact_as_of_few():
    """A whole prompt (16 query rows share their keys) against portions of 7 (one row each; a score in four chains of 144 terms), both against 64
    bits.  Rounding of a chain grows with its length: with a prompt's scores in two chains of 288 its error was 1.71 to 1.80 times that of the
    portions in six draws, in four 1.52 to 1.60 (its other products have longer chains than those of few rows)."""
    say("32-bit scores")
    whole = portions = 0.0
    for seed in range(3):
        cfg = config([(latent(heads=8, dim=128, rot_dim=64, vdim=128, kv_rank=512, scale=0.2), None)], width=256, vocab=300)
        w, toks = weights(cfg, seed=seed), tokens(cfg, 140, seed=seed)
        model, want = build(cfg, w, torch.float32), ref.forward(cfg, {k: v.double() for k, v in w.items()}, toks)
        whole += (run(model, toks, [140]).double().cpu() - want).norm().item()
        portions += (run(model, toks, [7] * 20).double().cpu() - want).norm().item()
    assert whole < 1.66 * portions, whole / portions


@pytest.mark.parametrize("experts", [7, 64, 65])
def test_choices_of_several_rows_side_by_side(experts):
    """Up to 64 rows choose in one workgroup, one, two or four rows to a wave: row counts at those borders, and experts of one and several to a lane."""
    say(f"choices of several rows, {experts} experts")
    cfg = config([(latent(), moe(experts=experts, top=6, ff=16))], vocab=50)
    w, toks = weights(cfg, seed=11), tokens(cfg, 65)
    model, want = build(cfg, w, torch.float32), ref.forward(cfg, {k: v.double() for k, v in w.items()}, toks)
    for n in (1, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65):
        check(run(model, toks[:n], [n]), want[:n], torch.float32, f"{n} rows")


@pytest.mark.parametrize("heads,rank,rot_dim", [(5, 512, 64), (1, 256, 32), (3, 200, 64), (2, 320, 0), (7, 512, 32)])
def test_32_bit_steps_whose_keys_are_shared_out(heads, rank, rot_dim):
    """Single tokens and portions of a few behind 0, 1, 63, 64, 65 and 300 cached ones: runs of keys that are empty, ragged or a single key, one and several
    shares of a row's keys, alone and for three sequences of different lengths."""
    say(f"32-bit steps, {heads} heads, rank {rank}, {rot_dim} rotated")
    cfg = config([(latent(heads=heads, dim=32, rot_dim=rot_dim, vdim=32, kv_rank=rank, scale=0.2), None)], width=128, vocab=90)
    w = weights(cfg, seed=5)
    model, w64 = build(cfg, w, torch.float32), {k: v.double() for k, v in w.items()}
    for cuts in ([1] * 5, [62, 1, 1, 1, 1], [300, 1, 2, 5], [63, 7]):
        n = sum(cuts)
        check(run(model, tokens(cfg, n), cuts), ref.forward(cfg, w64, tokens(cfg, n)), torch.float32, f"portions {cuts}")
    lengths = [3, 130, 65]
    seqs = [tokens(cfg, n + 2, seed=60 + n) for n in lengths]
    cache = model.new_cache(len(seqs), 160)
    for r, (s, n) in enumerate(zip(seqs, lengths)):
        alone = model.new_cache(1, 160)
        model.forward_last(ids(s[:n]), kv_cache=alone)
        cache.load_row(r, alone)
    for i in range(2):
        got = model.forward(torch.tensor([s[n + i:n + i + 1] for s, n in zip(seqs, lengths)], device=DEV), kv_cache=cache)
        for r, (s, n) in enumerate(zip(seqs, lengths)):
            check(got[r], ref.forward(cfg, w64, s[:n + i + 1])[-1:], torch.float32, f"step {i}, row {r}")


@pytest.mark.parametrize("width", [64, 512, 1024])
@pytest.mark.parametrize("ff", [2048, 2112, 1984])
def test_32_bit_shares_that_begin_in_the_middle_of_a_step(width, ff):
    """The output matrix of many rows in four shares of 33 half steps (ff = 2048), of 34 and of 32: a share may begin with the second half of a step.  Whole prompts against portions of few rows, which take other kernels."""
    say(f"shares, width {width}, ff {ff}")
    cfg = config([(retention(heads=1, dim=64, vdim=64, rot_dims=32), dense(ff=ff))] * 2, width=width, vocab=50)
    model = build(cfg, weights(cfg, seed=3), torch.float32)
    for n in (65, 80, 130, 400):
        toks = tokens(cfg, n)
        few = run(model, toks, [50] * (n // 50) + ([n % 50] if n % 50 else [])).cpu()
        for again in range(3):
            check(run(model, toks, [n]), few, torch.float32, f"{n} rows")


@pytest.mark.parametrize("dtype", DTYPES)
def test_rows_of_a_longer_prompt_have_the_same_bits(dtype):
    """From 65 tokens on a token's result is what it is in a shorter prompt that begins alike: one order of the sums for any number of rows."""
    say(f"prompts of other lengths, {dtype}")
    cfg = config([(latent(heads=8, dim=64), dense(ff=1100)), (retention(heads=2, dim=64, vdim=64, rot_dims=32), dense(ff=4096))], width=1024, vocab=50)
    model = build(cfg, weights(cfg, seed=3), dtype)
    toks = tokens(cfg, 700)
    want = run(model, toks, [700])
    for n in (65, 97, 333, 576):
        if dtype == torch.float32 or n >= 333:                # (bf16 latent attention changes its form between)
            assert torch.equal(run(model, toks[:n], [n]), want[:n]), n


@pytest.mark.parametrize("dtype", DTYPES)
def test_residual_stream_after_every_run(dtype):
    say(f"layer by layer, {dtype}")
    cfg, taps = CASES["odd"], []
    toks = tokens(cfg, 70)
    want = ref.forward(cfg, {k: v.double() for k, v in case_weights("odd").items()}, toks, taps)
    model = case_model("odd", dtype)
    logits, got = model.forward_tapped(ids(toks))
    check(logits[0], want, dtype, "logits")
    assert got.shape == (len(ref.layer_runs(cfg)), 1, 70, cfg["width"]) == (len(taps), 1, 70, cfg["width"])
    for i, t in enumerate(taps):
        check(got[i, 0], t, dtype, f"run {i}")


def mechanism(layer, mlp=None, **kw):
    return config([(layer, mlp)], width=64, vocab=50, **kw)


MECHANISMS = {
    "latent": mechanism(latent()),
    "latent, peaked scores": mechanism(latent(heads=2, dim=32, rot_dim=32, vdim=32, kv_rank=64, scale=1.5)),
    "retention": mechanism(retention()),
    "retention, slow decay": mechanism(retention(heads=2, dim=64, vdim=64, rot_dims=32, decay=[0.9993, 0.9985])),
    "retention, nothing kept and all kept": mechanism(retention(heads=2, dim=64, vdim=64, rot_dims=32, decay=[0.0, 1.0])),
    "dense": mechanism(retention(heads=1, dim=16, vdim=16, rot_dims=8), dense()),
    "experts": mechanism(retention(heads=1, dim=16, vdim=16, rot_dims=8), moe(experts=33, top=5)),
    "experts and shared": mechanism(retention(heads=1, dim=16, vdim=16, rot_dims=8), moe(shared=(40, 0.2))),
    "loop": mechanism(latent(heads=2), loop=(0, 1, 4)),
    "no layers in the loop": mechanism(latent(heads=2), loop=(1, 1, 2)),
}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", list(MECHANISMS))
def test_each_mechanism(name, dtype):
    """One layer of each kind: prompt at once, and token by token."""
    say(f"mechanism {name}, {dtype}")
    cfg = MECHANISMS[name]
    w = weights(cfg, seed=3)
    toks = tokens(cfg, 100)
    want = ref.forward(cfg, {k: v.double() for k, v in w.items()}, toks)
    model = build(cfg, w, dtype)
    # (a score of tens of units turns the rounding of a bf16 query into a change of weight)
    # and a head that sees one key only answers with its value times the sign of the score
    bar = {"latent, peaked scores": 0.15, "retention, nothing kept and all kept": 0.15}.get(name) if dtype == torch.bfloat16 else None
    check(run(model, toks, [100]), want, dtype, name, bar)
    check(run(model, toks, [1] * 100), want, dtype, name + ", token by token", bar)


def planted_mistakes():
    """(name, mechanism, function of the oracle that is replaced, replacement)."""
    def half_of_it(g, u, lim):
        return g.clamp(max=lim) * torch.sigmoid(1.702 * g.clamp(max=lim)) * (u.clamp(max=lim) + 1)

    def gate_on_both_sides(g, u, lim):
        return g.clamp(-lim, lim) * torch.sigmoid(1.702 * g.clamp(-lim, lim)) * (u.clamp(-lim, lim) + 1)

    return [("decay off by a thousandth", "retention, slow decay", "retention",
             lambda h, wt, c, eps: RETENTION(h, wt, dict(c, decay=[d * (1 - 1e-3) for d in c["decay"]]), eps)),
            ("rotation base a hundredth off", "latent, peaked scores", "rotate", lambda x, pos, base, dims: ROTATE(x, pos, base * 1.01, dims)),
            ("epsilon forgotten in the latent's norm", "latent", "rms_norm", lambda x, eps, weight=None: RMS_NORM(x, 0.03, weight)),
            ("weights not divided by their sum", "experts", "route", lambda h, r, top: torch.softmax(h @ r.T, -1).topk(top, -1)[::-1]),
            ("up not clamped below", "experts and shared", "clamped_glu", half_of_it),
            ("gate clamped below", "experts and shared", "clamped_glu", gate_on_both_sides),
            ("erf-like gelu", "dense", "gelu_tanh", lambda z: torch.nn.functional.gelu(z)),
            ("embedding output not added again", "loop", "layer_runs", lambda cfg: [(i, t if t == 0 else None) for i, t in LAYER_RUNS(cfg)])]


RETENTION, LAYER_RUNS, ROTATE, RMS_NORM = ref.retention, ref.layer_runs, ref.rotate, ref.rms_norm


@pytest.mark.parametrize("mistake", planted_mistakes(), ids=lambda m: m[0])
def test_bars_would_show_a_mistake(mistake, monkeypatch):
    """The same comparison with a mistake planted in the oracle fails clearly."""
    name, case, function, wrong = mistake
    say(f"planted mistake: {name}")
    cfg = MECHANISMS[case]
    w = weights(cfg, seed=3)
    toks = tokens(cfg, 100)
    w64 = {k: v.double() for k, v in w.items()}
    good = ref.forward(cfg, w64, toks)
    monkeypatch.setattr(ref, function, wrong)
    bad = ref.forward(cfg, w64, toks)
    got = run(build(cfg, w, torch.float32), toks, [len(toks)])
    check(got, good, torch.float32, name)
    err = rel_rms(got, bad)[-1].item()
    print(f"{name}: {err:.2e} at the last position")
    assert err > 5 * BAR[torch.float32]


# ------------------------------------------------------------------------------------------------ a far key that stands out
@pytest.mark.parametrize("dtype", DTYPES)
def test_keys_at_the_borders_of_the_kernels_blocks(dtype):
    """One key stands out for one query: the query's answer is that key's value.  Every place where a block of keys, a portion or a share
    of the keys begins or ends is visited, in prompts, in portions and in decoding."""
    say(f"keys that stand out, {dtype}")
    cfg = mechanism(latent(heads=2, dim=32, rot_dim=32, vdim=32, kv_rank=64, scale=0.3, base=2e5))
    w = weights(cfg, seed=5)
    # token 0 asks for token 1: their embeddings are opposite, and a query's unrotated part is minus the unrotated key of its own token
    W = cfg["width"]
    probe = torch.randn(W, generator=torch.Generator().manual_seed(9))
    w["embed"][1], w["embed"][0] = (3 * probe).bfloat16(), (-3 * probe).bfloat16()
    uk, q = w["l0.mix.uk"].float().view(2, 32, 64), w["l0.mix.q"].float().view(2, 64, W)
    q[:, :32] = -1.5 * uk @ w["l0.mix.dkv"].float()[:64]
    w["l0.mix.q"], w["l0.mix.o"] = q.view(-1, W).bfloat16(), 4 * w["l0.mix.o"]
    w64 = {k: v.double() for k, v in w.items()}
    n = 330
    model = build(cfg, w, dtype)
    g = torch.Generator().manual_seed(2)
    filler = torch.randint(2, cfg["vocab"], (n,), generator=g).tolist()
    bar = 6e-2 if dtype == torch.bfloat16 else None
    for key in (0, 1, 31, 32, 63, 64, 127, 128, 255, 256):
        toks = list(filler)
        toks[key] = 1
        for at in (key + 1, key + 2, 319, 320, n - 1):
            toks[at] = 0
        want = ref.forward(cfg, w64, toks)
        shifted = list(toks)
        shifted[key] = filler[key]
        there = rel_rms(ref.forward(cfg, w64, shifted), want)[n - 1].item()
        assert there > 0.3, (key, there)              # the answer at the end rests on this key
        check(run(model, toks, [n]), want, dtype, f"key {key}, whole", bar)
        check(run(model, toks, [63, 65, 2, 126, 64] + [1] * (n - 320)), want, dtype, f"key {key}, portions", bar)


# ------------------------------------------------------------------------------------------------ cuts
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["odd", "wide", "ones", "large_heads"])
def test_portions_and_decoding(name, dtype):
    say(f"cuts of one sequence, {name}, {dtype}")
    n = 150
    toks, model, want = tokens(CASES[name], n), case_model(name, dtype), oracle_logits(name, n)
    for cuts in ([2] * 75, [1] * 150, [33, 2, 64, 3, 31, 17], [149, 1], [1, 149], [64, 64, 22], [32, 32, 32, 54], [5, 140, 2, 2, 1]):
        check(run(model, toks, cuts), want, dtype, f"{name}, cuts {cuts[:6]}")


def test_long_decoding():
    say("long decoding")
    name, n = "odd", 420
    toks, want = tokens(CASES[name], n), oracle_logits(name, n)
    for dtype in DTYPES:
        check(run(case_model(name, dtype), toks, [20] + [1] * (n - 20), seq_len=1000), want, dtype, "20 + 400 tokens")


def test_results_do_not_depend_on_the_cache_length():
    say("cache length")
    toks, model = tokens(CASES["wide"], 40), case_model("wide", torch.bfloat16)
    a, b = (run(model, toks, [30] + [1] * 10, seq_len=s) for s in (40, 3000))
    assert rel_rms(a, b.double().cpu()).max().item() < 1e-2


# ------------------------------------------------------------------------------------------------ batches, slots
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["odd", "wide"])
def test_unequal_sequences_in_one_batch(name, dtype):
    """Sequences of different lengths share a cache: their decode steps equal those of each alone; then some rows end, and their
    slots take new sequences."""
    say(f"unequal batch, {name}, {dtype}")
    cfg, model = CASES[name], case_model(name, dtype)
    lengths, steps = [3, 70, 34, 1, 129], 6
    seqs = [tokens(cfg, n + 2 * steps, seed=10 + n) for n in lengths]
    w64 = {k: v.double() for k, v in case_weights(name).items()}
    cache = model.new_cache(len(seqs), 160)
    want = [ref.forward(cfg, w64, s) for s in seqs]

    def admit(row, toks):
        alone = model.new_cache(1, 160)
        got = model.forward_last(ids(toks), kv_cache=alone)
        cache.load_row(row, alone)
        return got[0]

    for r, (s, n) in enumerate(zip(seqs, lengths)):
        check(admit(r, s[:n])[None], want[r][n - 1:n], dtype, f"row {r} prompt")
    at = list(lengths)

    def step_all():
        col = torch.tensor([[s[p]] for s, p in zip(seqs, at)], dtype=torch.long, device=DEV)
        got = model.forward_last(col, kv_cache=cache)
        for r in range(len(seqs)):
            errors[r].append(rel_rms(got[r][None], want[r][at[r]:at[r] + 1]))
            at[r] += 1

    def run_steps():
        for e in errors:
            e.clear()
        for _ in range(steps):
            step_all()
        for r, e in enumerate(errors):
            judge(torch.cat(e), dtype, f"row {r} up to {at[r]}")
    errors = [[] for _ in seqs]
    run_steps()
    assert cache.cache_seqlens.tolist() == at
    # rows 1 and 4 end; new sequences take their slots, one of them token by token from an empty slot
    cache.reset_rows([1, 4])
    seqs[1], seqs[4] = tokens(cfg, 40, seed=77), tokens(cfg, 2 * steps, seed=78)
    want[1], want[4] = ref.forward(cfg, w64, seqs[1]), ref.forward(cfg, w64, seqs[4])
    admit(1, seqs[1][:30])
    at[1], at[4] = 30, 0
    run_steps()


@pytest.mark.parametrize("dtype", DTYPES)
def test_prompts_of_several_rows_at_once(dtype):
    say(f"several rows, {dtype}")
    cfg, model = CASES["wide"], case_model("wide", dtype)
    w64 = {k: v.double() for k, v in case_weights("wide").items()}
    seqs = [tokens(cfg, 90, seed=s) for s in (1, 2, 3)]
    for cuts in ([90], [40, 2, 48], [3] * 30):
        cache = model.new_cache(3, 90)
        at, outs = 0, []
        for n in cuts:
            outs.append(model.forward(torch.tensor([s[at:at + n] for s in seqs], device=DEV), kv_cache=cache))
            at += n
        got = torch.cat(outs, dim=1)
        for r, s in enumerate(seqs):
            check(got[r], ref.forward(cfg, w64, s), dtype, f"row {r} of 3, cuts {cuts[:3]}")


@pytest.mark.parametrize("mixer", [latent(heads=8, dim=32, kv_rank=200), latent(heads=3, kv_rank=56), retention(heads=2, dim=40, vdim=72), retention(heads=1, dim=128, vdim=128)])
@pytest.mark.parametrize("at", [0, 70, 95, 99])
def test_a_later_nan_does_not_reach_earlier_tokens(mixer, at):
    """A token whose embedding is NaN in the middle of the tokens that share its block of keys or its chunk, in 32-bit (in bfloat16 the matrix-core
    kernels have always multiplied masked weights): what comes before it is what it is without it, what comes after it is NaN."""
    say(f"a NaN at token {at}, {mixer['type']}")
    cfg = config([(mixer, None)], vocab=50)
    w, toks = weights(cfg, seed=12), [t or 1 for t in tokens(cfg, 100)]
    want = ref.forward(cfg, {k: v.double() for k, v in w.items()}, toks)
    w["embed"][0] = math.nan
    toks[at] = 0
    got = run(build(cfg, w, torch.float32), toks, [100])
    assert torch.isnan(got[at:]).all()
    if at:
        check(got[:at], want[:at], torch.float32, f"{at} tokens before a NaN")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("experts,top", [(4, 4), (4, 2), (16, 8), (1, 1)])
def test_experts_of_few_rows_have_the_same_sums_in_every_batch(experts, top, dtype):
    """64 sequences, 16 to 64 of them to an expert, against the same ones 20 and 33 at a time: tiles of 64 or of 32 rows, the same additions."""
    say(f"experts in batches, {top} of {experts}, {dtype}")
    cfg = config([(latent(), moe(experts=experts, top=top, ff=320))], width=320, vocab=70)
    model = build(cfg, weights(cfg, seed=9), dtype)
    toks = torch.arange(64, device=DEV)[:, None]
    want = model.forward_last(toks, kv_cache=model.new_cache(64, 2)).clone()
    for part in (20, 33):
        got = torch.cat([model.forward_last(p, kv_cache=model.new_cache(len(p), 2)).clone() for p in (toks[:part], toks[64 - part:])])
        assert torch.equal(got, torch.cat([want[:part], want[64 - part:]])), part


def spoiled_rows_leave_the_others_alone(cfg, rows, spoiled, dtype):
    """One token to each of `rows` sequences; those of `spoiled` bring a token whose embedding is NaN: the others' logits are what they are where
    every sequence is a healthy one, to the bit."""
    w = weights(cfg, seed=8)
    w["embed"][0] = math.nan
    model = build(cfg, w, dtype)
    healthy = torch.tensor([[1 + r % (cfg["vocab"] - 1)] for r in range(rows)], device=DEV)
    some = healthy.clone()
    some[spoiled] = 0
    want = model.forward_last(healthy, kv_cache=model.new_cache(rows, 4)).clone()
    got = model.forward_last(some, kv_cache=model.new_cache(rows, 4))
    rest = [r for r in range(rows) if r not in spoiled]
    assert torch.isfinite(want).all() and torch.isnan(got[spoiled]).all()
    assert torch.equal(got[rest], want[rest]), (got[rest] - want[rest]).abs().amax(1).tolist()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,spoiled", [(16, [0, 9]), (7, [6]), (2, [0]), (40, [3, 38])])
def test_rows_of_nan_scores_beside_others_that_share_their_expert(rows, spoiled, dtype):
    """Whichever experts a row of NaN scores chooses, the pairs of an expert past the first tile of 16 are computed as well."""
    say(f"NaN rows, 64 experts, {rows} rows, {dtype}")
    cfg = config([(latent(), moe(experts=64, top=48, ff=40)), (retention(), moe(experts=64, top=6, ff=64))], vocab=50)
    spoiled_rows_leave_the_others_alone(cfg, rows, spoiled, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("experts,top,rows", [(7, 7, 3), (20, 16, 16), (63, 5, 40), (70, 64, 9), (300, 20, 80)])
def test_rows_of_nan_scores_choose_experts_that_are_there(experts, top, rows, dtype):
    """Fewer experts than lanes (of one, four and sixteen experts each): a row of NaN scores chooses distinct ones of them, in small calls and in
    the larger ones that choose in a launch of their own."""
    say(f"NaN rows, {top} of {experts} experts, {rows} rows, {dtype}")
    cfg = config([(latent(), moe(experts=experts, top=top, ff=16)), (retention(), None)], vocab=50)
    spoiled_rows_leave_the_others_alone(cfg, rows, [1, rows - 1], dtype)


@pytest.mark.parametrize("bad", [math.nan, math.inf])
def test_experts_of_bad_scores(bad):
    """More experts whose scores are no numbers than choices that may avoid them: every logit is NaN, and the next call is as if it had not been."""
    say(f"router rows of {bad}")
    cfg = config([(latent(), moe(experts=20, top=16, ff=16)), (retention(), None)], vocab=50)
    w = weights(cfg, seed=8)
    model = build(cfg, w, torch.bfloat16)
    toks = ids(tokens(cfg, 9))
    want = model.forward(toks, kv_cache=model.new_cache(1, 9)).clone()
    spoiled = dict(w)
    spoiled["l0.mlp.router"] = w["l0.mlp.router"].clone()
    spoiled["l0.mlp.router"][3:15] = bad
    assert torch.isnan(build(cfg, spoiled, torch.bfloat16).forward(toks)).any()
    assert torch.equal(model.forward(toks, kv_cache=model.new_cache(1, 9)), want)


def test_a_slot_is_used_again_without_a_trace():
    say("slots used again")
    model, cfg = case_model("odd", torch.bfloat16), CASES["odd"]
    cache = model.new_cache(1, 120)
    first = model.forward(ids(tokens(cfg, 50)), kv_cache=cache).clone()
    for seed in (5, 6):
        cache.reset()
        model.forward(ids(tokens(cfg, 117, seed=seed)), kv_cache=cache)
        cache.reset()
        assert torch.equal(model.forward(ids(tokens(cfg, 50)), kv_cache=cache), first)


def test_taking_a_step_back():
    say("rewind")
    cfg, model = CASES["odd"], case_model("odd", torch.float32)
    toks = tokens(cfg, 40)
    cache = model.new_cache(1, 64)
    model.forward(ids(toks[:30]), kv_cache=cache)
    for t in toks[30:]:
        mark = cache.mark()
        model.forward_last(ids([(t + 7) % cfg["vocab"]]), kv_cache=cache)
        cache.rewind(1, mark)
        got = model.forward_last(ids([t]), kv_cache=cache)
    check(got, oracle_logits("odd", 40)[-1:], torch.float32, "after ten steps taken back")
    with pytest.raises(AssertionError):
        cache.rewind(2)


def test_chosen_places_and_errors():
    say("forward_at, refused calls")
    cfg, model = CASES["odd"], case_model("odd", torch.float32)
    toks = tokens(cfg, 33)
    every = model.forward(ids(toks))[0]
    assert torch.equal(model.forward_at(ids(toks), [32, 0, 5]), every[[32, 0, 5]])
    cache = model.new_cache(1, 33)
    assert model.forward_at(ids(toks[:20]), [], kv_cache=cache).shape == (0, cfg["vocab"]) and cache.get_pos() == 20
    assert torch.allclose(model.forward_at(ids(toks[20:]), [12], kv_cache=cache), every[32:], rtol=0, atol=1e-4)
    with pytest.raises(AssertionError):
        model.forward(ids([1]), kv_cache=cache)                      # full
    with pytest.raises(IndexError):
        model.forward(ids([1, cfg["vocab"]]))
    with pytest.raises(ValueError):
        Palilix.from_config(cfg, torch.float16)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("end", ["experts", "experts and shared", "dense", "recurrence", "wide"])
def test_rows_that_go_on_alone(end, dtype):
    """Behind the last mixers only the rows with logits go on, up to half of all and from two other rows (experts) or 256 (dense, width 192) on, and of many columns times rows the input matrix is two products
    then; the recurrence's read-out leaves out chunks without one.  The same logits as where all rows go on, cache and states as well, for places in any order, more than
    once, and for none.  (Other kernels: a rounding of one layer.)"""
    say(f"chosen rows, {end}, {dtype}")
    last = {"experts": moe(experts=20, top=3, ff=64), "experts and shared": moe(experts=20, top=3, ff=64, shared=(192, 0.5)), "dense": dense(ff=320), "recurrence": dense(ff=320),
            "wide": dense(ff=4096)}[end]
    first, mixer = retention(heads=1, dim=64, vdim=64, rot_dims=32), retention(heads=2, dim=64, vdim=64, rot_dims=32) if end == "recurrence" else latent()
    cfg = config([(first, dense(ff=64)), (mixer, last)], width=1024 if end == "wide" else 192, vocab=70)
    model = build(cfg, weights(cfg, seed=5), dtype)
    for B, T in ((1, 2), (1, 3), (20, 1), (1, 18), (1, 65), (3, 70), (1, 256), (1, 257), (2, 200)) if end != "wide" else ((1, 120), (2, 540)):
        toks = torch.tensor([tokens(cfg, T, seed=b + 1) for b in range(B)], device=DEV)
        full, some, none = (model.new_cache(B, T + 1) for _ in range(3))
        every = model.forward(toks, kv_cache=full).view(B * T, -1)
        places = [(7 * k) % (B * T) for k in range(max(1, B * T - 257))]
        for chosen in (None, places, [B * T - 1, 0, B * T - 1], list(range(B * T - 1)), list(range(1, B * T, 2))):
            some.reset()
            got = model.forward_last(toks, kv_cache=some) if chosen is None else model.forward_at(toks, chosen, kv_cache=some)
            check(got, every[[b * T + T - 1 for b in range(B)] if chosen is None else chosen].cpu(), dtype, f"{B} x {T}, {'last' if chosen is None else len(chosen)}")
        assert model.forward_at(toks, [], kv_cache=none).shape == (0, 70)
        step = torch.full((B, 1), 3, device=DEV)
        want = model.forward(step, kv_cache=full)
        for cache in (some, none):
            assert torch.equal(model.forward(step, kv_cache=cache), want), (B, T)


def test_chosen_rows_in_a_workspace_for_all_rows(monkeypatch):
    """Room for the logits of all rows is not always room for a gather of half of them: all rows go on then, and nothing is written behind the workspace."""
    say("chosen rows, workspace for all rows")
    cfg = config([(retention(heads=1, dim=64, vdim=64, rot_dims=32), dense(ff=64)), (latent(), moe(experts=20, top=3, ff=64))], width=192, vocab=70)
    model = build(cfg, weights(cfg, seed=5), torch.bfloat16)
    toks = torch.tensor([tokens(cfg, 300)], device=DEV)
    every = model.forward(toks).view(300, -1)
    guard, lib = [], ops._lib.stack_lib()

    def for_all(md, B, T, n_logits, keys):
        room = lib.nc_stack_workspace_bytes(ctypes.byref(md), B, T, B * T, keys)
        assert room < lib.nc_stack_workspace_bytes(ctypes.byref(md), B, T, n_logits, keys)
        t = torch.full((room + 4096,), 77, dtype=torch.uint8, device=DEV)
        off = -t.data_ptr() % 256
        guard.append(t[off + room:])
        return t.data_ptr() + off, room
    monkeypatch.setattr(model, "_workspace", for_all)
    chosen = list(range(1, 300, 2))
    check(model.forward_at(toks, chosen), every[chosen].cpu(), torch.bfloat16, "half of 300")
    assert len(guard) == 1 and bool((guard[0] == 77).all())


# ------------------------------------------------------------------------------------------------ generation
def test_greedy_generation_through_the_engine(tmp_path):
    """A folder on disk, the registry, the Engine's scheduler, the sampler: the ids are the oracle's greedy ids (32-bit)."""
    say("greedy generation")
    cfg = variant("odd", logit_scale=2.5)
    w = weights(cfg, seed=29)
    write_model(tmp_path, cfg, w)
    model, info = load_model(str(tmp_path), dtype=torch.float32)
    assert type(model) is Palilix and info["model_config"] == cfg
    w64 = {k: v.double() for k, v in w.items()}
    prompt, new = tokens(cfg, 37, seed=4), 24
    want = list(prompt)
    for _ in range(new):
        top = ref.forward(cfg, w64, want)[-1].topk(2)
        assert (top.values[0] - top.values[1]).item() > 1e-3           # no close call: the ids must agree
        want.append(top.indices[0].item())
    engine = Engine(model, SyntheticTokenizer())
    for kw in ({}, {"num_samples": 3}, {"prefill_chunk": 2}, {"prefill_chunk": 16, "num_samples": 2}):
        out, masks = engine.generate_batch(prompt, max_tokens=new, temperature=0.0, **kw)
        assert out == [want] * kw.get("num_samples", 1), kw
        assert masks[0] == [0] * len(prompt) + [1] * new
    # bf16, sampled: the stream is reproducible, rows differ
    half, _ = load_model(str(tmp_path))
    runs = [Engine(half, SyntheticTokenizer()).generate_batch(prompt, num_samples=4, max_tokens=12, temperature=1.0, top_k=20, seed=5)[0] for _ in range(2)]
    assert runs[0] == runs[1] and len({tuple(r) for r in runs[0]}) > 1


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_harness_on_a_model_folder(tmp_path, capsys, dtype):
    say(f"infer_bench --model, {dtype}")
    from nanochat_amd import infer_bench
    write_model(tmp_path, CASES["wide"], case_weights("wide"))
    infer_bench.main(["--model", str(tmp_path), "--dtype", dtype, "--prompt-tokens", "40", "--decode-tokens", "6", "--batch-sizes", "1,3"])
    card = json.loads(capsys.readouterr().out.strip().splitlines()[-1])
    assert card["model_config"] == CASES["wide"] and [s["batch_size"] for s in card["sweep"]] == [1, 3]
    assert card["kv_bytes_per_token"] == (512 + 64) * (2 if dtype == "bfloat16" else 4)


class ForcingTokenizer(SyntheticTokenizer):
    """Every sequence meets the tool-use tokens at once: <|python_start|> is whatever the model likes to say, so that the state machine
    forces tokens of its own and the step run ahead is taken back."""

    def __init__(self, start, end, out):
        self.ids = {"<|python_start|>": start, "<|python_end|>": end, "<|output_start|>": out, "<|output_end|>": out + 1, "<|assistant_end|>": 1 << 30}

    def encode_special(self, s):
        return self.ids[s]

    def encode(self, s, prepend=None):
        return [2, 3]

    def decode(self, toks):
        return "1+1"


def test_forced_tokens_take_the_step_back():
    say("forced tokens")
    cfg, model = CASES["odd"], case_model("odd", torch.float32)
    prompt = tokens(cfg, 9, seed=8)
    plain = Engine(model, SyntheticTokenizer()).generate_batch(prompt, max_tokens=10, temperature=0.0)[0][0][9:]
    # the second token opens the tool block, the first later one that differs from both its neighbours in kind closes it
    start = plain[1]
    end = next(t for i, t in enumerate(plain) if i >= 3 and t != start)
    tok = ForcingTokenizer(start, end, 120)
    out, masks = Engine(model, tok).generate_batch(prompt, max_tokens=24, temperature=0.0)
    assert 0 in masks[0][9:], "no token was forced"
    # the same ids, teacher-forced through the oracle: every sampled token is its greedy choice
    w64 = {k: v.double() for k, v in case_weights("odd").items()}
    logits = ref.forward(cfg, w64, out[0])
    for i in range(9, len(out[0])):
        if masks[0][i]:
            assert logits[i - 1].argmax().item() == out[0][i], i


def test_trace_replay(tmp_path):
    """bin/trace_run's own replay loop on two requests, one after the other, with a cache that is handed on."""
    say("trace replay")
    mod = trace_runner()
    cfg, model = CASES["odd"], case_model("odd", torch.float32)
    toks = tokens(cfg, 45)
    want = oracle_logits("odd", 45)
    replay = mod.Replay(model, 45)
    for name in ("a", "b"):
        got = replay.step([{"id": name, "tokens": toks[:20], "want": [0, 19]}], [])
        check(got, want[[0, 19]], torch.float32, name)
        assert replay.step([{"id": name, "tokens": toks[20:22], "want": []}], []).numel() == 0
        got = replay.step([{"id": name, "tokens": toks[22:44], "want": [3]}], [])
        check(got, want[25:26], torch.float32, name)
        got = replay.step([{"id": name, "tokens": toks[44:], "want": [0]}], [name])
        check(got, want[44:], torch.float32, name)
    assert len(replay.free) == 1 and not replay.live
    grown = mod.Replay(model, 10)                      # more tokens than were announced
    grown.step([{"id": "c", "tokens": toks[:10], "want": []}], [])
    check(grown.step([{"id": "c", "tokens": toks[10:45], "want": [34]}], ["c"]), want[44:], torch.float32, "grown")
