"""The C-ABI library loads and exports every function the public header declares (no GPU needed)."""
import ctypes
import os
import re
from concurrent.futures import ThreadPoolExecutor

import pytest
import torch

from nanochat_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_functions():
    text = open(os.path.join(ROOT, "include", "nanochat_amd.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(nc_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    names = declared_functions()
    assert len(names) >= 16
    lib = ctypes.CDLL(_lib.LIB_PATH)
    for n in names:
        assert hasattr(lib, n), f"{n} is declared in include/nanochat_amd.h but not exported"
    assert sorted(_lib.EXPORTS) == names


def test_binding_and_error_channel():
    lib = _lib.lib()
    assert lib.nc_abi_version() == 2
    # argument validation happens before any GPU call, so it can be exercised without a device
    rc = lib.nc_fp8_quantize_tensorwise(None, 0, 16, None, None, None, None, 0, None)
    assert rc == -1 and b"null pointer" in lib.nc_last_error()
    rc = lib.nc_fp8_gemm_tn(None, None, None, None, None, 1, None, 0, 0.0, 4, 4, 16, 4, 0, None, 0, None)
    assert rc == -1
    rc = lib.nc_sample(None, 1, 8, 8, 1.0, 0, None, None, None)
    assert rc == -1


def test_struct_layout_matches_header():
    # pointer-sized fields + ints: sizes as a C compiler lays them out on LP64
    assert ctypes.sizeof(_lib.LayerDesc) == 10 * 8 + 2 * 4
    assert ctypes.sizeof(_lib.ModelDesc) == 8 * 4 + 2 * 4 + 11 * 8
    assert ctypes.sizeof(_lib.CacheDesc) == 5 * 8 + 5 * 4 + 4


def test_library_was_built_from_these_sources():
    """A failed rebuild leaves the previous library in place; tests must not pass against a stale one.  The build writes the
    digest of its inputs next to the library."""
    from nanochat_amd import build as nb
    assert os.path.exists(nb.STAMP_PATH), "no build stamp next to the library: run python -m nanochat_amd.build"
    assert open(nb.STAMP_PATH).read().strip() == nb.sources_digest(), \
        "nanochat_amd/libnanochat_amd.so was built from other sources than the tree holds: run python -m nanochat_amd.build"


def test_hot_kernels_use_no_scratch_memory():
    """The streaming kernels keep their state in registers: a private-memory spill costs the decode attention 15 %.
    Compiles the sources that hold them with the resource-usage remarks on and reads the figures."""
    import subprocess
    from nanochat_amd import build as nb
    # bytes of scratch per lane allowed: the persistent GEMM keeps a few tile-level addresses there (outside its K loop); the
    # attention variants with 4 or 8 query heads per kv head reserve 20 bytes for a spilled scalar register's lane store and
    # touch them with no instruction
    hot = {"nc_attention.hip": {"attn_partial_kernel": 32},
           "nc_gemm_decode.hip": {"gemm_decode_kernel": 0, "finish_partials_kernel": 0},
           "nc_step.hip": {"step_kernel": 0},
           "nc_elementwise.hip": {"mix_norm_vec_kernel": 0, "kv_prefill_copy_kernel": 0, "qkv_rope_append_kernel": 0},
           "nc_gemm.hip": {"gemm_dl_kernel": 0, "gemm_dlp_kernel": 64},
           "nc_attention_prefill.hip": {"attn_prefill_kernel": 0},
           "nc_quantize.hip": {"amax_kernel": 0, "convert_kernel": 0, "transpose_u8_kernel": 0},
           "nc_sample.hip": {"sample_kernel": 0},
           "nc_stack_gemm.hip": {"linear_few_kernel": 0, "linear_tiled_kernel": 0},
           "nc_latent_attention.hip": {"latent_mfma_kernel": 0, "latent_expanded_kernel": 0, "latent_combine_kernel": 0, "latent_append_kernel": 0},
           "nc_stack_rows.hip": {"stack_row_add_kernel": 0, "route_sort_kernel": 0},
           "nc_window_attention.hip": {"window_few_kernel": 0, "window_prefill_kernel": 0, "window_combine_kernel": 0, "window_append_kernel": 0},
           "nc_selective_scan.hip": {"scan_kernel": 0, "scan_step_kernel": 0, "scan_chunks_kernel": 0, "scan_conv_kernel": 0}}

    def compile_remarks(src):
        cmd = ["hipcc", *nb.FLAGS, "-Rpass-analysis=kernel-resource-usage", "-c", os.path.join(nb.CSRC, src), "-o", os.devnull]
        return subprocess.run(cmd, capture_output=True, text=True)
    with ThreadPoolExecutor(max_workers=6) as ex:
        remarks = dict(zip(hot, ex.map(compile_remarks, hot)))
    for src, kernels in hot.items():
        r = remarks[src]
        assert r.returncode == 0, r.stderr[-2000:]
        name, seen = None, set()
        for line in r.stderr.splitlines():
            m = re.search(r"Function Name: (\S+)", line)
            if m:
                name = m.group(1)
            m = re.search(r"ScratchSize \[bytes/lane\]: (\d+)", line)
            if m and name:
                for k in kernels:
                    if k in name:
                        seen.add(k)
                        assert int(m.group(1)) <= kernels[k], f"{name} in {src} uses {m.group(1)} bytes of scratch per lane"
        assert seen == set(kernels), f"{src}: kernels not found in the compiler's report: {set(kernels) - seen}"


def test_prompt_rows_that_go_a_wave_to_a_row_bring_no_partial_sums():
    """The narrow projections of a prompt leave partial sums up to the row count at which the row pass of bf16 rows changes its form (models up to 768
    wide; the sums are the only part of the workspace that a further row makes smaller)."""
    def room(heads, rows):
        m = _lib.ModelDesc(n_layer=2, n_head=heads, n_kv_head=heads, n_embd=128 * heads, vocab_size=512)
        return _lib.lib().nc_gpt_workspace_bytes(ctypes.byref(m), 1, rows)
    for heads, line in ((2, 768), (3, 768), (4, 768), (5, 1024), (6, 1024)):
        shares = 4 * (line - 1) * 128 * heads * 2           # two shares at least
        assert room(heads, line - 1) - room(heads, line - 2) < shares / 2
        assert room(heads, line - 1) - room(heads, line) > shares / 2
        assert room(heads, 2 * line) < 2 * room(heads, line) + 4096
    assert room(7, 1024) > room(7, 1023)


def test_which_prompts_read_weights_ahead():
    """Calls whose linears are streams of the weight themselves (up to 64 rows, a step of any batch) read nothing ahead; from 65 to 128 rows those do whose
    layer comes while its attention runs."""
    def ahead(heads, B, T):
        m = _lib.ModelDesc(n_layer=2 * heads, n_head=heads, n_kv_head=heads, n_embd=128 * heads, vocab_size=32768)
        return _lib.lib().nc_gpt_reads_ahead(ctypes.byref(m), B, T)
    assert not any(ahead(13, B, T) for B, T in [(1, 16), (1, 64), (4, 16), (1, 65), (4, 20), (1, 128), (500, 1), (200, 2), (10, 15)])
    assert all(ahead(13, B, T) for B, T in [(1, 129), (9, 16), (1, 1792), (8, 1024)])
    assert [ahead(10, 1, T) for T in (16, 64, 65, 128, 129)] == [0, 0, 1, 1, 1]


def test_a_launch_that_meets_has_a_word_for_every_workgroup():
    """The words' size follows from the most workgroups that may meet, and no shape is let in that has one more (257 tiles of 256 x 256)."""
    lib = _lib.lib()
    assert lib.nc_fp8_meeting_bytes() == 4 * (256 + 256 // 32)
    assert [lib.nc_fp8_gemm_relu2_e4m3_fits(M, 4096, 512) for M in (4096, 4097)] == [1, 0]


def _step_descriptors():
    """A step of one row, three layers of width 256, complete and nowhere in memory: its host checks look at no device."""
    at = 1 << 20
    layers = (_lib.LayerDesc * 3)()
    for ly in layers:
        for name, kind in _lib.LayerDesc._fields_:
            setattr(ly, name, -1 if name == "window_left" else 0 if name == "reserved" else at)
    model = _lib.ModelDesc(n_layer=3, n_head=2, n_kv_head=2, n_embd=256, vocab_size=512, padded_vocab=512, rope_len=64, softcap=15.0)
    for name, kind in _lib.ModelDesc._fields_:
        if kind is ctypes.c_void_p:
            setattr(model, name, at)
    model.layers = ctypes.cast(layers, type(model.layers))
    cache = _lib.CacheDesc(k_cache=at, v_cache=at, cache_seqlens=at, prev_out=at, batch=1, max_seq_len=64)
    return model, layers, cache


@pytest.mark.skipif(torch.cuda.is_available(), reason="descriptors of no memory: a check that is missing would reach a launch")
@pytest.mark.parametrize("what, field, value, message", [
    ("layer", "w_qkv", None, b"no FP8 weights"), ("layer", "inv_attn_proj", None, b"no weight scales"), ("layer", "inv_fc", None, b"no weight scales"),
    ("layer", "inv_mlp_proj", None, b"no weight scales"), ("layer", "ve_gate_w", None, b"gate weights"),
    *[("layer", w, (1 << 20) + 8, b"16-byte aligned") for w in ("w_qkv", "w_attn_proj", "w_fc", "w_mlp_proj")],
    ("model", "cos", None, b"rotary"), ("model", "sin", None, b"rotary"), ("model", "rope_len", 0, b"rotary"), ("model", "resid_lambdas", None, b"lambdas"),
    ("model", "x0_lambdas", None, b"lambdas"), ("cache", "max_seq_len", 0, b"cache of 0 tokens")])
def test_a_step_in_one_launch_refuses_what_the_separate_launches_refuse(what, field, value, message):
    """The last layer's pointers, the tables and the cache's length are looked at before anything is launched."""
    lib = _lib.lib()
    model, layers, cache = _step_descriptors()
    room = lib.nc_gpt_workspace_bytes(ctypes.byref(model), 1, 1)
    setattr({"layer": layers[2], "model": model, "cache": cache}[what], field, value)
    assert lib.nc_gpt_forward(ctypes.byref(model), ctypes.byref(cache), 1 << 20, 1, 1, 1 << 20, 1, 1 << 20, room, None) == -1
    assert message in lib.nc_last_error()


@pytest.mark.skipif(torch.cuda.is_available(), reason="descriptors of no memory")
def test_a_model_without_backout_takes_the_separate_launches():
    """They leave the subtraction out; the one launch reads its factor."""
    lib = _lib.lib()
    model, _, cache = _step_descriptors()
    model.backout_lambda = None
    room = lib.nc_gpt_workspace_bytes(ctypes.byref(model), 1, 1)
    assert lib.nc_gpt_forward_present(ctypes.byref(model), ctypes.byref(cache), 1 << 20, 1, 1 << 20, 1 << 20, room, 1, None) == -1
    assert b"not a step that one launch takes" in lib.nc_last_error()


def test_how_long_a_step_in_one_launch_waits_for_its_workgroups():
    """The smaller the team it would begin with, the longer, as a round of tiles more costs by the model's weights; a bound of some 8 ms; not longer for half of them."""
    def polls(heads, layers, registered, B=1, keys=64, windows=(-1,)):
        each = (_lib.LayerDesc * layers)(*[_lib.LayerDesc(window_left=windows[i % len(windows)]) for i in range(layers)])
        m = _lib.ModelDesc(n_layer=layers, n_head=heads, n_kv_head=heads, n_embd=128 * heads, vocab_size=512, layers=each)
        return _lib.lib().nc_gpt_step_list_polls(ctypes.byref(m), B, keys, registered)
    for heads, layers, wgs in ((2, 4, 128), (5, 10, 128), (8, 16, 128), (10, 20, 256), (13, 26, 256)):
        waits = [polls(heads, layers, n) for n in range(1, wgs + 1)]
        assert waits == sorted(waits, reverse=True) and set(waits[wgs // 2 - 1:]) == {64} and waits[0] <= 64 + (1 << 14)
        assert waits[wgs // 4 - 1] - 64 == 2 * (waits[wgs // 3] - 64) > 0           # four rounds and three
    assert polls(13, 26, 32) > 2 * polls(5, 10, 32) > 2 * polls(2, 4, 32)
    assert polls(13, 26, 8) > 1 << 13 and polls(2, 4, 8) < 256
    assert polls(13, 26, 8, B=9) == 0
    # 100 are most of 128, and few of 256: as many are wanted of narrow models with many keys, in the mean of their layers
    for heads, layers, B, line in ((2, 4, 8, 6144), (6, 12, 8, 2048), (8, 16, 1, 12288)):
        assert [polls(heads, layers, 100, B, keys) > 64 for keys in (1, line - 1, line, 4 * line)] == [False, False, True, True]
        assert [polls(heads, layers, 100, B, 4 * line, (0, w)) > 64 for w in (line, 2 * line - 1, 2 * line, -1)] == [False, False, True, True]
