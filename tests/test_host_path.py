"""The library's host code without a GPU: which kernels a call launches.

tests/host_runtime.cpp links the library and defines the HIP runtime calls it
makes; its commands run entry points over host memory and print the launches.
"""
import os
import subprocess

import pytest
import torch

from llminfer_amd import _lib, ops
from tests.conftest import ROOT


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    """run(command, *args, env={}) -> [(what, [word, ...]), ...]"""
    exe = tmp_path_factory.mktemp("host") / "host_runtime"
    lib = _lib.LIB_PATH
    subprocess.run(["g++", "-std=c++17", "-O1", "-rdynamic", "-D__HIP_PLATFORM_AMD__",
                    f"-I{ROOT}/include", "-I/opt/rocm/include", f"{ROOT}/tests/host_runtime.cpp",
                    str(lib), f"-Wl,-rpath,{lib.parent}", "-Wl,-rpath-link,/opt/rocm/lib",
                    "-o", str(exe)], check=True)

    def run(*args, env=None):
        out = subprocess.run([str(exe), *map(str, args)], check=True, capture_output=True,
                             text=True, timeout=60, env={**os.environ, **(env or {})}).stdout
        return [(line.split()[0], line.split()[1:]) for line in out.splitlines()]
    return run


@pytest.mark.parametrize("place,joint", [
    ("apart", True), ("keys_in_values", False), ("values_in_keys", False),
    ("keys_in_output", False), ("keys_unaligned", False)])
def test_gated_prefill_rows_share_a_launch_only_where_order_does_not_matter(host, place, joint):
    got = dict(host("gated", 40, 24, 16, 4, 256, 64, place))
    assert got["status"] == ["0"]
    rows = got["launches"][:-1]
    if joint:
        assert rows == ["attention_rows"]
    else:  # the keys, the values, the queries
        keys = "norm_rope_rows" if place == "keys_unaligned" else "norm_rope_tile"
        assert rows == [keys, "kv_append_vec", "norm_rope_tile"]


@pytest.mark.parametrize("mxcsr", [0, 0x8040])  # the default, and FTZ + DAZ
def test_logits_are_exact_in_any_float_mode(host, mxcsr):
    """Every fp16 value as a logit, read by a thread that flushes denormals
    (torch.set_flush_denormal(True) sets the same two bits)."""
    got = dict(host("logits", mxcsr))
    assert got["status"] == ["0"] and got["wrong"] == ["0"]


# The kernel of each record's name.
KERNELS = {"kvAppend": "kv_append_vec", "gqaDecodeSplitK": "gqa_decode_split_kernel",
           "gqaDecodeMerge": "gqa_decode_merge_kernel", "gqaPrefillMfma": "gqa_prefill",
           "gqaPrefillGated": "gqa_prefill", "gqaPrefillMerge": "gqa_prefill_merge_kernel",
           "gqaPrefillMergeGated": "gqa_prefill_merge_kernel", "gqaGeneric": "gqa_generic",
           "attentionRows": "attention_rows"}


@pytest.mark.parametrize("T,past,hq,hkv,d", [
    (2, 0, 16, 4, 256), (61, 511, 16, 4, 256), (61, 512, 16, 4, 256), (2, 4000, 16, 4, 128),
    (40, 700, 8, 1, 256), (512, 2000, 8, 8, 128), (2048, 2048, 16, 4, 256), (3, 600, 4, 2, 64)])
@pytest.mark.parametrize("call", ["gqa", "append", "gated"])
def test_records_name_what_is_launched(host, call, T, past, hq, hkv, d):
    if call == "gated":
        got = dict(host("gated", T, past, hq, hkv, d, 32, "apart"))
        if d < 128:
            assert got["status"] != ["0"] and got["names"] == []
            return
    else:
        got = dict(host("gqa", T, past, hq, hkv, d, int(call == "append")))
    assert got["status"] == ["0"]
    assert len(got["names"]) == len(got["launches"])
    for name, kernel in zip(got["names"], got["launches"]):
        assert kernel.startswith(KERNELS[name])


NO_LIMIT = 2 ** 63


@pytest.mark.parametrize("tokens,limit,divided", [
    (61, NO_LIMIT, True), (61, 8 << 20, False), (1, NO_LIMIT, None)])
def test_session_step_runs_undivided_where_the_partials_find_no_room(host, tokens, limit, divided):
    got = dict(host("session", 16411, tokens, limit))
    assert got["status"] == ["0"] and got["past"] == [str(16411 + tokens)]
    if divided is not None:
        merges = [n for n in got["launches"] if "prefill_merge" in n]
        assert len(merges) == divided
        assert got["names"].count("gqaPrefillMerge") == divided
        assert got["names"].count("gqaPrefillMfma") == 1


def test_session_step_without_a_decode_workspace_is_refused(host):
    got = dict(host("session", 16411, 1, 1 << 16))
    assert got["status"] == [str(_lib.WORKSPACE)] and got["launches"] == []
    assert got["past"] == ["16411"]


def test_model_step_runs_undivided_where_the_partials_find_no_room(host):
    past, tokens = 640, 300
    merges = lambda names: sum("refill_merge" in n or "PrefillMerge" in n for n in names)
    full = dict(host("model", past, tokens, NO_LIMIT))
    assert full["status"] == full["run"] == ["0"]
    assert merges(full["launches"]) == merges(full["again"]) == merges(full["names"]) == 1
    partials = _lib.load().llmi_hip_gqa_workspace_bytes(_lib.GqaParams(tokens, 4, 2, 256, past))
    partials = (partials + 255) // 256 * 256
    everything = int(full["scratch"][0])
    for limit in (everything - 1, everything - partials):
        got = dict(host("model", past, tokens, limit))
        assert got["status"] == got["run"] == ["0"]
        assert merges(got["launches"]) == merges(got["again"]) == merges(got["names"]) == 0
        assert int(got["scratch"][0]) == everything - partials
        assert int(got["count"][0]) == len(got["names"]) == len(full["names"]) - 1
        assert [n for n in full["launches"] if "prefill_merge" not in n] == got["launches"]
    short = dict(host("model", past, tokens, everything - partials - 1))
    assert short["status"] == [str(_lib.WORKSPACE)] and short["launches"] == []


def test_prefill_takes_no_workspace_where_torch_has_none(monkeypatch):
    def full(need, device):
        raise torch.cuda.OutOfMemoryError
    calls = []
    lib = _lib.load()
    monkeypatch.setattr(ops, "workspace", full)
    monkeypatch.setattr(ops, "_require", lambda *a: None)  # (host tensors)
    monkeypatch.setattr(ops, "_stream", lambda: None)

    class Recorded:
        llmi_hip_gqa_workspace_bytes = lib.llmi_hip_gqa_workspace_bytes
        llmi_hip_causal_gqa = llmi_hip_kv_append_causal_gqa = llmi_hip_gated_attention = \
            staticmethod(lambda *a: calls.append(a[-3:-1]) or _lib.OK)
    monkeypatch.setattr(_lib, "load", lambda: Recorded)
    monkeypatch.setattr(ops, "kernel_names", lambda *a: ["attention"])
    f16 = lambda *s: torch.zeros(s, dtype=torch.float16)
    cache, w = f16(700, 4, 256), torch.zeros(256)
    for T in (61, 1):
        q, k, qp, out = f16(T, 16, 256), f16(T, 4, 256), f16(T, 16, 512), f16(T, 16, 256)
        for call in (lambda: ops.causal_gqa(q, cache, cache, 600),
                     lambda: ops.kv_append_causal_gqa(q, k, k, cache, cache, 600),
                     lambda: ops.gated_attention(qp, k, k, w, w, cache, cache, 600, 64),
                     lambda: ops.bind_causal_gqa(q, cache, cache, out, 600)(),
                     lambda: ops.bind_kv_append_causal_gqa(q, k, k, cache, cache, out, 600)()):
            if T == 1:
                with pytest.raises(torch.cuda.OutOfMemoryError):
                    call()
            else:
                call()
    assert calls == [(None, 0)] * 5


@pytest.mark.parametrize("T", [20, 61, 500])
@pytest.mark.parametrize("past", [0, 4096])
@pytest.mark.parametrize("forced", ["0", "1"])
def test_prefill_kernel_switch_holds_for_divided_keys_too(host, T, past, forced):
    """LLMI_PREFILL_HALVES at the heads that the key-split kernel takes (four a
    workgroup; a short undivided prefill serves two, by the other kernel)."""
    got = dict(host("gqa", T, past, 16, 4, 256, 0, env={"LLMI_PREFILL_HALVES": forced}))
    assert got["status"] == ["0"] and len(got["launches"]) == (2 if past else 1)
    halves = forced == "1" and (past > 0 or T == 500)
    assert got["launches"][0] == ("gqa_prefill_halves_kernel" if halves else "gqa_prefill_kernel")


@pytest.mark.parametrize("rows,width,wave", [
    (100, 8, 16), (131072, 8, 16), (100000, 32, 16), (100, 40, 8), (100000, 64, 8),
    (16384, 72, 4), (16385, 72, 8), (16384, 256, 4), (100000, 128, 8)])
def test_row_norms_rows_a_wave(host, rows, width, wave):
    got = dict(host("rows", rows, width))
    assert got["status"] == ["0", "0"]
    assert got["launches"] == ["l2_norm_tile", "gated_rms_norm_tile"]
    assert got["grids"] == [str(-(-rows // wave))] * 2


@pytest.mark.parametrize("T,channels,offset,pairs", [
    (1, 8192, 0, False), (2, 8192, 0, False), (6, 8192, 0, False), (7, 8192, 0, True),
    (1024, 2, 0, True), (1024, 8191, 0, False), (1024, 8192, 1, False), (1024, 8192, 2, True)])
def test_convolution_pairs_channels_from_seven_tokens(host, T, channels, offset, pairs):
    got = dict(host("conv", T, channels, offset))
    assert got["status"] == ["0"]
    assert got["launches"] == ["causal_conv_k4_pairs" if pairs else "causal_conv_k4"]
