"""Host-side logic of the library checked on the CPU with g++: the C ABI's device resolution
(csrc/device_select.h) and the attention kernels' schedules (csrc/attn_sched.h).

Device resolution.

An entry point works on its stream's device, not on the calling thread's current
device: the CU count that shapes a grid, a kernel's LDS limit and the address of
the allocation-free entry's scratch array are all looked up for the device the
stream belongs to, and per-device one-time set-up runs once under std::call_once
(an XLA FFI handler may be called from several threads with any device current).
The host-side logic is
compiled with g++ against stand-in lookups and run here; on the GPU the same code
runs with hipStreamGetDevice / hipGetDevice behind it.
"""

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_device_select_host_logic(tmp_path):
    exe = tmp_path / "device_select_test"
    src = os.path.join(HERE, "cpp", "device_select_test.cpp")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", src, "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stderr
    assert "all checks passed" in out.stdout


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_attention_schedules(tmp_path):
    """The CPU replay of every attention launcher's schedule (tests/cpp/attn_schedule_test.cpp):
    grid orders, the split kernels' shares, ring loads, waits and reads from the kernels' own
    schedule header, over lengths 64..4096 (and 8192) and several head counts: every output row
    written once, every ring read served by a completed load of the right tile, no region refilled
    under a reader; and every planted schedule mistake caught."""
    exe = tmp_path / "attn_schedule_test"
    src = os.path.join(HERE, "cpp", "attn_schedule_test.cpp")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", src, "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr[-4000:]
    assert "all checks passed" in out.stdout


def test_internal_entry_points_match_their_header():
    """_hip.INTERNAL binds exactly what csrc/internal_api.h declares, and none of it is in the C ABI."""
    import os
    import re

    from ferrite import _hip
    from tests.conftest import ROOT

    text = open(os.path.join(ROOT, "ferrite-tpu_amd", "csrc", "internal_api.h")).read()
    declared = set(re.findall(r"^(?:int|int64_t) (ferrite_internal_\w+)\(", text, re.M))
    assert declared == set(_hip.INTERNAL) and not declared & set(_hip.SIGNATURES)


def _on_gpu(*shape, dtype=None):
    """What the rules ask of a tensor on a GPU."""
    from types import SimpleNamespace

    import torch

    return SimpleNamespace(shape=shape, ndim=len(shape), dtype=dtype or torch.float32, device="cuda:0", is_cuda=True,
                           numel=lambda: int(torch.Size(shape).numel()))


def test_embedding_rules_stay_within_a_launch():
    """A block of 256 threads per token and position, and under 2^32 threads along a grid's x: the rules
    leave more to torch's indexing, and the entry points refuse it before a launch."""
    import torch

    from ferrite import _hip
    from ferrite.model import gpt
    from ferrite.serving import engine

    tensor, i64, bf16, most = _on_gpu, torch.int64, torch.bfloat16, (1 << 24) - 1
    for n, takes in ((most, True), (most + 1, False)):
        assert gpt._one_kernel_embedding(tensor(256, 8), tensor(4, 8), tensor(n, 1, dtype=i64), bf16) == takes
        assert gpt._one_kernel_embedding(tensor(256, 8), tensor(n, 8), tensor(3, 4, dtype=i64), bf16) == takes
        assert engine._one_kernel_embedding(tensor(256, 8), tensor(4, 8), tensor(n, dtype=i64), tensor(n, dtype=i64),
                                            bf16) == takes
        assert _hip.lib().ferrite_internal_embed(None, None, None, None, None, n, 8, 256, 4, 4, 0, 0, None) == 1
        assert ("null" if takes else "sizes") in _hip.last_error()
        assert (_hip.lib().ferrite_internal_embed_bwd_workspace(12, 4, 8, 256, n) > 0) == takes


def test_training_embedding_keeps_to_where_it_is_faster():
    """Every side of the rule's lines: vocabularies past 512 tokens with wide rows stay with torch's sorted sums."""
    import torch

    from ferrite.model import gpt

    for tokens, dim, vocab, takes in [(16384, 512, 1000, True), (16384, 513, 1000, False), (16384, 513, 512, True),
                                      (8192, 1024, 1024, True), (2048, 2048, 1024, True), (4096, 2048, 1024, False), (131072, 256, 1024, True),
                                      (131072, 4096, 512, True), (4, 64, 1025, False)]:
        got = gpt._one_kernel_embedding(_on_gpu(vocab, dim), _on_gpu(8, dim), _on_gpu(tokens // 4, 4, dtype=torch.int64),
                                        torch.bfloat16)
        assert got == takes, (tokens, dim, vocab)
