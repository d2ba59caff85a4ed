"""CPU tests of the serving engine (reference: tests/test_serving.py:11-36): bucket
selection, and the engine's prefill + cached decode against re-running the full model
each step, on the torch route (graphs off, on the CPU)."""

import numpy as np
import pytest
import torch

from ferrite.model.gpt import GPTConfig, init_params
from ferrite.serving.engine import Engine, ServeConfig, bucket_for, reference_greedy

CFG = GPTConfig(vocab_size=256, seq_len=256, d_model=128, n_head=1, n_layer=2, d_ff=256, dtype=torch.float32)
XLA = dict(attention="xla", norm="xla", linear="xla", loss="xla")


def test_bucket_selection():
    assert bucket_for(1, (64, 128)) == 64 and bucket_for(64, (64, 128)) == 64 and bucket_for(65, (64, 128)) == 128
    with pytest.raises(ValueError):
        bucket_for(129, (64, 128))


def test_engine_matches_reference_greedy_on_cpu():
    cfg = CFG.replace(**XLA)
    params = init_params(0, cfg)
    eng = Engine(params, cfg, ServeConfig(batch=2, max_len=256, buckets=(128,), prefill_kernels="xla",
                                          decode_kernels="xla", graphs=False))
    assert eng.n_compiles == 2  # one prefill bucket + decode
    prompts = [[1, 2, 3, 4, 5, 6, 7, 8, 9, 10], [42, 7, 99]]
    gen, stats = eng.generate(prompts, max_new_tokens=6)
    assert gen.shape == (2, 6) and stats["ttft_ms"] > 0
    for i, p in enumerate(prompts):
        np.testing.assert_array_equal(gen[i], reference_greedy(params, cfg, p, 6))


def test_engine_validation():
    params = init_params(0, CFG.replace(**XLA))
    with pytest.raises(ValueError):
        Engine(params, CFG.replace(**XLA), ServeConfig(max_len=512, graphs=False))
    eng = Engine(params, CFG.replace(**XLA), ServeConfig(batch=1, max_len=64, buckets=(32,), prefill_kernels="xla",
                                                         decode_kernels="xla", graphs=False))
    with pytest.raises(ValueError):
        eng.generate([[1] * 30], max_new_tokens=40)
    with pytest.raises(ValueError):
        eng.prefill([[1], [2]])


def test_closed_engine_refuses_to_serve():
    """close() ends an engine's use: prefill, decode and generate raise instead of failing deep
    inside (a missing bucket) or quietly capturing a new graph."""
    cfg = CFG.replace(**XLA)
    params = init_params(0, cfg)
    with Engine(params, cfg, ServeConfig(batch=1, max_len=64, buckets=(32,), prefill_kernels="xla",
                                         decode_kernels="xla", graphs=False)) as eng:
        tok, pos, _, _ = eng.prefill([[1, 2, 3]])
    for call in (lambda: eng.prefill([[1, 2, 3]]), lambda: eng.decode(tok, pos), lambda: eng.generate([[1, 2]], 2)):
        with pytest.raises(RuntimeError, match="engine closed"):
            call()
    eng.close()  # closing again is harmless


def test_capture_window_holds_off_the_cycle_collector():
    """ferrite.graphs.capture_window: no cyclic collection inside a capture, the collector's
    previous state restored afterwards (also when the capture raises)."""
    import gc

    from ferrite.graphs import capture_window

    assert gc.isenabled()
    with capture_window():
        assert not gc.isenabled()
    assert gc.isenabled()
    try:
        with capture_window():
            raise RuntimeError("capture failed")
    except RuntimeError:
        pass
    assert gc.isenabled()
    gc.disable()
    try:
        with capture_window():
            assert not gc.isenabled()
        assert not gc.isenabled()
    finally:
        gc.enable()


def test_one_kernel_embedding_takes_only_alike_tables():
    """The decode step's embedding kernel is kept to what it reads: two tables of one dtype and width,
    a position for each token. Anything else goes through torch's indexing, which is also the result."""
    from ferrite.serving.engine import _embed, _one_kernel_embedding

    f32, bf16 = torch.float32, torch.bfloat16
    tok, pe = torch.randn(9, 16), torch.randn(5, 16)
    t, p = torch.tensor([1, -1, 3]), torch.tensor([0, 4, 2], dtype=torch.int32)
    assert _one_kernel_embedding(tok, pe, t, p, bf16) and _one_kernel_embedding(tok.bfloat16(), pe.bfloat16(), t, p, f32)
    for case in ((tok, pe.bfloat16(), t, p), (tok.bfloat16(), pe, t, p), (tok.half(), pe.half(), t, p),
                 (tok, pe[:, :1], t, p), (tok, pe, t, p[:1]), (tok, pe, t, p[0])):
        assert not _one_kernel_embedding(*case, bf16)
        got = _embed({"tok_emb": case[0], "pos_emb": case[1]}, case[2], case[3], CFG.replace(dtype=bf16), True)
        assert torch.equal(got, (case[0][case[2]] + case[1][case[3].long()]).to(bf16))
    assert not _one_kernel_embedding(tok, pe, t, p, torch.float16)


def test_one_kernel_embedding_leaves_other_devices_to_indexing():
    """Tokens may lie on the CPU beside tables on a GPU: the decode step's embedding kernel does not take
    them, torch's indexing does. (The meta device stands in for the second one.)"""
    from ferrite.serving.engine import _one_kernel_embedding

    tok, pe = torch.randn(9, 16), torch.randn(5, 16)
    t, p = torch.tensor([1, 3]), torch.tensor([0, 4], dtype=torch.int32)
    assert _one_kernel_embedding(tok, pe, t, p, torch.bfloat16)
    for at in range(4):
        case = [tok, pe, t, p]
        case[at] = case[at].to("meta")
        assert not _one_kernel_embedding(*case, torch.bfloat16)


def test_few_rows_head_keeps_to_where_it_is_faster():
    """Every side of the rule's lines, as measured: a float embedding's copy costs more than a bf16 one's."""
    from ferrite.serving.engine import _few_rows_head

    f32, bf16 = torch.float32, torch.bfloat16
    cases = [(8, 1000, 512, f32, True), (32, 8192, 2048, f32, True), (33, 8192, 2048, f32, False),
             (64, 8192, 1024, f32, True), (65, 256, 256, f32, False), (1, 8193, 2048, f32, False),
             (32, 8192, 512, bf16, True), (33, 8192, 512, bf16, False), (8, 1000, 1024, bf16, False),
             (64, 256, 512, bf16, True), (32, 300, 129, bf16, False), (8, 32768, 512, bf16, False), (8, 256, 256, torch.float16, False),
             (8, 256, 960, bf16, True), (4, 1000, 704, bf16, True), (16, 1000, 768, bf16, False), (16, 16384, 904, bf16, True),
             (17, 16384, 904, bf16, False), (32, 2048, 520, bf16, True), (32, 1000, 704, bf16, False), (33, 256, 960, bf16, False),
             (8, 8192, 1224, bf16, False), (8, 256, 1024, bf16, False)]
    for rows, v, d, dtype, takes in cases:
        emb = torch.empty(v, d, dtype=dtype, device="meta")
        assert _few_rows_head(torch.empty(rows, d, dtype=bf16, device="meta"), emb) == takes, (rows, v, d, dtype)
        assert not _few_rows_head(torch.empty(rows, d, dtype=f32, device="meta"), emb)
