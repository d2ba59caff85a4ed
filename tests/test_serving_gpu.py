"""GPU tests of the decode-attention kernel (csrc/decode.hip) and the serving engine
(reference: src/ferrite/serving/engine.py, tests/test_serving.py:11-32).

Pins for the kernel: the reference's own math (engine.py:89-104: write the new
rows, f32 scores over keys <= pos masked with -1e30, softmax, P.V), restated in
torch on the same inputs, at positions on and across the edges of waves' and workgroups' rows;
the caches hold the new rows at pos and nothing else changed; out-of-range
positions write nothing and give NaN; reruns are bitwise equal. For the engine:
greedy tokens equal re-running the full model per step (the reference's own
test), decode logits equal the full forward's, and graph replay equals eager.
"""

import math

import numpy as np
import pytest
import torch

from ferrite.kernels.decode_attention import decode_attention, decode_attention_reference
from ferrite.model.gpt import GPTConfig, forward, init_params
from ferrite.serving.engine import Engine, ServeConfig, decode_step, prefill, reference_greedy
from tests._util import bf16_ulp

pytestmark = pytest.mark.gpu


def _case(dev, b, h, L, d, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    mk = lambda *s: torch.randn(*s, generator=g).to(dev, dtype)
    return mk(b, h, d), mk(b, h, d), mk(b, h, d), mk(b, h, L, d), mk(b, h, L, d)


@pytest.mark.parametrize("b,h,L,d,dtype,pos", [
    (2, 3, 1000, 64, torch.bfloat16, [0, 999]),
    (2, 3, 1000, 64, torch.bfloat16, [255, 256]),
    (3, 2, 600, 128, torch.bfloat16, [511, 1, 300]),
    (1, 2, 256, 128, torch.float32, [100]),       # one workgroup of 16 waves: direct output
    (2, 1, 300, 256, torch.bfloat16, [257, 299]),
    (4, 12, 2048, 64, torch.float32, [2047, 1024, 3, 1500]),
    # 128 heads: 1024-key chunks (the grid within 512 workgroups)
    (4, 32, 4096, 128, torch.bfloat16, [4095, 1023, 1024, 2500]),
    (2, 64, 4096, 64, torch.float32, [0, 4095]),
    # 128 heads over 16384 keys: four 4096-key chunks; positions at chunk and
    # row-step edges (a step of loads covers 32 rows at D = 64)
    (2, 64, 16384, 64, torch.bfloat16, [16383, 4096]),
    (2, 64, 16384, 64, torch.bfloat16, [4095, 8223]),
    # 640 heads: one 1024-key chunk holds all 1000 keys (direct output)
    (4, 160, 1000, 64, torch.float32, [999, 0, 500, 31]),
])
def test_decode_attention_matches_reference(dev, b, h, L, d, dtype, pos):
    q, kn, vn, kc, vc = _case(dev, b, h, L, d, dtype, sum(pos) + L)
    p = torch.tensor(pos, dtype=torch.int32, device=dev)
    kc0, vc0 = kc.clone(), vc.clone()
    kr, vr = kc.clone(), vc.clone()
    ref = decode_attention_reference(q, kn, vn, kr, vr, p)
    out = decode_attention(q, kn, vn, kc, vc, p)
    torch.cuda.synchronize()
    assert torch.equal(kc, kr) and torch.equal(vc, vr)  # the new rows at pos, nothing else
    for i, pi in enumerate(pos):
        kc0[i, :, pi] = kn[i]
        vc0[i, :, pi] = vn[i]
    assert torch.equal(kc, kc0) and torch.equal(vc, vc0)
    # the reference output, in f64 for the tolerance: softmax weights in f32 on both sides
    ref64 = torch.stack([
        (torch.softmax(torch.einsum("hd,hkd->hk", q[i].double(), kr[i, :, : pi + 1].double()) / math.sqrt(d), -1)[..., None]
         * vr[i, :, : pi + 1].double()).sum(1) for i, pi in enumerate(pos)])
    got = out.double()
    if dtype == torch.float32:
        assert float((got - ref64).abs().max()) <= 1e-5
    else:
        r = ref64.cpu().numpy()
        assert np.all(np.abs(got.cpu().numpy() - r) <= bf16_ulp(r.astype(np.float32)) + 1e-5)
        assert float((out.float() - ref.float()).abs().max()) <= 2e-2
    again = decode_attention(q, kn, vn, kc.clone(), vc.clone(), p)
    assert torch.equal(out, again)


def test_decode_attention_out_of_range_position(dev):
    q, kn, vn, kc, vc = _case(dev, 2, 2, 512, 64, torch.bfloat16, 3)
    kc0, vc0 = kc.clone(), vc.clone()
    out = decode_attention(q, kn, vn, kc, vc, torch.tensor([-1, 512], dtype=torch.int32, device=dev))
    torch.cuda.synchronize()
    assert torch.isnan(out.float()).all()
    assert torch.equal(kc, kc0) and torch.equal(vc, vc0)


CFG = GPTConfig(vocab_size=256, seq_len=256, d_model=256, n_head=2, n_layer=2, d_ff=512, dtype=torch.float32)
XLA = dict(attention="xla", norm="xla", linear="xla", loss="xla")


def test_engine_matches_reference_greedy(dev):
    """tests/test_serving.py:11-21 on the HIP kernels, f32: prefill and decode replayed from graphs."""
    params = init_params(0, CFG, device=dev)
    eng = Engine(params, CFG, ServeConfig(batch=2, max_len=256, buckets=(128,)))
    assert eng.n_compiles == 2 and eng._decode.graph is not None
    prompts = [[1, 2, 3, 4, 5, 6, 7, 8, 9, 10], [42, 7, 99]]
    gen, stats = eng.generate(prompts, max_new_tokens=6)
    assert gen.shape == (2, 6) and stats["ttft_ms"] > 0
    for i, p in enumerate(prompts):
        np.testing.assert_array_equal(gen[i], reference_greedy(params, CFG.replace(**XLA), p, 6))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_decode_logits_match_full_forward(dev, dtype):
    """After a prefill, each decode step's logits equal the full model's logits at that position
    (f32: 1e-4; bf16: 3e-2, the bf16 activations of two different operation orders)."""
    cfg = CFG.replace(dtype=dtype, linear="pallas")
    params = init_params(1, cfg, device=dev)
    toks = [5, 17, 200, 3, 9, 77, 31]
    lengths = torch.tensor([4], dtype=torch.int32, device=dev)
    t = torch.tensor([toks[:4] + [0] * 60], device=dev)
    logits, kc, vc = prefill(params, t, lengths, cfg, 256)
    full = forward(params, torch.tensor([toks], device=dev), cfg)
    tol = 1e-4 if dtype == torch.float32 else 3e-2
    assert float((logits[0] - full[0, 3]).abs().max()) <= tol
    for step in range(4, len(toks)):
        lg = decode_step(params, torch.tensor([toks[step]], device=dev),
                         torch.tensor([step], dtype=torch.int32, device=dev), kc, vc, cfg)
        assert float((lg[0] - full[0, step]).abs().max()) <= tol, step


def test_graph_replay_matches_eager_engine(dev):
    """bf16, batch 3, two buckets: the graph-replayed engine and an eager one give the same tokens."""
    cfg = CFG.replace(dtype=torch.bfloat16, linear="pallas", n_head=4)
    params = init_params(2, cfg, device=dev)
    prompts = [[3, 1, 4, 1, 5], [9, 2, 6, 5, 3, 5, 8, 9, 7, 9] * 7, [2, 7]]
    a = Engine(params, cfg, ServeConfig(batch=3, max_len=256, buckets=(32, 128)))
    b = Engine(params, cfg, ServeConfig(batch=3, max_len=256, buckets=(32, 128), graphs=False))
    ga, _ = a.generate(prompts, 12)
    gb, _ = b.generate(prompts, 12)
    np.testing.assert_array_equal(ga, gb)
    ga2, _ = a.generate([p[:3] for p in prompts], 5)  # the small bucket, after the large one
    gb2, _ = b.generate([p[:3] for p in prompts], 5)
    np.testing.assert_array_equal(ga2, gb2)


def test_engines_built_after_dropped_ones(dev):
    """Engines are built, used and dropped in a loop, as the serving benchmark does: a dropped
    engine's graphs must be gone before the next engine captures (no graph may be destroyed
    during a capture), so each new engine still matches the eager one."""
    import gc
    import weakref

    cfg = CFG.replace(dtype=torch.bfloat16, n_head=4)
    params = init_params(3, cfg, device=dev)
    ref = Engine(params, cfg, ServeConfig(batch=2, max_len=128, buckets=(32,), graphs=False))
    want, _ = ref.generate([[1, 2, 3], [4, 5]], 6)
    for batch_kernels in ("pallas", "xla", "pallas"):
        eng = Engine(params, cfg, ServeConfig(batch=2, max_len=128, buckets=(32,), decode_kernels=batch_kernels))
        got, _ = eng.generate([[1, 2, 3], [4, 5]], 6)
        if batch_kernels == "pallas":
            np.testing.assert_array_equal(got, want)
        alive = weakref.ref(eng._decode)
        del eng
        assert alive() is None  # freed without waiting for the cycle collector
    gc.collect()


def test_engine_close_releases_graphs(dev):
    """Explicit lifetime: leaving a ``with Engine(...)`` block destroys every captured graph, and
    an engine built after that captures and serves as before."""
    cfg = CFG.replace(dtype=torch.bfloat16, n_head=4)
    params = init_params(3, cfg, device=dev)
    with Engine(params, cfg, ServeConfig(batch=2, max_len=128, buckets=(32,))) as eng:
        want, _ = eng.generate([[1, 2, 3], [4, 5]], 6)
        decode = eng._decode
        assert decode.graph is not None
    assert decode.graph is None and not eng._prefill
    with Engine(params, cfg, ServeConfig(batch=2, max_len=128, buckets=(32,))) as eng2:
        got, _ = eng2.generate([[1, 2, 3], [4, 5]], 6)
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("b,h,L,d,dtype", [
    (3, 2, 512, 128, torch.bfloat16),   # one workgroup of 16 waves per head
    (2, 3, 513, 128, torch.bfloat16),   # one row more: chunks and a second pass
    (1, 2, 128, 64, torch.bfloat16),    # one workgroup of 4 waves
    (2, 1, 130, 256, torch.float32),
    (24, 22, 300, 64, torch.bfloat16),  # many heads: one workgroup of 4 waves, rows not a power of two
])
def test_decode_attention_reads_a_projection_in_place(dev, b, h, L, d, dtype):
    """q, k and v as thirds of one [B, 3, H, D] projection give bitwise what dense copies do, and both
    match the torch restatement (f32 sums in another order; one bf16 rounding of the output)."""
    g = torch.Generator(device=dev).manual_seed(b * L)
    qkv = torch.randn(b, 3, h, d, device=dev, generator=g).to(dtype)
    pos = torch.randint(0, L, (b,), device=dev, generator=g, dtype=torch.int32)
    pos[0] = L - 1
    caches = [torch.randn(b, h, L, d, device=dev, generator=g).to(dtype) for _ in range(2)]
    outs = []
    for dense in (False, True):
        kc, vc = (c.clone() for c in caches)
        q, k, v = (t.contiguous() if dense else t for t in qkv.unbind(1))
        outs.append((decode_attention(q, k, v, kc, vc, pos), kc, vc))
    assert all(torch.equal(a, c) for a, c in zip(*outs))
    kc, vc = (c.clone() for c in caches)
    ref = decode_attention_reference(*qkv.unbind(1), kc, vc, pos)
    assert torch.equal(kc, outs[0][1]) and torch.equal(vc, outs[0][2])
    bar = 2.0**-7 if dtype == torch.bfloat16 else 1e-5
    assert ((outs[0][0].float() - ref.float()).abs() <= bar * ref.float().abs() + 1e-5).all()


@pytest.mark.parametrize("edt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d", [64, 520])
def test_decode_embedding_and_head(dev, edt, d):
    """The decode step's one-kernel embedding is bitwise the gathers, sum and cast, negative indices
    included, and the few-rows head is the rounded embedding's product to f32 sums."""
    from ferrite import _hip

    g = torch.Generator(device=dev).manual_seed(d)
    tok, pe = (torch.randn(n, d, device=dev, generator=g).to(edt) for n in (300, 70))
    t = torch.tensor([0, 299, -1, 17], device=dev)
    p = torch.tensor([69, 0, 3, -70], dtype=torch.int32, device=dev)
    for dt in (torch.bfloat16, torch.float32):
        assert torch.equal(_hip.native().embed(t, p, tok, pe, dt), (tok[t] + pe[p.long()]).to(dt))
    y = torch.randn(5, d, device=dev, generator=g).bfloat16()
    ref = y.double() @ tok.bfloat16().double().t()
    bound = 2.0**-20 * (y.double().abs() @ tok.bfloat16().double().abs().t())
    assert ((_hip.native().tied_logits(y, tok).double() - ref).abs() <= bound).all()


def test_decode_step_takes_tokens_from_the_cpu(dev):
    """decode_step indexes the tables on the GPU with token ids on the CPU, as torch's indexing does."""
    cfg = CFG.replace(dtype=torch.bfloat16, linear="pallas")
    params = init_params(2, cfg, device=dev)
    kc, vc = (torch.randn(cfg.n_layer, 3, cfg.n_head, 64, cfg.head_dim, device=dev).to(cfg.dtype) for _ in range(2))
    token, pos = torch.tensor([5, 200, 31]), torch.tensor([9, 63, 0], dtype=torch.int32, device=dev)
    want = decode_step(params, token.to(dev), pos, kc.clone(), vc.clone(), cfg)
    got = decode_step(params, token, pos, kc.clone(), vc.clone(), cfg)
    assert torch.equal(got, want)  # the embedding is the same sum, rounded the same


@pytest.mark.parametrize("edt", [torch.float32, torch.bfloat16])
def test_decode_step_of_no_sequences(dev, edt):
    """An empty batch gives logits [0, V], through the few-rows head too."""
    cfg = CFG.replace(dtype=torch.bfloat16, linear="pallas")
    params = init_params(2, cfg, device=dev, param_dtype=edt)
    kc, vc = (torch.zeros(cfg.n_layer, 0, cfg.n_head, 64, cfg.head_dim, device=dev, dtype=cfg.dtype) for _ in range(2))
    token, pos = (torch.zeros(0, dtype=dt, device=dev) for dt in (torch.long, torch.int32))
    logits = decode_step(params, token, pos, kc, vc, cfg)
    assert logits.shape == (0, cfg.vocab_size) and logits.dtype == torch.float32


@pytest.mark.parametrize("L", [129, 256])
@pytest.mark.parametrize("d,dtype", [(256, torch.float32), (256, torch.bfloat16), (64, torch.float32)])
def test_decode_attention_of_a_short_cache_needs_no_workspace(dev, L, d, dtype):
    """The entry point takes caches of up to 256 rows without a workspace, and a longer one that it cuts
    only with one."""
    from ferrite import _hip

    def call(length, q, kn, vn, kc, vc, pos):
        out = torch.full_like(q, float("nan"))
        return out, _hip.lib().ferrite_hip_decode_attention(
            *(t.data_ptr() for t in (q, kn, vn, kc, vc, pos, out)), 2, 3, length, d, _hip.dtype_code(dtype), d**-0.5,
            None, 0, _hip.stream_of(q))

    q, kn, vn, kc, vc = _case(dev, 2, 3, L, d, dtype, L + d)
    pos = torch.tensor([L - 1, 5], dtype=torch.int32, device=dev)
    ref = decode_attention_reference(q, kn, vn, kc.clone(), vc.clone(), pos)
    out, rc = call(L, q, kn, vn, kc, vc, pos)
    _hip.check(rc, "decode")
    bar = 2.0**-7 if dtype == torch.bfloat16 else 1e-5  # two f32 sums, and one rounding to bf16 each
    assert ((out.float() - ref.float()).abs() <= bar * ref.float().abs() + 1e-5).all()
    q, kn, vn, kc, vc = _case(dev, 2, 3, 2000, d, dtype, 1)
    assert call(2000, q, kn, vn, kc, vc, pos)[1] == 1 and "workspace" in _hip.last_error()


def test_decode_attention_sums_of_many_chunks(dev):
    """Float32 over 125 chunks of 128 rows: the second pass's sums keep the error of a few dozen terms. Mean
    relative error over 24 heads, each a call of its own: 2.55e-7 with 63 chunks of 256 rows in one chain,
    3.1e-7 with 125 in one."""
    g = torch.Generator(device=dev).manual_seed(3)
    err = []
    for _ in range(24):
        q, kn, vn = (torch.randn(1, 1, 64, device=dev, generator=g) for _ in range(3))
        kc, vc = (torch.randn(1, 1, 16000, 64, device=dev, generator=g) for _ in range(2))
        out = decode_attention(q, kn, vn, kc, vc, torch.tensor([15999], dtype=torch.int32, device=dev))
        p = torch.softmax((kc.double() * q.double().unsqueeze(2)).sum(-1) / 8, -1)
        ref = (p.unsqueeze(-1) * vc.double()).sum(2)
        err.append(float((out.double() - ref).norm() / ref.norm()))
    assert np.mean(err) <= 2.6e-7, np.mean(err)


@pytest.mark.parametrize("L,d,dtype", [
    (4096, 64, torch.bfloat16), (4097, 64, torch.bfloat16),  # the last in chunks of 128 rows, the first in 256
    (8192, 64, torch.float32), (8193, 64, torch.float32),
    (2500, 256, torch.bfloat16),
])
def test_decode_attention_of_every_chunk_count(dev, L, d, dtype):
    """Positions in each of the first 18 chunks and the last: whole and ragged batches of the second pass, and
    whole caches on both sides of the chunks' rule, against the restatement in float64."""
    pos = [128 * i + (7 * i) % 128 for i in range(18)] + [L - 1, L - 2, 127, 128]
    q, kn, vn, kc, vc = _case(dev, 1, 2, L, d, dtype, L)
    for p in pos:
        k, v = kc.clone(), vc.clone()
        out = decode_attention(q, kn, vn, k, v, torch.tensor([p], dtype=torch.int32, device=dev))
        k, v = (t[0, :, : p + 1].double() for t in (k, v))
        ref = (torch.softmax((k * q[0].double().unsqueeze(1)).sum(-1) * d**-0.5, -1).unsqueeze(-1) * v).sum(1)
        # one rounding to bf16 (half an ulp, 2^-9 of the value); f32 sums as in the cases above
        assert ((out[0].double() - ref).abs() <= (2.0**-8 if dtype == torch.bfloat16 else 0.0) * ref.abs() + 1e-5).all(), p
