"""The workloads by which this library's speed is judged: what a program has it do through its
public entry points, from a single short prompt to a training step.

    listed()            the fixed cases
    draw(rng)           one more case from the same ranges
    prepare(case, seed) the inputs, weights and moments a program has in hand before the call
    run(state)          one pass; returns its outputs
    work(case)          bytes and operations one pass cannot do without
    tolerance(case)     how far another correct implementation's outputs may lie
    exact(case, seed)   the same outputs in 64 bits, by plain torch
"""

from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ferrite-tpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from ferrite.kernels.cross_entropy import cross_entropy  # noqa: E402
from ferrite.kernels.decode_attention import decode_attention  # noqa: E402
from ferrite.kernels.flash_attention import BlockSizes, flash_attention  # noqa: E402
from ferrite.kernels.matmul import matmul, mlp_gelu  # noqa: E402
from ferrite.kernels.rmsnorm import rmsnorm  # noqa: E402
from ferrite.model.gpt import GPTConfig, init_params, named_leaves, unflatten  # noqa: E402
from ferrite.model.train import TrainConfig, build_train_step, lr_at  # noqa: E402
from ferrite.serving.engine import decode_step  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
SIZE = {"bf16": 2, "f32": 4}


def listed() -> list[dict]:
    return [
        # A short prompt through one attention layer of the default model: the smallest call, one launch.
        _attention("attn_prefill", 1, 4, 256, 256, 128, "bf16", causal=True, grad=False),
        # Self-attention of a training step: the reference's headline shape, forward and backward.
        _attention("attn_causal", 4, 16, 2048, 2048, 128, "bf16", causal=True, grad=True),
        # Its long-context variant: few heads, long rows, a narrow head.
        _attention("attn_long", 1, 8, 8192, 8192, 64, "bf16", causal=True, grad=True),
        # Attention over another sequence: no mask, unequal and ragged lengths, a padded head dim.
        _attention("attn_cross", 2, 8, 1000, 1408, 80, "bf16", causal=False, grad=True),
        # Training in float32 (`--dtype float32`): true fp32 products.
        _attention("attn_f32", 2, 8, 1024, 1024, 64, "f32", causal=True, grad=True),
        # One decode token per sequence over a long cache, sequences of different lengths.
        {"name": "attn_decode", "kind": "decode", "b": 8, "h": 32, "max_len": 8192, "d": 128, "dtype": "bf16"},
        # A linear layer whose sizes fit no tile, forward and backward.
        {"name": "matmul_ragged", "kind": "matmul", "m": 2100, "k": 1003, "n": 2050, "dtype": "bf16", "grad": True},
        # The transformer MLP of the 12-layer model at batch 8 x 1024, forward and backward.
        {"name": "mlp_train", "kind": "mlp", "t": 8192, "d": 768, "f": 3072},
        # The residual add and norm between its sub-layers, forward and backward.
        {"name": "norm_train", "kind": "norm", "rows": 8192, "dim": 768, "dtype": "bf16", "residual": True, "grad": True},
        # The loss over its vocabulary, forward and backward.
        {"name": "loss_train", "kind": "loss", "n": 8192, "v": 32768},
        # One whole step of the training program at its defaults (batch 64 x 256, byte vocabulary).
        {"name": "train_step", "kind": "train", "layers": 4, "d": 512, "heads": 4, "f": 2048, "vocab": 256, "seq": 256,
         "batch": 64, "linear": "pallas", "params": "f32"},
        # One decode step of the serving benchmark's model for eight users, replayed from a graph as the engine does.
        {"name": "serve_decode", "kind": "serve", "layers": 4, "d": 512, "heads": 4, "f": 2048, "vocab": 256, "seq": 512,
         "batch": 8, "linear": "pallas", "params": "f32"},
    ]


def _attention(name, b, h, sq, sk, d, dtype, causal, grad) -> dict:
    return {"name": name, "kind": "attention", "b": b, "h": h, "sq": sq, "sk": sk, "d": d, "dtype": dtype, "causal": causal,
            "grad": grad}


# ---------------------------------------------------------------- drawn cases


def _log_int(rng, lo: int, hi: int) -> int:
    """An integer of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _size(rng, lo: int, hi: int, step: int) -> int:
    """Like _log_int; half of them multiples of `step`, as most programs' sizes are, the others any number."""
    n = _log_int(rng, lo, hi)
    return n if rng.random() < 0.5 else min(hi // step, max(1, round(n / step))) * step


def draw(rng) -> dict:
    # Matmuls are drawn twice as often: they carry the widest range of shapes and two directions.
    kind = rng.choice(["attention", "attention", "attention", "decode", "matmul", "matmul", "mlp", "norm", "norm", "loss",
                       "train", "serve"])
    return globals()["_draw_" + kind](rng)


def _draw_attention(rng) -> dict:
    while True:
        causal, grad = rng.random() < 0.7, rng.random() < 0.7
        dtype = "bf16" if rng.random() < 0.75 else "f32"
        b, h = _log_int(rng, 1, 16), _log_int(rng, 1, 32)
        d = rng.choice([32, 48, 64, 64, 64, 80, 96, 128, 128, 128, 256])
        sk = 128 * _log_int(rng, 1, 64)
        sq = sk if causal or rng.random() < 0.3 else 8 * _log_int(rng, 1, 512)
        case = _attention("", b, h, sq, sk, d, dtype, causal, grad)
        del case["name"]
        # No more than the headline shape: f32 products run at a sixteenth of bf16's rate.
        if work(case)["flops"] * (16 if dtype == "f32" else 1) <= 1.6e11 * (1.5 if grad else 1):
            return case


def _draw_decode(rng) -> dict:
    while True:
        case = {"kind": "decode", "b": _log_int(rng, 1, 64), "h": _log_int(rng, 1, 32), "max_len": _log_int(rng, 64, 16384),
                "d": rng.choice([64, 128, 128, 256]), "dtype": "bf16" if rng.random() < 0.75 else "f32"}
        if case["b"] * case["h"] * case["max_len"] * case["d"] * SIZE[case["dtype"]] <= 1 << 29:
            return case


def _draw_matmul(rng) -> dict:
    while True:
        dtype, grad = ("bf16" if rng.random() < 0.7 else "f32"), rng.random() < 0.5
        m, k, n = _size(rng, 1, 8192, 128), _size(rng, 32, 8192, 128), _size(rng, 32, 8192, 128)
        if m * k * n * (3 if grad else 1) * (16 if dtype == "f32" else 1) <= 3 * 4096**3:
            return {"kind": "matmul", "m": m, "k": k, "n": n, "dtype": dtype, "grad": grad}


def _draw_mlp(rng) -> dict:
    while True:
        t, d = _size(rng, 64, 16384, 128), 64 * _log_int(rng, 2, 64)
        if t * d * d <= 8192 * 768 * 768 * 4:
            return {"kind": "mlp", "t": t, "d": d, "f": 4 * d}


def _draw_norm(rng) -> dict:
    while True:
        rows, dim = _log_int(rng, 1, 65536), _size(rng, 64, 8192, 128)
        if rows * dim <= 1 << 26:
            return {"kind": "norm", "rows": rows, "dim": dim, "dtype": "bf16" if rng.random() < 0.75 else "f32",
                    "residual": rng.random() < 0.75, "grad": rng.random() < 0.6}


def _draw_loss(rng) -> dict:
    while True:
        n, v = _log_int(rng, 32, 16384), rng.choice([256, 50257, 32768, _log_int(rng, 256, 131072)])
        if n * v <= 1 << 28:
            return {"kind": "loss", "n": n, "v": v}


def _draw_model(rng, d_most) -> dict:
    hd = rng.choice([64, 128])
    heads = rng.randint(2, d_most // hd)
    return {"layers": rng.randint(1, 4), "d": hd * heads, "heads": heads, "f": 4 * hd * heads,
            "vocab": rng.choice([256, 1000, 8192]), "linear": rng.choice(["pallas", "pallas", "xla"]),
            "params": rng.choice(["f32", "bf16"])}


def _draw_train(rng) -> dict:
    m, seq = _draw_model(rng, 512), 128 * rng.choice([1, 2, 3, 4, 8])
    return {"kind": "train", **m, "seq": seq, "batch": _log_int(rng, 1, 16384 // seq)}


def _draw_serve(rng) -> dict:
    m = _draw_model(rng, 1024)
    return {"kind": "serve", **m, "seq": 128 * rng.randint(2, 16), "batch": _log_int(rng, 1, 32)}


# ---------------------------------------------------------------- inputs


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, shape, dtype, scale: float = 1.0, loc: float = 0.0):
    return (loc + scale * torch.randn(shape, generator=g, device="cuda")).to(dtype)


def _uniform(g, shape, dtype):
    return (2 * torch.rand(shape, generator=g, device="cuda") - 1).to(dtype)


def _positions(b: int, max_len: int, seed: int):
    """The cache rows' last indices: sequences filled from a third to all of the cache, in an order of the seed's."""
    fill = [math.ceil(max_len * (1 / 3 + 2 / 3 * (i + 1) / b)) - 1 for i in range(b)]
    order = torch.randperm(b, generator=torch.Generator().manual_seed(seed))
    return torch.tensor(fill, dtype=torch.int32)[order].cuda()


def prepare(case: dict, seed: int) -> dict:
    return {"case": case, **globals()["_prepare_" + case["kind"]](case, seed)}


def _prepare_attention(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    q = _normal(g, (c["b"], c["h"], c["sq"], c["d"]), dt)
    k, v = (_normal(g, (c["b"], c["h"], c["sk"], c["d"]), dt) for _ in range(2))
    do = _normal(g, q.shape, dt)
    if c["grad"]:
        q, k, v = (t.requires_grad_() for t in (q, k, v))
    # Blocks have to divide the lengths: multiples of 8 queries and of 128 keys.
    bq = 128 if c["sq"] % 128 == 0 else 8
    return {"q": q, "k": k, "v": v, "do": do, "blocks": BlockSizes(bq, 128, bq, 128)}


def _prepare_decode(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    q, k, v = (_normal(g, (c["b"], c["h"], c["d"]), dt) for _ in range(3))
    kc, vc = (torch.empty((c["b"], c["h"], c["max_len"], c["d"]), dtype=dt, device="cuda").normal_(generator=g) for _ in range(2))
    return {"q": q, "k": k, "v": v, "kc": kc, "vc": vc, "pos": _positions(c["b"], c["max_len"], seed)}


def _prepare_matmul(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    x, y = _uniform(g, (c["m"], c["k"]), dt), _uniform(g, (c["k"], c["n"]), dt)
    go = _normal(g, (c["m"], c["n"]), dt)
    if c["grad"]:
        x, y = x.requires_grad_(), y.requires_grad_()
    return {"x": x, "y": y, "go": go}


def _prepare_mlp(c, seed):
    g, dt = _gen(seed), torch.bfloat16
    x = _normal(g, (c["t"], c["d"]), dt).requires_grad_()
    w1 = _normal(g, (c["d"], c["f"]), dt, c["d"] ** -0.5).requires_grad_()
    w2 = _normal(g, (c["f"], c["d"]), dt, c["f"] ** -0.5).requires_grad_()
    return {"x": x, "w1": w1, "w2": w2, "go": _normal(g, (c["t"], c["d"]), dt)}


def _prepare_norm(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    x, r, dh, dy = (_normal(g, (c["rows"], c["dim"]), dt) for _ in range(4))
    w = _normal(g, (c["dim"],), dt, 0.1, 1.0)
    if c["grad"]:
        x, r, w = (t.requires_grad_() for t in (x, r, w))
    return {"x": x, "r": r if c["residual"] else None, "w": w, "dh": dh, "dy": dy}


def _prepare_loss(c, seed):
    g = _gen(seed)
    logits = torch.empty((c["n"], c["v"]), device="cuda").normal_(generator=g).mul_(2.0).requires_grad_()
    targets = torch.randint(0, c["v"], (c["n"],), generator=g, device="cuda")
    return {"logits": logits, "targets": targets}


def _gpt(c) -> GPTConfig:
    return GPTConfig(vocab_size=c["vocab"], seq_len=c["seq"], d_model=c["d"], n_head=c["heads"], n_layer=c["layers"],
                     d_ff=c["f"], linear=c["linear"])


def _prepare_train(c, seed):
    """A run under way: moments of the size that clipped gradients leave, step 100 of 200."""
    params = init_params(seed, _gpt(c), device="cuda", param_dtype=DTYPES[c["params"]])
    g = _gen(seed)
    leaves = [t for _, t in named_leaves(params)]
    s = sum(t.numel() for t in leaves) ** -0.5  # a gradient of norm 1, spread evenly
    m = unflatten(params, [_normal(g, t.shape, torch.float32, 0.3 * s) for t in leaves])
    v = unflatten(params, [s * s * (0.5 + torch.rand(t.shape, generator=g, device="cuda")) for t in leaves])
    x = torch.randint(0, c["vocab"], (c["batch"], c["seq"] + 1), generator=g, device="cuda")
    return {"params": params, "opt": {"m": m, "v": v, "step": 99}, "x": x[:, :-1].contiguous(), "y": x[:, 1:].contiguous(),
            "step": build_train_step(_gpt(c), TrainConfig(batch=c["batch"]))}


def _serve_inputs(c, seed):
    cfg, g = _gpt(c), _gen(seed)
    params = init_params(seed, cfg, device="cuda", param_dtype=DTYPES[c["params"]])
    shape = (cfg.n_layer, c["batch"], cfg.n_head, c["seq"], cfg.head_dim)
    kc, vc = (_normal(g, shape, cfg.dtype) for _ in range(2))
    tokens = torch.randint(0, c["vocab"], (c["batch"],), generator=g, device="cuda")
    return {"params": params, "kc": kc, "vc": vc, "tokens": tokens, "pos": _positions(c["batch"], c["seq"], seed)}


def _prepare_serve(c, seed):
    """The weights, a cache that prompts have filled, and the decode step captured once into a graph."""
    s, cfg = _serve_inputs(c, seed), _gpt(c)

    def step():
        return decode_step(s["params"], s["tokens"], s["pos"], s["kc"], s["vc"], cfg)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        logits = step()
    return {**s, "graph": graph, "logits": logits}


# ---------------------------------------------------------------- one pass


def run(state: dict):
    return globals()["_run_" + state["case"]["kind"]](state)


def _run_attention(s):
    out = flash_attention(s["q"], s["k"], s["v"], causal=s["case"]["causal"], block_sizes=s["blocks"])
    if not s["case"]["grad"]:
        return out
    return (out.detach(), *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["do"]))


def _run_decode(s):
    return decode_attention(s["q"], s["k"], s["v"], s["kc"], s["vc"], s["pos"]), s["kc"], s["vc"]


def _run_matmul(s):
    out = matmul(s["x"], s["y"])
    return (out.detach(), *torch.autograd.grad(out, (s["x"], s["y"]), s["go"])) if s["case"]["grad"] else out


def _run_mlp(s):
    out = mlp_gelu(s["x"], s["w1"], s["w2"])
    return (out.detach(), *torch.autograd.grad(out, (s["x"], s["w1"], s["w2"]), s["go"]))


def _run_norm(s):
    x, r, w = s["x"], s["r"], s["w"]
    if r is None:
        y = rmsnorm(x, w)
        return (y.detach(), *torch.autograd.grad(y, (x, w), s["dy"])) if s["case"]["grad"] else y
    h, y = rmsnorm(x, w, residual=r)
    return (h.detach(), y.detach(), *torch.autograd.grad((h, y), (x, r, w), (s["dh"], s["dy"]))) if s["case"]["grad"] else (h, y)


def _run_loss(s):
    loss = cross_entropy(s["logits"], s["targets"])
    return loss.detach(), *torch.autograd.grad(loss, s["logits"])


def _run_train(s):
    params, s["opt"], loss, gnorm = s["step"](s["params"], s["opt"], s["x"], s["y"])
    return {"loss": loss, "gnorm": gnorm, "params": dict(named_leaves(params)), "m": dict(named_leaves(s["opt"]["m"]))}


def _run_serve(s):
    s["graph"].replay()
    return s["logits"], s["kc"], s["vc"]


# ---------------------------------------------------------------- work


def work(case: dict) -> dict:
    return dict(zip(("bytes", "flops"), globals()["_work_" + case["kind"]](case)))


def _work_attention(c):
    flops = 4 * c["b"] * c["h"] * c["sq"] * c["sk"] * c["d"] * (0.5 if c["causal"] else 1.0)
    rows = c["b"] * c["h"] * c["d"] * SIZE[c["dtype"]]
    if c["grad"]:  # q, do, o, dq and k, v, dk, dv
        return rows * 4 * (c["sq"] + c["sk"]), 3.5 * flops
    return rows * 2 * (c["sq"] + c["sk"]), flops


def _filled(b: int, max_len: int) -> int:
    return sum(math.ceil(max_len * (1 / 3 + 2 / 3 * (i + 1) / b)) for i in range(b))


def _work_decode(c):
    rows = c["h"] * _filled(c["b"], c["max_len"])
    return 2 * rows * c["d"] * SIZE[c["dtype"]], 4 * rows * c["d"]


def _work_matmul(c):
    m, k, n, passes = c["m"], c["k"], c["n"], 2 if c["grad"] else 1  # with gradients: x, y, g in and out, dx, dy out
    return (passes * (m * k + k * n + m * n)) * SIZE[c["dtype"]], (3 if c["grad"] else 1) * 2 * m * k * n


def _work_mlp(c):
    t, d, f = c["t"], c["d"], c["f"]  # x, g, w1, w2 in; out, dx, dw1, dw2 out
    return 2 * (4 * t * d + 4 * d * f), 12 * t * d * f


def _work_norm(c):
    streams = (4 if c["residual"] else 2) + ((3 if c["residual"] else 2) if c["grad"] else 0)
    return streams * c["rows"] * c["dim"] * SIZE[c["dtype"]], 0


def _work_loss(c):
    return 8 * c["n"] * c["v"], 0


def _dense(c):
    """Parameters of the layers, and of all."""
    layers = c["layers"] * (4 * c["d"] ** 2 + 2 * c["d"] * c["f"])
    return layers, layers + (c["vocab"] + c["seq"] + 2 * c["layers"] + 1) * c["d"]


def _work_train(c):
    layers, every = _dense(c)
    tokens = c["batch"] * c["seq"]
    flops = 6 * tokens * (layers + c["vocab"] * c["d"]) + 3.5 * 2 * tokens * c["seq"] * c["d"] * c["layers"]
    return every * (2 * SIZE[c["params"]] + 16), flops  # weights and two f32 moments, in and out


def _work_serve(c):
    layers, _ = _dense(c)
    weights = layers + c["vocab"] * c["d"]
    rows = _filled(c["batch"], c["seq"]) * c["layers"]
    return weights * SIZE[c["params"]] + 2 * rows * c["d"] * 2 + c["batch"] * c["vocab"] * 4, 2 * weights * c["batch"] + 4 * rows * c["d"]


# ---------------------------------------------------------------- tolerances


def tolerance(case: dict):
    """About four times the distance of the outputs from `exact` on an MI355X. bf16 (0.0017 to
    0.0031): one rounding of each output, at most 2^-9 of it, and of what lies between two
    products. f32 (3e-7 to 8e-7, the loss's exponentials 1e-7): sums in another order, up to
    8192 terms, and another rounding of the exponentials' arguments."""
    kind, f32 = case["kind"], case.get("dtype") == "f32"
    if kind in ("train", "serve"):  # 0.0045 and 0.0085: roundings to bf16 travel through every layer
        return {"rel": 0.02 if kind == "train" else 0.03, "max": 0.5}
    if f32 or kind == "loss":
        return {"rel": 5e-6, "max": 1e-4}
    return {"rel": 0.012, "max": 0.1}


# ---------------------------------------------------------------- 64 bits


def exact(case: dict, seed: int):
    with torch.no_grad():
        return globals()["_exact_" + case["kind"]](case, seed)


def _exact_attention(c, seed):
    s = _prepare_attention(c, seed)
    scale, out = c["d"] ** -0.5, []
    for b in range(c["b"]):
        for h in range(c["h"]):
            q, k, v, do = (s[n][b, h].detach().double() for n in ("q", "k", "v", "do"))
            p = (q @ k.T).mul_(scale)
            if c["causal"]:
                p.masked_fill_(torch.ones_like(p, dtype=torch.bool).triu_(1), -math.inf)
            p = torch.softmax(p, -1)
            o = p @ v
            if not c["grad"]:
                out.append((o,))
                continue
            ds = (do @ v.T).sub_((do * o).sum(-1, keepdim=True)).mul_(p).mul_(scale)
            out.append((o, ds @ k, ds.T @ q, p.T @ do))
    got = tuple(torch.stack(t).view(c["b"], c["h"], *t[0].shape) for t in zip(*out))
    return got if c["grad"] else got[0]


def _exact_decode(c, seed):
    s = _prepare_decode(c, seed)
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    for b, p in enumerate(s["pos"].tolist()):
        out[b] = _attend_cache(s["q"][b].double(), s["kc"][b, :, :p], s["vc"][b, :, :p], s["k"][b], s["v"][b])
    return out, None, None


def _attend_cache(q, kc, vc, k, v):
    """One query per head [H, D] over the cached rows [H, P, D] and the new one [H, D]."""
    keys = torch.cat([kc.double(), k.double().unsqueeze(1)], 1)
    vals = torch.cat([vc.double(), v.double().unsqueeze(1)], 1)
    p = torch.softmax((keys * q.unsqueeze(1)).sum(-1) * q.shape[-1] ** -0.5, -1)
    return (p.unsqueeze(-1) * vals).sum(1)


def _exact_matmul(c, seed):
    s = _prepare_matmul(c, seed)
    x, y, g = (s[n].detach().double() for n in ("x", "y", "go"))
    return (x @ y, g @ y.T, x.T @ g) if c["grad"] else x @ y


def _gelu(u):
    return 0.5 * u * (1 + torch.tanh(math.sqrt(2 / math.pi) * (u + 0.044715 * u**3)))


def _exact_mlp(c, seed):
    s = _prepare_mlp(c, seed)
    with torch.enable_grad():
        x, w1, w2 = (s[n].detach().double().requires_grad_() for n in ("x", "w1", "w2"))
        out = _gelu(x @ w1) @ w2
        return (out.detach(), *torch.autograd.grad(out, (x, w1, w2), s["go"].double()))


def _rms(h, w, eps=1e-6):
    return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + eps) * w


def _exact_norm(c, seed):
    s = _prepare_norm(c, seed)
    x, w = s["x"].detach().double(), s["w"].detach().double()
    h = x if s["r"] is None else x + s["r"].detach().double()
    y = _rms(h, w)
    if not c["grad"]:
        return y if s["r"] is None else (h, y)
    dy = s["dy"].double()
    inv = torch.rsqrt(h.square().mean(-1, keepdim=True) + 1e-6)
    g = dy * w
    dx = inv * (g - h * inv * (g * h * inv).mean(-1, keepdim=True))
    dw = (dy * h * inv).sum(0)
    if s["r"] is None:
        return y, dx, dw
    dx = dx + s["dh"].double()
    return h, y, dx, dx, dw


def _exact_loss(c, seed):
    s = _prepare_loss(c, seed)
    logits, at = s["logits"].detach().double(), torch.arange(c["n"], device="cuda")
    lse = torch.logsumexp(logits, -1)
    loss = (lse - logits[at, s["targets"]]).mean()
    grad = logits.sub_(lse.unsqueeze(-1)).exp_()
    grad[at, s["targets"]] -= 1
    return loss, grad.div_(c["n"])


def _heads(t, c):
    """[B, S, 3 d] -> q, k, v [B, H, S, hd]."""
    b, s, _ = t.shape
    return t.view(b, s, 3, c["heads"], -1).permute(2, 0, 3, 1, 4)


def _exact_train(c, seed):
    s = _prepare_train(c, seed)
    cfg, step = TrainConfig(batch=c["batch"]), s["opt"]["step"] + 1
    b1, b2, eps = 0.9, 0.95, 1e-8
    leaves = {n: t.detach().double() for n, t in named_leaves(s["params"])}
    with torch.enable_grad():
        p = unflatten(s["params"], [t.requires_grad_() for t in leaves.values()])
        h = p["tok_emb"][s["x"]] + p["pos_emb"][: c["seq"]]
        hidden = torch.ones((c["seq"], c["seq"]), dtype=torch.bool, device="cuda").triu_(1)
        for layer in p["layers"]:
            q, k, v = _heads(_rms(h, layer["ln1"]) @ layer["wqkv"], c)
            w = torch.softmax((q @ k.transpose(-1, -2) * q.shape[-1] ** -0.5).masked_fill(hidden, -math.inf), -1)
            h = h + (w @ v).transpose(1, 2).reshape(h.shape) @ layer["wo"]
            h = h + _gelu(_rms(h, layer["ln2"]) @ layer["w1"]) @ layer["w2"]
        logits = (_rms(h, p["ln_f"]) @ p["tok_emb"].T).view(-1, c["vocab"])
        loss = torch.nn.functional.cross_entropy(logits, s["y"].reshape(-1))
        grads = torch.autograd.grad(loss, list(leaves.values()))
    gnorm = math.sqrt(sum(float(g.square().sum()) for g in grads))
    clip, lr = min(1.0, cfg.clip / (gnorm + 1e-6)), lr_at(step, cfg)
    params, moments = {}, {}
    for (n, t), g, (_, m), (_, v) in zip(leaves.items(), grads, named_leaves(s["opt"]["m"]), named_leaves(s["opt"]["v"])):
        g = g * clip
        m, v = b1 * m.double() + (1 - b1) * g, b2 * v.double() + (1 - b2) * g * g
        decay = cfg.weight_decay if t.ndim >= 2 else 0.0
        params[n] = t.detach() - lr * ((m / (1 - b1**step)) / ((v / (1 - b2**step)).sqrt() + eps) + decay * t.detach())
        moments[n] = m
    return {"loss": loss.detach(), "gnorm": gnorm, "params": params, "m": moments}


def _exact_serve(c, seed):
    s = _serve_inputs(c, seed)
    p = unflatten(s["params"], [t.double() for _, t in named_leaves(s["params"])])
    h, kc, vc = p["tok_emb"][s["tokens"]] + p["pos_emb"][s["pos"].long()], s["kc"].double(), s["vc"].double()
    for i, layer in enumerate(p["layers"]):
        q, k, v = _heads((_rms(h, layer["ln1"]) @ layer["wqkv"]).unsqueeze(1), c).squeeze(3)
        a = torch.empty_like(h)
        for b, at in enumerate(s["pos"].tolist()):
            kc[i, b, :, at], vc[i, b, :, at] = k[b], v[b]
            a[b] = _attend_cache(q[b], kc[i, b, :, :at], vc[i, b, :, :at], k[b], v[b]).reshape(-1)
        h = h + a @ layer["wo"]
        h = h + _gelu(_rms(h, layer["ln2"]) @ layer["w1"]) @ layer["w2"]
    return _rms(h, p["ln_f"]) @ p["tok_emb"].T, kc, vc
