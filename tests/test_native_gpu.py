"""The autograd functions of csrc/native.cpp beyond the kernels' own tests: the linear layer and the
MLP that round their weights, saved-tensor hooks, streams of the backward, and what they refuse."""

import pytest
import torch

from ferrite.kernels.flash_attention import flash_attention
from ferrite.kernels.matmul import linear, matmul, mlp_gelu_rounded
from ferrite.kernels.rmsnorm import rmsnorm

pytestmark = pytest.mark.gpu


def _rand(dev, *shape, seed=0, dtype=torch.bfloat16, scale=1.0):
    g = torch.Generator(device=dev).manual_seed(seed)
    return (scale * torch.randn(shape, generator=g, device=dev)).to(dtype)


@pytest.mark.parametrize("rows", [(1,), (4, 16), (65,), (3, 50)])  # 64 rows read a float weight in place
@pytest.mark.parametrize("wdt", [torch.float32, torch.bfloat16])
def test_linear_rounds_its_weight(dev, rows, wdt):
    """linear(x, w) equals matmul(x, w rounded) bitwise where both run the same kernel's sums, and
    its weight gradient is the unrounded product for a float weight, rounded once otherwise."""
    x, w = _rand(dev, *rows, 128, seed=1).requires_grad_(), _rand(dev, 128, 72, seed=2, dtype=wdt).requires_grad_()
    y = linear(x, w)
    ref = matmul(x.detach().reshape(-1, 128), w.detach().bfloat16()).view(*rows, 72)
    assert y.shape == (*rows, 72) and torch.equal(y, ref)
    g = _rand(dev, *rows, 72, seed=3)
    dx, dw = torch.autograd.grad(y, (x, w), g)
    assert dx.dtype == x.dtype and dw.dtype == wdt and dx.shape == x.shape
    dx64 = g.double() @ w.detach().bfloat16().double().t()
    dw64 = x.detach().reshape(-1, 128).double().t() @ g.reshape(-1, 72).double()
    # sums of 72 and up to 150 f32 products, and one bf16 rounding where the result is bf16
    assert (dx.double() - dx64).abs().max() <= 2.0**-8 * dx64.abs().max()
    assert (dw.double() - dw64).abs().max() <= (1e-5 if wdt == torch.float32 else 2.0**-8) * dw64.abs().max()


@pytest.mark.parametrize("rows", [7, 200])
def test_mlp_rounds_its_weights(dev, rows):
    """Float weights give the outputs and input gradient of their rounded copies."""
    x = _rand(dev, rows, 64, seed=4).requires_grad_()
    w1, w2 = _rand(dev, 64, 256, seed=5, dtype=torch.float32, scale=0.1), _rand(dev, 256, 64, seed=6, dtype=torch.float32, scale=0.1)
    g = _rand(dev, rows, 64, seed=7)
    outs = []
    for a, b in ((w1, w2), (w1.bfloat16(), w2.bfloat16())):
        a, b = a.requires_grad_(), b.requires_grad_()
        y = mlp_gelu_rounded(x, a, b)
        outs.append((y.detach(), *torch.autograd.grad(y, (x, a, b), g)))
    for u, v in zip(*outs):
        assert (u.double() - v.double()).abs().max() <= 2.0**-7 * v.double().abs().max()
    assert outs[0][2].dtype == outs[0][3].dtype == torch.float32


@pytest.mark.parametrize("rows", [1, 64])
def test_few_rows_keep_the_forward_weights(dev, rows):
    """A float weight read in place (no backward recorded) gives the recorded call's output, whose
    backward uses the weights of the forward also after they were updated in place."""
    x = _rand(dev, rows, 128, seed=20).requires_grad_()
    w1 = _rand(dev, 128, 256, seed=21, dtype=torch.float32, scale=0.1).requires_grad_()
    w2 = _rand(dev, 256, 72, seed=22, dtype=torch.float32, scale=0.1).requires_grad_()
    g1, g2 = _rand(dev, rows, 256, seed=23), _rand(dev, rows, 72, seed=24)
    for call, ws, g in ((linear, (w1,), g1), (mlp_gelu_rounded, (w1, w2), g2)):
        want = torch.autograd.grad(call(x, *ws), (x, *ws), g)
        y = call(x, *ws)
        with torch.no_grad():
            # the same f32 sums up to their order, rounded to bf16 (the MLP: twice)
            assert (call(x, *ws).float() - y.float()).abs().max() <= 2.0**-7 * y.float().abs().max()
            keep = [w.clone() for w in ws]
            for w in ws:
                w.mul_(2)
        got = torch.autograd.grad(y, (x, *ws), g)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        with torch.no_grad():
            for w, k in zip(ws, keep):
                w.copy_(k)


def test_hooks_streams_and_views(dev):
    """Saved-tensor hooks see what is saved, a backward runs on its forward's stream, and
    non-contiguous inputs and gradients give what dense ones do."""
    x, w = _rand(dev, 32, 256, seed=8).requires_grad_(), _rand(dev, 256, seed=9).requires_grad_()
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.to(dev)):
        h, y = rmsnorm(x, w, residual=x)
    assert len(packed) == 2
    want = torch.autograd.grad(rmsnorm(x, w, residual=x), (x, w), (torch.ones_like(h), torch.ones_like(y)))
    got = torch.autograd.grad((h, y), (x, w), (torch.ones_like(h), torch.ones_like(y)))
    assert all(torch.equal(a, b) for a, b in zip(got, want))

    qkv = [_rand(dev, 2, 128, 3, 64, seed=10 + i).requires_grad_() for i in range(3)]  # [B, S, H, D]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        o = flash_attention(*(t.transpose(1, 2) for t in qkv), causal=True)
    torch.cuda.current_stream().wait_stream(side)
    got = torch.autograd.grad(o, qkv, torch.ones(1, device=dev, dtype=o.dtype).expand_as(o))
    dense = [t.detach().transpose(1, 2).contiguous().requires_grad_() for t in qkv]
    want = torch.autograd.grad(flash_attention(*dense, causal=True), dense, torch.ones_like(o))
    assert all(torch.equal(a, b.transpose(1, 2)) for a, b in zip(got, want))


def test_refusals(dev):
    x, w = _rand(dev, 4, 8, 64), _rand(dev, 64)
    with pytest.raises(RuntimeError, match="functorch"):
        torch.vmap(lambda a: rmsnorm(a, w))(x)
    with pytest.raises(RuntimeError, match="functorch"):
        torch.func.grad(lambda a: matmul(a, a.t()).float().sum())(x[0])
    with pytest.raises(RuntimeError):
        import torch.autograd.forward_ad as fwd

        with fwd.dual_level():
            linear(fwd.make_dual(x, x), _rand(dev, 64, 64))
    with pytest.raises(ValueError, match="float32 or bfloat16"):
        matmul(x[0].half(), x[0].half().t())
    with pytest.raises(RuntimeError):
        rmsnorm(x[..., :0], w[:0])
