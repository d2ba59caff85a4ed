"""The training step's embedding and its gradients against the tables' indexing in torch."""

import pytest
import torch

from ferrite import _hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,s,seq,d,vocab", [
    (1, 1, 1, 1, 1),
    (5, 13, 20, 65, 256),  # odd columns, rows not of whole batches, positions past the sequences
    (64, 256, 256, 512, 256),  # the training program's defaults
    (3, 128, 256, 130, 257),
    (9, 100, 100, 48, 1000),
    (2, 64, 64, 264, 1024),
])
@pytest.mark.parametrize("edt,dt", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.bfloat16),
                                    (torch.float32, torch.float32)])
def test_embedding_and_gradients(dev, b, s, seq, d, vocab, edt, dt):
    g = torch.Generator(device=dev).manual_seed(b * s + d)
    tok, pe = (torch.randn(n, d, device=dev, generator=g).to(edt).requires_grad_() for n in (vocab, seq))
    t = torch.randint(-vocab, vocab, (b, s), device=dev, generator=g)
    dh = torch.randn(b, s, d, device=dev, generator=g).to(dt)
    out = _hip.autograd().embed_tokens(t, tok, pe, dt)
    assert torch.equal(out, (tok[t] + pe[:s]).to(dt))
    dtok, dpos = torch.autograd.grad(out, (tok, pe), dh)
    assert dtok.dtype == dpos.dtype == edt
    ref = torch.zeros(vocab, d, dtype=torch.float64, device=dev)
    mag = torch.zeros_like(ref)
    at = (t % vocab).reshape(-1)
    ref.index_add_(0, at, dh.double().view(-1, d))
    mag.index_add_(0, at, dh.double().abs().view(-1, d))
    most = int(torch.bincount(at).max())
    # one rounding of the f32 sum: half a unit in the last of bf16's 8 significant bits, 2^-8 of the value
    ulp = 2.0**-8 if edt == torch.bfloat16 else 0.0
    # f32 sums of n terms in any order: n 2^-24 of the terms' magnitudes
    assert ((dtok.double() - ref).abs() <= (most + 64) * 2.0**-24 * mag + ulp * ref.abs() * 1.01).all()
    ref, mag = dh.double().sum(0), dh.double().abs().sum(0)
    assert ((dpos[:s].double() - ref).abs() <= (b + 4) * 2.0**-24 * mag + ulp * ref.abs() * 1.01).all()
    assert (dpos[s:] == 0).all()
    again = torch.autograd.grad(_hip.autograd().embed_tokens(t, tok, pe, dt), (tok, pe), dh)
    assert torch.equal(again[0], dtok) and torch.equal(again[1], dpos)


def test_a_gradient_that_is_not_finite_stays_in_its_rows(dev):
    tok, pe = torch.zeros(8, 64, device=dev, requires_grad=True), torch.zeros(4, 64, device=dev, requires_grad=True)
    t = torch.tensor([[1, 2, 3, 1], [5, 5, 6, 7]], device=dev)
    dh = torch.ones(2, 4, 64, device=dev)
    dh[0, 1], dh[1, 2, 0] = float("inf"), float("nan")
    dtok, dpos = torch.autograd.grad(_hip.autograd().embed_tokens(t, tok, pe, torch.float32), (tok, pe), dh)
    want = torch.zeros(8, 64, device=dev).index_add_(0, t.view(-1), dh.view(-1, 64))
    assert torch.equal(dtok.nan_to_num(7e5), want.nan_to_num(7e5)) and torch.equal(dpos.nan_to_num(7e5), dh.sum(0).nan_to_num(7e5))
