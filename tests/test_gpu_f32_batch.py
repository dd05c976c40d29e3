"""The fp32 forward in batches of 8 chunks: lengths around a row, a chunk and
a batch, both widths of a workgroup, odd V, strided inputs, and the rule that
keeps the phase-by-phase kernel.  Bound: 1e-5 max-norm against the fp64
recurrence (fp32 sums over K and a chunk; the carried state decays)."""

import pytest
import torch

from oracle import gdn_oracle as ref

pytestmark = pytest.mark.gpu


def _inputs(B, T, H, K, V, seed, gate=0.1):
    gen = torch.Generator().manual_seed(seed)
    n = lambda *s: torch.randn(*s, generator=gen)
    return (ref.l2norm(n(B, T, H, K)), ref.l2norm(n(B, T, H, K)), n(B, T, H, V),
            gate * torch.nn.functional.logsigmoid(n(B, T, H)), torch.sigmoid(n(B, T, H)), n(B, H, K, V))


def _check(pkg, dev, ins, **kw):
    q, k, v, g, beta, h0 = ins
    o, fs = pkg.gdn_fwd(*(t.to(dev) for t in (q, k, v, g, beta, h0)), **kw)
    o_ref, h_ref = ref.recurrent(q, k, v, beta, g, ref.to_vk(h0), dtype=torch.float64)
    assert ref.rel_err(o_ref, o.cpu().double()) <= 1e-5
    assert ref.rel_err(ref.to_kv(h_ref), fs.cpu().double()) <= 1e-5


@pytest.mark.parametrize("K", [64, 128])
@pytest.mark.parametrize("T", [1, 31, 32, 33, 255, 256, 257, 300])
def test_f32_batch_lengths(pkg, cuda, T, K):
    print(f"[f32 batch] T={T} K={K}", flush=True)
    _check(pkg, cuda, _inputs(1, T, 2, K, 48, seed=T + K))


@pytest.mark.parametrize("B,T,H,V", [(9, 130, 8, 64), (9, 60, 8, 64), (40, 40, 8, 64), (1, 40, 70, 64), (6, 129, 20, 48)])
def test_f32_batch_widths_and_rule(pkg, cuda, B, T, H, V):
    """32 columns a workgroup, 16 where V is an odd multiple, the phased
    kernel for many short sequences."""
    print(f"[f32 batch] B={B} T={T} H={H} V={V}", flush=True)
    _check(pkg, cuda, _inputs(B, T, H, 64, V, seed=B))


def test_f32_batch_strides(pkg, cuda):
    B, T, H, K, V = 2, 70, 3, 64, 32
    q, k, v, g, beta, h0 = _inputs(B, T, H, K, V, seed=4)
    want = pkg.gdn_fwd(*(t.to(cuda) for t in (q, k, v, g, beta, h0)))
    hf = lambda t: t.to(cuda).transpose(1, 2).contiguous().transpose(1, 2)
    got = pkg.gdn_fwd(hf(q), hf(k), hf(v), g.to(cuda).transpose(0, 1).contiguous().transpose(0, 1), hf(beta),
                      ref.to_vk(h0).contiguous().to(cuda).transpose(2, 3))
    for a, b in zip(want, got):
        assert torch.equal(a, b)
