"""Cached launch plans of the backward: calls of one signature with other
pointers, with and without the state's gradient, misaligned rows after an
aligned call, and offsets of another integer type through autograd."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(cuda, T=70, H=2, K=64, V=32, dtype=torch.float16, seed=0):
    gen = torch.Generator(device=cuda).manual_seed(seed)
    n = lambda *s: torch.randn(*s, generator=gen, device=cuda)
    u = lambda x: (x / x.norm(dim=-1, keepdim=True)).to(dtype)
    return [u(n(1, T, H, K)), u(n(1, T, H, K)), n(1, T, H, V).to(dtype), -0.1 * n(1, T, H).abs(),
            torch.sigmoid(n(1, T, H)), n(1, H, K, V), n(1, T, H, V).to(dtype), n(1, H, K, V)]


def test_bwd_plans(pkg, cuda):
    q, k, v, g, beta, h0, do, dfin = _inputs(cuda)
    one = pkg.gdn_bwd(q, k, v, g, beta, h0, do, dfin)
    other = pkg.gdn_bwd(*_inputs(cuda, seed=1))
    again = pkg.gdn_bwd(q.clone(), k.clone(), v.clone(), g.clone(), beta.clone(), h0.clone(), do.clone(), dfin.clone())
    for a, b, c in zip(one, other, again):
        assert torch.equal(a, c) and not torch.equal(a, b)
    # the optional tensors and options are part of the signature
    none = pkg.gdn_bwd(q, k, v, g, beta, None, do, None, need_dh0=False)
    zero = pkg.gdn_bwd(q, k, v, g, beta, torch.zeros_like(h0), do, torch.zeros_like(dfin))
    assert none[5] is None
    for a, b in zip(none[:5], zero[:5]):
        assert torch.equal(a, b)
    half = pkg.gdn_bwd(q, k, v, g, beta, h0, do, dfin, scale=0.5)
    assert not torch.equal(half[0], one[0])
    # strides and shape of q unchanged, its rows no longer 16-byte aligned
    buf = torch.zeros(q.numel() + 8, dtype=q.dtype, device=cuda)
    with pytest.raises(ValueError, match="16-byte"):
        pkg.gdn_bwd(buf[1:1 + q.numel()].view(q.shape), k, v, g, beta, h0, do, dfin)


@pytest.mark.parametrize("cdtype", [torch.int32, torch.int64])
def test_packed_autograd_offsets(pkg, cuda, cdtype):
    q, k, v, g, beta, _, do, _ = _inputs(cuda, seed=2)
    cu = torch.tensor([0, 3, 40, 70], dtype=cdtype, device=cuda)
    leaves = [t.clone().requires_grad_(True) for t in (q, k, v, g, beta)]
    o, _ = pkg.chunk_gated_delta_rule(*leaves, scale=1.0, cu_seqlens=cu)
    got = torch.autograd.grad(o, leaves, do)
    want = pkg.gdn_bwd(q, k, v, g, beta, None, do, torch.zeros(3, 2, 64, 32, device=cuda), cu_seqlens=cu, need_dh0=False)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_packed_autograd_moved_offsets(pkg, cuda):
    """Saved-tensor hooks that hand the offsets back on the host: refused."""
    q, k, v, g, beta, _, do, _ = _inputs(cuda, seed=3)
    cu = torch.tensor([0, 3, 40, 70], dtype=torch.int64, device=cuda)
    leaves = [t.clone().requires_grad_(True) for t in (q, k, v, g, beta)]
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.cpu() if t.dtype == torch.int64 else t):
        o, _ = pkg.chunk_gated_delta_rule(*leaves, cu_seqlens=cu)
    with pytest.raises(ValueError, match="cu_seqlens must be on"):
        torch.autograd.grad(o, leaves, do)
