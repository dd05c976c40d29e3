"""fp32 sequences take their kernel by their own length (below 97 rows the
phase-by-phase one, where V leaves that more than 16 columns a workgroup): the
bits of a sequence do not depend on what it is batched or packed with, in
batches of few and of many workgroups, packed below, at and above the ranked
count, around the line.  The first of each is also checked against the fp64
recurrence (1e-5 max-norm)."""

import pytest
import torch

from oracle import gdn_oracle as ref

pytestmark = pytest.mark.gpu


def _inputs(B, T, H, K, V, N, seed):
    gen = torch.Generator().manual_seed(seed)
    n = lambda *s: torch.randn(*s, generator=gen)
    return [ref.l2norm(n(B, T, H, K)), ref.l2norm(n(B, T, H, K)), n(B, T, H, V),
            0.1 * torch.nn.functional.logsigmoid(n(B, T, H)), torch.sigmoid(n(B, T, H)), n(N, H, K, V)]


def _check(x, o, fs):
    q, k, v, g, beta, h0 = (t.cpu() for t in x)
    o_ref, h_ref = ref.recurrent(q, k, v, beta, g, ref.to_vk(h0), dtype=torch.float64)
    assert ref.rel_err(o_ref, o.cpu().double()) <= 1e-5
    assert ref.rel_err(ref.to_kv(h_ref), fs.cpu().double()) <= 1e-5


@pytest.mark.parametrize("B,H,K,V", [(3, 2, 64, 32), (9, 40, 64, 64), (5, 60, 128, 128), (4, 100, 128, 48),
                                     (20, 30, 64, 16)])
@pytest.mark.parametrize("T", [1, 33, 96, 97])
def test_f32_dense_equals_alone(pkg, cuda, T, B, H, K, V):
    """Fewer and more workgroups than CUs; K = 128 with 32 columns a workgroup."""
    x = [t.to(cuda) for t in _inputs(B, T, H, K, V, B, seed=T + V)]
    print(f"[f32 routes] B={B} T={T} H={H} K={K} V={V}", flush=True)
    o, fs = pkg.gdn_fwd(*x)
    for i in (0, B - 1):
        so, sf = pkg.gdn_fwd(*(t[i:i + 1] for t in x))
        assert torch.equal(o[i:i + 1], so) and torch.equal(fs[i:i + 1], sf), i
    # two heads alone: a workgroup of 16 columns
    so, sf = pkg.gdn_fwd(*(t[:1, :, :2] for t in x[:5]), x[5][:1, :2])
    assert torch.equal(o[:1, :, :2], so) and torch.equal(fs[:1, :2], sf)
    _check([t[:1, :, :2] for t in x[:5]] + [x[5][:1, :2]], so, sf)


@pytest.mark.parametrize("N", [1, 7, 64, 65, 150])
@pytest.mark.parametrize("H,K,V", [(2, 64, 32), (3, 128, 48), (16, 128, 64)])
def test_f32_packed_equals_separate(pkg, cuda, N, H, K, V):
    lens = [(0, 1, 40, 96, 97, 130, 3, 300)[(5 * i + N) % 8] if i % 9 else 97 for i in range(N)]
    if N == 1:
        lens = [60]
    x = [t.to(cuda) for t in _inputs(1, sum(lens), H, K, V, N, seed=N + V)]
    c = [sum(lens[:i]) for i in range(N + 1)]
    print(f"[f32 routes] packed N={N} H={H} K={K} V={V}", flush=True)
    o, fs = pkg.gdn_fwd(*x, cu_seqlens=torch.tensor(c, device=cuda))
    for i, (a, b) in enumerate(zip(c, c[1:])):
        if a == b:
            assert torch.equal(fs[i], x[5][i])
            continue
        part = [t[:, a:b] for t in x[:5]] + [x[5][i:i + 1]]
        so, sf = pkg.gdn_fwd(*part)
        assert torch.equal(o[:, a:b], so) and torch.equal(fs[i], sf[0]), (i, b - a)
        if i < 5:
            _check(part, so, sf)
