"""Packed sequences run longest first (up to 64 of them) and take one record
job per chunk slot: every batch gives the bits of its sequences run one by
one, with empty and equal lengths, below, at and above the ranked count, and
in segments shorter than the longest sequence."""

import random

import pytest
import torch

from oracle import gdn_oracle as ref

pytestmark = pytest.mark.gpu


def _batch(lens, H, K, V, dtype, seed, dev):
    gen = torch.Generator().manual_seed(seed)
    n = lambda *s: torch.randn(*s, generator=gen)
    T, N = sum(lens), len(lens)
    q, k = ref.l2norm(n(1, T, H, K)).to(dtype), ref.l2norm(n(1, T, H, K)).to(dtype)
    g, beta = 0.3 * torch.nn.functional.logsigmoid(n(1, T, H)), torch.sigmoid(n(1, T, H))
    ins = (q, k, n(1, T, H, V).to(dtype), g, beta, 0.1 * n(N, H, K, V), n(1, T, H, V).to(dtype), n(N, H, K, V))
    cu = torch.tensor([sum(lens[:i]) for i in range(N + 1)], dtype=torch.int64)
    return [t.to(dev) for t in ins], cu.to(dev)


@pytest.mark.parametrize("N", [1, 5, 64, 65])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_packed_longest_first_equals_separate_runs(pkg, cuda, dtype, N):
    rng = random.Random(N)
    lens = [rng.choice([0, 1, 31, 32, 33, 64, 70, 70, 129]) for _ in range(N)]
    lens[-1] = 161    # the longest last
    H, K, V = 3, 64, 32
    (q, k, v, g, beta, h0, do, dfin), cu = _batch(lens, H, K, V, dtype, N, cuda)
    print(f"[packed order] {dtype} N={N}", flush=True)
    o, fs = pkg.gdn_fwd(q, k, v, g, beta, h0, cu_seqlens=cu)
    o2, fs2 = pkg.gdn_fwd(q, k, v, g, beta, h0, cu_seqlens=cu, max_segment_chunks=2)
    grads = pkg.gdn_bwd(q, k, v, g, beta, h0, do, dfin, cu_seqlens=cu)
    torch.cuda.synchronize()
    c = cu.tolist()
    for i in range(N):
        a, b = c[i], c[i + 1]
        if a == b:
            assert torch.equal(fs[i], h0[i]) and torch.equal(fs2[i], h0[i])
            continue
        part = [t[:, a:b] for t in (q, k, v, g, beta)]
        so, sf = pkg.gdn_fwd(*part, h0[i:i + 1])
        assert torch.equal(o[:, a:b], so) and torch.equal(fs[i], sf[0]), i
        so, sf = pkg.gdn_fwd(*part, h0[i:i + 1], max_segment_chunks=2)
        assert torch.equal(o2[:, a:b], so) and torch.equal(fs2[i], sf[0]), i
        sg = pkg.gdn_bwd(*part, h0[i:i + 1], do[:, a:b], dfin[i:i + 1])
        for x, y in zip(grads[:5], sg[:5]):
            assert torch.equal(x[:, a:b], y), i
        assert torch.equal(grads[5][i], sg[5][0]), i
