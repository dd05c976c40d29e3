"""GPU test of the 16-bit backward's 32-column walks, which dense batches of
many heads take: a batch past that rule's line against its sequences run in
parts below the line (16 columns a workgroup).  Both sum in the same order,
so the results are bit-equal; the first sequence is also checked against
reverse-mode differentiation of the fp64 recurrence, with the bound of
test_gpu_bwd.py (1e-3 plus one rounding to the storage dtype, max-norm).
"""

import pytest
import torch

from oracle import gdn_oracle as ref

pytestmark = pytest.mark.gpu

EPS = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
NAMES = ("dq", "dk", "dv", "dg", "dbeta", "dh0")


# workgroups of 16 and of 32 columns that run at once on 256 CUs
ROUND = {128: (512, 512), 64: (768, 512), 32: (1024, 768)}


def _wide(B, H, K, V):
    """The launcher's rule: 32 columns where they take fewer rounds."""
    units, (n16, n32) = B * H * (V // 16), ROUND[K]
    return V % 32 == 0 and -(-units // n32) < -(-2 * units // n16)


# 2 B H V / 16 workgroups of 16 columns: over 512 at K = 128, 768 at 64, 1024 at 32
@pytest.mark.parametrize("B,T,H,K,V", [(3, 1, 45, 128, 32), (3, 33, 16, 128, 96), (3, 95, 12, 128, 128),
                                       (3, 64, 17, 64, 128), (3, 70, 90, 32, 32)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("spread", [0, 14])
def test_wide_walks(pkg, cuda, dtype, B, T, H, K, V, spread):
    assert _wide(B, H, K, V) and not _wide(1, H, K, V)
    gen = torch.Generator().manual_seed(T + K + V)
    n = lambda *s: torch.randn(*s, generator=gen)
    q, k = ref.l2norm(n(B, T, H, K)), ref.l2norm(n(B, T, H, K))
    v, g, beta = n(B, T, H, V), 0.3 * torch.nn.functional.logsigmoid(n(B, T, H)), torch.sigmoid(n(B, T, H))
    h0, do, dfs = 0.1 * n(B, H, K, V), n(B, T, H, V), n(B, H, K, V)
    if dtype == torch.bfloat16:
        # the two 16-column blocks of a workgroup in different ranges
        for x in (v, h0, do, dfs):
            x[..., 16:32] *= 2.0 ** -spread
    q, k, v, do = (x.to(dtype) for x in (q, k, v, do))
    ins = (q, k, v, g, beta, h0, do, dfs)
    d = [x.to(cuda) for x in ins]
    print(f"[wide] {dtype} B={B} T={T} H={H} K={K} V={V}", flush=True)
    got = pkg.gdn_bwd(*d, scale=0.5)
    parts = [pkg.gdn_bwd(*[x[i:i + 1] for x in d], scale=0.5) for i in range(B)]
    torch.cuda.synchronize()
    for i, name in enumerate(NAMES):
        assert torch.equal(got[i], torch.cat([p[i] for p in parts])), name
    dq, dk, dv, dbeta, dg, dh0 = ref.recurrent_grads(*[x[:1, :, :2] for x in (q, k, v, beta, g)], h0[:1, :2],
                                                     do[:1, :, :2], dfs[:1, :2], scale=0.5)
    for i, (name, want) in enumerate(zip(NAMES, (dq, dk, dv, dg, dbeta, dh0))):
        a = got[i][:1, :2] if name == "dh0" else got[i][:1, :, :2]
        err = ref.rel_err(want, a.cpu().double())
        assert err <= 1e-3 + EPS[dtype], (name, err)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,T,H,K,V", [(3, 70, 12, 128, 128), (3, 40, 17, 64, 128)])
def test_wide_walks_do_row_offset(pkg, cuda, dtype, B, T, H, K, V):
    """dO rows that start 4-byte aligned only: the bits of a dense dO."""
    assert _wide(B, H, K, V)
    gen = torch.Generator().manual_seed(K)
    n = lambda *s: torch.randn(*s, generator=gen)
    q, k = ref.l2norm(n(B, T, H, K)).to(dtype), ref.l2norm(n(B, T, H, K)).to(dtype)
    v, g, beta = n(B, T, H, V).to(dtype), 0.3 * torch.nn.functional.logsigmoid(n(B, T, H)), torch.sigmoid(n(B, T, H))
    d = [x.to(cuda) for x in (q, k, v, g, beta, 0.1 * n(B, H, K, V))]
    buf = 1e-3 * n(B, T, H, V + 8).to(dtype).to(cuda)
    do, dfs = buf[..., 2:2 + V], 1e-3 * n(B, H, K, V).to(cuda)
    assert do.data_ptr() % 16 == 4
    print(f"[wide] {dtype} K={K} V={V} dO rows at 4 bytes", flush=True)
    got = pkg.gdn_bwd(*d, do, dfs, scale=0.5)
    want = pkg.gdn_bwd(*d, do.contiguous(), dfs, scale=0.5)
    for name, a, b in zip(NAMES, got, want):
        assert torch.equal(a, b), name
