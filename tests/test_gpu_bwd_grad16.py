"""GPU parity of the gradient kernel of the 16-bit backward at the edges of
its tiles: V of one to several blocks of its V steps and odd multiples of 16,
every K, partial chunks, rows that take element accesses, and bf16 slices
whose range shifts lie far apart.

Bounds as in test_gpu_bwd.py: 1e-3 plus one rounding to the storage dtype,
max-norm, against reverse-mode differentiation of the fp64 recurrence.
"""

import pytest
import torch

from oracle import gdn_oracle as ref

pytestmark = pytest.mark.gpu

EPS = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _inputs(T, H, K, V, seed, gate=0.3):
    gen = torch.Generator().manual_seed(seed)
    n = lambda *s: torch.randn(*s, generator=gen)
    q, k = ref.l2norm(n(1, T, H, K)), ref.l2norm(n(1, T, H, K))
    return (q, k, n(1, T, H, V), gate * torch.nn.functional.logsigmoid(n(1, T, H)), torch.sigmoid(n(1, T, H)),
            0.1 * n(1, H, K, V), n(1, T, H, V), n(1, H, K, V))


def _run(pkg, dev, ins):
    d = [t.to(dev) for t in ins]
    got = pkg.gdn_bwd(*d[:5], d[5], d[6], d[7], scale=0.5)
    torch.cuda.synchronize()
    return [t.cpu().double() for t in got]


def _want(ins):
    q, k, v, g, beta, h0, do, dfin = ins
    dq, dk, dv, dbeta, dg, dh0 = ref.recurrent_grads(q, k, v, beta, g, h0, do, dfin, scale=0.5)
    return [dq, dk, dv, dg, dbeta, dh0]


@pytest.mark.parametrize("K,V,T", [(32, 16, 31), (32, 80, 40), (64, 96, 33), (64, 16, 64), (128, 144, 50),
                                   (128, 256, 65), (128, 48, 1), (64, 272, 37)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_grad16_shapes(pkg, cuda, dtype, K, V, T):
    ins = list(_inputs(T, 2, K, V, seed=K + V + T))
    for i in (0, 1, 2, 6):
        ins[i] = ins[i].to(dtype)
    print(f"[grad16] {dtype} K={K} V={V} T={T}", flush=True)
    for name, a, b in zip(("dq", "dk", "dv", "dg", "dbeta", "dh0"), _run(pkg, cuda, ins), _want(ins)):
        assert ref.rel_err(b, a) <= 1e-3 + EPS[dtype], (name, ref.rel_err(b, a))


@pytest.mark.parametrize("spread", [3, 20, 50])
def test_grad16_slices_of_different_range(pkg, cuda, spread):
    """bf16 columns 0-15 of v, h0, dO and d_final_state 2^spread times the
    others, and zero in the first chunk: its dq and dk come from the small
    columns alone and stay within the bound of their own magnitude."""
    K, V, T, C = 64, 64, 96, 32
    ins = list(_inputs(T, 2, K, V, seed=spread))
    ins[3] = ins[3] * 20.0    # the chunks hardly see each other
    for i in (2, 5, 6, 7):
        ins[i][..., :16] *= 2.0 ** spread
    ins[2][:, :C, :, :16] = 0
    ins[6][:, :C, :, :16] = 0
    ins[5][..., :16] = 0
    for i in (0, 1, 2, 6):
        ins[i] = ins[i].to(torch.bfloat16)
    print(f"[grad16] bf16 slices 2^{spread} apart", flush=True)
    got, want = _run(pkg, cuda, ins), _want(ins)
    tol = 1e-3 + EPS[torch.bfloat16]
    for i, name in ((0, "dq"), (1, "dk"), (2, "dv"), (3, "dg"), (4, "dbeta")):
        assert ref.rel_err(want[i], got[i]) <= tol, name
    # the first chunk's rows but its last few, which still see the next
    # chunk's state gradient through the decay
    for i, name in ((0, "dq"), (1, "dk")):
        a, b = got[i][:, :C // 2], want[i][:, :C // 2]
        assert ref.rel_err(b, a) <= tol, (name, ref.rel_err(b, a))
    for j in range(0, V, 16):
        assert ref.rel_err(want[2][..., j:j + 16], got[2][..., j:j + 16]) <= tol, j
