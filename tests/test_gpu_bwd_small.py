"""GPU tests of the 16-bit backward where gradients, rows or inputs are far
smaller than the largest of their sequence: each output's rows stay within the
bound of their own magnitude (2-norm), against reverse-mode differentiation of
the fp64 recurrence."""

import pytest
import torch

from oracle import gdn_oracle as ref

pytestmark = pytest.mark.gpu

# one rounding to the storage dtype
EPS = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
NAMES = ("dq", "dk", "dv", "dg", "dbeta", "dh0")


def _inputs(T, H, K, V, dtype, seed, gate=1.0):
    gen = torch.Generator().manual_seed(seed)
    n = lambda *s: torch.randn(*s, generator=gen)
    return {"q": ref.l2norm(n(1, T, H, K)), "k": ref.l2norm(n(1, T, H, K)), "v": n(1, T, H, V),
            "g": gate * torch.nn.functional.logsigmoid(n(1, T, H)), "beta": torch.sigmoid(n(1, T, H)),
            "h0": 0.1 * n(1, H, K, V), "do": n(1, T, H, V), "dfs": n(1, H, K, V)}


def _grads(pkg, dev, x, dtype, scale):
    x = {n: t.to(dtype) if n in ("q", "k", "v", "do") else t for n, t in x.items()}
    d = {n: t.to(dev) for n, t in x.items()}
    got = pkg.gdn_bwd(d["q"], d["k"], d["v"], d["g"], d["beta"], d["h0"], d["do"], d["dfs"], scale=scale)
    torch.cuda.synchronize()
    dq, dk, dv, dbeta, dg, dh0 = ref.recurrent_grads(x["q"], x["k"], x["v"], x["beta"], x["g"], x["h0"], x["do"],
                                                     x["dfs"], scale=scale)
    return dict(zip(NAMES, (t.cpu().double() for t in got))), dict(zip(NAMES, (dq, dk, dv, dg, dbeta, dh0)))


def _err(got, want, rows=slice(None)):
    """Relative 2-norm error over some rows."""
    a, b = got[:, rows], want[:, rows]
    return ((a - b).norm() / b.norm()).item()


@pytest.mark.parametrize("K,V", [(128, 64), (64, 48), (32, 32)])
def test_small_du(pkg, cuda, K, V):
    """bf16 dO near 2^-14 beside a final state's gradient near 1, a small scale
    and gates that leave each row to itself: du of the first chunk is near
    2^-20 of the walk's unit, and dv = beta T^T du keeps its own precision.
    Bound: one rounding, and 2^-10 for dO's elements below 2^-17 (subnormal in
    fp16) and P (entries near 2^-4 to 2^-25)."""
    dtype = torch.bfloat16
    x = _inputs(96, 2, K, V, dtype, seed=K + V, gate=20.0)
    x["do"] *= 2.0 ** -14
    print(f"[small] du {dtype} K={K} V={V}", flush=True)
    got, want = _grads(pkg, cuda, x, dtype, scale=0.125)
    err = _err(got["dv"], want["dv"], slice(0, 32))
    print(f"  dv {err:.2e}", flush=True)
    assert err <= EPS[dtype] + 2.0 ** -10


@pytest.mark.parametrize("K,V", [(128, 48), (128, 96), (64, 64)])
def test_small_gradients_f16(pkg, cuda, K, V):
    """fp16 gradients near 2^-13 (the walks do not shift fp16): dbeta, an fp32
    output.  Bound: 2^-10, of which the carried state gradient (an fp16 pair to
    2^-25, entries near 2^-14) is half."""
    dtype = torch.float16
    x = _inputs(300, 4, K, V, dtype, seed=5, gate=0.3)
    x["do"] *= 2.0 ** -13
    x["dfs"] *= 2.0 ** -13
    print(f"[small] {dtype} K={K} V={V}", flush=True)
    got, want = _grads(pkg, cuda, x, dtype, scale=0.3)
    err = _err(got["dbeta"], want["dbeta"])
    print(f"  dbeta {err:.2e}", flush=True)
    assert err <= 2.0 ** -10


@pytest.mark.parametrize("K,V", [(128, 128), (64, 128), (128, 48), (32, 80)])
@pytest.mark.parametrize("p", [14, 18, 22])
def test_small_do(pkg, cuda, K, V, p):
    """bf16 dO 2^-p below a final state's gradient near 1, gates near 1 a row:
    dq depends on dO alone and keeps its own precision wherever dO lies in
    the walk's unit (one rounding of each element, 2^-10 for the fp16 states)."""
    dtype = torch.bfloat16
    x = _inputs(96, 2, K, V, dtype, seed=K + V + p, gate=0.3)
    x["do"] *= 2.0 ** -p
    print(f"[small] do 2^-{p} K={K} V={V}", flush=True)
    got, want = _grads(pkg, cuda, x, dtype, scale=0.3)
    err = _err(got["dq"], want["dq"])
    print(f"  dq {err:.2e}", flush=True)
    assert err <= EPS[dtype] + 2.0 ** -10


@pytest.mark.parametrize("K,V", [(128, 128), (64, 128), (32, 64)])
@pytest.mark.parametrize("p", [10, 17, 24])
def test_small_do_rows(pkg, cuda, K, V, p):
    """bf16: most rows of dO 2^-p below every seventh: dq of every row keeps the
    bound of its own magnitude (as above).  Slices of different range, too."""
    dtype = torch.bfloat16
    x = _inputs(70, 2, K, V, dtype, seed=K + V + p, gate=0.3)
    for spread in (0, 3, 9):
        y = dict(x)
        y["do"] = x["do"] * torch.where(torch.arange(70) % 7 == 0, 1.0, 2.0 ** -p).view(1, -1, 1, 1)
        for n in ("v", "h0", "do", "dfs"):
            y[n] = y[n].clone()
            y[n][..., 16:32] *= 2.0 ** (6 + spread)    # out of the range that is left as it is
        print(f"[small] rows 2^-{p} K={K} V={V} spread {spread}", flush=True)
        got, want = _grads(pkg, cuda, y, dtype, scale=0.3)
        a, b = got["dq"], want["dq"]
        err = ((a - b).norm(dim=-1) / b.norm(dim=-1)).max().item()
        print(f"  dq {err:.2e}", flush=True)
        assert err <= EPS[dtype] + 2.0 ** -10


@pytest.mark.parametrize("which,p", [("q", 13), ("k", 20), ("k", 40)])
@pytest.mark.parametrize("K", [128, 64, 32])
def test_small_q_k(pkg, cuda, which, p, K):
    """bf16 q or k near 2^-p in one chunk (what carries from chunk to chunk goes
    through the walks, which take q and k as fp16 holds them, and P to 2^-25): dq
    of small k, dk of small q keep the bound of their own magnitude."""
    dtype = torch.bfloat16
    x = _inputs(30, 2, K, 48, dtype, seed=K + p, gate=0.3)
    x[which] *= 2.0 ** -p
    x["h0"] *= 0.0
    x["dfs"] *= 0.0
    print(f"[small] {which} 2^-{p} K={K}", flush=True)
    got, want = _grads(pkg, cuda, x, dtype, scale=0.3)
    name = "dk" if which == "q" else "dq"
    err = _err(got[name], want[name])
    print(f"  {name} {err:.2e}", flush=True)
    assert err <= EPS[dtype] + 2.0 ** -10


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,V", [(128, 128), (64, 48), (32, 32)])
def test_dbeta_precision(pkg, cuda, dtype, K, V):
    """dbeta, an fp32 output, does not see the chunk states' fp16: 5e-6 (fp32 sums
    of u and z, whose operands are fp16 pairs), with beta down to 2^-9, also
    negative; where beta is zero the products with S take over (2^-10)."""
    x = _inputs(200, 2, K, V, dtype, seed=K + V, gate=0.05)
    x["beta"][:, ::3] *= 2.0 ** -7
    x["beta"][:, 1::5] *= -1.0
    x["beta"][:, 2::9] = 0.0
    print(f"[small] dbeta {dtype} K={K} V={V}", flush=True)
    got, want = _grads(pkg, cuda, x, dtype, scale=0.3)
    zero = x["beta"] == 0
    a, b = got["dbeta"], want["dbeta"]
    err = [((a - b)[m].norm() / b[m].norm()).item() for m in (~zero, zero)]
    print(f"  dbeta {err[0]:.2e} {err[1]:.2e}", flush=True)
    assert err[0] <= 5e-6 and err[1] <= 2.0 ** -10


@pytest.mark.parametrize("T,K,V", [(32, 64, 48), (97, 64, 96), (97, 128, 80)])
def test_small_v_and_gradients_f16(pkg, cuda, T, K, V):
    """fp16 v near 2^-10 and gradients near 2^-16: u and z are far below 1, the
    unit of fp16 inputs; dg and dbeta, fp32 outputs, keep 2^-9 (the carried
    state gradient, an fp16 pair to 2^-25, gives half of that)."""
    dtype = torch.float16
    x = _inputs(T, 4, K, V, dtype, seed=T + V, gate=0.3)
    for n, p in (("v", 10), ("do", 16), ("dfs", 16)):
        x[n] *= 2.0 ** -p
    print(f"[small] fp16 v and gradients T={T} K={K} V={V}", flush=True)
    got, want = _grads(pkg, cuda, x, dtype, scale=0.3)
    for n in ("dg", "dbeta"):
        err = _err(got[n], want[n])
        print(f"  {n} {err:.2e}", flush=True)
        assert err <= 2.0 ** -9, n


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_dbeta_before_a_bad_row(pkg, cuda, dtype, bad):
    """v not finite in one row: dbeta of the chunk's first row, which does not
    see it, is that of finite values."""
    x = _inputs(8, 2, 64, 32, dtype, seed=8)
    want, _ = _grads(pkg, cuda, x, dtype, scale=0.3)
    x["v"][:, 5, :, 3] = bad
    print(f"[small] {dtype} v {bad} in row 5", flush=True)
    d = {n: t.to(dtype).to(cuda) if n in ("q", "k", "v", "do") else t.to(cuda) for n, t in x.items()}
    got = pkg.gdn_bwd(d["q"], d["k"], d["v"], d["g"], d["beta"], d["h0"], d["do"], d["dfs"], scale=0.3)[4].cpu()
    assert torch.isfinite(got[:, 0]).all()
    # by the products with the fp16 chunk state: 2^-10
    assert ((got[:, 0] - want["dbeta"][:, 0]).norm() / want["dbeta"][:, 0].norm()).item() <= 2.0 ** -10
