"""The step-by-step walk of sequences of at most 4 rows: around that length,
dense and inside packed batches, for every state layout and output dtype,
against the fp64 recurrence (the walk is fp32 throughout: 2e-6 on fp32 outputs,
one rounding more on 16-bit ones), and bit-equal between packed and separate
runs."""

import ctypes

import pytest
import torch

from oracle import gdn_oracle as ref

pytestmark = pytest.mark.gpu

EPS = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 0.0}


def _inputs(B, T, H, K, V, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    n = lambda *s: torch.randn(*s, generator=gen)
    return (ref.l2norm(n(B, T, H, K)).to(dtype), ref.l2norm(n(B, T, H, K)).to(dtype), n(B, T, H, V).to(dtype),
            0.3 * torch.nn.functional.logsigmoid(n(B, T, H)), torch.sigmoid(n(B, T, H)), n(B, H, K, V))


@pytest.mark.parametrize("K,V", [(64, 16), (64, 96), (128, 128), (128, 48)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T", [1, 3, 4, 5])
def test_short_rows(pkg, cuda, dtype, T, K, V):
    B, H = 3, 5
    q, k, v, g, beta, h0 = _inputs(B, T, H, K, V, dtype, seed=T + K + V)
    d = lambda t: t.to(cuda)
    args = [d(t) for t in (q, k, v, g, beta)]
    print(f"[short] {dtype} T={T} K={K} V={V}", flush=True)
    o_ref, h_ref = ref.recurrent(q, k, v, beta, g, ref.to_vk(h0), dtype=torch.float64)
    # no step beyond 4 rows is fp32: those take the 16-bit bound
    tol = 2e-6 if T <= 4 else 1e-3
    for odt in (dtype, torch.float32):
        o, fs = pkg.gdn_fwd(*args, d(h0), output_dtype=odt)
        assert ref.rel_err(o_ref, o.cpu().double()) <= tol + EPS[odt]
        assert ref.rel_err(ref.to_kv(h_ref), fs.cpu().double()) <= tol
    # a state laid out [B, H, V, K] and one with no unit stride, zero state
    for h in (d(ref.to_vk(h0).contiguous()).transpose(2, 3), d(torch.stack((h0, h0), -1))[..., 0]):
        o2, fs2 = pkg.gdn_fwd(*args, h, output_dtype=torch.float32)
        assert torch.equal(o2, o) and torch.equal(fs2, fs)
    o3, hk = pkg.gdn_chunk_fwd(*args[:3], args[4], args[3])
    o4, fs4 = pkg.gdn_fwd(*args, torch.zeros_like(d(h0)))
    assert torch.equal(o3, o4) and torch.equal(hk.transpose(2, 3), fs4)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lens", [[1] * 70, [4, 5, 1, 0, 33, 3], [2, 300, 4]])
def test_short_rows_packed(pkg, cuda, dtype, lens):
    H, K, V = 2, 128, 96
    q, k, v, g, beta, _ = _inputs(1, sum(lens), H, K, V, dtype, seed=len(lens))
    h0 = torch.randn(len(lens), H, K, V, generator=torch.Generator().manual_seed(3))
    q, k, v, g, beta, h0 = (t.to(cuda) for t in (q, k, v, g, beta, h0))
    c = [sum(lens[:i]) for i in range(len(lens) + 1)]
    print(f"[short] packed {dtype} N={len(lens)}", flush=True)
    o, fs = pkg.gdn_fwd(q, k, v, g, beta, h0, cu_seqlens=torch.tensor(c, device=cuda))
    o2, fs2 = pkg.gdn_fwd(q, k, v, g, beta, h0, cu_seqlens=torch.tensor(c, device=cuda), max_segment_chunks=2)
    for i, (a, b) in enumerate(zip(c, c[1:])):
        so, sf = pkg.gdn_fwd(*(t[:, a:b] for t in (q, k, v, g, beta)), h0[i:i + 1])
        assert torch.equal(o[:, a:b], so) and torch.equal(fs[i], sf[0]), i
        so, sf = pkg.gdn_fwd(*(t[:, a:b] for t in (q, k, v, g, beta)), h0[i:i + 1], max_segment_chunks=2)
        assert torch.equal(o2[:, a:b], so) and torch.equal(fs2[i], sf[0]), i


@pytest.mark.parametrize("dtype,T,H", [(torch.float16, 1, 3), (torch.bfloat16, 4, 3), (torch.bfloat16, 2, 3000)])
def test_short_rows_workspace(pkg, cuda, dtype, T, H):
    """The C entry points with no workspace, an empty one, an unaligned one and
    one of a few bytes, and gdn_fwd_launch_noalloc (3000 bf16 heads: more
    records than its array holds), all give gdn_fwd's bits."""
    L, B, K, V = pkg._lib, 1, 128, 16
    lib = L.load_library()
    q, k, v, g, beta, h0 = (t.to(cuda) for t in _inputs(B, T, H, K, V, dtype, seed=T))
    want = pkg.gdn_fwd(q, k, v, g, beta, h0)
    ws = torch.empty(1024, dtype=torch.uint8, device=cuda)
    P = L.GdnFwdParams()
    code = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}
    for n, t in (("q", q), ("k", k), ("v", v), ("g", g), ("beta", beta), ("h0", h0)):
        setattr(P, n, t.data_ptr())
        getattr(P, f"{n}_stride")[:] = t.stride() if n in ("g", "beta", "h0") else t.stride()[:3]
    P.o_stride[:], P.fs_stride[:] = v.stride()[:3], h0.stride()
    P.B, P.T, P.H, P.K, P.V, P.scale, P.chunk_size = B, T, H, K, V, 1.0, 32
    P.qkv_dtype = P.o_dtype = code[dtype]
    P.g_dtype, P.beta_dtype = code[g.dtype], code[beta.dtype]
    assert lib.gdn_fwd_workspace_size(ctypes.byref(P)) == 0
    for fn, ptr, nbytes in ((lib.gdn_fwd_launch, None, 0), (lib.gdn_fwd_launch, ws.data_ptr(), 0),
                            (lib.gdn_fwd_launch, ws.data_ptr() + 16, 0), (lib.gdn_fwd_launch, ws.data_ptr(), 512),
                            (lib.gdn_fwd_launch_noalloc, None, 0)):
        o, fs = torch.full_like(v, float("nan")), torch.full_like(h0, float("nan"))
        P.o, P.final_state, P.workspace, P.workspace_bytes = o.data_ptr(), fs.data_ptr(), ptr, nbytes
        print(f"[short] {dtype} T={T} H={H} {fn.__name__} workspace {nbytes}", flush=True)
        rc = fn(ctypes.byref(P), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert rc == 0, L.status_string(rc)
        assert torch.equal(o, want[0]) and torch.equal(fs, want[1])
