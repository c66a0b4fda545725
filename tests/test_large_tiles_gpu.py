"""The products of the feed-forward and of the bf16 head on 256 x 256 tiles where these are ragged:
rows, columns and k past a tile, whole and split over k, each stored layout; the block's direct and
summed stores into one or two weight gradients, in bf16 and f32. Every case states the tile and the
k ranges it is meant for and checks them, so that a change of the rule that chooses them cannot take
the test elsewhere.
"""

import ctypes

import numpy as np
import pytest

from helpers import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _plan(product, M, N, K):
    from algebraic_amd import _lib as L
    tile, split = ctypes.c_int(), ctypes.c_int()
    L.check(L.load().alg_ffn_plan(product, M, N, K, tile, split), "alg_ffn_plan")
    return tile.value, split.value


@pytest.mark.parametrize("a_trans,b_trans", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K,split", [(4104, 4104, 200, 1), (2056, 4104, 1096, 1), (1032, 1032, 8200, 8),
                                         (4360, 4104, 2056, 2)])
def test_ragged_products(M, N, K, split, a_trans, b_trans):
    from algebraic_amd import _lib as L
    lib = L.load()
    assert _plan(L.FFN_GEMM, M, N, K) == (256, split)
    print(f"[ffn large] M={M} N={N} K={K} {a_trans} {b_trans}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    B = torch.randn(K, N, device="cuda", generator=g).to(torch.bfloat16)
    a = A.t().contiguous() if a_trans else A
    b = B.t().contiguous() if b_trans else B
    ws_b = lib.alg_ffn_gemm_workspace_size(M, N, K)
    ws = torch.full((max(ws_b, 1),), 0x7F, dtype=torch.uint8, device="cuda")
    c = torch.full((M + 1, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    L.check(lib.alg_ffn_gemm(L.stream_of(a), M, N, K, L.ptr(a), a.shape[1], int(a_trans), L.ptr(b), b.shape[1],
                             int(b_trans), L.ptr(c), N, L.ptr(ws), ws_b), "alg_ffn_gemm")
    torch.cuda.synchronize()
    ref = A.float() @ B.float()
    tol = ref.abs() * 2.0 ** -8 + (A.float().abs() @ B.float().abs()) * 2.0 ** -20
    bad = ((c[:M].float() - ref).abs() > tol) | c[:M].float().isnan()
    assert not bool(bad.any()), f"{int(bad.sum())} entries off, first {bad.nonzero()[:4].tolist()}"
    assert bool(c[M].isnan().all())  # nothing past the last row


# The first shape splits all four plain products over k (their sums go through the summing kernel),
# the second runs both weight gradients whole (stored from the accumulators).
@pytest.mark.parametrize("dtypes", ["bbb", "fff", "fbf"])
@pytest.mark.parametrize("N,d,F,dw_splits", [(4100, 1032, 2816, (2, 4)), (2060, 1544, 4224, (1, 1))])
def test_ragged_block(N, d, F, dw_splits, dtypes):
    from algebraic_amd import _lib as L
    from algebraic_amd.kernels.ffn import alu_glu_ffn
    from oracle import ffn as OF
    from oracle.numerics import round_bf16
    assert _plan(L.FFN_GATE_UP, N, F, d)[0] == _plan(L.FFN_DY, N, F, d)[0] == 256
    assert _plan(L.FFN_GEMM, N, d, F)[0] == _plan(L.FFN_GEMM, N, d, 2 * F)[0] == 256
    assert (_plan(L.FFN_GEMM, d, 2 * F, N), _plan(L.FFN_GEMM, F, d, N)) == tuple((256, s) for s in dw_splits)
    print(f"[ffn large block] N={N} d={d} F={F} {dtypes}", flush=True)
    rng = np.random.default_rng(N + d + F)
    mk = lambda *s: round_bf16(rng.standard_normal(s).astype(np.float32) / np.float32(np.sqrt(s[0])))
    x = round_bf16(rng.standard_normal((N, d)).astype(np.float32))
    do = round_bf16(rng.standard_normal((N, d)).astype(np.float32))
    wg, wu, wd = mk(d, F), mk(d, F), mk(F, d)
    dt = {"b": torch.bfloat16, "f": torch.float32}
    tx, tg, tu, td = (torch.tensor(a, device="cuda").to(dt[c]).requires_grad_(True)
                      for a, c in zip((x, wg, wu, wd), "b" + dtypes))
    y = alu_glu_ffn(tx, tg, tu, td)
    got = [y.detach(), *torch.autograd.grad(y, (tx, tg, tu, td), torch.tensor(do, device="cuda").to(torch.bfloat16))]
    out, *_ = OF.ffn_forward(x, wg, wu, wd)
    want = [out, *OF.ffn_backward(x, wg, wu, wd, do)[:4]]
    edge = np.s_[-(N % 256):, :], np.s_[-(N % 256):, :], np.s_[-(d % 256):, :], np.s_[-(d % 256):, :], np.s_[:, -(d % 256):]
    for name, a, b, w, e in zip(("out", "dx", "dw_g", "dw_u", "dw_d"), got, want, (tx, tx, tg, tu, td), edge):
        assert a.dtype == w.dtype and a.is_contiguous()
        a = a.float().cpu().numpy()
        assert rel_l2(a, b) < 1e-2, name
        assert rel_l2(a[e], np.asarray(b)[e]) < 1e-2, f"{name} in the ragged tiles"


@pytest.mark.parametrize("schedule", ["residual", "recompute"])
@pytest.mark.parametrize("e_dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("N,d,V,dh_split,de_split", [(1030, 1032, 8200, 10, 1), (2060, 1032, 4104, 5, 2)])
def test_ragged_head(N, d, V, dh_split, de_split, e_dtype, schedule, monkeypatch):
    from algebraic_amd import _lib as L
    from algebraic_amd.kernels import fused_head as FH
    from oracle import head as OH
    from oracle.numerics import round_bf16
    monkeypatch.setattr(FH, "SCHEDULE", schedule)
    tile, split = ctypes.c_int(), ctypes.c_int()
    for product, ranges in ((L.HEAD_LOGITS, 1), (L.HEAD_DH, dh_split), (L.HEAD_DE, de_split)):
        L.check(L.load().alg_head_plan(L.DTYPE_BF16, product, N, d, V, tile, split), "alg_head_plan")
        assert (tile.value, split.value) == (256, ranges)
    print(f"head large tiles N{N} d{d} V{V} {e_dtype} {schedule}", flush=True)
    rng = np.random.default_rng(N + d + V)
    h = round_bf16(rng.standard_normal((N, d)).astype(np.float32))
    E = round_bf16((rng.standard_normal((V, d)) * 0.05).astype(np.float32))
    t = rng.integers(0, V, N).astype(np.int32)
    th = torch.tensor(h, device="cuda").to(torch.bfloat16).requires_grad_(True)
    tE = torch.tensor(E, device="cuda").to(e_dtype).requires_grad_(True)
    obj, pt = FH.fused_head(th, tE, torch.tensor(t, device="cuda"), kind="alg_ce", n=8, c=2.0, block_n=N)
    dh, dE = torch.autograd.grad(obj * 0.7, (th, tE))
    obj_r, pt_r = OH.dense_forward(h, E, t, n=8, c=2.0)
    dh_r, dE_r = OH.dense_backward(h, E, t, 0.7, n=8, c=2.0)
    np.testing.assert_allclose(obj.item(), obj_r, rtol=2e-3, atol=2e-4)
    np.testing.assert_allclose(pt.cpu().numpy(), pt_r, rtol=1e-4, atol=1e-9)  # f32 sums of exact products
    for got, want, rows in ((dh, dh_r, N), (dE, dE_r, V)):
        got = got.float().cpu().numpy()
        assert rel_l2(got, want) < 1e-2
        edge = np.s_[-(rows % 256):, :], np.s_[:, -(d % 256):]
        assert all(rel_l2(got[e], want[e]) < 1e-2 for e in edge)
