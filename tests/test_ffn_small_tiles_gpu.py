"""The feed-forward products on 64 x 64 and 128 x 128 tiles (short inputs): one row and column of
tiles more or less than whole, k of one step, under one, and with a remainder, each stored layout,
k splits, a row length and tile count that take the plain tile order; the two fused epilogues around
the sizes where the tile changes. Products against a
float32 product of the same bf16 operands (one bf16 rounding, and the order of the f32 sums).
"""

import numpy as np
import pytest

from helpers import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("a_trans,b_trans", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(64, 64, 64), (72, 56, 40), (128, 192, 320), (200, 136, 1000), (8, 520, 192),
                                   (304, 1024, 4096), (1016, 776, 2056), (776, 4088, 1016), (320, 768, 136)])
def test_small_products(M, N, K, a_trans, b_trans):
    from algebraic_amd import _lib as L
    lib = L.load()
    print(f"[ffn small] M={M} N={N} K={K} {a_trans} {b_trans}", flush=True)
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


@pytest.mark.parametrize("dtypes", ["bbb", "fff", "bfb", "fbf"])
@pytest.mark.parametrize("N,d,F", [(1, 64, 128), (64, 72, 128), (65, 128, 256), (129, 192, 640), (1000, 256, 1024),
                                   (1025, 320, 2048)])
def test_small_block(N, d, F, dtypes):
    """Weights in bf16 (b) or f32 (f): the products run on their bf16 values, an f32 weight's gradient
    is the f32 sum, which the oracle rounds to bf16."""
    from algebraic_amd.kernels.ffn import alu_glu_ffn
    from oracle import ffn as OF
    from oracle.numerics import round_bf16
    print(f"[ffn small block] N={N} d={d} F={F} {dtypes}", flush=True)
    rng = np.random.default_rng(N + d + F)
    mk = lambda *s: round_bf16(rng.standard_normal(s).astype(np.float32) / np.sqrt(s[0] if len(s) == 2 else 1))
    x = round_bf16(rng.standard_normal((N, d)).astype(np.float32))
    do = round_bf16(rng.standard_normal((N, d)).astype(np.float32))
    wg, wu, wd = mk(d, F), mk(d, F), mk(F, d)
    dt = {"b": torch.bfloat16, "f": torch.float32}
    tx, tg, tu, td = (torch.tensor(a, device="cuda").to(dt[c]).requires_grad_(True)
                      for a, c in zip((x, wg, wu, wd), "b" + dtypes))
    with torch.no_grad():  # f32 weights that bf16 does not hold
        for w in (tg, tu, td):
            if w.dtype == torch.float32:
                w.mul_(1 + 2.0 ** -12)
    y = alu_glu_ffn(tx, tg, tu, td)
    got = [y.detach(), *torch.autograd.grad(y, (tx, tg, tu, td), torch.tensor(do, device="cuda").to(torch.bfloat16))]
    out, *_ = OF.ffn_forward(x, wg, wu, wd)
    want = [out, *OF.ffn_backward(x, wg, wu, wd, do)[:4]]
    for name, a, b, w in zip(("out", "dx", "dw_g", "dw_u", "dw_d"), got, want, (tx, tx, tg, tu, td)):
        assert a.dtype == w.dtype and a.is_contiguous()
        assert rel_l2(a.float().cpu().numpy(), b) < 1e-2, name


@pytest.mark.parametrize("host", [0, 1, 2])
def test_weight_on_the_host_is_refused(host):
    """A weight on another device than the input is refused before any pointer reaches a kernel."""
    from algebraic_amd.kernels.ffn import alu_glu_ffn
    x = torch.zeros(8, 64, dtype=torch.bfloat16, device="cuda")
    w = [torch.zeros(s, dtype=torch.bfloat16, device="cuda") for s in ((64, 128), (64, 128), (128, 64))]
    w[host] = w[host].cpu()
    with pytest.raises(RuntimeError, match="weights"):
        alu_glu_ffn(x, *w)
