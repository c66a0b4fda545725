"""The f32 head's products on the bf16 matrix cores (three bf16 planes an operand, csrc/head.hip):
sizes at the edges of the 128 x 128 and 256 x 256 tiles, of the 64-deep k steps and of the vocabulary
and token splits, against the float64 dense oracle at the f32 bars; inputs that are not finite, which
the f32 kernels take, against those kernels (the streamed schedule runs them always) and numpy.
"""

import ctypes

import numpy as np
import pytest

from helpers import rel_l2
from oracle import head as OH
from oracle.numerics import head_clamp

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# (N, d, V) and the (tile, ranges) of the logits, dh and dE: one k step, a partial one, several; N and V
# one past and at a tile; d past a tile; vocabulary ranges of dh, token ranges of the dE tail. Under
# 256 tokens (tile 0) the f32 kernels run.
SHAPES = [((256, 64, 256), (128, 1), (128, 1), (128, 1)), ((257, 72, 513), (128, 1), (128, 2), (128, 1)),
          ((255, 128, 255), (0, 1), (0, 1), (0, 1)), ((513, 264, 1032), (128, 1), (128, 4), (128, 1)),
          ((100, 200, 4100), (0, 1), (0, 16), (0, 1)), ((2050, 192, 700), (128, 1), (128, 2), (256, 2)),
          # Logits on 256 tiles ragged in N and V (V % 256 under 128: the last tile has one row of
          # 128-entry partials); dh of 7 and 16 ranges and dE on 256 tiles, split over the tokens in one.
          ((1030, 1032, 4200), (256, 1), (256, 7), (256, 1)), ((520, 776, 8200), (256, 1), (256, 16), (256, 1)),
          ((2049, 520, 4360), (256, 1), (256, 7), (256, 2))]


def _plans(N, d, V):
    from algebraic_amd import _lib as L
    out = []
    for product in (L.HEAD_LOGITS, L.HEAD_DH, L.HEAD_DE):
        tile, split = ctypes.c_int(), ctypes.c_int()
        L.check(L.load().alg_head_plan(L.DTYPE_F32, product, N, d, V, tile, split), "alg_head_plan")
        out.append((tile.value, split.value))
    return tuple(out)


def _run(h, E, t, e_dtype=torch.float32, g=1.0, n=8):
    from algebraic_amd.kernels.fused_head import fused_head
    th = torch.tensor(h, device="cuda", requires_grad=True)
    tE = torch.tensor(E, device="cuda").to(e_dtype).requires_grad_(True)
    obj, pt = fused_head(th, tE, torch.tensor(t, device="cuda"), kind="alg_ce", n=n, c=2.0, block_n=len(h))
    dh, dE = torch.autograd.grad(obj * g, (th, tE))
    f = lambda x: x.detach().float().cpu().numpy().astype(np.float64)
    return float(obj.detach()), f(pt), f(dh), f(dE)


@pytest.mark.parametrize("n", [8, 16])
@pytest.mark.parametrize("case", SHAPES, ids=lambda s: "x".join(map(str, s[0])))
def test_split_products_match_dense(case, n):
    (N, d, V), *plans = case
    assert _plans(N, d, V) == tuple(plans)
    print(f"f32 head split N{N} d{d} V{V} n{n}", flush=True)
    rng = np.random.default_rng(N + d + V)
    h = rng.standard_normal((N, d)).astype(np.float32)
    E = (rng.standard_normal((V, d)) * 0.15).astype(np.float32)
    t = rng.integers(0, V, N).astype(np.int32)
    obj, pt, dh, dE = _run(h, E, t, g=0.7, n=n)
    obj_r, pt_r = OH.dense_forward(h, E, t, n=n, c=2.0)
    dh_r, dE_r = OH.dense_backward(h, E, t, 0.7, n=n, c=2.0)
    np.testing.assert_allclose(obj, obj_r, rtol=1e-5)
    # pt = (rho stat)^n: n times the relative error of its factors, 1e-5 allowed at n = 8.
    np.testing.assert_allclose(pt, pt_r, rtol=1e-5 * n / 8)
    # A plane dropped or taken twice shows as 2^-9, 2^-17 or 2^-25 of the whole; the f32 sums
    # themselves stay within the f32 bar (the weights multiply a logit's error by n).
    assert rel_l2(dh, dh_r) < 3e-6 * n / 8
    assert rel_l2(dE, dE_r) < 3e-6 * n / 8


def test_columns_of_very_different_sizes_keep_their_precision():
    """Columns of E up to 1e12 times smaller than others, met by columns of h as much larger, weigh
    alike in the logits: each column of dh and dE, on its own scale, keeps the f32 bar."""
    rng = np.random.default_rng(11)
    N, d, V = 300, 128, 600
    s = (10.0 ** rng.uniform(-12, 12, d)).astype(np.float32)
    h = rng.standard_normal((N, d)).astype(np.float32) * s
    E = ((rng.standard_normal((V, d)) * 0.15).astype(np.float32) / s).astype(np.float32)
    t = rng.integers(0, V, N).astype(np.int32)
    _, pt, dh, dE = _run(h, E, t)
    _, pt_r = OH.dense_forward(h, E, t, n=8, c=2.0)
    dh_r, dE_r = OH.dense_backward(h, E, t, 1.0, n=8, c=2.0)
    np.testing.assert_allclose(pt, pt_r, rtol=1e-5)
    for j in range(d):
        assert rel_l2(dh[:, j] * s[j], dh_r[:, j] * s[j]) < 3e-6, j
        assert rel_l2(dE[:, j] / s[j], dE_r[:, j] / s[j]) < 3e-6, j


def test_small_values_keep_their_precision():
    """Gradient scales down to 1e-20: the planes hold the same 24 bits there."""
    rng = np.random.default_rng(3)
    h = rng.standard_normal((300, 128)).astype(np.float32)
    E = (rng.standard_normal((500, 128)) * 0.15).astype(np.float32)
    t = rng.integers(0, 500, 300).astype(np.int32)
    _, _, dh, dE = _run(h, E, t, g=1e-20)
    dh_r, dE_r = OH.dense_backward(h, E, t, 1e-20, n=8, c=2.0)
    assert rel_l2(dh, dh_r) < 3e-6 and rel_l2(dE, dE_r) < 3e-6


@pytest.mark.parametrize("h_scale,E_scale,g", [(1.0, 1.0, 1e-32), (1e16, 1e-35, 1e4), (1e-30, 1e30, 1.0),
                                               (1e-35, 1e16, 1e4)])
def test_whole_f32_range_keeps_its_precision(h_scale, E_scale, g):
    """Upstream gradients, hidden states and embeddings whose planes would be subnormal bf16 (or whose
    scaled products would overflow): the results keep the f32 bar."""
    rng = np.random.default_rng(5)
    h = (rng.standard_normal((300, 128)) * h_scale).astype(np.float32)
    E = (rng.standard_normal((500, 128)) * 0.15 * E_scale).astype(np.float32)
    t = rng.integers(0, 500, 300).astype(np.int32)
    _, pt, dh, dE = _run(h, E, t, g=g)
    _, pt_r = OH.dense_forward(h, E, t, n=8, c=2.0)
    dh_r, dE_r = OH.dense_backward(h, E, t, g, n=8, c=2.0)
    np.testing.assert_allclose(pt, pt_r, rtol=1e-5)
    # The norms of such values underflow: scaled to about 1 first.
    for got, want in ((dh, dh_r), (dE, dE_r)):
        m = np.abs(want).max()
        assert rel_l2(got / m, want / m) < 3e-6


@pytest.mark.parametrize("g", [float("inf"), float("nan")])
def test_upstream_gradient_not_finite(g, monkeypatch):
    """As the f32 kernels (the streamed schedule) give it."""
    from algebraic_amd.kernels import fused_head as FH
    rng = np.random.default_rng(6)
    h = np.abs(rng.standard_normal((300, 64))).astype(np.float32)  # one sign: infinities stay infinities
    E = (rng.standard_normal((500, 64)) * 0.15).astype(np.float32)
    t = rng.integers(0, 250, 300).astype(np.int32)
    _, _, dh, dE = _run(h, E, t, g=g)
    monkeypatch.setattr(FH, "SCHEDULE", "streamed")
    _, _, dh_s, dE_s = _run(h, E, t, g=g)
    np.testing.assert_array_equal(dh, dh_s)
    np.testing.assert_array_equal(dE, dE_s)
    if g > 0:
        assert np.isinf(dE[300:]).all()  # entries that are no token's target


@pytest.mark.parametrize("where", ["h_inf", "h_nan", "E_inf", "E_huge"])
def test_not_finite_inputs(where, monkeypatch):
    from algebraic_amd.kernels import fused_head as FH
    rng = np.random.default_rng(7)
    N, d, V = 300, 128, 600
    h = rng.standard_normal((N, d)).astype(np.float32)
    E = (rng.standard_normal((V, d)) * 0.15).astype(np.float32)
    t = rng.integers(0, V, N).astype(np.int32)
    if where == "h_inf":
        h[17, 5] = np.inf
    elif where == "h_nan":
        h[17, 5] = np.nan
    elif where == "E_inf":
        E[33, 2] = -np.inf
    else:
        E[33, 2] = 3.4e38  # finite, but not in bf16
    obj, pt, dh, dE = _run(h, E, t)
    monkeypatch.setattr(FH, "SCHEDULE", "streamed")
    obj_s, pt_s, dh_s, dE_s = _run(h, E, t)
    np.testing.assert_equal(obj, obj_s)
    np.testing.assert_equal(pt, pt_s)
    for got, want in ((dh, dh_s), (dE, dE_s)):
        np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
        np.testing.assert_allclose(got, want, rtol=1e-4, atol=1e-9)
    # The formula in numpy f32: min(z/c, X) takes X for a NaN logit.
    with np.errstate(all="ignore"):
        z = (h.astype(np.float64) @ E.T.astype(np.float64)).astype(np.float32)
        x = np.fmin(z / np.float32(2), np.float32(head_clamp(V, 8)))
        rad = 1 + x * x
        w = ((x + rad * (1 / np.sqrt(rad))) ** 8).astype(np.float64)
        pt_r = w[np.arange(N), t] / w.sum(1)
    same = np.isfinite(pt_r)
    assert same.sum() >= N - 1 if where.startswith("h") else True
    rows = same & (np.arange(N) != 17)
    np.testing.assert_allclose(pt[rows], pt_r[rows], rtol=1e-4, atol=1e-12)
