"""The bf16 head on 128 x 128 tiles (few tokens or a small vocabulary) and at the sizes where it
changes to 256 x 256: tiles one short, whole and one over in tokens, vocabulary and width, k of less
than a step and with a remainder, vocabulary splits of the dh product; against the float64 dense
oracle at the head's bars, for the residual and the recompute schedule, and the evaluation head."""

import numpy as np
import pytest

from helpers import rel_l2
from oracle import head as OH
from oracle.numerics import round_bf16

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# (N, d, V); 256 tiles of 128 in the last but two, one row of tiles more in the last but one; the
# last has ragged 256 x 256 tiles.
SHAPES = [(1, 64, 127), (127, 72, 129), (129, 200, 1000), (128, 136, 8200), (300, 1032, 700), (100, 256, 32768),
          (100, 64, 32769), (1100, 320, 4300)]


@pytest.mark.parametrize("schedule", ["residual", "recompute"])
@pytest.mark.parametrize("e_dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_small_tiles(shape, e_dtype, schedule, monkeypatch):
    from algebraic_amd.kernels import fused_head as FH
    monkeypatch.setattr(FH, "SCHEDULE", schedule)
    N, d, V = shape
    print(f"head small tiles N{N} d{d} V{V} {e_dtype} {schedule}", flush=True)
    rng = np.random.default_rng(N + d + V)
    h = round_bf16(rng.standard_normal((N, d)).astype(np.float32))
    E = round_bf16((rng.standard_normal((V, d)) * 0.1).astype(np.float32))
    t = rng.integers(0, V, N).astype(np.int32)
    th = torch.tensor(h, device="cuda").to(torch.bfloat16).requires_grad_(True)
    tE = torch.tensor(E, device="cuda").to(e_dtype).requires_grad_(True)
    tt = torch.tensor(t, device="cuda")
    obj, pt = FH.fused_head(th, tE, tt, kind="alg_ce", n=8, c=2.0, block_n=N)
    dh, dE = torch.autograd.grad(obj * 0.7, (th, tE))
    obj_r, pt_r = OH.dense_forward(h, E, t, n=8, c=2.0)
    dh_r, dE_r = OH.dense_backward(h, E, t, 0.7, n=8, c=2.0)
    np.testing.assert_allclose(obj.item(), obj_r, rtol=2e-3, atol=2e-4)
    np.testing.assert_allclose(pt.cpu().numpy(), pt_r, rtol=1e-4, atol=1e-9)  # f32 sums of exact products
    assert rel_l2(dh.float().cpu().numpy(), dh_r) < 1e-2
    assert rel_l2(dE.float().cpu().numpy(), dE_r) < 1e-2
    lp, am = FH.head_logprob(th.detach(), tE.detach(), tt, n=8, c=2.0)
    lp_r, am_r, z = OH.eval_logprob(h, E, t, n=8, c=2.0)
    np.testing.assert_allclose(lp.cpu().numpy(), lp_r, atol=1e-4, rtol=0)
    zr = z[np.arange(N), am.cpu().numpy()]
    np.testing.assert_allclose(zr, z.max(axis=1), rtol=1e-5, atol=1e-5)
