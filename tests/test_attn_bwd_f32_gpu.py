"""The f32 attention backward kernel at the sizes where its 64-key blocks and 32 x 32 wave blocks can
go wrong, and on both sides of the launch rule (one or two workgroups to a CU), against the
float64 dense oracle at the f32 bar; dK and dV, which no atomics form, the same bits on every
call."""

import numpy as np
import pytest

from helpers import rel_l2
from oracle import attention as OA

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

VARIANTS = {"guarded": dict(range_guard=True), "shifted": dict(shift=True), "clipped": dict()}
# (B, H, T, D): one key, blocks one short, whole and one over, an odd number of query tiles; the
# last has 1152 key blocks, two to a CU (run once).
CASES = [(1, 2, 1, 64), (1, 3, 63, 64), (2, 1, 64, 128), (1, 2, 65, 64), (1, 1, 97, 128), (1, 2, 130, 64),
         (1, 2, 320, 128), (1, 2, 321, 64), (8, 16, 520, 64)]
RUNS = [(c, v, lay) for c in CASES for v in VARIANTS for lay in ("bhtd", "bthd")
        if c[0] * c[1] < 100 or (v, lay) == ("guarded", "bhtd")]


@pytest.mark.parametrize("shape,variant,layout", RUNS, ids=lambda x: "x".join(map(str, x)) if isinstance(x, tuple) else x)
def test_f32_backward(shape, variant, layout):
    from algebraic_amd.kernels.flash import flash_attention
    B, H, T, D = shape
    kw = VARIANTS[variant]
    print(f"[f32 bwd] {shape} {kw} {layout}", flush=True)
    rng = np.random.default_rng(B + H + T + D)
    q, k, v, do = (rng.standard_normal((B, H, T, D)).astype(np.float32) for _ in range(4))
    q, k = (x / np.sqrt(np.mean(x * x, -1, keepdims=True) + 1e-5) for x in (q, k))
    sink = (rng.standard_normal(H) * 0.1).astype(np.float32)
    tr = (lambda x: x.transpose(0, 2, 1, 3)) if layout == "bthd" else (lambda x: x)
    mk = lambda x: torch.tensor(np.ascontiguousarray(tr(x)), device="cuda")
    tq, tk, tv = (mk(x).requires_grad_(True) for x in (q, k, v))
    ts = torch.tensor(sink, device="cuda", requires_grad=True)
    runs = []
    for _ in range(2):
        o = flash_attention(tq, tk, tv, ts, kind="asinh", n=16, c=8.0, block=T, layout=layout, **kw)
        runs.append(torch.autograd.grad(o, (tq, tk, tv, ts), mk(do)))
    want = OA.dense_backward(q, k, v, sink, do, n=16, c=8.0)
    for name, g, w in zip(("dq", "dk", "dv", "dsink"), runs[0], want):
        a = g.double().cpu().numpy()
        assert rel_l2(tr(a) if a.ndim == 4 else a, w) < 1e-5, name
    assert torch.equal(runs[0][1], runs[1][1]) and torch.equal(runs[0][2], runs[1][2])
