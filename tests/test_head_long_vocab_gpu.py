"""The head over a vocabulary whose rows of the logit gradient and of the residual (2 V bytes each,
256 of them in a tile) lie more than 2^32 bytes apart inside one tile: every token's dh against
float64 torch in vocabulary chunks."""

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

N, D, V = 256, 8, 9_000_000
HEAD_N, HEAD_C = 8, 2.0
CHUNK = 1_000_000


def _reference(h, E, t):
    h = h.double()
    chunks = range(0, V, CHUNK)

    def weights(v0):
        x = (h @ E[v0:v0 + CHUNK].double().t().contiguous()) / HEAD_C
        return x, torch.exp(HEAD_N * torch.asinh(x))

    total = sum(weights(v0)[1].sum(-1) for v0 in chunks)
    dh, size = torch.zeros_like(h), torch.zeros_like(h)
    rows = torch.arange(N, device=h.device)
    for v0 in chunks:
        x, w = weights(v0)
        dz = w / total[:, None]
        mine = (t >= v0) & (t < v0 + CHUNK)
        dz[rows[mine], t[mine] - v0] -= 1.0
        dz *= torch.rsqrt(1 + x * x) * (HEAD_N / HEAD_C / N)
        dh += dz @ E[v0:v0 + CHUNK].double()
        size += dz.abs() @ E[v0:v0 + CHUNK].double().abs()
    return dh, size


# f32: V / 16 additions (an MFMA adds 16 products) of 2^-24 of the sum of magnitudes each, as a random
# walk, four times over. bf16: the rounding of dZ's and E's entries and of dh.
@pytest.mark.parametrize("dtype,bar", [("f32", 4 * (V / 16) ** 0.5 * 2.0 ** -24), ("bf16", 2e-2)])
def test_rows_over_4_gib_apart(dtype, bar):
    from algebraic_amd.kernels.fused_head import fused_head
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    g = torch.Generator(device="cuda")
    g.manual_seed(4)
    h = torch.randn(N, D, device="cuda", generator=g).to(dt).requires_grad_(True)
    E = (0.3 * torch.randn(V, D, device="cuda", generator=g)).to(dt)
    t = torch.randint(0, V, (N,), device="cuda", generator=g)
    obj, _ = fused_head(h, E, t, kind="alg_ce", n=HEAD_N, c=HEAD_C, block_n=N)
    (dh,) = torch.autograd.grad(obj, (h,))
    want, size = _reference(h.detach(), E, t)
    assert float((want.norm(dim=-1) / size.norm(dim=-1)).min()) > 4 * bar  # a lost row would show
    err = (dh.double() - want).norm(dim=-1) / size.norm(dim=-1)
    assert float(err.max()) < bar, f"token {int(err.argmax())}: {float(err.max()):.2e}"
