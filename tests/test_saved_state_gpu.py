"""What the attention saves for its backward, seen through saved-tensor hooks that store floating
tensors in fewer bits (as activation compression does): only the rounding of the stored values may
show, never another branch of the guard."""

import pytest

from helpers import attention_inputs

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _pack(t):
    return (t.dtype, t.to(torch.bfloat16) if t.is_floating_point() else t)


def _unpack(saved):
    return saved[1].to(saved[0])


@pytest.mark.parametrize("prologue", [False, True])
@pytest.mark.parametrize("range_guard", [False, True])
def test_guard_flag_survives_reduced_precision_storage(prologue, range_guard):
    from algebraic_amd.kernels.flash import flash_attention
    from algebraic_amd.kernels.prologue import cayley_table_geometric, qk_norm_rotary_flash_attention
    B, H, T, D = 2, 3, 150, 64
    q, k, v, do, sink = (torch.tensor(a, device="cuda") for a in attention_inputs(B, H, T, D))
    bf = torch.bfloat16
    args = [t.to(bf).requires_grad_(True) for t in (q, k, v)] + [sink.requires_grad_(True)]
    kw = dict(kind="asinh", n=16, c=8.0, range_guard=range_guard)

    def grads():
        if prologue:
            cs, sn = cayley_table_geometric(D, T, device="cuda")
            o = qk_norm_rotary_flash_attention(*args, None, None, cs, sn, **kw)
        else:
            o = flash_attention(*args, **kw)
        return torch.autograd.grad(o, args, do.to(bf))

    want = grads()
    with torch.autograd.graph.saved_tensors_hooks(_pack, _unpack):
        got = grads()
    for a, b in zip(got, want):
        a, b = a.float(), b.float()
        # The prologue's 1/rms and gains in bf16: 2^-9 each.
        assert float((a - b).norm() / b.norm()) < 2e-2
