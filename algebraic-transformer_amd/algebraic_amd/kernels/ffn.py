"""ALU-GLU feed-forward block on MI355X with the activation fused into the products.

``alu_glu_ffn(h2, w_g, w_u, w_d, beta)`` is ``(h2 @ w_g * alu(h2 @ w_u, beta)) @ w_d`` as the
model's block computes it (src/algebraic/model.py:185-193, ffn="alu_glu"; alu and its custom VJP
src/algebraic/algebraic.py:86-113), differentiable in h2 and the three weights. The gate/up
product over the packed weights [w_g | w_u] carries the activation in its epilogue (one
HIP kernel writes y = gate*alu(up) and the gate/up residuals); in the backward, the product
dout @ w_d^T carries the activation's VJP in its epilogue (one HIP kernel writes
[d_gate | d_up]). The four remaining products are plain GEMMs on the same MFMA core, each operand
read in its stored layout (no transposed copies): y @ w_d, [d_gate | d_up] @ [w_g | w_u]^T,
h2^T @ [d_gate | d_up], y^T @ dout. Each direction is one library call (``alg_ffn_block_fwd``,
``alg_ffn_block_bwd``). Activations in bf16, products in bf16 with f32 sums; bf16 or f32 weights
(others go through bf16), whose gradients come back in their dtype, f32 ones as the f32 sum. d_ff
must be a multiple of 128 and the widths multiples of 8. No CPU fallback.
"""

import torch

from .. import _lib


_DTYPES = {torch.bfloat16: _lib.DTYPE_BF16, torch.float32: _lib.DTYPE_F32}


def _weight(w):
    """``w`` as the library reads it (bf16 or f32, contiguous, aligned) and its dtype code."""
    if w.dtype not in _DTYPES:
        w = w.to(torch.bfloat16)
    return _lib.aligned16(w), _DTYPES[w.dtype]


def _grad_like(w_dtype, rows, cols, dev):
    """An empty weight gradient in the weight's dtype (bf16 where the library writes no other)."""
    dt = w_dtype if w_dtype in _DTYPES else torch.bfloat16
    return torch.empty((rows, cols), dtype=dt, device=dev), _DTYPES[dt]


def _parts(act):
    """Pointers of the three (N, F) bf16 matrices of one (3, N, F) allocation."""
    base, step = act.data_ptr(), act.numel() // 3 * 2
    return base, base + step, base + 2 * step


class _FfnFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, h2, w_g, w_u, w_d, beta):
        lib = _lib.load()
        shape = h2.shape
        d = shape[-1]
        x = _lib.aligned16(h2).reshape(-1, d)
        dev, bf = x.device, torch.bfloat16
        N, F, dm = x.shape[0], w_g.shape[1], w_d.shape[1]
        (wg, gt), (wu, ut), (wd, dt) = _weight(w_g), _weight(w_u), _weight(w_d)
        w_gu = torch.empty((d, 2 * F), dtype=bf, device=dev)
        wd16 = torch.empty((F, dm), dtype=bf, device=dev) if dt == _lib.DTYPE_F32 else None
        act = torch.empty((3, N, F), dtype=bf, device=dev)  # y, gate, up
        out = torch.empty((N, dm), dtype=bf, device=dev)
        nbytes = lib.alg_ffn_block_workspace_size(N, d, F, dm, 0)
        ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=dev)
        p = _lib.ptr
        _lib.check(lib.alg_ffn_block_fwd(_lib.stream_of(x), N, d, F, dm, p(x), p(wg), gt, p(wu), ut, p(wd), dt,
                                         float(beta), p(w_gu), p(wd16), *_parts(act), p(out), p(ws), nbytes),
                   "alu_glu_ffn")
        ctx.save_for_backward(x, w_gu, wd if wd16 is None else wd16, act)
        ctx.meta = (shape, beta, w_g.dtype, w_u.dtype, w_d.dtype)
        return out.reshape(*shape[:-1], dm)

    @staticmethod
    def backward(ctx, dout):
        x, w_gu, wd, act = ctx.saved_tensors
        shape, beta, tg, tu, td = ctx.meta
        lib = _lib.load()
        dev = x.device
        N, d = x.shape
        F, dm = wd.shape
        do = _lib.aligned16(dout.to(torch.bfloat16)).reshape(N, dm)
        dx = torch.empty_like(x)
        (dwg, gt), (dwu, ut), (dwd, dt) = (_grad_like(t, r, c, dev) for t, r, c in ((tg, d, F), (tu, d, F), (td, F, dm)))
        nbytes = lib.alg_ffn_block_workspace_size(N, d, F, dm, 1)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        p = _lib.ptr
        _lib.check(lib.alg_ffn_block_bwd(_lib.stream_of(x), N, d, F, dm, p(x), p(w_gu), p(wd), *_parts(act), p(do),
                                         float(beta), p(dx), p(dwg), gt, p(dwu), ut, p(dwd), dt, p(ws), nbytes),
                   "alu_glu_ffn backward")
        return dx.reshape(shape), dwg.to(tg), dwu.to(tu), dwd.to(td), None


def alu_glu_ffn(h2, w_g, w_u, w_d, beta: float = 0.5):
    """(h2 @ w_g * alu(h2 @ w_u, beta)) @ w_d for bfloat16 GPU tensors (model.py:185-193)."""
    if h2.dtype != torch.bfloat16:
        raise NotImplementedError(f"dtype {h2.dtype}: the gfx950 feed-forward takes bfloat16 activations")
    d = h2.shape[-1]
    if w_g.shape != w_u.shape or w_g.shape[0] != d or w_d.shape[0] != w_g.shape[1]:
        raise ValueError("w_g, w_u must be (d, d_ff) and w_d (d_ff, d_out)")
    if not h2.is_cuda:
        raise RuntimeError("alu_glu_ffn needs GPU tensors (no CPU fallback)")
    # The library packs the weights by pointer, so nothing else would notice one on another device.
    if any(w.device != h2.device for w in (w_g, w_u, w_d)):
        raise RuntimeError(f"alu_glu_ffn needs its weights on {h2.device}")
    return _FfnFn.apply(h2, w_g, w_u, w_d, float(beta))
