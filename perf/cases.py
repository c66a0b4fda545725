"""The work that users of this package have it do, as measurable cases.

Each case is one pass through a public entry point on inputs of the distributions the model
meets: QK RMS-normalised scores, a learned per-head sink, embeddings of std 0.02, uniform
targets, the algebraic preset's exponents (attention n = 16, c = 8 with the range guard; head
n = 8, c = 2). ``listed`` names the sizes that stand for the range, ``draw`` gives others of
the same range, ``exact`` states the same maths in float64 with plain torch.
"""

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path.cwd() / "algebraic-transformer_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from algebraic_amd.kernels.ffn import alu_glu_ffn  # noqa: E402
from algebraic_amd.kernels.flash import flash_attention  # noqa: E402
from algebraic_amd.kernels.fused_head import fused_head, head_logprob  # noqa: E402
from algebraic_amd.kernels.norm import rms_norm  # noqa: E402
from algebraic_amd.kernels.prologue import cayley_table_geometric, qk_norm_rotary_flash_attention  # noqa: E402

ATTN_N, ATTN_C = 16, 8.0
HEAD_N, HEAD_C = 8, 2.0
EPS = 1e-5
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # Attention of the 1B shape, one training microbatch: the headline configuration.
        dict(name="attention_1b_train", kind="attention", dtype="bf16", B=8, H=16, T=2048, D=128, train=True),
        # The whole attention layer between the projections (norm, rotation, attention, and back)
        # at the 350M shape, in the projections' own storage order.
        dict(name="attention_layer_350m_train", kind="layer", dtype="bf16", B=8, H=16, T=2048, D=64, train=True),
        # Single-precision training at the 125M shape (the reference's CPU configuration).
        dict(name="attention_125m_f32_train", kind="attention", dtype="f32", B=2, H=12, T=1024, D=64, train=True),
        # Prefill over a long context, forward only.
        dict(name="attention_prefill_16k", kind="attention", dtype="bf16", B=1, H=16, T=16384, D=128, train=False),
        # One short sequence of odd length: launches and latency count.
        dict(name="attention_short_train", kind="attention", dtype="bf16", B=1, H=12, T=197, D=64, train=True),
        # The head of the 1B shape, one training microbatch: the headline configuration.
        dict(name="head_1b_train", kind="head", dtype="bf16", N=16384, d=2048, V=32000, embed="bf16"),
        # The head of the 125M shape with its odd vocabulary.
        dict(name="head_125m_train", kind="head", dtype="bf16", N=8192, d=768, V=50257, embed="bf16"),
        # Single-precision training of the 125M head on one microbatch.
        dict(name="head_125m_f32_train", kind="head", dtype="f32", N=2048, d=768, V=32768, embed="f32"),
        # The model's tail (final norm, then the head) on a small microbatch of odd size, with the
        # embedding kept in f32 as the optimiser keeps it.
        dict(name="tail_350m_small_train", kind="tail", dtype="bf16", N=1000, d=1024, V=32768, embed="f32"),
        # Scoring a few sequences: log-probabilities and greedy tokens, forward only.
        dict(name="head_350m_score", kind="score", dtype="bf16", N=1531, d=1024, V=32768, embed="bf16"),
        # Feed-forward block of the 1B preset, one training microbatch.
        dict(name="ffn_1b_train", kind="ffn", N=16384, d=1536, F=4224, weights="bf16"),
        # Feed-forward block of the 125M preset on one sequence, weights kept in f32.
        dict(name="ffn_125m_small_train", kind="ffn", N=1024, d=768, F=2048, weights="f32"),
    ]


# --- drawn cases ---------------------------------------------------------------------------

def _logint(rng, lo, hi, step=1):
    """A whole number of [lo, hi], uniform over its logarithm, a multiple of `step`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def _fit(value, cost, limit, lo, step=1):
    """`value` lowered (to a multiple of `step`, not under `lo`) until cost(value) <= limit."""
    while value > lo and cost(value) > limit:
        value = max(lo, int(value * 0.8) // step * step)
    return value


def draw(rng):
    kind = rng.choice(["attention", "attention", "layer", "head", "head", "tail", "score", "ffn", "ffn"])
    if kind in ("attention", "layer"):
        f32 = kind == "attention" and rng.random() < 0.25
        D = 64 if f32 else rng.choice([64, 128])
        H = rng.choice([4, 8, 12, 16, 24])
        T = _logint(rng, 48, 2048 if f32 else 4096)
        if rng.random() < 0.5:
            T = max(64, T // 64 * 64)
        limit = 2 * 12 * 1024 ** 2 * 64 if f32 else 8 * 16 * 2048 ** 2 * 128
        B = _fit(_logint(rng, 1, 16), lambda b: b * H * T * T * D, limit, 1)
        T = _fit(T, lambda t: B * H * t * t * D, limit, 48)
        train = kind == "layer" or rng.random() < 0.75
        return dict(kind=kind, dtype="f32" if f32 else "bf16", B=B, H=H, T=T, D=D, train=train)
    if kind == "ffn":
        d = _logint(rng, 512, 2048, 64)
        F = _logint(rng, 1024, 5632, 128)
        N = _fit(_logint(rng, 100, 16384), lambda n: n * d * F, 16384 * 1536 * 4224, 100)
        if rng.random() < 0.5:
            N = max(128, N // 128 * 128)
        return dict(kind=kind, N=N, d=d, F=F, weights=rng.choice(["bf16", "f32"]))
    f32 = kind == "head" and rng.random() < 0.25
    d = _logint(rng, 256, 1024 if f32 else 2048, 64)
    V = rng.choice([4096, 8192, 32000, 32768, 50257, _logint(rng, 4000, 51200)])
    limit = 2048 * 768 * 32768 if f32 else 16384 * 2048 * 32000
    N = _fit(_logint(rng, 100, 4096 if f32 else 16384), lambda n: n * d * V, limit, 100)
    if rng.random() < 0.5:
        N = max(128, N // 128 * 128)
    embed = "f32" if f32 else rng.choice(["bf16", "f32"])
    return dict(kind=kind, dtype="f32" if f32 else "bf16", N=N, d=d, V=V, embed=embed)


# --- inputs ---------------------------------------------------------------------------------

def _randn(seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))
    return g, (lambda *shape: torch.randn(*shape, device=dev, generator=g, dtype=torch.float32))


def _normed(x):
    return x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt()


def prepare(case, seed):
    g, rn = _randn(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind in ("attention", "layer"):
        B, H, T, D = (case[k] for k in "BHTD")
        dt, train = DTYPES[case["dtype"]], case["train"]
        shape = (B, H, T, D) if kind == "attention" else (B, T, H, D)
        q, k, v = rn(*shape), rn(*shape), rn(*shape)
        if kind == "attention":  # the layer normalises its own raw projections
            q, k = _normed(q), _normed(k)
        for name, t in (("q", q), ("k", k), ("v", v)):
            s[name] = t.to(dt).requires_grad_(train)
        s["sink"] = (0.1 * rn(H)).requires_grad_(train)
        if train:
            s["do"] = rn(*shape).to(dt)
        if kind == "layer":
            s["gq"] = (1 + 0.1 * rn(D)).requires_grad_(train)
            s["gk"] = (1 + 0.1 * rn(D)).requires_grad_(train)
            s["cos"], s["sin"] = cayley_table_geometric(D, T, device="cuda")
        return s
    if kind == "ffn":
        N, d, F = case["N"], case["d"], case["F"]
        dt = DTYPES[case["weights"]]
        s["x"] = _normed(rn(N, d)).to(torch.bfloat16).requires_grad_(True)
        for name, a, b in (("wg", d, F), ("wu", d, F), ("wd", F, d)):
            s[name] = (rn(a, b) / math.sqrt(a)).to(dt).requires_grad_(True)
        s["do"] = rn(N, d).to(torch.bfloat16)
        return s
    N, d, V = case["N"], case["d"], case["V"]
    train = kind != "score"
    h = rn(N, d)
    s["h"] = (h if kind == "tail" else _normed(h)).to(DTYPES[case["dtype"]]).requires_grad_(train)
    if kind == "tail":
        s["gain"] = (1 + 0.1 * rn(d)).requires_grad_(True)
    s["E"] = (0.02 * rn(V, d)).to(DTYPES[case["embed"]]).requires_grad_(train)
    s["t"] = torch.randint(0, V, (N,), device=h.device, generator=g, dtype=torch.int32)
    return s


# --- one pass --------------------------------------------------------------------------------

def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind in ("attention", "layer"):
        kw = dict(kind="asinh", n=ATTN_N, c=ATTN_C, block=case["T"], range_guard=True)
        if kind == "attention":
            o = flash_attention(s["q"], s["k"], s["v"], s["sink"], **kw)
            wrt = (s["q"], s["k"], s["v"], s["sink"])
        else:
            o = qk_norm_rotary_flash_attention(s["q"], s["k"], s["v"], s["sink"], s["gq"], s["gk"], s["cos"], s["sin"],
                                               eps=EPS, layout="bthd", **kw)
            wrt = (s["q"], s["k"], s["v"], s["sink"], s["gq"], s["gk"])
        if not case["train"]:
            return [o]
        return [o, *torch.autograd.grad(o, wrt, s["do"])]
    if kind == "ffn":
        y = alu_glu_ffn(s["x"], s["wg"], s["wu"], s["wd"])
        return [y, *torch.autograd.grad(y, (s["x"], s["wg"], s["wu"], s["wd"]), s["do"])]
    if kind == "score":
        return list(head_logprob(s["h"], s["E"], s["t"], n=HEAD_N, c=HEAD_C))
    h, wrt = s["h"], (s["h"], s["E"])
    if kind == "tail":
        h, wrt = rms_norm(h, s["gain"], EPS), (s["h"], s["gain"], s["E"])
    obj, pt = fused_head(h, s["E"], s["t"], kind="alg_ce", n=HEAD_N, c=HEAD_C, block_n=case["N"])
    return [obj, pt, *torch.autograd.grad(obj, wrt)]


# --- what a pass cannot do without ----------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("attention", "layer"):
        B, H, T, D = (case[k] for k in "BHTD")
        size = 2 if case["dtype"] == "bf16" else 4
        fwd = 4.0 * B * H * T * T * D / 2
        # q, k, v in and o out; backward: dO in, dq, dk, dv out.
        tensors = 8 if case["train"] else 4
        return {"bytes": tensors * B * H * T * D * size, "flops": fwd * (3.5 if case["train"] else 1.0)}
    if kind == "ffn":
        N, d, F = case["N"], case["d"], case["F"]
        w = 3 * d * F * (2 if case["weights"] == "bf16" else 4)
        # x, dout in, out, dx out; the weights in and their gradients out.
        return {"bytes": 4 * N * d * 2 + 2 * w, "flops": 3 * 3 * 2.0 * N * d * F}
    N, d, V = case["N"], case["d"], case["V"]
    hb = N * d * (2 if case["dtype"] == "bf16" else 4)
    eb = V * d * (2 if case["embed"] == "bf16" else 4)
    if kind == "score":
        return {"bytes": hb + eb + N * 16, "flops": 2.0 * N * d * V}
    return {"bytes": 2 * hb + 2 * eb + N * 8, "flops": 3 * 2.0 * N * d * V}


def tolerance(case):
    if case.get("dtype") == "f32":
        return {"rel": 1e-5, "max": 1e-3}
    if case["kind"] == "score":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.002}
    return {"rel": 1.5e-2, "max": 0.5}


# --- the same maths in 64 bits ---------------------------------------------------------------

def _f64(t):
    return t.detach().double()


def _attention64(q, k, v, sink, do, rows=1024):
    """Causal attention of one head with weights softmax(n asinh(s / c)) over the keys and the
    sink, and its gradients for the cotangent `do`; blocks of query rows bound the memory."""
    T, D = q.shape
    alpha = 1.0 / (math.sqrt(D) * ATTN_C)
    kt = k.t().contiguous()
    vt = v.t().contiguous()
    o = torch.empty_like(q)
    dq, dk, dv, dsink = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v), torch.zeros_like(sink)
    xb = sink / ATTN_C
    for r0 in range(0, T, rows):
        r1 = min(T, r0 + rows)
        x = (q[r0:r1] @ kt[:, :r1].contiguous()) * alpha
        a = ATTN_N * torch.asinh(x)
        dead = torch.arange(r1, device=q.device)[None, :] > torch.arange(r0, r1, device=q.device)[:, None]
        a.masked_fill_(dead, -math.inf)
        ab = ATTN_N * torch.asinh(xb)
        m = torch.maximum(a.max(-1, keepdim=True).values, ab)
        w = torch.exp(a - m)
        wb = torch.exp(ab - m)
        z = w.sum(-1, keepdim=True) + wb
        p, pb = w / z, wb / z
        o[r0:r1] = p @ v[:r1]
        if do is None:
            continue
        g = do[r0:r1]
        di = (g * o[r0:r1]).sum(-1, keepdim=True)
        ds = p * (g @ vt[:, :r1].contiguous() - di) * ATTN_N * torch.rsqrt(1 + x * x)
        dq[r0:r1] = (ds @ k[:r1]) * alpha
        dk[:r1] += (ds.t().contiguous() @ q[r0:r1]) * alpha
        dv[:r1] += p.t().contiguous() @ g
        dsink += -(pb * di).sum() * ATTN_N * torch.rsqrt(1 + xb * xb) / ATTN_C
    return o, dq, dk, dv, dsink


def _heads64(q, k, v, sink, do):
    B, H = q.shape[:2]
    outs = [torch.empty_like(q) for _ in range(4)]
    dsink = torch.zeros_like(sink)
    for b in range(B):
        for h in range(H):
            got = _attention64(q[b, h], k[b, h], v[b, h], sink[h], None if do is None else do[b, h])
            for out, t in zip(outs, got):
                out[b, h] = t
            dsink[h] += got[4]
    return (*outs, dsink)


def _norm64(x, gain):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gain


def _rotate64(x, cos, sin):
    a, b = x.chunk(2, -1)
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def _cayley64(D, T, device):
    half = D // 2
    w = 0.5 * 10000.0 ** (-torch.arange(half, device=device, dtype=torch.float64) / half)
    angle = 2 * torch.arange(T, device=device, dtype=torch.float64)[:, None] * torch.atan(w)
    return torch.cos(angle), torch.sin(angle)


def _head64(h, E, t):
    z = h @ E.t().contiguous()
    a = HEAD_N * torch.asinh(z / HEAD_C)
    p = torch.softmax(a, -1)
    del a
    N = h.shape[0]
    at = torch.arange(N, device=h.device)
    pt = p[at, t.long()].clone()
    p[at, t.long()] -= 1
    p *= torch.rsqrt(1 + (z / HEAD_C).square_())
    del z
    p *= HEAD_N / HEAD_C / N
    return (1 - pt).mean(), pt, p @ E, p.t().contiguous() @ h


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "attention":
        do = _f64(s["do"]) if case["train"] else None
        got = _heads64(*(_f64(s[n]) for n in ("q", "k", "v", "sink")), do)
        return list(got) if case["train"] else [got[0]]
    if kind == "layer":
        head_first = lambda t: t.permute(0, 2, 1, 3).contiguous()  # noqa: E731
        q, k = (_f64(s[n]).requires_grad_(True) for n in ("q", "k"))
        gq, gk = (_f64(s[n]).requires_grad_(True) for n in ("gq", "gk"))
        cos, sin = _cayley64(case["D"], case["T"], q.device)
        with torch.enable_grad():
            qr, kr = (_rotate64(_norm64(head_first(x), g), cos, sin) for x, g in ((q, gq), (k, gk)))
        o, dqr, dkr, dv, dsink = _heads64(qr.detach(), kr.detach(), head_first(_f64(s["v"])), _f64(s["sink"]),
                                          head_first(_f64(s["do"])))
        dq, dgq = torch.autograd.grad(qr, (q, gq), dqr)
        dk, dgk = torch.autograd.grad(kr, (k, gk), dkr)
        return [head_first(o), dq, dk, head_first(dv), dsink, dgq, dgk]
    if kind == "ffn":
        x, wg, wu, wd = (_f64(s[n]).requires_grad_(True) for n in ("x", "wg", "wu", "wd"))
        with torch.enable_grad():
            up = x @ wu
            bz = 0.5 * up
            y = (x @ wg * (0.5 * up * (1 + bz * torch.rsqrt(1 + bz * bz)))) @ wd
        return [y.detach(), *torch.autograd.grad(y, (x, wg, wu, wd), _f64(s["do"]))]
    E, t = _f64(s["E"]), s["t"]
    if kind == "score":
        z = _f64(s["h"]) @ E.t().contiguous()
        lp = torch.log_softmax(HEAD_N * torch.asinh(z / HEAD_C), -1)
        return [lp[torch.arange(z.shape[0], device=z.device), t.long()], z.argmax(-1)]
    if kind == "head":
        return list(_head64(_f64(s["h"]), E, t))
    x, gain = (_f64(s[n]).requires_grad_(True) for n in ("h", "gain"))
    with torch.enable_grad():
        h = _norm64(x, gain)
    obj, pt, dh, dE = _head64(h.detach(), E, t)
    dx, dgain = torch.autograd.grad(h, (x, gain), dh)
    return [obj, pt, dx, dgain, dE]
