"""CPU: which tiles the feed-forward's and the head's products take. Each line is a size at which both
forms were timed on an MI355X (us), so that a rule that is fitted again cannot go back to the slower
one unseen."""

import ctypes

import pytest


def plan(kind, *args):
    from algebraic_amd import _lib
    tile, split = ctypes.c_int(), ctypes.c_int()
    lib = _lib.load()
    fn = lib.alg_ffn_plan if kind == "ffn" else lib.alg_head_plan
    assert fn(*args, ctypes.byref(tile), ctypes.byref(split)) == _lib.ALG_OK
    return tile.value, split.value


# product, M, N, K (gate/up and dy: N = d_ff), tile, us on that tile, us on the other one
FFN = [
    ("GATE_UP", 512, 4096, 1024, 128, 17.6, 28.7),
    ("GATE_UP", 300, 2816, 1024, 128, 26.5, 33.6),
    ("GATE_UP", 2048, 1408, 512, 128, 20.4, 22.0),
    ("GATE_UP", 6528, 1280, 960, 128, 51.9, 63.5),
    ("GATE_UP", 400, 5632, 2048, 256, 56.8, 88.9),
    ("GATE_UP", 1000, 2816, 1024, 256, 36.2, 39.9),
    ("GATE_UP", 3500, 2816, 1024, 256, 66.8, 119.7),
    ("GATE_UP", 16384, 4224, 1536, 256, None, None),
    ("DY", 1500, 2816, 1024, 64, 27.7, 41.6),
    ("DY", 2500, 2048, 768, 64, 25.3, 36.2),
    ("DY", 1300, 5632, 2048, 256, 54.9, 62.1),
    ("DY", 4096, 2816, 1024, 256, 43.7, 47.3),
    ("GEMM", 1024, 8192, 300, 256, 18.6, 23.0),
    ("GEMM", 1536, 8448, 197, 256, 20.5, 28.2),
    ("GEMM", 5632, 2048, 300, 256, 19.0, 25.9),
    ("GEMM", 4096, 1024, 3500, 128, 38.2, 45.3),
    ("GEMM", 512, 1536, 8448, 64, 28.8, 37.9),
]


@pytest.mark.parametrize("product,M,N,K,tile,us,other", FFN)
def test_ffn_tile(product, M, N, K, tile, us, other):
    from algebraic_amd import _lib
    assert plan("ffn", getattr(_lib, "FFN_" + product), M, N, K)[0] == tile


# dtype, product, N, d, V, tile, us on that tile, us on the other one (with its best split)
HEAD = [
    ("BF16", "DH", 2500, 1536, 8192, 256, 87.3, 125.4),
    ("BF16", "DH", 700, 1536, 8192, 256, 56.2, 76.9),
    ("BF16", "DH", 300, 2048, 16384, 256, 61.7, 76.9),
    ("BF16", "DH", 512, 512, 8192, 128, 33.9, 46.2),
    ("BF16", "DH", 127, 72, 129, 128, None, None),  # a vocabulary shorter than a range keeps the choice
    ("BF16", "DH", 128, 1024, 32000, 128, 44.4, 76.7),
    ("BF16", "DE", 200, 256, 50257, 256, 22.7, 35.1),
    ("BF16", "DE", 300, 768, 16384, 256, 21.1, 27.3),
    ("BF16", "DE", 100, 896, 8192, 128, 15.0, 21.4),
    ("F32", "DE", 300, 768, 8192, 256, 58.7, 69.4),
    ("BF16", "LOGITS", 128, 1024, 32768, 128, 23, 37),
    ("BF16", "LOGITS", 200, 2048, 32000, 256, 59, 74),
]


@pytest.mark.parametrize("dtype,product,N,d,V,tile,us,other", HEAD)
def test_head_tile(dtype, product, N, d, V, tile, us, other):
    from algebraic_amd import _lib
    assert plan("head", getattr(_lib, "DTYPE_" + dtype), getattr(_lib, "HEAD_" + product), N, d, V)[0] == tile


def test_plan_queries_refuse_bad_arguments():
    from algebraic_amd import _lib
    lib = _lib.load()
    a, b = ctypes.c_int(), ctypes.c_int()
    assert lib.alg_ffn_plan(3, 64, 64, 64, a, b) == _lib.ALG_ERR_INVALID
    assert lib.alg_ffn_plan(0, 64, 0, 64, a, b) == _lib.ALG_ERR_INVALID
    assert lib.alg_ffn_plan(0, 64, 64, 64, None, b) == _lib.ALG_ERR_INVALID
    assert lib.alg_head_plan(7, 0, 64, 64, 64, a, b) == _lib.ALG_ERR_INVALID
    assert lib.alg_head_plan(0, 3, 64, 64, 64, a, b) == _lib.ALG_ERR_INVALID
    assert plan("head", _lib.DTYPE_F32, _lib.HEAD_DH, 255, 64, 4096)[0] == 0  # the f32 kernels
