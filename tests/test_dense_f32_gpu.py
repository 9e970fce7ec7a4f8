"""Dense f32 matrices (dense.hip) against the oracle's matmul_f32
(matmul.rs:150-157, 377-391), bit for bit: column counts around the four-way
chains, the chunks of 64 and 256 elements and a tail, row and token tile
edges, unaligned activations, and non-finite values."""
import ctypes as C

import numpy as np
import pytest

import prana_amd as P
from oracle import oracle as O
from prana_amd import check, load

pytestmark = pytest.mark.gpu


def same_bits(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))


def make(rows, cols, n):
    r = np.random.default_rng(rows * 7 + cols * 3 + n)
    return r.standard_normal((rows, cols)).astype(np.float32), r.standard_normal((n, cols)).astype(np.float32)


@pytest.mark.parametrize("n", [1, 2, 4, 5, 8, 9, 16, 17, 31, 33])
@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 3), (17, 4), (15, 7), (16, 64), (65, 63), (64, 256), (130, 257),
                                       (33, 260), (100, 1028), (48, 1535)])
def test_dense_shapes(rows, cols, n):
    w, x = make(rows, cols, n)
    raw = w.view(np.uint8)
    assert same_bits(P.Matrix(P.F32, rows, cols, raw).apply(x), O.Mat.from_ggml(P.F32, rows, cols, raw).apply(x))


# 16-, 32- and 64-token tiles
@pytest.mark.parametrize("rows,cols,n", [(640, 96, 67), (2049, 68, 481), (4100, 36, 515)])
def test_dense_batches(rows, cols, n):
    test_dense_shapes(rows, cols, n)


def test_dense_unaligned_activations_and_residual_zero_signs():
    rows, cols, n = 70, 132, 20
    w, x = make(rows, cols, n)
    w[3] = -0.0
    x[5] = 0.0
    w[9, 11], w[10, 12], x[7, 40] = np.inf, -np.inf, 3e38
    raw = w.view(np.uint8)
    m, want = P.Matrix(P.F32, rows, cols, raw), O.Mat.from_ggml(P.F32, rows, cols, raw).apply(x)
    for k in (3, n):
        buf = P.DeviceArray.from_host(np.concatenate([np.zeros(1, np.float32), x[:k].ravel()]))
        out = P.DeviceArray((k, rows), np.float32)
        check(load().prana_matmul(m.h, C.c_void_p(buf.ptr.value + 4), k, out.ptr, None))
        got = out.to_host()
        nan = np.isnan(want[:k])
        assert np.array_equal(np.isnan(got), nan)
        assert same_bits(got[~nan], want[:k][~nan])
