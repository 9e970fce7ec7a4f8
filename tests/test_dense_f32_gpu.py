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


# groups of eight tokens (few tiles), and 32- and 64-token tiles of one chunk or two
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


def narrow(rows, cols, n):
    """Whether a lane per class and row takes the call, without staging (narrow_takes)."""
    if n == 1 and rows >= 16000 and cols <= (200 if rows >= 24000 else 140):
        return True
    if n == 2 and 16000 <= rows <= 40000 and cols <= 110:
        return True
    most = ((3600000 if n <= 16 else 2000000) if cols < 4 else 26000000 if cols <= 17
            else (15000000 if n <= 16 else 9000000) if cols <= 24 else 6000000 if n <= 4 else 3200000 if rows > 5000 else 4000000 if rows < 1000
            else 13500000 if cols <= 56 else 6000000)
    return cols < 96 and rows * n * (cols + 4) <= most


# narrow matrices over many rows, both sides of the line: last row groups part
# filled, a tail of 1-3 columns and none, activations 4 bytes off
@pytest.mark.parametrize("rows,cols,n,taken", [(24001, 200, 1, True), (24001, 201, 1, False), (16001, 110, 2, True),
                                               (16001, 111, 2, False), (10007, 3, 28, True), (20011, 2, 33, False),
                                               (9001, 17, 137, True), (9001, 17, 138, False), (33001, 24, 16, True),
                                               (1003, 56, 224, True), (1003, 56, 225, False), (5001, 26, 21, True),
                                               (5001, 26, 22, False), (1003, 95, 20, True), (1003, 96, 20, False)])
@pytest.mark.parametrize("shift", [0, 1])
def test_dense_narrow(rows, cols, n, taken, shift):
    assert narrow(rows, cols, n) == taken
    w, x = make(rows, cols, n)
    w[rows // 2, 0], x[0, cols - 1] = -0.0, -0.0
    raw = w.view(np.uint8)
    buf = P.DeviceArray.from_host(np.concatenate([np.zeros(shift, np.float32), x.ravel()]))
    out = P.DeviceArray((n, rows), np.float32)
    m = P.Matrix(P.F32, rows, cols, raw)
    check(load().prana_matmul(m.h, C.c_void_p(buf.ptr.value + 4 * shift), n, out.ptr, None))
    assert same_bits(out.to_host(), O.Mat.from_ggml(P.F32, rows, cols, raw).apply(x))


def batch_tile(rows, n):
    """Tokens per tile of the batch kernel, 0 where groups of eight tokens run instead (launch_dense)."""
    jobs = lambda tt: -(-rows // 64) * -(-n // tt)  # (rows of 96 columns and more)
    if n <= 16 or jobs(16) < 400:
        return 0
    return 64 if jobs(64) >= 512 else 32 if jobs(32) >= 512 else 16


# every tile of the batch kernel over five and more chunks of 64 columns (both
# staging buffers are reused): rows of any and of whole 16-byte words, with a
# tail of 1-3 columns and without, and whole words 4 bytes off
@pytest.mark.parametrize("rows,cols,n,tile", [(2048, 389, 301, 16), (2048, 388, 301, 16), (2049, 325, 481, 32),
                                              (2049, 324, 481, 32), (4100, 323, 515, 64), (4100, 320, 515, 64)])
@pytest.mark.parametrize("shift", [0, 1])
def test_dense_batch_tiles(rows, cols, n, tile, shift):
    assert batch_tile(rows, n) == tile
    w, x = make(rows, cols, n)
    raw = w.view(np.uint8)
    buf = P.DeviceArray.from_host(np.concatenate([np.zeros(shift, np.float32), x.ravel()]))
    out = P.DeviceArray((n, rows), np.float32)
    m = P.Matrix(P.F32, rows, cols, raw)
    check(load().prana_matmul(m.h, C.c_void_p(buf.ptr.value + 4 * shift), n, out.ptr, None))
    assert same_bits(out.to_host(), O.Mat.from_ggml(P.F32, rows, cols, raw).apply(x))
