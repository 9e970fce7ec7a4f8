"""quantize_acts with four elements per lane (16-byte aligned rows) and one
element per lane (any alignment) against the oracle (matmul.rs:105-127): part
workgroups, ties, zero, subnormal and non-finite blocks."""
import ctypes as C

import numpy as np
import pytest

import prana_amd as P
from oracle import oracle as O
from prana_amd import check, load

pytestmark = pytest.mark.gpu


def values(n, k):
    x = np.random.default_rng(n * 31 + k).standard_normal((n, k)).astype(np.float32)
    x[0, :32] = 0.0
    x[-1, -32:] = np.arange(32, dtype=np.float32) * 0.5      # halves of a step
    x[-1, -1] = 63.5
    if k > 96:
        x[0, 32:64] *= 1e-41
        x[0, 64], x[0, 70], x[0, 96] = np.inf, np.nan, 3e38
    return x


@pytest.mark.parametrize("n,k", [(1, 32), (1, 96), (1, 1024), (3, 1056), (7, 4864), (33, 288)])
@pytest.mark.parametrize("shift", [0, 1])
def test_quantize_acts_alignments(n, k, shift):
    x = values(n, k)
    buf = P.DeviceArray.from_host(np.concatenate([np.zeros(shift, np.float32), x.ravel()]))
    q, s, m = P.DeviceArray((n * k,), np.int8), P.DeviceArray((n * k // 32,), np.float32), P.DeviceArray((n * k // 32,),
                                                                                                       np.int32)
    check(load().prana_quantize_acts(C.c_void_p(buf.ptr.value + 4 * shift), n, k, q.ptr, s.ptr, m.ptr, None))
    wq, ws, wm = (np.concatenate([np.ravel(a) for a in p]) for p in zip(*[O.quantize_acts(r) for r in x]))
    sc = s.to_host()
    assert np.array_equal(q.to_host(), wq) and np.array_equal(m.to_host(), wm)
    assert np.array_equal(np.isnan(sc), np.isnan(ws)) and np.array_equal(sc[~np.isnan(ws)], ws[~np.isnan(ws)])
