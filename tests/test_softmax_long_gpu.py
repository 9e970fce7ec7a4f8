"""Chunked softmax over long rows (softmax.hip) against the oracle's softmax
(norms.rs:44-56), bit for bit: chunk edges, several rows, sums whose rounding
drifts away from the predicted binades (terms below half a unit of the sum),
ties, subnormal terms, non-finite rows, and in-place calls."""
import numpy as np
import pytest

import prana_amd as P
from oracle import oracle as O
from prana_amd import check, load

pytestmark = pytest.mark.gpu


def same(got, want):
    got, want = np.asarray(got, np.float32).ravel(), np.asarray(want, np.float32).ravel()
    gn, wn = np.isnan(got), np.isnan(want)
    return np.array_equal(gn, wn) and np.array_equal(got[~gn].view(np.uint32), want[~wn].view(np.uint32))


def rows_like(kind, rows, n):
    r = np.random.default_rng(n + rows)
    x = r.standard_normal((rows, n)).astype(np.float32)
    if kind == "flat":            # every term 1: ties once the sum passes 2^24 / n steps of an odd grid
        x[:] = 0.25
    elif kind == "peak":          # one large term, the rest below half a unit of the sum
        x -= 19.0
        x[:, 5] = 0.0
    elif kind == "late":          # nothing until the last chunk
        x -= 60.0
        x[:, -3:] = 1.0
    elif kind == "ramp":          # the sum doubles every few hundred terms
        x[:] = np.linspace(-90.0, 0.0, n, dtype=np.float32)
    elif kind == "subnormal":
        x[:] = -95.0 - np.abs(x)
        x[:, 0] = 0.0
    elif kind == "wide":
        x *= 12.0
    return x


@pytest.mark.parametrize("kind", ["normal", "flat", "peak", "late", "ramp", "subnormal", "wide"])
@pytest.mark.parametrize("rows,n", [(1, 7168), (3, 7169), (2, 9217), (1, 32000), (1, 151936)])
def test_softmax_long(kind, rows, n):
    x = rows_like(kind, rows, n)
    got = P.softmax(x)
    for i in range(rows):
        assert same(got[i], O.softmax(x[i])), (kind, i)


# the last row count of each range on the chunked launches, and the next one on
# a workgroup per row
@pytest.mark.parametrize("rows,n", [(64, 7168), (65, 7999), (96, 8000), (97, 9999), (192, 10000), (193, 11999),
                                    (768, 12000), (769, 12999), (769, 13000)])
def test_softmax_row_counts(rows, n):
    x = rows_like("normal", rows, n)
    x[rows // 2] = rows_like("ramp", 1, n)
    got = P.softmax(x)
    for i in (0, 1, rows // 2, rows - 2, rows - 1):
        assert same(got[i], O.softmax(x[i])), i
    assert np.all(np.abs(got.sum(1, dtype=np.float64) - 1) < 1e-4)  # every row was written (the 32-bit sum drifts by < 3e-9 n)


def test_softmax_long_many_rows_and_past_2_24():
    x = rows_like("normal", 70, 7500)
    got = P.softmax(x)
    assert all(same(g, O.softmax(v)) for g, v in zip(got, x))
    flat = np.zeros(17_000_001, np.float32)  # the sum stops growing at 2^24
    assert same(P.softmax(flat)[0], O.softmax(flat))


# 1000 and 1001 chunks: the row's maximum and the sums before each chunk from
# every chunk's workgroup, and from launches of their own (a full and a part
# round of 1024 chunks)
@pytest.mark.parametrize("rows,n", [(1, 1024000), (2, 1024001), (1, 1048577), (2, 1100003)])
@pytest.mark.parametrize("kind", ["normal", "peak", "late", "ramp", "wide", "nonfinite"])
def test_softmax_many_chunks(kind, rows, n):
    x = rows_like(kind, rows, n)
    if kind == "nonfinite":
        x[0, n // 2] = np.nan
        x[-1, : n - 700] = -np.inf
    got = P.softmax(x)
    for i in range(rows):
        assert same(got[i], O.softmax(x[i])), (kind, i)


def test_softmax_long_nonfinite_and_in_place():
    x = rows_like("normal", 5, 9000)
    x[0, 4000] = np.nan
    x[1, 8000] = np.inf
    x[2, :4500] = -np.inf
    x[3, :] = -np.inf
    got = P.softmax(x)
    for i in range(5):
        assert same(got[i], O.softmax(x[i])), i
    d = P.DeviceArray.from_host(x[4])
    check(load().prana_softmax(d.ptr, 1, 9000, d.ptr, None))
    assert same(d.to_host(), O.softmax(x[4]))
