"""Tiled prefill attention (prefill_attention.hip) against the oracle's
`attention` (attention.rs:236-284), bit for bit: block and tile edges (16 / 32 / 64
query rows, 128 / 256 keys), head widths that fill a lane tile or leave part
of it empty, several blocks per workgroup, and non-finite K and V rows."""
import ctypes as C

import numpy as np
import pytest

import prana_amd as P
from oracle import oracle as O
from prana_amd import check, load
from prana_amd import models as M

pytestmark = pytest.mark.gpu


def same_bits(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))


def qkv(seq, nh, nkv, hd):
    r = np.random.default_rng(seq * 1000 + hd)
    return [r.standard_normal(seq * n * hd).astype(np.float32) for n in (nh, nkv, nkv)]


# (seq, query heads, KV heads, head width), by query rows per block: 16 (the
# first group; lane tiles filled or partly empty, edges of 16 rows, 64-key
# groups and 256-key tiles), 32 (from 640 such blocks, compiled for three
# workgroups per compute unit from 1000), 64 (from 1024)
@pytest.mark.parametrize("seq,nh,nkv,hd", [
    (16, 44, 4, 64), (17, 48, 48, 4), (63, 16, 2, 128), (65, 12, 6, 48), (129, 8, 1, 20), (257, 5, 5, 256),
    (200, 5, 5, 80), (255, 3, 1, 96), (256, 8, 8, 100), (300, 4, 1, 132), (1000, 14, 2, 64),
    (350, 64, 8, 64), (321, 64, 16, 128), (319, 64, 64, 8), (330, 60, 4, 160),
    (350, 96, 8, 48), (340, 96, 12, 72),
    (513, 128, 8, 64), (520, 128, 16, 72), (1025, 64, 8, 12)])
def test_prefill_tile(seq, nh, nkv, hd):
    q, k, v = qkv(seq, nh, nkv, hd)
    assert same_bits(P.attention_prefill(q, k, v, seq, nh, nkv, hd), O.attention(q, k, v, seq, nh, nkv, hd))


def block_rows(seq, nh, hd):
    """Query rows per block of the tiled kernel, and its workgroups per compute unit (pt_plan)."""
    jobs = lambda bq: -(-seq // bq) * nh
    bq = 64 if jobs(64) >= 1024 else 32 if jobs(32) >= 640 else 16
    if bq == 64 and hd > 128:
        bq = 32
    if bq == 16:
        return bq, 3
    return bq, 3 if hd <= (64 if bq == 64 else 128) and jobs(bq) >= 1000 else 2


# both sides of the row count from which a shape takes the tiled kernel
@pytest.mark.parametrize("seq,nh,nkv,hd", [
    (2099, 1, 1, 32), (2100, 1, 1, 32), (725, 2, 1, 16), (724, 2, 1, 16), (58, 18, 6, 48), (57, 18, 6, 48),
    (400, 4, 1, 36), (260, 4, 4, 64), (280, 5, 5, 80), (279, 5, 5, 80), (255, 6, 2, 96), (180, 6, 1, 112), (179, 6, 1, 112),
    (180, 6, 2, 128), (179, 6, 2, 128), (138, 8, 8, 256), (137, 8, 8, 256)])
def test_prefill_line(seq, nh, nkv, hd):
    test_prefill_tile(seq, nh, nkv, hd)


# few heads over windows of up to 2048 positions: pairs of 8-row blocks
# (attention.hip), the middle block of an odd count taken once, a part block at
# the end; the first and last window of each width's range, and the tiled
# kernel on the other side of each line
@pytest.mark.parametrize("seq,nh,nkv,hd", [
    (950, 1, 1, 128), (949, 1, 1, 128), (594, 2, 1, 128), (593, 2, 1, 128), (699, 4, 2, 128), (1024, 8, 8, 128), (1025, 3, 1, 128), (2048, 4, 2, 128),
    (1025, 1, 1, 64), (1024, 2, 1, 64), (1500, 4, 2, 64), (2041, 3, 3, 64), (2048, 4, 1, 64), (2049, 2, 2, 64),
    (1200, 7, 7, 64)])
def test_prefill_few_heads(seq, nh, nkv, hd):
    test_prefill_tile(seq, nh, nkv, hd)


# v at any f32 address runs the same kernel as an aligned one (its slots of
# scratch), with the same bits; q or k off 16 bytes runs the one-launch kernel
@pytest.mark.parametrize("seq,nh,nkv,hd", [(350, 6, 2, 128), (320, 128, 16, 64), (129, 8, 1, 20), (300, 4, 1, 132),
                                            (1200, 2, 1, 64)])
@pytest.mark.parametrize("shift", [(0, 0, 1), (0, 0, 2), (0, 0, 3), (1, 0, 0), (0, 3, 0)])
def test_prefill_unaligned(seq, nh, nkv, hd, shift):
    host = qkv(seq, nh, nkv, hd)
    d = [P.DeviceArray.from_host(np.concatenate([np.zeros(s, np.float32), a])) for s, a in zip(shift, host)]
    out = P.DeviceArray((seq * nh * hd,), np.float32)
    check(load().prana_attention_prefill(*[C.c_void_p(a.ptr.value + 4 * s) for s, a in zip(shift, d)], seq, nh, nkv,
                                         hd, out.ptr, None))
    assert same_bits(out.to_host(), O.attention(*host, seq, nh, nkv, hd).ravel())


def test_prefill_tile_nonfinite():
    # a key's infinite or NaN row must not reach the rows before it, whose
    # products never include it
    seq, nh, nkv, hd = 150, 6, 1, 64
    q, k, v = qkv(seq, nh, nkv, hd)
    v = v.reshape(seq, hd)
    v[40, 3], v[70, 5], v[100, 7] = np.inf, np.nan, -np.inf
    k = k.reshape(seq, hd)
    k[120] = np.nan
    k[130, 0] = np.inf
    got = P.attention_prefill(q, k, v, seq, nh, nkv, hd)
    want = O.attention(q, k.ravel(), v.ravel(), seq, nh, nkv, hd)
    gn, wn = np.isnan(got), np.isnan(want)
    assert np.array_equal(gn, wn)  # NaN payloads are not part of the contract
    assert np.array_equal(got[~gn].view(np.uint32), want[~wn].view(np.uint32))


@pytest.mark.parametrize("seq,nh,hd,rows", [(350, 64, 64, 32), (140, 256, 128, 32), (330, 64, 160, 32),
                                             (193, 256, 64, 64), (193, 256, 128, 64)])
def test_prefill_tile_nonfinite_larger_blocks(seq, nh, hd, rows):
    assert block_rows(seq, nh, hd)[0] == rows
    q, k, v = qkv(seq, nh, 1, hd)
    v = v.reshape(seq, hd)
    v[40, 3], v[70, 5], v[100, hd - 1] = np.inf, np.nan, -np.inf
    k = k.reshape(seq, hd)
    k[120] = np.nan
    k[130, 0] = np.inf
    got = P.attention_prefill(q, k, v, seq, nh, 1, hd)
    want = O.attention(q, k.ravel(), v.ravel(), seq, nh, 1, hd)
    gn, wn = np.isnan(got), np.isnan(want)
    assert np.array_equal(gn, wn)
    assert np.array_equal(got[~gn].view(np.uint32), want[~wn].view(np.uint32))


# the int8 copy of the output that wo reads (head widths of whole 32-blocks),
# from every block size, width and workgroup count: the second layer's K and V
# rows hold what the first layer's attention gave
@pytest.mark.parametrize("seq,nh,nkv,hd,plan", [
    (100, 12, 4, 96, (16, 3)), (40, 64, 8, 128, (16, 3)), (50, 32, 4, 160, (16, 3)), (50, 32, 4, 224, (16, 3)),
    (350, 64, 8, 64, (32, 2)), (70, 256, 16, 128, (32, 2)), (350, 96, 8, 96, (32, 3)), (140, 256, 16, 64, (32, 3)),
    (129, 256, 16, 128, (32, 3)), (330, 64, 8, 160, (32, 2)), (321, 64, 4, 224, (32, 2)), (197, 160, 8, 256, (32, 2)),
    (193, 256, 16, 32, (64, 3)), (193, 256, 16, 64, (64, 3)), (193, 256, 16, 128, (64, 2)), (200, 256, 8, 96, (64, 2))])
def test_prefill_tile_quantized_output(seq, nh, nkv, hd, plan):
    assert block_rows(seq, nh, hd) == plan
    cfg = M.config(64, 96, 2, nh, nkv, 96, seq + 1, head_dim=hd)
    t = M.synth_tensors(cfg, lambda name, cols: P.Q8_0, 5)
    gc, oc = P.Model(cfg, t).cache(seq), O.Model(cfg, t).cache(seq)
    prompt = np.random.default_rng(seq).integers(0, cfg["vocab_size"], seq).astype(np.uint32)
    gc.prefill(prompt)
    oc.prefill(prompt)
    for which in (0, 1):
        assert np.array_equal(gc.read(1, which, seq), oc.read(1, which, seq)), which
