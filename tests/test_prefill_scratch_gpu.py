"""Device memory of a prefill attention: the score rows of the kernel that takes
the shape and no more (32 heads x 5000 positions on the tiled kernel 1.0 GB,
where the one-launch kernel's rows are 3.2; 256-wide heads run 32-row blocks in
512 slots)."""
import numpy as np
import pytest
import torch

import prana_amd as P
from oracle import oracle as O
from prana_amd import models as M

pytestmark = pytest.mark.gpu

STRIDE = 256  # score rows are padded to whole tiles of keys


@pytest.mark.parametrize("seq,nh,nkv,hd,slot_rows", [(5000, 32, 32, 4, 768 * 64), (2048, 32, 2, 256, 512 * 32)])
def test_prefill_scratch_is_the_kernels_own(seq, nh, nkv, hd, slot_rows):
    g = P.Graph()
    q, k, v = (g.input(seq) for _ in range(3))
    g.attention(q, k, v, nh, nkv, hd)
    for node, heads in ((q, nh), (k, nkv), (v, nkv)):
        g.set_input(node, np.zeros((seq, heads * hd), np.float32))
    free = torch.cuda.mem_get_info()[0]
    g.execute()
    taken = free - torch.cuda.mem_get_info()[0]
    want = 4 * (slot_rows * -(-seq // STRIDE) * STRIDE + seq * nh * hd)
    assert want // 2 < taken < want + (32 << 20), (taken, want)  # (allocations come in pages of a few MiB)


def leave_little_memory():
    """Buffers that leave about 200 MB of the card's memory."""
    torch.cuda.empty_cache()
    piece = 64 << 20
    held = []
    try:
        # (the free memory that is reported and what can be allocated differ by a few pieces)
        held.append(P.DeviceArray((torch.cuda.mem_get_info()[0] - 2 * piece,), np.uint8))
        for _ in range(64):
            held.append(P.DeviceArray((piece,), np.uint8))
    except P.PranaError:
        pass
    if not 4 < len(held) < 65:
        pytest.skip("free memory of this card cannot be narrowed down")
    return held[:-3]


def test_prefill_without_room_for_scratch():
    # 403 MB of score rows with about 200 MB left: the window runs without
    seq, nh, nkv, hd = 2048, 32, 32, 4
    r = np.random.default_rng(3)
    host = [r.standard_normal((seq, n * hd)).astype(np.float32) for n in (nh, nkv, nkv)]
    g = P.Graph()
    nodes = [g.input(seq) for _ in range(3)]
    out = g.attention(*nodes, nh, nkv, hd)
    for node, a in zip(nodes, host):
        g.set_input(node, a)
    held = leave_little_memory()
    try:
        g.execute()
    finally:
        held.clear()
    got = np.asarray(g.output_f32(out), np.float32)
    want = O.attention(*(a.ravel() for a in host), seq, nh, nkv, hd)
    assert np.array_equal(got.ravel().view(np.uint32), np.asarray(want, np.float32).ravel().view(np.uint32))


def test_model_runs_on_after_a_batch_that_does_not_fit():
    # a prompt whose logits (1.2 GB) do not fit is refused, and the next call
    # finds its buffers again
    cfg = M.config(64, 96, 1, 2, 2, 100000, 3000, head_dim=32)
    t = M.synth_tensors(cfg, lambda name, cols: P.Q8_0, 9)
    g, o = P.Model(cfg, t), O.Model(cfg, t)
    gc, oc = g.cache(3000), o.cache(3000)
    assert np.array_equal(gc.forward(5, 0), oc.forward(5, 0))
    held = leave_little_memory()
    try:
        with pytest.raises(P.PranaError) as e:
            gc.prefill(np.zeros(3000, np.uint32))
        assert e.value.code == -3  # PRANA_ERR_NOMEM
        assert np.array_equal(gc.forward(7, 1), oc.forward(7, 1))
    finally:
        held.clear()
