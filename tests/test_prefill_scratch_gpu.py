"""Device memory of a prefill attention: the score rows of the kernel that takes
the shape and no more (32 heads x 5000 positions on the tiled kernel 1.0 GB,
where the one-launch kernel's rows are 3.2; 256-wide heads run 32-row blocks in
512 slots)."""
import numpy as np
import pytest
import torch

import prana_amd as P

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
