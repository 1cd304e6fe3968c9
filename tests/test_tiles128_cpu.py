"""When a 256x256 plan runs on 128x128 ring tiles (TX_FLAG_TILES_128).

The flag changes neither the plan's block nor its workspace; it is set where
the 256x256 tiles leave CUs idle and the split that fills them costs more than
the smaller tile, and never on a block asked for.
"""
import pytest

import triton_ext_amd as tx
from triton_ext_amd import capi


@pytest.mark.parametrize("M,N,K,t,mode,c,ring", [
    (1000, 4000, 4000, tx.BF16, tx.SCALE_NONE, tx.BF16, True),     # 38 us against 52
    (512, 8192, 8192, tx.I8, tx.SCALE_ROWCOL, tx.BF16, True),      # 40 / 55
    (1280, 3200, 1024, tx.F8E4M3, tx.SCALE_MX32, tx.F32, True),    # 12.7 / 19.6
    (2048, 2800, 8192, tx.F8E4M3, tx.SCALE_NONE, tx.F32, False),   # 70.9 / 63.0: two rounds
    (1792, 3584, 4096, tx.BF16, tx.SCALE_NONE, tx.BF16, False),    # 68.6 / 66.6
    (2048, 2800, 8192, tx.F4E2M1, tx.SCALE_MX32, tx.F32, False),   # 65.9 / 61.2
    (4096, 4096, 4096, tx.BF16, tx.SCALE_NONE, tx.BF16, False),    # 256 tiles fill the chip
])
def test_choice(M, N, K, t, mode, c, ring):
    k = 64 if t == tx.BF16 else 256 if t == tx.F4E2M1 else 128
    p = tx.plan(tx.make_desc(M, N, K, t, c, scale_mode=mode))
    assert (p.desc.block_m, p.desc.block_n, p.desc.block_k) == (256, 256, k)
    assert bool(p.desc.flags & capi.FLAG_TILES_128) == ring
    q = tx.plan(tx.make_desc(M, N, K, t, c, scale_mode=mode, block=(256, 256, k)))
    assert not q.desc.flags & capi.FLAG_TILES_128
    assert q.grid_x == p.grid_x and q.block_threads == p.block_threads
