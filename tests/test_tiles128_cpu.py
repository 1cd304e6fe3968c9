"""When a 256x256 plan runs on 128x128 ring tiles (TX_FLAG_TILES_128).

The flag changes neither the plan's block nor its workspace; it is set where
the 256x256 tiles leave CUs idle and the split that fills them costs more than
the smaller tile, and never on a block asked for.
"""
import ctypes

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


@pytest.mark.parametrize("M,N,K,t", [
    (128, 16384, 262112, tx.F4E2M1), (128, 1048576, 4064, tx.F4E2M1),  # 131056 / 2032 packed rows
    (128, 2097152, 2016, tx.F4E2M1), (65, 2097152, 1952, tx.F4E2M1),
    (128, 1048576, 2016, tx.F8E4M3), (128, 2097152, 992, tx.F8E5M2),
])
def test_wide_mx_plans(M, N, K, t):
    """The planner and the launch layer hold the ring tiles to one bound, 128 rows of B past K
    within 2^32 bytes (e2m1: packed rows, K / 2 of them): what the planner chooses is planned."""
    k = 256 if t == tx.F4E2M1 else 128
    p = tx.plan(tx.make_desc(M, N, K, t, tx.F32, scale_mode=tx.SCALE_MX32))
    assert (p.desc.block_m, p.desc.block_n, p.desc.block_k) == (256, 256, k)
    if not tx.load().tx_device_available():  # the launch's own checks accept it (dummy pointers)
        a = ctypes.c_void_p(1 << 20)
        assert tx.load().tx_dot_launch(ctypes.byref(p), a, a, a, a, a, a, p.workspace_bytes,
                                       None) == tx.ERR_NO_DEVICE


@pytest.mark.parametrize("K,ld,ok", [
    (128, (1 << 24) - 16, True),   # 255 rows of B, of 2^24 - 16 bytes: below 2^32
    (127, 1 << 24, True),          # 255 rows of 2^24
    (128, 1 << 24, False),         # 256 of them
])
def test_ring_bound(K, ld, ok):
    d = tx.make_desc(300, 512, K, tx.F8E4M3, tx.F32, block=(256, 256, 128), ldb=ld, ldc=512,
                     lda=128, flags=capi.FLAG_TILES_128)
    p = capi.DotPlan()
    rc = tx.load().tx_dot_plan_create(ctypes.byref(d), ctypes.byref(p))
    assert rc == (tx.OK if ok else tx.ERR_UNSUPPORTED)
    # left to itself the planner takes the 256x256 tile past the bound
    d = tx.make_desc(300, 512, K, tx.F8E4M3, tx.F32, ldb=ld, ldc=512, lda=128)
    p = tx.plan(d)
    assert ok or not p.desc.flags & capi.FLAG_TILES_128


def test_ring_group_m():
    """plan.group_m is what the launch takes: 4 tile rows on the ring tiles whatever K, 2 on the
    8-bit 256x256 tile once K spans 8192 bytes."""
    for block, gm in (((0, 0, 0), 4), ((256, 256, 128), 2)):
        p = tx.plan(tx.make_desc(512, 8192, 8192, tx.I8, tx.BF16, scale_mode=tx.SCALE_ROWCOL,
                                 block=block))
        assert bool(p.desc.flags & capi.FLAG_TILES_128) == (gm == 4) and p.group_m == gm
