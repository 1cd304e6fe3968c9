"""GPU parity of the MX decode kernels (dot_scaled with a few rows of A) against the oracle.

MX x MX (decode_f8.h's MX form): the scaled MFMA's own bound (test_mx_gpu.check_mx).
Shapes sit at the edges: slices of 16 .. 64 rows, N and K that fill no strip
or batch, scale rows that start at every byte of a dword, split K, and more than one
segment of staged scales (K past 4096 in one split).
"""
import numpy as np
import pytest

import triton_ext_amd as tx
from dotcase import say, to_device
from test_mx_gpu import check_mx, mx_case, ref_of, run_gpu

pytestmark = pytest.mark.gpu


def _plan(M, N, K, a, b, sm=tx.SCALE_MX32):
    r = lambda x, q: -(-x // q) * q
    return tx.plan(tx.make_desc(M, N, K, a, tx.F32, b_type=b, lda=r(K, 32), ldb=r(N, 16),
                                ldc=r(N, 4), scale_mode=sm))


@pytest.mark.parametrize("fa,fb", [("e4m3", "e4m3"), ("e5m2", "e4m3"), ("e4m3", "e5m2"),
                                   ("e2m1", "e2m1")])
@pytest.mark.parametrize("M,N,K", [(1, 136, 1056), (16, 1024, 8192), (17, 300, 2080), (33, 129, 608),
                                   (48, 128, 32), (64, 272, 4128), (65, 128, 256)])
def test_mx_decode_vs_oracle(gpu, fa, fb, M, N, K):
    t = {"e4m3": tx.F8E4M3, "e5m2": tx.F8E5M2, "e2m1": tx.F4E2M1}
    p = _plan(M, N, K, t[fa], t[fb])
    assert p.kernel == (tx.KERNEL_DECODE_F8 if M <= 64 else tx.KERNEL_GEMM_MX)
    say(f"mx decode {fa}x{fb} {M}x{N}x{K} split={p.split_k}")
    cs = mx_case(M, N, K, fa, fb, seed=M + N + K)
    for out in ("f32", "bf16"):
        check_mx(run_gpu(gpu, cs, out), ref_of(cs, out), cs, out, f"mx decode {out}")


@pytest.mark.parametrize("fmt,K", [("e4m3", 4352), ("e2m1", 8448)])
def test_mx_decode_scale_segments(gpu, fmt, K):
    """One split of more than one segment of staged scales; sampled columns."""
    M, N = 5, 16640
    p = _plan(M, N, K, FMT_TX[fmt], FMT_TX[fmt])
    assert p.kernel == tx.KERNEL_DECODE_F8 and p.split_k == 1
    say(f"mx decode segments {fmt} K={K}")
    cs = mx_case(M, N, K, fmt, fmt, seed=7)
    got = run_gpu(gpu, cs)
    cols = np.sort(np.random.default_rng(1).choice(N, 96, replace=False))
    part = dict(cs, b=np.ascontiguousarray(cs["b"][:, cols]),
                bc=np.ascontiguousarray(cs["bc"][:, cols]), sb=np.ascontiguousarray(cs["sb"][cols]))
    check_mx(np.ascontiguousarray(got[:, cols]), ref_of(part), part, "f32", "segments")


FMT_TX = {"e4m3": tx.F8E4M3, "e5m2": tx.F8E5M2, "e2m1": tx.F4E2M1}


def test_mx_decode_acc_and_repeat(gpu):
    """acc + dot is the dot plus acc in one fp32 addition, and launches repeat bit for bit."""
    import torch
    say("mx decode acc")
    M, N, K = 20, 640, 8192
    cs = mx_case(M, N, K, "e2m1", "e2m1", seed=3)
    dev = {k: to_device(cs[k], gpu) for k in ("a", "sa", "b", "sb")}
    run = lambda **kw: tx.dot_scaled(dev["a"], dev["sa"], "e2m1", dev["b"], dev["sb"], "e2m1", **kw)
    c0, c1 = run(), run()
    acc = torch.randn((M, N), device=gpu)
    got = run(acc=acc)
    torch.cuda.synchronize()
    assert torch.equal(c0.view(torch.int32), c1.view(torch.int32))
    assert torch.equal(got.view(torch.int32), (acc + c0).view(torch.int32))
