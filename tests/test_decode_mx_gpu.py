"""GPU parity of the MX decode kernels (dot_scaled with a few rows of A) against the oracle.

MX x MX (decode_f8.h's MX form): the scaled MFMA's own bound (test_mx_gpu.check_mx).
bf16 x MX and e4m3 scales (decode16.h's WQ form): the operand upcast is exact, so the
result is within fp32 summation error of the oracle, K 2^-24 sum |a b|, plus one bf16 ulp
for bf16 C.  Shapes sit at the edges: slices of 16 .. 96 rows, N and K that fill no strip
or batch, scale rows that start at every byte of a dword, split K, and more than one
segment of staged scales (K past 4096 in one split).
"""
import numpy as np
import pytest

import oracle
import test_mx_gpu
import triton_ext_amd as tx
from dotcase import bits_to_f32, from_device, say, to_device
from test_mx_gpu import FMT, check_mx, mx_bf16_case, mx_case, ref_of, run_gpu

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


@pytest.mark.parametrize("fmt", ["e2m1", "e4m3", "e5m2"])
@pytest.mark.parametrize("out", ["f32", "bf16"])
@pytest.mark.parametrize("M,N,K", [(1, 250, 480), (16, 128, 256), (33, 272, 416), (64, 136, 512),
                                   (80, 300, 288), (96, 256, 992), (97, 128, 256)])
def test_mx_bf16_decode_small(gpu, fmt, out, M, N, K):
    """One split on both sides: bit for bit the bf16 dot of the host upcast, and the oracle."""
    p = _plan(M, N, K, tx.BF16, FMT_TX[fmt])
    assert p.kernel == (tx.KERNEL_DECODE_MX_BF16 if M <= 96 else tx.KERNEL_GEMM_MX_BF16)
    test_mx_gpu.test_mx_bf16_vs_oracle(gpu, "b", fmt, out, M, N, K)


@pytest.mark.parametrize("fmt", ["e2m1", "e4m3", "e5m2"])
def test_mx_bf16_decode_scale_range(gpu, fmt):
    """Scales over [1, 239] (pair conversion and the fp32 path beside it): bit for bit the
    bf16 dot of the host upcast; NaN scales make exactly their columns NaN."""
    import torch
    say(f"bf16 x {fmt} decode scale range")
    M, N, K = 32, 272, 512
    cs = mx_bf16_case(M, N, K, "b", fmt, seed=78 + len(fmt))
    cs["s"] = np.random.default_rng(3).integers(1, 240, size=cs["s"].shape).astype(np.uint8)
    cs["b16"] = test_mx_gpu.upcast_bf16(cs["codes"], cs["s"], fmt, "b")
    bf = lambda x: to_device(x.view(np.int16), gpu).view(torch.bfloat16)
    run = lambda s: from_device(tx.dot_scaled(bf(cs["a16"]), None, "bf16", to_device(cs["b"], gpu),
                                              to_device(s, gpu), fmt))
    got = run(cs["s"])
    want = from_device(tx.dot(bf(cs["a16"]), bf(cs["b16"]), out_dtype=torch.float32))
    assert np.array_equal(got.view(np.int32), want.view(np.int32))
    s = cs["s"].copy()
    s[1::2, 5] = 255
    nan = np.isnan(run(s))
    # (e5m2 terms reach 2^127: an even column's sum may itself be inf - inf)
    assert nan[:, 1::2].all() and np.array_equal(nan[:, 0::2], np.isnan(got[:, 0::2]))


@pytest.mark.parametrize("lhs,rhs,fmt", [("bf16", "e2m1", "mx"), ("bf16", "e4m3", "mx"),
                                         ("bf16", "e2m1", "nv"), ("e2m1", "e2m1", "nv")])
@pytest.mark.parametrize("M,N,K", [(3, 600, 8256), (40, 16640, 4352)])
def test_wq_decode_split_and_segments(gpu, lhs, rhs, fmt, M, N, K):
    """Split K, and one split of several scale segments; sampled columns against the oracle."""
    import torch
    nv = fmt == "nv"
    p = _plan(M, N, K, FMT_TX.get(lhs, tx.BF16), FMT_TX[rhs], tx.SCALE_NV16 if nv else tx.SCALE_MX32)
    assert p.kernel == tx.KERNEL_DECODE_MX_BF16 and (p.split_k > 1) == (N == 600)
    say(f"wq decode {lhs}x{rhs} {fmt} {M}x{N}x{K} split={p.split_k}")
    rng = np.random.default_rng(M + N)
    grp, lo, hi = (16, 0x20, 0x50) if nv else (32, 117, 138)
    bc = test_mx_gpu.codes(rng, (K, N), rhs)
    sb = rng.integers(lo, hi, size=(N, K // grp)).astype(np.uint8)
    b = test_mx_gpu.pack(bc, 0) if rhs == "e2m1" else bc
    if lhs == "bf16":
        a, sa = test_mx_gpu.upcast_bf16(rng.integers(0, 16, size=(M, K)).astype(np.uint8),
                                        np.full((M, K // 32), 127, np.uint8), "e2m1", "a"), None
        da = to_device(a.view(np.int16), gpu).view(torch.bfloat16)
    else:
        a = test_mx_gpu.pack(rng.integers(0, 16, size=(M, K)).astype(np.uint8), 1)
        sa = rng.integers(lo, hi, size=(M, K // grp)).astype(np.uint8)
        da = to_device(a, gpu)
    e4 = lambda x: None if x is None else (to_device(x, gpu).view(torch.float8_e4m3fn) if nv
                                           else to_device(x, gpu))
    got = from_device(tx.dot_scaled(da, e4(sa), lhs, to_device(b, gpu), e4(sb), rhs))
    cols = np.sort(rng.choice(N, 64, replace=False))
    ref = oracle.dot_scaled(a, sa, FMT[lhs] if lhs != "bf16" else oracle.BF16,
                            np.ascontiguousarray(b[:, cols]), np.ascontiguousarray(sb[cols]),
                            FMT[rhs], K=K, nv16=nv)
    k = np.arange(K) // grp
    dec = (lambda s: torch.from_numpy(s).view(torch.float8_e4m3fn).double().numpy()) if nv else \
        (lambda s: np.exp2(s.astype(np.float64) - 127))
    bv = np.abs(oracle.mx_decode(bc[:, cols], FMT[rhs]) * dec(np.ascontiguousarray(sb[cols]))[:, k].T)
    av = np.abs(bits_to_f32(a, "bf16").astype(np.float64)) if lhs == "bf16" else \
        np.abs(oracle.mx_decode(np.stack([a & 15, a >> 4], 2).reshape(M, K), FMT[lhs]) * dec(sa)[:, k])
    bound = K * 2.0 ** -24 * (av @ bv) + 1e-30
    d = np.abs(got[:, cols].astype(np.float64) - ref)
    assert (d <= bound).all(), f"worst d/bound {(d / bound).max():.3g}"


@pytest.mark.parametrize("fmt,M,N,K", [("e4m3", 22, 6656, 7296), ("e4m3", 69, 3296, 4160),
                                       ("e2m1", 16, 704, 8128), ("e2m1", 3, 17000, 4096),
                                       ("e4m3", 9, 384, 2400)])
def test_wq_decode_error(gpu, fmt, M, N, K):
    """fp32 C against 64 bits: no further off than the upcast and the 256x256 bf16 tile (an
    explicit block) are, over long ranges of K, uneven ones and 16 splits.  (Both errors are
    2-norms over M N elements and three seeds: they scatter by about a percent, 2 at the
    smallest.)"""
    import torch
    say(f"wq decode error {fmt} {M}x{N}x{K}")
    mag = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6], device=gpu, dtype=torch.float64)
    mag = torch.cat([mag, -mag])
    err = [0.0, 0.0]
    for seed in (1, 2, 3):
        g = torch.Generator(device=gpu)
        g.manual_seed(seed)
        a = tx.aligned_rows(torch.randn((M, K), generator=g, device=gpu).bfloat16())
        s = torch.randint(124, 131, (N, K // 32), generator=g, device=gpu, dtype=torch.uint8)
        if fmt == "e2m1":
            b = torch.randint(0, 256, (K // 2, N), generator=g, device=gpu, dtype=torch.uint8)
            bv = mag[torch.stack([b & 15, b >> 4], 1).long()].view(K, N)
        else:
            b = torch.randn((K, N), generator=g, device=gpu).to(torch.float8_e4m3fn)
            bv = b.float().double()
        bv = bv * torch.exp2(s.double() - 127).repeat_interleave(32, 1).t()
        want = a.double() @ bv
        for i, block in enumerate(((0, 0, 0), (256, 256, 64))):
            p = tx.plan(tx.make_desc(M, N, K, tx.BF16, tx.F32, b_type=FMT_TX[fmt],
                                     scale_mode=tx.SCALE_MX32, block=block, lda=a.stride(0),
                                     ldb=-(-N // 16) * 16, ldc=-(-N // 4) * 4))
            assert p.kernel == (tx.KERNEL_GEMM_MX_BF16 if i else tx.KERNEL_DECODE_MX_BF16)
            got = tx.dot_scaled(a, None, "bf16", tx.aligned_rows(b, col_ok=False), s, fmt, plan=p)
            err[i] += float((got.double() - want).norm() / want.norm())
    assert err[0] <= 1.03 * err[1], err
