"""GPU parity of the 128x128 ring tiles (TX_FLAG_TILES_128, gemm_ring.h): every operand kind
and layout at tile edges, K tails of one byte to a whole step, split K and a single step,
against the 256x256 tiles the same plan names without the flag (explicit block).

int8 sums are exact and must be equal.  The others add the same products in fp32, in K order
within a range (16-bit, fp8: one MFMA chain per range; block-scaled: one fma per 128 K), so
two results differ by at most the rounding of the sums: (K / 16 + 8) 2^-23 sum |a b| here,
plus one ulp of a 16-bit C.
"""
import numpy as np
import pytest

import triton_ext_amd as tx
from dotcase import say

pytestmark = pytest.mark.gpu

SHAPES = [(97, 128, 512), (129, 257, 2049), (300, 131, 4100), (128, 640, 64), (513, 1000, 1111)]


def _padded(torch, x, junk):
    """x in rows 16 bytes apart, the padding and the row after the last full of `junk`."""
    es = x.element_size()
    ld = (x.shape[1] * es + 15) // 16 * 16 // es + 16 // es
    buf = torch.empty((x.shape[0] + 1, ld), dtype=x.dtype, device=x.device)
    buf.view(torch.uint8).fill_(junk)
    buf[:x.shape[0], :x.shape[1]] = x
    return buf[:x.shape[0], :x.shape[1]]


def _both(dot, desc_args, flags=0):
    """The dot on the plan with TX_FLAG_TILES_128 and on the 256x256 tiles."""
    out = []
    for f in (tx.FLAG_TILES_128, 0):
        p = tx.plan(tx.make_desc(flags=flags | f, **desc_args))
        assert (p.desc.block_m, p.desc.block_n) == (256, 256)
        assert bool(p.desc.flags & tx.FLAG_TILES_128) == bool(f)
        out.append(dot(p))
    return out


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("kind", ["bf16", "f16_f32", "int8", "w8a8", "fp8", "fp8_mix", "fp8b",
                                  "fp8b_f32"])
@pytest.mark.parametrize("kmajor", [False, True])
def test_tiles128_vs_256(gpu, kind, kmajor, M, N, K):
    import torch
    say(f"tiles128 {kind} kmajor={kmajor} {M}x{N}x{K}")
    g = torch.Generator(device=gpu)
    g.manual_seed(M + N + K)
    a, b = (torch.randn(s, generator=g, device=gpu) for s in ((M, K), (N, K) if kmajor else (K, N)))
    sa = sb = None
    mode, out, junk = tx.SCALE_NONE, torch.float32, 0x7F
    if kind in ("bf16", "f16_f32"):
        t = torch.bfloat16 if kind == "bf16" else torch.float16
        out = torch.bfloat16 if kind == "bf16" else torch.float32
        a, b, junk = a.to(t), b.to(t), 0xFF
    elif kind in ("int8", "w8a8"):
        a, b = (torch.round(x * 40).clamp(-127, 127).to(torch.int8) for x in (a, b))
        out = torch.int32 if kind == "int8" else torch.bfloat16
        if kind == "w8a8":
            mode, sa, sb = tx.SCALE_ROWCOL, torch.rand(M, device=gpu), torch.rand(N, device=gpu)
    else:
        a = a.to(torch.float8_e4m3fn)
        b = b.to(torch.float8_e5m2 if kind == "fp8_mix" else torch.float8_e4m3fn)
        if kind in ("fp8b", "fp8b_f32"):
            mode, out = tx.SCALE_BLOCK128, torch.bfloat16 if kind == "fp8b" else torch.float32
            kb = -(-K // 128)
            sa = torch.rand((M, kb), device=gpu) + 0.5
            sb = torch.rand((kb, -(-N // 128)), device=gpu) + 0.5
    a, b = _padded(torch, a, junk), _padded(torch, b, junk)
    c = tx.new_output(M, N, out, gpu)
    bv = b.t() if kmajor else b
    desc = dict(M=M, N=N, K=K, a_type=tx.tx_type(a), b_type=tx.tx_type(b), c_type=tx.tx_type(c),
                scale_mode=mode, block=(256, 256, 64 if a.element_size() == 2 else 128),
                lda=a.stride(0), ldb=b.stride(0), ldc=c.stride(0))

    def run(p):
        r = tx.new_output(M, N, out, gpu)
        tx.dot(a, bv, out=r, scale_a=sa, scale_b=sb, plan=p)
        return r.clone()
    got, want = _both(run, desc, tx.FLAG_B_KMAJOR if kmajor else 0)
    torch.cuda.synchronize()
    if kind in ("int8", "w8a8"):
        assert torch.equal(got, want)
        return
    f = lambda x: x.to(torch.float32).double().abs()
    if mode == tx.SCALE_BLOCK128:
        S = (f(a) * sa.double().repeat_interleave(128, 1)[:, :K]) @ \
            (f(bv) * sb.double().repeat_interleave(128, 0)[:K].repeat_interleave(128, 1)[:, :N])
    else:
        S = f(a) @ f(bv)
    bound = (K / 16 + 8) * 2.0 ** -23 * S + 1e-30
    if out == torch.bfloat16:
        bound = bound + 2.0 ** -7 * f(want)
    d = (got.double() - want.double()).abs()
    assert torch.isfinite(got.double()).all() and (d <= bound).all(), float((d / bound).max())


@pytest.mark.parametrize("M,N,K", [(97, 128, 512), (129, 257, 2080), (300, 131, 4128), (128, 640, 64)])
@pytest.mark.parametrize("fa,fb", [("e4m3", "e4m3"), ("e5m2", "e4m3"), ("e2m1", "e2m1")])
@pytest.mark.parametrize("out", ["f32", "bf16"])
def test_tiles128_mx(gpu, fa, fb, out, M, N, K):
    """The planner's choice at these sizes is the ring tile; against the oracle."""
    from test_decode_mx_gpu import FMT_TX
    from test_mx_gpu import check_mx, mx_case, ref_of, run_gpu
    r = lambda x, q: -(-x // q) * q
    p = tx.plan(tx.make_desc(M, N, K, FMT_TX[fa], tx.F32, b_type=FMT_TX[fb], lda=r(K, 32),
                             ldb=r(N, 16), ldc=r(N, 4), scale_mode=tx.SCALE_MX32))
    assert p.kernel == tx.KERNEL_GEMM_MX and p.desc.flags & tx.FLAG_TILES_128
    assert (p.split_k > 1) == (K >= 4096 or (K > 2048 and fa != "e2m1"))
    say(f"tiles128 mx {fa}x{fb} {out} {M}x{N}x{K} split={p.split_k}")
    cs = mx_case(M, N, K, fa, fb, seed=M + N + K)
    check_mx(run_gpu(gpu, cs, out), ref_of(cs, out), cs, out, f"tiles128 mx {out}")


def test_tiles128_acc_noalloc_and_repeat(gpu):
    """acc + dot is the dot plus acc in one fp32 addition, split and whole; launches repeat
    bit for bit; the no-allocation launch gives the same bits."""
    import ctypes

    import torch
    say("tiles128 acc / noalloc")
    for M, N, K in ((200, 300, 4096), (700, 900, 512)):
        a = torch.randn((M, K), device=gpu).bfloat16()
        b = torch.randn((K, N), device=gpu).bfloat16()
        b = tx.aligned_rows(b)
        p = tx.plan_for(a, b, tx.F32, ldc=-(-N // 4) * 4)
        assert p.desc.flags & tx.FLAG_TILES_128 and (p.split_k > 1) == (K == 4096)
        c0, c1 = (tx.dot(a, b, out_dtype=torch.float32) for _ in range(2))
        acc = torch.randn((M, N), device=gpu)
        got = tx.dot(a, b, acc=acc)
        c2 = tx.new_output(M, N, torch.float32, gpu)
        tx.check(tx.load().tx_dot_launch_noalloc(ctypes.byref(p), a.data_ptr(), b.data_ptr(),
                                                 c2.data_ptr(), None, None,
                                                 torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert torch.equal(c0.view(torch.int32), c1.view(torch.int32))
        assert torch.equal(c0, c2) and torch.equal(got, acc + c0)
        want = a.double() @ b.double()
        assert ((c0.double() - want).abs() <= 1e-5 * (a.double().abs() @ b.double().abs())).all()
        assert np.isfinite(c0.sum().item())


def test_tiles128_wide_mxfp4(gpu):
    """e2m1 B of nearly 2^31 bytes, whose offsets past K lie above 2^31: the same sums as the
    256x256 tile's, whose K order is the same within 8 steps (the module's bound; |a b| summed
    over slices of columns)."""
    import torch
    M, N, K = 128, 1048576, 4064
    say(f"tiles128 mxfp4 {M}x{N}x{K}")
    g = torch.Generator(device=gpu)
    g.manual_seed(11)
    a = torch.randint(0, 256, (M, K // 2), generator=g, device=gpu, dtype=torch.uint8)
    b = torch.randint(0, 256, (K // 2, N), generator=g, device=gpu, dtype=torch.uint8)
    sa = torch.randint(124, 131, (M, K // 32), generator=g, device=gpu, dtype=torch.uint8)
    sb = torch.randint(124, 131, (N, K // 32), generator=g, device=gpu, dtype=torch.uint8)
    a = tx.aligned_rows(a, col_ok=False)
    p = tx.plan(tx.make_desc(M, N, K, tx.F4E2M1, tx.F32, scale_mode=tx.SCALE_MX32,
                             lda=2 * a.stride(0), ldb=N, ldc=N))
    assert p.desc.flags & tx.FLAG_TILES_128
    got = tx.dot_scaled(a, sa, "e2m1", b, sb, "e2m1", plan=p)
    want = tx.dot_scaled(a, sa, "e2m1", b, sb, "e2m1", block=(256, 256, 256))
    torch.cuda.synchronize()
    mag = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6] * 2, device=gpu, dtype=torch.float64)

    def values(codes, s):  # |rows of codes times their scales| [R, K]
        x = mag[torch.stack([codes & 15, codes >> 4], 2).long()].view(codes.shape[0], -1)
        return x * torch.exp2(s.double() - 127).repeat_interleave(32, 1)
    fa = values(a, sa)
    for n in (0, N // 2 - 512, N - 1024):
        S = fa @ values(b[:, n:n + 1024].t().contiguous(), sb[n:n + 1024]).t().contiguous()
        d = (got[:, n:n + 1024].double() - want[:, n:n + 1024].double()).abs()
        assert (d <= (K / 16 + 8) * 2.0 ** -23 * S).all()
    assert torch.isfinite(got).all() and float((got - want).abs().max()) < 1e-2 * float(want.abs().max())


@pytest.mark.parametrize("kind", ["bf16", "fp8", "mxw"])
def test_tiles128_noalloc_split(gpu, kind):
    """The no-allocation launch splits K as the ring tiles do (2 ranges, 12 or 16 MiB of partials),
    whatever the 256x256 tiles' own split would take (8 ranges, past the scratch): the bits of
    the launch with a workspace, over several launches."""
    import ctypes

    import torch
    M, N, K = (384, 4096, 4096) if kind == "mxw" else (256, 8192, 8192)
    say(f"tiles128 noalloc split {kind} {M}x{N}x{K}")
    g = torch.Generator(device=gpu)
    g.manual_seed(9)
    sb = None
    a = torch.randn((M, K), generator=g, device=gpu).bfloat16()
    if kind == "mxw":
        b = torch.randint(0, 256, (K // 2, N), generator=g, device=gpu, dtype=torch.uint8)
        sb = torch.randint(124, 131, (N, K // 32), generator=g, device=gpu, dtype=torch.uint8)
        p = tx.plan(tx.make_desc(M, N, K, tx.BF16, tx.F32, b_type=tx.F4E2M1,
                                 scale_mode=tx.SCALE_MX32, ldb=N, ldc=N))
        run = lambda: tx.dot_scaled(a, None, "bf16", b, sb, "e2m1", plan=p)
    else:
        b = torch.randn((K, N), generator=g, device=gpu).bfloat16()
        if kind == "fp8":
            a, b = a.to(torch.float8_e4m3fn), b.to(torch.float8_e4m3fn)
        p = tx.plan_for(a, b, tx.F32)
        run = lambda: tx.dot(a, b, plan=p, out=torch.empty((M, N), device=gpu))
    assert p.desc.flags & tx.FLAG_TILES_128 and p.split_k == 8
    assert p.workspace_bytes > tx.NOALLOC_SCRATCH_BYTES
    want = run()
    for _ in range(3):
        got = torch.empty_like(want)
        tx.check(tx.load().tx_dot_launch_noalloc(
            ctypes.byref(p), a.data_ptr(), b.data_ptr(), got.data_ptr(), None,
            None if sb is None else sb.data_ptr(), torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("M,N,K,split", [(700, 1100, 512, False), (300, 700, 8192, True)])
def test_tiles128_group_m(gpu, M, N, K, split):
    """A caller's plan.group_m, past the tile rows too, changes the tile order alone."""
    import torch
    say(f"tiles128 group_m {M}x{N}x{K}")
    a, b = (torch.randint(-127, 128, s, device=gpu, dtype=torch.int8) for s in ((M, K), (K, N)))
    b = tx.aligned_rows(b)
    p = tx.plan_for(a, b, tx.I32, ldc=-(-N // 4) * 4)
    assert p.desc.flags & tx.FLAG_TILES_128 and (p.split_k > 1) == split
    want = a.double() @ b.double()
    for gm in (1, 2, 3, 4, 100, 2 ** 31 - 1):
        p.group_m = gm
        out = tx.new_output(M, N, torch.int32, gpu)
        assert torch.equal(tx.dot(a, b, plan=p, out=out).double(), want)


@pytest.mark.parametrize("K,ld", [(100, 1 << 24), (126, (1 << 24) + 16)])
def test_tiles128_long_rows(gpu, K, ld):
    """A few columns of a matrix of 2^24 columns, rows past K up to just below 2^32 bytes: the
    bits of the same dot on a copy of those columns."""
    import torch
    M, N = 300, 512
    say(f"tiles128 {M}x{N}x{K} of rows {ld} bytes apart")
    g = torch.Generator(device=gpu)
    g.manual_seed(K)
    a = torch.randn((M, K), generator=g, device=gpu).to(torch.float8_e4m3fn)
    whole = torch.zeros((K, ld), device=gpu, dtype=torch.uint8)
    whole.fill_(0x7F)  # NaN
    b = whole.view(torch.float8_e4m3fn)[:, :N]
    b.copy_(torch.randn((K, N), generator=g, device=gpu).to(torch.float8_e4m3fn))
    a = tx.aligned_rows(a, col_ok=False)
    p = tx.plan_for(a, b, tx.F32)
    assert p.desc.flags & tx.FLAG_TILES_128 and p.desc.ldb == ld
    got = tx.dot(a, b, plan=p, out=torch.empty((M, N), device=gpu))
    assert torch.equal(got, tx.dot(a, b.contiguous(), out_dtype=torch.float32))
    want = a.float().double() @ b.float().double()
    assert (got.double() - want).norm() < 1e-4 * want.norm()
