"""GPU parity of the attention forward at few programs, where (at fp16 / bf16, head dims up to
64 and blocks left to the planner) 4 groups of waves split a row's keys: against float64
attention (o within 2^-8 of its size, M within 1e-4), and against the one-group kernel, whose
rounding of p it keeps: groups without a block, odd block counts, causal and not, strided
[Z, N, H, D] operands, scores of -inf, values near the type's lowest."""
import math

import numpy as np
import pytest

import triton_ext_amd as tx
from dotcase import say

pytestmark = pytest.mark.gpu


def exact(q, k, v, causal, scale):
    import torch
    s = q.double() @ k.double().transpose(2, 3) * scale
    if causal:
        n = s.shape[-1]
        s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=s.device).triu(1), -math.inf)
    return torch.softmax(s, 3) @ v.double(), torch.logsumexp(s, 3) / math.log(2.0)


@pytest.mark.parametrize("Z,H,N,D", [
    (1, 1, 128, 64), (1, 2, 256, 16), (1, 3, 384, 32), (1, 1, 640, 64), (2, 4, 1152, 64),  # 4 groups
    (1, 5, 128, 128), (1, 11, 1024, 64), (1, 9, 896, 128), (2, 16, 512, 32),  # one, or 4 at 32
    (1, 17, 1152, 128), (1, 32, 1024, 64), (3, 8, 1280, 32), (1, 33, 1024, 32)])  # one
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_attn_key_groups(gpu, dtype, causal, Z, H, N, D):
    import torch
    say(f"attn key groups {dtype} causal={causal} {Z}x{H}x{N}x{D}")
    dt = torch.float16 if dtype == "fp16" else torch.bfloat16
    g = torch.Generator(device=gpu)
    g.manual_seed(N + D)
    q, k, v = (torch.randn((Z, N, H, D), generator=g, device=gpu).to(dt).permute(0, 2, 1, 3)
               for _ in range(3))
    o, M = tx.attention(q, k, v, causal, D ** -0.5, return_lse=True)
    o2, M2 = tx.attention(q, k, v, causal, D ** -0.5, return_lse=True)
    torch.cuda.synchronize()
    assert torch.equal(o, o2) and torch.equal(M, M2)
    eo, em = exact(q, k, v, causal, D ** -0.5)
    # p and o each rounded once to the operands' type: 2^-9 (bf16) or 2^-12 (fp16) of the
    # largest |v| a row averages, twice, plus fp32 sums
    u = 2.0 ** -9 if dtype == "bf16" else 2.0 ** -12
    vmax = v.double().abs().amax(dim=(2, 3), keepdim=True)
    assert ((o.double() - eo).abs() <= 2 * u * vmax + 1e-5).all()
    assert (M.double() - em).abs().max() < 1e-4


def test_attn_key_groups_inf_scores(gpu):
    """Keys whose scores are -inf for every row fill a later group's first blocks: they add
    nothing, as after finite blocks in one group."""
    import torch
    say("attn key groups, -inf scores")
    Z, H, N, D = 1, 2, 512, 64
    g = torch.Generator(device=gpu)
    g.manual_seed(3)
    q = torch.rand((Z, H, N, D), generator=g, device=gpu).bfloat16() + 1
    k = torch.randn((Z, H, N, D), generator=g, device=gpu).bfloat16()
    v = torch.randn((Z, H, N, D), generator=g, device=gpu).bfloat16()
    k[:, :, 128:256, 0] = -math.inf
    k[:, :, 448:, 3] = -math.inf
    o, M = tx.attention(q, k, v, False, 0.125, return_lse=True)
    torch.cuda.synchronize()
    eo, em = exact(q, k, v, False, 0.125)
    assert torch.isfinite(o).all() and np.isfinite(M.sum().item())
    assert (o.double() - eo).abs().max() <= 2 ** -8 * float(v.abs().max()) + 1e-5
    assert (M.double() - em).abs().max() < 1e-4


def rel(x, y):
    x, y = x.double(), y.double()
    return float((x - y).norm() / y.norm())


@pytest.mark.parametrize("Z,H,N,D", [(1, 2, 256, 16), (1, 1, 384, 64), (1, 8, 1024, 64),
                                     (1, 16, 1024, 32), (2, 1, 4096, 64), (1, 16, 1024, 128),
                                     (1, 32, 1024, 64)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_attn_key_groups_round_as_one(gpu, dtype, causal, Z, H, N, D):
    """p is rounded against the row's running maximum whatever the groups: o differs from the
    64 x 64 blocks' (always one group) by the order of fp32 sums alone.  Relative differences of
    2^-20 before o is rounded flip at most that over half a unit u of o's roundings, u each:
    u sqrt(2^-19 / u), 9e-5 (bf16) and 3e-5 (fp16); rounding p otherwise gives about u / 3.
    With the blocks given there is one group: the same bits as 64 x 64's without the mask."""
    import torch
    say(f"attn key groups as one {dtype} causal={causal} {Z}x{H}x{N}x{D}")
    dt = torch.float16 if dtype == "fp16" else torch.bfloat16
    u = 2.0 ** -11 if dtype == "fp16" else 2.0 ** -8
    g = torch.Generator(device=gpu)
    g.manual_seed(N + D)
    q, k, v = (torch.randn((Z, N, H, D), generator=g, device=gpu).to(dt).permute(0, 2, 1, 3)
               for _ in range(3))
    o, M = tx.attention(q, k, v, causal, D ** -0.5, return_lse=True)
    o1, M1 = tx.attention(q, k, v, causal, D ** -0.5, return_lse=True, block=(64, 64))
    o2, M2 = tx.attention(q, k, v, causal, D ** -0.5, return_lse=True, block=(128, 64))
    torch.cuda.synchronize()
    assert rel(o, o1) < u / 10 and (M - M1).abs().max() < 1e-5
    if not causal:
        assert torch.equal(o2, o1) and torch.equal(M2, M1)
    if D == 128 or Z * H * N > 128 * (128 if D <= 32 else 64):  # one group by itself
        assert torch.equal(o, o2) and torch.equal(M, M2)


def test_attn_key_groups_large_values(gpu):
    """Values near bf16's lowest whose keys' weights underflow next to the row's earlier keys:
    they add nothing (a group's own maximum would weigh them 1, and sum them to -inf)."""
    import torch
    say("attn key groups, large values of no weight")
    Z, H, N, D = 1, 2, 1024, 64
    g = torch.Generator(device=gpu)
    g.manual_seed(5)
    q = torch.ones((Z, H, N, D), device=gpu, dtype=torch.bfloat16)
    k = torch.randn((Z, H, N, D), generator=g, device=gpu).bfloat16()
    v = torch.randn((Z, H, N, D), generator=g, device=gpu).bfloat16()
    k[:, :, :64] = 32.0  # scores of 256 log2(e), against some units
    v[:, :, 512:] = torch.finfo(torch.bfloat16).min
    o, M = tx.attention(q, k, v, False, 0.125, return_lse=True)
    o1, M1 = tx.attention(q, k, v, False, 0.125, return_lse=True, block=(64, 64))
    torch.cuda.synchronize()
    assert torch.isfinite(o).all() and rel(o, o1) < 2.0 ** -8 / 10
    assert (M - M1).abs().max() < 1e-4


@pytest.mark.parametrize("N", [512, 896])
@pytest.mark.parametrize("causal", [False, True])
def test_attn_key_groups_inf_as_one(gpu, causal, N):
    """Blocks of -inf scores, first in a later group and in the maximum pass: as in one group."""
    import torch
    say(f"attn key groups, -inf scores as one causal={causal} N={N}")
    g = torch.Generator(device=gpu)
    g.manual_seed(7)
    q = torch.rand((1, 2, N, 32), generator=g, device=gpu).bfloat16() + 1
    k, v = (torch.randn((1, 2, N, 32), generator=g, device=gpu).bfloat16() for _ in range(2))
    k[:, :, 64:192, 0] = -math.inf
    k[:, :, N - 64:, 3] = -math.inf
    o, M = tx.attention(q, k, v, causal, 0.125, return_lse=True)
    o1, M1 = tx.attention(q, k, v, causal, 0.125, return_lse=True, block=(64, 64))
    torch.cuda.synchronize()
    assert torch.isfinite(o).all() and rel(o, o1) < 2.0 ** -8 / 10
    assert (M - M1).abs().max() < 1e-5
