"""GPU parity of the attention forward where a row's keys are split among groups of waves
(fp16 / bf16 at the default block, few programs): against the oracle at the bars of
test_attn_gpu (o within 2^-8 of its size, M within 1e-4), and float64 attention, at every form
of the split: groups without a block, odd block counts, causal and not, strided [Z, N, H, D]
operands, scores of -inf."""
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
    (1, 1, 128, 64), (1, 2, 256, 16), (1, 3, 384, 32), (1, 1, 640, 64), (2, 4, 1152, 64),  # 32 x 4
    (1, 5, 128, 128), (1, 11, 1024, 64), (1, 9, 896, 128), (2, 16, 512, 32),  # 64 x 2
    (1, 17, 1152, 128), (1, 32, 1024, 64), (3, 8, 1280, 32), (1, 33, 1024, 32)])  # 128 x 2
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
