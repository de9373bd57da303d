"""The forward's choice between 256-row blocks (the 8-wave kernel) and 128-row
ones (one pass of the 4-wave kernel), every row against float64.

TOL: the probabilities are rounded to 16 bits before the PV product and O once
(f16 2^-11, bf16 2^-8 relative each); with |V| up to about 4.5 and weights
summing to one the first is at most 4.5 * 2^-11 (2^-8) and in practice a tenth.
"""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.float16: 2e-3, torch.bfloat16: 1.5e-2}


def reference(q, k, v, causal):
    B, H, S, D = q.shape
    o = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    lse = torch.empty((B, H, S), dtype=torch.float64, device=q.device)
    hide = torch.ones(S, S, dtype=torch.bool, device=q.device).triu_(1) if causal else None
    for b in range(B):
        for h in range(H):
            j = h // (H // k.shape[1])
            s = q[b, h].double() @ k[b, j].double().t().contiguous() / math.sqrt(D)
            if causal:
                s.masked_fill_(hide, -math.inf)
            lse[b, h] = torch.logsumexp(s, 1)
            o[b, h] = torch.softmax(s, 1) @ v[b, j].double()
    return o, lse


# On 256 CUs: 128-row blocks because they are at most one a CU (the first
# five), or because they pad less on several rounds (300, 513); 256-row blocks
# (256, 1000, 640).
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,S", [(1, 1, 1, 1), (1, 2, 1, 127), (1, 3, 3, 129), (2, 4, 2, 500),
                                         (1, 32, 8, 1000), (2, 72, 8, 300), (3, 50, 10, 513),
                                         (4, 40, 8, 256), (2, 64, 8, 1000), (1, 61, 61, 640)])
def test_every_row(wave, dev, dt, causal, B, Hq, Hkv, S):
    g = torch.Generator(device=dev).manual_seed(S)
    q, k, v = (torch.randn(s, generator=g, device=dev).to(dt)
               for s in ((B, Hq, S, 128), (B, Hkv, S, 128), (B, Hkv, S, 128)))
    o, lse = wave.flash_attention_lse(q, k, v, causal=causal)
    torch.cuda.synchronize()
    ref, lref = reference(q, k, v, causal)
    half_ulp = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    over = ((o.double() - ref).abs() - half_ulp * ref.abs()).max().item()
    assert over <= TOL[dt], over
    assert (lse.double() - lref).abs().max().item() <= (1e-3 if dt == torch.float16 else 5e-3)
    assert torch.equal(o, wave.flash_attention(q, k, v, causal=causal))
    if S <= 640:  # inputs within a bound: the fixed-max kernels
        bound = 0.5 if dt == torch.float16 else 1.0
        qb, kb = (t.clamp(-bound, bound) for t in (q, k))
        ob = wave.flash_attention(qb, kb, v, causal=causal, qk_max_abs=bound)
        rb, _ = reference(qb, kb, v, causal)
        over = ((ob.double() - rb).abs() - half_ulp * rb.abs()).max().item()
        assert over <= TOL[dt], over


# Causal blocks by length (heads a multiple of the 8 XCDs): long and short pairs
# of 128-row blocks (1100 and 2300: a last run of blocks that is not full; 300;
# 257: four blocks a CU, mostly padding) and 256-row blocks (1537, 777), odd
# lengths throughout, K and V of one head up to all of them.
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,Hq,Hkv,S", [(1, 32, 8, 1100), (2, 8, 1, 2300), (2, 72, 8, 300),
                                         (8, 40, 8, 257), (1, 40, 40, 1537), (4, 24, 8, 777)])
def test_blocks_by_length(wave, dev, dt, B, Hq, Hkv, S):
    test_every_row(wave, dev, dt, True, B, Hq, Hkv, S)
