"""flash_attention_f32 through the library: a grid of 16-row x 32- or
128-column units whose waves share the keys (fa_small.hip), against float64.

The probabilities enter the second product as f16 relative to the running max in
key order (at most 1, relative error 2^-11, absolute 2^-25 below the normal range),
so |O - O_ref| <= (2^-11 + S 2^-25) max|V| plus fp32 rounding: 6e-4 max|V| covers
S up to 4096.
"""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def check(wave, q, k, v):
    o = wave.flash_attention_f32(q, k, v)
    torch.cuda.synchronize()
    s = (q.double() @ k.double().t()) * math.log(2.0)
    ref = torch.softmax(s, dim=1) @ v.double()
    err = (o.double() - ref).abs().max().item()
    assert err <= 6e-4 * v.double().abs().max().item(), err


def inputs(M, S, D, dev, seed, offset=0):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(M, D, generator=g) * (math.log2(math.e) / math.sqrt(D))

    def at(t):
        buf = torch.empty(t.numel() + offset, dtype=torch.float16, device=dev)
        out = buf[offset:].view(t.shape)
        out.copy_(t)
        return out

    return tuple(at(t) for t in (q, torch.randn(S, D, generator=g), torch.randn(S, D, generator=g)))


@pytest.mark.parametrize("M,S,D", [
    # one to 17 key blocks (waves with one block, with none beyond, with two),
    # ragged keys; head dims below, at and between the register steps
    (16, 1, 64), (16, 31, 64), (15, 32, 32), (17, 33, 128), (1, 511, 8), (16, 512, 64),
    (33, 513, 120), (31, 545, 72), (64, 4096, 128), (5, 1025, 56),
    # any head dim: 4-byte rows, one column, several 128-column units
    (16, 100, 1), (40, 70, 31), (20, 300, 250), (9, 64, 1000),
    # 128-column units
    (4096, 96, 128), (2200, 700, 96), (9000, 40, 20)])
def test_sizes(wave, dev, M, S, D):
    check(wave, *inputs(M, S, D, dev, 1))


@pytest.mark.parametrize("offset", [1, 2, 4])
def test_unaligned_buffers(wave, dev, offset):
    check(wave, *inputs(20, 200, 64, dev, 2, offset))


def in_key_order(q, k, v):
    """The kernel's own steps in float64: blocks of 32 keys in order, each block's
    probabilities relative to the running max and rounded to f16, the sums so far
    rescaled when the max rises; row sums of the unrounded probabilities."""
    s = q.double() @ k.double().t()
    M = s.shape[0]
    m = torch.full((M, 1), -math.inf, dtype=torch.float64, device=s.device)
    l = torch.zeros_like(m)
    acc = torch.zeros((M, v.shape[1]), dtype=torch.float64, device=s.device)
    for n0 in range(0, s.shape[1], 32):
        b = s[:, n0:n0 + 32]
        top = torch.maximum(m, b.amax(dim=1, keepdim=True))
        p, f = torch.exp2(b - top), torch.exp2(m - top)
        l = l * f + p.sum(dim=1, keepdim=True)
        acc = acc * f + p.half().double() @ v[n0:n0 + 32].double()
        m = top
    return acc / l


@pytest.mark.parametrize("M,S,D,ramp", [
    # every register step and both column widths, one to nine rounds of blocks;
    # scores that grow or shrink along the keys move the running max at most
    # blocks or at none
    (64, 1024, 64, 1.0), (64, 1000, 64, 4.0), (33, 4096, 128, 1.0), (16, 2080, 128, 0.25),
    (40, 700, 31, 4.0), (20, 900, 250, 1.0), (2200, 700, 96, 4.0), (9000, 545, 20, 1.0)])
def test_rounds_as_one_running_max(wave, dev, M, S, D, ramp):
    """What the waves share is summed as one pass over the keys would: each
    probability is rounded relative to the running max at its own block.  fp32
    and the rare f16 rounding that goes the other way (0.4 % of them at a score
    error of 2^-22: 2^-11 * 0.004^0.5) give 3e-5 in the 2-norm; probabilities
    rounded relative to any other max, 2e-4."""
    q, k, v = inputs(M, S, D, dev, 5)
    k *= torch.linspace(1.0, ramp, S, device=dev).half()[:, None]
    o = wave.flash_attention_f32(q, k, v).double()
    ref = in_key_order(q, k, v)
    assert ((o - ref).norm() / ref.norm()).item() < 6e-5


@pytest.mark.parametrize("D", [32, 64, 96, 100])
def test_scores_far_apart(wave, dev, D):
    """Blocks whose scores lie hundreds apart, rising and falling: factors and
    probabilities down to zero (below 2^-126 and to 2^-149 among them)."""
    q, k, v = inputs(48, 900, D, dev, 8)
    k *= ((torch.arange(900, device=dev) // 40 * 5 % 7).half() * 12)[:, None]
    o = wave.flash_attention_f32(q, k, v).double()
    ref = in_key_order(q, k, v)
    assert bool(o.isfinite().all())
    # A score of up to 2^9 carries an fp32 error of 2^-13, and so does its power.
    assert ((o - ref).norm() / ref.norm()).item() < 2e-4


def test_excluded_leading_block_is_nan(wave, dev):
    """With every score of the first 32 keys at -inf the running max starts at
    -inf and the row is NaN, as in one pass over the keys."""
    q, k, v = inputs(16, 256, 64, dev, 6)
    q = q.abs() + 0.01
    k[:32] = -math.inf
    assert bool(wave.flash_attention_f32(q, k, v).isnan().all())


def test_grid_beyond_one_dimension(wave, dev):
    """More units than one grid dimension holds threads for (2^32)."""
    M, S = 16 * ((1 << 23) + 3), 256
    q = torch.zeros((M, 1), dtype=torch.float16, device=dev)
    q[-40:] = 1.0
    k = torch.linspace(-2, 2, S, device=dev).half()[:, None]
    v = torch.linspace(3, 7, S, device=dev).half()[:, None]
    o = wave.flash_attention_f32(q, k, v)
    for part, x in ((o[:-40], 0.0), (o[-40:], 1.0)):
        w = torch.softmax(k.double() * x * math.log(2.0), dim=0)
        ref = (w * v.double()).sum().item()
        assert float((part.double() - ref).abs().max()) <= 6e-4 * 7


def test_blocks_of_excluded_keys(wave, dev):
    """Keys with a score of -inf fill whole blocks, so that some waves see no
    finite score at all; the others' result stands."""
    q, k, v = inputs(16, 256, 64, dev, 3)
    q = q.abs() + 0.01
    k[32:160] = -math.inf
    check(wave, q, k, v)


def test_infinite_scores_stay_nan(wave, dev):
    """A row with a +inf score is NaN (inf - inf), and only that row."""
    q, k, v = inputs(16, 256, 64, dev, 4)
    k[100, 0] = math.inf
    q[:, 0] = 0.5
    q[3, 0] = -0.5
    o = wave.flash_attention_f32(q, k, v)
    nan = o.isnan().all(dim=1)
    assert bool(nan[torch.arange(16, device=dev) != 3].all())
    assert bool(o[3].isfinite().all())
