"""flash_attention_f32 through the library: a grid of 16-row x 32- or
128-column units whose waves share the keys (fa_small.hip), against float64.

The probabilities enter the second product as f16 relative to a wave's running
max (at most 1, relative error 2^-11, absolute 2^-25 below the normal range),
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
