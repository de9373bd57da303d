"""wave_mxfp8_quantize_launch against the same formula as tensor operations
(ops._mxfp8_quantize_formula), byte for byte, on the kernels' three routes:
rows (blocks along the last dimension), columns, and element by element.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]


def values(shape, dtype, seed):
    """Random signs and magnitudes over the dtype's whole range, with every
    special value the encoding treats apart among them."""
    g = torch.Generator().manual_seed(seed)
    n = 1
    for d in shape:
        n *= d
    lo, hi = {torch.float32: (-149, 128), torch.bfloat16: (-133, 128),
              torch.float16: (-24, 16)}[dtype]
    # Runs of 512 values share an exponent to within 16, so that most blocks
    # hold elements of many codes and not one large value and zeros.
    centre = torch.randint(lo, hi, (n // 512 + 1,), generator=g).repeat_interleave(512)[:n]
    e = (centre - torch.randint(0, 16, (n,), generator=g)).double()
    x = torch.exp2(e) * (1 + torch.rand(n, generator=g, dtype=torch.float64))
    x = torch.where(torch.rand(n, generator=g) < 0.5, -x, x)
    one = torch.tensor(1.0, dtype=dtype)
    below = torch.nextafter(one.float(), torch.zeros(())) if dtype == torch.float32 else 1 - \
        torch.finfo(dtype).eps / 2
    special = [0.0, -0.0, float("inf"), -float("inf"), float("nan"), 1.0, float(below), 448.0,
               -464.0, 480.0]
    x = x.to(dtype)
    at = torch.randperm(n, generator=g)[:max(1, n // 200)]
    x[at] = torch.tensor(special, dtype=dtype)[torch.arange(len(at)) % len(special)]
    if n > 256:
        x[64:128] = 0.0
        x[128:192] = -0.0
        x[200] = float("nan")
    return x.reshape(shape)


def check(wave, x, dim):
    got = wave.mxfp8_quantize(x, dim=dim)
    torch.cuda.synchronize()
    want = wave.ops._mxfp8_quantize_formula(x, dim % x.dim())
    for name, a, b in zip(("elements", "scales"), got, want):
        assert a.shape == b.shape and a.dtype == b.dtype and a.is_contiguous()
        # A NaN's sign is not part of the encoding's value: 0x7f and 0xff.
        if name == "elements":
            nan = (b & 0x7F) == 0x7F
            assert torch.equal((a & 0x7F) == 0x7F, nan)
            a, b = a.masked_fill(nan, 0), b.masked_fill(nan, 0)
        bad = (a != b).sum().item()
        assert bad == 0, f"{name}: {bad} of {a.numel()} bytes differ"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape,dim", [
    ((1, 32), -1), ((3, 5, 96, 128), -1), ((1031, 64), 1),          # rows
    ((2, 3, 64, 128), 2), ((2, 3, 50, 128), 2), ((1, 1, 4), 1),     # columns: whole and cut
    ((37, 33, 20), 1), ((31, 128), 0), ((4097, 4), 0),              # blocks, odd unit counts
    ((5, 100), 1), ((3, 96, 7), 1), ((1,), 0), ((2, 31), 1),        # element by element
])
def test_bytes_match_the_formula(wave, dev, dtype, shape, dim):
    check(wave, values(shape, dtype, 1).to(dev), dim)


@pytest.mark.parametrize("dtype", DTYPES)
def test_views(wave, dev, dtype):
    """Unaligned starts and strided inputs."""
    flat = values((8 * 64 * 128 + 8,), dtype, 3).to(dev)
    check(wave, flat[1:1 + 64 * 128].view(64, 128), -1)
    check(wave, flat[2:2 + 64 * 128].view(64, 128), 0)
    check(wave, flat[:8 * 64 * 128].view(8, 64, 128).transpose(0, 1), -1)
    check(wave, flat[:8 * 64 * 128].view(64, 8, 128)[:, ::2], 0)


def test_f32_below_powers_of_two(wave, dev):
    """Largest values just under 2^k, where log2 rounds: one block each."""
    k = torch.arange(-126, 128, dtype=torch.float64)
    p = torch.exp2(k).float()
    x = torch.zeros(len(k) * 4, 32)
    bits = p.view(torch.int32)
    for j in range(4):
        x[j::4, 5] = (bits - j).view(torch.float32)
        x[j::4, 9] = -p * 0.3
    check(wave, x.to(dev), -1)


def test_other_dtypes_and_graphs(wave, dev):
    x = values((4, 64), torch.float32, 5).nan_to_num(0.0, 1.0, -1.0).to(dev)
    d, s = wave.mxfp8_quantize(x.double()), wave.mxfp8_quantize(x)
    assert torch.equal(d[0], s[0]) and torch.equal(d[1], s[1])
    h = x.half()
    wave.mxfp8_quantize(h)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        e, sc = wave.mxfp8_quantize(h)
    for seed in (6, 7, 8):
        h.copy_(values((4, 64), torch.float16, seed).to(dev))
        graph.replay()
        torch.cuda.synchronize()
        we, ws = wave.mxfp8_quantize(h)
        assert torch.equal(e, we) and torch.equal(sc, ws)


def test_jit_trace_is_refused(wave, dev):
    """A trace would record the output allocations without the launch between
    them; it takes the formula, whose uint8 views torch.jit.trace refuses."""
    x = values((4, 64), torch.float32, 9).to(dev)
    with pytest.raises(RuntimeError):
        torch.jit.trace(lambda t: wave.mxfp8_quantize(t), (x,), check_trace=False)


@pytest.mark.parametrize("dim", [0, 1])
def test_lazy_tensors(wave, dev, dim):
    """Views that are negated when read, and zero tensors without memory."""
    x = values((64, 96), torch.float32, 10).nan_to_num().to(dev)
    neg = torch._neg_view(x)
    assert neg.is_neg()
    for got, want in zip(wave.mxfp8_quantize(neg, dim), wave.mxfp8_quantize(-x, dim)):
        assert torch.equal(got, want)
    # The imaginary part of a conjugate: negated and strided.
    z = torch.complex(x, x.flip(0)).conj().imag
    assert z.is_neg()
    for got, want in zip(wave.mxfp8_quantize(z, dim), wave.mxfp8_quantize(-x.flip(0), dim)):
        assert torch.equal(got, want)
    zero = torch._efficientzerotensor((64, 96), device=dev)
    for got, want in zip(wave.mxfp8_quantize(zero, dim),
                         wave.mxfp8_quantize(torch.zeros((64, 96), device=dev), dim)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("dim", [0, 1])
def test_beyond_32_bits(wave, dev, dim):
    """2^32 + 64 blocks of one value: columns past 2^32 (across), and more blocks
    than one grid dimension holds threads for (along)."""
    n, part = (1 << 32) + 64, 1 << 20
    x = torch.full((n,), 1.5, dtype=torch.bfloat16, device=dev)
    ends = (slice(0, part), slice((1 << 31) - part, 1 << 31), slice(n - part, n))
    for i, at in enumerate(ends):
        x[at] = values((part,), torch.bfloat16, 11 + i).nan_to_num().to(dev)
    got = [t.view(n) for t in wave.mxfp8_quantize(x.view((1, n) if dim == 0 else (n, 1)), dim)]
    for at in ends:
        want = wave.ops._mxfp8_quantize_formula(x[at].view((1, part) if dim == 0 else (part, 1)),
                                                dim)
        for a, b in zip(got, want):
            assert torch.equal(a[at], b.view(part))
    # 1.5 = 384 * 2^-8, everywhere between.
    assert bool((got[0][part:(1 << 31) - part] == 0x7C).all())
    assert bool((got[1][1 << 31:n - part] == 127 - 8).all())
