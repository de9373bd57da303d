"""Which dK/dV kernel the backward takes, without a GPU: bwd_key_block of
attention_bwd.hip (a C++ function, so by its mangled name) on 256 CUs.
"""

import ctypes

import pytest

from test_attention_bwd_gpu import HALF_SHAPES


def key_block(wave, B, Hq, Hkv, S, causal):
    fn = wave.runtime.lib()._ZN4wave9attention13bwd_key_blockEiiiibi
    fn.restype = ctypes.c_int
    fn.argtypes = [ctypes.c_int] * 4 + [ctypes.c_bool, ctypes.c_int]
    return fn(B, Hq, Hkv, S, causal, 256)


@pytest.mark.parametrize("causal", [False, True])
def test_half_shapes_take_64_keys(wave, causal):
    for shape in HALF_SHAPES:
        assert key_block(wave, *shape, causal) == 64, shape


# (B, Hq, Hkv, S, causal, keys): the faster one as measured.  With 128 keys a block
# half of the last one lies past the sequence: 33 us against 26 in the first row, 247
# / 208 in the second, 534 / 488 in the sixth.
@pytest.mark.parametrize("B,Hq,Hkv,S,causal,keys", [
    (32, 16, 16, 64, False, 64), (256, 16, 16, 64, True, 64), (64, 32, 8, 64, True, 64),
    (24, 12, 12, 192, False, 64), (128, 16, 16, 192, True, 64), (64, 16, 16, 448, True, 64),
    # many items a block, chunks, or little past the sequence
    (1, 64, 1, 64, True, 128), (128, 16, 2, 192, True, 128), (16, 32, 8, 192, False, 128),
    (32, 16, 16, 320, False, 128), (64, 16, 16, 576, True, 128), (2, 16, 4, 1984, True, 128),
    (4, 32, 32, 4032, False, 128),
    # whole blocks of 128
    (32, 16, 16, 128, False, 128), (2, 16, 4, 2048, True, 128)])
def test_key_block_by_shape(wave, B, Hq, Hkv, S, causal, keys):
    assert key_block(wave, B, Hq, Hkv, S, causal) == keys


def workspace(wave, B, Hq, Hkv, S, causal):
    fn = wave.runtime.lib()._ZN4wave9attention19bwd_workspace_bytesEiiiibi
    fn.restype = ctypes.c_size_t
    fn.argtypes = [ctypes.c_int] * 4 + [ctypes.c_bool, ctypes.c_int]
    return fn(B, Hq, Hkv, S, causal, 256)


# (B, Hq, Hkv, S, causal, chunks): whether cutting the blocks was the faster, as
# measured (first row 35 us in chunks, 29 whole; third 4167, 3810).
@pytest.mark.parametrize("B,Hq,Hkv,S,causal,chunks", [
    (1, 64, 16, 128, False, False), (1, 64, 16, 128, True, False), (1, 64, 8, 8192, True, False),
    (1, 64, 8, 7680, True, False), (2, 64, 8, 4096, True, False), (1, 40, 8, 7168, True, False),
    (4, 16, 2, 6976, True, False), (2, 32, 8, 4096, True, False),
    (1, 32, 8, 128, False, True), (2, 32, 4, 128, False, True), (1, 64, 8, 6144, True, True),
    (1, 64, 8, 4096, True, True), (1, 64, 4, 8192, True, True), (1, 48, 12, 6144, True, True),
    (2, 128, 16, 1984, True, True), (2, 16, 4, 2048, True, True), (1, 8, 8, 2048, True, True),
    (1, 64, 8, 5120, False, True), (2, 256, 32, 128, False, True), (1, 4, 1, 64, False, True)])
def test_chunks_by_shape(wave, B, Hq, Hkv, S, causal, chunks):
    assert (workspace(wave, B, Hq, Hkv, S, causal) > 0) == chunks
    # The most a call asks for: three rounds of 128 KiB partials.
    assert workspace(wave, B, Hq, Hkv, S, causal) <= 3 * 256 * (128 << 10)
