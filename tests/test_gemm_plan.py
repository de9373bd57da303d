"""Host side of the GEMM dispatch, without a GPU: the tags of split launches and
the kernel a shape takes."""

import pytest

import gemm_plan
from test_gemm_block_gpu import (BLOCK_SHAPES, GRAPH_SHAPES, SPLIT_SHAPES, TILE_SHAPES,
                                 UNALIGNED_SHAPES)
from test_streamk_gpu import AUTO_SHAPES, FLOAT_SHAPES, auto_workers, short_m_plan


def test_split_tags_are_drawn_from_sixty_bits(wave):
    """A counter word of a split launch counts only under that launch's tag, and
    the workspace it lies in may hold anything: the tag has to differ from it in
    any of its 60 bits, not in half of a word or by a step from launch to launch."""
    lib = wave.runtime.lib()
    tags = [gemm_plan.split_tag(lib) for _ in range(4096)]
    assert all(t and t & 15 == 0 for t in tags)
    assert len(set(tags)) == len(tags)
    for bit in range(4, 64):  # each bit about half the time (12 sigma)
        assert abs(sum(t >> bit & 1 for t in tags) - 2048) < 400, bit
        flips = sum((a ^ b) >> bit & 1 for a, b in zip(tags, tags[1:]))
        assert abs(flips - 2048) < 400, bit


@pytest.mark.parametrize("M,N,K", [(1 << 18, 1 << 18, 1), (1 << 18, 1 << 18, 5),
                                   (1 << 24, 4096, 1), ((1 << 18) - 64, 1 << 18, 1),
                                   (1 << 17, 1 << 17, 4), (1 << 28, 32, 4)])
def test_block_grids_stay_below_2_32_threads(wave, M, N, K):
    p = gemm_plan.plan(wave.runtime.lib(), M, N, K)
    if p.bm:
        assert -(-M // p.bm) * -(-N // p.bn) * p.splits * 256 < 1 << 32


# What the GPU tests' shapes take on 256 CUs, as their comments say.
def test_block_shapes_take_every_block(wave):
    lib = wave.runtime.lib()
    plans = [gemm_plan.plan(lib, *s) for s in BLOCK_SHAPES]
    assert {(p.bm, p.bn) for p in plans[:-2]} == {(32, 32), (32, 64), (64, 64), (128, 64),
                                                  (128, 128)}
    assert [p.bm for p in plans[-2:]] == [0, 0]
    plans = [gemm_plan.plan(lib, *s) for s in UNALIGNED_SHAPES]
    assert all((p.bm, p.bn) == (64, 64) for p in plans[:-2])
    assert [p.bm for p in plans[-2:]] == [0, 0]
    assert all(gemm_plan.plan(lib, M, N, K, vec4=K % 4 == 0 and off % 4 == 0).bm == 0
               for M, N, K, off in TILE_SHAPES)


# (M, N, K, block): the faster kernel as measured, element by element.
@pytest.mark.parametrize("M,N,K,bm", [
    (4293, 7657, 51, 0), (2472, 4628, 23, 0), (1927, 7182, 49, 0), (2758, 7945, 11, 0),
    (6651, 1032, 311, 0), (3000, 3000, 1001, 0), (1872, 2891, 21, 64), (1141, 4300, 215, 64),
    (7038, 664, 43, 64), (2007, 1464, 4845, 64), (2048, 2048, 1001, 64), (1000, 1000, 1001, 64)])
def test_unaligned_rows_by_shape(wave, M, N, K, bm):
    assert gemm_plan.plan(wave.runtime.lib(), M, N, K).bm == bm


# Operands beyond the last-level cache: no 64x64 blocks in several rounds where
# rows lie off its lines.
@pytest.mark.parametrize("M,N,K,bm", [
    (5421, 905, 18996, 0), (1332, 3665, 36640, 0), (627, 7008, 37280, 0), (746, 6165, 34196, 0),
    (1553, 2621, 36652, 0), (1121, 4345, 26000, 0), (2319, 1678, 22072, 64),
    (1937, 2465, 27840, 64), (2539, 1669, 17440, 64)])
def test_long_k_by_shape(wave, M, N, K, bm):
    assert gemm_plan.plan(wave.runtime.lib(), M, N, K).bm == bm


def auto(lib, M, N, K):
    return gemm_plan.auto_plan(lib, M, N, K, short_m_plan(M, N, K, 256),
                               auto_workers(M, N, K, 256))


def test_split_shapes_split_every_block(wave):
    plans = [auto(wave.runtime.lib(), *s) for s in SPLIT_SHAPES]
    assert all(p.splits > 1 for p in plans)
    assert {(p.bm, p.bn) for p in plans} == {(32, 32), (32, 64), (64, 64), (128, 64), (128, 128)}
    assert {p.splits for p in plans} >= {2, 3, 4, 5, 6, 8}
    assert [auto(wave.runtime.lib(), *s).splits for s in FLOAT_SHAPES] == [2, 4]
    small, large = (auto(wave.runtime.lib(), *s) for s in GRAPH_SHAPES)
    assert small.splits > 1 and large.splits > 1
    top = auto_workers(*GRAPH_SHAPES[0], 256) * 2 * 256 * 256 * 4  # end of its slots
    M, N, _ = GRAPH_SHAPES[1]
    assert -(-M // large.bm) * -(-N // large.bn) * large.splits * large.bm * large.bn * 4 >= top


def test_auto_shapes_take_what_they_name(wave):
    lib = wave.runtime.lib()
    for shape, kind in AUTO_SHAPES:
        p = auto(lib, *shape)
        got = ("stream-k" if p.workers else "tiles" if p.bm == 0 else
               "split" if p.splits > 1 else "blocks")
        assert got == kind, (shape, p)
