"""Host side of the GEMM dispatch, without a GPU: the tags of split launches and
the kernel a shape takes."""

import pytest

import gemm_plan


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
