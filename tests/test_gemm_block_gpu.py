"""The small-block GEMM kernels (gemm_block.hpp) and the rule that chooses
between them, the 256x256 tiles and Stream-K (gemm_plan), against the CPU
oracle: bucket inputs make every fp32 sum exact whatever its order (K < 2^18),
so every kernel, block size and K split has to give the oracle's bits.
"""

import pytest
import torch

import gemm_plan
from conftest import to_dev
from test_gemm_gpu import ODT, TDT, assert_exact, run_gemm

pytestmark = pytest.mark.gpu


# Edges of every block (32, 64, 128) in M and N, K from one element group to
# several ring depths with and without a remainder of the 64-deep stage.  On 256
# CUs every block size is among the plans, and 256x256 tiles for the last two
# (test_gemm_plan.py).
BLOCK_SHAPES = [
    (1, 1, 4), (31, 33, 64), (32, 32, 60), (33, 31, 68), (64, 65, 128), (63, 127, 640),
    (1, 4096, 704), (32, 5000, 128), (100, 1030, 196),                      # few rows
    (500, 300, 1100), (515, 1021, 64), (400, 1600, 260), (1000, 1000, 132),
    (1024, 1536, 192), (1290, 1270, 72), (129, 8192, 324),                  # 64 and 128 edges
    (1536, 2048, 256), (2000, 1500, 100), (16400, 256, 64),
    (64, 96, 256), (64, 96, 320), (1536, 2048, 128), (1536, 2048, 192),     # with and without ring
    (3000, 3000, 132), (3072, 3300, 64)]


@pytest.mark.parametrize("in_dt,out_dt,layout", [(1, 0, "row"), (1, 1, "col"), (2, 2, "row"),
                                                 (2, 0, "col"), (1, 2, "row"), (2, 1, "col")])
@pytest.mark.parametrize("shape", BLOCK_SHAPES)
def test_blocks_bit_exact(wave, oracle, dev, in_dt, out_dt, layout, shape):
    M, N, K = shape
    _, _, c, ref = run_gemm(wave, oracle, dev, M, N, K, in_dt, out_dt, layout, seed=21)
    assert_exact(oracle, c, ref, out_dt)


# K not a multiple of 4: element-by-element loads, 64x64 blocks, and for the last
# two shapes (short K, many blocks) the 256x256 tiles (test_gemm_plan.py).
UNALIGNED_SHAPES = [(1, 1, 1), (64, 64, 63), (65, 129, 65), (200, 300, 130),
                    (1000, 70, 1001), (1872, 891, 21), (3000, 3000, 65), (1450, 7431, 87)]


@pytest.mark.parametrize("layout,out_dt", [("row", 2), ("col", 0)])
@pytest.mark.parametrize("shape", UNALIGNED_SHAPES)
def test_unaligned_k_bit_exact(wave, oracle, dev, layout, out_dt, shape):
    M, N, K = shape
    _, _, c, ref = run_gemm(wave, oracle, dev, M, N, K, 2, out_dt, layout, seed=22)
    assert_exact(oracle, c, ref, out_dt)


# Large enough for 256x256 tiles, in each of that kernel's modes: whole tiles on
# the DMA path (one, two and five 64-deep stages); whole tiles with K off the
# stage (a 32-deep tail after 0, 1 and 2 stages); ragged tiles on the DMA ring
# with K % 8 == 0 and K % 4 == 0 (tails of 8, 20, 36 and 4, the first two below a
# stage) and C lines off 16 bytes; element by element.  The last number is A's
# start in elements past a 16-byte boundary: 4 takes the K % 4 path, 1 the
# element-by-element one.
TILE_SHAPES = [
    (1280, 3328, 64, 0), (1280, 3328, 128, 0), (1280, 3328, 320, 0),
    (2560, 3328, 32, 0), (2560, 3328, 96, 0), (2560, 3328, 160, 0),
    (2555, 3273, 8, 0), (2554, 3272, 72, 0), (2554, 3273, 200, 0),
    (2554, 3272, 20, 0), (2555, 3272, 36, 0), (2554, 3273, 452, 0), (2560, 3328, 64, 4),
    (3834, 3784, 65, 0), (2554, 3273, 641, 0), (4096, 4096, 64, 1)]


@pytest.mark.parametrize("in_dt", [1, 2])
@pytest.mark.parametrize("shape", TILE_SHAPES)
def test_tiles_bit_exact(wave, oracle, dev, in_dt, shape):
    M, N, K, off = shape
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    p = gemm_plan.plan(wave.runtime.lib(), M, N, K, cus,
                       vec4=K % 4 == 0 and off % 4 == 0)
    assert cus != 256 or p.bm == 0, p
    a, b = oracle.gemm_inputs(M, K, in_dt, 26, 0), oracle.gemm_inputs(N, K, in_dt, 26, 1)
    buf = torch.empty(M * K + 8, dtype=TDT[in_dt], device=dev)
    A, B = buf[off:off + M * K].view(M, K), to_dev(b, TDT[in_dt], dev)
    A.copy_(to_dev(a, TDT[in_dt], dev))
    ref = oracle.gemm_nt(a, b, in_dt)
    for out_dt in (0, 1, 2):
        for layout in ("row", "col"):
            c = wave.gemm(A, B, out_dtype=ODT[out_dt], layout=layout)
            torch.cuda.synchronize()
            assert_exact(oracle, c if layout == "row" else c.t(), ref, out_dt)


@pytest.mark.parametrize("out_dt", [0, 1])
@pytest.mark.parametrize("a_off,b_off,c_off", [(4, 0, 0), (0, 2, 0), (1, 3, 0), (0, 0, 1),
                                               (4, 4, 4)])
@pytest.mark.parametrize("shape", [(70, 66, 132), (600, 500, 192)])
def test_unaligned_buffers(wave, oracle, dev, shape, out_dt, a_off, b_off, c_off):
    """A, B and C starting that many elements past a 16-byte boundary."""
    M, N, K = shape
    a, b = oracle.gemm_inputs(M, K, 1, 23, 0), oracle.gemm_inputs(N, K, 1, 23, 1)

    def at(t, off):
        buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=dev)
        v = buf[off:off + t.numel()].view(t.shape)
        v.copy_(t)
        return v

    A, B = at(to_dev(a, TDT[1], dev), a_off), at(to_dev(b, TDT[1], dev), b_off)
    guard = torch.full((M * N + 16,), 7.0, dtype=ODT[out_dt], device=dev)
    C = guard[8 + c_off:8 + c_off + M * N].view(M, N)
    wave.gemm(A, B, out_dtype=ODT[out_dt], out=C)
    torch.cuda.synchronize()
    assert_exact(oracle, C, oracle.gemm_nt(a, b, 1), out_dt)
    assert bool((guard[:8 + c_off] == 7).all()) and bool((guard[8 + c_off + M * N:] == 7).all())


# The shape-driven entry point with its workspace: K split over 2 to 8 CTAs of
# 32x32 to 128x128 blocks (test_gemm_plan.py), split K ranges of unequal length, a
# K remainder (the last split's), and M <= 128 with its counters.
SPLIT_SHAPES = [
    (130, 200, 4100), (300, 260, 8260), (512, 512, 16384), (200, 2000, 8256), (1000, 1000, 16384),
    (1100, 900, 16390 // 4 * 4), (2048, 1024, 16384), (1, 1024, 16384), (33, 1500, 16448),
    (128, 16384, 4096), (100, 5000, 12288), (3, 2048, 16384), (128, 3000, 16448),
    (1, 1024, 32768), (33, 1024, 32768)]


@pytest.mark.parametrize("in_dt,out_dt,layout", [(1, 1, "row"), (2, 2, "col"), (2, 0, "row")])
@pytest.mark.parametrize("shape", SPLIT_SHAPES)
def test_auto_splits_bit_exact(wave, oracle, dev, in_dt, out_dt, layout, shape):
    M, N, K = shape
    a, b = oracle.gemm_inputs(M, K, in_dt, 24, 0), oracle.gemm_inputs(N, K, in_dt, 24, 1)
    ref = oracle.gemm_nt(a, b, in_dt)
    A, B = to_dev(a, TDT[in_dt], dev), to_dev(b, TDT[in_dt], dev)
    need = wave.gemm_auto_workspace_bytes(M, N, K)
    assert need > 0
    guard = torch.full((need + 256,), 0xFF, dtype=torch.uint8, device=dev)
    ws = guard[:need]
    for _ in range(3):  # a dirty workspace, then what the launch before left
        c = wave.gemm_auto(A, B, out_dtype=ODT[out_dt], layout=layout, workspace=ws)
        torch.cuda.synchronize()
        assert_exact(oracle, c.t() if layout == "col" else c, ref, out_dt)
    assert bool((guard[need:] == 0xFF).all())


# Both split on 256 CUs (test_gemm_plan.py); the second's partials reach to where
# the first's counters lie (the top 32 KiB of 16 MiB).
GRAPH_SHAPES = [(512, 512, 16384), (2048, 1024, 16384)]


def test_split_graph_replays(wave, oracle, dev):
    """A captured split launch (a fixed tag) replayed between eager launches of
    another shape on the same workspace, after the words it counts on were
    written over, and twice in a row."""
    ops = []
    for i, (M, N, K) in enumerate(GRAPH_SHAPES):
        a, b = oracle.gemm_inputs(M, K, 1, 25 + i, 0), oracle.gemm_inputs(N, K, 1, 25 + i, 1)
        ops.append((to_dev(a, TDT[1], dev), to_dev(b, TDT[1], dev), oracle.gemm_nt(a, b, 1)))
    need = max(wave.gemm_auto_workspace_bytes(*s) for s in GRAPH_SHAPES)
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=dev)
    (A, B, ref), (A1, B1, ref1) = ops
    out = wave.gemm_auto(A, B, out_dtype="f32", workspace=ws)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        wave.gemm_auto(A, B, out_dtype="f32", workspace=ws, out=out)
    noise = torch.randn(need // 4, device=dev).view(torch.uint8)
    for i in range(4):
        other = wave.gemm_auto(A1, B1, out_dtype="f32", workspace=ws)
        if i & 1:
            ws[:need // 4 * 4].copy_(noise)
        for _ in range(2):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert_exact(oracle, out, ref, 0)
        assert_exact(oracle, other, ref1, 0)


@pytest.mark.parametrize("shape", [(512, 512, 16384), (100, 5000, 12288)])
def test_counter_words_of_other_launches(wave, oracle, dev, shape):
    """Workspaces full of words that earlier launches left half counted: other
    tags, with every count (both places where counters lie)."""
    M, N, K = shape
    a, b = oracle.gemm_inputs(M, K, 1, 27, 0), oracle.gemm_inputs(N, K, 1, 27, 1)
    ref = oracle.gemm_nt(a, b, 1)
    A, B = to_dev(a, TDT[1], dev), to_dev(b, TDT[1], dev)
    need = wave.gemm_auto_workspace_bytes(M, N, K)
    for count in range(16):
        word = gemm_plan.split_tag(wave.runtime.lib()) | count
        ws = torch.full((need // 8,), word - (1 << 64) * (word >> 63), dtype=torch.int64,
                        device=dev).view(torch.uint8)
        c = wave.gemm_auto(A, B, out_dtype="f32", workspace=ws)
        torch.cuda.synchronize()
        assert_exact(oracle, c, ref, 0)
