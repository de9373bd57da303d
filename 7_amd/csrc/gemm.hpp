// gemm.hpp -- host-side launch interface of the tiled / Stream-K GEMM
// kernels in gemm.hip (used by the C ABI in wave_runtime.cpp).
#pragma once

#include <hip/hip_runtime.h>

namespace wave {
namespace gemm {

struct GemmArgs {
  const void *A = nullptr;  // [M x K] row-major, f16 or bf16
  const void *B = nullptr;  // [N x K] row-major, same type as A
  void *C = nullptr;        // [M x N] row-major or [N x M] (column-major)
  int M = 0, N = 0, K = 0;
  int in_dtype = 1;         // wave::kF16 / wave::kBF16
  int out_dtype = 1;        // wave::kF32 / kF16 / kBF16
  bool col_major = false;
  int group_m = 0;          // tile-row group size; 0 = default (4)
  void *scratch = nullptr;  // Stream-K fp32 partials (workers*2*256*256)
  void *counters = nullptr; // Stream-K per-tile arrival counters (zeroed)
  int workers = 0;          // > 0 selects the Stream-K kernel
  bool force_masked = false;
  int cus = 256;            // compute units of the device, for the block choice
  // MXFP4 (in_dtype kMXFP4): A [M][K/2], B [N][K/2] packed fp4; e8m0 scales
  // group-major [K/32][M] and [K/32][N].
  const void *a_scale = nullptr;
  const void *b_scale = nullptr;
  // MXFP4 with B and both scales in the AITER preshuffled layouts.
  bool aiter = false;
  // Tile-packed C for the reference blocking (bm, bn, wave_m_tiles,
  // wave_n_tiles); computed in the column-major orientation.
  bool packed = false;
  int pk_bm = 1, pk_bn = 1, pk_wmt = 1, pk_wnt = 1;
};

constexpr int kTileEdge = 256;
constexpr int kKStage = 64;

int tiles_for(int extent);
int k_iterations(int K);
hipError_t launch(const GemmArgs &args, hipStream_t stream);
// MXFP4 scaled GEMM (gemm_mxfp4.hip): M, N % 256 == 0, K % 128 == 0.
hipError_t launch_mxfp4(const GemmArgs &args, hipStream_t stream);

// The kernel `launch_auto` runs for a shape.  bm = 0: the 256x256 tiles
// (Stream-K when workers > 0), else a bm x bn block over `splits` K ranges
// (gemm_block.hpp).
struct GemmPlan {
  int bm = 0, bn = 0, splits = 1;
  int workers = 0;
};
// Limits a caller's workspace puts on a split: fp32 partial slots and 64-bit
// counter words (two a block).
struct SplitLimits {
  size_t slot_bytes = 0, counter_words = 0;
};
// vec4: K % 4 == 0 and A, B 8-byte aligned (rows_vec4); c_vec: C's lines start at
// multiples of 16 bytes (lines_vec16); workers: what Stream-K would run with (0: not
// offered).
GemmPlan gemm_plan(int M, int N, int K, int cus, bool vec4, bool c_vec, int workers,
                   const SplitLimits &limits);
bool rows_vec4(const GemmArgs &args);
bool lines_vec16(const GemmArgs &args);
// A small-block launch: `slots` / `counters` for splits > 1 (any contents: a
// counter word counts only under this launch's `tag`; left zero),
// and zero_words 64-bit words at `zero` left zero.
struct BlockWorkspace {
  float *slots = nullptr;
  unsigned long long *counters = nullptr, *zero = nullptr;
  size_t zero_words = 0;
  uint64_t tag = 0;  // split_tag()
};
// Counts share a word with their launch's tag: the low bits, up to kMaxSplits.
constexpr unsigned long long kCountMask = 15;
constexpr int kMaxSplits = 8;
static_assert(kMaxSplits <= (int)kCountMask, "a count fits its bits");
// A tag for one split launch: nonzero, kCountMask's bits zero, the others drawn
// anew each time (any thread).
uint64_t split_tag();
hipError_t launch_blocks(const GemmArgs &args, const GemmPlan &plan, const BlockWorkspace &ws,
                         hipStream_t stream);

// The workspace contract of the shape-driven entry point for M <= 128:
// partial slots of `splits` x (128 x bn) fp32 per bn columns, then two 64-bit
// words per bn columns, which every launch that is given them leaves zero.
// splits == 0: no workspace.
struct SplitPlan {
  int splits = 0;
  int bn = 128;
};
SplitPlan short_m_workspace(int M, int N, int K, int cus);
size_t short_m_slot_bytes(int N, const SplitPlan &plan);
size_t short_m_counter_count(int N, const SplitPlan &plan);

} // namespace gemm
} // namespace wave
