// gemm_dispatch.hip -- host-side selection of the GEMM kernel variant
// (aligned DMA path vs masked path, dtype/layout, tiled vs Stream-K).
#include "gemm_block.hpp"
#include "gemm_kernels.hpp"

#ifndef WAVE_GEMM_GROUP_M
#define WAVE_GEMM_GROUP_M 4
#endif

#include <sys/random.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <type_traits>
#include <vector>

namespace wave {
namespace gemm {

#define WAVE_GEMM_EXTERN(IN, OUT, SK)                                          \
  extern template hipError_t launch_variant<IN, OUT, false, SK>(               \
      const Params &, int, hipStream_t);                                       \
  extern template hipError_t launch_variant<IN, OUT, true, SK>(                \
      const Params &, int, hipStream_t);
#define WAVE_GEMM_EXTERN_IN(IN)                                                \
  WAVE_GEMM_EXTERN(IN, kF32, false)                                            \
  WAVE_GEMM_EXTERN(IN, kF16, false)                                            \
  WAVE_GEMM_EXTERN(IN, kBF16, false)                                           \
  WAVE_GEMM_EXTERN(IN, kF32, true)                                             \
  WAVE_GEMM_EXTERN(IN, kF16, true)                                             \
  WAVE_GEMM_EXTERN(IN, kBF16, true)
WAVE_GEMM_EXTERN_IN(kF16)
WAVE_GEMM_EXTERN_IN(kBF16)

namespace block {
#define WAVE_BLOCK_EXTERN(IN, OUT)                                             \
  extern template hipError_t launch_block<IN, OUT>(const BlockParams &, int,   \
                                                   int, bool, bool, hipStream_t);
WAVE_BLOCK_EXTERN(kF16, kF32)
WAVE_BLOCK_EXTERN(kF16, kF16)
WAVE_BLOCK_EXTERN(kF16, kBF16)
WAVE_BLOCK_EXTERN(kBF16, kF32)
WAVE_BLOCK_EXTERN(kBF16, kF16)
WAVE_BLOCK_EXTERN(kBF16, kBF16)
} // namespace block

template <int IN, int OUT>
static hipError_t launch_out(const Params &p, bool cm, bool sk, int mode,
                             hipStream_t s) {
  if (sk)
    return cm ? launch_variant<IN, OUT, true, true>(p, mode, s)
              : launch_variant<IN, OUT, false, true>(p, mode, s);
  return cm ? launch_variant<IN, OUT, true, false>(p, mode, s)
            : launch_variant<IN, OUT, false, false>(p, mode, s);
}

template <int IN>
static hipError_t launch_in(const Params &p, int out, bool cm, bool sk,
                            int mode, hipStream_t s) {
  if (out == kF32)
    return launch_out<IN, kF32>(p, cm, sk, mode, s);
  if (out == kF16)
    return launch_out<IN, kF16>(p, cm, sk, mode, s);
  return launch_out<IN, kBF16>(p, cm, sk, mode, s);
}

static bool aligned_to(const void *ptr, size_t bytes) {
  return ((uintptr_t)ptr % bytes) == 0;
}

// Counter maintenance for the Stream-K workspace.  A fill kernel rather than
// hipMemsetAsync so the reset can sit inside a captured HIP graph.
__global__ void zero_u32_kernel(uint32_t *p, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    p[i] = 0u;
}

hipError_t zero_counters(uint32_t *counters, size_t count, hipStream_t stream) {
  if (count == 0)
    return hipSuccess;
  hipLaunchKernelGGL(zero_u32_kernel, dim3((unsigned)((count + 255) / 256)),
                     dim3(256), 0, stream, counters, count);
  return hipGetLastError();
}

hipError_t count_nonzero(const uint32_t *counters, size_t count, int *result,
                         hipStream_t stream) {
  std::vector<uint32_t> host(count);
  hipError_t e = hipMemcpyAsync(host.data(), counters, count * sizeof(uint32_t),
                                hipMemcpyDeviceToHost, stream);
  if (e != hipSuccess)
    return e;
  e = hipStreamSynchronize(stream);
  if (e != hipSuccess)
    return e;
  int n = 0;
  for (uint32_t v : host)
    n += v != 0u;
  *result = n;
  return hipSuccess;
}

int tiles_for(int extent) { return (extent + kTile - 1) / kTile; }
int k_iterations(int K) { return (K + kSKUnit - 1) / kSKUnit; }

bool rows_vec4(const GemmArgs &g) {
  return g.K % 4 == 0 && aligned_to(g.A, 8) && aligned_to(g.B, 8);
}
bool lines_vec16(const GemmArgs &g) {
  const size_t line = (size_t)(g.col_major ? g.M : g.N) * (g.out_dtype == kF32 ? 4 : 2);
  return aligned_to(g.C, 16) && line % 16 == 0;
}

// ---- which kernel a shape takes --------------------------------------------
// Each candidate's time is estimated (microseconds) and the least taken.  The
// constants are a fit to measured launches: f16, one MI355X (256 CUs), three
// operand sets in turn, 3400 random shapes (M, N 1 to 16384, K 32 to 16384,
// half of them M <= 128) times every block size and 1 to 8 splits.  On those
// shapes the choice is on average 2 % from the best candidate and never more
// than 8 % slower than the 256x256 / 32-column kernels it chose between
// before, 2.6 times as fast in the mean.
//
// A block's stage (64 of K) costs s0 on an idle chip and s1 with a CTA on
// every CU (its DMA is bound by what a CU fetches, 80 to 110 GB/s); further
// CTAs queue (s2 a stage, `round` a CTA).  A split's exchange costs e0 plus
// what all partials cost to publish (e1 a MB) and the last arriver to read
// (e2 a 16 KiB slot).  No candidate beats its operands' time from HBM (4.2
// TB/s; 5.0 when CTAs work on different K ranges); the two limits meet
// smoothly, so that of two HBM-bound candidates the one with the faster loop
// wins.
namespace {
struct BlockCost {
  int bm, bn;
  float base, s0, s1, s2, round, e0, e1, e2;
};
constexpr BlockCost kBlocks[] = {
    {128, 128, 4.10f, .328f, .514f, .531f, 4.46f, 2.08f, .152f, .362f},
    {128, 64, 3.64f, .228f, .282f, .331f, 3.56f, 1.44f, .228f, .600f},
    {64, 64, 3.18f, .151f, .184f, .185f, 1.40f, .843f, .273f, 1.02f},
    {32, 64, 3.09f, .107f, .132f, .123f, 1.25f, .814f, .503f, 1.95f},
    {32, 32, 3.13f, .0735f, .0789f, .0765f, 1.09f, .801f, .979f, 3.82f},
};
// Rows off 8 bytes (element-by-element loads through registers): a stage of
// the 256x256 kernel, and of a 64x64 block alone on its CU or sharing it with
// others (1000^2 x 1001 60.3 us in tiles, 15.8 in blocks; 2048^2 59.8 / 32.7;
// 3000^2 62.8 / about 70).  Short K: storing C counts, a round of tiles 23.5 us
// without its stages, of blocks 2.7 a CTA (10.3 and 1.6 where C's lines start at 16
// bytes).  us, tiles / blocks: 4293 x 7657 x 51 62 / 91, 2472 x 4628 x 23 30.0 /
// 38.4, 1450 x 7431 x 87 31 / 41, 1872 x 2891 x 21 24.6 / 19.6, 1141 x 4300 x 215
// 34.5 / 26.9, 7038 x 664 x 43 13.6 / 11.8.
constexpr float kMaskedTile = 3.35f, kMaskedBlock = .8f, kMaskedShared = .46f;
constexpr float kMaskedTileStore[2] = {23.5f, 10.3f}, kMaskedBlockStore[2] = {2.7f, 1.6f};
constexpr int kMinSplitStages = 4;  // stages a split keeps
// Operands that the 256 MB last-level cache does not hold, with rows off its lines:
// blocks on more than one round fetch their panels, shared lines and all, again and
// again from HBM.  f16 us, tiles / 64x64 blocks: 5421 x 905 x 18996 (240 MB) 519 /
// 578, 1332 x 3665 x 36640 839 / 993, 627 x 7008 x 37280 865 / 988; 128x64 ones: 2982
// x 1372 x 35408 902 / 976, 1402 x 3089 x 33568 749 / 800.  Below, 2319 x 1678 x 22072
// (176 MB) 592 / 503; whole lines, 1937 x 2465 x 27840 (245 MB) 570 / 548.
constexpr float kFarMB = 235.f, kFarStage = 1.25f;

int64_t up(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The cube of a block launch's estimate (the smooth maximum of its own time
// and its operands' time from HBM, without the root).
float block_cost3(const BlockCost &c, int64_t tiles, int64_t nk, int splits, int cus,
                  float hbm_mb, bool off_lines) {
  const int64_t ctas = tiles * splits, stages = up(nk, splits), load = up(ctas, cus);
  const bool far = off_lines && hbm_mb > kFarMB;
  const float stage = ctas <= cus ? c.s0 + (c.s1 - c.s0) * (float)ctas / (float)cus
                                  : c.s2 * (float)load * (far ? kFarStage : 1.f);
  float t = c.base + stage * (float)stages + (float)(load - 1) * c.round;
  if (splits > 1)
    t += c.e0 + c.e1 * (float)(ctas * (c.bm * c.bn)) * 4e-6f +
         c.e2 * (float)((splits - 1) * (c.bm * c.bn / 4096.f));
  const float hbm = c.base + hbm_mb / (splits > 1 ? 5.0f : 4.2f);
  return t * t * t + hbm * hbm * hbm;
}

// 256x256 tiles: a stage costs 1.0 (up to a quarter of the chip busy) to 1.5
// (all of it); ragged edges or a K remainder 3 more a launch.
float tile_stage(float busy, bool vec4) {
  return vec4 ? 1.0f + 0.5f * std::min(1.0f, std::max(0.0f, (busy - 0.25f) / 0.75f))
              : kMaskedTile;
}
float cube(float t) { return t * t * t; }
} // namespace

GemmPlan gemm_plan(int M, int N, int K, int cus, bool vec4, bool c_vec, int workers,
                   const SplitLimits &limits) {
  GemmPlan plan;
  // Block row and column numbers are ints with room for a block's edge; far
  // smaller shapes fill the chip with 256x256 tiles.
  if (M > (1 << 28) || N > (1 << 28))
    return plan;
  const int64_t nk = up(K, 64), big = up(M, 256) * up(N, 256), rounds = up(big, cus);
  const bool ragged = M % 256 || N % 256 || K % 64;
  float best =
      vec4 ? cube(7.f + (float)rounds * tile_stage((float)big / (float)(rounds * cus), true) *
                            (float)nk + (float)(rounds - 1) * 4.f + (ragged ? 3.f : 0.f))
           : cube(1.f + (float)rounds * (kMaskedTileStore[c_vec] + kMaskedTile * (float)nk));
  if (workers > 0) {
    // Stream-K: a worker's share of the stages, and 32 for the counter fill,
    // the publish and the reduction.
    const float t = cube(32.f + (float)(big * nk) / (float)workers *
                                    tile_stage((float)workers / (float)cus, vec4));
    if (t < best) {
      best = t;
      plan.workers = workers;
    }
  }
  const float hbm_mb = 2e-6f * (float)K * ((float)M + (float)N);
  for (const BlockCost &c : kBlocks) {
    const int64_t tiles = up(M, c.bm) * up(N, c.bn);
    // A grid holds fewer than 2^32 threads, 256 a block.
    if (tiles >= (1 << 24) || (!vec4 && (c.bm != 64 || c.bn != 64)))
      continue;
    for (int splits = 1; splits <= (vec4 ? kMaxSplits : 1); ++splits) {
      if (splits > 1 &&
          (K / 64 < splits * kMinSplitStages || tiles * splits > 2 * cus ||
           (size_t)(tiles * splits * c.bm * c.bn) * sizeof(float) > limits.slot_bytes ||
           (size_t)tiles * 2 > limits.counter_words))
        break;
      const float t =
          vec4 ? block_cost3(c, tiles, nk, splits, cus, hbm_mb, K % 64 != 0)
               : cube(c.base +
                      (float)nk * std::max(kMaskedBlock, kMaskedShared * (float)up(tiles, cus)) +
                      (float)(up(tiles, cus) - 1) * kMaskedBlockStore[c_vec]);
      if (t < best) {
        best = t;
        plan.bm = c.bm;
        plan.bn = c.bn;
        plan.splits = splits;
        plan.workers = 0;
      }
    }
  }
  return plan;
}

SplitPlan short_m_workspace(int M, int N, int K, int cus) {
  SplitPlan plan;
  if (M > 128 || N < 1024 || K % 64 != 0 || (uint64_t)K * 2u * 128u >= (1ull << 32) ||
      (uint64_t)N * K * 2u >= (1ull << 32))
    return plan;
  // Columns in blocks of 64 when they leave room for at least two splits on
  // the device's CUs, else of 128; at most 4 splits (at least 2 when the
  // columns fill the CUs 32 at a time), at least 8 stages of 64 a split;
  // none when a split keeps less than 4096 of K (2048 where M > 96 and the
  // columns fill the CUs 32 at a time).
  const int nk = K / 64;
  const int narrow = (N + 31) / 32;
  for (int bn : {64, 128}) {
    const int tiles = (N + bn - 1) / bn;
    int s = std::min(cus / tiles, 4);
    if (s < 2 && bn == 128 && narrow > cus)
      s = 2;
    while (s > 1 && nk < 8 * s)
      --s;
    if (s < 2)
      continue;
    const int ks = K / s;
    if (ks < 2048 || (ks < 4096 && (M <= 96 || narrow < cus)))
      return plan;
    plan.splits = s;
    plan.bn = bn;
    return plan;
  }
  return plan;
}

size_t short_m_slot_bytes(int N, const SplitPlan &plan) {
  return (size_t)((N + plan.bn - 1) / plan.bn) * plan.splits * 128 * plan.bn * sizeof(float);
}

size_t short_m_counter_count(int N, const SplitPlan &plan) {
  return 2 * (size_t)((N + plan.bn - 1) / plan.bn);
}

uint64_t split_tag() {
  // A counter through the output function of SplitMix64 (Steele, Lea, Flood 2014),
  // a bijection that spreads it over all 64 bits; its start comes from the
  // kernel's random source, or the clock and an address.
  static std::atomic<uint64_t> state{[] {
    uint64_t seed = 0;
    if (getrandom(&seed, sizeof seed, GRND_NONBLOCK) != (ssize_t)sizeof seed)
      seed = (uint64_t)std::chrono::steady_clock::now().time_since_epoch().count() ^
             (uint64_t)(uintptr_t)&seed << 20;
    return seed;
  }()};
  for (;;) {
    uint64_t z = state.fetch_add(0x9E3779B97F4A7C15ull, std::memory_order_relaxed);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z = (z ^ (z >> 31)) & ~(uint64_t)kCountMask;
    if (z)
      return z;
  }
}

hipError_t launch_blocks(const GemmArgs &g, const GemmPlan &plan, const BlockWorkspace &ws,
                         hipStream_t stream) {
  if (plan.bm == 0 || plan.splits < 1 ||
      (plan.splits > 1 && (!ws.slots || !ws.counters || !ws.tag || (ws.tag & kCountMask) ||
                           plan.splits > kMaxSplits || g.K / 64 < plan.splits)))
    return hipErrorInvalidValue;
  block::BlockParams p{};
  p.A = static_cast<const uint16_t *>(g.A);
  p.B = static_cast<const uint16_t *>(g.B);
  p.C = g.C;
  p.M = g.M;
  p.N = g.N;
  p.K = g.K;
  p.ldc = g.col_major ? g.M : g.N;
  p.c_vec_ok = lines_vec16(g);
  p.splits = plan.splits;
  p.slots = ws.slots;
  p.counters = ws.counters;
  p.tag = ws.tag;
  p.zero = ws.zero;
  p.zero_words = (uint32_t)ws.zero_words;
  const bool vec4 = rows_vec4(g);
  auto in = [&](auto tag) {
    constexpr int IN = decltype(tag)::value;
    if (g.out_dtype == kF32)
      return block::launch_block<IN, kF32>(p, plan.bm, plan.bn, vec4, g.col_major, stream);
    if (g.out_dtype == kF16)
      return block::launch_block<IN, kF16>(p, plan.bm, plan.bn, vec4, g.col_major, stream);
    return block::launch_block<IN, kBF16>(p, plan.bm, plan.bn, vec4, g.col_major, stream);
  };
  if (g.in_dtype == kF16)
    return in(std::integral_constant<int, kF16>{});
  return in(std::integral_constant<int, kBF16>{});
}

hipError_t launch(const GemmArgs &g, hipStream_t stream) {
  if (g.workers == 0 && !g.force_masked && !g.packed) {
    const GemmPlan plan = gemm_plan(g.M, g.N, g.K, g.cus, rows_vec4(g), lines_vec16(g), 0,
                                    SplitLimits{});
    if (plan.bm)
      return launch_blocks(g, plan, BlockWorkspace{}, stream);
  }
  Params p{};
  p.A = static_cast<const uint16_t *>(g.A);
  p.B = static_cast<const uint16_t *>(g.B);
  p.C = g.C;
  p.M = g.M;
  p.N = g.N;
  p.K = g.K;
  p.tiles_m = tiles_for(g.M);
  p.tiles_n = tiles_for(g.N);
  p.group_m = g.group_m > 0 ? g.group_m : WAVE_GEMM_GROUP_M;
  if (p.group_m > p.tiles_m)
    p.group_m = p.tiles_m;
  const bool cm = g.col_major || g.packed;
  p.ldc = cm ? g.M : g.N;
  const size_t out_bytes = g.out_dtype == kF32 ? 4 : 2;
  p.c_vec_ok = (p.ldc % 4 == 0) && aligned_to(g.C, 4 * out_bytes);
  if (g.packed) {
    p.pk = 1;
    p.pk_bm = g.pk_bm;
    p.pk_bn = g.pk_bn;
    p.pk_wmt = g.pk_wmt;
    p.pk_wnt = g.pk_wnt;
    p.pk_nblocks = g.N / (16 * g.pk_bn * g.pk_wnt);
    p.c_vec_ok = aligned_to(g.C, 4 * out_bytes);  // M % 16 == 0: whole 4-row groups
  }
  p.scratch = static_cast<float *>(g.scratch);
  p.counters = static_cast<uint32_t *>(g.counters);
  p.workers = g.workers;
  // Whole tiles take the DMA path when K is a whole number of 64-deep stages
  // (the tiled and the Stream-K kernel).
  const bool sk = g.workers > 0;
  const int stage_k = TileCfg::BK;
  const bool fast = (g.M % kTile == 0) && (g.N % kTile == 0) &&
                    (g.K % stage_k == 0) && aligned_to(g.A, 16) &&
                    aligned_to(g.B, 16) && p.c_vec_ok && !g.force_masked;
  // Ragged M / N or K off the stage: the hybrid DMA path (rows every 8
  // bytes at least, so each 16-byte DMA access is dword-aligned), unless
  // the caller forces the bounds-checked one or C is tile-packed.
  const bool hybrid = !g.force_masked && !g.packed;
  int mode = 1;
  if (fast)
    mode = 0;
  else if (g.K % 8 == 0 && aligned_to(g.A, 16) && aligned_to(g.B, 16))
    mode = hybrid ? kModeHybrid8 : 8;
  else if (g.K % 4 == 0 && aligned_to(g.A, 8) && aligned_to(g.B, 8))
    mode = hybrid ? kModeHybrid4 : 4;
  if (g.in_dtype == kF16)
    return launch_in<kF16>(p, g.out_dtype, cm, sk, mode, stream);
  return launch_in<kBF16>(p, g.out_dtype, cm, sk, mode, stream);
}

} // namespace gemm
} // namespace wave
