// attention_fwd.hip -- instantiation and host launch of the gfx950
// flash-attention forward kernels: the 12-wave three-group kernel
// (attention_fwd3.hpp), the 8-wave ping-pong kernel (attention_kernels.hpp)
// and the 4-wave kernel (attention_fwd4.hpp).
#include "attention_fwd3.hpp"
#include "attention_fwd4.hpp"
#include "attention_kernels.hpp"

#include <algorithm>
#include <cmath>

namespace wave {
namespace attention {

hipError_t launch_fwd(const FwdArgs &a, hipStream_t stream) {
  Params p{};
  p.Q = static_cast<const uint16_t *>(a.Q);
  p.K = static_cast<const uint16_t *>(a.K);
  p.V = static_cast<const uint16_t *>(a.V);
  p.O = static_cast<uint16_t *>(a.O);
  p.batch = a.batch;
  p.q_heads = a.q_heads;
  p.kv_heads = a.kv_heads;
  p.seq_q = a.seq_q;
  p.seq_k = a.seq_k;
  // The default (8 waves a 256-row block, one CTA a CU) gives way to the 4-wave
  // kernel on 128-row blocks where those are at most one a CU (half as many
  // 256-row ones would leave CUs idle: B1 Hq32 Hkv8 S1000 causal bf16 30.1 -> 25.2
  // us, B1 H8 S512 16.8 -> 13.0, B1 H16 S1024 28.8 -> 23.1; at 384 blocks of 128
  // the 8-wave kernel is ahead, 24.8 / 28.0), or where, on more than one
  // round of 256-row blocks, they save more padded rows than their rate costs
  // (about 13 % behind on a full chip: B8 H64 S300 57.9 -> 43.3, B7 H11 S777
  // causal 54.1 -> 34.4, S1024 level; within one round the 8-wave kernel keeps
  // ahead, B1 H61 S640 24.3 / 25.7).
  // Causal blocks are of uneven length: where the heads divide over the XCDs they
  // go by length (block_coords).  8-wave kernel, head by head -> by length:
  // B1 Hq32 Hkv32 S3000 107 -> 84 us, B4 H16 S2048 104 -> 78, B2 Hq32 Hkv8
  // S4096 309 -> 277, B1 Hq64 Hkv8 S8192 1013 -> 979.  The heads then side by
  // side read their K and V at once, which the 256 MB last-level cache has to
  // hold: 32 MB in all (B1 Hq32 Hkv4 S16384) 1965 -> 1937 us, 256 MB (B4 H32
  // S4096, B8 H32 S2048) 623 -> 587 and 383 -> 351, 512 MB (B2 H64 S8192) 2063 ->
  // 2228.  In long and short pairs the 4-wave kernel's blocks are ahead up to two
  // of them a CU: B2 Hq16 Hkv4 S2048 59 (8-wave, head by head), 53 (8-wave, by
  // length), 47 (pairs); B1 H16 S4096 103, 98, 91; with four a CU B1 Hq64 Hkv8
  // S2048 114, 77, 82.  One block a CU has nothing to order (B1 Hq32 Hkv8 S1000 3 %
  // slower by length).
  const int64_t heads = (int64_t)a.batch * a.q_heads;
  const int64_t n128 = ((a.seq_q - 1) / kF4PassRows + 1) * heads,
                n256 = ((a.seq_q - 1) / 256 + 1) * heads;
  const int64_t kv_bytes = (int64_t)a.batch * a.kv_heads * a.seq_k * (2 * kKRowBytes);
  bool by_length = a.causal && heads % 8 == 0 && kv_bytes <= (256 << 20);
  const bool narrow = a.waves == kPPWaves && (n128 <= (by_length ? 2 * a.cus : a.cus) ||
                                              (n256 > a.cus && 113 * n128 < 200 * n256));
  // 256-row blocks of short sequences do little work on each K and V row: half of
  // that cache (B48 H16 S448, 176 MB, 126 head by head, 134 by length; B64 Hq32 Hkv8
  // S768, 201 MB, 562, 600; below, B64 Hq32 Hkv8 S512, 134 MB, level).
  if (!narrow && a.seq_k < 1024 && kv_bytes > (128 << 20))
    by_length = false;
  const int rows = a.waves == kR3Waves ? kR3Rows
                   : narrow            ? kF4PassRows
                                       : 32 * kPPWaves;  // 4 waves: two passes of 128
  p.q_blocks = (a.seq_q + rows - 1) / rows;
  p.by_length = !by_length || p.q_blocks * heads <= a.cus ? 0
                : narrow                                  ? std::max(a.cus / 8, 1)
                                                          : 1;
  p.causal = a.causal;
  const float scale = a.scale > 0.f ? a.scale : 1.0f / std::sqrt((float)a.head_dim);
  p.scale_log2 = scale * kLog2e;
  p.lse = a.lse;
  // Fixed-max mode: |s * scale| <= head_dim * qk_max_abs^2 * scale, in log2
  // units (wave_flash_attention.py:108-113 with scale = 1/sqrt(128)).
  p.fixed_max = (float)((double)kLog2e * scale * a.head_dim * a.qk_max_abs * a.qk_max_abs);
  const bool fixed = a.qk_max_abs > 0.f;
  if (a.waves == kF4Waves || narrow) {
    // 4 waves x 32 query rows per pass, two passes a CTA (the same 256-row
    // blocks) or one.
    const dim3 grid(p.q_blocks * a.batch * a.q_heads), block(64 * kF4Waves);
    auto go = [&](auto dt, auto fix) {
      constexpr int DT = decltype(dt)::value;
      constexpr bool FIXED = decltype(fix)::value;
      if (narrow)
        hipLaunchKernelGGL((fwd4_kernel<DT, FIXED, 1>), grid, block, 0, stream, p);
      else
        hipLaunchKernelGGL((fwd4_kernel<DT, FIXED, 2>), grid, block, 0, stream, p);
    };
    if (a.dtype == kF16)
      fixed ? go(I_<kF16>{}, std::true_type{}) : go(I_<kF16>{}, std::false_type{});
    else
      fixed ? go(I_<kBF16>{}, std::true_type{}) : go(I_<kBF16>{}, std::false_type{});
    return hipGetLastError();
  }
  if (a.waves == kR3Waves) {
    // 12 waves x 32 query rows per CTA, three rotating groups of 4 waves.
    const dim3 grid(p.q_blocks * a.batch * a.q_heads), block(64 * kR3Waves);
    if (a.dtype == kF16) {
      if (fixed)
        hipLaunchKernelGGL((fwd3_kernel<kF16, true>), grid, block, 0, stream, p);
      else
        hipLaunchKernelGGL((fwd3_kernel<kF16, false>), grid, block, 0, stream, p);
    } else {
      if (fixed)
        hipLaunchKernelGGL((fwd3_kernel<kBF16, true>), grid, block, 0, stream, p);
      else
        hipLaunchKernelGGL((fwd3_kernel<kBF16, false>), grid, block, 0, stream, p);
    }
    return hipGetLastError();
  }
  // 8 waves x 32 query rows per CTA, two ping-pong groups of 4 waves.
  const dim3 grid(p.q_blocks * a.batch * a.q_heads), block(64 * kPPWaves);
  if (a.dtype == kF16) {
    if (fixed)
      hipLaunchKernelGGL((fwd_pp_kernel<kF16, true>), grid, block, 0, stream, p);
    else
      hipLaunchKernelGGL((fwd_pp_kernel<kF16, false>), grid, block, 0, stream, p);
  } else {
    if (fixed)
      hipLaunchKernelGGL((fwd_pp_kernel<kBF16, true>), grid, block, 0, stream, p);
    else
      hipLaunchKernelGGL((fwd_pp_kernel<kBF16, false>), grid, block, 0, stream, p);
  }
  return hipGetLastError();
}

} // namespace attention
} // namespace wave
