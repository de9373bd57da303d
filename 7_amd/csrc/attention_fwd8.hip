// attention_fwd8.hip -- host launch of the block-scaled FP8 flash-attention
// forward (attention_fwd8.hpp).
#include "attention_fwd8.hpp"

#include <cmath>

namespace wave {
namespace attention {

hipError_t launch_fwd_fp8(const Fp8FwdArgs &a, hipStream_t stream) {
  Fp8Params p{};
  p.Q = static_cast<const uint8_t *>(a.Q);
  p.K = static_cast<const uint8_t *>(a.K);
  p.V = static_cast<const uint8_t *>(a.V);
  p.Qs = static_cast<const uint8_t *>(a.Q_scale);
  p.Ks = static_cast<const uint8_t *>(a.K_scale);
  p.Vs = static_cast<const uint8_t *>(a.V_scale);
  p.O = static_cast<uint16_t *>(a.O);
  p.batch = a.batch;
  p.q_heads = a.q_heads;
  p.kv_heads = a.kv_heads;
  p.seq_q = a.seq_q;
  p.seq_k = a.seq_k;
  p.q_blocks = (a.seq_q + k8Rows - 1) / k8Rows;
  p.causal = a.causal;
  const float scale = a.scale > 0.f ? a.scale : 1.0f / std::sqrt((float)kD);
  p.scale_log2 = scale * kLog2e;
  p.lse = a.lse;
  // Causal blocks by length where the heads divide over the XCDs and K and V, which
  // the heads side by side read at once, fit the 256 MB last-level cache, as in
  // launch_fwd.  Head by head -> by length: B2 Hq32 Hkv8 S2048 85.8 -> 55.6 us (two
  // blocks a CU, a long and a short one), B1 H32 S3000 81.7 -> 58.5, B4 H32 S4096
  // 421 -> 344, B2 H64 S8192 (256 MB) 1442 -> 1285; one block a CU level.  Not up to
  // 384 rows, whose two blocks are of nearly one length (B48 H16 S384 69 -> 74), and
  // below 1024 to three quarters of that cache (B120 H12 S640, 236 MB, 261 -> 277;
  // S512, 189 MB, 208 -> 176).
  const int64_t heads = (int64_t)a.batch * a.q_heads;
  const int64_t kv_bytes = (int64_t)a.batch * a.kv_heads * a.seq_k * (2 * kD);
  p.by_length = a.causal && heads % 8 == 0 && a.seq_q > 384 &&
                kv_bytes <= ((a.seq_k < 1024 ? 192 : 256) << 20);
  const dim3 grid(p.q_blocks * a.batch * a.q_heads), block(64 * k8Waves);
  if (a.out_dtype == kF16) {
    if (a.causal)
      hipLaunchKernelGGL((fwd8_kernel<kF16, true>), grid, block, 0, stream, p);
    else
      hipLaunchKernelGGL((fwd8_kernel<kF16, false>), grid, block, 0, stream, p);
  } else {
    if (a.causal)
      hipLaunchKernelGGL((fwd8_kernel<kBF16, true>), grid, block, 0, stream, p);
    else
      hipLaunchKernelGGL((fwd8_kernel<kBF16, false>), grid, block, 0, stream, p);
  }
  return hipGetLastError();
}

} // namespace attention
} // namespace wave
