// fa_small.hip -- host launch of flash_attention_f32 through the library: the
// math of fa_small.hpp (the reference's single-workgroup kernel, which the
// code objects keep) on a grid.
//
// A CTA owns 16 query rows x 16 TC output columns; its W waves deal the
// 32-key blocks among themselves (wave w takes blocks w, w + W, ...), each with
// its own running max, row sums and accumulators, and the results are merged
// through LDS in wave order.  Nothing here is near a rate of the chip: the work
// is a chain of load -> QK -> max -> exp2 -> PV steps, so its length is what
// counts, and the loads of a wave's next block are in flight while it works on
// the current one; V goes through LDS for the transposing read (gathered 2 bytes
// a lane it took 13 us where this takes 9).  Measured (us, one workgroup / this
// grid): 64 queries x 1024 keys x 64 130 / 9.0 (8 CTAs x 16 waves), 16 x 4096 x
// 128 957 / 36, 4096 x 2048 x 128 11700 / 30.
#include "attention.hpp"
#include "fa_small.hpp"

namespace wave {
namespace attention {

namespace {

constexpr int kSplitWaves = 16;

// ND: 32-wide steps of the head dimension held in registers (D <= 32 ND, D a
// multiple of 8, 16-byte aligned rows), or 0 for any D and alignment.
// TC: 16-column tiles a CTA owns.
template <int TC> constexpr int max_waves() { return TC > 2 ? kSplitWaves / 2 : kSplitWaves; }

template <int ND, int TC>
__global__ __launch_bounds__(64 * max_waves<TC>()) void small_split_kernel(
    const _Float16 *Q, const _Float16 *K, const _Float16 *V, float *O, int block_m, int seq_n,
    int D, int col_units) {
  constexpr int NF = ND > 0 ? ND : 1;
  constexpr int MAXW = max_waves<TC>();
  // A wave's LDS: its V block of 32 keys x 16 TC columns (ND > 0), then, after
  // the loop, its sums -- both 1 KiB a tile, and no other wave's.
  __shared__ f32x4 part[MAXW][TC][64];
  __shared__ float wave_m[MAXW][16], wave_l[MAXW][16];
  const int W = blockDim.x >> 6, wave = (int)uniform(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  const int unit = blockIdx.x;
  const int q0 = unit / col_units * 16, c0 = unit % col_units * (16 * TC);
  const int qrow = q0 + col;
  const bool q_ok = qrow < block_m;
  const uint16_t *vh = reinterpret_cast<const uint16_t *>(V);
  const u32x4 zero4 = {0u, 0u, 0u, 0u};

  // 8 halves of row `row` (valid) at column d, zero past D.
  auto chunk = [&](const _Float16 *base, int row, int d) {
    return d < D ? *reinterpret_cast<const u32x4 *>(base + (size_t)row * D + d) : zero4;
  };
  u32x4 qf[NF];
  if constexpr (ND > 0) {
#pragma unroll
    for (int s = 0; s < ND; ++s)
      qf[s] = q_ok ? chunk(Q, qrow, 32 * s + 8 * grp) : zero4;
  }

  // One block's operands: K rows n0 + 16h + col and, as rows of 16-byte pieces
  // (ND > 0), V; piece i of a lane is row (lane + 64 i) / (2 TC), chunk
  // (lane + 64 i) % (2 TC).
  struct Block {
    u32x4 k[2][NF], v[TC];
  };
  auto load = [&](Block &b, int n0) {
    if constexpr (ND > 0) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int key = min(n0 + 16 * h + col, seq_n - 1);  // masked below
#pragma unroll
        for (int s = 0; s < ND; ++s)
          b.k[h][s] = chunk(K, key, 32 * s + 8 * grp);
      }
#pragma unroll
      for (int i = 0; i < TC; ++i) {
        const int piece = lane + 64 * i, key = n0 + piece / (2 * TC);
        b.v[i] = key < seq_n ? chunk(V, key, c0 + 8 * (piece % (2 * TC))) : zero4;
      }
    }
  };
  // V^T as the PV product's A operand: column c0 + 16t + col, keys in the order
  // the scores come out (4 grp + 0..3, 16 + 4 grp + 0..3).  ND > 0: through the
  // transposing LDS read (lane 16g + i of a group receives element i of the
  // four rows that lanes 16g + 4j + 0..3 address), else gathered.
  auto key_of = [&](int n0, int j) { return n0 + (j < 4 ? 4 * grp + j : 16 + 4 * grp + j - 4); };
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const uint32_t vbase = lds_addr(part) + wave * (TC * 1024);
  auto store_v = [&](const Block &b) {
#pragma unroll
    for (int i = 0; i < TC; ++i)
      part[wave][i][lane] = __builtin_bit_cast(f32x4, b.v[i]);
  };
  auto v_operand = [&](int t, int n0) {
    if constexpr (ND > 0) {
      const uint32_t row = 4 * grp + (col >> 2);
      const uint32_t at = vbase + row * (32 * TC) + 32 * t + 8 * (col & 3);
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(uintptr_t)at);
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_s16x4 *)(uintptr_t)(at + 16 * 32 * TC));
      const u32x2 a = __builtin_bit_cast(u32x2, lo), b = __builtin_bit_cast(u32x2, hi);
      return u32x4{a[0], a[1], b[0], b[1]};
    } else {
      const int c = c0 + 16 * t + col;
      u32x4 w = zero4;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = key_of(n0, j);
        const uint32_t x = vh[(size_t)min(key, seq_n - 1) * D + min(c, D - 1)];
        w[j >> 1] |= (key < seq_n && c < D ? x : 0u) << (16 * (j & 1));
      }
      return w;
    }
  };

  f32x4 acc[TC];
#pragma unroll
  for (int t = 0; t < TC; ++t)
    acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -__builtin_inff(), l = 0.f;
  const int step = 32 * W;
  Block cur, nxt;
  load(cur, 32 * wave);  // W <= blocks: every wave has one
  for (int n0 = 32 * wave; n0 < seq_n; n0 += step) {
    if (n0 + step < seq_n)
      load(nxt, n0 + step);
    if constexpr (ND > 0) {
      // The previous block's reads of this LDS are done (its values are in
      // MFMA operands); the stores below land before this block's reads.
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      store_v(cur);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    auto qk = [&](int h, u32x4 kf, u32x4 q) {
      s[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, kf),
                                                    __builtin_bit_cast(f16x8, q), s[h], 0, 0, 0);
    };
    if constexpr (ND > 0) {
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          qk(h, cur.k[h][d], qf[d]);
    } else {
      for (int d0 = 0; d0 < D; d0 += 32) {
        const u32x4 q = small_load8(Q, qrow, q_ok, d0 + 8 * grp, D, D);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int key = n0 + 16 * h + col;
          qk(h, small_load8(K, key, key < seq_n, d0 + 8 * grp, D, D), q);
        }
      }
    }
    float p[8], cmax = -__builtin_inff();
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      p[j] = key_of(n0, j) < seq_n ? s[j >> 2][j & 3] : -__builtin_inff();
      cmax = fmaxf(cmax, p[j]);
    }
    const float m_new = fmaxf(m, small_wave_max4(cmax));
    // A wave whose scores are all -inf so far contributes nothing (another
    // wave's may be finite).
    const float base = m_new == -__builtin_inff() ? 0.f : m_new;
    const float alpha = exp2f(m - base);
    m = m_new;
    float psum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      p[j] = exp2f(p[j] - base);
      psum += p[j];
    }
    l = l * alpha + psum;
    const u32x4 pf = {small_pack_f16(p[0], p[1]), small_pack_f16(p[2], p[3]),
                      small_pack_f16(p[4], p[5]), small_pack_f16(p[6], p[7])};
#pragma unroll
    for (int t = 0; t < TC; ++t) {
      acc[t] *= alpha;
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
          __builtin_bit_cast(f16x8, v_operand(t, n0)), __builtin_bit_cast(f16x8, pf), acc[t], 0, 0,
          0);
    }
    cur = nxt;
  }

  // Merge: O = sum_w 2^(m_w - m) acc_w / sum_w 2^(m_w - m) l_w, in wave order.
  l = small_wave_sum4(l);
  if (grp == 0) {
    wave_m[wave][col] = m;
    wave_l[wave][col] = l;
  }
#pragma unroll
  for (int t = 0; t < TC; ++t)
    part[wave][t][lane] = acc[t];
  __syncthreads();
  float top = -__builtin_inff();
  for (int w = 0; w < W; ++w)
    top = fmaxf(top, wave_m[w][col]);
  float total = 0.f;
  for (int w = 0; w < W; ++w)
    total += wave_l[w][col] * exp2f(wave_m[w][col] - top);
  const float inv = 1.0f / total;
  for (int t = wave; t < TC; t += W) {
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < W; ++w)
      o += part[w][t][lane] * exp2f(wave_m[w][col] - top);
    // O^T rows are output columns: registers hold columns 4 grp .. +3.
    const int c = c0 + 16 * t + 4 * grp;
    if (q_ok) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (c + i < D)
          O[(size_t)qrow * D + c + i] = o[i] * inv;
    }
  }
}

template <int TC>
hipError_t launch_tc(const _Float16 *Q, const _Float16 *K, const _Float16 *V, float *O, int block_m,
                     int seq_n, int D, hipStream_t stream) {
  const int blocks = (seq_n - 1) / 32 + 1, most = max_waves<TC>();
  const int waves = blocks < most ? blocks : most;
  const int col_units = (D - 1) / (16 * TC) + 1;
  const dim3 grid((unsigned)((block_m - 1) / 16 + 1) * (unsigned)col_units), block(64 * waves);
  const bool vec = D % 8 == 0 && ((reinterpret_cast<uintptr_t>(Q) |
                                   reinterpret_cast<uintptr_t>(K) |
                                   reinterpret_cast<uintptr_t>(V)) & 15) == 0;
  if (vec && D <= 64)
    hipLaunchKernelGGL((small_split_kernel<2, TC>), grid, block, 0, stream, Q, K, V, O, block_m,
                       seq_n, D, col_units);
  else if (vec && D <= 128)
    hipLaunchKernelGGL((small_split_kernel<4, TC>), grid, block, 0, stream, Q, K, V, O, block_m,
                       seq_n, D, col_units);
  else
    hipLaunchKernelGGL((small_split_kernel<0, TC>), grid, block, 0, stream, Q, K, V, O, block_m,
                       seq_n, D, col_units);
  return hipGetLastError();
}

} // namespace

hipError_t launch_small(const void *Q, const void *K, const void *V, float *O,
                        int block_m, int seq_n, int head_dim, hipStream_t stream) {
  const _Float16 *q = static_cast<const _Float16 *>(Q), *k = static_cast<const _Float16 *>(K),
                 *v = static_cast<const _Float16 *>(V);
  // 32 columns a CTA while those CTAs fit the chip (each computes its rows'
  // scores again), 128 beyond.
  const int64_t narrow = (int64_t)((block_m - 1) / 16 + 1) * ((head_dim - 1) / 32 + 1);
  return narrow <= 512 ? launch_tc<2>(q, k, v, O, block_m, seq_n, head_dim, stream)
                       : launch_tc<8>(q, k, v, O, block_m, seq_n, head_dim, stream);
}

} // namespace attention
} // namespace wave
