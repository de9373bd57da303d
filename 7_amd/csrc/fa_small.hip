// fa_small.hip -- host launch of flash_attention_f32 through the library: the
// math of fa_small.hpp (the reference's single-workgroup kernel, which the
// code objects keep) on a grid.
//
// A CTA owns 16 query rows x 16 TC output columns and takes the keys in rounds of
// one 32-key block a wave.  Every result is, bit for bit, that of one wave going
// through the blocks in order, which is what the single-workgroup kernel does:
// the waves share the round's block maxima, so each rounds its probabilities
// relative to the running max at its block, and the sums over blocks (rescale,
// then one MFMA) are done in block order by one wave a column tile.  That chain
// is short (about 45 cycles a block); scores, exp2 and loads are what the waves
// do side by side.  (Waves with running maxima of their own, merged at the end,
// round the probabilities otherwise: results 2e-4 away.)
//
// Nothing here is near a rate of the chip: a round is a chain of load -> QK ->
// maxima -> exp2 -> PV steps, with the next round's loads in flight, and four waves
// share a SIMD's VALU.  Measured (us, one workgroup / this grid): 64 queries x 1024
// keys x 64 130 / 7.9 (8 CTAs x 16 waves), 16 x 4096 x 128 957 / 35.5, 4096 x 2048 x
// 128 11700 / 29.  Keeping the query fragments in LDS lets the D = 128 step fit 128
// registers (in registers it spilled: 16 x 4096 x 128 47.8, 64 x 1024 x 64 10.9);
// maxima without LDS shuffles and masks, and the exp2 instruction for P, took 64 x
// 1024 x 64 from 8.4 to 7.9 and 1 x 4096 x 16 from 19.1 to 16.1; rounds of even length
// 64 x 600 x 48 from 5.8 to 5.3; V gathered a round ahead 64 x 1024 x 63 from 29.2 to
// 26.5.
#include "attention.hpp"
#include "fa_small.hpp"

#include <type_traits>

namespace wave {
namespace attention {

namespace {

constexpr int kSplitWaves = 16;

// ND: 32-wide steps of the head dimension held in registers (D <= 32 ND, D a
// multiple of 8, 16-byte aligned rows), or 0 for any D and alignment.
// TC: 16-column tiles a CTA owns.
// Largest of the four lanes l % 16 + 16 {0..3}, in all of them: rows of 16 lanes
// exchanged by the VALU (an xor shuffle goes through LDS and takes seven more
// instructions).
__device__ __forceinline__ float rows_max4(float v) {
  const uint32_t a = __builtin_bit_cast(uint32_t, v);
  const auto x = __builtin_amdgcn_permlane16_swap(a, a, false, false);
  v = fmaxf(__builtin_bit_cast(float, (uint32_t)x[0]), __builtin_bit_cast(float, (uint32_t)x[1]));
  const uint32_t b = __builtin_bit_cast(uint32_t, v);
  const auto y = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return fmaxf(__builtin_bit_cast(float, (uint32_t)y[0]), __builtin_bit_cast(float, (uint32_t)y[1]));
}

template <int TC> constexpr int max_waves() { return TC > 2 ? kSplitWaves / 2 : kSplitWaves; }

template <int ND, int TC>
__global__ __launch_bounds__(64 * max_waves<TC>()) void small_split_kernel(
    const _Float16 *Q, const _Float16 *K, const _Float16 *V, float *O, int block_m, int seq_n,
    int D, int col_units, uint32_t units) {
  constexpr int NF = ND > 0 ? ND : 1;
  constexpr int MAXW = max_waves<TC>();
  // What the waves leave for a round's chain, by key block: V (32 keys x 16 TC
  // columns; ND = 0: TC operands of 64 lanes), P as the product's operand, each
  // lane's sum of its P, each query's factor of the earlier sums and block max.
  __shared__ f32x4 sv[MAXW][TC][64];
  __shared__ u32x4 sp[MAXW][64], sq[NF][64];
  __shared__ float ssum[MAXW][64], salpha[MAXW][16];
  __shared__ __attribute__((aligned(16))) float smax[16][MAXW + 4];  // padded: no bank conflicts
  const uint32_t unit = blockIdx.y * gridDim.x + blockIdx.x;
  if (unit >= units)
    return;  // the whole CTA
  const int W = blockDim.x >> 6, wave = (int)uniform(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  const int q0 = (int)(unit / col_units) * 16, c0 = (int)(unit % col_units) * (16 * TC);
  const int qrow = q0 + col;
  const bool q_ok = qrow < block_m;
  const uint16_t *vh = reinterpret_cast<const uint16_t *>(V);
  const u32x4 zero4 = {0u, 0u, 0u, 0u};

  // 8 halves of row min(row, rows) at column d (d a multiple of 8), zero past the
  // rows and past D: those lanes read past the buffer, which gives zeros ((rows +
  // 1) * D < 2^30, so the bytes of row `rows` lie below 2^31).
  auto rsrc = [&](const _Float16 *base, int rows) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(base), 0,
                                             (uint32_t)rows * (uint32_t)D * 2u, 0x00020000);
  };
  const uint32_t pitch = (uint32_t)D * 2u;
  auto past = [&](int d) { return (uint32_t)((D - 8 - d) >> 31) & 0x80000000u; };
  auto chunk = [&](__amdgpu_buffer_rsrc_t r, int rows, int row, int d) {
    const uint32_t at = (uint32_t)min(row, rows) * pitch + ((uint32_t)d * 2u + past(d));
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0));
  };
  const __amdgpu_buffer_rsrc_t rk = rsrc(K, seq_n), rv = rsrc(V, seq_n);

  // One block's operands: K rows n0 + 16h + col and, as rows of 16-byte pieces
  // (ND > 0), V; piece i of a lane is row (lane + 64 i) / (2 TC), chunk
  // (lane + 64 i) % (2 TC).
  u32x4 kf[2][NF], vf[TC];
  auto load_k = [&](int n0) {
    if constexpr (ND > 0) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int key = n0 + 16 * h + col;
#pragma unroll
        for (int s = 0; s < ND; ++s)
          kf[h][s] = chunk(rk, seq_n, key, 32 * s + 8 * grp);
      }
    }
  };
  auto key_of = [&](int n0, int j) { return n0 + (j < 4 ? 4 * grp + j : 16 + 4 * grp + j - 4); };
  uint32_t vr[ND > 0 ? 1 : TC][8];  // ND = 0: the operands' halves, gathered
  auto load_v = [&](int n0) {
#pragma unroll
    for (int i = 0; i < TC; ++i) {
      if constexpr (ND > 0) {
        const int piece = lane + 64 * i, key = n0 + piece / (2 * TC);
        vf[i] = chunk(rv, seq_n, key, c0 + 8 * (piece % (2 * TC)));
      } else {
        const int c = c0 + 16 * i + col;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          vr[i][j] = vh[(size_t)min(key_of(n0, j), seq_n - 1) * D + min(c, D - 1)];
      }
    }
  };
  auto store_v = [&](int n0) {
#pragma unroll
    for (int i = 0; i < TC; ++i) {
      if constexpr (ND == 0) {
        const bool in = c0 + 16 * i + col < D;
        u32x4 w = zero4;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          w[j >> 1] |= (in && key_of(n0, j) < seq_n ? vr[i][j] : 0u) << (16 * (j & 1));
        vf[i] = w;
      }
      sv[wave][i][lane] = __builtin_bit_cast(f32x4, vf[i]);
    }
  };
  // V^T of block b of the round as the PV product's A operand: column c0 + 16t +
  // col, keys in the order the scores come out (4 grp + 0..3, 16 + 4 grp + 0..3).
  // ND > 0: through the transposing LDS read (lane 16g + i of a group receives
  // element i of the four rows that lanes 16g + 4j + 0..3 address).
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const uint32_t vbase = lds_addr(sv) + (4 * grp + (col >> 2)) * (32 * TC) + 8 * (col & 3);
  auto v_operand = [&](int b, int t) {
    if constexpr (ND > 0) {
      const uint32_t at = vbase + b * (TC * 1024) + 32 * t;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(uintptr_t)at);
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_s16x4 *)(uintptr_t)(at + 16 * 32 * TC));
      const u32x2 x = __builtin_bit_cast(u32x2, lo), y = __builtin_bit_cast(u32x2, hi);
      return u32x4{x[0], x[1], y[0], y[1]};
    } else {
      return __builtin_bit_cast(u32x4, sv[b][t][lane]);
    }
  };

  // Waves 0 .. TC-1 carry a column tile each (W >= TC) through the chain.
  const bool carries = wave < TC && c0 + 16 * wave < D;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  float m = -__builtin_inff(), l = 0.f;
  const int blocks = (seq_n - 1) / 32 + 1;
  // The query fragments, the same for every wave: in LDS, not 4 ND registers.
  u32x4 qr[NF];
  if constexpr (ND > 0) {
    if (wave == 0) {
#pragma unroll
      for (int s = 0; s < ND; ++s)
        qr[s] = chunk(rsrc(Q, block_m), block_m, qrow, 32 * s + 8 * grp);
    }
  }
  load_k(32 * wave);
  if (ND > 0 || wave < blocks)
    load_v(32 * wave);
  if constexpr (ND > 0) {
    if (wave == 0) {
#pragma unroll
      for (int s = 0; s < ND; ++s)
        sq[s][lane] = qr[s];
    }
    lds_barrier();
  }
  for (int b0 = 0; b0 < blocks; b0 += W) {
    const int here = min(W, blocks - b0);  // the round's blocks
    const bool mine = wave < here;
    const int n0 = (int)(32u * (uint32_t)(b0 + wave));
    float p[8], top = -__builtin_inff();
    if (mine) {
      f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
      auto qk = [&](int h, u32x4 k, u32x4 q) {
        s[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, k),
                                                      __builtin_bit_cast(f16x8, q), s[h], 0, 0, 0);
      };
      if constexpr (ND > 0) {
        u32x4 q[NF];
#pragma unroll
        for (int d = 0; d < ND; ++d)
          q[d] = sq[d][lane];
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            qk(h, kf[h][d], q[d]);
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
      load_k(n0 + 32 * W);  // the next round's, early; zeros past the last key
#pragma unroll
      for (int j = 0; j < 8; ++j)
        p[j] = s[j >> 2][j & 3];
      if (n0 + 31 >= seq_n) {  // the last block
#pragma unroll
        for (int j = 0; j < 8; ++j)
          p[j] = key_of(n0, j) < seq_n ? p[j] : -__builtin_inff();
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
        top = fmaxf(top, p[j]);
      top = rows_max4(top);
    }
    if (grp == 0)
      smax[col][wave] = top;  // -inf without a block
    lds_barrier();  // the round's maxima; the last round's chain is done
    float before = m;
#pragma unroll
    for (int w4 = 0; w4 < MAXW; w4 += 4) {
      if (w4 >= W)
        break;
      const f32x4 x = *reinterpret_cast<const f32x4 *>(&smax[col][w4]);
      if (w4 + 4 <= wave) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          before = fmaxf(before, x[i]);
      } else if (w4 < wave) {
#pragma unroll
        for (int i = 0; i < 3; ++i)
          before = fmaxf(before, w4 + i < wave ? x[i] : -__builtin_inff());
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        m = fmaxf(m, w4 + i < W ? x[i] : -__builtin_inff());
    }
    if (mine) {
      const float m_new = fmaxf(before, top);
      float psum = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        // Below 2^-126 the instruction gives 0 where exp2f is subnormal: nothing in
        // f16, nor in a row's sum, one of whose terms is 1.
        p[j] = __builtin_amdgcn_exp2f(p[j] - m_new);
        psum += p[j];
      }
      sp[wave][lane] = u32x4{small_pack_f16(p[0], p[1]), small_pack_f16(p[2], p[3]),
                             small_pack_f16(p[4], p[5]), small_pack_f16(p[6], p[7])};
      ssum[wave][lane] = psum;
      if (grp == 0)
        salpha[wave][col] = exp2f(before - m_new);
      store_v(n0);
      if (ND > 0 || wave < blocks - b0 - W)
        load_v(n0 + 32 * W);
    }
    lds_barrier();  // the round's P, V, sums and factors
    if (carries) {
      // N blocks from b on: their operands read together, then multiplied in order.
      auto chain = [&](int b, auto group) {
        constexpr int N = decltype(group)::value;
        u32x4 pb[N], vb[N];
        float alpha[N], psum[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
          alpha[i] = salpha[b + i][col];
          psum[i] = ssum[b + i][lane];
          pb[i] = sp[b + i][lane];
          vb[i] = v_operand(b + i, wave);
        }
#pragma unroll
        for (int i = 0; i < N; ++i) {
          l = l * alpha[i] + psum[i];
          acc *= alpha[i];
          acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, vb[i]),
                                                       __builtin_bit_cast(f16x8, pb[i]), acc, 0, 0,
                                                       0);
        }
      };
      constexpr int G = 4;
      int b = 0;
#pragma unroll 1
      for (; b + G <= here; b += G)
        chain(b, std::integral_constant<int, G>{});
#pragma unroll 1
      for (; b < here; ++b)
        chain(b, std::integral_constant<int, 1>{});
    }
  }
  if (!carries)
    return;
  const float inv = 1.0f / small_wave_sum4(l);
  if (!q_ok)
    return;
  // O^T rows are output columns: registers hold columns 4 grp .. +3.
  const int c = c0 + 16 * wave + 4 * grp;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (c + i < D)
      O[(size_t)qrow * D + c + i] = acc[i] * inv;
}

template <int TC>
hipError_t launch_tc(const _Float16 *Q, const _Float16 *K, const _Float16 *V, float *O, int block_m,
                     int seq_n, int D, hipStream_t stream) {
  const int blocks = (seq_n - 1) / 32 + 1, most = max_waves<TC>();
  // Rounds of even length.
  const int rounds = (blocks - 1) / most + 1, even = (blocks - 1) / rounds + 1;
  const int waves = even < TC ? TC : even;
  const int col_units = (D - 1) / (16 * TC) + 1;
  // At most 2^27 units (block_m * D < 2^31); a grid dimension holds fewer than 2^32
  // threads.
  const uint32_t units = ((uint32_t)(block_m - 1) / 16 + 1) * (uint32_t)col_units, row = 1u << 21;
  const dim3 grid(units < row ? units : row, (units - 1) / row + 1), block(64 * waves);
  const int64_t rows = (int64_t)(block_m > seq_n ? block_m : seq_n) + 1;
  const uintptr_t at = reinterpret_cast<uintptr_t>(Q) | reinterpret_cast<uintptr_t>(K) |
                       reinterpret_cast<uintptr_t>(V);
  const bool vec = D % 8 == 0 && at % 16 == 0 && rows * D < (1 << 30);
  auto go = [&](auto nd) {
    hipLaunchKernelGGL((small_split_kernel<decltype(nd)::value, TC>), grid, block, 0, stream, Q, K,
                       V, O, block_m, seq_n, D, col_units, units);
  };
  if (!vec || D > 128)
    go(std::integral_constant<int, 0>{});
  else if (D <= 32)
    go(std::integral_constant<int, 1>{});
  else if (D <= 64)
    go(std::integral_constant<int, 2>{});
  else if (D <= 96)
    go(std::integral_constant<int, 3>{});
  else
    go(std::integral_constant<int, 4>{});
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
