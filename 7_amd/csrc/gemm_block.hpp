#pragma once
// gemm_block.hpp -- C = A . B^T in small blocks: the products whose 256x256
// tiles (gemm_kernels.hpp) would leave most of the chip's CUs idle, and the
// short-M ones bound by streaming B.
//
// Bound by what a CU's DMA fetches (80 to 110 GB/s, an LDS ring of any depth)
// and, from 256 CTAs of 128x128 on, by the matrix cores (without the DMA
// 2048^2 x 8192 takes 55 us of its 64).  So the block is the largest that
// still gives every CU one, down to 32x32, where half of a stage is operand
// A.  Measured (f16, us, 256x256 tiles or Stream-K or 32-column kernel / these
// blocks): 32x32x64 7.6 / 3.7, 256^2 x 8192 77 / 10.3, 512^3 14.6 / 3.8,
// 1024^3 22.3 / 5.8, 2048^3 39.8 / 19.5, 2048^2 x 8192 91 / 64, 16 x 4096 x
// 4096 15.7 / 7.7, 128 x 2048 x 8192 32.6 / 16.1, 8192 x 512 x 4096 62 / 34.
// A K loop that starts at another stage in each CTA (to spread HBM channels)
// loses the panels that CTAs share in L2: 2048^2 x 8192 67 / 135.
//
// One CTA (4 waves) owns a BM x BN block of C over one of `splits` contiguous
// K ranges.  K is consumed 64 deep per LDS stage (A rows, then B rows, 128
// bytes each, 16-byte chunks XOR-swizzled by row so that the 32 rows of one
// fragment read cover all banks); NS stages form a ring filled by
// global->LDS DMA.  Wave w computes an RM x RN part of the block (WM x WN
// waves) on 32x32x16 MFMAs from one of two register sets: while stage k is
// multiplied out of one, stage k + 1 is read into the other.  One barrier a
// stage, at its start: there every wave holds stage k in registers, so the
// barrier frees the slot for stage k + NS, and stage k + 1 has landed.
//
// Rows past M and N are fetched from the last valid row (their products only
// reach elements of C that are never stored).  The K remainder (K % 64) is
// loaded into registers before the ring starts, zero past K, and written to
// LDS and multiplied after the last whole stage, so its latency hides under
// the main loop.  VEC 1 (K not a multiple of 4, or rows not 8-byte aligned)
// has no DMA: every stage goes through registers with bounds checks.
//
// splits > 1: each contributor of a block takes an arrival ticket when its K
// range is done.  All but the last store their fp32 partials to their slot
// with device-coherent stores and, once those are acknowledged, count
// themselves published; the last waits for that count, reads the partials
// with device-coherent loads and sums them in split order (its own from its
// accumulators), so the result does not depend on arrival order.  Counter
// words are 64-bit: the launch's tag (split_tag(), nonzero) in the high 60 bits,
// a count in the low four; a word with any other tag counts as zero, so a
// workspace needs no clearing, and the last arriver leaves zeros, which keeps
// replays of a captured launch (a fixed tag) correct.  Tags are drawn from all
// of their 60 bits, so a word that holds anything else (partial sums of another
// shape, recycled memory) matches with a chance of 2^-60.

#include "gemm.hpp"
#include "gemm_kernels.hpp"

namespace wave {
namespace gemm {
namespace block {

constexpr int kBK = 64;
constexpr int kRB = 128;  // bytes per operand row per stage

typedef unsigned long long u64;

struct BlockParams {
  const uint16_t *A, *B;
  void *C;
  int M, N, K, ldc;
  int c_vec_ok;          // C's lines start at multiples of 16 bytes
  int tiles_m, tiles_n, group_m;
  int splits;
  float *slots;          // [tiles * splits][BM * BN] (splits > 1)
  u64 *counters;         // [tiles][2] arrived, published (tag | count)
  u64 tag;               // split_tag() of this launch
  u64 *zero;             // zero_words words left zero (BlockWorkspace)
  uint32_t zero_words;
};

// WM x WN x WK waves: WK > 1 deals a stage's four 16-deep slices over WK
// waves of the same part, summed through LDS after the K loop.
template <int BM_, int BN_> struct BlockCfg {
  static constexpr int BM = BM_, BN = BN_;
  static constexpr int WN = BN == 32 ? 1 : 2;
  static constexpr int WM = BM == 32 ? 1 : 2, WK = 4 / (WM * WN);
  static_assert(WM * WN * WK == 4, "four waves");
  static constexpr int KS = 4 / WK;                     // slices a wave multiplies
  static constexpr int OWNERS = 64 * WM * WN;           // threads that hold the block's sums
  static constexpr int RM = BM / WM, RN = BN / WN;      // a wave's part
  static_assert(RM % 32 == 0 && RN % 32 == 0, "whole MFMA tiles");
  static constexpr int TI = RM / 32, TJ = RN / 32;
  static constexpr int NG = TI * TJ * 4;                // 16-byte groups of a wave's part
  static constexpr int AB = BM * kRB, STAGE = AB + BN * kRB;
  // Blocks up to 64x64 run two CTAs a CU (80 KiB each), larger ones a 120 or
  // 128 KiB ring.  (All 160 KiB for one CTA measured no faster: the loop is
  // bound by what a CU's DMA fetches, about 80 to 110 GB/s.)
  static constexpr int OCC = BM * BN <= 64 * 64 ? 2 : 1;
  static constexpr int NS = (OCC == 2 ? 80 : 128) * 1024 / STAGE;
  static constexpr int AI = BM / 32, BI = BN / 32;      // DMA issues per wave a stage
  static constexpr int DMA = AI + BI;
  static constexpr int SLOT = BM * BN;                  // floats per partial slot
  // Up to SHORT stages go without the ring, whose other slots would be filled for
  // nothing: 1 x 6976 x 64 3.32 -> 3.12 us (rocprofv3), 64 x 5696 x 128 3.64 -> 3.40,
  // 32 x 4096 x 256 3.72 -> 3.36; 1536 x 2048 x 256 in blocks of 128x128 6.92 -> 7.16,
  // so two stages there.
  static constexpr int SHORT = OCC == 2 ? 4 : 2;
  static_assert(SHORT <= NS, "a slot a stage");
  static_assert(DMA * (NS - 2) < 64, "vmcnt budget");
};

__device__ __forceinline__ uint32_t sw8(uint32_t r) { return (r ^ (r >> 3)) & 7u; }

__device__ __forceinline__ uint32_t tag_count(u64 w, u64 tag) {
  return (w & ~kCountMask) == tag ? (uint32_t)(w & kCountMask) : 0u;
}
// Counts one arrival on *c for this launch and returns the count before it.
// The first guess is the zero every launch leaves, so the common first
// arrival takes one atomic round trip; each failed exchange means another
// contributor's succeeded (at most splits - 1) or the word was stale.
__device__ __forceinline__ uint32_t tag_increment(u64 *c, u64 tag) {
  u64 old = 0;
  for (;;) {
    const uint32_t n = tag_count(old, tag);
    if (__hip_atomic_compare_exchange_strong(c, &old, tag | (n + 1u),
                                             __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT))
      return n;
  }
}

template <class X, int IN_DT, int OUT_DT, bool COL_MAJOR, int VEC>
__global__ __launch_bounds__(256, X::OCC) void block_kernel(BlockParams p) {
  constexpr int TI = X::TI, TJ = X::TJ, NG = X::NG, NS = X::NS;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[NS * X::STAGE];
  const uint32_t wave = uniform(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63;
  // Workgroup i runs on XCD i % 8: renumber so that one XCD's CTAs are
  // consecutive (the first gridDim % 8 XCDs hold one more); a block's splits
  // are consecutive then, and blocks run in bands of group_m, which share
  // operand panels in that XCD's L2.
  const uint32_t xcd = blockIdx.x & 7;
  const int id = (int)(xcd * (gridDim.x >> 3) + min(xcd, gridDim.x & 7) + (blockIdx.x >> 3));
  for (uint32_t w = blockIdx.x * 256 + threadIdx.x; w < p.zero_words; w += gridDim.x * 256)
    p.zero[w] = 0ull;
  const int tile = id / p.splits, split = id - tile * p.splits;
  int tm, tn;
  tile_coords(tile, p.tiles_m, p.tiles_n, p.group_m, false, tm, tn);
  const int m0 = __builtin_amdgcn_readfirstlane(tm * X::BM);
  const int n0 = __builtin_amdgcn_readfirstlane(tn * X::BN);
  const int nk = p.K / kBK;  // whole stages, dealt evenly over the splits
  const int q = nk / p.splits, rem = nk - q * p.splits;
  const int k0 = split * q + min(split, rem);
  const int len = q + (split < rem ? 1 : 0);
  // The K remainder belongs to the last split.
  const bool tail = (p.K % kBK) != 0 && split == p.splits - 1;
  const uint32_t rowbytes = (uint32_t)p.K * 2u;

  // Chunk copies of a stage: copy i of this wave covers local rows R = 8 *
  // (wave * AI + i) + lane / 8 of A (i < AI), then of B, 8 lanes a row; lane
  // slot lane % 8 of row R holds chunk (lane % 8) ^ sw8(R).
  const uint32_t slot8 = lane & 7, row8 = lane >> 3;
  auto a_row = [&](int i) { return (wave * X::AI + i) * 8 + row8; };
  auto b_row = [&](int i) { return (wave * X::BI + i) * 8 + row8; };
  const uint32_t ring = lds_addr(smem);

  // Registers of one stage's chunks, zero past K.
  u32x4 va[X::AI], vb[X::BI];
  auto load_regs = [&](int kt) {
#pragma unroll
    for (int i = 0; i < X::AI; ++i) {
      const uint32_t R = a_row(i);
      const int kc = kt * kBK + (int)((slot8 ^ sw8(R)) * 8);
      const uint16_t *row = p.A + (size_t)min(m0 + (int)R, p.M - 1) * p.K;
      va[i] = VEC == 4 ? load_chunk_k4(row, kc, p.K) : load_chunk<1>(row, kc, p.K);
    }
#pragma unroll
    for (int i = 0; i < X::BI; ++i) {
      const uint32_t R = b_row(i);
      const int kc = kt * kBK + (int)((slot8 ^ sw8(R)) * 8);
      const uint16_t *row = p.B + (size_t)min(n0 + (int)R, p.N - 1) * p.K;
      vb[i] = VEC == 4 ? load_chunk_k4(row, kc, p.K) : load_chunk<1>(row, kc, p.K);
    }
  };
  auto store_regs = [&](int s) {
    uint8_t *st = smem + s * X::STAGE + lane * 16;
#pragma unroll
    for (int i = 0; i < X::AI; ++i)
      *reinterpret_cast<u32x4 *>(st + (wave * X::AI + i) * 1024) = va[i];
#pragma unroll
    for (int i = 0; i < X::BI; ++i)
      *reinterpret_cast<u32x4 *>(st + X::AB + (wave * X::BI + i) * 1024) = vb[i];
  };

  // Fragments: MFMA tile i of the wave's rows / j of its columns, lane row
  // lane % 32, K half lane / 32 of a 16-deep slice.
  const uint32_t wk = wave / (X::WM * X::WN);
  const uint32_t wm = wave / X::WN % X::WM, wn = wave % X::WN;
  const uint32_t rr = lane & 31, h = lane >> 5;
  uint32_t offa[TI], swa[TI], offb[TJ], swb[TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i) {
    const uint32_t ra = wm * X::RM + i * 32 + rr;
    offa[i] = ra * kRB;
    swa[i] = sw8(ra) ^ h;
  }
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    const uint32_t rb = wn * X::RN + j * 32 + rr;
    offb[j] = X::AB + rb * kRB;
    swb[j] = sw8(rb) ^ h;
  }
  // Fragments of one whole stage: the wave's 16-deep slices of its rows.
  struct Frag {
    u32x4 a[X::KS][TI], b[X::KS][TJ];
  };
  constexpr int NR = X::KS * (TI + TJ);  // LDS reads a stage
  auto read1 = [&](Frag &f, int s, int r) {
    const uint8_t *st = smem + s * X::STAGE;
    const int kk = r / (TI + TJ), t = r % (TI + TJ);
    const uint32_t x = 2 * (wk * X::KS + kk);
    if (t < TI)
      f.a[kk][t] = *reinterpret_cast<const u32x4 *>(st + offa[t] + ((x ^ swa[t]) << 4));
    else
      f.b[kk][t - TI] =
          *reinterpret_cast<const u32x4 *>(st + offb[t - TI] + ((x ^ swb[t - TI]) << 4));
  };
  auto read = [&](Frag &f, int s) {
#pragma unroll
    for (int r = 0; r < NR; ++r)
      read1(f, s, r);
  };
  f32x16 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
      acc[i][j] = f32x16{};
  // The stage's NM MFMAs, each followed by its share of other work: hook(m).
  constexpr int NM = X::KS * TI * TJ;
  auto multiply = [&](const Frag &f, auto hook) {
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const int kk = m / (TI * TJ), i = (m / TJ) % TI, j = m % TJ;
      // Row-major C: MFMA rows = n (B), columns = m (A); column-major: swapped.
      acc[i][j] = COL_MAJOR ? mfma32x32x16<IN_DT>(f.a[kk][i], f.b[kk][j], acc[i][j])
                            : mfma32x32x16<IN_DT>(f.b[kk][j], f.a[kk][i], acc[i][j]);
      hook(m);
    }
  };
  auto whole_stage = [&](int s) {
    Frag f;
    read(f, s);
    multiply(f, [](int) {});
  };

  if constexpr (VEC == 4) {
    if (tail)
      load_regs(nk);
    if (len > 0) {
      uint32_t goa[X::AI], gob[X::BI];
#pragma unroll
      for (int i = 0; i < X::AI; ++i) {
        const uint32_t R = a_row(i);
        goa[i] = min(R, (uint32_t)(p.M - 1 - m0)) * rowbytes + ((slot8 ^ sw8(R)) << 4);
      }
#pragma unroll
      for (int i = 0; i < X::BI; ++i) {
        const uint32_t R = b_row(i);
        gob[i] = min(R, (uint32_t)(p.N - 1 - n0)) * rowbytes + ((slot8 ^ sw8(R)) << 4);
      }
      const char *a0 = reinterpret_cast<const char *>(p.A) + (size_t)m0 * rowbytes;
      const char *b0 = reinterpret_cast<const char *>(p.B) + (size_t)n0 * rowbytes;
      // DMA d of stage k of this CTA's range into slot s.  Past the last stage
      // every lane fetches the block's first 16 bytes instead (one cache line
      // an instruction): each iteration issues one stage, so the vmcnt budget
      // is constant, and a short K range costs no second fetch of its stages.
      auto issue1 = [&](int s, int k, int d) {
        const uint32_t l = ring + s * X::STAGE;
        const bool in = k < len;
        const uint32_t keep = in ? ~0u : 0u;
        const size_t at = in ? (size_t)(k0 + k) * kRB : 0;
        if (d < X::AI)
          dma16(l + (wave * X::AI + d) * 1024, a0 + at, goa[d] & keep);
        else
          dma16(l + X::AB + (wave * X::BI + d - X::AI) * 1024, b0 + at, gob[d - X::AI] & keep);
      };
      asm volatile("" ::: "memory");  // the remainder's loads stay ahead of the DMA
      if (len <= X::SHORT) {
        // A few stages: no ring to fill behind them.
        for (int s = 0; s < len; ++s)
#pragma unroll
          for (int d = 0; d < X::DMA; ++d)
            issue1(s, s, d);
        vm_wait_barrier();
        for (int s = 0; s < len; ++s)
          whole_stage(s);
        lds_barrier();  // every wave is done with the ring
      } else {
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
          for (int d = 0; d < X::DMA; ++d)
            issue1(s, s, d);
        vm_wait_barrier<X::DMA *(NS - 1)>();
        // Stage k from registers, stage k + 1 read into the other set and stage
        // k + NS issued into stage k's slot, spread over the MFMAs (the reads
        // over the first three quarters, so that the next barrier finds them
        // done).
        constexpr int RM = NM * 3 / 4 > 0 ? NM * 3 / 4 : 1;
        int s = 0;
        auto step = [&](const Frag &cur, Frag &nxt, int k) {
          // Stage k + 1 has landed (stages k + 2 .. k + NS - 1 may be in
          // flight) and every wave holds stage k in registers.
          vm_wait_barrier<X::DMA *(NS - 2)>();
          const int free_slot = s;
          s = s == NS - 1 ? 0 : s + 1;
          multiply(cur, [&](int m) {
#pragma unroll
            for (int r = 0; r < NR; ++r)
              if (r * RM / NR == m)
                read1(nxt, s, r);
#pragma unroll
            for (int d = 0; d < X::DMA; ++d)
              if (d * NM / X::DMA == m)
                issue1(free_slot, k + NS, d);
            __builtin_amdgcn_sched_barrier(0);
          });
        };
        Frag f[2];
        read(f[0], 0);
        int k = 0;
        for (; k + 1 < len; k += 2) {
          step(f[0], f[1], k);
          step(f[1], f[0], k + 1);  // past the last stage the reads go unused
        }
        if (k < len)
          multiply(f[0], [](int) {});
        vm_wait_barrier();  // the DMA past the end, before the ring is written again
      }
    }
    if (tail) {
      store_regs(0);
      lds_barrier();
      whole_stage(0);
    }
  } else {
    const int end = k0 + len + (tail ? 1 : 0);
    if (k0 < end) {
      load_regs(k0);
      store_regs(0);
      lds_barrier();
      for (int k = k0; k < end; ++k) {
        if (k + 1 < end)
          load_regs(k + 1);
        whole_stage((k - k0) & 1);
        if (k + 1 < end)
          store_regs((k + 1 - k0) & 1);
        lds_barrier();
      }
    }
  }

  // 16-byte group g (0 .. NG-1) of the thread's part: MFMA tile (g / (4 TJ),
  // g / 4 % TJ), accumulator registers 4 * (g % 4) .. +3.
  auto group = [&](int g) {
    const f32x16 &a = acc[g / (4 * TJ)][(g / 4) % TJ];
    const int e = g & 3;
    return f32x4{a[4 * e], a[4 * e + 1], a[4 * e + 2], a[4 * e + 3]};
  };
  f32x4 out[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g)
    out[g] = group(g);
  // WK > 1: the waves of slice set 0 add the others' sums, in order; only
  // they hold the block from here on.
  const bool owner = X::WK == 1 || wk == 0;
  if constexpr (X::WK > 1) {
    f32x4 *sums = reinterpret_cast<f32x4 *>(smem);
    lds_barrier();  // every wave is done with the ring
    if (!owner) {
#pragma unroll
      for (int g = 0; g < NG; ++g)
        sums[g * 256 + threadIdx.x] = out[g];
    }
    lds_barrier();
    if (owner) {
#pragma unroll
      for (int w = 1; w < X::WK; ++w)
#pragma unroll
        for (int g = 0; g < NG; ++g)
          out[g] += sums[g * 256 + w * X::OWNERS + threadIdx.x];
    }
  }
  if (p.splits > 1) {
    // The ticket goes through the ring's first word (a separate LDS word would
    // push two 80 KiB rings past the CU's 160 KiB): every wave is done with it.
    uint32_t *arrival = reinterpret_cast<uint32_t *>(smem);
    __syncthreads();
    if (threadIdx.x == 0)
      *arrival = tag_increment(&p.counters[2 * tile], p.tag);
    __syncthreads();
    if (*arrival != (uint32_t)p.splits - 1) {
      const __amdgpu_buffer_rsrc_t mine =
          coherent_rsrc(p.slots + (size_t)id * X::SLOT, X::SLOT * 4);
      if (owner) {
#pragma unroll
        for (int g = 0; g < NG; ++g)
          coherent_store16(mine, (g * X::OWNERS + threadIdx.x) * 16, out[g]);
      }
      // Every wave's stores are acknowledged at the coherence point before
      // the barrier, so thread 0's count, issued after it, needs no release.
      vm_wait_barrier();
      if (threadIdx.x == 0)
        tag_increment(&p.counters[2 * tile + 1], p.tag);
      return;
    }
    // Every other contributor has its ticket, so it is resident and publishes
    // without waiting on anything: the wait ends.  It is bounded all the same
    // (2^20 polls, about a second), for a counter word that already held this
    // launch's tag (a chance of 2^-60 a word for arbitrary contents).
    if (threadIdx.x == 0) {
      for (uint32_t poll = 0;
           poll < (1u << 20) &&
           tag_count(__hip_atomic_load(&p.counters[2 * tile + 1], __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT),
                     p.tag) != (uint32_t)p.splits - 1;
           ++poll)
        __builtin_amdgcn_s_sleep(1);
      __hip_atomic_store(&p.counters[2 * tile], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(&p.counters[2 * tile + 1], 0ull, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    // The others' partials in split order (other o is split o + (o >= split)),
    // KB of them in flight at once, this CTA's accumulators at their place.
    constexpr int KB = 32 / NG > 4 ? 4 : 32 / NG;
    const __amdgpu_buffer_rsrc_t peers = coherent_rsrc(
        p.slots + (size_t)tile * p.splits * X::SLOT, (uint32_t)p.splits * X::SLOT * 4);
    const int others = owner ? p.splits - 1 : 0;
    f32x4 sum[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g)
      sum[g] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int o0 = 0; o0 < others; o0 += KB) {
      f32x4 x[KB][NG];
#pragma unroll
      for (int b = 0; b < KB; ++b) {
        if (o0 + b < others) {
          const uint32_t c = o0 + b + (o0 + b >= split ? 1 : 0);
#pragma unroll
          for (int g = 0; g < NG; ++g)
            x[b][g] = coherent_load16(peers, c * (X::SLOT * 4) + threadIdx.x * 16,
                                      g * X::OWNERS * 16);
        }
      }
#pragma unroll
      for (int b = 0; b < KB; ++b) {
        if (o0 + b < others) {
          if (o0 + b == split) {
#pragma unroll
            for (int g = 0; g < NG; ++g)
              sum[g] += out[g];
          }
#pragma unroll
          for (int g = 0; g < NG; ++g)
            sum[g] += x[b][g];
        }
      }
    }
#pragma unroll
    for (int g = 0; g < NG; ++g)
      out[g] = split == others ? sum[g] + out[g] : sum[g];
  }

  // Store through LDS: each group holds 4 consecutive values along C's
  // contiguous dimension P, but a store instruction of them would touch 32
  // lines with 8 or 16 bytes each.  The block is laid out as QB lines of PB
  // values (16-byte chunk c of line q at c ^ (q mod CH)) and written as runs of
  // whole lines, 16 bytes a lane.
  constexpr int OB = OUT_DT == kF32 ? 4 : 2;
  constexpr int PB = COL_MAJOR ? X::BM : X::BN, QB = COL_MAJOR ? X::BN : X::BM;
  constexpr int LINE = PB * OB, CH = LINE / 16, EPC = 16 / OB;
  constexpr int PIECES = QB * CH;  // 16-byte pieces of the block
  static_assert(QB * LINE <= NS * X::STAGE, "C block in the ring");
  lds_barrier();  // every wave is done with the ring
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    if (!owner)
      break;
    const int i = g / (4 * TJ), j = (g / 4) % TJ;
    const uint32_t e0 = 8 * (g & 3) + 4 * h;
    const uint32_t ml = wm * X::RM + 32 * i, nl = wn * X::RN + 32 * j;
    const uint32_t ql = (COL_MAJOR ? nl : ml) + rr;
    const uint32_t byte = ((COL_MAJOR ? ml : nl) + e0) * OB;
    uint8_t *dst = smem + ql * LINE + (((byte >> 4) ^ (ql & (CH - 1))) << 4) + (byte & 15);
    if constexpr (OUT_DT == kF32)
      *reinterpret_cast<f32x4 *>(dst) = out[g];
    else
      *reinterpret_cast<u32x2 *>(dst) =
          u32x2{pack2<OUT_DT>(out[g][0], out[g][1]), pack2<OUT_DT>(out[g][2], out[g][3])};
  }
  lds_barrier();
  const int Q0 = COL_MAJOR ? n0 : m0, P0 = COL_MAJOR ? m0 : n0;
  const int Qext = COL_MAJOR ? p.N : p.M, Pext = COL_MAJOR ? p.M : p.N;
#pragma unroll
  for (int it = 0; it < (PIECES + 255) / 256; ++it) {
    const uint32_t flat = it * 256 + threadIdx.x;
    if (PIECES % 256 != 0 && flat >= PIECES)
      break;
    const uint32_t ql = flat / CH, c = flat % CH;
    const u32x4 v =
        *reinterpret_cast<const u32x4 *>(smem + ql * LINE + ((c ^ (ql & (CH - 1))) << 4));
    const int qq = Q0 + (int)ql, pp = P0 + (int)c * EPC;
    if (qq >= Qext || pp >= Pext)
      continue;
    uint8_t *dst = static_cast<uint8_t *>(p.C) + ((size_t)qq * p.ldc + pp) * OB;
    if (p.c_vec_ok && pp + EPC <= Pext) {
      *reinterpret_cast<u32x4 *>(dst) = v;
    } else {
#pragma unroll
      for (int e = 0; e < EPC; ++e)
        if (pp + e < Pext) {
          if constexpr (OUT_DT == kF32)
            reinterpret_cast<uint32_t *>(dst)[e] = v[e];
          else
            reinterpret_cast<uint16_t *>(dst)[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
        }
    }
  }
}

template <class X, int IN, int OUT, int VEC>
hipError_t launch_cfg(BlockParams p, bool cm, hipStream_t s) {
  p.tiles_m = (p.M - 1) / X::BM + 1;
  p.tiles_n = (p.N - 1) / X::BN + 1;
  p.group_m = p.tiles_m < 4 ? p.tiles_m : 4;
  const dim3 grid((unsigned)p.tiles_m * (unsigned)p.tiles_n * (unsigned)p.splits), block(256);
  if (cm)
    hipLaunchKernelGGL((block_kernel<X, IN, OUT, true, VEC>), grid, block, 0, s, p);
  else
    hipLaunchKernelGGL((block_kernel<X, IN, OUT, false, VEC>), grid, block, 0, s, p);
  return hipGetLastError();
}

// (bm, bn): one of 128x128, 128x64, 64x64, 32x64, 32x32; vec4: rows at 8-byte boundaries
// (K % 4 == 0, A and B 8-byte aligned), else 64x64 unsplit only.
template <int IN, int OUT>
hipError_t launch_block(const BlockParams &p, int bm, int bn, bool vec4, bool cm,
                        hipStream_t s) {
  if (!vec4)
    return launch_cfg<BlockCfg<64, 64>, IN, OUT, 1>(p, cm, s);
  if (bm == 32)
    return bn == 32 ? launch_cfg<BlockCfg<32, 32>, IN, OUT, 4>(p, cm, s)
                    : launch_cfg<BlockCfg<32, 64>, IN, OUT, 4>(p, cm, s);
  if (bm == 64)
    return launch_cfg<BlockCfg<64, 64>, IN, OUT, 4>(p, cm, s);
  if (bn == 64)
    return launch_cfg<BlockCfg<128, 64>, IN, OUT, 4>(p, cm, s);
  return launch_cfg<BlockCfg<128, 128>, IN, OUT, 4>(p, cm, s);
}

} // namespace block
} // namespace gemm
} // namespace wave
