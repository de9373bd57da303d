// attention_bwd.hip -- flash-attention backward for gfx950, head_dim 128.
//
// Gradients of O = softmax(scale * Q K^T) V (optional causal mask key >
// query, grouped-query heads kv_head = q_head / (Hq / Hkv)) given dO, O and
// the forward's row log-sum-exp lse = ln sum_k exp(scale * q.k):
//   P   = exp(scale * Q K^T - lse)         (recomputed, never stored)
//   dV  = P^T dO                          (summed over a KV head's q heads)
//   dP  = dO V^T
//   dS  = P o (dP - delta),  delta = rowsum(dO o O)
//   dQ  = scale * dS K,      dK = scale * dS^T Q
// The reference has no backward; this is the standard flash-attention-2
// recomputation scheme, checked against a float64 CPU restatement of the
// formulas above (oracle.py fa_backward) that is itself checked against
// torch autograd.
//
// Three or four kernels a call, deterministic (no atomics):
//  * bwd_delta_kernel: -delta[row] = -sum_d dO[row][d] * O[row][d] in fp32
//    (into the caller's scratch).
//  * bwd_kv_pp_kernel: one CTA (8 waves, two groups of 4 one segment apart)
//    per 128-key block of one KV head (the last block's second half may lie
//    past the sequence); it loops over the query blocks of every q head of the
//    group (causal: the blocks at or after the key block), with each block's
//    Q, dO, lse and -delta arriving by LDS DMA, and accumulates dK, dV in
//    registers.  Where those blocks are fewer than the CUs, or causal ones of
//    uneven length, a block's loop is cut into chunks for several CTAs, which
//    leave fp32 partials that bwd_kv_sum_kernel adds in chunk order.
//    bwd_kv_kernel (one CTA of 4 waves per 64-key block, Q and dO staged through
//    registers) takes over where half a block of 128 past the sequence costs more
//    (half_blocks).
//  * bwd_q_kernel: one CTA per 64-query block of one q head; it loops over
//    the key blocks (causal: up to the diagonal) and accumulates dQ.
// Every product is an "NT" product C[m][n] = sum_k A[m][k] B[n][k] of 32x32
// tiles on v_mfma_f32_32x32x16.  The operands fixed for a CTA (K, V in the
// dK/dV kernels; Q, dO in the dQ kernel) are held as MFMA fragments in
// registers; the rest are read as 16-byte row chunks from LDS.  Operands
// needed K-contiguous the other way (Q^T, dO^T, K^T as the B operand of
// dK, dV, dQ) are read from the row-major Q, dO, K tiles by transposing LDS
// reads (ds_read_b64_tr_b16), and P^T / dS^T (dS for dQ) go through LDS
// between the score products and the gradient products.  LDS tiles are
// unpadded with XOR-swizzled 16-byte chunks (swz below), conflict-free for
// every read these kernels make: 130 KiB (bwd_kv_pp_kernel, one CTA per
// CU), 48 KiB (bwd_kv_kernel) and 72 KiB (dQ) of LDS, two CTAs per CU.
#include "attention.hpp"
#include "wave_common.hpp"

#include <algorithm>
#include <cmath>

namespace wave {
namespace attention {

namespace {

constexpr int kBD = 128;               // head dim
constexpr int kBlk = 64;               // query or key rows per block
constexpr int kWide = kBlk * 256;      // [64][128] 16-bit tile: 16 KiB
constexpr int kNarrowS = kBlk * 128;   // [64][64] tile: 8 KiB
constexpr float kLog2eB = 1.4426950408889634f;

// Byte offset of (row r, byte b) in a tile of ROWB-byte rows: 16-byte chunk
// c of row r at c ^ swz(r).  256-byte rows: swz(r) = 4 (r % 4) + (r / 4) % 4,
// under which both access patterns of these tiles are free of LDS bank
// conflicts on gfx950 (measured: a 16-byte row-fragment read of 32
// consecutive rows, and the transposing 8-byte reads of tr_frag, which
// touch rows k .. k+3 and k+8 .. k+11 in one instruction; c ^ (r % 16)
// served the first but made the second 2.6x slower).  128-byte rows:
// swz(r) = (r / 2) % 8.
template <int ROWB> __device__ __forceinline__ uint32_t swz(uint32_t r) {
  return ROWB == 256 ? (((r & 3u) << 2) | ((r >> 2) & 3u)) : ((r >> 1) & 7u);
}
template <int ROWB> __device__ __forceinline__ uint32_t toff(uint32_t r, uint32_t b) {
  return r * ROWB + ((((b >> 4) ^ swz<ROWB>(r))) << 4) + (b & 15u);
}

struct BwdParams {
  const uint16_t *Q, *K, *V, *O, *dO;
  const float *lse;
  float *delta;
  uint16_t *dQ, *dK, *dV;
  int batch, q_heads, kv_heads, seq;
  int causal;
  float scale;        // softmax scale
  float scale_log2;   // scale * log2(e)
  float inv_scale;    // 1 / scale
  // dK/dV work split: chunks of at most `chunk` items (0: one CTA a block),
  // `per_head` CTAs a KV head, partials [CTA][16][512] f32x4.
  int chunk, per_head;
  f32x4 *part;
  // Causal CTA order (head_coords) of the dK/dV and the dQ kernel.
  int kv_by_length, q_by_length;
};

// Two NT products over K = 128 that share their A rows: c0 += A0 . b0^T and
// c1 += A1 . b1^T, with A rows a0 .. a0+31 of two [rows][128] 16-bit LDS
// tiles (256-byte rows) and B as per-slice register fragments (lane l: row
// l % 32 of B, elements 16 kk + 8 (l / 32) .. +8).  The two accumulation
// chains alternate (each MFMA's predecessor on its chain is two MFMAs
// back), and each A fragment is read kPF slices ahead of its MFMA.
template <int DT, int kPF = 2>
__device__ __forceinline__ void mma2_nt_reg(f32x16 &c0, const uint8_t *A0, const u32x4 (&b0)[8],
                                            f32x16 &c1, const uint8_t *A1, const u32x4 (&b1)[8],
                                            uint32_t a0) {
  const uint32_t lane = threadIdx.x & 63, ra = a0 + (lane & 31);
  const uint32_t sw = (lane >> 5) ^ swz<256>(ra);
  auto frag = [&](const uint8_t *A, int kk) {
    return *reinterpret_cast<const u32x4 *>(A + ra * 256 + (((2u * kk) ^ sw) << 4));
  };
  u32x4 f0[8], f1[8];
#pragma unroll
  for (int kk = 0; kk < kPF; ++kk) {
    f0[kk] = frag(A0, kk);
    f1[kk] = frag(A1, kk);
  }
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) {
    if (kk + kPF < 8) {
      f0[kk + kPF] = frag(A0, kk + kPF);
      f1[kk + kPF] = frag(A1, kk + kPF);
    }
    c0 = mfma32x32x16<DT>(f0[kk], b0[kk], c0);
    c1 = mfma32x32x16<DT>(f1[kk], b1[kk], c1);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The B operand of a gradient product from a row-major [K][128] 16-bit LDS
// tile R of 256-byte rows, columns c0 .. c0+31, slice kk (K rows 16 kk ..
// 16 kk + 15), by transposing reads (ds_read_b64_tr_b16: in each 16-lane
// group source lane 4a + p addresses R[k + a][c + 4p .. +3] and lane i then
// holds R[k .. k+3][c + i]).  Lane l reads rows 16 kk + 8 (l / 32) + 4 r +
// (l >> 2) % 4, columns c0 + 16 ((l >> 4) % 2) + 4 (l % 4), r = 0, 1: the 8
// K values of its B fragment, in order.  So no transposed copy of R is
// needed.
__device__ __forceinline__ u32x4 tr_frag(uint32_t rbase, int kk, uint32_t c0) {
  typedef short s4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s4 lds_s4;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t rb = 16 * kk + 8 * (lane >> 5) + ((lane >> 2) & 3);
  const uint32_t cb = 2 * c0 + 32 * ((lane >> 4) & 1) + 8 * (lane & 3);
  const u32x2 lo = __builtin_bit_cast(
      u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(uintptr_t)(rbase + toff<256>(rb, cb))));
  const u32x2 hi = __builtin_bit_cast(
      u32x2,
      __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(uintptr_t)(rbase + toff<256>(rb + 4, cb))));
  return u32x4{lo[0], lo[1], hi[0], hi[1]};
}

// 2 NT gradient chains over K = 64 (4 slices): for tile pair i < NT and
// t = 0, 1, acc[2i + t] += A_i . R_i[:, c_t .. c_t + 31], with A_i rows
// a0 .. a0+31 of a 128-byte-row LDS tile and R_i a row-major [64][128] LDS
// tile read transposed (tr_frag).  Steps (slice kk, pair i) run in order,
// two MFMAs each, and the fragments of step n + GPF are read before the
// MFMAs of step n.
template <int DT, int NT, int GPF = 1>
__device__ __forceinline__ void mma_grad(f32x16 (&acc)[2 * NT], const uint8_t *const (&A)[NT],
                                         uint32_t a0, const uint8_t *const (&R)[NT],
                                         uint32_t c0, uint32_t c1) {
  const uint32_t lane = threadIdx.x & 63, ra = a0 + (lane & 31);
  const uint32_t sw = (lane >> 5) ^ swz<128>(ra);
  constexpr int NS = 4 * NT, NB = GPF + 1;
  u32x4 fa[NB], fb[NB][2];
  auto load = [&](int n, int slot) {
    const int kk = n / NT, i = n % NT;
    fa[slot] = *reinterpret_cast<const u32x4 *>(A[i] + ra * 128 + (((2u * kk) ^ sw) << 4));
    fb[slot][0] = tr_frag(lds_addr(R[i]), kk, c0);
    fb[slot][1] = tr_frag(lds_addr(R[i]), kk, c1);
  };
#pragma unroll
  for (int n = 0; n < GPF && n < NS; ++n)
    load(n, n % NB);
#pragma unroll
  for (int n = 0; n < NS; ++n) {
    if (n + GPF < NS)
      load(n + GPF, (n + GPF) % NB);
    const int i = n % NT;
    acc[2 * i] = mfma32x32x16<DT>(fa[n % NB], fb[n % NB][0], acc[2 * i]);
    acc[2 * i + 1] = mfma32x32x16<DT>(fa[n % NB], fb[n % NB][1], acc[2 * i + 1]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// One gradient product over K = 64 (4 slices) for 64 rows: acc[2a + t] +=
// A[32a .. 32a+31] . R[:, c_t .. c_t + 31] (a, t = 0, 1), A a 128-byte-row
// LDS tile (rows r and r + 32 share swz<128>), R a row-major [64][128] tile
// read transposed.  Per slice two A and two B fragments feed four MFMAs:
// 1 KiB of LDS reads an MFMA, against 1.5 KiB for mma_grad's two products
// of 32 rows each (whose A fragment feeds two MFMAs but each B one).  The
// fragments of slice kk + GPF are read before the MFMAs of slice kk.
template <int DT, int GPF = 1>
__device__ __forceinline__ void mma_grad_rows2(f32x16 (&acc)[4], const uint8_t *A,
                                               const uint8_t *R, uint32_t c0, uint32_t c1) {
  const uint32_t lane = threadIdx.x & 63, ra = lane & 31;
  const uint32_t sw = (lane >> 5) ^ swz<128>(ra);
  constexpr int NB = GPF + 1;
  u32x4 fa[NB][2], fb[NB][2];
  auto load = [&](int kk, int slot) {
    const uint32_t cb = ((2u * kk) ^ sw) << 4;
    fa[slot][0] = *reinterpret_cast<const u32x4 *>(A + ra * 128 + cb);
    fa[slot][1] = *reinterpret_cast<const u32x4 *>(A + (ra + 32) * 128 + cb);
    fb[slot][0] = tr_frag(lds_addr(R), kk, c0);
    fb[slot][1] = tr_frag(lds_addr(R), kk, c1);
  };
#pragma unroll
  for (int kk = 0; kk < GPF && kk < 4; ++kk)
    load(kk, kk % NB);
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    if (kk + GPF < 4)
      load(kk + GPF, (kk + GPF) % NB);
    const int sl = kk % NB;
    acc[0] = mfma32x32x16<DT>(fa[sl][0], fb[sl][0], acc[0]);
    acc[1] = mfma32x32x16<DT>(fa[sl][0], fb[sl][1], acc[1]);
    acc[2] = mfma32x32x16<DT>(fa[sl][1], fb[sl][0], acc[2]);
    acc[3] = mfma32x32x16<DT>(fa[sl][1], fb[sl][1], acc[3]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// MFMA fragments of 32 rows of a [rows][128] global block (row0 = the
// lane's row): lane l holds elements 16 kk + 8 (l / 32) .. +8 for kk < 8.
__device__ __forceinline__ void load_frags(const uint16_t *row, u32x4 (&f)[8]) {
  const uint32_t lane = threadIdx.x & 63;
#pragma unroll
  for (int kk = 0; kk < 8; ++kk)
    f[kk] = *reinterpret_cast<const u32x4 *>(row + 16 * kk + 8 * (lane >> 5));
}

// A [64][128] block of rows (row stride 128 elements) in flight through
// registers: fetch() issues the global loads, put() writes the rows to LDS
// (wide tile R).
// Thread t handles row pairs x 16-byte chunks: unit u = t + 256*i, row pair
// u / 16, chunk u % 16.
struct BlockRegs {
  u32x4 a[2], b[2];
  __device__ __forceinline__ void fetch(const uint16_t *src) {
    const uint32_t t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t u = t + 256u * i, rp = u >> 4, c = u & 15u;
      a[i] = *reinterpret_cast<const u32x4 *>(src + (size_t)(2 * rp) * kBD + 8 * c);
      b[i] = *reinterpret_cast<const u32x4 *>(src + (size_t)(2 * rp + 1) * kBD + 8 * c);
    }
  }
  __device__ __forceinline__ void put(uint8_t *R) const {
    const uint32_t t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t u = t + 256u * i, rp = u >> 4, c = u & 15u;
      *reinterpret_cast<u32x4 *>(R + toff<256>(2 * rp, 16 * c)) = a[i];
      *reinterpret_cast<u32x4 *>(R + toff<256>(2 * rp + 1, 16 * c)) = b[i];
    }
  }
};

// CTA id -> work index with the CTAs of one head on one XCD (the
// dispatcher places workgroup i on XCD i % 8), so they share that head's
// K/V or Q/dO rows in the XCD's L2.
__device__ __forceinline__ int xcd_pid(int raw, int total) {
  const int xcd = raw & 7;  // the first total % 8 XCDs hold one more
  return xcd * (total >> 3) + min(xcd, total & 7) + (raw >> 3);
}

// CTA id -> head and the head's CTA i of n; by_length (heads a multiple of 8):
// an XCD runs CTA 0 of each of its heads, then CTA 1 of each, and so on.
__device__ __forceinline__ void head_coords(int raw, int heads, int n, int by_length, int &head,
                                            int &i) {
  if (by_length) {
    const int hx = heads >> 3, j = raw >> 3;  // heads of an XCD
    i = j / hx;
    head = (raw & 7) * hx + j - i * hx;
    return;
  }
  const int pid = xcd_pid(raw, heads * n);
  head = pid / n;
  i = pid - head * n;
}

// Store a 32x32 fp32 accumulator tile (rows row0.., columns col0..) of a
// [rows][128] 16-bit output, times mul.
template <int DT>
__device__ __forceinline__ void store_tile32(uint16_t *dst, int row0, int col0, const f32x16 &acc,
                                             float mul) {
  const uint32_t lane = threadIdx.x & 63;
  const int col = col0 + (int)(lane & 31);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = row0 + 8 * (r >> 2) + 4 * (int)(lane >> 5) + (r & 3);
    dst[(size_t)row * kBD + col] = to_bits<DT>(acc[r] * mul);
  }
}

} // namespace

// delta[row] = -sum_d dO[row][d] * O[row][d] (stored negated: it is the
// start value of the dP accumulators); 16 lanes per row, 8 elements a lane.
template <int DT>
__global__ __launch_bounds__(256) void bwd_delta_kernel(BwdParams p, int rows) {
  const int row = (int)(blockIdx.x * 16 + (threadIdx.x >> 4));
  const int c = threadIdx.x & 15;
  float s = 0.f;
  if (row < rows) {
    const u32x4 a = *reinterpret_cast<const u32x4 *>(p.dO + (size_t)row * kBD + 8 * c);
    const u32x4 b = *reinterpret_cast<const u32x4 *>(p.O + (size_t)row * kBD + 8 * c);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s += from_bits<DT>((uint16_t)(a[e] & 0xffffu)) * from_bits<DT>((uint16_t)(b[e] & 0xffffu));
      s += from_bits<DT>((uint16_t)(a[e] >> 16)) * from_bits<DT>((uint16_t)(b[e] >> 16));
    }
  }
#pragma unroll
  for (int m = 8; m >= 1; m >>= 1)
    s += __shfl_xor(s, m, 16);
  if (row < rows && c == 0)
    p.delta[row] = -s;
}

// dK, dV of one 64-key block of one KV head.
template <int DT, bool CAUSAL>
__global__ __launch_bounds__(256, 2) void bwd_kv_kernel(BwdParams p) {
  __shared__ __attribute__((aligned(16))) uint8_t smem[2 * kWide + 2 * kNarrowS];
  uint8_t *sQ = smem, *sdO = sQ + kWide, *sPt = sdO + kWide, *sdSt = sPt + kNarrowS;
  const int nb = p.seq / kBlk;
  int bhk, kb;
  head_coords((int)blockIdx.x, p.batch * p.kv_heads, nb, 0, bhk, kb);
  const int b = bhk / p.kv_heads, hkv = bhk - b * p.kv_heads;
  const int group = p.q_heads / p.kv_heads;
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const size_t kv_off = ((size_t)bhk * p.seq + (size_t)kb * kBlk) * kBD;

  // Score tiles: wave w computes S[q][key] for q half w&1, key half w>>1;
  // lane l holds key kh2*32 + l%32 and queries qh2*32 + 8g + 4(l/32) + e.
  const int qh2 = wave & 1, kh2 = wave >> 1;
  // Gradient tiles: key half w&1, d quarters 2(w>>1), 2(w>>1)+1.
  const int kh = wave & 1, dq = wave >> 1;
  // K and V rows of this wave's key half as B fragments, for the whole CTA.
  u32x4 kf[8], vf[8];
  load_frags(p.K + kv_off + (size_t)(kh2 * 32 + (lane & 31)) * kBD, kf);
  load_frags(p.V + kv_off + (size_t)(kh2 * 32 + (lane & 31)) * kBD, vf);
  // Gradient accumulators: dV columns (2 dq) * 32 and (2 dq + 1) * 32, then
  // dK's.
  f32x16 g[4] = {f32x16{}, f32x16{}, f32x16{}, f32x16{}};
  const int key = kb * kBlk + kh2 * 32 + (int)(lane & 31);
  // Work items: (q head h of the group, query block qb), h major (causal:
  // the blocks at or after the key block); the next item's Q and dO rows
  // and its lse / delta are fetched while this one's products run.
  const int qb0 = CAUSAL ? kb : 0, items = group * (nb - qb0);
  auto rows_of = [&](int h, int q) {  // first row of item (h, q) in [B*Hq*S]
    return ((size_t)b * p.q_heads + (size_t)hkv * group + h) * p.seq + (size_t)q * kBlk;
  };
  // This wave's score rows of an item: lse and -delta of rows
  // qh2*32 + 8 g + 4 (l / 32) + e as the accumulators' start values.
  f32x16 s, dp;
  auto load_stats = [&](size_t rb) {
    const size_t r0 = rb + qh2 * 32 + 4 * (lane >> 5);
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const f32x4 a = *reinterpret_cast<const f32x4 *>(p.lse + r0 + 8 * g4);
      const f32x4 d = *reinterpret_cast<const f32x4 *>(p.delta + r0 + 8 * g4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[4 * g4 + e] = a[e];
        dp[4 * g4 + e] = d[e];
      }
    }
  };
  int h = 0, qb = qb0;
  BlockRegs rq, rdo;
  rq.fetch(p.Q + rows_of(0, qb0) * kBD);
  rdo.fetch(p.dO + rows_of(0, qb0) * kBD);
  load_stats(rows_of(0, qb0));
  for (int it = 0; it < items; ++it) {
    int hn = h, qbn = qb + 1;
    if (qbn == nb) {
      qbn = qb0;
      ++hn;
    }
    const bool more = it + 1 < items;
    __syncthreads();  // the previous item's readers are done
    rq.put(sQ);
    rdo.put(sdO);
    if (more) {
      rq.fetch(p.Q + rows_of(hn, qbn) * kBD);
      rdo.fetch(p.dO + rows_of(hn, qbn) * kBD);
    }
    // The score accumulator starts at -lse / scale and dP's at -delta, so
    // exp2(c * s) = P and dp = dP - delta after the products.
#pragma unroll
    for (int r = 0; r < 16; ++r)
      s[r] *= -p.inv_scale;
    __syncthreads();
    mma2_nt_reg<DT>(s, sQ, kf, dp, sdO, vf, qh2 * 32);
    // P and dS; P^T / dS^T rows = keys, 4 consecutive queries per store.
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      float pv[4], dsv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * g4 + e;
        const int q = qb * kBlk + qh2 * 32 + 8 * g4 + 4 * (int)(lane >> 5) + e;
        float pr = __builtin_amdgcn_exp2f(s[r] * p.scale_log2);
        if (CAUSAL && key > q)
          pr = 0.f;
        pv[e] = pr;
        dsv[e] = pr * dp[r];
      }
      const uint32_t off =
          toff<128>(kh2 * 32 + (lane & 31), 2 * (qh2 * 32 + 8 * g4 + 4 * (lane >> 5)));
      *reinterpret_cast<u32x2 *>(sPt + off) = u32x2{pack2<DT>(pv[0], pv[1]), pack2<DT>(pv[2], pv[3])};
      *reinterpret_cast<u32x2 *>(sdSt + off) =
          u32x2{pack2<DT>(dsv[0], dsv[1]), pack2<DT>(dsv[2], dsv[3])};
    }
    __syncthreads();
    const uint8_t *const ga[2] = {sPt, sdSt};
    const uint8_t *const gr[2] = {sdO, sQ};
    mma_grad<DT, 2>(g, ga, kh * 32, gr, (2 * dq) * 32, (2 * dq + 1) * 32);
    if (more)
      load_stats(rows_of(hn, qbn));
    h = hn;
    qb = qbn;
  }
  uint16_t *dK = p.dK + kv_off, *dV = p.dV + kv_off;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    store_tile32<DT>(dV, kh * 32, (2 * dq + t) * 32, g[t], 1.f);
    store_tile32<DT>(dK, kh * 32, (2 * dq + t) * 32, g[2 + t], p.scale);
  }
}

// Work items of 128-key block kb2 of a KV head: (q head of the group, 64-query
// block); causal: the blocks at or after the key block.
__host__ __device__ __forceinline__ int kv_items(int group, int nb, int kb2, bool causal) {
  return group * (nb - (causal ? 2 * kb2 : 0));
}
__host__ __device__ __forceinline__ int kv_chunks(int items, int chunk) {
  return chunk > 0 ? (items + chunk - 1) / chunk : 1;
}
// The first item of chunk `index` of `count`: items * index / count rounded down,
// whose product does not fit 32 bits where a block has millions of items (from 1.4
// million query heads of 128 rows on one KV head on: Q, O, dO and dQ of 46 GB).
__host__ __device__ constexpr int kv_first(int items, int index, int count) {
  return items / count * index + items % count * index / count;
}
static_assert(kv_first(1 << 24, 700, 768) == (int)(((int64_t)1 << 24) * 700 / 768) &&
                  kv_first(1 << 24, 768, 768) == 1 << 24 && kv_first(128, 2, 3) == 85 &&
                  kv_first(5, 1, 3) == 1 && kv_first(5, 2, 3) == 3,
              "chunk bounds");

// CTA c (0 .. per_head-1) of a KV head -> its block, its chunk of the block's
// items and how many the block has.
struct KvChunk {
  int kb2, index, count;
};
template <bool CAUSAL>
__device__ __forceinline__ KvChunk kv_chunk(const BwdParams &p, int group, int nb, int c) {
  if (!CAUSAL || p.chunk == 0) {
    const int n = kv_chunks(group * nb, p.chunk);
    return {c / n, c % n, n};
  }
  for (int kb2 = 0;; ++kb2) {
    const int n = kv_chunks(kv_items(group, nb, kb2, true), p.chunk);
    if (c < n)
      return {kb2, c, n};
    c -= n;
  }
}

// dK, dV of a 128-key block of one KV head as two groups of four waves:
// group g (waves 4g .. 4g+3) owns keys 64 g .. 64 g + 63 of the block and
// does for them what bwd_kv_kernel does for its 64 keys (the same products), on
// the same work items.  The groups share each item's Q
// and dO rows and its rows' lse and -delta, which arrive by LDS DMA into a
// 3-buffer ring (so no global load is waited for inside the loop), and run
// one segment apart ("ping-pong"), so that on every SIMD one wave's MFMAs
// run next to the other group's softmax:
//
//   segment    2i              2i+1            2i+2
//   group 0    M2(i-1) M1(i)   SM(i)           M2(i) M1(i+1)
//   group 1    SM(i-1)         M2(i-1) M1(i)   SM(i)
//
// M1(i): S and dP of item i (A fragments from its Q / dO buffer); SM(i): P
// and dS of item i into the group's P^T / dS^T tiles; M2(i): dV, dK += the
// products of those tiles with Q / dO of item i (transposing reads).  Every
// segment ends with a workgroup barrier (2 * items + 2 of them for every
// wave).  Buffers: item i's Q / dO sit in ring slot i % 3, read from
// segment 2i (group 0's M1(i)) to 2i+3 (group 1's M2(i)); group 1's waves
// issue the DMA of item j+1 at the start of segment 2j (their SM(j-1),
// shorter than group 0's matrix segment beside it, which the DMA issues
// used to lengthen: 4-5 % of the kernel's time), after slot (j+1) % 3's
// previous item (j-2) was last read in segment 2j-1, and every wave waits
// for it at the end of segment 2j+1.  A group's P^T / dS^T are written in
// SM(i) and read in M2(i), the next segment of that group.
#ifndef WAVE_BWD_PF
#define WAVE_BWD_PF 3  // score products: A fragments read this many slices ahead
#endif
#ifndef WAVE_BWD_GPF
#define WAVE_BWD_GPF 2  // gradient products: fragments read this many steps ahead
#endif
template <int DT, bool CAUSAL>
__global__ __launch_bounds__(512, 1) void bwd_kv_pp_kernel(BwdParams p) {
  // One ring slot: an item's Q and dO rows (32 KiB), then its 64 rows' lse
  // and -delta (256 B each).
  constexpr uint32_t kStats = 2 * kWide, kQD = kStats + 512;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[3 * kQD + 4 * kNarrowS];
  const int nb = p.seq / kBlk;
  int bhk, cta;
  head_coords((int)blockIdx.x, p.batch * p.kv_heads, p.per_head, p.kv_by_length, bhk, cta);
  const int b = bhk / p.kv_heads, hkv = bhk - b * p.kv_heads;
  const int group = p.q_heads / p.kv_heads;
  const uint32_t wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const uint32_t grp = wave >> 2, wg = wave & 3;
  const KvChunk chunk = kv_chunk<CAUSAL>(p, group, nb, cta);
  const int kb2 = chunk.kb2;
  // This group's 64-key block; past the sequence (the last block's second half
  // when nb is odd) it repeats the last one and stores nothing.
  const bool keys_in = 2 * kb2 + (int)grp < nb;
  const int kb = keys_in ? 2 * kb2 + (int)grp : nb - 1;
  const size_t kv_off = ((size_t)bhk * p.seq + (size_t)kb * kBlk) * kBD;
  uint8_t *sPt = smem + 3 * kQD + grp * 2 * kNarrowS, *sdSt = sPt + kNarrowS;
  const uint32_t lds0 = lds_addr(smem);
  // Wave roles within the group.  Score products: query half qh2, key half
  // kh2.  Gradient products: wave role 0 accumulates dV, role 1 dK, each for
  // all 64 keys of the group and d columns 64 dq .. 64 dq + 63.
  const int qh2 = wg & 1, kh2 = wg >> 1, role = wg & 1, dq = wg >> 1;
  u32x4 kf[8], vf[8];
  load_frags(p.K + kv_off + (size_t)(kh2 * 32 + (lane & 31)) * kBD, kf);
  load_frags(p.V + kv_off + (size_t)(kh2 * 32 + (lane & 31)) * kBD, vf);
  f32x16 g[4] = {f32x16{}, f32x16{}, f32x16{}, f32x16{}};
  const int key = kb * kBlk + kh2 * 32 + (int)(lane & 31);
  // Work items (q head h, query block qb), h major; causal: the blocks at
  // or after group 0's key block (group 1's first one is wholly masked).
  const int qb0 = CAUSAL ? 2 * kb2 : 0, block_items = group * (nb - qb0);
  const int first = kv_first(block_items, chunk.index, chunk.count);
  const int items = kv_first(block_items, chunk.index + 1, chunk.count) - first;
  struct Cursor {
    int h, qb;
  };
  auto advance = [&](Cursor &c) {
    if (++c.qb == nb) {
      c.qb = qb0;
      ++c.h;
    }
  };
  auto rows_of = [&](const Cursor &c) {
    return ((size_t)b * p.q_heads + (size_t)hkv * group + c.h) * p.seq + (size_t)c.qb * kBlk;
  };
  // DMA of an item into ring slot `slot`, issued by group 1's waves: wave
  // wg fills Q and dO rows 16 wg .. 16 wg + 15 (four 1 KiB windows each),
  // lane l row 4 win + l / 16, slot l % 16, which holds chunk (l % 16) ^
  // swz(row); waves wg = 0 and 1 add the rows' lse and -delta (256 B each,
  // 4 bytes a lane).
  auto dma_item = [&](const Cursor &c, uint32_t slot) {
    const size_t rb = rows_of(c);
    const uint32_t l = lds0 + slot * kQD;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t win = 4 * wg + j, r = 4 * win + (lane >> 4);
      const uint32_t off = r * 256 + (((lane & 15) ^ swz<256>(r)) << 4);
      dma16(l + win * 1024, p.Q + rb * kBD, off);
      dma16(l + kWide + win * 1024, p.dO + rb * kBD, off);
    }
    if (wg < 2)
      dma4(l + kStats + wg * 256, wg == 0 ? (const void *)(p.lse + rb) : (const void *)(p.delta + rb),
           4 * lane);
  };
  f32x16 s, dp;
  // This wave's score rows' lse and -delta (rows qh2*32 + 8 g + 4 (l / 32)
  // + e) from the item's ring slot: the accumulators' start values.
  auto load_stats = [&](const uint8_t *q) {
    const float *r0 = reinterpret_cast<const float *>(q + kStats) + qh2 * 32 + 4 * (lane >> 5);
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const f32x4 a = *reinterpret_cast<const f32x4 *>(r0 + 8 * g4);
      const f32x4 d = *reinterpret_cast<const f32x4 *>(r0 + 64 + 8 * g4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[4 * g4 + e] = a[e];
        dp[4 * g4 + e] = d[e];
      }
    }
  };
  const int h0 = first / (nb - qb0);
  Cursor dmac{h0, qb0 + first - h0 * (nb - qb0)}, cur = dmac;
  if (grp == 1)
    dma_item(dmac, 0);
  advance(dmac);
  vm_wait_barrier();
  // Waited for here: a kernel argument still on its way counts as an LDS read to
  // the compiler, which then drains all reads at each fragment's wait in the loop
  // (B1 Hq64 Hkv8 S8192 7.39 ms, 7.65 without).
  f32x4 *part0 = p.part;
  asm volatile("" : "+s"(part0));
  const int nseg = 2 * items + 2;
  for (int sg = 0; sg < nseg; ++sg) {
    if ((sg & 1) == 0 && (sg >> 1) + 1 < items) {
      if (grp == 1)
        dma_item(dmac, (uint32_t)(((sg >> 1) + 1) % 3));
      advance(dmac);
    }
    const int ls = sg - (int)grp;
    if (ls >= 0 && ls <= 2 * items) {
      const int i = ls >> 1;
      if ((ls & 1) == 0) {
        if (i >= 1) {  // M2(i-1)
          const uint8_t *q = smem + ((i - 1) % 3) * kQD;
          // dV += P^T dO, dK += dS^T Q (scaled at the store).
          mma_grad_rows2<DT, WAVE_BWD_GPF>(g, role ? sdSt : sPt, role ? q : q + kWide,
                                           (2 * dq) * 32, (2 * dq + 1) * 32);
        }
        if (i < items) {  // M1(i): S starts at -lse / scale, dP at -delta
          const uint8_t *q = smem + (i % 3) * kQD;
          load_stats(q);
#pragma unroll
          for (int r = 0; r < 16; ++r)
            s[r] *= -p.inv_scale;
          mma2_nt_reg<DT, WAVE_BWD_PF>(s, q, kf, dp, q + kWide, vf, qh2 * 32);
        }
      } else {  // SM(i)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          float pv[4], dsv[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = 4 * g4 + e;
            const int q = cur.qb * kBlk + qh2 * 32 + 8 * g4 + 4 * (int)(lane >> 5) + e;
            float pr = __builtin_amdgcn_exp2f(s[r] * p.scale_log2);
            if (CAUSAL && key > q)
              pr = 0.f;
            pv[e] = pr;
            dsv[e] = pr * dp[r];
          }
          const uint32_t off =
              toff<128>(kh2 * 32 + (lane & 31), 2 * (qh2 * 32 + 8 * g4 + 4 * (lane >> 5)));
          *reinterpret_cast<u32x2 *>(sPt + off) =
              u32x2{pack2<DT>(pv[0], pv[1]), pack2<DT>(pv[2], pv[3])};
          *reinterpret_cast<u32x2 *>(sdSt + off) =
              u32x2{pack2<DT>(dsv[0], dsv[1]), pack2<DT>(dsv[2], dsv[3])};
        }
        advance(cur);
      }
    }
    if (sg & 1)
      vm_wait_barrier();  // the DMA of item (sg >> 1) + 1 has landed
    else
      lds_barrier();
  }
  if (chunk.count > 1) {
    f32x4 *part = part0 + (size_t)(bhk * p.per_head + cta) * (16 * 512) + threadIdx.x;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        part[(4 * t + r) * 512] =
            f32x4{g[t][4 * r], g[t][4 * r + 1], g[t][4 * r + 2], g[t][4 * r + 3]};
    return;
  }
  if (!keys_in)
    return;
  uint16_t *dst = (role ? p.dK : p.dV) + kv_off;
  const float sc = role ? p.scale : 1.f;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int t = 0; t < 2; ++t)
      store_tile32<DT>(dst, a * 32, (2 * dq + t) * 32, g[2 * a + t], sc);
}

// dK, dV of the blocks that bwd_kv_pp_kernel cut into chunks: the partials'
// sum in chunk order, rounded once.  One CTA a 32x32 tile set t (0 .. 3) of a
// block, its threads standing for that kernel's.
template <int DT, bool CAUSAL>
__global__ __launch_bounds__(512) void bwd_kv_sum_kernel(BwdParams p) {
  const int nb = p.seq / kBlk, nkb = (nb + 1) / 2, group = p.q_heads / p.kv_heads;
  const int t = blockIdx.x & 3, kb2 = (int)(blockIdx.x >> 2) % nkb, bhk = (int)(blockIdx.x >> 2) / nkb;
  const int n = kv_chunks(kv_items(group, nb, kb2, CAUSAL), p.chunk);
  if (n == 1)
    return;
  int slot = bhk * p.per_head;  // the block's first CTA
  if (CAUSAL) {
    for (int k = 0; k < kb2; ++k)
      slot += kv_chunks(kv_items(group, nb, k, true), p.chunk);
  } else {
    slot += kb2 * n;
  }
  const f32x4 *part = p.part + (size_t)slot * (16 * 512) + 4 * t * 512 + threadIdx.x;
  f32x16 sum = {};
  for (int c = 0; c < n; ++c) {
    f32x4 v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      v[r] = part[(size_t)c * (16 * 512) + r * 512];
#pragma unroll
    for (int r = 0; r < 16; ++r)
      sum[r] += v[r >> 2][r & 3];
  }
  const uint32_t wave = threadIdx.x >> 6, wg = wave & 3;
  const int role = wg & 1, dq = wg >> 1, kb = 2 * kb2 + (int)(wave >> 2);
  if (kb >= nb)
    return;
  uint16_t *dst = (role ? p.dK : p.dV) + ((size_t)bhk * p.seq + (size_t)kb * kBlk) * kBD;
  store_tile32<DT>(dst, (t >> 1) * 32, (2 * dq + (t & 1)) * 32, sum, role ? p.scale : 1.f);
}

// dQ of one 64-query block of one q head.
#ifndef WAVE_BWDQ_PF
#define WAVE_BWDQ_PF 2  // score products: A fragments read this many slices ahead
#endif
#ifndef WAVE_BWDQ_GPF
#define WAVE_BWDQ_GPF 1  // dQ product: fragments read this many steps ahead
#endif
template <int DT, bool CAUSAL>
__global__ __launch_bounds__(256, 2) void bwd_q_kernel(BwdParams p) {
  // K and V rows of a key block arrive by LDS DMA into a 2-slot ring: the
  // DMA of block kb + 1 goes into the slot block kb - 1 used, after the
  // barrier that starts iteration kb, and is waited for at the barrier that
  // starts iteration kb + 1.
  constexpr uint32_t kKV = 2 * kWide;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * kKV + kNarrowS];
  uint8_t *sdS = smem + 2 * kKV;
  const int nb = p.seq / kBlk;
  // Causal: the longest query blocks first, so that the short ones fill the
  // last round.
  int bh, i;
  head_coords((int)blockIdx.x, p.batch * p.q_heads, nb, p.q_by_length, bh, i);
  const int qb = CAUSAL ? nb - 1 - i : i;
  const int b = bh / p.q_heads, hq = bh - b * p.q_heads;
  const int hkv = hq / (p.q_heads / p.kv_heads);
  const uint32_t wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const size_t q_off = ((size_t)bh * p.seq + (size_t)qb * kBlk) * kBD;
  // Score tiles: wave w computes S^T[key][q] for key half w&1, q half w>>1;
  // lane l holds query qh2*32 + l%32 and keys kh2*32 + 8g + 4(l/32) + e.
  const int kh2 = wave & 1, qh2 = wave >> 1;
  // dQ tiles: q half w&1, d quarters 2(w>>1), 2(w>>1)+1.
  const int qh = wave & 1, dq = wave >> 1;
  // Q and dO rows of this wave's query half as B fragments, for the whole CTA.
  u32x4 qf[8], dof[8];
  load_frags(p.Q + q_off + (size_t)(qh2 * 32 + (lane & 31)) * kBD, qf);
  load_frags(p.dO + q_off + (size_t)(qh2 * 32 + (lane & 31)) * kBD, dof);
  const int q = qb * kBlk + qh2 * 32 + (int)(lane & 31);
  const size_t row = (size_t)bh * p.seq + q;
  const float l2 = p.lse[row] * kLog2eB, ndl = p.delta[row];  // -delta
  f32x16 dqa[2] = {f32x16{}, f32x16{}};
  const size_t kv_base = (size_t)(b * p.kv_heads + hkv) * p.seq * kBD;
  const int kb_end = CAUSAL ? qb + 1 : nb;
  const uint32_t lds0 = lds_addr(smem);
  // DMA of key block kb into ring slot kb % 2: wave w fills K and V rows
  // 16w .. 16w+15 (four 1 KiB windows each), lane l row 4 win + l / 16,
  // slot l % 16, which holds chunk (l % 16) ^ swz(row).
  auto dma_block = [&](int kb) {
    const size_t r0 = kv_base + (size_t)kb * kBlk * kBD;
    const uint32_t l = lds0 + (kb & 1) * kKV;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t win = 4 * wave + j, r = 4 * win + (lane >> 4);
      const uint32_t off = r * 256 + (((lane & 15) ^ swz<256>(r)) << 4);
      dma16(l + win * 1024, p.K + r0, off);
      dma16(l + kWide + win * 1024, p.V + r0, off);
    }
  };
  dma_block(0);
  for (int kb = 0; kb < kb_end; ++kb) {
    // Block kb's DMA has landed everywhere, and every wave is done with
    // iteration kb - 1's LDS reads (of the slot block kb + 1 takes, and of
    // dS, which this iteration rewrites).
    vm_wait_barrier();
    if (kb + 1 < kb_end)
      dma_block(kb + 1);
    const uint8_t *sK = smem + (kb & 1) * kKV, *sV = sK + kWide;
    f32x16 st = {}, dpt = {};
    mma2_nt_reg<DT, WAVE_BWDQ_PF>(st, sK, qf, dpt, sV, dof, kh2 * 32);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float dsv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * g + e;
        const int key = kb * kBlk + kh2 * 32 + 8 * g + 4 * (int)(lane >> 5) + e;
        float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(st[r], p.scale_log2, -l2));
        if (CAUSAL && key > q)
          pr = 0.f;
        dsv[e] = pr * (dpt[r] + ndl);
      }
      // dS row q, 4 consecutive keys.
      const uint32_t off =
          toff<128>(qh2 * 32 + (lane & 31), 2 * (kh2 * 32 + 8 * g + 4 * (lane >> 5)));
      *reinterpret_cast<u32x2 *>(sdS + off) =
          u32x2{pack2<DT>(dsv[0], dsv[1]), pack2<DT>(dsv[2], dsv[3])};
    }
    __syncthreads();
    const uint8_t *const ga[1] = {sdS};
    const uint8_t *const gr[1] = {sK};
    mma_grad<DT, 1, WAVE_BWDQ_GPF>(dqa, ga, qh * 32, gr, (2 * dq) * 32, (2 * dq + 1) * 32);
  }
  uint16_t *dQ = p.dQ + q_off;
#pragma unroll
  for (int t = 0; t < 2; ++t)
    store_tile32<DT>(dQ, qh * 32, (2 * dq + t) * 32, dqa[t], p.scale);
}

namespace {
// The dK/dV kernel's split: the chunk length and the CTAs a KV head then has.
struct KvPlan {
  int chunk = 0, per_head = 0;
  bool sum = false;   // some block has several chunks
  bool half = false;  // bwd_kv_kernel's 64-key blocks
};

// Whether bwd_kv_kernel's 64-key blocks are the faster whole blocks of an odd
// number nb of them.  128-key blocks spend half of the last one on keys past the
// sequence, one CTA a CU; 64-key ones run two a CU, with more LDS traffic an item.
// us a CTA to start and end, and an item, fitted to 130 measured shapes: 3.6 (3.3
// in many rounds) and 1.75; 1.1 and 2.07 (alone on its CU), 2.85 and 2.5 (two a CU).
// Causal blocks by length end level (0.86, but the longest come in whole rounds);
// head by head, two or four lengths in turn fall on the same CUs each time (1.25 over
// many rounds).  The backward (us, 128-key / 64-key): S64 B32 H16 32.9 / 26.3, B256
// H16 247 / 208, B1 H8 15.5 / 13.8, Hq64 Hkv1 130 / 154; S192 B24 H12 62.5 / 54.5,
// B128 Hq16 Hkv2 254 / 282; S320 B32 H16 180 / 188; causal S448 B64 H16 534 / 488,
// S960 B32 H16 745 / 758.
bool half_blocks(int64_t heads, int group, int nb, bool causal, bool by_length, int cus) {
  const int nkb = (nb + 1) / 2;
  const double longest = (double)group * nb, mean = (double)group * nkb;  // causal: of a block
  const double n128 = (double)heads * nkb, n64 = (double)heads * nb;      // CTAs
  const double one128 = 3.6 + 1.75 * longest, one64 = 1.1 + 2.07 * longest,
               two64 = 2.85 + 2.5 * longest;
  double t128, t64;
  if (causal && nb > 1) {
    const double turns = by_length ? 0.86
                         : (nkb == 2 || nkb == 4) && n128 >= 8 * cus ? 1.25
                                                                     : 1.0;
    t128 = std::max(one128 * (by_length ? std::ceil((double)heads / cus) : 1.0),
                    n128 > cus ? turns * (3.3 + 1.75 * mean) * n128 / cus : 0.0);
    t64 = n64 <= cus ? one64 : std::max(two64, (2.85 + 2.5 * mean) * n64 / (2 * cus));
  } else {
    const double rounds = std::floor(n64 / (2 * cus)), rest = n64 - rounds * 2 * cus;
    t128 = one128 * std::ceil(n128 / cus);
    t64 = rounds * two64 + (rest == 0 ? 0.0 : rest <= cus ? one64 : two64);
  }
  return t64 < t128;
}

// A CTA takes 1.75 us an item (measured) and 4 to start and end; a CU runs one
// at a time.  Splitting adds the sum kernel: 4 us and 0.06 a CTA (its 128 KiB
// partial written and read; 0.1 with chunks of one item: Hq64 Hkv16 S128, 128 of
// them, 35.2 against 28.9 whole; Hq32 Hkv8, 64 of them, 26.5 / 28.6).  Whole blocks on
// n > CUs: the CUs share the total, and the last blocks run up to half a block's time
// alone; causal ones by length end with the shortest, and their time is the total's
// share or the longest.
// So do those of one head an XCD, or of heads that each fill an XCD's CUs, the
// longest first: Hq64 Hkv8 S8192 3810 whole, 4167 in chunks, B2 Hq64 Hkv8 S4096 2046 /
// 2205, but S6144 (the longest counts) 2417 / 2341.
// Candidates: whole blocks, or the shortest chunks for which the CTAs fill the
// chip once, twice or three times.  B2 Hq16 Hkv4 S2048 causal (128 blocks of 8 to
// 128 items): whole 229 us, chunks of 43 items (256 CTAs) 105 to 111 and the sum
// 7.5.  S1984 (a half block at the end): the backward 346 -> 196 us, against 64-key
// blocks of one CTA each.  B2 Hq32 Hkv8 S4096 (512 blocks, two a CU): whole by
// length 1014, chunks 1156, whole head by head 1051 for the whole backward; S2048
// (256 blocks): whole 358, chunks 308.
// split: with the chunks among the candidates.
KvPlan kv_plan(int batch, int kv_heads, int group, int nb, bool causal, bool by_length, int cus,
               bool split) {
  const int64_t heads = (int64_t)batch * kv_heads;
  const int nkb = (nb + 1) / 2, longest = group * nb;
  auto per_head = [&](int chunk) {
    if (!causal)
      return (int64_t)nkb * kv_chunks(longest, chunk);
    int64_t n = 0;
    for (int k = 0; k < nkb; ++k)
      n += kv_chunks(kv_items(group, nb, k, true), chunk);
    return n;
  };
  int64_t total = 0;  // items of a head
  for (int k = 0; k < nkb; ++k)
    total += kv_items(group, nb, k, causal);
  auto time = [&](int64_t ctas, int len) {
    const double share = (double)total * heads / cus;
    return 4 + 1.75 * (ctas <= cus ? (double)len : share + 0.5 * len + 2);
  };
  KvPlan plan;
  plan.per_head = nkb;
  const bool level =
      by_length || (causal && heads % 8 == 0 && (heads == 8 || nkb >= std::max(cus / 8, 1)));
  double best = level ? 4 + 1.75 * std::max((double)longest, (double)total * heads / cus + 2)
                      : time(heads * nkb, longest);
  for (int rounds = 1; split && rounds <= 3; ++rounds) {
    const int64_t most = (int64_t)rounds * cus / heads;
    if (most <= nkb)
      continue;
    int lo = 1, hi = longest;  // the least chunk with per_head(chunk) <= most
    while (lo < hi) {
      const int mid = (lo + hi) / 2;
      if (per_head(mid) <= most)
        hi = mid;
      else
        lo = mid + 1;
    }
    const int64_t n = per_head(lo);
    if (lo == longest || n == nkb)
      continue;
    const double t = time(heads * n, lo) + 4 + (lo == 1 ? 0.1 : 0.06) * (double)(heads * n);
    if (t < best) {
      best = t;
      plan.chunk = lo;
      plan.per_head = (int)n;
      plan.sum = true;
    }
  }
  if (!plan.sum && nb % 2 && half_blocks(heads, group, nb, causal, by_length, cus)) {
    plan.half = true;
    plan.per_head = nb;
  }
  return plan;
}

constexpr size_t kPartBytes = 16 * 512 * sizeof(f32x4);  // a CTA's dK, dV in fp32

template <int DT, bool CAUSAL>
hipError_t launch_bwd_dt(const BwdParams &p, const KvPlan &plan, hipStream_t stream) {
  const int rows = p.batch * p.q_heads * p.seq;
  hipLaunchKernelGGL((bwd_delta_kernel<DT>), dim3((rows + 15) / 16), dim3(256), 0, stream, p,
                     rows);
  const int nb = p.seq / kBlk, heads = p.batch * p.kv_heads;
  if (plan.half)
    hipLaunchKernelGGL((bwd_kv_kernel<DT, CAUSAL>), dim3(nb * heads), dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL((bwd_kv_pp_kernel<DT, CAUSAL>), dim3(p.per_head * heads), dim3(512), 0,
                       stream, p);
  if (plan.sum)
    hipLaunchKernelGGL((bwd_kv_sum_kernel<DT, CAUSAL>), dim3((nb + 1) / 2 * heads * 4), dim3(512),
                       0, stream, p);
  hipLaunchKernelGGL((bwd_q_kernel<DT, CAUSAL>), dim3(nb * p.batch * p.q_heads), dim3(256), 0,
                     stream, p);
  return hipGetLastError();
}

// Causal blocks go by length where the heads divide over the XCDs and what those
// side by side read at once (rows of two tensors) is at most half the last-level
// cache: with 256 MB (the dK/dV kernel's Q and dO of B8 H32 S2048) the backward
// takes 1268 us head by head and 1375 by length, with 128 MB (B4) 649 and 610.
// Smaller: B1 Hkv32 S1984 186 -> 145 us, B8 H16 S512 84 -> 71, B8 Hq32 Hkv8 S1024
// 404 -> 321.
bool by_length(int64_t heads, int64_t read_heads, int seq, bool causal) {
  return causal && heads % 8 == 0 && read_heads * seq * (4 * kBD) <= (128 << 20);
}
bool kv_order(int batch, int q_heads, int kv_heads, int seq, bool causal) {
  return by_length((int64_t)batch * kv_heads, (int64_t)batch * q_heads, seq, causal);
}
} // namespace

size_t bwd_workspace_bytes(int batch, int q_heads, int kv_heads, int seq, bool causal, int cus) {
  const KvPlan plan = kv_plan(batch, kv_heads, q_heads / kv_heads, seq / kBlk, causal,
                              kv_order(batch, q_heads, kv_heads, seq, causal), cus, true);
  return plan.sum ? (size_t)batch * kv_heads * plan.per_head * kPartBytes : 0;
}

int bwd_key_block(int batch, int q_heads, int kv_heads, int seq, bool causal, int cus) {
  const KvPlan plan = kv_plan(batch, kv_heads, q_heads / kv_heads, seq / kBlk, causal,
                              kv_order(batch, q_heads, kv_heads, seq, causal), cus, true);
  return plan.half ? kBlk : 2 * kBlk;
}

hipError_t launch_bwd(const BwdArgs &a, hipStream_t stream) {
  BwdParams p{};
  p.Q = static_cast<const uint16_t *>(a.Q);
  p.K = static_cast<const uint16_t *>(a.K);
  p.V = static_cast<const uint16_t *>(a.V);
  p.O = static_cast<const uint16_t *>(a.O);
  p.dO = static_cast<const uint16_t *>(a.dO);
  p.lse = a.lse;
  p.delta = a.delta;
  p.dQ = static_cast<uint16_t *>(a.dQ);
  p.dK = static_cast<uint16_t *>(a.dK);
  p.dV = static_cast<uint16_t *>(a.dV);
  p.batch = a.batch;
  p.q_heads = a.q_heads;
  p.kv_heads = a.kv_heads;
  p.seq = a.seq;
  p.causal = a.causal;
  p.scale = a.scale > 0.f ? a.scale : 1.0f / __builtin_sqrtf((float)kBD);
  p.scale_log2 = p.scale * kLog2eB;
  p.inv_scale = 1.0f / p.scale;
  const int group = a.q_heads / a.kv_heads, nb = a.seq / kBlk;
  const bool kv_whole_order = kv_order(a.batch, a.q_heads, a.kv_heads, a.seq, a.causal != 0);
  auto plan_for = [&](bool split) {
    return kv_plan(a.batch, a.kv_heads, group, nb, a.causal != 0, kv_whole_order, a.cus, split);
  };
  KvPlan plan = plan_for(a.workspace != nullptr);
  if (plan.sum && a.workspace_bytes < (size_t)a.batch * a.kv_heads * plan.per_head * kPartBytes)
    plan = plan_for(false);
  p.chunk = plan.chunk;
  p.per_head = plan.per_head;
  p.part = static_cast<f32x4 *>(a.workspace);
  p.kv_by_length = kv_whole_order && !plan.sum;
  // Two or three query blocks a head on more than one round (two CTAs a CU) have
  // little to level and read K and V once more each: head by head -> by length, the
  // backward, B64 H16 S192 168.8 -> 171.7, B32 H16 S192 88 -> 92, B128 Hq32 Hkv8 S128
  // 283 -> 287; within a round B8 Hq16 Hkv4 S192 43.3 -> 41.7.
  p.q_by_length = by_length((int64_t)a.batch * a.q_heads, (int64_t)a.batch * a.kv_heads, a.seq,
                            a.causal != 0) &&
                  (nb >= 4 || (int64_t)nb * a.batch * a.q_heads <= 2 * a.cus);
  if (a.dtype == kF16)
    return a.causal ? launch_bwd_dt<kF16, true>(p, plan, stream)
                    : launch_bwd_dt<kF16, false>(p, plan, stream);
  return a.causal ? launch_bwd_dt<kBF16, true>(p, plan, stream)
                  : launch_bwd_dt<kBF16, false>(p, plan, stream);
}

} // namespace attention
} // namespace wave
