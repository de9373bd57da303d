// mxfp8_quant.hip -- OCP MX-FP8 encoding of f32 / f16 / bf16 tensors (the
// input format of attention_fwd8.hpp): blocks of 32 values share the e8m0
// scale 2^(floor(log2(amax)) - 8), and each value is x / scale rounded to
// e4m3 (RNE, saturated at +-448).
//
// Bound by HBM: each value is read once and its byte written once, where the
// same steps as tensor operations take about ten passes over float32
// copies.  Three kernels for X [outer][n][inner], blocks along n:
//  * rows (inner = 1, n % 32 == 0): the tensor is one run of blocks; a
//    thread takes half a block (16 values: 32 bytes of 16-bit input, one
//    16-byte store) and its lane pair the block.
//  * cols (inner % 4 == 0): a thread takes 16 rows x 4 columns of a block
//    column, lanes l and l + 32 the two row halves, so every load and store
//    instruction covers runs of 32 * 4 consecutive columns.
//  * any other shape or alignment: one thread a block, element by element.
// Measured at B2 Hq32 Hkv8 S2048 D128 bf16 (rocprofv3): q through the rows
// kernel 9.4 us (50 MB: 5.4 TB/s, against 4.8 for a large device copy), k 5.5
// us, v through the columns kernel 5.6 us (12.6 MB each: mostly launch); the
// three as tensor operations 350 us, in about 30 launches.
#include "mxfp8_quant.hpp"

#include "wave_common.hpp"

namespace wave {
namespace quant {

namespace {

constexpr int kBlock = 32;       // values a scale covers
constexpr uint32_t kInf = 0x7F800000u;

template <int DT> constexpr int elem_bytes() { return DT == kF32 ? 4 : 2; }

// Value i of a run of packed input dwords, as float.
template <int DT> __device__ __forceinline__ float unpack(const uint32_t *w, int i) {
  if constexpr (DT == kF32)
    return __builtin_bit_cast(float, w[i]);
  else
    return from_bits<DT>((uint16_t)(w[i >> 1] >> (16 * (i & 1))));
}

template <int DT> __device__ __forceinline__ float load1(const void *x, size_t i) {
  if constexpr (DT == kF32)
    return static_cast<const float *>(x)[i];
  else
    return from_bits<DT>(static_cast<const uint16_t *>(x)[i]);
}

__device__ __forceinline__ uint32_t abs_bits(float v) {
  return __builtin_bit_cast(uint32_t, v) & 0x7FFFFFFFu;
}

// Exponent of a block whose largest |value| has these bits (compared as
// integers, so a NaN anywhere makes it a NaN): floor(log2(amax)) - 8 within
// [-127, 127]; -127 for an all-zero block and for one with a NaN, 127 with an
// infinity.  16-bit inputs read the exponent field (values below 2^-119 all
// end at -127); f32 ones take floor(log2f(amax)), which rounds up for the
// last few values below a power of two, as the tensor formula does.
template <int DT> __device__ __forceinline__ int block_exponent(uint32_t amax) {
  if (amax == 0u || amax > kInf)
    return -127;
  if (amax == kInf)
    return 127;
  int e;
  if constexpr (DT == kF32)
    e = (int)floorf(log2f(__builtin_bit_cast(float, amax))) - 8;
  else
    e = (int)(amax >> 23) - 127 - 8;
  return e < -127 ? -127 : e > 127 ? 127 : e;
}

// 2^-e, e in [-127, 127] (2^-127 is subnormal): x * 2^-e is x / 2^e rounded
// once, as the division rounds it.
__device__ __forceinline__ float inv_scale(int e) {
  return __builtin_bit_cast(float, e == 127 ? 0x00400000u : (uint32_t)(127 - e) << 23);
}

__device__ __forceinline__ float saturate(float q) {
  return fminf(fmaxf(q, -448.0f), 448.0f);
}

// Four scaled values -> four e4m3 bytes, the first in the low byte.
__device__ __forceinline__ uint32_t pack4(float a, float b, float c, float d) {
  int w = __builtin_amdgcn_cvt_pk_fp8_f32(saturate(a), saturate(b), 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(saturate(c), saturate(d), w, true);
}

// The byte of one value of a block that holds a NaN (its scale is 2^-127).
__device__ __forceinline__ uint32_t byte_nan_block(float x, float inv) {
  if (abs_bits(x) > kInf)
    return 0x7Fu | (__builtin_bit_cast(uint32_t, x) >> 31 << 7);
  return pack4(x * inv, 0.f, 0.f, 0.f) & 0xFFu;
}

// v[0..N) scaled and packed, N a multiple of 4.
template <int N>
__device__ __forceinline__ void encode(const float (&v)[N], uint32_t amax, float inv,
                                       uint32_t (&out)[N / 4]) {
  if (amax > kInf) {
#pragma unroll
    for (int i = 0; i < N / 4; ++i) {
      out[i] = 0u;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        out[i] |= byte_nan_block(v[4 * i + j], inv) << (8 * j);
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < N / 4; ++i)
    out[i] = pack4(v[4 * i] * inv, v[4 * i + 1] * inv, v[4 * i + 2] * inv, v[4 * i + 3] * inv);
}

// Blocks in two grid dimensions: one holds fewer than 2^32 threads.
dim3 grid_of(size_t blocks) {
  constexpr size_t kRow = (size_t)1 << 22;
  return blocks <= kRow ? dim3((unsigned)blocks)
                        : dim3((unsigned)kRow, (unsigned)((blocks + kRow - 1) / kRow));
}
__device__ __forceinline__ size_t linear_block() {
  return (size_t)blockIdx.y * gridDim.x + blockIdx.x;
}

template <int DT>
__global__ __launch_bounds__(256) void rows_kernel(const uint8_t *X, uint8_t *E, uint8_t *S,
                                                   size_t halves) {
  const size_t t = linear_block() * 256 + threadIdx.x;
  if (t >= halves)
    return;  // halves is even: lane pairs stay whole
  constexpr int NW = 16 * elem_bytes<DT>() / 4;
  uint32_t w[NW];
  const u32x4 *src = reinterpret_cast<const u32x4 *>(X + t * (16 * elem_bytes<DT>()));
#pragma unroll
  for (int i = 0; i < NW / 4; ++i) {
    const u32x4 q = src[i];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[4 * i + j] = q[j];
  }
  float v[16];
  uint32_t amax = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    v[i] = unpack<DT>(w, i);
    amax = max(amax, abs_bits(v[i]));
  }
  amax = max(amax, (uint32_t)__shfl_xor((int)amax, 1));
  const int e = block_exponent<DT>(amax);
  uint32_t out[4];
  encode<16>(v, amax, inv_scale(e), out);
  *reinterpret_cast<u32x4 *>(E + t * 16) = u32x4{out[0], out[1], out[2], out[3]};
  if ((t & 1) == 0)
    S[t >> 1] = (uint8_t)(e + 127);
}

// units = outer * blocks * groups, groups = inner / 4; all below 2^31.
template <int DT>
__global__ __launch_bounds__(256) void cols_kernel(const uint8_t *X, uint8_t *E, uint8_t *S,
                                                   uint32_t units, uint32_t n, uint32_t blocks,
                                                   uint32_t groups) {
  const uint32_t lane = threadIdx.x & 63;
  const size_t u = (linear_block() * 4 + (threadIdx.x >> 6)) * 32 + (lane & 31);
  if (u >= units)
    return;  // both halves of a unit leave together
  const uint32_t ob = (uint32_t)u / groups, cg = (uint32_t)u - ob * groups;
  const uint32_t o = ob / blocks, blk = ob - o * blocks;
  const uint32_t row0 = blk * kBlock + (lane >> 5) * 16;
  const size_t inner = (size_t)groups * 4, col = (size_t)cg * 4;
  const size_t base = ((size_t)o * n + row0) * inner + col;
  const uint32_t rows = row0 < n ? min(n - row0, 16u) : 0u;
  constexpr int NW = elem_bytes<DT>();  // dwords of 4 values
  uint32_t w[16][NW];
#pragma unroll
  for (uint32_t r = 0; r < 16; ++r) {
    if (r < rows) {
      const uint8_t *src = X + (base + r * inner) * elem_bytes<DT>();
      if constexpr (DT == kF32) {
        const u32x4 q = *reinterpret_cast<const u32x4 *>(src);
#pragma unroll
        for (int j = 0; j < NW; ++j)
          w[r][j] = q[j];
      } else {
        const u32x2 q = *reinterpret_cast<const u32x2 *>(src);
        w[r][0] = q[0];
        w[r][1] = q[1];
      }
    } else {
#pragma unroll
      for (int j = 0; j < NW; ++j)
        w[r][j] = 0u;
    }
  }
  uint32_t amax[4] = {0, 0, 0, 0};
#pragma unroll
  for (int r = 0; r < 16; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c)
      amax[c] = max(amax[c], abs_bits(unpack<DT>(w[r], c)));
  float inv[4];
  uint32_t scales = 0, worst = 0;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    amax[c] = max(amax[c], (uint32_t)__shfl_xor((int)amax[c], 32));
    const int e = block_exponent<DT>(amax[c]);
    inv[c] = inv_scale(e);
    scales |= (uint32_t)(e + 127) << (8 * c);
    worst = max(worst, amax[c]);
  }
#pragma unroll
  for (uint32_t r = 0; r < 16; ++r) {
    if (r < rows) {
      float v[4];
#pragma unroll
      for (int c = 0; c < 4; ++c)
        v[c] = unpack<DT>(w[r], c);
      uint32_t q;
      if (worst > kInf) {
        q = 0;
#pragma unroll
        for (int c = 0; c < 4; ++c)
          q |= byte_nan_block(v[c], inv[c]) << (8 * c);
      } else {
        q = pack4(v[0] * inv[0], v[1] * inv[1], v[2] * inv[2], v[3] * inv[3]);
      }
      *reinterpret_cast<uint32_t *>(E + base + r * inner) = q;
    }
  }
  if (lane < 32)
    *reinterpret_cast<uint32_t *>(S + (size_t)ob * inner + col) = scales;
}

template <int DT>
__global__ __launch_bounds__(256) void any_kernel(const void *X, uint8_t *E, uint8_t *S,
                                                  size_t total, size_t n, size_t blocks,
                                                  size_t inner) {
  const size_t t = linear_block() * 256 + threadIdx.x;  // (outer, block, inner)
  if (t >= total)
    return;
  const size_t ob = t / inner, i = t - ob * inner;
  const size_t o = ob / blocks, blk = ob - o * blocks;
  const size_t row0 = blk * kBlock, rows = min(n - row0, (size_t)kBlock);
  const size_t base = (o * n + row0) * inner + i;
  uint32_t amax = 0;
  for (size_t r = 0; r < rows; ++r)
    amax = max(amax, abs_bits(load1<DT>(X, base + r * inner)));
  const int e = block_exponent<DT>(amax);
  const float inv = inv_scale(e);
  for (size_t r = 0; r < rows; ++r)
    E[base + r * inner] = (uint8_t)byte_nan_block(load1<DT>(X, base + r * inner), inv);
  S[t] = (uint8_t)(e + 127);
}

template <int DT>
hipError_t launch_dt(const void *X, void *E, void *S, size_t outer, size_t n, size_t inner,
                     hipStream_t stream) {
  const size_t blocks = (n + kBlock - 1) / kBlock;
  const uint8_t *x = static_cast<const uint8_t *>(X);
  uint8_t *e = static_cast<uint8_t *>(E), *s = static_cast<uint8_t *>(S);
  const uintptr_t xa = (uintptr_t)X, ea = (uintptr_t)E, sa = (uintptr_t)S;
  const size_t groups = inner / 4, units = outer * blocks * groups;
  size_t threads;
  // The vector kernels where a block's values sit in whole aligned vectors:
  // 16-byte loads and stores along the row, or 4 columns (8 or 16 bytes in,
  // 4 out) across it.
  if (inner == 1 && n % kBlock == 0 && (xa | ea) % 16 == 0 &&
      outer * n / 16 < ((size_t)1 << 39)) {
    threads = outer * n / 16;
    hipLaunchKernelGGL((rows_kernel<DT>), grid_of((threads + 255) / 256), dim3(256), 0,
                       stream, x, e, s, threads);
  } else if (inner % 4 == 0 && n < ((size_t)1 << 31) && units < ((size_t)1 << 31) &&
             xa % (4 * elem_bytes<DT>()) == 0 && (ea | sa) % 4 == 0) {
    hipLaunchKernelGGL((cols_kernel<DT>), grid_of((units + 127) / 128), dim3(256), 0,
                       stream, x, e, s, (uint32_t)units, (uint32_t)n, (uint32_t)blocks,
                       (uint32_t)groups);
  } else {
    threads = outer * blocks * inner;
    if (threads >= ((size_t)1 << 39))
      return hipErrorInvalidValue;
    hipLaunchKernelGGL((any_kernel<DT>), grid_of((threads + 255) / 256), dim3(256), 0,
                       stream, X, e, s, threads, n, blocks, inner);
  }
  return hipGetLastError();
}

} // namespace

hipError_t launch_mxfp8(const void *X, void *E, void *S, size_t outer, size_t n, size_t inner,
                        int dtype, hipStream_t stream) {
  if (dtype == kF32)
    return launch_dt<kF32>(X, E, S, outer, n, inner, stream);
  if (dtype == kF16)
    return launch_dt<kF16>(X, E, S, outer, n, inner, stream);
  return launch_dt<kBF16>(X, E, S, outer, n, inner, stream);
}

} // namespace quant
} // namespace wave
