// qmlp_pack.hip -- load-time weight preparation kernels: canonical bfp8 quantisation, packing into
// the tiled layout (qmlp_common.h), the inverse unpack, and an audit dequantiser that reuses the
// GEMM's in-register dequant routine.
#include "qmlp_common.h"
#include "qmlp_internal.h"

namespace qmlp {

// ---------------------------------------------------------------- canonical quantisation
//
// One thread per 16-value group.  Exact integer arithmetic on the bf16 words: a value is
// sig * 2^ex0 with sig < 256; its frexp exponent is bitlen(sig) + ex0.  The shared exponent is the
// largest of the group; q = round-half-even(sig * 2^(ex0 - (e8-127))) clamped to 2^MB - 1.
// MB magnitude bits: 7 (bfp8) or 3 (bf4).
template <int MB>
__global__ void quantize_kernel(const uint16_t* __restrict__ w, int rows, int cols, int8_t* __restrict__ q,
                                uint8_t* __restrict__ e8, uint32_t* bad) {
  const int groups = cols / 16;
  const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= (long)rows * groups) return;
  const int r = (int)(gid / groups), g = (int)(gid % groups);
  const uint16_t* src = w + (size_t)r * cols + (size_t)g * 16;
  const u32x4 lo = *(const u32x4*)src;
  const u32x4 hi = *(const u32x4*)(src + 8);
  uint16_t v[16];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = (uint16_t)(lo[i] & 0xffffu);
    v[2 * i + 1] = (uint16_t)(lo[i] >> 16);
    v[8 + 2 * i] = (uint16_t)(hi[i] & 0xffffu);
    v[8 + 2 * i + 1] = (uint16_t)(hi[i] >> 16);
  }
  int sig[16], ex0[16];
  int shared = -100000;
  bool finite = true, any = false;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int ef = (v[i] >> 7) & 0xff, mf = v[i] & 0x7f;
    if (ef == 0xff) finite = false;
    if (ef == 0) {
      sig[i] = mf;
      ex0[i] = -133;
    } else {
      sig[i] = 128 | mf;
      ex0[i] = ef - 134;
    }
    if (sig[i]) {
      any = true;
      const int e = (32 - __clz(sig[i])) + ex0[i];
      shared = e > shared ? e : shared;
    }
  }
  uint32_t out[4] = {0u, 0u, 0u, 0u};
  uint8_t ebyte = 0;
  if (!finite) {
    if (bad) atomicAdd(bad, 1u);
  } else if (any) {
    int e = shared + 127 - MB;
    e = e < 1 ? 1 : (e > 254 ? 254 : e);
    ebyte = (uint8_t)e;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int s = (e - 127) - ex0[i];  // right shift, >= 1 by construction
      int m;
      if (s >= 10) {
        m = 0;  // sig < 2^8, so sig / 2^s < 1/2
      } else {
        m = sig[i] >> s;
        const int rem = sig[i] & ((1 << s) - 1), half = 1 << (s - 1);
        if (rem > half || (rem == half && (m & 1))) ++m;
      }
      m = m > (1 << MB) - 1 ? (1 << MB) - 1 : m;
      const int qv = (v[i] & 0x8000) ? -m : m;
      out[i / 4] |= ((uint32_t)(qv & 0xff)) << (8 * (i % 4));
    }
  }
  *(u32x4*)(q + (size_t)r * cols + (size_t)g * 16) = u32x4{out[0], out[1], out[2], out[3]};
  e8[(size_t)r * groups + g] = ebyte;
}

// ---------------------------------------------------------------- packing

// Writes the whole 256-byte trailer (zero padding), so a packed buffer's bytes depend only on the
// weights -- packed buffers compare bit-for-bit and cache files are reproducible.
__global__ void trailer_init_kernel(Trailer* t) {
  uint32_t* words = (uint32_t*)t;
  for (int i = threadIdx.x; i < kTrailer / 4; i += blockDim.x) words[i] = 0u;
  __syncthreads();
  if (threadIdx.x == 0) t->magic = kTrailerMagic;
}

// One workgroup (256 threads) per row: row base exponent, rowexp, L2 norm, flushed-group count.
__global__ void rowinfo_bfp8_kernel(const int8_t* __restrict__ q, const uint8_t* __restrict__ e8,
                                    int rows, int cols, int* __restrict__ rowexp, Trailer* trailer) {
  __shared__ int smax[256];
  __shared__ double ssum[256];
  __shared__ unsigned sflush[256];
  const int r = blockIdx.x, groups = cols / 16;
  const uint8_t* er = e8 + (size_t)r * groups;
  int mx = 0;
  for (int g = threadIdx.x; g < groups; g += 256) mx = max(mx, (int)er[g]);
  smax[threadIdx.x] = mx;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) smax[threadIdx.x] = max(smax[threadIdx.x], smax[threadIdx.x + s]);
    __syncthreads();
  }
  const int base = smax[0];
  double acc = 0.0;
  unsigned flushed = 0;
  for (int g = threadIdx.x; g < groups; g += 256) {
    const int e = er[g];
    if (!e) continue;
    if (e - base + 20 < 1) ++flushed;
    const int8_t* qg = q + (size_t)r * cols + (size_t)g * 16;
    int sq = 0;
    for (int i = 0; i < 16; ++i) sq += (int)qg[i] * (int)qg[i];
    acc += ldexp((double)sq, 2 * (e - 127));
  }
  ssum[threadIdx.x] = acc;
  sflush[threadIdx.x] = flushed;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
      ssum[threadIdx.x] += ssum[threadIdx.x + s];
      sflush[threadIdx.x] += sflush[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    rowexp[r] = base - 132;
    const double n = sqrt(ssum[0]);
    atomicMax(&trailer->max_row_norm_bits, (unsigned long long)__double_as_longlong(n));
    if (sflush[0]) atomicAdd(&trailer->flushed_groups, sflush[0]);
  }
}

__global__ void rowinfo_bf16_kernel(const uint16_t* __restrict__ w, int rows, int cols,
                                    int* __restrict__ rowexp, Trailer* trailer) {
  __shared__ double ssum[256];
  const int r = blockIdx.x;
  double acc = 0.0;
  for (int k = threadIdx.x; k < cols; k += 256) {
    const double v = (double)bf16_to_f32(w[(size_t)r * cols + k]);
    acc += v * v;
  }
  ssum[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) ssum[threadIdx.x] += ssum[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    rowexp[r] = 0;
    atomicMax(&trailer->max_row_norm_bits, (unsigned long long)__double_as_longlong(sqrt(ssum[0])));
  }
}

// Exponent dword of lane l of block (t, sb): byte j = E5 << 2 of the lane's group in K-step j.
__device__ __forceinline__ uint32_t lane_exponents(const uint8_t* e8, int cols, int row, int sb, int qq,
                                                   const int* rowexp) {
  const int groups = cols / 16;
  const int base = rowexp[row] + 132;
  uint32_t dw = 0;
  for (int jj = 0; jj < kSteps; ++jj) {
    const int e = e8[(size_t)row * groups + sb * 16 + jj * 4 + qq];
    const int e5 = e - base + 20;
    dw |= ((e && e5 >= 1) ? (uint32_t)(e5 << 2) : 0u) << (8 * jj);
  }
  return dw;
}

// One thread per (block u, K-step j, lane l): 16 mantissa bytes; j == 0 threads also write the
// lane's exponent dword.
__global__ void pack_bfp8_kernel(const int8_t* __restrict__ q, const uint8_t* __restrict__ e8,
                                 int rows, int cols, const int* __restrict__ rowexp,
                                 uint8_t* __restrict__ packed) {
  const int C = cols / kSuperK;
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = (long)(rows / kTileRows) * C * kSteps * 64;
  if (tid >= total) return;
  const int l = (int)(tid & 63);
  const int j = (int)((tid >> 6) & 3);
  const long u = tid >> 8;
  const int t = (int)(u / C), sb = (int)(u % C);
  const int r = l & 15, qq = l >> 4;
  const int row = t * kTileRows + r;
  const int k0 = sb * kSuperK + j * 64 + qq * 16;
  const u32x4 src = *(const u32x4*)(q + (size_t)row * cols + k0);
  uint8_t* blk = packed + (size_t)u * kBfp8Block;
  *(u32x4*)(blk + j * 1024 + l * 16) = src ^ u32x4{0x80808080u, 0x80808080u, 0x80808080u, 0x80808080u};
  if (j == 0) *(uint32_t*)(blk + 4096 + l * 4) = lane_exponents(e8, cols, row, sb, qq, rowexp);
}

// bf4: one thread per (block u, K-step pair p, lane l): 2 x 16 mantissas -> 16 nibble bytes.
__device__ __forceinline__ uint32_t nibbles8(const int8_t* v) {  // values v[0..7] -> one dword
  uint32_t d = 0;
#pragma unroll
  for (int b = 0; b < 4; ++b)
    d |= ((uint32_t)(v[b] + 8) | ((uint32_t)(v[b + 4] + 8) << 4)) << (8 * b);
  return d;
}

__global__ void pack_bf4_kernel(const int8_t* __restrict__ q, const uint8_t* __restrict__ e8, int rows, int cols,
                                const int* __restrict__ rowexp, uint8_t* __restrict__ packed) {
  const int C = cols / kSuperK;
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = (long)(rows / kTileRows) * C * 2 * 64;
  if (tid >= total) return;
  const int l = (int)(tid & 63);
  const int pp = (int)((tid >> 6) & 1);
  const long u = tid >> 7;
  const int t = (int)(u / C), sb = (int)(u % C);
  const int qq = l >> 4, row = t * kTileRows + (l & 15);
  uint32_t out[4];
#pragma unroll
  for (int sub = 0; sub < 2; ++sub) {
    const int j = 2 * pp + sub;
    int8_t v[16];
    const int8_t* src = q + (size_t)row * cols + sb * kSuperK + j * 64 + qq * 16;
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = src[i];
    out[2 * sub] = nibbles8(v);
    out[2 * sub + 1] = nibbles8(v + 8);
  }
  uint8_t* blk = packed + (size_t)u * kBf4Block;
  *(u32x4*)(blk + pp * 1024 + l * 16) = u32x4{out[0], out[1], out[2], out[3]};
  if (pp == 0) *(uint32_t*)(blk + 2048 + l * 4) = lane_exponents(e8, cols, row, sb, qq, rowexp);
}

// Inverse of pack_bf4_kernel (same thread mapping).
__global__ void unpack_bf4_kernel(const uint8_t* __restrict__ packed, int rows, int cols,
                                  const int* __restrict__ rowexp, int8_t* __restrict__ q, uint8_t* __restrict__ e8) {
  const int C = cols / kSuperK;
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = (long)(rows / kTileRows) * C * 2 * 64;
  if (tid >= total) return;
  const int l = (int)(tid & 63);
  const int pp = (int)((tid >> 6) & 1);
  const long u = tid >> 7;
  const int t = (int)(u / C), sb = (int)(u % C);
  const int qq = l >> 4, row = t * kTileRows + (l & 15);
  const uint8_t* blk = packed + (size_t)u * kBf4Block;
  const u32x4 m = *(const u32x4*)(blk + pp * 1024 + l * 16);
  const uint32_t dw = *(const uint32_t*)(blk + 2048 + l * 4);
  const int base = rowexp[row] + 132;
#pragma unroll
  for (int sub = 0; sub < 2; ++sub) {
    const int j = 2 * pp + sub;
    int8_t* dst = q + (size_t)row * cols + sb * kSuperK + j * 64 + qq * 16;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t d = m[2 * sub + h];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        dst[8 * h + b] = (int8_t)((int)((d >> (8 * b)) & 0xfu) - 8);
        dst[8 * h + b + 4] = (int8_t)((int)((d >> (8 * b + 4)) & 0xfu) - 8);
      }
    }
    const int e5 = (int)((dw >> (8 * j)) & 0xffu) >> 2;
    e8[(size_t)row * (cols / 16) + sb * 16 + j * 4 + qq] = (uint8_t)(e5 ? e5 - 20 + base : 0);
  }
}

// Audit dequantiser for bf4: the GEMM's dq16_bf4 routine, then the row scale.
__global__ void dequant_bf4_kernel(const uint8_t* __restrict__ packed, int rows, int cols,
                                   const int* __restrict__ rowexp, float* __restrict__ out) {
  const int C = cols / kSuperK;
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = (long)(rows / kTileRows) * C * kSteps * 64;
  if (tid >= total) return;
  const int l = (int)(tid & 63);
  const int j = (int)((tid >> 6) & 3);
  const long u = tid >> 8;
  const int t = (int)(u / C), sb = (int)(u % C);
  const int row = t * kTileRows + (l & 15), qq = l >> 4;
  const uint8_t* blk = packed + (size_t)u * kBf4Block;
  const u32x2 m = *(const u32x2*)(blk + (j >> 1) * 1024 + l * 16 + (j & 1) * 8);
  const uint32_t dw = *(const uint32_t*)(blk + 2048 + l * 4);
  f16x8 a0, a1;
  dq16_bf4(m.x, m.y, scale_pair(dw, j), a0, a1);
  const int re = rowexp[row];
  float* o = out + (size_t)row * cols + sb * kSuperK + j * 64 + qq * 16;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    o[i] = __builtin_amdgcn_ldexpf((float)a0[i], re);
    o[8 + i] = __builtin_amdgcn_ldexpf((float)a1[i], re);
  }
}

// One thread per (block, K-step, half, lane): 8 bf16 values (16 bytes).
__global__ void pack_bf16_kernel(const uint16_t* __restrict__ w, int rows, int cols,
                                 uint8_t* __restrict__ packed) {
  const int C = cols / kSuperK;
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = (long)(rows / kTileRows) * C * kSteps * 2 * 64;
  if (tid >= total) return;
  const int l = (int)(tid & 63);
  const int h = (int)((tid >> 6) & 1);
  const int j = (int)((tid >> 7) & 3);
  const long u = tid >> 9;
  const int t = (int)(u / C), sb = (int)(u % C);
  const int row = t * kTileRows + (l & 15);
  const int k0 = sb * kSuperK + j * 64 + (l >> 4) * 16 + h * 8;
  *(u32x4*)(packed + (size_t)u * kBf16Block + j * 2048 + h * 1024 + l * 16) =
      *(const u32x4*)(w + (size_t)row * cols + k0);
}

// Inverse of pack_bfp8_kernel (same thread mapping).
__global__ void unpack_bfp8_kernel(const uint8_t* __restrict__ packed, int rows, int cols,
                                   const int* __restrict__ rowexp, int8_t* __restrict__ q,
                                   uint8_t* __restrict__ e8) {
  const int C = cols / kSuperK;
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = (long)(rows / kTileRows) * C * kSteps * 64;
  if (tid >= total) return;
  const int l = (int)(tid & 63);
  const int j = (int)((tid >> 6) & 3);
  const long u = tid >> 8;
  const int t = (int)(u / C), sb = (int)(u % C);
  const int row = t * kTileRows + (l & 15), qq = l >> 4;
  const uint8_t* blk = packed + (size_t)u * kBfp8Block;
  const u32x4 m = *(const u32x4*)(blk + j * 1024 + l * 16);
  *(u32x4*)(q + (size_t)row * cols + sb * kSuperK + j * 64 + qq * 16) =
      m ^ u32x4{0x80808080u, 0x80808080u, 0x80808080u, 0x80808080u};
  const uint32_t dw = *(const uint32_t*)(blk + 4096 + l * 4);
  const int e5 = (int)((dw >> (8 * j)) & 0xffu) >> 2;
  const int base = rowexp[row] + 132;
  e8[(size_t)row * (cols / 16) + sb * 16 + j * 4 + qq] = (uint8_t)(e5 ? e5 - 20 + base : 0);
}

// Audit dequantiser: the GEMM's dq16 routine, then the row scale.
__global__ void dequant_bfp8_kernel(const uint8_t* __restrict__ packed, int rows, int cols,
                                    const int* __restrict__ rowexp, float* __restrict__ out) {
  const int C = cols / kSuperK;
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = (long)(rows / kTileRows) * C * kSteps * 64;
  if (tid >= total) return;
  const int l = (int)(tid & 63);
  const int j = (int)((tid >> 6) & 3);
  const long u = tid >> 8;
  const int t = (int)(u / C), sb = (int)(u % C);
  const int row = t * kTileRows + (l & 15), qq = l >> 4;
  const uint8_t* blk = packed + (size_t)u * kBfp8Block;
  const u32x4 m = *(const u32x4*)(blk + j * 1024 + l * 16);
  const uint32_t dw = *(const uint32_t*)(blk + 4096 + l * 4);
  f16x8 a0, a1;
  dq16(m, scale_pair(dw, j), a0, a1);
  const int re = rowexp[row];
  float* o = out + (size_t)row * cols + sb * kSuperK + j * 64 + qq * 16;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    o[i] = __builtin_amdgcn_ldexpf((float)a0[i], re);
    o[8 + i] = __builtin_amdgcn_ldexpf((float)a1[i], re);
  }
}

__global__ void dequant_bf16_kernel(const uint8_t* __restrict__ packed, int rows, int cols,
                                    float* __restrict__ out) {
  const int C = cols / kSuperK;
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = (long)(rows / kTileRows) * C * kSteps * 2 * 64;
  if (tid >= total) return;
  const int l = (int)(tid & 63);
  const int h = (int)((tid >> 6) & 1);
  const int j = (int)((tid >> 7) & 3);
  const long u = tid >> 9;
  const int t = (int)(u / C), sb = (int)(u % C);
  const int row = t * kTileRows + (l & 15);
  const int k0 = sb * kSuperK + j * 64 + (l >> 4) * 16 + h * 8;
  const u32x4 v = *(const u32x4*)(packed + (size_t)u * kBf16Block + j * 2048 + h * 1024 + l * 16);
  float* o = out + (size_t)row * cols + k0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[2 * i] = bf16_to_f32((uint16_t)(v[i] & 0xffffu));
    o[2 * i + 1] = bf16_to_f32((uint16_t)(v[i] >> 16));
  }
}

// ---------------------------------------------------------------- quantise and pack in one pass
//
// bf16 weights -> packed layout, the same bytes as quantize_kernel / rowinfo / pack kernels leave,
// with one read of the weights and one write of the packed matrix.  Those passes write and re-read
// the canonical mantissas and exponents.  us per 27B matrix, 17408 x 5120 and 5120 x 17408: bfp8
// 77 + 205 + 34 and 77 + 68 + 34 there, 62 and 74 here (4.4 and 3.7 TB/s); bf4 80 + 202 + 26, here
// 56; bf16 weights 215 + 60 and 130 + 60, here 89 and 83.
//
// Bound by memory.  One block of 8 waves per 16-row tile; lane l = 16 quarter + row holds one
// 16-value group, the unit of the packed layout, so a wave's step reads 128 contiguous bytes of 16
// rows and writes 1 KB.  The mantissas do not depend on the row's base exponent and leave at once;
// the shared exponents wait (in LDS, or in their own place in the packed matrix for rows too long
// for it) until the row's largest is known.  The next superblock is in flight while one is
// converted (64 KB per block).  The 5120-row matrix has 320 blocks for 256 CUs, hence its lower rate.
//
// Row norms are sums in double precision in rowinfo's order -- accumulator t of 256 takes the
// groups t, t + 256, ..., then halves are added, t + 128 first -- so that they are the same bits:
// wave w takes superblocks w, w + 8, ..., whose groups belong to accumulators 16 (sb % 16) + 4 j +
// quarter, i.e. 2 x 4 per lane.

constexpr int kPackWaves = 8;
constexpr int kPackLdsExp = 176;  // superblocks whose exponent words fit beside the norm sums in 64 KB of LDS

struct PackedGroup {
  uint32_t d[4];  // bfp8: 16 bytes excess-128; bf4: two dwords of nibbles excess-8
  uint32_t e;     // shared exponent, 0: all zero or not finite
  int sq;         // sum of the squared mantissas
  bool finite;
};

// One group: q = round-half-even(v * 2^(127 - e)) clamped to 2^MB - 1 magnitudes, e from the largest
// magnitude.  v has 8 significant bits and the scale is a power of two, so the product is exact
// (or far below 1/2); adding 1.5 * 2^23 rounds it half to even into the low mantissa bits.
template <int MB>
__device__ __forceinline__ PackedGroup quantize_group(u32x4 lo, u32x4 hi) {
  PackedGroup o;
  uint32_t mx = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    mx = max(mx, max(lo[i] & 0x7fffu, (lo[i] >> 16) & 0x7fffu));
    mx = max(mx, max(hi[i] & 0x7fffu, (hi[i] >> 16) & 0x7fffu));
  }
  o.finite = mx < 0x7f80u;
  const bool live = o.finite && mx != 0;
  const int e = max(1, (int)(mx >> 7) + 1 - MB);
  o.e = live ? (uint32_t)e : 0u;
  constexpr float TOP = (float)((1 << MB) - 1);
  constexpr float BIAS = 12582912.0f + (float)(1 << MB);  // 1.5 * 2^23: round, and the excess
  uint32_t u[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const uint32_t w = i < 8 ? lo[i / 2] : hi[i / 2 - 4];
    const float v = __uint_as_float((i & 1) ? (w & 0xffff0000u) : (w << 16));
    const float x = fminf(fmaxf(__builtin_amdgcn_ldexpf(v, 127 - e), -TOP), TOP);
    u[i] = live ? __float_as_uint(x + BIAS) & 0xffu : (uint32_t)(1 << MB);
  }
  uint32_t b[4];  // bytes in value order
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = u[4 * i] | (u[4 * i + 1] << 8) | (u[4 * i + 2] << 16) | (u[4 * i + 3] << 24);
  int sq = MB == 7 ? 0 : 16 * 64;  // bf4: sum (u - 8)^2 = sum u^2 - 16 sum u + 16 * 64
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (MB == 7) {
      const int m = (int)(b[i] ^ 0x80808080u);
      sq = __builtin_amdgcn_sdot4(m, m, sq, false);
    } else {
      sq = __builtin_amdgcn_sdot4((int)b[i], (int)b[i], sq, false);
      sq = __builtin_amdgcn_sdot4((int)b[i], (int)0xf0f0f0f0u, sq, false);  // -16 in every byte
    }
  }
  o.sq = sq;
  if constexpr (MB == 7) {
#pragma unroll
    for (int i = 0; i < 4; ++i) o.d[i] = b[i];
  } else {  // byte b of dword h: u[8 h + b] | u[8 h + b + 4] << 4
    o.d[0] = b[0] | (b[1] << 4);
    o.d[1] = b[2] | (b[3] << 4);
    o.d[2] = o.d[3] = 0;
  }
  return o;
}

// The block's row norms from acc[wave][j][lane] (accumulators t and t + 128 already added), by wave
// 0: row lane % 16, the result in lanes 0..15; then the trailer's maximum.
__device__ __forceinline__ void finish_norms(double sum, int lane, Trailer* tr) {
  unsigned long long n = (unsigned long long)__double_as_longlong(sqrt(sum));
  if (lane >= 16) n = 0;
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) {
    const unsigned long long other = __shfl_xor(n, o);
    n = n > other ? n : other;
  }
  if (lane == 0) atomicMax(&tr->max_row_norm_bits, n);
}

template <int MB, bool EXP_LDS>
__global__ __launch_bounds__(kPackWaves * 64, 4) void quantize_pack_kernel(const uint16_t* __restrict__ w, int cols,
                                                                       uint8_t* __restrict__ packed,
                                                                       int* __restrict__ rowexp, PackTrailer* tr) {
  constexpr int BLK = MB == 7 ? kBfp8Block : kBf4Block;
  extern __shared__ uint32_t s_e[];  // EXP_LDS: [C][64] shared exponents, byte j of a lane's word: K-step j
  __shared__ double s_acc[kPackWaves][kSteps][64];
  __shared__ int s_max[kPackWaves][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, C = cols / kSuperK;
  const int row = blockIdx.x * kTileRows + (lane & 15);
  const uint16_t* src = w + (size_t)row * cols + (lane >> 4) * 16;
  uint8_t* dst = packed + (size_t)blockIdx.x * C * BLK;
  u32x4 v[kSteps][2];
  auto load = [&](int j, int sb) {
    const uint16_t* s = src + (size_t)min(sb, C - 1) * kSuperK + j * 64;
    v[j][0] = *(const u32x4*)s;
    v[j][1] = *(const u32x4*)(s + 8);
  };
  auto exponents = [&](int sb) {
    return EXP_LDS ? s_e + sb * 64 + lane : (uint32_t*)(dst + (size_t)sb * BLK + (BLK - 256) + lane * 4);
  };
  double acc[2][kSteps] = {};
  int emax = 0;
  uint32_t bad = 0;
  // converts superblock sb and requests the wave's next one, K-step by K-step
  auto convert = [&](int sb, double(&a)[kSteps]) {
    uint8_t* blk = dst + (size_t)sb * BLK;
    uint32_t ew = 0;
    u32x4 pair;  // bf4: two K-steps share a 16-byte slot
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
      const PackedGroup g = quantize_group<MB>(v[j][0], v[j][1]);
      load(j, sb + kPackWaves);
      if constexpr (MB == 7) {
        *(u32x4*)(blk + j * 1024 + lane * 16) = u32x4{g.d[0], g.d[1], g.d[2], g.d[3]};
      } else {
        pair[2 * (j & 1)] = g.d[0];
        pair[2 * (j & 1) + 1] = g.d[1];
        if (j & 1) *(u32x4*)(blk + (j >> 1) * 1024 + lane * 16) = pair;
      }
      ew |= g.e << (8 * j);
      emax = max(emax, (int)g.e);
      bad += g.finite ? 0u : 1u;
      a[j] += ldexp((double)g.sq, 2 * ((int)g.e - 127));
    }
    *exponents(sb) = ew;
  };
#pragma unroll
  for (int j = 0; j < kSteps; ++j) load(j, wave);
  for (int sb = wave; sb < C; sb += 2 * kPackWaves) {
    convert(sb, acc[0]);
    if (sb + kPackWaves < C) convert(sb + kPackWaves, acc[1]);
  }
  emax = max(emax, __shfl_xor(emax, 16));
  emax = max(emax, __shfl_xor(emax, 32));
  if (lane < 16) s_max[wave][lane] = emax;
#pragma unroll
  for (int j = 0; j < kSteps; ++j) s_acc[wave][j][lane] = acc[0][j] + acc[1][j];
  if (bad) atomicAdd(&tr->bad_groups, bad);
  __syncthreads();
  int base = 0;
#pragma unroll
  for (int v = 0; v < kPackWaves; ++v) base = max(base, s_max[v][lane & 15]);
  uint32_t flushed = 0;
  for (int sb = wave; sb < C; sb += kPackWaves) {
    const uint32_t ew = *exponents(sb);  // this thread's own words
    uint32_t o = 0;
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
      const int e = (int)((ew >> (8 * j)) & 0xffu), e5 = e - base + 20;
      if (e && e5 < 1) ++flushed;
      o |= ((e && e5 >= 1) ? (uint32_t)(e5 << 2) : 0u) << (8 * j);
    }
    *(uint32_t*)(dst + (size_t)sb * BLK + (BLK - 256) + lane * 4) = o;
  }
  if (flushed) atomicAdd(&tr->flushed_groups, flushed);
  if (wave == 0) {
    double s[kSteps];
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {  // accumulator bits 6, 5, 4: waves v + 4, v + 2, v + 1
      double t[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) t[v] = s_acc[v][j][lane] + s_acc[v + 4][j][lane];
      s[j] = (t[0] + t[2]) + (t[1] + t[3]);
    }
    double sum = (s[0] + s[2]) + (s[1] + s[3]);  // bits 3, 2: K-steps
    sum += __shfl_xor(sum, 32);                  // bits 1, 0: quarters
    sum += __shfl_xor(sum, 16);
    if (lane < 16) rowexp[row] = base - 132;
    finish_norms(sum, lane, tr);
  }
}

// bf16 weights: the packed layout is a permutation; wave (j, h) moves its 8 values per lane of every
// superblock in order, which are accumulators t = 64 j + 16 quarter + 8 h + 0..7 of the row norm.
__global__ __launch_bounds__(kPackWaves * 64) void pack_bf16_fused_kernel(const uint16_t* __restrict__ w, int cols,
                                                                         uint8_t* __restrict__ packed,
                                                                         int* __restrict__ rowexp, Trailer* tr) {
  constexpr int DEPTH = 4;  // superblocks in flight per wave
  __shared__ double s_acc[kPackWaves][8][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, C = cols / kSuperK;
  const int j = wave >> 1, h = wave & 1;
  const int row = blockIdx.x * kTileRows + (lane & 15);
  const uint16_t* src = w + (size_t)row * cols + j * 64 + (lane >> 4) * 16 + h * 8;
  uint8_t* dst = packed + (size_t)blockIdx.x * C * kBf16Block + j * 2048 + h * 1024 + lane * 16;
  double acc[8] = {};
  u32x4 v[DEPTH];
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) v[d] = *(const u32x4*)(src + (size_t)min(d, C - 1) * kSuperK);
  for (int s0 = 0; s0 < C; s0 += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const int sb = s0 + d;
      if (sb < C) {
        const u32x4 t = v[d];
        v[d] = *(const u32x4*)(src + (size_t)min(sb + DEPTH, C - 1) * kSuperK);
        *(u32x4*)(dst + (size_t)sb * kBf16Block) = t;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const double x = (double)__uint_as_float((i & 1) ? (t[i / 2] & 0xffff0000u) : (t[i / 2] << 16));
          acc[i] += x * x;
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) s_acc[wave][i][lane] = acc[i];
  __syncthreads();
  if (wave != 0) return;
  double s[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    double t[2];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {  // bits 7, 6: K-steps; bits 5, 4: quarters
      t[hh] = (s_acc[hh][i][lane] + s_acc[4 + hh][i][lane]) + (s_acc[2 + hh][i][lane] + s_acc[6 + hh][i][lane]);
      t[hh] += __shfl_xor(t[hh], 32);
      t[hh] += __shfl_xor(t[hh], 16);
    }
    s[i] = t[0] + t[1];  // bit 3: half
  }
  const double sum = ((s[0] + s[4]) + (s[2] + s[6])) + ((s[1] + s[5]) + (s[3] + s[7]));
  if (lane < 16) rowexp[row] = 0;
  finish_norms(sum, lane, tr);
}

__global__ void fill_zero_kernel(u32x4* __restrict__ p, size_t n16) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (size_t)gridDim.x * blockDim.x)
    p[i] = u32x4{0u, 0u, 0u, 0u};
}

// ---------------------------------------------------------------- host launchers

static inline unsigned blocks_for(long n, int threads) { return (unsigned)((n + threads - 1) / threads); }

int launch_quantize(const void* w, int rows, int cols, void* q, void* e8, uint32_t* bad, int mbits, hipStream_t s) {
  const long n = (long)rows * (cols / 16);
  if (mbits == 3)
    hipLaunchKernelGGL(quantize_kernel<3>, dim3(blocks_for(n, 256)), dim3(256), 0, s, (const uint16_t*)w, rows, cols,
                       (int8_t*)q, (uint8_t*)e8, bad);
  else
    hipLaunchKernelGGL(quantize_kernel<7>, dim3(blocks_for(n, 256)), dim3(256), 0, s, (const uint16_t*)w, rows, cols,
                       (int8_t*)q, (uint8_t*)e8, bad);
  return check_launch("quantize_kernel");
}

int launch_pack(const void* src0, const void* src1, int rows, int cols, int fmt, void* packed, hipStream_t s) {
  uint8_t* base = (uint8_t*)packed;
  int* rowexp = (int*)(base + rowexp_offset(rows, cols, fmt));
  Trailer* tr = (Trailer*)(base + trailer_offset(rows, cols, fmt));
  hipLaunchKernelGGL(trailer_init_kernel, dim3(1), dim3(64), 0, s, tr);
  if (fmt == 1 || fmt == 2) {
    hipLaunchKernelGGL(rowinfo_bfp8_kernel, dim3(rows), dim3(256), 0, s, (const int8_t*)src0,
                       (const uint8_t*)src1, rows, cols, rowexp, tr);
    if (fmt == 1) {
      const long n = (long)(rows / kTileRows) * (cols / kSuperK) * kSteps * 64;
      hipLaunchKernelGGL(pack_bfp8_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, (const int8_t*)src0,
                         (const uint8_t*)src1, rows, cols, (const int*)rowexp, base);
    } else {
      const long n = (long)(rows / kTileRows) * (cols / kSuperK) * 2 * 64;
      hipLaunchKernelGGL(pack_bf4_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, (const int8_t*)src0,
                         (const uint8_t*)src1, rows, cols, (const int*)rowexp, base);
    }
  } else {
    hipLaunchKernelGGL(rowinfo_bf16_kernel, dim3(rows), dim3(256), 0, s, (const uint16_t*)src0, rows, cols,
                       rowexp, tr);
    const long n = (long)(rows / kTileRows) * (cols / kSuperK) * kSteps * 2 * 64;
    hipLaunchKernelGGL(pack_bf16_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, (const uint16_t*)src0, rows,
                       cols, base);
  }
  return check_launch("pack kernels");
}

int launch_quantize_pack(const void* w, int rows, int cols, int fmt, void* packed, hipStream_t s) {
  uint8_t* base = (uint8_t*)packed;
  int* rowexp = (int*)(base + rowexp_offset(rows, cols, fmt));
  PackTrailer* tr = (PackTrailer*)(base + trailer_offset(rows, cols, fmt));
  const dim3 grid(rows / kTileRows), block(kPackWaves * 64);
  hipLaunchKernelGGL(trailer_init_kernel, dim3(1), dim3(64), 0, s, (Trailer*)tr);
  if (fmt == 0) {
    hipLaunchKernelGGL(pack_bf16_fused_kernel, grid, block, 0, s, (const uint16_t*)w, cols, base, rowexp,
                       (Trailer*)tr);
  } else {
    const int C = cols / kSuperK;
    const bool in_lds = C <= kPackLdsExp;
    auto kern = fmt == 1 ? (in_lds ? quantize_pack_kernel<7, true> : quantize_pack_kernel<7, false>)
                         : (in_lds ? quantize_pack_kernel<3, true> : quantize_pack_kernel<3, false>);
    hipLaunchKernelGGL(kern, grid, block, in_lds ? (size_t)C * 256 : 0, s, (const uint16_t*)w, cols, base, rowexp, tr);
  }
  return check_launch("quantize_pack_kernel");
}

int launch_unpack(const void* packed, int rows, int cols, int fmt, void* q, void* e8, hipStream_t s) {
  const uint8_t* base = (const uint8_t*)packed;
  const int* rowexp = (const int*)(base + rowexp_offset(rows, cols, fmt));
  if (fmt == 2) {
    const long n = (long)(rows / kTileRows) * (cols / kSuperK) * 2 * 64;
    hipLaunchKernelGGL(unpack_bf4_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, base, rows, cols, rowexp,
                       (int8_t*)q, (uint8_t*)e8);
  } else {
    const long n = (long)(rows / kTileRows) * (cols / kSuperK) * kSteps * 64;
    hipLaunchKernelGGL(unpack_bfp8_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, base, rows, cols, rowexp,
                       (int8_t*)q, (uint8_t*)e8);
  }
  return check_launch("unpack kernel");
}

int launch_dequant(const void* packed, int rows, int cols, int fmt, float* out, hipStream_t s) {
  const uint8_t* base = (const uint8_t*)packed;
  if (fmt == 1) {
    const long n = (long)(rows / kTileRows) * (cols / kSuperK) * kSteps * 64;
    hipLaunchKernelGGL(dequant_bfp8_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, base, rows, cols,
                       (const int*)(base + rowexp_offset(rows, cols, 1)), out);
  } else if (fmt == 2) {
    const long n = (long)(rows / kTileRows) * (cols / kSuperK) * kSteps * 64;
    hipLaunchKernelGGL(dequant_bf4_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, base, rows, cols,
                       (const int*)(base + rowexp_offset(rows, cols, 2)), out);
  } else {
    const long n = (long)(rows / kTileRows) * (cols / kSuperK) * kSteps * 2 * 64;
    hipLaunchKernelGGL(dequant_bf16_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, base, rows, cols, out);
  }
  return check_launch("dequant kernels");
}

int launch_fill_zero(void* p, size_t bytes, hipStream_t s) {
  const size_t n16 = bytes / 16;
  if (n16) {
    unsigned blocks = (unsigned)((n16 + 255) / 256);
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(fill_zero_kernel, dim3(blocks), dim3(256), 0, s, (u32x4*)p, n16);
  }
  return check_launch("fill_zero_kernel");
}

}  // namespace qmlp
