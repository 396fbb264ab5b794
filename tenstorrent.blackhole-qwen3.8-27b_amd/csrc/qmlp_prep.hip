// qmlp_prep.hip -- the activation pass that runs before the projection kernels: the RMSNorm, the
// fp16 conversion with per-token scales of the many-token block-float path, or both.
#include "qmlp_common.h"
#include "qmlp_internal.h"

namespace qmlp {

// ---------------------------------------------------------------- one pass over the token rows
//
// CONV (block-float weights, many tokens): x bf16 -> x16 = fp16(x * 2^tx[m]) with a per-token power
// of two that puts max|x[m]| in [2^14, 2^15), and th[m] from the Cauchy-Schwarz bound
// |h| <= |x_m|^2 max|Wg_n| max|Wu_n| (row norms from the packed trailers) so that h * 2^th[m] fits
// fp16.  NORM: the decoder's ffn_norm first, n = bf16(x * (1 / sqrt(mean(x^2) + eps)) * (1 + w))
// (docker/qwen-c2-graft/graft/layer.py:110-112,228-237, add_unit_offset); without CONV n itself is
// the output.  Norm and conversion share one launch and one read of x.
//
// Bound by latency: a row's load, one or two block reductions and its store.  One block of 256
// threads per row, so that a few dozen rows still spread over the chip and every load of a row is
// in flight at once (rows of up to 8192 values stay in registers; longer ones are re-read from
// L2).  One wave per row, four rows per block, took 5.2-5.9 us at 64-201 rows for the conversion
// and 14 us for the norm, whose loop over the row kept one load in flight.  Reductions run in a
// fixed order (deterministic).
constexpr int kRowThreads = 256;
constexpr int kRowRegCh = 4;  // 16-byte chunks per thread held in registers

template <typename T, typename F>
__device__ __forceinline__ T row_reduce(T v, T* lds, F&& op) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = op(v, __shfl_xor(v, o));
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  return op(op(lds[0], lds[1]), op(lds[2], lds[3]));
}

__device__ __forceinline__ float lo_f32(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi_f32(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

template <bool NORM, bool CONV, bool REGS>
__global__ __launch_bounds__(kRowThreads) void rows_kernel(const uint16_t* __restrict__ x,
                                                          const uint16_t* __restrict__ w, float eps, int H,
                                                          const Trailer* tg, const Trailer* tu,
                                                          uint16_t* __restrict__ out, int* __restrict__ tx,
                                                          int* __restrict__ th) {
  __shared__ float s_norm[4], s_max[4];
  __shared__ double s_sum[4];
  const int m = blockIdx.x, nch = H / 8, tid = threadIdx.x;
  const u32x4* xr = (const u32x4*)(x + (size_t)m * H);
  const u32x4* wr = (const u32x4*)w;
  u32x4* orow = (u32x4*)(out + (size_t)m * H);
  u32x4 v[REGS ? kRowRegCh : 1];
  u32x4 g[REGS && NORM ? kRowRegCh : 1];
  if constexpr (REGS) {
#pragma unroll
    for (int i = 0; i < kRowRegCh; ++i) {
      const int c = min(tid + i * kRowThreads, nch - 1);
      v[i] = xr[c];
      if constexpr (NORM) g[i] = wr[c];
    }
  }
  // f(chunk index, value, norm weight) over the thread's chunks
  auto each = [&](auto&& f) {
    if constexpr (REGS) {
#pragma unroll
      for (int i = 0; i < kRowRegCh; ++i)
        if (tid + i * kRowThreads < nch) f(tid + i * kRowThreads, v[i], g[NORM ? i : 0]);
    } else {
      for (int c = tid; c < nch; c += kRowThreads) {
        u32x4 t = xr[c], u = NORM ? wr[c] : u32x4{0u, 0u, 0u, 0u};
        f(c, t, u);
      }
    }
  };
  float rs = 1.f;
  auto normed = [&](u32x4 t, u32x4 u) {
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = (uint32_t)f32_to_bf16(lo_f32(t[i]) * rs * (1.0f + lo_f32(u[i]))) |
             ((uint32_t)f32_to_bf16(hi_f32(t[i]) * rs * (1.0f + hi_f32(u[i]))) << 16);
    return o;
  };
  if constexpr (NORM) {
    float ss = 0.f;
    each([&](int, u32x4& t, u32x4&) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ss = fmaf(lo_f32(t[i]), lo_f32(t[i]), ss);
        ss = fmaf(hi_f32(t[i]), hi_f32(t[i]), ss);
      }
    });
    ss = row_reduce(ss, s_norm, [](float a, float b) { return a + b; });
    rs = 1.0f / sqrtf(ss / (float)H + eps);
    if constexpr (!CONV) {
      each([&](int c, u32x4& t, u32x4& u) { orow[c] = normed(t, u); });
      return;
    }
    if constexpr (REGS) each([&](int, u32x4& t, u32x4& u) { t = normed(t, u); });
  }
  if constexpr (CONV) {
    float mx = 0.f;
    double ss = 0.0;
    auto value = [&](const u32x4& t, const u32x4& u) {
      if constexpr (NORM && !REGS) return normed(t, u);
      return t;
    };
    each([&](int, u32x4& t, u32x4& u) {
      const u32x4 n = value(t, u);
      float cs = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        mx = fmaxf(mx, fmaxf(fabsf(lo_f32(n[i])), fabsf(hi_f32(n[i]))));
        cs = fmaf(lo_f32(n[i]), lo_f32(n[i]), cs);
        cs = fmaf(hi_f32(n[i]), hi_f32(n[i]), cs);
      }
      ss += (double)cs;
    });
    // both reductions behind one barrier
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      mx = fmaxf(mx, __shfl_xor(mx, o));
      ss += __shfl_xor(ss, o);
    }
    if ((tid & 63) == 0) {
      s_max[tid >> 6] = mx;
      s_sum[tid >> 6] = ss;
    }
    __syncthreads();
    mx = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
    ss = (s_sum[0] + s_sum[1]) + (s_sum[2] + s_sum[3]);
    int e = 0;
    if (mx > 0.f) frexpf(mx, &e);
    const int txm = mx > 0.f ? 15 - e : 0;
    if (tid == 0) {
      const double gn = __longlong_as_double((long long)tg->max_row_norm_bits);
      const double un = __longlong_as_double((long long)tu->max_row_norm_bits);
      const double bound = ss * gn * un * (1.0 + 1.0 / 64.0);
      int eb = 0;
      if (bound > 0.0) frexp(bound, &eb);
      tx[m] = txm;
      th[m] = bound > 0.0 ? 15 - eb : 0;
    }
    each([&](int c, u32x4& t, u32x4& u) {
      const u32x4 n = value(t, u);
      u32x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        o[i] = (uint32_t)f32_to_f16_bits(__builtin_amdgcn_ldexpf(lo_f32(n[i]), txm)) |
               ((uint32_t)f32_to_f16_bits(__builtin_amdgcn_ldexpf(hi_f32(n[i]), txm)) << 16);
      orow[c] = o;
    });
  }
}

template <bool NORM, bool CONV>
static int launch_rows(const void* x, const void* w, float eps, int M, int H, const Trailer* tg, const Trailer* tu,
                       void* out, int* tx, int* th, hipStream_t s) {
  auto kern = H <= 8 * kRowThreads * kRowRegCh ? rows_kernel<NORM, CONV, true> : rows_kernel<NORM, CONV, false>;
  hipLaunchKernelGGL(kern, dim3(M), dim3(kRowThreads), 0, s, (const uint16_t*)x, (const uint16_t*)w, eps, H, tg, tu,
                     (uint16_t*)out, tx, th);
  return check_launch("rows_kernel");
}

int launch_rmsnorm(const void* x, const void* w, float eps, int M, int H, void* xn, hipStream_t s) {
  return launch_rows<true, false>(x, w, eps, M, H, nullptr, nullptr, xn, nullptr, nullptr, s);
}

int launch_prep(const ForwardArgs& a, hipStream_t s) {
  const WsLayout L = ws_layout(a.M, a.H, a.I, a.fmt);
  const Trailer* tg = (const Trailer*)(a.wg + trailer_offset(a.I, a.H, a.fmt));
  const Trailer* tu = (const Trailer*)(a.wu + trailer_offset(a.I, a.H, a.fmt));
  uint8_t* x16 = a.ws + L.x16;
  int *tx = (int*)(a.ws + L.tx), *th = (int*)(a.ws + L.th);
  return a.normw ? launch_rows<true, true>(a.x, a.normw, a.eps, a.M, a.H, tg, tu, x16, tx, th, s)
                 : launch_rows<false, true>(a.x, nullptr, 0.f, a.M, a.H, tg, tu, x16, tx, th, s);
}

}  // namespace qmlp
