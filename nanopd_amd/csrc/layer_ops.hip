// The elementwise passes of a decoder layer around its GEMMs: residual add +
// RMSNorm, and the SwiGLU product. The reference leaves them to Hugging Face
// modules (nanoPD/engine/model_runner.py:8-13 wraps the whole model). As
// separate tensor operations they re-read and re-write every activation. 527
// tokens of 4096 columns (12288 in the MLP), rocprof: add 5.1 + norm 7.2 us
// against 5.8 here; silu 11.2 + product 9.6 against 7.5.
//
// Both are bound by HBM / L2 bytes at many tokens and by one load -> store
// latency at few. Every element is read and written once, in 16-byte accesses.
#include "common.h"

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int kThreads = 256;

// One workgroup per row of E = 8 * chunks elements; a thread holds its NCH
// chunks tid + 256 e in registers between the statistic and the output.
// kAdd: x becomes half(x + delta) first (stored back), as a separate addition
// would round it; the norm reads the rounded sum. y = half(x * rstd * w) with
// the mean square in fp32, rounded once.
template <class TT, int NCH, bool kAdd>
__global__ __launch_bounds__(kThreads) void rms_norm_kernel(u32x4* __restrict__ out,
                                                            u32x4* x, const u32x4* __restrict__ delta,
                                                            const u32x4* __restrict__ w, int chunks,
                                                            float inv_e, float eps) {
  __shared__ float s_sum[kThreads / 64];
  const int tid = threadIdx.x;
  const int64_t row = (int64_t)blockIdx.x * chunks;
  u32x4 v[NCH], wv[NCH];
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < NCH; ++e) {
    const int c = tid + kThreads * e;
    v[e] = u32x4{0, 0, 0, 0};
    if (c < chunks) {
      v[e] = x[row + c];
      wv[e] = w[c];
      if (kAdd) {
        const u32x4 d = delta[row + c];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          v[e][i] = TT::pack2(TT::lo(v[e][i]) + TT::lo(d[i]), TT::hi(v[e][i]) + TT::hi(d[i]));
        x[row + c] = v[e];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ss = fmaf(TT::lo(v[e][i]), TT::lo(v[e][i]), ss);
      ss = fmaf(TT::hi(v[e][i]), TT::hi(v[e][i]), ss);
    }
  }
  ss = npd::wave_sum_f(ss);
  if ((tid & 63) == 0) s_sum[tid >> 6] = ss;
  __syncthreads();
  const float r = rsqrtf(((s_sum[0] + s_sum[1]) + (s_sum[2] + s_sum[3])) * inv_e + eps);
#pragma unroll
  for (int e = 0; e < NCH; ++e) {
    const int c = tid + kThreads * e;
    if (c >= chunks) continue;
    u32x4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      y[i] = TT::pack2(TT::lo(v[e][i]) * r * TT::lo(wv[e][i]), TT::hi(v[e][i]) * r * TT::hi(wv[e][i]));
    out[row + c] = y;
  }
}

// out[t, i] = silu(gate) * up over rows [gate (I) | up (I)] of gu; silu is
// rounded to the dtype before the product, as the separate operations round it
// (a layer's output then differs from theirs by the last bit of a few values
// only). A thread takes 8 elements of a row.
template <class TT>
__global__ __launch_bounds__(kThreads) void silu_mul_kernel(u32x4* __restrict__ out,
                                                            const u32x4* __restrict__ gu,
                                                            int64_t total, int chunks) {
  const int64_t at = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (at >= total) return;
  const int64_t row = at / chunks;
  const int64_t src = at + row * chunks;   // row * 2 * chunks + column
  const u32x4 g = gu[src], u = gu[src + chunks];
  auto silu = [](float x) {
    // x / (1 + e^-x): 0 at -inf's side (e^-x overflows to inf), x at +inf's. Of
    // a quarter of the divisor, whose reciprocal is a normal number: below -87.3
    // that of the divisor itself is not, and v_rcp_f32 would make it 0.
    const float e = __builtin_amdgcn_exp2f(x * -1.4426950408889634f);
    return x * 0.25f * __builtin_amdgcn_rcpf(fmaf(e, 0.25f, 0.25f));
  };
  u32x4 y;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t s = TT::pack2(silu(TT::lo(g[i])), silu(TT::hi(g[i])));
    y[i] = TT::pack2(TT::lo(s) * TT::lo(u[i]), TT::hi(s) * TT::hi(u[i]));
  }
  out[at] = y;
}

template <class TT, bool kAdd>
void launch_norm(void* out, void* x, const void* delta, const void* w, int64_t rows, int chunks,
                 float eps, hipStream_t st) {
  const dim3 g((unsigned)rows), b(kThreads);
  auto* o = static_cast<u32x4*>(out);
  auto* xp = static_cast<u32x4*>(x);
  auto* dp = static_cast<const u32x4*>(delta);
  auto* wp = static_cast<const u32x4*>(w);
  const float inv = 1.f / (8.f * (float)chunks);
  if (chunks <= kThreads)
    hipLaunchKernelGGL((rms_norm_kernel<TT, 1, kAdd>), g, b, 0, st, o, xp, dp, wp, chunks, inv, eps);
  else if (chunks <= 2 * kThreads)
    hipLaunchKernelGGL((rms_norm_kernel<TT, 2, kAdd>), g, b, 0, st, o, xp, dp, wp, chunks, inv, eps);
  else
    hipLaunchKernelGGL((rms_norm_kernel<TT, 4, kAdd>), g, b, 0, st, o, xp, dp, wp, chunks, inv, eps);
}

}  // namespace

extern "C" int npd_add_rms_norm(void* out, void* x, const void* delta, const void* weight,
                                int64_t rows, int64_t width, float eps, int32_t dtype,
                                void* stream) {
  using namespace npd;
  const char* name = "npd_add_rms_norm";
  if (dtype != NPD_DTYPE_F16 && dtype != NPD_DTYPE_BF16)
    return fail(NPD_E_DTYPE, "%s: unsupported dtype code %d (fp16/bf16 only)", name, dtype);
  if (rows < 0 || rows > INT32_MAX || width <= 0 || width % 8 != 0 || width > 8192)
    return fail(NPD_E_INVALID, "%s: %lld rows of %lld (a multiple of 8 up to 8192 wanted)", name,
                (long long)rows, (long long)width);
  if (!(eps >= 0.f)) return fail(NPD_E_INVALID, "%s: eps must be non-negative", name);
  if (rows == 0) return NPD_OK;
  if (!out || !x || !weight) return fail(NPD_E_INVALID, "%s: null pointer", name);
  if (!aligned16(out) || !aligned16(x) || !aligned16(weight) || !aligned16(delta))
    return fail(NPD_E_ALIGN, "%s: pointers must be 16-byte aligned", name);
  hipStream_t st = as_stream(stream);
  const int chunks = (int)(width / 8);
  if (dtype == NPD_DTYPE_BF16) {
    if (delta) launch_norm<BF16, true>(out, x, delta, weight, rows, chunks, eps, st);
    else launch_norm<BF16, false>(out, x, delta, weight, rows, chunks, eps, st);
  } else {
    if (delta) launch_norm<F16, true>(out, x, delta, weight, rows, chunks, eps, st);
    else launch_norm<F16, false>(out, x, delta, weight, rows, chunks, eps, st);
  }
  return check_launch(name);
}

extern "C" int npd_silu_mul(void* out, const void* gate_up, int64_t rows, int64_t width,
                            int32_t dtype, void* stream) {
  using namespace npd;
  const char* name = "npd_silu_mul";
  if (dtype != NPD_DTYPE_F16 && dtype != NPD_DTYPE_BF16)
    return fail(NPD_E_DTYPE, "%s: unsupported dtype code %d (fp16/bf16 only)", name, dtype);
  if (rows < 0 || width <= 0 || width % 8 != 0 || width > INT32_MAX)
    return fail(NPD_E_INVALID, "%s: %lld rows of %lld (a multiple of 8 wanted)", name,
                (long long)rows, (long long)width);
  if (rows == 0) return NPD_OK;
  if (!out || !gate_up) return fail(NPD_E_INVALID, "%s: null pointer", name);
  if (!aligned16(out) || !aligned16(gate_up))
    return fail(NPD_E_ALIGN, "%s: pointers must be 16-byte aligned", name);
  const int64_t chunks = width / 8;
  if (rows > INT64_MAX / chunks || (rows * chunks + kThreads - 1) / kThreads > INT32_MAX)
    return fail(NPD_E_INVALID, "%s: too many elements", name);
  const int64_t total = rows * chunks;
  const dim3 g((unsigned)((total + kThreads - 1) / kThreads)), b(kThreads);
  hipStream_t st = as_stream(stream);
  auto* o = static_cast<u32x4*>(out);
  auto* s = static_cast<const u32x4*>(gate_up);
  if (dtype == NPD_DTYPE_BF16)
    hipLaunchKernelGGL((silu_mul_kernel<BF16>), g, b, 0, st, o, s, total, (int)chunks);
  else
    hipLaunchKernelGGL((silu_mul_kernel<F16>), g, b, 0, st, o, s, total, (int)chunks);
  return check_launch(name);
}
