// Fused attention prologue for Qwen3-style layers: per-head RMSNorm of q and k
// (q_norm / k_norm), rotate-half RoPE at each token's position, and the paged
// KV store of the rotated k and of v by slot -- one launch per layer, reading
// the fused QKV projection output as it is. Without norm weights (null
// pointers) the same launch serves Qwen2 / Llama layers, whose attention has
// no q / k norm (the reference applies them only when the module has them,
// nanoPD/engine/model_runner.py:101-104): RoPE of q and k as projected.
//
// Reference: per layer, paged_forward runs HF Qwen3Attention's q_norm / k_norm
// and apply_rotary_pos_emb (nanoPD/engine/model_runner.py:97-115), transposes
// and copies k / v (.contiguous(), :142-143, :191-192) and calls
// paged_kv_store (:146, :189): about a dozen elementwise launches plus the
// copies. Here one workgroup takes one token and every head row of it:
//   rows [0, H)           q heads: normalise, rotate, write q_out
//   rows [H, H + KV)      k heads: normalise, rotate, store to k_cache[slot]
//   rows [H + KV, H + 2KV) v heads: store to v_cache[slot]
// A row of D elements takes D / 16 lanes (head dims 64, 128, 256: 4, 8, 16).
// Lane j holds elements 8j .. 8j+7 and their rotate-half partners D/2 + 8j ..,
// two 16-byte loads, so RoPE needs no data exchange; the RMS statistic is a
// DPP reduction over the row's lanes. cos and sin depend on the token only:
// the workgroup computes each angle once, into LDS, and a lane keeps its eight
// in registers for every row it takes.
// Bound: HBM (each element read and written once), at few tokens the latency
// of one load -> angle -> store chain. rocprof, one workgroup per token
// against one wave per row with 2-byte accesses and a sincosf per element:
//   2048 tokens, 32 q / 8 kv heads of 128 (50 MB)          12.6 / 49.3 us
//   2647 tokens, 64 / 8 heads over an FP8 pool (92 MB)     24.1 / 100 us
//   1351 tokens, 16 / 8 heads of 256 (39 MB)               12.6 / 23.5 us
//   527 tokens, 32 / 8 heads                                6.9 / 13.4 us
// Loading the norm weights ahead with the rows (80 VGPRs) was 5-10% slower.
// RMSNorm rounds as HF Qwen3RMSNorm does (transformers modeling_qwen3):
// n = half(half(x * rsqrt(mean(x^2) + eps)) * w), with the mean in fp32.
// RoPE then rotates n in fp32 with cos / sin of pos * inv_freq[i] (inv_freq
// from the caller, fp32) and rounds once. The reference's HF
// apply_rotary_pos_emb rounds cos / sin and each product to the model dtype
// first; the fp32 rotation here is the more accurate of the two and differs
// from it by a few half-precision ulps at most.
// FP8 pools (kF8): the rotated k and the raw v, rounded to the 2-byte type as
// above, are stored as e4m3 bytes of value / scale[kv head] (the rounding of
// npd_paged_kv_store_slots_fp8, so both paths write the same bytes).
#include "common.h"

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kMaxThreads = 256;   // most threads of a workgroup (one token)

struct RopeArgs {
  uint16_t* q_out;
  void* k_cache;   // 2-byte elements, or e4m3 bytes (kF8)
  void* v_cache;
  const float* k_scale;   // kF8: per-kv-head scales
  const float* v_scale;
  const uint16_t* qkv;
  const int32_t* slots;
  const int32_t* positions;
  const float* inv_freq;
  const uint16_t* q_w;
  const uint16_t* k_w;
  int heads, kv_heads, block_size, num_blocks;
  int64_t qkv_stride, q_stride;
  float eps;
};

// Lane ^ 4 within each 8 lanes: the upper four of a bank pair read down, the
// lower four up (row_shl:4 / row_shr:4, each on its half of the banks).
__device__ __forceinline__ float xor4(float x) {
  const int v = __builtin_bit_cast(int, x);
  const int up = __builtin_amdgcn_update_dpp(0, v, 0x104, 0xF, 0x5, false);   // lane + 4
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(up, v, 0x114, 0xF, 0xA, false));
}

// Sum of eight values of each of the L lanes of a row, L in {4, 8, 16}: over
// the lanes value by value, then pairwise over the eight -- the summation tree
// of one (i, i + D/2) pair per lane and a butterfly from the farthest lane in.
template <int L>
__device__ __forceinline__ float row_sum(float (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if (L >= 16) v[i] += npd::dpp<npd::kDppRor8>(v[i]);
    if (L >= 8) v[i] += xor4(v[i]);
    v[i] += npd::dpp<npd::kDppXor2>(v[i]);
    v[i] += npd::dpp<npd::kDppXor1>(v[i]);
  }
  return ((v[0] + v[4]) + (v[2] + v[6])) + ((v[1] + v[5]) + (v[3] + v[7]));
}

// Eight consecutive elements. kVec: one 16-byte access; otherwise (pointers
// or strides off 16 bytes) one access per element.
template <bool kVec>
__device__ __forceinline__ u32x4 ld8(const uint16_t* p) {
  if constexpr (kVec) return *reinterpret_cast<const u32x4*>(p);
  u32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = (uint32_t)p[2 * i] | ((uint32_t)p[2 * i + 1] << 16);
  return v;
}
template <bool kVec>
__device__ __forceinline__ void st8(uint16_t* p, u32x4 v) {
  if constexpr (kVec) {
    *reinterpret_cast<u32x4*>(p) = v;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[2 * i] = (uint16_t)v[i];
      p[2 * i + 1] = (uint16_t)(v[i] >> 16);
    }
  }
}
// Eight elements as the e4m3 bytes of value / scale (one 8-byte access).
template <class TT, bool kVec>
__device__ __forceinline__ void st8_fp8(uint8_t* p, u32x4 v, float scale) {
  u32x2 w;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    w[i] = npd::e4m3_byte(TT::lo(v[2 * i]), scale) | (npd::e4m3_byte(TT::hi(v[2 * i]), scale) << 8) |
           (npd::e4m3_byte(TT::lo(v[2 * i + 1]), scale) << 16) |
           (npd::e4m3_byte(TT::hi(v[2 * i + 1]), scale) << 24);
  if constexpr (kVec) {
    *reinterpret_cast<u32x2*>(p) = w;
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = (uint8_t)(w[i / 4] >> (8 * (i % 4)));
  }
}

template <class TT, bool kF8, int D, bool kVec>
__global__ __launch_bounds__(kMaxThreads) void qk_norm_rope_store_kernel(RopeArgs a) {
  constexpr int HALF = D / 2;
  constexpr int L = HALF / 8;                 // lanes per row
  __shared__ __attribute__((aligned(16))) float s_cos[HALF], s_sin[HALF];
  const int tid = threadIdx.x;
  const int64_t t = blockIdx.x;
  const int i0 = (tid % L) * 8;               // this lane's first pair
  const int R = a.heads + 2 * a.kv_heads;
  const int step = blockDim.x / L;            // rows per pass (blockDim is a multiple of 64)
  const uint16_t* src = a.qkv + t * a.qkv_stride + i0;
  const bool norm = a.q_w != nullptr;

  // the first row's loads are in flight while the angles are computed
  int row = tid / L;
  u32x4 x0{}, x1{};
  if (row < R) {
    x0 = ld8<kVec>(src + (int64_t)row * D);
    x1 = ld8<kVec>(src + (int64_t)row * D + HALF);
  }
  const int slot = a.slots[t];
  const bool store = slot >= 0 && slot < a.num_blocks * a.block_size;
  const int64_t blk = store ? slot / a.block_size : 0;
  const int off = store ? slot - (int)blk * a.block_size : 0;
  const float pos = (float)a.positions[t];
  for (int i = tid; i < HALF; i += blockDim.x) {
    float s, c;
    sincosf(pos * a.inv_freq[i], &s, &c);
    s_cos[i] = c;
    s_sin[i] = s;
  }
  __syncthreads();
  float cs[8], sn[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    cs[i] = s_cos[i0 + i];
    sn[i] = s_sin[i0 + i];
  }

  while (row < R) {
    const int next = row + step;
    u32x4 nx0{}, nx1{};
    if (next < R) {   // the next row's loads run under this row's arithmetic
      nx0 = ld8<kVec>(src + (int64_t)next * D);
      nx1 = ld8<kVec>(src + (int64_t)next * D + HALF);
    }
    const bool is_q = row < a.heads, is_v = row >= a.heads + a.kv_heads;
    if (!is_v) {
      // no norm weight (Qwen2 / Llama layers): RoPE of the projection output
      // as it is. Uniform over a row's lanes, so the row reduction runs on
      // every lane it exchanges with.
      if (norm) {
        const uint16_t* w = (is_q ? a.q_w : a.k_w) + i0;
        const u32x4 w0 = ld8<kVec>(w), w1 = ld8<kVec>(w + HALF);
        float sq[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float a0 = TT::lo(x0[i]), b0 = TT::lo(x1[i]), a1 = TT::hi(x0[i]), b1 = TT::hi(x1[i]);
          sq[2 * i] = a0 * a0 + b0 * b0;
          sq[2 * i + 1] = a1 * a1 + b1 * b1;
        }
        const float r = rsqrtf(row_sum<L>(sq) * (1.f / D) + a.eps);
        auto scaled = [&](uint32_t x, uint32_t wv) {
          const uint32_t n = TT::pack2(TT::lo(x) * r, TT::hi(x) * r);
          return TT::pack2(TT::lo(n) * TT::lo(wv), TT::hi(n) * TT::hi(wv));
        };
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          x0[i] = scaled(x0[i], w0[i]);
          x1[i] = scaled(x1[i], w1[i]);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a0 = TT::lo(x0[i]), b0 = TT::lo(x1[i]), a1 = TT::hi(x0[i]), b1 = TT::hi(x1[i]);
        const float c0 = cs[2 * i], s0 = sn[2 * i], c1 = cs[2 * i + 1], s1 = sn[2 * i + 1];
        x0[i] = TT::pack2(a0 * c0 - b0 * s0, a1 * c1 - b1 * s1);
        x1[i] = TT::pack2(b0 * c0 + a0 * s0, b1 * c1 + a1 * s1);
      }
    }
    if (is_q) {
      uint16_t* dst = a.q_out + t * a.q_stride + (int64_t)row * D + i0;
      st8<kVec>(dst, x0);
      st8<kVec>(dst + HALF, x1);
    } else if (store) {
      const int kh = is_v ? row - a.heads - a.kv_heads : row - a.heads;
      const int64_t e = ((blk * a.kv_heads + kh) * a.block_size + off) * D + i0;
      void* cache = is_v ? a.v_cache : a.k_cache;
      if constexpr (kF8) {
        uint8_t* dst = static_cast<uint8_t*>(cache) + e;
        const float sc = is_v ? a.v_scale[kh] : a.k_scale[kh];
        st8_fp8<TT, kVec>(dst, x0, sc);
        st8_fp8<TT, kVec>(dst + HALF, x1, sc);
      } else {
        uint16_t* dst = static_cast<uint16_t*>(cache) + e;
        st8<kVec>(dst, x0);
        st8<kVec>(dst + HALF, x1);
      }
    }
    x0 = nx0;
    x1 = nx1;
    row = next;
  }
}

template <class TT, bool kF8, int D>
void launch_rope_d(bool vec, int threads, int64_t tokens, hipStream_t st, const RopeArgs& a) {
  const dim3 g((unsigned)tokens), b((unsigned)threads);
  if (vec)
    hipLaunchKernelGGL((qk_norm_rope_store_kernel<TT, kF8, D, true>), g, b, 0, st, a);
  else
    hipLaunchKernelGGL((qk_norm_rope_store_kernel<TT, kF8, D, false>), g, b, 0, st, a);
}

template <class TT, bool kF8>
void launch_rope(int64_t head_dim, bool vec, int threads, int64_t tokens, hipStream_t st,
                 const RopeArgs& a) {
  switch (head_dim) {
    case 64: launch_rope_d<TT, kF8, 64>(vec, threads, tokens, st, a); break;
    case 128: launch_rope_d<TT, kF8, 128>(vec, threads, tokens, st, a); break;
    default: launch_rope_d<TT, kF8, 256>(vec, threads, tokens, st, a); break;
  }
}

}  // namespace

namespace {

// Shared by the 2-byte and the FP8 entry points (k_scale / v_scale null for
// 2-byte pools).
int rope_impl(void* q_out, void* k_cache, void* v_cache, const void* qkv,
              const int32_t* slot_mapping, const int32_t* positions, const float* inv_freq,
              const void* q_norm_weight, const void* k_norm_weight, const float* k_scale,
              const float* v_scale, int64_t num_tokens, int64_t num_heads, int64_t num_kv_heads,
              int64_t head_dim, int64_t num_blocks, int64_t block_size, int64_t qkv_stride_token,
              int64_t q_stride_token, float eps, int32_t dtype, void* stream, bool fp8,
              const char* name) {
  using namespace npd;
  if (dtype != NPD_DTYPE_F16 && dtype != NPD_DTYPE_BF16)
    return fail(NPD_E_DTYPE, "%s: unsupported dtype code %d (fp16/bf16 only)", name, dtype);
  if (head_dim != 64 && head_dim != 128 && head_dim != 256)
    return fail(NPD_E_INVALID, "%s: head_dim %lld not in {64, 128, 256}", name,
                (long long)head_dim);
  if (num_tokens < 0 || num_heads <= 0 || num_kv_heads <= 0 || num_blocks <= 0 || block_size <= 0)
    return fail(NPD_E_INVALID, "%s: bad sizes", name);
  if (num_blocks * block_size > INT32_MAX)
    return fail(NPD_E_INVALID, "%s: pool exceeds int32 slot indexing", name);
  if (qkv_stride_token < (num_heads + 2 * num_kv_heads) * head_dim || q_stride_token < num_heads * head_dim)
    return fail(NPD_E_INVALID, "%s: token strides shorter than a token's heads", name);
  if (!(eps >= 0.f))
    return fail(NPD_E_INVALID, "%s: eps must be non-negative", name);
  if (num_tokens == 0) return NPD_OK;
  if (!q_out || !k_cache || !v_cache || !qkv || !slot_mapping || !positions || !inv_freq ||
      (fp8 && (!k_scale || !v_scale)))
    return fail(NPD_E_INVALID, "%s: null pointer", name);
  if ((q_norm_weight == nullptr) != (k_norm_weight == nullptr))
    return fail(NPD_E_INVALID, "%s: pass both norm weights (Qwen3) or neither (Qwen2 / Llama)",
                name);
  const int64_t rows = num_tokens * (num_heads + 2 * num_kv_heads);
  if (rows / 4 > INT32_MAX) return fail(NPD_E_INVALID, "%s: too many rows", name);
  // a workgroup per token, its threads cut so that the passes over the token's
  // rows are as full as whole waves allow (48 rows of 8 lanes: 2 x 192)
  const int64_t lanes = (num_heads + 2 * num_kv_heads) * (head_dim / 16);
  const int64_t passes = (lanes + kMaxThreads - 1) / kMaxThreads;
  const int threads = (int)(((lanes + passes - 1) / passes + 63) / 64 * 64);
  // 16-byte accesses where every row starts on 16 bytes (FP8 cache rows: 8)
  auto on16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  const bool vec = on16(q_out) && on16(k_cache) && on16(v_cache) && on16(qkv) &&
                   on16(q_norm_weight) && on16(k_norm_weight) && qkv_stride_token % 8 == 0 &&
                   q_stride_token % 8 == 0;
  RopeArgs a;
  a.q_out = static_cast<uint16_t*>(q_out);
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.k_scale = k_scale;
  a.v_scale = v_scale;
  a.qkv = static_cast<const uint16_t*>(qkv);
  a.slots = slot_mapping;
  a.positions = positions;
  a.inv_freq = inv_freq;
  a.q_w = static_cast<const uint16_t*>(q_norm_weight);
  a.k_w = static_cast<const uint16_t*>(k_norm_weight);
  a.heads = (int)num_heads;
  a.kv_heads = (int)num_kv_heads;
  a.block_size = (int)block_size;
  a.num_blocks = (int)num_blocks;
  a.qkv_stride = qkv_stride_token;
  a.q_stride = q_stride_token;
  a.eps = eps;
  hipStream_t st = as_stream(stream);
  if (dtype == NPD_DTYPE_BF16) {
    if (fp8) launch_rope<BF16, true>(head_dim, vec, threads, num_tokens, st, a);
    else launch_rope<BF16, false>(head_dim, vec, threads, num_tokens, st, a);
  } else {
    if (fp8) launch_rope<F16, true>(head_dim, vec, threads, num_tokens, st, a);
    else launch_rope<F16, false>(head_dim, vec, threads, num_tokens, st, a);
  }
  return check_launch(name);
}

}  // namespace

extern "C" int npd_qk_norm_rope_store(void* q_out, void* k_cache, void* v_cache, const void* qkv,
                                      const int32_t* slot_mapping, const int32_t* positions,
                                      const float* inv_freq, const void* q_norm_weight,
                                      const void* k_norm_weight, int64_t num_tokens,
                                      int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
                                      int64_t num_blocks, int64_t block_size,
                                      int64_t qkv_stride_token, int64_t q_stride_token, float eps,
                                      int32_t dtype, void* stream) {
  return rope_impl(q_out, k_cache, v_cache, qkv, slot_mapping, positions, inv_freq, q_norm_weight,
                   k_norm_weight, nullptr, nullptr, num_tokens, num_heads, num_kv_heads, head_dim,
                   num_blocks, block_size, qkv_stride_token, q_stride_token, eps, dtype, stream,
                   false, "npd_qk_norm_rope_store");
}

extern "C" int npd_qk_norm_rope_store_fp8(void* q_out, void* k_cache, void* v_cache,
                                          const void* qkv, const int32_t* slot_mapping,
                                          const int32_t* positions, const float* inv_freq,
                                          const void* q_norm_weight, const void* k_norm_weight,
                                          const float* k_scale, const float* v_scale,
                                          int64_t num_tokens, int64_t num_heads,
                                          int64_t num_kv_heads, int64_t head_dim,
                                          int64_t num_blocks, int64_t block_size,
                                          int64_t qkv_stride_token, int64_t q_stride_token,
                                          float eps, int32_t dtype, void* stream) {
  return rope_impl(q_out, k_cache, v_cache, qkv, slot_mapping, positions, inv_freq, q_norm_weight,
                   k_norm_weight, k_scale, v_scale, num_tokens, num_heads, num_kv_heads, head_dim,
                   num_blocks, block_size, qkv_stride_token, q_stride_token, eps, dtype, stream,
                   true, "npd_qk_norm_rope_store_fp8");
}
