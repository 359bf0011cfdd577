// Chunked-prefill attention over a paged prefix plus the new chunk (MFMA).
//
// Reference: the prefill branch of ModelRunner.paged_forward
// (nanoPD/engine/model_runner.py:152-168) runs F.scaled_dot_product_attention
// over the chunk's own K/V with a block-diagonal causal mask and never reads
// the prefix already in the pool. This op computes what that code means for a
// chunk on a prefix: query row i of sequence s, at position
// p = context_lens[s] - q_len + i, attends causally to keys 0..p of the paged
// cache (the chunk's K/V are stored before the call, as the reference stores
// them before attending, model_runner.py:146). For an empty prefix both agree.
//
// MI355X design (gfx950, v_mfma_f32_32x32x16_{bf16,f16}, wave64):
//   head dim D = 64, 128 or 256 (prefill_kernel<.., D, ..>; the other multiples
//   of 32 up to 224, and 256 over an FP8 pool, run prefill_generic_kernel below);
//   workgroup = 8 waves = one (sequence, kv-head, tile of 256 rows, key part)
//   -- 4 waves and 128 rows, without the half-step shift below, at head dim 256
//   (no key parts) and for few tiles at 128.
//   Rows are (token, head) pairs of the kv head's G query heads, flattened as
//   token * G + head: any G fills its tiles, and a wave's 32 rows span 32 / G
//   tokens, so its causal range ends with the tile's. With 8 waves, two share a
//   SIMD, 256 VGPRs each. All waves read the 64-key K/V tiles that the workgroup
//   gathers from the pool into LDS (GQA and row reuse).
//   per step of 64 keys, each wave:
//     S^T = K . Q^T   -- A = K rows from LDS, B = the wave's query rows, kept
//                        in registers for the whole key loop;
//     softmax          -- lane l holds 32 keys of query row l % 32, lane l ^ 32
//                        the others. Scale and reference are one FMA before
//                        exp2; the row sum is a v_dot2 of the rounded P pair
//                        with (1, 1). No maximum is taken in the usual step:
//                        whether the reference must move is read off the packed
//                        P values or their sum (Bound), and only then the
//                        maxima are taken, O rescaled and P formed again (head
//                        dim 256: the maximum of every step, kExactMax);
//     O^T += V^T . P^T -- P^T is the S^T accumulator, already in B-operand
//                        layout (packed with v_cvt_pk_bf16_f32); V stays
//                        row-major in LDS like K, and the V^T A operand is two
//                        ds_read_b64_tr_b16 (gfx950 transposing LDS read: in a
//                        group of 16 lanes, lane j receives element j%4 of the
//                        8-byte chunks addressed by lanes 4e + j/4, e = 0..3).
//   K/V tiles load straight into LDS (global_load_lds, 16 bytes per lane),
//   three steps ahead, with a swizzle in place of padded rows: no ring
//   registers, no LDS stores. The two waves of a SIMD run half a step apart:
//   one's MFMAs with the other's softmax. Keys past the visible range are
//   clamped to the last visible key (a real, finite context row) and masked.
//   Operand layouts of v_mfma_f32_32x32x16 (checked on the hardware):
//     A[m = lane%32][k = 8*(lane/32) + e], B[k = 8*(lane/32) + e][n = lane%32],
//     D[m = 8*(i/4) + 4*(lane/32) + i%4][n = lane%32].
//
// What bounds it: power, then issue. 12000 tokens of 32 / 8 heads run at 3009
// cycles per step against 2048 of MFMA, at 1.8 GHz (all-zero inputs, which draw
// less, hold 2.4 GHz and take 0.76x the time): 1027 to 1122 us over several
// boxes = 1.05 to 1.15 PFLOP/s of useful work, where a plain 8192^3 product
// reaches 1.47. Before (16x16x32 MFMAs, K/V through a register ring, maxima in
// every step): 1328 to 1383 us. A step without the tile loads takes the same
// cycles at a higher clock; more operand reads ahead (6 to 12) change nothing;
// the dot2 row sums cost 11 cycles each under the other wave's MFMAs, 4 alone.
//
// Key splits: tiles are cut into nsp <= splits_max near-equal key parts run by
// separate workgroups where that shortens the launch (prefill_item; in the
// fixed order of very many tiles at ks_steps). Each part publishes its
// unnormalised O, exponent reference and row sum with device-coherent stores,
// then takes a ticket from a per-tile counter; the last of the nsp to arrive
// merges the others into its registers
//   M = max_j m_j,  L = sum_j l_j 2^(m_j - M),  O = sum_j O_j 2^(m_j - M) / L
// writes the output and resets the counter to 0.
#include <type_traits>

#include "common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kWaveRows = 32;    // flattened (token, head) rows per wave
constexpr int tile_rows(int nw) { return nw * kWaveRows; }   // ... and per workgroup of nw waves
constexpr int kKT = 64;          // keys per step
constexpr int kBufK = 4;         // K tiles in LDS
constexpr int kBufV = 5;         // V tiles in LDS
constexpr int kListBlocks = 2048;     // blocks of the key range listed in LDS at a time (8 KB)
constexpr int kMaxTableBlocks = 16384;  // widest block table accepted
constexpr int kSchedMfma = 0x8, kSchedDsRead = 0x100;   // sched_group_barrier classes
constexpr int kWaitVm0 = 0x0f70;       // s_waitcnt vmcnt(0), the other counters free
constexpr float kNoRef = 3.402823466e38f;     // exponent offset of a row without a reference
constexpr int kSplitSteps = 16;       // a key range longer than this many steps is split
constexpr int kMaxSplits = 8;
constexpr int kFixedSplits = 4;       // parts in the fixed order of a full launch
constexpr int kAhead = 4;             // LDS operand reads ahead of their MFMA
constexpr int kSlots = 8;             // tiles per lane of the work list
constexpr int kListTiles = 64 * kSlots;
constexpr int kSmallDiv = 1 << 21;    // dividends small_div takes for any divisor
constexpr int kMinPart = 4;           // shortest part the work list cuts (steps)
constexpr int kItemSteps = 4;         // an item's prologue and output, in steps
constexpr int kMergeSteps = 4;        // publishing and merging a part, in steps
constexpr float kLog2e = 1.4426950408889634f;
// partial record of one wave (32 rows, one split) at head dim d, floats:
// [db*8 + i/2][lane][2] over the O^T accumulators, db < d / 32
constexpr int rec_o(int d) { return d / 8 * 2 * 64 * 2; }
constexpr int kRecML = 2 * 64 * 2;       // [lane][m, l] (half of it used)

struct PrefillArgs {
  uint16_t* out;
  const uint16_t* q;
  const u32x4* k_cache;
  const u32x4* v_cache;
  const int32_t* block_tables;
  const int32_t* cu_seqlens_q;
  const int32_t* context_lens;
  int* counters;
  float* part_o;
  float* part_ml;
  const float* k_scale;   // FP8 pools: per-kv-head scales (element = e4m3 byte * scale)
  const float* v_scale;
  int num_seqs, num_kv_heads, group, block_size, bs_shift, num_blocks, max_bps;
  int tiles_max, subtiles, splits_max;   // subtiles: 32-row subtiles per (sequence, kv head)
  int ks_steps;                          // key steps per split (fixed order)
  bool list;                             // items by the work list (else in the fixed order)
  int max_items;                         // items per kv head the grid has room for
  int even_items;                        // ... to be used where no tile outlasts the mean load
  int num_cus;                           // compute units of the device (work-list sizing)
  float scale_log2;
  int64_t q_stride_token, q_stride_head, out_stride_token, out_stride_head;
};

template <class TT>
struct Mfma;
template <>
struct Mfma<npd::BF16> {
  typedef bf16x8 V8;
  static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(V8, a),
                                                   __builtin_bit_cast(V8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x16 mma32(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(V8, a),
                                                 __builtin_bit_cast(V8, b), c, 0, 0, 0);
  }
};
template <>
struct Mfma<npd::F16> {
  typedef f16x8 V8;
  static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(V8, a),
                                                  __builtin_bit_cast(V8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x16 mma32(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(V8, a),
                                                 __builtin_bit_cast(V8, b), c, 0, 0, 0);
  }
};

// When a row's reference moves (head dims 64 and 128). bf16: the reference sits kBias above the
// maximum it was taken from, P is <= 2^-7 then, and a P of 2 or more (bit 14 of
// any packed half; also inf and NaN) asks for a new one: one v_or3 per two
// pairs. fp16 keeps its reference at the maximum (a bias would cost small P
// their bits) and asks where a lane's P of the step, which are summed anyway,
// come to kPast = 2^8: one compare, and every P is below 2^8 where none asks.
// (A packed integer maximum over the 16 registers instead: 291 against 266 us
// for three chunks of 300-1000 tokens of 64 / 8 heads on prefixes to 4096, FP8
// pool.) The lane's up to 32 P of such a step have one of 2^3 or more, so that
// its row moves (kMove). Either way P stays exact enough between moves: fp32
// sums, relative rounding of the pair.
template <class TT>
struct Bound;
template <>
struct Bound<npd::BF16> {
  static constexpr float kBias = 7.f, kMove = 0.f, kPast = 0.f;
};
template <>
struct Bound<npd::F16> {
  static constexpr float kBias = 0.f, kMove = 2.f, kPast = 256.f;
};
// bf16: any P of 2 or more
template <int KB>
__device__ __forceinline__ bool past_two(const u32x4 (&pb)[KB]) {
  uint32_t o = 0;
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    o = o | pb[kb][0] | pb[kb][1];
    o = o | pb[kb][2] | pb[kb][3];
  }
  return (o & 0x40004000u) != 0;
}

// Max / sum over the 4 key groups of a query row (lanes l, l^16, l^32, l^48).
using npd::row_max4;
using npd::row_sum4;

typedef short s16x4 __attribute__((ext_vector_type(4)));
// ds_read_b64_tr_b16 on an LDS address given as a generic pointer to __shared__
__device__ __forceinline__ u32x2 lds_read_tr(const uint16_t* p) {
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p)));
}

// x / d for 0 <= x < 2^31, d > 0 and quotients below 2^21: the fp32 estimate
// is off by at most one. A handful of instructions against some 35 of the
// integer division.
__device__ __forceinline__ int small_div(int x, int d) {
  int q = (int)((float)x * __builtin_amdgcn_rcpf((float)d));
  const int r = x - q * d;
  return q + (r >= d ? 1 : 0) - (r < 0 ? 1 : 0);
}

// The work item of this workgroup, derived by its first wave: the sequence s,
// its tile t of TR flattened (token, head) rows, key part j of nsp, kv
// head kh, the sequence's first query row, chunk length and context, the
// tile's keys 0 .. nkeys - 1 and the part's steps st0 .. st1 - 1. false: no
// item, the workgroup exits.
struct Item {
  int s, t, j, nsp, kh, q0, qlen, ctx, nkeys, st0, st1;
};
// one past the last position that tile t of a chunk sees
template <int TR>
__device__ __forceinline__ int tile_keys(const PrefillArgs& a, int t, int qlen, int ctx) {
  const int fr = qlen * a.group, fe = (t + 1) * TR;
  const int last = fe >= fr ? qlen - 1   // position in the chunk of the tile's last row
                            : (fe < kSmallDiv ? small_div(fe - 1, a.group) : (fe - 1) / a.group);
  const int nk = ctx - qlen + last + 1;
  return nk < 0 ? 0 : nk;
}
template <int TR, int KT>
__device__ __forceinline__ bool prefill_item(const PrefillArgs& a, int lane, Item& it) {
  int s, t, j, kh, nsp, nsteps, q0, qlen, ctx;
  const int cap = a.max_bps * a.block_size;
  const int per_item = a.num_kv_heads;   // workgroups per (sequence, tile, part)
  const int tiles = a.num_seqs * a.tiles_max;
  if (a.list) {
    // Work list in longest-processing-time order, derived from the sequence
    // lengths. Slot (k, lane) stands for tile index i = 64 k +
    // lane: sequence i / tiles_max, tile i % tiles_max, n key steps. The
    // kv-head is the fastest-varying index and every count is a multiple of
    // the kv-head count, so with 8 kv-heads each XCD (workgroups go to XCDs
    // round-robin by blockIdx) serves one kv-head and its K/V stays in that
    // XCD's L2.
    int n[kSlots], c0[kSlots], ql[kSlots], cx[kSlots];
    bool valid[kSlots];
#pragma unroll
    for (int k = 0; k < kSlots; ++k) {
      valid[k] = 64 * k + lane < tiles;
      n[k] = c0[k] = ql[k] = cx[k] = 0;
      if (64 * k < tiles && valid[k]) {
        const int ls = small_div(64 * k + lane, a.tiles_max);
        c0[k] = a.cu_seqlens_q[ls];
        ql[k] = a.cu_seqlens_q[ls + 1];
        cx[k] = a.context_lens[ls];
      }
    }
    int tot = 0, nmax = 0, ntiles = 0;
#pragma unroll
    for (int k = 0; k < kSlots; ++k)
      if (64 * k < tiles) {
        const int lt = 64 * k + lane - small_div(64 * k + lane, a.tiles_max) * a.tiles_max;
        ql[k] -= c0[k];
        cx[k] = cx[k] < 0 ? 0 : (cx[k] < cap ? cx[k] : cap);
        valid[k] = valid[k] && lt * TR < ql[k] * a.group;
        if (valid[k]) n[k] = (tile_keys<TR>(a, lt, ql[k], cx[k]) + KT - 1) / KT;
        tot += n[k];
        nmax = max(nmax, n[k]);
        ntiles += __popcll(__ballot(valid[k]));
      }
    // a lane adds up its slots before the wave does: one DPP reduction, not one
    // per slot row (300 chunks of 60 tokens of 32 / 8 heads 264 -> 246 us)
    tot = npd::wave_sum_i(tot);   // wave-uniform
    nmax = npd::wave_max_i(nmax);
    // Parts per tile: a tile of n steps runs as nsp = ceil(n / ks) near-equal
    // parts (a short tail part would pay a whole item's prologue and merge for
    // a few steps), ks = nmax / p for the p whose estimated time is least: the
    // longest item where one round of the compute units takes them all, else
    // their mean load plus a share of the longest item (what a greedy
    // longest-first order leaves uneven; less with every further round, none
    // from three on). An item costs kItemSteps steps on top of its own, one that
    // publishes and merges kMergeSteps more. Three rounds of whole tiles are not
    // cut, unless the longest outlasts the mean load: one long prefix among many
    // prompts ends the launch by itself (12 chunks of 512 tokens of 32 / 8
    // heads, one on a prefix of 100000: 2050 us whole, 787 cut).
    auto nsp_of = [&](int k, int step) {
      const int p = small_div(n[k] + step - 1, step);
      return !valid[k] ? 0 : (p < 1 ? 1 : (p > a.splits_max ? a.splits_max : p));
    };
    int ks = nmax < 1 ? 1 : nmax;
    const int units = a.num_cus < per_item ? 1 : small_div(a.num_cus, per_item);
    const bool tail = (float)(nmax + kItemSteps) * units > (float)tot + (float)(ntiles * kItemSteps);
    if (a.splits_max > 1 && (ntiles < 3 * units || tail)) {
      const int room = tail ? a.max_items : a.even_items;
      float best = 0.f;
      for (int p = 1; p <= a.splits_max; ++p) {
        const int kp = small_div(nmax + p - 1, p);
        if (p > 1 && kp < kMinPart) break;
        int sums = 0;   // parts, and parts of cut tiles (16 bits each: at most 8 * 512)
#pragma unroll
        for (int k = 0; k < kSlots; ++k)
          if (64 * k < tiles) {
            const int c = nsp_of(k, kp < 1 ? 1 : kp);
            sums += c + (c > 1 ? c << 16 : 0);
          }
        sums = npd::wave_sum_i(sums);
        const int items = sums & 0xffff, cut = sums >> 16;
        if (p > 1 && items > room) break;
        const float longest = (float)(kp + kItemSteps + (p > 1 ? kMergeSteps : 0));
        const float mean = (float)(tot + items * kItemSteps + cut * kMergeSteps) / units;
        const float est = items <= units ? longest
                                         : fmaxf(longest, mean + 0.35f * longest * max(3 * units - items, 0) / (2 * units));
        if (p == 1 || est < 0.97f * best) best = est, ks = kp < 1 ? 1 : kp;
      }
    }
    // Items by part length (bucket len = ceil(n / nsp)), longest first; within
    // a bucket by tile, part and then kv-head.
    int cut[kSlots], len[kSlots], lenmax = 0;
#pragma unroll
    for (int k = 0; k < kSlots; ++k) {
      cut[k] = 0;
      len[k] = -1;
      if (64 * k < tiles) {
        cut[k] = nsp_of(k, ks);
        if (valid[k]) len[k] = small_div(n[k] + cut[k] - 1, cut[k]);
        lenmax = max(lenmax, len[k]);
      }
    }
    lenmax = npd::wave_max_i(lenmax);
    // items in buckets >= b, non-increasing in b; item id is in the last
    // bucket b with from(b) > id (binary search over DPP wave sums)
    auto from = [&](int b) -> int {
      int c = 0;
#pragma unroll
      for (int k = 0; k < kSlots; ++k)
        if (64 * k < tiles) c += len[k] >= b ? cut[k] : 0;
      return npd::wave_sum_i(c) * per_item;
    };
    int id = blockIdx.x;
    if (id >= from(0)) return false;   // past the last item
    int lo = 0, hi = lenmax;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (from(mid) > id) lo = mid; else hi = mid - 1;
    }
    id -= from(lo + 1);
    // the bucket's tile holding item id: the slot row by its sum, then the
    // lane by an inclusive scan over the row
    bool found = false;
    s = t = j = kh = nsp = nsteps = q0 = qlen = ctx = 0;
#pragma unroll
    for (int k = 0; k < kSlots; ++k)
      if (64 * k < tiles && !found) {
        const int c = len[k] == lo ? cut[k] : 0;
        const int sum = npd::wave_scan_i(c);
        const int all = __builtin_amdgcn_readlane(sum, 63) * per_item;
        if (id < all) {
          const int sel = __builtin_ctzll(__ballot(sum * per_item > id));
          nsp = __builtin_amdgcn_readlane(c, sel);
          id -= (__builtin_amdgcn_readlane(sum, sel) - nsp) * per_item;
          s = small_div(64 * k + sel, a.tiles_max);
          t = 64 * k + sel - s * a.tiles_max;
          nsteps = __builtin_amdgcn_readlane(n[k], sel);
          q0 = __builtin_amdgcn_readlane(c0[k], sel);
          qlen = __builtin_amdgcn_readlane(ql[k], sel);
          ctx = __builtin_amdgcn_readlane(cx[k], sel);
          found = true;
        } else {
          id -= all;
        }
      }
    if (!found) return false;   // never: id is below from(lo)
    j = small_div(id, per_item);
    kh = id - j * per_item;
  } else {
    // Fixed order: key part, sequence, tile (the last, with the most keys,
    // first), kv head. The kv head varies fastest, as above, so the tiles of a
    // sequence that run together on an XCD read the same K/V.
    const int id = blockIdx.x;
    int u = id / per_item;
    kh = id - u * per_item;
    const int v = u / a.tiles_max;
    t = a.tiles_max - 1 - (u - v * a.tiles_max);
    j = v / a.num_seqs;
    s = v - j * a.num_seqs;
    q0 = a.cu_seqlens_q[s];
    qlen = a.cu_seqlens_q[s + 1] - q0;
    if (t * TR >= qlen * a.group) return false;
    ctx = a.context_lens[s];
    ctx = ctx < 0 ? 0 : (ctx < cap ? ctx : cap);
    nsteps = (tile_keys<TR>(a, t, qlen, ctx) + KT - 1) / KT;
    nsp = (nsteps + a.ks_steps - 1) / a.ks_steps;
    nsp = nsp < 1 ? 1 : (nsp > a.splits_max ? a.splits_max : nsp);
    if (j >= nsp) return false;
  }
  // near-equal parts, the first nsteps % nsp one step longer
  const int base = small_div(nsteps, nsp), rem = nsteps - base * nsp;
  const int st0 = j * base + (j < rem ? j : rem);
  it = Item{s, t, j, nsp, kh, q0, qlen, ctx, tile_keys<TR>(a, t, qlen, ctx), st0,
            st0 + base + (j < rem ? 1 : 0)};
  return true;
}

// LDS position of 16-byte chunk `chunk` of tile row `row` is chunk ^ swz(row):
// rows are D * 2 bytes apart with no padding (the direct-to-LDS loads write
// 1 KB runs), and the swizzle spreads both reads of a tile over all banks --
// 32 rows at one chunk (K), 4 rows x 4 chunks (transposing V reads). Bits of a
// row index above the fourth do not enter, so rows 16 apart share offsets.
template <int D>
__device__ __forceinline__ int swz(int row) {
  if (D == 64)   // two rows per 256 bytes
    return (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
  return ((row & 3) << 2) | (((row >> 2) & 1) << 1) | ((row >> 3) & 1);
}
// chunk offset bits (bytes) that differ between rows r and r + 8
template <int D>
constexpr int swz8() { return D == 64 ? 32 : 16; }

// 64 lanes x 16 bytes from base + off (per lane) straight into LDS at
// lds .. lds + 1023, lane i at lds + 16 i. Counts in vmcnt; the caller waits.
__device__ __forceinline__ void load_to_lds(uint32_t lds, uint32_t off, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void load_to_lds(uint32_t lds, const void* p) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :: "s"(lds), "v"(p) : "memory", "m0");
}
// All but the last L LDS accesses of this wave are done and at most N of its
// direct-to-LDS loads are still in flight; then the workgroup's barrier.
template <int N, int L = 0>
__device__ __forceinline__ void wait_and_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(%1)\n\ts_barrier" :: "n"(N), "n"(L) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// NW: waves per workgroup, 8 (two per SIMD, 256 registers each) or 4 (one per
// SIMD, up to 512: head dim 256 keeps O in accumulation registers).
// kOff32: every K/V element of the pool lies within 4 GiB of the cache base,
// so gather offsets are 32-bit. kF8: the pool holds OCP e4m3 bytes, converted
// exactly to TT pairs on the way into LDS (through registers); the per-kv-head
// scales go into the score scale and the output.
template <class TT, int D, int NW, bool kOff32, bool kF8>
__global__ __launch_bounds__(64 * NW) void prefill_kernel(PrefillArgs a) {
  static_assert(D == 64 || D == 128 || (D == 256 && !kF8), "head dims of this kernel");
  constexpr int KT = kKT;                              // keys per step
  constexpr int NT = 64 * NW;                          // threads
  constexpr int RB = 2 * D;                            // bytes of a tile row
  constexpr int TB = KT * RB;                         // bytes of a K or V tile
  constexpr int NI = TB / (1024 * NW);             // 1 KB loads per wave and tile (D 128: 2)
  constexpr int NC = D / 16;                           // head-dim chunks of QK
  constexpr int NS = KT / 32;                         // 32-key blocks of S
  constexpr int KB = KT / 16;                         // 16-key blocks of PV
  constexpr int DB = D / 32;                           // 32-dim blocks of O
  constexpr int kRecO = rec_o(D);
  // Head dim 256 keeps the running maximum of a row as its reference, so that
  // the largest P is 1 and exact: one that lags leaves 3 to 9% more error in the
  // output where few keys dominate a row. The 128 accumulators of O are rescaled
  // in most of the first steps then (one of 32 rows has a new maximum), so steps
  // are of 64 keys (of 32: 127 against 103 us for three chunks of 300 to 700
  // tokens of 16 / 8 heads on prefixes to 1500; a lagging reference 88), and two
  // tiles of 32 KB each are what fits: the next one loads during the step.
  constexpr bool kExactMax = D == 256;
  constexpr int NBK = kExactMax ? 2 : kBufK, NBV = kExactMax ? 2 : kBufV;
  static_assert(NI * 1024 * NW == TB, "tile shape");
  __shared__ __attribute__((aligned(1024))) char s_k[NBK * TB];
  __shared__ __attribute__((aligned(1024))) char s_v[NBV * TB];
  __shared__ int s_row[kListBlocks];   // first K/V row of each block of the key range
  __shared__ int s_ticket;
  __shared__ Item s_item;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int hf = lane >> 5, c32 = lane & 31;

  // The first wave derives the item: eight waves sharing the SIMDs for the same
  // answer took 5.1 us where this takes 4.4 (32 tiles, four part counts tried;
  // 3 us where none is, 1.1 in the fixed order). Block ids, queries and the
  // first tiles follow one after another in 4 us; asking for the block ids ahead
  // of the queries gave nothing and cost FP8 pools 15%.
  if (wave == 0) {
    Item it{};
    it.nsp = 0;
    prefill_item<tile_rows(NW), KT>(a, lane, it);
    if (lane == 0) s_item = it;
  }
  __syncthreads();
  auto uni = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  const int nsp = uni(s_item.nsp);
  if (nsp == 0) return;   // no item
  const int s = uni(s_item.s), t = uni(s_item.t), j = uni(s_item.j), kh = uni(s_item.kh);
  const int q0 = uni(s_item.q0), qlen = uni(s_item.qlen), ctx = uni(s_item.ctx), G = a.group;
  const int nkeys = uni(s_item.nkeys), st0 = uni(s_item.st0), st1 = uni(s_item.st1);

  // flattened rows f = token * G + head: the tile's 256, this wave's 32 and
  // this lane's one (clamped to the chunk's last; outputs past it are not stored)
  const int prefix = ctx - qlen;                       // position of the chunk's first token
  const int frows = qlen * G;
  const int wsub = t * NW + wave;                  // 32-row subtile of the (sequence, kv head)
  const int f0 = wsub * kWaveRows;
  const bool row_ok = f0 + c32 < frows;
  const int f = row_ok ? f0 + c32 : frows - 1;
  const int tok = frows < kSmallDiv ? small_div(f, G) : f / G;
  const int h = kh * G + (f - tok * G);
  const int pos = prefix + tok;                        // this lane's query position
  const int wpos0 = __builtin_amdgcn_readfirstlane(pos);
  const int wpos1 = __builtin_amdgcn_readlane(pos, 31);   // the wave's first and last position
  const int bs = a.block_size;
  const int kend = st1 * KT < nkeys ? st1 * KT : nkeys;

  uint16_t* op = a.out + (int64_t)(q0 + tok) * a.out_stride_token + (int64_t)h * a.out_stride_head;
  if (st0 >= st1) {
    // no key at all (every row of the tile sits before position 0): zero rows
    if (row_ok)
#pragma unroll
      for (int e = 0; e < D / 8; ++e) *reinterpret_cast<u32x2*>(op + e * 8 + hf * 4) = u32x2{0, 0};
    return;
  }

  // the lane's query row as B operands: qb[c] = Q[row][c*16 + 8 hf .. +8]
  u32x4 qb[NC];
  {
    const uint16_t* qp = a.q + (int64_t)(q0 + tok) * a.q_stride_token +
                         (int64_t)h * a.q_stride_head + hf * 8;
#pragma unroll
    for (int c = 0; c < NC; ++c) qb[c] = *reinterpret_cast<const u32x4*>(qp + c * 16);
  }

  // Tile loads. 2-byte pools: 1 KB run e of this wave's NI covers tile bytes
  // (wave * NI + e) * 1024 ..; lane i's 16 bytes are the chunk that the swizzle
  // puts at byte 16 i of the run. FP8 pools: through registers, NF loads of
  // F8B bytes (F8B / 8 chunks) per thread. Keys past the split's range are
  // clamped to its last key: a real, finite context row that the causal mask
  // removes (only keys past the tile's last position are clamped).
  constexpr int F8B = D == 64 ? 8 : 16;
  constexpr int LROW = kF8 ? D / F8B : RB / 16;        // lanes per row
  constexpr int NR = kF8 ? KT * D / (NT * F8B) : NI;
  static_assert(!kF8 || NR * NT * F8B == KT * D, "FP8 tile shape");
  int lrow[NR], lcol[NR];   // tile row and source column (bytes) of this lane's loads
#pragma unroll
  for (int e = 0; e < NR; ++e) {
    if (kF8) {
      lrow[e] = (tid + NT * e) / LROW;
      lcol[e] = (tid + NT * e) % LROW * F8B;
    } else {
      const int o = (wave * NI + e) * 1024 + lane * 16;
      lrow[e] = o / RB;
      lcol[e] = ((o % RB / 16) ^ swz<D>(lrow[e])) * 16;
    }
  }
  int blk0 = 0;   // first block of the list in s_row
  // pool row of tile row lrow[e] of step `step` (< 2^31, host check)
  auto pool_row = [&](int step, int e) {
    int tk = step * KT + lrow[e];
    tk = tk < kend ? tk : kend - 1;
    const int lb = a.bs_shift >= 0 ? tk >> a.bs_shift : tk / bs;
    return s_row[lb - blk0] + (tk - (a.bs_shift >= 0 ? lb << a.bs_shift : lb * bs));
  };
  const uint32_t lds_k = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)s_k;
  const uint32_t lds_v = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)s_v;
  typedef uint32_t raw16 __attribute__((ext_vector_type(F8B / 4), aligned(8)));
  struct Raw {
    raw16 k[kF8 ? NR : 1], v[kF8 ? NR : 1];
  };
  int rows[NR];   // pool rows of the tile loaded next
  auto find_rows = [&](int step) {
#pragma unroll
    for (int e = 0; e < NR; ++e) rows[e] = pool_row(step, e);
  };
  // 2-byte pools: the tile of `rows` into LDS buffers kb, vb
  auto load = [&](int kb, int vb) {
#pragma unroll
    for (int e = 0; e < NR; ++e) {
      const uint32_t run = (uint32_t)(wave * NI + e) * 1024u;
      if (kOff32) {
        const uint32_t off = (uint32_t)rows[e] * (uint32_t)RB + (uint32_t)lcol[e];
        load_to_lds(lds_k + kb * TB + run, off, a.k_cache);
        load_to_lds(lds_v + vb * TB + run, off, a.v_cache);
      } else {
        const int64_t off = (int64_t)rows[e] * RB + lcol[e];
        load_to_lds(lds_k + kb * TB + run, reinterpret_cast<const char*>(a.k_cache) + off);
        load_to_lds(lds_v + vb * TB + run, reinterpret_cast<const char*>(a.v_cache) + off);
      }
    }
  };
  // FP8 pools: the tile of `rows` into registers; registers into LDS
  auto fetch = [&](Raw& r) {
#pragma unroll
    for (int e = 0; e < NR; ++e) {
      const int64_t off = kOff32 ? (int64_t)((uint32_t)rows[e] * (uint32_t)D + (uint32_t)lcol[e])
                                 : (int64_t)rows[e] * D + lcol[e];
      r.k[e] = *reinterpret_cast<const raw16*>(reinterpret_cast<const char*>(a.k_cache) + off);
      r.v[e] = *reinterpret_cast<const raw16*>(reinterpret_cast<const char*>(a.v_cache) + off);
    }
  };
  auto stash = [&](const Raw& r, int kb, int vb) {
#pragma unroll
    for (int e = 0; e < NR; ++e)
#pragma unroll
      for (int x = 0; x < F8B / 8; ++x) {
        const int at = lrow[e] * RB + (((lcol[e] / 8 + x) ^ swz<D>(lrow[e])) << 4);
        auto put = [&](char* tile, const raw16& w) {
          *reinterpret_cast<u32x4*>(tile + at) =
              u32x4{npd::e4m3x2_to<TT, false>(w[2 * x]), npd::e4m3x2_to<TT, true>(w[2 * x]),
                    npd::e4m3x2_to<TT, false>(w[2 * x + 1]), npd::e4m3x2_to<TT, true>(w[2 * x + 1])};
        };
        put(s_k + kb * TB, r.k[e]);
        put(s_v + vb * TB, r.v[e]);
      }
  };

  f32x16 oacc[DB];   // O^T[d = db*32 + 8*(i/4) + 4 hf + i%4][row c32]
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[db][i] = 0.f;
  // reference of the row's exponents (log2 units; -inf: none yet), what is
  // added to the scaled scores (-mref; large before the first reference, so
  // that any visible score asks for one), and the row sum of this lane's keys
  float mref = -INFINITY, nmref = kNoRef, lsum = 0.f;
  const float c2 = kF8 ? a.scale_log2 * a.k_scale[kh] : a.scale_log2;
  const float oscale = kF8 ? a.v_scale[kh] : 1.f;

  const int kofs = c32 * RB + ((hf ^ swz<D>(c32)) << 4);
  // K operand x of a step: head-dim chunk x / NS of 32-key block x % NS
  auto read_k = [&](int kb, int x) {
    return *reinterpret_cast<const u32x4*>(s_k + ((kb * TB + kofs) ^ (x / NS << 5)) + x % NS * 32 * RB);
  };
  auto qk = [&](int kb, const u32x4 (&kpre)[kAhead], f32x16 (&sacc)[NS]) {
#pragma unroll
    for (int n = 0; n < NS; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) sacc[n][i] = 0.f;
#pragma unroll
    for (int x = 0; x < NS * NC; ++x) {
      const u32x4 ka = x < kAhead ? kpre[x] : read_k(kb, x);
      sacc[x % NS] = Mfma<TT>::mma32(ka, qb[x / NS], sacc[x % NS]);
    }
  };
  auto softmax = [&](int step, f32x16 (&sacc)[NS], u32x4 (&pb)[KB]) {
    const int key0 = step * KT;
    if (__builtin_expect(key0 + KT - 1 > wpos0, 0)) {   // some key here is after some row
      const int lim = pos - key0 - 4 * hf;
#pragma unroll
      for (int n = 0; n < NS; ++n)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (n * 32 + 8 * (i >> 2) + (i & 3) > lim) sacc[n][i] = -INFINITY;
    }
    // P = 2^(s*c - m), packed: pb[kb] is the B operand of keys kb*16 .. +16 in
    // slots e < 4 -> key 4 hf + e, e >= 4 -> 8 + 4 hf + e - 4
    auto expo = [&]() {
#pragma unroll
      for (int n = 0; n < NS; ++n)
#pragma unroll
        for (int i = 0; i < 16; i += 2)
          pb[n * 2 + (i >> 3)][(i & 7) >> 1] =
              TT::pack2(__builtin_amdgcn_exp2f(fmaf(sacc[n][i], c2, nmref)),
                        __builtin_amdgcn_exp2f(fmaf(sacc[n][i + 1], c2, nmref)));
    };
    // sum of this lane's P of the step on top of x
    auto sum_p = [&](float x) {
      float ps[4] = {x, 0.f, 0.f, 0.f};   // four short chains
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) ps[i] = TT::dot2(pb[kb][i], TT::kOne2, ps[i]);
      return (ps[0] + ps[1]) + (ps[2] + ps[3]);
    };
    // the row's scaled maximum of the step
    auto row_max = [&]() {
      float mx = fmaxf(fmaxf(sacc[0][0], sacc[0][1]), sacc[0][2]);
#pragma unroll
      for (int e = 3; e + 1 < 16 * NS; e += 2)
        mx = fmaxf(fmaxf(mx, sacc[e >> 4][e & 15]), sacc[(e + 1) >> 4][(e + 1) & 15]);
      return npd::half_max(fmaxf(mx, sacc[NS - 1][15])) * c2;
    };
    // a row whose maximum passed its reference by `move` takes it, plus `bias`,
    // as the new one
    auto move_ref = [&](float mx, float move, float bias) {
      const bool nd = mx > mref + move;
      const float mnew = nd ? mx + bias : mref;
      const float alpha = nd ? __builtin_amdgcn_exp2f(mref - mnew) : 1.f;   // 0 from -inf
#pragma unroll
      for (int db = 0; db < DB; ++db) oacc[db] *= alpha;
      lsum *= alpha;
      mref = mnew;
      nmref = mnew == -INFINITY ? kNoRef : -mnew;
    };
    if constexpr (kExactMax) {
      const float mx = row_max();
      if (__ballot(mx > mref) != 0) move_ref(mx, 0.f, 0.f);
      expo();
      lsum = sum_p(lsum);
      return;
    }
    expo();
    // The reference moves only when an exponential grew past a bound, read off
    // the packed values or their sum: the maximum is taken in that rare case
    // only.
    constexpr bool kBySum = std::is_same<TT, npd::F16>::value;
    float st = 0.f;
    bool past;
    if constexpr (kBySum) {
      st = sum_p(0.f);
      past = st >= Bound<TT>::kPast;
    } else {
      past = past_two(pb);
    }
    if (__builtin_expect(__ballot(past) != 0, 0)) {
      move_ref(row_max(), Bound<TT>::kMove, Bound<TT>::kBias);
      expo();
      if constexpr (kBySum) st = sum_p(0.f);
    }
    if constexpr (kBySum) lsum += st;
    else lsum = sum_p(lsum);
  };
  // O^T += V^T . P^T ; A = V^T[d = db*32 + c32][keys as pb's slots]: two
  // transposing reads, in each of which lane i of a group of 16 addresses key
  // i/4 (+ 4 hf) and dims 16*(group & 1) + 4*(i%4) .. +3
  const int vrow = 4 * hf + ((lane & 15) >> 2);
  const int vofs = vrow * RB + (((((lane >> 4) & 1) * 2 + ((lane & 3) >> 1)) ^ swz<D>(vrow)) << 4) +
                   (lane & 1) * 8;
  auto pv = [&](int vb, const u32x4 (&pb)[KB]) {
    const int vt = vb * TB + vofs;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const int at = vt ^ (db << 6);
        const u32x2 lo = lds_read_tr(reinterpret_cast<const uint16_t*>(s_v + at + kb * 16 * RB));
        const u32x2 hi = lds_read_tr(
            reinterpret_cast<const uint16_t*>(s_v + (at ^ swz8<D>()) + (kb * 16 + 8) * RB));
        oacc[db] = Mfma<TT>::mma32(u32x4{lo.x, lo.y, hi.x, hi.y}, pb[kb], oacc[db]);
      }
  };

  // Order of the interval's LDS reads and MFMAs (NS * NC QK, then KB * DB PV):
  // operand reads stay kAhead MFMAs ahead (the first kAhead K operands were
  // read before the barrier), so that none waits on LDS latency. Left to itself
  // the compiler keeps one pair of K reads in flight.
  auto interleave = [&]() {
    constexpr int kQ = NS * NC, kP = KB * DB;
#pragma unroll
    for (int i = 0; i < kQ - kAhead; ++i) {
      __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 1, 0);
      __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
    }
#pragma unroll
    for (int i = 0; i < kP; ++i) {
      __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 2, 0);
      __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(kSchedMfma, kAhead, 0);
  };
  // Two waves share each SIMD (waves w and w + 4), kept half a step apart: in
  // every interval between two barriers one of them runs its MFMAs (QK of its
  // step and PV of the step before), the other its softmax.
  //   interval       2i                2i + 1
  //   waves 0-3   QK(i), PV(i-1)     softmax(i)
  //   waves 4-7   softmax(i-1)       QK(i), PV(i-1)
  // Each wave starts its share of tile i + 3 before softmax(i) (over an FP8
  // pool at head dim 64, where the MFMAs are the shorter half and the share is
  // conversions too, before those of step i: 32 / 8 heads, 1684 + 994 tokens
  // 43.0 against 44.5 us, 6000 on a prefix of 2000 314 against 324, 8 chunks of
  // 200 on 3000 72 against 75, 4 of 1024 in fp16 73.3 against 72.7; 2-byte pools
  // gain nothing), in interval 2i at the earliest, into the buffers of K tile
  // i - 1 and V tile i - 2 (4 K, 5 V buffers), last read in interval 2i - 1. Its share of tile i + 2
  // has landed when its softmax(i) is done (interval 2i + 1 or 2i + 2), so the
  // whole tile has when a wave reads its first K operands ahead of step i + 2,
  // at the end of interval 2i + 3 or 2i + 4.
  constexpr bool kLoadFirst = D == 64 && kF8;
  const bool late = NW == 8 && wave >= NW / 2;
  const int list_steps = (int)((int64_t)(kListBlocks - 2) * bs / KT);   // steps the list covers
  const int seg = list_steps < 1 ? 1 : list_steps;
  for (int sb = st0; sb < st1; sb += seg) {
    const int n = (sb + seg < st1 ? sb + seg : st1) - sb;
    // first rows of the blocks of this segment's keys (ids clamped into the pool)
    auto div_bs = [&](int x) { return a.bs_shift >= 0 ? x >> a.bs_shift : x / bs; };
    blk0 = div_bs(sb * KT);
    const int ke = (sb + n) * KT < kend ? (sb + n) * KT : kend;
    const int nblk = div_bs(ke - 1) + 1 - blk0;
    if (sb != st0) __syncthreads();   // the last segment's reads are done
    for (int e = tid; e < nblk; e += NT) {
      int bid = a.block_tables[(int64_t)s * a.max_bps + blk0 + e];
      bid = bid < 0 ? 0 : (bid >= a.num_blocks ? a.num_blocks - 1 : bid);
      s_row[e] = (bid * a.num_kv_heads + kh) * bs;
    }
    // nothing of the compiler's own loads stays in flight: its waits inside
    // the loop would cover the tile loads too
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    __syncthreads();
    // steps in which some row of this wave sees a key (the causal mask only
    // ever ends a wave's steps): later ones it spends in the barriers
    int nact = wpos1 < sb * KT ? 0 : wpos1 / KT - sb + 1;
    nact = nact < n ? nact : n;
    u32x4 pb[KB];
    if constexpr (kExactMax) {
      // One wave per SIMD: QK, softmax and PV of a step in turn, one barrier
      // per step. Past it tile i has landed and every wave has left step i - 1,
      // whose buffers tile i + 1 loads into.
      find_rows(sb);
      load(0, 0);
      for (int i = 0; i < n; ++i) {
        const int b = i & 1;
        wait_and_barrier<0>();
        if (i + 1 < n) {
          find_rows(sb + i + 1);
          load(b ^ 1, b ^ 1);
        }
        if (i >= nact) continue;
        f32x16 sacc[NS];
        u32x4 kpre[kAhead];
#pragma unroll
        for (int x = 0; x < kAhead; ++x) kpre[x] = read_k(b, x);
        qk(b, kpre, sacc);
        softmax(sb + i, sacc, pb);
        pv(b, pb);
      }
      continue;
    }
    // P of the step before the segment: none. Its V tile (the last buffer) is
    // zeroed too, so that the first interval's PV adds nothing.
#pragma unroll
    for (int e = 0; e < KB; ++e) pb[e] = u32x4{0, 0, 0, 0};
    for (int e = tid; e < TB / 16; e += NT)
      *reinterpret_cast<u32x4*>(s_v + (kBufV - 1) * TB + e * 16) = u32x4{0, 0, 0, 0};
    Raw raw;   // FP8: the bytes of the tile stashed next
    if constexpr (kF8) {
      Raw r1, r2;
      find_rows(sb);
      fetch(raw);
      if (n > 1) { find_rows(sb + 1); fetch(r1); }
      if (n > 2) { find_rows(sb + 2); fetch(r2); }
      stash(raw, 0, 0);
      if (n > 1) stash(r1, 1, 1);
      if (n > 2) stash(r2, 2, 2);
      if (n > 3) { find_rows(sb + 3); fetch(raw); }
      wait_and_barrier<63>();
    } else {
      find_rows(sb);
      load(0, 0);
      if (n > 1) { find_rows(sb + 1); load(1, 1); }
      if (n > 2) { find_rows(sb + 2); load(2, 2); }
      if (n > 3) find_rows(sb + 3);
      if (n > 2) wait_and_barrier<2 * NR>(); else wait_and_barrier<0>();   // tiles 0 and 1
    }
    // buffers of the step's tile, of V tile i - 1 and of tile i + 3
    int kb = 0, vb = 0, vp = kBufV - 1, kb3 = 3, vb3 = 3;
    // the first K operands of step i + 1, read ahead of its barrier; and tile
    // i + 2 has landed, i + 3 may be in flight
    u32x4 kpre[kAhead];
    auto softmax_done = [&](int i) {
      if (i + 1 < n)
#pragma unroll
        for (int x = 0; x < kAhead; ++x) kpre[x] = read_k(kb, x);
      if (!kF8 && i + 3 < n) wait_and_barrier<2 * NR, kAhead>();
      else wait_and_barrier<kF8 ? 63 : 0, kAhead>();
    };
    auto next_tile = [&](int i) {   // tile i + 3, and the rows (FP8: the bytes) of tile i + 4
      if (i + 3 < n) {
        if constexpr (kF8) stash(raw, kb3, vb3); else load(kb3, vb3);
        if (i + 4 < n) {
          find_rows(sb + i + 4);
          if constexpr (kF8) fetch(raw);
        }
      }
    };
    auto advance = [&]() {   // to step i + 1's buffers
      kb = (kb + 1) & 3;
      kb3 = (kb3 + 1) & 3;
      vp = vb;
      vb = vb == kBufV - 1 ? 0 : vb + 1;
      vb3 = vb3 == kBufV - 1 ? 0 : vb3 + 1;
    };
    static_assert(kBufK == 4 && kBufV == 5, "buffer rotation");
#pragma unroll
    for (int x = 0; x < kAhead; ++x) kpre[x] = read_k(kb, x);
    if (late) wait_and_barrier<63>();
    int i = 0;
    for (; i < nact; ++i) {
      f32x16 sacc[NS];   // S^T[key = n*32 + 8*(i/4) + 4 hf + i%4][row c32]
      if (kLoadFirst) next_tile(i);
      __builtin_amdgcn_s_setprio(1);
      qk(kb, kpre, sacc);
      pv(vp, pb);
      interleave();
      wait_and_barrier<63>();
      __builtin_amdgcn_s_setprio(0);
      if (!kLoadFirst) next_tile(i);
      advance();
      softmax(sb + i, sacc, pb);
      softmax_done(i);
    }
    pv(vp, pb);
    for (; i < n; ++i) {
      if (kLoadFirst) next_tile(i);
      wait_and_barrier<63>();
      if (!kLoadFirst) next_tile(i);
      advance();
      softmax_done(i);
    }
    if (!late) wait_and_barrier<63>();   // as many barriers as waves 4-7
  }

  float l = npd::half_sum(lsum);   // the row's keys are in lanes c32 and c32 + 32

  if (nsp > 1) {
    // publish this split's partial (register order: every store is 512
    // contiguous bytes), then the last split of the tile to arrive merges
    const int64_t rec = (((int64_t)s * a.num_kv_heads + kh) * a.subtiles + wsub) * a.splits_max;
    {
      float* po = a.part_o + (rec + j) * kRecO + lane * 2;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          npd::st_coherent2(po + (db * 8 + i) * 128, oacc[db][2 * i], oacc[db][2 * i + 1]);
      npd::st_coherent2(a.part_ml + (rec + j) * kRecML + lane * 2, mref, l);
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);   // every store of this wave has completed
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    const int64_t cidx = ((int64_t)s * a.tiles_max + t) * a.num_kv_heads + kh;
    if (tid == 0)
      s_ticket = __hip_atomic_fetch_add(a.counters + cidx, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (s_ticket != nsp - 1) return;
    for (int jj = 0; jj < nsp; ++jj) {
      if (jj == j) continue;
      float mp, lp;
      npd::ld_coherent2(a.part_ml + (rec + jj) * kRecML + lane * 2, mp, lp);
      const float mm = fmaxf(mref, mp);
      const float wa = mref == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mref - mm);
      const float wb = mp == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mp - mm);
      l = l * wa + lp * wb;
      mref = mm;
      const float* po = a.part_o + (rec + jj) * kRecO + lane * 2;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float x0, x1;
          npd::ld_coherent2(po + (db * 8 + i) * 128, x0, x1);
          oacc[db][2 * i] = oacc[db][2 * i] * wa + x0 * wb;
          oacc[db][2 * i + 1] = oacc[db][2 * i + 1] * wa + x1 * wb;
        }
    }
    if (tid == 0) __hip_atomic_store(a.counters + cidx, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // normalise and store: lane writes d = db*32 + 8e + 4 hf .. +3 of its row
  if (!row_ok) return;
  const float inv = (l > 0.f && pos >= 0) ? oscale / l : 0.f;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      u32x2 w;
      w.x = TT::pack2(oacc[db][4 * e] * inv, oacc[db][4 * e + 1] * inv);
      w.y = TT::pack2(oacc[db][4 * e + 2] * inv, oacc[db][4 * e + 3] * inv);
      *reinterpret_cast<u32x2*>(op + db * 32 + e * 8 + hf * 4) = w;
    }
}

// The head dims whose rows are not a power of two of 16-byte chunks (32, 96,
// 160, 192, 224), and 256 over an FP8 pool. One workgroup of 4 waves per
// (sequence, query head, 64-row query tile); wave w owns query rows
// 16w .. 16w + 15 of the tile. Per step of 64 keys the workgroup copies the kv
// head's K and V rows into LDS (keys past the visible range clamped to the
// last visible key, as in prefill_kernel), then every wave computes
//   S^T = K . Q^T     (v_mfma_f32_16x16x32, D/32 chunks of the head dim x
//                      4 blocks of 16 keys; Q rows held in registers),
//   a causal mask and an online softmax in fp32 (log2 units; O and the row
//   sum rescaled whenever a row's running max grows),
//   O^T += V^T . P^T  (D/16 blocks of 16 dims x 2 chunks of 32 keys; V^T via
//                      the transposing LDS read, P^T from the S^T layout).
// The operand layouts, the P packing and the normalisation (the row sum adds
// the rounded P values) are those of prefill_kernel. The next step's K/V
// chunks load into registers during the step (two workgroups per CU, at most
// 246 VGPRs); the workgroups of one (sequence, kv head) share K/V through one
// XCD's L2 rather than one LDS tile, and there are no key splits. Rows with no
// visible key are written as zeros.
template <class TT, int D, bool kF8>
__global__ __launch_bounds__(256, 2) void prefill_generic_kernel(PrefillArgs a) {
  constexpr int kGT = 256;                      // threads
  constexpr int RW = D + 16;                    // LDS row (elements); 16-byte multiple
  constexpr int CPR = D / 8;                    // 8-element chunks per K/V row
  constexpr int NPASS = kKT * CPR / kGT;        // chunks of the 64-key tile per thread
  constexpr int NC = D / 32;                    // head-dim chunks of QK
  constexpr int NB = D / 16;                    // 16-dim blocks of O
  static_assert(D % 32 == 0 && D >= 32 && D <= 256, "head dims of this kernel");
  static_assert(NPASS * kGT == kKT * CPR && RW % 8 == 0, "tile shape");
  __shared__ __attribute__((aligned(16))) uint16_t s_k[kKT * RW];
  __shared__ __attribute__((aligned(16))) uint16_t s_v[kKT * RW];

  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int g = lane >> 4, r = lane & 15;
  // Every workgroup of one (sequence, kv head) reads the same keys from 0 up:
  // they all run on one XCD (workgroups go to XCDs round-robin by blockIdx),
  // one after another in that XCD's order, so the K/V rows come from its L2
  // after the first read. Groups go longest context first (up to 64
  // sequences; more keep their order); within a group the last tile (the
  // most keys) first, the group's query heads of a tile together.
  const int per = a.tiles_max * a.group;        // workgroups per (sequence, kv head)
  const int xcd = (int)(blockIdx.x & 7u), p = (int)(blockIdx.x >> 3);
  const int gi = (p / per) * 8 + xcd;           // (sequence rank, kv head) index
  if (gi >= a.num_seqs * a.num_kv_heads) return;
  const int u = p - (p / per) * per;
  const int rank = gi / a.num_kv_heads;
  const int t = a.tiles_max - 1 - u / a.group;
  const int h = (gi - rank * a.num_kv_heads) * a.group + (u - (u / a.group) * a.group);
  const int cap = a.max_bps * a.block_size;
  int s = rank;
  if (a.num_seqs <= 64) {
    // lane i stands for sequence i; its rank counts the sequences with a
    // longer context (ties: the lower index first)
    int n = -1;
    if (lane < a.num_seqs) {
      n = a.context_lens[lane];
      n = n < 0 ? 0 : (n < cap ? n : cap);
    }
    int rk = 0;
    for (int i = 0; i < a.num_seqs; ++i) {
      const int ni = __builtin_amdgcn_readlane(n, i);
      rk += (ni > n || (ni == n && i < lane)) ? 1 : 0;
    }
    const uint64_t m = __ballot(lane < a.num_seqs && rk == rank);
    s = __builtin_amdgcn_readfirstlane(__builtin_ctzll(m));
  }
  const int q0 = a.cu_seqlens_q[s];
  const int qlen = a.cu_seqlens_q[s + 1] - q0;
  if (t * 64 >= qlen) return;
  int ctx = a.context_lens[s];
  ctx = ctx < 0 ? 0 : (ctx < cap ? ctx : cap);
  const int kh = h / a.group;
  const int prefix = ctx - qlen;                 // position of query row 0
  const int rows = (qlen - t * 64) < 64 ? (qlen - t * 64) : 64;
  int nkeys = prefix + t * 64 + rows;            // keys 0 .. the tile's last position
  nkeys = nkeys < 0 ? 0 : nkeys;
  const int nsteps = (nkeys + kKT - 1) / kKT;
  const int bs = a.block_size;
  const int row = t * 64 + wave * 16 + r;        // this lane's query row (S^T column r)
  const int pos = prefix + row;

  u32x4 qb[NC];   // B operand: Q[row][c*32 + 8g .. +8]; rows past the chunk read its last row
  {
    const int rq = row < qlen ? row : qlen - 1;
    const uint16_t* qp = a.q + (int64_t)(q0 + rq) * a.q_stride_token +
                         (int64_t)h * a.q_stride_head + g * 8;
#pragma unroll
    for (int c = 0; c < NC; ++c) qb[c] = *reinterpret_cast<const u32x4*>(qp + c * 32);
  }
  f32x4 oacc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) oacc[nb] = f32x4{0, 0, 0, 0};
  float m = -INFINITY, l = 0.f;
  const float c2 = kF8 ? a.scale_log2 * a.k_scale[kh] : a.scale_log2;
  const float oscale = kF8 ? a.v_scale[kh] : 1.f;

  // K/V of the step's tile: raw chunks loaded into registers one step ahead
  // (in flight during the previous step's MFMAs), converted and copied into
  // LDS at the step's start. Keys past the visible range are clamped to the
  // last visible key (a real, finite row; the causal mask removes them).
  // Chunk tid + 256e of the tile (e < NPASS) is chunk col_of(e) of key
  // key_of(e): every thread moves whole 16-byte chunks, also when D / 8 is
  // not a power of two.
  typedef typename std::conditional<kF8, u32x2, u32x4>::type raw_t;   // 8 elements
  raw_t kr[NPASS], vr[NPASS];
  auto key_of = [&](int e) { return (tid + kGT * e) / CPR; };
  auto col_of = [&](int e) { return (tid + kGT * e) % CPR; };
  auto fetch = [&](int step) {
#pragma unroll
    for (int e = 0; e < NPASS; ++e) {
      const int col = col_of(e);
      int tok = step * kKT + key_of(e);
      tok = tok < nkeys ? tok : nkeys - 1;
      const int lb = a.bs_shift >= 0 ? tok >> a.bs_shift : tok / bs;
      int blk = a.block_tables[(int64_t)s * a.max_bps + lb];
      blk = blk < 0 ? 0 : (blk >= a.num_blocks ? a.num_blocks - 1 : blk);
      const int64_t ri = ((int64_t)blk * a.num_kv_heads + kh) * bs + (tok - lb * bs);
      if constexpr (kF8) {   // D-byte rows, 8-byte chunks
        kr[e] = *reinterpret_cast<const u32x2*>(reinterpret_cast<const char*>(a.k_cache) + ri * D + col * 8);
        vr[e] = *reinterpret_cast<const u32x2*>(reinterpret_cast<const char*>(a.v_cache) + ri * D + col * 8);
      } else {
        const int64_t idx = ri * CPR + col;   // 16-byte units
        kr[e] = a.k_cache[idx];
        vr[e] = a.v_cache[idx];
      }
    }
  };
  auto pairs = [](raw_t w) -> u32x4 {
    if constexpr (kF8)
      return u32x4{npd::e4m3x2_to<TT, false>(w.x), npd::e4m3x2_to<TT, true>(w.x),
                   npd::e4m3x2_to<TT, false>(w.y), npd::e4m3x2_to<TT, true>(w.y)};
    else
      return w;
  };
  if (nsteps > 0) fetch(0);
  for (int step = 0; step < nsteps; ++step) {
    __syncthreads();   // every wave is done with the previous tile
#pragma unroll
    for (int e = 0; e < NPASS; ++e) {
      const int kk = key_of(e), col = col_of(e);
      *reinterpret_cast<u32x4*>(&s_k[kk * RW + col * 8]) = pairs(kr[e]);
      *reinterpret_cast<u32x4*>(&s_v[kk * RW + col * 8]) = pairs(vr[e]);
    }
    __syncthreads();
    if (step + 1 < nsteps) fetch(step + 1);

    // S^T[key n*16 + 4g + i][query r]
    f32x4 sacc[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) sacc[n] = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const u32x4 ka = *reinterpret_cast<const u32x4*>(&s_k[(n * 16 + r) * RW + c * 32 + g * 8]);
        sacc[n] = Mfma<TT>::mma(ka, qb[c], sacc[n]);
      }
    const int key0 = step * kKT;
    float v[16];
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = key0 + n * 16 + 4 * g + i;
        v[n * 4 + i] = key <= pos ? sacc[n][i] : -INFINITY;
      }
    float mx = v[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, v[e]);
    mx = row_max4(mx);
    const float mnew = fmaxf(m, mx * c2);
    const float mref = mnew == -INFINITY ? 0.f : mnew;
    const float alpha = __builtin_amdgcn_exp2f(m - mref);   // 0 from the initial -inf
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) oacc[nb] *= alpha;
    l *= alpha;
    m = mnew;
    uint32_t packed[8];
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
      const float p0 = __builtin_amdgcn_exp2f(fmaf(v[e], c2, -mref));
      const float p1 = __builtin_amdgcn_exp2f(fmaf(v[e + 1], c2, -mref));
      const uint32_t u = TT::pack2(p0, p1);
      l = TT::dot2(u, TT::kOne2, l);
      packed[e / 2] = u;
    }
    // B operand of keys kc*32 .. +32: slots e < 4 -> key 4g + e, e >= 4 -> 16 + 4g + e - 4
    const u32x4 pb[2] = {u32x4{packed[0], packed[1], packed[2], packed[3]},
                         u32x4{packed[4], packed[5], packed[6], packed[7]}};
    const uint16_t* vlane = s_v + (g * 4 + (r >> 2)) * RW + 4 * (r & 3);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        const u32x2 lo = lds_read_tr(vlane + (kc * 32) * RW + nb * 16);
        const u32x2 hi = lds_read_tr(vlane + (kc * 32 + 16) * RW + nb * 16);
        oacc[nb] = Mfma<TT>::mma(u32x4{lo.x, lo.y, hi.x, hi.y}, pb[kc], oacc[nb]);
      }
  }
  l = row_sum4(l);
  if (row >= qlen) return;
  const float inv = (l > 0.f && pos >= 0) ? oscale / l : 0.f;
  uint16_t* op = a.out + (int64_t)(q0 + row) * a.out_stride_token + (int64_t)h * a.out_stride_head;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const f32x4 o = oacc[nb];
    u32x2 w;
    w.x = TT::pack2(o[0] * inv, o[1] * inv);
    w.y = TT::pack2(o[2] * inv, o[3] * inv);
    *reinterpret_cast<u32x2*>(op + nb * 16 + g * 4) = w;
  }
}

template <class TT, bool kF8>
int launch_generic(int64_t head_dim, const PrefillArgs& a, int64_t grid, hipStream_t st,
                   const char* name) {
  const dim3 g((unsigned)grid), b(256);
  switch (head_dim) {
    case 32: hipLaunchKernelGGL((prefill_generic_kernel<TT, 32, kF8>), g, b, 0, st, a); break;
    case 96: hipLaunchKernelGGL((prefill_generic_kernel<TT, 96, kF8>), g, b, 0, st, a); break;
    case 160: hipLaunchKernelGGL((prefill_generic_kernel<TT, 160, kF8>), g, b, 0, st, a); break;
    case 192: hipLaunchKernelGGL((prefill_generic_kernel<TT, 192, kF8>), g, b, 0, st, a); break;
    case 224: hipLaunchKernelGGL((prefill_generic_kernel<TT, 224, kF8>), g, b, 0, st, a); break;
    default:
      if constexpr (kF8) {
        if (head_dim == 256) {
          hipLaunchKernelGGL((prefill_generic_kernel<TT, 256, kF8>), g, b, 0, st, a);
          break;
        }
      }
      return npd::fail(NPD_E_INVALID, "%s: head_dim %lld", name, (long long)head_dim);
  }
  return npd::check_launch(name);
}

template <class TT, int D, int NW, bool kF8>
void launch_d(bool off32, const PrefillArgs& a, int64_t grid, hipStream_t st) {
  const dim3 g((unsigned)grid), b(64 * NW);
  if (off32) hipLaunchKernelGGL((prefill_kernel<TT, D, NW, true, kF8>), g, b, 0, st, a);
  else hipLaunchKernelGGL((prefill_kernel<TT, D, NW, false, kF8>), g, b, 0, st, a);
}

template <class TT, bool kF8>
int launch_dt(int64_t head_dim, int waves, bool off32, const PrefillArgs& a, int64_t grid,
              hipStream_t st, const char* name) {
  if (head_dim == 256) {
    if constexpr (!kF8) launch_d<TT, 256, 4, false>(off32, a, grid, st);
  } else if (head_dim == 64) launch_d<TT, 64, 8, kF8>(off32, a, grid, st);
  else if (waves == 8) launch_d<TT, 128, 8, kF8>(off32, a, grid, st);
  else launch_d<TT, 128, 4, kF8>(off32, a, grid, st);
  return npd::check_launch(name);
}

// Workspace: [counter region (kCounterBytes) | O partials | (m, l) partials].
// Sized for the most records any group size can address: a (sequence, kv head)
// of G heads has 8 * ceil(max_q_len * G / 256) <= G * (ceil(max_q_len / 32) + 7)
// subtiles of 32 flattened rows (no more with 4-wave tiles).
struct Layout {
  int splits, ks_steps;
  int64_t o_off, ml_off, total;
};

Layout prefill_layout(int64_t num_seqs, int64_t num_heads, int64_t head_dim, int64_t max_q_len,
                      int64_t max_context_len) {
  Layout L{1, kSplitSteps, 0, 0, 0};
  if (max_context_len > 0) {
    // splits of kSplitSteps steps, longer ones when that would exceed kMaxSplits
    const int64_t steps = (max_context_len + kKT - 1) / kKT;
    int64_t ks = (steps + kMaxSplits - 1) / kMaxSplits;
    ks = ks < kSplitSteps ? kSplitSteps : ks;
    L.ks_steps = (int)ks;
    L.splits = (int)((steps + ks - 1) / ks);
  }
  if (L.splits <= 1 || num_seqs <= 0 || num_heads <= 0 || max_q_len <= 0) {
    L.splits = 1;
    return L;
  }
  const int64_t t32 = (max_q_len + kWaveRows - 1) / kWaveRows + 7;
  const int64_t units = num_seqs * t32 * num_heads;
  const int64_t nrec = units * L.splits;
  L.o_off = npd::kCounterBytes;
  L.ml_off = L.o_off + nrec * rec_o((int)head_dim) * 4;
  L.total = L.ml_off + nrec * kRecML * 4;
  return L;
}

}  // namespace

extern "C" int64_t npd_paged_prefill_workspace_size(int64_t num_seqs, int64_t total_q,
                                                    int64_t num_heads, int64_t head_dim,
                                                    int64_t max_q_len, int64_t max_context_len) {
  (void)total_q;
  // head dims other than 64 and 128 are not cut and need no workspace
  if (head_dim != 64 && head_dim != 128) return 0;
  return prefill_layout(num_seqs, num_heads, head_dim, max_q_len, max_context_len).total;
}

namespace {

// Shared by the 2-byte and the FP8 entry points: k_scale / v_scale are null
// for 2-byte pools.
int prefill_impl(void* out, const void* query, const void* key_cache, const void* value_cache,
                 const int32_t* block_tables, const int32_t* cu_seqlens_q,
                 const int32_t* context_lens, const float* k_scale, const float* v_scale,
                 int64_t num_seqs, int64_t total_q, int64_t num_heads, int64_t num_kv_heads,
                 int64_t head_dim, int64_t num_blocks, int64_t block_size,
                 int64_t max_blocks_per_seq, int64_t max_q_len, int64_t max_context_len,
                 float scale, int64_t q_stride_token, int64_t q_stride_head,
                 int64_t out_stride_token, int64_t out_stride_head, void* workspace,
                 int64_t workspace_bytes, int32_t dtype, void* stream, bool fp8,
                 const char* name) {
  using namespace npd;
  if (dtype != NPD_DTYPE_F16 && dtype != NPD_DTYPE_BF16)
    return fail(NPD_E_DTYPE, "%s: unsupported dtype code %d (fp16/bf16 only)", name, dtype);
  if (num_seqs < 0 || total_q < 0 || num_heads <= 0 || num_kv_heads <= 0 || num_blocks <= 0 ||
      block_size <= 0 || max_blocks_per_seq <= 0 || max_q_len < 0)
    return fail(NPD_E_INVALID, "%s: bad sizes", name);
  if (head_dim < 32 || head_dim > 256 || head_dim % 32 != 0)
    return fail(NPD_E_INVALID, "%s: head_dim %lld is not a multiple of 32 in [32, 256]", name,
                (long long)head_dim);
  // head dims 64, 128 and 256: prefill_kernel (256 without key splits: its
  // callers bring no workspace); every other one, and 256 over an FP8 pool
  // (three chunks of 300 to 700 tokens of 16 / 8 heads on prefixes to 1500:
  // 100.5 us, prefill_kernel with the exact maximum 121): prefill_generic_kernel
  const bool generic = head_dim != 64 && head_dim != 128 && (head_dim != 256 || fp8);
  if (num_heads % num_kv_heads != 0)
    return fail(NPD_E_INVALID, "%s: num_heads %lld is not a multiple of num_kv_heads %lld", name,
                (long long)num_heads, (long long)num_kv_heads);
  const int64_t g = num_heads / num_kv_heads;
  if (num_blocks * block_size * num_kv_heads > INT32_MAX || max_blocks_per_seq * block_size > INT32_MAX)
    return fail(NPD_E_INVALID, "%s: pool exceeds int32 row indexing", name);
  if ((head_dim == 64 || head_dim == 128) && max_blocks_per_seq > kMaxTableBlocks)
    return fail(NPD_E_INVALID, "%s: block tables wider than %d blocks are not supported", name,
                kMaxTableBlocks);
  if (q_stride_token % 8 || q_stride_head % 8 || out_stride_token % 4 || out_stride_head % 4 ||
      q_stride_token < 0 || q_stride_head < 0 || out_stride_token < 0 || out_stride_head < 0)
    return fail(NPD_E_ALIGN, "%s: query strides must be multiples of 8 elements, out strides of 4",
                name);
  if (!(scale > 0.f) || scale == INFINITY)   // the row maxima are taken before scaling
    return fail(NPD_E_INVALID, "%s: scale must be positive and finite", name);
  if (num_seqs == 0 || total_q == 0 || max_q_len == 0) return NPD_OK;
  if (!out || !query || !key_cache || !value_cache || !block_tables || !cu_seqlens_q || !context_lens)
    return fail(NPD_E_INVALID, "%s: null pointer", name);
  if (fp8 && (!k_scale || !v_scale)) return fail(NPD_E_INVALID, "%s: null scale pointer", name);
  const uintptr_t cache_align = fp8 ? 7u : 15u;   // FP8 chunks are 8 bytes
  if (!aligned16(query) || (reinterpret_cast<uintptr_t>(key_cache) & cache_align) != 0 ||
      (reinterpret_cast<uintptr_t>(value_cache) & cache_align) != 0 ||
      (reinterpret_cast<uintptr_t>(out) & 7u) != 0)
    return fail(NPD_E_ALIGN, "%s: query pointer must be 16-byte aligned, caches %d-byte, out 8-byte",
                name, fp8 ? 8 : 16);
  if (generic) {
    const int64_t tiles = (max_q_len + 63) / 64;
    const int64_t grid = (num_seqs * num_kv_heads + 7) / 8 * 8 * tiles * g;
    if (grid > INT32_MAX) return fail(NPD_E_INVALID, "%s: too many tiles", name);
    PrefillArgs a{};
    a.out = static_cast<uint16_t*>(out);
    a.q = static_cast<const uint16_t*>(query);
    a.k_cache = static_cast<const u32x4*>(key_cache);
    a.v_cache = static_cast<const u32x4*>(value_cache);
    a.block_tables = block_tables;
    a.cu_seqlens_q = cu_seqlens_q;
    a.context_lens = context_lens;
    a.k_scale = k_scale;
    a.v_scale = v_scale;
    a.num_seqs = (int)num_seqs;
    a.num_kv_heads = (int)num_kv_heads;
    a.group = (int)g;
    a.block_size = (int)block_size;
    a.bs_shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctzll((unsigned long long)block_size) : -1;
    a.num_blocks = (int)num_blocks;
    a.max_bps = (int)max_blocks_per_seq;
    a.tiles_max = (int)tiles;
    a.scale_log2 = scale * kLog2e;
    a.q_stride_token = q_stride_token;
    a.q_stride_head = q_stride_head;
    a.out_stride_token = out_stride_token;
    a.out_stride_head = out_stride_head;
    hipStream_t st = as_stream(stream);
    if (dtype == NPD_DTYPE_BF16)
      return fp8 ? launch_generic<BF16, true>(head_dim, a, grid, st, name)
                 : launch_generic<BF16, false>(head_dim, a, grid, st, name);
    return fp8 ? launch_generic<F16, true>(head_dim, a, grid, st, name)
               : launch_generic<F16, false>(head_dim, a, grid, st, name);
  }
  const Layout L = head_dim == 256 ? Layout{1, 1 << 30, 0, 0, 0}
                                   : prefill_layout(num_seqs, num_heads, head_dim, max_q_len, max_context_len);
  if (L.total > 0) {
    if (!workspace || workspace_bytes < L.total)
      return fail(NPD_E_WORKSPACE, "%s: workspace of %lld bytes needed, %lld given", name,
                  (long long)L.total, (long long)workspace_bytes);
    if ((reinterpret_cast<uintptr_t>(workspace) & 255u) != 0)
      return fail(NPD_E_ALIGN, "%s: workspace must be 256-byte aligned", name);
  }
  if (max_q_len * g > INT32_MAX - 256)
    return fail(NPD_E_INVALID, "%s: too many query rows", name);
  // most tiles of tr rows there can be (a chunk's last one may be part full)
  auto tiles_of = [&](int64_t tr) {
    const int64_t by_max = num_seqs * ((max_q_len * g + tr - 1) / tr), by_rows = total_q * g / tr + num_seqs;
    return by_max < by_rows ? by_max : by_rows;
  };
  // Tiles of 256 rows (8 waves, two per SIMD: one's softmax under the other's
  // MFMAs), or of 128 (4 waves): at head dim 256, whose accumulators and
  // queries need more than the 256 registers of two waves per SIMD (4 / 8
  // waves: two chunks of 4096 tokens 425 / 463 us, 500 tokens 35 / 64 us), and
  // at 128 where the 256-row tiles take half the compute units at most (500
  // tokens of 32 / 8 heads 23.4 / 25.9 us, 64 on a prefix of 6000 43.0 / 50.8).
  // Head dim 64 gains nothing from it (17.9 / 18.1 us).
  const bool few = tiles_of(tile_rows(8)) * num_kv_heads * 2 <= device_cus();
  const int waves = head_dim == 256 || (head_dim == 128 && few) ? 4 : 8;
  const int64_t tr = tile_rows(waves);
  const int64_t tiles = (max_q_len * g + tr - 1) / tr;
  if (L.total > 0 && num_seqs * tiles * num_kv_heads > kMaxCounters)
    return fail(NPD_E_INVALID, "%s: too many query tiles for the %lld merge counters", name,
                (long long)kMaxCounters);
  // Whether the longest context there can be outlasts the mean load of a
  // compute unit, as far as the host can tell: total_q rows make no fewer than
  // `rows` tiles, whose steps are least where all chunks are alike and without
  // a prefix.
  const int kt = kKT;
  const int64_t longest = (max_context_len + kt - 1) / kt, rows = total_q * g / tr;
  const bool tail = (longest + kItemSteps) * device_cus() >
                    rows * num_kv_heads * (kItemSteps + total_q / num_seqs / (2 * kt));
  // Up to kListTiles (sequence, tile) pairs the kernel cuts key ranges by the
  // work it finds. More run whole, in a fixed order, unless they leave compute
  // units idle (many short chunks on long prefixes) or one may end the launch
  // by itself. Then a part there is not costs an empty workgroup of 1 us, so
  // these are at most kFixedSplits (32 / 8 heads, whole / 2 / 4 / 8 parts: 700
  // chunks of 60 tokens and one of 256 on a prefix of 32512 1625 / 1358 / 1340 /
  // 1509 us, 16 of 2048 and one of 64 on 131072 3302 / 1941 / 1309 / 1169, 40 of
  // 100 and one of 2048 on 30000, whose tiles fill the chip whole, 952 / 979 /
  // 1024 / 1148).
  // Three rounds or more of tiles that cannot be cut and are nearly all there
  // need no list either, which costs an item 2 us and more (16 chunks of 512
  // tokens of 32 / 8 heads 150 us by the list, 130 in the fixed order; 300 of 60
  // tokens 246, 206; 4 of 2048 169, 160).
  const bool even = L.splits == 1 && num_seqs * tiles * num_kv_heads >= 3LL * device_cus() &&
                    4 * num_seqs * tiles <= 5 * rows;
  const bool list = num_seqs * tiles <= kListTiles && !even;
  const bool full = !list && total_q * num_heads >= 2LL * device_cus() * tr;
  const int splits = !full ? L.splits : !tail ? 1 : L.splits < kFixedSplits ? L.splits : kFixedSplits;
  const int ks_steps = splits == L.splits ? L.ks_steps : (int)((longest + splits - 1) / splits);
  // Grid: the tiles there can be, or two rounds of the compute units where the
  // kernel may cut that many parts; a workgroup without an item ends after the
  // work list. Where one of several sequences may outlast the others, its parts
  // have a further round (parts no shorter than the mean load are no more; with
  // two or three rounds of room the greedy schedules of 400 random skewed
  // batches end no sooner).
  const int64_t whole_tiles = tiles_of(tr);
  const int64_t round = (device_cus() + num_kv_heads - 1) / num_kv_heads;
  const int64_t two_rounds = (2LL * device_cus() + num_kv_heads - 1) / num_kv_heads;
  const int64_t even_items = !list ? splits * num_seqs * tiles
                             : splits > 1 && whole_tiles < two_rounds ? two_rounds : whole_tiles;
  const int64_t max_items = list && tail && splits > 1 && num_seqs > 1 && whole_tiles + round > even_items
                                ? whole_tiles + round : even_items;
  const int64_t grid = max_items * num_kv_heads;
  if (grid > INT32_MAX) return fail(NPD_E_INVALID, "%s: too many tiles", name);

  PrefillArgs a;
  a.out = static_cast<uint16_t*>(out);
  a.q = static_cast<const uint16_t*>(query);
  a.k_cache = static_cast<const u32x4*>(key_cache);
  a.v_cache = static_cast<const u32x4*>(value_cache);
  a.block_tables = block_tables;
  a.cu_seqlens_q = cu_seqlens_q;
  a.context_lens = context_lens;
  char* ws = static_cast<char*>(workspace);
  a.counters = L.total > 0 ? reinterpret_cast<int*>(ws) : nullptr;
  a.part_o = L.total > 0 ? reinterpret_cast<float*>(ws + L.o_off) : nullptr;
  a.part_ml = L.total > 0 ? reinterpret_cast<float*>(ws + L.ml_off) : nullptr;
  a.k_scale = k_scale;
  a.v_scale = v_scale;
  a.num_seqs = (int)num_seqs;
  a.num_kv_heads = (int)num_kv_heads;
  a.group = (int)g;
  a.block_size = (int)block_size;
  a.bs_shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctzll((unsigned long long)block_size) : -1;
  a.num_blocks = (int)num_blocks;
  a.max_bps = (int)max_blocks_per_seq;
  a.tiles_max = (int)tiles;
  a.subtiles = (int)(tiles * waves);
  a.splits_max = splits;
  a.ks_steps = ks_steps;
  a.list = list;
  a.max_items = (int)max_items;
  a.even_items = (int)even_items;
  a.num_cus = device_cus();
  a.scale_log2 = scale * kLog2e;
  a.q_stride_token = q_stride_token;
  a.q_stride_head = q_stride_head;
  a.out_stride_token = out_stride_token;
  a.out_stride_head = out_stride_head;
  hipStream_t st = as_stream(stream);
  const int64_t elt = fp8 ? 1 : 2;
  const bool off32 = num_blocks * num_kv_heads * block_size * head_dim * elt <= (int64_t)UINT32_MAX;
  if (dtype == NPD_DTYPE_BF16)
    return fp8 ? launch_dt<BF16, true>(head_dim, waves, off32, a, grid, st, name)
               : launch_dt<BF16, false>(head_dim, waves, off32, a, grid, st, name);
  return fp8 ? launch_dt<F16, true>(head_dim, waves, off32, a, grid, st, name)
             : launch_dt<F16, false>(head_dim, waves, off32, a, grid, st, name);
}

}  // namespace

extern "C" int npd_paged_prefill_attention(
    void* out, const void* query, const void* key_cache, const void* value_cache,
    const int32_t* block_tables, const int32_t* cu_seqlens_q, const int32_t* context_lens,
    int64_t num_seqs, int64_t total_q, int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
    int64_t num_blocks, int64_t block_size, int64_t max_blocks_per_seq, int64_t max_q_len,
    int64_t max_context_len, float scale, int64_t q_stride_token, int64_t q_stride_head,
    int64_t out_stride_token, int64_t out_stride_head, void* workspace, int64_t workspace_bytes,
    int32_t dtype, void* stream) {
  return prefill_impl(out, query, key_cache, value_cache, block_tables, cu_seqlens_q,
                      context_lens, nullptr, nullptr, num_seqs, total_q, num_heads, num_kv_heads,
                      head_dim, num_blocks, block_size, max_blocks_per_seq, max_q_len,
                      max_context_len, scale, q_stride_token, q_stride_head, out_stride_token,
                      out_stride_head, workspace, workspace_bytes, dtype, stream, false,
                      "npd_paged_prefill_attention");
}

extern "C" int npd_paged_prefill_attention_fp8(
    void* out, const void* query, const void* key_cache, const void* value_cache,
    const int32_t* block_tables, const int32_t* cu_seqlens_q, const int32_t* context_lens,
    const float* k_scale, const float* v_scale, int64_t num_seqs, int64_t total_q,
    int64_t num_heads, int64_t num_kv_heads, int64_t head_dim, int64_t num_blocks,
    int64_t block_size, int64_t max_blocks_per_seq, int64_t max_q_len, int64_t max_context_len,
    float scale, int64_t q_stride_token, int64_t q_stride_head, int64_t out_stride_token,
    int64_t out_stride_head, void* workspace, int64_t workspace_bytes, int32_t dtype,
    void* stream) {
  return prefill_impl(out, query, key_cache, value_cache, block_tables, cu_seqlens_q,
                      context_lens, k_scale, v_scale, num_seqs, total_q, num_heads, num_kv_heads,
                      head_dim, num_blocks, block_size, max_blocks_per_seq, max_q_len,
                      max_context_len, scale, q_stride_token, q_stride_head, out_stride_token,
                      out_stride_head, workspace, workspace_bytes, dtype, stream, true,
                      "npd_paged_prefill_attention_fp8");
}
