// What the attention kernels share: launch parameters, operand types, conversions to the attention's
// 16-bit type, the matrix instruction, the key order of its rows.
#pragma once
#include "varq_common.h"

namespace varq_attn {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16_t;
typedef __attribute__((__vector_size__(4 * sizeof(u32)))) u32 u32x4_t;

constexpr float kLog2e = 1.4426950408889634f;
constexpr int BN = 64;   // keys per tile

constexpr int kMaxSegments = 16;
constexpr int kMaxSplits_v = 8;        // shares of a query block's keys in the general kernel
constexpr int kMaxKeyShares_v = 64;    // ... and in the kernel for few queries

struct AttnParams {
  const __bf16 *q;
  __bf16 *out;
  const u32 *k_words, *v_words;
  const float *k_scale, *k_zp, *v_scale, *v_zp;
  // per-(head, channel) quantization (CHAN kernels): fp32 [Hkv, D] tables shared by all
  // tokens and batch entries; the per-key pointers above are unused then
  const float *k_chan_scale, *k_chan_zp, *v_chan_scale, *v_chan_zp;
  // the tables may change along the keys: keys [seg_end[s-1], seg_end[s]) use table s
  // (fp32 [nseg, Hkv, D]); this is a cache that was quantized step by step
  int nseg;
  int seg_end[kMaxSegments];
  const int32_t *head_map;
  const int32_t *kv_limit;
  int B, Hq, Hkv, Lq, Lk, Lstride;
  int q_tiles, bh_total;
  float scale_log2e;
  // the keys of a query block may be shared out over nsplit workgroups; each leaves its
  // normalized output (fp32 [nsplit][B*Hkv*Lq][D]) and softmax statistics (reference,
  // denominator: fp32 [nsplit][B*Hkv*Lq][2]) for the combining kernel.  nsplit = 1: no
  // workspace, the output is written directly.
  int nsplit;
  float *ws_o, *ws_ml;
  // the caller asked for exact codes in the MFMA operands where such a kernel exists (host side only)
  int exact_codes;
  int k_shift, v_shift;   // log2 of the channels per scale group (fused_attn.hip)
  int f16;   // q, out and the MFMA operands are fp16 (host side only: it selects the instantiation)
  int fq_share_blocks;   // few-queries kernel: 32-key blocks per share of the keys
  int key_waves;         // fused_attn.hip: wavefronts that share a block of 32 queries, 1, 2 or 4 (host side only)
  int few_waves;         // ... and wavefronts of a workgroup, 4 or 8 (host side only)
  // memory layout, in rows (a row = the D values of one token of one head):
  // q row = b*q_bs + h*q_hs + i*q_ts, out row likewise with o_*, key row = b*kv_bs + slot*kv_hs + j*kv_ts.
  // BHLc: (H*L, L, 1); BLHc (the layout of the flash-attention call): (L*H, 1, H).
  int64_t q_bs, q_hs, q_ts, o_bs, o_hs, o_ts, kv_bs, kv_hs, kv_ts;
};

// above 64 KiB of LDS the limit has to be raised, once per device the process launches on
inline void allow_lds(const void *kernel, int bytes, bool (&configured)[64]) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
  if (dev >= 0 && configured[dev]) return;
  (void)hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (dev >= 0) configured[dev] = true;
}

__device__ __forceinline__ u32 pack_bf16_rne(float lo, float hi) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  typedef float f2 __attribute__((ext_vector_type(2)));
  f2 v = {lo, hi};
  bf2 b = __builtin_convertvector(v, bf2);
  return __builtin_bit_cast(u32, b);
}
__device__ __forceinline__ u32 pack_f16_rne(float lo, float hi) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  typedef float f2 __attribute__((ext_vector_type(2)));
  f2 v = {lo, hi};
  h2 b = __builtin_convertvector(v, h2);
  return __builtin_bit_cast(u32, b);
}
// two fp32 values rounded to nearest-even into a pair of the attention's 16-bit type
template <bool F16> __device__ __forceinline__ u32 pack_io_rne(float lo, float hi) {
  if constexpr (F16) return pack_f16_rne(lo, hi);
  else return pack_bf16_rne(lo, hi);
}
// D (32x32 fp32) += A (32x16) B (16x32), operands in the attention's 16-bit type
template <bool F16> __device__ __forceinline__ floatx16_t mfma_32x32x16(u32x4_t a, u32x4_t b, floatx16_t c) {
  if constexpr (F16) {
    typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
}
// sum[0..3] += this lane's four numbers of w, on the matrix pipe: of the sixteen 4 x 4 products of the instruction, each with four contraction
// steps, lane l holds column l % 4 of product l / 4, so ones in the place of A add up a lane's own four numbers.
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
template <bool F16> __device__ __forceinline__ f32x4_t add4(f32x4_t sum, uint2 w) {
  if constexpr (F16) {
    typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_4x4x4f16(f16x4_t{1, 1, 1, 1}, __builtin_bit_cast(f16x4_t, w), sum, 0, 0, 0);
  } else {
    typedef short s16x4_t __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(s16x4_t{0x3f80, 0x3f80, 0x3f80, 0x3f80}, __builtin_bit_cast(s16x4_t, w), sum, 0, 0, 0);
  }
}
// The sum of a lane's weights of 8 keys as rounded for the matrix product.  v_dot2, a pair at a time, runs on the matrix pipe too and keeps it from
// the products beside it for 17 cycles; this takes 8 for four numbers.  4096 queries x 10521 keys, 32 pairs, D=128, with the quantizer and the
// expansion 625-637 -> 613-619 us; 13 scales of 128 pairs 4550 -> 4480-4515.
template <bool F16> __device__ __forceinline__ float sum_weights(u32x4_t w) {
  return add4<F16>(add4<F16>(f32x4_t{0.f, 0.f, 0.f, 0.f}, make_uint2(w[0], w[1])), make_uint2(w[2], w[3]))[0];
}
// The smallest or largest of the values of a wavefront's first ROWS rows of 16 lanes (the other rows hold copies), the same for all lanes.
template <bool IS_MAX, int ROWS> __device__ __forceinline__ int wave_fold(int v) {
  auto op = [](int a, int b) { return IS_MAX ? max(a, b) : min(a, b); };
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0xb1, 0xf, 0xf, false));    // quad_perm:[1,0,3,2]
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x4e, 0xf, 0xf, false));    // quad_perm:[2,3,0,1]
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xf, 0xf, false));   // row_half_mirror
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xf, 0xf, false));   // row_mirror
  int r = __builtin_amdgcn_readlane(v, 0);
#pragma unroll
  for (int i = 1; i < ROWS; ++i) r = op(r, __builtin_amdgcn_readlane(v, 16 * i));
  return r;
}
// The largest key limit of the N queries from row `first` on.  Every wavefront looks at all of them: as an atomic maximum in LDS, which takes the
// lanes one at a time, and two barriers, this was 7 000 to 10 000 of the 58 000 cycles of a workgroup that attends 680 keys (a whole
// sequence of 680 tokens under the block-causal rule, [8,680,16,64]: append and attention 40.3 -> 37.1 us).
template <int N> __device__ __forceinline__ int block_limit(const int32_t *kv_limit, int first, int Lq, int Lk) {
  static_assert(N % 64 == 0, "whole wavefronts");
  int m = 0;
#pragma unroll
  for (int i = 0; i < N / 64; ++i) {
    const int row = first + i * 64 + (int)(threadIdx.x & 63), limit = kv_limit[min(row, Lq - 1)];   // (past the end: the last row's again)
    m = max(m, min(limit, Lk));
  }
  return wave_fold<true, 4>(m);
}
// MFMA row r (0..31) of the S^T block carries key kperm(r) of the 32-key block
// (bits 2 and 3 of r swapped), so accumulator register i of a lane in half h
// holds key 16*(i/8) + 8*h + i%8.
__device__ __forceinline__ int kperm(int r) { return (r & 0x13) | ((r & 4) << 1) | ((r & 8) >> 1); }

// Workgroup `slot` of an XCD that has `groups` (batch, head) pairs of q_tiles query tiles, under a key limit that grows
// with the query (the block-causal rule), which makes the query tiles of a pair differ in length: windows of `win` pairs
// one after the other, in a window the last query tiles of all its pairs first, so that the short ones even out what is left.
struct HeavyFirst {
  int grp, qt;
  __device__ __forceinline__ HeavyFirst(int slot, int q_tiles, int groups, int win) {
    const int first = slot / (win * q_tiles) * win, n = min(win, groups - first);
    const int r = slot - first * q_tiles;
    qt = q_tiles - 1 - r / n;
    grp = first + r % n;
  }
};

// A cache whose heads have several bit-widths, all classes in one launch: pair k of the launch belongs to the
// class that its range falls in (8-bit codes first: the longest workgroups start first), and the workgroup
// runs that class's code.  The registers and the LDS are those of the most demanding class, which is no
// more than each class takes alone (see launch_shape); what is gained are the launches -- and that the
// classes, which have a few heads each, fill the device together.  Three widths, one launch per class ->
// one launch, us: [2,16,128] 100 queries x 600 keys 66 -> 18, [8,16,128] 256 x 500 78 -> 28, 576 x 1497 140 ->
// 117, 1024 x 2521 230 -> 200 (the last two with a stream for each class).
struct ClassParams {
  const u32 *k_words, *v_words;
  const float *k_scale, *k_zp, *v_scale, *v_zp;
  const int32_t *head_map;
  int heads, first;   // packed heads of the class; its first pair of the launch
};
struct ClassTable { ClassParams c[3]; };   // of 8, 4 and 2 bits; a width that the cache does not have has no heads
__device__ __forceinline__ void enter_class(AttnParams &p, const ClassParams &c) {
  p.k_words = c.k_words; p.v_words = c.v_words;
  p.k_scale = c.k_scale; p.k_zp = c.k_zp; p.v_scale = c.v_scale; p.v_zp = c.v_zp;
  p.head_map = c.head_map;
  p.Hkv = c.heads;
  p.kv_bs = (int64_t)c.heads * p.Lstride;
}
// F(bits, pair within the class, pair of the output) for the class of pair k
template <class F> __device__ __forceinline__ void in_class(AttnParams &p, const ClassTable &t, int k, F &&f) {
  const int H = p.Hq;
  auto run = [&](auto bits, const ClassParams &c) __attribute__((always_inline)) {
    enter_class(p, c);
    const int bh = k - c.first;
    f(bits, bh, bh / c.heads * H + c.head_map[bh % c.heads]);
  };
  if (k < t.c[1].first) run(std::integral_constant<int, 8>{}, t.c[0]);
  else if (k < t.c[2].first) run(std::integral_constant<int, 4>{}, t.c[1]);
  else run(std::integral_constant<int, 2>{}, t.c[2]);
}

// ---- few queries (few_attn.hip) ----
constexpr int kFewBlock = 32;   // keys per block
constexpr int kFewGroups = 2;   // scale groups of a row, at most
// p.q_tiles: tiles of 32 queries (up to 16 queries are one of 16); p.nsplit, p.fq_share_blocks, p.ws_*: the shares of the keys
void launch_few(const AttnParams &p, int D, int bits, int k_group, int v_group, hipStream_t st);
void launch_few_classes(const AttnParams &p, int D, const ClassTable &t, int group, hipStream_t st);

// ---- the wide path (wide_attn.hip): K and V expanded once, then attended by many query blocks ----
struct WidePlan {
  int waves;            // wavefronts of a workgroup: 8 (blocks of 256 queries) or 4 (128)
  int n_wgs, rounds;    // workgroups of the attention kernel; blocks that each of them takes whole
  size_t tile_bytes;    // the expanded tiles, at the start of the workspace
  size_t ws_bytes;      // ... and the partial results behind them
};
// Whether a launch takes workgroups of four wavefronts.
bool wide_four(int64_t bh, int Lq, int Lk, int D, int cus, bool limits);
// share: whether blocks may be shared out; limits: whether the queries have key limits
WidePlan plan_wide(int64_t bh, int Lq, int Lk, int D, int cus, bool share, bool limits);
// Expands the packed cache of p (per-key groups of k_group / v_group channels, or the per-channel
// tables) into `tiles`, pair after pair.
void launch_expand(const AttnParams &p, int D, int bits, int k_group, int v_group, bool chan, char *tiles, hipStream_t st);
// ... and a cache whose heads have several bit-widths, every class to the places of its heads among the p.Hq heads of the cache.
void launch_expand_classes(const AttnParams &p, int D, const ClassTable &t, int group, char *tiles, hipStream_t st);
// Attends the expanded tiles at the start of `ws`.
void launch_wide(const AttnParams &p, int D, const WidePlan &plan, char *ws, hipStream_t st);

}  // namespace varq_attn
