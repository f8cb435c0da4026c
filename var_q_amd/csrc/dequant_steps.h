// Dequantizing the cache of a stepwise quantizer: shared by the launch that does only that (dequant.hip) and the
// one that quantizes a step as well (quant_general.hip).
#pragma once
#include "varq_common.h"

namespace varq_deq {

typedef u32 u32x4 __attribute__((ext_vector_type(4)));

template <bool STREAM, class T> __device__ __forceinline__ void put(T *at, T v) {
  if constexpr (STREAM) __builtin_nontemporal_store(v, at);
  else *at = v;
}
// STREAM: past the caches (whole octets only)
template <int ODT, bool STREAM = false> __device__ __forceinline__ void store8(void *out, int64_t elem, const float (&f)[8], int n_valid) {
  if (ODT == VARQ_F32) {
    float *o = reinterpret_cast<float *>(out) + elem;
    if (n_valid == 8) {
      reinterpret_cast<float4 *>(o)[0] = make_float4(f[0], f[1], f[2], f[3]);
      reinterpret_cast<float4 *>(o)[1] = make_float4(f[4], f[5], f[6], f[7]);
    } else {
      for (int j = 0; j < n_valid; ++j) o[j] = f[j];
    }
  } else {
    uint16_t *o = reinterpret_cast<uint16_t *>(out) + elem;
    if (ODT == VARQ_BF16 && n_valid == 8) {
      // hardware round-to-nearest-even conversion, two values per instruction
      typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
      typedef float f2 __attribute__((ext_vector_type(2)));
      u32 w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f2 v = {f[2 * j], f[2 * j + 1]};
        w[j] = __builtin_bit_cast(u32, __builtin_convertvector(v, bf2));
      }
      put<STREAM>(reinterpret_cast<u32x4 *>(o), u32x4{w[0], w[1], w[2], w[3]});
      return;
    }
    uint16_t h[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) h[j] = (ODT == VARQ_BF16) ? f32_to_bf16_rne(f[j]) : f32_to_f16_rne(f[j]);
    if (n_valid == 8) {
      put<STREAM>(reinterpret_cast<u32x4 *>(o),
                  u32x4{h[0] | ((u32)h[1] << 16), h[2] | ((u32)h[3] << 16), h[4] | ((u32)h[5] << 16), h[6] | ((u32)h[7] << 16)});
    } else {
      for (int j = 0; j < n_valid; ++j) o[j] = h[j];
    }
  }
}

// The cache of a stepwise quantizer, one table of scales per step.  A pair is a (batch, head) (heads first)
// or a batch entry (tokens first); its tokens lie one after the other in words and output, `octs` octets each,
// so an octet's place is its number and only its table depends on the token.  HBM-bound by its output: per
// element 4 bytes (or 2) written and bits/8 read; the tables stay in the caches.  (Reading the scales
// expanded over the tokens instead, four more bytes per element, took 8.9 against 5.9 us at [8,680,30,64],
// and the expansion had to be written first.)
struct StepParams {
  const u32 *words;
  const float *scale, *zp;
  void *out;
  int64_t pair_words, pair_octs;   // words of a pair in the buffer, octets of a pair that are read
  int64_t out_pair_octs;           // octets of a pair in the output
  int octs, H, c, nseg;
  FastDiv by_octs;
  int head_in_pair;                // 1: heads first, the pair's head is pair % H
  int64_t row;                     // H * c: floats of a table
  int seg_oct[16];                 // first octet of a pair that is past segment s
};

// the step that octet o lies in (those past the last one end where the pair does)
__device__ __forceinline__ int step_of(const StepParams &p, int o) {
  int seg = 0;
#pragma unroll
  for (int s = 0; s < 15; ++s) seg += o >= p.seg_oct[s] ? 1 : 0;
  return seg;
}

// Block `block` of pair `pair`: NT threads, U octets each, all of whose loads are under way before the first is used.  (One octet after the other, each
// with its search for the step in LDS and a trip for its scales, a workgroup was a chain of some 4 us, and what the launches of
// a schedule took: [8,n,30,64], ten steps to fp32, 173 -> 169 us.)
template <int ODT, int BITS, int NT, int U>
__device__ __forceinline__ void dequant_steps_block(const StepParams &p, int64_t pair, int block) {
  const u32 *words = p.words + pair * p.pair_words;
  const float *scale = p.scale + (p.head_in_pair ? (pair % p.H) * p.c : 0);
  const float *zp = p.zp ? p.zp + (p.head_in_pair ? (pair % p.H) * p.c : 0) : nullptr;
  const int first = block * (NT * U), last = (int)p.pair_octs - 1, o0 = first + threadIdx.x;
  auto segment = [&](int o) __attribute__((always_inline)) { return step_of(p, o); };
  // most blocks lie in one step (with an octet per lane, looking for it comes to as much as for the octets')
  const int seg0 = U > 1 ? segment(first) : 0;
  const bool one_seg = U > 1 && seg0 == segment(min(first + NT * U - 1, last));
  u32 w0[U], w1[U];
  int64_t at[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int o = min(o0 + u * NT, last);
    w1[u] = 0;
    if (BITS == 8) { const uint2 t = *reinterpret_cast<const uint2 *>(words + 2 * (int64_t)o); w0[u] = t.x; w1[u] = t.y; }
    else if (BITS == 4) w0[u] = words[o];
    else w0[u] = words[o >> 1] >> ((o & 1) * 16);
    at[u] = seg0 * p.row + (int)((u32)o - p.by_octs((u32)o) * (u32)p.octs) * 8;
    if (!one_seg) at[u] += (segment(o) - seg0) * p.row;
  }
  float4 s[U][2], z[U][2];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s[u][h] = *reinterpret_cast<const float4 *>(scale + at[u] + 4 * h);
      if (zp) z[u][h] = *reinterpret_cast<const float4 *>(zp + at[u] + 4 * h);
    }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int o = o0 + u * NT;
    if (o > last) return;
    const float sv[8] = {s[u][0].x, s[u][0].y, s[u][0].z, s[u][0].w, s[u][1].x, s[u][1].y, s[u][1].z, s[u][1].w};
    float f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      f[j] = (float)(int)(BITS == 8 ? __builtin_amdgcn_sbfe((int)(j < 4 ? w0[u] : w1[u]), 8 * (j & 3), 8) : __builtin_amdgcn_sbfe((int)w0[u], BITS * j, BITS));
    if (zp) {
      const float zv[8] = {z[u][0].x, z[u][0].y, z[u][0].z, z[u][0].w, z[u][1].x, z[u][1].y, z[u][1].z, z[u][1].w};
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = (f[j] - zv[j]) * sv[j];
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = f[j] * sv[j];
    }
    store8<ODT>(p.out, (pair * p.out_pair_octs + o) * 8, f, 8);
  }
}

// The same to 32 bits, by pieces of 16 bytes: a wavefront stores 1 KiB with each, where an octet takes two stores 32 bytes apart.  All tokens of ten steps, in a
// graph, us, by octets / by pieces: [8,680,30,64] 8 bits 12.3 / 10.0, 4 bits affine 12.7 / 10.5, [32,30,680,64] 37.0 / 34.2, [2,16,680,128] 2 bits affine 6.5 both.  Beside workgroups
// that quantize, whose stores are octets by their groups, twice the loads cost more (the ten steps of [8,n,30,64] one by one 167.4 / 169.9).
template <int BITS, int NT, int U>
__device__ __forceinline__ void dequant_steps_halves(const StepParams &p, int64_t pair, int block) {
  constexpr int N = 2 * U;   // pieces of a lane
  typedef float f4 __attribute__((ext_vector_type(4)));
  const char *const words = reinterpret_cast<const char *>(p.words + pair * p.pair_words);
  const int64_t head = p.head_in_pair ? (pair % p.H) * p.c : 0;
  const float *const scale = p.scale + head, *const zp = p.zp ? p.zp + head : nullptr;
  const int first = block * (NT * U), last = (int)p.pair_octs - 1, o0 = first + (int)threadIdx.x / 2, half = threadIdx.x & 1;
  const int seg0 = U > 1 ? step_of(p, first) : 0;
  const bool one_seg = U > 1 && seg0 == step_of(p, min(first + NT * U - 1, last));
  u32 w[N];
  int64_t at[N];
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const int o = min(o0 + u * (NT / 2), last);
    const char *const src = words + ((int64_t)o * 2 + half) * (BITS / 2);
    if constexpr (BITS == 8) w[u] = *reinterpret_cast<const u32 *>(src);
    else if constexpr (BITS == 4) w[u] = *reinterpret_cast<const uint16_t *>(src);
    else w[u] = *reinterpret_cast<const unsigned char *>(src);
    at[u] = seg0 * p.row + (int)((u32)o - p.by_octs((u32)o) * (u32)p.octs) * 8 + half * 4;
    if (!one_seg) at[u] += (step_of(p, o) - seg0) * p.row;
  }
  f4 s[N], z[N];
#pragma unroll
  for (int u = 0; u < N; ++u) {
    s[u] = *reinterpret_cast<const f4 *>(scale + at[u]);
    if (zp) z[u] = *reinterpret_cast<const f4 *>(zp + at[u]);
  }
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const int o = o0 + u * (NT / 2);
    if (o > last) return;
    f4 f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float q = (float)(int)__builtin_amdgcn_sbfe((int)w[u], BITS * j, BITS);
      f[j] = zp ? (q - z[u][j]) * s[u][j] : q * s[u][j];
    }
    reinterpret_cast<f4 *>(p.out)[(pair * p.out_pair_octs + o) * 2 + half] = f;
  }
}

// The launch parameters for `nseg` steps that end at host_seg_end[..]; false where the octets of a pair exceed
// 31 bits or a dim the grid's 65535.  p.out_pair_octs is that of an output which holds these tokens and no others.
inline bool set_steps(StepParams &p, const int32_t *words, const float *scale, const float *zp, int nseg, const int32_t *host_seg_end, int B, int H,
                      int64_t capacity, int c, int bits, bool tokens_first, void *out) {
  if (B > 65535 || (!tokens_first && H > 65535)) return false;
  const int64_t tokens = nseg ? host_seg_end[nseg - 1] : 0;
  p.words = reinterpret_cast<const u32 *>(words); p.scale = scale; p.zp = zp; p.out = out;
  p.H = H; p.c = c; p.nseg = nseg; p.row = (int64_t)H * c;
  p.head_in_pair = tokens_first ? 0 : 1;
  p.octs = (tokens_first ? H * c : c) / 8;
  p.by_octs = FastDiv::by(p.octs);
  if (tokens * p.octs >= (1ll << 31) - 2048) return false;
  for (int s = 0; s < 16; ++s) p.seg_oct[s] = (s < nseg ? host_seg_end[s] : (int)tokens) * p.octs;
  p.pair_octs = p.out_pair_octs = tokens * p.octs;
  p.pair_words = capacity * p.octs * 8 * bits / 32;
  return true;
}

}  // namespace varq_deq
