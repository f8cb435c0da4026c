// Attention of few queries over a packed cache: reading the cache and dequantizing it once is the work.
//
// The kernels for many queries (fused_attn.hip, wide_attn.hip) have workgroups of 256 queries; with a few dozen they
// leave most of their wavefronts without queries and spend barriers per key tile on the rest.  Here all wavefronts of a
// workgroup serve the SAME 16 * NQC queries, and each takes its own blocks of 32 keys of the workgroup's share: from global
// memory to registers to the matrix instructions, nothing shared between wavefronts inside the key loop, no barrier in
// it, and no way through LDS for K or V:
//  * S^T = K Q^T with v_mfma_f32_16x16x32 (r = lane % 16, g = lane / 16): lane (r, g) dequantizes D / 4 channels of the
//    keys 8 (r / 4) + 4 t + r % 4, t = 0, 1, of the block.  The contraction does not mind the order of the channels, so a
//    lane takes D / 4 consecutive ones (one 16-byte load of a row of 4-bit codes at D = 128), and Q^T has them in that order;
//  * these rows leave the logits of the keys 8 g + 0..7 of query r in lane (r, g), which is what it has to hold of P^T as
//    the operand of O^T = V^T P^T;
//  * V^T: lane (r, g) loads the codes of its D / 16 consecutive channels of the keys 8 g + 0..7, so that it has the
//    eight keys of every one of its channels: matrix instruction m takes channel m of every lane.  Row r of its
//    result is channel (D / 16) r + m, and the order is undone at the end, when the wavefronts' results are put together.
// K and V enter the products as (code - zp) * scale in fp32 rounded to the attention's 16-bit type, the operands that
// the other kernels have -- but for V of a group whose zero-point is no whole number or beyond +-896: there (code - near) * scale is rounded,
// near the whole number within +-896 next to the zero-point, and (near - zp) * scale, the same for all channels of the group, is summed with the weights in
// fp32 and added to the result (another operand, nearer to the unrounded value).  Online softmax per lane against a reference that moves only when a weight would pass 2^16
// (2^15 in fp16).
// The wavefronts' partial results meet in LDS, the workgroups' shares of the keys in the workspace (combine_splits_kernel).
//
// What bounds it: 4-bit codes at D = 128 are 23 vector instructions per eight elements, 446 per block and wavefront with the
// softmax and the addresses (and 520 per wavefront around the loop), most of them of the classes that issue once in four cycles: the vector ALU is busy for 0.64 of
// the launch over [2,16,10521,128], 0.76 over four times as many keys; [7,8,41576,128], 2 queries: 73 us without the
// loads of the loop, 68 us without the dequantization, 91 us whole (335 MB, 3.7 TB/s; INT8 121 us, 5.2 TB/s).  The kernel that this one replaced (32
// queries to a wavefront, V transposed through LDS, one scale group at D = 128 only) took 140 and 167 us.  [2,16,10521,128], 16 queries, with the
// launch that combines the shares: 25.4 -> 20.6 us over one cache again and again, out of the Infinity Cache, 26.2 -> 21.9 over 24 in turn, out of HBM; D = 64, [15,30,5049,64] 2-bit in groups of 32, 28 queries, on the kernel for many queries: 123 -> 62.
#include <type_traits>

#include "attn_common.h"

using namespace varq_attn;

namespace {

constexpr int BK = kFewBlock;
// Wavefronts of a SIMD, for the registers
template <int D, int NQC, int NW> constexpr int kWaves = NW == 8 ? 2 : D == 128 ? (NQC == 1 ? 3 : 2) : (NQC == 1 ? 4 : 3);

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
template <bool F16> __device__ __forceinline__ f32x4_t mfma_16x16x32(u32x4_t a, u32x4_t b, f32x4_t c) {
  if constexpr (F16) {
    typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
}

// How a code becomes a value.  The 10 low bits of 1024 in fp16 count ones, so code + kHalf (kHalf = 2^(BITS - 1)) or'ed into
// them makes a number of two codes at once; a packed fp16 addition of kZero - zp, kZero = -1024 - kHalf, leaves
// code - zp, and v_fma_mix_f32 takes its fp16 halves as they are: (code - zp) * scale with one rounding, the product that
// the reference rounds (VAR_Q/quant.py:123-124).  About three instructions per element with the rounding to the attention's type.
// (Bytes through v_cvt_f32_ubyte, a subtraction and a product are four, and the kernel is bound by their number.)
// fp16 holds the integers up to 2048, so zero-points are split: what is beyond +-896 and the fraction, times the scale, is
// `rest`.  K's rides on the fma (a product of a code and a scale plus 0 is that product); V's, the same for all channels of a
// group, is summed with the weights on the side, in blocks that have one that is not 0.
struct GroupScales {
  float scale[BK], rest[BK];   // rest: -scale * (zp - what `zero` holds of it)
  _Float16 zero[BK];
};
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
template <int BITS> struct Codes {
  static constexpr u32 kHalf = 1u << (BITS - 1), kField = (1u << BITS) - 1u;
  // two codes of w, in bits i * BITS.. of its halves (8 bits: its bytes 2 i and 2 i + 1), as 1024 + kHalf + code
  __device__ static __forceinline__ u32 pair(u32 w, int i) {
    if constexpr (BITS == 8) return __builtin_amdgcn_perm(0x64646464u, w, i ? 0x04030402u : 0x04010400u) ^ (kHalf * 0x10001u);
    else return ((w >> (BITS * i)) & (kField * 0x10001u)) ^ (0x64006400u + kHalf * 0x10001u);
  }
  __device__ static __forceinline__ f16x2_t number(u32 pair, f16x2_t zero) { return __builtin_bit_cast(f16x2_t, pair) + zero; }
};

template <int D, int NG, int NQC, int NW> struct FewLds {
  static constexpr bool kQ = D * NQC > 128;                            // Q^T in LDS (registers: a wavefront per SIMD more)
  static constexpr int kWave = 2 * NG * (int)sizeof(GroupScales);     // [K, V][scale groups of a row]: the scales of a block
  static constexpr int kQat = NW * kWave;                             // Q^T: [NQC][D / 32][64 lanes] 16 bytes
  static constexpr int kSlots = NW * D * 16 * 4;                      // the wavefronts' accumulators of 16 queries (after the key loop)
  static constexpr int kMl = kSlots;
  static constexpr int kBytes = kMl + NW * NQC * 16 * 8;              // [NW][NQC * 16 queries] reference and denominator
  static_assert(kQat + (kQ ? NQC * (D / 32) * 1024 : 0) <= kSlots, "the key loop's part lies under the accumulators");
};

// The channels of a lane's slice of a K row, in the order in which they become operands: the slot s of chunk c
template <int BITS> __host__ __device__ constexpr int k_channel(int c, int s) {
  if (BITS == 8) return 8 * c + s;
  if (BITS == 4) return 8 * c + s / 2 + 4 * (s % 2);
  return 16 * (c / 2) + 4 * (c % 2) + s / 2 + 8 * (s % 2);
}

template <int D, int BITS, int NG, int NQC, int NW, bool F16>
__device__ __forceinline__ void attend_few(const AttnParams &p, int k_shift, int v_shift, int bh, int out_pair, int qt, int split) {
  constexpr int WPR = D * BITS / 32, NCH = D / 32, NT = D / 16;
  constexpr int KW = WPR / 4;                            // words of a lane's quarter of a K row
  constexpr int VB = NT * BITS;                          // bits of a lane's NT channels of a V row
  constexpr int VW = VB >= 32 ? VB / 32 : 1;
  using Lds = FewLds<D, NG, NQC, NW>;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, quarter = lane >> 4;
  GroupScales *const par = reinterpret_cast<GroupScales *>(lds_raw + wave * Lds::kWave);   // [K, V][NG]
  float2 *const lds_ml = reinterpret_cast<float2 *>(lds_raw + Lds::kMl);             // [NW][NQC * 16]

  const int b = bh / p.Hkv, hs = bh % p.Hkv;
  const int hq = p.head_map ? p.head_map[hs] : hs;

  int limit[NQC], qrow[NQC];
  int kv_end = 0, minlim = p.Lk;
#pragma unroll
  for (int n = 0; n < NQC; ++n) {
    qrow[n] = (qt * NQC + n) * 16 + r16;
    limit[n] = p.kv_limit ? max(min(p.kv_limit[min(qrow[n], p.Lq - 1)], p.Lk), 0) : p.Lk;
    if (qrow[n] < p.Lq) { kv_end = max(kv_end, limit[n]); minlim = min(minlim, limit[n]); }
  }
  // (every wavefront holds the same queries, and every quarter of it: the largest and the smallest limit need no exchange between them)
  if (p.kv_limit) {
    kv_end = wave_fold<true, 1>(kv_end);
    minlim = wave_fold<false, 1>(minlim);
  } else {
    kv_end = p.Lk; minlim = p.Lk;
  }
  // the share's blocks: a fixed number per share (set by the host from Lk), cut at the queries' last key
  const int nb = (kv_end + BK - 1) / BK;
  const int b_begin = split * p.fq_share_blocks, b_end = min(b_begin + p.fq_share_blocks, nb);
  // Block j of the share goes to wavefront (j + rot) % NW: the wavefront that gets the odd block more differs between
  // workgroups that are likely to sit on one compute unit.  (A function of the (batch, head) pair, the query tile and the
  // share only: the two cache layouts add up in the same order.)
  const int slot_s = ((bh >> 3) * p.q_tiles + qt) * p.nsplit + split;
  const int rot = (slot_s + (slot_s >> 5)) % NW;
  const int blk0 = b_begin + (wave + NW - rot) % NW;

  // Loads of a block: requested as soon as the registers of the block before are used up, about a block ahead of
  // their use, and without conditions around them (past the wavefront's last block they read that block's last row
  // again, and a missing zero-point array reads the scales): behind a branch the compiler no longer knows how many are in flight.
  // 32-bit byte offsets from uniform bases (the host checks that they fit).
  const int64_t kv_row0 = b * p.kv_bs + hs * p.kv_hs;
  const char *const kw_base = reinterpret_cast<const char *>(p.k_words + kv_row0 * WPR);
  const char *const vw_base = reinterpret_cast<const char *>(p.v_words + kv_row0 * WPR);
  const bool of_v = lane >= BK;   // the scales of key lane % 32: the lower half of the lanes K's, the upper half V's
  const int g_shift = of_v ? v_shift : k_shift, groups = D >> g_shift;
  const float *const sc = of_v ? p.v_scale : p.k_scale, *const zp = of_v ? p.v_zp : p.k_zp;
  const char *const s_base = reinterpret_cast<const char *>(sc + kv_row0 * groups);
  const char *const z_base = reinterpret_cast<const char *>((zp ? zp : sc) + kv_row0 * groups);
  const bool has_zp = zp != nullptr;
  const u32 row_b = (u32)p.kv_ts * (WPR * 4), par_b = (u32)p.kv_ts * 4 * groups;
  const int last_blk = blk0 + max(b_end - 1 - blk0, 0) / NW * NW;   // (this wavefront's last block, if it has any)
  const u32 last_key = (u32)min(last_blk * BK + BK - 1, p.Lk - 1);
  const u32 k_lane = quarter * (KW * 4), v_lane = r16 * VB / 32 * 4;
  // where a lane has 16 or 8 bits of a key: those of two keys' words, in the halves of one
  const u32 v_at = r16 * VB % 32 / 8, v_sel = VB == 16 ? v_at * 0x01010101u + 0x05040100u : v_at * 0x00010001u + 0x0c040c00u;
  // (offsets of the next block's rows, moved on and clamped; the products of key and stride once)
  const u32 row_step = NW * BK * row_b, par_step = NW * BK * par_b;
  const u32 k_last = last_key * row_b + k_lane, v_last = last_key * row_b + v_lane, p_last = last_key * par_b;
  u32 k_off = (blk0 * BK + 8 * (r16 >> 2) + (r16 & 3)) * row_b + k_lane, v_off = (blk0 * BK + 8 * quarter) * row_b + v_lane;
  u32 p_off = (blk0 * BK + (lane & (BK - 1))) * par_b;
  auto umin = [](u32 x, u32 y) { return x < y ? x : y; };
  u32 kraw[2][KW], vraw[8][VW];
  float sraw[NG], zraw[NG];
  auto request_p = [&]() {
    const u32 o = umin(p_off, p_last);
    p_off += par_step;
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      const u32 oi = o + 4 * min(i, groups - 1);   // (a group that the row does not have: its last one again)
      sraw[i] = *reinterpret_cast<const float *>(s_base + oi);
      zraw[i] = *reinterpret_cast<const float *>(z_base + oi);
    }
  };
  auto load_words = [](const char *src, auto &dst) __attribute__((always_inline)) {
    constexpr int N = sizeof(dst) / 4;
    if constexpr (N % 4 == 0) {
#pragma unroll
      for (int i = 0; i < N; i += 4) {
        const u32x4_t t = *reinterpret_cast<const u32x4_t *>(src + 4 * i);
        dst[i] = t[0]; dst[i + 1] = t[1]; dst[i + 2] = t[2]; dst[i + 3] = t[3];
      }
    } else if constexpr (N == 2) {
      const uint2 t = *reinterpret_cast<const uint2 *>(src);
      dst[0] = t.x; dst[1] = t.y;
    } else {
      dst[0] = *reinterpret_cast<const u32 *>(src);
    }
  };
  auto request_k = [&]() {
#pragma unroll
    for (int t = 0; t < 2; ++t) load_words(kw_base + umin(k_off + 4 * t * row_b, k_last), kraw[t]);
    k_off += row_step;
  };
  auto request_v = [&]() {
#pragma unroll
    for (int j = 0; j < 8; ++j) load_words(vw_base + umin(v_off + j * row_b, v_last), vraw[j]);
    v_off += row_step;
  };

  request_p();
  // ---- Q^T, in the order of the K operands ----
  u32x4_t qreg[NQC][NCH];
  u32x4_t *const q_lds = reinterpret_cast<u32x4_t *>(lds_raw + Lds::kQat);
#pragma unroll
  for (int n = 0; n < NQC; ++n) {
    if (Lds::kQ && wave != n) continue;   // (each wavefront has one column to put there)
    const __bf16 *qp = p.q + (b * p.q_bs + hq * p.q_hs + min(qrow[n], p.Lq - 1) * p.q_ts) * D + quarter * (D / 4);
    u32 raw[NCH * 4];
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const u32x4_t t = *reinterpret_cast<const u32x4_t *>(qp + c * 8);
      raw[4 * c] = t[0]; raw[4 * c + 1] = t[1]; raw[4 * c + 2] = t[2]; raw[4 * c + 3] = t[3];
    }
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      u32x4_t o;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c0 = k_channel<BITS>(c, 2 * i), c1 = k_channel<BITS>(c, 2 * i + 1);
        // channel c0 of the lane's below channel c1
        const u32 sel = (c0 & 1 ? 0x0302u : 0x0100u) | (c1 & 1 ? 0x07060000u : 0x05040000u);
        o[i] = __builtin_amdgcn_perm(raw[c1 >> 1], raw[c0 >> 1], sel);
      }
      if constexpr (Lds::kQ) q_lds[(n * NCH + c) * 64 + lane] = o;
      else qreg[n][c] = o;
    }
  }
  auto qop = [&](int n, int c) __attribute__((always_inline)) {
    if constexpr (Lds::kQ) return q_lds[(n * NCH + c) * 64 + lane];
    else return qreg[n][c];
  };
  request_k();
  request_v();
  if constexpr (Lds::kQ) __syncthreads();

  f32x4_t oacc[NT][NQC];
  float m_ref[NQC], l_part[NQC], v_rest[NG][NQC];   // v_rest: the sum of the weights times `rest`, by group
#pragma unroll
  for (int n = 0; n < NQC; ++n) {
    m_ref[n] = 0.f; l_part[n] = 0.f;
#pragma unroll
    for (int g = 0; g < NG; ++g) v_rest[g][n] = 0.f;
#pragma unroll
    for (int m = 0; m < NT; ++m) oacc[m][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  bool first = true;
  const int k_group = quarter * (D / 4) >> k_shift, v_group = r16 * NT >> v_shift;

  // One block of 32 keys.
  auto block = [&](const int blk, const bool rest) __attribute__((always_inline)) {
    const int t0 = blk * BK;

    // ---- S^T = K Q^T ----
    f32x4_t sacc[2][NQC];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int key = 8 * (r16 >> 2) + 4 * t + (r16 & 3);
      const float ks = par[k_group].scale[key], kc = par[k_group].rest[key];
      const _Float16 kz = par[k_group].zero[key];
#pragma unroll
      for (int n = 0; n < NQC; ++n) sacc[t][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        u32x4_t a;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          u32 pair;
          if constexpr (BITS == 8) pair = Codes<8>::pair(kraw[t][2 * c + i / 2], i % 2);
          else if constexpr (BITS == 4) pair = Codes<4>::pair(kraw[t][c], i);
          else pair = Codes<2>::pair(kraw[t][c / 2], 4 * (c % 2) + i);
          const f16x2_t x = Codes<BITS>::number(pair, f16x2_t{kz, kz});
          a[i] = pack_io_rne<F16>(__builtin_fmaf((float)x[0], ks, kc), __builtin_fmaf((float)x[1], ks, kc));
        }
#pragma unroll
        for (int n = 0; n < NQC; ++n) sacc[t][n] = mfma_16x16x32<F16>(a, qop(n, c), sacc[t][n]);
      }
    }
    request_k();

    // ---- softmax of the block: register i of half t is key t0 + 8 quarter + 4 t + i ----
    u32x4_t pop[NQC];
#pragma unroll
    for (int n = 0; n < NQC; ++n) {
      float z[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) z[i] = __builtin_fmaf(p.scale_log2e, sacc[i >> 2][n][i & 3], -m_ref[n]);
      if (t0 + BK > minlim) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (t0 + 8 * quarter + i >= limit[n]) z[i] = -INFINITY;
      }
      // Moves the reference to the row's current maximum: up only once something has been accumulated;
      // the first block takes its maximum as it is (the accumulators are zero).
      auto move_reference = [&]() {
        float zmax = z[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) zmax = fmaxf(zmax, z[i]);
        zmax = fmaxf(zmax, __shfl_xor(zmax, 16, 64));
        zmax = fmaxf(zmax, __shfl_xor(zmax, 32, 64));
        const float delta = first ? ((zmax == -INFINITY) ? 0.f : zmax) : fmaxf(zmax, 0.f);
        m_ref[n] += delta;
#pragma unroll
        for (int i = 0; i < 8; ++i) z[i] -= delta;
        if (!first) {
          const float alpha = __builtin_amdgcn_exp2f(-delta);
#pragma unroll
          for (int m = 0; m < NT; ++m) oacc[m][n] *= alpha;
          l_part[n] *= alpha;
#pragma unroll
          for (int g = 0; g < NG; ++g) v_rest[g][n] *= alpha;
        }
      };
      float bsum;
      auto weights = [&]() {
        bsum = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
          const u32 w = pack_io_rne<F16>(__builtin_amdgcn_exp2f(z[i]), __builtin_amdgcn_exp2f(z[i + 1]));
          pop[n][i >> 1] = w;
          // the sum grows by the weights as rounded for the matrix product
          if constexpr (F16) {
            typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
            bsum = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, w), __builtin_bit_cast(f16x2_t, 0x3c003c00u), bsum, false);
          } else {
            typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
            bsum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w), __builtin_bit_cast(bf16x2_t, 0x3f803f80u), bsum, false);
          }
        }
      };
      constexpr float kMoveAt = F16 ? 32768.f : 65536.f;
      if (first) move_reference();
      weights();
      if (!first && __any(!(bsum <= kMoveAt))) {
        move_reference();
        weights();
      }
      l_part[n] += bsum;
    }
    first = false;

    // ---- O^T += V^T P^T ----
    if (rest) {
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int n = 0; n < NQC; ++n)
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const u32 w = pop[n][j >> 1] >> (16 * (j & 1));
            const float weight = F16 ? (float)__builtin_bit_cast(_Float16, (uint16_t)w) : u2f(w << 16);
            v_rest[g][n] = __builtin_fmaf(weight, par[NG + g].rest[8 * quarter + j], v_rest[g][n]);
          }
    }
    float vs[8];
    f16x2_t vz[4];   // of two keys
    {
      const GroupScales &g = par[NG + v_group];
#pragma unroll
      for (int j = 0; j < 8; ++j) vs[j] = g.scale[8 * quarter + j];
#pragma unroll
      for (int j = 0; j < 4; ++j) vz[j] = reinterpret_cast<const f16x2_t *>(g.zero)[4 * quarter + j];
    }
    // the codes of keys j, j + 1 as pairs: of two channels of one key, or, where a lane has at most 16 bits of a key, of both keys
    auto values = [&](int j, u32 pair0, u32 pair1, int half0, int half1) __attribute__((always_inline)) {
      const f16x2_t x0 = __builtin_bit_cast(f16x2_t, pair0), x1 = __builtin_bit_cast(f16x2_t, pair1);
      return pack_io_rne<F16>(__builtin_fmaf((float)x0[half0], vs[j], 0.f), __builtin_fmaf((float)x1[half1], vs[j + 1], 0.f));
    };
    auto multiply = [&](int m, const u32x4_t &a) __attribute__((always_inline)) {
#pragma unroll
      for (int n = 0; n < NQC; ++n) oacc[m][n] = mfma_16x16x32<F16>(a, pop[n], oacc[m][n]);
    };
    if constexpr (VB >= 32) {
#pragma unroll
      for (int i = 0; i < NT / 2; ++i) {
        u32 pair[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const _Float16 z = vz[j >> 1][j & 1];
          const u32 raw = BITS == 8 ? Codes<8>::pair(vraw[j][i / 2], i % 2) : Codes<BITS>::pair(vraw[j][0], i);
          pair[j] = __builtin_bit_cast(u32, Codes<BITS>::number(raw, f16x2_t{z, z}));
        }
        if (i == NT / 2 - 1) request_v();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          u32x4_t a;
#pragma unroll
          for (int j = 0; j < 8; j += 2) a[j >> 1] = values(j, pair[j], pair[j + 1], h, h);
          multiply(BITS == 8 ? 2 * i + h : i + 4 * h, a);   // (as in k_channel)
        }
      }
    } else {
      u32 w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = __builtin_amdgcn_perm(vraw[2 * j + 1][0], vraw[2 * j][0], v_sel);
      request_v();
#pragma unroll
      for (int m = 0; m < NT; ++m) {
        u32x4_t a;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const u32 pair = __builtin_bit_cast(u32, Codes<BITS>::number(Codes<BITS>::pair(w[j], m), vz[j]));
          a[j] = values(2 * j, pair, pair, 0, 1);
        }
        multiply(m, a);
      }
    }
  };
  // The scales of the block go through LDS to the lanes that need them (one wavefront: its requests are served in order).
  // Returns whether a V scale has a rest.
  auto put_scales = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    bool rest = false;
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      GroupScales &g = par[(of_v ? NG : 0) + i];
      const int key = lane & (BK - 1);
      const float z = has_zp ? zraw[i] : 0.f, near = __builtin_amdgcn_fmed3f(__builtin_rintf(z), -896.f, 896.f);
      g.scale[key] = sraw[i];
      g.rest[key] = -(z - near) * sraw[i];
      g.zero[key] = (_Float16)(-1024.f - (float)Codes<BITS>::kHalf - near);
      rest = rest || (of_v && z != near);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    request_p();
    return __any(rest) != 0;
  };
  for (int blk = blk0; blk < b_end; blk += NW) {
    const bool rest = put_scales();
    block(blk, rest);
  }

  // ---- the wavefronts' partial results meet in LDS, 16 queries at a time ----
  // The row 4 quarter + i of result m is channel NT (4 quarter + i) + m: the values of four consecutive m are
  // four consecutive channels.  Unit (i, h): the channels 4 h.. of rows 4 quarter + i, one float4 per lane.
  float l_own[NQC];
#pragma unroll
  for (int n = 0; n < NQC; ++n) {
    l_own[n] = l_part[n] + __shfl_xor(l_part[n], 16, 64);
    l_own[n] += __shfl_xor(l_own[n], 32, 64);
    if (quarter == 0) lds_ml[(wave * NQC + n) * 16 + r16] = make_float2(m_ref[n], l_own[n]);
  }
  // (the sums on the side belong to every channel of their group; result m has channels NT (4 quarter + i) + m in it)
#pragma unroll
  for (int n = 0; n < NQC; ++n) {
    float sum[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      sum[g] = v_rest[g][n] + __shfl_xor(v_rest[g][n], 16, 64);
      sum[g] += __shfl_xor(sum[g], 32, 64);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float add = NG == 2 && (NT * (4 * quarter + i)) >> v_shift ? sum[NG - 1] : sum[0];
#pragma unroll
      for (int m = 0; m < NT; ++m) oacc[m][n][i] += add;
    }
  }
  float4 *const slots = reinterpret_cast<float4 *>(lds_raw);   // [NW][4][NT / 4][64]
#pragma unroll
  for (int n = 0; n < NQC; ++n) {
    __syncthreads();   // (the scales, or the 16 queries before, are done with)
    float M = 0.f;
    bool any_live = false;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float2 ml = lds_ml[(w * NQC + n) * 16 + r16];
      if (ml.y != 0.f) { M = any_live ? fmaxf(M, ml.x) : ml.x; any_live = true; }
    }
    float l_sum = 0.f;   // (summed in the same order by every wavefront)
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float2 ml = lds_ml[(w * NQC + n) * 16 + r16];
      l_sum = __builtin_fmaf(ml.y, ml.y != 0.f ? __builtin_amdgcn_exp2f(ml.x - M) : 0.f, l_sum);
    }
    const float wt = l_own[n] != 0.f ? __builtin_amdgcn_exp2f(m_ref[n] - M) : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int h = 0; h < NT / 4; ++h)
        slots[((wave * 4 + i) * (NT / 4) + h) * 64 + lane] =
            make_float4(oacc[4 * h][n][i] * wt, oacc[4 * h + 1][n][i] * wt, oacc[4 * h + 2][n][i] * wt, oacc[4 * h + 3][n][i] * wt);
    __syncthreads();
    const float inv = l_sum > 0.f ? 1.0f / l_sum : 0.f;
    for (int u = wave; u < NT; u += NW) {
      float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float4 o = slots[(w * NT + u) * 64 + lane];
        acc[0] += o.x; acc[1] += o.y; acc[2] += o.z; acc[3] += o.w;
      }
      if (qrow[n] >= p.Lq) continue;
      const int ch = NT * (4 * quarter + u / (NT / 4)) + u % (NT / 4) * 4;
      if (p.nsplit > 1) {
        const int64_t prow = ((int64_t)split * p.bh_total + out_pair) * p.Lq + qrow[n];
        if (u == 0 && quarter == 0) *reinterpret_cast<float2 *>(p.ws_ml + prow * 2) = make_float2(M, l_sum);
        *reinterpret_cast<float4 *>(p.ws_o + prow * D + ch) = make_float4(acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
      } else {
        *reinterpret_cast<uint2 *>(p.out + (b * p.o_bs + hq * p.o_hs + qrow[n] * p.o_ts) * D + ch) =
            make_uint2(pack_io_rne<F16>(acc[0] * inv, acc[1] * inv), pack_io_rne<F16>(acc[2] * inv, acc[3] * inv));
      }
    }
  }
}

// Workgroup -> (pair, query tile, share): the grid is (8, shares, groups of eight (batch, head) x query tiles); x runs fastest in
// the dispatch order, so the workgroups of one (batch, head) sit on one XCD (one L2).
struct FewBlockOf {
  int pair, qt, split;
  __device__ __forceinline__ explicit FewBlockOf(const AttnParams &p) {
    const int xcd = blockIdx.x, slot = blockIdx.z, grp = p.q_tiles == 1 ? slot : slot / p.q_tiles;
    split = blockIdx.y;
    qt = slot - grp * p.q_tiles;
    pair = p.kv_hs == 1 && p.kv_ts > 1 ? xcd * ((p.bh_total + 7) >> 3) + grp : grp * 8 + xcd;   // (as in BlockOf)
  }
};
template <int D, int BITS, int NG, int NQC, int NW, bool F16>
__global__ __launch_bounds__(NW * 64, (kWaves<D, NQC, NW>)) void few_attn_kernel(AttnParams p, int k_shift, int v_shift) {
  const FewBlockOf k(p);
  if (k.pair >= p.bh_total) return;
  attend_few<D, BITS, NG, NQC, NW, F16>(p, k_shift, v_shift, k.pair, k.pair, k.qt, k.split);
}
template <int D, int NG, int NQC, int NW, bool F16>
__global__ __launch_bounds__(NW * 64, (kWaves<D, NQC, NW>)) void few_attn_classes_kernel(AttnParams p, ClassTable t, int shift) {
  const FewBlockOf k(p);
  if (k.pair >= p.bh_total) return;
  in_class(p, t, k.pair, [&](auto bits, int bh, int out_pair) __attribute__((always_inline)) {
    attend_few<D, decltype(bits)::value, NG, NQC, NW, F16>(p, shift, shift, bh, out_pair, k.qt, k.split);
  });
}

dim3 few_grid(const AttnParams &p) { return dim3(8, (unsigned)p.nsplit, (unsigned)((p.bh_total + 7) / 8 * p.q_tiles)); }
template <int D, int BITS, int NG, int NQC, int NW, bool F16> void launch_one(const AttnParams &p, int k_shift, int v_shift, hipStream_t st) {
  constexpr int lds = FewLds<D, NG, NQC, NW>::kBytes;
  static bool configured[64] = {false};
  if (lds > 64 * 1024) allow_lds(reinterpret_cast<const void *>(&few_attn_kernel<D, BITS, NG, NQC, NW, F16>), lds, configured);
  hipLaunchKernelGGL((few_attn_kernel<D, BITS, NG, NQC, NW, F16>), few_grid(p), dim3(NW * 64), lds, st, p, k_shift, v_shift);
}
template <int D, int NG, int NQC, int NW, bool F16> void launch_classes(const AttnParams &p, const ClassTable &t, int shift, hipStream_t st) {
  constexpr int lds = FewLds<D, NG, NQC, NW>::kBytes;
  static bool configured[64] = {false};
  if (lds > 64 * 1024) allow_lds(reinterpret_cast<const void *>(&few_attn_classes_kernel<D, NG, NQC, NW, F16>), lds, configured);
  hipLaunchKernelGGL((few_attn_classes_kernel<D, NG, NQC, NW, F16>), few_grid(p), dim3(NW * 64), lds, st, p, t, shift);
}

// f(scale groups, columns of 16 queries, wavefronts)
template <class F> void shape_of(const AttnParams &p, bool one_group, F &&f) {
  using std::integral_constant;
  auto groups = [&](auto columns, auto waves) {
    if (one_group) f(integral_constant<int, 1>{}, columns, waves);
    else f(integral_constant<int, 2>{}, columns, waves);
  };
  auto queries = [&](auto waves) {
    if (p.Lq <= 16) groups(integral_constant<int, 1>{}, waves);
    else groups(integral_constant<int, 2>{}, waves);
  };
  if (p.few_waves == 8) queries(integral_constant<int, 8>{});
  else queries(integral_constant<int, 4>{});
}
template <int D, bool F16> void launch_bits(const AttnParams &p, int bits, int k_shift, int v_shift, hipStream_t st) {
  shape_of(p, D >> k_shift == 1 && D >> v_shift == 1, [&](auto ng, auto nqc, auto nw) {
    constexpr int NG = decltype(ng)::value, NQC = decltype(nqc)::value, NW = decltype(nw)::value;
    if (bits == 4) launch_one<D, 4, NG, NQC, NW, F16>(p, k_shift, v_shift, st);
    else if (bits == 8) launch_one<D, 8, NG, NQC, NW, F16>(p, k_shift, v_shift, st);
    else launch_one<D, 2, NG, NQC, NW, F16>(p, k_shift, v_shift, st);
  });
}
template <int D, bool F16> void launch_classes_shape(const AttnParams &p, const ClassTable &t, int shift, hipStream_t st) {
  shape_of(p, D >> shift == 1, [&](auto ng, auto nqc, auto nw) {
    launch_classes<D, decltype(ng)::value, decltype(nqc)::value, decltype(nw)::value, F16>(p, t, shift, st);
  });
}

}  // namespace

namespace varq_attn {

void launch_few(const AttnParams &p, int D, int bits, int k_group, int v_group, hipStream_t st) {
  const int ks = varq_log2_exact(k_group), vs = varq_log2_exact(v_group);
  if (D == 128) launch_bits<128, false>(p, bits, ks, vs, st);
  else if (p.f16) launch_bits<64, true>(p, bits, ks, vs, st);
  else launch_bits<64, false>(p, bits, ks, vs, st);
}

void launch_few_classes(const AttnParams &p, int D, const ClassTable &t, int group, hipStream_t st) {
  const int shift = varq_log2_exact(group);
  if (D == 128) launch_classes_shape<128, false>(p, t, shift, st);
  else if (p.f16) launch_classes_shape<64, true>(p, t, shift, st);
  else launch_classes_shape<64, false>(p, t, shift, st);
}

}  // namespace varq_attn
