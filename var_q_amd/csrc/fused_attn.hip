// Fused dequant flash-attention for gfx950.
//
//   out = softmax(scale * Q K^T + mask) V,   K = (kq - kzp) * ks,  V = (vq - vzp) * vs
//
// with K/V held as packed INT2/4/8 codes plus per-token group scales.  Replaces
// "unpack whole cache -> fp32 dequant -> external attention" of
// VAR_Q/quant.py:216-230 + VAR/models/basic_var.py:156-162 /
// Infinity/infinity/models/basic.py:339-351; the mask is the block-causal
// next-scale rule of VAR/models/var.py:110-114 expressed as a per-query key
// limit.
//
// Design (one workgroup = 8 wavefronts = 256 queries of one (batch, head)):
//  * Both contractions run on v_mfma_f32_32x32x16_bf16 in transposed form,
//    S^T = K Q^T and O^T = V^T P^T, so that a lane owns one query column: row
//    max/sum are per-lane (one cross-half exchange per tile) and the S^T
//    accumulator registers are directly the B operand of the second MFMA.
//  * Packed K and V go HBM -> registers, requested a tile ahead, are widened once per workgroup and put into LDS as rows of
//    16-bit values, which are the MFMA A operands of the first product; those of the second, which runs over keys, are read
//    from the rows of V with the transposing LDS read.  The tiles are double-buffered, with one workgroup barrier per tile; at head
//    dim 64 there is also an instantiation with one buffer, for launches of many small workgroups (launch_d64).
//  * Launches that leave compute units idle have workgroups of 128 or 64 queries, the same eight wavefronts, two or four of which
//    share the keys of their queries and put their outputs together in LDS at the end (KS, choose_shares).
//  * Key rows are fed to the first MFMA in a permuted order chosen so that each
//    lane's accumulator registers hold 8 consecutive keys per 16-key chunk, which is the order of the V^T operand.
//  * Online softmax in the log2 domain against a reference that is only moved when a logit
//    gets 16 octaves above the maximum it was set from, and that is found out from the weights
//    (their sum, or the exponent bits of the packed bf16 pairs), not by a search for the row
//    maximum: the common tile needs no maximum, no subtraction and no rescale of the output
//    accumulators; the rare one is computed twice.
//  * Two forms of the operands:
//    - dequantized (the default of every kernel): (code - zp) * scale in fp32, rounded to the
//      attention's 16-bit type (bf16, or fp16 for the VAR path) when a tile is widened -- the
//      operands the reference's attention sees -- and a plain flash attention behind it (attend_tiles);
//    - exact codes (opt-in, attend_codes; one group per key of 4- or 2-bit codes at head dim 128, bf16): the MFMA operands
//      are exact small numbers derived from the codes, never scaled or rounded.  A code lands in
//      the top mantissa bits of a bf16 1.x (raw = (code + kOff) / kMul), which costs one shift and
//      one and-or per two elements.  Scales are applied in fp32, zero-points ride on extra MFMA
//      work:
//         S[l,q]  = ck[l] * ( sum_d rawK[l,d] q[d]  -  (kzp[l]+kOff)/kMul * sum_d q[d] )
//         O[q,:]  = ( kMul * sum_l p'[l,q] rawV[l,:]  -  sum_l p'[l,q] (vzp[l]+kOff) ) / sum_l p[l,q]
//      The second term of S is a rank-1 update: both factors are split into three bf16 pieces
//      and laid on the 16 contraction slots of one more MFMA per key block.  The second term of
//      O is one more row of V^T (one more 32-row MFMA block whose row 0 carries vzp+kOff).
//      p' = bf16(p * vs[l]): log2(vs)/ck is added to S through spare slots of the rank-1 MFMA,
//      so exp2 yields p * vs directly, and the denominator is accumulated as sum_l p'[l,q] / vs[l]
//      by rows 4..6 of the extra block (1/vs in three bf16 pieces): numerator and denominator
//      then use the same rounded weights.  V zero-points beyond +-kZmax (data offset by hundreds
//      of quantization steps) or with a fractional part are split zp = zp_c + zp_r; the remainder
//      goes through an fp32 correction term on tiles that have one.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "attn_common.h"
#include "../../include/varq_testing.h"

using namespace varq_attn;

namespace {

constexpr int NW = 8;          // wavefronts per workgroup
constexpr int BM = NW * 32;    // queries per workgroup (32 per wavefront)
// (The D=64 kernels also exist with four wavefronts per workgroup, for launches of many (batch,
// head) pairs with at most 128 queries each -- the first steps of a scale schedule at a large
// batch -- see launch().)
constexpr float kHeadroom = 15.f;   // exact-code kernels: octaves between a fresh softmax reference and the row maximum

// ---- V side code widening ----------------------------------------------------
// The V^T operand of the second MFMA holds, like the K operand of the first, an
// affine image `raw` of the code (code = kMul * raw - kOff) that costs one shift
// and one and-or per two elements.  `pairs` widens octet `oct` of two adjacent key
// rows at once: out[j] = {raw(row0, channel j), raw(row1, channel j)} as a bf16
// pair, which is one dword of the transposed tile.  The zero-point is not folded
// in here; it rides on an extra MFMA row (see the kernel).  kZmax bounds the
// part of the zero-point handled that way: kOff + zp must be a bf16-exact integer.
template <int BITS> struct VCodec;
template <> struct VCodec<4> {
  static constexpr float kMul = 16.f, kOff = 24.f, kZmax = 232.f;
  static constexpr u32 kStageXor = 0x88888888u;   // applied once when the tile is staged: nibble -> code + 8
  __device__ static __forceinline__ void pairs(const u32 *row0, const u32 *row1, int oct, u32 M, u32 (&o)[8]) {
    const u32 w0 = row0[oct], w1 = row1[oct];
    constexpr u32 B = 0x3f803f80u;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      // byte k of both rows, 16 bits apart: nibbles 2k and 2k+1
      const u32 x = __builtin_amdgcn_perm(w1, w0, 0x0c000c00u | (u32)k | ((u32)(4 + k) << 16));
      o[2 * k] = ((x << 3) & M) | B;
      o[2 * k + 1] = ((x >> 1) & M) | B;
    }
  }
};
template <> struct VCodec<2> {
  static constexpr float kMul = 4.f, kOff = 6.f, kZmax = 250.f;
  static constexpr u32 kStageXor = 0xaaaaaaaau;
  __device__ static __forceinline__ void pairs(const u32 *row0, const u32 *row1, int oct, u32 M, u32 (&o)[8]) {
    // the octet is half a word: put the two rows' halves side by side
    const u32 x = __builtin_amdgcn_perm(row1[oct >> 1], row0[oct >> 1], 0x05040100u + (u32)(oct & 1) * 0x02020202u);
    constexpr u32 B = 0x3f803f80u;
    o[0] = ((x << 5) & M) | B;
    o[1] = ((x << 3) & M) | B;
    o[2] = ((x << 1) & M) | B;
    o[3] = ((x >> 1) & M) | B;
    o[4] = ((x >> 3) & M) | B;
    o[5] = ((x >> 5) & M) | B;
    o[6] = ((x >> 7) & M) | B;
    o[7] = ((x >> 9) & M) | B;
  }
};
// x = h0 + h1 + h2 exactly, each piece a bf16 (returned as its 16 bits): three
// 8-bit slices of the 24-bit significand
__device__ __forceinline__ void split3_bf16(float x, u32 &h0, u32 &h1, u32 &h2) {
  const float x0 = u2f(f2u(x) & 0xffff0000u);
  const float r1 = x - x0;
  const float x1 = u2f(f2u(r1) & 0xffff0000u);
  const float x2 = r1 - x1;
  h0 = f2u(x0) >> 16; h1 = f2u(x1) >> 16; h2 = f2u(x2) >> 16;
}

// ---- code widening ---------------------------------------------------------
// K side: 8 codes of one octet -> 8 bf16 (4 dwords) holding code*kMul'+const,
// i.e. code = kMul * raw - kOff.  `slot_d(j)` is the channel (within the octet)
// that lands in operand slot j; the Q operand is gathered in the same order.
template <int BITS> struct KCodec;

template <> struct KCodec<4> {
  // nibble u = code+8 goes to the top 4 mantissa bits of bf16 1.0:
  // raw = 1 + u/16 = (code + 24)/16.
  static constexpr float kMul = 16.f, kOff = 24.f;
  __device__ static __forceinline__ int slot_d(int j) { return (j >> 1) + 4 * (j & 1); }
  static constexpr u32 kStageXor = 0x88888888u;   // applied once when the tile is staged
  static constexpr u32 kMask = 0x00780078u;
  // `M` is kMask held in a vector register, which lets each output be one shift and one v_and_or_b32
  __device__ static __forceinline__ void expand(const u32 *lds_row, int oct, u32 M, u32 (&o)[4]) {
    const u32 w = lds_row[oct];
    constexpr u32 B = 0x3f803f80u;
    o[0] = ((w << 3) & M) | B;   // nibbles 0,4
    o[1] = ((w >> 1) & M) | B;   // 1,5
    o[2] = ((w >> 5) & M) | B;   // 2,6
    o[3] = ((w >> 9) & M) | B;   // 3,7
  }
};

template <> struct KCodec<2> {
  // field u = code+2 goes to the top 2 mantissa bits: raw = 1 + u/4 = (code + 6)/4.
  static constexpr float kMul = 4.f, kOff = 6.f;
  // an octet is half a word: fields 0..7 of the half; dword m holds fields (m, m+4)
  __device__ static __forceinline__ int slot_d(int j) { return (j >> 1) + 4 * (j & 1); }
  static constexpr u32 kStageXor = 0xaaaaaaaau;
  static constexpr u32 kMask = 0x00600060u;
  __device__ static __forceinline__ void expand(const u32 *lds_row, int oct, u32 M, u32 (&o)[4]) {
    const u32 w = (lds_row[oct >> 1] >> ((oct & 1) * 16)) & 0xffffu;
    // fields m (bits 2m) and m+4 (bits 2m+8): move to bits 5..6 and 21..22
    const u32 t = (w & 0xffu) | ((w & 0xff00u) << 8);  // low byte: fields 0-3, byte 2: fields 4-7
    constexpr u32 B = 0x3f803f80u;
    o[0] = ((t << 5) & M) | B;
    o[1] = ((t << 3) & M) | B;
    o[2] = ((t << 1) & M) | B;
    o[3] = ((t >> 1) & M) | B;
  }
};

// octet (8-channel unit) of K that lane-half h contracts in 16-channel chunk ch
__device__ __forceinline__ int k_octet(int ch, int h) { return h * 8 + ch; }

// LDS layout of the kernel with exact codes (bytes), shared by kernel and launcher.
template <int BITS> struct ExactLds {
  static constexpr int D = 128, WPR = D * BITS / 32;
  static constexpr int RSV = WPR + 1;       // packed V row stride (words): odd, bank spread
  static constexpr int kParFloats = 2 * 64;
  // Widened tiles and packed V have two buffers, what the kernel reads while it attends three.
  static constexpr int RSR = 64 + 8;        // stride (bf16) of the rows feeding the extra PV MFMA
  static constexpr int KXS = D + 8;         // stride (bf16) of a widened K row: 16-byte rows, bank spread
  static constexpr int kKx = 0;             // widened K
  static constexpr int kVp = kKx + 2 * 64 * KXS * 2;
  static constexpr int kVt = (kVp + 2 * 64 * RSV * 4 + 15) / 16 * 16;
  static constexpr int kKz = kVt + 2 * D * (64 + 8) * 2;   // rank-1 operands of S^T, 2 x 16 bytes per key
  static constexpr int kWz = kKz + 3 * 64 * 32;            // 8 rows per slot for the extra PV MFMA
  static constexpr int kPar = kWz + 3 * 8 * RSR * 2;
  static constexpr int kFlag = kPar + 3 * kParFloats * 4;
  static constexpr int kBytes = kFlag + 16;
};

// A lane's column of O^T (16 registers of every block of 32 channels) to its place: the output, or with the keys shared out the normalized fp32
// output and (reference, denominator) of this share, for the combining kernel.
template <int D, bool F16, class Value>
__device__ __forceinline__ void store_block(const AttnParams &p, int b, int hq, int qrow, bool q_live, int half, int split, int out_pair, float m_ref, float l_sum,
                                            const floatx16_t (&oacc)[D / 32], Value &&value) {
  const float inv = l_sum > 0.f ? 1.0f / l_sum : 0.f;
  if (!q_live) return;
  __bf16 *optr = p.out + (b * p.o_bs + hq * p.o_hs + qrow * p.o_ts) * D;
  const bool shared_out = p.nsplit > 1;
  const int64_t prow = ((int64_t)split * p.bh_total + out_pair) * p.Lq + qrow;
  float *wptr = p.ws_o + prow * D;
  if (shared_out && half == 0) *reinterpret_cast<float2 *>(p.ws_ml + prow * 2) = make_float2(m_ref, l_sum);
#pragma unroll
  for (int d = 0; d < D / 32; ++d) {
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      // registers 4*g4 .. 4*g4+3 are rows d*32 + 8*g4 + 4*half + 0..3 of O^T
      const float o0 = value(oacc[d][4 * g4 + 0]) * inv, o1 = value(oacc[d][4 * g4 + 1]) * inv;
      const float o2 = value(oacc[d][4 * g4 + 2]) * inv, o3 = value(oacc[d][4 * g4 + 3]) * inv;
      if (shared_out) *reinterpret_cast<float4 *>(wptr + d * 32 + 8 * g4 + 4 * half) = make_float4(o0, o1, o2, o3);
      else *reinterpret_cast<uint2 *>(optr + d * 32 + 8 * g4 + 4 * half) = make_uint2(pack_io_rne<F16>(o0, o1), pack_io_rne<F16>(o2, o3));
    }
  }
}

// The opt-in kernel with exact codes: one group per key of 4- or 2-bit codes at D=128.
// One workgroup's work: query tile qt of packed pair bh (= batch * p.Hkv + packed head), share `split` of its
// keys; partial results go to the rows of pair `out_pair`.
template <int BITS>
__device__ __forceinline__ void attend_codes(const AttnParams &p, int bh, int out_pair, int qt, int split) {
  using L = ExactLds<BITS>;
  constexpr int D = L::D, NT = NW * 64, WPR = L::WPR;
  constexpr int NCH = D / 16;               // contraction chunks of QK^T
  constexpr int NDB = D / 32;               // 32-row blocks of O^T
  constexpr int VTS = BN + 8;               // V^T row stride (bf16 elements)

  // Pipelined LDS buffers (one workgroup barrier per tile):
  //   packed V, the widened K and the widened V^T of tile t live in slot t % 2 (packed V is
  //   read one iteration before its tile is attended, so tile t+2 may take its slot then), the
  //   per-key parameters in slot t % 3.
  // While tile t is being attended, K and V of tile t+1 are widened (K straight
  // from the registers it was loaded into one iteration earlier, once per
  // workgroup, so the eight wavefronts share the work) and packed V of tile t+2 is
  // written from its registers.
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  uint16_t *const lds_kx = reinterpret_cast<uint16_t *>(lds_raw + L::kKx);  // [2][BN][KXS] widened K codes (MFMA A operands)
  u32 *const lds_vp = reinterpret_cast<u32 *>(lds_raw + L::kVp);          // [2][BN][RSV]
  uint16_t *const lds_vt = reinterpret_cast<uint16_t *>(lds_raw + L::kVt);  // [2][D][VTS]  raw V codes, transposed
  u32x4_t *const lds_kz = reinterpret_cast<u32x4_t *>(lds_raw + L::kKz);  // [3][BN][2] rank-1 A operands (per lane half)
  // [3][8][RSR] bf16 rows of the extra PV MFMA: row 0 = vzp_c + kOff,
  // rows 4..6 = the three bf16 pieces of 1/vs, row 7 = zeros
  uint16_t *const lds_wz = reinterpret_cast<uint16_t *>(lds_raw + L::kWz);
  float *const lds_par = reinterpret_cast<float *>(lds_raw + L::kPar);    // [3][kParFloats]: ck [BN], vr [BN]
  int *const lds_flag = reinterpret_cast<int *>(lds_raw + L::kFlag);      // [3] tile+1 if that tile has a zero-point remainder
  constexpr int KXS = L::KXS, RSV = L::RSV, RSR = L::RSR, P_VR = BN;

  const int b = bh / p.Hkv, hs = bh % p.Hkv;
  const int hq = p.head_map ? p.head_map[hs] : hs;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 31, half = lane >> 5;

  // ---- this lane's query ----------------------------------------------------
  const int qrow = qt * BM + wave * 32 + col;
  const bool q_live = qrow < p.Lq;
  const bool wave_live = qt * BM + wave * 32 < p.Lq;   // wave-uniform
  const int qrow_c = q_live ? qrow : p.Lq - 1;
  const __bf16 *qptr = p.q + (b * p.q_bs + hq * p.q_hs + qrow_c * p.q_ts) * D;
  int limit = p.kv_limit ? min(p.kv_limit[qrow_c], p.Lk) : p.Lk;
  if (limit < 0) limit = 0;

  // Q^T operands, gathered in the slot order of the K codec
  u32x4_t qb[NCH];
  u32x4_t bq;
  // The K zero-point term -(kzp+kOff)/kMul * sum(q) is a rank-1 update of S^T and
  // rides on one more MFMA per key block.  Both factors are split into
  // three bf16 pieces (a0+a1+a2, b0+b1+b2, exact) and the 9 products are laid on
  // the 16 contraction slots: slots 0..7 (lower lane half) carry
  // A = a0 a0 a0 a1 a1 a1 a2 a2 against B = b0 b1 b2 b0 b1 b2 b0 b1 (a2*b2, 2^-32 of
  // the term, is dropped).  Slots 0..2 of the upper half add
  // log2(vs)/ck (three pieces against 1.0), which makes exp2(logit) come out as
  // p * vs without a multiplication; the other upper slots are zero.
  // (the raw values were requested into qb earlier -- the prologue does, to overlap the trip
  // with its other loads)
  auto load_q = [&]() {
    float qsum = 0.f;
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
      // the octet's eight channels, loaded in one 16-byte piece, into the codec's slot order
      const u32x4_t raw = qb[ch];
#pragma unroll
      for (int j2 = 0; j2 < 4; ++j2) {
        // operand slots 2*j2 and 2*j2+1, one dword
        const int d0 = KCodec<BITS>::slot_d(2 * j2), d1 = KCodec<BITS>::slot_d(2 * j2 + 1);   // channels within the octet
        const u32 lo = (raw[d0 >> 1] >> (16 * (d0 & 1))) << 16, hi = (raw[d1 >> 1] >> (16 * (d1 & 1))) << 16;
        qb[ch][j2] = (lo >> 16) | hi;
        qsum += u2f(lo) + u2f(hi);
      }
    }
    qsum += __shfl_xor(qsum, 32, 64);
    u32 b0, b1, b2;
    split3_bf16(qsum, b0, b1, b2);
    if (half == 0) bq = u32x4_t{b0 | (b1 << 16), b2 | (b0 << 16), b1 | (b2 << 16), b0 | (b1 << 16)};
    else bq = u32x4_t{0x3f803f80u, 0x00003f80u, 0u, 0u};
  };
  // ---- tile range: every lane of the workgroup runs the same number of tiles ----
  const int kv_end = p.kv_limit ? block_limit<BM>(p.kv_limit, qt * BM, p.Lq, p.Lk) : p.Lk;   // without limits every query sees all keys
  int n_tiles = (kv_end + BN - 1) / BN, tbase = 0;   // tbase: this workgroup's first tile in the block's tile sequence
  if (p.nsplit > 1) {
    // this workgroup's share of the tiles: [t_begin, t_end) of the block's tile sequence
    const int t_begin = n_tiles * split / p.nsplit, t_end = n_tiles * (split + 1) / p.nsplit;
    tbase = t_begin;
    n_tiles = t_end - t_begin;
  }
  const int tile_base = tbase * BN;   // first key of this workgroup's tiles
  // The K prefetch and the V prefetch each walk the tiles in order.
  int pk_tile = 0, pv_tile = 0;
  // the keys that every query of this wavefront sees, and those that some query sees
  int wave_minlim = p.Lk, wave_end = kv_end;
  if (p.kv_limit) {   // (the two halves of the wavefront hold the same queries)
    wave_minlim = wave_fold<false, 2>(q_live ? limit : p.Lk);
    wave_end = wave_fold<true, 2>(q_live ? limit : 0);
  }

  floatx16_t oacc[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) oacc[i][j] = 0.f;
  // extra O^T block: row 0: sum_l p'[l] * (vzp_c + kOff); rows 4..6: pieces of the
  // softmax denominator sum_l p'[l] / vs, i.e. the sum of the weights as rounded for the MFMA
  floatx16_t racc;
#pragma unroll
  for (int j = 0; j < 16; ++j) racc[j] = 0.f;
  float m_ref = 0.f;                 // softmax reference (log2 domain)
  float r_run = 0.f;                 // sum_l p' * vzp_r, only fed on tiles with a remainder

  const int64_t kv_row0 = b * p.kv_bs + hs * p.kv_hs;
  const int64_t kv_ts = p.kv_ts;
  const u32 *kw = p.k_words + kv_row0 * WPR;
  const u32 *vw = p.v_words + kv_row0 * WPR;

  constexpr int QUADS = BN * WPR / 4;                 // 16-byte pieces per packed tile
  constexpr int LPT = (QUADS + NT - 1) / NT;          // pieces per thread
  u32x4_t kreg[LPT], vreg[LPT];
  float ksc = 0.f, kzp = 0.f, vsc = 0.f, vzp = 0.f, ksc0 = 0.f;

  auto prefetch_k = [&]() {   // the next tile of the K stream
    const int t0 = tile_base + pk_tile * BN;
    ++pk_tile;
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int piece = tid + i * NT;
      if (LPT * NT == QUADS || piece < QUADS) {
        const int key = min(t0 + piece / (WPR / 4), p.Lk - 1);
        kreg[i] = *reinterpret_cast<const u32x4_t *>(kw + key * kv_ts * WPR + (piece % (WPR / 4)) * 4);
      }
    }
  };
  auto prefetch = [&]() {   // the next tile of the V stream
    const int t0 = tile_base + pv_tile * BN;
    ++pv_tile;
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int piece = tid + i * NT;
      if (LPT * NT == QUADS || piece < QUADS) {
        const int key = min(t0 + piece / (WPR / 4), p.Lk - 1);
        vreg[i] = *reinterpret_cast<const u32x4_t *>(vw + key * kv_ts * WPR + (piece % (WPR / 4)) * 4);
      }
    }
    // scales: thread t handles key t % 64; wavefront 0 takes K's and the last one V's, which puts the K and the V arithmetic on
    // different wavefronts
    const int key = min(t0 + (tid & 63), p.Lk - 1), seg = tid >> 6, vseg = NW - 1 - seg;
    if (seg < 1) {
      const int64_t g = kv_row0 + key * kv_ts;
      ksc = p.k_scale[g];
      kzp = p.k_zp ? p.k_zp[g] : 0.f;
    }
    if (vseg < 1) {
      const int64_t g = kv_row0 + key * kv_ts;
      vsc = p.v_scale[g];
      vzp = p.v_zp ? p.v_zp[g] : 0.f;
      ksc0 = p.k_scale[g];
    }
  };

  // registers -> LDS slot of `tile` (packed words as they are, parameters precombined)
  auto stage = [&](int tile) {
    const int sl = tile % 3;
    u32 *vp = lds_vp + tile % 2 * BN * RSV;
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int piece = tid + i * NT;
      if (LPT * NT == QUADS || piece < QUADS) {
        const int key = piece / (WPR / 4), w4 = (piece % (WPR / 4)) * 4;
        constexpr u32 VX = VCodec<BITS>::kStageXor;
        // V rows use an odd stride (bank spread for the column reads of the widening step)
#pragma unroll
        for (int j = 0; j < 4; ++j) vp[key * RSV + w4 + j] = vreg[i][j] ^ VX;
      }
    }
    float *par = lds_par + sl * L::kParFloats;
    const int key = tid & 63, seg = tid >> 6, vseg = NW - 1 - seg;
    // |ck| is kept away from zero so that log2(vs)/ck stays finite for a constant group
    auto ck_of = [&](float ks) {
      const float c = ks * p.scale_log2e * KCodec<BITS>::kMul;
      return __builtin_fabsf(c) < 1e-30f ? 1e-30f : c;
    };
    if (seg < 1) {
      par[key] = ck_of(ksc);
      u32 a0, a1, a2;
      split3_bf16(-(kzp + KCodec<BITS>::kOff) * (1.f / KCodec<BITS>::kMul), a0, a1, a2);
      lds_kz[(sl * BN + key) * 2] = u32x4_t{a0 | (a0 << 16), a0 | (a1 << 16), a1 | (a1 << 16), a2 | (a2 << 16)};
    }
    if (vseg < 1) {
      u32 l0, l1, l2;
      split3_bf16(__builtin_amdgcn_logf(vsc) * __builtin_amdgcn_rcpf(ck_of(ksc0)), l0, l1, l2);
      lds_kz[(sl * BN + key) * 2 + 1] = u32x4_t{l0 | (l1 << 16), l2, 0u, 0u};
      // integer part of the zero-point within +-kZmax rides on the MFMA, the rest (none
      // for zero-points produced by the quantizer of ordinary data) on the fp32 remainder
      const float zc = __builtin_amdgcn_fmed3f(__builtin_rintf(vzp), -VCodec<BITS>::kZmax, VCodec<BITS>::kZmax);
      const float zr = vzp - zc;
      par[P_VR + key] = zr;
      uint16_t *rows = lds_wz + sl * 8 * RSR;
      rows[key] = (uint16_t)(f2u(zc + VCodec<BITS>::kOff) >> 16);
      u32 i0, i1, i2;
      split3_bf16(__builtin_amdgcn_rcpf(vsc), i0, i1, i2);
      rows[4 * RSR + key] = (uint16_t)i0;
      rows[5 * RSR + key] = (uint16_t)i1;
      rows[6 * RSR + key] = (uint16_t)i2;
      if (!(zr == 0.f)) lds_flag[sl] = tile + 1;   // benign race: every writer stores the same tag
    }
  };

  u32 kmask = KCodec<BITS>::kMask;
  asm volatile("" : "+v"(kmask));   // keep the mask in a vector register (see KCodec::expand)

  // row of the extra PV block this lane feeds (as element offset)
  const int rowsel = (col == 0 ? 0 : (col >= 4 && col < 7) ? col : 7) * RSR;

  // packed V of `tile` -> V^T bf16: a work item is 2 adjacent keys x 8 channels (one
  // packed word of each key), written as 8 dwords of the transposed tile
  auto widen_v = [&](int tile) {
    const u32 *vp = lds_vp + (tile % 2) * BN * RSV;
    uint16_t *vt = lds_vt + (tile % 2) * D * VTS;
    static_assert((BN / 2) * (D / 8) == NT, "an item for every thread");
    const int kp2 = tid & (BN / 2 - 1), oct = tid / (BN / 2);
    const u32 *row = &vp[kp2 * 2 * RSV];
    u32 pr[8];
    VCodec<BITS>::pairs(row, row + RSV, oct, kmask, pr);
#pragma unroll
    for (int j = 0; j < 8; ++j) *reinterpret_cast<u32 *>(&vt[(oct * 8 + j) * VTS + kp2 * 2]) = pr[j];
  };

  // packed K of `tile` (in kreg) -> widened bf16 rows: each piece holds OPQ octets
  // of one key, every octet becomes one 16-byte MFMA A operand
  auto widen_k = [&](int tile) {
    uint16_t *kx = lds_kx + (tile % 2) * BN * KXS;
    constexpr int OPQ = 16 / BITS;       // octets per piece
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int piece = tid + i * NT;
      if (LPT * NT == QUADS || piece < QUADS) {
        const int key = piece / (WPR / 4), oct0 = (piece % (WPR / 4)) * OPQ;
        constexpr u32 KX = KCodec<BITS>::kStageXor;
        u32 q4[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) q4[w] = kreg[i][w] ^ KX;
#pragma unroll
        for (int j = 0; j < OPQ; ++j) {
          u32 a[4];
          KCodec<BITS>::expand(q4, j, kmask, a);
          *reinterpret_cast<u32x4_t *>(&kx[key * KXS + (oct0 + j) * 8]) = u32x4_t{a[0], a[1], a[2], a[3]};
        }
      }
    }
  };

  // ---- prologue: V tiles 0 and 1 staged, K and V of tile 0 widened, K of tile 1 and V
  //      of tile 2 in registers ------------------------------------------------------------
  if (tid < 3) lds_flag[tid] = 0;
  for (int i = tid; i < 3 * RSR; i += NT) lds_wz[((i / RSR) * 8 + 7) * RSR + i % RSR] = 0;   // the all-zero row of each slot
  if (n_tiles > 0) { prefetch_k(); prefetch(); }
  // the query values, behind the first tile's requests
#pragma unroll
  for (int ch = 0; ch < NCH; ++ch) qb[ch] = *reinterpret_cast<const u32x4_t *>(qptr + k_octet(ch, half) * 8);
  __syncthreads();
  load_q();
  if (n_tiles > 0) { stage(0); widen_k(0); }
  if (n_tiles > 1) { prefetch_k(); prefetch(); stage(1); }
  __syncthreads();
  if (n_tiles > 0) widen_v(0);
  if (n_tiles > 2) prefetch();
  __syncthreads();

  // ---- the three phases of one 32-key block, as lambdas over per-tile state --------
  // LDS operands are requested ahead of their use where the registers allow it (the
  // scheduling fences keep the requests where they are written).
  int t0 = 0;
  const uint16_t *kx = nullptr, *vt = nullptr, *wz = nullptr;
  const float *par = nullptr;
  const u32x4_t *kz = nullptr;
  bool tile_rem = false, first = true;
  // register i of this lane <-> key kb*32 + 16*(i/8) + 8*half + i%8 of the tile
  floatx16_t sacc;
  u32 pop[2][4];          // P'^T operands: p * vs as bf16, [16-key chunk][dword]
  float ckv[16];
  u32x4_t vta[NDB], wza;

  auto begin_tile = [&](int tile) {
    t0 = tile_base + tile * BN;
    kx = lds_kx + (tile % 2) * BN * KXS;
    par = lds_par + (tile % 3) * L::kParFloats;
    vt = lds_vt + (tile % 2) * D * VTS;
    kz = lds_kz + (tile % 3) * BN * 2;
    wz = lds_wz + (tile % 3) * 8 * RSR;
    tile_rem = lds_flag[tile % 3] == tile + 1;   // tagged with the tile, so stale tags never match
    // slot (tile+2)%3 was last read during tile-1 (before the barrier): refill it
    if (tile + 2 < n_tiles) stage(tile + 2);
    if (tile + 3 < n_tiles) prefetch();
  };
  // with the PV MFMAs of a block in flight: widen the next tile's K and V into the other slots
  auto widen_next = [&](int tile) {
    if (tile + 1 < n_tiles) {
      widen_v(tile + 1);
      widen_k(tile + 1);
      if (tile + 2 < n_tiles) prefetch_k();
    }
  };
  auto load_scales = [&](int kb) {
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const int key = kb * 32 + 16 * (i4 >> 1) + 8 * half + 4 * (i4 & 1);
      const float4 t = *reinterpret_cast<const float4 *>(&par[key]);
      ckv[4 * i4] = t.x; ckv[4 * i4 + 1] = t.y; ckv[4 * i4 + 2] = t.z; ckv[4 * i4 + 3] = t.w;
    }
  };
  auto load_v_operands = [&](int kb, int c) {
#pragma unroll
    for (int d = 0; d < NDB; ++d)
      vta[d] = *reinterpret_cast<const u32x4_t *>(&vt[(d * 32 + col) * VTS + (kb * 2 + c) * 16 + half * 8]);
    wza = *reinterpret_cast<const u32x4_t *>(&wz[rowsel + (kb * 2 + c) * 16 + half * 8]);
  };

  // (raised priority around the matrix instructions: see attend_tiles)
  constexpr bool MFMA_PRIO = BITS == 4;
  // S^T = K Q^T for one 32-key block; the A operands are the widened K rows in LDS
  auto qk = [&](int kb) {
    if constexpr (MFMA_PRIO) __builtin_amdgcn_s_setprio(1);
    const int krow_i = kb * 32 + kperm(col);
    floatx16_t zero;
#pragma unroll
    for (int j = 0; j < 16; ++j) zero[j] = 0.f;
    // starts the accumulator with the zero-point term (see bq above)
    sacc = mfma_32x32x16<false>(kz[krow_i * 2 + half], bq, zero);
    const uint16_t *krow = &kx[krow_i * KXS];
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) sacc = mfma_32x32x16<false>(*reinterpret_cast<const u32x4_t *>(&krow[k_octet(ch, half) * 8]), qb[ch], sacc);
    if constexpr (MFMA_PRIO) __builtin_amdgcn_s_setprio(0);
  };

  // logits -> P'^T operands of one block: online softmax against a lazily moved reference
  auto softmax = [&](int kb) {
    float z[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = __builtin_fmaf(ckv[i], sacc[i], -m_ref);
    // mask: block-causal key limit and the ragged last tile
    if (t0 + BN > wave_minlim) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = t0 + kb * 32 + 16 * (i >> 3) + 8 * half + (i & 7);
        if (key >= limit) z[i] = -INFINITY;
      }
    }
    // Moves the softmax reference kHeadroom octaves above the row's current maximum: up only (never down) once
    // something has been accumulated; the very first block takes its maximum as it is, negative
    // or not (the accumulators are still zero, so alpha = 1 is exact).
    auto move_reference = [&]() {
      float zmax = z[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) zmax = fmaxf(zmax, z[i]);
      // the other lane half of the same query, without a trip through LDS
      const auto sw = __builtin_amdgcn_permlane32_swap(f2u(zmax), f2u(zmax), false, false);
      zmax = fmaxf(u2f(sw[0]), u2f(sw[1]));
      const float delta = first ? ((zmax == -INFINITY) ? 0.f : zmax + kHeadroom) : fmaxf(zmax + kHeadroom, 0.f);
      const float alpha = first ? 1.f : __builtin_amdgcn_exp2f(-delta);
      m_ref += delta;
#pragma unroll
      for (int i = 0; i < 16; ++i) z[i] -= delta;
#pragma unroll
      for (int d = 0; d < NDB; ++d)
#pragma unroll
        for (int j = 0; j < 16; ++j) oacc[d][j] *= alpha;
#pragma unroll
      for (int j = 0; j < 16; ++j) racc[j] *= alpha;
      r_run *= alpha;
    };
    // exp2 of the logits, rounded to bf16 pairs for the MFMA
    auto weights = [&]() {
      float pv[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) pv[i] = __builtin_amdgcn_exp2f(z[i]);
#pragma unroll
      for (int i = 0; i < 16; i += 2) pop[i >> 3][(i & 7) >> 1] = pack_bf16_rne(pv[i], pv[i + 1]);
    };
    // The denominator is summed by the MFMA, so there is no sum to look at (as in attend_tiles); the packed
    // weights themselves are: all are >= 0, so bit 14 of a bf16 (the top exponent bit) says
    // "this weight is 2 or more" (infinities included), and an OR over the block's eight words
    // finds one.  The reference is put kHeadroom octaves above the maximum when it moves, so
    // weights start at 2^-kHeadroom or below -- bf16 and the fp32 sums keep their relative
    // precision there -- and it moves again only for a logit 1 + kHeadroom octaves above that
    // maximum.
    if (first) move_reference();
    weights();
    if (!first) {
      u32 any_w = 0;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) any_w |= pop[h][j];
      if (__any((any_w & 0x40004000u) != 0)) {
        move_reference();
        weights();
      }
    }
    first = false;
    if (tile_rem) {
      // the remainder term must see the same bf16-rounded weights as the MFMA
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const int key = kb * 32 + 16 * (i >> 3) + 8 * half + (i & 7);
        const u32 pk = pop[i >> 3][(i & 7) >> 1];
        r_run = __builtin_fmaf(u2f(pk << 16), par[P_VR + key], r_run);
        r_run = __builtin_fmaf(u2f(pk & 0xffff0000u), par[P_VR + key + 1], r_run);
      }
    }
  };

  // O^T += V^T P'^T for the 32 keys of one block; one more MFMA per chunk
  // feeds the extra block: its row 0 collects the zero-point sum and rows
  // 4..6 the softmax denominator
  auto pv_mfma = [&](int kb) {
    if constexpr (MFMA_PRIO) __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      u32x4_t av[NDB];
#pragma unroll
      for (int d = 0; d < NDB; ++d) av[d] = vta[d];
      const u32x4_t aw = wza;
      if (c == 0) {
        load_v_operands(kb, 1);   // in flight under this chunk's MFMAs
        __builtin_amdgcn_sched_barrier(0);
      }
      const u32x4_t bv = {pop[c][0], pop[c][1], pop[c][2], pop[c][3]};
#pragma unroll
      for (int d = 0; d < NDB; ++d) oacc[d] = mfma_32x32x16<false>(av[d], bv, oacc[d]);
      racc = mfma_32x32x16<false>(aw, bv, racc);
    }
    if constexpr (MFMA_PRIO) __builtin_amdgcn_s_setprio(0);
  };

  // (the key blocks behind the last key that a query of this wavefront sees: see attend_tiles)
  const int wave_tiles = __builtin_amdgcn_readfirstlane(wave_live ? min(n_tiles, (max(wave_end - tile_base, 0) + BN - 1) / BN) : 0);
  auto attend = [&](int tile) {
    begin_tile(tile);
    const bool half_tile = wave_end - t0 <= 32;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      if (kb == 1 && half_tile) continue;
      load_scales(kb);
      qk(kb);
      load_v_operands(kb, 0);   // used after the softmax arithmetic
      __builtin_amdgcn_sched_barrier(0);
      softmax(kb);
      pv_mfma(kb);
      if (kb == 0) widen_next(tile);
    }
  };
  int tile = 0;
  for (; tile < wave_tiles; ++tile) {
    attend(tile);
    __syncthreads();   // the one barrier per tile
  }
  // from there on (a wavefront without queries: from the start) the wavefront only helps with staging and
  // widening, at the same barrier count as the others
  for (; tile < n_tiles; ++tile) {
    if (tile + 2 < n_tiles) stage(tile + 2);
    if (tile + 3 < n_tiles) prefetch();
    widen_next(tile);
    __syncthreads();
  }
  if (!wave_live) return;

  // ---- epilogue -------------------------------------------------------------------
  r_run += __shfl_xor(r_run, 32, 64);
  // rows 4..6 of racc are registers 0..2 of the upper lane half, row 0 register 0 of the lower
  const float l_sum = __shfl(racc[0] + racc[1] + racc[2], col + 32, 64);
  const float r = __shfl(racc[0], col, 64) + r_run;
  constexpr float VM = VCodec<BITS>::kMul;
  store_block<D, false>(p, b, hq, qrow, q_live, half, split, out_pair, m_ref, l_sum, oacc, [&](float o) { return VM * o - r; });
}

// ---- the kernel that dequantizes ----------------------------------------------------------------
// K and V of a tile are widened alike, straight from the registers they were loaded into: a thread takes an eighth of a key's
// channels, of K and of V, dequantizes them -- (code - zp) * scale in fp32, rounded to the attention's 16-bit type, the very
// operands that the reference's attention sees after its dequantize and downcast (VAR_Q/quant.py:216-224,
// VAR/models/basic_var.py:158) -- and puts them into LDS as a row of that key.  The rows of K are operands of S^T = K Q^T as they lie; the
// operands of O^T = V^T P^T, 8 keys of one channel, come out of the rows of V through the transposing LDS read (ds_read_b64_tr_b16).
// Before, V went to LDS packed and its parameters with it, was read back, and was written transposed two keys at a time; a table without
// zero-points cost as much as one with.  Attention calls, before -> now, us: [64,256,16,64] over 680 keys, 8 bits, ten tables 95 -> 81, its
// ten scales with the quantizers 401 -> 372..392 (boxes differ); 128 pairs x 680 tokens block-causal, 4 bits in groups of 32 34 -> 31.
// What bounds it: at D=64 and four wavefronts per SIMD the vector ALU (some 200 instructions per wavefront and tile beside 24
// matrix instructions); with one workgroup per compute unit the chain through a tile, 1.6 us at D=64 and 2.1 to 2.5 at D=128.
//
// A thread's codes as numbers, divided by kUnit: a power of two, which the scale and the zero-point take up exactly.
template <int BITS> struct Widen {
  static constexpr float kUnit = BITS == 8 ? 1.f : BITS == 4 ? 16.f : 4.f;
  // octet `o` of the piece that begins at w; the low four bits of a word as a signed number, a sixteenth of it, are one instruction
  __device__ static __forceinline__ void octet(const u32 *w, int o, float (&f)[8]) {
    if constexpr (BITS == 8) {
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = (float)(int)__builtin_amdgcn_sbfe((int)w[2 * o + (j >> 2)], 8 * (j & 3), 8);
    } else if constexpr (BITS == 4) {
      u32 low = w[o], high = low >> 4;
      asm("" : "+v"(high));   // (a register of its own, whose bytes the conversions take as they lie; the compiler would shift each out of w)
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = __builtin_amdgcn_cvt_off_f32_i4((int)__builtin_amdgcn_ubfe(j & 1 ? high : low, 8 * (j >> 1), 8));
    } else {
      const u32 h = w[o >> 1] >> (16 * (o & 1));
      u32 x[4] = {(h << 2) & 0xccccu, h & 0xccccu};   // even and odd fields in the upper halves of nibbles
      x[2] = x[0] >> 4; x[3] = x[1] >> 4;
      asm("" : "+v"(x[2]), "+v"(x[3]));
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = __builtin_amdgcn_cvt_off_f32_i4((int)__builtin_amdgcn_ubfe(x[j & 3], 8 * (j >> 2), 8));
    }
  }
};
// Rows of K and V in LDS (stride in elements).  K: 16 lanes read 16 bytes of 16 rows each, 4 banks apart.  V: 32 lanes read 64 bytes of four
// rows each, at D=128 16 banks apart (4 banks apart, as K's, they got in one another's way); at D=64 they are 4 apart too, where 16 measured the same.
template <int D> constexpr int kKRow = D + 8;
template <int D> constexpr int kVRow = D + (D == 128 ? 32 : 8);
template <int D, int TB = BN> constexpr int kKBuf = TB * kKRow<D>;   // a tile of TB keys (elements)
template <int D, int TB = BN> constexpr int kVBuf = TB * kVRow<D>;
// LDS of the kernel (bytes).  ONE: one buffer instead of two, so that more workgroups are resident; a tile is widened and
// attended before the next one is widened (see launch_d64 for when that is the better way).
// KS: wavefronts that share a block of 32 queries, each with a block of 32 keys of every tile (of 64 keys, 128 with four of them).  Where a launch has fewer
// workgroups than the device has compute units the chain through a tile is what it takes, and with half the work of a tile in each of twice the workgroups, which all
// widen it, that chain is two thirds as long (D=128 2.1 us a tile of 64 keys alone, 1.35 with two, 0.95 with four; D=64 1.4, 0.85, 0.55): see choose_shares.
template <int KS> constexpr int kTileKeys = KS <= 2 ? BN : KS * 32;
template <int D, bool ONE, int KS = 1> struct TileLds {
  static constexpr int kBufs = ONE ? 1 : 2;
  static constexpr int kTables = kBufs * (kKBuf<D, kTileKeys<KS>> + kVBuf<D, kTileKeys<KS>>) * 2;   // behind K's and V's buffers: the per-channel tables of the launch
  // ... and, in the place of all of them when the last tile is attended, what the wavefronts of a block of queries tell one another (see join_shares)
  static constexpr int kStats = 8 * 32 * 8, kJoin = KS == 1 ? 0 : kStats + 8 / KS * (KS - 1) * (D / 8) * 1024;
};

// CHAN: scales and zero-points per (head, channel) instead of per (key, channel group), in up to 16 tables that change along the
// keys (a cache quantized step by step has one per step): K[l,d] = (code[l,d] - zk_s[d]) * sk_s[d] with s the segment of key l, and
// likewise V.  The tables of the head sit in LDS; a tile inside one segment reads that segment's rows, a tile that
// straddles segments looks the segment up per key.
// KS: see TileLds.
// F16: q, out and the MFMA operands are fp16 instead of bf16 (dequantized K and V are rounded to fp16, as the reference's fp16
// attention call sees them: VAR/models/basic_var.py:157-158 under the fp16 autocast of scripts/inference_multi_VAR.py:123).
// One workgroup's work: query tile qt of packed pair bh (= batch * p.Hkv + packed head), share `split` of its
// keys; partial results go to the rows of pair `out_pair`.
template <int D, int BITS, bool CHAN, int NWV, bool F16, bool ONE = false, int KS = 1>
__device__ __forceinline__ void attend_tiles(const AttnParams &p, int bh, int out_pair, int qt, int split) {
  constexpr int NT = NWV * 64, BM = NWV / KS * 32, TB = kTileKeys<KS>;
  constexpr int WPR = D * BITS / 32;        // packed words per key row
  constexpr int NCH = D / 16;               // contraction chunks of QK^T
  constexpr int NDB = D / 32;               // 32-row blocks of O^T
  constexpr int CH = D / 8, OCT = CH / 8;   // channels and octets of a thread's piece of a row
  constexpr int PB = CH * BITS / 8, PW = PB < 4 ? 1 : PB / 4;   // bytes and words of it
  constexpr int IT = TB * 8 / NT;           // pieces of a tile per thread
  constexpr int KBUF = kKBuf<D, TB>, VBUF = kVBuf<D, TB>;
  using L = TileLds<D, ONE, KS>;
  constexpr int KR = kKRow<D>, VR = kVRow<D>;
  constexpr float kUnit = Widen<BITS>::kUnit;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  uint16_t *const lds_k = reinterpret_cast<uint16_t *>(lds_raw);   // [kBufs][TB][KR]
  uint16_t *const lds_v = lds_k + L::kBufs * KBUF;                 // [kBufs][TB][VR]
  float *const lds_tab = reinterpret_cast<float *>(lds_raw + L::kTables);   // [nseg][2 or 4][D]: scales of K and V times kUnit, zero-points over kUnit
  const bool has_zp = p.k_chan_zp || p.v_chan_zp;
  const int tab_rows = has_zp ? 4 : 2;

  const int b = bh / p.Hkv, hs = bh % p.Hkv;
  const int hq = p.head_map ? p.head_map[hs] : hs;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 31, half = lane >> 5;
  const int qwave = wave % (NWV / KS), share = wave / (NWV / KS);   // the wavefront's block of queries, and of keys of a tile

  // ---- this lane's query ----------------------------------------------------
  const int qrow = qt * BM + qwave * 32 + col;
  const bool q_live = qrow < p.Lq;
  const bool wave_live = qt * BM + qwave * 32 < p.Lq;   // wave-uniform
  const int qrow_c = q_live ? qrow : p.Lq - 1;
  const __bf16 *const qptr = p.q + (b * p.q_bs + hq * p.q_hs + qrow_c * p.q_ts) * D + half * 8;
  const int limit = p.kv_limit ? max(min(p.kv_limit[qrow_c], p.Lk), 0) : p.Lk;

  // ---- tile range: every lane of the workgroup runs the same number of tiles ----
  const int kv_end = p.kv_limit ? block_limit<BM>(p.kv_limit, qt * BM, p.Lq, p.Lk) : p.Lk;   // without limits every query sees all keys
  int n_tiles = (kv_end + TB - 1) / TB, tbase = 0;   // tbase: this workgroup's first tile in the block's tile sequence
  if (p.nsplit > 1) {
    const int t_begin = n_tiles * split / p.nsplit, t_end = n_tiles * (split + 1) / p.nsplit;
    tbase = t_begin;
    n_tiles = t_end - t_begin;
  }
  const int tile_base = tbase * TB;   // first key of this workgroup's tiles
  // the keys that every query of this wavefront sees, and those that some query sees
  int wave_minlim = p.Lk, wave_end = kv_end;
  if (p.kv_limit) {   // (the two halves of the wavefront hold the same queries)
    wave_minlim = wave_fold<false, 2>(q_live ? limit : p.Lk);
    wave_end = wave_fold<true, 2>(q_live ? limit : 0);
  }
  // segment ends in LDS: indexing the kernel arguments with a run-time index would move
  // the whole argument block to scratch memory (literal indices only, for the same reason)
  __shared__ int lds_seg_end[kMaxSegments];
  if constexpr (CHAN) {
    if (p.nseg > 1 && tid == 0) {
#define VARQ_SEG(S) lds_seg_end[S] = p.seg_end[S];
      VARQ_SEG(0) VARQ_SEG(1) VARQ_SEG(2) VARQ_SEG(3) VARQ_SEG(4) VARQ_SEG(5) VARQ_SEG(6) VARQ_SEG(7)
      VARQ_SEG(8) VARQ_SEG(9) VARQ_SEG(10) VARQ_SEG(11) VARQ_SEG(12) VARQ_SEG(13) VARQ_SEG(14) VARQ_SEG(15)
#undef VARQ_SEG
      static_assert(kMaxSegments == 16, "the list above names every segment");
    }
    // (read behind the prologue's first barrier)
  }

  // ---- loads: piece i of the thread is eighth `part` of key tid / 8 + i * NT / 8 of the tile ----
  const int part = tid & 7, key_l = tid >> 3;
  const int64_t kv_row0 = b * p.kv_bs + hs * p.kv_hs;
  const int k_groups = CHAN ? 0 : D >> p.k_shift, v_groups = CHAN ? 0 : D >> p.v_shift;
  const int64_t word_row = p.kv_ts * (WPR * 4), ks_row = p.kv_ts * (4 * k_groups), vs_row = p.kv_ts * (4 * v_groups);   // bytes from key to key
  const char *const kw = reinterpret_cast<const char *>(p.k_words) + kv_row0 * (WPR * 4), *const vw = reinterpret_cast<const char *>(p.v_words) + kv_row0 * (WPR * 4);
  // (without zero-points the scales are read in their place and not used: a branch around each load costs more)
  const bool k_has_zp = p.k_zp != nullptr, v_has_zp = p.v_zp != nullptr;
  const char *const ksc = reinterpret_cast<const char *>(p.k_scale) + kv_row0 * (4 * k_groups);
  const char *const kzp = reinterpret_cast<const char *>(k_has_zp ? p.k_zp : p.k_scale) + kv_row0 * (4 * k_groups);
  const char *const vsc = reinterpret_cast<const char *>(p.v_scale) + kv_row0 * (4 * v_groups);
  const char *const vzp = reinterpret_cast<const char *>(v_has_zp ? p.v_zp : p.v_scale) + kv_row0 * (4 * v_groups);
  const int k_g4 = CHAN ? 0 : (part * CH >> p.k_shift) * 4, v_g4 = CHAN ? 0 : (part * CH >> p.v_shift) * 4;
  // (two bytes stay two until they are used: widened where the two ways of request() meet, they would be waited for there)
  using Raw = std::conditional_t<PB == 2, uint16_t, u32>;
  struct Piece { Raw k[PW], v[PW]; float ks, kz, vs, vz; } next[IT];
  auto load_piece = [](const char *src, Raw (&dst)[PW]) __attribute__((always_inline)) {
    if constexpr (PB == 16) {
      const u32x4_t t = *reinterpret_cast<const u32x4_t *>(src);
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[i] = t[i];
    } else if constexpr (PB == 8) {
      const uint2 t = *reinterpret_cast<const uint2 *>(src);
      dst[0] = t.x; dst[1] = t.y;
    } else if constexpr (PB == 4) {
      dst[0] = *reinterpret_cast<const u32 *>(src);
    } else {
      dst[0] = *reinterpret_cast<const uint16_t *>(src);
    }
  };
  // The tiles are requested in order, at scalar addresses that go on from one to the next; a lane adds its own 32 bits of an offset.  (With each
  // lane's address made anew in 64 bits, nine of the slow multiplications and forty scalar instructions of every wavefront and tile: scales in
  // groups, 4 bits, the quantizer of the step included, us: 128 pairs x 680 tokens block-causal, D=64 36.7 -> 34.9; 32 pairs, 1024 x 2521, D=128 74.2 -> 71.2.)
  int64_t w_tile = tile_base * word_row, ks_tile = tile_base * ks_row, vs_tile = tile_base * vs_row;
  int last = p.Lk - 1 - tile_base;   // (rows past the end: the last row's)
  auto request = [&]() {
    auto load = [&](Piece &x, auto w_at, auto ks_at, auto vs_at) __attribute__((always_inline)) {
      load_piece(kw + w_tile + w_at, x.k);
      load_piece(vw + w_tile + w_at, x.v);
      if constexpr (!CHAN) {
        x.ks = *reinterpret_cast<const float *>(ksc + ks_tile + ks_at);
        x.kz = *reinterpret_cast<const float *>(kzp + ks_tile + ks_at);
        x.vs = *reinterpret_cast<const float *>(vsc + vs_tile + vs_at);
        x.vz = *reinterpret_cast<const float *>(vzp + vs_tile + vs_at);
      }
    };
    if (word_row < 1 << 24) {   // (no row of scales is longer than one of codes)
#pragma unroll
      for (int i = 0; i < IT; ++i) {
        const u32 key = (u32)min(key_l + i * (NT / 8), last);
        load(next[i], (u32)__umul24(key, (u32)word_row) + part * PB, (u32)__umul24(key, (u32)ks_row) + k_g4, (u32)__umul24(key, (u32)vs_row) + v_g4);
      }
    } else {
#pragma unroll
      for (int i = 0; i < IT; ++i) {
        const int64_t key = min(key_l + i * (NT / 8), last);
        load(next[i], key * word_row + part * PB, key * ks_row + k_g4, key * vs_row + v_g4);
      }
      asm volatile("");   // (or the compiler makes the loads of both ways one, with 64 bits of an offset)
    }
    w_tile += TB * word_row; ks_tile += TB * ks_row; vs_tile += TB * vs_row; last -= TB;
  };

  // CHAN: segment of the first key of the next tile to be widened, and where that segment ends
  // (wave-uniform; the tiles are widened in order)
  int wseg = 0, wseg_end = p.Lk;
  // the requested tile -> rows of K and V
  auto widen = [&](int tile) {
    uint16_t *const kx = lds_k + tile % L::kBufs * KBUF, *const vx = lds_v + tile % L::kBufs * VBUF;
    bool one_seg = true;
    if constexpr (CHAN) {
      const int t0w = tile_base + tile * TB;
      while (wseg + 1 < p.nseg && t0w >= wseg_end) {
        ++wseg;
        wseg_end = __builtin_amdgcn_readfirstlane(lds_seg_end[wseg]);
      }
      one_seg = wseg + 1 >= p.nseg || t0w + TB <= wseg_end;
    }
    auto put = [&](auto zp_tag) __attribute__((always_inline)) {
      constexpr bool ZP = decltype(zp_tag)::value;
#pragma unroll
      for (int i = 0; i < IT; ++i) {
        const int key = key_l + i * (NT / 8);
        const float *tab = lds_tab;
        if constexpr (CHAN) {
          int sg = wseg;
          if (!one_seg) {
            const int k = min(tile_base + tile * TB + key, p.Lk - 1);
            while (sg + 1 < p.nseg && k >= lds_seg_end[sg]) ++sg;
          }
          tab += sg * (tab_rows * D) + part * CH;
        }
        auto rows = [&](const Raw (&raw)[PW], float s, float z, int row, uint16_t *dst) __attribute__((always_inline)) {
          u32 w[PW];
#pragma unroll
          for (int j = 0; j < PW; ++j) w[j] = raw[j];
          const float s1 = s * kUnit, z1 = z * (1.f / kUnit);
#pragma unroll
          for (int o = 0; o < OCT; ++o) {
            float f[8];
            Widen<BITS>::octet(w, o, f);
            u32x4_t r;
            if constexpr (CHAN) {
              const float4 sa = *reinterpret_cast<const float4 *>(tab + row * D + o * 8), sb = *reinterpret_cast<const float4 *>(tab + row * D + o * 8 + 4);
              const float sc[8] = {sa.x, sa.y, sa.z, sa.w, sb.x, sb.y, sb.z, sb.w};
              if constexpr (ZP) {
                const float4 za = *reinterpret_cast<const float4 *>(tab + (row + 2) * D + o * 8), zb = *reinterpret_cast<const float4 *>(tab + (row + 2) * D + o * 8 + 4);
                const float zc[8] = {za.x, za.y, za.z, za.w, zb.x, zb.y, zb.z, zb.w};
#pragma unroll
                for (int j = 0; j < 8; ++j) f[j] -= zc[j];
              }
#pragma unroll
              for (int j = 0; j < 4; ++j) r[j] = pack_io_rne<F16>(f[2 * j] * sc[2 * j], f[2 * j + 1] * sc[2 * j + 1]);
            } else {
#pragma unroll
              for (int j = 0; j < 4; ++j) r[j] = pack_io_rne<F16>((f[2 * j] - z1) * s1, (f[2 * j + 1] - z1) * s1);
            }
            *reinterpret_cast<u32x4_t *>(dst + o * 8) = r;
          }
        };
        rows(next[i].k, next[i].ks, k_has_zp ? next[i].kz : 0.f, 0, kx + key * KR + part * CH);
        rows(next[i].v, next[i].vs, v_has_zp ? next[i].vz : 0.f, 1, vx + key * VR + part * CH);
      }
    };
    if constexpr (CHAN) {
      if (has_zp) put(std::true_type{});
      else put(std::false_type{});
    } else {
      put(std::true_type{});
    }
  };

  // ---- prologue: tile 0 widened, tile 1 requested ----
  if (n_tiles > 0) request();
  // the query values, behind the first tile's requests and ahead of the table loads: one round trip for all three
  u32x4_t qb[NCH];
#pragma unroll
  for (int ch = 0; ch < NCH; ++ch) qb[ch] = *reinterpret_cast<const u32x4_t *>(qptr + ch * 16);
  if constexpr (CHAN) {
    // The head's tables (see lds_tab): row by row, NT / D of them at a time.  kTabLoads rows are
    // under way before the first is used: one after the other, each a trip to memory, they were what a launch began with, 1.6 us (five
    // segments) to 4.1 us (eight, four wavefronts) of the 10 to 20 that the smaller steps of a schedule take.
    constexpr int kTabLoads = 8, G = NT / D;
    static_assert(NT % D == 0 && D % 64 == 0, "the row that a thread loads is the same for a wavefront");
    const int row0 = __builtin_amdgcn_readfirstlane(tid / D), d = tid % D, rows = p.nseg * tab_rows;
    for (int first = row0; first < rows; first += kTabLoads * G) {
      float x[kTabLoads] = {};
#pragma unroll
      for (int u = 0; u < kTabLoads; ++u) {
        const int r = min(first + u * G, rows - 1), which = r & (tab_rows - 1), seg = r >> (has_zp ? 2 : 1);
        const float *const of_k = which & 2 ? p.k_chan_zp : p.k_chan_scale, *const of_v = which & 2 ? p.v_chan_zp : p.v_chan_scale;
        // (as a global pointer: behind the choice the compiler no longer knows it for one, and flat loads wait for LDS too)
        const auto src = (const __attribute__((address_space(1))) float *)(uintptr_t)(which & 1 ? of_v : of_k);
        if (src) x[u] = src[((int64_t)seg * p.Hkv + hs) * D + d];
      }
#pragma unroll
      for (int u = 0; u < kTabLoads; ++u) {
        const int r = first + u * G;
        if (r < rows) lds_tab[r * D + d] = r & 2 & tab_rows >> 1 ? x[u] * (1.f / kUnit) : x[u] * kUnit;
      }
    }
    __syncthreads();
    if (p.nseg > 1) wseg_end = __builtin_amdgcn_readfirstlane(lds_seg_end[0]);   // (a share of the keys may begin mid-cache: widen goes on to its segment)
  }
  if constexpr (!ONE) {
    if (n_tiles > 0) widen(0);
    if (n_tiles > 1) request();
    __syncthreads();
  }

  // (the queries are there: otherwise the compiler has the key loop wait for them, and with them for the tile that is on its way)
#pragma unroll
  for (int ch = 0; ch < NCH; ++ch) asm volatile("" : "+v"(qb[ch]));

  floatx16_t oacc[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) oacc[i][j] = 0.f;
  float l_part = 0.f;   // the softmax denominator, from the weights as rounded for the MFMA (this lane's keys; the lane halves are added in the epilogue)
  float m_ref = 0.f;    // softmax reference (log2 domain)
  bool first = true;

  // A wavefront raises its priority while it issues the MFMAs of a phase.  Measured per kernel
  // (same run, bit-identical results): at D=128 that is worth 5 % for 4-bit codes (0.725 against
  // 0.762 ms at the configuration-4 shape) and costs 1-3.5 % for 2-bit and 8-bit codes, whose
  // widening has more to do beside the MFMAs; at D=64 it makes no difference.
  constexpr bool MFMA_PRIO = !(D == 128 && BITS != 4);
  // LDS operands are requested ahead of their use where the registers allow it (the
  // scheduling fences keep the requests where they are written).
  floatx16_t sacc;
  u32 pop[2][4];       // P^T operands, [16-key chunk][dword]
  u32x4_t vta[NDB];
  int t0 = 0;
  const uint16_t *kx = nullptr, *vx = nullptr;
  // V^T operand of block kb, chunk c, rows d: the lane's 8 keys of channel d * 32 + col, four of them by each read (16 lanes read 4 keys x 16
  // channels, 8 bytes each, and are handed a channel's four keys)
  const uint16_t *const v_lane = lds_v + (half * 8 + (lane & 15) / 4) * VR + (lane & 16) + (lane & 3) * 4;
  typedef short s16x4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4_t *lds_s16x4;
  auto load_v_operands = [&](int kb, int c) {
#pragma unroll
    for (int d = 0; d < NDB; ++d) {
      const uint16_t *at = vx + (kb * 32 + c * 16) * VR + d * 32;
      const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(at)));
      const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(at + 4 * VR)));
      vta[d] = u32x4_t{lo.x, lo.y, hi.x, hi.y};
    }
  };
  auto qk = [&](int kb) {
    if constexpr (MFMA_PRIO) __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int j = 0; j < 16; ++j) sacc[j] = 0.f;
    const uint16_t *const krow = kx + (kb * 32 + kperm(col)) * KR + half * 8;
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) sacc = mfma_32x32x16<F16>(*reinterpret_cast<const u32x4_t *>(krow + ch * 16), qb[ch], sacc);
    if constexpr (MFMA_PRIO) __builtin_amdgcn_s_setprio(0);
  };

  // logits -> P^T operands of one block: online softmax against a lazily moved reference
  auto softmax = [&](int kb) {
    float z[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = __builtin_fmaf(p.scale_log2e, sacc[i], -m_ref);
    // mask: block-causal key limit and the ragged last tile (register i of this lane <-> key kb*32 + 16*(i/8) + 8*half + i%8 of the tile)
    if (t0 + (KS == 1 ? BN : kb * 32 + 32) > wave_minlim) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = t0 + kb * 32 + 16 * (i >> 3) + 8 * half + (i & 7);
        if (key >= limit) z[i] = -INFINITY;
      }
    }
    // Moves the softmax reference to the row's current maximum: up only (never down) once
    // something has been accumulated; the very first block takes its maximum as it is, negative
    // or not (the accumulators are still zero, so alpha = 1 is exact).
    auto move_reference = [&]() {
      float zmax = z[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) zmax = fmaxf(zmax, z[i]);
      // the other lane half of the same query, without a trip through LDS
      const auto sw = __builtin_amdgcn_permlane32_swap(f2u(zmax), f2u(zmax), false, false);
      zmax = fmaxf(u2f(sw[0]), u2f(sw[1]));
      const float delta = first ? (zmax == -INFINITY ? 0.f : zmax) : fmaxf(zmax, 0.f);
      m_ref += delta;
#pragma unroll
      for (int i = 0; i < 16; ++i) z[i] -= delta;
      if (!first) {
        const float alpha = __builtin_amdgcn_exp2f(-delta);
#pragma unroll
        for (int d = 0; d < NDB; ++d)
#pragma unroll
          for (int j = 0; j < 16; ++j) oacc[d][j] *= alpha;
        l_part *= alpha;
      }
    };
    // exp2 of the logits, rounded to pairs of the attention's type for the MFMA, and their sum (this lane's keys)
    float blk = 0.f;
    auto weights = [&]() {
      float pv[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) pv[i] = __builtin_amdgcn_exp2f(z[i]);
      blk = 0.f;
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const u32 w = pack_io_rne<F16>(pv[i], pv[i + 1]);
        pop[i >> 3][(i & 7) >> 1] = w;
      }
      float part[4];   // (four of its weights each, and no sum waits for another)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < 2; ++i) part[2 * c + i] = add4<F16>(f32x4_t{0.f, 0.f, 0.f, 0.f}, make_uint2(pop[c][2 * i], pop[c][2 * i + 1]))[0];
      blk = (part[0] + part[1]) + (part[2] + part[3]);
    };
    // The reference has to move when a logit exceeds it by 2^16.  Rather than look for the
    // row maximum in every block (eleven instructions of sixty), the weights are computed
    // against the reference as it stands and their sum is looked at, which the denominator
    // needs anyway: a weight above 2^16 (or an overflow to infinity) shows in it, and the block
    // is then redone with the reference moved.  (A sum above 2^16 without such a weight moves
    // the reference too, which is harmless.)
    // (fp16 weights end at 65504: there the reference moves at a block sum of 2^15, which keeps
    // every weight of an accepted block finite; an overflowed one makes the sum infinite)
    constexpr float kMoveAt = F16 ? 32768.f : 65536.f;
    if (first) move_reference();
    weights();
    if (!first && __any(!(blk <= kMoveAt))) {
      move_reference();
      weights();
    }
    l_part += blk;
    first = false;
  };

  // O^T += V^T P^T for the 32 keys of one block
  auto pv_mfma = [&](int kb) {
    if constexpr (MFMA_PRIO) __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      u32x4_t av[NDB];
#pragma unroll
      for (int d = 0; d < NDB; ++d) av[d] = vta[d];
      if (c == 0) {
        load_v_operands(kb, 1);   // in flight under this chunk's MFMAs
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int d = 0; d < NDB; ++d) oacc[d] = mfma_32x32x16<F16>(av[d], u32x4_t{pop[c][0], pop[c][1], pop[c][2], pop[c][3]}, oacc[d]);
    }
    if constexpr (MFMA_PRIO) __builtin_amdgcn_s_setprio(0);
  };

  // The key blocks behind the last key that a query of this wavefront sees add nothing (every weight there
  // would be exp2(-inf) = 0): the end of the cache and, under a key limit, whatever the workgroup's other
  // wavefronts still need.  A whole sequence of 680 tokens in ten steps, [8,680,16,64] fp16: a quarter of
  // the workgroups' key blocks; with the order of the query tiles (BlockOf) append and attention 47.5 -> 39.7 us.
  const int block0 = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(share * 32);   // the first key of a tile that the wavefront attends
  const int wave_tiles = __builtin_amdgcn_readfirstlane(wave_live ? min(n_tiles, (max(wave_end - tile_base - block0, 0) + TB - 1) / TB) : 0);
  // with the MFMAs of a block in flight: the next tile is widened into the other buffers
  auto widen_next = [&](int tile) {
    if (tile + 1 >= n_tiles) return;
    widen(tile + 1);
    if (tile + 2 < n_tiles) request();
  };
  auto attend = [&](int tile) {
    t0 = tile_base + tile * TB + block0;
    kx = lds_k + tile % L::kBufs * KBUF + block0 * KR;
    vx = v_lane + tile % L::kBufs * VBUF + block0 * VR;
    const bool half_tile = wave_end - t0 <= 32;
#pragma unroll
    for (int kb = 0; kb < (KS == 1 ? 2 : 1); ++kb) {
      if (kb == 1 && half_tile) continue;
      qk(kb);
      load_v_operands(kb, 0);   // used after the softmax arithmetic
      __builtin_amdgcn_sched_barrier(0);
      softmax(kb);
      pv_mfma(kb);
      if (!ONE && kb == 0) widen_next(tile);
    }
  };
  int tile = 0;
  if constexpr (ONE) {
    // one of each buffer: a tile is widened and attended in turn, with the next one's loads in flight
    for (; tile < n_tiles; ++tile) {
      if (tile) __syncthreads();   // (the tile before is attended)
      widen(tile);
      if (tile + 1 < n_tiles) request();
      __syncthreads();
      if (tile < wave_tiles) attend(tile);
    }
  } else {
    for (; tile < wave_tiles; ++tile) {
      attend(tile);
      __syncthreads();   // the one barrier per tile
    }
    // from there on (a wavefront without queries: from the start) the wavefront only helps with the
    // widening, at the same barrier count as the others
    for (; tile < n_tiles; ++tile) {
      widen_next(tile);
      __syncthreads();
    }
  }
  // ---- epilogue -------------------------------------------------------------------
  if constexpr (KS == 1) {
    if (!wave_live) return;
    const float l_sum = l_part + __shfl_xor(l_part, 32, 64);
    store_block<D, F16>(p, b, hq, qrow, q_live, half, split, out_pair, m_ref, l_sum, oacc, [](float o) { return o; });
  } else {
    // The wavefronts of a block of queries: each hands the others the quads of rows of O^T (four registers, u-th of D / 8) that those put together, weighted
    // by the softmax mass against the largest reference of all (none where it saw no key; a NaN counts, and makes the result one).
    constexpr int OWN = D / 8 / KS;
    if constexpr (ONE) __syncthreads();   // (every tile is attended)
    float2 *const stats = reinterpret_cast<float2 *>(lds_raw);                       // [NWV / KS][KS][32]
    float4 *const handed = reinterpret_cast<float4 *>(lds_raw + L::kStats);          // [NWV / KS][to: KS][from: KS - 1][OWN][64]
    const float l_own = l_part + __shfl_xor(l_part, 32, 64);
    if (l_own == 0.f) {   // (the query sees none of the share's keys: an infinity or NaN among them, times 0, has no say either)
#pragma unroll
      for (int d = 0; d < NDB; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[d][i] = 0.f;
    }
    if (half == 0) stats[(qwave * KS + share) * 32 + col] = make_float2(m_ref, l_own);
    __syncthreads();
    float M = -INFINITY, l_sum = 0.f, w_own = 0.f;
    float2 of[KS];
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      of[i] = stats[(qwave * KS + i) * 32 + col];
      if (of[i].y != 0.f) M = fmaxf(M, of[i].x);
    }
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const float w = of[i].y != 0.f ? __builtin_amdgcn_exp2f(of[i].x - M) : 0.f;
      l_sum = __builtin_fmaf(w, of[i].y, l_sum);
      if (i == share) w_own = w;
    }
    if (wave_live) {
#pragma unroll
      for (int to = 0; to < KS; ++to) {
        if (to == share) continue;
        float4 *const dst = handed + ((qwave * KS + to) * (KS - 1) + (share < to ? share : share - 1)) * OWN * 64 + lane;
#pragma unroll
        for (int u = 0; u < OWN; ++u) {
          const int r = to * OWN + u;
          dst[u * 64] = make_float4(oacc[r / 4][r % 4 * 4] * w_own, oacc[r / 4][r % 4 * 4 + 1] * w_own, oacc[r / 4][r % 4 * 4 + 2] * w_own, oacc[r / 4][r % 4 * 4 + 3] * w_own);
        }
      }
    }
    __syncthreads();
    if (!q_live) return;
    const float inv = l_sum > 0.f ? 1.0f / l_sum : 0.f;
    const bool shared_out = p.nsplit > 1;
    __bf16 *const optr = p.out + (b * p.o_bs + hq * p.o_hs + qrow * p.o_ts) * D;
    const int64_t prow = ((int64_t)split * p.bh_total + out_pair) * p.Lq + qrow;
    float *const wptr = p.ws_o + prow * D;
    if (shared_out && half == 0 && share == 0) *reinterpret_cast<float2 *>(p.ws_ml + prow * 2) = make_float2(M == -INFINITY ? 0.f : M, l_sum);
#pragma unroll
    for (int to = 0; to < KS; ++to) {   // (registers are named at compile time)
      if (to != share) continue;
      const float4 *const src = handed + (qwave * KS + to) * (KS - 1) * OWN * 64 + lane;
#pragma unroll
      for (int u = 0; u < OWN; ++u) {
        const int r = to * OWN + u;
        float4 o = make_float4(oacc[r / 4][r % 4 * 4] * w_own, oacc[r / 4][r % 4 * 4 + 1] * w_own, oacc[r / 4][r % 4 * 4 + 2] * w_own, oacc[r / 4][r % 4 * 4 + 3] * w_own);
#pragma unroll
        for (int from = 0; from < KS - 1; ++from) {
          const float4 x = src[(from * OWN + u) * 64];
          o.x += x.x; o.y += x.y; o.z += x.z; o.w += x.w;
        }
        o.x *= inv; o.y *= inv; o.z *= inv; o.w *= inv;
        const int at = r / 4 * 32 + 8 * (r % 4) + 4 * half;
        if (shared_out) *reinterpret_cast<float4 *>(wptr + at) = o;
        else *reinterpret_cast<uint2 *>(optr + at) = make_uint2(pack_io_rne<F16>(o.x, o.y), pack_io_rne<F16>(o.z, o.w));
      }
    }
  }
}

// Workgroup -> (pair, query tile, share of the keys).  XCD-aware: consecutive workgroup ids go to different
// XCDs (8 of them), so ids congruent mod 8 share an L2.  An XCD takes a run of the pairs' query tiles and shares, pair after pair, an eighth
// of all: a pair's packed K/V stay in one L2 (or two), as do the cache lines that neighbouring heads of a token-major cache share.  (Whole pairs to an
// XCD are one for six of them and none for two where there are six, and four for some where there are 25: of 104 random forms whose pairs are no multiple of
// eight this order alone makes the launches 1.05 times as fast on the geometric mean, up to 1.78 and none slower than 0.98 without limits; of 296 others 1.00, 0.96 to 1.06.)
// Under key limits the tiles that see the most keys come first: in windows of an XCD's pairs (HeavyFirst), or with fewer than 64 pairs that are no
// multiple of eight, which whole pairs would spread unevenly, over all pairs.  (Without shares the division by their number is left out there: 0.5 % of a launch.)
struct BlockOf {
  int pair, qt, split;
  __device__ __forceinline__ explicit BlockOf(const AttnParams &p) {
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    if (p.kv_limit && p.q_tiles > 1) {
      if (spread_limits(p.bh_total)) {
        const int unit = p.nsplit > 1 ? blockIdx.x / p.nsplit : blockIdx.x, back = unit / p.bh_total;
        split = blockIdx.x - unit * p.nsplit;
        pair = back < p.q_tiles ? unit - back * p.bh_total : p.bh_total;
        qt = p.q_tiles - 1 - back;
        return;
      }
      // (windows of the pairs whose workgroups are resident together, 64 on an XCD at two per compute unit)
      const int groups = (p.bh_total + 7) >> 3, rest = p.nsplit > 1 ? slot / p.nsplit : slot;   // pairs of an XCD
      const HeavyFirst k(rest, p.q_tiles, groups, max(64 / p.q_tiles, 1));
      split = slot - rest * p.nsplit;
      qt = k.qt;
      pair = p.kv_hs == 1 && p.kv_ts > 1 ? xcd * groups + k.grp : k.grp * 8 + xcd;
      return;
    }
    const int unit = xcd * ((p.bh_total * p.q_tiles * p.nsplit + 7) >> 3) + slot, tile = unit / p.nsplit;
    split = unit - tile * p.nsplit;
    pair = tile / p.q_tiles;
    qt = tile - pair * p.q_tiles;
  }
  __host__ __device__ static bool spread_limits(int pairs) { return pairs < 64 && pairs % 8 != 0; }
  static dim3 grid(const AttnParams &p) {
    if (p.kv_limit && p.q_tiles > 1 && !spread_limits(p.bh_total)) return dim3((unsigned)((p.bh_total + 7) / 8 * 8 * p.q_tiles * p.nsplit));
    return dim3((unsigned)(((int64_t)p.bh_total * p.q_tiles * p.nsplit + 7) / 8 * 8));
  }
};

// WPS: wavefronts per SIMD the register allocation aims at (2, or 4: two 8-wavefront workgroups
// per compute unit at 128 registers, which the D=64 kernels afford)
template <int D, int BITS, bool CHAN, int NWV, int WPS, bool F16, bool ONE, int KS>
__global__ __launch_bounds__(NWV * 64, WPS) void fused_attn_kernel(AttnParams p) {
  const BlockOf k(p);
  if (k.pair >= p.bh_total) return;
  attend_tiles<D, BITS, CHAN, NWV, F16, ONE, KS>(p, k.pair, k.pair, k.qt, k.split);
}

template <int D, int NWV, int WPS, bool F16, int KS>
__global__ __launch_bounds__(NWV * 64, WPS) void fused_attn_classes_kernel(AttnParams p, ClassTable t) {
  const BlockOf k(p);
  if (k.pair >= p.bh_total) return;
  p.kv_ts = 1;   // (heads first, which a constant tells the compiler: rows as far apart as they are long)
  in_class(p, t, k.pair, [&](auto bits, int bh, int out_pair) __attribute__((always_inline)) {
    attend_tiles<D, decltype(bits)::value, false, NWV, F16, false, KS>(p, bh, out_pair, k.qt, k.split);
  });
}

// ... and with exact codes
template <int BITS>
__global__ __launch_bounds__(NW * 64, 2) void exact_attn_kernel(AttnParams p) {
  const BlockOf k(p);
  if (k.pair >= p.bh_total) return;
  attend_codes<BITS>(p, k.pair, k.pair, k.qt, k.split);
}

// Where four channels of a packed row go.  (Rows fit 32 bits: so many, times the shares of a partial result, are more than any memory.  Divided in
// 64 bits they were half of the combining kernels' instructions.)
template <int D> __device__ __forceinline__ __bf16 *out_of_row(const AttnParams &p, u32 row, int c0) {
  const u32 bh = row / (u32)p.Lq, qrow = row - bh * (u32)p.Lq, b = bh / (u32)p.Hkv, hs = bh - b * (u32)p.Hkv;
  const int hq = p.head_map ? p.head_map[hs] : (int)hs;
  return p.out + ((int64_t)b * p.o_bs + hq * p.o_hs + (int64_t)qrow * p.o_ts) * D + c0;
}

// The shares' outputs weighted by their softmax mass l * 2^(m - M), M the largest reference among
// the shares that saw a key.  (A share that saw none has the mass 0; one whose logits held a NaN has NaN for its mass, which
// is not to be taken for 0, or the result would be finite where the unshared kernel's is NaN.)  A workgroup of 256 threads serves 2 query rows x (D/4) channel quads
// x G groups of shares (G = 4 at D=128, 8 at D=64: the threads of a quad split the shares among
// them): the weights of a row's shares are formed once, in LDS, and every thread then sums its
// shares' quads with nothing between the loads but the weights.
template <int D, bool F16>
__global__ __launch_bounds__(256) void combine_splits_kernel(AttnParams p) {
  constexpr int QUADS = D / 4, ROWS = 2, G = 256 / (ROWS * QUADS);
  constexpr int kMaxS = 64, kEarly = 4;
  static_assert(G >= 1 && kMaxS >= kMaxKeyShares_v && kMaxS >= kMaxSplits_v, "share counts");
  __shared__ float w_lds[ROWS][kMaxS];
  const int64_t rows = (int64_t)p.bh_total * p.Lq;
  const int tid = threadIdx.x;
  const int64_t row0 = (int64_t)blockIdx.x * ROWS;
  const int r = tid / (QUADS * G), gq = tid % (QUADS * G), grp = gq / QUADS, c0 = (gq % QUADS) * 4;
  const int64_t row = row0 + r, row_c = row < rows ? row : rows - 1;
  // The thread's first shares are requested along with the statistics, and a row's weights are formed by the wavefront whose lanes are its
  // shares: one trip to memory instead of two, and no loop over the shares (16 shares of 512 rows, D=128, with the launch before it: 20.4 -> 19.4 us).
  const float *const o_row = p.ws_o + row_c * D + c0;
  float4 o[kEarly];
#pragma unroll
  for (int u = 0; u < kEarly; ++u) o[u] = *reinterpret_cast<const float4 *>(o_row + (int64_t)min(grp + u * G, p.nsplit - 1) * rows * D);
  static_assert(kMaxS == 64 && ROWS * kMaxS <= 256, "one wavefront per row, one lane per share");
  if (tid < ROWS * kMaxS) {
    const int wr = tid / kMaxS, wsh = tid % kMaxS;
    float2 ml = make_float2(0.f, 0.f);   // (denominator 0: an empty share)
    if (wsh < p.nsplit && row0 + wr < rows) ml = *reinterpret_cast<const float2 *>(p.ws_ml + ((int64_t)wsh * rows + row0 + wr) * 2);
    const float m_max = group_allreduce<64, true>(ml.y != 0.f ? ml.x : -INFINITY);
    w_lds[wr][wsh] = ml.y != 0.f ? ml.y * __builtin_amdgcn_exp2f(ml.x - m_max) : 0.f;
  }
  __syncthreads();
  float acc[4] = {0.f, 0.f, 0.f, 0.f}, wsum = 0.f;
  auto add = [&](int share, float4 x) {
    const float w = w_lds[r][share];
    acc[0] = __builtin_fmaf(w, x.x, acc[0]); acc[1] = __builtin_fmaf(w, x.y, acc[1]);
    acc[2] = __builtin_fmaf(w, x.z, acc[2]); acc[3] = __builtin_fmaf(w, x.w, acc[3]);
    wsum += w;
  };
#pragma unroll
  for (int u = 0; u < kEarly; ++u)
    if (grp + u * G < p.nsplit) add(grp + u * G, o[u]);
#pragma unroll 4
  for (int s_ = grp + kEarly * G; s_ < p.nsplit; s_ += G) add(s_, *reinterpret_cast<const float4 *>(o_row + (int64_t)s_ * rows * D));
  if constexpr (G > 1) {
    // the groups of a row's shares meet through LDS (group 0 collects)
    __shared__ float part[256][5];
    part[tid][0] = acc[0]; part[tid][1] = acc[1]; part[tid][2] = acc[2]; part[tid][3] = acc[3]; part[tid][4] = wsum;
    __syncthreads();
    if (grp != 0) return;
#pragma unroll
    for (int g2 = 1; g2 < G; ++g2) {
      const float *o = part[tid + g2 * QUADS];
      acc[0] += o[0]; acc[1] += o[1]; acc[2] += o[2]; acc[3] += o[3]; wsum += o[4];
    }
  }
  if (row >= rows) return;
  const float inv = wsum > 0.f ? 1.0f / wsum : 0.f;
  *reinterpret_cast<uint2 *>(out_of_row<D>(p, (u32)row, c0)) = make_uint2(pack_io_rne<F16>(acc[0] * inv, acc[1] * inv), pack_io_rne<F16>(acc[2] * inv, acc[3] * inv));
}

// The same for a handful of shares and many rows: a thread sums four channels of one row over all
// shares, nothing passes through LDS.  (With the kernel above, two rows and three barriers to a
// workgroup, two shares of 32 768 rows took 18.9 us for the 50 MB they are.)
// NS: the shares, or the most of them; U: rows of a thread (two shares, D=128, 1024 queries of 32 pairs, the call with its producer and
// attention: one row 77.5 us, two 76.7, four 77.7; 77.9 with rows divided in 64 bits).
template <int D, bool F16, int NS, int U>
__global__ __launch_bounds__(256) void combine_few_splits_kernel(AttnParams p) {
  const int64_t rows = (int64_t)p.bh_total * p.Lq;
  const int64_t row0 = (int64_t)blockIdx.x * (U * 1024 / D) + threadIdx.x / (D / 4);
  const int c0 = threadIdx.x % (D / 4) * 4, n = NS == 2 ? 2 : p.nsplit;
  float2 ml[U][NS];
  float4 o[U][NS];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t row = row0 + u * (1024 / D);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      ml[u][s] = make_float2(0.f, 0.f);
      if (s < n && row < rows) {
        ml[u][s] = *reinterpret_cast<const float2 *>(p.ws_ml + ((int64_t)s * rows + row) * 2);
        o[u][s] = *reinterpret_cast<const float4 *>(p.ws_o + ((int64_t)s * rows + row) * D + c0);
      }
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t row = row0 + u * (1024 / D);
    if (row >= rows) return;
    float M = -INFINITY;
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (ml[u][s].y != 0.f) M = fmaxf(M, ml[u][s].x);
    float acc[4] = {0.f, 0.f, 0.f, 0.f}, wsum = 0.f;
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (s < n && ml[u][s].y != 0.f) {
        const float w = ml[u][s].y * __builtin_amdgcn_exp2f(ml[u][s].x - M);
        acc[0] = __builtin_fmaf(w, o[u][s].x, acc[0]); acc[1] = __builtin_fmaf(w, o[u][s].y, acc[1]);
        acc[2] = __builtin_fmaf(w, o[u][s].z, acc[2]); acc[3] = __builtin_fmaf(w, o[u][s].w, acc[3]);
        wsum += w;
      }
    const float inv = wsum > 0.f ? 1.0f / wsum : 0.f;
    *reinterpret_cast<uint2 *>(out_of_row<D>(p, (u32)row, c0)) =
        make_uint2(pack_io_rne<F16>(acc[0] * inv, acc[1] * inv), pack_io_rne<F16>(acc[2] * inv, acc[3] * inv));
  }
}

template <int D, bool F16> void launch_combine(const AttnParams &p, hipStream_t st) {
  const int64_t rows = (int64_t)p.bh_total * p.Lq;
  // (few rows: the threads of a row sharing its shares out are what fills the device)
  constexpr int R = 1024 / D;
  if (p.nsplit == 2 && rows >= 4096)
    hipLaunchKernelGGL((combine_few_splits_kernel<D, F16, 2, 2>), dim3((unsigned)((rows + 2 * R - 1) / (2 * R))), dim3(256), 0, st, p);
  else if (p.nsplit <= kMaxSplits_v && rows >= 4096)
    hipLaunchKernelGGL((combine_few_splits_kernel<D, F16, kMaxSplits_v, 1>), dim3((unsigned)((rows + R - 1) / R)), dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL((combine_splits_kernel<D, F16>), dim3((unsigned)((rows + 1) / 2)), dim3(256), 0, st, p);
}

template <int D, int BITS, bool CHAN, int NWV, int WPS = 2, bool F16 = false, bool ONE = false, int KS = 1>
void launch_shape(const AttnParams &p, hipStream_t st) {
  // (the per-channel tables take LDS by the number of segments of the launch, and half of it without zero-points)
  using L = TileLds<D, ONE, KS>;
  constexpr int lds_base = L::kTables, lds_max = std::max(lds_base + (CHAN ? kMaxSegments * 4 * D * 4 : 0), L::kJoin);
  static_assert(lds_max <= 160 * 1024, "LDS budget");
  const int lds_bytes = std::max(lds_base + (CHAN ? p.nseg * (p.k_chan_zp || p.v_chan_zp ? 4 : 2) * D * 4 : 0), L::kJoin);
  static bool configured[64] = {false};
  allow_lds(reinterpret_cast<const void *>(&fused_attn_kernel<D, BITS, CHAN, NWV, WPS, F16, ONE, KS>), lds_max, configured);
  hipLaunchKernelGGL((fused_attn_kernel<D, BITS, CHAN, NWV, WPS, F16, ONE, KS>), BlockOf::grid(p), dim3(NWV * 64), lds_bytes, st, p);
  if (p.nsplit > 1) launch_combine<D, F16>(p, st);
}
template <int BITS> void launch_exact(const AttnParams &p, hipStream_t st) {
  constexpr int lds_bytes = ExactLds<BITS>::kBytes;
  static bool configured[64] = {false};
  allow_lds(reinterpret_cast<const void *>(&exact_attn_kernel<BITS>), lds_bytes, configured);
  hipLaunchKernelGGL((exact_attn_kernel<BITS>), BlockOf::grid(p), dim3(NW * 64), lds_bytes, st, p);
  if (p.nsplit > 1) launch_combine<128, false>(p, st);
}

// The workgroups at D=64, F16 or not.
template <int BITS, bool CHAN, bool F16> void launch_d64(const AttnParams &p, hipStream_t st) {
  if (p.key_waves == 2) return launch_shape<64, BITS, CHAN, 8, 4, F16, false, 2>(p, st);
  if (p.key_waves == 4) return launch_shape<64, BITS, CHAN, 8, 4, F16, false, 4>(p, st);
  // More (batch, head) pairs than compute units, at most four wavefronts of queries each:
  // workgroups of four wavefronts (same arithmetic, same results).  Also for one or two
  // wavefronts of queries: the wavefronts without queries share the widening
  // of the tiles, which is what such a workgroup spends its time on.
  // Such a workgroup is a chain of loads, barriers and short computations, so what counts is how many are resident.  Two of each
  // buffer are 36 864 bytes: four workgroups to a compute unit, three with the tables of eight steps or more (four with zero-points) behind
  // them and, by its registers (132), with 8-bit codes in groups.  One of each: four always, though for 8-bit codes in groups at the price of
  // 24 bytes of spills.  From more pairs on than one round of three, one buffer gains where two would leave three workgroups, and elsewhere
  // they come out the same; 2-bit codes in groups lose a little and keep two.  Two buffers / one, us, fp16 [64,n,16,64] (1024 pairs), 36 queries x
  // 91 keys, 64 x 155, 100 x 600, 128 x 1250: 8 bits with ten tables 14.7 / 11.1, 19.6 / 14.8, 43.8 / 38.1, 81.3 / 71.1, with five
  // 10.5 / 10.3, 13.4 / 13.7, 37.2 / 36.9, 70.8 / 70.8, in groups of 32 10.6 / 10.4, 16.4 / 15.5, 43.5 / 42.5, 85.2 / 81.2; 4 bits in groups 9.6 /
  // 9.6, 13.8 / 13.5, 39.9 / 40.2, 78.8 / 79.1; 2 bits in groups 10.0 / 10.0, 13.9 / 13.8, 41.3 / 42.1, 79.8 / 80.4; 768 pairs, 8 bits with ten tables
  // 9.6 / 9.8, 11.9 / 12.5, 31.4 / 31.3, 56.9 / 56.8, in groups 8.2 / 9.0, 11.1 / 12.3, 32.5 / 33.4, 63.4 / 64.7.  A single tile of keys has nothing to pipeline, and one
  // buffer is the same with tables (64 queries x 64 keys, three tables, 512 pairs 6.5 / 6.6, 1920 16.3 / 16.1); in groups it is behind,
  // 4 bits 5.6 / 5.8, 13.6 / 13.8, 8 bits 5.6 / 6.5, 15.6 / 16.4.
  if (p.Lq <= 128 && p.bh_total > device_cus()) {
    const bool rounds = (int64_t)p.bh_total * p.nsplit > 3 * device_cus() && (CHAN || BITS != 2);
    if (p.Lk <= BN || rounds) launch_shape<64, BITS, CHAN, 4, 4, F16, true>(p, st);
    else launch_shape<64, BITS, CHAN, 4, 3, F16>(p, st);
    return;
  }
  // (114 to 122 registers, no spills: two resident workgroups per compute unit hide each other's prologue and barriers)
  launch_shape<64, BITS, CHAN, 8, 4, F16>(p, st);
}

template <int D, int BITS, bool CHAN> void launch(const AttnParams &p, hipStream_t st) {
  if constexpr (D == 64) {
    // fp16 operands (the VAR path; every VAR model has head dim 64) or bf16 ones
    if (p.f16) launch_d64<BITS, CHAN, true>(p, st);
    else launch_d64<BITS, CHAN, false>(p, st);
  } else if (p.key_waves == 2) {
    launch_shape<D, BITS, CHAN, 8, 2, false, false, 2>(p, st);
  } else if (p.key_waves == 4) {
    launch_shape<D, BITS, CHAN, 8, 2, false, CHAN, 4>(p, st);
  } else {
    launch_shape<D, BITS, CHAN, 8>(p, st);
  }
}
template <bool CHAN> void launch_any(const AttnParams &p, int D, int bits, hipStream_t st) {
  if (D == 128) {
    if (bits == 4) launch<128, 4, CHAN>(p, st);
    else if (bits == 8) launch<128, 8, CHAN>(p, st);
    else launch<128, 2, CHAN>(p, st);
  } else {
    if (bits == 4) launch<64, 4, CHAN>(p, st);
    else if (bits == 8) launch<64, 8, CHAN>(p, st);
    else launch<64, 2, CHAN>(p, st);
  }
}

// the scale groups that are served
bool groups_served(int D, int gk, int gv) {
  return ((gk == gv && (gk == 128 || gk == 64 || gk == 32)) || (gk == 32 && gv == 64)) && gk <= D;
}

template <int D, int NWV, int WPS, bool F16, int KS = 1>
void launch_classes_shape(const AttnParams &p, const ClassTable &t, hipStream_t st) {
  constexpr int lds = std::max(TileLds<D, false, KS>::kTables, TileLds<D, false, KS>::kJoin);
  static bool configured[64] = {false};
  allow_lds(reinterpret_cast<const void *>(&fused_attn_classes_kernel<D, NWV, WPS, F16, KS>), lds, configured);
  hipLaunchKernelGGL((fused_attn_classes_kernel<D, NWV, WPS, F16, KS>), BlockOf::grid(p), dim3(NWV * 64), lds, st, p, t);
  if (p.nsplit > 1) launch_combine<D, F16>(p, st);
}
// (the workgroup sizes by the rules of launch())
template <int D> void launch_classes(const AttnParams &p, const ClassTable &t, hipStream_t st) {
  if constexpr (D == 64) {
    const bool four = p.Lq <= 128 && p.bh_total > device_cus();
    if (p.key_waves == 2) { if (p.f16) launch_classes_shape<D, 8, 4, true, 2>(p, t, st); else launch_classes_shape<D, 8, 4, false, 2>(p, t, st); return; }
    if (p.key_waves == 4) { if (p.f16) launch_classes_shape<D, 8, 4, true, 4>(p, t, st); else launch_classes_shape<D, 8, 4, false, 4>(p, t, st); return; }
    if (p.f16) { if (four) launch_classes_shape<D, 4, 3, true>(p, t, st); else launch_classes_shape<D, 8, 4, true>(p, t, st); }
    else { if (four) launch_classes_shape<D, 4, 3, false>(p, t, st); else launch_classes_shape<D, 8, 4, false>(p, t, st); }
  } else if (p.key_waves == 2) {
    launch_classes_shape<D, 8, 2, false, 2>(p, t, st);
  } else if (p.key_waves == 4) {
    launch_classes_shape<D, 8, 2, false, 4>(p, t, st);
  } else {
    launch_classes_shape<D, 8, 2, false>(p, t, st);
  }
}

int set_layout(AttnParams &p, int layout, const char *who) {
  if (layout == VARQ_LAYOUT_BHLC || layout == VARQ_LAYOUT_BHLC_OUT_BLHC) {
    p.q_bs = (int64_t)p.Hq * p.Lq; p.q_hs = p.Lq; p.q_ts = 1;
    p.kv_bs = (int64_t)p.Hkv * p.Lstride; p.kv_hs = p.Lstride; p.kv_ts = 1;
  } else if (layout == VARQ_LAYOUT_BLHC) {
    p.q_bs = (int64_t)p.Lq * p.Hq; p.q_hs = 1; p.q_ts = p.Hq;
    p.kv_bs = (int64_t)p.Lstride * p.Hkv; p.kv_hs = 1; p.kv_ts = p.Hkv;
  } else {
    return varq_set_error(VARQ_ERR_INVALID, "%s: layout must be VARQ_LAYOUT_BHLC (0), VARQ_LAYOUT_BLHC (1) or VARQ_LAYOUT_BHLC_OUT_BLHC (2), got %d", who, layout);
  }
  p.o_bs = p.q_bs; p.o_hs = p.q_hs; p.o_ts = p.q_ts;
  if (layout == VARQ_LAYOUT_BHLC_OUT_BLHC) { p.o_bs = (int64_t)p.Lq * p.Hq; p.o_hs = 1; p.o_ts = p.Hq; }
  return VARQ_OK;
}

// ---- sharing the keys of a query block out over several workgroups ---------------------
constexpr int kMaxSplits = kMaxSplits_v;

size_t split_workspace_bytes(int splits, int64_t rows, int D) {
  return splits > 1 ? (size_t)splits * (size_t)rows * (size_t)(D + 2) * sizeof(float) : 0;
}

// How the keys of a block of 256 queries are shared out: over `splits` workgroups, whose partial results take a second launch, and with `waves` 2 or 4
// over that many wavefronts of a workgroup, which then serves a half or a quarter of the queries and widens every tile for them alone.
struct KeyShares { int waves, splits; };

// The shares that minimize a launch's modelled time: workgroups run one per compute unit in rounds, an eighth of them on each XCD (see
// BlockOf); a workgroup costs its tiles (of 128 keys where four wavefronts share them) plus a fixed prologue and epilogue, and with shares of wavefronts their
// joining.  Fitted to 386 random forms (6 to 960 pairs, 16 to 1100 queries, 17 to 4800 keys, groups and tables, 2, 4 and 8 bits), each with every choice: what this
// takes is 0.5 % behind the best of all on the geometric mean and 9 % ahead of workgroups alone, and in 5 of them behind those by more than 2.5 %.  4 bits in groups,
// us, workgroups alone / this: D=128, 32 pairs, 256 queries x 521 keys 22.6 / 16.5, 400 x 921 32.4 / 22.8, 64 pairs, 144 x 300 16.8 / 12.0, 256 x 521
// 27.2 / 17.4, 400 x 921 40.9 / 30.5, 128 pairs, 256 x 521 28.6 / 22.8; D=64, 32 pairs, 256 x 521 15.7 / 11.6, 1024 x 2521 50.1 / 43.4, 128 pairs, 256 x 521 19.1 / 15.1.
// Tables take a workgroup 0.1 us per KiB beyond the first one (their LDS, at D=64 with four wavefronts beyond 80 KiB one workgroup per compute unit instead of two): of 600 forms with 1, 5, 10 and
// 16 tables without that 31 were more than 3 % behind workgroups alone, by up to 28 %, with it 19, by up to 11 %, and 9.7 -> 10.1 % ahead of them on the geometric mean.
double tables_us(int nseg, int D) { return 0.1 * (nseg - 1) * (4 * D * 4) / 1024.0; }
// alone: what workgroups alone would be, where that is asked too (it is what the first round of the loop ends with).
KeyShares choose_shares(int64_t bh, int Lq, int Lk, int D, int nseg, int most_waves, int cus, KeyShares *alone = nullptr) {
  static const double tile_us[2][3] = {{1.45, 0.85, 1.1}, {2.07, 1.35, 1.9}};
  const double per_xcd = cus / 8.0;
  const bool wide = D == 128;
  KeyShares best = {1, 1};
  double best_us = 0.0;
  for (int waves = 1, i = 0; waves <= most_waves; waves *= 2, ++i) {
    // (a single tile has nothing to share; and what up to 128 queries, the first steps of a schedule, come to does not go by how many pairs a launch has,
    // which would gain up to a tenth in tables: 64 queries x 600 keys, 128 pairs, D=64 15.9 / 13.5, D=128 20.8 / 18.7)
    if (waves > 1 && (Lk <= BN || Lq <= 128)) break;
    const int tiles = (Lk + (waves == 4 ? 2 * BN : BN) - 1) / (waves == 4 ? 2 * BN : BN);
    const int64_t blocks = bh * ((Lq + BM / waves - 1) / (BM / waves));
    // (up to 128 queries half of the wavefronts have none, and widen only)
    const double tile = tile_us[wide][i] * (waves == 1 && Lq <= 128 ? 0.7 : 1.0), fixed = (wide ? 2.8 : 2.2) + (waves > 1 ? 1.1 : 0.0) + tables_us(nseg, D);
    for (int n = 1; n <= kMaxSplits; ++n) {
      if (n > 1 && (Lk + BN - 1) / BN / n < 2) break;
      double us = std::ceil((double)((blocks * n + 7) / 8) / per_xcd) * ((double)((tiles + n - 1) / n) * tile + fixed);
      if (n > 1) us += 2.4 + 2.0 * (double)split_workspace_bytes(n, bh * Lq, D) / 4.4e6;   // written and read
      if ((waves == 1 && n == 1) || us < best_us) { best_us = us; best = {waves, n}; }
    }
    if (waves == 1 && alone) *alone = best;
  }
  return best;
}
// Fills the fields of the shares of p from the caller's request.  splits: 0 = as the model above
// says, reduced to what the workspace holds; 1 = none; 2..8 = exactly that many.  limited: what limited_shares says, or null.
// (The device is asked for once, and the model too: every step of a schedule pays for it.)
int set_splits(AttnParams &p, int D, int most_waves, const KeyShares *limited, int splits, void *workspace, size_t workspace_bytes, const char *who) {
  p.nsplit = 1; p.ws_o = nullptr; p.ws_ml = nullptr;
  p.key_waves = 1;
  if (splits < 0 || splits > kMaxSplits)
    return varq_set_error(VARQ_ERR_INVALID, "%s: splits must be 0 (automatic) or 1..%d (got %d)", who, kMaxSplits, splits);
  const int64_t rows = (int64_t)p.bh_total * p.Lq;
  const bool unaligned = workspace && ((uintptr_t)workspace & 15);
  int n = splits;
  KeyShares alone = {1, 1}, k = {1, 1};
  if (splits == 0 && (!limited || unaligned)) k = choose_shares(p.bh_total, p.Lq, p.Lk, D, p.nseg, limited ? 1 : most_waves, device_cus(), &alone);
  // (a workspace that cannot be used is an error wherever workgroups alone would use it, and is not used otherwise)
  if (unaligned && alone.splits > 1 && workspace_bytes >= split_workspace_bytes(2, rows, D))
    return varq_set_error(VARQ_ERR_INVALID, "%s: the workspace must be 16-byte aligned", who);
  if (limited) {
    p.key_waves = limited->waves;
    n = unaligned ? 1 : limited->splits;
  } else if (splits == 0) {
    n = alone.splits;
    if (k.waves > 1 && (k.splits == 1 || (workspace && !unaligned && workspace_bytes >= split_workspace_bytes(k.splits, rows, D)))) {
      p.key_waves = k.waves;
      n = k.splits;
    }
  }
  p.q_tiles = (p.Lq + BM / p.key_waves - 1) / (BM / p.key_waves);
  if (splits > 1 && (!workspace || workspace_bytes < split_workspace_bytes(n, rows, D)))
    return varq_set_error(VARQ_ERR_INVALID, "%s: %d splits need a workspace of %zu bytes (got %zu)", who, n,
                          split_workspace_bytes(n, rows, D), workspace ? workspace_bytes : (size_t)0);
  while (n > 1 && (!workspace || workspace_bytes < split_workspace_bytes(n, rows, D))) --n;
  if (n <= 1) return VARQ_OK;
  if ((uintptr_t)workspace & 15) return varq_set_error(VARQ_ERR_INVALID, "%s: the workspace must be 16-byte aligned", who);
  if ((int64_t)((p.bh_total + 7) / 8 * 8) * p.q_tiles * n >= (1ll << 31))
    return varq_set_error(VARQ_ERR_INVALID, "%s: grid too large for %d splits", who, n);
  p.nsplit = n;
  p.ws_o = reinterpret_cast<float *>(workspace);
  p.ws_ml = p.ws_o + (size_t)n * (size_t)rows * (size_t)D;
  return VARQ_OK;
}


// ---- few queries (few_attn.hip) -----------------------------------------------------------------
// Launches of at most kFewQueries queries per (batch, head), in tiles of 32 that each dequantize the cache for themselves,
// against 256 a workgroup and staged tiles of 64 keys in the kernel above.  Measured, us, the kernel above / that one, 4-bit
// codes, one group, pairs of (batch, head) x queries x keys: up to 16 queries it is faster everywhere, D=64 32 x 16 x 32 3.9 / 3.8, 128 x 16 x 4096 40.4 /
// 18.1, 240 x 16 x 1024 19.7 / 8.6, D=128 32 x 8 x 21 4.7 / 4.6, 240 x 16 x 1024 28.1 / 17.5.  More queries have two columns of 16 to prepare first: from the
// second tile of keys on, D=64 32 x 24 x 64 4.1 / 5.0, x 128 5.1 / 5.0, x 256 7.1 / 5.9; D=128 5.2 / 6.6, 6.7 / 6.7.  Several tiles of queries that do not fit the device
// at once pay with longer caches only, D=64 240 x 64 (480 tiles) x 128 5.7 / 6.7, x 256 7.7 / 8.1, x 400 10.6 / 10.6, x 1024 20.3 / 17.4, 480 x 64 (960) x 256 10.6 / 12.7, x 512
// 17.7 / 18.4, x 768 25.0 / 24.2; three and four tiles not beyond the device, 240 x 100 x 1024 21.4 / 29.0, and not where the widening dominates, 128 x
// 100 x 1024 18.5 / 17.2, x 2048 27.1 / 29.5, x 4096 43.1 / 53.4.  (The kernel above got faster since these lines were drawn: where they cross at 256, 512 and
// 2048 keys it is up to a tenth ahead by now, at D=128, 128 x 100 x 2048, 37.5 / 44.1; 8-bit codes the same.)
constexpr int kFewQueries = 128;
constexpr int kMaxKeyShares = kMaxKeyShares_v;
bool fewq_eligible(int B, int Hkv, int Lq, int Lk, int D, int k_group, int v_group) {
  // (the kernel keeps 32-bit byte offsets inside one (batch, head): rows of up to D bytes, up to
  // Hkv rows from one key to the next, a few blocks of overshoot before the clamp)
  const int64_t q_tiles = (Lq + 31) / 32, tiles = (int64_t)B * Hkv * q_tiles;
  if (!((D == 64 || D == 128) && D % k_group == 0 && D % v_group == 0 && D / k_group <= kFewGroups && D / v_group <= kFewGroups && Lq > 0 &&
        Lq <= kFewQueries && ((int64_t)Lk + 32 * kFewBlock) * Hkv * D < (1ll << 32) && ((int64_t)B * Hkv + 7) / 8 * q_tiles <= 65535))   // (the grid's z extent)
    return false;
  if (Lq <= 16) return true;
  const int cus = device_cus();
  if (q_tiles > 2 && (tiles > 2 * cus || Lk > 2048)) return false;
  return Lk > (q_tiles == 1 || tiles <= cus ? 64 : tiles <= 2 * cus ? 255 : 511);
}
// Over how many workgroups the keys of a tile of queries are shared out: as many as are resident together (more would
// be a second round: 56 pairs x 2 queries x 41576 keys, ten shares each 108 us, nine 92), at least eight blocks each, and not
// at all for a cache so short that the second launch costs more.
int fewq_shares(int bh_total, int Lq, int Lk, int D, int k_group, int v_group) {
  const int64_t tiles = (int64_t)((bh_total + 7) / 8 * 8) * ((Lq + 31) / 32), nb = (Lk + kFewBlock - 1) / kFewBlock;
  if (nb < 24) return 1;
  const int64_t resident = D == 128 && k_group == D && v_group == D ? 2 * (int64_t)device_cus() : (int64_t)device_cus();
  const int64_t s = std::min(std::min(resident / tiles, nb / 8), (int64_t)kMaxKeyShares);
  return s < 1 ? 1 : (int)s;
}

// The split fields of a launch of the few-queries kernel: no more shares than the workspace holds.
void set_few(AttnParams &p, int D, int k_group, int v_group, void *workspace, size_t workspace_bytes) {
  const int64_t rows = (int64_t)p.bh_total * p.Lq;
  int n = fewq_shares(p.bh_total, p.Lq, p.Lk, D, k_group, v_group);
  while (n > 1 && (!workspace || ((uintptr_t)workspace & 15) || workspace_bytes < split_workspace_bytes(n, rows, D))) --n;
  p.q_tiles = (p.Lq + 31) / 32;
  p.nsplit = n;
  p.fq_share_blocks = ((p.Lk + kFewBlock - 1) / kFewBlock + n - 1) / n;
  // Eight wavefronts instead of four halve the chain of blocks of a share; where several workgroups run on a compute unit they
  // only cost registers (two columns of queries: one workgroup instead of three).  Below 1024 keys this does not go by the
  // number of pairs.  A pair's result is then the same whatever others the launch has, bit for bit, up to 736 keys and 16 queries: from 24 blocks
  // on fewq_shares goes by it, and beyond 16 queries fewq_eligible.
  const int nb = (p.Lk + kFewBlock - 1) / kFewBlock;
  const bool alone = nb < 32 ? p.Lq <= 16 : (int64_t)p.bh_total * p.q_tiles * n <= device_cus();
  p.few_waves = p.fq_share_blocks > 8 && alone ? 8 : 4;
  p.ws_o = n > 1 ? reinterpret_cast<float *>(workspace) : nullptr;
  p.ws_ml = n > 1 ? p.ws_o + (size_t)n * (size_t)rows * (size_t)D : nullptr;
}
// ... the second launch of one with shares
void combine_few(const AttnParams &p, int D, hipStream_t st) {
  if (p.nsplit <= 1) return;
  if (D == 128) launch_combine<128, false>(p, st);
  else if (p.f16) launch_combine<64, true>(p, st);
  else launch_combine<64, false>(p, st);
}

// ---- many queries: K and V expanded once, then a plain flash attention (wide_attn.hip) ----------
// The expanded K and V of a call take at most 1 GiB of the caller's memory at a time; a larger batch is expanded and attended
// part after part.  2.1 GB at once gain nothing over two parts, smaller parts end up to 8 % later (256 MiB / 512 MiB /
// 1 GiB / no bound, us, 4 bits): 384 pairs, 4096 x 10521, 7710 / 7710 / 7715 / 7760-8000; 1600 x 4121 1576 / 1508 / 1460 / 1460-1500; D=64,
// 960 pairs, 1600 x 4121 2312 / 2243 / 2214 / 2220.
constexpr int64_t kExpandBytes = 1ll << 30;
// That many batch entries are a part (0: not even one fits, and the call takes the kernel above).
int wide_batch(int B, int Hkv, int Lk, int D) {
  const int64_t most = kExpandBytes / ((int64_t)Hkv * ((Lk + BN - 1) / BN) * (2 * BN * D * 2));
  if (most >= B || most == 0) return most ? B : 0;
  const int64_t parts = (B + most - 1) / most;
  return (int)((B + parts - 1) / parts);
}
// Worth it from five (D = 128) or six blocks of 256 queries per (batch, head) on: expanding costs what
// widening costs the kernel above in a block or two, and then its way through memory; and on a device
// that is not nearly full the three launches cost more than they save.  Measured (us, 4-bit codes in groups, 8-bit ones with five tables,
// the kernel above / this): D=128 B=2 H=16 1024 x 2521 69.8 / 71.3, 63.3 / 71.8, 1300 x 3000 107 / 95, 104 / 95, 1600 x 4121 145 / 123, 138 / 125,
// 2304 x 6425 331 / 232, 329 / 243; B=8 1024 x 2521 191 / 194, 191 / 204, 1300 x 3000 318 / 285, 308 / 300, 2304 x 6425 1085 / 884, 1081 / 914; B=1 H=8
// 1600 x 4121 55 / 60, 54 / 63; D=64 B=2 1600 x 4121 98 / 90, 95 / 86, B=8 1300 x 3000 182 / 178, 177 / 180, 1600 x 4121 317 / 285, 304 / 294, 2304 x 6425 626 / 553,
// 607 / 567, but B=30 1600 x 4121 1030 / 1047, 995 / 1062.
// Under key limits (measured with the block-causal rule over a whole sequence, pairs x tokens): D=128 all of 16 to 128
// pairs x 2521 to 10521 are faster, 16 x 2521 91 / 86, 128 x 2521 339 / 322, 48 x 2952 228 / 183, 32 x 4121
// 284 / 197, 32 x 10521 1325 / 1038.  D=64 gains where the longest query blocks are the whole of the time, up to about
// a block and a quarter per compute unit, 16 x 2521 62.6 / 56.8, 24 x 3256 84.5 / 76.8 (though 16 x 4121 85.6 / 88.2), and in long sequences,
// 32 x 6425 322 / 272, 128 x 6425 1142 / 1050; in between it goes either way, 32 x 3256 89.5 / 100, 128 x 4121 513 / 489,
// 320 x 2952 645 / 683, 48 x 5417 328 / 319.  (Few pairs: wide_four.)
bool wide_eligible(int B, int Hkv, int Lq, int Lk, int D, bool limits, int cus = device_cus()) {
  const int64_t bh = (int64_t)wide_batch(B, Hkv, Lk, D) * Hkv, blocks = bh * ((Lq + 255) / 256);
  if (bh > 0 && wide_four(bh, Lq, Lk, D, cus, limits)) return true;
  if (limits && D == 64 && Lq < 6144 && blocks > cus * 5 / 4) return false;
  return Lq >= (D == 128 ? 1280 : 1536) && Lk >= 2048 && blocks >= 160 && bh <= 65535;
}
// Under key limits, whose blocks end at different keys that only the device knows; taken for a sequence's own, of which a block sees a quarter
// more than its share.  The time is that of the longest workgroup or of all of them evenly dealt out, and more where both are alike.  Shares of wavefronts also
// with splits = 1 (most = 1).  waves 0: K and V are expanded instead.  Fitted to 452 forms (2 to 360 pairs, whole sequences of 129 to 6000 tokens) with
// every choice: 1.2 % behind the best on the geometric mean, 18 % ahead of the rules before, blocks of 128 queries for few pairs (wide_four) and shares as without
// limits.  4 bits in groups, us, before / this: D=64, 2 pairs x 4500 tokens 52.7 / 31, 16 x 300 12.4 / 9.0, x 680 17.6 / 12.4, x 1500 29.1 / 24.6, 32 x 524 17.2 / 12.9, 48 x 1000 27.3 / 23.0;
// D=128, 2 x 4500 93 / 46, 16 x 680 24.8 / 17.3, 24 x 600 24.6 / 16.6, x 1000 33.9 / 28.9, 32 x 854 34.0 / 27.1, 90 x 249 16.7 / 13.7.
KeyShares limited_shares(int B, int Hkv, int Lq, int Lk, int D, int nseg, int most, bool may_expand, int cus) {
  const int64_t bh = (int64_t)B * Hkv;
  const bool four = may_expand && wide_four((int64_t)wide_batch(B, Hkv, Lk, D) * Hkv, Lq, Lk, D, cus, true);
  if (may_expand && !four && wide_eligible(B, Hkv, Lq, Lk, D, true, cus)) return {0, 1};
  if (Lq <= 128 || Lk <= 128) return {1, most == 1 ? 1 : choose_shares(bh, Lq, Lk, D, nseg, 1, cus).splits};
  struct Cost { double tile, fixed, again, load; };   // us of a tile, of a workgroup, of one that is not the longest; of the whole load
  static const Cost cost[2][3] = {{{1.32, 5.8, 4.7, 0.9}, {0.87, 6.0, 4.9, 1.03}, {1.15, 5.6, 4.6, 1.03}}, {{2.1, 4.7, 3.8, 1.0}, {1.4, 6.6, 5.4, 1.14}, {1.9, 6.1, 5.0, 1.14}}};
  static const Cost expanded[2] = {{0.9, 10.0, 4.0, 0.92}, {1.4, 14.0, 4.0, 0.95}};
  const double tables = tables_us(nseg, D);
  auto us = [&](const Cost &c, int block, int keys, int n, double tables = 0.0) {
    const double blocks = (Lq + block - 1) / block, part = std::floor(0.8 * blocks), tiles = (double)Lk / keys * (1.25 * part * (part + 1.0) / (2.0 * blocks) + blocks - part) + 0.5 * blocks;
    const double longest = c.fixed + tables + c.tile * (((Lk + keys - 1) / keys + n - 1) / n), load = c.load * (double)bh * (blocks * n * (c.again + tables) + tiles * c.tile) / cus;
    const double two = longest * longest, four = load * load;
    return std::sqrt(std::sqrt(two * two + four * four));
  };
  const int d = D == 128;
  KeyShares best = {1, 1};
  double best_us = us(cost[d][0], BM, BN, 1, tables);
  if (four) {
    const double t = us(expanded[d], 128, BN, 1);
    if (t < best_us) { best_us = t; best = {0, 1}; }
  }
  for (int i = 0; i < 3; ++i)
    for (int n = 1; n <= most && (n == 1 || (Lk + BN - 1) / BN / n >= 2); ++n) {
      double t = us(cost[d][i], BM >> i, i == 2 ? 2 * BN : BN, n, tables) * (i ? 1.05 : 1.0);
      if (n > 1) t += 2.8 + 2.0 * (double)split_workspace_bytes(n, bh * Lq, D) / 4.0e6;
      if (t < best_us) { best_us = t; best = {1 << i, n}; }
    }
  return best;
}
constexpr int kLimitedSplits = 6;   // (more gain nothing)
// What a call does, whose caller asks expand_bytes, which knows of no tables, whether it expands.
KeyShares limited_call(int B, int Hkv, int Lq, int Lk, int D, int nseg, int most, int cus) {
  const KeyShares k = limited_shares(B, Hkv, Lq, Lk, D, 1, most, true, cus);
  return k.waves && nseg > 1 ? limited_shares(B, Hkv, Lq, Lk, D, nseg, most, false, cus) : k;
}
// The largest workspace of the parts that the call is done in.
size_t wide_bytes(int B, int Hkv, int Lq, int Lk, int D, bool share, bool limits) {
  const int n = wide_batch(B, Hkv, Lk, D), last = B - (B - 1) / n * n;
  auto bytes = [&](int b) { return plan_wide((int64_t)b * Hkv, Lq, Lk, D, device_cus(), share, limits).ws_bytes; };
  return std::max(bytes(n), bytes(last));
}
// The launches of the wide path, part after part, or false when the workspace does not hold what they need.
// expand(p, first, ws): the tiles of the batch entries first.. of the call, p.B of them.
template <class Expand>
bool run_wide(const AttnParams &p, int D, int splits, void *workspace, size_t workspace_bytes, hipStream_t st, Expand &&expand) {
  const bool share = splits == 0, limits = p.kv_limit != nullptr;
  if (!workspace || ((uintptr_t)workspace & 15) || workspace_bytes < wide_bytes(p.B, p.Hkv, p.Lq, p.Lk, D, share, limits)) return false;
  char *const ws = reinterpret_cast<char *>(workspace);
  const int n = wide_batch(p.B, p.Hkv, p.Lk, D);
  for (int first = 0; first < p.B; first += n) {
    AttnParams c = p;
    c.B = std::min(n, p.B - first);
    c.bh_total = c.B * p.Hkv;
    c.q += first * p.q_bs * D;
    c.out += first * p.o_bs * D;
    expand(c, first, ws);
    launch_wide(c, D, plan_wide(c.bh_total, p.Lq, p.Lk, D, device_cus(), share, limits), ws, st);
  }
  return true;
}
// The packed K and V of batch entry `first` and on (rows of D channels of `bits` bits; per-key scales of `groups` per row).
void skip_entries(AttnParams &p, int first, int D, int bits, int k_groups, int v_groups) {
  const int64_t rows = first * p.kv_bs, words = rows * (D * bits / 32);
  p.k_words += words; p.v_words += words;
  if (p.k_scale) { p.k_scale += rows * k_groups; p.v_scale += rows * v_groups; }
  if (p.k_zp) p.k_zp += rows * k_groups;
  if (p.v_zp) p.v_zp += rows * v_groups;
}
// What limited_shares says of a call, if it is asked: once with the expansion, and again without where the workspace does not hold it.
class Limited {
  const AttnParams &p;
  int B, D, most;   // most: 0 without limits, or where the caller says how the keys are shared out
  KeyShares k = {0, 1};

 public:
  Limited(const AttnParams &p_, int B_, int D_, int splits) : p(p_), B(B_), D(D_), most(!p_.kv_limit || splits > 1 ? 0 : splits == 1 ? 1 : kLimitedSplits) {
    if (most) k = limited_call(B, p.Hkv, p.Lq, p.Lk, D, p.nseg, most, device_cus());
  }
  bool expands() const { return k.waves == 0; }   // (or is not asked)
  const KeyShares *shares() {
    if (!most) return nullptr;
    if (k.waves == 0) k = limited_shares(B, p.Hkv, p.Lq, p.Lk, D, p.nseg, most, false, device_cus());
    return &k;
  }
};

size_t expand_bytes(int B, int Hkv, int Lq, int Lk, int D, bool limits) {
  if (B <= 0 || Hkv <= 0 || Lq <= 0 || Lk <= 0 || (D != 64 && D != 128)) return 0;
  const int cus = device_cus();   // (a call into the runtime)
  if (!wide_eligible(B, Hkv, Lq, Lk, D, limits, cus) || (limits && limited_shares(B, Hkv, Lq, Lk, D, 1, kLimitedSplits, true, cus).waves)) return 0;
  return wide_bytes(B, Hkv, Lq, Lk, D, true, limits);
}

}  // namespace

namespace {
// Bytes for the shares of a call without key limits, with them, or either and in any operand form.
enum { kPlain = 1, kLimits = 2 };
size_t shares_bytes(int B, int Hkv, int Lq, int Lk, int D, int nseg, int splits, int of) {
  if (B <= 0 || Hkv <= 0 || Lq <= 0 || Lk <= 0 || (D != 64 && D != 128) || splits < 0 || splits > kMaxSplits) return 0;
  nseg = std::min(std::max(nseg, 1), kMaxSegments);
  const int64_t bh = (int64_t)B * Hkv, rows = bh * Lq;
  int n = splits;
  if (!splits) {   // (every call asks: up to 128 queries or keys what wavefronts share, and what the limits say, come to the same as workgroups alone)
    const int cus = device_cus();
    const bool waves = of & kPlain && Lq > 128 && Lk > BN, limits = of & kLimits && Lq > 128 && Lk > 128;
    KeyShares alone = {1, 1};
    if (limits) n = limited_shares(B, Hkv, Lq, Lk, D, nseg, kLimitedSplits, false, cus).splits;
    if (!limits || of & kPlain) n = std::max(n, choose_shares(bh, Lq, Lk, D, nseg, waves ? 4 : 1, cus, &alone).splits);
    if (of == (kPlain | kLimits)) n = std::max(n, alone.splits);   // (the form with exact codes has no shares of wavefronts)
    // (the group sizes are not known here: room for the few-queries kernel's shares whenever the
    // other sizes would admit it)
    if (fewq_eligible(B, Hkv, Lq, Lk, D, D, D)) n = std::max(n, fewq_shares(B * Hkv, Lq, Lk, D, D, D));
  }
  return split_workspace_bytes(n, rows, D);
}
}  // namespace

extern "C" size_t varq_fused_attn_workspace_bytes(int B, int Hkv, int Lq, int Lk, int D, int nseg, int splits) {
  return shares_bytes(B, Hkv, Lq, Lk, D, nseg, splits, kPlain | kLimits);
}
extern "C" size_t varq_fused_attn_workspace_bytes_call(int B, int Hkv, int Lq, int Lk, int D, int nseg, int splits, int limits) {
  return shares_bytes(B, Hkv, Lq, Lk, D, nseg, splits, limits ? kLimits : kPlain);
}

extern "C" int varq_fused_attn_key_waves(int B, int Hkv, int Lq, int Lk, int D, int nseg, int limits) {
  if (B <= 0 || Hkv <= 0 || Lq <= 0 || Lk <= 0 || (D != 64 && D != 128) || nseg < 1) return -1;
  const int cus = device_cus();
  return limits ? limited_call(B, Hkv, Lq, Lk, D, nseg, kLimitedSplits, cus).waves : choose_shares((int64_t)B * Hkv, Lq, Lk, D, nseg, 4, cus).waves;
}

extern "C" size_t varq_fused_attn_expand_bytes(int B, int Hkv, int Lq, int Lk, int D) {
  return expand_bytes(B, Hkv, Lq, Lk, D, false);
}
extern "C" size_t varq_fused_attn_expand_bytes_limits(int B, int Hkv, int Lq, int Lk, int D) { return expand_bytes(B, Hkv, Lq, Lk, D, true); }

extern "C" int varq_fused_attn_key_shares(int B, int Hkv, int Lq, int Lk, int D, int k_group, int v_group) {
  if (B <= 0 || Hkv <= 0 || Lq <= 0 || Lk <= 0 || (D != 64 && D != 128)) return 0;
  if (fewq_eligible(B, Hkv, Lq, Lk, D, k_group, v_group)) return fewq_shares(B * Hkv, Lq, Lk, D, k_group, v_group);
  return choose_shares((int64_t)B * Hkv, Lq, Lk, D, 1, 4, device_cus()).splits;
}

extern "C" int varq_fused_attn(const void *q, void *out,
                               const int32_t *k_words, const float *k_scale, const float *k_zp, int k_bits, int k_group,
                               const int32_t *v_words, const float *v_scale, const float *v_zp, int v_bits, int v_group,
                               int B, int Hq, int Hkv, const int32_t *head_map,
                               int Lq, int Lk, int Lk_stride, int D,
                               const int32_t *kv_limit, float softmax_scale, int layout, int io_dtype, int operand_form,
                               void *workspace, size_t workspace_bytes, int splits, void *stream) {
  VARQ_CHECK_ARG(B > 0 && Hq > 0 && Hkv > 0 && Lq >= 0 && Lk >= 0 && Lk_stride >= Lk, "fused_attn: bad sizes");
  VARQ_CHECK_ARG(io_dtype == VARQ_BF16 || io_dtype == VARQ_F16, "fused_attn: io_dtype must be VARQ_BF16 (1) or VARQ_F16 (2), got %d", io_dtype);
  VARQ_CHECK_ARG(operand_form == VARQ_ATTN_REFERENCE_ROUNDING || operand_form == VARQ_ATTN_EXACT_CODES,
                 "fused_attn: operand_form must be 0 (reference rounding) or 1 (exact codes), got %d", operand_form);
  if (io_dtype == VARQ_F16 && D != 64)
    return varq_set_error(VARQ_ERR_UNSUPPORTED, "fused_attn: fp16 queries need D = 64 (got %d); D = 128 is served in bf16", D);
  // (no queries: nothing to do, and q and out may be the null pointers of empty tensors)
  VARQ_CHECK_ARG(Lq == 0 || (q && out), "fused_attn: null pointer");
  VARQ_CHECK_ARG(Lq == 0 || Lk == 0 || (k_words && v_words && k_scale && v_scale), "fused_attn: null pointer");
  VARQ_CHECK_ARG(head_map || Hkv == Hq, "fused_attn: Hkv != Hq needs a head map");
  VARQ_CHECK_ARG(D == 64 || D == 128, "fused_attn: D must be 64 or 128 (got %d)", D);
  VARQ_CHECK_ARG(k_bits == 2 || k_bits == 4 || k_bits == 8, "fused_attn: bits must be 2, 4 or 8 (got %d)", k_bits);
  if (k_bits != v_bits)
    return varq_set_error(VARQ_ERR_UNSUPPORTED, "fused_attn: K and V bit-widths must match (%d vs %d)", k_bits, v_bits);
  VARQ_CHECK_ARG(k_group > 0 && v_group > 0 && D % k_group == 0 && D % v_group == 0, "fused_attn: groups must divide D");
  if (Lq == 0 || Lk == 0) {
    if (Lq > 0) return varq_set_error(VARQ_ERR_INVALID, "fused_attn: no keys to attend");
    return VARQ_OK;
  }
  VARQ_CHECK_ARG((int64_t)B * Hkv * Lk_stride * D < (1ll << 40), "fused_attn: cache too large");
  VARQ_CHECK_ARG(((uintptr_t)q & 15) == 0 && ((uintptr_t)out & 7) == 0, "fused_attn: q must be 16-byte and out 8-byte aligned");

  AttnParams p;
  p.q = reinterpret_cast<const __bf16 *>(q);
  p.out = reinterpret_cast<__bf16 *>(out);
  p.k_words = reinterpret_cast<const u32 *>(k_words);
  p.v_words = reinterpret_cast<const u32 *>(v_words);
  p.k_scale = k_scale; p.k_zp = k_zp; p.v_scale = v_scale; p.v_zp = v_zp;
  p.k_chan_scale = nullptr; p.k_chan_zp = nullptr; p.v_chan_scale = nullptr; p.v_chan_zp = nullptr;
  p.nseg = 1;
  for (int s = 0; s < kMaxSegments; ++s) p.seg_end[s] = Lk;
  p.head_map = head_map; p.kv_limit = kv_limit;
  p.B = B; p.Hq = Hq; p.Hkv = Hkv; p.Lq = Lq; p.Lk = Lk; p.Lstride = Lk_stride;
  p.q_tiles = (Lq + BM - 1) / BM;
  p.bh_total = B * Hkv;
  p.fq_share_blocks = 0;
  p.scale_log2e = softmax_scale * kLog2e;
  p.f16 = io_dtype == VARQ_F16;
  p.exact_codes = operand_form == VARQ_ATTN_EXACT_CODES && !p.f16;
  if (int e = set_layout(p, layout, "fused_attn")) return e;
  hipStream_t st = (hipStream_t)stream;
  // few queries, left to the library: the kernel whose wavefronts share the keys (it has no exact form)
  const bool exact_form = p.exact_codes && D == 128 && k_group == D && v_group == D && k_bits != 8;
  if (splits == 0 && !exact_form && groups_served(D, k_group, v_group) && fewq_eligible(B, Hkv, Lq, Lk, D, k_group, v_group)) {
    set_few(p, D, k_group, v_group, workspace, workspace_bytes);
    launch_few(p, D, k_bits, k_group, v_group, st);
    combine_few(p, D, st);
    VARQ_CHECK_LAUNCH("fused_attn");
    return VARQ_OK;
  }
  Limited limited(p, B, D, exact_form ? 2 : splits);
  if ((splits == 0 || splits == 1) && limited.expands() && !p.exact_codes && groups_served(D, k_group, v_group) && wide_eligible(B, p.Hkv, Lq, Lk, D, kv_limit != nullptr) &&
      run_wide(p, D, splits, workspace, workspace_bytes, st, [&](AttnParams c, int first, char *ws) {
        skip_entries(c, first, D, k_bits, D / k_group, D / v_group);
        launch_expand(c, D, k_bits, k_group, v_group, false, ws, st);
      })) {
    VARQ_CHECK_LAUNCH("fused_attn");
    return VARQ_OK;
  }
  if (int e = set_splits(p, D, exact_form ? 1 : 4, limited.shares(), splits, workspace, workspace_bytes, "fused_attn")) return e;
  if (!groups_served(D, k_group, v_group))
    return varq_set_error(VARQ_ERR_UNSUPPORTED, "fused_attn: no kernel for D=%d bits=%d k_group=%d v_group=%d", D, k_bits,
                          k_group, v_group);
  p.k_shift = varq_log2_exact(k_group);
  p.v_shift = varq_log2_exact(v_group);
  if (exact_form) {
    if (k_bits == 4) launch_exact<4>(p, st);
    else launch_exact<2>(p, st);
  } else {
    launch_any<false>(p, D, k_bits, st);
  }
  VARQ_CHECK_LAUNCH("fused_attn");
  return VARQ_OK;
}

extern "C" int varq_fused_attn_channel(const void *q, void *out,
                                       const int32_t *k_words, const float *k_chan_scale, const float *k_chan_zp,
                                       const int32_t *v_words, const float *v_chan_scale, const float *v_chan_zp,
                                       int nseg, const int32_t *host_seg_end,
                                       int bits, int B, int Hq, int Hkv, const int32_t *head_map,
                                       int Lq, int Lk, int Lk_stride, int D,
                                       const int32_t *kv_limit, float softmax_scale, int layout, int io_dtype,
                                       void *workspace, size_t workspace_bytes, int splits, void *stream) {
  VARQ_CHECK_ARG(io_dtype == VARQ_BF16 || io_dtype == VARQ_F16, "fused_attn_channel: io_dtype must be VARQ_BF16 (1) or VARQ_F16 (2), got %d", io_dtype);
  if (io_dtype == VARQ_F16 && D != 64)
    return varq_set_error(VARQ_ERR_UNSUPPORTED, "fused_attn_channel: fp16 queries need D = 64 (got %d); D = 128 is served in bf16", D);
  // (no queries: nothing to do, and q and out may be the null pointers of empty tensors)
  VARQ_CHECK_ARG(Lq == 0 || (q && out), "fused_attn_channel: null pointer");
  VARQ_CHECK_ARG(Lq == 0 || Lk == 0 || (k_words && v_words && k_chan_scale && v_chan_scale), "fused_attn_channel: null pointer");
  VARQ_CHECK_ARG(nseg >= 1 && nseg <= kMaxSegments, "fused_attn_channel: nseg must be 1..%d (got %d)", kMaxSegments, nseg);
  VARQ_CHECK_ARG(nseg == 1 || host_seg_end, "fused_attn_channel: segment ends missing");
  VARQ_CHECK_ARG(B > 0 && Hq > 0 && Hkv > 0 && Lq >= 0 && Lk >= 0 && Lk_stride >= Lk, "fused_attn_channel: bad sizes");
  VARQ_CHECK_ARG(head_map || Hkv == Hq, "fused_attn_channel: Hkv != Hq needs a head map");
  VARQ_CHECK_ARG(D == 64 || D == 128, "fused_attn_channel: D must be 64 or 128 (got %d)", D);
  VARQ_CHECK_ARG(bits == 2 || bits == 4 || bits == 8, "fused_attn_channel: bits must be 2, 4 or 8 (got %d)", bits);
  if (Lq == 0 || Lk == 0) {
    if (Lq > 0) return varq_set_error(VARQ_ERR_INVALID, "fused_attn_channel: no keys to attend");
    return VARQ_OK;
  }
  VARQ_CHECK_ARG((int64_t)B * Hkv * Lk_stride * D < (1ll << 40), "fused_attn_channel: cache too large");
  VARQ_CHECK_ARG(((uintptr_t)q & 15) == 0 && ((uintptr_t)out & 7) == 0,
                 "fused_attn_channel: q must be 16-byte and out 8-byte aligned");
  VARQ_CHECK_ARG(((uintptr_t)k_chan_scale & 15) == 0 && ((uintptr_t)k_chan_zp & 15) == 0 &&
                     ((uintptr_t)v_chan_scale & 15) == 0 && ((uintptr_t)v_chan_zp & 15) == 0,
                 "fused_attn_channel: the tables must be 16-byte aligned");

  AttnParams p;
  p.q = reinterpret_cast<const __bf16 *>(q);
  p.out = reinterpret_cast<__bf16 *>(out);
  p.k_words = reinterpret_cast<const u32 *>(k_words);
  p.v_words = reinterpret_cast<const u32 *>(v_words);
  p.k_scale = nullptr; p.k_zp = nullptr; p.v_scale = nullptr; p.v_zp = nullptr;
  p.k_chan_scale = k_chan_scale; p.k_chan_zp = k_chan_zp; p.v_chan_scale = v_chan_scale; p.v_chan_zp = v_chan_zp;
  p.nseg = nseg;
  for (int s = 0, prev = 0; s < nseg; ++s) {
    // the last segment runs to the end of the keys whatever the caller's table says
    const int e = (s == nseg - 1 || !host_seg_end) ? Lk : host_seg_end[s];
    VARQ_CHECK_ARG(e > prev || (s == nseg - 1 && e >= prev), "fused_attn_channel: segment ends must increase");
    VARQ_CHECK_ARG(e <= Lk, "fused_attn_channel: segment end %d beyond Lk=%d", e, Lk);
    p.seg_end[s] = e;
    prev = e;
  }
  for (int s = nseg; s < kMaxSegments; ++s) p.seg_end[s] = Lk;
  p.head_map = head_map; p.kv_limit = kv_limit;
  p.B = B; p.Hq = Hq; p.Hkv = Hkv; p.Lq = Lq; p.Lk = Lk; p.Lstride = Lk_stride;
  p.q_tiles = (Lq + BM - 1) / BM;
  p.bh_total = B * Hkv;
  p.fq_share_blocks = 0;
  p.scale_log2e = softmax_scale * kLog2e;
  p.f16 = io_dtype == VARQ_F16;
  p.exact_codes = 0;
  if (int e = set_layout(p, layout, "fused_attn_channel")) return e;
  hipStream_t st = (hipStream_t)stream;
  Limited limited(p, B, D, splits);
  if ((splits == 0 || splits == 1) && limited.expands() && wide_eligible(B, p.Hkv, Lq, Lk, D, kv_limit != nullptr) &&
      run_wide(p, D, splits, workspace, workspace_bytes, st, [&](AttnParams c, int first, char *ws) {
        skip_entries(c, first, D, bits, 0, 0);
        launch_expand(c, D, bits, D, D, true, ws, st);
      })) {
    VARQ_CHECK_LAUNCH("fused_attn_channel");
    return VARQ_OK;
  }
  if (int e = set_splits(p, D, 4, limited.shares(), splits, workspace, workspace_bytes, "fused_attn_channel"))
    return e;
  launch_any<true>(p, D, bits, st);
  VARQ_CHECK_LAUNCH("fused_attn_channel");
  return VARQ_OK;
}

// One call for all bit-width classes of a cache: see ClassTable.
extern "C" int varq_fused_attn_classes(const void *q, void *out, const varq_kv_class *host_classes, int n_classes, int group,
                                       int B, int H, int Lq, int Lk, int Lk_stride, int D,
                                       const int32_t *kv_limit, float softmax_scale, int layout, int io_dtype,
                                       void *workspace, size_t workspace_bytes, int splits, void *stream) {
  VARQ_CHECK_ARG(B > 0 && H > 0 && Lq >= 0 && Lk >= 0 && Lk_stride >= Lk, "fused_attn_classes: bad sizes");
  VARQ_CHECK_ARG(io_dtype == VARQ_BF16 || io_dtype == VARQ_F16, "fused_attn_classes: io_dtype must be VARQ_BF16 (1) or VARQ_F16 (2), got %d", io_dtype);
  VARQ_CHECK_ARG(D == 64 || D == 128, "fused_attn_classes: D must be 64 or 128 (got %d)", D);
  if (io_dtype == VARQ_F16 && D != 64)
    return varq_set_error(VARQ_ERR_UNSUPPORTED, "fused_attn_classes: fp16 queries need D = 64 (got %d); D = 128 is served in bf16", D);
  VARQ_CHECK_ARG(layout == VARQ_LAYOUT_BHLC || layout == VARQ_LAYOUT_BHLC_OUT_BLHC, "fused_attn_classes: a heads-first cache is needed (layout %d)", layout);
  VARQ_CHECK_ARG(host_classes && n_classes >= 1 && n_classes <= 3, "fused_attn_classes: 1..3 classes (got %d)", n_classes);
  VARQ_CHECK_ARG(group == 32 || group == 64 || (group == 128 && D == 128), "fused_attn_classes: no kernel for D=%d group=%d", D, group);
  VARQ_CHECK_ARG(Lq == 0 || (q && out), "fused_attn_classes: null pointer");
  VARQ_CHECK_ARG((int64_t)B * H * Lk_stride * D < (1ll << 40) && (int64_t)B * H < (1 << 24), "fused_attn_classes: cache too large");
  VARQ_CHECK_ARG(((uintptr_t)q & 15) == 0 && ((uintptr_t)out & 7) == 0, "fused_attn_classes: q must be 16-byte and out 8-byte aligned");
  if (Lq == 0) return VARQ_OK;
  VARQ_CHECK_ARG(Lk > 0, "fused_attn_classes: no keys to attend");
  ClassTable t = {};
  int heads = 0;
  for (int i = 0; i < n_classes; ++i) {
    const varq_kv_class &c = host_classes[i];
    VARQ_CHECK_ARG(c.bits == 2 || c.bits == 4 || c.bits == 8, "fused_attn_classes: bits must be 2, 4 or 8 (got %d)", c.bits);
    VARQ_CHECK_ARG(c.heads > 0 && c.head_map && c.k_words && c.v_words && c.k_scale && c.v_scale, "fused_attn_classes: incomplete class %d", i);
    ClassParams &d = t.c[c.bits == 8 ? 0 : c.bits == 4 ? 1 : 2];
    VARQ_CHECK_ARG(!d.heads, "fused_attn_classes: two classes of %d bits", c.bits);
    d = {reinterpret_cast<const u32 *>(c.k_words), reinterpret_cast<const u32 *>(c.v_words), c.k_scale, c.k_zp, c.v_scale, c.v_zp, c.head_map, c.heads, 0};
    heads += c.heads;
  }
  VARQ_CHECK_ARG(heads == H, "fused_attn_classes: the classes have %d heads, not %d", heads, H);
  t.c[1].first = B * t.c[0].heads;
  t.c[2].first = t.c[1].first + B * t.c[1].heads;

  AttnParams p = {};
  p.q = reinterpret_cast<const __bf16 *>(q);
  p.out = reinterpret_cast<__bf16 *>(out);
  p.nseg = 1;
  for (int s = 0; s < kMaxSegments; ++s) p.seg_end[s] = Lk;
  p.kv_limit = kv_limit;
  p.B = B; p.Hq = H; p.Hkv = H; p.Lq = Lq; p.Lk = Lk; p.Lstride = Lk_stride;
  p.q_tiles = (Lq + BM - 1) / BM;
  p.bh_total = B * H;
  p.scale_log2e = softmax_scale * kLog2e;
  p.f16 = io_dtype == VARQ_F16;
  if (int e = set_layout(p, layout, "fused_attn_classes")) return e;
  hipStream_t st = (hipStream_t)stream;
  Limited limited(p, B, D, splits);
  if (splits == 0 && fewq_eligible(B, H, Lq, Lk, D, group, group)) {
    set_few(p, D, group, group, workspace, workspace_bytes);
    launch_few_classes(p, D, t, group, st);
    combine_few(p, D, st);
  } else if ((splits == 0 || splits == 1) && limited.expands() && wide_eligible(B, p.Hkv, Lq, Lk, D, kv_limit != nullptr) &&
             run_wide(p, D, splits, workspace, workspace_bytes, st, [&](const AttnParams &part, int first, char *ws) {
               ClassTable of = t;   // the part's batch entries of every class
               int pairs = 0;
               for (int i = 0; i < 3; ++i) {
                 ClassParams &d = of.c[i];
                 d.first = pairs;
                 if (!d.heads) continue;
                 const int64_t rows = (int64_t)first * d.heads * Lk_stride, words = rows * (D * (8 >> i) / 32), groups = rows * (D / group);
                 d.k_words += words; d.v_words += words;
                 d.k_scale += groups; d.v_scale += groups;
                 if (d.k_zp) d.k_zp += groups;
                 if (d.v_zp) d.v_zp += groups;
                 pairs += part.B * d.heads;
               }
               launch_expand_classes(part, D, of, group, ws, st);
             })) {
  } else {
    if (int e = set_splits(p, D, 4, limited.shares(), splits, workspace, workspace_bytes, "fused_attn_classes")) return e;
    p.k_shift = p.v_shift = varq_log2_exact(group);
    if (D == 128) launch_classes<128>(p, t, st);
    else launch_classes<64>(p, t, st);
  }
  VARQ_CHECK_LAUNCH("fused_attn_classes");
  return VARQ_OK;
}
