// Attention of many queries over a packed cache in two launches: the packed K and V of every
// (batch, head) are dequantized ONCE into the operands of the matrix instructions, and a plain flash
// attention then streams those.
//
// fused_attn.hip widens a key tile in every workgroup, i.e. once per 256 queries; behind that it
// computes with the very same operands, (code - zp) * scale in fp32 rounded to the attention's
// 16-bit type.  With several blocks of 256 queries per (batch, head) the widening is the same
// work over and over, it takes a fifth to a quarter of that kernel's time, and its registers and
// instructions keep the rest from overlapping.
#include <type_traits>

#include "attn_common.h"

using namespace varq_attn;

namespace {

// A tile holds 64 keys of one (batch, head): first K, then V, 64 * D * 2 bytes each, as 1 KiB
// fragments that are operands of v_mfma_f32_16x16x32 for a wavefront, 16 bytes per lane (r = lane % 16,
// g = lane / 16):
//   K fragment [kb][ch][t] (half t of the 32 keys kb, 32 channels ch): lane holds key kb*32 + 8*(r/4) + 4*t + r%4,
//                          channels ch*32 + g*8 + 0..7
//   V fragment [kb][d]     (16 channels d, the 32 keys kb): lane holds channel d*16 + r, keys kb*32 + g*8 + 0..7
// so that the attention kernel copies tiles to LDS as they are and reads every operand with one
// conflict-free ds_read_b128.  The order of the keys in the two K fragments of a block is the one
// that leaves the logits of 8 consecutive keys in a lane of S^T = K Q^T, which is what the lane
// holds of P^T in O^T = V^T P^T.  Keys past Lk hold zeros.
template <int D> constexpr int kHalfTile = BN * D * 2;

struct ExpandParams {
  AttnParams a;
  char *tiles;
  int n_tiles, kg_shift, vg_shift;   // log2 of the channels per scale group
};

// the eight codes of octet `oct` of a packed row, as they lie, and as numbers
template <int BITS> __device__ __forceinline__ uint2 load_codes(const u32 *row, int oct) {
  if constexpr (BITS == 8) return *reinterpret_cast<const uint2 *>(row + 2 * oct);
  else if constexpr (BITS == 4) return make_uint2(row[oct], 0u);
  else return make_uint2(row[oct >> 1] >> ((oct & 1) * 16), 0u);
}
template <int BITS> __device__ __forceinline__ void code_values(uint2 w, float (&f)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j)
    f[j] = (float)(int)__builtin_amdgcn_sbfe((int)(BITS == 8 && j >= 4 ? w.y : w.x), BITS * (BITS == 8 ? j & 3 : j), BITS);
}

// One workgroup = one tile of one (batch, head).  HBM-bound by its writes: all codes and per-key parameters of the
// tile are requested before the first is used, and the segment that a tile's keys belong to is looked up once (key by
// key, and with each octet's loads behind a check of its key, [2,16,10521,128] took 51 us at 4 bits in groups and 76 at
// 8 bits with 13 per-channel tables; now 43 and 49, 5.0 and 5.3 TB/s).
constexpr int kTransposed = BN + 8;   // keys of a row of the transposed tile
// (vt: [D][kTransposed], seg_end: [kMaxSegments] in LDS; place: the pair of the tile buffer)
template <int D, int BITS, bool CHAN, bool F16>
__device__ __forceinline__ void expand_tile(const ExpandParams &e, const AttnParams &p, int tile, int bh, int place, uint16_t *vt, int *seg_end) {
  constexpr int WPR = D * BITS / 32, NF = D / 16, OCT = D / 8;   // NF: fragments per 32 keys
  constexpr int VTS = kTransposed;
  const int tid = threadIdx.x;
  const int b = bh / p.Hkv, hs = bh - b * p.Hkv;
  const int64_t kv_row0 = b * p.kv_bs + hs * p.kv_hs;
  char *const out = e.tiles + ((int64_t)place * e.n_tiles + tile) * (2 * kHalfTile<D>);
  constexpr int VI = BN / 2 * OCT / 256, KI = BN * OCT / 256;   // items of a thread: two keys' octets of V, one of K
  const int key0 = tile * BN;
  auto k_key = [&](int i) {
    const int item = tid + i * 256, r = item & 15, frag = item >> 6;
    return key0 + frag / NF * 32 + 8 * (r >> 2) + 4 * (frag & 1) + (r & 3);
  };
  auto k_oct = [&](int i) { const int item = tid + i * 256; return (item >> 6) % NF / 2 * 4 + ((item >> 4) & 3); };
  auto v_key = [&](int i) { return key0 + (tid + i * 256) / OCT * 2; };
  const int v_oct = tid % OCT;
  // everything the tile needs is requested before the first use (rows past the end: the last row's)
  uint2 kc[KI], vc[VI][2];
  float ks[CHAN ? 1 : KI], kz[CHAN ? 1 : KI], vs[CHAN ? 1 : VI][2], vz[CHAN ? 1 : VI][2];
  auto request = [&](const u32 *words, const float *scale, const float *zp, int g_shift, int key, int oct, uint2 &code, float &s, float &z) {
    const int64_t row = kv_row0 + min(key, p.Lk - 1) * p.kv_ts;
    code = load_codes<BITS>(words + row * WPR, oct);
    if constexpr (!CHAN) {
      const int64_t g = row * (D >> g_shift) + (oct * 8 >> g_shift);
      s = scale[g];
      z = zp ? zp[g] : 0.f;
    }
  };
#pragma unroll
  for (int i = 0; i < VI; ++i)
#pragma unroll
    for (int n = 0; n < 2; ++n) request(p.v_words, p.v_scale, p.v_zp, e.vg_shift, v_key(i) + n, v_oct, vc[i][n], vs[CHAN ? 0 : i][n], vz[CHAN ? 0 : i][n]);
#pragma unroll
  for (int i = 0; i < KI; ++i) request(p.k_words, p.k_scale, p.k_zp, e.kg_shift, k_key(i), k_oct(i), kc[i], ks[CHAN ? 0 : i], kz[CHAN ? 0 : i]);
  // the segment of the tile's first key: of the ends that are not the last, how many are not behind it
  int seg0 = 0;
  bool one_seg = true;
  if constexpr (CHAN) {
    if (tid < kMaxSegments) seg_end[tid] = p.seg_end[tid];
    __syncthreads();
    const int lane = tid & 63;
    seg0 = __popcll(__ballot(lane + 1 < p.nseg && key0 >= seg_end[lane & (kMaxSegments - 1)]));
    one_seg = seg0 + 1 >= p.nseg || key0 + BN <= seg_end[seg0];
  }
  const bool ragged = key0 + BN > p.Lk;
  auto values = [&](uint2 code, float s1, float z1, const float *cscale, const float *czp, int key, int oct, float (&f)[8]) {
    code_values<BITS>(code, f);
    if constexpr (CHAN) {
      int seg = seg0;
      if (!one_seg) while (seg + 1 < p.nseg && key >= seg_end[seg]) ++seg;
      const int64_t t = ((int64_t)seg * p.Hkv + hs) * D + oct * 8;
      const float4 sa = *reinterpret_cast<const float4 *>(cscale + t), sb = *reinterpret_cast<const float4 *>(cscale + t + 4);
      const float s[8] = {sa.x, sa.y, sa.z, sa.w, sb.x, sb.y, sb.z, sb.w};
      if (czp) {
        const float4 za = *reinterpret_cast<const float4 *>(czp + t), zb = *reinterpret_cast<const float4 *>(czp + t + 4);
        const float z[8] = {za.x, za.y, za.z, za.w, zb.x, zb.y, zb.z, zb.w};
#pragma unroll
        for (int j = 0; j < 8; ++j) f[j] = (f[j] - z[j]) * s[j];
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) f[j] = f[j] * s[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = (f[j] - z1) * s1;
    }
    if (ragged && key >= p.Lk) {
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = 0.f;
    }
  };
  // V: two adjacent keys x 8 channels -> the transposed tile in LDS
#pragma unroll
  for (int i = 0; i < VI; ++i) {
    float f0[8], f1[8];
    const int c = CHAN ? 0 : i;
    values(vc[i][0], vs[c][0], vz[c][0], p.v_chan_scale, p.v_chan_zp, v_key(i), v_oct, f0);
    values(vc[i][1], vs[c][1], vz[c][1], p.v_chan_scale, p.v_chan_zp, v_key(i) + 1, v_oct, f1);
#pragma unroll
    for (int j = 0; j < 8; ++j) *reinterpret_cast<u32 *>(&vt[(v_oct * 8 + j) * VTS + (tid + i * 256) / OCT * 2]) = pack_io_rne<F16>(f0[j], f1[j]);
  }
  // K: one octet of one key is one lane's 16 bytes
#pragma unroll
  for (int i = 0; i < KI; ++i) {
    float f[8];
    values(kc[i], ks[CHAN ? 0 : i], kz[CHAN ? 0 : i], p.k_chan_scale, p.k_chan_zp, k_key(i), k_oct(i), f);
    u32x4_t w;
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = pack_io_rne<F16>(f[2 * j], f[2 * j + 1]);
    *reinterpret_cast<u32x4_t *>(out + (tid + i * 256) * 16) = w;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < KI; ++i) {
    const int item = tid + i * 256, r = item & 15, g = (item >> 4) & 3, frag = item >> 6;
    *reinterpret_cast<u32x4_t *>(out + kHalfTile<D> + item * 16) =
        *reinterpret_cast<const u32x4_t *>(&vt[((frag % NF) * 16 + r) * VTS + (frag / NF) * 32 + g * 8]);
  }
}

template <int D, int BITS, bool CHAN, bool F16>
__global__ __launch_bounds__(256) void expand_tiles_kernel(ExpandParams e) {
  __shared__ uint16_t vt[D * kTransposed];
  __shared__ int seg_end[kMaxSegments];
  expand_tile<D, BITS, CHAN, F16>(e, e.a, blockIdx.x, blockIdx.y, blockIdx.y, vt, seg_end);
}
// All bit-widths of a cache in one launch, each head's tiles to its place among the heads: [8,16,n,128] with 8, 3 and 5 heads
// of 8, 4 and 2 bits, us, a launch per width -> one: n = 4121 88 -> 77, 6425 123 -> 111, 10521 192 -> 179 (5.3 TB/s).
template <int D, bool F16>
__global__ __launch_bounds__(256) void expand_classes_kernel(ExpandParams e, ClassTable t) {
  __shared__ uint16_t vt[D * kTransposed];
  AttnParams p = e.a;
  in_class(p, t, blockIdx.y, [&](auto bits, int bh, int place) __attribute__((always_inline)) {
    expand_tile<D, decltype(bits)::value, false, F16>(e, p, blockIdx.x, bh, place, vt, nullptr);
  });
}

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;
// D (16x16 fp32) += A (16x32) B (32x16), operands in the attention's 16-bit type
template <bool F16> __device__ __forceinline__ floatx4_t mfma_16x16x32(u32x4_t a, u32x4_t b, floatx4_t c) {
  if constexpr (F16) {
    typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
}

// A wavefront copies N KiB from global memory (`src`: the lane's 16 bytes of the first) to LDS, from address `dst` on,
// past the registers.  The compiler does not count these loads: wait_copies<N> waits until at most the N KiB last asked
// for are under way.
// (m0 is written here and named for it: the compiler sets it for instructions of its own and may take a value to be still there.  It
// warns of every reserved register that is named.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <int N> __device__ __forceinline__ void to_lds(const char *src, u32 dst) {
  static_assert(N == 1 || N == 2 || N == 4, "N");
  dst = __builtin_amdgcn_readfirstlane(dst);
  if constexpr (N == 1)
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(dst) : "m0", "memory");
  else if constexpr (N == 2)
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off\n\tglobal_load_lds_dwordx4 %0, off offset:1024" ::"v"(src), "s"(dst) : "m0", "memory");
  else
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off\n\tglobal_load_lds_dwordx4 %0, off offset:1024\n\t"
                 "global_load_lds_dwordx4 %0, off offset:2048\n\tglobal_load_lds_dwordx4 %0, off offset:3072" ::"v"(src), "s"(dst) : "m0", "memory");
}
#pragma clang diagnostic pop
template <int N> __device__ __forceinline__ void wait_copies() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// Work comes in blocks of 256 queries (128: see wide_four) of one (batch, head), block bh * q_tiles + qt, and is dealt out to
// n workgroups in rounds: in each of the first `rounds` rounds workgroup w takes block round * n + w
// whole; the blocks left over are shared out by the key tile, workgroup w taking units [T w / n, T (w + 1) / n)
// of their T = blocks * tiles units, and a block that falls on several workgroups is put together
// from their partial results.  With n = the number of compute units all of them finish together.
// Whole rounds first, because the workgroups of an XCD then read the same few tile streams at a time
// through their L2.  (Consecutive w sit on one XCD: ids congruent mod 8 share an L2.)
struct WideParams {
  AttnParams a;
  const char *tiles;
  int all_tiles, rounds;
  float *ws_o, *ws_ml;   // partial results: slot 2w the first shared block of workgroup w, slot 2w + 1 its last; [slot][256][D], [slot][256][2]
};
struct SharedUnits {
  int64_t first, total;   // the first unit that is shared out, and how many are
  int n;
  __device__ __forceinline__ SharedUnits(const WideParams &e, int n_wgs) : n(n_wgs) {
    first = (int64_t)e.rounds * n_wgs * e.all_tiles;
    total = max((int64_t)e.a.bh_total * e.a.q_tiles * e.all_tiles - first, (int64_t)0);   // (a padded grid covers more than there is)
  }
  __device__ __forceinline__ int64_t begin(int w) const { return first + total * w / n; }
  __device__ __forceinline__ int owner(int64_t unit) const { return (int)(((unit - first + 1) * n - 1) / total); }   // the last w with begin(w) <= unit
};

// Workgroups of an XCD in a window of HeavyFirst: four rounds over its 32 compute units.  One, two and four rounds, us
// under the block-causal rule: D=128, 24 pairs of 4121 tokens 201 / 169 / 170, 128 of 2952 465 / 491 / 453, 64 of 10521
// 2147 / 2123 / 2202; D=64, 32 of 4121 172 / 171 / 145, 128 of 5021 725 / 721 / 669.
constexpr int kLimitWindow = 128;

// One workgroup = NW wavefronts = 32 NW queries of one (batch, head) at a time (8; 4: see wide_four); a wavefront owns
// 32 queries (two columns of 16) and walks blocks of 32 keys, transposed: S^T = K Q^T, O^T = V^T P^T.
// The tiles go to LDS past the registers: with loads and LDS stores of the wavefront's own, a block of 128 queries took 12 % longer
// (1024 x 2521, 32 pairs, D=128: 66 -> 57 us; 680 x 680, 128 pairs, D=64: 44 -> 32), and
// blocks of 256, where two wavefronts of a SIMD cover for one another, 2-3 % (4096 x 10521, 32 pairs, with its quantizer
// and the expansion 623 -> 607; 13 scales of 128 pairs 4600 -> 4497).  Also measured and the same: operands requested eight fragments
// ahead, scheduling fences after every fragment, 32x32x16 instructions (2-6 % slower).
template <int D, bool F16, int NW>
__global__ __launch_bounds__(NW * 64, NW / 4) void wide_attn_kernel(WideParams e) {
  constexpr int NT = NW * 64, NF = D / 16, HT = kHalfTile<D>, PIECES = HT / (NT * 16);
  constexpr int BQ = NW * 32;   // queries of a block
  extern __shared__ __attribute__((aligned(16))) char lds[];   // K slots [4][HT], V slots [4][HT]
  const AttnParams &p = e.a;
  const int all_tiles = e.all_tiles, n_wgs = gridDim.x;
  const int w = (blockIdx.x & 7) * (n_wgs >> 3) + min(blockIdx.x & 7, n_wgs & 7) + (blockIdx.x >> 3);
  const SharedUnits shared(e, n_wgs);
  int64_t unit = shared.begin(w);
  const int64_t unit_end = shared.begin(w + 1);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, quarter = lane >> 4;
  const float scale = p.scale_log2e;
  const char *const frag0 = lds + lane * 16;

  for (int round = 0; round < e.rounds || unit < unit_end; ++round) {
  int qblock = round * n_wgs + w, tbase = 0, tlast = all_tiles;
  if (round >= e.rounds) {
    qblock = (int)(unit / all_tiles);
    tbase = (int)(unit - (int64_t)qblock * all_tiles);
    tlast = (int)min((int64_t)all_tiles, tbase + (unit_end - unit));
    unit += tlast - tbase;
  }
  const bool partial = tlast - tbase < all_tiles;
  if (round > 0) __syncthreads();   // (the block before is done with the LDS)

  int bh = qblock / p.q_tiles, qt = qblock - bh * p.q_tiles;
  if (p.kv_limit) {   // (whole blocks, one round: see plan_wide)
    const HeavyFirst k(blockIdx.x >> 3, p.q_tiles, (p.bh_total + 7) >> 3, max(kLimitWindow / p.q_tiles, 1));
    bh = k.grp * 8 + (blockIdx.x & 7);
    qt = k.qt;
    if (bh >= p.bh_total) return;
  }
  const int b = bh / p.Hkv, hs = bh - b * p.Hkv;
  const int hq = p.head_map ? p.head_map[hs] : hs;
  const int qrow0 = qt * BQ + wave * 32;
  const bool wave_live = qrow0 < p.Lq;   // wave-uniform
  int limit[2], qrow_c[2];
  int minlim = p.Lk;
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const int row = qrow0 + n * 16 + r16;
    qrow_c[n] = min(row, p.Lq - 1);
    limit[n] = p.kv_limit ? max(min(p.kv_limit[qrow_c[n]], p.Lk), 0) : p.Lk;
    if (row < p.Lq) minlim = min(minlim, limit[n]);
  }
  const int kv_end = p.kv_limit ? block_limit<BQ>(p.kv_limit, qt * BQ, p.Lq, p.Lk) : p.Lk;
  const int n_tiles = __builtin_amdgcn_readfirstlane(max(min((kv_end + BN - 1) / BN, tlast) - tbase, 0));
  // tiles that no query of the wavefront has to mask
  const int n_full = __builtin_amdgcn_readfirstlane(min(max(wave_fold<false, 1>(minlim) / BN - tbase, 0), n_tiles));

  const char *const src = e.tiles + ((int64_t)bh * all_tiles + tbase) * (2 * HT);
  // Tile t of K and of V sits in slot t % 4.  The copies to LDS go past the registers, each wavefront its own stretch of a
  // tile; their addresses are a scalar and what the lane adds to it.
  const int my_part = __builtin_amdgcn_readfirstlane(wave * (PIECES * 1024));
  const u32 my_lds = (u32)(uintptr_t)(__attribute__((address_space(3))) char *)lds + my_part;
  const char *const my_src = src + my_part + lane * 16;
  auto copy_k = [&](int t) __attribute__((always_inline)) {   // (past the end: the last tile again, never used)
    to_lds<PIECES>(my_src + (int64_t)min(t, n_tiles - 1) * (2 * HT), (t & 3) * HT + my_lds);
  };
  auto copy_v = [&](int t) __attribute__((always_inline)) {
    to_lds<PIECES>(my_src + (int64_t)min(t, n_tiles - 1) * (2 * HT) + HT, (4 + (t & 3)) * HT + my_lds);
  };

  // ---- prologue: K of tiles 0 and 1 and V of tile 0 in LDS, K of tile 2 and V of tile 1 on their way;
  //      the V slot of "tile -1" holds zeros ----
  u32x4_t qb[2][NF / 2];
  if (n_tiles > 0) {
    copy_k(0); copy_v(0); copy_k(1);
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const __bf16 *qptr = p.q + (b * p.q_bs + hq * p.q_hs + qrow_c[n] * p.q_ts) * D + quarter * 8;
#pragma unroll
      for (int ch = 0; ch < NF / 2; ++ch) qb[n][ch] = *reinterpret_cast<const u32x4_t *>(qptr + ch * 32);
    }
#pragma unroll
    for (int i = 0; i < PIECES; ++i) *reinterpret_cast<u32x4_t *>(lds + 7 * HT + i * (NT * 16) + tid * 16) = u32x4_t{0, 0, 0, 0};
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
    copy_k(2); copy_v(1);
  }
  __syncthreads();

  if (!wave_live) {
    for (int t = 0; t < n_tiles; ++t) {
      copy_k(t + 3); copy_v(t + 2);
      wait_copies<2 * PIECES>();
      __syncthreads();
    }
    wait_copies<0>();
    continue;
  }

  floatx4_t oacc[NF][2];                // [16 channels][16 queries]
  floatx4_t sacc[2][2][2];              // [block parity][half of the keys][16 queries]
  u32x4_t pop[2][2];                    // [block parity][16 queries]: weights of 8 keys
  float l_part[2], m_ref[2];
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    l_part[n] = 0.f; m_ref[n] = 0.f;
    pop[0][n] = pop[1][n] = u32x4_t{0, 0, 0, 0};
#pragma unroll
    for (int d = 0; d < NF; ++d) oacc[d][n] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  }

  // logit of key 8*quarter + i of the block, query column n
  auto logit = [&](const floatx4_t (&s)[2][2], int n, int i, int key0, auto mask_tag) __attribute__((always_inline)) {
    const float z = __builtin_fmaf(scale, s[i >> 2][n][i & 3], -m_ref[n]);
    if constexpr (decltype(mask_tag)::value) return key0 + 8 * quarter + i >= limit[n] ? -INFINITY : z;
    else return z;
  };
  // largest of a query's logits over the block: four lanes hold them
  auto row_max = [&](const floatx4_t (&s)[2][2], int n, int key0, auto mask_tag) __attribute__((always_inline)) {
    float zmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; ++i) zmax = fmaxf(zmax, logit(s, n, i, key0, mask_tag));
    zmax = fmaxf(zmax, __shfl_xor(zmax, 16, 64));
    return fmaxf(zmax, __shfl_xor(zmax, 32, 64));
  };

  // operands of the next matrix instructions, requested ahead: K and V fragments i sit in slot i % 4
  u32x4_t kf[4], vf[4];
  auto frag = [&](const char *base, int i) __attribute__((always_inline)) { return *reinterpret_cast<const u32x4_t *>(base + i * 1024); };

  // One pipeline step: S^T of the next block (K fragments at kp), the weights of this block
  // (s_in -> p_out), O^T of the block before (V fragments at vp, p_in): three independent streams.
  // kn, vn: the fragments of the step after.
  auto step = [&](const char *kp, const char *vp, const char *kn, const char *vn, const floatx4_t (&s_in)[2][2], floatx4_t (&s_out)[2][2],
                  const u32x4_t (&p_in)[2], u32x4_t (&p_out)[2], int key0, auto mask_tag) __attribute__((always_inline)) {
    constexpr int HALVES = 16 / (2 * NF);   // exponentials per fragment
    float blk[2], z[16], e[16];   // element h: query column h / 8, key h % 8
    auto form = [&](int j) __attribute__((always_inline)) {   // the logits of pair j
      z[2 * j] = logit(s_in, j >> 2, (2 * j) & 7, key0, mask_tag);
      z[2 * j + 1] = logit(s_in, j >> 2, (2 * j + 1) & 7, key0, mask_tag);
    };
    auto pack = [&](int j) __attribute__((always_inline)) {   // the weights of pair j are rounded, kept and summed
      const u32 w = pack_io_rne<F16>(e[2 * j], e[2 * j + 1]);
      p_out[j >> 2][j & 3] = w;
      if (j % 4 == 3) blk[j >> 2] = sum_weights<F16>(p_out[j >> 2]);
    };
    form(0);
    floatx4_t acc[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t) acc[t][0] = acc[t][1] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    int nk = 0, nv = 0;
#pragma unroll
    for (int o = 0; o < 2 * NF; ++o) {
      // K K V K K V ...: S^T is done a few instructions before the step ends, where the next one reads it
      if (nk < NF && o % 3 != 2) {
#pragma unroll
        for (int n = 0; n < 2; ++n) acc[nk & 1][n] = mfma_16x16x32<F16>(kf[nk % 4], qb[n][nk >> 1], acc[nk & 1][n]);
        kf[nk % 4] = nk + 4 < NF ? frag(kp, nk + 4) : frag(kn, nk + 4 - NF);
        ++nk;
      } else {
#pragma unroll
        for (int n = 0; n < 2; ++n) oacc[nv][n] = mfma_16x16x32<F16>(vf[nv % 4], p_in[n], oacc[nv][n]);
        vf[nv % 4] = nv + 4 < NF ? frag(vp, nv + 4) : frag(vn, nv + 4 - NF);
        ++nv;
      }
      // exponential h: its pair's logits were formed a pair ahead, its pair is packed a pair behind
#pragma unroll
      for (int h = o * HALVES; h < (o + 1) * HALVES; ++h) {
        const int j = h / 2;
        if (h % 2 == 0 && j + 1 < 8) form(j + 1);
        e[h] = __builtin_amdgcn_exp2f(z[h]);
        if (h % 2 == 1 && j > 0) pack(j - 1);
      }
    }
    pack(7);
#pragma unroll
    for (int t = 0; t < 2; ++t) { s_out[t][0] = acc[t][0]; s_out[t][1] = acc[t][1]; }
    // The softmax reference moves only when a weight would pass 2^16 (2^15 in fp16, whose weights
    // end at 65504); the block's sum of weights shows it, and the block is redone.
    constexpr float kMoveAt = F16 ? 32768.f : 65536.f;
    if (__any(!(blk[0] <= kMoveAt) || !(blk[1] <= kMoveAt))) {
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const float delta = fmaxf(row_max(s_in, n, key0, mask_tag), 0.f);
        const float alpha = __builtin_amdgcn_exp2f(-delta);
        m_ref[n] += delta;
#pragma unroll
        for (int d = 0; d < NF; ++d) oacc[d][n] *= alpha;
        l_part[n] *= alpha;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        form(j);
        e[2 * j] = __builtin_amdgcn_exp2f(z[2 * j]);
        e[2 * j + 1] = __builtin_amdgcn_exp2f(z[2 * j + 1]);
        pack(j);
      }
    }
    l_part[0] += blk[0];
    l_part[1] += blk[1];
  };

  if (n_tiles > 0) {
#pragma unroll
    for (int t = 0; t < 2; ++t) sacc[0][t][0] = sacc[0][t][1] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NF; ++i)
#pragma unroll
      for (int n = 0; n < 2; ++n) sacc[0][i & 1][n] = mfma_16x16x32<F16>(frag(frag0, i), qb[n][i >> 1], sacc[0][i & 1][n]);
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const float zmax = row_max(sacc[0], n, tbase * BN, std::true_type{});
      m_ref[n] = zmax == -INFINITY ? 0.f : zmax;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) { kf[i] = frag(frag0 + NF * 1024, i); vf[i] = frag(frag0 + 7 * HT + NF * 1024, i); }
  }
  auto tile_step = [&](int t, auto mask_tag) __attribute__((always_inline)) {
    copy_k(t + 3); copy_v(t + 2);
    const int key0 = (tbase + t) * BN;
    const char *const ka = frag0 + (t & 3) * HT + NF * 1024, *const va = frag0 + (4 + ((t + 3) & 3)) * HT + NF * 1024;
    const char *const kb = frag0 + ((t + 1) & 3) * HT, *const vb = frag0 + (4 + (t & 3)) * HT;
    step(ka, va, kb, vb, sacc[0], sacc[1], pop[1], pop[0], key0, mask_tag);
    step(kb, vb, kb + NF * 1024, vb + NF * 1024, sacc[1], sacc[0], pop[0], pop[1], key0 + 32, mask_tag);
    wait_copies<2 * PIECES>();   // (what the tile before asked for: the next tile reads it)
    __syncthreads();
  };
  int t = 0;
  for (; t < n_full; ++t) tile_step(t, std::false_type{});
  for (; t < n_tiles; ++t) tile_step(t, std::true_type{});
  if (n_tiles > 0) {
    wait_copies<0>();   // (none may be under way when the next block fills the slots, or when the workgroup ends)
    const char *vp = frag0 + (4 + ((n_tiles - 1) & 3)) * HT + NF * 1024;
#pragma unroll
    for (int i = 0; i < NF; ++i)
#pragma unroll
      for (int n = 0; n < 2; ++n) oacc[i][n] = mfma_16x16x32<F16>(frag(vp, i), pop[1][n], oacc[i][n]);
  }

#pragma unroll
  for (int n = 0; n < 2; ++n) {
    float l_sum = l_part[n] + __shfl_xor(l_part[n], 16, 64);
    l_sum += __shfl_xor(l_sum, 32, 64);
    const float inv = l_sum > 0.f ? 1.0f / l_sum : 0.f;
    const int qrow = qrow0 + n * 16 + r16;
    if (qrow >= p.Lq) continue;
    // register i of tile d is channel 16*d + 4*quarter + i
    if (partial) {
      const int64_t prow = (int64_t)(2 * w + (round == e.rounds ? 0 : 1)) * BQ + wave * 32 + n * 16 + r16;
      if (quarter == 0) *reinterpret_cast<float2 *>(e.ws_ml + prow * 2) = make_float2(m_ref[n], l_sum);
      float *wptr = e.ws_o + prow * D + 4 * quarter;
#pragma unroll
      for (int d = 0; d < NF; ++d)
        *reinterpret_cast<float4 *>(wptr + d * 16) = make_float4(oacc[d][n][0] * inv, oacc[d][n][1] * inv, oacc[d][n][2] * inv, oacc[d][n][3] * inv);
    } else {
      __bf16 *optr = p.out + (b * p.o_bs + hq * p.o_hs + qrow * p.o_ts) * D + 4 * quarter;
#pragma unroll
      for (int d = 0; d < NF; ++d)
        *reinterpret_cast<uint2 *>(optr + d * 16) =
            make_uint2(pack_io_rne<F16>(oacc[d][n][0] * inv, oacc[d][n][1] * inv), pack_io_rne<F16>(oacc[d][n][2] * inv, oacc[d][n][3] * inv));
    }
  }
  }
}

// The query blocks that fell on several workgroups: the partial outputs weighted by their softmax
// mass l * 2^(m - M) (0: it saw no key; a NaN counts, and makes the result one).  A workgroup serves 1024 / D rows of one block, a thread four channels of a row.
template <int D, bool F16>
__global__ __launch_bounds__(256) void wide_combine_kernel(WideParams e, int n_wgs) {
  const AttnParams &p = e.a;
  const SharedUnits shared(e, n_wgs);
  const int qblock = e.rounds * n_wgs + blockIdx.y, tid = threadIdx.x;
  const int row = blockIdx.x * (1024 / D) + tid / (D / 4), c0 = tid % (D / 4) * 4;
  const int64_t u0 = (int64_t)qblock * e.all_tiles;
  const int w0 = shared.owner(u0), w1 = shared.owner(u0 + e.all_tiles - 1);
  const int bh = qblock / p.q_tiles, qrow = (qblock - bh * p.q_tiles) * 256 + row;
  if (w0 == w1 || qrow >= p.Lq) return;
  // (a workgroup whose units start inside the block or with it has it as its first, any other as its last)
  // (those behind w0, the last that starts at or before u0, start inside; asked of each, a division in 64 bits)
  const int first_slot = shared.begin(w0) >= u0 ? 0 : 1;
  auto slot_row = [&](int w) { return (int64_t)(2 * w + (w == w0 ? first_slot : 0)) * 256 + row; };
  // (kAhead parts are requested before the first is used: one by one, each a trip to memory, and with the division above for each, 32 blocks of 256
  // queries took 13.9 us, now 10.1)
  constexpr int kAhead = 4;
  float M = -INFINITY;
  for (int w = w0; w <= w1; w += kAhead) {
    float2 ml[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) ml[i] = *reinterpret_cast<const float2 *>(e.ws_ml + slot_row(min(w + i, w1)) * 2);
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
      if (ml[i].y != 0.f) M = fmaxf(M, ml[i].x);
  }
  float acc[4] = {0.f, 0.f, 0.f, 0.f}, sum = 0.f;
  for (int w = w0; w <= w1; w += kAhead) {
    float2 ml[kAhead];
    float4 o[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int64_t r = slot_row(min(w + i, w1));
      ml[i] = *reinterpret_cast<const float2 *>(e.ws_ml + r * 2);
      o[i] = *reinterpret_cast<const float4 *>(e.ws_o + r * D + c0);
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
      if (w + i <= w1 && ml[i].y != 0.f) {
        const float wt = ml[i].y * __builtin_amdgcn_exp2f(ml[i].x - M);
        acc[0] = __builtin_fmaf(wt, o[i].x, acc[0]); acc[1] = __builtin_fmaf(wt, o[i].y, acc[1]);
        acc[2] = __builtin_fmaf(wt, o[i].z, acc[2]); acc[3] = __builtin_fmaf(wt, o[i].w, acc[3]);
        sum += wt;
      }
  }
  const float inv = sum > 0.f ? 1.0f / sum : 0.f;
  const int b = bh / p.Hkv, hs = bh - b * p.Hkv;
  const int hq = p.head_map ? p.head_map[hs] : hs;
  *reinterpret_cast<uint2 *>(p.out + (b * p.o_bs + hq * p.o_hs + qrow * p.o_ts) * D + c0) =
      make_uint2(pack_io_rne<F16>(acc[0] * inv, acc[1] * inv), pack_io_rne<F16>(acc[2] * inv, acc[3] * inv));
}

template <int D, int BITS> void expand_bits(const ExpandParams &e, bool chan, dim3 grid, hipStream_t st) {
  if constexpr (D == 64) {
    if (e.a.f16) {
      if (chan) hipLaunchKernelGGL((expand_tiles_kernel<D, BITS, true, true>), grid, dim3(256), 0, st, e);
      else hipLaunchKernelGGL((expand_tiles_kernel<D, BITS, false, true>), grid, dim3(256), 0, st, e);
      return;
    }
  }
  if (chan) hipLaunchKernelGGL((expand_tiles_kernel<D, BITS, true, false>), grid, dim3(256), 0, st, e);
  else hipLaunchKernelGGL((expand_tiles_kernel<D, BITS, false, false>), grid, dim3(256), 0, st, e);
}

template <int D, bool F16, int NW> void launch_wide_shape(const WideParams &e, int n_wgs, hipStream_t st) {
  constexpr int lds_bytes = 8 * kHalfTile<D>;
  static bool configured[64] = {false};
  allow_lds(reinterpret_cast<const void *>(&wide_attn_kernel<D, F16, NW>), lds_bytes, configured);
  hipLaunchKernelGGL((wide_attn_kernel<D, F16, NW>), dim3((unsigned)n_wgs), dim3(NW * 64), lds_bytes, st, e);
}
template <int D, bool F16> void launch_wide_waves(const WideParams &e, const WidePlan &plan, hipStream_t st) {
  if (plan.waves == 4) {
    launch_wide_shape<D, F16, 4>(e, plan.n_wgs, st);
    return;
  }
  launch_wide_shape<D, F16, 8>(e, plan.n_wgs, st);
  const int64_t left = (int64_t)e.a.bh_total * e.a.q_tiles - (int64_t)e.rounds * plan.n_wgs;   // (none under key limits)
  if (left > 0)
    hipLaunchKernelGGL((wide_combine_kernel<D, F16>), dim3(256 / (1024 / D), (unsigned)left), dim3(256), 0, st, e, plan.n_wgs);
}

}  // namespace

namespace varq_attn {

// A sequence attended as a whole under key limits ends when its last query blocks do, which see every key: with few pairs
// most of the device waits for them, and blocks of 128 queries are done sooner (a tile takes four wavefronts 1.25 us where it takes eight 1.8)
// and are twice as many to fill it with.  Block-causal rule, 4-bit codes, us, the kernel that widens per workgroup / blocks of
// 256 / of 128: D=64, 16 pairs of 680 tokens 19.3 / 21.8 / 16.7, of 2440 61.1 / 56.0 / 42.1, of 5064 130 / 114 / 116; 32 pairs of 255
// 10.9 / 14.8 / 11.5, of 680 21.9 / 23.5 / 18.7, of 1656 43.4 / 45.2 / 35.6, of 2440 63.7 / 61.8 / 63.6, of 3464 130 / 139 / 116; D=128, 16 of 680 29.4 / 31.6 / 24.2,
// of 2440 89.2 / 83.5 / 64.6, of 5064 176 / 156 / 184; 32 of 680 32.2 / 35.6 / 28.7, of 1656 63.6 / 65.0 / 59.7, of 2440 91 / 86 / 99.  With 64 pairs the
// device is full: 680 tokens 22.3 / 26.9 / 23.1 and 33.3 / 41.4 / 41.4.  With fewer than ten pairs the shares of the keys do
// better (8 pairs, widening / 128: D=64 1656 tokens 26.0 / 27.7, 2440 35.5 / 37.8; 10 pairs of 2440 43.8 / 39.0,
// of 5064 127 / 106; D=128 44.5 / 40.9 at 1656, 178 / 185 at 5064), and 155 tokens are too few (11.3 / 15.0).
// (The kernel that widens has since got shares of wavefronts, which are ahead of these blocks up to about 2000 tokens: limited_shares has the last word.)
// Without limits, where the shares of the keys fill the device, a block of 128 gains at most a tenth, and only where it takes exactly the
// device and the keys are few.  All launches, 4-bit codes, us, widening per workgroup with its shares / blocks of 256 / of 128 (the last
// measured earlier and on another card than the others, by up to a tenth slower):
//   D=128, queries x keys   16 pairs          32 pairs          64 pairs           128 pairs
//    256 x  521         19.5 / 27.4 / 21.6   23.4 / 30.6 / 25.0   26.4 / 37.8 / 32.2   27.5 / 42.4 / 38.6
//    256 x 2521         27.2 / 34.8 / 61.9   33.4 / 41.3 / 64.6   41.2 / 56.8 / 67.0   62.3 / 98.2 / 87.1
//    512 x  521         22.8 / 27.3 / 21.9   26.3 / 31.0 / 25.1   26.9 / 37.7 / 34.2   30.1 / 44.0 / 49.1
//    512 x 1024         28.3 / 35.4 / 29.5   34.0 / 44.9 / 37.8   42.6 / 51.3 / 46.0   45.9 / 60.0 / 67.9
//    512 x 2521         35.0 / 38.0 / 62.0   42.4 / 47.4 / 64.9   62.5 / 74.6 / 70.1   97.1 / 114 / 135
//   1024 x 1024         35.1 / 38.2 / 30.6   42.0 / 46.5 / 40.3   46.2 / 56.2 / 62.9   88.8 / 92.6 / 107
//   1024 x 2521         45.2 / 45.0 / 62.8   62.1 / 66.3 / 66.6   97.3 / 97.2 / 114    190 / 195 / 230
//   D=64
//    256 x  521         12.9 / 18.4 / 15.4   14.9 / 19.8 / 17.0   17.8 / 22.9 / 21.0   18.2 / 31.2 / 28.4
//    512 x 1024         17.7 / 25.6 / 21.6   21.8 / 28.5 / 25.5   28.6 / 35.6 / 33.0   30.2 / 45.1 / 47.8
//   1024 x 1024         23.5 / 25.5 / 21.8   28.4 / 28.9 / 26.1   30.4 / 37.7 / 41.5   48.9 / 58.9 / 61.7
//   1024 x 2521         32.1 / 37.5 / 42.7   47.5 / 45.8 / 51.8   63.6 / 67.8 / 72.7   111 / 118 / 124
// (8-bit codes within 7 % of these.)
bool wide_four(int64_t bh, int Lq, int Lk, int D, int cus, bool limits) {
  return limits && Lk <= Lq && Lq > 192 && bh * 26 >= cus && bh * 8 <= cus && bh * ((Lq + 127) / 128) * 4 <= (D == 128 ? 7 : 10) * (int64_t)cus;
}
WidePlan plan_wide(int64_t bh, int Lq, int Lk, int D, int cus, bool share, bool limits) {
  WidePlan w;
  w.waves = wide_four(bh, Lq, Lk, D, cus, limits) ? 4 : 8;
  const int block = 32 * w.waves;
  const int64_t blocks = bh * ((Lq + block - 1) / block), tiles = (Lk + BN - 1) / BN;
  w.tile_bytes = (size_t)bh * (size_t)tiles * (size_t)(2 * BN * D * 2);
  w.n_wgs = (int)blocks;
  w.rounds = 1;
  w.ws_bytes = w.tile_bytes;
  if (limits) {
    // Blocks of unequal length that only the device knows: a workgroup each, dealt out by the hardware in the order of
    // HeavyFirst (an XCD takes every eighth pair; the grid is padded to whole eighths).  Dealt out beforehand in equal
    // numbers of blocks, or of all tiles, the longest workgroup has as much to do as without limits: 32 pairs of 10521
    // tokens, D=128, block-causal, 1386 us against 1057 like this (1598 without limits).
    w.n_wgs = (int)((bh + 7) / 8 * 8 * ((Lq + block - 1) / block));
    return w;
  }
  // One workgroup runs on a compute unit.  Whole blocks take ceil(blocks / cus) rounds; sharing the
  // last, unfilled round out evenly takes its fraction of a round, and the way of the partial results
  // through memory.
  const double tile_us = D == 128 ? 1.9 : 1.2, fixed_us = 6.0;
  const int64_t rounds = blocks / cus, left = (blocks - rounds * cus) * tiles;
  int64_t n = rounds ? cus : left / 4 < cus ? left / 4 : cus;
  if (share && n > 1 && left) {
    const double whole = (double)tiles * tile_us + fixed_us;
    const double pieces = (double)(n + blocks - rounds * cus);   // at most this many partial results, written and read at 5 TB/s
    const double shared = (double)left / (double)n * tile_us + 2.0 * fixed_us + 5.0 + 2.0 * pieces * 256.0 * D * 4.0 / 5.0e6;
    if (shared < whole) {
      w.n_wgs = (int)n;
      w.rounds = (int)rounds;
      w.ws_bytes += (size_t)(2 * n) * 256 * (size_t)(D + 2) * sizeof(float);
    }
  }
  return w;
}

void launch_expand(const AttnParams &p, int D, int bits, int k_group, int v_group, bool chan, char *tiles, hipStream_t st) {
  ExpandParams e;
  e.a = p;
  e.tiles = tiles;
  e.n_tiles = (p.Lk + BN - 1) / BN;
  e.kg_shift = varq_log2_exact(k_group);
  e.vg_shift = varq_log2_exact(v_group);
  dim3 grid((unsigned)e.n_tiles, (unsigned)p.bh_total);
#define VARQ_EXPAND(D_)                                        \
  do {                                                         \
    if (bits == 4) expand_bits<D_, 4>(e, chan, grid, st);      \
    else if (bits == 8) expand_bits<D_, 8>(e, chan, grid, st); \
    else expand_bits<D_, 2>(e, chan, grid, st);                \
  } while (0)
  if (D == 128) VARQ_EXPAND(128);
  else VARQ_EXPAND(64);
#undef VARQ_EXPAND
}

void launch_expand_classes(const AttnParams &p, int D, const ClassTable &t, int group, char *tiles, hipStream_t st) {
  ExpandParams e;
  e.a = p;
  e.tiles = tiles;
  e.n_tiles = (p.Lk + BN - 1) / BN;
  e.kg_shift = e.vg_shift = varq_log2_exact(group);
  dim3 grid((unsigned)e.n_tiles, (unsigned)p.bh_total);
  if (D == 128) hipLaunchKernelGGL((expand_classes_kernel<128, false>), grid, dim3(256), 0, st, e, t);
  else if (p.f16) hipLaunchKernelGGL((expand_classes_kernel<64, true>), grid, dim3(256), 0, st, e, t);
  else hipLaunchKernelGGL((expand_classes_kernel<64, false>), grid, dim3(256), 0, st, e, t);
}

void launch_wide(const AttnParams &p, int D, const WidePlan &plan, char *ws, hipStream_t st) {
  WideParams e;
  e.a = p;
  e.tiles = ws;
  e.all_tiles = (p.Lk + BN - 1) / BN;
  e.rounds = plan.rounds;
  e.ws_o = reinterpret_cast<float *>(ws + plan.tile_bytes);
  e.ws_ml = e.ws_o + (size_t)(2 * plan.n_wgs) * 256 * (size_t)D;
  e.a.q_tiles = (p.Lq + 32 * plan.waves - 1) / (32 * plan.waves);
  if (D == 128) launch_wide_waves<128, false>(e, plan, st);
  else if (p.f16) launch_wide_waves<64, true>(e, plan, st);
  else launch_wide_waves<64, false>(e, plan, st);
}

}  // namespace varq_attn
