// Unpack + dequantize in one pass: what VAR_Q/quant.py:216-224 does with two
// unpack launches per field, a stack, a sign-extension and a multiply
// (VAR_Q/pack_unpack.py:198-211, VAR_Q/quant.py:123-124), plus the affine form
// (q - zp) * scale.  HBM-bound; the output (fp32 in the reference, 4 B/element)
// dominates the traffic, so bf16/fp16 outputs are offered too.
//
// One lane produces 8 consecutive channels.  A block stays inside one (i0,i1)
// pair so the scale base and the input-window row base are block-uniform.
#include "dequant_steps.h"
#include <type_traits>

using namespace varq_deq;

namespace {

struct DeqParams {
  const int32_t *words;
  const int8_t *codes;
  const float *scale;
  const float *zp;
  void *out;
  RowMap in_map;           // (i0,i1,i2) -> input row
  int64_t n1, n2;
  int64_t ss0, ss1, ss2, ss3;
  int64_t octets_per_pair;
  int c, c8, wpr, bits, group;
  int c8_shift;            // log2(c8) when c8 is a power of two, else -1
};

// Any codes, groups, strides and alignments; U items (octets) per lane, 256 lanes apart.
template <int ODT, int U>
__global__ __launch_bounds__(256) void dequant_kernel(DeqParams p) {
  // grid = (tiles of 256*U octets, i1, i0): no division to find the block's place
  const int64_t i0 = blockIdx.z, i1 = blockIdx.y;
  const int o0 = blockIdx.x * (256 * U) + threadIdx.x;   // first octet inside the (i0, i1) pair, < 2^31
  const int64_t sbase0 = i0 * p.ss0 + i1 * p.ss1;
  const int64_t in_base = i0 * p.in_map.os0 + i1 * p.in_map.os1 + p.in_map.off;
  const int64_t out_base = (i0 * p.n1 + i1) * p.n2;
#pragma unroll 1
  for (int u = 0; u < U; ++u) {
  const int o = o0 + u * 256;
  if (o >= p.octets_per_pair) return;
  int i2, col;
  if (p.c8_shift >= 0) { i2 = o >> p.c8_shift; col = o & (p.c8 - 1); }
  else { i2 = o / p.c8; col = o - i2 * p.c8; }
  const int ch0 = col * 8;
  const int n_valid = min(8, p.c - ch0);
  const int64_t in_row = in_base + i2 * p.in_map.os2;
  const int64_t out_row = out_base + i2;

  int q[8];
  if (p.codes) {
    const int8_t *src = p.codes + in_row * p.c + ch0;
    if (n_valid == 8 && (p.c & 7) == 0) {
      uint2 b = *reinterpret_cast<const uint2 *>(src);
#pragma unroll
      for (int j = 0; j < 4; ++j) { q[j] = __builtin_amdgcn_sbfe((int)b.x, 8 * j, 8); q[4 + j] = __builtin_amdgcn_sbfe((int)b.y, 8 * j, 8); }
    } else {
      for (int j = 0; j < 8; ++j) q[j] = j < n_valid ? src[j] : 0;
    }
  } else {
    const int32_t *src = p.words + in_row * p.wpr;
    if (p.bits == 4) {
      const int w = src[col];
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = __builtin_amdgcn_sbfe(w, 4 * j, 4);
    } else if (p.bits == 8) {
      const int w0 = src[col * 2];
      const int w1 = (col * 2 + 1 < p.wpr) ? src[col * 2 + 1] : 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) { q[j] = __builtin_amdgcn_sbfe(w0, 8 * j, 8); q[4 + j] = __builtin_amdgcn_sbfe(w1, 8 * j, 8); }
    } else {
      const int w = src[col >> 1] >> ((col & 1) * 16);
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = __builtin_amdgcn_sbfe(w, 2 * j, 2);
    }
  }

  const int64_t sbase = sbase0 + i2 * p.ss2;
  float f[8];
  if ((p.group & 7) == 0) {
    const int64_t g = sbase + (ch0 / p.group) * p.ss3;
    const float s = p.scale[g];
    if (p.zp) {
      const float z = p.zp[g];
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = ((float)q[j] - z) * s;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = (float)q[j] * s;
    }
  } else if (p.group == 1 && p.ss3 == 1 && n_valid == 8 && ((sbase + ch0) & 3) == 0) {
    // one scale per channel, contiguous: two 16-byte loads
    const float4 *sp = reinterpret_cast<const float4 *>(p.scale + sbase + ch0);
    const float4 sa = sp[0], sb = sp[1];
    const float sv[8] = {sa.x, sa.y, sa.z, sa.w, sb.x, sb.y, sb.z, sb.w};
    if (p.zp) {
      const float4 *zq = reinterpret_cast<const float4 *>(p.zp + sbase + ch0);
      const float4 za = zq[0], zb = zq[1];
      const float zv[8] = {za.x, za.y, za.z, za.w, zb.x, zb.y, zb.z, zb.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = ((float)q[j] - zv[j]) * sv[j];
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = (float)q[j] * sv[j];
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int ch = min(ch0 + j, p.c - 1);
      const int64_t g = sbase + (ch / p.group) * p.ss3;
      const float s = p.scale[g];
      f[j] = p.zp ? ((float)q[j] - p.zp[g]) * s : (float)q[j] * s;
    }
  }
  store8<ODT>(p.out, out_row * p.c + ch0, f, ((p.c & 7) == 0) ? 8 : n_valid);
  }
}

// Packed words whose scales lie in groups of whole octets (TABLE = 0) or one per channel (1; 2: the tokens of a pair share them, and the
// lane's pieces are the same channels of U tokens, with one load): everything else takes dequant_kernel.
// Bound by HBM.  A lane stores U pieces of 16 bytes, a wavefront 1 KiB with each (two stores of 16 bytes, 32 apart, for the octet of 32-bit values: 68 us where this
// takes 55), and all loads of a lane are under way before the first is used.  Widths, divisors and kind of scales are known when the kernel is compiled or
// come as multipliers: with branches and integer divisions between the loads a launch took 2 to 3 us more at any size.  In a graph, us, before -> now: groups of
// 32, 4 bits, [3,7,1511,96] fp32 6.4 -> 4.3, bf16 5.1 -> 3.2; 2 bits [2,16,2048,128] bf16 7.0 -> 5.2; 8 bits [4,30,1000,64] fp32 10.3 -> 7.1; 4 bits [16,16,2000,128]
// fp32 77 -> 43, [16,16,4000,128] bf16 76 -> 49; a scale per (head, channel) [8,30,100,64] 8 bits fp32 4.4 -> 3.3, [2,8,8000,40] 4 bits bf16 7.2 -> 5.1.
// One piece per lane: 55 -> 83 us at 262 MB of fp32, four: 57, with the small launches the same.  But pairs of up to 256 pieces, whose second round would load and
// store nothing, have one, and their wavefronts without any end at once: a scale per (row, channel), 8 bits to bf16, 30 rows of 64 channels, 4096 pairs 8.5 -> 6.5 us (the general
// kernel 7.6), 20000 28.3 -> 19.0 (22.6), one row 24.9 -> 10.5 (15.5); groups of whole rows 1.06 times as fast, a table per head 1.12.
// STREAM: an output that does not fit the Infinity Cache with its codes goes past it (262 MB, alone / with a copy that reads it: fp32 55 / 158 -> 43 / 152, bf16 58 / 158 -> 49 / 154); a
// smaller one would be read from memory by whoever reads it next (98 MB fp32 18.6 / 48.5 -> 16.3 / 54.3, 84 MB bf16 19.0 / 43.7 -> 18.1 / 48.9).
constexpr int64_t kStreamBytes = 240ll << 20;
struct WordsParams {
  const char *words;
  const float *scale, *zp;
  void *out;
  int64_t os0, os1, off;            // input row of pair (i0, i1)
  int64_t ss0, ss1;
  int64_t n1;
  u32 row_bytes, token_bytes;       // bytes of a row of words, and from a token of a pair to the next
  int ss2, ss3;                     // floats from a token's scales to the next one's, and from a group's to the next
  int octets;                       // of a pair
  int c8;
  FastDiv by_c8, by_g8;             // octets of a row, and of a group
};
template <int ODT, int BITS, int TABLE, int U, bool STREAM>
__global__ __launch_bounds__(256) void dequant_words_kernel(WordsParams p) {
  // grid = (tiles of 256 * U pieces, i1, i0)
  constexpr int Q = ODT == VARQ_F32 ? 4 : 8, PER = 8 / Q;   // channels of a piece, pieces of an octet
  const int64_t i0 = blockIdx.z, i1 = blockIdx.y;
  const u32 first = blockIdx.x * (256 * U) + threadIdx.x, n = (u32)p.octets * PER;
  if (U == 1 && first >= n) return;
  const char *const words = p.words + (i0 * p.os0 + i1 * p.os1 + p.off) * p.row_bytes;
  const int64_t table = i0 * p.ss0 + i1 * p.ss1;
  const float *const scale = p.scale + table, *const zp = p.zp ? p.zp + table : nullptr;
  constexpr int V = TABLE ? Q / 4 : 1, N = TABLE == 2 ? 1 : U;   // vectors of scales of a piece; pieces with scales of their own
  typedef float f4 __attribute__((ext_vector_type(4)));
  u32 w0[U], w1[U];
  f4 s[N][V], z[N][V];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const u32 i = min(first + u * 256, n - 1), o = i / PER, i2 = p.by_c8(o), col = o - i2 * p.c8, ch = col * 8 + i % PER * Q;
    const char *const src = words + (size_t)(i2 * p.token_bytes + ch * BITS / 8);
    w1[u] = 0;
    if constexpr (BITS * Q == 64) { const uint2 t = *reinterpret_cast<const uint2 *>(src); w0[u] = t.x; w1[u] = t.y; }
    else if constexpr (BITS * Q == 32) w0[u] = *reinterpret_cast<const u32 *>(src);
    else if constexpr (BITS * Q == 16) w0[u] = *reinterpret_cast<const uint16_t *>(src);
    else w0[u] = *reinterpret_cast<const unsigned char *>(src);
    if (u < N) {
      if constexpr (TABLE) {
#pragma unroll
        for (int h = 0; h < V; ++h) {
          const u32 g = (TABLE == 1 ? i2 * (u32)p.ss2 : 0) + ch + 4 * h;
          s[u][h] = *reinterpret_cast<const f4 *>(scale + g);
          if (zp) z[u][h] = *reinterpret_cast<const f4 *>(zp + g);
        }
      } else {
        const u32 g = i2 * (u32)p.ss2 + p.by_g8(col) * (u32)p.ss3;
        s[u][0][0] = scale[g];
        if (zp) z[u][0][0] = zp[g];
      }
    }
  }
  const int64_t pair = (i0 * p.n1 + i1) * n;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const u32 i = first + u * 256;
    const int m = TABLE == 2 ? 0 : u;
    if (i >= n) return;
    float f[8];
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      f[j] = (float)(int)(BITS == 8 ? __builtin_amdgcn_sbfe((int)(j < 4 ? w0[u] : w1[u]), 8 * (j & 3), 8) : __builtin_amdgcn_sbfe((int)w0[u], BITS * j, BITS));
      const float sj = TABLE ? s[m][j / 4 % V][j % 4] : s[m][0][0];
      f[j] = zp ? (f[j] - (TABLE ? z[m][j / 4 % V][j % 4] : z[m][0][0])) * sj : f[j] * sj;
    }
    if constexpr (Q == 4) put<STREAM>(reinterpret_cast<f4 *>(p.out) + (pair + i), f4{f[0], f[1], f[2], f[3]});
    else store8<ODT, STREAM>(p.out, (pair + i) * 8, f, 8);
  }
}

template <int ODT> void launch_words(const WordsParams &w, const int64_t *s, int bits, bool table, hipStream_t st) {
  constexpr int PER = ODT == VARQ_F32 ? 2 : 1;
  const bool stream = s[0] * s[1] * (int64_t)w.octets * 16 * PER >= kStreamBytes;
  auto pieces = [&](auto b, auto t, auto u) {
    dim3 grid((unsigned)(((int64_t)w.octets * PER + 256 * u() - 1) / (256 * u())), (unsigned)s[1], (unsigned)s[0]);
    if (stream) hipLaunchKernelGGL((dequant_words_kernel<ODT, b(), t(), u(), true>), grid, dim3(256), 0, st, w);
    else hipLaunchKernelGGL((dequant_words_kernel<ODT, b(), t(), u(), false>), grid, dim3(256), 0, st, w);
  };
  auto kind = [&](auto b, auto t) {
    if ((int64_t)w.octets * PER <= 256) pieces(b, t, std::integral_constant<int, 1>{});
    else pieces(b, t, std::integral_constant<int, 2>{});
  };
  auto width = [&](auto b) {
    if (!table) kind(b, std::integral_constant<int, 0>{});
    else if (w.ss2 == 0 && 256 % (w.c8 * PER) == 0) kind(b, std::integral_constant<int, 2>{});
    else kind(b, std::integral_constant<int, 1>{});
  };
  if (bits == 4) width(std::integral_constant<int, 4>{});
  else if (bits == 8) width(std::integral_constant<int, 8>{});
  else width(std::integral_constant<int, 2>{});
}

template <int ODT, int BITS, int U>
__global__ __launch_bounds__(256) void dequant_steps_kernel(StepParams p) {
  if constexpr (ODT == VARQ_F32) dequant_steps_halves<BITS, 256, U>(p, (int64_t)blockIdx.z * gridDim.y + blockIdx.y, blockIdx.x);
  else dequant_steps_block<ODT, BITS, 256, U>(p, (int64_t)blockIdx.z * gridDim.y + blockIdx.y, blockIdx.x);
}

}  // namespace

extern "C" int varq_dequant_steps(const int32_t *words, const float *scale, const float *zp, int nseg, const int32_t *host_seg_end,
                                  int B, int H, int64_t capacity, int c, int bits, int tokens_first, void *out, int out_dtype, void *stream) {
  VARQ_CHECK_ARG(words && scale && out && host_seg_end, "dequant_steps: null pointer");
  VARQ_CHECK_ARG(nseg >= 1 && nseg <= 16 && B > 0 && H > 0 && c > 0 && c % 8 == 0, "dequant_steps: bad sizes (1..16 segments, whole octets of channels)");
  VARQ_CHECK_ARG((bits == 2 || bits == 4 || bits == 8) && (c * bits) % 32 == 0, "dequant_steps: bits must be 2, 4 or 8 and rows whole words");
  VARQ_CHECK_ARG(out_dtype >= 0 && out_dtype <= 2, "dequant_steps: bad output dtype %d", out_dtype);
  VARQ_CHECK_ARG((((uintptr_t)scale | (uintptr_t)zp | (uintptr_t)out) & 15) == 0 && ((uintptr_t)words & 7) == 0, "dequant_steps: misaligned operand");
  StepParams p;
  const int64_t tokens = host_seg_end[nseg - 1];
  for (int s = 0, prev = 0; s < nseg; prev = host_seg_end[s++])
    VARQ_CHECK_ARG(host_seg_end[s] >= prev, "dequant_steps: segment ends must increase");
  VARQ_CHECK_ARG(tokens <= capacity && set_steps(p, words, scale, zp, nseg, host_seg_end, B, H, capacity, c, bits, tokens_first, out),
                 "dequant_steps: more tokens than the buffer or the grid holds");
  if (tokens <= 0) return VARQ_OK;
  hipStream_t st = (hipStream_t)stream;
  auto launch = [&](auto odt, auto width, auto per) {
    // (pair b * H + h is block (h, b): the grid's limit holds for each dim, as in varq_dequant)
    dim3 grid((unsigned)((p.pair_octs + 256 * per() - 1) / (256 * per())), (unsigned)(tokens_first ? 1 : H), (unsigned)B);
    hipLaunchKernelGGL((dequant_steps_kernel<odt(), width(), per()>), grid, dim3(256), 0, st, p);
  };
  // An octet per lane up to four workgroups per compute unit: a chain of one, where four cost the small launches their idle rounds and the search for the
  // block's steps.  All tokens of the first 1, 2 and 5 of ten steps, five forms of [1..32,n,6..30,64..128], in a graph, us, four / one: to fp32 2.73 / 2.24, 3.66 / 2.32,
  // 4.15 / 3.04, to 16 bits 2.59 / 2.13, 3.05 / 2.15, 3.36 / 2.71; from 2^18 octets on it goes either way, one up to 15 % behind.
  const bool few = (int64_t)B * (tokens_first ? 1 : H) * p.pair_octs <= 1 << 18;
  auto of = [&](auto odt, auto width) {
    if (few) launch(odt, width, std::integral_constant<int, 1>{});
    else launch(odt, width, std::integral_constant<int, 4>{});
  };
#define VARQ_STEPS(ODT_)                                        \
  do {                                                          \
    std::integral_constant<int, ODT_> odt;                      \
    if (bits == 8) of(odt, std::integral_constant<int, 8>{});   \
    else if (bits == 4) of(odt, std::integral_constant<int, 4>{}); \
    else of(odt, std::integral_constant<int, 2>{});             \
  } while (0)
  if (out_dtype == VARQ_F32) VARQ_STEPS(VARQ_F32);
  else if (out_dtype == VARQ_BF16) VARQ_STEPS(VARQ_BF16);
  else VARQ_STEPS(VARQ_F16);
#undef VARQ_STEPS
  VARQ_CHECK_LAUNCH("dequant_steps");
  return VARQ_OK;
}

extern "C" int varq_dequant(const int32_t *words, const int8_t *codes_i8, const float *scale, const float *zp,
                            const int64_t *host_shape4, const int64_t *host_scale_strides4, int group, int bits,
                            const int64_t *host_in_rowmap, void *out, int out_dtype, void *stream) {
  VARQ_CHECK_ARG(host_shape4 && host_scale_strides4, "dequant: null shape/strides");
  const int64_t *s = host_shape4;
  VARQ_CHECK_ARG(s[0] >= 0 && s[1] >= 0 && s[2] >= 0 && s[3] > 0 && s[3] <= (1 << 20), "dequant: bad shape");
  // (a tensor without rows may come as null pointers: nothing to do)
  if (s[0] * s[1] * s[2] == 0) return VARQ_OK;
  VARQ_CHECK_ARG((words != nullptr) != (codes_i8 != nullptr), "dequant: exactly one of words/codes must be given");
  VARQ_CHECK_ARG(!words || bits == 2 || bits == 4 || bits == 8, "dequant: bits must be 2, 4 or 8 (got %d)", bits);
  VARQ_CHECK_ARG(out_dtype >= 0 && out_dtype <= 2, "dequant: bad output dtype %d", out_dtype);
  VARQ_CHECK_ARG(group >= 1 && group <= s[3], "dequant: bad group %d", group);
  const int64_t rows = s[0] * s[1] * s[2];
  if (rows == 0) return VARQ_OK;
  VARQ_CHECK_ARG(scale && out, "dequant: null pointer");

  DeqParams p;
  p.words = words; p.codes = codes_i8; p.scale = scale; p.zp = zp; p.out = out;
  p.n1 = s[1]; p.n2 = s[2];
  p.c = (int)s[3];
  p.c8 = (p.c + 7) / 8;
  p.bits = bits; p.group = group;
  p.wpr = words ? (p.c + 32 / bits - 1) / (32 / bits) : 0;
  p.ss0 = host_scale_strides4[0]; p.ss1 = host_scale_strides4[1];
  p.ss2 = host_scale_strides4[2]; p.ss3 = host_scale_strides4[3];
  if (host_in_rowmap) {
    p.in_map = varq_rowmap_from_host(host_in_rowmap, rows);
    VARQ_CHECK_ARG(p.in_map.n0 == s[0] && p.in_map.n1 == s[1] && p.in_map.n2 == s[2], "dequant: row map dims differ from shape");
    VARQ_CHECK_ARG(p.in_map.slot_dim < 0, "dequant: slot tables are not supported on input maps");
  } else {
    p.in_map.n0 = s[0]; p.in_map.n1 = s[1]; p.in_map.n2 = s[2];
    p.in_map.os0 = s[1] * s[2]; p.in_map.os1 = s[2]; p.in_map.os2 = 1; p.in_map.off = 0; p.in_map.slot_dim = -1;
  }
  p.octets_per_pair = s[2] * p.c8;
  p.c8_shift = -1;
  for (int sh = 0; sh < 20; ++sh)
    if ((1 << sh) == p.c8) p.c8_shift = sh;
  // a pair with few rows wastes lanes of its last block only; pairs map to grid.y/z (limit 65535 each)
  VARQ_CHECK_ARG(p.octets_per_pair < (1ll << 31) - 1024 && s[1] <= 65535 && s[0] <= 65535, "dequant: shape exceeds the grid limits");
  hipStream_t st = (hipStream_t)stream;
  const bool table = group == 1 && p.ss3 == 1 && (s[2] == 1 || p.ss2 % 4 == 0) && (s[0] == 1 || p.ss0 % 4 == 0) && (s[1] == 1 || p.ss1 % 4 == 0) && (((uintptr_t)scale | (uintptr_t)zp) & 15) == 0;
  const int64_t token_bytes = p.in_map.os2 * p.wpr * 4;
  // (places inside a pair are counted in 32 bits)
  if (words && s[3] % 8 == 0 && (bits != 8 || ((uintptr_t)words & 7) == 0) && (group % 8 == 0 || table) && ((uintptr_t)out & 15) == 0 && token_bytes >= 0 &&
      token_bytes <= (1ll << 32) / s[2] - 1 && p.ss2 >= 0 && p.ss3 >= 0 && p.ss2 <= (1ll << 30) / s[2] && p.ss3 <= (1ll << 30) / s[3]) {
    WordsParams w;
    w.words = reinterpret_cast<const char *>(words); w.scale = scale; w.zp = zp; w.out = out;
    w.os0 = p.in_map.os0; w.os1 = p.in_map.os1; w.off = p.in_map.off; w.ss0 = p.ss0; w.ss1 = p.ss1; w.n1 = s[1];
    w.row_bytes = (u32)p.wpr * 4; w.token_bytes = (u32)token_bytes; w.ss2 = (int)p.ss2; w.ss3 = (int)p.ss3;
    w.octets = (int)p.octets_per_pair; w.c8 = p.c8; w.by_c8 = FastDiv::by(p.c8); w.by_g8 = FastDiv::by(table ? 1 : group / 8);
    if (out_dtype == VARQ_F32) launch_words<VARQ_F32>(w, s, bits, table, st);
    else if (out_dtype == VARQ_BF16) launch_words<VARQ_BF16>(w, s, bits, table, st);
    else launch_words<VARQ_F16>(w, s, bits, table, st);
    VARQ_CHECK_LAUNCH("dequant");
    return VARQ_OK;
  }
  // The octets of a lane follow one another: four where a pair has the work for it, two where four would leave more than a twelfth of the last block's lanes idle
  // (four / two, us: int8 codes [3,6,173,128] fp16 4.0 / 3.1, [8,6,662,64] fp32 6.0 / 5.1, packed rows of 100 channels [12,30,177,100] fp16 15.4 / 12.3).
  int U = p.octets_per_pair >= 2048 ? 4 : 1;
  if (U == 4 && !(group == 1 && p.ss3 == 1 && p.ss2 == 0)) {
    const int64_t t4 = (p.octets_per_pair + 1023) / 1024;
    if ((t4 * 1024 - p.octets_per_pair) * 12 > t4 * 1024) U = 2;
  }
  const int64_t tiles = (p.octets_per_pair + 256 * U - 1) / (256 * U);
  dim3 grid((unsigned)tiles, (unsigned)s[1], (unsigned)s[0]);
#define VARQ_DEQ(ODT_)                                                                     \
  do {                                                                                     \
    if (U == 4) hipLaunchKernelGGL((dequant_kernel<ODT_, 4>), grid, dim3(256), 0, st, p);  \
    else if (U == 2) hipLaunchKernelGGL((dequant_kernel<ODT_, 2>), grid, dim3(256), 0, st, p);  \
    else hipLaunchKernelGGL((dequant_kernel<ODT_, 1>), grid, dim3(256), 0, st, p);         \
  } while (0)
  if (out_dtype == VARQ_F32) VARQ_DEQ(VARQ_F32);
  else if (out_dtype == VARQ_BF16) VARQ_DEQ(VARQ_BF16);
  else VARQ_DEQ(VARQ_F16);
#undef VARQ_DEQ
  VARQ_CHECK_LAUNCH("dequant");
  return VARQ_OK;
}
