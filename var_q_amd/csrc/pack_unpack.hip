// Stand-alone bit packing and unpacking of int8 codes, the operations of
// VAR_Q/pack_unpack.py:107-162 (Triton wrappers) and 177-211 (layout
// definition).  Pure byte shuffling, HBM-bound: one thread per four 32-bit words
// (16 bytes of words, 16 to 64 bytes of codes, all in 16-byte accesses) when a row is a
// whole number of words and both buffers are 16-byte aligned; otherwise one thread per word
// (packing, the words that are left over, and unpacking short rows or few words) or per 16 codes (unpacking other rows that do not fill their last word).
#include <algorithm>
#include <type_traits>

#include "varq_common.h"
#include "../../include/varq_testing.h"

namespace {

// 4 bytes -> their low `BITS` bits, concatenated (byte k -> field k).
template <int BITS> __device__ __forceinline__ u32 squeeze4(u32 b) {
  if (BITS == 8) return b;
  if (BITS == 4) {
    u32 t = b & 0x0f0f0f0fu;
    t = (t | (t >> 4)) & 0x00ff00ffu;
    return (t | (t >> 8)) & 0xffffu;
  }
  u32 t = b & 0x03030303u;
  t = (t | (t >> 6)) & 0x000f000fu;
  return (t | (t >> 12)) & 0xffu;
}

// field k of the low 4*BITS bits -> sign-extended byte k.
template <int BITS> __device__ __forceinline__ u32 spread4(u32 f) {
  if (BITS == 8) return f;
  u32 t;
  if (BITS == 4) {
    t = f & 0xffffu;
    t = (t | (t << 8)) & 0x00ff00ffu;
    t = (t | (t << 4)) & 0x0f0f0f0fu;
    const u32 s = t & 0x08080808u;       // sign bit of each field
    return t | ((s << 5) - (s << 1));     // fill bits 4..7 of negative fields
  }
  t = f & 0xffu;
  t = (t | (t << 12)) & 0x000f000fu;
  t = (t | (t << 6)) & 0x03030303u;
  const u32 s = t & 0x02020202u;
  return t | ((s << 7) - (s << 1));       // fill bits 2..7
}

template <int BITS> __device__ __forceinline__ u32 pack_word(const u32 *src) {   // 32/BITS codes -> one word
  if (BITS == 8) return src[0];
  if (BITS == 4) return squeeze4<4>(src[0]) | (squeeze4<4>(src[1]) << 16);
  return squeeze4<2>(src[0]) | (squeeze4<2>(src[1]) << 8) | (squeeze4<2>(src[2]) << 16) | (squeeze4<2>(src[3]) << 24);
}
template <int BITS> __device__ __forceinline__ void unpack_word(u32 x, u32 *dst) {   // one word -> 32/BITS codes
  if (BITS == 8) dst[0] = x;
  else if (BITS == 4) { dst[0] = spread4<4>(x); dst[1] = spread4<4>(x >> 16); }
  else { dst[0] = spread4<2>(x); dst[1] = spread4<2>(x >> 8); dst[2] = spread4<2>(x >> 16); dst[3] = spread4<2>(x >> 24); }
}

// Four words per thread: one 16-byte piece of words, DPW 16-byte pieces of codes.  (n_quads =
// n_words / 4; the host sends the words that are left to the per-word kernel.)
template <int BITS>
__global__ __launch_bounds__(256) void pack_quad_kernel(const int8_t *codes, int32_t *words, int64_t n_quads) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n_quads) return;
  constexpr int DPW = 8 / BITS;   // dwords of codes per word: 1, 2 or 4
  const uint4 *src = reinterpret_cast<const uint4 *>(codes) + i * DPW;
  u32 q[4 * DPW];
#pragma unroll
  for (int k = 0; k < DPW; ++k) {
    const uint4 t = src[k];
    q[4 * k] = t.x; q[4 * k + 1] = t.y; q[4 * k + 2] = t.z; q[4 * k + 3] = t.w;
  }
  reinterpret_cast<uint4 *>(words)[i] =
      make_uint4(pack_word<BITS>(q), pack_word<BITS>(q + DPW), pack_word<BITS>(q + 2 * DPW), pack_word<BITS>(q + 3 * DPW));
}

// Unpacking writes most of the bytes, so there a thread owns one 16-byte piece of codes:
// BITS / 2 words (n_pieces = n_words / (BITS / 2)).
template <int BITS>
__global__ __launch_bounds__(256) void unpack_piece_kernel(const int32_t *words, int8_t *codes, int64_t n_pieces) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n_pieces) return;
  constexpr int WPT = BITS / 2, DPW = 8 / BITS;   // words per thread, dwords of codes per word
  const u32 *src = reinterpret_cast<const u32 *>(words) + i * WPT;
  u32 x[WPT];
  if constexpr (WPT == 4) { const uint4 t = *reinterpret_cast<const uint4 *>(src); x[0] = t.x; x[1] = t.y; x[2] = t.z; x[3] = t.w; }
  else if constexpr (WPT == 2) { const uint2 t = *reinterpret_cast<const uint2 *>(src); x[0] = t.x; x[1] = t.y; }
  else x[0] = src[0];
  u32 q[4];
#pragma unroll
  for (int k = 0; k < WPT; ++k) unpack_word<BITS>(x[k], q + k * DPW);
  reinterpret_cast<uint4 *>(codes)[i] = make_uint4(q[0], q[1], q[2], q[3]);
}

// one word per thread, from word `w0` on
template <int BITS>
__global__ __launch_bounds__(256) void pack_flat_kernel(const int8_t *codes, int32_t *words, int64_t w0, int64_t n_words) {
  const int64_t w = w0 + (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (w >= n_words) return;
  constexpr int VALS = 32 / BITS;
  words[w] = (int32_t)pack_word<BITS>(reinterpret_cast<const u32 *>(codes + w * VALS));
}

template <int BITS>
__global__ __launch_bounds__(256) void unpack_flat_kernel(const int32_t *words, int8_t *codes, int64_t w0, int64_t n_words) {
  const int64_t w = w0 + (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (w >= n_words) return;
  constexpr int VALS = 32 / BITS;
  unpack_word<BITS>((u32)words[w], reinterpret_cast<u32 *>(codes + w * VALS));
}

// Rows that do not fill their last word (zero padding on pack, dropped on unpack), and code buffers
// off a 16-byte boundary.  Both kernels count rows, words and codes in 32 bits: the host hands them
// so many rows that neither the words nor the codes reach 2^31 (row_chunks).
//
// Packing reads most of the bytes: one word per thread, its 32 / BITS codes in one load of 4 to 16
// bytes at whatever byte they begin (global loads take any address), also where the row ends inside:
// what follows are codes of the next row, masked away.  Only the words that would read past the last row go
// by bytes.  Bound by memory: 400000 rows of 255 4-bit codes take 29.2 us (5.2 TB/s) where a
// load per code and a 64-bit division per word took 67.9, 40009 rows of 100 2.4 where it took 4.3.
template <int BITS>
__global__ __launch_bounds__(256) void pack_ragged_kernel(const int8_t *codes, int32_t *words, u32 n_codes, u32 n_words, u32 c, u32 wpr, FastDiv by_wpr) {
  const u32 t = blockIdx.x * 256 + threadIdx.x;
  if (t >= n_words) return;
  constexpr u32 VALS = 32 / BITS, DPW = 8 / BITS;
  const u32 r = by_wpr(t), ch = (t - r * wpr) * VALS, at = r * c + ch;
  const u32 n = min(VALS, c - ch);
  u32 w;
  if (at + VALS <= n_codes) {
    u32 q[DPW];
    __builtin_memcpy(q, codes + at, VALS);
    w = pack_word<BITS>(q);
  } else {
    w = 0;
    for (u32 j = 0; j < n; ++j) w |= ((u32)(int)codes[at + j] & ((1u << BITS) - 1u)) << (j * BITS);
  }
  words[t] = (int32_t)(w & (0xffffffffu >> ((VALS - n) * BITS)));
}

// Unpacking writes most of the bytes: one piece of 16 codes per thread, stored whole, whichever rows
// they belong to (two at most: rows are of 15 codes or more).  The words of a row hold its codes as one run of bits, so the piece's
// part of a row is BITS / 2 words of that run, shifted into place from one word more; where the piece goes on
// in the next row, the same window is taken so far before that row's first word that its codes
// land in their places, and the two are joined by a mask.
// Bound by memory: 400000 rows of 255 4-bit codes take 28.3 us where a word per thread, stored by bytes, takes 68.0; of 100 11.8 / 29.5.
// The pieces whose windows would end behind the last word take them word by word, and store what there is of the last one by bytes.
template <int BITS> struct Window {   // 16 codes
  static constexpr u32 VALS = 32 / BITS, WIN = BITS / 2;
  u32 x[WIN + 1], shift;
  template <bool INSIDE> __device__ __forceinline__ void take(const u32 *words, u32 n_words, u32 field) {   // from `field` on, counted in fields
    const u32 w = field / VALS;
    shift = field % VALS * BITS;
    if constexpr (INSIDE) {
      __builtin_memcpy(x, words + w, sizeof x);
    } else {
#pragma unroll
      for (u32 k = 0; k <= WIN; ++k) x[k] = words[min(w + k, n_words - 1)];   // (the codes that are there lie in words that are there)
    }
  }
  __device__ __forceinline__ u32 word(u32 k) const { return __builtin_amdgcn_alignbit(x[k + 1], x[k], shift); }
};
template <int BITS>
__global__ __launch_bounds__(256) void unpack_ragged_kernel(const int32_t *words, int8_t *codes, u32 n_codes, u32 n_words, u32 c, u32 wpr, FastDiv by_c) {
  const u32 at = (blockIdx.x * 256 + threadIdx.x) * 16;
  if (at >= n_codes) return;
  constexpr u32 VALS = 32 / BITS, WIN = BITS / 2, DPW = 8 / BITS;
  const u32 *const src = reinterpret_cast<const u32 *>(words);
  const u32 r = by_c(at), ch = at - r * c, first = r * wpr * VALS + ch, got = c - ch;   // got: codes of the piece in the first row
  const u32 second = first - ch + wpr * VALS - got;   // (a field that is there: c <= wpr * VALS)
  u32 q[4];
  auto piece = [&](auto inside) __attribute__((always_inline)) {
    Window<BITS> a, b;
    a.template take<inside()>(src, n_words, first);
    u32 w[WIN];
#pragma unroll
    for (u32 k = 0; k < WIN; ++k) w[k] = a.word(k);
    if (got < 16) {
      b.template take<inside()>(src, n_words, second);
#pragma unroll
      for (u32 k = 0; k < WIN; ++k) {
        const u32 in = got > k * VALS ? min(got - k * VALS, VALS) : 0u;   // fields of this word that are the first row's
        const u32 m = in ? 0xffffffffu >> ((VALS - in) * BITS) : 0u;
        w[k] = (w[k] & m) | (b.word(k) & ~m);
      }
    }
#pragma unroll
    for (u32 k = 0; k < WIN; ++k) unpack_word<BITS>(w[k], q + k * DPW);
  };
  if (at + 16 <= n_codes && (got < 16 ? second : first) / VALS + WIN < n_words) {
    piece(std::true_type{});
    __builtin_memcpy(codes + at, q, 16);
  } else {
    piece(std::false_type{});
#pragma unroll
    for (u32 j = 0; j < 16; ++j)
      if (at + j < n_codes) codes[at + j] = (int8_t)(q[j / 4] >> (8 * (j % 4)));
  }
}
// A word per thread, its codes stored by bytes: rows of less than 15 codes (by pieces of 16 and a window per row, 1.8-2.2 us where it takes 1.75-2.1
// had become 3.1-4.9), and 4 and 8 bits up to 2^19 codes, whose pieces at the end are a longer chain (us, pieces / this: 300 rows of
// 201 codes, 8 bits, 2.44 / 2.11, 4 bits 2.47 / 2.04, but 30000 rows of 145 2.97 / 4.5 and 2.95 / 5.4; 2 bits, 16 stores of a byte, 300 x 201 2.33 / 2.57).
template <int BITS>
__global__ __launch_bounds__(256) void unpack_short_kernel(const int32_t *words, int8_t *codes, u32 n_words, u32 c, u32 wpr, FastDiv by_wpr) {
  const u32 t = blockIdx.x * 256 + threadIdx.x;
  if (t >= n_words) return;
  constexpr u32 VALS = 32 / BITS;
  const u32 r = by_wpr(t), ch = (t - r * wpr) * VALS, at = r * c + ch, n = min(VALS, c - ch);
  u32 q[8 / BITS];
  unpack_word<BITS>((u32)words[t], q);
#pragma unroll
  for (u32 j = 0; j < VALS; ++j)
    if (j < n) codes[at + j] = (int8_t)(q[j / 4] >> (8 * (j % 4)));
}

// Launches f(first row, rows) over stretches of rows that the ragged kernels can count: `fields` codes at most, padding included.
constexpr int64_t kStretch = (1ll << 31) - 4096;
template <class F> void row_chunks(int64_t rows, int wpr, int vals, int64_t fields, F f) {
  const int64_t most = std::max<int64_t>(1, fields / ((int64_t)wpr * vals));
  for (int64_t r0 = 0; r0 < rows; r0 += most) f(r0, std::min(most, rows - r0));
}

int check_common(const void *a, const void *b, int64_t rows, int c, int bits, const char *who) {
  if (!(bits == 2 || bits == 4 || bits == 8)) return varq_set_error(VARQ_ERR_INVALID, "%s: bits must be 2, 4 or 8 (got %d)", who, bits);
  if (rows < 0 || c <= 0) return varq_set_error(VARQ_ERR_INVALID, "%s: bad shape rows=%lld c=%d", who, (long long)rows, c);
  if (rows > 0 && (!a || !b)) return varq_set_error(VARQ_ERR_INVALID, "%s: null pointer", who);
  const int vals = 32 / bits;
  const int64_t wpr = (c + vals - 1) / vals;
  if (rows * wpr >= (1ll << 39)) return varq_set_error(VARQ_ERR_INVALID, "%s: too large", who);
  return 0;
}

int pack_codes(const int8_t *codes, int64_t rows, int c, int bits, int32_t *words, int64_t stretch, void *stream) {
  if (int rc = check_common(codes, words, rows, c, bits, "pack")) return rc;
  if (rows == 0) return VARQ_OK;
  hipStream_t st = (hipStream_t)stream;
  const int vals = 32 / bits;
  const int wpr = (c + vals - 1) / vals;
  const int64_t n_words = rows * wpr;
  if (c % vals == 0 && ((uintptr_t)codes % 16) == 0) {
    // whole words only: the tensor is one flat run of words; four per thread where the words are
    // 16-byte aligned too, the last 0..3 (or all of them) one per thread
    const int64_t n_quads = ((uintptr_t)words % 16) == 0 ? n_words / 4 : 0;
    const int64_t w0 = n_quads * 4;
    dim3 qgrid((unsigned)((n_quads + 255) / 256)), tgrid((unsigned)((n_words - w0 + 255) / 256));
#define VARQ_PACK(B_)                                                                                           \
  {                                                                                                             \
    if (n_quads) hipLaunchKernelGGL(pack_quad_kernel<B_>, qgrid, dim3(256), 0, st, codes, words, n_quads);      \
    if (w0 < n_words) hipLaunchKernelGGL(pack_flat_kernel<B_>, tgrid, dim3(256), 0, st, codes, words, w0, n_words); \
  }
    if (bits == 8) VARQ_PACK(8) else if (bits == 4) VARQ_PACK(4) else VARQ_PACK(2)
#undef VARQ_PACK
  } else {
    row_chunks(rows, wpr, vals, stretch, [&](int64_t r0, int64_t n) {
      const u32 nc = (u32)(n * c), nw = (u32)(n * wpr);
      auto *const kernel = bits == 8 ? pack_ragged_kernel<8> : bits == 4 ? pack_ragged_kernel<4> : pack_ragged_kernel<2>;
      hipLaunchKernelGGL(kernel, dim3((nw + 255) / 256), dim3(256), 0, st, codes + r0 * c, words + r0 * wpr, nc, nw, (u32)c, (u32)wpr, FastDiv::by(wpr));
    });
  }
  VARQ_CHECK_LAUNCH("pack");
  return VARQ_OK;
}

// by_pieces: 0 or 1 for the tests, which reach both kernels at sizes of their own (rows of 15 codes or more), or -1
int unpack_words(const int32_t *words, int64_t rows, int c, int bits, int8_t *codes, int64_t stretch, int by_pieces, void *stream) {
  if (int rc = check_common(words, codes, rows, c, bits, "unpack")) return rc;
  if (rows == 0) return VARQ_OK;
  hipStream_t st = (hipStream_t)stream;
  const int vals = 32 / bits;
  const int wpr = (c + vals - 1) / vals;
  const int64_t n_words = rows * wpr;
  if (c % vals == 0 && ((uintptr_t)codes % 16) == 0) {
    const int wpt = bits / 2;   // words per 16 bytes of codes
    const int64_t n_pieces = ((uintptr_t)words % 16) == 0 ? n_words / wpt : 0;
    const int64_t w0 = n_pieces * wpt;
    dim3 qgrid((unsigned)((n_pieces + 255) / 256)), tgrid((unsigned)((n_words - w0 + 255) / 256));
#define VARQ_UNPACK(B_)                                                                                           \
  {                                                                                                               \
    if (n_pieces) hipLaunchKernelGGL(unpack_piece_kernel<B_>, qgrid, dim3(256), 0, st, words, codes, n_pieces);   \
    if (w0 < n_words) hipLaunchKernelGGL(unpack_flat_kernel<B_>, tgrid, dim3(256), 0, st, words, codes, w0, n_words); \
  }
    if (bits == 8) VARQ_UNPACK(8) else if (bits == 4) VARQ_UNPACK(4) else VARQ_UNPACK(2)
#undef VARQ_UNPACK
  } else {
    row_chunks(rows, wpr, vals, stretch, [&](int64_t r0, int64_t n) {
      const u32 nc = (u32)(n * c), nw = (u32)(n * wpr);
      if (c < 15 || (by_pieces < 0 ? bits > 2 && (int64_t)nw * vals <= 1 << 19 : !by_pieces)) {
        auto *const kernel = bits == 8 ? unpack_short_kernel<8> : bits == 4 ? unpack_short_kernel<4> : unpack_short_kernel<2>;
        hipLaunchKernelGGL(kernel, dim3((nw + 255) / 256), dim3(256), 0, st, words + r0 * wpr, codes + r0 * c, nw, (u32)c, (u32)wpr, FastDiv::by(wpr));
        return;
      }
      auto *const kernel = bits == 8 ? unpack_ragged_kernel<8> : bits == 4 ? unpack_ragged_kernel<4> : unpack_ragged_kernel<2>;
      hipLaunchKernelGGL(kernel, dim3((nc + 4095) / 4096), dim3(256), 0, st, words + r0 * wpr, codes + r0 * c, nc, nw, (u32)c, (u32)wpr, FastDiv::by(c));
    });
  }
  VARQ_CHECK_LAUNCH("unpack");
  return VARQ_OK;
}

}  // namespace

extern "C" int varq_pack(const int8_t *codes, int64_t rows, int c, int bits, int32_t *words, void *stream) {
  return pack_codes(codes, rows, c, bits, words, kStretch, stream);
}
extern "C" int varq_unpack(const int32_t *words, int64_t rows, int c, int bits, int8_t *codes, void *stream) {
  return unpack_words(words, rows, c, bits, codes, kStretch, -1, stream);
}
extern "C" int varq_pack_stretches(const int8_t *codes, int64_t rows, int c, int bits, int32_t *words, int64_t stretch, void *stream) {
  return pack_codes(codes, rows, c, bits, words, std::min(std::max<int64_t>(stretch, 1), kStretch), stream);
}
extern "C" int varq_unpack_stretches(const int32_t *words, int64_t rows, int c, int bits, int8_t *codes, int64_t stretch, int by_pieces, void *stream) {
  return unpack_words(words, rows, c, bits, codes, std::min(std::max<int64_t>(stretch, 1), kStretch), by_pieces, stream);
}
