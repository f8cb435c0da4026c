// General two-phase quantizer: groups that span rows (the six grouping methods
// of VAR_Q/quant.py:75-95, which all reduce over the batch dim, plus any other
// reduce set).  Where workgroups can hold the rows in registers, one launch reads the input once (quant_one_kernel,
// quant_shared_kernel); otherwise:
//   phase A  group min/max (or max-abs): one partial per (chunk, group) in the
//            workspace, no atomics (tiled path below)
//   finalize fold the partials -> scale / zero-point      (VAR_Q/quant.py:112-116)
//   phase B  re-read input (L2 / Infinity-Cache resident for KV-sized tensors),
//            divide, round half-to-even, clamp, pack    (VAR_Q/quant.py:118-121,
//            VAR_Q/pack_unpack.py:177-196)
// min/max are exactly associative, so the result does not depend on the order
// in which partial results meet.  Channel counts that are not a multiple of 8 and
// rows wider than 512 channels take scalar kernels with ordered-integer atomics.
#include "dequant_steps.h"
#include "../../include/varq_testing.h"
#include <algorithm>
#include <mutex>
#include <type_traits>

#ifndef VARQ_GEN_NRO_MIN
#define VARQ_GEN_NRO_MIN 256
#endif
#ifndef VARQ_FIN_THREADS
#define VARQ_FIN_THREADS 65536
#endif
#ifndef VARQ_GEN_BLOCKS
#define VARQ_GEN_BLOCKS 2048
#endif

using namespace varq_deq;

namespace {

// Octets of earlier tokens up to which they share the step's launch (see quant_one_step_kernel): beyond, a launch of
// their own with all of a compute unit's wavefronts and registers is the better way through memory.  Symmetric /
// affine (whose quantizing workgroups' LDS leaves fewer of them resident), two launches -> one, us: 0.8 million 24.5 ->
// 18.5 / 1.0 million 24.4 -> 20.8; 2.0 20.3 -> 17.1 / 1.9 25.7 -> 27.3; 3.8 40.2 -> 42.3 / 8.2 33 -> 42; 5.1 42.5 -> 52.6.
constexpr int64_t kStepMostSym = 3ll << 20, kStepMostAsym = 3ll << 19;
constexpr int kStepOctets = 1024;   // octets of earlier tokens that a workgroup dequantizes

// Order-preserving float <-> uint map so that integer atomicMin/Max implement
// float min/max.
__device__ __forceinline__ u32 enc_ord(float f) {
  u32 u = f2u(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float dec_ord(u32 e) {
  return u2f((e & 0x80000000u) ? (e & 0x7fffffffu) : ~e);
}

// Where the scale of group g goes when it is written once per token that it serves (and the zero-point like it): elements
// (g / gi) go + (g % gi) ge + off + i + o * s_out, i < r_in, o < r_out.
struct Spread {
  int on;
  FastDiv by_gi, by_in;
  u32 gi, r_in, reps;        // reps = r_in * r_out
  int64_t go, ge, off, s_out;
  float *scale, *zp, *scale1, *zp1;   // where they go once each as well, in the order of the groups (or null)
};

struct GenParams {
  const void *x;
  u32 *ws;       // [n_groups] encoded max (or max-abs), behind them [n_groups] encoded min (asym only)
  float *scale, *zp;
  int32_t *words;
  int8_t *codes;
  int64_t n1, n2;          // the last two leading dims
  int64_t gs0, gs1, gs2;   // group-id stride of each leading dim (0 = reduced)
  int64_t rows;            // n0*n1*n2
  int64_t n_groups;
  int c, c8;               // channels, octets per row
  int keepc;               // last dim kept (one group per channel) or reduced
  int bits, qmin, qmax, wpr; // wpr = words per row
  int asym;
  float eps;
  // Output rows (codes / words) may land in a larger buffer: input row r goes to output row
  // r + (r / out_inner) * out_delta + out_off -- a step [B,H,n,c] into tokens len.. of a cache
  // [B,H,cap,..] is (n, cap - n, len), a step [B,n,H,c] into [B,cap,H,..] is (n*H, (cap - n)*H, len*H).
  int out_mapped;
  int64_t out_inner, out_delta, out_off;
  FastDiv by_inner;
  Spread spread;
  // a second tensor of the same shape in the same launches (blockIdx.y == 1): its input,
  // its outputs and the distance (in 4-byte words) to its part of the workspace
  const void *x1;
  float *scale1, *zp1;
  int32_t *words1;
  int8_t *codes1;
  int64_t ws1;
};

// the tensor a workgroup of the tiled kernels works on
__device__ __forceinline__ bool take_second(GenParams &p) {
  if (blockIdx.y == 0) return false;
  p.x = p.x1; p.scale = p.scale1; p.zp = p.zp1; p.words = p.words1; p.codes = p.codes1;
  p.spread.scale = p.spread.scale1; p.spread.zp = p.spread.zp1;
  return true;
}

// The parameters of a workgroup's 2^shift groups, in LDS, to all their places, by all `NT` threads; group_of(t): the number of a group (or less
// than 0: no such group).  Adjacent threads write adjacent places: those of a token, or of a row of a table, unless the groups' own are adjacent.
// (G_TOKEN in layout BLHc, two tensors of [64,324,16,64] in three launches, 1024 places a group: 65 us with the groups first, in as many workgroups as
// the fold takes; so 50.)
template <bool ASYM, int NT, class F>
__device__ __forceinline__ void spread_parameters(const GenParams &p, int shift, const float *par_s, const float *par_z, F &&group_of) {
  auto put = [&](int t, int64_t g, u32 rep) __attribute__((always_inline)) {
    const u32 o = p.spread.by_in(rep), a = p.spread.by_gi((u32)g);
    const int64_t at = a * p.spread.go + (int64_t)((u32)g - a * p.spread.gi) * p.spread.ge + p.spread.off + (rep - o * p.spread.r_in) + o * p.spread.s_out;
    p.scale[at] = par_s[t];
    if (ASYM) p.zp[at] = par_z[t];
  };
  if ((p.spread.gi > 1 ? p.spread.ge : p.spread.go) == 1) {
    for (u32 i = threadIdx.x; i < p.spread.reps << shift; i += NT) {
      const int t = i & ((1u << shift) - 1);
      const int64_t g = group_of(t);
      if (g >= 0) put(t, g, i >> shift);
    }
  } else {   // (a wavefront per group, or all threads by as many groups as there are)
    const int lanes = max(6, __builtin_ctz((unsigned)NT) - shift);
    for (int t = threadIdx.x >> lanes; t < 1 << shift; t += NT >> lanes) {
      const int64_t g = group_of(t);
      if (g < 0) continue;
      for (u32 rep = threadIdx.x & ((1u << lanes) - 1); rep < p.spread.reps; rep += 1u << lanes) put(t, g, rep);
    }
  }
}

__device__ __forceinline__ int64_t out_row(const GenParams &p, int64_t row) {
  return p.out_mapped ? row + (row / p.out_inner) * p.out_delta + p.out_off : row;
}
// (rows of the tiled kernels fit 31 bits)
__device__ __forceinline__ int64_t out_row32(const GenParams &p, int64_t row) {
  return p.out_mapped ? row + (int64_t)p.by_inner((u32)row) * p.out_delta + p.out_off : row;
}

__global__ void init_ws_kernel(u32 *ws_max, u32 *ws_min, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    ws_max[i] = 0u;
    if (ws_min) ws_min[i] = 0xffffffffu;
  }
}

__device__ __forceinline__ void row_to_idx(const GenParams &p, int64_t r, int64_t &i0, int64_t &i1, int64_t &i2) {
  i2 = r % p.n2;
  int64_t t = r / p.n2;
  i1 = t % p.n1;
  i0 = t / p.n1;
}

// ---- fast path (c % 8 == 0, at most 512 channels): tiled, atomic-free -------------
// The leading dims are brought to a canonical form on the host (Plan): a linear
// index `ko` over kept outer dims, a linear index `ro` over reduced outer dims,
// and along contiguous rows either a kept extent Q (d2 kept) or a reduced extent
// RI (d2 reduced):
//     row   = ko*ko_rs + ro*ro_rs + (q | ri)
//     group = ko*ko_gs + q*q_gs  (+ channel when the channel dim is kept)
// A workgroup is 256 threads = R row lanes x c8p column lanes (8 channels each) and
// owns one (ko, tile of Q, chunk z of the reduced steps).  Every thread sees a
// single group (per channel) for its whole life: no group lookups and no integer
// divisions in the loop.  Phase A leaves one partial min/max per (z, group) in the
// workspace (plain stores, each written exactly once), the finalize kernel folds
// the Z partials, phase B walks the same decomposition with the group's scale,
// reciprocal and zero-point in registers.
struct Plan {
  int64_t ko_rs, ro_rs, ko_gs, q_gs;
  int nko, nro, Q, RI;
  int lanesQ, sub, tilesQ;     // row lanes spent on q; positions folded into the rest; tiles over Q
  int fold_ro;                 // 1: the spare row lanes fold consecutive ro (RI == 1), 0: consecutive rows of RI
  int T;                       // steps per ro along RI (inner reduced), 1 when d2 is kept
  int steps, Z, steps_per_chunk;
  int R, c8, c8p, shift;
};
// The arguments of the two tiled kernels fill seven cache lines: eight bytes more take the three launches 0.2 us longer ([32,30,680,64] bf16,
// 8 bits 63.6 -> 64.0 us, 4 bits affine 60.6 -> 61.0).
static_assert(sizeof(GenParams) + sizeof(Plan) + 2 * sizeof(void *) <= 448, "kernel arguments");

// decode the workgroup and lane; returns false for an idle lane
struct Lane {
  int ko, q, f, col, z;
  bool live;
};
__device__ __forceinline__ Lane decode(const Plan &pl) {
  Lane l;
  const int bid = blockIdx.x;
  l.z = bid % pl.Z;
  const int kb = bid / pl.Z;
  const int tq = kb % pl.tilesQ;
  l.ko = kb / pl.tilesQ;
  l.col = threadIdx.x & (pl.c8p - 1);
  const int rowlane = threadIdx.x >> pl.shift;
  const int lq = rowlane % pl.lanesQ;
  l.f = rowlane / pl.lanesQ;
  l.q = tq * pl.lanesQ + lq;
  l.live = l.col < pl.c8 && l.f < pl.sub && l.q < pl.Q;
  return l;
}

// Calls body(row, v) for every row of this thread, in step order, with the row's 8 values of
// this lane's octet.
template <int DT, typename F>
__device__ __forceinline__ void for_rows(const GenParams &p, const Plan &pl, const Lane &l, F body) {
  // (scalars: the rows of a step differ between the lanes by what lane_row holds)
  const int s0 = __builtin_amdgcn_readfirstlane(l.z * pl.steps_per_chunk), s1 = min(s0 + pl.steps_per_chunk, pl.steps);
  const int64_t lane_row = (int64_t)l.ko * pl.ko_rs + l.q + (pl.fold_ro ? l.f * pl.ro_rs : l.f);
  const char *const lane_x = reinterpret_cast<const char *>(p.x) + (lane_row * p.c + l.col * 8) * In8<DT>::kBytes;
  const int64_t row_bytes = (int64_t)p.c * In8<DT>::kBytes;
  auto take = [&](int64_t step_row) __attribute__((always_inline)) {
    float v[8];
    In8<DT>::load(lane_x + step_row * row_bytes, 0, v);
    body((u32)lane_row + (u32)step_row, v);
  };
  // (one load in flight per lane: issuing two steps' loads before either is used, or the next
  // row's load ahead of the current row's arithmetic, was measured 5-15 % slower on both phases)
  if (pl.fold_ro) {
    // d2 kept: a step is `sub` consecutive reduced positions
    for (int s = s0; s < s1; ++s)
      if (s * pl.sub + l.f < pl.nro) take((int64_t)s * pl.sub * pl.ro_rs);
  } else {
    // d2 reduced: a step is `sub` (= R) consecutive rows of one ro
    int ro = s0 / pl.T, t = s0 - ro * pl.T;
    for (int s = s0; s < s1; ++s) {
      if (t * pl.sub + l.f < pl.RI) take((int64_t)ro * pl.ro_rs + t * pl.sub);
      if (++t == pl.T) { t = 0; ++ro; }
    }
  }
}

template <int DT, bool ASYM, bool KEEPC>
__global__ __launch_bounds__(256) void minmax_tiled_kernel(GenParams p, Plan pl, float *part_max, float *part_min) {
  constexpr int NV = KEEPC ? 8 : 1;
  __shared__ float lds_mx[256 * NV];
  __shared__ float lds_mn[ASYM ? 256 * NV : 1];
  if (take_second(p)) { part_max += p.ws1; part_min += p.ws1; }
  const Lane l = decode(pl);
  float mx[NV], mn[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) { mx[j] = ASYM ? -INFINITY : 0.f; mn[j] = INFINITY; }
  if (l.live) {
    for_rows<DT>(p, pl, l, [&](u32, const float (&v)[8]) {
      if (KEEPC) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (ASYM) { mx[j] = fmaxf(mx[j], v[j]); mn[j] = fminf(mn[j], v[j]); }
          else mx[j] = fmaxf(mx[j], fabsf(v[j]));
        }
      } else if (ASYM) {
        mx[0] = fmaxf(mx[0], fmaxf(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])), fmaxf(fmaxf(v[4], v[5]), fmaxf(v[6], v[7]))));
        mn[0] = fminf(mn[0], fminf(fminf(fminf(v[0], v[1]), fminf(v[2], v[3])), fminf(fminf(v[4], v[5]), fminf(v[6], v[7]))));
      } else {
        mx[0] = fmaxf(mx[0], fmaxf(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))),
                                   fmaxf(fmaxf(fabsf(v[4]), fabsf(v[5])), fmaxf(fabsf(v[6]), fabsf(v[7])))));
      }
    });
  }
  if (!KEEPC) {
    // fold the column lanes of a row (c8p <= 64: a row never spans wavefronts; idle lanes hold the identity)
    for (int off = 1; off < pl.c8p; off <<= 1) {
      mx[0] = fmaxf(mx[0], __shfl_xor(mx[0], off, 64));
      if (ASYM) mn[0] = fminf(mn[0], __shfl_xor(mn[0], off, 64));
    }
  }
  // fold the `sub` row lanes that share q (lane index = (f*lanesQ + lq)*c8p + col, so the
  // positions f of one (q, col) lie `stride` lanes apart): inside a wavefront by lane exchanges
  // when the stride is a power of two below 64, the rest -- at most one value per wavefront
  // then -- through LDS.  (Idle lanes hold the identity of max / min.)
  if (pl.sub > 1) {
    const int stride = pl.lanesQ * pl.c8p;
    int fstep = 1;                       // distance in f between the values still to fold
    if (stride < 64 && (stride & (stride - 1)) == 0) {
      for (int off = stride; off < 64; off <<= 1) {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          mx[j] = fmaxf(mx[j], __shfl_xor(mx[j], off, 64));
          if (ASYM) mn[j] = fminf(mn[j], __shfl_xor(mn[j], off, 64));
        }
      }
      fstep = 64 / stride;
    }
    if (fstep < pl.sub) {
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        lds_mx[j * 256 + threadIdx.x] = mx[j];
        if (ASYM) lds_mn[j * 256 + threadIdx.x] = mn[j];
      }
      __syncthreads();
      if (l.f == 0) {
        for (int f = fstep; f < pl.sub; f += fstep)
#pragma unroll
          for (int j = 0; j < NV; ++j) {
            mx[j] = fmaxf(mx[j], lds_mx[j * 256 + threadIdx.x + f * stride]);
            if (ASYM) mn[j] = fminf(mn[j], lds_mn[j * 256 + threadIdx.x + f * stride]);
          }
      }
    }
  }
  if (l.f != 0 || l.q >= pl.Q || l.col >= pl.c8 || (!KEEPC && l.col != 0)) return;
  const int64_t g = (int64_t)l.ko * pl.ko_gs + (int64_t)l.q * pl.q_gs + (KEEPC ? l.col * 8 : 0);
  float *dmx = part_max + (int64_t)l.z * p.n_groups + g;
  float *dmn = part_min + (int64_t)l.z * p.n_groups + g;
  if (KEEPC) {
    reinterpret_cast<float4 *>(dmx)[0] = make_float4(mx[0], mx[1], mx[2], mx[3]);
    reinterpret_cast<float4 *>(dmx)[1] = make_float4(mx[4 % NV], mx[5 % NV], mx[6 % NV], mx[7 % NV]);
    if (ASYM) {
      reinterpret_cast<float4 *>(dmn)[0] = make_float4(mn[0], mn[1], mn[2], mn[3]);
      reinterpret_cast<float4 *>(dmn)[1] = make_float4(mn[4 % NV], mn[5 % NV], mn[6 % NV], mn[7 % NV]);
    }
  } else {
    dmx[0] = mx[0];
    if (ASYM) dmn[0] = mn[0];
  }
}

// partials -> scale, zero-point, reciprocal and the flag of the exact-quotient shortcut.
// 256 threads = ZL z-lanes x 256/ZL adjacent groups; the z-lanes of a group meet in LDS.
template <bool ASYM>
__global__ __launch_bounds__(256) void finalize_tiled_kernel(GenParams p, int Z, int ZL, const float *part_max,
                                                             const float *part_min, float *rinv, u32 *plain) {
  __shared__ float lds_mx[256];
  __shared__ float lds_mn[256];
  if (take_second(p)) { part_max += p.ws1; part_min += p.ws1; rinv += p.ws1; plain += p.ws1; }
  const int gpb = 256 / ZL;                       // groups per block
  const int gl = threadIdx.x % gpb, zl = threadIdx.x / gpb;
  const int64_t g = (int64_t)blockIdx.x * gpb + gl;
  float mx = ASYM ? -INFINITY : 0.f, mn = INFINITY;
  if (g < p.n_groups) {
    for (int z = zl; z < Z; z += ZL) {
      mx = fmaxf(mx, part_max[(int64_t)z * p.n_groups + g]);
      if (ASYM) mn = fminf(mn, part_min[(int64_t)z * p.n_groups + g]);
    }
  }
  lds_mx[threadIdx.x] = mx;
  lds_mn[threadIdx.x] = mn;
  __syncthreads();
  for (int h = ZL >> 1; h > 0; h >>= 1) {
    if (zl < h) {
      lds_mx[threadIdx.x] = fmaxf(lds_mx[threadIdx.x], lds_mx[threadIdx.x + h * gpb]);
      lds_mn[threadIdx.x] = fminf(lds_mn[threadIdx.x], lds_mn[threadIdx.x + h * gpb]);
    }
    __syncthreads();
  }
  const bool spread = p.spread.on;
  if (zl == 0 && g < p.n_groups) {
    mx = lds_mx[threadIdx.x];
    mn = lds_mn[threadIdx.x];
    float s, z = 0.f;
    if (ASYM) {
      s = fmaxf((mx - mn) / (float)((1 << p.bits) - 1), p.eps);
      z = (float)p.qmin - rintf(mn / s);
      (spread ? p.spread.zp : p.zp)[g] = z;
    } else {
      s = fmaxf(mx / (float)p.qmax, p.eps);
    }
    (spread ? p.spread.scale : p.scale)[g] = s;
    rinv[g] = 1.0f / s;
    // whether exact_quotient holds (about x/s = -zp: the values of a group may lie far from 0 in a narrow range)
    plain[g] = (s > 0x1p-96f && s < 0x1p96f && (f2u(s) & 0x7fffffu) != 0x7fffffu && fabsf(z) <= 0x1p120f) ? 1u : 0u;
    lds_mx[threadIdx.x] = s;
    lds_mn[threadIdx.x] = z;
  }
  if (!spread) return;
  __syncthreads();
  spread_parameters<ASYM, 256>(p, __builtin_ctz((u32)gpb), lds_mx, lds_mn,
                               [&](int t) { const int64_t of = (int64_t)blockIdx.x * gpb + t; return of < p.n_groups ? of : -1; });
}

// x/s == RN(q0 + (x - q0*s)*r) with q0 = RN(x*r), r = RN(1/s), for every finite x unless the significand of s is all ones, the
// residual can underflow or the quotient comes near the largest float
__device__ __forceinline__ float exact_quotient(float x, float s, float r) {
  const float q0 = x * r;
  return __builtin_fmaf(__builtin_fmaf(-q0, s, x), r, q0);
}
// The codes of an octet by division
template <int NV>
__device__ __forceinline__ void divided(const float (&v)[8], const float (&s)[NV], const float (&z)[NV], float qmin, float qmax, int (&q)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) q[j] = (int)__builtin_amdgcn_fmed3f(rintf(v[j] / s[j % NV]) + z[j % NV], qmin, qmax);
}
// Quantizes and stores one octet (column `col`) of row `row`: s, z the scale and the zero-point of the octet's groups (one per channel or one).
// also(codes): what else the caller wants from them.
__device__ __forceinline__ void store_codes(const GenParams &p, int64_t row, int col, const int (&q)[8], u32 mask) {
  const int64_t orow = out_row32(p, row);
  if (p.codes || p.bits == 8) {
    const u32 lo = (q[0] & 0xff) | ((q[1] & 0xff) << 8) | ((q[2] & 0xff) << 16) | ((u32)q[3] << 24);
    const u32 hi = (q[4] & 0xff) | ((q[5] & 0xff) << 8) | ((q[6] & 0xff) << 16) | ((u32)q[7] << 24);
    if (p.codes) *reinterpret_cast<uint2 *>(p.codes + (orow * p.c8 + col) * 8) = make_uint2(lo, hi);
    if (p.words && p.bits == 8) *reinterpret_cast<uint2 *>(p.words + orow * p.wpr + col * 2) = make_uint2(lo, hi);
  }
  if (p.words && p.bits != 8) {
    u32 w = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) w |= ((u32)q[j] & mask) << (j * p.bits);
    if (p.bits == 4) {
      p.words[orow * p.wpr + col] = (int32_t)w;
    } else {  // 2 bits: 16 codes per word = two adjacent octets (c % 16 == 0 on this path)
      const u32 other = __shfl_xor(w, 1, 64);
      if ((col & 1) == 0) p.words[orow * p.wpr + (col >> 1)] = (int32_t)(w | (other << 16));
    }
  }
}
template <int NV, class F>
__device__ __forceinline__ void store_octet(const GenParams &p, int64_t row, int col, const float (&v)[8], const float (&s)[NV],
                                            const float (&z)[NV], F &&also) {
  int q[8];
  divided<NV>(v, s, z, (float)p.qmin, (float)p.qmax, q);
  also(q);
  store_codes(p, row, col, q, (1u << p.bits) - 1u);
}

// The groups of one octet (one per channel or one) where all scales allow exact_quotient and the zero-points are
// below 2^21: clamp(rint(t) + z, qmin, qmax) = rint(clamp(t, qmin - z, qmax - z)) + z, adding 1.5 * 2^23 rounds to nearest-even and leaves
// the integer in the low bits, four of them are a dword of bytes, and the zero-points are added to its bytes at once.  About eight
// instructions per element with the conversion; store_octet takes twelve, and the quantizing kernels are bound by their number as
// much as by the bytes.
template <int NV, bool ASYM> struct FastOctet {
  float s[NV], r[NV], lo[NV], span, hi;
  u32 zw[ASYM ? 2 : 1];   // zero-points, one byte per channel
  __device__ __forceinline__ FastOctet(const GenParams &p, const float (&s_)[NV], const float (&r_)[NV], const float (&z)[NV]) {
    span = (float)(p.qmax - p.qmin); hi = (float)p.qmax;
#pragma unroll
    for (int j = 0; j < NV; ++j) { s[j] = s_[j]; r[j] = r_[j]; lo[j] = ASYM ? (float)p.qmin - z[j] : (float)p.qmin; }
    if constexpr (ASYM) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        zw[h] = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) zw[h] |= ((u32)(int)z[(4 * h + j) % NV] & 0xffu) << (8 * j);
      }
    }
  }
  // number(j): the code of v[j] less its zero-point, in the low bits of a float of 1.5 * 2^23
  __device__ __forceinline__ float number(float x, int j) const {
    const int n = j % NV;
    return __builtin_amdgcn_fmed3f(exact_quotient(x, s[n], r[n]), lo[n], ASYM ? lo[n] + span : hi) + 12582912.f;
  }
  __device__ __forceinline__ u32 bytes(const float (&u)[8], int h) const {
    const u32 a = __builtin_amdgcn_perm(f2u(u[4 * h + 1]), f2u(u[4 * h]), 0x0c0c0400u), b = __builtin_amdgcn_perm(f2u(u[4 * h + 3]), f2u(u[4 * h + 2]), 0x0c0c0400u);
    const u32 w = __builtin_amdgcn_perm(b, a, 0x05040100u);
    if constexpr (ASYM) return ((w & 0x7f7f7f7fu) + (zw[h] & 0x7f7f7f7fu)) ^ ((w ^ zw[h]) & 0x80808080u);
    else return w;
  }
  // Quantizes and stores an octet; also(u): what else the caller wants from its numbers.
  template <class F> __device__ __forceinline__ void store(const GenParams &p, int64_t orow, int col, const float (&v)[8], F &&also) const {
    float u[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) u[j] = number(v[j], j);
    also(u);
    const u32 lo8 = bytes(u, 0), hi8 = bytes(u, 1);
    if (p.codes) *reinterpret_cast<uint2 *>(p.codes + (orow * p.c8 + col) * 8) = make_uint2(lo8, hi8);
    if (!p.words) return;
    if (p.bits == 8) {
      *reinterpret_cast<uint2 *>(p.words + orow * p.wpr + col * 2) = make_uint2(lo8, hi8);
    } else if (p.bits == 4) {
      const u32 a = lo8 & 0x0f0f0f0fu, b = hi8 & 0x0f0f0f0fu;
      p.words[orow * p.wpr + col] = (int32_t)__builtin_amdgcn_perm(b | b >> 4, a | a >> 4, 0x06040200u);
    } else {  // 2 bits: 16 codes per word = two adjacent octets (c % 16 == 0 on this path), the partner lane's in the upper half
      auto four = [](u32 w) { w &= 0x03030303u; w |= w >> 6; return (w & 0xfu) | (w >> 12 & 0xf0u); };
      const u32 w = four(lo8) | four(hi8) << 8;
      const u32 other = (u32)__builtin_amdgcn_update_dpp(0, (int)w, 0xB1, 0xf, 0xf, false);
      if ((col & 1) == 0) p.words[orow * p.wpr + (col >> 1)] = (int32_t)(w | (other << 16));
    }
  }
};

template <int DT, bool ASYM, bool KEEPC>
__global__ __launch_bounds__(256) void quant_tiled_kernel(GenParams p, Plan pl, const float *rinv, const u32 *plain) {
  constexpr int NV = KEEPC ? 8 : 1;
  if (take_second(p)) { rinv += p.ws1; plain += p.ws1; }
  const Lane l = decode(pl);
  if (!l.live) return;   // (only the 2-bit path exchanges between lanes, and there c8 is even: partners are live together)
  const int64_t g = (int64_t)l.ko * pl.ko_gs + (int64_t)l.q * pl.q_gs + (KEEPC ? l.col * 8 : 0);
  float s[NV], r[NV], z[NV] = {};
  bool fast = true;
  if constexpr (KEEPC) {
    // the lane's eight groups are adjacent and start at a multiple of 8: 16-byte loads (the
    // workspace and the outputs are 16-byte aligned; checked on the host)
    auto ld8 = [&](const float *src, float (&dst)[NV]) {
      const float4 a = reinterpret_cast<const float4 *>(src + g)[0], b = reinterpret_cast<const float4 *>(src + g)[1];
      dst[0] = a.x; dst[1] = a.y; dst[2] = a.z; dst[3] = a.w; dst[4 % NV] = b.x; dst[5 % NV] = b.y; dst[6 % NV] = b.z; dst[7 % NV] = b.w;
    };
    ld8(p.scale, s);
    ld8(rinv, r);
    if (ASYM) ld8(p.zp, z);
    const uint4 pa = reinterpret_cast<const uint4 *>(plain + g)[0], pb = reinterpret_cast<const uint4 *>(plain + g)[1];
    fast = (pa.x & pa.y & pa.z & pa.w & pb.x & pb.y & pb.z & pb.w) != 0u;
  } else {
    s[0] = p.scale[g];
    r[0] = rinv[g];
    if (ASYM) z[0] = p.zp[g];
    fast = plain[g] != 0u;
  }
  // (The longer arithmetic of the two: with FastOctet's, the chunks run ahead of what the Infinity Cache serves.  us for the three launches, this /
  // that: a scale per (head, channel) of [32,30,680,64] 8 bits 51.0 / 53.0, fp32 78.4 / 79.8, 4 bits affine 49.0 / 51.1, of [2,16,10521,128] 52.5 / 54.5,
  // [64,256,16,64] 26.5 / 27.1; one scale 50.8 / 52.0; but one per (token, head) 48.8 / 47.8.)
  const float qmin = (float)p.qmin, qmax = (float)p.qmax;
  const u32 mask = (1u << p.bits) - 1u;
  for_rows<DT>(p, pl, l, [&](u32 row, const float (&v)[8]) {
    int q[8];
    if (fast) {
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = (int)__builtin_amdgcn_fmed3f(rintf(exact_quotient(v[j], s[j % NV], r[j % NV])) + z[j % NV], qmin, qmax);
    } else {
      divided<NV>(v, s, z, qmin, qmax, q);
    }
    store_codes(p, row, l.col, q, mask);
  });
}

// ---- one launch: a workgroup holds all rows of its groups -----------------------------------------
// Where the rows of a group fit the registers of a workgroup (16 rows of an octet per thread, 8 in fp32) the
// three launches become one, and the input is read once: load, fold, derive the parameters, quantize what
// the registers hold.  The steps of a schedule are bound by the number of their launches and by latency, not
// by bytes.  K and V of a step, 8-bit, one scale per channel and head, fp16 [64,n,16,64] / bf16 [2,16,n,128],
// three launches -> one: n = 1 12.7 -> 4.4 us / 9.9 -> 4.7, n = 16 11.8 -> 8.6 / 9.9 -> 4.6, n = 64 22.7 ->
// 14.7, n = 400 14.3 -> 9.9, n = 1024 22.6 -> 16.5.
// A workgroup owns, for one ko, 2^lq_shift kept inner indices x c8s column lanes; thread
// ((lq * sub + f) * c8s + col) takes the reduced rows f, f + sub, ... of its q.  A row is straight-line code, once per held row and pass: what it
// costs are its instructions, issued and fetched.  With two divisions of 64-bit rows, the conversion to integers and
// the division's own path in every row, 45 KB for 16 rows, and that kernel for four rows as well, the launches of fp16 [64,n,16,64]
// took 13.1 us (n = 9), 15.3 (25), 13.1 (36) and 20.6 (64); now 6.8, 10.2, 11.8 and 18.6; with the dequantized cache, [8,n,30,64] to
// fp32, 11.4 -> 7.8 (n = 25), 12.4 -> 10.3 (64), 21.5 -> 19.3 (256).  With the channel dim kept
// the columns are cut into slices of c8s octets, one workgroup each, until there are workgroups enough: the
// steps of one batch have few groups, and narrow slices (64, 32, then 16 bytes of a row, whose cache lines
// the slices of one XCD share) still read faster than few workgroups do.
// The extremes over the lanes whose numbers differ in the bits from `from` up to below `to` (powers of two; all lanes are active), in every one of them.  From
// rows of 16 lanes up by rotations inside the row and swaps of rows, a few cycles each where an exchange through LDS waits for some
// hundred.  The small launches are one chain of such waits: with this fold, the wavefronts' extremes requested together and no divisions, us: ten steps with the
// dequantized cache, [8,n,30,64] to fp32, 178 -> 173; with attention, [64,n,16,64] 375 -> 370.  In quant_shared_kernel,
// whose registers are full, the same fold costs (K of [32,30,680,64] 63.1 -> 64.1, unpacking included), so it keeps the exchange.
template <bool ASYM, int NV> __device__ __forceinline__ void fold_lanes(float (&mx)[NV], float (&mn)[NV], int from, int to) {
  auto with = [&](auto &&other) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      mx[j] = fmaxf(mx[j], other(mx[j]));
      if (ASYM) mn[j] = fminf(mn[j], other(mn[j]));
    }
  };
  if (to < 16) {
    for (int off = from; off < to; off <<= 1) with([&](float v) __attribute__((always_inline)) { return __shfl_xor(v, off, 64); });
    return;
  }
  if (from <= 1) with([](float v) __attribute__((always_inline)) { return dpp_f<0x121>(v); });   // row_ror:1
  if (from <= 2) with([](float v) __attribute__((always_inline)) { return dpp_f<0x122>(v); });
  if (from <= 4) with([](float v) __attribute__((always_inline)) { return dpp_f<0x124>(v); });
  if (from <= 8) with([](float v) __attribute__((always_inline)) { return dpp_f<0x128>(v); });
  // (of a value swapped with itself one half is the other rows' and the other half the lane's own)
  auto swapped = [&](auto &&swap) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const auto a = swap(f2u(mx[j]));
      mx[j] = fmaxf(u2f(a[0]), u2f(a[1]));
      if (ASYM) { const auto b = swap(f2u(mn[j])); mn[j] = fminf(u2f(b[0]), u2f(b[1])); }
    }
  };
  if (from <= 16 && to > 16) swapped([](u32 v) __attribute__((always_inline)) { return __builtin_amdgcn_permlane16_swap(v, v, false, false); });
  if (from <= 32 && to > 32) swapped([](u32 v) __attribute__((always_inline)) { return __builtin_amdgcn_permlane32_swap(v, v, false, false); });
}

struct OnePlan {
  int64_t ko_rs, ro_rs, ko_gs, q_gs;
  int nko, Q, RR, RI;           // kept outer, kept inner; reduced rows, of which RI are contiguous
  FastDiv by_RI;
  int c8s_shift, sub_shift, lq_shift;
  int slices, tilesQ, steps;
  int blocks;                   // nko * tilesQ
  FastDiv by_slices, by_tilesQ;
};

// also(row, col, codes less their zero-points, scales): what else is made of an octet once it is quantized
template <int DT, bool ASYM, bool KEEPC, int NT, int NI, class F>
__device__ __forceinline__ void quant_one_block(const GenParams &p, const OnePlan &pl, F &&also) {
  constexpr int NV = KEEPC ? 8 : 1, MAXG = 2048;
  __shared__ float lds_mx[MAXG];
  __shared__ float lds_mn[ASYM ? MAXG : 1];
  __shared__ float par_s[MAXG], par_r[MAXG];
  __shared__ float par_z[ASYM ? MAXG : 1];
  // the slices of a block on one XCD (ids congruent mod 8 share an L2): they share the rows' cache lines
  const int bid = blockIdx.x, of_eight = (int)pl.by_slices((u32)bid >> 3), slice = (bid >> 3) - of_eight * pl.slices, blk = of_eight * 8 + (bid & 7);
  if (blk >= pl.blocks) return;
  const int ko = (int)pl.by_tilesQ((u32)blk), tq = blk - ko * pl.tilesQ;
  const int tid = threadIdx.x, c8s = 1 << pl.c8s_shift, sub = 1 << pl.sub_shift;
  const int lcol = tid & (c8s - 1), col = slice * c8s + lcol, f = (tid >> pl.c8s_shift) & (sub - 1), lq = tid >> (pl.c8s_shift + pl.sub_shift);
  const int q = (tq << pl.lq_shift) + lq;
  const bool live = col < p.c8 && q < pl.Q && lq < (1 << pl.lq_shift);
  // (the tensors are at most 128 MiB, so rows and byte offsets fit 32 bits)
  const u32 row0 = (u32)ko * (u32)pl.ko_rs + (live ? q : 0);
  auto row_of = [&](int j) {
    const u32 o = pl.by_RI((u32)j);
    return row0 + o * (u32)pl.ro_rs + ((u32)j - o * (u32)pl.RI);
  };
  auto octet_at = [&](u32 row) { return reinterpret_cast<const Raw8<DT> *>(reinterpret_cast<const char *>(p.x) + (row * (u32)p.c + col * 8) * (u32)In8<DT>::kBytes); };

  Raw8<DT> raw[NI];
#pragma unroll
  for (int s = 0; s < NI; ++s) {
    const int j = (s << pl.sub_shift) + f;
    if (s < pl.steps && live && j < pl.RR)
      raw[s] = *octet_at(row_of(j));
  }
  float mx[NV], mn[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) { mx[j] = ASYM ? -INFINITY : 0.f; mn[j] = INFINITY; }
#pragma unroll
  for (int s = 0; s < NI; ++s) {
    if (s >= pl.steps || !live || (s << pl.sub_shift) + f >= pl.RR) continue;
    float v[8];
    raw[s].widen(v);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (ASYM) { mx[j % NV] = fmaxf(mx[j % NV], v[j]); mn[j % NV] = fminf(mn[j % NV], v[j]); }
      else mx[j % NV] = fmaxf(mx[j % NV], fabsf(v[j]));
    }
  }
  // fold over f (and, with the channel dim reduced, over the columns), inside the wavefront first;
  // what is left is one value per wavefront and column, or per q where a q has less than a wavefront
  const int q_lanes = sub << pl.c8s_shift;         // threads of a q
  fold_lanes<ASYM>(mx, mn, KEEPC ? c8s : 1, q_lanes);
  const int gcols = KEEPC ? c8s * 8 : 1;           // groups of a q in this workgroup
  const int parts = q_lanes > 64 ? q_lanes >> 6 : 1, lane_in_part = q_lanes > 64 ? tid & 63 : tid & (q_lanes - 1);
  const int part = q_lanes > 64 ? tid >> 6 : tid >> (pl.sub_shift + pl.c8s_shift);      // = lq * parts + wavefront of the q
  if (lane_in_part < (KEEPC ? c8s : 1)) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      lds_mx[part * gcols + lcol * NV + j] = mx[j];
      if (ASYM) lds_mn[part * gcols + lcol * NV + j] = mn[j];
    }
  }
  __syncthreads();
  // one thread per group
  const int n_par = gcols << pl.lq_shift;
  for (int t = tid; t < n_par; t += NT) {
    const int tl = KEEPC ? t >> (pl.c8s_shift + 3) : t, g8 = t - tl * gcols, tqi = (tq << pl.lq_shift) + tl;
    float m = ASYM ? -INFINITY : 0.f, n = INFINITY;
    // (all of them requested at once, the last one again where they are fewer)
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
      const int at = (tl * parts + min(w, parts - 1)) * gcols + g8;
      m = fmaxf(m, lds_mx[at]);
      if (ASYM) n = fminf(n, lds_mn[at]);
    }
    const bool mine = tqi < pl.Q && (!KEEPC || slice * c8s * 8 + g8 < p.c);
    float s, zp = 0.f;
    if (ASYM) {
      s = fmaxf((m - n) / (float)((1 << p.bits) - 1), p.eps);
      zp = (float)p.qmin - rintf(n / s);
      par_z[t] = zp;
    } else {
      s = fmaxf(m / (float)p.qmax, p.eps);
    }
    par_s[t] = s;
    // (exact_quotient, where FastOctet's rounding holds the zero-point; 0: this group takes the division)
    par_r[t] = (s > 0x1p-96f && s < 0x1p96f && (f2u(s) & 0x7fffffu) != 0x7fffffu && fabsf(zp) <= 0x1p21f) ? 1.0f / s : 0.f;
    float *const once = KEEPC || !p.spread.on ? p.scale : p.spread.scale;
    if (mine && once) {
      const int64_t g = (int64_t)ko * pl.ko_gs + (int64_t)tqi * pl.q_gs + (KEEPC ? slice * c8s * 8 + g8 : 0);
      once[g] = s;
      if (ASYM) (KEEPC || !p.spread.on ? p.zp : p.spread.zp)[g] = zp;
    }
  }
  __syncthreads();
  if constexpr (!KEEPC) {
    auto group_of = [&](int t) { const int q = (tq << pl.lq_shift) + t; return q < pl.Q ? (int64_t)ko * pl.ko_gs + (int64_t)q * pl.q_gs : -1; };
    if (p.spread.on) spread_parameters<ASYM, NT>(p, pl.lq_shift, par_s, par_z, group_of);
  }
  if (!live) return;   // (2-bit words take two adjacent columns, which are live together: c is a multiple of 16 there)
  const int t0 = lq * gcols + lcol * (KEEPC ? 8 : 0);
  float s[NV], r[NV], z[NV] = {};
  bool plain = true;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    s[j] = par_s[t0 + j];
    r[j] = par_r[t0 + j];
    if (ASYM) z[j] = par_z[t0 + j];
    plain = plain && r[j] != 0.f;
  }
  if (__any(!plain)) {   // (rare, and once in the code: the rows are read again)
    for (int j = f; j < pl.RR; j += sub) {
      const u32 row = row_of(j);
      float v[8];
      octet_at(row)->widen(v);
      store_octet<NV>(p, row, col, v, s, z, [&](const int (&codes)[8]) {
        float x[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = ASYM ? (float)codes[k] - z[k % NV] : (float)codes[k];
        also(row, col, x, s);
      });
    }
    return;
  }
  const FastOctet<NV, ASYM> o(p, s, r, z);
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int j = (i << pl.sub_shift) + f;
    if (i >= pl.steps || j >= pl.RR) continue;
    float v[8];
    raw[i].widen(v);
    const u32 row = row_of(j);
    o.store(p, out_row32(p, row), col, v, [&](const float (&u)[8]) {
      float x[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) x[k] = u[k] - 12582912.f;
      also(row, col, x, s);
    });
    __builtin_amdgcn_sched_barrier(0);   // (rows started ahead of their turn cost registers that the held ones need)
  }
}
template <int DT, bool ASYM, bool KEEPC, int NT, int NI>
__global__ __launch_bounds__(NT) void quant_one_kernel(GenParams p, OnePlan pl) {
  take_second(p);
  quant_one_block<DT, ASYM, KEEPC, NT, NI>(p, pl, [](u32, int, const auto &, const auto &) {});
}

// ---- one pass by workgroups that share their groups ----------------------------------------------
// Where the rows of a group are too many for a workgroup: `n` workgroups of 256 threads take a block's rows, full rows of 256 bytes
// together with their neighbours', hold 16 octets (fp32: 8) per thread, exchange the extremes and quantize what they hold.  All of them
// are on the chip at once, four to a compute unit, and rows beyond the held ones are read again, the last ones first.  Bound by memory: the input
// is read once where the three launches read it twice, and where one launch holds a group in one workgroup, pieces of 16 bytes of
// a row cost it a request to the L2 each.  What the exchange costs, with the launch that clears its words, is about 9 us.  Three launches or one -> this,
// us, 8 bits, a scale per (head, channel): fp16 [64,n,16,64], two tensors, n = 100 23.8 -> 18.1, 169 31.0 -> 24.0, 256 40.9 -> 32.7; bf16
// [2,16,4096,128], two, 36.3 -> 32.1; affine, 2 bits, [B,30,680,64] B = 8 21.6 -> 16.8, 32 45.3 -> 38.5; fp32 B = 16 42.3 -> 29.2, 80 207 -> 168;
// bf16 [600,30,680,64] 940 -> 859; one scale per head, [32,30,680,64] 4 bits 44.7 -> 34.9, one per token 45.7 -> 34.7.
// The workgroups that share the groups of a block (see quant_shared_kernel): `n` of them, what they exchange and how long one
// waits for the others, in ticks of 10 ns.
struct Shards {
  int n;
  FastDiv by_n;
  u32 *mx, *mn;                 // per group, `stride` words apart
  u32 *words;                   // per block, `spacing` words apart, four of them a quarter of that from one another: see quant_shared_kernel
  int stride, spacing;
  u32 ticks;
};
constexpr int kSharedGroups = 1024;   // groups of a workgroup, and values of its fold
__global__ __launch_bounds__(256) void clear_shards_kernel(GenParams p, Shards sh, int64_t n_groups, int blocks) {
  if (take_second(p)) { sh.mx += p.ws1; sh.mn += p.ws1; sh.words += p.ws1; }
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n_groups) { sh.mx[i * sh.stride] = 0u; sh.mn[i * sh.stride] = 0xffffffffu; }
  if (i < blocks)
    for (int w = 0; w < 4; ++w) sh.words[sh.spacing * i + sh.spacing / 4 * w] = 0u;
}
template <int DT, bool ASYM, bool KEEPC>
__global__ __launch_bounds__(256, 4) void quant_shared_kernel(GenParams p, OnePlan pl, Shards sh) {
  constexpr int NV = KEEPC ? 8 : 1, NI = DT == VARQ_F32 ? 8 : 16, kAhead = NI / 4;   // octets held; requested at once beyond them
  __shared__ float lds_mx[kSharedGroups];
  __shared__ float lds_mn[ASYM ? kSharedGroups : 1];
  __shared__ float par_s[kSharedGroups], par_r[kSharedGroups];
  __shared__ float par_z[ASYM ? kSharedGroups : 1];
  __shared__ u32 lds_next;
  if (take_second(p)) { sh.mx += p.ws1; sh.mn += p.ws1; sh.words += p.ws1; }
  const int blk = (int)sh.by_n(blockIdx.x), shard = blockIdx.x - blk * sh.n, ko = (int)pl.by_tilesQ((u32)blk), tq = blk - ko * pl.tilesQ;
  const int tid = threadIdx.x, c8s = 1 << pl.c8s_shift, sub = 1 << pl.sub_shift;
  const int col = tid & (c8s - 1), f = (tid >> pl.c8s_shift) & (sub - 1), lq = tid >> (pl.c8s_shift + pl.sub_shift);
  const int f0 = shard * (pl.steps << pl.sub_shift) + f, q = (tq << pl.lq_shift) + lq;   // f0: the thread's first row
  const bool live = col < p.c8 && q < pl.Q;
  // (rows fit 31 bits and the bytes of a tensor 32)
  const u32 row0 = (u32)ko * (u32)pl.ko_rs + (live ? q : 0);
  auto row_at = [&](int step) { return (step << pl.sub_shift) + f0; };
  auto has = [&](int step) { return step < pl.steps && row_at(step) < pl.RR; };
  auto row_of = [&](int j) {
    const u32 o = pl.by_RI((u32)j);
    return row0 + o * (u32)pl.ro_rs + ((u32)j - o * (u32)pl.RI);
  };
  auto octet_at = [&](u32 row) { return reinterpret_cast<const Raw8<DT> *>(reinterpret_cast<const char *>(p.x) + (row * (u32)p.c + col * 8) * (u32)In8<DT>::kBytes); };

  Raw8<DT> raw[NI];
#pragma unroll
  for (int s = 0; s < NI; ++s)
    if (live && has(s)) raw[s] = *octet_at(row_of(row_at(s)));
  float mx[NV], mn[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) { mx[j] = ASYM ? -INFINITY : 0.f; mn[j] = INFINITY; }
  auto extend = [&](const Raw8<DT> &octet) __attribute__((always_inline)) {
    float v[8];
    octet.widen(v);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (ASYM) { mx[j % NV] = fmaxf(mx[j % NV], v[j]); mn[j % NV] = fminf(mn[j % NV], v[j]); }
      else mx[j % NV] = fmaxf(mx[j % NV], fabsf(v[j]));
    }
  };
#pragma unroll
  for (int s = 0; s < NI; ++s)
    if (live && has(s)) extend(raw[s]);
  if (live) {
    for (int i = NI; i < pl.steps; i += kAhead) {
      Raw8<DT> more[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) if (has(i + u)) more[u] = *octet_at(row_of(row_at(i + u)));
#pragma unroll
      for (int u = 0; u < kAhead; ++u) if (has(i + u)) extend(more[u]);
    }
  }
  // fold over f (and, with the channel dim reduced, over the columns), inside the wavefront first, as in quant_one_block
  const int q_lanes = sub << pl.c8s_shift, gcols = KEEPC ? c8s * 8 : 1;
  const int parts = q_lanes > 64 ? q_lanes >> 6 : 1, lane_in_part = q_lanes > 64 ? tid & 63 : tid & (q_lanes - 1);
  const int part = q_lanes > 64 ? tid >> 6 : tid >> (pl.sub_shift + pl.c8s_shift);
  auto fold = [&]() __attribute__((always_inline)) {
    for (int off = KEEPC ? c8s : 1; off < 64 && off < q_lanes; off <<= 1) {
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        mx[j] = fmaxf(mx[j], __shfl_xor(mx[j], off, 64));
        if (ASYM) mn[j] = fminf(mn[j], __shfl_xor(mn[j], off, 64));
      }
    }
    if (lane_in_part < (KEEPC ? c8s : 1)) {
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        lds_mx[part * gcols + col * NV + j] = mx[j];
        if (ASYM) lds_mn[part * gcols + col * NV + j] = mn[j];
      }
    }
    __syncthreads();
  };
  // body(t, whether there is such a group, its number, its extremes in this workgroup), a thread per group
  const int n_par = gcols << pl.lq_shift;
  auto per_group = [&](auto &&body) __attribute__((always_inline)) {
    for (int t = tid; t < n_par; t += 256) {
      const int tl = KEEPC ? t >> (pl.c8s_shift + 3) : t, g8 = t - tl * gcols, tqi = (tq << pl.lq_shift) + tl;
      float m = ASYM ? -INFINITY : 0.f, n = INFINITY;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int at = (tl * parts + min(w, parts - 1)) * gcols + g8;
        m = fmaxf(m, lds_mx[at]);
        if (ASYM) n = fminf(n, lds_mn[at]);
      }
      body(t, tqi < pl.Q && (!KEEPC || g8 < p.c), (int64_t)ko * pl.ko_gs + (int64_t)tqi * pl.q_gs + (KEEPC ? g8 : 0), m, n);
    }
  };
  // The extremes of all workgroups of the block meet in memory.  Nothing but these words goes from one workgroup to another, and every
  // access to them is an atomic of the device's scope, which all XCDs perform at one place: an extreme whose old value has come back is
  // there, the count goes up after that, and who has seen the count reads behind it.  (A release and an acquire instead write back and drop
  // whole L2s, once per workgroup: [64,256,16,64] fp16, two tensors, 33 -> 76 us.)  The last to arrive sets a word of its own,
  // half a `spacing` from the count, which the others look at: with all of them polling the counts, side by side, 56 us.
  //
  // The others may be waiting for a place on the chip, for as long as other launches please.  After `ticks` those that are here read the parts of the block's
  // rows over again, each part once, by whoever asks for it next (an extreme may be raised twice): the extremes are complete when all have arrived or all parts are
  // read, whichever is first.  And so that no workgroup depends on another one's progress, whoever finds no part left and has waited `ticks` for
  // those who read the last ones reads all rows by itself.  (With all rows read by everyone who had waited, us, beside 1000 workgroups of
  // another stream that keep their places for 2.2 ms, then / now / three launches: fp32 [2,3,35001,128] 2791 / 1310 / 1257, [60,3,35001,64] 2350 to 34000 /
  // 2378 / 2154, bf16 [300,30,680,64] affine 4467 / 2168 / 1932; on a device of their own after 3 us of patience, [2,3,35001,128] 1577 / 67,
  // [32,30,680,64] affine 291 / 62, a scale per head 267 / 55; waiting 55, 54, 50.)
  u32 *const arrived = sh.words + sh.spacing * blk, *const asked = arrived + sh.spacing / 4, *const all = arrived + sh.spacing / 2, *const read = all + sh.spacing / 4;
  constexpr u32 kOwn = ~0u, kEvery = ~0u - 1, kMet = ~0u - 2;   // what a round has read: the own part, all rows, or the part of that number; kMet: nothing is left to read
  const u32 n_shards = (u32)sh.n;
  for (u32 what = kOwn;;) {
    fold();
    per_group([&](int, bool mine, int64_t g, float m, float n) __attribute__((always_inline)) {
      if (!mine) return;
      const u32 a = __hip_atomic_fetch_max(sh.mx + g * sh.stride, ASYM ? enc_ord(m) : f2u(m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      u32 b = 0;
      if (ASYM) b = __hip_atomic_fetch_min(sh.mn + g * sh.stride, enc_ord(n), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("" :: "v"(a), "v"(b) : "memory");   // (the old values have come back)
    });
    __syncthreads();
    if (tid == 0) {
      auto wait = [&](u32 here) {
        const long long t0 = wall_clock64();
        while (here < n_shards && wall_clock64() - t0 < sh.ticks) {
          __builtin_amdgcn_s_sleep(8);
          here = __hip_atomic_load(all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return here;
      };
      u32 here = n_shards;
      if (what != kEvery) here = __hip_atomic_fetch_add(what == kOwn ? arrived : read, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
      if (here == n_shards) __hip_atomic_store(all, here, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else if (what == kOwn) here = wait(here);
      else here = __hip_atomic_load(all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      u32 next = kMet;
      if (here < n_shards) {
        next = __hip_atomic_fetch_add(asked, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (next >= n_shards) next = wait(0u) < n_shards ? kEvery : kMet;
      }
      lds_next = next;
    }
    __syncthreads();
    what = lds_next;
    if (what == kMet) break;
    if (live) {
      const int first = what == kEvery ? f : (int)what * (pl.steps << pl.sub_shift) + f, last = what == kEvery ? pl.RR : min(pl.RR, (int)(what + 1) * (pl.steps << pl.sub_shift));
      for (int j = first; j < last; j += kAhead << pl.sub_shift) {
        Raw8<DT> more[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) if (j + (u << pl.sub_shift) < last) more[u] = *octet_at(row_of(j + (u << pl.sub_shift)));
#pragma unroll
        for (int u = 0; u < kAhead; ++u) if (j + (u << pl.sub_shift) < last) extend(more[u]);
      }
    }
  }
  per_group([&](int t, bool mine, int64_t g, float m, float n) __attribute__((always_inline)) {
    if (mine) {
      const u32 a = __hip_atomic_load(sh.mx + g * sh.stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      m = ASYM ? dec_ord(a) : u2f(a);
      if (ASYM) n = dec_ord(__hip_atomic_load(sh.mn + g * sh.stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    }
    float s, zp = 0.f;
    if (ASYM) {
      s = fmaxf((m - n) / (float)((1 << p.bits) - 1), p.eps);
      zp = (float)p.qmin - rintf(n / s);
      par_z[t] = zp;
    } else {
      s = fmaxf(m / (float)p.qmax, p.eps);
    }
    par_s[t] = s;
    // (as in quant_one_block)
    par_r[t] = (s > 0x1p-96f && s < 0x1p96f && (f2u(s) & 0x7fffffu) != 0x7fffffu && fabsf(zp) <= 0x1p21f) ? 1.0f / s : 0.f;
    float *const once = KEEPC || !p.spread.on ? p.scale : p.spread.scale;
    if (mine && shard == 0 && once) {
      once[g] = s;
      if (ASYM) (KEEPC || !p.spread.on ? p.zp : p.spread.zp)[g] = zp;
    }
  });
  __syncthreads();
  if constexpr (!KEEPC) {
    auto group_of = [&](int t) { const int q = (tq << pl.lq_shift) + t; return q < pl.Q ? (int64_t)ko * pl.ko_gs + (int64_t)q * pl.q_gs : -1; };
    if (p.spread.on && shard == 0) spread_parameters<ASYM, 256>(p, pl.lq_shift, par_s, par_z, group_of);
  }
  if (!live) return;   // (2-bit words take two adjacent columns, which are live together: c is a multiple of 16 there)
  const int t0 = lq * gcols + col * (KEEPC ? 8 : 0);
  float s[NV], r[NV], z[NV] = {};
  bool plain = true;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    s[j] = par_s[t0 + j];
    r[j] = par_r[t0 + j];
    if (ASYM) z[j] = par_z[t0 + j];
    plain = plain && r[j] != 0.f;
  }
  if (__any(!plain)) {   // (rare, and once in the code: the rows are read again)
    for (int i = 0; has(i); ++i) {
      const u32 row = row_of(row_at(i));
      float v[8];
      octet_at(row)->widen(v);
      store_octet<NV>(p, row, col, v, s, z, [](const int (&)[8]) {});
    }
    return;
  }
  const FastOctet<NV, ASYM> o(p, s, r, z);
  auto finish = [&](int step, const Raw8<DT> &octet) __attribute__((always_inline)) {
    float v[8];
    octet.widen(v);
    o.store(p, out_row32(p, row_of(row_at(step))), col, v, [](const float (&)[8]) {});
  };
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    if (!has(i)) continue;
    finish(i, raw[i]);
    __builtin_amdgcn_sched_barrier(0);   // (rows started ahead of their turn cost registers that the held ones need)
  }
  // (those read last are the likeliest to be in a cache still)
  for (int i = NI + (pl.steps - 1 - NI) / kAhead * kAhead; i >= NI; i -= kAhead) {
    Raw8<DT> more[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) if (has(i + u)) more[u] = *octet_at(row_of(row_at(i + u)));
#pragma unroll
    for (int u = 0; u < kAhead; ++u) if (has(i + u)) finish(i + u, more[u]);
  }
}

// A step of a quantizer with a scale per (head, channel), and the whole cache dequantized behind it, in one launch:
// the first workgroups quantize the step and write its dequantized values from the codes in their registers, the
// others dequantize the earlier tokens.  The values are those of the two launches.  Bound by launches and by
// the chain of loads and barriers in the quantizing workgroups, under which the others now work.  8 bits, fp16 to fp32,
// two launches -> one, us: [8,n,30,64] 1 token behind none 8.3 -> 6.0, 36 behind 55 11.0 -> 8.6, 256 behind 424 24.5 -> 18.5.
struct StepOut {
  StepParams earlier;             // the tokens before this step (none: nseg = 0)
  int64_t inner, delta, off;      // input row r is output row r + r / inner * delta + off
  FastDiv by_inner;
  int odt, q_blocks, pair_blocks; // workgroups that quantize; workgroups of a pair of `earlier`
};
template <int DT, bool ASYM, int ODT, int NT, int NI>
__global__ __launch_bounds__(NT) void quant_one_step_kernel(GenParams p, OnePlan pl, StepOut o) {
  if ((int)blockIdx.x >= o.q_blocks) {
    constexpr int U = kStepOctets / NT;
    const int b = blockIdx.x - o.q_blocks, pair = b / o.pair_blocks, block = b - pair * o.pair_blocks;
    if (p.bits == 8) dequant_steps_block<ODT, 8, NT, U>(o.earlier, pair, block);
    else if (p.bits == 4) dequant_steps_block<ODT, 4, NT, U>(o.earlier, pair, block);
    else dequant_steps_block<ODT, 2, NT, U>(o.earlier, pair, block);
    return;
  }
  quant_one_block<DT, ASYM, true, NT, NI>(p, pl, [&](u32 row, int col, const auto &x, const auto &s) __attribute__((always_inline)) {
    float f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = x[j] * s[j];
    const int64_t orow = row + (int64_t)o.by_inner(row) * o.delta + o.off;
    store8<ODT>(o.earlier.out, orow * p.c + col * 8, f, 8);
  });
}

// ---- phase A, any c: one thread per element --------------------------------
template <int DT, bool ASYM>
__global__ void minmax_scalar_kernel(GenParams p) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= p.rows * p.c) return;
  const int64_t r = e / p.c;
  const int ch = (int)(e - r * p.c);
  int64_t i0, i1, i2;
  row_to_idx(p, r, i0, i1, i2);
  const int64_t g = i0 * p.gs0 + i1 * p.gs1 + i2 * p.gs2 + (p.keepc ? ch : 0);
  const float v = In8<DT>::load1(p.x, e);
  if (ASYM) {
    atomicMax(&p.ws[g], enc_ord(v));
    atomicMin(&p.ws[p.n_groups + g], enc_ord(v));
  } else {
    atomicMax(&p.ws[g], f2u(fabsf(v)));
  }
}

// ---- finalize: min/max -> scale, zero-point --------------------------------
template <bool ASYM>
__global__ void finalize_kernel(GenParams p) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= p.n_groups) return;
  if (ASYM) {
    const float mx = dec_ord(p.ws[g]), mn = dec_ord(p.ws[p.n_groups + g]);
    const float s = fmaxf((mx - mn) / (float)((1 << p.bits) - 1), p.eps);
    p.scale[g] = s;
    p.zp[g] = (float)p.qmin - rintf(mn / s);
  } else {
    p.scale[g] = fmaxf(u2f(p.ws[g]) / (float)p.qmax, p.eps);
  }
}

__device__ __forceinline__ int quant_one(float v, float s, float zp, bool asym, float qmin, float qmax) {
  float n = rintf(v / s);
  if (asym) n += zp;
  return (int)__builtin_amdgcn_fmed3f(n, qmin, qmax);
}

// ---- phase B, any c: one thread per output word (or per code group) ---------
template <int DT>
__global__ void quant_scalar_kernel(GenParams p) {
  const int vals = p.words ? 32 / p.bits : 4;
  const int wpr = (p.c + vals - 1) / vals;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= p.rows * wpr) return;
  const int64_t r = t / wpr;
  const int wi = (int)(t - r * wpr);
  int64_t i0, i1, i2;
  row_to_idx(p, r, i0, i1, i2);
  const int64_t gb = i0 * p.gs0 + i1 * p.gs1 + i2 * p.gs2;
  const u32 mask = (p.bits == 32) ? ~0u : ((1u << p.bits) - 1u);
  u32 w = 0;
  for (int j = 0; j < vals; ++j) {
    const int ch = wi * vals + j;
    if (ch >= p.c) break;
    const int64_t g = gb + (p.keepc ? ch : 0);
    const int q = quant_one(In8<DT>::load1(p.x, r * p.c + ch), p.scale[g], p.asym ? p.zp[g] : 0.f, p.asym,
                            (float)p.qmin, (float)p.qmax);
    if (p.codes) p.codes[out_row(p, r) * p.c + ch] = (int8_t)q;
    w |= ((u32)q & mask) << (j * p.bits);
  }
  if (p.words) p.words[out_row(p, r) * wpr + wi] = (int32_t)w;
}

// The leading dims in canonical form (see Plan).
struct Canonical { int64_t nko, nro, Q, RI, ko_rs, ro_rs, ko_gs, q_gs; };
Canonical canonical(const int64_t *sh, int reduce_mask) {
  const int64_t n0 = sh[0], n1 = sh[1], n2 = sh[2], c = sh[3], rows = n0 * n1 * n2;
  const bool k0 = !(reduce_mask & 1), k1 = !(reduce_mask & 2), k2 = !(reduce_mask & 4), kc = !(reduce_mask & 8);
  int64_t stride = kc ? c : 1;
  const int64_t gs2 = k2 ? stride : 0; if (k2) stride *= n2;
  const int64_t gs1 = k1 ? stride : 0; if (k1) stride *= n1;
  const int64_t gs0 = k0 ? stride : 0;
  Canonical k = {1, 1, 1, 1, 0, 0, 0, 0};
  if (k2) {
    k.Q = n2; k.q_gs = gs2;
    if (k1) {
      k.Q = n1 * n2;                                   // gs1 == gs2 * n2: q runs over (i1, i2)
      if (k0) k.Q = rows;                              // every row its own group
      else { k.nro = n0; k.ro_rs = n1 * n2; }
    } else if (k0) { k.nko = n0; k.ko_rs = n1 * n2; k.ko_gs = gs0; k.nro = n1; k.ro_rs = n2; }
    else { k.nro = n0 * n1; k.ro_rs = n2; }
  } else {
    k.RI = n2;
    if (!k1) {
      k.RI = n1 * n2;
      if (!k0) k.RI = rows;
      else { k.nko = n0; k.ko_rs = n1 * n2; k.ko_gs = gs0; }
    } else if (k0) { k.nko = n0 * n1; k.ko_rs = n2; k.ko_gs = gs1; }     // gs0 == gs1 * n1
    else { k.nko = n1; k.ko_rs = n2; k.ko_gs = gs1; k.nro = n0; k.ro_rs = n1 * n2; }
  }
  return k;
}

// Host side of the tiled path: the launch shape.  Returns false when the shape needs the scalar kernels.
bool make_plan(const int64_t *sh, int reduce_mask, int64_t n_groups, Plan &pl) {
  const int64_t c = sh[3];
  const int64_t rows = sh[0] * sh[1] * sh[2];
  if (c % 8 != 0 || rows <= 0 || rows >= (1ll << 31) - 512) return false;
  pl.c8 = (int)(c / 8);
  int c8p = 1, shl = 0;
  while (c8p < pl.c8) { c8p <<= 1; ++shl; }
  if (c8p > 64) return false;
  pl.c8p = c8p; pl.shift = shl; pl.R = 256 / c8p;
  const Canonical k = canonical(sh, reduce_mask);
  const int64_t nko = k.nko, nro = k.nro, Q = k.Q, RI = k.RI;
  pl.ko_rs = k.ko_rs; pl.ro_rs = k.ro_rs; pl.ko_gs = k.ko_gs; pl.q_gs = k.q_gs;
  pl.nko = (int)nko; pl.nro = (int)nro; pl.Q = (int)Q; pl.RI = (int)RI;
  pl.lanesQ = (int)(Q < pl.R ? Q : pl.R);
  if (RI == 1 && nro >= VARQ_GEN_NRO_MIN) {
    // Groups indexed by the innermost leading dim, many reduced rows each (the reference's default
    // method in layout BLHc): few row lanes on q -- rows of at least 128 channels per wavefront
    // segment -- and the others on consecutive reduced rows, which fold inside the workgroup.  More
    // tiles over q, hence fewer chunks and fewer partials for the finalize kernel to fold.
    int cap = 1;
    while (cap * 2 * c <= 128) cap *= 2;
    if (pl.lanesQ > cap) pl.lanesQ = cap;
  }
  pl.sub = pl.R / pl.lanesQ;
  pl.tilesQ = (int)((Q + pl.lanesQ - 1) / pl.lanesQ);
  pl.fold_ro = (RI == 1);
  int64_t steps;
  if (pl.fold_ro) { pl.T = 1; steps = (nro + pl.sub - 1) / pl.sub; }
  else { pl.T = (int)((RI + pl.sub - 1) / pl.sub); steps = nro * pl.T; }
  const int64_t kept_blocks = nko * pl.tilesQ;
  int64_t Z = (VARQ_GEN_BLOCKS + kept_blocks - 1) / kept_blocks;
  const int64_t zcap = (8ll << 20) / (n_groups > 0 ? n_groups : 1);   // partials stay below 64 MiB
  if (Z > zcap) Z = zcap;
  // ... and below a sixteenth of the input: with few kept blocks (groups indexed by the
  // innermost leading dim only, the BLHc layouts) thousands of chunks would write and re-read
  // as many partials as half the tensor
  const int64_t zvol = rows * c / (16 * (n_groups > 0 ? n_groups : 1));
  if (Z > zvol) Z = zvol;
  if (Z > steps) Z = steps;
  if (Z < 1) Z = 1;
  const int64_t spc = (steps + Z - 1) / Z;
  Z = (steps + spc - 1) / spc;                     // no empty chunk: every (z, group) partial gets written
  if (steps >= (1ll << 31) || kept_blocks * Z >= (1ll << 31)) return false;
  pl.steps = (int)steps; pl.Z = (int)Z; pl.steps_per_chunk = (int)spc;
  return true;
}

// Whether the one-launch kernel takes less time than the other way: workgroups that share their groups where `shared`, or the three launches, with their
// 2048 workgroups on either side of the fold.  Workgroups that share take 11 us and 0.37 per MiB (0.25 in fp32) as launches from the host, two less in a graph, where one launch is
// a tenth below what is said here: that / one, in a graph, us, [2,16,n,128] 8 bits, two tensors, 16 MiB 14.1 / 10.7, 25 17.7 / 15.2, 36 21.0 / 21.2, 64 31.9 / 36.3; [64,n,16,64] 9 12.6 / 10.7, 16
// 14.9 / 15.4; one tensor 4.5 10.9 / 9.0, 8 12.3 / 12.6; [B,30,680,64] fp32 20 13.0 / 11.9, 30 15.0 / 16.2, 40 17.8 / 21.7, affine 20 14.3 / 12.6, 40 18.8 / 20.2.
// The three take 12.4 us and 0.44 per MiB (of padded rows), for two tensors 16.2 and 0.41.  A workgroup of 1024 threads of the one-launch
// kernel, which has a compute unit to itself, takes 4.5 us and 0.22 per KiB in pieces of 16 bytes, 0.175 while there are no more than 128 of them, 0.135
// in pieces of 32 (0.17 where the rows lie multiples of 1 KiB apart), 0.10 in longer ones.  Three / one, us, 8 bits, a scale per (head, channel), two tensors:
// [2,16,n,128] 16 MiB 23.3 / 12.5, 25 25.0 / 18.9, 36 29.5 / 24.5, 64 44.2 / 39.4; [32,n,30,64] 23 24.7 / 18.6, 40 32.2 / 27.2, 60 42.1 / 38.2;
// [8,n,16,128] 36 30.2 / 28.4, 64 44.1 / 51.0; [64,n,16,64] 16 23.8 / 18.3, 25 25.4 / 27.8, 64 43.3 / 63.9; [4,8,n,128] 16 24.5 / 17.7, 25 25.7 / 27.0;
// [64,n,8,64] 12.5 21.3 / 24.2; one tensor: [64,n,16,64] 8 17.0 / 15.9, 12.5 18.0 / 24.2; [32,n,30,64] 11.7 16.9 / 15.1, 20 20.6 / 23.9; [16,n,12,64]
// 6 14.9 / 15.6, 9.4 15.7 / 23.9; [64,n,8,64] 6.2 15.8 / 22.9, 16 19.6 / 51.6; [2,16,n,128] 12.5 17.6 / 14.7, 18 19.3 / 20.6; fp32 [2,16,1600,128] 50 31.2 / 22.2.
// (The line was 16 MiB in all.)  Groups of whole rows keep to the sizes at which the one launch is never behind: up to 48 MiB symmetric, [32,30,L,64] bf16, one
// scale per (token, head), 24 MiB 22.8 / 18.1, 32 24.0 / 23.9, 48 36.1 / 32.0, 64 37.8 / 42.3, two tensors 48 33.6 / 32.1, 64 38.1 / 44.6; affine up to 16, 8 MiB
// 13.8 / 8.6, 16 17.0 / 17.2, 24 22.3 / 23.4, 48 33.9 / 42.8.  Other forms would gain beyond these lines: [64,16,L,64] fp16 64 MiB 37.7 / 31.1, affine 24
// 22.5 / 17.8, 64 36.8 / 40.5; [8,16,L,128] fp32 96 MiB 45.5 / 32.4, affine 43.3 / 40.7; one scale per token, [32,30,L,64] bf16 96 62.0 / 51.6, affine 48 34.2 / 28.7.  With the step dequantized in the same launch the other way has one
// more, whose work the one launch does beside: three and that / one, per tensor to fp32, [64,100,16,64] 40 / 74, [32,169,16,64] 41 / 64, [32,256,16,64]
// 51 / 71, [32,12,256,64] 46 / 62, [64,100,8,64] 26 / 30, [32,169,30,64] 58 / 48, [16,256,8,128] 43 / 38, [32,100,16,64] 25 / 19.
bool one_launch_pays(const OnePlan &pl, int c8, int c8p, int threads, bool keepc, double mib, int elem, int tensors, bool asym, bool with_values, bool shared) {
  if (!keepc) return mib <= (asym ? 16 : 48);
  if (threads == 256) return mib <= 16;
  const int64_t wgs = (int64_t)pl.blocks * pl.slices * tensors, cus = device_cus();
  const int piece = (8 * elem) << pl.c8s_shift;
  const bool apart = pl.RI == 1 && pl.ro_rs * c8 * 8 * elem % 1024 == 0;
  const double per_kib = piece <= 16 ? (wgs <= 128 ? 0.175 : 0.22) : piece == 32 ? (apart ? 0.17 : 0.135) : 0.10;
  const double one = 4.5 + per_kib * (asym ? 1.1 : 1.0) * mib * 1024.0 / (double)wgs * (double)((wgs + cus - 1) / cus);
  const double pad = (double)c8p / c8;
  // (32 bits, one round, long pieces, or heads first where lanes of the other way idle and a thread has few rows: the estimates of both ways are too
  // far off, and the one launch stays where it was before workgroups could share. One / shared: [32,30,55,96] two tensors affine 14.9 / 18.3,
  // [16,112,24,96] tokens first, two 12.8 / 15.2, [8,476,30,96] 15.9 / 17.9, [3,24,973,128] 12.7 / 14.2, [2,16,1779,128] two affine 19.1 / 21.1,
  // [4,24,987,128] 16.9 / 17.9, but [1,2611,12,128] two affine 15.1 / 14.7, [4,838,20,128] affine 17.4 / 15.2; short pieces, [8,16,498,72] 9.5 /
  // 12.5, [1,16,4718,72] 10.1 / 13.3, [2,6,3020,72] two 12.5 / 13.7, [8,30,708,40] affine 14.4 / 15.7, of eight rows [16,16,494,72] affine 23.2 /
  // 18.9)
  if (shared && elem == 4 && wgs <= cus && (piece >= 64 || (pl.RI > 1 && pad >= 1.6 && pl.steps <= 6))) shared = false;
  if (shared) return 0.9 * one < 11.0 + (elem == 4 ? 0.25 : 0.37) * mib * pad + (asym ? 1.0 : 0.0) + (with_values ? 10.5 : 0.0);
  const double three = (tensors == 2 ? 16.2 + 0.41 * mib * pad : 12.4 + 0.44 * mib * pad) + (asym ? 3.0 : 0.0) + (with_values ? 10.5 : 0.0);
  return one < three;
}

// The one-launch plan, or false when a group has too many rows for a workgroup's registers.
bool make_one_plan(const int64_t *sh, int reduce_mask, int elem, int tensors, int bits, bool asym, bool with_values, bool shared, OnePlan &pl, int &threads) {
  const int64_t c = sh[3], rows = sh[0] * sh[1] * sh[2];
  const int row_steps = elem == 4 ? 8 : 16;
  if (c % 8 != 0 || c > 512 || rows <= 0 || rows >= (1ll << 31) - 512) return false;
  const Canonical k = canonical(sh, reduce_mask);
  const int64_t rr = k.nro * k.RI;
  const double mib = (double)(rows * c * elem * tensors) / (1 << 20);
  if (rr > 8192 || mib > 128) return false;   // (rows and byte offsets of the kernel are of 32 bits)
  const bool keepc = !(reduce_mask & 8);
  const int c8 = (int)(c / 8);
  int c8p_shift = 0;
  while ((1 << c8p_shift) < c8) ++c8p_shift;
  pl.ko_rs = k.ko_rs; pl.ro_rs = k.ro_rs; pl.ko_gs = k.ko_gs; pl.q_gs = k.q_gs;
  pl.nko = (int)k.nko; pl.Q = (int)k.Q; pl.RR = (int)rr; pl.RI = (int)k.RI; pl.by_RI = FastDiv::by(k.RI);
  int rr_shift = 0;
  while ((1 << rr_shift) < rr) ++rr_shift;
  // column slices (channel dim kept): whole rows while that makes workgroups enough, 64 bytes of a row at least
  pl.c8s_shift = keepc && c8p_shift > 4 ? 4 : c8p_shift;
  // Narrower slices mean more workgroups and smaller pieces of each row, down to 32 bytes where dequantized values are
  // stored as well or a word of 2-bit codes takes two octets, to 16 otherwise.
  // A workgroup of 1024 threads holds its rows in the registers of a whole compute unit, so slices are halved only
  // while that leaves one for each of the 256, from 128 workgroups at most: K and V [64,n,16,64] fp16, 8 bits, 128 -> 256,
  // n = 64 24.9 -> 19.6 us, n = 16 9.9 -> 8.5; one tensor [8,256,36,64] 144 -> 288 11.2 -> 18.1, [2,1024,18,128] the
  // same 11.4 -> 18.0, [8,256,40,64] 160 -> 320 12.1 -> 18.6, [4,400,24,128] 192 -> 384 13.5 -> 19.4.
  // Several workgroups of 256 threads are resident on one, and more of them are no loss: [8,64,36,64] 144 -> 288 6.8 ->
  // 6.0, [8,64,48,64] 192 -> 384 6.8 -> 6.2; [2,400,18,128] 7.9 either way.  The dequantized values of a step in 32-byte pieces from
  // twice as many workgroups take a schedule of [8,n,30,64] from 208 to 227 us.
  const int narrowest = bits == 2 || with_values ? 1 : 0;
  for (;; --pl.c8s_shift) {
    pl.slices = keepc ? (c8 + (1 << pl.c8s_shift) - 1) >> pl.c8s_shift : 1;
    // 256 threads where their rows suffice, 1024 otherwise; the row lanes of a q no more than its rows
    for (threads = 256; ; threads = 1024) {
      const int shift = (threads == 256 ? 8 : 10) - pl.c8s_shift;
      pl.sub_shift = rr_shift < shift ? rr_shift : shift;
      // (few rows: a step or two more per thread and fewer lanes per q would only make fewer workgroups)
      pl.lq_shift = shift - pl.sub_shift;
      while (pl.lq_shift > 0 && (1ll << (pl.lq_shift - 1)) >= k.Q) --pl.lq_shift;
      pl.steps = (int)((rr + (1 << pl.sub_shift) - 1) >> pl.sub_shift);
      if (pl.steps <= 4 || threads == 1024) break;
    }
    pl.tilesQ = (int)((k.Q + (1 << pl.lq_shift) - 1) >> pl.lq_shift);
    pl.blocks = pl.nko * pl.tilesQ;
    pl.by_slices = FastDiv::by(pl.slices); pl.by_tilesQ = FastDiv::by(pl.tilesQ);
    const bool fits = pl.steps <= row_steps;
    const int enough = with_values ? 128 : threads == 1024 ? 129 : 160;
    if (fits && ((int64_t)pl.blocks * pl.slices * tensors >= enough || !keepc || pl.c8s_shift <= narrowest)) return one_launch_pays(pl, c8, 1 << c8p_shift, threads, keepc, mib, elem, tensors, asym, with_values, shared);
    if (!keepc || pl.c8s_shift <= narrowest) return false;
  }
}

// The plan of workgroups that share their groups, in `words` of workspace per tensor, or false where it does not pay whatever one launch
// takes; three_wgs: the workgroups of either of the large ones among the three launches.  Tokens first, tensors of 16 bits lose beyond 192 MiB, where the second
// read comes from memory and 256 bytes of a row in eight sets of workgroups are the worse way through it: [64,n,16,64] fp16 125 MiB 71.8 -> 63.5 us, 187
// 105 -> 99, 250 135 -> 144, 500 266 -> 301; fp32 250 119 -> 107, 375 195 -> 174.  Heads first they lose from there on (lanes that idle counted in) where the three
// launches come out as one round of eight workgroups per compute unit, three -> this: [2199,8,256,72] 618 MiB 357 -> 486, [4,24,17568,72] 232 125 -> 148, [8,16,14491,64] 226
// 109 -> 116, [39,8,6115,64] 233 affine 115 -> 126, a scale per head of [635,16,508,40] 394 240 -> 296; with 2050 to 2070 workgroups, where a few are a second round,
// the three take longer: [402,24,517,64] 609 397 -> 322, [162,30,169,128] 201 110 -> 90, unless nearly half of the lanes idle, [339,20,680,72] 633
// 483 -> 518, [2,30,40914,72] 337 230 -> 274 (against [3184,12,169,40] 493 370 -> 355).  Of 394 forms of 16 bits from 11 to 880 MiB 51 were slower by more than 2.5 % than the three
// without this line and that of `few`, six with them, the worst of which are tokens first in idle lanes ([2223,36,30,40] 104 -> 134).  Groups of whole rows gain from 48 MiB: 8 bits affine, a scale per head of [B,30,680,64] bf16, 20 MiB
// 18.1 -> 21.9, 30 22.6 -> 19.4, 40 27.4 -> 31.3, 50 33.1 -> 27.6, 80 48.9 -> 38.0, per token 50 34.2 -> 25.7.
bool make_shared_plan(const int64_t *sh, int reduce_mask, int64_t n_groups, int elem, int tensors, size_t words, int64_t three_wgs, OnePlan &pl, Shards &s) {
  const int64_t c = sh[3], rows = sh[0] * sh[1] * sh[2];
  if (c % 8 != 0 || c > 512 || rows <= 0 || rows >= (1ll << 31) - 512) return false;
  const Canonical k = canonical(sh, reduce_mask);
  const int64_t rr = k.nro * k.RI;
  const int64_t bytes = rows * c * elem * tensors;
  const bool keepc = !(reduce_mask & 8);
  if (rows * c * elem > (1ll << 31)) return false;   // (rows and byte offsets of the kernel are of 32 bits)
  if (!keepc && bytes < (48ll << 20)) return false;
  if (k.RI == 1 && elem == 2 && bytes > (192ll << 20)) return false;
  const int c8 = (int)(c / 8);
  int c8p_shift = 0;
  while ((1 << c8p_shift) < c8) ++c8p_shift;
  const bool half_idle = 7 * c8 <= 4 << c8p_shift;
  if (k.RI > 1 && elem == 2 && (half_idle || three_wgs <= 8 * (int64_t)device_cus()) && (bytes / c8 << c8p_shift) > (192ll << 20)) return false;
  pl.ko_rs = k.ko_rs; pl.ro_rs = k.ro_rs; pl.ko_gs = k.ko_gs; pl.q_gs = k.q_gs;
  pl.nko = (int)k.nko; pl.Q = (int)k.Q; pl.RR = (int)rr; pl.RI = (int)k.RI; pl.by_RI = FastDiv::by(k.RI);
  pl.c8s_shift = c8p_shift; pl.slices = 1;
  // pieces of 256 bytes
  pl.lq_shift = 0;
  while (k.RI == 1 && (2 << pl.lq_shift) <= k.Q && ((8 * elem) << (c8p_shift + pl.lq_shift)) < 256) ++pl.lq_shift;
  if (8 - c8p_shift - pl.lq_shift < 0) return false;
  pl.sub_shift = 8 - c8p_shift - pl.lq_shift;
  pl.tilesQ = (int)((k.Q + (1 << pl.lq_shift) - 1) >> pl.lq_shift);
  if (k.nko * pl.tilesQ > 512) return false;
  pl.blocks = pl.nko * pl.tilesQ;
  pl.by_slices = FastDiv::by(1); pl.by_tilesQ = FastDiv::by(pl.tilesQ);
  // as many workgroups as the chip holds at once, of at least four steps (groups of whole rows: eight), and no more than meet quickly; of
  // fewer than three per compute unit, or than nearly four where lanes idle, the three launches read faster (two heads: fp32 [1,2,381944,72], one scale per
  // head, 103 -> 128 us, fp16 [2,2,381944,72] 139 -> 261; three: fp16 [2,3,23148,72] 22.3 -> 23.6, but fp32 [5,3,28645,128] 104 -> 87), in 16 bits also of fewer than
  // three and a half where more rows are read again than half of those that the registers hold (three heads, 768 workgroups: 16 steps 31.8 -> 30.9, 18 31.5 -> 30.4,
  // 25 38.5 -> 40.1, 48 62.5 -> 65.1, 89 109 -> 139, 283 417 -> 537)
  const int64_t least = (keepc ? 4ll : 8ll) << pl.sub_shift;
  int64_t n = std::min<int64_t>({(int64_t)device_cus() * 4 / ((int64_t)pl.blocks * tensors), (rr + least - 1) / least, 256});
  if (n < 2 || n * pl.blocks * tensors * 4 < (int64_t)device_cus() * (c8 == 1 << c8p_shift ? 12 : 15)) return false;
  pl.steps = (int)((rr + (n << pl.sub_shift) - 1) / (n << pl.sub_shift));
  n = (rr + ((int64_t)pl.steps << pl.sub_shift) - 1) / ((int64_t)pl.steps << pl.sub_shift);
  const bool few = n * pl.blocks * tensors * 2 < (int64_t)device_cus() * 7;
  if (elem == 2 && few && pl.steps > 24) return false;
  const int n_par = (keepc ? 8 << c8p_shift : 1) << pl.lq_shift, fold_vals = n_par * std::max(1, (1 << (pl.sub_shift + c8p_shift)) / 64);
  if (n < 2 || std::max(n_par, fold_vals) > kSharedGroups) return false;
  // (lines of their own for the extremes of each group of whole rows and for the words of a block, and as far apart as there is room
  // otherwise: atomics on one line wait for one another.  One scale per head of 30 heads, 60 or 61 chunks of the three launches and thus room for
  // half a line: fp32 [60,30,66,128] affine 36.4 -> 19.7 us (side by side / 16 words apart; three launches 28.1), [3,30,3843,40] 33.7 -> 21.0 (26.4))
  s.n = (int)n; s.by_n = FastDiv::by(n);
  for (s.stride = keepc ? 1 : 32; s.stride > 1 && 2 * (size_t)s.stride * (size_t)n_groups + 64 * (size_t)pl.blocks > words;) s.stride /= 2;
  const size_t left = words - std::min(words, 2 * s.stride * (size_t)n_groups);
  for (s.spacing = 64; s.spacing >= 8 && (size_t)s.spacing * pl.blocks > left;) s.spacing /= 2;
  s.ticks = (u32)(10000 + (bytes >> 20) * 100);   // 0.1 ms, and 1 us for each MiB, several times what it takes
  return s.spacing >= 8;
}

template <int DT, bool ASYM, bool KEEPC>
void launch_one(const GenParams &p, const OnePlan &pl, int threads, hipStream_t st) {
  constexpr int NI = DT == VARQ_F32 ? 8 : 16;
  dim3 grid((unsigned)((pl.blocks + 7) / 8 * 8 * pl.slices), p.x1 ? 2u : 1u);
  // (256 threads have at most four steps, see make_one_plan; a kernel for more has their code and registers)
  if (threads == 1024 && pl.steps > 4) hipLaunchKernelGGL((quant_one_kernel<DT, ASYM, KEEPC, 1024, NI>), grid, dim3(1024), 0, st, p, pl);
  else if (threads == 1024) hipLaunchKernelGGL((quant_one_kernel<DT, ASYM, KEEPC, 1024, 4>), grid, dim3(1024), 0, st, p, pl);
  else if (pl.steps <= 2) hipLaunchKernelGGL((quant_one_kernel<DT, ASYM, KEEPC, 256, 2>), grid, dim3(256), 0, st, p, pl);
  else hipLaunchKernelGGL((quant_one_kernel<DT, ASYM, KEEPC, 256, 4>), grid, dim3(256), 0, st, p, pl);
}
template <int DT> void run_one(const GenParams &p, const OnePlan &pl, int threads, hipStream_t st) {
  if (p.asym) { if (p.keepc) launch_one<DT, true, true>(p, pl, threads, st); else launch_one<DT, true, false>(p, pl, threads, st); }
  else { if (p.keepc) launch_one<DT, false, true>(p, pl, threads, st); else launch_one<DT, false, false>(p, pl, threads, st); }
}

template <int DT, bool ASYM, int ODT> void launch_one_step(const GenParams &p, const OnePlan &pl, int threads, const StepOut &o, unsigned blocks, hipStream_t st) {
  constexpr int NI = DT == VARQ_F32 ? 8 : 16;
  if (threads == 1024 && pl.steps > 4) hipLaunchKernelGGL((quant_one_step_kernel<DT, ASYM, ODT, 1024, NI>), dim3(blocks), dim3(1024), 0, st, p, pl, o);
  else if (threads == 1024) hipLaunchKernelGGL((quant_one_step_kernel<DT, ASYM, ODT, 1024, 4>), dim3(blocks), dim3(1024), 0, st, p, pl, o);
  else if (pl.steps <= 2) hipLaunchKernelGGL((quant_one_step_kernel<DT, ASYM, ODT, 256, 2>), dim3(blocks), dim3(256), 0, st, p, pl, o);
  else hipLaunchKernelGGL((quant_one_step_kernel<DT, ASYM, ODT, 256, 4>), dim3(blocks), dim3(256), 0, st, p, pl, o);
}
template <int DT> void run_one_step(const GenParams &p, const OnePlan &pl, int threads, const StepOut &o, unsigned blocks, hipStream_t st) {
  auto typed = [&](auto odt) {
    constexpr int ODT = decltype(odt)::value;
    if (p.asym) launch_one_step<DT, true, ODT>(p, pl, threads, o, blocks, st);
    else launch_one_step<DT, false, ODT>(p, pl, threads, o, blocks, st);
  };
  if (o.odt == VARQ_F32) typed(std::integral_constant<int, VARQ_F32>{});
  else if (o.odt == VARQ_BF16) typed(std::integral_constant<int, VARQ_BF16>{});
  else typed(std::integral_constant<int, VARQ_F16>{});
}

template <int DT, bool ASYM, bool KEEPC>
void launch_shared(const GenParams &p, const OnePlan &pl, const Shards &sh, hipStream_t st) {
  const unsigned nt = p.x1 ? 2u : 1u;
  const int64_t n = std::max(p.n_groups, (int64_t)pl.blocks);
  hipLaunchKernelGGL(clear_shards_kernel, dim3((unsigned)((n + 255) / 256), nt), dim3(256), 0, st, p, sh, p.n_groups, pl.blocks);
  hipLaunchKernelGGL((quant_shared_kernel<DT, ASYM, KEEPC>), dim3((unsigned)(pl.blocks * sh.n), nt), dim3(256), 0, st, p, pl, sh);
}
template <int DT> void run_shared(const GenParams &p, const OnePlan &pl, const Shards &sh, hipStream_t st) {
  if (p.asym) { if (p.keepc) launch_shared<DT, true, true>(p, pl, sh, st); else launch_shared<DT, true, false>(p, pl, sh, st); }
  else { if (p.keepc) launch_shared<DT, false, true>(p, pl, sh, st); else launch_shared<DT, false, false>(p, pl, sh, st); }
}

// workgroups of the min/max launch, and of the one that quantizes
int64_t large_wgs(const Plan &pl) { return (int64_t)pl.nko * pl.tilesQ * pl.Z; }
size_t plan_workspace_bytes(const Plan &pl, int64_t n_groups) {
  return (size_t)n_groups * (2 + 2 * (size_t)pl.Z) * sizeof(float);
}

template <int DT>
int run_tiled(GenParams &p, const Plan &pl, void *workspace, hipStream_t st) {
  const int64_t ng = p.n_groups;
  float *rinv = reinterpret_cast<float *>(workspace);
  u32 *plain = reinterpret_cast<u32 *>(rinv + ng);
  float *part_max = rinv + 2 * ng;
  float *part_min = part_max + (int64_t)pl.Z * ng;
  const unsigned nt = p.x1 ? 2u : 1u;   // tensors per launch (grid.y)
  p.ws1 = (int64_t)(plan_workspace_bytes(pl, ng) / sizeof(float));
  dim3 grid((unsigned)large_wgs(pl), nt);
  if (p.asym) {
    if (p.keepc) hipLaunchKernelGGL((minmax_tiled_kernel<DT, true, true>), grid, dim3(256), 0, st, p, pl, part_max, part_min);
    else hipLaunchKernelGGL((minmax_tiled_kernel<DT, true, false>), grid, dim3(256), 0, st, p, pl, part_max, part_min);
  } else {
    if (p.keepc) hipLaunchKernelGGL((minmax_tiled_kernel<DT, false, true>), grid, dim3(256), 0, st, p, pl, part_max, part_min);
    else hipLaunchKernelGGL((minmax_tiled_kernel<DT, false, false>), grid, dim3(256), 0, st, p, pl, part_max, part_min);
  }
  // z-lanes per group in the finalize kernel: enough threads in total, no more lanes than partials
  int ZL = 1;
  while (ZL < 256 && ZL < pl.Z && ng * ZL < VARQ_FIN_THREADS) ZL <<= 1;
  // ... and where each group's parameters have many places, so many workgroups as there are compute units (or groups)
  if (p.spread.on)
    while (ZL < 256 && (256 / ZL) * (int64_t)p.spread.reps > 1024 && ng * ZL < 256 * 256) ZL <<= 1;
  dim3 fgrid((unsigned)((ng + 256 / ZL - 1) / (256 / ZL)), nt);
  if (p.asym)
    hipLaunchKernelGGL((finalize_tiled_kernel<true>), fgrid, dim3(256), 0, st, p, pl.Z, ZL, part_max, part_min, rinv, plain);
  else
    hipLaunchKernelGGL((finalize_tiled_kernel<false>), fgrid, dim3(256), 0, st, p, pl.Z, ZL, part_max, part_min, rinv, plain);
  // the parameters as the last launch reads them, one after the other by group, are where a caller takes them once each
  if (p.spread.on) { p.scale = p.spread.scale; p.zp = p.spread.zp; p.scale1 = p.spread.scale1; p.zp1 = p.spread.zp1; }
  // phase B walks the same chunks (its per-thread parameters are eight 16-byte loads; chunks of 4 to 8 steps
  // per thread measured alike, longer ones slower)
  const Plan &pb = pl;
  dim3 bgrid((unsigned)((int64_t)pb.nko * pb.tilesQ * pb.Z), nt);
  // Five workgroups on a compute unit instead of eight (by LDS that they do not use) for large tensors of 32 bits with long
  // groups: fewer chunks are read at once, and more of the second read comes out of the Infinity Cache.  Eight / five, us for the three
  // launches on tensors in turn, a scale per (head, channel), 8 bits, then 4 bits affine: [B,30,680,64] fp32, 80 MiB 43.1 / 43.7, 43.6 / 44.3; 120 62.0 / 61.5,
  // 59.0 / 59.1; 194 94.6 / 91.9, 87.8 / 86.7; 264 139 / 133, 130 / 122; 319 170 / 164, 160 / 150; 398 209 / 208, 195 / 193; 702 364 / 358, 328 / 315; [B,30,680,128]
  // the same, one scale for all of it 319 MiB 168 / 162, 156 / 147; the same tensor again and again, its dequantization behind it, 1-3 % at all of them.  Tensors of
  // 16 bits, whose launch has more instructions per byte, lose by it up to 256 MiB and go either way beyond: bf16 120 MiB 70.7 / 73.3, 65.9 / 70.1; 159
  // 91.0 / 93.3, 82.0 / 89.7; 192 109 / 114, 98 / 101; 264 174 / 164, 164 / 154 (D=128 154 / 154, 139 / 145); 401 233 / 238, 222 / 225; 513 339 / 318, 320 / 297 (292 / 294, 274 / 277).
  const bool large = DT == VARQ_F32 && !p.x1 && p.rows * p.c * In8<DT>::kBytes >= (128ll << 20) && pl.Z >= 16;
  const unsigned lds = large ? 32000 : 0;
  if (p.asym) {
    if (p.keepc) hipLaunchKernelGGL((quant_tiled_kernel<DT, true, true>), bgrid, dim3(256), lds, st, p, pb, rinv, plain);
    else hipLaunchKernelGGL((quant_tiled_kernel<DT, true, false>), bgrid, dim3(256), lds, st, p, pb, rinv, plain);
  } else {
    if (p.keepc) hipLaunchKernelGGL((quant_tiled_kernel<DT, false, true>), bgrid, dim3(256), lds, st, p, pb, rinv, plain);
    else hipLaunchKernelGGL((quant_tiled_kernel<DT, false, false>), bgrid, dim3(256), lds, st, p, pb, rinv, plain);
  }
  return 0;
}

// any shape: one thread per element / per output word, group min/max by ordered-integer atomics
template <int DT>
int run_general(GenParams &p, hipStream_t st) {
  const int64_t ng = p.n_groups;
  hipLaunchKernelGGL(init_ws_kernel, dim3((unsigned)((ng + 255) / 256)), dim3(256), 0, st, p.ws,
                     p.asym ? p.ws + ng : (u32 *)nullptr, ng);
  {
    const int64_t n = p.rows * p.c;
    dim3 grid((unsigned)((n + 255) / 256));
    if (p.asym) hipLaunchKernelGGL((minmax_scalar_kernel<DT, true>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((minmax_scalar_kernel<DT, false>), grid, dim3(256), 0, st, p);
  }
  {
    dim3 grid((unsigned)((ng + 255) / 256));
    if (p.asym) hipLaunchKernelGGL((finalize_kernel<true>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((finalize_kernel<false>), grid, dim3(256), 0, st, p);
  }
  {
    const int vals = p.words ? 32 / p.bits : 4;
    const int64_t n = p.rows * ((p.c + vals - 1) / vals);
    dim3 grid((unsigned)((n + 255) / 256));
    hipLaunchKernelGGL((quant_scalar_kernel<DT>), grid, dim3(256), 0, st, p);
  }
  return 0;
}

int64_t count_groups(const int64_t *s, int reduce_mask) {
  int64_t n = 1;
  for (int d = 0; d < 4; ++d)
    if (!(reduce_mask & (1 << d))) n *= s[d];
  return n;
}

}  // namespace

extern "C" size_t varq_quant_workspace_bytes(const int64_t *host_shape4, int reduce_mask) {
  if (!host_shape4) return 0;
  const int64_t ng = count_groups(host_shape4, reduce_mask);
  Plan pl;
  if (make_plan(host_shape4, reduce_mask, ng, pl)) return plan_workspace_bytes(pl, ng);
  return (size_t)ng * 2 * sizeof(u32);
}

namespace {
// the launches that a tensor (or two of one shape) takes
enum class Way { kOne, kShared, kThree, kAnyShape };
Way choose_way(const int64_t *sh, int reduce_mask, int64_t n_groups, int elem, int tensors, int word_bits, bool asym, bool with_values, bool may_share, size_t words_each,
               int64_t three_wgs, OnePlan &one, int &threads, OnePlan &by_many, Shards &shards) {
  const bool shared = may_share && make_shared_plan(sh, reduce_mask, n_groups, elem, tensors, words_each, three_wgs, by_many, shards);
  if (make_one_plan(sh, reduce_mask, elem, tensors, word_bits, asym, with_values, shared, one, threads)) return Way::kOne;
  return shared ? Way::kShared : Way::kThree;
}

// x1 != NULL: a second tensor of the same shape with its own outputs, in the same launches
// where the tiled kernels apply, one after the other through the same workspace otherwise
int quant_pack_impl(const void *x, const void *x1, int x_dtype, const int64_t *host_shape4, int reduce_mask, int bits,
                    int asym, float eps, int32_t *words, int8_t *codes, float *scale, float *zp,
                    int32_t *words1, int8_t *codes1, float *scale1, float *zp1,
                    const int64_t *host_out_map, void *workspace, size_t workspace_bytes, void *stream,
                    StepOut *step = nullptr, int64_t step_pairs = 0, const int64_t *host_scale_map = nullptr, float *const *once = nullptr, const u32 *host_wait_ticks = nullptr) {
  VARQ_CHECK_ARG(host_shape4, "quant_pack: null shape");
  const int64_t *s = host_shape4;
  VARQ_CHECK_ARG(s[0] >= 0 && s[1] >= 0 && s[2] >= 0 && s[3] > 0 && s[3] <= (1 << 20), "quant_pack: bad shape");
  VARQ_CHECK_ARG(x_dtype >= 0 && x_dtype <= 2, "quant_pack: bad dtype %d", x_dtype);
  VARQ_CHECK_ARG(reduce_mask >= 0 && reduce_mask < 16, "quant_pack: bad reduce mask");
  VARQ_CHECK_ARG(bits > 1 && bits <= 8, "quant_pack: bits must be in 2..8 (got %d)", bits);
  VARQ_CHECK_ARG(!words || bits == 2 || bits == 4 || bits == 8, "quant_pack: packing implements 2/4/8 bits only (got %d)", bits);
  const int64_t rows = s[0] * s[1] * s[2];
  if (rows == 0) return VARQ_OK;
  VARQ_CHECK_ARG(words || codes, "quant_pack: no output requested");
  VARQ_CHECK_ARG(scale && (!asym || zp), "quant_pack: scale/zp output missing");
  VARQ_CHECK_ARG(x && (workspace || host_scale_map), "quant_pack: null pointer");
  if (x1) {
    VARQ_CHECK_ARG((!words == !words1) && (!codes == !codes1) && scale1 && (!asym || zp1),
                   "quant_pack: the second tensor needs the same kinds of output as the first");
  }
  const int64_t ng = count_groups(s, reduce_mask);
  Plan pl;
  // the tiled kernels pack whole words per octet: c*bits must fill words (always true for 4 and 8 bits)
  const bool tiled = make_plan(s, reduce_mask, ng, pl) && (!words || (s[3] * bits) % 32 == 0);
  const size_t need = tiled ? plan_workspace_bytes(pl, ng) * (x1 ? 2 : 1) : (size_t)ng * 2 * sizeof(u32);
  if (workspace_bytes < need && (!host_scale_map || workspace))
    return varq_set_error(VARQ_ERR_WORKSPACE, "quant_pack: workspace %zu < %zu bytes", workspace_bytes, need);
  VARQ_CHECK_ARG(rows * s[3] < (1ll << 40), "quant_pack: tensor too large");
  // only the tiled kernels that keep the channel dim move scales, zero-points and partials in
  // 16-byte pieces; every other path reads and writes them one word at a time
  const uintptr_t par_align = (tiled && !(reduce_mask & 8)) ? 15 : 3;
  VARQ_CHECK_ARG((((uintptr_t)workspace | (uintptr_t)scale | (uintptr_t)zp | (uintptr_t)scale1 | (uintptr_t)zp1) & par_align) == 0,
                 "quant_pack: scale, zp and workspace must be %d-byte aligned for this shape", (int)par_align + 1);

  GenParams p;
  p.x = x;
  p.ws = reinterpret_cast<u32 *>(workspace);
  p.scale = scale; p.zp = zp; p.words = words; p.codes = codes;
  p.x1 = nullptr; p.scale1 = nullptr; p.zp1 = nullptr; p.words1 = nullptr; p.codes1 = nullptr; p.ws1 = 0;
  p.out_mapped = 0; p.out_inner = 1; p.out_delta = 0; p.out_off = 0;
  if (host_out_map) {
    VARQ_CHECK_ARG(host_out_map[0] > 0 && host_out_map[1] >= 0 && host_out_map[2] >= 0 && rows % host_out_map[0] == 0,
                   "quant_pack: output map {rows per block, extra rows per block, first row} = {%lld, %lld, %lld} does not fit %lld rows",
                   (long long)host_out_map[0], (long long)host_out_map[1], (long long)host_out_map[2], (long long)rows);
    p.out_mapped = 1; p.out_inner = host_out_map[0]; p.out_delta = host_out_map[1]; p.out_off = host_out_map[2];
  }
  p.by_inner = FastDiv::by(p.out_inner);
  p.spread.on = 0;
  if (const int64_t *m = host_scale_map) {
    VARQ_CHECK_ARG(m[0] > 0 && m[4] > 0 && m[5] > 0 && (reduce_mask & 8), "quant_pack: scales of whole rows can be spread, over at least one place each");
    // (places counted in 32 bits, times the 512 groups that a workgroup has at most)
    if (m[4] > (1 << 22) || m[4] * m[5] > (1 << 22))
      return varq_set_error(VARQ_ERR_UNSUPPORTED, "quant_pack: scales are spread over at most 4 million places each");
    VARQ_CHECK_ARG(!once || !once[0] || ((!asym || once[1]) && (!x1 || (once[2] && (!asym || once[3])))), "quant_pack: scales once per group come with zero-points, and for both tensors");
    p.spread = {1, FastDiv::by(m[0]), FastDiv::by(m[4]), (u32)std::min(m[0], (int64_t)0x7fffffff), (u32)m[4], (u32)(m[4] * m[5]), m[1], m[2], m[3], m[6],
                once ? once[0] : nullptr, once ? once[1] : nullptr, once ? once[2] : nullptr, once ? once[3] : nullptr};
  }
  p.n1 = s[1]; p.n2 = s[2];
  p.c = (int)s[3];
  p.keepc = !(reduce_mask & 8);
  // group-id strides of the kept leading dims, row-major over the kept dims
  int64_t stride = p.keepc ? p.c : 1;
  p.gs2 = (reduce_mask & 4) ? 0 : stride; if (!(reduce_mask & 4)) stride *= s[2];
  p.gs1 = (reduce_mask & 2) ? 0 : stride; if (!(reduce_mask & 2)) stride *= s[1];
  p.gs0 = (reduce_mask & 1) ? 0 : stride;
  p.rows = rows;
  p.n_groups = ng;
  p.c8 = (p.c + 7) / 8;
  p.bits = bits; p.qmin = -(1 << (bits - 1)); p.qmax = (1 << (bits - 1)) - 1;
  p.wpr = words ? (p.c + 32 / bits - 1) / (32 / bits) : 0;
  p.asym = asym ? 1 : 0;
  p.eps = eps;
  hipStream_t st = (hipStream_t)stream;
  OnePlan one;
  int threads;
  const size_t words_each = tiled ? plan_workspace_bytes(pl, ng) / sizeof(u32) : 0;
  OnePlan by_many;
  Shards sh = {};
  const Way way = tiled ? choose_way(s, reduce_mask, ng, x_dtype == VARQ_F32 ? 4 : 2, x1 ? 2 : 1, words ? bits : 8, asym != 0, step != nullptr, !host_scale_map || workspace,
                                     words_each, large_wgs(pl), one, threads, by_many, sh)
                        : Way::kAnyShape;
  if (way == Way::kOne) {
    if (step) {
      step->q_blocks = (one.blocks + 7) / 8 * 8 * one.slices;
      step->pair_blocks = (int)((step->earlier.pair_octs + kStepOctets - 1) / kStepOctets);
      const int64_t blocks = step->q_blocks + step_pairs * step->pair_blocks;
      if (blocks < (1ll << 31)) {
        const unsigned n = (unsigned)blocks;
        if (x_dtype == VARQ_F32) run_one_step<VARQ_F32>(p, one, threads, *step, n, st);
        else if (x_dtype == VARQ_BF16) run_one_step<VARQ_BF16>(p, one, threads, *step, n, st);
        else run_one_step<VARQ_F16>(p, one, threads, *step, n, st);
        VARQ_CHECK_LAUNCH("quant_step_dequant");
        step->q_blocks = -1;   // done
        return VARQ_OK;
      }
    }
    if (x1) { p.x1 = x1; p.scale1 = scale1; p.zp1 = zp1; p.words1 = words1; p.codes1 = codes1; }
    if (x_dtype == VARQ_F32) run_one<VARQ_F32>(p, one, threads, st);
    else if (x_dtype == VARQ_BF16) run_one<VARQ_BF16>(p, one, threads, st);
    else run_one<VARQ_F16>(p, one, threads, st);
  } else if (way == Way::kShared) {
    if (x1) { p.x1 = x1; p.scale1 = scale1; p.zp1 = zp1; p.words1 = words1; p.codes1 = codes1; }
    p.ws1 = (int64_t)words_each;
    sh.mx = p.ws; sh.mn = p.ws + ng * sh.stride; sh.words = p.ws + 2 * ng * sh.stride;
    if (host_wait_ticks) sh.ticks = *host_wait_ticks;
    if (x_dtype == VARQ_F32) run_shared<VARQ_F32>(p, by_many, sh, st);
    else if (x_dtype == VARQ_BF16) run_shared<VARQ_BF16>(p, by_many, sh, st);
    else run_shared<VARQ_F16>(p, by_many, sh, st);
  } else if (host_scale_map && (way == Way::kAnyShape || !workspace || !p.spread.scale)) {
    return varq_set_error(VARQ_ERR_UNSUPPORTED, "quant_pack: spread scales come with groups that one launch quantizes, or with a workspace and the scales once per group");
  } else if (way == Way::kThree) {
    if (x1) { p.x1 = x1; p.scale1 = scale1; p.zp1 = zp1; p.words1 = words1; p.codes1 = codes1; }
    if (x_dtype == VARQ_F32) run_tiled<VARQ_F32>(p, pl, workspace, st);
    else if (x_dtype == VARQ_BF16) run_tiled<VARQ_BF16>(p, pl, workspace, st);
    else run_tiled<VARQ_F16>(p, pl, workspace, st);
  } else {
    for (int t = 0; t < (x1 ? 2 : 1); ++t) {   // stream order keeps the shared workspace safe
      if (t == 1) { p.x = x1; p.scale = scale1; p.zp = zp1; p.words = words1; p.codes = codes1; }
      if (x_dtype == VARQ_F32) run_general<VARQ_F32>(p, st);
      else if (x_dtype == VARQ_BF16) run_general<VARQ_BF16>(p, st);
      else run_general<VARQ_F16>(p, st);
    }
  }
  VARQ_CHECK_LAUNCH("quant_pack");
  return VARQ_OK;
}
}  // namespace

extern "C" int varq_quant_pack(const void *x, int x_dtype, const int64_t *host_shape4, int reduce_mask, int bits,
                               int asym, float eps, int32_t *words, int8_t *codes, float *scale, float *zp,
                               const int64_t *host_out_map, void *workspace, size_t workspace_bytes, void *stream) {
  return quant_pack_impl(x, nullptr, x_dtype, host_shape4, reduce_mask, bits, asym, eps, words, codes, scale, zp,
                         nullptr, nullptr, nullptr, nullptr, host_out_map, workspace, workspace_bytes, stream);
}

extern "C" int varq_quant_pack2(const void *x0, const void *x1, int x_dtype, const int64_t *host_shape4, int reduce_mask,
                                int bits, int asym, float eps, int32_t *words0, int8_t *codes0, float *scale0, float *zp0,
                                int32_t *words1, int8_t *codes1, float *scale1, float *zp1,
                                const int64_t *host_out_map, void *workspace, size_t workspace_bytes, void *stream) {
  // (tensors without rows may come as null pointers: nothing to do, as in varq_quant_pack)
  if (host_shape4 && host_shape4[0] >= 0 && host_shape4[1] >= 0 && host_shape4[2] >= 0 &&
      host_shape4[0] * host_shape4[1] * host_shape4[2] == 0 && host_shape4[3] > 0)
    return VARQ_OK;
  VARQ_CHECK_ARG(x1, "quant_pack2: null second tensor");
  return quant_pack_impl(x0, x1, x_dtype, host_shape4, reduce_mask, bits, asym, eps, words0, codes0, scale0, zp0,
                         words1, codes1, scale1, zp1, host_out_map, workspace, workspace_bytes, stream);
}

extern "C" int varq_quant_pack_wait(const void *x, int x_dtype, const int64_t *host_shape4, int reduce_mask, int bits, int asym, float eps, int32_t *words,
                                    int8_t *codes, float *scale, float *zp, const int64_t *host_out_map, uint32_t wait_ticks, void *workspace,
                                    size_t workspace_bytes, void *stream) {
  return quant_pack_impl(x, nullptr, x_dtype, host_shape4, reduce_mask, bits, asym, eps, words, codes, scale, zp, nullptr, nullptr, nullptr, nullptr,
                         host_out_map, workspace, workspace_bytes, stream, nullptr, 0, nullptr, nullptr, &wait_ticks);
}

extern "C" int varq_quant_pack_shards(const int64_t *host_shape4, int reduce_mask, int x_dtype, int tensors, int word_bits, int asym) {
  const int64_t ng = count_groups(host_shape4, reduce_mask);
  Plan pl;
  if (!make_plan(host_shape4, reduce_mask, ng, pl) || (host_shape4[3] * word_bits) % 32 != 0) return 0;
  OnePlan one, by_many;
  Shards sh = {};
  int threads;
  const Way way = choose_way(host_shape4, reduce_mask, ng, x_dtype == VARQ_F32 ? 4 : 2, tensors, word_bits, asym != 0, false, true, plan_workspace_bytes(pl, ng) / sizeof(u32),
                             large_wgs(pl), one, threads, by_many, sh);
  return way == Way::kShared ? sh.n : way == Way::kOne ? 1 : 0;
}

extern "C" int varq_quant_pack_spread_room(const void *x0, const void *x1, int x_dtype, const int64_t *host_shape4, int reduce_mask, int bits, int asym,
                                           float eps, int32_t *words0, float *scale0, float *zp0, int32_t *words1, float *scale1, float *zp1,
                                           float *once_scale0, float *once_zp0, float *once_scale1, float *once_zp1,
                                           const int64_t *host_out_map, const int64_t *host_scale_map, void *workspace, size_t workspace_bytes, void *stream) {
  VARQ_CHECK_ARG(host_scale_map, "quant_pack_spread: null scale map");
  float *const once[4] = {once_scale0, once_zp0, once_scale1, once_zp1};
  return quant_pack_impl(x0, x1, x_dtype, host_shape4, reduce_mask, bits, asym, eps, words0, nullptr, scale0, zp0, words1, nullptr, scale1, zp1,
                         host_out_map, workspace, workspace_bytes, stream, nullptr, 0, host_scale_map, once);
}

extern "C" int varq_quant_pack_spread_once(const void *x0, const void *x1, int x_dtype, const int64_t *host_shape4, int reduce_mask, int bits, int asym,
                                           float eps, int32_t *words0, float *scale0, float *zp0, int32_t *words1, float *scale1, float *zp1,
                                           float *once_scale0, float *once_zp0, float *once_scale1, float *once_zp1,
                                           const int64_t *host_out_map, const int64_t *host_scale_map, void *stream) {
  return varq_quant_pack_spread_room(x0, x1, x_dtype, host_shape4, reduce_mask, bits, asym, eps, words0, scale0, zp0, words1, scale1, zp1,
                                     once_scale0, once_zp0, once_scale1, once_zp1, host_out_map, host_scale_map, nullptr, 0, stream);
}

extern "C" int varq_quant_pack_spread(const void *x0, const void *x1, int x_dtype, const int64_t *host_shape4, int reduce_mask, int bits, int asym,
                                      float eps, int32_t *words0, float *scale0, float *zp0, int32_t *words1, float *scale1, float *zp1,
                                      const int64_t *host_out_map, const int64_t *host_scale_map, void *stream) {
  return varq_quant_pack_spread_once(x0, x1, x_dtype, host_shape4, reduce_mask, bits, asym, eps, words0, scale0, zp0, words1, scale1, zp1,
                                     nullptr, nullptr, nullptr, nullptr, host_out_map, host_scale_map, stream);
}

// Quantizes a step into its tokens of the cache buffer and dequantizes the whole cache: in one launch where the step
// takes one by itself and the cache is not much more work than it (see kStepMostSym), in the launches of the two calls otherwise.
extern "C" int varq_quant_step_dequant(const void *x, int x_dtype, int B, int H, int n, int c, int tokens_first, int bits, int asym, float eps,
                                       int32_t *words, int64_t capacity, float *scale, float *zp, int nseg, const int32_t *host_seg_end,
                                       void *out, int out_dtype, void *workspace, size_t workspace_bytes, void *stream) {
  VARQ_CHECK_ARG(x && words && scale && out && host_seg_end && (!asym || zp), "quant_step_dequant: null pointer");
  VARQ_CHECK_ARG(nseg >= 1 && nseg <= 16 && B > 0 && H > 0 && n > 0 && c > 0 && c % 8 == 0 && c <= (1 << 20),
                 "quant_step_dequant: bad sizes (1..16 steps, whole octets of channels)");
  VARQ_CHECK_ARG((bits == 2 || bits == 4 || bits == 8) && (c * bits) % 32 == 0, "quant_step_dequant: bits must be 2, 4 or 8 and rows whole words");
  VARQ_CHECK_ARG(out_dtype >= 0 && out_dtype <= 2, "quant_step_dequant: bad output dtype %d", out_dtype);
  VARQ_CHECK_ARG((((uintptr_t)x | (uintptr_t)scale | (uintptr_t)zp | (uintptr_t)out) & 15) == 0 && ((uintptr_t)words & 7) == 0, "quant_step_dequant: misaligned operand");
  for (int s = 0, prev = 0; s < nseg; prev = host_seg_end[s++])
    VARQ_CHECK_ARG(host_seg_end[s] >= prev, "quant_step_dequant: segment ends must increase");
  const int64_t start = nseg > 1 ? host_seg_end[nseg - 2] : 0, tokens = host_seg_end[nseg - 1], per = tokens_first ? H : 1, row = (int64_t)H * c;
  VARQ_CHECK_ARG(tokens - start == n && tokens <= capacity, "quant_step_dequant: the last step has %d tokens and the buffer room for %lld", n, (long long)capacity);
  const int64_t shape[4] = {B, tokens_first ? n : H, tokens_first ? H : n, c}, map[3] = {n * per, (capacity - n) * per, start * per};
  StepOut o;
  const int64_t pairs = tokens_first ? B : (int64_t)B * H;
  // (refused before the step is quantized)
  VARQ_CHECK_ARG(set_steps(o.earlier, words, scale, asym ? zp : nullptr, nseg, host_seg_end, B, H, capacity, c, bits, tokens_first, out),
                 "quant_step_dequant: more tokens or pairs than the grid holds");
  set_steps(o.earlier, words, scale, asym ? zp : nullptr, nseg - 1, host_seg_end, B, H, capacity, c, bits, tokens_first, out);
  const bool fits = pairs * start * o.earlier.octs <= (asym ? kStepMostAsym : kStepMostSym);
  o.earlier.out_pair_octs = tokens * o.earlier.octs;
  o.inner = map[0]; o.by_inner = FastDiv::by(map[0]); o.delta = (tokens - n) * per; o.off = map[2];
  o.odt = out_dtype; o.q_blocks = 0; o.pair_blocks = 0;
  float *const s = scale + (nseg - 1) * row, *const z = asym ? zp + (nseg - 1) * row : nullptr;
  if (const int e = quant_pack_impl(x, nullptr, x_dtype, shape, tokens_first ? 0b0011 : 0b0101, bits, asym, eps, words, nullptr, s, z, nullptr, nullptr,
                                    nullptr, nullptr, map, workspace, workspace_bytes, stream, fits ? &o : nullptr, pairs))
    return e;
  if (o.q_blocks < 0) return VARQ_OK;
  return varq_dequant_steps(words, scale, asym ? zp : nullptr, nseg, host_seg_end, B, H, capacity, c, bits, tokens_first, out, out_dtype, stream);
}

// ---- the entry point that allocates nothing ------------------------------------------
// Its workspace is this array, which every device the library runs on holds from the load
// of the code object to the end of the process.  Host code never uses the array's name as
// an address: scratch_for_current_device() asks the runtime once per device where that
// device's copy lives and hands out that pointer.
static __device__ __align__(256) unsigned char scratch[VARQ_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

int scratch_for_current_device(void **out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return varq_set_error(VARQ_ERR_LAUNCH, "quant_pack_static: hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices)
    return varq_set_error(VARQ_ERR_UNSUPPORTED, "quant_pack_static: device index %d beyond %d", dev, kMaxDevices - 1);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return varq_set_error(VARQ_ERR_LAUNCH, "quant_pack_static: hipGetSymbolAddress: %s", hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return VARQ_OK;
}
}  // namespace

// Also the warm-up call: it looks the current device's copy of the array up (a runtime query that
// must not happen while a stream is being captured into a graph), so that the entry point below
// finds the address already there.  Without a usable device it only reports the size.
extern "C" size_t varq_quant_static_scratch_bytes(void) {
  void *ws = nullptr;
  (void)scratch_for_current_device(&ws);
  return (size_t)VARQ_STATIC_SCRATCH_BYTES;
}

extern "C" int varq_quant_pack_static(const void *x, int x_dtype, const int64_t *host_shape4, int reduce_mask, int bits,
                                      int asym, float eps, int32_t *words, int8_t *codes, float *scale, float *zp,
                                      const int64_t *host_out_map, void *stream) {
  VARQ_CHECK_ARG(host_shape4, "quant_pack_static: null shape");
  VARQ_CHECK_ARG(reduce_mask >= 0 && reduce_mask < 16, "quant_pack_static: bad reduce mask");
  const size_t need = varq_quant_workspace_bytes(host_shape4, reduce_mask);
  if (need > (size_t)VARQ_STATIC_SCRATCH_BYTES)
    return varq_set_error(VARQ_ERR_WORKSPACE,
                          "quant_pack_static: this shape and grouping need %zu bytes of partial results, the static "
                          "scratch holds %zu; use varq_quant_pack with a workspace of the caller's",
                          need, (size_t)VARQ_STATIC_SCRATCH_BYTES);
  void *ws = nullptr;
  const int rc = scratch_for_current_device(&ws);
  if (rc != VARQ_OK) return rc;
  // every partial and parameter the kernels read is written earlier in the same call (plain
  // stores, or the fill kernel of the scalar path), so what an earlier call left behind is
  // never seen and nothing needs clearing here
  return quant_pack_impl(x, nullptr, x_dtype, host_shape4, reduce_mask, bits, asym, eps, words, codes, scale, zp,
                         nullptr, nullptr, nullptr, nullptr, host_out_map, ws, (size_t)VARQ_STATIC_SCRATCH_BYTES, stream);
}
