// kvf_quantize.hip - the KV append step: fp32 rows quantized on the GPU and
// scattered to their physical rows (kvf_quantize_place, kvf_append_tokens),
// bit-exact with runtime/kvf_host.h:72-135,166-184.
//
// Bound by memory: a row of d floats is read once and its codes and (scale,
// zero) words are written once. The arithmetic has to stay below that, so a
// lane holds 8 neighbouring elements (two 16-byte loads, one store of 4, 8 or
// 16 bytes of codes), a row takes d / 8 lanes, a group of 32, 64 or 128
// elements is 4, 8 or 16 neighbouring lanes, and its minimum and maximum are
// DPP steps inside a row of 16 lanes.
#include "kvf_kernels.hpp"

namespace kvf {
namespace gfx950 {
namespace {

// Exact i / div for i < 2^31: (i * mul) >> (31 + l) with mul = ceil(2^(31+l) / div),
// l = ceil(log2 div); the rounding of mul adds less than 1 / div to i / div.
struct FastDiv {
  uint32_t div = 1, mul = 1u << 31, l = 0;
  FastDiv() = default;
  explicit FastDiv(uint32_t d) : div(d) {
    while ((1ull << l) < d) ++l;
    mul = (uint32_t)(((1ull << (31 + l)) + d - 1) / d);
  }
  __device__ uint32_t quot(uint32_t i) const { return __umulhi(i << 1, mul) >> l; }
};

// Where the rows come from and go. Work item i is a row in the order of the
// physical layout, so that neighbouring lanes write neighbouring rows: sequence
// by sequence, head by head (head-major) or token by token (token-major: a
// token's rows of all heads lie side by side, and a head at a time would write
// every line in Hkv pieces from different workgroups).
struct Place {
  uint32_t rows;        // B * Hkv * n
  int n, Hkv, order, bt, max_blocks;
  FastDiv inner, outer; // sizes of the two inner dimensions of a work item
  FastDiv page;         // bt (1 for contiguous)
  const int *table;
};

// One step of a minimum / maximum over the lanes of a group: the value of the
// lane that DPP control CTRL names.
template <int CTRL> __device__ __forceinline__ float dpp(float x) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}
// Reduction over the 4, 8 or 16 lanes of a group: pairs and quads by quad
// permutation, then the mirror of 8 and the mirror of 16 lanes (each lane
// then meets a lane of the other half, all of which hold their half's value).
template <int LANES, class F> __device__ __forceinline__ float over_group(float x, F f) {
  x = f(x, dpp<0xB1>(x));                          // quad_perm 1,0,3,2
  x = f(x, dpp<0x4E>(x));                          // quad_perm 2,3,0,1
  if constexpr (LANES >= 8) x = f(x, dpp<0x141>(x));  // row_half_mirror
  if constexpr (LANES >= 16) x = f(x, dpp<0x140>(x)); // row_mirror
  return x;
}

// Rows and codes need only their element's alignment (the hardware takes
// unaligned addresses), as with element-wise accesses.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u1u __attribute__((aligned(1)));
typedef uint32_t u2u __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t u4u __attribute__((ext_vector_type(4), aligned(2)));

// round(x / sc) clamped to [0, levels] as the reference computes it: the
// correctly rounded quotient, rounded half away from zero. `r` is the
// correctly rounded 1 / sc; one residual step then gives the correctly rounded
// quotient (Markstein, 1990): q = a r, q + (a - q sc) r. It needs finite
// operands and no underflow in the residual; sc is a binary16 value >= 2^-24
// and a quotient below 2^-2 rounds to 0 whatever its last bit is, so only
// sc = 0 and non-finite sc or zero point need the division itself.
// The rounding: adding the largest float below 1/2 and truncating equals
// rounding half away from zero for 0 <= q < 2^23.
__device__ __forceinline__ uint32_t code_fast(float a, float sc, float r, float levels) {
  const float q0 = a * r;
  const float q = fmaf(fmaf(-q0, sc, a), r, q0);
  return (uint32_t)(fminf(fmaxf(q, 0.f), levels) + 0.49999997f);
}
__device__ __forceinline__ uint32_t code_div(float a, float sc, float levels) {
  return (uint32_t)(fminf(fmaxf(__fdiv_rn(a, sc), 0.f), levels) + 0.49999997f);
}

// Quantizes a row's 8 elements [8c, 8c + 8) and writes them, and the group's
// (scale, zero) from its first lane, to physical row `prow`. All lanes of a
// row call it together (the reductions stay inside a row). NT: the codes pass
// the caches by (a whole prompt's rows), or stay for the step that reads them.
template <int FMT, int D, int GQ, bool NT>
__device__ __forceinline__ void put_row(f4u v0, f4u v1, int c, long long prow, unsigned char *data, uint32_t *meta) {
  constexpr int ROW = D * bits_of<FMT>() / 8;
  float e[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) e[k] = k < 4 ? v0[k % 4] : v1[k % 4];
  unsigned char *to = data + prow * ROW + c * (8 * bits_of<FMT>() / 8);
  if constexpr (FMT == FMT_F16) {
    u4u w;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      w[k] = __builtin_bit_cast(uint32_t, (half2_t){(_Float16)e[2 * k], (_Float16)e[2 * k + 1]});
    if constexpr (NT) __builtin_nontemporal_store(w, reinterpret_cast<u4u *>(to));
    else *reinterpret_cast<u4u *>(to) = w;
  } else {
    constexpr float LEVELS = FMT == FMT_INT8 ? 255.f : 15.f;
    constexpr int LPG = GQ / 8; // lanes per group
    auto mn = [](float a, float b) { return fminf(a, b); };
    auto mx = [](float a, float b) { return fmaxf(a, b); };
    // signalling NaNs are made quiet first: the three-operand minimum that the
    // compiler forms returns a NaN for one, and the next drops what was so far
    // the minimum along with it (quiet ones are skipped, as in the reference;
    // 8 instructions a lane: int4 31.7 -> 32.4 us for 4 x 4093 tokens, int8 none)
#pragma unroll
    for (int k = 0; k < 8; ++k) e[k] = __builtin_canonicalizef(e[k]);
    float lo = e[0], hi = e[0];
#pragma unroll
    for (int k = 1; k < 8; ++k) {
      lo = fminf(lo, e[k]);
      hi = fmaxf(hi, e[k]);
    }
    lo = over_group<LPG>(lo, mn);
    hi = over_group<LPG>(hi, mx);
    const _Float16 zero_h = (_Float16)lo;
    float scale = __fdiv_rn(hi - lo, LEVELS);
    if (scale <= 0.f) scale = 1.f;
    const _Float16 scale_h = (_Float16)scale;
    const float zero = (float)zero_h;
    const float sc = (float)scale_h;
    if (c % LPG == 0)
      meta[prow * (D / GQ) + c / LPG] = (uint32_t)__builtin_bit_cast(uint16_t, scale_h) |
                                           ((uint32_t)__builtin_bit_cast(uint16_t, zero_h) << 16);
    uint32_t q[8];
    if (sc > 0.f && sc < INFINITY && fabsf(zero) < INFINITY) {
      const float r = __fdiv_rn(1.f, sc);
#pragma unroll
      for (int k = 0; k < 8; ++k) q[k] = code_fast(e[k] - zero, sc, r, LEVELS);
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) q[k] = code_div(e[k] - zero, sc, LEVELS);
    }
    if constexpr (FMT == FMT_INT8) {
      u2u w;
#pragma unroll
      for (int k = 0; k < 2; ++k)
        w[k] = q[4 * k] | q[4 * k + 1] << 8 | q[4 * k + 2] << 16 | q[4 * k + 3] << 24;
      if constexpr (NT) __builtin_nontemporal_store(w, reinterpret_cast<u2u *>(to));
      else *reinterpret_cast<u2u *>(to) = w;
    } else {
      uint32_t w = 0;
#pragma unroll
      for (int k = 0; k < 8; ++k) w |= q[k] << (4 * k); // even elements in the low nibble
      if constexpr (NT) __builtin_nontemporal_store(w, reinterpret_cast<u1u *>(to));
      else *reinterpret_cast<u1u *>(to) = w;
    }
  }
}

// A wave takes 512 / D neighbouring work items, a load of 16 bytes twice a
// lane. Items' (sequence, head, token) come from one scalar division per wave,
// its first item's, and a carry per lane (per-lane divisions were as many
// cycles as the quantizing). More items a wave, 2, 4 or 8 loads in flight a
// lane, were each slower than more waves (2: 64.8, 4: 68.2, 8: 76.5 us where 1
// takes 62.3); the codes' stores are nontemporal, the rows' loads are not (they
// are often still cached: with nontemporal loads 8000 tokens 16.8 -> 18.5 us).
// Measured on MI355X, K and V of one layer with 8 KV heads of 128: 32768
// tokens in int8:64, head-major contiguous, 339 -> 59 us (5.8 TB/s read and
// written; a large copy reaches 5.3); 4 x 4093 tokens in int4:32, paged
// token-major, 180 -> 32 us (4.8 TB/s). Before, a wave took one row, a lane
// single elements with byte stores, and every element one division.
template <int FMT, int D, int GQ>
__global__ void __launch_bounds__(256)
quantize_place_kernel(const float *__restrict__ x, unsigned char *__restrict__ data, uint32_t *__restrict__ meta,
                      const Place p) {
  constexpr int LPR = D / 8;    // lanes per row
  constexpr int RPW = 64 / LPR; // rows per wave
  const int lane = threadIdx.x & 63;
  const int c = lane % LPR;     // the lane's elements are [8c, 8c + 8)
  const uint32_t i0 = (blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * RPW, o = lane / LPR;
  const bool ok = i0 + o < p.rows;
  // past the end: the last row again, loaded and not stored
  const uint32_t item = ok ? i0 + o : p.rows - 1;
  uint32_t in, mid, b;
  if (p.inner.div >= RPW && i0 + RPW <= p.rows) {
    const uint32_t rest0 = p.inner.quot(i0), b0 = p.outer.quot(rest0);
    in = i0 - rest0 * p.inner.div + o;
    mid = rest0 - b0 * p.outer.div;
    b = b0;
    if (in >= p.inner.div) {
      in -= p.inner.div;
      ++mid;
    }
    if (mid >= p.outer.div) {
      mid = 0;
      ++b;
    }
  } else {
    const uint32_t rest = p.inner.quot(item);
    in = item - rest * p.inner.div;
    b = p.outer.quot(rest);
    mid = rest - b * p.outer.div;
  }
  const uint32_t h = p.order == ORD_HEAD ? mid : in;
  const uint32_t t = p.order == ORD_HEAD ? in : mid;
  // logical row (b Hkv + h) n + t; head-major items are in that order already
  const uint32_t src = p.order == ORD_HEAD ? item : (b * p.Hkv + h) * p.n + t;
  const float *xr = x + (long long)src * D + c * 8;
  const f4u v0 = *reinterpret_cast<const f4u *>(xr), v1 = *reinterpret_cast<const f4u *>(xr + 4);
  long long prow = item; // the physical row; contiguous: the item itself
  if (p.bt) {
    const uint32_t blk = p.page.quot(t), off = t - blk * p.bt;
    prow = (long long)p.table[(long long)b * p.max_blocks + blk] * (p.Hkv * p.bt) +
           (p.order == ORD_HEAD ? h * p.bt + off : off * p.Hkv + h);
  }
  // (a row's lanes go together: the group reductions stay inside a row)
  if (ok) put_row<FMT, D, GQ, true>(v0, v1, c, prow, data, meta);
}

// One token per sequence: a workgroup is one wave on 64 * 8 / D neighbouring
// heads of sequence blockIdx.y (and y + 65535, ...). A handful of rows: nothing
// but the chain argument -> position -> page id -> store bounds it, so the
// arguments are 14 dwords that arrive preloaded, the rows' loads go out ahead of
// the chain, and position and page are scalar. (Captured steps of 8 layers for 4
// sequences, 16 calls beside 16 other kernels: 118.3 -> 114.7 us a graph against
// appending through the kernel above.)
template <int FMT, int D, int GQ>
__global__ void __launch_bounds__(64)
append_kernel(const float *__restrict__ x, const int *__restrict__ positions, const int *__restrict__ table,
              unsigned char *__restrict__ data, uint32_t *__restrict__ meta, const int Hkv, const int limit,
              const uint32_t bt_order, const int max_blocks, const int B) {
  constexpr int LPR = D / 8;
  const int c = threadIdx.x % LPR;
  const int h = blockIdx.x * (64 / LPR) + threadIdx.x / LPR;
  const uint32_t bt = bt_order & 0x7fffffffu;
  const bool head_major = !(bt_order >> 31);
  int b = blockIdx.y; // the grid has no y past B
  do {
    const float *xr = x + ((long long)b * Hkv + min(h, Hkv - 1)) * D + c * 8;
    const f4u v0 = *reinterpret_cast<const f4u *>(xr), v1 = *reinterpret_cast<const f4u *>(xr + 4);
    const int pos = positions[b];
    // a position outside the layout writes nothing (no branch: one would hold
    // back the rows' loads until the position is there)
    const bool ok = pos >= 0 && pos < limit;
    const uint32_t t = ok ? (uint32_t)pos : 0u;
    long long prow;
    if (bt) {
      uint32_t blk, in;
      if ((bt & (bt - 1)) == 0) {
        blk = t >> __builtin_ctz(bt);
        in = t & (bt - 1);
      } else {
        blk = t / bt;
        in = t - blk * bt;
      }
      const long long base = (long long)table[(long long)b * max_blocks + blk] * ((long long)Hkv * bt);
      prow = base + (head_major ? (long long)h * bt + in : (long long)in * Hkv + h);
    } else {
      prow = head_major ? ((long long)b * Hkv + h) * limit + t : ((long long)b * limit + t) * Hkv + h;
    }
    if (ok && h < Hkv) put_row<FMT, D, GQ, false>(v0, v1, c, prow, data, meta);
    b += 65535;
  } while (b < B);
}

// What a call names: fmt, group, rows and layout (positions: one token per
// sequence).
struct Call {
  int fmt, group;
  const float *x;
  int B, Hkv, n;
  const int *positions;
  int order, bt;
  const int *table;
  int max_blocks;
  unsigned char *data;
  uint32_t *meta;
};

template <int FMT, int D, int GQ> hipError_t launch_quantize(const Call &q, hipStream_t st) {
  constexpr uint32_t RPW = 64 / (D / 8);
  if (q.positions) {
    const long long limit = q.bt ? (long long)q.max_blocks * q.bt : q.n;
    const dim3 grid((unsigned)((q.Hkv + RPW - 1) / RPW), (unsigned)std::min(q.B, 65535));
    const uint32_t bt_order = (uint32_t)q.bt | (q.order == ORD_HEAD ? 0u : 1u << 31);
    hipLaunchKernelGGL((append_kernel<FMT, D, GQ>), grid, dim3(64), 0, st, q.x, q.positions, q.table, q.data, q.meta,
                       q.Hkv, (int)std::min(limit, 0x7fffffffLL), bt_order, q.max_blocks, q.B);
    return hipGetLastError();
  }
  Place p;
  p.rows = (uint32_t)((long long)q.B * q.Hkv * q.n);
  p.n = q.n;
  p.Hkv = q.Hkv;
  p.order = q.order;
  p.bt = q.bt;
  p.max_blocks = q.max_blocks;
  p.inner = FastDiv(q.order == ORD_HEAD ? q.n : q.Hkv);
  p.outer = FastDiv(q.order == ORD_HEAD ? q.Hkv : q.n);
  p.page = FastDiv(q.bt ? q.bt : 1);
  p.table = q.table;
  const dim3 grid((p.rows + 4 * RPW - 1) / (4 * RPW));
  hipLaunchKernelGGL((quantize_place_kernel<FMT, D, GQ>), grid, dim3(256), 0, st, q.x, q.data, q.meta, p);
  return hipGetLastError();
}

template <int D> hipError_t launch_format(const Call &q, hipStream_t st) {
  switch (q.fmt) {
  case FMT_F16:
    return launch_quantize<FMT_F16, D, D>(q, st);
  case FMT_INT8:
    if (q.group == 32) return launch_quantize<FMT_INT8, D, 32>(q, st);
    if (q.group == 64) return launch_quantize<FMT_INT8, D, 64>(q, st);
    return launch_quantize<FMT_INT8, D, D>(q, st);
  case FMT_INT4:
    if (q.group == 32) return launch_quantize<FMT_INT4, D, 32>(q, st);
    if (q.group == 64) return launch_quantize<FMT_INT4, D, 64>(q, st);
    return launch_quantize<FMT_INT4, D, D>(q, st);
  default:
    return hipErrorInvalidValue;
  }
}

hipError_t quantize_rows(const Call &q, int d, hipStream_t st) {
  if (!q.x || !q.data || q.B < 1 || q.Hkv < 1 || q.n < 1 || (d != 64 && d != 128)) return hipErrorInvalidValue;
  if (q.order != ORD_HEAD && q.order != ORD_TOKEN) return hipErrorInvalidValue;
  if (q.bt < 0 || (q.bt > 0 && (!q.table || q.max_blocks * q.bt < q.n))) return hipErrorInvalidValue;
  if (q.fmt != FMT_F16) {
    if (!q.meta || (q.group != 32 && q.group != 64 && q.group != 128) || q.group > d) return hipErrorInvalidValue;
  }
  // A grid dimension holds 2^32 - 1 work-items, and a row takes d / 8 of x: all
  // rows of a bulk call, one sequence's of an append, in whole workgroups (256
  // and 64 threads). That is 2^28 (d 128) and 2^29 rows (d 64), and row numbers
  // fit 31 bits below it.
  const int per_group = (q.positions ? 64 : 256) / (d / 8);
  const long long most = 0xffffffffLL / (d / 8) / per_group * per_group;
  const long long heads = q.positions ? q.Hkv : (long long)q.B * q.Hkv;
  if (heads > most || (!q.positions && heads * q.n > most)) return hipErrorInvalidValue;
  return d == 64 ? launch_format<64>(q, st) : launch_format<128>(q, st);
}

} // namespace
} // namespace gfx950
} // namespace kvf

extern "C" hipError_t kvf_quantize_place(int fmt, int group, int d, const float *x, int B,
                                         int Hkv, int n, int order, int block_tokens,
                                         const int *block_table, int max_blocks,
                                         unsigned char *data, void *meta, hipStream_t st) {
  return kvf::gfx950::quantize_rows({fmt, group, x, B, Hkv, n, nullptr, order, block_tokens, block_table, max_blocks,
                                     data, static_cast<uint32_t *>(meta)}, d, st);
}

extern "C" hipError_t kvf_append_tokens(int fmt, int group, int d, const float *x, int B, int Hkv,
                                        int n, const int *positions, int order,
                                        int block_tokens, const int *block_table,
                                        int max_blocks, unsigned char *data, void *meta,
                                        hipStream_t st) {
  if (!positions) return hipErrorInvalidValue;
  return kvf::gfx950::quantize_rows({fmt, group, x, B, Hkv, n, positions, order, block_tokens, block_table, max_blocks,
                                     data, static_cast<uint32_t *>(meta)}, d, st);
}
