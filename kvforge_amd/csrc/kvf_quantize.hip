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
  uint32_t rows;        // B * Hkv * (n, or 1 when appending)
  int n, Hkv, order, bt, max_blocks;
  FastDiv inner, outer; // sizes of the two inner dimensions of a work item
  FastDiv page;         // bt (1 for contiguous)
  const int *table;
  const int *positions; // append: sequence b's token; null: tokens 0..n-1
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

// A wave takes R * 512 / D neighbouring work items; all their loads go out
// before the first is used. The items' (sequence, head, token) come from one
// scalar division per load of a wave, its first item's, and a carry per lane
// (per-lane divisions were as many cycles as the quantizing).
// Measured on MI355X, K and V of one layer with 8 KV heads of 128: 32768
// tokens in int8:64, head-major contiguous, 339 -> 68 us (5.0 TB/s read and
// written, a large copy's 5.2); 4 x 4093 tokens in int4:32, paged token-major,
// 180 -> 36 us (4.3 TB/s). Before, a wave took one row, a lane single elements
// with byte stores, and every element one division. Appending one token to
// each of 4 sequences (16 calls in a graph of 8 layers' steps): the graph
// 154 -> 126 us.
template <int FMT, int D, int GQ, int R>
__global__ void __launch_bounds__(256)
quantize_place_kernel(const float *__restrict__ x, unsigned char *__restrict__ data, uint32_t *__restrict__ meta,
                      const Place p) {
  constexpr int LPR = D / 8;         // lanes per row
  constexpr int RPW = 64 / LPR;      // rows per wave and load
  constexpr int ROW = D * bits_of<FMT>() / 8;
  const int lane = threadIdx.x & 63;
  const uint32_t wave = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane % LPR;          // the lane's elements are [8c, 8c + 8)
  bool ok[R];
  uint32_t b[R], h[R], t[R], item[R];
  int page[R];
  f4u v[R][2];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const uint32_t i0 = (wave * R + j) * RPW, o = lane / LPR;
    ok[j] = i0 + o < p.rows;
    // past the end: the last row again, loaded and not stored
    const uint32_t i = item[j] = ok[j] ? i0 + o : p.rows - 1;
    uint32_t in, mid;
    if (p.inner.div >= RPW && i0 + RPW <= p.rows) {
      const uint32_t rest0 = p.inner.quot(i0), b0 = p.outer.quot(rest0);
      in = i0 - rest0 * p.inner.div + o;
      mid = rest0 - b0 * p.outer.div;
      b[j] = b0;
      if (in >= p.inner.div) {
        in -= p.inner.div;
        ++mid;
      }
      if (mid >= p.outer.div) {
        mid = 0;
        ++b[j];
      }
    } else {
      const uint32_t rest = p.inner.quot(i);
      in = i - rest * p.inner.div;
      b[j] = p.outer.quot(rest);
      mid = rest - b[j] * p.outer.div;
    }
    // appending, the inner dimension is the heads and the outer one is 1
    const bool head_inner = p.positions || p.order != ORD_HEAD;
    h[j] = head_inner ? in : mid;
    t[j] = head_inner ? mid : in;
  }
#pragma unroll
  for (int j = 0; j < R; ++j) {
    // logical row (b Hkv + h) n + t; head-major and appended rows are in that order already
    const uint32_t src = p.positions || p.order == ORD_HEAD ? item[j] : (b[j] * p.Hkv + h[j]) * p.n + t[j];
    const float *xr = x + (long long)src * D + c * 8;
    v[j][0] = *reinterpret_cast<const f4u *>(xr);
    v[j][1] = *reinterpret_cast<const f4u *>(xr + 4);
  }
  if (p.positions) {
#pragma unroll
    for (int j = 0; j < R; ++j) {
      // a position outside the layout writes nothing
      const int pos = p.positions[b[j]];
      const bool in = pos >= 0 && pos < (p.bt ? p.max_blocks * p.bt : p.n);
      ok[j] = ok[j] && in;
      t[j] = in ? (uint32_t)pos : 0u;
    }
  }
  if (p.bt) {
#pragma unroll
    for (int j = 0; j < R; ++j) page[j] = p.table[(long long)b[j] * p.max_blocks + p.page.quot(t[j])];
  }
#pragma unroll
  for (int j = 0; j < R; ++j) {
    // a row's lanes leave together (the group reductions stay inside a row)
    if (!ok[j]) continue;
    long long prow; // the physical row
    if (p.bt) {
      const uint32_t in = t[j] - p.page.quot(t[j]) * p.bt;
      prow = (long long)page[j] * (p.Hkv * p.bt) + (p.order == ORD_HEAD ? h[j] * p.bt + in : in * p.Hkv + h[j]);
    } else if (p.positions) {
      prow = p.order == ORD_HEAD ? (long long)item[j] * p.n + t[j] : ((long long)b[j] * p.n + t[j]) * p.Hkv + h[j];
    } else {
      prow = item[j];
    }
    float e[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) e[k] = v[j][k / 4][k % 4];
    unsigned char *to = data + prow * ROW + c * (8 * bits_of<FMT>() / 8);
    if constexpr (FMT == FMT_F16) {
      u4u w;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        w[k] = __builtin_bit_cast(uint32_t, (half2_t){(_Float16)e[2 * k], (_Float16)e[2 * k + 1]});
      *reinterpret_cast<u4u *>(to) = w;
    } else {
      constexpr float LEVELS = FMT == FMT_INT8 ? 255.f : 15.f;
      constexpr int LPG = GQ / 8; // lanes per group
      auto mn = [](float a, float b) { return fminf(a, b); };
      auto mx = [](float a, float b) { return fmaxf(a, b); };
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
        *reinterpret_cast<u2u *>(to) = w;
      } else {
        uint32_t w = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) w |= q[k] << (4 * k); // even elements in the low nibble
        *reinterpret_cast<u1u *>(to) = w;
      }
    }
  }
}

template <int FMT, int D, int GQ>
hipError_t launch_quantize(const float *x, unsigned char *data, uint32_t *meta, const Place &p, hipStream_t st) {
  // 4 loads a lane in flight where the rows give every SIMD of the chip two
  // waves of them; fewer rows spread over more waves
  constexpr uint32_t RPW = 64 / (D / 8);
  if (p.rows >= 2048u * 4 * RPW) {
    const dim3 grid((p.rows + 16 * RPW - 1) / (16 * RPW));
    hipLaunchKernelGGL((quantize_place_kernel<FMT, D, GQ, 4>), grid, dim3(256), 0, st, x, data, meta, p);
  } else {
    const dim3 grid((p.rows + 4 * RPW - 1) / (4 * RPW));
    hipLaunchKernelGGL((quantize_place_kernel<FMT, D, GQ, 1>), grid, dim3(256), 0, st, x, data, meta, p);
  }
  return hipGetLastError();
}

template <int D>
hipError_t launch_format(int fmt, int group, const float *x, unsigned char *data, uint32_t *meta, const Place &p,
                         hipStream_t st) {
  switch (fmt) {
  case FMT_F16:
    return launch_quantize<FMT_F16, D, D>(x, data, meta, p, st);
  case FMT_INT8:
    if (group == 32) return launch_quantize<FMT_INT8, D, 32>(x, data, meta, p, st);
    if (group == 64) return launch_quantize<FMT_INT8, D, 64>(x, data, meta, p, st);
    return launch_quantize<FMT_INT8, D, D>(x, data, meta, p, st);
  case FMT_INT4:
    if (group == 32) return launch_quantize<FMT_INT4, D, 32>(x, data, meta, p, st);
    if (group == 64) return launch_quantize<FMT_INT4, D, 64>(x, data, meta, p, st);
    return launch_quantize<FMT_INT4, D, D>(x, data, meta, p, st);
  default:
    return hipErrorInvalidValue;
  }
}

hipError_t quantize_rows(int fmt, int group, int d, const float *x, int B, int Hkv, int n,
                         const int *positions, int order, int block_tokens,
                         const int *block_table, int max_blocks, unsigned char *data,
                         void *meta, hipStream_t st) {
  if (!x || !data || B < 1 || Hkv < 1 || n < 1 || (d != 64 && d != 128)) return hipErrorInvalidValue;
  if (order != ORD_HEAD && order != ORD_TOKEN) return hipErrorInvalidValue;
  if (block_tokens < 0 || (block_tokens > 0 && (!block_table || max_blocks * block_tokens < n)))
    return hipErrorInvalidValue;
  if (fmt != FMT_F16) {
    if (!meta || (group != 32 && group != 64 && group != 128) || group > d) return hipErrorInvalidValue;
  }
  const long long rows = (long long)B * Hkv * (positions ? 1 : n);
  // work items are 31-bit (a grid of one row per 64 threads ended at 2^26 rows)
  if (rows > 0x7fffffffLL) return hipErrorInvalidValue;
  Place p;
  p.rows = (uint32_t)rows;
  p.n = n;
  p.Hkv = Hkv;
  p.order = order;
  p.bt = block_tokens;
  p.max_blocks = max_blocks;
  p.inner = FastDiv(positions ? Hkv : order == ORD_HEAD ? n : Hkv);
  p.outer = FastDiv(positions ? 1 : order == ORD_HEAD ? Hkv : n);
  p.page = FastDiv(block_tokens ? block_tokens : 1);
  p.table = block_table;
  p.positions = positions;
  uint32_t *m = static_cast<uint32_t *>(meta);
  return d == 64 ? launch_format<64>(fmt, group, x, data, m, p, st)
                 : launch_format<128>(fmt, group, x, data, m, p, st);
}

} // namespace
} // namespace gfx950
} // namespace kvf

extern "C" hipError_t kvf_quantize_place(int fmt, int group, int d, const float *x, int B,
                                         int Hkv, int n, int order, int block_tokens,
                                         const int *block_table, int max_blocks,
                                         unsigned char *data, void *meta, hipStream_t st) {
  return kvf::gfx950::quantize_rows(fmt, group, d, x, B, Hkv, n, nullptr, order, block_tokens, block_table,
                                    max_blocks, data, meta, st);
}

extern "C" hipError_t kvf_append_tokens(int fmt, int group, int d, const float *x, int B, int Hkv,
                                        int n, const int *positions, int order,
                                        int block_tokens, const int *block_table,
                                        int max_blocks, unsigned char *data, void *meta,
                                        hipStream_t st) {
  if (!positions) return hipErrorInvalidValue;
  return kvf::gfx950::quantize_rows(fmt, group, d, x, B, Hkv, n, positions, order, block_tokens, block_table,
                                    max_blocks, data, meta, st);
}
