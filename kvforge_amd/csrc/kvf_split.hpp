// kvf_split.hpp - which tokens a split covers, for the launcher, the kernels
// and, compiled by itself, the host tests (no HIP here).
//
// Lengths are ints up to 2^31 - 1, and a last split's end or a chunk rounded up
// to tiles may lie past that, so all of it is worked out in 32 unsigned bits:
// splits * chunk stays below len + 2^16 * 33 < 2^32.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define KVF_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define KVF_HOST_DEVICE inline
#endif

namespace kvf {
namespace gfx950 {

constexpr int TT = 32; // tokens per tile (PV MFMA k)

// Tokens of a split of `len` tokens in contiguous chunks: the reference's
// ceil(len / splits) (runtime/kvf_kernels.cuh:147-150), or that rounded up to
// whole tiles.
KVF_HOST_DEVICE uint32_t split_chunk(int len, int splits, bool whole_tiles) {
  const uint32_t per = ((uint32_t)len + (uint32_t)splits - 1) / (uint32_t)splits;
  return whole_tiles ? (per + TT - 1) / TT * TT : per;
}

// Tokens [t0, t1) of split `split` in chunks of `chunk`; empty, at len, for the
// splits past the end.
struct TokenRange {
  int t0, t1;
};
KVF_HOST_DEVICE TokenRange split_range(int len, uint32_t chunk, int split) {
  const uint32_t at = (uint32_t)split * chunk, end = (uint32_t)len;
  const uint32_t t0 = at < end ? at : end;
  const uint32_t n = end - t0;
  return {(int)t0, (int)(t0 + (chunk < n ? chunk : n))};
}

// Tiles, aligned to absolute token positions, that the first `len` tokens touch.
KVF_HOST_DEVICE int tiles_of(int len) { return (int)(((uint32_t)len + TT - 1) / TT); }

} // namespace gfx950
} // namespace kvf
