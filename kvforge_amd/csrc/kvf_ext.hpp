// kvf_ext.hpp - what travels beside kvf::Args into the gfx950 kernels, and the
// extended launcher every dispatch variant provides.
//
// Args stays byte-identical to the reference's (runtime/kvf_kernels.cuh:29-46);
// the variable-length / binary16 / fused-merge extension and the launch mode
// (split kernel only, kernel-bound timing events) are passed separately.
#pragma once

#include "kvf_abi.h"

#include <hip/hip_runtime.h>

namespace kvf {
namespace gfx950 {

// Ext::flags, the launch's form in one word that reaches the split kernel in
// a preloaded register (see decode_partial).
constexpr uint32_t KX_VARLEN = 1;      // per-sequence lengths
constexpr uint32_t KX_LPT = 2;         // longest first
constexpr uint32_t KX_Q16 = 4;         // binary16 query
constexpr uint32_t KX_HGDIV = 8;       // XCD-affine grid over more than one sequence
constexpr int KX_NX_SHIFT = 4;         // 4 bits: XCDs of an XCD-affine grid, 0 for (splits, head groups, B)
constexpr int KX_BS_SHIFT = 8;         // 4 bits: Args::block_shift
constexpr uint32_t KX_GQ1 = 1u << 12;  // one query head per KV head
constexpr int KX_MB_SHIFT = 13;        // 19 bits: Args::max_blocks, all ones when it is larger
constexpr uint32_t KX_MB_MAX = (1u << 19) - 1;

// Extension fields beside Args; all null by default.
struct Ext {
  const int *seq_lens = nullptr; // per-sequence lengths (Args::n is the maximum)
  const _Float16 *q16 = nullptr; // binary16 query instead of Args::q
  _Float16 *out16 = nullptr;     // binary16 output instead of Args::out
  bool longest_first = false;    // workgroup slots take sequences by decreasing length (B <= 64)
  unsigned *counters = nullptr;  // [B][head groups][KVF_COUNTER_STRIDE] split counters: fused merge
  // persistent step: [0] the item queue's claim counter, [KVF_COUNTER_STRIDE]
  // the count of workgroups done (both zero between calls); the grid is then
  // 1-D and `slots` caps it (0: as many workgroups as are resident at once)
  unsigned *queue = nullptr;
  int slots = 0;
  // fused step: the workgroups that do not merge run the merge code dry, to
  // bring it into the instruction cache for the one that does (set by the
  // launcher when the whole grid is resident at once)
  bool dry_merge = false;
  // set by the launcher from the fields above and Args: the query in the
  // format that KX_Q16 names, KX_* bits, and the tokens of a split (uniform
  // lengths)
  const void *q = nullptr;
  uint32_t flags = 0;
  uint32_t chunk = 0;
};

// How a decode step is enqueued: the split kernel alone (partial_only), and
// optionally with HIP events bound to the split kernel's own dispatch
// (hipExtLaunchKernelGGL), which time the kernel itself rather than the
// stream around it.
struct Launch {
  bool partial_only = false;
  hipEvent_t ev_start = nullptr;
  hipEvent_t ev_stop = nullptr;
};

// Extended launcher of one variant (defined in kvf_kernels.hpp, explicitly
// instantiated per variant by the generated kvf_inst_*.hip files).
template <int FMT, int D, int G, int U, int ORD, bool PAGED>
hipError_t launch_ext(const Args &a, const Ext &x, const Launch &l, hipStream_t st);

} // namespace gfx950
} // namespace kvf
