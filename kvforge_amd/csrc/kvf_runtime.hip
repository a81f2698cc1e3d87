// kvf_runtime.hip - C-ABI entry points of libkvf_hip.so.
//
//   kvf_launch_variant / kvf_launch_varlen_variant / kvf_launch_partial_variant
//       dispatch a decode step by the reference's variant id
//       (src/codegen.cpp:59-65), the way bench/sweep.cu:180-186 does through
//       kvf::Registry;
//   kvf_launch_merge
//       the log-sum-exp merge alone.
// The KV append step's entry points are in kvf_quantize.hip.
#include "kvf_kernels.hpp"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

namespace kvf {
namespace gfx950 {
namespace {

Registry &registry() {
  static Registry reg;
  static std::once_flag once;
  std::call_once(once, [] { kvf_register_all(reg); });
  return reg;
}

LaunchXFn extended(const char *id) { return id ? registry().findx(id) : nullptr; }

// GQA pack size of a variant id ("_g{G}_"), 1 when absent.
int pack_of(const char *id) {
  const char *g = std::strstr(id, "_g");
  return g ? std::max(1, std::atoi(g + 2)) : 1;
}

// Whether `words` unsigned ints hold the fused step's merge counters for `a`
// (one KVF_COUNTER_STRIDE line per (sequence, head group)).
bool counters_fit(const char *id, const kvf_args_t &a, size_t words) {
  if (a.B < 1 || a.H < 1 || a.Hkv < 1) return false;
  const size_t groups = pack_of(id) > 1 ? (size_t)a.Hkv : (size_t)a.H;
  return words >= KVF_COUNTER_WORDS(a.B, groups);
}

Ext ext_of(const kvf_varlen_args_t *va) {
  Ext x;
  if (va) {
    x.seq_lens = va->seq_lens;
    x.q16 = static_cast<const _Float16 *>(va->q16);
    x.out16 = static_cast<_Float16 *>(va->out16);
    x.longest_first = (va->flags & KVF_VARLEN_LONGEST_FIRST) != 0;
  }
  return x;
}

std::vector<std::string> &variant_ids() {
  static std::vector<std::string> ids;
  static std::once_flag once;
  std::call_once(once, [] {
    for (const auto &kv : registry().fn) ids.push_back(kv.first);
    std::sort(ids.begin(), ids.end());
  });
  return ids;
}

} // namespace
} // namespace gfx950
} // namespace kvf

using namespace kvf;
using namespace kvf::gfx950;

extern "C" hipError_t kvf_launch_variant(const char *id, const kvf_args_t *a, hipStream_t st) {
  if (!a) return hipErrorInvalidValue;
  const LaunchFn fn = registry().find(id ? id : "");
  if (!fn) return hipErrorNotFound;
  return fn(*a, st);
}

extern "C" hipError_t kvf_launch_varlen_variant(const char *id, const kvf_args_t *a,
                                                const kvf_varlen_args_t *va, hipStream_t st) {
  if (!a) return hipErrorInvalidValue;
  const LaunchXFn fx = extended(id);
  if (!fx) return hipErrorNotFound;
  return fx(*a, ext_of(va), Launch{}, st);
}

extern "C" hipError_t kvf_launch_fused_variant(const char *id, const kvf_args_t *a,
                                               const kvf_varlen_args_t *va, unsigned *counters,
                                               size_t counter_words, hipStream_t st) {
  if (!a || !counters) return hipErrorInvalidValue;
  const LaunchXFn fx = extended(id);
  if (!fx) return hipErrorNotFound;
  if (!counters_fit(id, *a, counter_words)) return hipErrorInvalidValue;
  Ext x = ext_of(va);
  x.counters = counters;
  return fx(*a, x, Launch{}, st);
}

extern "C" hipError_t kvf_launch_persistent_variant(const char *id, const kvf_args_t *a,
                                                    const kvf_varlen_args_t *va, unsigned *counters,
                                                    size_t counter_words, unsigned *queue,
                                                    size_t queue_words, int workgroups, hipStream_t st) {
  if (!a || !queue || workgroups < 0) return hipErrorInvalidValue;
  const LaunchXFn fx = extended(id);
  if (!fx) return hipErrorNotFound;
  if (queue_words < KVF_QUEUE_WORDS) return hipErrorInvalidValue;
  if (counters && !counters_fit(id, *a, counter_words)) return hipErrorInvalidValue;
  Ext x = ext_of(va);
  x.counters = counters;
  x.queue = queue;
  x.slots = workgroups;
  return fx(*a, x, Launch{}, st);
}

// ---- the entry point that allocates nothing ----------------------------------
// The one-launch step's device memory beyond inputs and outputs (its merge
// counters and the split partials) lives in `scratch`, a file-scope device
// array of KVF_SCRATCH_BYTES that every GPU holds from module load until the
// process ends. In host code `scratch` names a host-side stand-in, not a
// device address: its address on each device comes from hipGetSymbolAddress,
// called once per device with that device current, and only that address is
// handed to kernels. Layout: [0, 64 KiB) merge counters (zero at load, and
// every completed step leaves them at zero again), then part_ml, then part_o,
// each 256-byte aligned. Calls that overlap on one GPU share the array and
// race.
static __device__ __align__(256) unsigned char scratch[KVF_SCRATCH_BYTES];

namespace {
constexpr size_t SCRATCH_COUNTERS = 64 * 1024;
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[MAX_DEVICES] = {};

hipError_t scratch_of_current_device(unsigned char **out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= MAX_DEVICES) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    g_scratch_ptr[dev] = p;
  }
  *out = static_cast<unsigned char *>(g_scratch_ptr[dev]);
  return hipSuccess;
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }
} // namespace

extern "C" hipError_t kvf_launch_fused_variant_noalloc(const char *id, const kvf_args_t *a,
                                                       const kvf_varlen_args_t *va,
                                                       hipStream_t st) {
  if (!a || a->B < 1 || a->H < 1 || a->Hkv < 1 || a->splits < 1) return hipErrorInvalidValue;
  const LaunchXFn fx = extended(id);
  if (!fx) return hipErrorNotFound;
  // counters: one per (sequence, head group); the pack size comes from the id
  const size_t counters = KVF_COUNTER_WORDS(a->B, pack_of(id) > 1 ? a->Hkv : a->H) * sizeof(unsigned);
  const size_t heads = (size_t)a->B * a->H * a->splits;
  const size_t d = std::strstr(id, "_d64") ? 64 : 128;
  const size_t ml_bytes = align256(heads * 2 * sizeof(float));
  const size_t o_bytes = align256(heads * d * sizeof(float));
  if (counters > SCRATCH_COUNTERS || SCRATCH_COUNTERS + ml_bytes + o_bytes > KVF_SCRATCH_BYTES)
    return hipErrorInvalidValue;
  unsigned char *base = nullptr;
  const hipError_t e = scratch_of_current_device(&base);
  if (e != hipSuccess) return e;
  kvf_args_t b = *a;
  b.part_ml = reinterpret_cast<float *>(base + SCRATCH_COUNTERS);
  b.part_o = reinterpret_cast<float *>(base + SCRATCH_COUNTERS + ml_bytes);
  Ext x = ext_of(va);
  x.counters = reinterpret_cast<unsigned *>(base);
  return fx(b, x, Launch{}, st);
}

extern "C" hipError_t kvf_launch_partial_variant(const char *id, const kvf_args_t *a,
                                                 hipStream_t st) {
  if (!a) return hipErrorInvalidValue;
  const LaunchXFn fx = extended(id);
  if (!fx) return hipErrorNotFound;
  if (!a->part_o || !a->part_ml) return hipErrorInvalidValue;
  Launch l;
  l.partial_only = true;
  return fx(*a, Ext{}, l, st);
}

extern "C" hipError_t kvf_launch_partial_variant_timed(const char *id, const kvf_args_t *a,
                                                       hipStream_t st, hipEvent_t start,
                                                       hipEvent_t stop) {
  if (!a) return hipErrorInvalidValue;
  const LaunchXFn fx = extended(id);
  if (!fx) return hipErrorNotFound;
  if (!a->part_o || !a->part_ml || !start || !stop) return hipErrorInvalidValue;
  Launch l;
  l.partial_only = true;
  l.ev_start = start;
  l.ev_stop = stop;
  return fx(*a, Ext{}, l, st);
}

extern "C" hipError_t kvf_launch_partial_varlen_variant_timed(const char *id, const kvf_args_t *a,
                                                              const kvf_varlen_args_t *va,
                                                              hipStream_t st, hipEvent_t start,
                                                              hipEvent_t stop) {
  if (!a) return hipErrorInvalidValue;
  const LaunchXFn fx = extended(id);
  if (!fx) return hipErrorNotFound;
  if (!a->part_o || !a->part_ml || !start || !stop) return hipErrorInvalidValue;
  Launch l;
  l.partial_only = true;
  l.ev_start = start;
  l.ev_stop = stop;
  return fx(*a, ext_of(va), l, st);
}

extern "C" hipError_t kvf_launch_step_timed(const char *id, const kvf_args_t *a,
                                            const kvf_varlen_args_t *va, unsigned *counters,
                                            size_t counter_words, hipStream_t st, hipEvent_t start,
                                            hipEvent_t stop) {
  if (!a || !start || !stop) return hipErrorInvalidValue;
  const LaunchXFn fx = extended(id);
  if (!fx) return hipErrorNotFound;
  if (counters && !counters_fit(id, *a, counter_words)) return hipErrorInvalidValue;
  Ext x = ext_of(va);
  x.counters = counters;
  Launch l;
  l.ev_start = start;
  l.ev_stop = stop;
  return fx(*a, x, l, st);
}

extern "C" hipError_t kvf_launch_merge(int d, const kvf_args_t *a, hipStream_t st) {
  if (!a || a->splits < 1 || a->B < 1 || a->H < 1 || !a->part_o || !a->part_ml || !a->out)
    return hipErrorInvalidValue;
  if (d == 128) return launch_merge_kernel<128>(*a, Ext{}, st);
  if (d == 64) return launch_merge_kernel<64>(*a, Ext{}, st);
  return hipErrorInvalidValue;
}

extern "C" int kvf_variant_count(void) { return (int)variant_ids().size(); }

extern "C" const char *kvf_variant_id(int i) {
  const auto &ids = variant_ids();
  return (i >= 0 && i < (int)ids.size()) ? ids[i].c_str() : nullptr;
}

extern "C" const char *kvf_version(void) { return "kvforge-mi355x 0.3 (gfx950, ABI 2)"; }

extern "C" int kvf_abi_version(void) { return KVF_ABI_VERSION; }
