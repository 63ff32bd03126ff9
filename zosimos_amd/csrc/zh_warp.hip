// zh_warp.hip -- the registered affine layer-stack kernels (zh_spec.h
// ZH_WARP_LIST): instantiations of the bodies in zh_warp_kernels.h, their
// registry and launchers.  Forms not registered here are compiled at run time
// from the same bodies (zh_jit.cpp).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cstring>

#include "zh_warp_kernels.h"

namespace zh {
namespace spec {

template <class V>
__global__ __launch_bounds__(kBlock, min_waves<V>()) void k_warp(const StageDesc* dd, uint32_t run) {
  warp_stage<V>(dd, run);
}

// Stages of at most one tile per compute unit: the kernel without a choice of path.
template <class V>
__global__ __launch_bounds__(kBlock) void k_warp_few(const StageDesc* dd, uint32_t run) {
  warp_stage<V, false>(dd, run);
}

template <class V>
__global__ __launch_bounds__(kBlock, min_waves<V>()) void k_warp_batch(const BatchDesc* bb, uint32_t run) {
  warp_batch<V>(bb, run);
}

// LDS-staged tiles of one-source separable forms (staged_tile).
template <class V>
__global__ __launch_bounds__(kBlock) void k_warp_staged(const StageDesc* dd, uint32_t) {
  warp_staged_stage<V>(dd);
}

template <class V>
__global__ __launch_bounds__(kBlock) void k_warp_staged_batch(const BatchDesc* bb, uint32_t) {
  warp_staged_batch<V>(bb);
}

// The registered forms have runs: zh_launch_warp deals them all so.
#define ZH_WARP_RUNS(name, src, f, mat, ...) static_assert(f != FMT_F32, #name);
ZH_WARP_LIST(ZH_WARP_RUNS)
#undef ZH_WARP_RUNS

template <class V>
constexpr void (*few_fn())(const StageDesc*, uint32_t) {
  if constexpr (warp_has_few(V::SRC, V::F)) return k_warp_few<V>;
  else return nullptr;
}
template <class V>
constexpr void (*staged_fn())(const StageDesc*, uint32_t) {
  if constexpr (V::SEP && V::SRC == WSRC_ONE) return k_warp_staged<V>;
  else return nullptr;
}
template <class V>
constexpr void (*staged_batch_fn())(const BatchDesc*, uint32_t) {
  if constexpr (V::SEP && V::SRC == WSRC_ONE) return k_warp_staged_batch<V>;
  else return nullptr;
}

// ---- registry ------------------------------------------------------------------
#define ZH_WARP_TYPE(name, src, f, mat, ...)                         \
  typedef Warp<src, f, mat != 0, Prog<__VA_ARGS__>, false> V_##name;    \
  typedef Warp<src, f, mat != 0, Prog<__VA_ARGS__>, true> VS_##name;    \
  static const uint16_t WP_##name[] = {__VA_ARGS__};
ZH_WARP_LIST(ZH_WARP_TYPE)
#undef ZH_WARP_TYPE

// Kernel index 2 i: form i with general affine maps; 2 i + 1: separable.
enum {
#define ZH_WARP_ENUM(name, ...) WI_##name, WIS_##name,
  ZH_WARP_LIST(ZH_WARP_ENUM)
#undef ZH_WARP_ENUM
  kNumWarps
};

struct WarpEntry {
  const char* name;
  uint32_t src, fmt, mat;
  const uint16_t* post;
  int n;
  void (*fn)(const StageDesc*, uint32_t);
  void (*few)(const StageDesc*, uint32_t);     // null: no such form
  void (*batch)(const BatchDesc*, uint32_t);
  void (*staged)(const StageDesc*, uint32_t);  // separable one-source forms: LDS-staged tiles
  void (*staged_batch)(const BatchDesc*, uint32_t);
};

#define ZH_WARP_ENTRY(name, src, f, mat, ...)                                                          \
  {#name, src, f, mat, WP_##name, (int)(sizeof(WP_##name) / sizeof(uint16_t)), k_warp<V_##name>,         \
   few_fn<V_##name>(), k_warp_batch<V_##name>, nullptr, nullptr},                                         \
  {#name "_sep", src, f, mat, WP_##name, (int)(sizeof(WP_##name) / sizeof(uint16_t)), k_warp<VS_##name>, \
   few_fn<VS_##name>(), k_warp_batch<VS_##name>, staged_fn<VS_##name>(), staged_batch_fn<VS_##name>()},
static const WarpEntry kWarps[] = {ZH_WARP_LIST(ZH_WARP_ENTRY)};
#undef ZH_WARP_ENTRY

}  // namespace spec
}  // namespace zh

extern "C" {

int zh_warp_lookup(uint32_t src, uint32_t fmt, uint32_t mat, const uint16_t* post, int n) {
  for (int i = 0; i < zh::spec::kNumWarps; i += 2) {
    const auto& e = zh::spec::kWarps[i];
    if (e.src == src && e.fmt == fmt && e.mat == mat && e.n == n &&
        std::memcmp(e.post, post, sizeof(uint16_t) * (size_t)n) == 0)
      return i;
  }
  return -1;
}

const char* zh_warp_name(int index) {
  return index >= 0 && index < zh::spec::kNumWarps ? zh::spec::kWarps[index].name : "";
}

int zh_warp_form_of(int index, uint32_t* src, uint32_t* fmt, uint32_t* mat, const uint16_t** post, int* n) {
  if (index < 0 || index >= zh::spec::kNumWarps) return 0;
  const auto& e = zh::spec::kWarps[index];
  *src = e.src;
  *fmt = e.fmt;
  *mat = e.mat;
  *post = e.post;
  *n = e.n;
  return 1;
}

int zh_warp_has_staged(int index) {
  return index >= 0 && index < zh::spec::kNumWarps && zh::spec::kWarps[index].staged != nullptr;
}

// Grid of a warp launch over `tiles` tiles, `resident` workgroups fitting a
// compute unit: blocks of run tiles for the dispatcher to balance, or a persistent
// grid (run 0): where asked for (the staged kernels' pipelined loop, forms without
// runs); per_cu workgroups per compute unit, which keeps more of each one's taps
// in the L1; and grids that are resident as a whole, where nothing is left to
// balance (two 640x480 layers rotated, 300 tiles, 6.65 us against 7.67 in runs).
// layers: of a stage whose kernel loads the 8-bit tables (0: none or a batch).
void zh_warp_grid(uint32_t tiles, uint32_t resident, uint32_t cus, uint32_t per_cu, int persistent, uint32_t layers,
                  uint32_t* blocks, uint32_t* run) {
  if (per_cu || persistent || tiles <= resident * cus) {
    *run = 0;
    *blocks = std::min(tiles, (per_cu ? std::min(per_cu, resident) : resident) * cus);
    return;
  }
  // Runs of up to 8 tiles, while that leaves 12 runs for every resident
  // workgroup: longer runs repeat less of the set-up (tables, the batch's
  // stage search) and share more source rows, shorter ones balance better.
  // 256-image batch (95 and 150 tiles per resident workgroup), run 1 / 4 / 8 /
  // 16: 1604 / 1340 / 1315 / 1327 us, persistent 1442; 8 layers at 3840x2160
  // (6 tiles per resident workgroup), run 1 / 2 / 4: 132 / 134 / 149 us,
  // persistent 150.
  *run = std::max(1u, std::min(8u, tiles / (12u * resident * cus)));
  // A run loads the tables anew, which one layer's taps do not hide: two tiles a
  // run from 2.5 per resident workgroup on (one RGBA16F layer to RGBA8 at 3840x2160,
  // 6.4: 35.4-36.6 us, in twos 32.3-33.8; 2560x1440, 2.8: 19.1 and 18.3-18.5).  Two
  // layers gain or lose by the map (3840x2160 RGBA8 49.6 and 50.9).
  if (layers == 1 && (uint64_t)tiles * 2 >= (uint64_t)resident * cus * 5) *run = std::max(*run, 2u);
  *blocks = (tiles + *run - 1) / *run;
}

hipError_t zh_launch_warp(int index, int staged, int few, const zh::StageDesc* d_dev, uint32_t tiles, uint32_t layers,
                          uint32_t cus, uint32_t per_cu, hipStream_t stream) {
  if (index < 0 || index >= zh::spec::kNumWarps) return hipErrorInvalidValue;
  const auto& e = zh::spec::kWarps[index];
  const auto fn = staged ? e.staged : few ? e.few : e.fn;
  if (!fn) return hipErrorInvalidValue;
  static uint32_t resident[2][zh::spec::kNumWarps] = {};
  uint32_t& res = resident[staged ? 1 : 0][index];
  if (!res) res = zh::resident_blocks((const void*)(staged ? e.staged : e.fn), 1);
  uint32_t blocks, run;
  zh_warp_grid(tiles, res, cus, per_cu, staged, layers, &blocks, &run);
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(fn, dim3(blocks), dim3(zh::kBlock), 0, stream, d_dev, run);
  return hipGetLastError();
}

hipError_t zh_launch_warp_batch(int index, int staged, const zh::BatchDesc* b_dev, uint32_t total_tiles,
                                uint32_t cus, uint32_t per_cu, hipStream_t stream) {
  if (index < 0 || index >= zh::spec::kNumWarps) return hipErrorInvalidValue;
  const auto& e = zh::spec::kWarps[index];
  if (staged && !e.staged_batch) return hipErrorInvalidValue;
  const auto fn = staged ? e.staged_batch : e.batch;
  static uint32_t resident[2][zh::spec::kNumWarps] = {};
  uint32_t& res = resident[staged ? 1 : 0][index];
  if (!res) res = zh::resident_blocks((const void*)fn, 1);
  uint32_t blocks, run;
  zh_warp_grid(total_tiles, res, cus, per_cu, staged, 0, &blocks, &run);
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(fn, dim3(blocks), dim3(zh::kBlock), 0, stream, b_dev, run);
  return hipGetLastError();
}

}  // extern "C"
