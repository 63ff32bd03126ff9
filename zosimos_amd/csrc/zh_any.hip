// zh_any.hip -- pointwise stages of the common shapes in any texel format and
// row pitch: conversions (with or without a 3x3 matrix) and the 'over' of two
// images.  Formats within a class of slots are uniform arguments (zh_any.h),
// so no compile and no registration stands between a format pair and its
// kernel.  They stream: measured (and on the interpreter they replace) 26.6 us
// (221) for 10-bit Bt.2020 to RGBA16F and 29.9 us (139) for RGBA16F to 16-bit
// sRGB at 3840x2160, 3.7 and 4.4 TB/s; 13.5 us (64) for the 'over' of two
// 1919x1079 RGBA8 images with padded rows, of which some 6 us are the launch
// and the tables.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>

#include "zh_any.h"

namespace zh {
namespace any {

// A lane's group: where its texels are, and the codes of its loads.
struct Group {
  uint64_t x0, y;
  int n;
  Codes a, b;
};

__device__ __forceinline__ const gbyte* texels(const Src& s, const Group& g) {
  return (const gbyte*)s.ptr + (g.y * s.stride + g.x0 * s.bpp);
}

template <int A, int B>
__device__ __forceinline__ void fetch(const Src& a, const Src& b, Group& g) {
  if (A != SRC_F32 && a.bpp != 16) load_group(texels(a, g), a.bpp, g.n, g.a);
  if constexpr (B >= 0)
    if (B != SRC_F32 && b.bpp != 16) load_group(texels(b, g), b.bpp, g.n, g.b);
}

// The colour of the group under the shape's program.  The arithmetic is the
// interpreter's, instruction by instruction (zh_kernels.hip run()).
template <int A, int B, bool POW>
__device__ __forceinline__ void colour(const Src& a, const Src& b, bool mat, const float* m, const Group& g, Px& X,
                                       const float* ta, const float* tb) {
  decode_group<A, POW>(a, texels(a, g), g.n, g.a, X, ta);
  if constexpr (B >= 0) {
    Px U;
    decode_group<B, POW>(b, texels(b, g), g.n, g.b, U, tb);
#pragma unroll
    for (int i = 0; i < kPix; ++i) {
      const float4 dn = make_float4(X[i].x * X[i].w, X[i].y * X[i].w, X[i].z * X[i].w, X[i].w);
      const float4 up = make_float4(U[i].x * U[i].w, U[i].y * U[i].w, U[i].z * U[i].w, U[i].w);
      const float k = 1.0f - up.w;
      const float4 v = make_float4(fmaf(dn.x, k, up.x), fmaf(dn.y, k, up.y), fmaf(dn.z, k, up.z), fmaf(dn.w, k, up.w));
      const float r = v.w > 0.0f ? __builtin_amdgcn_rcpf(v.w) : 0.0f;
      X[i] = make_float4(v.x * r, v.y * r, v.z * r, v.w);
    }
  }
  if (mat) {  // uniform
#pragma unroll
    for (int i = 0; i < kPix; ++i) {
      const float r = row3(m, X[i]), gr = row3(m + 3, X[i]), bl = row3(m + 6, X[i]);
      X[i] = make_float4(r, gr, bl, X[i].w);
    }
  }
}

// A persistent grid striding over the stage's groups of kPix texels: the
// whole image as one row when every slot is tight (flat), else
// ceil(width / kPix) groups a row, the last of a row partial.  A lane's next
// loads are issued once its codes are decoded, the first ones before the
// workgroup fills its tables.
// A, B: classes of the loads (B -1: none); D: class of the store; POW:
// transfers of power functions per pixel.
template <int A, int B, int D, bool POW>
__global__ __launch_bounds__(kBlock) void k_any(const StageDesc* dd) {
  const CDesc d = as_const(dd);
  __shared__ float ta[has_table(A) ? kTable : 1];
  __shared__ float tb[has_table(B) ? kTable : 1];
  __shared__ typename LutOf<D == DST_U8>::type lut_mem;
  Luts* const luts = (Luts*)&lut_mem;
  const uint32_t last = d->n_instr - 1;
  const Src a = source<A>(ldc(&d->slot[instr_slot(d, 0)]), &d->table[0]);
  const Src b = B >= 0 ? source<B>(ldc(&d->slot[instr_slot(d, 2)]), &d->table[1]) : a;
  const Dst o = target<D>(ldc(&d->slot[instr_slot(d, last)]));
  const bool flat = d->flat != 0;
  const uint64_t w = flat ? (uint64_t)d->width * d->height : d->width;
  const uint32_t gpr = (uint32_t)((w + kPix - 1) / kPix);
  const uint32_t groups = flat ? gpr : gpr * d->height;  // below 2^32 (the planner's check)
  const uint32_t stride = gridDim.x * kBlock;
  auto at = [&](uint32_t g, Group& r) {
    const uint32_t y = flat ? 0u : g / gpr;
    r.y = y;
    r.x0 = (uint64_t)(g - y * gpr) * kPix;
    r.n = r.x0 + kPix <= w ? kPix : (int)(w - r.x0);
  };
  Group r;
  uint32_t g = blockIdx.x * kBlock + threadIdx.x;
  const bool any = g < groups;
  if (any) {
    at(g, r);
    fetch<A, B>(a, b, r);
  }
  const bool mat = last == (B >= 0 ? 7u : 2u);
  const uint32_t mq = mat ? d->code[last - 1].arg : 0u;
  float m[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) m[k] = d->params[mq + k];
  fill_table<A>(a, d, ta);
  if constexpr (B >= 0) fill_table<B>(b, d, tb);
  if constexpr (D == DST_U8) {
    if (o.transfer == 5) load_lut(d, luts);
  }
  __syncthreads();
  if (!any) return;
  while (true) {
    Px X;
    colour<A, B, POW>(a, b, mat, m, r, X, ta, tb);
    gbyte* const q = (gbyte*)o.ptr + (r.y * o.stride + r.x0 * o.bpp);
    const int n = r.n;
    const bool more = groups - g > stride;
    if (more) {
      g += stride;
      at(g, r);
      fetch<A, B>(a, b, r);
    }
    put_group<D, POW>(o, q, n, X, luts);
    if (!more) break;
  }
}

typedef void (*Kernel)(const StageDesc*);

// Kernel of a shape (zh_stage.h AnyShape): conversions for every pair of
// classes; the 'over' of two images for tables and half floats in any mix into
// 8-bit and float targets, the rest through SRC_ANY.  Power functions are
// carried only where a class can need them.
template <int A, int B, int D>
Kernel pick(bool pow) {
  if constexpr (A >= SRC_WIDE || D >= DST_CODE) {
    if (pow) return k_any<A, B, D, true>;
  }
  return k_any<A, B, D, false>;
}
template <int A, int B>
Kernel pick(int dst, bool pow) {
  switch (dst) {
    case DST_U8: return pick<A, B, DST_U8>(pow);
    case DST_F16: return pick<A, B, DST_F16>(pow);
    case DST_F32: return pick<A, B, DST_F32>(pow);
    case DST_CODE: return pick<A, B, DST_CODE>(pow);
    default: return pick<A, B, DST_WIDE>(pow);
  }
}
template <int A, int B>
Kernel pick_plain(int dst) {
  return dst == DST_U8 ? k_any<A, B, DST_U8, false> : dst == DST_F16 ? k_any<A, B, DST_F16, false>
                                                                    : k_any<A, B, DST_F32, false>;
}
static Kernel kernel_of(uint32_t shape) {
  const int a = (int)any_src(shape, 0), b = (int)any_src(shape, 1), dst = (int)any_dst(shape);
  const bool pow = (shape & ANY_POW) != 0;
  if (!(shape & ANY_OVER)) {
    switch (a) {
      case SRC_TABLE: return pick<SRC_TABLE, -1>(dst, pow);
      case SRC_F16: return pick<SRC_F16, -1>(dst, pow);
      case SRC_F32: return pick<SRC_F32, -1>(dst, pow);
      default: return pick<SRC_WIDE, -1>(dst, pow);
    }
  }
  if (dst < DST_CODE) {
    if (a == SRC_TABLE && b == SRC_TABLE) return pick_plain<SRC_TABLE, SRC_TABLE>(dst);
    if (a == SRC_TABLE && b == SRC_F16) return pick_plain<SRC_TABLE, SRC_F16>(dst);
    if (a == SRC_F16 && b == SRC_TABLE) return pick_plain<SRC_F16, SRC_TABLE>(dst);
    if (a == SRC_F16 && b == SRC_F16) return pick_plain<SRC_F16, SRC_F16>(dst);
  }
  return pick<SRC_ANY, SRC_ANY>(dst, pow);
}

}  // namespace any
}  // namespace zh

extern "C" {

hipError_t zh_launch_any(uint32_t shape, const zh::StageDesc* d_dev, uint32_t width, uint32_t height, int flat,
                         uint32_t cus, hipStream_t stream) {
  if (shape >= zh::kAnyShapes) return hipErrorInvalidValue;
  static std::atomic<uint32_t> resident[zh::kAnyShapes];
  const zh::any::Kernel fn = zh::any::kernel_of(shape);
  uint32_t res = resident[shape].load(std::memory_order_relaxed);
  if (!res) {
    res = zh::resident_blocks((const void*)fn, 1);
    resident[shape].store(res, std::memory_order_relaxed);
  }
  const uint64_t gpr = ((flat ? (uint64_t)width * height : width) + zh::kPix - 1) / zh::kPix;
  const uint64_t groups = flat ? gpr : gpr * height;
  if (groups >= (1ull << 32)) return hipErrorInvalidValue;
  const uint64_t blocks = std::min<uint64_t>((groups + zh::kBlock - 1) / zh::kBlock, (uint64_t)res * cus);
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(fn, dim3((uint32_t)blocks), dim3(zh::kBlock), 0, stream, d_dev);
  return hipGetLastError();
}

}  // extern "C"
