// zh_move.hip -- nearest paints that move texels: inscribe, crop and nearest
// affine placements whose images all hold one format that decodes and encodes
// to the same bytes (native RGBA8 / BGRA8, linear RGBA16F and RGBA32F).  No
// texel is decoded: a pixel takes the bytes of the topmost layer that covers
// it, else of the base, and reads nothing else.
//
// A workgroup covers 64 columns x 16 rows, a wave 4 rows of 64 columns, so
// every load and store of an unscaled paint is one contiguous run per row.
// Maps are evaluated in FP64 as the interpreter's are (zh_device.h map_pt: the
// same contraction, and its division by 1 dropped), so coverage and texels are
// the same; an axis-aligned map's column coordinate is computed once for the
// lane's 4 rows.  The interpreter decoded base and layers for every pixel at
// two waves per SIMD, with four FP64 divisions a pixel: 143 us for a 1920x1080
// RGBA8 picture pasted into a 3840x2160 frame, 17.6 us here (66 MB, 3.8 TB/s).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "zh_any.h"

namespace zh {
namespace any {

template <int W> struct TexelT { typedef uint32_t type; };
template <> struct TexelT<2> { typedef w2 type; };
template <> struct TexelT<4> { typedef w4 type; };

// Halves pass through float, as decode and encode take them (a signalling NaN
// comes out quiet).
__device__ __forceinline__ uint32_t halves(uint32_t v) { return f2h(h2f(v & 0xffffu)) | (f2h(h2f(v >> 16)) << 16); }
template <int W>
__device__ __forceinline__ typename TexelT<W>::type canonical(typename TexelT<W>::type v) {
  if constexpr (W == 2) return w2{halves(v.x), halves(v.y)};
  else return v;
}

template <int W>
__device__ __forceinline__ typename TexelT<W>::type solid(CDesc d, uint32_t at, const Slot& o) {
  const uint4 v = encode_texel<true>(o, make_float4(d->params[at], d->params[at + 1], d->params[at + 2], d->params[at + 3]),
                                     (const Luts*)d->srgb_lut);
  if constexpr (W == 1) return v.x;
  else if constexpr (W == 2) return w2{v.x, v.y};
  else return w4{v.x, v.y, v.z, v.w};
}

// W: 32-bit words of a texel.
template <int W>
__global__ __launch_bounds__(kBlock) void k_move(const StageDesc* dd) {
  typedef typename TexelT<W>::type T;
  constexpr int kRows = 4;
  const CDesc d = as_const(dd);
  const Slot o = ldc(&d->slot[instr_slot(d, d->post_begin)]);
  const uint32_t X = blockIdx.x * 64 + (threadIdx.x & 63u);
  const uint32_t Y = blockIdx.y * 16 + (threadIdx.x >> 6) * kRows;
  const uint32_t wd = d->width, ht = d->height;
  // Per row: the texel's address, or none (a solid base, or past a source).
  uint64_t src[kRows];
  bool done[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    src[r] = 0;
    done[r] = false;
  }
  const double px = (double)(int)X + 0.5;
  for (uint32_t l = d->n_layers; l-- > 0;) {  // topmost first
    const Layer L = ldc(&d->layer[l]);
    const Slot s = ldc(&d->slot[instr_slot(d, L.prog_begin)]);
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const double py = (double)(int)(Y + r) + 0.5;
      const double u = fma(L.inv[0], px, L.inv[1] * py) + L.inv[2];
      const double v = fma(L.inv[3], px, L.inv[4] * py) + L.inv[5];
      const bool in = !done[r] && u >= L.cover[0] && u < L.cover[2] && v >= L.cover[1] && v < L.cover[3];
      if (in) {
        const int x = (int)floor(u), y = (int)floor(v);
        done[r] = true;
        src[r] = x >= 0 && y >= 0 && x < (int)s.width && y < (int)s.height
                     ? s.ptr + ((uint64_t)(uint32_t)y * s.row_stride + (uint64_t)(uint32_t)x * (4 * W))
                     : 0;
      }
    }
  }
  // The base where no layer covers.
  T fill{};
  T t[kRows];
  if (d->base_end > d->base_begin) {  // uniform
    if ((((CWords)&d->code[d->base_begin])[0] & 255u) == OP_LOAD) {
      const Slot s = ldc(&d->slot[instr_slot(d, d->base_begin)]);
#pragma unroll
      for (int r = 0; r < kRows; ++r)
        if (!done[r] && X < s.width && Y + r < s.height)
          src[r] = s.ptr + ((uint64_t)(Y + r) * s.row_stride + (uint64_t)X * (4 * W));
    } else {
      fill = solid<W>(d, d->code[d->base_begin].arg, o);
    }
  }
  const bool col = X < wd;
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    t[r] = done[r] ? T{} : fill;
    if (col && Y + r < ht && src[r]) t[r] = canonical<W>(nt_get<T>((const gbyte*)src[r]));
  }
#pragma unroll
  for (int r = 0; r < kRows; ++r)
    if (col && Y + r < ht) nt_put<T>((gbyte*)o.ptr + ((uint64_t)(Y + r) * o.row_stride + (uint64_t)X * (4 * W)), t[r]);
}

}  // namespace any
}  // namespace zh

extern "C" {

hipError_t zh_launch_move(int words, const zh::StageDesc* d_dev, uint32_t width, uint32_t height, hipStream_t stream) {
  const dim3 grid((width + 63) / 64, (height + 15) / 16), block(zh::kBlock);
  if (width == 0 || height == 0 || grid.y > 65535) return hipErrorInvalidValue;
  switch (words) {
    case 1: hipLaunchKernelGGL(zh::any::k_move<1>, grid, block, 0, stream, d_dev); break;
    case 2: hipLaunchKernelGGL(zh::any::k_move<2>, grid, block, 0, stream, d_dev); break;
    case 4: hipLaunchKernelGGL(zh::any::k_move<4>, grid, block, 0, stream, d_dev); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // extern "C"
