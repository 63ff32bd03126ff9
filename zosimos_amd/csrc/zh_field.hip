// zh_field.hip -- stages whose value depends on the pixel's place: the 3x3
// filter (box3.frag), fractal noise, the bilinear and normal-distribution
// generators, and the palette lookup at a generated coordinate (resize).  One
// kernel per operation and class of slots (zh_any.h); the arithmetic is the
// interpreter's (zh_kernels.hip run()), so the outputs are the same bytes.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>

#include "zh_any.h"
#include "zh_field.h"

namespace zh {
namespace any {

typedef const __attribute__((address_space(4))) float* CParams;

// ---- 3x3 filter ------------------------------------------------------------------
// A lane filters 4 columns of a strip of rows, one input row at a time.  A row
// adds its part to three outputs: it is the last row of the one above, the
// middle row of its own and the first row of the one below, which is the
// order the weighted sum runs in, so two partial sums a pixel carry it (24
// registers) and every texel is loaded and decoded once per strip (plus the
// lane's two neighbour columns).  The interpreter fetched and decoded 9 texels
// a pixel: 237 us for a 3840x2160 RGBA8 frame, 31 us here, bound by the vector
// instructions (280 a wave and row) and their latency at 5 waves a SIMD.
template <int S>
struct Row {
  Codes mid;                 // the lane's group
  uint32_t l[2], r[2];       // the columns left and right of it
};

// The texels of row y around the group at x0 (columns clamped to the image).
template <int S>
__device__ __forceinline__ void fetch_row(const Src& s, uint32_t x0, int n, uint32_t w, uint32_t y, Row<S>& t) {
  if (S == SRC_F32 || s.bpp == 16) return;
  const gbyte* row = (const gbyte*)s.ptr + (uint64_t)y * s.stride;
  load_group(row + (uint64_t)x0 * s.bpp, s.bpp, n, t.mid);
  const uint32_t xl = x0 ? x0 - 1 : 0u, xr = min(x0 + kPix, w - 1);
  load_code(row + (uint64_t)xl * s.bpp, s.bpp, t.l[0], t.l[1]);
  load_code(row + (uint64_t)xr * s.bpp, s.bpp, t.r[0], t.r[1]);
}

// Colours of the six columns x0 - 1 .. x0 + 4 of row y.  (In a row's last group
// load_group repeats the last texel for the columns past the image.)
template <int S, bool POW>
__device__ __forceinline__ void decode_row(const Src& s, uint32_t x0, int n, uint32_t w, uint32_t y, const Row<S>& t,
                                           float3* c, const float* tab) {
  Px X;
  const gbyte* row = (const gbyte*)s.ptr + (uint64_t)y * s.stride;
  decode_group<S, POW>(s, row + (uint64_t)x0 * s.bpp, n, t.mid, X, tab);
#pragma unroll
  for (int i = 0; i < kPix; ++i) c[1 + i] = make_float3(X[i].x, X[i].y, X[i].z);
  // The two outer columns as one more (half used) group.
  Codes e;
  e.lo[0] = t.l[0]; e.hi[0] = t.l[1];
  e.lo[1] = t.r[0]; e.hi[1] = t.r[1];
  e.lo[2] = e.lo[3] = e.hi[2] = e.hi[3] = 0u;
  if (S == SRC_F32 || s.bpp == 16) {
    const uint32_t xl = x0 ? x0 - 1 : 0u, xr = min(x0 + kPix, w - 1);
    X[0] = f4_bits(gld<w4>(row + (uint64_t)xl * 16));
    X[1] = f4_bits(gld<w4>(row + (uint64_t)xr * 16));
    X[2] = X[3] = X[0];
  }
  decode_codes<S, POW>(s, e, X, tab);
  c[0] = make_float3(X[0].x, X[0].y, X[0].z);
  c[5] = make_float3(X[1].x, X[1].y, X[1].z);
}

// acc += the three columns of kernel row w on every pixel.  A derivative has
// three zero weights; a zero times a finite colour adds nothing (no sum here
// is -0: each starts at +0), so integer texels skip them where their transfer
// decodes every code to a finite value.
template <bool TABLE>
__device__ __forceinline__ void add_row(const float* w, bool finite, const float3* c, float3* acc) {
#pragma unroll
  for (int dx = 0; dx < 3; ++dx) {
    if (TABLE && finite && w[dx] == 0.0f) continue;  // uniform
#pragma unroll
    for (int i = 0; i < kPix; ++i) {
      acc[i].x = fmaf(w[dx], c[i + dx].x, acc[i].x);
      acc[i].y = fmaf(w[dx], c[i + dx].y, acc[i].y);
      acc[i].z = fmaf(w[dx], c[i + dx].z, acc[i].z);
    }
  }
}

template <int S, int D, bool POW>
__global__ __launch_bounds__(kBlock) void k_box3(const StageDesc* dd, uint32_t rows) {
  const CDesc d = as_const(dd);
  __shared__ float tab[has_table(S) ? kTable : 1];
  __shared__ typename LutOf<D == DST_U8>::type lut_mem;
  Luts* const luts = (Luts*)&lut_mem;
  const Src s = source<S>(ldc(&d->slot[instr_slot(d, 0)]), &d->table[0]);
  const Dst o = target<D>(ldc(&d->slot[instr_slot(d, 1)]));
  const uint32_t W = d->width, H = d->height, gpr = (W + kPix - 1) / kPix;
  const uint32_t strips = (H + rows - 1) / rows;
  const uint32_t g = blockIdx.x * kBlock + threadIdx.x;  // fewer than 2^32 groups (the planner's check)
  const uint32_t strip = g / gpr, x0 = (g - strip * gpr) * kPix;
  const bool any = strip < strips;
  const int n = (int)min((uint32_t)kPix, W - x0);
  const uint32_t y0 = strip * rows, y1 = min(y0 + rows, H);
  Row<S> t;
  if (any) fetch_row<S>(s, x0, n, W, y0 ? y0 - 1 : 0u, t);
  float w[9];
  const uint32_t q = d->code[0].arg;
#pragma unroll
  for (int k = 0; k < 9; ++k) w[k] = d->params[q + k];
  fill_table<S>(s, d, tab);
  if constexpr (D == DST_U8) {
    if (o.transfer == 5) load_lut(d, luts);
  }
  __syncthreads();
  if (!any) return;
  const bool finite = s.transfer != 3;  // (SMPTE 240: NaN between its segments)
  float3 first[kPix], second[kPix];     // sums over one and two rows
#pragma unroll
  for (int i = 0; i < kPix; ++i) first[i] = second[i] = make_float3(0.0f, 0.0f, 0.0f);
  // Input rows y0 - 1 .. y1 (clamped to the image); row y completes output y - 1.
  for (uint32_t k = 0; k <= y1 - y0 + 1; ++k) {
    const uint32_t y = min(y0 + k ? y0 + k - 1 : 0u, H - 1);
    float3 c[kPix + 2];
    decode_row<S, POW>(s, x0, n, W, y, t, c, tab);
    if (k <= y1 - y0) fetch_row<S>(s, x0, n, W, min(y0 + k, H - 1), t);
    add_row<S == SRC_TABLE>(w + 6, finite, c, second);
    Px X;
#pragma unroll
    for (int i = 0; i < kPix; ++i) X[i] = make_float4(second[i].x, second[i].y, second[i].z, 1.0f);
    add_row<S == SRC_TABLE>(w + 3, finite, c, first);
#pragma unroll
    for (int i = 0; i < kPix; ++i) {
      second[i] = first[i];
      first[i] = make_float3(0.0f, 0.0f, 0.0f);
    }
    add_row<S == SRC_TABLE>(w, finite, c, first);
    if (k >= 2)
      put_group<D, POW>(o, (gbyte*)o.ptr + ((uint64_t)(y0 + k - 2) * o.stride + (uint64_t)x0 * o.bpp), n, X, luts);
  }
}

// ---- generators --------------------------------------------------------------------
// bilinear.frag at the pixel centre of column x, row coordinate v; mix(a, b, t)
// is evaluated as a + (b - a) t, exact where a = b.
__device__ __forceinline__ float4 grid_value(CParams q, float u, float v) {
  const float uv = u * v;
  float r[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    r[k] = fmaf(q[4 + k] - q[k], u, q[k]) + fmaf(q[12 + k] - q[8 + k], v, q[8 + k]) +
           fmaf(q[20 + k] - q[16 + k], uv, q[16 + k]);
  return make_float4(r[0], r[1], r[2], r[3]);
}

// Noise corners cached in LDS: the tile of 64 x 16 pixels a workgroup works on
// meets few cells of the low octaves (a cell is many pixels wide), and its
// pixels share their corners.  The cells that the tile can meet are hashed once, a
// corner per lane, in batches of the octaves that fit the cache together, with
// the difference to the corner below that the blend takes; the hash is 10
// quarter-rate multiplies a corner, four corners a pixel and octave without the
// cache: 92 us for four octaves at 2048x2048, 50 with it, bound by the blend's
// vector instructions.  Octaves whose box does not fit (cells smaller than a
// pixel) hash directly, as does a lane with a pixel whose rounded coordinate
// falls outside the box.
constexpr uint32_t kCorners = 1024;  // 32 KB of values and differences
constexpr uint32_t kBoxes = 8;       // octaves cached

struct NoiseBox {
  int32_t x, y;   // first cell
  uint32_t w, h;  // corners a row (one more than cells), rows of cells (one less than of corners)
  // Its corners in the cache, [at, end), while its batch is there.  A box of
  // no cells (w = h = 0) is not cached.
  uint32_t at, end;
};

// v += amp (mix of the cell's corners): a, da the left corner's value and
// difference, b, db the right's.
__device__ __forceinline__ float4 blend_cell(float4 v, float4 a, float4 da, float4 b, float4 db, float ux, float uy,
                                             float amp) {
#pragma clang fp contract(off)
  const float vx = 1.0f - ux;
  v.x = v.x + amp * (a.x * vx + b.x * ux + da.x * uy * vx + db.x * ux * uy);
  v.y = v.y + amp * (a.y * vx + b.y * ux + da.y * uy * vx + db.y * ux * uy);
  v.z = v.z + amp * (a.z * vx + b.z * ux + da.z * uy * vx + db.z * ux * uy);
  v.w = v.w + amp * (a.w * vx + b.w * ux + da.w * uy * vx + db.w * ux * uy);
  return v;
}

// The corner (cx, cy) and the difference to the one below.
__device__ __forceinline__ void corner_at(uint32_t cx, uint32_t cy, float4& v, float4& dv) {
#pragma clang fp contract(off)
  v = cell_value(cx, cy);
  const float4 c = cell_value(cx, cy + 1u);
  dv = make_float4(c.x - v.x, c.y - v.y, c.z - v.z, c.w - v.w);
}

// The next octave's coordinates (fractal_noise.frag's rotation and doubling).
__device__ __forceinline__ void next_octave(float& x, float& y) {
#pragma clang fp contract(off)
  const float kc = 1.75516512378075f, ks = 0.958851077208406f;
  const float nx = kc * x + -ks * y, ny = ks * x + kc * y;
  x = nx;
  y = ny;
}

template <int D, bool POW>
__global__ __launch_bounds__(kBlock) void k_noise(const StageDesc* dd) {
#pragma clang fp contract(off)
  const CDesc d = as_const(dd);
  // Two arrays: neighbouring corners of one lie in neighbouring banks.
  __shared__ float4 value[kCorners], below[kCorners];
  __shared__ NoiseBox box[kBoxes];
  __shared__ uint32_t batch_end;
  __shared__ typename LutOf<D == DST_U8>::type lut_mem;
  Luts* const luts = (Luts*)&lut_mem;
  const Dst o = target<D>(ldc(&d->slot[instr_slot(d, 1)]));
  const CParams q = d->params + d->code[0].arg;
  const float sx = q[0], sy = q[1], damping = q[3];
  const uint32_t octaves = (uint32_t)q[4];
  const uint32_t cached = min(octaves, kBoxes);
  const uint32_t W = d->width, H = d->height;
  const uint32_t tx = (W + 63) / 64, tiles = tx * ((H + 15) / 16);
  if constexpr (D == DST_U8) {
    if (o.transfer == 5) load_lut(d, luts);
  }
  const uint32_t lx = threadIdx.x & 15u, ly = threadIdx.x >> 4;
  for (uint32_t t = blockIdx.x; t < tiles; t += gridDim.x) {
    const uint32_t tyi = t / tx, X0 = (t - tyi * tx) * 64, Y0 = tyi * 16;
    __syncthreads();  // the previous tile's reads
    if (threadIdx.x < cached) {
      // Box of this lane's octave: the cells of the tile's corner pixels (an
      // affine map takes the tile into their hull) and one cell of margin.
      const float xa = ((float)X0 + 0.5f) / (float)W, xb = ((float)min(X0 + 63, W - 1) + 0.5f) / (float)W;
      const float ya = ((float)Y0 + 0.5f) / (float)H, yb = ((float)min(Y0 + 15, H - 1) + 0.5f) / (float)H;
      float px[4] = {xa, xb, xa, xb}, py[4] = {ya, ya, yb, yb};
      for (uint32_t k = 0; k < threadIdx.x; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) next_octave(px[i], py[i]);
      float x0 = px[0] * sx, x1 = x0, y0 = py[0] * sy, y1 = y0;
#pragma unroll
      for (int i = 1; i < 4; ++i) {
        x0 = fminf(x0, px[i] * sx);
        x1 = fmaxf(x1, px[i] * sx);
        y0 = fminf(y0, py[i] * sy);
        y1 = fmaxf(y1, py[i] * sy);
      }
      NoiseBox b{0, 0, 0u, 0u, 0u, 0u};
      // Coordinates small enough that a float resolves a thousandth of a cell.
      if (fmaxf(fmaxf(fabsf(x0), fabsf(x1)), fmaxf(fabsf(y0), fabsf(y1))) < 16384.0f) {
        b.x = (int32_t)floorf(x0) - 1;
        b.y = (int32_t)floorf(y0) - 1;
        b.w = (uint32_t)((int32_t)floorf(x1) + 3 - b.x);
        b.h = (uint32_t)((int32_t)floorf(y1) + 2 - b.y);
        if (b.w > kCorners || b.h >= kCorners || b.w * (b.h + 1u) > kCorners) b.w = b.h = 0u;
      }
      box[threadIdx.x] = b;
    }
    const uint32_t x0 = X0 + lx * kPix, y = Y0 + ly;
    const float v = ((float)y + 0.5f) / (float)H;
    float x[kPix], yy[kPix];
    Px X;
#pragma unroll
    for (int i = 0; i < kPix; ++i) {
      x[i] = ((float)(x0 + i) + 0.5f) / (float)W;
      yy[i] = v;
      X[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    float amp = q[2];
    uint32_t k = 0;
    do {  // uniform
      // The next batch: octaves while their corners fit the cache together.
      __syncthreads();  // the boxes; the previous batch's reads
      if (threadIdx.x == 0) {
        uint32_t used = 0, e = k;
        for (; e < cached; ++e) {
          const uint32_t n = box[e].w * (box[e].h + 1u);
          if (n > kCorners - used) break;
          box[e].at = used;
          used += n;
          box[e].end = used;
        }
        batch_end = e;
      }
      __syncthreads();
      uint32_t end = __builtin_amdgcn_readfirstlane(batch_end);
      const uint32_t used = end > k ? __builtin_amdgcn_readfirstlane(box[end - 1].end) : 0u;
      for (uint32_t e = threadIdx.x; e < used; e += kBlock) {
        uint32_t b = k;
        while (e >= box[b].end) ++b;
        const uint32_t i = e - box[b].at, r = i / box[b].w;
        value[e] = cell_value((uint32_t)(box[b].x + (int32_t)(i - r * box[b].w)), (uint32_t)(box[b].y + (int32_t)r));
      }
      __syncthreads();
      for (uint32_t e = threadIdx.x; e < used; e += kBlock) {
        uint32_t b = k;
        while (e >= box[b].end) ++b;
        if (e + box[b].w < box[b].end) {
          const float4 a = value[e], c = value[e + box[b].w];
          below[e] = make_float4(c.x - a.x, c.y - a.y, c.z - a.z, c.w - a.w);
        }
      }
      __syncthreads();
      if (end == k) end = octaves;  // past the cached octaves
      for (; k < end; ++k) {
        // An octave that is not cached has a box of no cells.
        uint32_t at = 0, bw = 1, bh = 0;
        int32_t bx = 0, by = 0;
        if (k < cached) {
          at = __builtin_amdgcn_readfirstlane(box[k].at);
          bx = __builtin_amdgcn_readfirstlane(box[k].x);
          by = __builtin_amdgcn_readfirstlane(box[k].y);
          bw = __builtin_amdgcn_readfirstlane(box[k].w);
          bh = __builtin_amdgcn_readfirstlane(box[k].h);
        }
        float ux[kPix], uy[kPix];
        uint32_t cx[kPix], cy[kPix], idx[kPix];
        bool in = true;
#pragma unroll
        for (int i = 0; i < kPix; ++i) {
          const float px = x[i] * sx, py = yy[i] * sy;
          const float flx = floorf(px), fly = floorf(py);
          const float fx = px - flx, fy = py - fly;
          cx[i] = cell_index(flx);
          cy[i] = cell_index(fly);
          ux[i] = fx * fx * (3.0f - 2.0f * fx);
          uy[i] = fy * fy * (3.0f - 2.0f * fy);
          const uint32_t rx = cx[i] - (uint32_t)bx, ry = cy[i] - (uint32_t)by;
          in = in && rx < bw - 1u && ry < bh;
          idx[i] = at + __umul24(ry, bw) + rx;
          next_octave(x[i], yy[i]);
        }
        if (in) {
#pragma unroll
          for (int i = 0; i < kPix; ++i) {
            const uint32_t e = idx[i];
            X[i] = blend_cell(X[i], value[e], below[e], value[e + 1], below[e + 1], ux[i], uy[i], amp);
          }
        } else {
          // One copy of the hash for the group's pixels: they rotate through
          // the registers.
#pragma unroll 1
          for (int i = 0; i < kPix; ++i) {
            float4 a, da, b, db;
            corner_at(cx[0], cy[0], a, da);
            corner_at(cx[0] + 1u, cy[0], b, db);
            const float4 r = blend_cell(X[0], a, da, b, db, ux[0], uy[0], amp);
#pragma unroll
            for (int j = 0; j + 1 < kPix; ++j) {
              X[j] = X[j + 1];
              cx[j] = cx[j + 1];
              cy[j] = cy[j + 1];
              ux[j] = ux[j + 1];
              uy[j] = uy[j + 1];
            }
            X[kPix - 1] = r;
          }
        }
        amp = amp * damping;
      }
    } while (k < octaves);
    if (x0 < W && y < H)
      put_group<D, POW>(o, (gbyte*)o.ptr + ((uint64_t)y * o.stride + (uint64_t)x0 * o.bpp),
                        (int)min((uint32_t)kPix, W - x0), X, luts);
  }
}

// The closed-form generators: a persistent grid of groups.
template <int OP, int D, bool POW>
__global__ __launch_bounds__(kBlock) void k_gen(const StageDesc* dd) {
  const CDesc d = as_const(dd);
  __shared__ typename LutOf<D == DST_U8>::type lut_mem;
  Luts* const luts = (Luts*)&lut_mem;
  const Dst o = target<D>(ldc(&d->slot[instr_slot(d, 1)]));
  const CParams q = d->params + d->code[0].arg;
  const uint32_t W = d->width, H = d->height, gpr = (W + kPix - 1) / kPix, groups = gpr * H;
  const uint32_t stride = gridDim.x * kBlock;
  if constexpr (D == DST_U8) {
    if (o.transfer == 5) load_lut(d, luts);
    __syncthreads();
  }
  uint32_t g = blockIdx.x * kBlock + threadIdx.x;
  if (g >= groups) return;
  while (true) {
    const uint32_t y = g / gpr, x0 = (g - y * gpr) * kPix;
    const int n = (int)min((uint32_t)kPix, W - x0);
    Px X;
    if constexpr (OP == OP_GRID) {
      const float v = ((float)y + 0.5f) / (float)H;
#pragma unroll
      for (int i = 0; i < kPix; ++i) X[i] = grid_value(q, ((float)(x0 + i) + 0.5f) / (float)W, v);
    } else {
      // distribution_normal2d.frag: the quadratic form of the inverse
      // covariance, read as the shader's column-major mat2 of the row-major
      // blob.
      const float py = 2.0f * (((float)y + 0.5f) / (float)H - 0.5f) - q[1];
      const float root = sqrtf(q[6]);
#pragma unroll
      for (int i = 0; i < kPix; ++i) {
        const float px = 2.0f * (((float)(x0 + i) + 0.5f) / (float)W - 0.5f) - q[0];
        const float e = 0.5f * (px * (q[2] * px + q[4] * py) + py * (q[3] * px + q[5] * py));
        const float v = expf(-e) / root;
        X[i] = make_float4(v, v, v, 1.0f);
      }
    }
    put_group<D, POW>(o, (gbyte*)o.ptr + ((uint64_t)y * o.stride + (uint64_t)x0 * o.bpp), n, X, luts);
    if (groups - g <= stride) break;
    g += stride;
  }
}

// resize: [grid quant palette store] -- the coordinate ramp rounded through
// RGBA8 (truncating codes), then the nearest texel of the palette.
template <int S, int D, bool POW>
__global__ __launch_bounds__(kBlock) void k_lookup(const StageDesc* dd) {
  const CDesc d = as_const(dd);
  __shared__ float tab[has_table(S) ? kTable : 1];
  __shared__ typename LutOf<D == DST_U8>::type lut_mem;
  Luts* const luts = (Luts*)&lut_mem;
  const Slot ps = ldc(&d->slot[instr_slot(d, 2)]);
  const Src s = source<S>(ps, &d->table[0]);
  const Dst o = target<D>(ldc(&d->slot[instr_slot(d, 3)]));
  const CParams ramp = d->params + d->code[0].arg, q = d->params + d->code[2].arg;
  const uint32_t W = d->width, H = d->height, gpr = (W + kPix - 1) / kPix, groups = gpr * H;
  const uint32_t stride = gridDim.x * kBlock;
  fill_table<S>(s, d, tab);
  if constexpr (D == DST_U8) {
    if (o.transfer == 5) load_lut(d, luts);
  }
  __syncthreads();
  const float w = (float)ps.width, h = (float)ps.height;
  uint32_t g = blockIdx.x * kBlock + threadIdx.x;
  if (g >= groups) return;
  while (true) {
    const uint32_t y = g / gpr, x0 = (g - y * gpr) * kPix;
    const int n = (int)min((uint32_t)kPix, W - x0);
    const float v = ((float)y + 0.5f) / (float)H;
    Px X;
    Codes c;
#pragma unroll
    for (int i = 0; i < kPix; ++i) {
      const float4 r = grid_value(ramp, ((float)(x0 + i) + 0.5f) / (float)W, v);
      const float4 k = make_float4(fd(qt(clamp01(r.x), 8), 255.0f), fd(qt(clamp01(r.y), 8), 255.0f),
                                   fd(qt(clamp01(r.z), 8), 255.0f), fd(qt(clamp01(r.w), 8), 255.0f));
      const float u = q[0] * k.x + q[1] * k.y + q[2] * k.z + q[3] * k.w + q[8];
      const float t = q[4] * k.x + q[5] * k.y + q[6] * k.z + q[7] * k.w + q[9];
      const int ix = (int)fminf(fmaxf(floorf(u * w), 0.0f), w - 1.0f);
      const int iy = (int)fminf(fmaxf(floorf(t * h), 0.0f), h - 1.0f);
      const gbyte* p = (const gbyte*)s.ptr + ((uint64_t)iy * s.stride + (uint64_t)ix * s.bpp);
      if (S == SRC_F32 || s.bpp == 16) X[i] = f4_bits(gld<w4>(p));
      else load_code(p, s.bpp, c.lo[i], c.hi[i]);
    }
    decode_codes<S, POW>(s, c, X, tab);
    put_group<D, POW>(o, (gbyte*)o.ptr + ((uint64_t)y * o.stride + (uint64_t)x0 * o.bpp), n, X, luts);
    if (groups - g <= stride) break;
    g += stride;
  }
}

// ---- kernels by shape -----------------------------------------------------------
typedef void (*FieldKernel)(const StageDesc*);
typedef void (*BoxKernel)(const StageDesc*, uint32_t);

// Instantiates K<..., D, POW> for a target class.
#define ZH_BY_DST(K, dst, pow, ...)                                                        \
  switch (dst) {                                                                           \
    case DST_U8: return K<__VA_ARGS__ DST_U8, false>;                                      \
    case DST_F16: return K<__VA_ARGS__ DST_F16, false>;                                    \
    case DST_F32: return K<__VA_ARGS__ DST_F32, false>;                                    \
    case DST_CODE: return pow ? K<__VA_ARGS__ DST_CODE, true> : K<__VA_ARGS__ DST_CODE, false>; \
    default: return pow ? K<__VA_ARGS__ DST_WIDE, true> : K<__VA_ARGS__ DST_WIDE, false>;  \
  }
#define ZH_COMMA ,

static BoxKernel box_kernel(uint32_t src, uint32_t dst, bool pow) {
  // Wide sources whose transfer is a power function per pixel take POW.
  if (src == SRC_TABLE) { ZH_BY_DST(k_box3, dst, pow, SRC_TABLE ZH_COMMA) }
  if (src == SRC_F16) { ZH_BY_DST(k_box3, dst, pow, SRC_F16 ZH_COMMA) }
  if (src == SRC_F32) { ZH_BY_DST(k_box3, dst, pow, SRC_F32 ZH_COMMA) }
  switch (dst) {
    case DST_U8: return k_box3<SRC_WIDE, DST_U8, true>;
    case DST_F16: return k_box3<SRC_WIDE, DST_F16, true>;
    case DST_F32: return k_box3<SRC_WIDE, DST_F32, true>;
    case DST_CODE: return k_box3<SRC_WIDE, DST_CODE, true>;
    default: return k_box3<SRC_WIDE, DST_WIDE, true>;
  }
}
static FieldKernel noise_kernel(uint32_t dst, bool pow) { ZH_BY_DST(k_noise, dst, pow, ) }
static FieldKernel grid_kernel(uint32_t dst, bool pow) { ZH_BY_DST(k_gen, dst, pow, OP_GRID ZH_COMMA) }
static FieldKernel normal_kernel(uint32_t dst, bool pow) { ZH_BY_DST(k_gen, dst, pow, OP_NORMAL2D ZH_COMMA) }
static FieldKernel lookup_kernel(uint32_t src, uint32_t dst, bool pow) {
  if (src == SRC_TABLE) { ZH_BY_DST(k_lookup, dst, pow, SRC_TABLE ZH_COMMA) }
  if (src == SRC_F16) { ZH_BY_DST(k_lookup, dst, pow, SRC_F16 ZH_COMMA) }
  switch (dst) {
    case DST_U8: return k_lookup<SRC_ANY, DST_U8, true>;
    case DST_F16: return k_lookup<SRC_ANY, DST_F16, true>;
    case DST_F32: return k_lookup<SRC_ANY, DST_F32, true>;
    case DST_CODE: return k_lookup<SRC_ANY, DST_CODE, true>;
    default: return k_lookup<SRC_ANY, DST_WIDE, true>;
  }
}
static FieldKernel field_kernel(uint32_t shape) {
  const uint32_t src = any_src(shape, 0), dst = any_dst(shape);
  const bool pow = (shape & ANY_POW) != 0;
  switch (field_kind(shape)) {
    case FIELD_NOISE: return noise_kernel(dst, pow);
    case FIELD_GRID: return grid_kernel(dst, pow);
    case FIELD_NORMAL: return normal_kernel(dst, pow);
    default: return lookup_kernel(src, dst, pow);
  }
}

}  // namespace any
}  // namespace zh

extern "C" {

hipError_t zh_launch_field(uint32_t shape, const zh::StageDesc* d_dev, uint32_t width, uint32_t height, uint32_t cus,
                           hipStream_t stream) {
  using namespace zh;
  if (shape >= kFieldShapes || width == 0 || height == 0) return hipErrorInvalidValue;
  const uint64_t gpr = (width + kPix - 1) / kPix;
  if (gpr * height >= (1ull << 32) - kBlock) return hipErrorInvalidValue;
  if (field_kind(shape) == FIELD_BOX3) {
    // Rows of a lane's strip: as few as let every strip be resident at once (a
    // strip reads two rows more than it writes, and a second round of
    // workgroups costs more: 41 us with 3 rows, 30.5 with 7, 35.6 with 10 at
    // 3840x2160, whose strips fill the chip at 7).
    const any::BoxKernel fn = any::box_kernel(any_src(shape, 0), any_dst(shape), (shape & ANY_POW) != 0);
    static std::atomic<uint32_t> resident[512];
    uint32_t res = resident[shape].load(std::memory_order_relaxed);
    if (!res) {
      res = resident_blocks((const void*)fn, 1);
      resident[shape].store(res, std::memory_order_relaxed);
    }
    const uint64_t lanes = (uint64_t)cus * res * kBlock;
    const uint32_t rows = (uint32_t)((gpr * height + lanes - 1) / lanes);
    const uint64_t strips = (height + rows - 1) / rows;
    hipLaunchKernelGGL(fn, dim3((uint32_t)((gpr * strips + kBlock - 1) / kBlock)), dim3(kBlock), 0, stream, d_dev, rows);
    return hipGetLastError();
  }
  static std::atomic<uint32_t> resident[kFieldShapes];
  const any::FieldKernel fn = any::field_kernel(shape);
  uint32_t res = resident[shape].load(std::memory_order_relaxed);
  if (!res) {
    res = resident_blocks((const void*)fn, 1);
    resident[shape].store(res, std::memory_order_relaxed);
  }
  const uint64_t work = field_kind(shape) == FIELD_NOISE ? (uint64_t)((width + 63) / 64) * ((height + 15) / 16)
                                                         : (gpr * height + kBlock - 1) / kBlock;
  const uint32_t blocks = (uint32_t)std::min<uint64_t>(work, (uint64_t)res * cus);
  hipLaunchKernelGGL(fn, dim3(blocks), dim3(kBlock), 0, stream, d_dev);
  return hipGetLastError();
}

}  // extern "C"
