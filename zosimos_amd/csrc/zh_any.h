// zh_any.h -- codecs of whole lane groups for every texel format, device code
// of the kernels in zh_any.hip.
//
// A slot's format is uniform over the grid, so each step of a codec is one
// scalar branch around straight-line code for the lane's kPix pixels: nothing
// is called out of line and no texel is tested on its own.  (The interpreter's
// codecs are functions called per texel with the format in vector registers:
// 174 VGPRs and scratch, two waves per SIMD.)
//
// Integer texels of up to 10 bits per channel decode through a table in LDS:
// a workgroup evaluates the transfer function once per code (four 10-bit codes
// per lane) instead of once per pixel and channel, and every pixel's channel
// is a bit-field extract and a read.  The entries are the values the
// per-texel codec computes, so the decode is the same bit for bit.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "zh_device.h"

namespace zh {
namespace any {

// Groups move as dwords wherever their address is a multiple of 4 (a group of
// kPix texels is a whole number of dwords in every format).
typedef uint32_t w2 __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t w3 __attribute__((ext_vector_type(3), aligned(4)));
typedef uint32_t w4 __attribute__((ext_vector_type(4), aligned(4)));

template <typename T>
__device__ __forceinline__ T nt_get(const gbyte* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const __attribute__((address_space(1))) T*>(p));
}
template <typename T>
__device__ __forceinline__ void nt_put(gbyte* p, T v) {
  __builtin_nontemporal_store(v, reinterpret_cast<__attribute__((address_space(1))) T*>(p));
}

// Codes of a lane's texels: lo holds up to 4 bytes, hi the rest of 6- and
// 8-byte texels.
struct Codes {
  uint32_t lo[kPix], hi[kPix];
};

__device__ __forceinline__ float4 f4_bits(w4 v) {
  return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
}

// One texel's code (bpp 1, 3 at any address, 2 and 6 at even ones, 4 and 8 at
// multiples of 4).
__device__ __forceinline__ void load_code(const gbyte* p, uint32_t bpp, uint32_t& lo, uint32_t& hi) {
  hi = 0u;
  switch (bpp) {  // uniform
    case 1: lo = gld<uint8_t>(p); break;
    case 2: lo = gld<uint16_t>(p); break;
    case 3:
      lo = (uint32_t)gld<uint8_t>(p) | ((uint32_t)gld<uint8_t>(p + 1) << 8) | ((uint32_t)gld<uint8_t>(p + 2) << 16);
      break;
    case 4: lo = gld<uint32_t>(p); break;
    case 6:
      lo = (uint32_t)gld<uint16_t>(p) | ((uint32_t)gld<uint16_t>(p + 2) << 16);
      hi = gld<uint16_t>(p + 4);
      break;
    case 8: {
      const w2 v = gld<w2>(p);
      lo = v.x;
      hi = v.y;
      break;
    }
    default: lo = 0u;
  }
}

// The group's texels at q: all kPix by dwords, or one by one where the group is
// a row's last (its first n >= 1 texels; the others repeat the last one and
// their results are not stored) or its address is no multiple of 4.  16-byte
// texels have no codes: load_floats reads them.
__device__ __forceinline__ void load_group(const gbyte* q, uint32_t bpp, int n, Codes& c) {
#pragma unroll
  for (int i = 0; i < kPix; ++i) c.lo[i] = c.hi[i] = 0u;
  if (n == kPix && ((uintptr_t)q & 3u) == 0) {
    switch (bpp) {  // uniform
      case 1: {
        const uint32_t v = nt_get<uint32_t>(q);
#pragma unroll
        for (int i = 0; i < kPix; ++i) c.lo[i] = (v >> (8 * i)) & 255u;
        break;
      }
      case 2: {
        const w2 v = nt_get<w2>(q);
        c.lo[0] = v.x & 0xffffu;
        c.lo[1] = v.x >> 16;
        c.lo[2] = v.y & 0xffffu;
        c.lo[3] = v.y >> 16;
        break;
      }
      case 3: {
        const w3 v = nt_get<w3>(q);
        c.lo[0] = v.x & 0xffffffu;
        c.lo[1] = __builtin_amdgcn_alignbyte(v.y, v.x, 3) & 0xffffffu;
        c.lo[2] = __builtin_amdgcn_alignbyte(v.z, v.y, 2) & 0xffffffu;
        c.lo[3] = v.z >> 8;
        break;
      }
      case 4: {
        const w4 v = nt_get<w4>(q);
        c.lo[0] = v.x;
        c.lo[1] = v.y;
        c.lo[2] = v.z;
        c.lo[3] = v.w;
        break;
      }
      case 6: {
        const w4 v = nt_get<w4>(q);
        const w2 u = nt_get<w2>(q + 16);
        c.lo[0] = v.x;
        c.hi[0] = v.y & 0xffffu;
        c.lo[1] = __builtin_amdgcn_alignbyte(v.z, v.y, 2);
        c.hi[1] = v.z >> 16;
        c.lo[2] = v.w;
        c.hi[2] = u.x & 0xffffu;
        c.lo[3] = __builtin_amdgcn_alignbyte(u.y, u.x, 2);
        c.hi[3] = u.y >> 16;
        break;
      }
      case 8: {
        const w4 v = nt_get<w4>(q), u = nt_get<w4>(q + 16);
        c.lo[0] = v.x;
        c.hi[0] = v.y;
        c.lo[1] = v.z;
        c.hi[1] = v.w;
        c.lo[2] = u.x;
        c.hi[2] = u.y;
        c.lo[3] = u.z;
        c.hi[3] = u.w;
        break;
      }
      default: break;
    }
  } else {
#pragma unroll
    for (int i = 0; i < kPix; ++i) load_code(q + (uint32_t)min(i, n - 1) * bpp, bpp, c.lo[i], c.hi[i]);
  }
}

__device__ __forceinline__ void load_floats(const gbyte* q, int n, Px& X) {
#pragma unroll
  for (int i = 0; i < kPix; ++i) X[i] = f4_bits(nt_get<w4>(q + 16 * min(i, n - 1)));
}

__device__ __forceinline__ void store_code(gbyte* p, uint32_t bpp, uint32_t lo, uint32_t hi) {
  switch (bpp) {  // uniform
    case 1: gst<uint8_t>(p, (uint8_t)lo); break;
    case 2: gst<uint16_t>(p, (uint16_t)lo); break;
    case 3:
      gst<uint8_t>(p, (uint8_t)lo);
      gst<uint8_t>(p + 1, (uint8_t)(lo >> 8));
      gst<uint8_t>(p + 2, (uint8_t)(lo >> 16));
      break;
    case 4: gst<uint32_t>(p, lo); break;
    case 6:
      gst<uint16_t>(p, (uint16_t)lo);
      gst<uint16_t>(p + 2, (uint16_t)(lo >> 16));
      gst<uint16_t>(p + 4, (uint16_t)hi);
      break;
    case 8: gst<w2>(p, w2{lo, hi}); break;
    default: break;
  }
}

__device__ __forceinline__ void store_group(gbyte* q, uint32_t bpp, int n, const Codes& c) {
  // Values, not elements of c: left in the branches, their loads are merged
  // into one from a variable index and c ends up in memory.
  const uint32_t l0 = c.lo[0], l1 = c.lo[1], l2 = c.lo[2], l3 = c.lo[3];
  const uint32_t h0 = c.hi[0], h1 = c.hi[1], h2 = c.hi[2], h3 = c.hi[3];
  if (n == kPix && ((uintptr_t)q & 3u) == 0) {
    switch (bpp) {  // uniform
      case 1: nt_put<uint32_t>(q, l0 | (l1 << 8) | (l2 << 16) | (l3 << 24)); break;
      case 2: nt_put<w2>(q, w2{l0 | (l1 << 16), l2 | (l3 << 16)}); break;
      case 3:
        nt_put<w3>(q, w3{l0 | (l1 << 24), (l1 >> 8) | (l2 << 16), (l2 >> 16) | (l3 << 8)});
        break;
      case 4: nt_put<w4>(q, w4{l0, l1, l2, l3}); break;
      case 6:
        nt_put<w4>(q, w4{l0, h0 | (l1 << 16), (l1 >> 16) | (h1 << 16), l2});
        nt_put<w2>(q + 16, w2{h2 | (l3 << 16), (l3 >> 16) | (h3 << 16)});
        break;
      case 8:
        nt_put<w4>(q, w4{l0, h0, l1, h1});
        nt_put<w4>(q + 16, w4{l2, h2, l3, h3});
        break;
      default: break;
    }
  } else {
    store_code(q, bpp, l0, h0);  // n >= 1
    if (n > 1) store_code(q + bpp, bpp, l1, h1);
    if (n > 2) store_code(q + 2 * bpp, bpp, l2, h2);
    if (n > 3) store_code(q + 3 * bpp, bpp, l3, h3);
  }
}
static_assert(kPix == 4, "a group holds 4 texels");

__device__ __forceinline__ void store_floats(gbyte* q, int n, const Px& X) {
  w4 v[kPix];
#pragma unroll
  for (int i = 0; i < kPix; ++i)
    v[i] = w4{__float_as_uint(X[i].x), __float_as_uint(X[i].y), __float_as_uint(X[i].z), __float_as_uint(X[i].w)};
  nt_put<w4>(q, v[0]);  // n >= 1
  if (n > 1) nt_put<w4>(q + 16, v[1]);
  if (n > 2) nt_put<w4>(q + 32, v[2]);
  if (n > 3) nt_put<w4>(q + 48, v[3]);
}

// ---- transfers ---------------------------------------------------------------
// One channel of untransfer (zh_codec.h), for the decode tables.  The planner
// keeps LabLch, which mixes channels, off these kernels.
__device__ __forceinline__ float untransfer1(float v, uint32_t t) {
  switch (t) {
    case 5: return eo_srgb(v);
    case 0: case 6: case 7: return eo_bt709(v);
    case 1: return powf(v, 2.2f);
    case 2: return oe_bt709(v);
    case 3: return eo_smpte240(v);
    case 8: return eo_pq(v);
  }
  return v;
}

// f on the colour of every pixel in turn through one copy of its code: the
// group rotates through the registers (a power function is some 100
// instructions; twelve copies of each would not stay in the instruction
// cache).
template <class Fn>
__device__ __forceinline__ void each_px(Px& X, Fn f) {
#pragma unroll 1
  for (int i = 0; i < kPix; ++i) {
    const float4 v = X[0];
#pragma unroll
    for (int k = 0; k + 1 < kPix; ++k) X[k] = X[k + 1];
    const float r = f(v.x);
    __builtin_amdgcn_sched_barrier(0);
    const float g = f(v.y);
    __builtin_amdgcn_sched_barrier(0);
    const float b = f(v.z);
    __builtin_amdgcn_sched_barrier(0);
    X[kPix - 1] = make_float4(r, g, b, v.w);
  }
}

// POW: the kernel also carries the transfers made of power functions.  Without
// them it holds twice the waves per SIMD.
template <bool POW>
__device__ __forceinline__ void untransfer_group(Px& X, uint32_t t) {
  if (t == 5) {  // uniform
#pragma unroll
    for (int i = 0; i < kPix; ++i) X[i] = make_float4(eo_srgb(X[i].x), eo_srgb(X[i].y), eo_srgb(X[i].z), X[i].w);
    return;
  }
  if constexpr (!POW) return;
  switch (t) {  // uniform
    case 0: case 6: case 7: each_px(X, [](float v) { return eo_bt709(v); }); break;
    case 1: each_px(X, [](float v) { return powf(v, 2.2f); }); break;
    case 2: each_px(X, [](float v) { return oe_bt709(v); }); break;
    case 3: each_px(X, [](float v) { return eo_smpte240(v); }); break;
    case 8: each_px(X, [](float v) { return eo_pq(v); }); break;
    default: break;
  }
}

template <bool POW>
__device__ __forceinline__ void transfer_group(Px& X, uint32_t t) {
  if (t == 5) {  // uniform
#pragma unroll
    for (int i = 0; i < kPix; ++i) X[i] = make_float4(oe_srgb(X[i].x), oe_srgb(X[i].y), oe_srgb(X[i].z), X[i].w);
    return;
  }
  if constexpr (!POW) return;
  switch (t) {  // uniform
    case 0: case 6: case 7: each_px(X, [](float v) { return oe_bt709(v); }); break;
    case 1: each_px(X, [](float v) { return powf(v, 1.0f / 2.2f); }); break;
    case 2: each_px(X, [](float v) { return eo_bt709(v); }); break;
    case 3: each_px(X, [](float v) { return oe_smpte240(v); }); break;
    case 8: each_px(X, [](float v) { return oe_pq(v); }); break;
    default: break;
  }
}

// ---- decode --------------------------------------------------------------------
// A kernel is compiled per class of slot (zh_stage.h SrcClass, DstClass); one
// kernel that carried every codec behind uniform branches took 41 us for
// 10-bit to RGBA16F at 3840x2160 (100 VGPRs, 80 KB of code that every launch
// fetches anew) where the class's own takes 26.7 us (the interpreter: 220 us).

// Floats of a decode table: two 10-bit segments (colour and alpha) and a
// short one, the most any layout takes.
constexpr uint32_t kTable = 1024 + 1024 + 64;

// A load's slot in scalar registers.
struct Src {
  uint64_t ptr, stride;
  uint32_t bpp, bits, parts, transfer, native;
  TableDesc t;  // SRC_TABLE
};

template <int S>
__device__ __forceinline__ Src source(const Slot& s, const __attribute__((address_space(4))) TableDesc* t) {
  Src r;
  r.ptr = s.ptr;
  r.stride = s.row_stride;
  r.bpp = S == SRC_F16 ? 8u : S == SRC_F32 ? 16u : s.bpp;
  r.bits = s.bits;
  r.parts = s.parts;
  r.transfer = s.transfer;
  r.native = s.native;
  if constexpr (S == SRC_TABLE || S == SRC_ANY) r.t = ldc(t);
  return r;
}
__device__ __forceinline__ bool is_wide(uint32_t bits) { return bits == 3 || (bits >= 11 && bits <= 13) || bits >= 18; }

// The slot's decode table; the caller synchronises the workgroup.
template <int S>
__device__ __forceinline__ void fill_table(const Src& s, CDesc d, float* tab) {
  if constexpr (S != SRC_TABLE && S != SRC_ANY) return;
  if (S == SRC_ANY && is_wide(s.bits)) return;  // uniform
  const float* dec = reinterpret_cast<const Luts*>(d->srgb_lut)->dec;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const TableChannel c = s.t.ch[k];
    if (!(c.flags & TABLE_OWNER)) continue;  // uniform
    const uint32_t n = c.mask / 4 + 1;
    for (uint32_t code = threadIdx.x; code < n; code += kBlock) {
      float v;
      if (s.native) {
        v = k < 3 && s.transfer == 5 ? dec[code] : (float)code * (1.0f / 255.0f);
      } else {
        v = n > 1 ? fd(code, (float)(n - 1)) : (c.flags & TABLE_ONE) ? 1.0f : 0.0f;
        if (k < 3) v = untransfer1(v, s.transfer);
      }
      tab[c.base / 4 + code] = v;
    }
  }
}

// u / 65535 correctly rounded for every 16-bit u: the product with the
// rounded reciprocal, corrected by its residual (equal to the division for
// all 65,536 values), in 3 instructions.
__device__ __forceinline__ float unorm16(uint32_t u) {
  const float n = (float)u, q = n * (1.0f / 65535.0f);
  return fmaf(fmaf(-q, 65535.0f, n), 1.0f / 65535.0f, q);
}

__device__ __forceinline__ void permute_group(Px& X, uint32_t parts) {
  if (parts_identity(parts) || parts == 10) return;  // uniform
#pragma unroll
  for (int i = 0; i < kPix; ++i) X[i] = parts_normalize(X[i], parts);
}

__device__ __forceinline__ void table_group(const TableDesc& t, const Codes& c, Px& X, const float* tab) {
#pragma unroll
  for (int i = 0; i < kPix; ++i) {
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t at = (__builtin_amdgcn_alignbit(c.lo[i], c.lo[i], t.ch[k].rot) & t.ch[k].mask) | t.ch[k].base;
      v[k] = *(const float*)((const char*)tab + at);
    }
    X[i] = make_float4(v[0], v[1], v[2], v[3]);
  }
}

template <bool POW>
__device__ __forceinline__ void wide_group(const Src& s, const Codes& c, Px& X) {
  if (s.bits == 18) {  // uniform; 19: load_floats filled X
#pragma unroll
    for (int i = 0; i < kPix; ++i) X[i] = dec_f16(c.lo[i], c.hi[i]);
  } else if (s.bits != 19) {
#pragma unroll
    for (int i = 0; i < kPix; ++i) {
      const float x = unorm16(c.lo[i] & 0xffffu);
      if (s.bits == 3) {
        X[i] = make_float4(x, x, x, x);
      } else {
        const float y = unorm16(c.lo[i] >> 16);
        if (s.bits == 11) X[i] = make_float4(x, y, 0.0f, 1.0f);
        else X[i] = make_float4(x, y, unorm16(c.hi[i] & 0xffffu), s.bits == 12 ? 1.0f : unorm16(c.hi[i] >> 16));
      }
    }
  }
  permute_group(X, s.parts);
  untransfer_group<POW>(X, s.transfer);
}

// X of a group's codes (16-byte texels: of the floats in X).
template <int S, bool POW>
__device__ __forceinline__ void decode_codes(const Src& s, const Codes& c, Px& X, const float* tab) {
  if constexpr (S == SRC_TABLE) {
    table_group(s.t, c, X, tab);
  } else if constexpr (S == SRC_F16) {
#pragma unroll
    for (int i = 0; i < kPix; ++i) X[i] = dec_f16(c.lo[i], c.hi[i]);
  } else if constexpr (S != SRC_F32) {
    if (S == SRC_ANY && !is_wide(s.bits)) table_group(s.t, c, X, tab);  // uniform
    else wide_group<POW>(s, c, X);
  }
}

// X of the fetched group at q (16-byte texels are read here).
template <int S, bool POW>
__device__ __forceinline__ void decode_group(const Src& s, const gbyte* q, int n, const Codes& c, Px& X,
                                             const float* tab) {
  if (S == SRC_F32 || (S >= SRC_WIDE && s.bits == 19)) load_floats(q, n, X);
  decode_codes<S, POW>(s, c, X, tab);
}

template <bool WITH> struct LutOf { typedef uint32_t type; };
template <> struct LutOf<true> { typedef Luts type; };
constexpr bool has_table(int s) { return s == SRC_TABLE || s == SRC_ANY; }

// ---- encode --------------------------------------------------------------------
struct Dst {
  uint64_t ptr, stride;
  uint32_t bpp, bits, parts, transfer, fmt;
};

template <int D>
__device__ __forceinline__ Dst target(const Slot& s) {
  return Dst{s.ptr, s.row_stride, D == DST_U8 ? 4u : D == DST_F16 ? 8u : D == DST_F32 ? 16u : s.bpp, s.bits, s.parts,
             s.transfer, s.fmt};
}

__device__ __forceinline__ void denormalize_group(Px& X, uint32_t parts) {
  if (parts_identity(parts)) return;  // uniform
#pragma unroll
  for (int i = 0; i < kPix; ++i) X[i] = parts_denormalize(X[i], parts);
}

// The codes of X (mux, stage.frag:533-641).  WIDE: 16-bit channels and float
// texels with other parts or transfers (16-byte texels' floats are X itself);
// else texels of up to 4 bytes.
template <bool WIDE, bool POW>
__device__ __forceinline__ void code_group(const Dst& s, Px& X, Codes& c) {
  transfer_group<POW>(X, s.transfer);
  denormalize_group(X, s.parts);
  if (WIDE && s.bits == 18) {  // uniform
#pragma unroll
    for (int i = 0; i < kPix; ++i) {
      round_f32(X[i]);
      c.lo[i] = pack_f16(X[i].x, X[i].y);
      c.hi[i] = pack_f16(X[i].z, X[i].w);
    }
    return;
  }
  if (WIDE && s.bits == 19) return;
#pragma unroll
  for (int i = 0; i < kPix; ++i) X[i] = make_float4(clamp01(X[i].x), clamp01(X[i].y), clamp01(X[i].z), clamp01(X[i].w));
#define ZH_MUX(B)                                                            \
  case B:                                                                    \
    _Pragma("unroll") for (int i = 0; i < kPix; ++i) {                       \
      c.lo[i] = mux(X[i], B);                                                \
      c.hi[i] = 0u;                                                          \
    }                                                                        \
    break;
  if constexpr (WIDE) {
    switch (s.bits) {  // uniform
      ZH_MUX(3)
      ZH_MUX(11)
      default:  // 12, 13
#pragma unroll
        for (int i = 0; i < kPix; ++i) {
          c.lo[i] = qt(X[i].x, 16) | (qt(X[i].y, 16) << 16);
          c.hi[i] = qt(X[i].z, 16) | (s.bits == 13 ? qt(X[i].w, 16) << 16 : 0u);
        }
    }
  } else {
    switch (s.bits) {  // uniform
      ZH_MUX(0) ZH_MUX(1) ZH_MUX(2) ZH_MUX(4) ZH_MUX(5) ZH_MUX(6) ZH_MUX(7) ZH_MUX(8) ZH_MUX(9) ZH_MUX(10)
      ZH_MUX(14) ZH_MUX(15) ZH_MUX(16) ZH_MUX(17)
      default: break;
    }
  }
#undef ZH_MUX
}

// Encode and store the lane's group at q.
template <int D, bool POW>
__device__ __forceinline__ void put_group(const Dst& s, gbyte* q, int n, Px& X, const Luts* L) {
  Codes c;
#pragma unroll
  for (int i = 0; i < kPix; ++i) c.lo[i] = c.hi[i] = 0u;
  if constexpr (D == DST_U8) {
    switch (s.fmt) {  // uniform
#define ZH_U8(F)                                                                     \
  case F:                                                                            \
    _Pragma("unroll") for (int i = 0; i < kPix; ++i) c.lo[i] = enc_u8<F>(X[i], L);   \
    break;
      ZH_U8(FMT_U8_SRGB_RGBA)
      ZH_U8(FMT_U8_SRGB_BGRA)
      ZH_U8(FMT_U8_LIN_RGBA)
      ZH_U8(FMT_U8_LIN_BGRA)
#undef ZH_U8
      default: break;
    }
    store_group(q, 4u, n, c);
  } else if constexpr (D == DST_F16) {
#pragma unroll
    for (int i = 0; i < kPix; ++i) {
      round_f32(X[i]);
      c.lo[i] = pack_f16(X[i].x, X[i].y);
      c.hi[i] = pack_f16(X[i].z, X[i].w);
    }
    store_group(q, 8u, n, c);
  } else if constexpr (D == DST_F32) {
    store_floats(q, n, X);
  } else {
    code_group<D == DST_WIDE, POW>(s, X, c);
    if (D == DST_WIDE && s.bits == 19) store_floats(q, n, X);
    else store_group(q, s.bpp, n, c);
  }
}

}  // namespace any
}  // namespace zh
