// Pieces shared by the kernels of the statequant layout ([B, HV, K, V], V
// contiguous): the split of a column's K rows over slices, the tree over the
// slices' partial sums, the residual codecs, and the vector accesses of one
// row's columns.
#pragma once

#include <type_traits>

#include "ck_capi_common.h"
#include "ck_device.h"
#include "ck_quant.h"
#include "ck_tiles.h"

namespace ck {
namespace qs {

constexpr int kResFp32 = CK_RES_FP32;
constexpr int kResFp16 = CK_RES_FP16;
constexpr int kResFp8 = CK_RES_FP8;
constexpr int kResInt8 = CK_RES_INT8;

// K-slices per workgroup, one half-wave each.
template <int K>
constexpr int kSlicesFor = K <= 128 ? 8 : K / 16;
template <int K, int GROUPS = kGroups>
constexpr int kThreadsFor = GROUPS * kSlicesFor<K>;

// fp8 e5m2 (OCP: sign | 5-bit exponent, bias 15 | 2-bit mantissa, with
// infinities and NaNs) through gfx950's conversion instructions: encoding
// rounds to nearest even, keeps subnormals (m * 2^-16) and sends values at or
// past the midpoint above the largest finite 57344 to infinity, the format's
// own definition (the reference's torch.float8_e5m2 casts). Two values per
// v_cvt_pk_bf8_f32 into one 16-bit half of the result; decoding picks a byte.
template <int CPT>
__device__ __forceinline__ uint32_t f32_to_e5m2(const float (&x)[CPT]) {
  if constexpr (CPT == 4) {
    const int lo = __builtin_amdgcn_cvt_pk_bf8_f32(x[0], x[1], 0, false);
    return (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(x[2], x[3], lo, true);
  } else {
    return (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(x[0], 0.0f, 0, false) & 0xffu;
  }
}

// Byte j (0..3, unrolled to a constant) of d as an e5m2 value.
__device__ __forceinline__ float e5m2_byte(uint32_t d, int j) {
  switch (j) {
    case 0: return __builtin_amdgcn_cvt_f32_bf8((int)d, 0);
    case 1: return __builtin_amdgcn_cvt_f32_bf8((int)d, 1);
    case 2: return __builtin_amdgcn_cvt_f32_bf8((int)d, 2);
    default: return __builtin_amdgcn_cvt_f32_bf8((int)d, 3);
  }
}

__device__ __forceinline__ float half_bits_to_f32(uint32_t h) {
  _Float16 x;
  const uint16_t b = (uint16_t)h;
  __builtin_memcpy(&x, &b, 2);
  return (float)x;
}

__device__ __forceinline__ uint32_t f32_to_half_bits(float f) {
  const _Float16 x = (_Float16)f;  // round to nearest even, subnormals kept
  uint16_t b;
  __builtin_memcpy(&b, &x, 2);
  return b;
}

// Balanced pairwise tree over the S slice partials of LDS column `col`.
template <int S, int NC>
__device__ __forceinline__ float slice_tree_sum(const float (*red)[NC], int col) {
  float c[S];
#pragma unroll
  for (int s = 0; s < S; ++s) c[s] = red[s][col];
#pragma unroll
  for (int w = 1; w < S; w *= 2)
#pragma unroll
    for (int i = 0; i + w < S; i += 2 * w) c[i] = c[i] + c[i + w];
  return c[0];
}

template <int S, int NC>
__device__ __forceinline__ float slice_max(const float (*red)[NC], int col) {
  float m = red[0][col];
#pragma unroll
  for (int s = 1; s < S; ++s) m = fmaxf(m, red[s][col]);
  return m;
}

// CPT consecutive columns of one row at p: CPT = 4 is one vector access at any
// alignment of the element (global memory takes those on this target), CPT = 1
// one element. 8-bit values travel packed in a dword (column j in byte j),
// 16-bit values two to a dword.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 __attribute__((aligned(4))) f32x4_u;
typedef u32x2 __attribute__((aligned(2))) b16x4_u;

template <int CPT>
__device__ __forceinline__ void ld_f32(const float* p, float (&x)[CPT]) {
  if constexpr (CPT == 4) {
    const f32x4 f = *reinterpret_cast<const f32x4_u*>(p);
    x[0] = f.x, x[1] = f.y, x[2] = f.z, x[3] = f.w;
  } else {
    x[0] = *p;
  }
}

template <int CPT>
__device__ __forceinline__ uint32_t ld_b8(const void* p) {
  if constexpr (CPT == 4) return *static_cast<const u32_u*>(p);
  else return *static_cast<const uint8_t*>(p);
}

template <int CPT>
__device__ __forceinline__ void ld_b16(const uint16_t* p, uint32_t (&w)[(CPT + 1) / 2]) {
  if constexpr (CPT == 4) {
    const u32x2 x = *reinterpret_cast<const b16x4_u*>(p);
    w[0] = x.x, w[1] = x.y;
  } else {
    w[0] = *p;
  }
}

template <int CPT>
__device__ __forceinline__ void st_f32(float* p, const float (&x)[CPT]) {
  if constexpr (CPT == 4) *reinterpret_cast<f32x4_u*>(p) = f32x4{x[0], x[1], x[2], x[3]};
  else *p = x[0];
}

template <int CPT>
__device__ __forceinline__ void st_b8(void* p, uint32_t x) {
  if constexpr (CPT == 4) *static_cast<u32_u*>(p) = x;
  else *static_cast<uint8_t*>(p) = (uint8_t)x;
}

template <int CPT>
__device__ __forceinline__ void st_b16(uint16_t* p, const uint32_t (&w)[(CPT + 1) / 2]) {
  if constexpr (CPT == 4) *reinterpret_cast<b16x4_u*>(p) = u32x2{w[0], w[1]};
  else *p = (uint16_t)w[0];
}

template <int FORM, int KP>
struct TileShape {
  static constexpr int CPT = FORM == kTileOne ? 1 : 4;
  static constexpr int GROUPS = FORM == kTileAny ? max_groups(KP) : kGroups;  // at most
  static constexpr int NC = GROUPS * CPT;                                 // columns, at most
};

// A lane's element offset in its matrix, from its row slice and column: 32 bits, so
// that it is one register beside a uniform base per row, and 64 in the form that
// matrices too large for it take (rows past K are not accessed: their offset may wrap).
template <int FORM>
using LaneOffset = std::conditional_t<FORM == kTileOne, int64_t, uint32_t>;

// A thread's place in its tile: column group, slice, first column (-1: none).
struct TilePlace {
  int cg, ks, col;
};
template <int FORM, int S>
__device__ __forceinline__ TilePlace tile_place(const ColTiles& tiles, int V, int vt) {
  constexpr int CPT = FORM == kTileOne ? 1 : 4;
  TilePlace pl;
  if constexpr (FORM == kTileAny) {
    const int t = min((int)threadIdx.x, tiles.groups * S - 1);
    pl.ks = (int)((uint32_t)t * tiles.inv >> 16);
    pl.cg = t - pl.ks * tiles.groups;
  } else {
    pl.cg = threadIdx.x % kGroups;
    pl.ks = threadIdx.x / kGroups;
  }
  const int c0 = vt * tiles.width + pl.cg * CPT;
  pl.col = c0 < V ? min(c0, V - CPT) : -1;
  return pl;
}

// Low bytes of the CPT codes, column j in byte j.
template <int CPT>
__device__ __forceinline__ uint32_t pack_codes(const uint32_t (&yb)[CPT]) {
  if constexpr (CPT == 4) return pack_low_bytes(yb[0], yb[1], yb[2], yb[3]);
  else return yb[0] & 0xffu;
}

// Bitwise OR of the addresses: its low bits are zero only if every pointer is
// aligned that far.
template <typename... P>
inline uintptr_t addr_bits(const P*... ptrs) {
  return (reinterpret_cast<uintptr_t>(ptrs) | ... | (uintptr_t)0);
}

// ---------------------------------------------------------------------------
// Quantizing a float state per column: scale = max(amax, 1e-12) / qmax, code =
// rne(x / scale). Two forms, equal on finite values of ordinary size:
//  IEEE: the quotient is an IEEE division's and the code is clamped, for columns
//    that hold infinities or NaN as well.
//  otherwise the reciprocal's quotient without the clamp, which cannot bind on
//    finite values; the shapes below have always had this form.
// ---------------------------------------------------------------------------
inline bool ingest_ieee(uintptr_t bits, int64_t M, int K, int V) {
  return !((bits & 15) == 0 && V % 4 == 0 && M <= 65535 && K >= 16 && K <= 256 && (K & (K - 1)) == 0);
}

// Amax of column `col` over the slices' maxima. The slices combine to eighths
// of the rows in IEEE order; across those the non-IEEE form takes the unsigned
// order of group_max (an eighth of NaNs only stays NaN).
template <bool IEEE, int S, int NC>
__device__ __forceinline__ float ingest_amax(const float (*red)[NC], int col) {
  float am = 0.0f;
#pragma unroll
  for (int i = 0; i < S; i += S / 8) {
    const float x = S == 8 ? red[i][col] : fmaxf(red[i][col], red[i + S / 8 - 1][col]);
    am = IEEE ? fmaxf(am, x) : __uint_as_float(max(__float_as_uint(am), __float_as_uint(x)));
  }
  return am;
}

// The code of x in the low byte; inv = recip_rn(s).
template <bool IEEE>
__device__ __forceinline__ uint32_t ingest_code(float x, float s, float inv, float qmax) {
  uint32_t yb;
  if constexpr (IEEE) {
    float q = exact_quotient(x, s, inv);
    if (!(s < 0x1p125f)) q = x / s;  // the reciprocal is no normal number
    yb = __float_as_uint(fminf(fmaxf(rintf(q), -qmax), qmax) + kMagic);
  } else {
    (void)quantize<kExact>(x, s, inv, yb);
  }
  return yb;
}

}  // namespace qs
}  // namespace ck
