// Fused GDN decode step in the statequant layout: state [B, HV, K, V] int8
// (V contiguous) with one scale per V-column (amax over K), error-feedback
// residual stored as fp32, fp16, fp8 e5m2 or int8 with a per-column scale.
// Out of place (in place also works: a workgroup reads its whole tile before
// writing it). Counterpart of statequant/kernel.py:260-341 (_gdn_quant_kernel),
// cuda/gdn_state_kernel.cu:141-246 and the launcher at :310-348; plus the fp32
// baseline step (statequant/kernel.py:211-248, cuda/gdn_state_kernel.cu:251-297).
//
// Work mapping. A workgroup covers one (request, head) and a tile of column
// groups; a thread owns one group of consecutive V-columns and one of S K-slices:
// S = 8 slices of K/8 rows for K <= 128, S = 16 slices of 16 rows at K = 256, so
// a thread's rows always fit its registers. Column sums over K are a sequential
// fma chain over the
// thread's rows, then the S slice partials are combined through LDS by a
// balanced pairwise tree (S = 8: ((s0+s1)+(s2+s3))+((s4+s5)+(s6+s7))). Four
// such exchanges per step (h.k, h.q, amax, and the int8 residual's amax), one
// barrier each.
//
// Any K in 1..256: the reference's CUDA launcher loops over its K rows
// (cuda/gdn_state_kernel.cu:141-246) and the Triton kernel masks its BK =
// next_pow2(K) rows (statequant/kernel.py:277-279). Here the rows are padded
// with zeros to KP = max(16, next_pow2(K)) and the KP kernel runs on them (MK:
// rows at or past K load nothing, contribute zero products and zero to every
// amax, and store nothing), so the sums keep the KP slice order.
//
// Columns per thread: four, one vector access per row at any alignment, with as
// many column groups in a workgroup as the tile's width needs or 32 (ck_tiles.h,
// TileForm); one column for V < 4 and from 2^32 elements on. Before, any V but a multiple of 4 with
// 16-byte aligned tensors took one column per thread, 32 to a workgroup (HV=32, us
// a call: K=100 V=130 B=16 fp32 residual 28.0 -> 18.2, fp16 25.1 -> 15.8, where the
// host's share is 15; K=256 V=130 B=16 fp32 70.0 -> 51.3, int8 48.5 -> 39.4;
// K=200 V=33 B=32 fp32 28.1 -> 18.1; fp32 step K=200 V=33 19.4 -> 11.7).
//
// Row addresses are a uniform base per row and one 32-bit lane offset (LaneOffset):
// as 64-bit lane addresses they held 16 to 20 VGPRs more, at K=128 one workgroup
// per CU with the fp16 residual (178 -> 162 VGPRs) and the fp32 step (146 -> 127).
// HV=32, K=V=128, B=64, us: fp16 39.2 -> 37.1, fp8 29.6 -> 28.1, int8 31.5 -> 30.7,
// fp32 level; V=130 K=100 B=16: fp8 15.5 -> 13.5, fp32 step 13.1 -> 10.7. k and q in
// LDS instead of registers freed 20 more and was slower (fp32 67.3, fp16 38.3):
// their load, a barrier and the LDS reads come before the first sum.
#include <hip/hip_runtime.h>

#include "ck_capi_common.h"
#include "ck_device.h"
#include "ck_quant.h"
#include "ck_statequant.h"

namespace ck {
namespace qs {

struct StepParams {
  const int8_t* h_in;
  const float* scale_in;
  const void* e_in;
  const float* e_scale_in;
  const float* q;
  const float* k;
  const float* v;
  const float* alpha;
  const float* beta;
  float* o;
  int8_t* h_out;
  float* scale_out;
  void* e_out;
  float* e_scale_out;
  int HV, V;
  ColTiles tiles;
  int K;  // rows that exist (the kernel's K template argument is the padded count)
  float qmax, rqmax;
};

template <int K, int RES, int MODE, int FORM, bool MK>
__global__ __launch_bounds__((kThreadsFor<K, TileShape<FORM, K>::GROUPS>)) void quant_step_kernel(const StepParams p) {
  constexpr int CPT = TileShape<FORM, K>::CPT;
  constexpr int S = kSlicesFor<K>;
  constexpr int RPS = K / S;            // rows per slice
  constexpr int NC = TileShape<FORM, K>::NC;  // columns per workgroup, at most
  __shared__ float red[4][S][NC];

  const int vt = blockIdx.x % p.tiles.nvt;
  const int w = blockIdx.x / p.tiles.nvt;  // (request, head)
  const TilePlace pl = tile_place<FORM, S>(p.tiles, p.V, vt);
  const int ks = pl.ks;
  const int lc = pl.cg * CPT;        // local column
  const int c0 = pl.col;
  const bool colok = c0 >= 0;
  const int r0 = ks * RPS;
  const int KA = MK ? p.K : K;       // rows that exist
  const int64_t mb = (int64_t)w * KA * p.V;
  const int64_t vb = (int64_t)w * p.V;
  const LaneOffset<FORM> off = (LaneOffset<FORM>)r0 * p.V + max(c0, 0);
  const float alpha = p.alpha[w];
  const float beta = p.beta[w];

  uint32_t cw[RPS];
  // the residual stays in its stored form until t = h + e (one dword per row
  // and 4 columns for 8-bit formats, two for fp16, four for fp32)
  constexpr int EWD = RES == kResFp32 ? CPT : RES == kResFp16 ? (CPT + 1) / 2 : 1;
  uint32_t ew[RPS][EWD];
  float sc[CPT], esc[CPT], vv[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) sc[j] = esc[j] = vv[j] = 0.f;
  float kk[RPS], qq[RPS];
#pragma unroll
  for (int r = 0; r < RPS; ++r) {
    kk[r] = qq[r] = 0.f;
    if (!MK || r0 + r < KA) {
      kk[r] = p.k[(int64_t)w * KA + r0 + r];
      qq[r] = p.q[(int64_t)w * KA + r0 + r];
    }
  }
  if (colok) {
    ld_f32<CPT>(p.scale_in + vb + c0, sc);
    ld_f32<CPT>(p.v + vb + c0, vv);
    if constexpr (RES == kResInt8) ld_f32<CPT>(p.e_scale_in + vb + c0, esc);
#pragma unroll
    for (int r = 0; r < RPS; ++r) {
      if (MK && r0 + r >= KA) {  // padding row: zero codes and residual (decodes to +0 in every format)
        cw[r] = 0;
#pragma unroll
        for (int j = 0; j < EWD; ++j) ew[r][j] = 0u;
        continue;
      }
      const int64_t i = mb + (int64_t)r * p.V;  // uniform; the lane's part is off
      cw[r] = ld_b8<CPT>(p.h_in + i + off);
      if constexpr (RES == kResFp32) {
        float e[CPT];
        ld_f32<CPT>(static_cast<const float*>(p.e_in) + i + off, e);
#pragma unroll
        for (int j = 0; j < CPT; ++j) ew[r][j] = __float_as_uint(e[j]);
      } else if constexpr (RES == kResFp16) {
        ld_b16<CPT>(static_cast<const uint16_t*>(p.e_in) + i + off, ew[r]);
      } else {
        ew[r][0] = ld_b8<CPT>(static_cast<const uint8_t*>(p.e_in) + i + off);
      }
    }
  } else {
#pragma unroll
    for (int r = 0; r < RPS; ++r) {
      cw[r] = 0;
#pragma unroll
      for (int j = 0; j < EWD; ++j) ew[r][j] = 0u;   // decodes to +0 in every format
    }
  }

  // dequantize + decay
  float h[RPS][CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const float sa = sc[j] * alpha;
#pragma unroll
    for (int r = 0; r < RPS; ++r) {
      const float code = code_i8(cw[r], j);
      h[r][j] = (MODE == kFast) ? code * sa : (code * sc[j]) * alpha;
    }
  }
  // rd = h^T k
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    float acc = h[0][j] * kk[0];
#pragma unroll
    for (int r = 1; r < RPS; ++r) acc = fmaf(h[r][j], kk[r], acc);
    red[0][ks][lc + j] = acc;
  }
  __syncthreads();
  float dv[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) dv[j] = beta * (vv[j] - slice_tree_sum<S, NC>(red[0], lc + j));
  // h += k dv; o = h^T q
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
#pragma unroll
    for (int r = 0; r < RPS; ++r) h[r][j] = madd<MODE>(kk[r], dv[j], h[r][j]);
    float acc = h[0][j] * qq[0];
#pragma unroll
    for (int r = 1; r < RPS; ++r) acc = fmaf(h[r][j], qq[r], acc);
    red[1][ks][lc + j] = acc;
  }
  // t = h + e (the residual decoded here)
#pragma unroll
  for (int r = 0; r < RPS; ++r) {
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      float ev;
      if constexpr (RES == kResFp32) {
        ev = __uint_as_float(ew[r][j]);
      } else if constexpr (RES == kResFp16) {
        ev = half_bits_to_f32(j % 2 ? ew[r][j / 2] >> 16 : ew[r][j / 2] & 0xffffu);
      } else if constexpr (RES == kResFp8) {
        ev = e5m2_byte(ew[r][0], j);
      } else {
        ev = code_i8(ew[r][0], j);
      }
      if constexpr (RES == kResInt8) {
        h[r][j] = madd<MODE>(ev, esc[j], h[r][j]);
      } else {
        h[r][j] = h[r][j] + ev;
      }
    }
  }
  // amax over K per column
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    float m = fabsf(h[0][j]);
#pragma unroll
    for (int r = 1; r < RPS; ++r) m = fmaxf(m, fabsf(h[r][j]));
    red[2][ks][lc + j] = m;
  }
  __syncthreads();
  if (ks == 0 && colok) {
    float o4[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) o4[j] = slice_tree_sum<S, NC>(red[1], lc + j);
    st_f32<CPT>(p.o + vb + c0, o4);
  }
  float s[CPT], inv[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    s[j] = fmaxf(div_small_int(slice_max<S, NC>(red[2], lc + j), p.qmax, p.rqmax), kEps);
    inv[j] = recip_rn(s[j]);
  }
  // requantize, store codes, form the residual
  float ea[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) ea[j] = 0.f;
#pragma unroll
  for (int r = 0; r < RPS; ++r) {
    uint32_t yb[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      const float code = quantize<MODE>(h[r][j], s[j], inv[j], yb[j]);
      h[r][j] = residual<MODE>(h[r][j], code, s[j]);
      ea[j] = fmaxf(ea[j], fabsf(h[r][j]));
    }
    if (colok && (!MK || r0 + r < KA)) st_b8<CPT>(p.h_out + mb + (int64_t)r * p.V + off, pack_codes<CPT>(yb));
  }
  if (ks == 0 && colok) st_f32<CPT>(p.scale_out + vb + c0, s);

  if constexpr (RES == kResInt8) {
#pragma unroll
    for (int j = 0; j < CPT; ++j) red[3][ks][lc + j] = ea[j];
    __syncthreads();
    float es[CPT], inv_e[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      es[j] = fmaxf(div_small_int(slice_max<S, NC>(red[3], lc + j), p.qmax, p.rqmax), kEps);
      inv_e[j] = recip_rn(es[j]);
    }
    if (colok) {
#pragma unroll
      for (int r = 0; r < RPS; ++r) {
        if (MK && r0 + r >= KA) continue;
        uint32_t eb[CPT];
#pragma unroll
        for (int j = 0; j < CPT; ++j) (void)quantize<MODE>(h[r][j], es[j], inv_e[j], eb[j]);
        st_b8<CPT>(static_cast<int8_t*>(p.e_out) + mb + (int64_t)r * p.V + off, pack_codes<CPT>(eb));
      }
      if (ks == 0) st_f32<CPT>(p.e_scale_out + vb + c0, es);
    }
  } else if (colok) {
#pragma unroll
    for (int r = 0; r < RPS; ++r) {
      if (MK && r0 + r >= KA) continue;
      const int64_t i = mb + (int64_t)r * p.V;
      if constexpr (RES == kResFp32) {
        st_f32<CPT>(static_cast<float*>(p.e_out) + i + off, h[r]);
      } else if constexpr (RES == kResFp16) {
        uint32_t hw[(CPT + 1) / 2];
#pragma unroll
        for (int j = 0; j < CPT; j += 2)
          hw[j / 2] = f32_to_half_bits(h[r][j]) | (j + 1 < CPT ? f32_to_half_bits(h[r][j + 1]) << 16 : 0u);
        st_b16<CPT>(static_cast<uint16_t*>(p.e_out) + i + off, hw);
      } else {
        st_b8<CPT>(static_cast<uint8_t*>(p.e_out) + i + off, f32_to_e5m2<CPT>(h[r]));
      }
    }
  }
}

struct Fp32Params {
  const float* h_in;
  const float* q;
  const float* k;
  const float* v;
  const float* alpha;
  const float* beta;
  float* o;
  float* h_out;
  int V;
  ColTiles tiles;
  int K;  // rows that exist (the kernel's K template argument is the padded count)
};

template <int K, int FORM, bool MK>
__global__ __launch_bounds__((kThreadsFor<K, TileShape<FORM, K>::GROUPS>)) void fp32_step_kernel(const Fp32Params p) {
  constexpr int CPT = TileShape<FORM, K>::CPT;
  constexpr int S = kSlicesFor<K>;
  constexpr int RPS = K / S;
  constexpr int NC = TileShape<FORM, K>::NC;
  __shared__ float red[2][S][NC];
  const int vt = blockIdx.x % p.tiles.nvt;
  const int w = blockIdx.x / p.tiles.nvt;
  const TilePlace pl = tile_place<FORM, S>(p.tiles, p.V, vt);
  const int ks = pl.ks;
  const int lc = pl.cg * CPT;
  const int c0 = pl.col;
  const bool colok = c0 >= 0;
  const int r0 = ks * RPS;
  const int KA = MK ? p.K : K;  // rows that exist
  const int64_t mb = (int64_t)w * KA * p.V;
  const int64_t vb = (int64_t)w * p.V;
  const LaneOffset<FORM> off = (LaneOffset<FORM>)r0 * p.V + max(c0, 0);
  const float alpha = p.alpha[w];
  const float beta = p.beta[w];
  float h[RPS][CPT], kk[RPS], qq[RPS], vv[CPT];
#pragma unroll
  for (int r = 0; r < RPS; ++r) {
    const bool rin = !MK || r0 + r < KA;
    kk[r] = qq[r] = 0.f;
    if (rin) {
      kk[r] = p.k[(int64_t)w * KA + r0 + r];
      qq[r] = p.q[(int64_t)w * KA + r0 + r];
    }
    float x[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) x[j] = 0.f;
    if (colok && rin) ld_f32<CPT>(p.h_in + mb + (int64_t)r * p.V + off, x);
#pragma unroll
    for (int j = 0; j < CPT; ++j) h[r][j] = x[j] * alpha;
  }
#pragma unroll
  for (int j = 0; j < CPT; ++j) vv[j] = 0.f;
  if (colok) ld_f32<CPT>(p.v + vb + c0, vv);
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    float acc = h[0][j] * kk[0];
#pragma unroll
    for (int r = 1; r < RPS; ++r) acc = fmaf(h[r][j], kk[r], acc);
    red[0][ks][lc + j] = acc;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const float dv = beta * (vv[j] - slice_tree_sum<S, NC>(red[0], lc + j));
#pragma unroll
    for (int r = 0; r < RPS; ++r) h[r][j] = fmaf(kk[r], dv, h[r][j]);
    float acc = h[0][j] * qq[0];
#pragma unroll
    for (int r = 1; r < RPS; ++r) acc = fmaf(h[r][j], qq[r], acc);
    red[1][ks][lc + j] = acc;
  }
  if (colok) {
#pragma unroll
    for (int r = 0; r < RPS; ++r)
      if (!MK || r0 + r < KA) st_f32<CPT>(p.h_out + mb + (int64_t)r * p.V + off, h[r]);
  }
  __syncthreads();
  if (ks == 0 && colok) {
    float o4[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) o4[j] = slice_tree_sum<S, NC>(red[1], lc + j);
    st_f32<CPT>(p.o + vb + c0, o4);
  }
}

template <int K, int MODE, int FORM, bool MK>
int launch_quant(const StepParams& p, int64_t grid, int res_fmt, hipStream_t s) {
  const dim3 g((unsigned)grid), b((unsigned)tile_threads(p.tiles, kSlicesFor<K>));
  switch (res_fmt) {
    case kResFp32: hipLaunchKernelGGL((quant_step_kernel<K, kResFp32, MODE, FORM, MK>), g, b, 0, s, p); break;
    case kResFp16: hipLaunchKernelGGL((quant_step_kernel<K, kResFp16, MODE, FORM, MK>), g, b, 0, s, p); break;
    case kResFp8: hipLaunchKernelGGL((quant_step_kernel<K, kResFp8, MODE, FORM, MK>), g, b, 0, s, p); break;
    default: hipLaunchKernelGGL((quant_step_kernel<K, kResInt8, MODE, FORM, MK>), g, b, 0, s, p); break;
  }
  return check_launch("ck_gdn_quant_step");
}

template <int MODE, int FORM, bool MK>
int launch_quant_kp(const StepParams& p, int64_t grid, int KP, int res_fmt, hipStream_t s) {
  switch (KP) {
    case 16: return launch_quant<16, MODE, FORM, MK>(p, grid, res_fmt, s);
    case 32: return launch_quant<32, MODE, FORM, MK>(p, grid, res_fmt, s);
    case 64: return launch_quant<64, MODE, FORM, MK>(p, grid, res_fmt, s);
    case 128: return launch_quant<128, MODE, FORM, MK>(p, grid, res_fmt, s);
    default: return launch_quant<256, MODE, FORM, MK>(p, grid, res_fmt, s);
  }
}

template <int MODE, int FORM>
int launch_quant_k(const StepParams& p, int64_t grid, int res_fmt, hipStream_t s) {
  const int KP = padded_k(p.K);
  return KP == p.K ? launch_quant_kp<MODE, FORM, false>(p, grid, KP, res_fmt, s)
                   : launch_quant_kp<MODE, FORM, true>(p, grid, KP, res_fmt, s);
}

template <int MODE>
int launch_quant_form(const StepParams& p, int64_t grid, int res_fmt, hipStream_t s) {
  switch (p.tiles.form) {
    case kTileFull: return launch_quant_k<MODE, kTileFull>(p, grid, res_fmt, s);
    case kTileAny: return launch_quant_k<MODE, kTileAny>(p, grid, res_fmt, s);
    default: return launch_quant_k<MODE, kTileOne>(p, grid, res_fmt, s);
  }
}

template <int FORM, bool MK>
int launch_fp32_kp(const Fp32Params& p, int64_t grid, int KP, hipStream_t s) {
  const dim3 g((unsigned)grid), b((unsigned)tile_threads(p.tiles, KP <= 128 ? 8 : 16));
  switch (KP) {
    case 16: hipLaunchKernelGGL((fp32_step_kernel<16, FORM, MK>), g, b, 0, s, p); break;
    case 32: hipLaunchKernelGGL((fp32_step_kernel<32, FORM, MK>), g, b, 0, s, p); break;
    case 64: hipLaunchKernelGGL((fp32_step_kernel<64, FORM, MK>), g, b, 0, s, p); break;
    case 128: hipLaunchKernelGGL((fp32_step_kernel<128, FORM, MK>), g, b, 0, s, p); break;
    default: hipLaunchKernelGGL((fp32_step_kernel<256, FORM, MK>), g, b, 0, s, p); break;
  }
  return check_launch("ck_gdn_fp32_step");
}

template <int FORM>
int launch_fp32(const Fp32Params& p, int64_t grid, hipStream_t s) {
  const int KP = padded_k(p.K);
  return KP == p.K ? launch_fp32_kp<FORM, false>(p, grid, KP, s) : launch_fp32_kp<FORM, true>(p, grid, KP, s);
}

}  // namespace qs
}  // namespace ck

extern "C" int ck_gdn_quant_step(const int8_t* h_in, const float* scale_in, const void* e_in,
                                 const float* e_scale_in,
                                 const float* q, const float* k, const float* v,
                                 const float* alpha, const float* beta,
                                 float* o, int8_t* h_out, float* scale_out, void* e_out, float* e_scale_out,
                                 int B, int HV, int K, int V, float qmax, int res_fmt, int quant_mode,
                                 void* stream) {
  using namespace ck;
  using namespace ck::qs;
  if (B < 0 || HV <= 0 || K <= 0 || V <= 0) return fail(CK_EINVAL, "bad sizes B=%d HV=%d K=%d V=%d", B, HV, K, V);
  if (!valid_k(K)) return fail(CK_EUNSUPPORTED, "K must be in 1..256, got %d", K);
  if (res_fmt < CK_RES_FP32 || res_fmt > CK_RES_INT8) return fail(CK_EINVAL, "unknown residual format %d", res_fmt);
  if (quant_mode != CK_QUANT_FAST && quant_mode != CK_QUANT_EXACT)
    return fail(CK_EINVAL, "quant_mode must be CK_QUANT_FAST or CK_QUANT_EXACT, got %d", quant_mode);
  const int iq = (int)qmax;
  if ((float)iq != qmax || iq < 1 || iq > 127) return fail(CK_EINVAL, "qmax must be an integer in 1..127");
  if (B == 0) return ok();
  if (!h_in || !scale_in || !e_in || !q || !k || !v || !alpha || !beta || !o || !h_out || !scale_out || !e_out)
    return fail(CK_EINVAL, "null pointer argument");
  if (res_fmt == CK_RES_INT8 && (!e_scale_in || !e_scale_out)) return fail(CK_EINVAL, "int8 residual needs e_scale");
  const bool int8_res = res_fmt == CK_RES_INT8;
  const uintptr_t fbits = addr_bits(scale_in, q, k, v, alpha, beta, o, scale_out) |
                          (int8_res ? addr_bits(e_scale_in, e_scale_out) : 0);
  const int esz = res_fmt == CK_RES_FP32 ? 4 : res_fmt == CK_RES_FP16 ? 2 : 1;
  const uintptr_t ebits = addr_bits(e_in, e_out);
  if ((fbits & 3) || (ebits & (esz - 1)))
    return fail(CK_EINVAL, "fp32 tensors must be 4-byte aligned and the residual %d-byte aligned", esz);
  StepParams p{};
  p.h_in = h_in;
  p.scale_in = scale_in;
  p.e_in = e_in;
  p.e_scale_in = e_scale_in;
  p.q = q;
  p.k = k;
  p.v = v;
  p.alpha = alpha;
  p.beta = beta;
  p.o = o;
  p.h_out = h_out;
  p.scale_out = scale_out;
  p.e_out = e_out;
  p.e_scale_out = e_scale_out;
  p.HV = HV;
  p.V = V;
  p.tiles = col_tiles(V, padded_k(K), res_fmt == CK_RES_FP32, false);
  p.K = K;
  volatile float one = 1.0f;
  p.qmax = qmax;
  p.rqmax = one / qmax;
  const int64_t grid = (int64_t)B * HV * p.tiles.nvt;
  if (grid > 0x7fffffff) return fail(CK_EUNSUPPORTED, "grid too large");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  return quant_mode == CK_QUANT_EXACT ? launch_quant_form<kExact>(p, grid, res_fmt, s)
                                      : launch_quant_form<kFast>(p, grid, res_fmt, s);
}

extern "C" int ck_gdn_fp32_step(const float* h_in, const float* q, const float* k, const float* v,
                                const float* alpha, const float* beta, float* o, float* h_out,
                                int B, int HV, int K, int V, void* stream) {
  using namespace ck;
  using namespace ck::qs;
  if (B < 0 || HV <= 0 || K <= 0 || V <= 0) return fail(CK_EINVAL, "bad sizes B=%d HV=%d K=%d V=%d", B, HV, K, V);
  if (!valid_k(K)) return fail(CK_EUNSUPPORTED, "K must be in 1..256, got %d", K);
  if (B == 0) return ok();
  if (!h_in || !q || !k || !v || !alpha || !beta || !o || !h_out) return fail(CK_EINVAL, "null pointer argument");
  const uintptr_t bits = addr_bits(h_in, q, k, v, alpha, beta, o, h_out);
  if (bits & 3) return fail(CK_EINVAL, "fp32 tensors must be 4-byte aligned");
  Fp32Params p{h_in, q, k, v, alpha, beta, o, h_out, V, col_tiles(V, padded_k(K), true, false), K};
  const int64_t grid = (int64_t)B * HV * p.tiles.nvt;
  if (grid > 0x7fffffff) return fail(CK_EUNSUPPORTED, "grid too large");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  switch (p.tiles.form) {
    case kTileFull: return launch_fp32<kTileFull>(p, grid, s);
    case kTileAny: return launch_fp32<kTileAny>(p, grid, s);
    default: return launch_fp32<kTileOne>(p, grid, s);
  }
}
