// Fused decode for any pool row length K in 1 .. 1024 and any row alignment:
// the reference masks its K lanes with o_k < K and loads zeros past K
// (vllm_integration/quantized_packed_decode.py:123-127, :158, :165-166,
// :196-202; BK = next_pow2(K) at :303), so a row of
// K codes computes as the same row padded with zeros to KP, the power of two
// >= max(K, 16) that the reference's BK also rounds to. This kernel runs the
// arithmetic of packed_decode_impl.h (process_item) on that padded row: the
// lane map of KP, every value past K zero in registers, stores of the K
// existing bytes only. A lane's codes come and go in one access of any
// alignment, two for rows of less than a lane (packed_decode_impl.h, kMaskLanes,
// kMaskTail and kMaskShort); the activations
// are loaded as raw words first, the state after them, and decoded while it is
// in flight. One item per workgroup. The bandwidth kernels cover aligned pools
// of the power-of-two K of real models, this one every other shape.
#pragma once

#include "ck_row_offset.h"
#include "packed_decode_impl.h"

namespace ck {
namespace pd {

// The register budget: the one-item kernel's.
template <int RPL, int WAVES, bool PER_HEAD>
constexpr int kMaskedWavesPerEU = kSingleWavesPerEU<RPL, WAVES, PER_HEAD>;

// The activations of one item, loaded as the aligned dwords that hold them and
// decoded later: byte offsets, from the token's row rounded down to a dword, of
// the rows' v and of this thread's share of [q | k], each padded to KP.
template <int KP, int RPL, int RPI, int QKT, int NT>
struct MaskedActs {
  const char* row;       // 4-byte aligned
  uint32_t v[RPL], qk[QKT];
  bool qk_in[QKT];       // not past p.K
  int dt;

  __device__ __forceinline__ MaskedActs(const PackedParams& p, const ItemCoord& ic, int row0) {
    dt = p.mixed_dtype();
    const int sh = dt == kF32 ? 2 : 1;
    const char* base = static_cast<const char*>(p.mixed) + (((int64_t)ic.n * p.stride_mixed) << sh);
    const uint32_t mis = (uint32_t)reinterpret_cast<uintptr_t>(base) & 3u;
    row = base - mis;
    const uint32_t v0 = 2u * p.H * p.K + (uint32_t)ic.hv * p.V;
    const uint32_t q0 = fdiv((uint32_t)ic.hv, p.div_grp) * p.K;
    const uint32_t v_last = ((v0 + (uint32_t)p.V - 1u) << sh) + mis;  // rows past V re-read row V-1
#pragma unroll
    for (int i = 0; i < RPL; ++i) v[i] = min(((v0 + (uint32_t)row0) << sh) + mis + ((uint32_t)(i * RPI) << sh), v_last);
#pragma unroll
    for (int j = 0; j < QKT; ++j) {
      const uint32_t e = min(threadIdx.x + j * NT, 2u * KP - 1u);
      const uint32_t kk = e & (KP - 1);
      qk_in[j] = kk < (uint32_t)p.K;
      qk[j] = ((q0 + min(kk, (uint32_t)p.K - 1u) + (e >= KP ? (uint32_t)(p.H * p.K) : 0u)) << sh) + mis;
    }
  }
  __device__ __forceinline__ uint32_t word(uint32_t off) const { return ld_at<uint32_t>(row, off & ~3u); }
  __device__ __forceinline__ uint32_t decode(uint32_t off, uint32_t w) const {
    if (dt == kF32) return w;
    const uint32_t h = w >> ((off & 2u) * 8u);
    return dt == kBF16 ? h << 16 : __float_as_uint(act_decode<kF16>(h));
  }
};

// The state of one live item, zero past p.K (kMaskTail: shifted at use).
template <int KP, int RPL, int WAVES, int RESID, bool PER_HEAD, int MASK>
__device__ __forceinline__ void load_item_masked(const PackedParams& p, const ItemCoord& ic, int row0, int c,
                                                 ItemRegs<RPL, Layout<KP, RPL, WAVES, RESID, PER_HEAD>::EW,
                                                          Layout<KP, RPL, WAVES, RESID, PER_HEAD>::QKT>& R) {
  using L = Layout<KP, RPL, WAVES, RESID, PER_HEAD>;
  constexpr int RKL = L::RK / L::LPR;  // residual bytes per lane: 8 (int4) or 16 (int8)
  // rows of whole lanes stream; a ragged row's ends share lines with other
  // instructions' rows, which cached loads read once (B=64, HV=32, V=128, us,
  // non-temporal against cached: K=100 int4 per head 28.1 / 25.0, int8 per row
  // 27.9 / 25.1; K=48 int4 per row 10.4 / 11.4; K=240 int4 per head B=8 9.3 / 10.1)
  constexpr bool STREAM = MASK == kMaskLanes;
  const int K = p.K;
  const int RKA = RESID == kResidInt4 ? K / 2 : K;
  const int8_t* sbase = p.state + ic.slot * p.stride_state + (int64_t)ic.hv * p.V * K;
  const int8_t* ebase = p.resid + ic.slot * p.stride_resid + (int64_t)ic.hv * p.V * RKA;
  const float* scb = p.sscale + ic.slot * p.stride_sscale + (int64_t)ic.hv * p.V;
  const float* rsb = p.rscale + ic.slot * p.stride_rscale + (int64_t)ic.hv * p.V;
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    const uint32_t r = (uint32_t)min(row0 + i * L::RPI, p.V - 1);  // rows past V re-read row V-1 (never stored)
    R.s_in[i] = ld_at<float>(scb, r * 4u);
    if constexpr (!PER_HEAD) R.es_in[i] = ld_at<float>(rsb, r * 4u);
  }
  if constexpr (PER_HEAD) R.es_in[0] = p.rscale[ic.slot * p.stride_rscale + ic.hv];
  if constexpr (MASK == kMaskShort) {  // one lane per row
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
      uint32_t w[4], e[L::EW];
      ld_pieces(sbase + clamped_row_offset(row0, i * L::RPI, K, p.V), K, w);
      ld_pieces(ebase + clamped_row_offset(row0, i * L::RPI, RKA, p.V), RKA, e);
      R.cw[i] = u32x4{w[0], w[1], w[2], w[3]};
#pragma unroll
      for (int j = 0; j < L::EW; ++j) R.ew[i][j] = e[j];
    }
  } else {
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
      R.cw[i] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < L::EW; ++j) R.ew[i][j] = 0u;
    }
    if (c * 16 < K) {
      // K >= 16 here, so the piece that ends with the row starts inside it
      const int sc = min(c * 16, K - 16), ec = min(c * RKL, RKA - RKL);
#pragma unroll
      for (int i = 0; i < RPL; ++i) {
        R.cw[i] = ld_16_u<STREAM>(sbase + (clamped_row_offset(row0, i * L::RPI, K, p.V) + (uint32_t)sc));
        const int8_t* e = ebase + (clamped_row_offset(row0, i * L::RPI, RKA, p.V) + (uint32_t)ec);
        if constexpr (RESID == kResidInt4) {
          const u32x2 e2 = ld_8_u<STREAM>(e);
          R.ew[i][0] = e2.x, R.ew[i][1] = e2.y;
        } else {
          const u32x4 e4 = ld_16_u<STREAM>(e);
          R.ew[i][0] = e4.x, R.ew[i][1] = e4.y, R.ew[i][2] = e4.z, R.ew[i][3] = e4.w;
        }
      }
    }
  }
}

template <int KP, int RPL, int WAVES, int RESID, bool PER_HEAD, int MODE, bool DST, int MASK>
__global__ __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(kMaskedWavesPerEU<RPL, WAVES, PER_HEAD>)))
void packed_decode_masked_kernel(const PackedParams p, const int32_t* __restrict__ idx,
                                 const int32_t* __restrict__ dst_idx) {
  using L = Layout<KP, RPL, WAVES, RESID, PER_HEAD>;
  __shared__ __attribute__((aligned(16))) float s_qk[4][2 * KP];  // [parity] staged, [2 + parity] raw
  __shared__ float s_red[2][WAVES];
  __shared__ float4 s_ek[1];  // unused: the per-head residual waits in VGPRs (EK_REGS)
  __shared__ float2 s_gate[1];

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int c = lane % L::LPR;
  const int g = lane / L::LPR;
  const Geom gm = geom_of(p);
  const ItemCoord ic = xcd_item_coord<DST>(p, gm, idx, dst_idx, (int)blockIdx.x, gm.share_n);  // share_n: xcd_base
  const int row0 = ic.vt * L::ROWS_WG + wave * L::ROWS_WAVE + g;
  const GateBits gbits = load_item_gate_bits(p, ic);  // before the item's loads (see stage_item_gates)
  ItemRegs<RPL, L::EW, L::QKT> R{};
  if (ic.live) load_item_masked<KP, RPL, WAVES, RESID, PER_HEAD, MASK>(p, ic, row0, c, R);
  __builtin_amdgcn_sched_barrier(0);
  const MaskedActs<KP, RPL, L::RPI, L::QKT, L::NT> acts(p, ic, row0);
  if (ic.live) {
#pragma unroll
    for (int j = 0; j < L::QKT; ++j) R.qk[j] = acts.word(acts.qk[j]);
#pragma unroll
    for (int i = 0; i < RPL; ++i) R.vv[i] = acts.word(acts.v[i]);
  }
  // wave 0 evaluates this item's gates into LDS, its loads in flight
  stage_item_gates(p, gbits, wave, lane, s_gate);
  if (ic.live) {  // (process_item runs with ACT = fp32 whatever the activation dtype)
#pragma unroll
    for (int j = 0; j < L::QKT; ++j) R.qk[j] = acts.qk_in[j] ? acts.decode(acts.qk[j], R.qk[j]) : 0u;
#pragma unroll
    for (int i = 0; i < RPL; ++i) R.vv[i] = acts.decode(acts.v[i], R.vv[i]);
  }
  if (PER_HEAD && threadIdx.x < WAVES) s_red[0][threadIdx.x] = 0.0f;  // a launch may have fewer waves
  __syncthreads();
  const float2 gab = s_gate[0];
  process_item<KP, RPL, WAVES, RESID, PER_HEAD, MODE, kF32, DST, MASK, true>(p, ic, row0, c, lane, wave, 0, gab.x,
                                                                            gab.y, R, s_qk, s_red, s_ek);
}

template <int KP, int RPL, int WAVES, int RESID, bool PER_HEAD, int MODE, bool DST, int MASK>
int launch_masked_cfg(PackedParams p, int B, hipStream_t stream) {
  using L = Layout<KP, RPL, WAVES, RESID, PER_HEAD>;
  const int nvt = PER_HEAD ? 1 : (p.V + L::ROWS_WG - 1) / L::ROWS_WG;
  const int64_t items = (int64_t)B * p.HV * nvt;
  if (items > 0x7fffffff) return fail(CK_EUNSUPPORTED, "%lld work items is too many", (long long)items);
  if (items == 0) return ok();
  const int64_t per_request = (int64_t)p.HV * nvt, most = max_workgroups(WAVES * 64);
  if (items > most) {  // consecutive launches over slices of the requests
    if (per_request > most) return fail(CK_EUNSUPPORTED, "%lld work items per request is too many", (long long)per_request);
    const int chunk = (int)(most / per_request);
    for (int64_t n0 = 0; n0 < B; n0 += chunk) {
      const int n = (int)min((int64_t)chunk, B - n0);
      const int rc = launch_masked_cfg<KP, RPL, WAVES, RESID, PER_HEAD, MODE, DST, MASK>(requests_from(p, (int)n0), n,
                                                                                       stream);
      if (rc != CK_OK) return rc;
    }
    return ok();
  }
  p.items = (int)items;
  p.div_nvt = make_fastdiv((uint32_t)nvt);
  p.div_hv = make_fastdiv((uint32_t)p.HV);
  p.cu_share_n = xcd_base(B, p.HV * nvt);  // the base of xcd_item_coord
  p.cu_shares = 0;
  // a head of fewer rows than the shape's takes the waves that hold a row (and
  // those that q and k take one value a thread from)
  int waves = WAVES;
  if (PER_HEAD && L::QKT == 1) waves = max((p.V + L::ROWS_WAVE - 1) / L::ROWS_WAVE, (2 * KP + 63) / 64);
  hipLaunchKernelGGL((packed_decode_masked_kernel<KP, RPL, WAVES, RESID, PER_HEAD, MODE, DST, MASK>), dim3((unsigned)items),
                     dim3((unsigned)min(waves, WAVES) * 64), 0, stream, p, p.idx, p.dst_idx);
  return check_launch("ck_gdn_packed_decode");
}

// Shapes. Per-row residual scales: 4 waves of two rows per lane from 1024 such
// tiles on, below that (and above K = 256) of one row, which spreads a small
// batch over more SIMDs (HV=16, V=100, K=100 int8, us, one row / two rows: B=24,
// 768 tiles 8.1 / 8.3; B=64, 2048 tiles 15.0 / 14.3; B=128 24.9 / 23.2); one row
// also where four waves of it cover the head, which two rows would leave to one or
// two of them (B=64, HV=32, us, one / two: K=36 V=64 int4 exact 10.6 / 12.3, K=200
// V=16 12.3 / 14.4, K=8 V=128 int8 8.3 / 9.3).
// A per-head scale needs the whole head in one workgroup: at KP=64 and 128 a
// head that four or eight waves of two rows per lane hold takes those, at
// KP=256 sixteen (fewer registers than four rows per lane, so more workgroups
// per CU), otherwise the fewest waves of four rows per lane that cover V. Waves
// that would hold no row of the head are not launched (per head) or skip the
// row work.
// Against the kernel that loaded 16-byte lanes, words or bytes by K and
// alignment, converted each activation next to its load and computed rows past
// V (B=64, HV=32, us): K=100 V=128 int4 per head 31.2 -> 25.0, int8 per row
// 28.7 -> 25.1; K=96 V=96 int4 per head 25.5 -> 21.4; K=200 int4 per head 82 ->
// 66; K=44 24.4 -> 15.1; K=101 V=77 int8 per head 83.5 -> 20.6; K=251 int8 per
// row 286 -> 69; K=34 V=64 int4 per head exact 23.1 -> 11.5.
template <int KP, int RESID, bool PER_HEAD, int MODE, bool DST, int MASK>
int launch_masked_shape(const PackedParams& p, int B, hipStream_t s) {
  constexpr int RPI = 64 / (KP / 16);
  if constexpr (!PER_HEAD) {
    if (KP <= 256 && p.V > RPI * 4 && (int64_t)B * p.HV * ((p.V + RPI * 8 - 1) / (RPI * 8)) >= 1024)
      return launch_masked_cfg<KP, 2, 4, RESID, false, MODE, DST, MASK>(p, B, s);
    return launch_masked_cfg<KP, 1, 4, RESID, false, MODE, DST, MASK>(p, B, s);
  } else {
    if constexpr (KP == 128) {
      if (p.V > RPI * 4 * 2 && p.V <= RPI * 2 * 8) return launch_masked_cfg<KP, 2, 8, RESID, true, MODE, DST, MASK>(p, B, s);
    }
    if constexpr (KP == 256) {
      if (p.V > RPI * 4 * 4 && p.V <= RPI * 2 * 16)
        return launch_masked_cfg<KP, 2, 16, RESID, true, MODE, DST, MASK>(p, B, s);
    }
    if constexpr (KP == 64) {
      if (p.V > RPI * 2 && p.V <= RPI * 2 * 4) return launch_masked_cfg<KP, 2, 4, RESID, true, MODE, DST, MASK>(p, B, s);
    }
    if (p.V <= RPI * 4 * 1) return launch_masked_cfg<KP, 4, 1, RESID, true, MODE, DST, MASK>(p, B, s);
    if (p.V <= RPI * 4 * 2) return launch_masked_cfg<KP, 4, 2, RESID, true, MODE, DST, MASK>(p, B, s);
    if (p.V <= RPI * 4 * 4) return launch_masked_cfg<KP, 4, 4, RESID, true, MODE, DST, MASK>(p, B, s);
    if (p.V <= RPI * 4 * 8) return launch_masked_cfg<KP, 4, 8, RESID, true, MODE, DST, MASK>(p, B, s);
    // rows of 512 or 1024 codes: 2 or 1 rows per wave instruction, so a head
    // of V = 128 or 64 rows takes 16 waves of 4 rows per lane
    constexpr int kMaxWaves = KP >= 512 ? 16 : 8;
    if constexpr (KP >= 512) {
      if (p.V <= RPI * 4 * 16) return launch_masked_cfg<KP, 4, 16, RESID, true, MODE, DST, MASK>(p, B, s);
    }
    return fail(CK_EUNSUPPORTED, "per-head residual scale supports V <= %d at K=%d, got V=%d", RPI * 4 * kMaxWaves,
                p.K, p.V);
  }
}

// Dispatch over residual format, scale granularity, mode and destination for
// one padded K and access mode.
template <int KP, int MASK>
int launch_masked_mode(const PackedParams& p, int B, int resid_fmt, int per_head, int mode, hipStream_t s) {
  const bool i4 = resid_fmt == CK_RESID_INT4;
  if (p.dst_idx) {  // out-of-place step: instantiated for the FAST arithmetic only
    if (mode != kFast) return fail(CK_EUNSUPPORTED, "dst_state_indices needs quant_mode FAST");
    return i4 ? (per_head ? launch_masked_shape<KP, kResidInt4, true, kFast, true, MASK>(p, B, s)
                          : launch_masked_shape<KP, kResidInt4, false, kFast, true, MASK>(p, B, s))
              : (per_head ? launch_masked_shape<KP, kResidInt8, true, kFast, true, MASK>(p, B, s)
                          : launch_masked_shape<KP, kResidInt8, false, kFast, true, MASK>(p, B, s));
  }
  if (mode == kFast)
    return i4 ? (per_head ? launch_masked_shape<KP, kResidInt4, true, kFast, false, MASK>(p, B, s)
                          : launch_masked_shape<KP, kResidInt4, false, kFast, false, MASK>(p, B, s))
              : (per_head ? launch_masked_shape<KP, kResidInt8, true, kFast, false, MASK>(p, B, s)
                          : launch_masked_shape<KP, kResidInt8, false, kFast, false, MASK>(p, B, s));
  return i4 ? (per_head ? launch_masked_shape<KP, kResidInt4, true, kExact, false, MASK>(p, B, s)
                        : launch_masked_shape<KP, kResidInt4, false, kExact, false, MASK>(p, B, s))
            : (per_head ? launch_masked_shape<KP, kResidInt8, true, kExact, false, MASK>(p, B, s)
                        : launch_masked_shape<KP, kResidInt8, false, kExact, false, MASK>(p, B, s));
}

template <int KP>
int launch_masked_k(const PackedParams& p, int B, int resid_fmt, int per_head, int mode, hipStream_t s);

#define CK_PD_DEFINE_MASKED_FOR_K(KP)                                                                        \
  template <>                                                                                                \
  int launch_masked_k<KP>(const PackedParams& p, int B, int resid_fmt, int per_head, int mode,               \
                          hipStream_t s) {                                                                   \
    if (p.K % 16 == 0) return launch_masked_mode<KP, kMaskLanes>(p, B, resid_fmt, per_head, mode, s);        \
    constexpr int kRest = KP == 16 ? kMaskShort : kMaskTail;                                                 \
    return launch_masked_mode<KP, kRest>(p, B, resid_fmt, per_head, mode, s);                                \
  }

}  // namespace pd
}  // namespace ck
