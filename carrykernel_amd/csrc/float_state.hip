// GDN decode step on an unquantized state pool (fp32 or bf16), vLLM's paged
// [slots, HV, V, K] layout, updated in place. This is the comparison arm for
// the quantized step: the semantics of the upstream packed decode that
// vllm_integration/quantized_packed_decode.py:1-7 replaces (same gates, GQA,
// optional L2 norm, NULL-slot padding), with vLLM's default bf16 state.
//
// It has the one-item form of the quantized decode (packed_decode_impl.h): one
// workgroup of 4 waves per (request, head, V-tile), a request's items on one
// XCD, the gates evaluated while the state loads, q/k staged in LDS, DPP row
// reductions. Per row:
//   h_j = h_j * alpha;  rd = sum_j h_j k_j;  dv = beta * (v - rd)
//   h_j = fma(k_j, dv, h_j);  o = sum_j h_j q_j;  state <- h (bf16: RNE)
//
// A lane computes 16 consecutive K of a row (a chunk: the sums' order), 64 bytes
// of fp32 or 32 of bf16, but its 16-byte accesses are not its own bytes: a load
// instruction takes 64 consecutive bytes per 4 lanes (fp32, K >= 128: 128 per 8
// lanes), and lanes swap the pieces by DPP (ChunkMap). Each lane loading its
// own bytes touched every line of the wave's rows in every instruction. HBM is
// the bound (the swaps are 2 VALU operations per fp32 element each way).
// Against the persistent kernel with a register prefetch and each lane's own
// bytes (HV=32, V=128, us), state sets that a last-level cache of 256 MB holds in
// part: bf16 K=128 B=64 31.7 -> 22.9 (192 MB in turn; with cold sets 30.3 -> 30.3, no
// gain); larger ones: bf16 B=128 60.7 -> 55.4 (4.9 TB/s), K=256 B=48 45.7 -> 40.2;
// fp32 K=128 B=8 12.6 -> 7.4, B=64 65.1 -> 50.5, B=128 122.6 -> 98.3 (5.6 TB/s), K=256
// B=48 91.9 -> 72.4.
#include <hip/hip_runtime.h>

#include "ck_capi_common.h"
#include "ck_device.h"
#include "packed_decode_impl.h"

namespace ck {
namespace fs {

using pd::ItemCoord;
using pd::PackedParams;

// 16-byte pieces of a chunk: 16 fp32 or 16 bf16.
template <bool BF16>
constexpr int kPieces = BF16 ? 2 : 4;

template <int RPL, int QKT, bool BF16>
struct FloatItemRegs {
  u32x4 sw[RPL][kPieces<BF16>];  // state, raw, as loaded
  uint32_t vv[RPL];              // v per row (raw activation bits)
  uint32_t qk[QKT];              // this thread's share of [q | k]
};

// Exchange with the lane whose index differs in the bit that `bit` tells: a
// becomes (own a, partner's a) where the bit is clear, (partner's b, own b)
// where it is set.
template <int CTRL>
__device__ __forceinline__ void swap_pieces(u32x4& a, u32x4& b, bool bit) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t x = a[j], y = b[j];
    const uint32_t px = dpp_u<CTRL>(x), py = dpp_u<CTRL>(y);
    a[j] = bit ? py : x;
    b[j] = bit ? y : px;
  }
}

// bf16 rows are cached, fp32 ones stream (us, cached / streaming loads: bf16 K=128
// B=64 24.5 / 30.3, B=128 55.9 / 56.3; fp32 K=128 B=8 9.3 / 7.8, B=64 54.5 / 50.8,
// B=128 109 / 98; cached stores bf16 B=64 23.2, fp32 no change).
// fp32 rows whose lanes take their own bytes (K = 16 and 32: an instruction touches
// a quarter of each line) are cached too (HV=32, B=200, us, streaming / cached: K=32
// V=128 77.2 / 42.0, V=200 125.6 / 59.0; K=16 V=128 46.1 / 25.7).
template <bool CACHED>
__device__ __forceinline__ u32x4 ld_state(const int8_t* p) {
  return CACHED ? ld_at<u32x4>(p, 0u) : ld_stream16(p);
}
template <bool CACHED>
__device__ __forceinline__ void st_state(int8_t* p, u32x4 v) {
  if constexpr (CACHED) st_at<u32x4>(p, 0u, v);
  else st_stream16(p, v);
}

// Which bytes of a row a lane's w-th access takes, which chunk it holds after
// the swaps, and the balanced tree over the chunks that this order needs.
// LPR lanes per row, c the lane's place among them.
//  bf16, LPR >= 4: access w of a quad is its 64 bytes 64 w ..; a swap of
//    neighbours leaves chunks 0, 2, 1, 3 in its lanes.
//  fp32, LPR = 4: access w is chunk w, a 4 x 4 transpose leaves chunk i in lane i.
//  fp32, LPR >= 8: access w is chunks 2 w (first quad of eight lanes) and 2 w + 1
//    (second quad); the transposes leave 0, 2, 4, 6 and, the second quad's
//    order turned round, 7, 5, 3, 1: a chunk's tree partner is the mirrored lane.
//  else (LPR <= 2): a lane's own bytes.
template <int LPR, bool BF16>
struct ChunkMap {
  static constexpr bool kSwap = LPR >= 4;
  static constexpr bool kEight = !BF16 && LPR >= 8;
  static constexpr bool kCached = BF16 || !kSwap;

  __device__ static __forceinline__ uint32_t piece_off(int c, int w) {  // byte offset in the row
    if constexpr (!kSwap) return (uint32_t)(c * kPieces<BF16> + w) * 16u;
    if constexpr (BF16) return (uint32_t)((c >> 2) * 8 + w * 4 + (c & 3)) * 16u;
    if constexpr (kEight) return (uint32_t)((c >> 3) * 32 + w * 8 + (c & 7)) * 16u;
    return (uint32_t)((c >> 2) * 16 + w * 4 + (c & 3)) * 16u;
  }
  __device__ static __forceinline__ int chunk(int c) {
    if constexpr (!kSwap) return c;
    const int i = c & 3;
    if constexpr (BF16) return (c & ~3) + (i >> 1) + 2 * (i & 1);
    if constexpr (kEight) return (c & ~7) + ((c & 4) ? 7 - 2 * i : 2 * i);
    return c;
  }
  // second quad of eight: accesses in reverse order
  __device__ static __forceinline__ void turn(int c, u32x4 (&s)[kPieces<BF16>]) {
    if constexpr (kEight) {
      const bool q = c & 4;
#pragma unroll
      for (int w = 0; w < 2; ++w) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t a = s[w][j], b = s[3 - w][j];
          s[w][j] = q ? b : a;
          s[3 - w][j] = q ? a : b;
        }
      }
    }
  }
  // the loaded pieces -> the lane's chunk, and (BACK) the reverse
  template <bool BACK>
  __device__ static __forceinline__ void swap(int c, u32x4 (&s)[kPieces<BF16>]) {
    if constexpr (kSwap && BF16) {
      swap_pieces<kDppQuadXor1>(s[0], s[1], c & 1);
    } else if constexpr (kSwap) {
      if constexpr (!BACK) turn(c, s);
      swap_pieces<kDppQuadXor1>(s[0], s[1], c & 1);
      swap_pieces<kDppQuadXor1>(s[2], s[3], c & 1);
      swap_pieces<kDppQuadXor2>(s[0], s[2], c & 2);
      swap_pieces<kDppQuadXor2>(s[1], s[3], c & 2);
      if constexpr (BACK) turn(c, s);
    }
  }
  __device__ static __forceinline__ float sum(float x) {
    if constexpr (!kSwap) {
      return group_sum<LPR>(x);
    } else {
      if constexpr (kEight) x = x + dpp_f<kDppRowHalfMirror>(x);
      if constexpr (BF16) x = x + dpp_f<kDppQuadXor2>(x);
      x = x + dpp_f<kDppQuadXor1>(x);
      if constexpr (!BF16) x = x + dpp_f<kDppQuadXor2>(x);
      if constexpr (BF16 && LPR >= 8) x = x + dpp_f<kDppRowHalfMirror>(x);
      if constexpr (LPR >= 16) x = x + dpp_f<kDppRowMirror>(x);
      return x;
    }
  }
};

template <int K, int RPL, int WAVES>
using FLayout = pd::Layout<K, RPL, WAVES, pd::kResidInt8, false>;

// All loads of one item; a dead item's collapse onto the first bytes of slot 0
// (see pd::load_item); rows past V re-read row V-1, where SHORT leaves
// out an instruction (rows from wave_row on) that has no other.
template <int K, int RPL, int WAVES, bool BF16, int ACT, bool SHORT>
__device__ __forceinline__ void load_fitem(const PackedParams& p, const ItemCoord& ic, int wave_row, int row0, int c,
                                           FloatItemRegs<RPL, FLayout<K, RPL, WAVES>::QKT, BF16>& R) {
  using L = FLayout<K, RPL, WAVES>;
  using M = ChunkMap<L::LPR, BF16>;
  constexpr uint32_t SB = BF16 ? 2u : 4u;  // state bytes per element
  constexpr int ESZ = act_bytes<ACT>;
  const uint32_t keep = ic.live ? 0xffffffffu : 0u;
  const int64_t slot = ic.live ? ic.slot : 0;
  const int hv = ic.live ? ic.hv : 0;
  const int8_t* sbase = p.state + (slot * p.stride_state + (int64_t)hv * p.V * K) * SB;
  const char* mrow = static_cast<const char*>(p.mixed) + (int64_t)ic.n * p.stride_mixed * ESZ;
  const char* vbase = mrow + (2 * (int64_t)p.H * K + (int64_t)hv * p.V) * ESZ;
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    if (SHORT && wave_row + i * L::RPI >= p.V) break;
    const uint32_t r = (uint32_t)min(row0 + i * L::RPI, p.V - 1) & keep;
#pragma unroll
    for (int w = 0; w < kPieces<BF16>; ++w)
      R.sw[i][w] = ld_state<M::kCached>(sbase + ((r * (K * SB) + M::piece_off(c, w)) & keep));
    R.vv[i] = load_act_raw<ESZ>(vbase, r * ESZ);
  }
  const char* qbase = mrow + (int64_t)pd::fdiv((uint32_t)hv, p.div_grp) * K * ESZ;
  const uint32_t koff = (uint32_t)((p.H - 1) * K);
#pragma unroll
  for (int j = 0; j < L::QKT; ++j) {
    const uint32_t e = min((uint32_t)threadIdx.x + j * L::NT, (uint32_t)(2 * K - 1));
    R.qk[j] = load_act_raw<ESZ>(qbase, ((e < K ? e : e + koff) * ESZ) & keep);
  }
}

template <int K, int RPL, int WAVES, bool BF16, int ACT, bool SHORT>
__device__ __forceinline__ void process_fitem(const PackedParams& p, const ItemCoord& ic, int wave_row, int row0,
                                              int c, float alpha, float beta, FloatItemRegs<RPL, FLayout<K, RPL, WAVES>::QKT, BF16>& R,
                                              float (*s_qk)[2 * K]) {
  using L = FLayout<K, RPL, WAVES>;
  using M = ChunkMap<L::LPR, BF16>;
  constexpr uint32_t SB = BF16 ? 2u : 4u;
  const int odt = p.out_dtype();
  char* obase = static_cast<char*>(p.out) + ((int64_t)ic.n * p.HV + ic.hv) * p.V * (odt == kF32 ? 4 : 2);
  if (!ic.live) {
    // NULL block (slot <= 0): zeros, no state access; out-of-range ids: NaN
    const float fill = (ic.slot <= 0) ? 0.0f : __uint_as_float(0x7fc00000u);
    if (c == 0) {
#pragma unroll
      for (int i = 0; i < RPL; ++i) {
        const int r = row0 + i * L::RPI;
        if (r < p.V) store_act_at(obase, (uint32_t)r, odt, fill);
      }
    }
    return;
  }
  pd::stage_qk<K, L::QKT, L::NT, ACT>(p, R.qk, c, 0, s_qk);
  const int ch = M::chunk(c);
  const float4* q4 = reinterpret_cast<const float4*>(s_qk[0] + ch * 16);
  const float4* k4 = reinterpret_cast<const float4*>(s_qk[0] + K + ch * 16);
  int8_t* sbase = p.state + (ic.slot * p.stride_state + (int64_t)ic.hv * p.V * K) * SB;
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    if (SHORT && wave_row + i * L::RPI >= p.V) break;
    const int r = row0 + i * L::RPI;
    asm volatile("" ::: "memory");  // re-read k, q from LDS for this row
    float kk[16], qq[16], h[16];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 b4 = k4[j];
      kk[4 * j] = b4.x, kk[4 * j + 1] = b4.y, kk[4 * j + 2] = b4.z, kk[4 * j + 3] = b4.w;
    }
    M::template swap<false>(c, R.sw[i]);
#pragma unroll
    for (int w = 0; w < kPieces<BF16>; ++w) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t x = R.sw[i][w][j];
        if constexpr (BF16) {
          h[8 * w + 2 * j] = __uint_as_float(x << 16) * alpha;
          h[8 * w + 2 * j + 1] = __uint_as_float(x & 0xffff0000u) * alpha;
        } else {
          h[4 * w + j] = __uint_as_float(x) * alpha;
        }
      }
    }
    float rd = h[0] * kk[0];
#pragma unroll
    for (int j = 1; j < 16; ++j) rd = fmaf(h[j], kk[j], rd);
    rd = M::sum(rd);
    const float dv = beta * (act_decode<ACT>(R.vv[i]) - rd);
#pragma unroll
    for (int j = 0; j < 16; ++j) h[j] = fmaf(kk[j], dv, h[j]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 a4 = q4[j];
      qq[4 * j] = a4.x, qq[4 * j + 1] = a4.y, qq[4 * j + 2] = a4.z, qq[4 * j + 3] = a4.w;
    }
    float o = h[0] * qq[0];
#pragma unroll
    for (int j = 1; j < 16; ++j) o = fmaf(h[j], qq[j], o);
    o = M::sum(o);
    asm volatile("" : "+v"(o));  // finish the sum here, where its DPP steps fuse into adds
    u32x4 out[kPieces<BF16>];
#pragma unroll
    for (int w = 0; w < kPieces<BF16>; ++w) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (BF16) {
          typedef float f2 __attribute__((ext_vector_type(2)));
          typedef __bf16 b2 __attribute__((ext_vector_type(2)));
          const b2 bb = __builtin_convertvector((f2){h[8 * w + 2 * j], h[8 * w + 2 * j + 1]}, b2);  // to nearest even
          uint32_t x;
          __builtin_memcpy(&x, &bb, 4);
          out[w][j] = x;
        } else {
          out[w][j] = __float_as_uint(h[4 * w + j]);
        }
      }
    }
    M::template swap<true>(c, out);
    if (r < p.V) {
      if (c == 0) store_act_at(obase, (uint32_t)r, odt, o);
#pragma unroll
      for (int w = 0; w < kPieces<BF16>; ++w) st_state<M::kCached>(sbase + ((uint32_t)r * (K * SB) + M::piece_off(c, w)), out[w]);
    }
  }
}

// One item per workgroup; the launch geometry in preloaded arguments (see
// pd::packed_decode_single_kernel). SHORT: waves without a row do no row work, for
// heads that leave a wave of their one tile empty: its re-reads of row V-1 cost
// (HV=32, B=200, us, without / with: fp32 K=128 V=1 26.1 / 13.3, V=16 30.9 / 20.9,
// bf16 K=128 V=16 20.2 / 14.7); with no such wave the branches do (+0-4 % at V=128).
template <int K, int RPL, int WAVES, bool BF16, int ACT, bool SHORT>
__global__ __launch_bounds__(WAVES * 64)
void float_decode_kernel(const int32_t* __restrict__ idx, int items, int stride_idx, uint32_t nvt_d, uint32_t nvt_m,
                         uint32_t nvt_sh, uint32_t hv_d, uint32_t hv_m, uint32_t hv_sh, int xcd_base, uint32_t grp_m,
                         uint32_t grp_w, const PackedParams p_arg) {
  using L = FLayout<K, RPL, WAVES>;
  const pd::Geom gm{items, stride_idx, 0, 0u, pd::FastDiv{nvt_d, nvt_m, nvt_sh}, pd::FastDiv{hv_d, hv_m, hv_sh}, items};
  PackedParams p = p_arg;
  p.div_grp = pd::quotient_fastdiv(grp_m, grp_w);
  __shared__ __attribute__((aligned(16))) float s_qk[4][2 * K];  // [0] staged, [2] raw
  __shared__ float2 s_gate[1];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int c = lane % L::LPR;
  const int g = lane / L::LPR;
  const ItemCoord ic = pd::xcd_item_coord<false>(p, gm, idx, nullptr, (int)blockIdx.x, xcd_base);
  const int wave_row = ic.vt * L::ROWS_WG + __builtin_amdgcn_readfirstlane(wave) * L::ROWS_WAVE;
  const int row0 = wave_row + g;
  FloatItemRegs<RPL, L::QKT, BF16> R;
  if constexpr (SHORT) R = {};
  load_fitem<K, RPL, WAVES, BF16, ACT, SHORT>(p, ic, wave_row, row0, c, R);
  __builtin_amdgcn_sched_barrier(0);  // the gate inputs' loads after the item's
  const pd::GateBits gbits = pd::load_item_gate_bits(p, ic);
  pd::stage_item_gates(p, gbits, wave, lane, s_gate);
  __syncthreads();
  const float2 gab = s_gate[0];
  process_fitem<K, RPL, WAVES, BF16, ACT, SHORT>(p, ic, wave_row, row0, c, gab.x, gab.y, R, s_qk);
}

template <int K, int RPL, bool BF16, int ACT>
int launch_fs_cfg(PackedParams p, int B, hipStream_t stream) {
  constexpr int WAVES = 4;
  using L = FLayout<K, RPL, WAVES>;
  const int nvt = (p.V + L::ROWS_WG - 1) / L::ROWS_WG;
  const int64_t items = (int64_t)B * p.HV * nvt;
  if (items > 0x7fffffff) return fail(CK_EUNSUPPORTED, "%lld work items is too many", (long long)items);
  if (items == 0) return ok();
  const int64_t cap = pd::one_item_cap(WAVES * 64);
  if (items > cap) {  // consecutive launches over slices of the requests
    const int64_t per_request = (int64_t)p.HV * nvt;
    if (per_request > cap) return fail(CK_EUNSUPPORTED, "%lld work items per request is too many", (long long)per_request);
    const int chunk = (int)(cap / per_request);
    for (int64_t n0 = 0; n0 < B; n0 += chunk) {
      const int n = (int)min((int64_t)chunk, B - n0);
      const int rc = launch_fs_cfg<K, RPL, BF16, ACT>(pd::requests_from(p, (int)n0), n, stream);
      if (rc != CK_OK) return rc;
    }
    return ok();
  }
  p.items = (int)items;
  p.div_nvt = pd::make_fastdiv((uint32_t)nvt);
  p.div_hv = pd::make_fastdiv((uint32_t)p.HV);
  auto fn = float_decode_kernel<K, RPL, WAVES, BF16, ACT, false>;
  if (p.V <= L::ROWS_WG - L::ROWS_WAVE) fn = float_decode_kernel<K, RPL, WAVES, BF16, ACT, true>;
  hipLaunchKernelGGL(fn, dim3((unsigned)items), dim3(WAVES * 64), 0, stream, p.idx, p.items, p.stride_idx, p.div_nvt.d,
                     p.div_nvt.m, p.div_nvt.sh, p.div_hv.d, p.div_hv.m, p.div_hv.sh, pd::xcd_base(B, p.HV * nvt),
                     p.div_grp.m, pd::quotient_word(p.div_grp), p);
  return check_launch("ck_gdn_packed_decode_float_state");
}

// Two rows per lane from 512 such tiles on, below that one (a small batch over
// more SIMDs), as the quantized decode with per-row scales; also two where a
// request's smaller tiles would pass the limit of items per launch.
template <int K, bool BF16, int ACT>
int launch_fs(const PackedParams& p, int B, hipStream_t stream) {
  constexpr int TILE = FLayout<K, 2, 4>::ROWS_WG;
  const int64_t cap = pd::one_item_cap(4 * 64);
  const int64_t small = (int64_t)p.HV * ((2 * (int64_t)p.V + TILE - 1) / TILE);
  if ((int64_t)B * p.HV * ((p.V + TILE - 1) / TILE) >= 512 || small > cap)
    return launch_fs_cfg<K, 2, BF16, ACT>(p, B, stream);
  return launch_fs_cfg<K, 1, BF16, ACT>(p, B, stream);
}

template <bool BF16, int ACT>
int launch_fs_k(const PackedParams& p, int B, int K, hipStream_t s) {
  switch (K) {
    case 16: return launch_fs<16, BF16, ACT>(p, B, s);
    case 32: return launch_fs<32, BF16, ACT>(p, B, s);
    case 64: return launch_fs<64, BF16, ACT>(p, B, s);
    case 128: return launch_fs<128, BF16, ACT>(p, B, s);
    case 256: return launch_fs<256, BF16, ACT>(p, B, s);
    default: return fail(CK_EUNSUPPORTED, "K must be one of 16, 32, 64, 128, 256, got %d", K);
  }
}

}  // namespace fs
}  // namespace ck

extern "C" int ck_gdn_packed_decode_float_state(const void* mixed_qkv, int qkv_dtype, int64_t stride_qkv_tok,
                                                const void* a, int a_dtype, int64_t stride_a_tok,
                                                const void* b, int b_dtype, int64_t stride_b_tok,
                                                const void* A_log, int A_log_dtype,
                                                const void* dt_bias, int dt_bias_dtype,
                                                float scale,
                                                void* state, int state_dtype, int64_t stride_state_slot,
                                                void* out, int out_dtype,
                                                const int32_t* ssm_state_indices, int64_t stride_indices,
                                                int64_t num_slots,
                                                int B, int H, int HV, int K, int V,
                                                int use_qk_l2norm, void* stream) {
  using namespace ck;
  if (B < 0 || H <= 0 || HV <= 0 || K <= 0 || V <= 0)
    return fail(CK_EINVAL, "bad sizes B=%d H=%d HV=%d K=%d V=%d", B, H, HV, K, V);
  if (HV % H != 0) return fail(CK_EINVAL, "HV (%d) must be a multiple of H (%d)", HV, H);
  if (!valid_dtype(qkv_dtype) || !valid_dtype(a_dtype) || !valid_dtype(b_dtype) || !valid_dtype(A_log_dtype) ||
      !valid_dtype(dt_bias_dtype) || !valid_dtype(out_dtype))
    return fail(CK_EINVAL, "unsupported dtype code");
  if (state_dtype != CK_DTYPE_F32 && state_dtype != CK_DTYPE_BF16)
    return fail(CK_EINVAL, "state dtype must be float32 or bfloat16");
  if (num_slots <= 0) return fail(CK_EINVAL, "num_slots must be positive");
  if (K != 16 && K != 32 && K != 64 && K != 128 && K != 256)
    return fail(CK_EUNSUPPORTED, "K must be one of 16, 32, 64, 128, 256, got %d", K);
  if (B == 0) return ok();
  if (!mixed_qkv || !a || !b || !A_log || !dt_bias || !state || !out || !ssm_state_indices)
    return fail(CK_EINVAL, "null pointer argument");
  const int sesz = state_dtype == CK_DTYPE_F32 ? 4 : 2;
  if ((reinterpret_cast<uintptr_t>(state) & 15) || ((stride_state_slot * sesz) % 16))
    return fail(CK_EINVAL, "state rows must be 16-byte aligned");
  // per-lane byte offsets inside one (slot, head) and one row of mixed_qkv are 32-bit
  if ((int64_t)V * K * sesz >= ((int64_t)1 << 31) || (2 * (int64_t)H * K + (int64_t)HV * V) * 4 >= ((int64_t)1 << 31))
    return fail(CK_EUNSUPPORTED, "head or activation row too large");
  const int64_t strides[] = {stride_qkv_tok, stride_a_tok, stride_b_tok, stride_state_slot, stride_indices};
  for (int64_t st : strides)
    if (st < 0 || st > INT32_MAX) return fail(CK_EUNSUPPORTED, "strides must be in [0, 2^31) elements");
  if (num_slots > INT32_MAX) return fail(CK_EUNSUPPORTED, "num_slots must be < 2^31");

  pd::PackedParams p{};
  p.mixed = mixed_qkv;
  p.a = a;
  p.b = b;
  p.A_log = A_log;
  p.dt_bias = dt_bias;
  p.state = static_cast<int8_t*>(state);  // fp32 / bf16 elements, addressed in bytes
  p.out = out;
  p.idx = ssm_state_indices;
  p.stride_mixed = (int32_t)stride_qkv_tok;
  p.stride_a = (int32_t)stride_a_tok;
  p.stride_b = (int32_t)stride_b_tok;
  p.stride_state = (int32_t)stride_state_slot;
  p.stride_idx = (int32_t)stride_indices;
  p.num_slots = (int32_t)num_slots;
  p.scale = scale;
  p.dtypes = qkv_dtype | (a_dtype << 4) | (b_dtype << 8) | (A_log_dtype << 12) | (dt_bias_dtype << 16) |
             (out_dtype << 20);
  p.H = H;
  p.HV = HV;
  p.div_grp = pd::make_fastdiv((uint32_t)(HV / H));
  p.V = V;
  p.l2norm = use_qk_l2norm ? 1 : 0;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const bool bf16 = state_dtype == CK_DTYPE_BF16;
  if (qkv_dtype == CK_DTYPE_F32)
    return bf16 ? fs::launch_fs_k<true, kF32>(p, B, K, s) : fs::launch_fs_k<false, kF32>(p, B, K, s);
  if (qkv_dtype == CK_DTYPE_BF16)
    return bf16 ? fs::launch_fs_k<true, kBF16>(p, B, K, s) : fs::launch_fs_k<false, kBF16>(p, B, K, s);
  return bf16 ? fs::launch_fs_k<true, kF16>(p, B, K, s) : fs::launch_fs_k<false, kF16>(p, B, K, s);
}
