// T decode steps of the statequant layout in one launch: the step of
// quant_step.hip (same operations in the same order, so the same bits) with
// the state kept in registers from one token to the next. A column of the
// state depends on no other column, so a wave owns a few columns of one
// (request, head) for all T steps; only q, k, v, alpha, beta are read and only o
// is written per token. Counterpart of statequant/kernel.py:436-452
// (gdn_quant_decode_fused), whose loop launches one step per token.
//
// What bounds it: each step's chain of dependent operations while few waves run,
// the VALU once the chip is full. So the S slices of a column's rows lie in
// neighbouring lanes (64 / S columns a wave) and every sum and maximum over K is
// a DPP butterfly inside the wave, the same tree as the step kernel's, with no
// barrier; the state's own accesses are 32 bytes wide that way, but are made
// once per launch. One column per lane also gives a short batch many waves and
// takes any V and alignment. Inputs come in chunks of 8 (K = 256: 4) tokens
// through LDS, the next chunk's loads in flight while one is computed.
// Measured (B=4, HV=16, K=V=128, fp32 residual, 16 tokens, whole call): one
// launch per token 318-329 us (6.6 us of device time per step, the rest the
// host's); one launch 24.3 us with the slices in the waves of a workgroup and
// sums through LDS, the initial quantization a launch of its own and inputs
// prefetched one token ahead; 15.2 us now.
#include <hip/hip_runtime.h>

#include <utility>

#include "ck_capi_common.h"
#include "ck_device.h"
#include "ck_quant.h"
#include "ck_statequant.h"

namespace ck {
namespace qs {

constexpr int kDecodeWaves = 4;

// Tokens whose inputs are staged in LDS together.
template <int K>
constexpr int kChunkFor = K <= 128 ? 8 : 4;

struct DecodeParams {
  const float* h0;  // the state before the first step, quantized as ck_quantize_cols does
  int8_t* h;        // the last step's codes, scales, residual and its scales
  float* scale;
  void* e;
  float* e_scale;
  const float* q;
  const float* k;
  const float* v;
  const float* alpha;
  const float* beta;
  float* o;
  int T, V, nvt;
  int K;  // rows that exist (the kernel's K template argument is the padded count)
  int heads;  // B * HV: stride of a token in (request, head) units
  bool ieee;  // the form of ck_quantize_cols that h0's shape takes (ck_statequant.h)
  float qmax, rqmax;
};

// The residual of one value as the next step reads it, and its stored bits.
template <int RES>
__device__ __forceinline__ uint32_t encode_resid(float r) {
  if constexpr (RES == kResFp32) {
    return __float_as_uint(r);
  } else if constexpr (RES == kResFp16) {
    return f32_to_half_bits(r);
  } else {
    const float x[1] = {r};
    return f32_to_e5m2<1>(x);
  }
}

template <int RES>
__device__ __forceinline__ float decode_resid(uint32_t bits) {
  if constexpr (RES == kResFp32) return __uint_as_float(bits);
  else if constexpr (RES == kResFp16) return half_bits_to_f32(bits & 0xffffu);
  else if constexpr (RES == kResFp8) return e5m2_byte(bits, 0);
  else return code_i8(bits, 0);
}

// f(0), f(1), ..., f(N - 1) with the index as a compile-time constant. Written
// out before the optimizer runs, so the per-row arrays below become scalars; an
// inner loop of the token loop is unrolled too late for that (the arrays turned
// into 16-dword vectors, copied whole: 226 VGPRs).
template <class F, int... I>
__device__ __forceinline__ void for_each_index(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
#define CK_ROWS(r) for_each_index(std::make_integer_sequence<int, RPS>{}, [&](auto r) __attribute__((always_inline))

template <int K, int RES, int MODE, bool MK>
__global__ __launch_bounds__(kDecodeWaves * 64) void quant_decode_kernel(const DecodeParams p) {
  constexpr int S = kSlicesFor<K>;
  constexpr int RPS = K / S;                // rows per slice
  constexpr int CW = 64 / S;                // columns per wave
  constexpr int NC = kDecodeWaves * CW;     // columns per workgroup
  constexpr int NT = kDecodeWaves * 64;
  constexpr int kChunk = kChunkFor<K>;
  constexpr int QKT = kChunk * 2 * K / NT;  // staged q/k values per thread and chunk
  static_assert(kChunk * 2 * K % NT == 0 && (NT % (2 * K) == 0 || 2 * K % NT == 0), "chunk shape");
  // a slice's q or k values, 16 of them 20 words apart: the slices' 16-byte
  // reads then fall in different banks
  constexpr int SLICE = RPS == 16 ? 20 : RPS;
  // per chunk parity: [token][q, k][slice], v, alpha and beta
  __shared__ __attribute__((aligned(16))) float s_qk[2][kChunk][2][S * SLICE];
  __shared__ float s_v[2][kChunk][NC];
  __shared__ float s_ab[2][2][kChunk];

  const int t = threadIdx.x;
  const int ks = t % S;
  const int cg = t / S;                     // column of the workgroup's
  const int vt = blockIdx.x % p.nvt;
  const int w = blockIdx.x / p.nvt;         // (request, head)
  const int col = vt * NC + cg;
  const bool colok = col < p.V;
  const int r0 = ks * RPS;
  const int KA = MK ? p.K : K;
  const int64_t mb = (int64_t)w * KA * p.V + col;
  const int64_t vb = (int64_t)w * p.V + col;
  const int64_t token_k = (int64_t)p.heads * KA;  // elements of q and k per token
  const int64_t token_v = (int64_t)p.heads * p.V;

  // this thread's share of a chunk's inputs: elements t, t + NT, ... of
  // [token][q | k], v of one token, alpha or beta of one; tokens past the last
  // re-read it
  float qk_r[QKT], v_r = 0.f, ab_r = 0.f;
  const int v_tok = t / NC, v_col = vt * NC + t % NC;
  const auto load_chunk = [&](int n0) __attribute__((always_inline)) {
    for_each_index(std::make_integer_sequence<int, QKT>{}, [&](auto j) __attribute__((always_inline)) {
      const int i = t + j * NT;
      const int kr = i % K;
      const float* src = i % (2 * K) < K ? p.q : p.k;
      qk_r[j] = !MK || kr < KA ? src[min(n0 + i / (2 * K), p.T - 1) * token_k + (int64_t)w * KA + kr] : 0.f;
    });
    if (v_tok < kChunk && v_col < p.V) v_r = p.v[min(n0 + v_tok, p.T - 1) * token_v + (int64_t)w * p.V + v_col];
    if (t < 2 * kChunk) ab_r = (t < kChunk ? p.alpha : p.beta)[(int64_t)min(n0 + t % kChunk, p.T - 1) * p.heads + w];
  };
  const auto stage_chunk = [&](int b) __attribute__((always_inline)) {
    for_each_index(std::make_integer_sequence<int, QKT>{}, [&](auto j) __attribute__((always_inline)) {
      const int i = t + j * NT;
      const int kr = i % K;
      s_qk[b][i / (2 * K)][i / K % 2][kr / RPS * SLICE + kr % RPS] = qk_r[j];
    });
    if (v_tok < kChunk) s_v[b][v_tok][t % NC] = v_r;
    if (t < 2 * kChunk) (&s_ab[b][0][0])[t] = ab_r;
  };

  uint32_t cb[RPS];  // state codes, low byte
  uint32_t eb[RPS];  // residual, stored form: zero at first, which decodes to +0 in every format
  float sc, es = 0.f;
  {
    float h0[RPS], m;
    CK_ROWS(r) {
      eb[r] = 0u;
      h0[r] = 0.f;
      if (colok && (!MK || r0 + r < KA)) h0[r] = p.h0[mb + (int64_t)(r0 + r) * p.V];
    });
    load_chunk(0);
    CK_ROWS(r) { m = r == 0 ? fabsf(h0[0]) : fmaxf(m, fabsf(h0[r])); });
    stage_chunk(0);
    // as ingest_amax: eighths of the rows in IEEE order, then unsigned unless ieee
    const float m8 = group_fmax<S / 8>(m);
    const float am = p.ieee ? fmaxf(group_fmax<S>(m), 0.f) : group_max<S>(m8);
    sc = fmaxf(am, kEps) / p.qmax;
    const float inv = recip_rn(sc);
    CK_ROWS(r) {
      cb[r] = p.ieee ? ingest_code<true>(h0[r], sc, inv, p.qmax) : ingest_code<false>(h0[r], sc, inv, p.qmax);
    });
    __syncthreads();
  }

  int n = 0, c = 0, b = 0;  // token, its place in its chunk, the chunk's buffer
  do {
    if (c == 0) load_chunk(n + kChunk);  // in flight while this chunk is computed
    const float alpha = s_ab[b][0][c], beta = s_ab[b][1][c], vv = s_v[b][c][cg];
    float qq[RPS], kk[RPS], h[RPS];
    constexpr int W = RPS >= 4 ? 4 : 2;  // values per LDS read
    typedef float vec __attribute__((ext_vector_type(W)));
    const vec* qv = reinterpret_cast<const vec*>(&s_qk[b][c][0][ks * SLICE]);
    const vec* kv = reinterpret_cast<const vec*>(&s_qk[b][c][1][ks * SLICE]);
    for_each_index(std::make_integer_sequence<int, RPS / W>{}, [&](auto j) __attribute__((always_inline)) {
      const vec x = kv[j], y = qv[j];
      for_each_index(std::make_integer_sequence<int, W>{}, [&](auto i) __attribute__((always_inline)) {
        kk[j * W + i] = x[int(i)];
        qq[j * W + i] = y[int(i)];
      });
    });

    // dequantize + decay; rd = h^T k
    const float sa = sc * alpha;
    float acc;
    CK_ROWS(r) {
      const float code = code_i8(cb[r], 0);
      h[r] = (MODE == kFast) ? code * sa : (code * sc) * alpha;
      acc = r == 0 ? h[0] * kk[0] : fmaf(h[r], kk[r], acc);
    });
    const float dv = beta * (vv - group_sum<S>(acc));
    // h += k dv; o = h^T q; t = h + e; amax over K
    float m;
    CK_ROWS(r) {
      h[r] = madd<MODE>(kk[r], dv, h[r]);
      acc = r == 0 ? h[0] * qq[0] : fmaf(h[r], qq[r], acc);
      const float ev = decode_resid<RES>(eb[r]);
      if constexpr (RES == kResInt8) h[r] = madd<MODE>(ev, es, h[r]);
      else h[r] = h[r] + ev;
      m = r == 0 ? fabsf(h[0]) : fmaxf(m, fabsf(h[r]));
    });
    acc = group_sum<S>(acc);
    if (ks == 0 && colok) p.o[n * token_v + vb] = acc;
    sc = fmaxf(div_small_int(group_fmax<S>(m), p.qmax, p.rqmax), kEps);
    const float inv = recip_rn(sc);
    // requantize, form the residual
    float ea = 0.f;
    CK_ROWS(r) {
      const float code = quantize<MODE>(h[r], sc, inv, cb[r]);
      h[r] = residual<MODE>(h[r], code, sc);
      if constexpr (RES == kResInt8) ea = fmaxf(ea, fabsf(h[r]));
      else eb[r] = encode_resid<RES>(h[r]);
    });
    if constexpr (RES == kResInt8) {
      es = fmaxf(div_small_int(group_fmax<S>(ea), p.qmax, p.rqmax), kEps);
      const float inv_e = recip_rn(es);
      CK_ROWS(r) { (void)quantize<MODE>(h[r], es, inv_e, eb[r]); });
    }
    if constexpr (MK) {  // rows past K hold zeros whatever the column's scale is
      CK_ROWS(r) {
        if (r0 + r >= KA) cb[r] = eb[r] = 0u;
      });
    }
    if (++c == kChunk) {
      // the other buffer's chunk was read before the last barrier
      c = 0, b ^= 1;
      stage_chunk(b);
      __syncthreads();
    }
  } while (++n < p.T);

  if (!colok) return;
  int64_t tail = mb + (int64_t)r0 * p.V;
  asm volatile("" : "+v"(tail));  // not the first loads' row addresses, kept over the token loop
  CK_ROWS(r) {
    if (MK && r0 + r >= KA) return;
    const int64_t i = tail + (int64_t)r * p.V;
    p.h[i] = (int8_t)cb[r];
    if constexpr (RES == kResFp32) static_cast<float*>(p.e)[i] = __uint_as_float(eb[r]);
    else if constexpr (RES == kResFp16) static_cast<uint16_t*>(p.e)[i] = (uint16_t)eb[r];
    else static_cast<uint8_t*>(p.e)[i] = (uint8_t)eb[r];
  });
  if (ks == 0) {
    p.scale[vb] = sc;
    if constexpr (RES == kResInt8) p.e_scale[vb] = es;
  }
}
#undef CK_ROWS

template <int K, int MODE, bool MK>
int launch_decode(const DecodeParams& p, int64_t grid, int res_fmt, hipStream_t s) {
  const dim3 g((unsigned)grid), b(kDecodeWaves * 64);
  switch (res_fmt) {
    case kResFp32: hipLaunchKernelGGL((quant_decode_kernel<K, kResFp32, MODE, MK>), g, b, 0, s, p); break;
    case kResFp16: hipLaunchKernelGGL((quant_decode_kernel<K, kResFp16, MODE, MK>), g, b, 0, s, p); break;
    case kResFp8: hipLaunchKernelGGL((quant_decode_kernel<K, kResFp8, MODE, MK>), g, b, 0, s, p); break;
    default: hipLaunchKernelGGL((quant_decode_kernel<K, kResInt8, MODE, MK>), g, b, 0, s, p); break;
  }
  return check_launch("ck_gdn_quant_decode");
}

template <int MODE, bool MK>
int launch_decode_kp(const DecodeParams& p, int64_t grid, int KP, int res_fmt, hipStream_t s) {
  switch (KP) {
    case 16: return launch_decode<16, MODE, MK>(p, grid, res_fmt, s);
    case 32: return launch_decode<32, MODE, MK>(p, grid, res_fmt, s);
    case 64: return launch_decode<64, MODE, MK>(p, grid, res_fmt, s);
    case 128: return launch_decode<128, MODE, MK>(p, grid, res_fmt, s);
    default: return launch_decode<256, MODE, MK>(p, grid, res_fmt, s);
  }
}

template <int MODE>
int launch_decode_k(const DecodeParams& p, int64_t grid, int res_fmt, hipStream_t s) {
  const int KP = padded_k(p.K);
  return KP == p.K ? launch_decode_kp<MODE, false>(p, grid, KP, res_fmt, s)
                   : launch_decode_kp<MODE, true>(p, grid, KP, res_fmt, s);
}

}  // namespace qs
}  // namespace ck

extern "C" int ck_gdn_quant_decode(const float* h0, int8_t* h, float* scale, void* e, float* e_scale,
                                   const float* q, const float* k, const float* v,
                                   const float* alpha, const float* beta, float* o,
                                   int T, int B, int HV, int K, int V, float qmax, int res_fmt, int quant_mode,
                                   void* stream) {
  using namespace ck;
  using namespace ck::qs;
  if (T < 0 || B < 0 || HV <= 0 || K <= 0 || V <= 0)
    return fail(CK_EINVAL, "bad sizes T=%d B=%d HV=%d K=%d V=%d", T, B, HV, K, V);
  if (!valid_k(K)) return fail(CK_EUNSUPPORTED, "K must be in 1..256, got %d", K);
  if (res_fmt < CK_RES_FP32 || res_fmt > CK_RES_INT8) return fail(CK_EINVAL, "unknown residual format %d", res_fmt);
  if (quant_mode != CK_QUANT_FAST && quant_mode != CK_QUANT_EXACT)
    return fail(CK_EINVAL, "quant_mode must be CK_QUANT_FAST or CK_QUANT_EXACT, got %d", quant_mode);
  const int iq = (int)qmax;
  if ((float)iq != qmax || iq < 1 || iq > 127) return fail(CK_EINVAL, "qmax must be an integer in 1..127");
  if (T == 0 || B == 0) return ok();
  if (!h0 || !h || !scale || !e || !q || !k || !v || !alpha || !beta || !o) return fail(CK_EINVAL, "null pointer argument");
  const bool int8_res = res_fmt == CK_RES_INT8;
  if (int8_res && !e_scale) return fail(CK_EINVAL, "int8 residual needs e_scale");
  const uintptr_t fbits = addr_bits(h0, scale, q, k, v, alpha, beta, o) | (int8_res ? addr_bits(e_scale) : 0);
  const int esz = res_fmt == CK_RES_FP32 ? 4 : res_fmt == CK_RES_FP16 ? 2 : 1;
  if ((fbits & 3) || (addr_bits(e) & (esz - 1)))
    return fail(CK_EINVAL, "fp32 tensors must be 4-byte aligned and the residual %d-byte aligned", esz);
  const int64_t heads = (int64_t)B * HV;
  const int cols = kDecodeWaves * (K <= 128 ? 8 : 4);  // columns per workgroup
  const int nvt = (V + cols - 1) / cols;
  if (heads > 0x7fffffff) return fail(CK_EUNSUPPORTED, "too many heads");
  volatile float one = 1.0f;
  const bool ieee = ingest_ieee(addr_bits(h0, h, scale), heads, K, V);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  return launch_slices(heads, nvt, kDecodeWaves * 64, [&](int64_t w0, int64_t n) {
    const int64_t m = w0 * K * V, c = w0 * V, r = w0 * K;  // the slice's first matrix, column and row
    const DecodeParams p{h0 + m, h + m, scale + c, static_cast<char*>(e) + m * esz, int8_res ? e_scale + c : nullptr,
                         q + r, k + r, v + c, alpha + w0, beta + w0, o + c, T, V, nvt, K, (int)heads, ieee, qmax,
                         one / qmax};
    return quant_mode == CK_QUANT_EXACT ? launch_decode_k<kExact>(p, n * nvt, res_fmt, s)
                                        : launch_decode_k<kFast>(p, n * nvt, res_fmt, s);
  });
}
