// State ingest: quantize a float state into the int8 pool.
//   ck_quantize_rows: rows of K (vLLM [.., V, K] layout), one scale per row,
//     init_quantized_state semantics (vllm_integration/quantized_packed_decode.py:347-351):
//     scale = max(amax, 1e-12) / qmax, code = clamp(rne(x / scale), +-qmax),
//     evaluated in the precision of x as torch evaluates that expression on a
//     tensor of x's dtype: fp32 and float64 arithmetic as such; for bf16 and
//     fp16 every operation is computed in fp32 and rounded (to nearest even)
//     to x's dtype, so the scale is the 16-bit value RN16(RN(max(amax, RN16(
//     1e-12)) / qmax)) and the quotient RN16(RN(x / scale)) is rounded to an
//     integer from there (it can reach qmax + 1 in bf16, where the clamp then
//     binds). A float64 scale is stored rounded to fp32.
//   ck_quantize_cols: [K, V] matrices, one scale per V-column (amax over K),
//     per_v_channel_quantize semantics (statequant/kernel.py:99-113).
// Both divide correctly rounded (IEEE division, or the reciprocal with
// Markstein's correction), so the codes equal torch.round(x / scale).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ck_capi_common.h"
#include "ck_device.h"
#include "ck_quant.h"
#include "ck_statequant.h"

namespace ck {
namespace {

// x rounded to nearest even to the 16-bit dtype DT and back to fp32 (fp32:
// unchanged); subnormal fp16 results are kept (the conversion honours fp16
// denormals), values past the largest finite fp16 become inf.
template <int DT>
__device__ __forceinline__ float round16(float x) {
  if constexpr (DT == kBF16) {
    return (float)(__bf16)x;  // v_cvt_pk_bf16_f32
  } else if constexpr (DT == kF16) {
    return (float)(_Float16)x;
  } else {
    return x;
  }
}

__device__ __forceinline__ float round16_rt(int dt, float x) {
  return dt == kBF16 ? round16<kBF16>(x) : dt == kF16 ? round16<kF16>(x) : x;
}

// Rows of K elements, a wave several rows at a time, in one pass: codes, scales
// and, where asked for, a zero residual of rk bytes per row and zero scales, which
// took the caller two launches and, with those that cleared the codes and scales
// before they were written, a pass over the pool. Two kernels, equal on finite
// values:
//  * K a power of two from 16 to 256, 16-byte aligned (quantize_rows16_kernel): 16
//    elements per lane, each through RN(1/s) with Markstein's correction (ck_quant.h,
//    EXACT mode), the correctly rounded quotient. |x / s| <= qmax (1 + 2^-23) < qmax +
//    1/2 since s >= RN(amax / qmax), so no code exceeds qmax and the clamp of the
//    reference never binds. The amax keeps a 16-element chunk of NaNs as NaN.
//  * any other (quantize_rows_tile_kernel), 16 bytes of a row per lane in one access
//    of any alignment, four rows in flight: IEEE quotients and the clamp (infinities,
//    scales that are no normal number), NaN codes 0 and NaNs no part of the amax.
// 16-bit dtypes in their own precision: RN16 after every fp32 operation.
// HBM bounds large fp32 states (5.6 TB/s at 257 slots of [32, 128, 128]); the VALU,
// with 16 operations an element (0.25 instructions per SIMD and cycle, fp32 0.06),
// 16-bit ones (6.7 TB/s). Row-level work is done
// once per 16 elements: 4 or 8 elements per lane in one access each, with the codes
// exchanged into 16-byte stores, were slower (us, so / now: 257 slots bf16 70.2 /
// 60.6, fp16 67.4 / 60.3, fp32 123.0 / 121.0; 8 slots bf16 6.0 / 4.2), and so were
// whole lines per access with the pieces swapped between lanes (257 slots bf16 64.7,
// fp32 124.0): the loads are cached, the next instruction's bytes L2 hits.
// init_quantized_state of a bf16 [64, 32, 128, 128] with an int4 residual (118 MB),
// four fills and a kernel / one pass: 35.1 / 22.0 us a call. [32, 32, 100, 100] int8:
// fp32 40.8 -> 14.7, bf16 42.1 -> 15.6 (two passes of one wave per row before).
struct RowsInit {
  int8_t* resid;    // or null
  int rk;           // residual bytes per row
  float* rscale;    // or null
  int64_t n_rscale;
};

struct RowsParams {
  const char* x;
  int64_t stride_row_bytes, rows;
  int K;
  float qmax;
  int8_t* codes;
  float* scale;
  RowsInit init;
};

// Unsigned maximum over groups of N lanes, up to a whole wave.
template <int N>
__device__ __forceinline__ float group_max_lanes(float x) {
  uint32_t u = __float_as_uint(group_max<(N < 16 ? N : 16)>(x));
  if constexpr (N >= 32) u = max(u, (uint32_t)__shfl_xor((int)u, 16));
  if constexpr (N >= 64) u = max(u, (uint32_t)__shfl_xor((int)u, 32));
  return __uint_as_float(u);
}

// The zero residual of rows r0 .. r0 + n - 1, by the lanes of a wave.
__device__ __forceinline__ void zero_residual_rows(const RowsInit& p, int64_t r0, int64_t n, int lane) {
  if (!p.resid) return;
  const int64_t total = n * p.rk;
  int8_t* z = p.resid + r0 * p.rk;
  for (int64_t i = lane * 16; i < total; i += 1024) {
    if (i + 16 <= total) {
      st_stream16_u(z + i, u32x4{0u, 0u, 0u, 0u});
    } else {
      for (int64_t b = i; b < total; ++b) z[b] = 0;
    }
  }
}

// The zero residual scales, by `threads` threads of which this is number t.
__device__ __forceinline__ void zero_scales(const RowsInit& p, int64_t t, int64_t threads) {
  for (int64_t i = t; i < p.n_rscale; i += threads) p.rscale[i] = 0.0f;
}

// The EPL elements of type DT in N dwords, as fp32.
template <int DT, int N, int EPL>
__device__ __forceinline__ void decode_elements(const uint32_t (&w)[N], float (&v)[EPL]) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if constexpr (DT == kF32) {
      v[j] = __uint_as_float(w[j]);
    } else {
      v[2 * j] = act_decode<DT>(w[j] & 0xffffu);
      v[2 * j + 1] = act_decode<DT>(w[j] >> 16);
    }
  }
}

// K = 16 * LPR, 16-byte aligned: 16 elements of a row per lane, its own bytes.
// The arguments that every wave needs before its first load are the first twelve
// dwords, which the dispatch preloads (with the number of waves read from the
// implicit arguments instead, fp32 8 slots 5.06 against 4.72 us).
template <int LPR, int DT, bool INIT>
__global__ __launch_bounds__(256) void quantize_rows16_kernel(const char* __restrict__ x, int64_t stride_row_bytes,
                                                              int64_t rows, int8_t* __restrict__ codes,
                                                              float* __restrict__ scale, float qmax, uint32_t nwaves,
                                                              const RowsInit init) {
  constexpr int NP = DT == kF32 ? 4 : 2;  // 16-byte pieces of a lane's elements
  constexpr int RPW = 64 / LPR;           // rows per wave
  constexpr int K = 16 * LPR;
  const int lane = threadIdx.x & 63;
  const int c = lane % LPR;
  const int g = lane / LPR;
  const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  for (int64_t r0 = wave * RPW; r0 < rows; r0 += (int64_t)nwaves * RPW) {
    const int64_t row = r0 + g;
    const bool valid = row < rows;
    const u32x4* xr = reinterpret_cast<const u32x4*>(x + (valid ? row : rows - 1) * stride_row_bytes) + c * NP;
    uint32_t bits[4 * NP];
#pragma unroll
    for (int w = 0; w < NP; ++w) {
      const u32x4 a = xr[w];
      bits[4 * w] = a.x, bits[4 * w + 1] = a.y, bits[4 * w + 2] = a.z, bits[4 * w + 3] = a.w;
    }
    if constexpr (INIT) zero_residual_rows(init, r0, min((int64_t)RPW, rows - r0), lane);
    float v[16];
    decode_elements<DT>(bits, v);
    float am = fabsf(v[0]);
#pragma unroll
    for (int j = 1; j < 16; ++j) am = fmaxf(am, fabsf(v[j]));
    am = group_max<LPR>(am);
    const float s = round16<DT>(fmaxf(am, round16<DT>(kEps)) / qmax);
    uint32_t yb[16];
    if (DT != kF16 || s > 0.0f) {
      const float inv = recip_rn(s);
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        if constexpr (DT == kF32) {
          (void)quantize<kExact>(v[j], s, inv, yb[j]);
        } else {
          const float q = round16<DT>(exact_quotient(v[j], s, inv));
          yb[j] = __float_as_uint(fminf(fmaxf(rintf(q), -qmax), qmax) + kMagic);
        }
      }
    } else {
      // RN16(1e-12) = 0 in fp16: the row's scale rounded to 0, so x / 0 is +-inf
      // (clamped to +-qmax) for x != 0 and NaN for x = 0, which the reference's
      // int8 conversion turns into 0
#pragma unroll
      for (int j = 0; j < 16; ++j)
        yb[j] = __float_as_uint((v[j] > 0.0f ? qmax : v[j] < 0.0f ? -qmax : 0.0f) + kMagic);
    }
    if (valid) {
      st_stream16(codes + row * K + c * 16,
                  u32x4{pack_low_bytes(yb[0], yb[1], yb[2], yb[3]), pack_low_bytes(yb[4], yb[5], yb[6], yb[7]),
                        pack_low_bytes(yb[8], yb[9], yb[10], yb[11]), pack_low_bytes(yb[12], yb[13], yb[14], yb[15])});
      if (c == 0) scale[row] = s;
    }
  }
  if constexpr (INIT) zero_scales(init, wave * 64 + lane, (int64_t)nwaves * 64);
}

// Any K from one lane's elements to 64 lanes': EPL elements per lane, the last
// lane taking the row's last EPL, some of them its neighbour's too (the same codes).
template <int W, int DT>
__global__ __launch_bounds__(256) void quantize_rows_tile_kernel(const RowsParams p) {
  constexpr int EPL = DT == kF32 ? 4 : 8;
  constexpr int ESZ = DT == kF32 ? 4 : 2;
  constexpr int RPI = 64 / W;           // rows per wave instruction
  constexpr int U = 4;
  constexpr int ROWS = RPI * U;         // rows per wave and iteration
  const int K = p.K;
  const int lane = threadIdx.x & 63;
  const int c = lane % W;
  const int g = lane / W;
  const int e0 = min(c * EPL, K - EPL);
  const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t nwaves = (int64_t)gridDim.x * 4;
  zero_scales(p.init, wave * 64 + lane, nwaves * 64);
  for (int64_t r0 = wave * ROWS; r0 < p.rows; r0 += nwaves * ROWS) {
    u32x4 raw[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t row = min(r0 + u * RPI + g, p.rows - 1);
      raw[u] = *reinterpret_cast<const u32x4_u*>(p.x + row * p.stride_row_bytes + e0 * ESZ);
    }
    zero_residual_rows(p.init, r0, min((int64_t)ROWS, p.rows - r0), lane);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t row = r0 + u * RPI + g;
      float v[EPL];
      const uint32_t bits[4] = {raw[u].x, raw[u].y, raw[u].z, raw[u].w};
      decode_elements<DT>(bits, v);
      float am = 0.0f;
#pragma unroll
      for (int j = 0; j < EPL; ++j) am = fmaxf(am, fabsf(v[j]));
      am = group_max_lanes<W>(am);
      const float s = round16<DT>(fmaxf(am, round16<DT>(kEps)) / p.qmax);
      const bool plain = s >= 0x1p-100f && s < 0x1p125f;
      const float inv = recip_rn(s);
      uint32_t yb[EPL];
#pragma unroll
      for (int j = 0; j < EPL; ++j) {
        float q = exact_quotient(v[j], s, inv);
        if (!plain) q = v[j] / s;
        q = round16<DT>(q);
        yb[j] = __float_as_uint((q != q ? 0.0f : fminf(fmaxf(rintf(q), -p.qmax), p.qmax)) + kMagic);
      }
      if (row < p.rows && c * EPL < K) {
        int8_t* dst = p.codes + row * K + e0;
        const uint32_t w0 = pack_low_bytes(yb[0], yb[1], yb[2], yb[3]);
        if constexpr (EPL == 8) {
          st_stream8_u(dst, u32x2{w0, pack_low_bytes(yb[4], yb[5], yb[6], yb[7])});
        } else {
          __builtin_nontemporal_store(w0, reinterpret_cast<u32_u*>(dst));
        }
      }
      if (row < p.rows && c == 0) p.scale[row] = s;
    }
  }
}

// Workgroups of four waves, each of which takes rows_per_wave rows at a time.
dim3 rows_grid(int64_t rows, int rows_per_wave, int most) {
  const int64_t waves = (rows + rows_per_wave - 1) / rows_per_wave;
  return dim3((unsigned)std::min<int64_t>((waves + 3) / 4, most));
}

template <int W>
void launch_rows_any_w(const RowsParams& p, int dtype, hipStream_t s) {
  const dim3 grid = rows_grid(p.rows, 64 / W * 4, 256 * 16), b(256);
  if (dtype == kF32) hipLaunchKernelGGL((quantize_rows_tile_kernel<W, kF32>), grid, b, 0, s, p);
  else if (dtype == kBF16) hipLaunchKernelGGL((quantize_rows_tile_kernel<W, kBF16>), grid, b, 0, s, p);
  else hipLaunchKernelGGL((quantize_rows_tile_kernel<W, kF16>), grid, b, 0, s, p);
}

void launch_rows_any(const RowsParams& p, int dtype, hipStream_t s) {
  const int lanes = (p.K + (dtype == kF32 ? 4 : 8) - 1) / (dtype == kF32 ? 4 : 8);
  if (lanes <= 2) launch_rows_any_w<2>(p, dtype, s);
  else if (lanes <= 4) launch_rows_any_w<4>(p, dtype, s);
  else if (lanes <= 8) launch_rows_any_w<8>(p, dtype, s);
  else if (lanes <= 16) launch_rows_any_w<16>(p, dtype, s);
  else if (lanes <= 32) launch_rows_any_w<32>(p, dtype, s);
  else launch_rows_any_w<64>(p, dtype, s);
}

template <int LPR, bool INIT>
void launch_rows16_init(const RowsParams& p, int dtype, hipStream_t s) {
  auto fn = dtype == kF32    ? quantize_rows16_kernel<LPR, kF32, INIT>
            : dtype == kBF16 ? quantize_rows16_kernel<LPR, kBF16, INIT>
                             : quantize_rows16_kernel<LPR, kF16, INIT>;
  const dim3 grid = rows_grid(p.rows, 64 / LPR, 256 * 32);
  hipLaunchKernelGGL(fn, grid, dim3(256), 0, s, p.x, p.stride_row_bytes, p.rows, p.codes, p.scale, p.qmax, grid.x * 4,
                     p.init);
}

template <int LPR>
void launch_rows16(const RowsParams& p, int dtype, hipStream_t s) {
  if (p.init.resid || p.init.n_rscale) launch_rows16_init<LPR, true>(p, dtype, s);
  else launch_rows16_init<LPR, false>(p, dtype, s);
}

// The zero residual and scales of the paths that do not write them themselves.
__global__ __launch_bounds__(256) void zero_residual_kernel(int8_t* __restrict__ resid, int64_t bytes,
                                                            float* __restrict__ rscale, int64_t n_rscale) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, n = (int64_t)gridDim.x * 256;
  for (int64_t i = t * 16; i < bytes; i += n * 16) {
    if (i + 16 <= bytes) {
      st_stream16_u(resid + i, u32x4{0u, 0u, 0u, 0u});
    } else {
      for (int64_t b = i; b < bytes; ++b) resid[b] = 0;
    }
  }
  for (int64_t i = t; i < n_rscale; i += n) rscale[i] = 0.0f;
}

void launch_zero_residual(int8_t* resid, int64_t bytes, float* rscale, int64_t n_rscale, hipStream_t s) {
  if (!resid) bytes = 0;
  if (!rscale) n_rscale = 0;
  if (bytes == 0 && n_rscale == 0) return;
  const int64_t blocks = (std::max(bytes / 16, n_rscale) + 255) / 256 + 1;
  hipLaunchKernelGGL(zero_residual_kernel, dim3((unsigned)std::min<int64_t>(blocks, 4096)), dim3(256), 0, s, resid,
                     bytes, rscale, n_rscale);
}

// Rows shorter or longer than the tile kernel takes: one wavefront per row; lanes
// stride over K. 16-bit
// dtypes in their own precision (RN16 after each fp32 operation).
__global__ __launch_bounds__(256) void quantize_rows_kernel(const void* __restrict__ x, int dtype, int64_t stride_row,
                                                            int64_t rows, int K, float qmax,
                                                            int8_t* __restrict__ codes, float* __restrict__ scale) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;  // whole wavefront exits together
  const int64_t base = row * stride_row;
  float am = 0.0f;
  for (int j = lane; j < K; j += 64) am = fmaxf(am, fabsf(load_act(x, base + j, dtype)));
  am = wave_max(am);
  const float s = round16_rt(dtype, fmaxf(am, round16_rt(dtype, kEps)) / qmax);
  for (int j = lane; j < K; j += 64) {
    // IEEE division: an fp16 scale that rounded to 0 gives +-inf (clamped to
    // +-qmax) for x != 0 and NaN for x = 0, which the int8 conversion of the
    // reference turns into 0
    const float q = round16_rt(dtype, load_act(x, base + j, dtype) / s);
    const float c = q != q ? 0.0f : fminf(fmaxf(rintf(q), -qmax), qmax);
    codes[row * K + j] = (int8_t)(int)c;
  }
  if (lane == 0) scale[row] = s;
}

// float64 rows (any K, alignment of a double): one wavefront per row, the
// arithmetic in float64 as torch does for a float64 h0; the scale is stored
// rounded to fp32 (the pool's scale dtype), the codes use the float64 scale.
__global__ __launch_bounds__(256) void quantize_rows_f64_kernel(const double* __restrict__ x, int64_t stride_row,
                                                                int64_t rows, int K, double qmax,
                                                                int8_t* __restrict__ codes, float* __restrict__ scale) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;  // whole wavefront exits together
  const double* xr = x + row * stride_row;
  double am = 0.0;
  for (int j = lane; j < K; j += 64) am = fmax(am, fabs(xr[j]));
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) am = fmax(am, __shfl_xor(am, m, 64));
  const double s = fmax(am, 1e-12) / qmax;
  for (int j = lane; j < K; j += 64) codes[row * K + j] = (int8_t)(int)fmin(fmax(rint(xr[j] / s), -qmax), qmax);
  if (lane == 0) scale[row] = (float)s;
}

// [M, K, V] matrices with K <= 256: the tile of the statequant step
// (ck_statequant.h). A workgroup covers up to 40 groups of CPT columns of one
// matrix, a thread one column group and one of S slices of the K rows (padded to
// the template K), so its rows stay in registers, the column amax takes one
// exchange through LDS, and a row of a slice is one contiguous access. CPT = 4
// at any alignment, 1 for V < 4.
// In the same pass, where asked for: the dequantized values (deq), a zero
// residual (e, e_bytes per element) and its zero scales, which took the caller
// a launch and a pass over memory each.
// Bound: HBM (4 bytes read, 1 written per element, more with deq or e): 5.8 TB/s at
// 8224 matrices of [128, 128], 117.0 us (cached code stores 121.8).
// Measured, init_quant_state of [16, 32, 128, 128] fp32 with an int8 residual
// (50.9 MB): 43.2 -> 12.3 us a call; before, a launch for the codes (8 lanes of
// 16 bytes per row), two torch passes for values that were dropped and two
// fills.
// IEEE: the form of ck_statequant.h that the shape takes (ingest_ieee).
// The arguments that a workgroup needs before its first load are the first twelve
// dwords, which the dispatch preloads. MORE: something is asked for besides codes
// and scales.
struct ColsInit {
  float* deq;      // or null
  char* e;         // or null
  int e_bytes;     // 1, 2 or 4
  float* e_scale;  // or null
};

struct ColsParams {
  const float* x;
  int8_t* codes;
  float* scale;
  int V, K;
  qs::ColTiles tiles;
  float qmax;
  ColsInit init;
};

template <int K, int FORM, bool MK, bool IEEE, bool MORE>
__global__ __launch_bounds__((qs::kThreadsFor<K, qs::TileShape<FORM, K>::GROUPS>)) void quantize_cols_tile_kernel(
    const float* __restrict__ x, int8_t* __restrict__ codes, float* __restrict__ scale, int V, int nvt, int width,
    int groups, uint32_t inv_groups, float qmax, int k_rows, const ColsInit init) {
  constexpr int CPT = qs::TileShape<FORM, K>::CPT;
  constexpr int S = qs::kSlicesFor<K>;
  constexpr int R = K / S;  // rows per slice
  constexpr int NC = qs::TileShape<FORM, K>::NC;
  __shared__ float red[S][NC];
  const int m = nvt == 1 ? blockIdx.x : blockIdx.x / nvt;
  const qs::ColTiles tiles{nvt, width, groups, inv_groups, (qs::TileForm)FORM};
  const qs::TilePlace pl = qs::tile_place<FORM, S>(tiles, V, blockIdx.x - m * nvt);
  const int ks = pl.ks;
  const int lc = pl.cg * CPT;
  const int c0 = pl.col;
  const bool colok = c0 >= 0;
  const int r0 = ks * R;
  const int KA = MK ? k_rows : K;  // rows that exist
  const int64_t base = (int64_t)m * KA * V + (int64_t)r0 * V + c0;
  float v[R][CPT];
#pragma unroll
  for (int r = 0; r < R; ++r) {
#pragma unroll
    for (int j = 0; j < CPT; ++j) v[r][j] = 0.0f;
    if (colok && (!MK || r0 + r < KA)) qs::ld_f32<CPT>(x + base + (int64_t)r * V, v[r]);
  }
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    float am = fabsf(v[0][j]);
#pragma unroll
    for (int r = 1; r < R; ++r) am = fmaxf(am, fabsf(v[r][j]));
    red[ks][lc + j] = am;
  }
  __syncthreads();
  if (!colok) return;
  float s[CPT], inv[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    s[j] = fmaxf(qs::ingest_amax<IEEE, S, NC>(red, lc + j), kEps) / qmax;
    inv[j] = recip_rn(s[j]);
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (MK && r0 + r >= KA) continue;
    uint32_t yb[CPT];
    float d[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      yb[j] = qs::ingest_code<IEEE>(v[r][j], s[j], inv[j], qmax);
      d[j] = code_i8(yb[j], 0) * s[j];
    }
    const int64_t i = base + (int64_t)r * V;
    if constexpr (FORM == qs::kTileFull) {  // whole 128-byte pieces of a row stream
      __builtin_nontemporal_store(qs::pack_codes<CPT>(yb), reinterpret_cast<u32_u*>(codes + i));
    } else {
      qs::st_b8<CPT>(codes + i, qs::pack_codes<CPT>(yb));
    }
    if constexpr (MORE) {
      if (init.deq) qs::st_f32<CPT>(init.deq + i, d);
      if (init.e) {
        const uint32_t zw[(CPT + 1) / 2] = {};
        const float zf[CPT] = {};
        if (init.e_bytes == 1) qs::st_b8<CPT>(init.e + i, 0u);
        else if (init.e_bytes == 2) qs::st_b16<CPT>(reinterpret_cast<uint16_t*>(init.e) + i, zw);
        else qs::st_f32<CPT>(reinterpret_cast<float*>(init.e) + i, zf);
      }
    }
  }
  if (ks == 0) {
    qs::st_f32<CPT>(scale + (int64_t)m * V + c0, s);
    if (MORE && init.e_scale) {
      const float zf[CPT] = {};
      qs::st_f32<CPT>(init.e_scale + (int64_t)m * V + c0, zf);
    }
  }
}

template <int KP, int FORM, bool MK, bool IEEE>
void launch_cols_kp(const ColsParams& p, int64_t M, hipStream_t s) {
  const ColsInit& in = p.init;
  auto fn = in.deq || in.e || in.e_scale ? quantize_cols_tile_kernel<KP, FORM, MK, IEEE, true>
                                         : quantize_cols_tile_kernel<KP, FORM, MK, IEEE, false>;
  const qs::ColTiles& t = p.tiles;
  hipLaunchKernelGGL(fn, dim3((unsigned)(M * t.nvt)), dim3((unsigned)qs::tile_threads(t, qs::kSlicesFor<KP>)), 0, s,
                     p.x, p.codes, p.scale, p.V, t.nvt, t.width, t.groups, t.inv, p.qmax, p.K, in);
}

template <int FORM, bool MK, bool IEEE>
void launch_cols(const ColsParams& p, int KP, int64_t M, hipStream_t s) {
  switch (KP) {
    case 16: launch_cols_kp<16, FORM, MK, IEEE>(p, M, s); break;
    case 32: launch_cols_kp<32, FORM, MK, IEEE>(p, M, s); break;
    case 64: launch_cols_kp<64, FORM, MK, IEEE>(p, M, s); break;
    case 128: launch_cols_kp<128, FORM, MK, IEEE>(p, M, s); break;
    default: launch_cols_kp<256, FORM, MK, IEEE>(p, M, s); break;
  }
}

template <int FORM>
void launch_cols_form(const ColsParams& p, int KP, int64_t M, bool ieee, hipStream_t s) {
  if (KP != p.K) launch_cols<FORM, true, true>(p, KP, M, s);
  else if (ieee) launch_cols<FORM, false, true>(p, KP, M, s);
  else launch_cols<FORM, false, false>(p, KP, M, s);  // V % 4 == 0: kTileOne past 2^30 columns
}

// K above 256, and many small matrices (few_columns): one thread per (matrix,
// V-column); consecutive threads take consecutive columns so every K-row access is
// coalesced. The two passes over a column's rows are what a small matrix waits
// for, and a narrow one's rows lie apart, so a residual and the dequantized values
// are written by launches of their own (us a call: [4, 8, 1024, 64] int8 residual
// 342 in the second pass, 286 so).
__global__ __launch_bounds__(256) void quantize_cols_kernel(const float* __restrict__ x, int64_t M, int K, int V,
                                                            float qmax, int8_t* __restrict__ codes,
                                                            float* __restrict__ scale) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= M * V) return;
  const int64_t m = t / V;
  const int c = (int)(t % V);
  const float* xm = x + m * K * V + c;
  float am = 0.0f;
  for (int j = 0; j < K; ++j) am = fmaxf(am, fabsf(xm[(int64_t)j * V]));
  const float s = fmaxf(am, kEps) / qmax;
  int8_t* cm = codes + m * K * V + c;
  for (int j = 0; j < K; ++j) {
    const float q = fminf(fmaxf(rintf(xm[(int64_t)j * V] / s), -qmax), qmax);
    cm[(int64_t)j * V] = (int8_t)(int)q;
  }
  scale[m * V + c] = s;
}

// deq = code * scale of those: a workgroup takes `per` of the M K rows at a time
// (1024 elements, or one row).
__global__ __launch_bounds__(256) void dequantize_cols_kernel(const int8_t* __restrict__ codes,
                                                              const float* __restrict__ scale, int64_t rows, int K,
                                                              int V, int per, float* __restrict__ deq) {
  for (int64_t r0 = (int64_t)blockIdx.x * per; r0 < rows; r0 += (int64_t)gridDim.x * per) {
    const int64_t m0 = r0 / K;
    const uint32_t k0 = (uint32_t)(r0 - m0 * K), n = (uint32_t)min((int64_t)per, rows - r0) * (uint32_t)V;
    for (uint32_t i = threadIdx.x; i < n; i += 256) {
      const uint32_t row = i / (uint32_t)V, c = i - row * (uint32_t)V;
      deq[r0 * V + i] = (float)codes[r0 * V + i] * scale[(m0 + (k0 + row) / (uint32_t)K) * V + c];
    }
  }
}

}  // namespace
}  // namespace ck

extern "C" int ck_quantize_rows(const void* x, int x_dtype, int64_t stride_row, int64_t rows, int K, float qmax,
                                int8_t* codes, float* scale, void* stream) {
  return ck_quantize_rows_init(x, x_dtype, stride_row, rows, K, qmax, codes, scale, nullptr, 0, nullptr, 0, stream);
}

extern "C" int ck_quantize_rows_init(const void* x, int x_dtype, int64_t stride_row, int64_t rows, int K, float qmax,
                                     int8_t* codes, float* scale, int8_t* resid, int resid_row_bytes, float* rscale,
                                     int64_t n_rscale, void* stream) {
  using namespace ck;
  if (rows < 0 || K <= 0 || stride_row < K) return fail(CK_EINVAL, "bad sizes rows=%lld K=%d", (long long)rows, K);
  if (!valid_dtype(x_dtype) && x_dtype != CK_DTYPE_F64) return fail(CK_EINVAL, "unsupported dtype code %d", x_dtype);
  if (!(qmax >= 1.0f && qmax <= 127.0f)) return fail(CK_EINVAL, "qmax must be in [1, 127]");
  if ((resid && resid_row_bytes <= 0) || (rscale && n_rscale <= 0))
    return fail(CK_EINVAL, "bad sizes of the residual: %d bytes per row, %lld scales", resid_row_bytes,
                (long long)n_rscale);
  if (rows == 0) return ok();
  if (!x || !codes || !scale) return fail(CK_EINVAL, "null pointer argument");
  if (!rscale) n_rscale = 0;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (x_dtype != CK_DTYPE_F64) {
    const int esz = x_dtype == kF32 ? 4 : 2, epl = 16 / esz;
    const bool aligned = ((reinterpret_cast<uintptr_t>(x) | (uintptr_t)(stride_row * esz) |
                           reinterpret_cast<uintptr_t>(codes)) & 15) == 0;
    if (K >= epl && K <= 64 * epl) {
      const RowsParams p{static_cast<const char*>(x), stride_row * esz, rows, K, qmax, codes, scale,
                         RowsInit{resid, resid_row_bytes, rscale, n_rscale}};
      switch (aligned ? K : 0) {
        case 16: launch_rows16<1>(p, x_dtype, s); break;
        case 32: launch_rows16<2>(p, x_dtype, s); break;
        case 64: launch_rows16<4>(p, x_dtype, s); break;
        case 128: launch_rows16<8>(p, x_dtype, s); break;
        case 256: launch_rows16<16>(p, x_dtype, s); break;
        default: launch_rows_any(p, x_dtype, s); break;
      }
      return check_launch("ck_quantize_rows");
    }
  }
  if (x_dtype == CK_DTYPE_F64 && (reinterpret_cast<uintptr_t>(x) & 7))
    return fail(CK_EINVAL, "float64 rows must be 8-byte aligned");
  const int64_t grid = (rows + 3) / 4;
  if (grid > 0x7fffffff) return fail(CK_EUNSUPPORTED, "too many rows");
  launch_zero_residual(resid, rows * resid_row_bytes, rscale, n_rscale, s);
  if (x_dtype == CK_DTYPE_F64)
    hipLaunchKernelGGL(quantize_rows_f64_kernel, dim3((unsigned)grid), dim3(256), 0, s, static_cast<const double*>(x),
                       stride_row, rows, K, (double)qmax, codes, scale);
  else
    hipLaunchKernelGGL(quantize_rows_kernel, dim3((unsigned)grid), dim3(256), 0, s, x, x_dtype, stride_row, rows, K,
                       qmax, codes, scale);
  return check_launch("ck_quantize_rows");
}

extern "C" int ck_quantize_cols(const float* x, int64_t M, int K, int V, float qmax, int8_t* codes, float* scale,
                                void* stream) {
  return ck_quantize_cols_init(x, M, K, V, qmax, codes, scale, nullptr, nullptr, 0, nullptr, stream);
}

extern "C" int ck_quantize_cols_init(const float* x, int64_t M, int K, int V, float qmax, int8_t* codes, float* scale,
                                     float* deq, void* e, int e_bytes, float* e_scale, void* stream) {
  using namespace ck;
  if (M < 0 || K <= 0 || V <= 0) return fail(CK_EINVAL, "bad sizes M=%lld K=%d V=%d", (long long)M, K, V);
  if (!(qmax >= 1.0f && qmax <= 127.0f)) return fail(CK_EINVAL, "qmax must be in [1, 127]");
  if (e && e_bytes != 1 && e_bytes != 2 && e_bytes != 4) return fail(CK_EINVAL, "e_bytes must be 1, 2 or 4");
  if (M == 0) return ok();
  if (!x || !codes || !scale) return fail(CK_EINVAL, "null pointer argument");
  if (e && (reinterpret_cast<uintptr_t>(e) & (e_bytes - 1))) return fail(CK_EINVAL, "misaligned residual");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const uintptr_t bits = qs::addr_bits(x, codes, scale);
  const int KP = K <= 256 ? qs::padded_k(K) : 0;
  const qs::ColTiles tiles = qs::col_tiles(V, KP, true, true);
  const bool ieee = qs::ingest_ieee(bits, M, K, V);
  if (K <= 256 && !(ieee && qs::few_columns(M, K, V))) {
    return launch_slices(M, tiles.nvt, qs::tile_threads(tiles, KP <= 128 ? 8 : 16), [&](int64_t m0, int64_t n) {
      const int64_t i = m0 * K * V, c = m0 * V;  // the slice's first matrix and column
      const ColsParams p{x + i, codes + i, scale + c, V, K, tiles, qmax,
                         ColsInit{deq ? deq + i : nullptr, e ? static_cast<char*>(e) + i * e_bytes : nullptr, e_bytes,
                                  e_scale ? e_scale + c : nullptr}};
      switch (tiles.form) {
        case qs::kTileFull: launch_cols_form<qs::kTileFull>(p, KP, n, ieee, s); break;
        case qs::kTileAny: launch_cols_form<qs::kTileAny>(p, KP, n, ieee, s); break;
        default: launch_cols_form<qs::kTileOne>(p, KP, n, ieee, s); break;
      }
      return check_launch("ck_quantize_cols");
    });
  }
  const int64_t grid = (M * V + 255) / 256;
  if (grid > 0x7fffffff) return fail(CK_EUNSUPPORTED, "too many columns");
  launch_zero_residual(static_cast<int8_t*>(e), M * K * V * e_bytes, e_scale, M * V, s);
  hipLaunchKernelGGL(quantize_cols_kernel, dim3((unsigned)grid), dim3(256), 0, s, x, M, K, V, qmax, codes, scale);
  if (deq) {
    const int64_t rows = M * K, per = std::max(1024 / V, 1), blocks = (rows + per - 1) / per;
    hipLaunchKernelGGL(dequantize_cols_kernel, dim3((unsigned)std::min<int64_t>(blocks, 1 << 16)), dim3(256), 0, s,
                       codes, scale, rows, K, V, (int)per, deq);
  }
  return check_launch("ck_quantize_cols");
}
