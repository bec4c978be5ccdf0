// rq_fp8.hip -- FP8 e4m3 activation encoding and GEMM on gfx950 matrix cores.
//
// Replaces ops::fp8_gemm (crates/runtimed-model/src/ops/fp8_gemm.rs:77-191):
//   - the reference encodes activations on the host, per element, with
//     f32_to_fp8_e4m3 (load_safetensors.rs:53-69) and no scale
//     (fp8_gemm.rs:94-101).  RQ_FP8_UNSCALED reproduces that encoder on the
//     device, bit for bit (nearest LUT value, ties to the lower magnitude).
//   - RQ_FP8_PER_TOKEN is the dynamic per-row scaling of the FP8 workload:
//     s = max|x|/448, codes e4m3_rne(x * (448/max|x|)).
//   - the product runs on v_mfma_f32_32x32x64_f8f6f4 (OCP e4m3 x e4m3, f32
//     accumulate) and applies x-scale * w-scale in the epilogue, where the
//     reference applies the per-channel scale as an extra broadcast_mul pass
//     (fp8_gemm.rs:180-186).
//
// GEMM tiling: a 256-thread workgroup computes a 256 x 256 tile of y with
// 128 x 128 per wave (4 x 4 MFMA tiles of 32 x 32, accumulators in AGPRs) for
// large problems (K-step 64 bytes, LDS rows of 80 bytes), or 128 x 128 with
// 64 x 64 per wave otherwise (K-step 128 bytes, rows of 144 bytes).  Two LDS
// buffers (double buffering); the row padding makes the 32 lanes that read
// one MFMA operand column touch distinct 16-byte bank groups.
//
// Roofline: MFMA-bound (fp8 dense peak 5.0 PFLOP/s); flops = 2*m*n*k.
#include "rq_e4m3.h"
#include "rq_epilogue.h"
#include "rq_internal.h"
#include "rq_pipe.h"

namespace rq {
namespace {

using namespace pipe;

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// One workgroup per activation row.
__global__ __launch_bounds__(256) void k_fp8_quant_rows(const void *__restrict__ x, int xtype,
                                                       int64_t k, int mode, uint8_t *__restrict__ xq,
                                                       float *__restrict__ xs) {
  __shared__ float red[4];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x;
  if (mode == RQ_FP8_UNSCALED) {
    for (int64_t t = tid; t < k; t += 256) xq[row * k + t] = (uint8_t)enc_e4m3_ref(load_x1(x, xtype, row * k + t));
    if (tid == 0) xs[row] = 1.0f;
    return;
  }
  float amax = 0.0f;
  for (int64_t t = tid; t < k; t += 256) amax = fmaxf(amax, fabsf(load_x1(x, xtype, row * k + t)));
  for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
  if ((tid & 63) == 0) red[tid >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  if (amax == 0.0f) {
    for (int64_t t = tid; t < k; t += 256) xq[row * k + t] = 0;
    if (tid == 0) xs[row] = 0.0f;
    return;
  }
  const float inv = 448.0f / amax;
  for (int64_t t = tid; t < k; t += 256) xq[row * k + t] = (uint8_t)enc_e4m3_rne(load_x1(x, xtype, row * k + t) * inv);
  if (tid == 0) xs[row] = amax / 448.0f;
}

// The same per-token encode with WPR waves per activation row (one, four rows
// a workgroup, or four): the row's maximum from 16-byte loads and a wave reduction,
// then the codes from a second pass over the row (an L2 hit, or the
// registers when the row is at most one batch), 4 (f32) or 8 (f16 / bf16)
// codes per store.  Same codes and scales as k_fp8_quant_rows (the maximum
// is exact in any order, enc_e4m3_rne_bf equals enc_e4m3_rne).  The
// activation type and the mode are template parameters: as run-time values
// the compiler turned each per-element choice into a branch.  One workgroup
// per row with scalar 2-byte loads took 21 us on 2048 x 4096 bf16.
template <int XT, bool SCALED, int WPR>
__global__ __launch_bounds__(256) void k_fp8_quant_waves(const void *__restrict__ x, int64_t m, int64_t k,
                                                        uint8_t *__restrict__ xq, float *__restrict__ xs) {
  constexpr bool F32X = XT == RQ_F32;
  constexpr int ES = F32X ? 4 : 8;  // elements per 16-byte chunk
  constexpr int T = 64 * WPR;  // threads a row
  const int lane = (int)threadIdx.x & (T - 1);
  const int64_t row = (int64_t)blockIdx.x * (4 / WPR) + threadIdx.x / T;
  if (row >= m) return;
  const int64_t nch = k / ES;
  const uint4 *src = reinterpret_cast<const uint4 *>(static_cast<const uint8_t *>(x) + row * k * (F32X ? 4 : 2));
  auto unpack = [&](const uint4 &v, float (&f)[ES]) {
    const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (F32X) {
        f[i] = __uint_as_float(u[i]);
      } else if constexpr (XT == RQ_BF16) {
        f[2 * i] = __uint_as_float(u[i] << 16);
        f[2 * i + 1] = __uint_as_float(u[i] & 0xFFFF0000u);
      } else {
        f[2 * i] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u[i] & 0xFFFFu));
        f[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u[i] >> 16));
      }
    }
  };
  // Batches of U chunks a lane, their loads issued together; a row of at
  // most one batch stays in registers between the two passes.
  constexpr int U = WPR == 1 ? 1 : F32X ? 4 : 2;
  uint4 buf[U];
  auto load_batch = [&](int64_t c0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t c = c0 + T * u;
      buf[u] = src[c < nch ? c : nch - 1];
    }
  };
  const bool resident = SCALED && nch <= T * U;
  float amax = 0.0f;
  bool nan = false;
  if constexpr (SCALED) {
    for (int64_t c0 = lane; c0 < nch; c0 += T * U) {
      load_batch(c0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float f[ES];
        unpack(buf[u], f);
        const bool live = c0 + T * u < nch;
#pragma unroll
        for (int i = 0; i < ES; ++i) {
          amax = fmaxf(amax, live ? fabsf(f[i]) : 0.0f);
          nan |= f[i] != f[i];
        }
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
    nan = __any(nan);
    if constexpr (WPR > 1) {
      __shared__ float red[WPR];
      __shared__ int bad[WPR];
      if ((lane & 63) == 0) red[lane >> 6] = amax, bad[lane >> 6] = nan;
      __syncthreads();
#pragma unroll
      for (int i = 0; i < WPR; ++i) amax = fmaxf(amax, red[i]), nan |= bad[i] != 0;
    }
  }
  // A row without NaN is encoded by the hardware conversion: for |v| <= 448
  // v_cvt_pk_fp8_f32 gives enc_e4m3_rne's code for every f32 input (compared
  // over all 2^32 of them on MI355X); v is clamped to +-448 first (the
  // product can exceed 448 by an ulp).  Rows with a NaN or an infinity (whose
  // product with inv = 0 is NaN) keep the software encoder, whose NaN code
  // differs.
  const bool hw = SCALED && !nan && amax != 0.0f && amax <= 3.4028235e38f;  // no NaN, no infinity
  // amax == 0: every code 0 (inv = 0 would turn NaN or infinite inputs into
  // NaN codes instead).
  const float inv = 448.0f / amax;
  const uint32_t keep = amax == 0.0f ? 0u : 0xFFu;
  uint8_t *dst = xq + row * k;
  for (int64_t c0 = lane; c0 < nch; c0 += T * U) {
    if (!resident) load_batch(c0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t c = c0 + T * u;
      float f[ES];
      unpack(buf[u], f);
      uint32_t word[ES / 4];
      if (hw) {
#pragma unroll
        for (int j = 0; j < ES / 4; ++j) {
          float v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = __builtin_amdgcn_fmed3f(f[4 * j + i] * inv, -448.0f, 448.0f);
          const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
          word[j] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], lo, true);
        }
      } else {
        uint32_t q[ES];
#pragma unroll
        for (int i = 0; i < ES; ++i) q[i] = SCALED ? enc_e4m3_rne_bf(f[i] * inv) & keep : enc_e4m3_ref(f[i]);
#pragma unroll
        for (int j = 0; j < ES / 4; ++j)
          word[j] = q[4 * j] | (q[4 * j + 1] << 8) | (q[4 * j + 2] << 16) | (q[4 * j + 3] << 24);
      }
      if (c < nch) {
        if constexpr (F32X) {
          *reinterpret_cast<uint32_t *>(dst + 4 * c) = word[0];
        } else {
          *reinterpret_cast<uint2 *>(dst + 8 * c) = make_uint2(word[0], word[1]);
        }
      }
    }
  }
  if (lane == 0) xs[row] = !SCALED ? 1.0f : amax == 0.0f ? 0.0f : amax / 448.0f;
}

// Scalar fallback for shapes the matrix-core kernels do not take (k % 16 != 0
// or misaligned operands).
__global__ __launch_bounds__(256) void k_fp8_gemm_scalar(const uint8_t *__restrict__ xq,
                                                        const float *__restrict__ xs, int64_t m,
                                                        const uint8_t *__restrict__ w,
                                                        const float *__restrict__ ws, int64_t n,
                                                        int64_t k, void *__restrict__ y, int ytype) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= m * n) return;
  const int64_t i = idx / n, j = idx - i * n;
  float acc = 0.0f;
  for (int64_t t = 0; t < k; ++t) acc = fmaf(dec_e4m3(xq[i * k + t]), dec_e4m3(w[j * k + t]), acc);
  const float sx = xs ? xs[i] : 1.0f, sw = ws ? ws[j] : 1.0f;
  store_out(y, ytype, idx, acc * (sx * sw));
}

// A BM x BN tile of y per 256-thread workgroup of WM x WN waves; each wave
// owns (BM/WM) x (BN/WN) = MI x NI MFMA tiles of 32 x 32.  With 128 x 128 wave
// tiles every 32-byte operand fragment read from LDS feeds four MFMAs.  BK is
// the K-step in bytes (64 or 128); LDS rows are BK + 16 bytes.
template <int BM, int BN, int WM, int WN, int BK>
__global__ __launch_bounds__(256) void k_fp8_gemm_mfma(const uint8_t *__restrict__ a,
                                                      const float *__restrict__ xs, int64_t m,
                                                      const uint8_t *__restrict__ b,
                                                      const float *__restrict__ ws, int64_t n,
                                                      int64_t k, void *__restrict__ y, int ytype) {
  static_assert(WM * WN == 4, "four waves");
  constexpr int LDS_STRIDE = BK + 16;
  constexpr int TPR = BK / 16;              // threads per row in a load round
  constexpr int RPR = 256 / TPR;            // rows per load round
  constexpr int MI = BM / WM / 32, NI = BN / WN / 32;
  constexpr int A_LOADS = BM / RPR, B_LOADS = BN / RPR;  // 16-byte loads per thread per step
  __shared__ __attribute__((aligned(16))) uint8_t As[2][BM * LDS_STRIDE];
  __shared__ __attribute__((aligned(16))) uint8_t Bs[2][BN * LDS_STRIDE];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int64_t m0 = (int64_t)blockIdx.y * BM, n0 = (int64_t)blockIdx.x * BN;

  // Global -> register staging: TPR threads per row, RPR rows per round.
  const int lrow = tid / TPR, lcol = (tid % TPR) * 16;
  uint4 ra[A_LOADS], rb[B_LOADS];
  auto gload = [&](int64_t k0) {
#pragma unroll
    for (int it = 0; it < A_LOADS; ++it) {
      const int64_t gm = m0 + lrow + RPR * it;
      ra[it] = gm < m ? *reinterpret_cast<const uint4 *>(a + gm * k + k0 + lcol) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int it = 0; it < B_LOADS; ++it) {
      const int64_t gn = n0 + lrow + RPR * it;
      rb[it] = gn < n ? *reinterpret_cast<const uint4 *>(b + gn * k + k0 + lcol) : make_uint4(0, 0, 0, 0);
    }
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int it = 0; it < A_LOADS; ++it)
      *reinterpret_cast<uint4 *>(&As[buf][(lrow + RPR * it) * LDS_STRIDE + lcol]) = ra[it];
#pragma unroll
    for (int it = 0; it < B_LOADS; ++it)
      *reinterpret_cast<uint4 *>(&Bs[buf][(lrow + RPR * it) * LDS_STRIDE + lcol]) = rb[it];
  };

  f32x16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = (f32x16){0};

  const int64_t nk = k / BK;
  gload(0);
  sstore(0);
  __syncthreads();
  for (int64_t kt = 0; kt < nk; ++kt) {
    const int buf = (int)(kt & 1);
    if (kt + 1 < nk) gload((kt + 1) * BK);
#pragma unroll
    for (int ks = 0; ks < BK / 64; ++ks) {
      const int kb = ks * 64 + 32 * (lane >> 5);
      i32x8 fa[MI], fb[NI];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int ar = wm * (BM / WM) + i * 32 + (lane & 31);
        const uint4 *pa = reinterpret_cast<const uint4 *>(&As[buf][ar * LDS_STRIDE + kb]);
        const uint4 a0 = pa[0], a1 = pa[1];
        fa[i] = (i32x8){(int)a0.x, (int)a0.y, (int)a0.z, (int)a0.w, (int)a1.x, (int)a1.y, (int)a1.z, (int)a1.w};
      }
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const int br = wn * (BN / WN) + j * 32 + (lane & 31);
        const uint4 *pb = reinterpret_cast<const uint4 *>(&Bs[buf][br * LDS_STRIDE + kb]);
        const uint4 b0 = pb[0], b1 = pb[1];
        fb[j] = (i32x8){(int)b0.x, (int)b0.y, (int)b0.z, (int)b0.w, (int)b1.x, (int)b1.y, (int)b1.z, (int)b1.w};
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[i], fb[j], acc[i][j], 0, 0,
                                                                      0, 0, 0, 0);
    }
    if (kt + 1 < nk) sstore(buf ^ 1);
    __syncthreads();
  }

  const bool vec = vec_stores_ok(y, n);
  float sx[MI][4], sw[NI][4];
#pragma unroll
  for (int i = 0; i < MI; ++i) tile_row_scales(xs, m, m0 + wm * (BM / WM) + i * 32, lane, sx[i]);
#pragma unroll
  for (int j = 0; j < NI; ++j) tile_col_scales(ws, n, n0 + wn * (BN / WN) + j * 32, lane, sw[j]);
  const Out o{y, nullptr, ytype, 0};
  const float nob[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  static_for<MI>([&](auto I) {
    static_for<NI>([&](auto J) {
      store_tile32<true>(acc[I][J], o, m, n, m0 + wm * (BM / WM) + I * 32, n0 + wn * (BN / WN) + J * 32, sx[I],
                         sw[J], nob, xs, ws, lane, vec);
    });
  });
}

// ---- few tiles: 16 MT rows x 32 columns a workgroup, K split over its waves ----
//
// Decode and verify rows (and more rows on narrow weights) leave the 128 x 128
// tiles on a fraction of the CUs, each walking the whole of K behind one
// barrier a step.  Here a workgroup owns 16 MT rows of x and 32 rows of w; its
// waves share K in steps of 128 inputs, each with its operands straight from
// global memory (no LDS, no barrier until the waves' sums meet): a lane loads
// two 16-byte pieces a row and step, four lanes 64 consecutive bytes of a row.
// One step of loads a wave is in flight: the wave then fits eight to a SIMD (48
// registers at MT = 1), which hides more than two, three or four steps in fewer
// waves did (5 x 14336 x 4096: 16.9 us against 17.7 / 24.5 / 18.7).  Plain loads:
// with non-temporal ones each half of a 128-byte line went to memory by itself
// (17.1 us against 13.1).  The order of the inputs inside a step
// is the same for both operands, so it need not be the natural one.  The
// codes are widened to f16, exactly, and the products summed on the f16 matrix
// cores: for these sizes as fast as the fp8 ones within 10 % and without their
// truncated sums (error against 64 bits 6e-8 instead of 1.4e-5).  Bound: the
// weight bytes (HBM) for few rows; 5 x 14336 x 4096 30.6 -> 13.1 us (4.5 TB/s),
// 5 x 4096 x 4096 30.1 -> 7.7, 512 x 2048 x 4096 29.9 -> 26.9, 100 x 2000 x 2048
// 20.9 -> 10.1 against the 128 x 128 tiles, 100 x 3000 x 2016 2479 -> 8.2 against
// one thread an output.  A row of x past m or of w past n
// re-reads the last one; its results are not stored.  TAIL: k % 128 != 0 (k %
// 16 == 0).
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

template <int MT, bool TAIL>
__global__ __launch_bounds__(512) void k_fp8_skinny(const uint8_t *__restrict__ a, const float *__restrict__ xs,
                                                    int64_t m, const uint8_t *__restrict__ b,
                                                    const float *__restrict__ ws, int64_t n, int64_t k,
                                                    void *__restrict__ y, int ytype, int tm) {
    extern __shared__ __attribute__((aligned(16))) float red[];  // [wave][2 MT tiles][4][64]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int W = (int)(blockDim.x >> 6);
  // XCD x (workgroups x, x + 8, ..) takes a run of consecutive tiles, rows of
  // x fastest, so that tiles sharing weights share an L2.
  const int T = (int)gridDim.x, xcd = (int)blockIdx.x & 7, qt = T >> 3, rt = T & 7;
  const int unit = xcd * qt + (xcd < rt ? xcd : rt) + ((int)blockIdx.x >> 3);
  const int nt = unit / tm, mt = unit - nt * tm;
  const int64_t m0 = 16 * MT * (int64_t)mt, n0 = 32 * (int64_t)nt;
  const int steps = (int)((k + 127) / 128);
  const int s0 = (int)((int64_t)steps * wave / W), s1 = (int)((int64_t)steps * (wave + 1) / W);
  const int r = lane & 15, g = lane >> 4;

  // Uniform tile bases, 32-bit lane offsets (32 or 64 rows of k <= 2^24 bytes).
  const uint8_t *const ta = a + m0 * k, *const tb = b + n0 * k;
  uint32_t oa[MT], ob[2];
#pragma unroll
  for (int i = 0; i < MT; ++i) oa[i] = (uint32_t)(m0 + 16 * i + r < m ? 16 * i + r : (int)(m - 1 - m0)) * (uint32_t)k;
#pragma unroll
  for (int j = 0; j < 2; ++j) ob[j] = (uint32_t)(n0 + 16 * j + r < n ? 16 * j + r : (int)(n - 1 - n0)) * (uint32_t)k;
  u32x4 fa[MT][2], fb[2][2];
  const int last = s1 > s0 ? s1 - 1 : 0;
  auto fill = [&](int s) __attribute__((always_inline)) {
    const int base = 128 * (s < last ? s : last);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int o = base + 16 * g + 64 * h;
      const uint32_t oc = !TAIL || o < (int)k ? o : 0;
#pragma unroll
      for (int j = 0; j < 2; ++j) fb[j][h] = *reinterpret_cast<const u32x4 *>(tb + (ob[j] + oc));
#pragma unroll
      for (int i = 0; i < MT; ++i) fa[i][h] = *reinterpret_cast<const u32x4 *>(ta + (oa[i] + oc));
    }
  };
  // Eight codes of a piece (half h) in f16, exactly.
  auto wide = [](const u32x4 &x, int h) __attribute__((always_inline)) {
    const uint32_t w0 = h ? x.z : x.x, w1 = h ? x.w : x.y;
    const f16x2 v0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, 1.0f, false);
    const f16x2 v1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, 1.0f, true);
    const f16x2 v2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, 1.0f, false);
    const f16x2 v3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, 1.0f, true);
    return (f16x8){v0[0], v0[1], v1[0], v1[1], v2[0], v2[1], v3[0], v3[1]};
  };
  f32x4 acc[MT][2];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (f32x4){0, 0, 0, 0};
  auto emit = [&](int s) __attribute__((always_inline)) {
    // Pieces past k hold the row's first piece: zeros in x's (w's codes are
    // finite there, or the row's sum is a NaN in any case).
    if (TAIL && s == steps - 1) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < MT; ++i)
          if (128 * s + 16 * g + 64 * h >= (int)k) fa[i][h] = (u32x4){0, 0, 0, 0};
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const f16x8 ob8 = wide(fb[j][p >> 1], p & 1);
#pragma unroll
        for (int i = 0; i < MT; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wide(fa[i][p >> 1], p & 1), ob8, acc[i][j], 0, 0, 0);
      }
  };
  fill(s0);
  for (int s = s0; s < s1; ++s) {
    emit(s);
    fill(s + 1);
  }

  // The waves' tiles summed in wave order.  Slot q of the tile: MFMA tile
  // q / 4 (row tile q / 8, column tile (q / 4) % 2), element q % 4: rows 16 i
  // + 4 (lane / 16) + q % 4, column 16 j + lane % 16.
  constexpr int Q = 8 * MT;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) red[(wave * Q + (2 * i + j) * 4 + e) * 64 + lane] = acc[i][j][e];
  __syncthreads();
  for (int q = wave; q < Q; q += W) {
    const int64_t row = m0 + 16 * (q >> 3) + 4 * (lane >> 4) + (q & 3);
    const int64_t col = n0 + 16 * ((q >> 2) & 1) + (lane & 15);
    if (row < m && col < n) {
      float v = red[q * 64 + lane];
      for (int w = 1; w < W; ++w) v += red[(w * Q + q) * 64 + lane];
      store_out(y, ytype, row * n + col, v * ((xs ? xs[row] : 1.0f) * (ws ? ws[col] : 1.0f)));
    }
  }
}

// ---- pipelined 256 x 256 kernel ------------------------------------------
//
// Four waves of 128 x 128 (4 x 4 MFMA tiles, 256 accumulators in AGPRs).  K
// advances 64 bytes per step through four LDS stages of 32 KB (A rows then B
// rows, 64 bytes each), filled by direct global -> LDS loads
// (global_load_lds_dwordx4: lane L of a wave lands at base + 16*L) issued
// three steps ahead, so about three steps of MFMA work cover the load latency
// without staging registers.  Rows carry no padding; instead the four 16-byte
// chunks of row r are stored XOR-swizzled by (r >> 2) & 3, so the 32 lanes
// that read one operand column of 32 rows hit 16 distinct 16-byte bank slots.

// Issue the direct loads of one stage.  The LDS pointer is __restrict__ so
// that, once inlined, the accesses carry scoped alias metadata and the
// compiler's wait insertion can tell the four stage buffers apart instead of
// draining every load before each LDS read.
__device__ __forceinline__ void pipe_issue(uint8_t *__restrict__ S, const uint8_t *const (&ga)[4],
                                           const uint8_t *const (&gb)[4], int64_t k0, int wave) {
#pragma unroll
  for (int j = 0; j < 4; ++j)
    __builtin_amdgcn_global_load_lds(ga[j] + k0, (lds_void *)(S + (64 * wave + 16 * j) * 64), 16, 0, 0);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    __builtin_amdgcn_global_load_lds(gb[j] + k0, (lds_void *)(S + P_B + (64 * wave + 16 * j) * 64), 16, 0, 0);
}

__device__ __forceinline__ i32x8 frag_a(const Frags &F, int i) {
  const u32x4 x0 = F.x[2 * i], x1 = F.x[2 * i + 1];
  return (i32x8){(int)x0.x, (int)x0.y, (int)x0.z, (int)x0.w, (int)x1.x, (int)x1.y, (int)x1.z, (int)x1.w};
}

// The 16 MFMAs of one K-step on `cur`, each followed by one LDS read of the
// next step's fragments into `nxt` (nullptr S: no next step), pinned in that
// order so the LDS reads run under the matrix work.
__device__ __forceinline__ void mfma_step(const Frags &cur, Frags &nxt, const uint8_t *__restrict__ S,
                                          f32x16 (&acc)[4][4], int wm, int wn, int lane) {
  static_for<4>([&](auto I) {
    const i32x8 fa = frag_a(cur, I);
    static_for<4>([&](auto J) {
      const i32x8 fb = frag_a(cur, 4 + J);
      acc[I][J] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc[I][J], 0, 0, 0, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (S) nxt.x[4 * I + J] = ds_read16(frag_addr(S, 4 * I + J, wm, wn, lane));
      __builtin_amdgcn_sched_barrier(0);
    });
  });
}

__global__ __launch_bounds__(256) void k_fp8_gemm_pipe(const uint8_t *__restrict__ a,
                                                      const float *__restrict__ xs, int64_t m,
                                                      const uint8_t *__restrict__ b,
                                                      const float *__restrict__ ws, int64_t n,
                                                      int64_t k, void *__restrict__ y, int ytype) {
  // four stages, one array: after the loop it holds the staged output tile
  __shared__ __attribute__((aligned(1024))) uint8_t SM[4 * P_STAGE];
  uint8_t *const S0 = SM, *const S1 = SM + P_STAGE, *const S2 = SM + 2 * P_STAGE, *const S3 = SM + 3 * P_STAGE;
  uint8_t *const SB[4] = {S0, S1, S2, S3};
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t m0 = (int64_t)blockIdx.y * 256, n0 = (int64_t)blockIdx.x * 256;
  const int64_t nk = k / 64;

  // Load assignment: wave w fills rows 64w .. 64w+63 of the A and B halves of
  // a stage, 16 rows (4 lanes x 16 bytes per row) per instruction.  Rows past
  // m or n re-read the last valid row; their results are never stored.
  const uint8_t *ga[4], *gb[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = 64 * wave + 16 * j + (lane >> 2);
    const int gc = (lane & 3) ^ swz(r);
    const int64_t gm = m0 + r < m ? m0 + r : m - 1;
    const int64_t gn = n0 + r < n ? n0 + r : n - 1;
    ga[j] = a + gm * k + 16 * gc;
    gb[j] = b + gn * k + 16 * gc;
  }

  f32x16 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (f32x16){0};

  // Stages 0..3 in flight; fragments of step 0 in registers.
#pragma unroll
  for (int s = 0; s < 4; ++s)
    if (s < nk) pipe_issue(SB[s], ga, gb, 64 * s, wave);
  if (nk > 3) wait_vm<24>();
  else if (nk > 2) wait_vm<16>();
  else if (nk > 1) wait_vm<8>();
  else wait_vm<0>();
  __builtin_amdgcn_s_barrier();
  Frags F0, F1;
  read_all(S0, F0, wm, wn, lane);
  wait_lds(F0);

  // Step t: stage t's fragments are in registers.  Make stage t+1 resident
  // (its loads landed in every wave: wait, then a bare barrier -- a release
  // fence would drain the younger stages too), refill buffer t%4 with stage
  // t+4 (everyone finished reading it before this barrier), then run step t's
  // MFMAs with the reads of step t+1 interleaved.
  auto step = [&](const Frags &cur, Frags &nxt, int64_t t, int buf) {
    const uint8_t *next = nullptr;
    if (t + 1 < nk) {
      if (t + 3 < nk) wait_vm<16>();
      else if (t + 2 < nk) wait_vm<8>();
      else wait_vm<0>();
      __builtin_amdgcn_s_barrier();
      if (t + 4 < nk) pipe_issue(SB[buf], ga, gb, 64 * (t + 4), wave);
      next = SB[(buf + 1) & 3];
    }
    mfma_step(cur, nxt, next, acc, wm, wn, lane);
    if (next) wait_lds(nxt);
  };
  for (int64_t t = 0; t < nk; t += 4) {
    step(F0, F1, t, 0);
    if (t + 1 < nk) step(F1, F0, t + 1, 1);
    if (t + 2 < nk) step(F0, F1, t + 2, 2);
    if (t + 3 < nk) step(F1, F0, t + 3, 3);
  }

  const bool vec = vec_stores_ok(y, n);
  float sx[4][4], sw[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) tile_row_scales(xs, m, m0 + 128 * wm + i * 32, lane, sx[i]);
#pragma unroll
  for (int j = 0; j < 4; ++j) tile_col_scales(ws, n, n0 + 128 * wn + j * 32, lane, sw[j]);
  if (ytype != RQ_F32 && vec && n % 8 == 0 && m0 + 256 <= m && n0 + 256 <= n) {
    __syncthreads();  // every wave's stage reads are done
    const float nob[4][4] = {};
    stage_block_2b<true>(acc, SM, 128 * wm, 128 * wn, ytype, sx, sw, nob, false, lane);
    __syncthreads();
    store_staged_2b(SM, y, n, m0, n0, threadIdx.x);
    return;
  }
  const Out o{y, nullptr, ytype, 0};
  const float nob[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  static_for<4>([&](auto I) {
    static_for<4>([&](auto J) {
      store_tile32<true>(acc[I][J], o, m, n, m0 + 128 * wm + I * 32, n0 + 128 * wn + J * 32, sx[I], sw[J], nob, xs,
                         ws, lane, vec);
    });
  });
}

// ---- the same with eight waves (two a SIMD) ------------------------------
//
// Eight waves of 128 (M) x 64 (N) on the 256 x 256 tile (4 x 2 MFMA tiles,
// 128 accumulators), two waves a SIMD: while one wave waits on its LDS reads
// or the step's barrier the other issues MFMAs (2048 x 14336 x 4096: 148-155
// -> 131-134 us against the four-wave kernel).  The four stages keep their A parts
// side by side (16 KB each) and their B parts side by side (64 KB above), so
// that one base register per operand and pass half reaches every stage and
// tile through the ds_read offset field; each wave fills 32 A rows and 32 B
// rows of a stage (two direct loads each), three steps ahead.
constexpr int F8_A = 16384, F8_B = 65536;

struct Frags8 {
  u32x4 x[12];  // A tiles 0..3 (halves 2t, 2t + 1), then B tiles 0..1 (8 + 2t, 9 + 2t)
};

__device__ __forceinline__ void wait_lds8(Frags8 &F) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(F.x[0]), "+v"(F.x[1]), "+v"(F.x[2]), "+v"(F.x[3]));
  asm volatile("" : "+v"(F.x[4]), "+v"(F.x[5]), "+v"(F.x[6]), "+v"(F.x[7]));
  asm volatile("" : "+v"(F.x[8]), "+v"(F.x[9]), "+v"(F.x[10]), "+v"(F.x[11]));
}

// Fragment f of stage ST (f < 8: A tile f / 2, else B tile (f - 8) / 2; half f % 2).
template <int ST, int F>
__device__ __forceinline__ u32x4 frag8(const uint32_t (&rd)[2][2]) {
  constexpr int t = F < 8 ? F / 2 : (F - 8) / 2;
  return ds_read16_off<ST * F8_A + 2048 * t>(rd[F & 1][F < 8 ? 0 : 1]);
}

__device__ __forceinline__ i32x8 frag8_op(const Frags8 &F, int f) {
  const u32x4 x0 = F.x[f], x1 = F.x[f + 1];
  return (i32x8){(int)x0.x, (int)x0.y, (int)x0.z, (int)x0.w, (int)x1.x, (int)x1.y, (int)x1.z, (int)x1.w};
}

// The 8 MFMAs of one K-step on `cur`; after MFMA f < 6, reads 2f and 2f + 1
// of the next step's fragments from stage ST.
template <int ST>
__device__ __forceinline__ void mfma_step8(const Frags8 &cur, Frags8 &nxt, const uint32_t (&rd)[2][2],
                                           f32x16 (&acc)[4][2]) {
  static_for<4>([&](auto I) {
    static_for<2>([&](auto J) {
      constexpr int f = 2 * decltype(I)::value + decltype(J)::value;
      acc[I][J] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(frag8_op(cur, 2 * I), frag8_op(cur, 8 + 2 * J),
                                                                  acc[I][J], 0, 0, 0, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (f < 6) {
        nxt.x[2 * f] = frag8<ST, 2 * f>(rd);
        nxt.x[2 * f + 1] = frag8<ST, 2 * f + 1>(rd);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  });
}

__global__ __launch_bounds__(512) void k_fp8_gemm_pipe8(const uint8_t *__restrict__ a,
                                                       const float *__restrict__ xs, int64_t m,
                                                       const uint8_t *__restrict__ b,
                                                       const float *__restrict__ ws, int64_t n,
                                                       int64_t k, void *__restrict__ y, int ytype) {
  __shared__ __attribute__((aligned(1024))) uint8_t SM[4 * P_STAGE];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 2, wn = wave & 3;
  const int64_t m0 = (int64_t)blockIdx.y * 256, n0 = (int64_t)blockIdx.x * 256;
  const int64_t nk = k / 64;

  // Wave w fills rows 32 w .. 32 w + 31 of the A and B parts of a stage, 16
  // rows (4 lanes x 16 bytes a row) an instruction, lane L at byte 16 L of
  // the instruction's kilobyte; rows past m or n re-read the last valid row.
  const uint8_t *ga[2], *gb[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = 32 * wave + 16 * j + (lane >> 2);
    const int gc = (lane & 3) ^ swz(r);
    const int64_t gm = m0 + r < m ? m0 + r : m - 1;
    const int64_t gn = n0 + r < n ? n0 + r : n - 1;
    ga[j] = a + gm * k + 16 * gc;
    gb[j] = b + gn * k + 16 * gc;
  }
  uint8_t *const dA = SM + 2048 * wave, *const dB = SM + F8_B + 2048 * wave;
  auto issue = [&](int st, int64_t k0) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      __builtin_amdgcn_global_load_lds(ga[j] + k0, (lds_void *)(dA + st * F8_A + 1024 * j), 16, 0, 0);
#pragma unroll
    for (int j = 0; j < 2; ++j)
      __builtin_amdgcn_global_load_lds(gb[j] + k0, (lds_void *)(dB + st * F8_A + 1024 * j), 16, 0, 0);
  };
  uint32_t rd[2][2];  // [half][A, B]
  {
    const uint32_t sa = lds_addr(SM), sb = sa + F8_B;
    const int l = lane & 31, g = lane >> 5, sw = (l >> 2) & 3;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      rd[h][0] = sa + 8192 * wm + 64 * l + 16 * ((2 * g + h) ^ sw);
      rd[h][1] = sb + 4096 * wn + 64 * l + 16 * ((2 * g + h) ^ sw);
    }
  }

  f32x16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (f32x16){0};

  // Stages 0..3 in flight; fragments of step 0 in registers.
#pragma unroll
  for (int s = 0; s < 4; ++s)
    if (s < nk) issue(s, 64 * s);
  if (nk > 3) wait_vm<12>();
  else if (nk > 2) wait_vm<8>();
  else if (nk > 1) wait_vm<4>();
  else wait_vm<0>();
  __builtin_amdgcn_s_barrier();
  Frags8 F0, F1;
  static_for<12>([&](auto Fc) { F0.x[decltype(Fc)::value] = frag8<0, decltype(Fc)::value>(rd); });
  wait_lds8(F0);

  // Step t (stage t % 4 in registers): make stage t + 1 resident (wait for its
  // loads, then a bare barrier), refill stage t % 4 with K-step t + 4 (every
  // wave has read it), then the MFMAs of step t with the reads of step t + 1.
  // The last step reads a stale stage (in bounds, never used), so that every
  // step has the same straight-line MFMA code (k % 256 == 0: whole groups of
  // four steps).
  auto step = [&](const Frags8 &cur, Frags8 &nxt, int64_t t, auto STc) {
    constexpr int ST = decltype(STc)::value;
    if (t + 3 < nk) wait_vm<8>();
    else if (t + 2 < nk) wait_vm<4>();
    else wait_vm<0>();
    __builtin_amdgcn_s_barrier();
    if (t + 4 < nk) issue(ST, 64 * (t + 4));
    mfma_step8<(ST + 1) & 3>(cur, nxt, rd, acc);
    wait_lds8(nxt);
  };
  for (int64_t t = 0; t < nk; t += 4) {
    step(F0, F1, t, std::integral_constant<int, 0>{});
    step(F1, F0, t + 1, std::integral_constant<int, 1>{});
    step(F0, F1, t + 2, std::integral_constant<int, 2>{});
    step(F1, F0, t + 3, std::integral_constant<int, 3>{});
  }

  const bool vec = vec_stores_ok(y, n);
  float sx[4][4], sw[2][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) tile_row_scales(xs, m, m0 + 128 * wm + i * 32, lane, sx[i]);
#pragma unroll
  for (int j = 0; j < 2; ++j) tile_col_scales(ws, n, n0 + 64 * wn + j * 32, lane, sw[j]);
  if (ytype != RQ_F32 && vec && n % 8 == 0 && m0 + 256 <= m && n0 + 256 <= n) {
    __syncthreads();  // every wave's stage reads are done
    const float nob[2][4] = {};
    stage_block_2b<true>(acc, SM, 128 * wm, 64 * wn, ytype, sx, sw, nob, false, lane);
    __syncthreads();
    store_staged_2b<512>(SM, y, n, m0, n0, tid);
    return;
  }
  const Out o{y, nullptr, ytype, 0};
  const float nob[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  static_for<4>([&](auto I) {
    static_for<2>([&](auto J) {
      store_tile32<true>(acc[I][J], o, m, n, m0 + 128 * wm + I * 32, n0 + 64 * wn + J * 32, sx[I], sw[J], nob, xs,
                         ws, lane, vec);
    });
  });
}

void launch_tiled(const uint8_t *xq, const float *xs, int64_t m, const uint8_t *w, const float *ws,
                  int64_t n, int64_t k, void *y, int ytype, hipStream_t s) {
  const dim3 grid((unsigned)((n + 127) / 128), (unsigned)((m + 127) / 128));
  hipLaunchKernelGGL((k_fp8_gemm_mfma<128, 128, 2, 2, 128>), grid, dim3(256), 0, s, xq, xs, m, w, ws, n, k, y, ytype);
}

template <int MT>
void launch_skinny(const uint8_t *xq, const float *xs, int64_t m, const uint8_t *w, const float *ws, int64_t n,
                   int64_t k, void *y, int ytype, hipStream_t s) {
  const int64_t tm = (m + 16 * MT - 1) / (16 * MT), wgs = tm * ((n + 31) / 32), steps = (k + 127) / 128;
  const int waves = (int)(steps < 8 ? steps : 8);
  const size_t lds = (size_t)waves * MT * 2048;  // at most 64 KB
#define RQ_SK(TAIL)                                                                                              \
  hipLaunchKernelGGL((k_fp8_skinny<MT, TAIL>), dim3((unsigned)wgs), dim3(64 * waves), lds, s, xq, xs, m, w, ws, n, k, y, \
                     ytype, (int)tm)
  if (k % 128 == 0) RQ_SK(false); else RQ_SK(true);
#undef RQ_SK
}

}  // namespace

int launch_fp8_quantize(const void *x, int xtype, int64_t m, int64_t k, int mode, uint8_t *xq,
                        float *xs, hipStream_t s) {
  if (m == 0) return RQ_OK;
  const bool f32x = xtype == RQ_F32;
  const int es = f32x ? 4 : 8;
  const bool vec = reinterpret_cast<uintptr_t>(x) % 16 == 0 && k % es == 0 && (k * (f32x ? 4 : 2)) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(xq) % es == 0;
  if (vec) {
    const bool sc = mode != RQ_FP8_UNSCALED;
    // Four waves a row unless one wave holds it in one chunk a lane (k = 4096,
    // f32: m = 5 4.3 -> 2.7 us, 512 4.8 -> 3.3, 2048 7.8 -> 6.9 against one wave
    // a row).
    const bool wide = k / es > 64;
    const dim3 grid((unsigned)(wide ? m : (m + 3) / 4));
#define RQ_QW(XT, SC)                                                                                                \
  if (wide) hipLaunchKernelGGL((k_fp8_quant_waves<XT, SC, 4>), grid, dim3(256), 0, s, x, m, k, xq, xs);              \
  else hipLaunchKernelGGL((k_fp8_quant_waves<XT, SC, 1>), grid, dim3(256), 0, s, x, m, k, xq, xs)
    if (xtype == RQ_F32) {
      if (sc) { RQ_QW(RQ_F32, true); } else { RQ_QW(RQ_F32, false); }
    } else if (xtype == RQ_BF16) {
      if (sc) { RQ_QW(RQ_BF16, true); } else { RQ_QW(RQ_BF16, false); }
    } else {
      if (sc) { RQ_QW(RQ_F16, true); } else { RQ_QW(RQ_F16, false); }
    }
#undef RQ_QW
  } else {
    hipLaunchKernelGGL(k_fp8_quant_rows, dim3((unsigned)m), dim3(256), 0, s, x, xtype, k, mode, xq, xs);
  }
  return hipGetLastError() == hipSuccess ? RQ_OK : set_error(RQ_E_DEVICE, "fp8 quantize launch failed");
}

int launch_fp8_gemm(const uint8_t *xq, const float *xs, int64_t m, const uint8_t *w,
                    const float *ws, int64_t n, int64_t k, void *y, int ytype, hipStream_t s) {
  if (m == 0 || n == 0) return RQ_OK;
  const bool aligned = (reinterpret_cast<uintptr_t>(xq) % 16 == 0) &&
                       (reinterpret_cast<uintptr_t>(w) % 16 == 0);
  // 16 MT x 32 tiles with K split over a workgroup's waves where the 128 x 128
  // tiles would leave CUs idle: up to 512 workgroups of 64 x 32 (at k = 4096 512
  // x 2048 26.9 against 29.9 us and 64 x 14336 31.2 against 30.8; 128 x 14336
  // 48.4 against 32.6), all of at most 32 rows (24 x 14336 17.8 against 33.4),
  // and every k that is not a multiple of 128.
  const int64_t sk_wgs = ((m + 63) / 64) * ((n + 31) / 32);
  const bool sk_ok = k % 16 == 0 && k <= (1 << 24) && sk_wgs <= 0x3FFFFFFF;
  if (aligned && k % 128 == 0 && !(sk_ok && (m <= 32 || sk_wgs <= 512))) {
    // 256 x 256 tiles when there are enough of them to cover the CUs (eight
    // waves of 128 x 64 for whole groups of four K-steps, else four of
    // 128 x 128), else 128 x 128.
    const int64_t big = ((m + 255) / 256) * ((n + 255) / 256);
    if (big >= 200) {
      const dim3 grid((unsigned)((n + 255) / 256), (unsigned)((m + 255) / 256));
      if (k % 256 == 0)
        hipLaunchKernelGGL(k_fp8_gemm_pipe8, grid, dim3(512), 0, s, xq, xs, m, w, ws, n, k, y, ytype);
      else
        hipLaunchKernelGGL(k_fp8_gemm_pipe, grid, dim3(256), 0, s, xq, xs, m, w, ws, n, k, y, ytype);
    } else {
      launch_tiled(xq, xs, m, w, ws, n, k, y, ytype, s);
    }
  } else if (aligned && sk_ok) {
    if (m <= 16) launch_skinny<1>(xq, xs, m, w, ws, n, k, y, ytype, s);
    else if (m <= 32) launch_skinny<2>(xq, xs, m, w, ws, n, k, y, ytype, s);
    else launch_skinny<4>(xq, xs, m, w, ws, n, k, y, ytype, s);
  } else {
    const int64_t total = m * n;
    hipLaunchKernelGGL(k_fp8_gemm_scalar, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, xq,
                       xs, m, w, ws, n, k, y, ytype);
  }
  return hipGetLastError() == hipSuccess ? RQ_OK : set_error(RQ_E_DEVICE, "fp8 gemm launch failed");
}

}  // namespace rq
