// Small-batch fp32 linear layers of the inference step: out = x W^T (+ bias),
// with the elementwise work around each of them folded in (engine/mamba.py
// step, :440-498, and the pre-norm residual loop of Mamba.step, :592-597):
//   kLinNorm   x is RMS-normalised on the way in (:82-89): the product runs
//              on x w and each row is scaled by rsqrt(mean(x^2) + eps) at the
//              end (the sum of squares rides along with the loads of x);
//   kLinSilu   the first nsilu outputs go through SiLU (the in_proj's
//              x branch);
//   kLinAdd    out = add + x W^T (the residual add after out_proj).
//
// Bound: at these batches (1 to a few hundred rows) a layer's projections are
// latency: W is read once from the last-level cache (6.6 MB of weights per
// layer at d_model 512) and the launches around them dominate.  So: one
// workgroup per 16 output columns and up to 64 rows, its waves splitting K in
// slices of 16 (kLinWaves slices at a time: every load of a wave is in flight
// before its first use), products on v_mfma_f32_16x16x4_f32 (fp32 inputs and
// accumulation: each product rounds once, as an FMA does), the waves' partial
// tiles summed in wave order through LDS.  A lane loads 16 bytes of a W row
// and of an x row: the four k of a float4 go to four MFMAs, so both operands
// use the same k order and no shuffle is needed.
//
// Measured at d_model 512 (in_proj 2048 x 512, x_proj 112 x 1024, dt_proj
// 1024 x 32, out_proj 512 x 1024): 5.4 / 6.0 / 3.0 / 5.3 us at 12 rows, 7.7 /
// 6.5 / 3.2 / 5.8 at 64 (11-12 each for the wide ones when 64 rows shared a
// workgroup), where the library's GEMMs took 7 us each, the norm 6.6 and the
// SiLU 3.8 in launches of their own: a layer 50 -> 33 us at 12 rows.

#include "rp_device.h"
#include "rp_launch.h"

namespace rp {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// RT: 16-row tiles per workgroup; MODE: bits of LinMode.
template <int RT, int MODE>
__global__ __launch_bounds__(kLinWaves* kWave) void linear_rows_kernel(LinearParams p) {
  constexpr bool NORM = MODE & kLinNorm;
  constexpr int OUTS = RT * 256;  // outputs of the workgroup (16 columns x 16 RT rows)
  __shared__ __align__(16) float sPart[kLinWaves][OUTS];
  __shared__ float sSq[NORM ? kLinWaves : 1][NORM ? RT * 16 : 1];
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  const int g = lane / 16, i = lane % 16;
  const int n0 = blockIdx.x * 16, r0 = blockIdx.y * (16 * RT);
  // rows beyond the matrices read the last one; their outputs are not stored
  const float* wrow = p.w + (int64_t)min(n0 + i, p.N - 1) * p.K;
  const float* xrow[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) xrow[t] = p.x + (int64_t)min(r0 + t * 16 + i, p.R - 1) * p.xsr;
  f32x4 acc[RT];
  float sq[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    sq[t] = 0.f;
  }
  // U slices of 16 k per turn, all loaded before the first is used; a slice
  // beyond K stays zero (the last one may be partial: K is a multiple of 4,
  // so a lane's float4 is inside or outside as a whole)
  constexpr int U = RT == 4 ? 2 : 4;
  const int nslice = (p.K + 15) / 16;
  for (int c0 = wave; c0 < nslice; c0 += U * kLinWaves) {
    f32x4 wv[U], nv[U], xv[U][RT];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int k = (c0 + j * kLinWaves) * 16 + g * 4;
      wv[j] = nv[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < RT; ++t) xv[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (k < p.K) {
        wv[j] = *reinterpret_cast<const f32x4*>(wrow + k);
        if constexpr (NORM) nv[j] = *reinterpret_cast<const f32x4*>(p.norm_w + k);
#pragma unroll
        for (int t = 0; t < RT; ++t) xv[j][t] = *reinterpret_cast<const f32x4*>(xrow[t] + k);
      }
    }
#pragma unroll
    for (int j = 0; j < U; ++j) {
#pragma unroll
      for (int t = 0; t < RT; ++t) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float xe = xv[j][t][e];
          if constexpr (NORM) {
            sq[t] = ffma(xe, xe, sq[t]);
            xe = fmul(xe, nv[j][e]);
          }
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[j][e], xe, acc[t], 0, 0, 0);
        }
      }
    }
  }
  // lane (g, i) holds outputs of columns n0 + 4 g + 0..3, row i of each tile
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    *reinterpret_cast<f32x4*>(&sPart[wave][t * 256 + lane * 4]) = acc[t];
    if constexpr (NORM) {
      float s = sq[t];
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      if (g == 0) sSq[wave][t * 16 + i] = s;
    }
  }
  __syncthreads();
  for (int o = tid; o < OUTS; o += kLinWaves * kWave) {
    const int t = o / 256, n = o % 16, r = o / 16 % 16;
    const int at = t * 256 + (n / 4) * 64 + r * 4 + n % 4;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < kLinWaves; ++w) v += sPart[w][at];
    if constexpr (NORM) {
      float s = 0.f;
#pragma unroll
      for (int w = 0; w < kLinWaves; ++w) s += sSq[w][t * 16 + r];
      v = fmul(v, rsqrtf(s * (1.f / (float)p.K) + p.eps));
    }
    const int row = r0 + t * 16 + r, col = n0 + n;
    if (row < p.R && col < p.N) {
      if (p.bias != nullptr) v += p.bias[col];
      if constexpr ((MODE & kLinSilu) != 0) {
        if (col < p.nsilu) v = v / (1.f + expf(-v));
      }
      if constexpr ((MODE & kLinAdd) != 0) v = p.add[(int64_t)row * p.asr + col] + v;
      p.out[(int64_t)row * p.osr + col] = v;
    }
  }
}

template <int MODE>
static hipError_t launch_linear_m(const LinearParams& p, hipStream_t st) {
  const int ctiles = (p.N + 15) / 16;
  auto rtiles = [&](int rt) { return (p.R + 16 * rt - 1) / (16 * rt); };
  // rows per workgroup: the fewest W reads that still leave a workgroup per CU
  int rt = 4;
  while (rt > 1 && ctiles * rtiles(rt) < 256) rt /= 2;
  const dim3 grid((unsigned)ctiles, (unsigned)rtiles(rt));
  const dim3 block(kLinWaves * kWave);
  if (rt == 1)
    hipLaunchKernelGGL((linear_rows_kernel<1, MODE>), grid, block, 0, st, p);
  else if (rt == 2)
    hipLaunchKernelGGL((linear_rows_kernel<2, MODE>), grid, block, 0, st, p);
  else
    hipLaunchKernelGGL((linear_rows_kernel<4, MODE>), grid, block, 0, st, p);
  return hipGetLastError();
}

hipError_t launch_linear(const LinearParams& p, int mode, hipStream_t st) {
  if (p.R == 0 || p.N == 0) return hipSuccess;
  switch (mode) {
    case 0: return launch_linear_m<0>(p, st);
    case kLinNorm | kLinSilu: return launch_linear_m<kLinNorm | kLinSilu>(p, st);
    case kLinAdd: return launch_linear_m<kLinAdd>(p, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace rp
