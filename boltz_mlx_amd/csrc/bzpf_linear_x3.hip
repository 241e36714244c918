// fp32 Linear over few rows (the s track's N rows) on split operands (bzpf_x3.h):
//   y[r][m] (epilogues 0 .. 3 of launch_gemm_nt) = x[r] . W[m] + bias[m], x [R][K], W [M][K], K a multiple of 32
// (boltz_mlx/layers/attentionv2.py:50-86, transition.py:27-54 at 384 channels).
// A row count of some hundreds leaves a 64 x 64-tile GEMM with a dozen workgroups walking K one stage after another. Here
// a workgroup takes 16 columns of W against 16 RB rows, and its 8 waves an eighth of K each: steps of 32 k, wave, wave + 8,
// ..., their operands straight from the caches and split in registers, the next step's loads in flight. The waves' sums
// are added over LDS in wave order, so an output's sum depends on K alone. 128 rows, K = 1536 -> 384: 31.1 -> 10.3 us, error
// against 64 bits 7.0e-7 -> 2.1e-7; K = 384 -> 1536 10.0 -> 6.5 us, 3.5e-7 -> 1.0e-7.
#include "bzpf_common.h"
#include "bzpf_kernels.h"
#include "bzpf_rowgemm_x3.h"

namespace bzpf {

namespace {

constexpr int LXW = 8;

template <int RB, typename TY>
__global__ __launch_bounds__(64 * LXW) void linear_x3_small_k(const float* __restrict__ x, const float* __restrict__ w,
                                                              const float* __restrict__ bias, TY* __restrict__ y,
                                                              int64_t R, int K, int M, int epi,
                                                              const float* __restrict__ gate, int64_t ld_gate,
                                                              int64_t gate_rows) {
  constexpr int ROWS = 16 * RB;
  __shared__ LDS_ALIGN float Part[LXW][ROWS][20];
  const int t = threadIdx.x, l = t & 63, g = l >> 4, r = l & 15;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int m0 = 16 * (int)blockIdx.x;
  const int64_t r0 = (int64_t)blockIdx.y * ROWS;
  const int steps = K / 32;
  const float* wp = w + (int64_t)min(m0 + r, M - 1) * K + 8 * g;
  const float* xp[RB];
#pragma unroll
  for (int rb = 0; rb < RB; rb++) xp[rb] = x + min(r0 + 16 * rb + r, R - 1) * K + 8 * g;
  f4 wr[2], xr[RB][2];
  const auto load = [&](int st) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      wr[h] = ld4(wp + 32 * st + 4 * h);
#pragma unroll
      for (int rb = 0; rb < RB; rb++) xr[rb][h] = ld4(xp[rb] + 32 * st + 4 * h);
    }
  };
  load(min(wave, steps - 1));
  f4 acc[RB] = {};
  for (int st = wave; st < steps; st += LXW) {
    bf16x8 wf[3], xf[RB][3];
    split8(wr[0], wr[1], wf[0], wf[1], wf[2]);
#pragma unroll
    for (int rb = 0; rb < RB; rb++) split8(xr[rb][0], xr[rb][1], xf[rb][0], xf[rb][1], xf[rb][2]);
    load(min(st + LXW, steps - 1));
#pragma unroll
    for (int q = 0; q < 6; q++)
#pragma unroll
      for (int rb = 0; rb < RB; rb++) acc[rb] = mfma_x3<false>(wf[X3_W[q]], xf[rb][X3_X[q]], acc[rb]);
  }
  if (wave_nonfinite(acc)) {  // (bzpf_rowgemm_x3.h)
#pragma unroll
    for (int rb = 0; rb < RB; rb++) acc[rb] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int st = 2 * wave; st < 2 * steps; st += (st & 1) ? 2 * LXW - 1 : 1) {  // halves 2 st, 2 st + 1 of a step
      const f4 wv = ld4(wp + 32 * (st >> 1) + 4 * (st & 1));
#pragma unroll
      for (int rb = 0; rb < RB; rb++) {
        const f4 xv = ld4(xp[rb] + 32 * (st >> 1) + 4 * (st & 1));
#pragma unroll
        for (int e = 0; e < 4; e++) acc[rb] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[e], xv[e], acc[rb], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int rb = 0; rb < RB; rb++) st4(&Part[wave][16 * rb + r][4 * g], acc[rb]);
  __syncthreads();
  // 4 outputs a thread: row t / 4, columns 4 (t % 4) .. + 3
  if (t >= 4 * ROWS) return;
  const int lr = t >> 2, m = m0 + 4 * (t & 3);
  const int64_t row = r0 + lr;
  if (row >= R || m >= M) return;  // M is a multiple of 4
  f4 v = ld4(&Part[0][lr][4 * (t & 3)]);
#pragma unroll
  for (int p = 1; p < LXW; p++) v = v + ld4(&Part[p][lr][4 * (t & 3)]);
  if (bias != nullptr) v += ld4(bias + m);
  TY* yp = y + row * M + m;
  if constexpr (sizeof(TY) == 4) {
    if (epi == 2) {
      const f4 gv = ld4(gate + (row % gate_rows) * ld_gate + m);
      v = f4{v[0] * sigmoidf_(gv[0]), v[1] * sigmoidf_(gv[1]), v[2] * sigmoidf_(gv[2]), v[3] * sigmoidf_(gv[3])};
    }
    if (epi >= 1) v += epi == 3 ? ld4(gate + row * ld_gate + m) : ld4(yp);
  }
  st4(yp, v);
}

template <int RB>
hipError_t run(const float* x, const float* w, const float* bias, void* y, int y_dt, int64_t R, int K, int M, int epi,
               const float* gate, int64_t ld_gate, int64_t gate_rows, hipStream_t st) {
  const dim3 grid((unsigned)((M + 15) / 16), (unsigned)((R + 16 * RB - 1) / (16 * RB)));
  if (y_dt == DT_F16)
    linear_x3_small_k<RB, half_t><<<grid, 64 * LXW, 0, st>>>(x, w, bias, static_cast<half_t*>(y), R, K, M, epi, gate,
                                                             ld_gate, gate_rows);
  else
    linear_x3_small_k<RB, float><<<grid, 64 * LXW, 0, st>>>(x, w, bias, static_cast<float*>(y), R, K, M, epi, gate,
                                                            ld_gate, gate_rows);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_linear_x3_small(const float* x, const float* w, const float* bias, void* y, int y_dt, int64_t R, int K,
                                  int M, int epi, const float* gate, int64_t ld_gate, int64_t gate_rows,
                                  hipStream_t st) {
  if (R < 1 || R > 65535 * 16 || K < 32 || K % 32 || M < 4 || M % 4) return hipErrorInvalidValue;
  return R <= 16 ? run<1>(x, w, bias, y, y_dt, R, K, M, epi, gate, ld_gate, gate_rows, st)
                 : run<2>(x, w, bias, y, y_dt, R, K, M, epi, gate, ld_gate, gate_rows, st);
}

}  // namespace bzpf
