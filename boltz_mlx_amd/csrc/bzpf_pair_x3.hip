// The fp32 row kernels of the pair track on the bf16 matrix cores (split operands: bzpf_rowgemm_x3.h). Same operations
// and buffers as the fp16 forms in bzpf_pair_gemm.hip:
//   trimul_proj, trimul_tail  (boltz_mlx/layers/triangular_mult.py:67-118, 143-170);
//   triattn_proj              (triangular_attention/attention.py:49-69, 100-104);
//   linear_resid_ln           (kernels_nax3.py:176-198);
//   transition                (transition.py:27-54, 148-154).
// The fp32 matrix instructions these ran on (v_mfma_f32_16x16x4_f32) take 2.7 times the six part products' time, and a
// short input was bound by one workgroup's chain of staging and tiles. us at N = 29 / 128 / 400 / 513 (launches of one kernel
// in a graph, fp32 MFMA form -> this one):
//   trimul_proj      42 / 46 / 224 / 363  ->  14 / 21 / 114 / 195   (0.207 TFLOP of part products at N = 513: 1.06 PFLOP/s)
//   trimul_tail      22 / 27 / 218 / 362  ->  14 / 19 / 124 / 196   (675 MB at N = 513: 3.4 TB/s)
//   triattn_proj     63 / 70 / 236 / 395  ->  15 / 23 / 152 / 241   (675 MB at N = 513: 2.8 TB/s)
//   linear_resid_ln  12 / 15 /  74 / 122  ->  14 / 17 /  68 / 119   (540 MB at N = 513: 4.5 TB/s)
//     transposed     13 / 15 /  82 / 136  ->  14 / 17 /  76 / 133
//   transition       84 / 88 / 573 / 962  ->  27 / 64 / 315 / 527   (1.18 PFLOP/s of part products)
// Sums that come out not finite are formed again on the fp32 instructions (wave_nonfinite, bzpf_rowgemm_x3.h).
#include <algorithm>
#include <type_traits>

#include "bzpf_common.h"
#include "bzpf_kernels.h"
#include "bzpf_rowgemm_x3.h"

namespace bzpf {

namespace {

constexpr int XW = 8, XT = 64 * XW;  // waves and threads of the persistent workgroups (2 per SIMD: 256 VGPRs)
constexpr int XTW = 32;              // positions of a wave tile: two row blocks of 16

// ---------------------------------------------------------------- triangle multiplication projection
// A workgroup holds 64 projection and their 64 gate rows (104 KB of LDS at KIN = 128; all 256 + 256 rows in three parts
// would take 418 KB) and streams tiles of 32 positions (i, k0 .. k0 + 31) of the padded rows; the 2 KIN / 64 groups of
// channels read the same x rows.
template <int KIN>
__global__ __launch_bounds__(XT) void trimul_proj_x3_k(const float* __restrict__ xn, const float* __restrict__ w,
                                                       const float* __restrict__ mask, float scale, int incoming,
                                                       float* __restrict__ ab, int64_t N, int64_t ld) {
  constexpr int NG = 2 * KIN / 64, PLANE_W = 128 * ldx<KIN>();
  __shared__ LDS_ALIGN __bf16 Ws[3 * PLANE_W];
  int grp, wg;
  weight_group<NG>(grp, wg);
  const int nwg = (int)gridDim.x / NG, c_lo = 64 * grp;
  const int tpr = (int)(ld / XTW), ntiles = (int)N * tpr, stride = nwg * XW;
  if (wg * XW >= ntiles) return;  // whole workgroup
  const int l = threadIdx.x & 63, g = l >> 4, r = l & 15;
  int t = __builtin_amdgcn_readfirstlane(wg * XW + (int)(threadIdx.x >> 6));
  RawRow<KIN> raw[2];
  float mk[2];
  const auto position = [&](int i, int64_t k) {  // of the xn row of output position (i, k)
    const int64_t kc = k < N ? k : N - 1;
    return incoming ? kc * N + i : (int64_t)i * N + kc;
  };
  const auto load = [&](int tt) {
    const int i = tt / tpr, k0 = (tt - i * tpr) * XTW;
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
      const int64_t src = position(i, k0 + 16 * rb + r);
      raw[rb].load(xn + src * KIN, g);
      mk[rb] = mask[src];
    }
  };
  load(min(t, ntiles - 1));
  stage_x3<128, KIN, XT>(Ws, PLANE_W,
                         [&](int rr) { return w + (int64_t)(rr < 64 ? c_lo + rr : 2 * KIN + c_lo + rr - 64) * KIN; });
  __syncthreads();
  for (; t < ntiles; t += stride) {
    const int i = t / tpr, k0 = (t - i * tpr) * XTW;
    X3Row<KIN> x[2];
    float mo[2][4];  // mask of output positions 16 rb + 4 g + e, from lane 4 g + e
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
      split_row(x[rb], raw[rb]);
      const float mv = k0 + 16 * rb + r < N ? mk[rb] * scale : 0.0f;
#pragma unroll
      for (int e = 0; e < 4; e++) mo[rb][e] = __shfl(mv, 4 * g + e);
    }
    load(min(t + stride, ntiles - 1));
    float* dst = ab + ((int64_t)(c_lo + r) * N + i) * ld + k0 + 4 * g;
#pragma unroll 1
    for (int cb = 0; cb < 4; cb++) {
      f4 pa[2] = {}, ga[2] = {};
      mma_x3<2, true, KIN>(pa, x, Ws + 16 * cb * ldx<KIN>(), PLANE_W);
      mma_x3<2, true, KIN>(ga, x, Ws + (64 + 16 * cb) * ldx<KIN>(), PLANE_W);
      const f4 all[4] = {pa[0], pa[1], ga[0], ga[1]};
      if (wave_nonfinite(all)) {
        const float* xr[2];
#pragma unroll
        for (int rb = 0; rb < 2; rb++) xr[rb] = xn + position(i, k0 + 16 * rb + r) * KIN;
        const float* wr = w + (int64_t)(c_lo + 16 * cb + r) * KIN;
        mma_f32<2, true, KIN>(pa, wr, xr);
        mma_f32<2, true, KIN>(ga, wr + (int64_t)2 * KIN * KIN, xr);
      }
#pragma unroll
      for (int rb = 0; rb < 2; rb++) {
        f4 v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = pa[rb][e] * sigmoidf_(ga[rb][e]) * mo[rb][e];
        st4(dst + (int64_t)16 * cb * N * ld + 16 * rb, v);
      }
    }
  }
}

// ---------------------------------------------------------------- triangle attention projection
// Four groups of weight rows: q, k, v and g with the bias block (16 rows, H of them used); rows of q, k and g permuted
// per 32 as in the fp16 form, so a lane holds 8 consecutive channels of its position.
template <int KIN>
__global__ __launch_bounds__(XT) void triattn_proj_x3_k(const float* __restrict__ xn, const float* __restrict__ w,
                                                        int trans, float q_scale, float b_scale,
                                                        float* __restrict__ qkg, float* __restrict__ vt,
                                                        float* __restrict__ tb, int64_t N, int64_t ldk, int H, int C) {
  constexpr int HC = 128, PLANE_W = (HC + 16) * ldx<KIN>();
  __shared__ LDS_ALIGN __bf16 Ws[3 * PLANE_W];
  int grp, wg;
  weight_group<4>(grp, wg);
  const int tpr = (int)(ldk / XTW), ntiles = (int)N * tpr, stride = (int)(gridDim.x / 4) * XW;
  if (wg * XW >= ntiles) return;  // whole workgroup
  const int l = threadIdx.x & 63, g = l >> 4, r = l & 15;
  int t = __builtin_amdgcn_readfirstlane(wg * XW + (int)(threadIdx.x >> 6));
  const int64_t NN = N * N;
  RawRow<KIN> raw[2];
  const auto xrow = [&](int i, int64_t j) {
    const int64_t jc = j < N ? j : N - 1;
    return xn + (trans ? jc * N + i : (int64_t)i * N + jc) * KIN;
  };
  const auto load = [&](int tt) {
    const int i = tt / tpr, j0 = (tt - i * tpr) * XTW;
#pragma unroll
    for (int rb = 0; rb < 2; rb++) raw[rb].load(xrow(i, j0 + 16 * rb + r), g);
  };
  load(min(t, ntiles - 1));
  const float* wg0 = w + (int64_t)grp * HC * KIN;
  const auto wrow = [&](int rr) -> const float* {
    if (rr >= HC) return rr - HC < H ? w + (int64_t)(4 * HC + rr - HC) * KIN : nullptr;
    if (grp == 2) return wg0 + rr * KIN;
    const int q = rr & 31, q16 = q & 15;
    return wg0 + ((rr & ~31) + 8 * (q16 >> 2) + 4 * (q >> 4) + (q16 & 3)) * KIN;
  };
  if (grp == 3) stage_x3<HC + 16, KIN, XT>(Ws, PLANE_W, wrow);
  else stage_x3<HC, KIN, XT>(Ws, PLANE_W, wrow);
  __syncthreads();
  for (; t < ntiles; t += stride) {
    const int i = t / tpr, j0 = (t - i * tpr) * XTW;
    X3Row<KIN> x[2];
#pragma unroll
    for (int rb = 0; rb < 2; rb++) split_row(x[rb], raw[rb]);
    load(min(t + stride, ntiles - 1));
    // a block again in fp32 (sums that are not finite): LDS weight rows rr0 .. rr0 + 15
    const auto again = [&](auto rows, f4 (&acc)[2], int rr0) {
      if (!wave_nonfinite(acc)) return;
      const float* wr = wrow(rr0 + r);
      const float* const xr[2] = {xrow(i, j0 + r), xrow(i, j0 + 16 + r)};
      mma_f32<2, decltype(rows)::value, KIN>(acc, wr != nullptr ? wr : w, xr);  // (no row: a bias row that is not stored)
    };
    // ROWS orientation: key j0 + 16 rb + 4 g + e is inside the row
    const auto valid = [&](int rb, int e) { return j0 + 16 * rb + 4 * g + e < N ? 1.0f : 0.0f; };
    if (grp == 2) {
#pragma unroll 1
      for (int cb = 0; cb < 8; cb++) {
        f4 acc[2] = {};
        mma_x3<2, true, KIN>(acc, x, Ws + 16 * cb * ldx<KIN>(), PLANE_W);
        again(std::true_type(), acc, 16 * cb);
        const int ch = 16 * cb + r, h = ch / C, d = ch - h * C;
        float* vp = vt + (((int64_t)h * N + i) * C + d) * ldk + j0 + 4 * g;
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
          __builtin_nontemporal_store(f4{acc[rb][0] * valid(rb, 0), acc[rb][1] * valid(rb, 1),
                                         acc[rb][2] * valid(rb, 2), acc[rb][3] * valid(rb, 3)},
                                      reinterpret_cast<f4*>(vp + 16 * rb));
      }
      continue;
    }
    const float sc = grp == 0 ? q_scale : 1.0f;
#pragma unroll 1
    for (int m = 0; m < 4; m++) {
      f4 a0[2] = {}, a1[2] = {};
      mma_x3<2, false, KIN>(a0, x, Ws + 32 * m * ldx<KIN>(), PLANE_W);
      mma_x3<2, false, KIN>(a1, x, Ws + (32 * m + 16) * ldx<KIN>(), PLANE_W);
      again(std::false_type(), a0, 32 * m);
      again(std::false_type(), a1, 32 * m + 16);
      const int within = 32 * m + 8 * g, h = within / C, d = within - h * C;
      const int64_t plane = (int64_t)(grp == 3 ? 2 : grp) * H + h;
#pragma unroll
      for (int rb = 0; rb < 2; rb++) {
        const int64_t j = j0 + 16 * rb + r;
        if (j >= N) continue;
        float* p = qkg + (plane * NN + (int64_t)i * N + j) * C + d;
        st4(p, a0[rb] * sc);
        st4(p + 4, a1[rb] * sc);
      }
    }
    if (grp == 3) {
      f4 acc[2] = {};
      mma_x3<2, true, KIN>(acc, x, Ws + HC * ldx<KIN>(), PLANE_W);
      again(std::true_type(), acc, HC);
      if (r < H) {
#pragma unroll
        for (int rb = 0; rb < 2; rb++) {
          const f4 v = acc[rb] * b_scale;
          st4(tb + tb_offset(r, i, j0 + 16 * rb + 4 * g, N, ldk),
              f4{v[0] * valid(rb, 0), v[1] * valid(rb, 1), v[2] * valid(rb, 2), v[3] * valid(rb, 3)});
        }
      }
    }
  }
}

// ---------------------------------------------------------------- triangle multiplication tail
// Tiles of 64 positions (i, j0 .. j0 + 63), 4 waves of 16 positions; the weights stream through LDS in chunks of 32 rows
// (p_out, then g_out), two chunks deep: a chunk's values are loaded while its predecessor computes, split and written
// to the other buffer. The o tile meets its transpose in the LDS the chunks take afterwards (52 KB in all, three
// workgroups per CU, whose barriers are independent).
template <int KIN>
__global__ __launch_bounds__(256, 3) void trimul_tail_x3_k(const float* __restrict__ o, const float* __restrict__ now,
                                                           const float* __restrict__ nob, float eps_out,
                                                           const float* __restrict__ w_po, const float* __restrict__ xn,
                                                           const float* __restrict__ w_go, float* __restrict__ z,
                                                           int accumulate, const float* __restrict__ lnw,
                                                           const float* __restrict__ lnb, float eps_next,
                                                           float* __restrict__ xn_next, int64_t N, int tpr, int64_t ld) {
  constexpr int D = KIN, CB = D / 16, NCH = D / 32, PLANE_W = 32 * ldx<D>(), LDT = D + 4;
  constexpr int WBYTES = 2 * 3 * PLANE_W * 2, TBYTES = 64 * LDT * 4;
  __shared__ LDS_ALIGN char lds[WBYTES > TBYTES ? WBYTES : TBYTES];
  float* Ts = reinterpret_cast<float*>(lds);
  const int i = (int)blockIdx.x / tpr, j0 = ((int)blockIdx.x - i * tpr) * 64;
  const int t = threadIdx.x, wave = t >> 6, l = t & 63, g = l >> 4, r = l & 15;
  const int64_t jp = j0 + 16 * wave + r, zr = jp < N ? (int64_t)i * N + jp : -1;
  const auto zrow = [&](int) { return zr; };
  const auto xrow = [&]() { return xn + ((int64_t)i * N + (jp < N ? jp : N - 1)) * D; };
  // o block of this thread: 4 channels 4 cq .. + 3, positions 4 (4 u + t % 4) .. + 3
  constexpr int UN = D / 64;  // (D / 4) x 16 blocks of the tile on 256 threads
#pragma unroll
  for (int u = 0; u < UN; u++) {
    const int e = u * 256 + t, pq = (e & 3) + 4 * (e / (4 * (D / 4))), cq = (e >> 2) % (D / 4);
    f4 v[4];
#pragma unroll
    for (int c = 0; c < 4; c++) v[c] = ld4(o + ((int64_t)(4 * cq + c) * N + i) * ld + j0 + 4 * pq);
#pragma unroll
    for (int p = 0; p < 4; p++)
      *reinterpret_cast<f4*>(Ts + (4 * pq + p) * LDT + 4 * cq) = f4{v[0][p], v[1][p], v[2][p], v[3][p]};
  }
  // chunk q: rows 32 (q % NCH) of p_out (q < NCH) or g_out; item e: row e / (D / 8), 8 channels
  constexpr int WI = 32 * D / 8 / 256;
  f4 pre[WI][2];
  const auto wload = [&](int q) {
    const float* src = (q < NCH ? w_po : w_go) + (int64_t)(q % NCH) * 32 * D;
#pragma unroll
    for (int v = 0; v < WI; v++) {
      pre[v][0] = ld4(src + (v * 256 + t) * 8);
      pre[v][1] = ld4(src + (v * 256 + t) * 8 + 4);
    }
  };
  const auto wstore = [&](int buf) {
    __bf16* W = reinterpret_cast<__bf16*>(lds) + buf * 3 * PLANE_W;
#pragma unroll
    for (int v = 0; v < WI; v++) {
      const int e = v * 256 + t;
      bf16x8 p0, p1, p2;
      split8(pre[v][0], pre[v][1], p0, p1, p2);
      __bf16* d = W + e / (D / 8) * ldx<D>() + e % (D / 8) * 8;
      *reinterpret_cast<bf16x8*>(d) = p0;
      *reinterpret_cast<bf16x8*>(d + PLANE_W) = p1;
      *reinterpret_cast<bf16x8*>(d + 2 * PLANE_W) = p2;
    }
  };
  wload(0);
  __syncthreads();
  // LN_out of this lane's position, channels D / 4 g .. + D / 4 - 1 (the rest in lanes l ^ 16, l ^ 32, l ^ 48)
  RawRow<D> of;
  of.load(Ts + (16 * wave + r) * LDT, g);
  const auto ln_out = [&]() {
    float sum = 0.f, ss = 0.f;
#pragma unroll
    for (int j = 0; j < D / 16; j++) sum += of.v[j][0] + of.v[j][1] + of.v[j][2] + of.v[j][3];
    const float mean = xgroups_sum(sum) * (1.0f / D);
#pragma unroll
    for (int j = 0; j < D / 16; j++) {
      of.v[j] = of.v[j] - mean;
      ss += of.v[j][0] * of.v[j][0] + of.v[j][1] * of.v[j][1] + of.v[j][2] * of.v[j][2] + of.v[j][3] * of.v[j][3];
    }
    const float rstd = 1.0f / sqrtf(xgroups_sum(ss) * (1.0f / D) + eps_out);
#pragma unroll
    for (int j = 0; j < D / 16; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int c = D / 4 * g + 4 * j + e;
        of.v[j][e] = of.v[j][e] * rstd * now[c] + nob[c];
      }
  };
  ln_out();
  __syncthreads();  // every wave has read its o rows: the chunks take the LDS
  wstore(0);
  wload(1);
  X3Row<D> x[1];
  split_row(x[0], of);
  f4 y[1][CB];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 2 * NCH; q++) {
    const __bf16* W = reinterpret_cast<const __bf16*>(lds) + (q & 1) * 3 * PLANE_W;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int cb = 2 * (q % NCH) + h;
      f4 acc[1] = {};
      mma_x3<1, false, D>(acc, x, W + 16 * h * ldx<D>(), PLANE_W);
      if (q >= NCH && wave_nonfinite(acc)) {
        const float* const xr[1] = {xrow()};
        mma_f32<1, false, D>(acc, opaque_ptr(w_go) + (16 * cb + r) * D, xr);
      }
#pragma unroll
      for (int e = 0; e < 4; e++) {
        if (q < NCH) y[0][cb][e] = acc[0][e];
        else y[0][cb][e] *= sigmoidf_(acc[0][e]);
      }
    }
    if (q == NCH - 1) {
      if (wave_nonfinite(y[0])) {
        const float* op = opaque_ptr(o) + ((int64_t)(D / 4 * g) * N + i) * ld + jp;
#pragma unroll
        for (int j = 0; j < D / 16; j++)
#pragma unroll
          for (int e = 0; e < 4; e++, op += N * ld) of.v[j][e] = *op;
        ln_out();
#pragma unroll
        for (int cb2 = 0; cb2 < CB; cb2++) y[0][cb2] = mma_f32<false, D>(w_po + (16 * cb2 + r) * D, of);
      }
      // the gates' input rows, loaded once the LN_out parts are done with
      RawRow<D> raw;
      raw.load(xrow(), g);
      split_row(x[0], raw);
    }
    if (q + 1 < 2 * NCH) {
      wstore((q + 1) & 1);  // last read in step q - 1, which every wave finished before the previous barrier
      if (q + 2 < 2 * NCH) wload(q + 2);
      __syncthreads();
    }
  }
  resid_ln_rows<float, 1>(y, zrow, z, accumulate, lnw, lnb, eps_next, xn_next);
}

// ---------------------------------------------------------------- linear_o + residual + next LayerNorm
// Persistent, 8 waves with W in LDS; a wave streams tiles of 16 rows, the next tile's rows and residual a tile ahead.
template <int DO>
__global__ __launch_bounds__(XT) void linear_resid_ln_x3_k(const float* __restrict__ x_in, const float* __restrict__ w,
                                                           int trans, float* __restrict__ z, int accumulate,
                                                           const float* __restrict__ lnw,
                                                           const float* __restrict__ lnb, float eps,
                                                           float* __restrict__ xn_next, int64_t N) {
  constexpr int K = 128, CB = DO / 16, PLANE_W = DO * ldx<K>();
  __shared__ LDS_ALIGN __bf16 Ws[3 * PLANE_W];
  __shared__ LnLds lns;
  const int64_t NN = N * N;
  const int ntiles = (int)((NN + 15) / 16), stride = gridDim.x * XW;
  const int l = threadIdx.x & 63, g = l >> 4, r = l & 15;
  int t = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * XW + (threadIdx.x >> 6)));
  const auto zrow_of = [&](int tt) -> int64_t {
    int64_t p = (int64_t)tt * 16 + r;
    if (p >= NN) return -1;
    if (trans) { const int64_t a = p / N; p = (p - a * N) * N + a; }
    return p;
  };
  RawRow<K> raw;
  f4 znext[1][CB];
  const auto load = [&](int tt) {
    raw.load(x_in + min((int64_t)tt * 16 + r, NN - 1) * K, g);
    const int64_t zr = zrow_of(tt);
    load_z_rows<1>(znext, [&](int) { return zr; }, z, accumulate);
  };
  load(min(t, ntiles - 1));
  stage_x3<DO, K, XT>(Ws, PLANE_W, [&](int rr) { return w + (int64_t)rr * K; });
  stage_ln(lns, lnw, lnb, DO);
  __syncthreads();
  const float* lw = lnw != nullptr ? lns.w : nullptr;
  for (; t < ntiles; t += stride) {
    X3Row<K> x[1];
    split_row(x[0], raw);
    f4 y[1][CB], zv[1][CB];
#pragma unroll
    for (int cb = 0; cb < CB; cb++) zv[0][cb] = znext[0][cb];
    load(min(t + stride, ntiles - 1));
#pragma unroll
    for (int cb = 0; cb < CB; cb++) {
      f4 acc[1] = {};
      mma_x3<1, false, K>(acc, x, Ws + 16 * cb * ldx<K>(), PLANE_W);
      y[0][cb] = acc[0];
      __builtin_amdgcn_sched_barrier(0);
    }
    if (wave_nonfinite(y[0])) {
      const float* const xr[1] = {x_in + min((int64_t)t * 16 + r, NN - 1) * K};
#pragma unroll
      for (int cb = 0; cb < CB; cb++) {
        f4 acc[1];
        mma_f32<1, false, K>(acc, w + (16 * cb + r) * K, xr);
        y[0][cb] = acc[0];
      }
    }
    const int64_t zr = zrow_of(t);
    resid_ln_apply<float, 1>(y, zv, [&](int) { return zr; }, z, lw, lns.b, eps, xn_next);
  }
}

// ---------------------------------------------------------------- pair bias = Linear(LN(z)) as [H][rows]
// (boltz_mlx/layers/attentionv2.py:40-48.) Persistent and bound by its read of z: a wave holds W's fragments (16 rows, H of
// them used) and streams tiles of 16 rows, the next tile loaded ahead; a row's LayerNorm stays in its four lanes. 160,000
// rows 36 us (through LDS, fp32 MFMA) -> 25, 263,169 rows 56 -> 35 (z's 135 MB at 5.2 TB/s: 26).
__global__ __launch_bounds__(256, 2) void pair_bias_x3_k(const float* __restrict__ z, const float* __restrict__ lnw,
                                                         const float* __restrict__ lnb, float eps,
                                                         const float* __restrict__ w, float* __restrict__ out,
                                                         int64_t rows, int H) {
  constexpr int D = 128;
  __shared__ LnLds lns;
  const int ntiles = (int)((rows + 15) / 16), stride = gridDim.x * 4;
  const int l = threadIdx.x & 63, g = l >> 4, r = l & 15;
  int t = grid_wave(4);
  RawRow<D> raw;
  const auto load = [&](int tt) { raw.load(z + min((int64_t)tt * 16 + r, rows - 1) * D, g); };
  load(min(t, ntiles - 1));
  X3Row<D> wx;
  {
    RawRow<D> wr = {};
    if (r < H) wr.load(w + (int64_t)r * D, g);
    split_row(wx, wr);
  }
  stage_ln(lns, lnw, lnb);
  __syncthreads();
  const auto ln = [&](RawRow<D>& v) {
    float sum = 0.f, ss = 0.f;
#pragma unroll
    for (int j = 0; j < D / 16; j++) sum += v.v[j][0] + v.v[j][1] + v.v[j][2] + v.v[j][3];
    const float mean = xgroups_sum(sum) * (1.0f / D);
#pragma unroll
    for (int j = 0; j < D / 16; j++) {
      v.v[j] = v.v[j] - mean;
      ss += v.v[j][0] * v.v[j][0] + v.v[j][1] * v.v[j][1] + v.v[j][2] * v.v[j][2] + v.v[j][3] * v.v[j][3];
    }
    const float rstd = 1.0f / sqrtf(xgroups_sum(ss) * (1.0f / D) + eps);
#pragma unroll
    for (int j = 0; j < D / 16; j++) {
      const int c = D / 4 * g + 4 * j;
      v.v[j] = v.v[j] * rstd * ld4(lns.w + c) + ld4(lns.b + c);
    }
  };
  for (; t < ntiles; t += stride) {
    ln(raw);
    X3Row<D> x;
    split_row(x, raw);
    load(min(t + stride, ntiles - 1));
    f4 acc = {};
#pragma unroll
    for (int q = 0; q < 6; q++)
#pragma unroll
      for (int s = 0; s < D / 32; s++) acc = mfma_x3<true>(wx.p[X3_W[q]][s], x.p[X3_X[q]][s], acc);
    const f4 all[1] = {acc};
    if (wave_nonfinite(all)) {
      RawRow<D> v;
      v.load(z + min((int64_t)t * 16 + r, rows - 1) * D, g);
      ln(v);
      acc = mma_f32<true, D>(w + (int64_t)min(r, H - 1) * D, v);
    }
    if (r < H) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int64_t p = (int64_t)t * 16 + 4 * g + e;
        if (p < rows) out[(int64_t)r * rows + p] = acc[e];
      }
    }
  }
}

// ---------------------------------------------------------------- transition
// h1, h2 = fc1 / fc2 rows . xn (16-unit blocks), a = silu(h1) * h2 in the accumulator layout, split in place: the B
// operand of out += fc3 a, a lane's k slots 8 g + t being units 16 (t / 4) + 4 g + t % 4 of a 32-unit slice.
__device__ __forceinline__ void split_units(X3Row<32>& b, const f4& lo, const f4& hi) {
  split8(lo, hi, b.p[0][0], b.p[1][0], b.p[2][0]);
}

// out = fc3 (silu(fc1 x) * fc2 x) over the 32-unit slices sl0, sl0 + step, ... on the fp32 matrix instructions, for a wave
// whose sums came out not finite (xr[rb]: the lane's rows of xn). A lane holds units 4 g + e of its row: step e of fc3.
template <int RB>
__device__ __forceinline__ void transition_f32(f4 (&out)[RB][8], const float* const (&xr)[RB], const float* w12,
                                               const float* w3, int hidden, int sl0, int step) {
  constexpr int D = 128;
  const int l = threadIdx.x & 63, g = l >> 4, r = l & 15;
  zero_acc(out);
#pragma unroll 1
  for (int u0 = 32 * sl0; u0 < hidden; u0 += (u0 & 16) ? 32 * step - 16 : 16) {
    f4 a[RB], h2[RB];
    mma_f32<RB, false, D>(a, w12 + (int64_t)(u0 + r) * D, xr);
    mma_f32<RB, false, D>(h2, w12 + (int64_t)(hidden + u0 + r) * D, xr);
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
      for (int e = 0; e < 4; e++) a[rb][e] = siluf_(a[rb][e]) * h2[rb][e];
#pragma unroll
    for (int ob = 0; ob < 8; ob++) {
      const f4 wv = ld4(w3 + (int64_t)(16 * ob + r) * hidden + u0 + 4 * g);
#pragma unroll
      for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int e = 0; e < 4; e++)
          out[rb][ob] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[e], a[rb][e], out[rb][ob], 0, 0, 0);
    }
  }
}
template <int RB, typename RowFn>
__device__ __forceinline__ void transition_finite(f4 (&out)[RB][8], const float* xn, RowFn row, int64_t rows_total,
                                                  const float* w12, const float* w3, int hidden, int sl0, int step) {
  bool bad = false;
#pragma unroll
  for (int rb = 0; rb < RB; rb++) bad = wave_nonfinite(out[rb]) || bad;
  if (!bad) return;
  const float* xr[RB];
#pragma unroll
  for (int rb = 0; rb < RB; rb++) xr[rb] = xn + min(row(rb), rows_total - 1) * 128;
  transition_f32<RB>(out, xr, w12, w3, hidden, sl0, step);
}

// Large inputs: tiles of 128 RB rows (8 waves of 16 RB), the hidden units streamed through LDS in chunks of 32 (fc1, fc2 rows
// and fc3 columns, split as they are written), the next chunk's values loaded while the current one computes.
// RB = 2 is at the 256 VGPRs of two waves per SIMD: 12 spill (52 bytes a lane), one 16-byte store and load of them a chunk.
constexpr int XH = 32;
template <int RB>
__global__ __launch_bounds__(XT) void transition_x3_k(const float* __restrict__ xn, const float* __restrict__ w12,
                                                      const float* __restrict__ w3, float* __restrict__ z,
                                                      int accumulate, const float* __restrict__ lnw,
                                                      const float* __restrict__ lnb, float eps,
                                                      float* __restrict__ xn_next, int64_t rows_total, int hidden) {
  constexpr int D = 128, LW = ldx<D>(), L3 = XH + 8, P12 = 2 * XH * LW, P3 = D * L3;
  __shared__ LDS_ALIGN __bf16 W12[3 * P12];
  __shared__ LDS_ALIGN __bf16 W3[3 * P3];
  const int t = threadIdx.x, wave = t >> 6, l = t & 63, g = l >> 4, r = l & 15;
  const int64_t r0 = (int64_t)blockIdx.x * (16 * RB * XW) + 16 * RB * wave;
  int64_t row[RB];
  X3Row<D> x[RB];
#pragma unroll
  for (int rb = 0; rb < RB; rb++) {
    row[rb] = r0 + 16 * rb + r;
    RawRow<D> raw;
    raw.load(xn + (row[rb] < rows_total ? row[rb] : rows_total - 1) * D, g);
    split_row(x[rb], raw);
  }
  // a chunk's items of this thread: fc1 and fc2 row t / 16, channels 8 (t % 16) .. + 7; fc3 channel t / 4, units
  // 8 (t % 4) .. + 7, stored at the slots the fragment reads take (unit 16 hi + 4 q + e at 8 q + 4 hi + e)
  f4 pre[3][2];
  const auto wload = [&](int h0) {
    const float* s1 = w12 + (int64_t)(h0 + (t >> 4)) * D + (t & 15) * 8;
    const float* s2 = s1 + (int64_t)hidden * D;
    const float* s3 = w3 + (int64_t)(t >> 2) * hidden + h0 + (t & 3) * 8;
#pragma unroll
    for (int v = 0; v < 2; v++) {
      pre[0][v] = ld4(s1 + 4 * v);
      pre[1][v] = ld4(s2 + 4 * v);
      pre[2][v] = ld4(s3 + 4 * v);
    }
  };
  const auto wstore = [&]() {
#pragma unroll
    for (int m = 0; m < 2; m++) {
      bf16x8 p[3];
      split8(pre[m][0], pre[m][1], p[0], p[1], p[2]);
      __bf16* d = W12 + (m * XH + (t >> 4)) * LW + (t & 15) * 8;
#pragma unroll
      for (int q = 0; q < 3; q++) *reinterpret_cast<bf16x8*>(d + q * P12) = p[q];
    }
    bf16x8 p[3];
    split8(pre[2][0], pre[2][1], p[0], p[1], p[2]);
    const int u = t & 3;
    __bf16* d = W3 + (t >> 2) * L3 + 16 * (u & 1) + 4 * (u >> 1);
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const uint4 v = __builtin_bit_cast(uint4, p[q]);
      *reinterpret_cast<uint2*>(d + q * P3) = uint2{v.x, v.y};
      *reinterpret_cast<uint2*>(d + q * P3 + 8) = uint2{v.z, v.w};
    }
  };
  f4 out[RB][8];
  zero_acc(out);
  wload(0);
  for (int h0 = 0; h0 < hidden; h0 += XH) {
    if (h0) __syncthreads();  // every wave is done with the previous chunk
    wstore();
    wload(h0 + XH < hidden ? h0 + XH : 0);
    __syncthreads();
    f4 a[RB][2];
#pragma unroll
    for (int hb = 0; hb < 2; hb++) {
      f4 h1[RB] = {}, h2[RB] = {};
      mma_x3<RB, false, D>(h1, x, W12 + 16 * hb * LW, P12);
      mma_x3<RB, false, D>(h2, x, W12 + (XH + 16 * hb) * LW, P12);
#pragma unroll
      for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int e = 0; e < 4; e++) a[rb][hb][e] = siluf_(h1[rb][e]) * h2[rb][e];
    }
    X3Row<32> b[RB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) split_units(b[rb], a[rb][0], a[rb][1]);
#pragma unroll
    for (int ob = 0; ob < 8; ob++) {
      const __bf16* wp = W3 + (16 * ob + r) * L3 + 8 * g;
      bf16x8 wf[3];
#pragma unroll
      for (int p = 0; p < 3; p++) wf[p] = *reinterpret_cast<const bf16x8*>(wp + p * P3);
#pragma unroll
      for (int q = 0; q < 6; q++)
#pragma unroll
        for (int rb = 0; rb < RB; rb++) out[rb][ob] = mfma_x3<false>(wf[X3_W[q]], b[rb].p[X3_X[q]][0], out[rb][ob]);
    }
  }
  transition_finite<RB>(out, xn, [&](int rb) { return row[rb]; }, rows_total, w12, w3, hidden, 0, 1);
  resid_ln_rows<float, RB>(out, [&](int rb) -> int64_t { return row[rb] < rows_total ? row[rb] : -1; }, z, accumulate,
                          lnw, lnb, eps, xn_next);
}

// Small inputs: a workgroup takes 16 RB rows and its 8 waves an eighth of the hidden units each (slices wave, wave + 8,
// ... of 32 units), the weights read straight from the caches and split in registers, the partial sums added over LDS
// in wave order; the rows' residual and LayerNorm then run on 32 / RB lanes per row.
template <int RB>
__global__ __launch_bounds__(XT) void transition_x3_small_k(const float* __restrict__ xn,
                                                            const float* __restrict__ w12,
                                                            const float* __restrict__ w3, float* __restrict__ z,
                                                            int accumulate, const float* __restrict__ lnw,
                                                            const float* __restrict__ lnb, float eps,
                                                            float* __restrict__ xn_next, int64_t rows_total,
                                                            int hidden) {
  constexpr int D = 128, LDO = D + 4, ROWS = 16 * RB;
  __shared__ LDS_ALIGN float Part[XW][ROWS][LDO];
  const int t = threadIdx.x, l = t & 63, g = l >> 4, r = l & 15;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t r0 = (int64_t)blockIdx.x * ROWS;
  const int nsl = hidden / 32;
  X3Row<D> x[RB];
  // weight block u of slice sl: 0, 1: fc1 / fc2 rows 0 .. 15 of the slice; 2, 3: rows 16 .. 31; raw holds one block,
  // step s of the next block is loaded as step s of this one has been split
  RawRow<D> raw;
  const auto wptr = [&](int sl, int u) {
    return w12 + (int64_t)((u & 1) * hidden + 32 * sl + 16 * (u >> 1) + r) * D + 32 * g;
  };
  const int sl0 = min(wave, nsl - 1);
  raw.load(wptr(sl0, 0) - 32 * g, g);
#pragma unroll
  for (int rb = 0; rb < RB; rb++) {
    const int64_t row = r0 + 16 * rb + r;
    RawRow<D> xr;
    xr.load(xn + (row < rows_total ? row : rows_total - 1) * D, g);
    split_row(x[rb], xr);
  }
  f4 out[RB][8];
  zero_acc(out);
  for (int sl = wave; sl < nsl; sl += XW) {
    f4 a[RB][2], h1[RB];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      f4 h[RB] = {};
      const float* nx = u < 3 ? wptr(sl, u + 1) : wptr(min(sl + XW, nsl - 1), 0);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        bf16x8 wf[3];
        split8(raw.v[2 * s], raw.v[2 * s + 1], wf[0], wf[1], wf[2]);
        raw.v[2 * s] = ld4(nx + 8 * s);
        raw.v[2 * s + 1] = ld4(nx + 8 * s + 4);
#pragma unroll
        for (int q = 0; q < 6; q++)
#pragma unroll
          for (int rb = 0; rb < RB; rb++) h[rb] = mfma_x3<false>(wf[X3_W[q]], x[rb].p[X3_X[q]][s], h[rb]);
      }
#pragma unroll
      for (int rb = 0; rb < RB; rb++) {
        if (u & 1) {
#pragma unroll
          for (int e = 0; e < 4; e++) a[rb][u >> 1][e] = siluf_(h1[rb][e]) * h[rb][e];
        } else {
          h1[rb] = h[rb];
        }
      }
    }
    X3Row<32> b[RB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) split_units(b[rb], a[rb][0], a[rb][1]);
    const float* wp = w3 + (int64_t)r * hidden + 32 * sl + 4 * g;
#pragma unroll
    for (int ob = 0; ob < 8; ob++) {
      bf16x8 wf[3];
      split8(ld4(wp + (int64_t)16 * ob * hidden), ld4(wp + (int64_t)16 * ob * hidden + 16), wf[0], wf[1], wf[2]);
#pragma unroll
      for (int q = 0; q < 6; q++)
#pragma unroll
        for (int rb = 0; rb < RB; rb++) out[rb][ob] = mfma_x3<false>(wf[X3_W[q]], b[rb].p[X3_X[q]][0], out[rb][ob]);
    }
  }
  transition_finite<RB>(out, xn, [&](int rb) { return r0 + 16 * rb + r; }, rows_total, w12, w3, hidden, wave, XW);
#pragma unroll
  for (int rb = 0; rb < RB; rb++)
#pragma unroll
    for (int ob = 0; ob < 8; ob++) st4(&Part[wave][16 * rb + r][16 * ob + 4 * g], out[rb][ob]);
  __syncthreads();
  // row lr of the tile on LPR lanes, VPL vectors of 4 channels each
  constexpr int LPR = 32 / RB, VPL = RB;
  const int lr = t / LPR, q0 = t % LPR;
  const int64_t row = r0 + lr, rc = row < rows_total ? row : rows_total - 1;
  f4 v[VPL];
  float s = 0.f;
#pragma unroll
  for (int u = 0; u < VPL; u++) {
    const int c = 4 * (q0 + LPR * u);
    f4 y = ld4(&Part[0][lr][c]);
#pragma unroll
    for (int p = 1; p < XW; p++) y = y + ld4(&Part[p][lr][c]);
    v[u] = accumulate ? y + ld4(z + rc * D + c) : y;
    s += v[u][0] + v[u][1] + v[u][2] + v[u][3];
    if (row < rows_total) st4(z + row * D + c, v[u]);
  }
  if (lnw == nullptr) return;
  const float mean = group_sum<LPR>(s) * (1.0f / D);
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < VPL; u++) {
    const f4 d = v[u] - mean;
    ss += d[0] * d[0] + d[1] * d[1] + d[2] * d[2] + d[3] * d[3];
  }
  const float rstd = 1.0f / sqrtf(group_sum<LPR>(ss) * (1.0f / D) + eps);
  if (row >= rows_total) return;
#pragma unroll
  for (int u = 0; u < VPL; u++) {
    const int c = 4 * (q0 + LPR * u);
    st4(xn_next + row * D + c, (v[u] - mean) * rstd * ld4(lnw + c) + ld4(lnb + c));
  }
}

template <typename Kern>
int x3_resident(Kern kernel, int (&cache)[kMaxDevices]) { return resident_grid(kernel, XT, cache); }

template <int KIN>
hipError_t proj_x3(const float* xn, const float* w, const float* mask, float scale, int incoming, float* ab, int64_t N,
                   int64_t ld, hipStream_t st) {
  static int cache[kMaxDevices];
  const int resident = x3_resident(trimul_proj_x3_k<KIN>, cache);
  if (resident <= 0) return hipErrorInvalidDevice;
  const int64_t ntiles = N * (ld / XTW);
  if (ntiles >= (1LL << 30)) return hipErrorInvalidValue;  // tile indices are 32-bit in the kernel
  trimul_proj_x3_k<KIN><<<group_grid(resident, 2 * KIN / 64, ntiles, XW), XT, 0, st>>>(xn, w, mask, scale, incoming, ab, N, ld);
  return hipGetLastError();
}

template <int KIN>
hipError_t tail_x3(const float* o, const float* now, const float* nob, float eps_out, const float* w_po,
                   const float* xn, const float* w_go, float* z, int accumulate, const float* lnw, const float* lnb,
                   float eps_next, float* xn_next, int64_t N, int64_t ld, hipStream_t st) {
  const int64_t tpr = (N + 63) / 64;  // ld is a multiple of 64 no smaller than N: a tile's o columns are inside the row
  if (N * tpr >= (1LL << 30)) return hipErrorInvalidValue;
  trimul_tail_x3_k<KIN><<<(unsigned)(N * tpr), 256, 0, st>>>(o, now, nob, eps_out, w_po, xn, w_go, z, accumulate, lnw,
                                                             lnb, eps_next, xn_next, N, (int)tpr, ld);
  return hipGetLastError();
}

template <int KIN>
hipError_t attn_proj_x3(const float* xn, const float* w, int trans, float q_scale, float b_scale, float* qkg, float* vt,
                        float* tb, int64_t N, int64_t ldk, int H, int C, hipStream_t st) {
  if (H * C != 128 || H > 16 || C % 8) return hipErrorInvalidValue;
  static int cache[kMaxDevices];
  const int resident = x3_resident(triattn_proj_x3_k<KIN>, cache);
  if (resident <= 0) return hipErrorInvalidDevice;
  const int64_t ntiles = N * (ldk / XTW);
  if (ntiles >= (1LL << 30)) return hipErrorInvalidValue;
  triattn_proj_x3_k<KIN><<<group_grid(resident, 4, ntiles, XW), XT, 0, st>>>(xn, w, trans, q_scale, b_scale, qkg, vt, tb, N,
                                                                      ldk, H, C);
  return hipGetLastError();
}

template <int DO>
hipError_t lrl_x3(const float* x, const float* w, int trans, float* z, int accumulate, const float* lnw,
                  const float* lnb, float eps, float* xn_next, int64_t N, hipStream_t st) {
  static int cache[kMaxDevices];
  const int resident = x3_resident(linear_resid_ln_x3_k<DO>, cache);
  if (resident <= 0) return hipErrorInvalidDevice;
  const int64_t ntiles = (N * N + 15) / 16;
  if (ntiles >= (1LL << 30)) return hipErrorInvalidValue;
  linear_resid_ln_x3_k<DO><<<(unsigned)std::min<int64_t>(resident, (ntiles + XW - 1) / XW), XT, 0, st>>>(
      x, w, trans, z, accumulate, lnw, lnb, eps, xn_next, N);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_trimul_proj_x3(const float* xn, const float* w, const float* mask, float scale, int incoming,
                                 float* ab, int64_t N, int64_t ld, int dim, hipStream_t st) {
  return (dim == 64 ? proj_x3<64> : proj_x3<128>)(xn, w, mask, scale, incoming, ab, N, ld, st);
}

hipError_t launch_trimul_tail_x3(const float* o, const float* now, const float* nob, float eps_out, const float* w_po,
                                 const float* xn, const float* w_go, float* z, int accumulate, const float* lnw,
                                 const float* lnb, float eps_next, float* xn_next, int64_t N, int64_t ld, int dim,
                                 hipStream_t st) {
  return (dim == 64 ? tail_x3<64> : tail_x3<128>)(o, now, nob, eps_out, w_po, xn, w_go, z, accumulate, lnw, lnb,
                                                  eps_next, xn_next, N, ld, st);
}

hipError_t launch_triattn_proj_x3(const float* xn, const float* w, int trans, float q_scale, float b_scale, float* qkg,
                                  float* vt, float* tb, int64_t N, int64_t ldk, int dim, int H, int C,
                                  hipStream_t st) {
  return (dim == 64 ? attn_proj_x3<64> : attn_proj_x3<128>)(xn, w, trans, q_scale, b_scale, qkg, vt, tb, N, ldk, H, C,
                                                            st);
}

hipError_t launch_linear_resid_ln_x3(const float* x, const float* w, int trans, float* z, int accumulate,
                                     const float* lnw, const float* lnb, float eps, float* xn_next, int64_t N, int dim,
                                     hipStream_t st) {
  return (dim == 64 ? lrl_x3<64> : lrl_x3<128>)(x, w, trans, z, accumulate, lnw, lnb, eps, xn_next, N, st);
}

hipError_t launch_pair_bias_x3(const float* z, const float* lnw, const float* lnb, float eps, const float* w, float* out,
                               int64_t rows, int H, hipStream_t st) {
  static int cache[kMaxDevices];
  const int resident = resident_grid(pair_bias_x3_k, 256, cache);
  if (resident <= 0) return hipErrorInvalidDevice;
  const int64_t ntiles = (rows + 15) / 16;
  if (rows < 1 || H < 1 || H > 16 || ntiles >= (1LL << 30)) return hipErrorInvalidValue;
  pair_bias_x3_k<<<(unsigned)std::min<int64_t>(resident, (ntiles + 3) / 4), 256, 0, st>>>(z, lnw, lnb, eps, w, out, rows, H);
  return hipGetLastError();
}

hipError_t launch_transition_x3(const float* xn, const float* w12, const float* w3, float* z, int accumulate,
                                const float* lnw, const float* lnb, float eps, float* xn_next, int64_t rows,
                                int hidden, hipStream_t st) {
  if (hidden % 32 || rows > (1LL << 34)) return hipErrorInvalidValue;
  // Whole rounds of one 256-row tile a CU (the kernel's LDS lets one workgroup in), then the remaining rows in the form that
  // takes them soonest (transition_split). On 256 CUs, 512 hidden units, us: 16-row tiles with the hidden units split over
  // the waves 27 up to 4,096 rows, 32-row ones 31 a round of 8,192 rows (16,384: 64), 128-row tiles 74 up to 32,768
  // (32-row ones 120), 256-row tiles 105 to 128 up to 65,536. 263,169 rows: 538 (1,029 256-row tiles alone 561, fp32 MFMA
  // 935).
  static int cache[kMaxDevices];
  const int cus = x3_resident(transition_x3_k<2>, cache);
  if (cus <= 0) return hipErrorInvalidDevice;
  const auto part = [&](int64_t r0, int64_t n, auto kernel, int64_t tile) {
    kernel<<<(unsigned)((n + tile - 1) / tile), XT, 0, st>>>(xn + r0 * 128, w12, w3, z + r0 * 128, accumulate, lnw, lnb,
                                                             eps, xn_next != nullptr ? xn_next + r0 * 128 : nullptr, n,
                                                             hidden);
    return hipGetLastError();
  };
  const TransitionSplit split = transition_split(rows, cus);
  const int64_t full = split.full, rem = rows - full;
  if (full > 0) {
    const hipError_t e = part(0, full, transition_x3_k<2>, 256);
    if (e != hipSuccess || rem == 0) return e;
  }
  switch (split.tile) {
    case 16: return part(full, rem, transition_x3_small_k<1>, 16);
    case 32: return part(full, rem, transition_x3_small_k<2>, 32);
    case 128: return part(full, rem, transition_x3_k<1>, 128);
    default: return part(full, rem, transition_x3_k<2>, 256);
  }
}

}  // namespace bzpf
