// fp32 flash triangle-attention core on the bf16 matrix cores, head width C = 32: every fp32 operand (Q, K, V and the
// probabilities) is split exactly into three bf16 parts and a product is its six leading part products with fp32 sums
// (bzpf_x3.h), so logits, softmax, probabilities and sums all keep fp32 accuracy.
//
// What bounds it: a 32-key x 32-query tile costs 24 v_mfma_f32_32x32x16_bf16 (768 cycles) and about 210 VALU
// instructions (the probabilities' split is 88 of them); at N = 640 (807 us, 1.02 M tiles on 1,024 SIMDs) a tile takes about
// 1,940 cycles of its SIMD at the nominal 2.4 GHz (fewer at the clock held under load): the two pipes overlap little. N = 400: 249 us (132 TFLOP/s of the 32.8
// GFLOP without padding), against 2,405 us on the VALU kernel (kept for the other head widths and as the caller's choice);
// the true fp32 MFMA (v_mfma_f32_32x32x2f32) would need 2,048 cycles a tile.
//
// Work unit: one (head h, row i, 128 queries), 4 waves of 32 queries; 128 VGPRs and 31 KB of LDS, so four workgroups
// share a CU (64-key stages at 187 VGPRs and two workgroups took 1.14 times as long). S^T = K Q^T as in the fp16 core: lane l = 32 hl + q
// owns query q and keys 8 (e / 4) + 4 hl + e % 4 of each 32-key tile, so its statistics need one cross-half step and its
// probabilities are, split in place, already the B operand of O^T = V^T P^T for V^T staged in the matching key order.
// 32 keys of K and V^T per stage are loaded a stage ahead, split by the threads that loaded them and written to one of
// two LDS buffers (one barrier per stage: the buffer written in stage kb was last read in stage kb - 2, which every wave
// finished before the barrier of kb - 1); the bias arrives in the fragment order of tb_offset, straight into registers,
// and starts the logits' accumulators.
// Logits are base 2. A stage that masks a key adds the mask's bias in the reference's order, (q.k + mask) + bias, so a
// row whose keys are all masked gets the uniform weights that fp32 rounding gives. Stages after the row's last
// unmasked key are skipped where that cannot change a bit: a masked key's logit is about inf*log2(e) below the
// maximum, and 2^x is exactly zero in fp32 below x = -150 (inf >= 1e6 leaves room for any spread of the logits).
// The maximum is raised lazily: probabilities are formed against the current one, and only a lane whose sum of a tile's
// passes 2^15 (or is not a number) makes the wave raise it. v_exp_f32 gives 0 below 2^-126, so a key whose weight is less than
// 2^-126 of the row's largest has none. A wave whose sums come out not finite (an operand without parts, bzpf_rowgemm_x3.h;
// values so large that 2^15 of them overflow) forms its queries again in fp32.
// Reference behaviour: boltz_mlx/layers/triangular_attention/attention.py:27-93, kernels.py:538-600.
#include "bzpf_common.h"
#include "bzpf_kernels.h"
#include "bzpf_x3.h"

namespace bzpf {

namespace {

constexpr int NXCD = 8;

__device__ __forceinline__ float halves_max(float v) {
  const unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ float halves_sum(float v) {
  const unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}

// eight fp32 values as the three bf16 parts of a fragment (part p: values 0 .. 7 in order)
__device__ __forceinline__ void split3_8(const float (&x)[8], bf16x8 (&p)[3]) {
  u32x4_t w[3];
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const Pair3 s = split3_pair(x[2 * e], x[2 * e + 1]);
#pragma unroll
    for (int q = 0; q < 3; q++) w[q][e] = s.p[q];
  }
#pragma unroll
  for (int q = 0; q < 3; q++) p[q] = __builtin_bit_cast(bf16x8, w[q]);
}

constexpr int XBK = 32;            // keys per stage
constexpr int XLDK = 32 + 8;       // K rows: 32 channels (pitch 80 B: 16 lanes on 16 rows meet distinct banks)
constexpr int XLDV = XBK + 8;      // V^T rows: 32 keys (likewise)
constexpr int XKP = XBK * XLDK;    // one part plane of K
constexpr int XVP = 32 * XLDV;     // one part plane of V^T

__global__ __launch_bounds__(256, 3) void triattn_core_x3_k(const float* __restrict__ qkg, const float* __restrict__ vt,
                                                            const float* __restrict__ tb,
                                                            const float* __restrict__ mask, int64_t mask_si,
                                                            int64_t mask_sk, float inf, float* __restrict__ out, int N,
                                                            int ldk, int H, int64_t units, int64_t per_xcd) {
  constexpr int C = 32, WQ = 128;
  constexpr float LOG2E = 1.4426950408889634f;
  constexpr float PLIM = 32768.0f;
  __shared__ LDS_ALIGN __bf16 Ks[2][3 * XKP];
  __shared__ LDS_ALIGN __bf16 Vs[2][3 * XVP];
  __shared__ LDS_ALIGN float Mb[4][64];  // (written by all 64 lanes; keys 0 .. 31 are read)
  __shared__ int kend_w[4];

  const int64_t u = (int64_t)(blockIdx.x % NXCD) * per_xcd + blockIdx.x / NXCD;
  if (u >= units) return;  // whole workgroup
  const int nqb = (N + WQ - 1) / WQ;
  const int qb = (int)(u % nqb);
  const int64_t hi = u / nqb;
  const int i = (int)(hi % N), h = (int)(hi / N);
  const int64_t NN = (int64_t)N * N;
  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), l = t & 63;
  const int hl = l >> 5, qi = l & 31;
  const float* qp = qkg + ((int64_t)h * NN + (int64_t)i * N) * C;
  const float* kp = qkg + ((int64_t)(H + h) * NN + (int64_t)i * N) * C;
  const float* gp = qkg + ((int64_t)(2 * H + h) * NN + (int64_t)i * N) * C;
  const float* vp = vt + ((int64_t)h * N + i) * C * ldk;
  const float* mrow = mask + (int64_t)i * mask_si;
  const int jq = qb * WQ + 32 * wave + qi;
  const bool wact = qb * WQ + 32 * wave < N;  // wave-uniform: the wave has queries (else it only stages)

  // the row's key extent (1 + its last unmasked key; every key when none is unmasked), 256 keys at a time from the end
  int kend = 0;
  for (int base = N - 256;; base -= 256) {  // workgroup-uniform
    const int kq = base + t;                // < N
    const uint64_t b = __ballot(kq >= 0 && mrow[(int64_t)kq * mask_sk] != 0.0f);
    if (l == 0) kend_w[wave] = b ? base + 64 * wave + 64 - __clzll(b) : 0;
    __syncthreads();
    kend = max(max(kend_w[0], kend_w[1]), max(kend_w[2], kend_w[3]));
    __syncthreads();  // kend_w is written again by the next step
    if (kend > 0 || base <= 0) break;
  }
  if (kend <= 0 || inf < 1e6f) kend = N;
  const int nblk = (kend + XBK - 1) / XBK;

  // Q fragments: part p of slab m holds channels 16 m + 8 hl .. + 7 of the lane's query
  bf16x8 qf[2][3];
  {
    const int jc = jq < N ? jq : N - 1;
#pragma unroll
    for (int m = 0; m < 2; m++) {
      const f4 a = *reinterpret_cast<const f4*>(qp + (int64_t)jc * C + 16 * m + 8 * hl);
      const f4 b = *reinterpret_cast<const f4*>(qp + (int64_t)jc * C + 16 * m + 8 * hl + 4);
      const float x[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
      split3_8(x, qf[m]);
    }
  }
  f16x oacc;
#pragma unroll
  for (int e = 0; e < 16; e++) oacc[e] = 0.f;
  float m_run = -INFINITY, lsum = 0.f;

  // staging roles: thread t loads channels 4 (t % 8) .. + 3 of key t / 8 and keys 4 (t % 8) .. + 3 of channel t / 8
  const int srow = t >> 3, s4 = (t & 7) * 4;
  constexpr int RSRC_CFG = 0x00020000;  // raw buffer, 32-bit data format; loads past the extent read as zeros
  const __amdgpu_buffer_rsrc_t krs =
      __builtin_amdgcn_make_buffer_rsrc((void*)kp, 0, (int)xcore_k_extent(N, C), RSRC_CFG);
  const __amdgpu_buffer_rsrc_t vrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)vp, 0, (int)xcore_v_extent(ldk, C), RSRC_CFG);
  const __amdgpu_buffer_rsrc_t mrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)mrow, 0, (int)core_m_extent(N, mask_sk), RSRC_CFG);
  const int njt = (N + 31) / 32, nkb = ldk / 64;
  __amdgpu_buffer_rsrc_t brs;
  {
    int jt = qb * (WQ / 32) + wave;
    if (jt >= njt) jt = njt - 1;
    brs = __builtin_amdgcn_make_buffer_rsrc((void*)(tb + (((int64_t)h * njt + jt) * nkb) * 2048), 0,
                                            (int)xcore_b_extent(ldk), RSRC_CFG);
  }
  const int koff = xcore_k_lane(t, C), voff = xcore_v_lane(t, ldk), mvo = core_m_lane(qi, mask_sk);
  f4 kreg, vreg, bcur[4];
  float mraw;
  auto ldb = [](const __amdgpu_buffer_rsrc_t& r, int vo, int so) {
    return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(r, vo, so, 0));
  };
  auto prefetch = [&](int kb) {
    kreg = ldb(krs, koff, xcore_k_stage(kb, C));
    vreg = ldb(vrs, voff, xcore_v_stage(kb));
    mraw = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(mrs, mvo, xcore_m_stage(kb, mask_sk), 0));
  };
  auto prefetch_bias = [&](int kb) {
#pragma unroll
    for (int v = 0; v < 4; v++) bcur[v] = ldb(brs, xcore_b_lane(v, l), xcore_b_stage(kb));
  };
  prefetch(0);
  if (wact) prefetch_bias(0);

  for (int kb = 0; kb < nblk; kb++) {
    const int k0 = kb * XBK, buf = kb & 1;
    __bf16* Kb = Ks[buf];
    __bf16* Vb = Vs[buf];
    {
      const Pair3 lo = split3_pair(kreg[0], kreg[1]), hi = split3_pair(kreg[2], kreg[3]);
#pragma unroll
      for (int q = 0; q < 3; q++)
        *reinterpret_cast<uint2*>(Kb + q * XKP + srow * XLDK + s4) = uint2{lo.p[q], hi.p[q]};
    }
    {
      if (k0 + XBK > N) {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (k0 + s4 + e >= N) vreg[e] = 0.0f;
      }
      // within each 16-key slab, key 8 a + 4 h + e sits at 8 h + 4 a + e: the 8 keys of a lane half (4 hl .. + 3 and
      // 8 + 4 hl .. + 3) are one 16-byte read
      const Pair3 lo = split3_pair(vreg[0], vreg[1]), hi = split3_pair(vreg[2], vreg[3]);
      const int u = t & 7;
      __bf16* d = Vb + srow * XLDV + 16 * (u >> 2) + 8 * (u & 1) + 4 * ((u >> 1) & 1);
#pragma unroll
      for (int q = 0; q < 3; q++) *reinterpret_cast<uint2*>(d + q * XVP) = uint2{lo.p[q], hi.p[q]};
    }
    // key-mask bias of key k0 + qi (keys past N: -inf); the same in every wave, so each wave decides by itself
    const float mbias = k0 + qi < N ? inf * (mraw - 1.0f) * LOG2E : -INFINITY;
    const bool masked = __any(mbias != 0.0f);
    if (masked) Mb[wave][l] = mbias;
    __syncthreads();
    prefetch(kb + 1 < nblk ? kb + 1 : nblk - 1);
    if (!wact) continue;

    f16x s;
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int e = 0; e < 4; e++) s[4 * q + e] = masked ? 0.0f : bcur[q][e];
#pragma unroll
    for (int m = 0; m < 2; m++) {
      bf16x8 kf[3];
#pragma unroll
      for (int p = 0; p < 3; p++)
        kf[p] = *reinterpret_cast<const bf16x8*>(Kb + p * XKP + qi * XLDK + 16 * m + 8 * hl);
      s = mfma_parts6(kf, qf[m], s);
    }
    if (masked) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const f4 mb = *reinterpret_cast<const f4*>(&Mb[wave][8 * q + 4 * hl]);
#pragma unroll
        for (int e = 0; e < 4; e++) s[4 * q + e] = (s[4 * q + e] + mb[e]) + bcur[q][e];
      }
    }
    prefetch_bias(kb + 1 < nblk ? kb + 1 : nblk - 1);
    // probabilities relative to the current maximum; a lane whose sum of them passes PLIM (the first tile, a logit that
    // far above the maximum, an overflow) raises it and forms them again
    float p[16], psum = 0.f;
    const auto probs = [&]() {
      psum = 0.f;
#pragma unroll
      for (int e = 0; e < 16; e++) {
        p[e] = __builtin_amdgcn_exp2f(s[e] - m_run);
        psum += p[e];
      }
    };
    probs();
    if (__any(jq < N && !(psum <= PLIM))) {
      float mx = fmaxf(s[0], s[1]);
#pragma unroll
      for (int e = 2; e < 16; e += 2) mx = fmaxf(fmaxf(mx, s[e]), s[e + 1]);
      const float mn = fmaxf(m_run, halves_max(mx));
      const float corr = __builtin_amdgcn_exp2f(m_run - mn);
      oacc *= corr;
      lsum *= corr;
      m_run = mn;
      probs();
    }
    lsum += psum;
#pragma unroll
    for (int sl = 0; sl < 2; sl++) {
      const float ps[8] = {p[8 * sl], p[8 * sl + 1], p[8 * sl + 2], p[8 * sl + 3],
                           p[8 * sl + 4], p[8 * sl + 5], p[8 * sl + 6], p[8 * sl + 7]};
      bf16x8 pf[3], vf[3];
      split3_8(ps, pf);
#pragma unroll
      for (int q = 0; q < 3; q++)
        vf[q] = *reinterpret_cast<const bf16x8*>(Vb + q * XVP + qi * XLDV + 16 * sl + 8 * hl);
      oacc = mfma_parts6(vf, pf, oacc);
    }
  }
  if (!wact) return;
  float t0 = lsum * 0.f;
#pragma unroll
  for (int e = 0; e < 16; e++) t0 = fmaf(oacc[e], 0.f, t0);
  if (__any(jq < N && t0 != t0)) {
    // Sums that are not finite: the wave's queries again in fp32 throughout (v_mfma_f32_32x32x2_f32, one k of each lane
    // half a step), operands straight from memory, probabilities relative to the true running maximum.
    const float* qr = qp + (int64_t)(jq < N ? jq : N - 1) * C + 4 * hl;
    const float* vr = vp + (int64_t)qi * ldk + 4 * hl;
    m_run = -INFINITY;
    lsum = 0.f;
#pragma unroll
    for (int e = 0; e < 16; e++) oacc[e] = 0.f;
#pragma unroll 1
    for (int kb = 0; kb < nblk; kb++) {
      const int k0 = kb * XBK;
      const float* kr = kp + (int64_t)min(k0 + qi, N - 1) * C + 4 * hl;
      f16x s;
#pragma unroll
      for (int e = 0; e < 16; e++) s[e] = 0.f;
#pragma unroll 1
      for (int c = 0; c < C; c += 8) {
        const f4 kv = *reinterpret_cast<const f4*>(kr + c), qv = *reinterpret_cast<const f4*>(qr + c);
#pragma unroll
        for (int e = 0; e < 4; e++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[e], qv[e], s, 0, 0, 0);
      }
      float mx = -INFINITY;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const f4 b = ldb(brs, xcore_b_lane(q, l), xcore_b_stage(kb));
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int k = k0 + 8 * q + 4 * hl + e;
          const float mb = k < N ? inf * (mrow[(int64_t)k * mask_sk] - 1.0f) * LOG2E : -INFINITY;
          s[4 * q + e] = k < N ? (s[4 * q + e] + mb) + b[e] : -INFINITY;
          mx = fmaxf(mx, s[4 * q + e]);
        }
      }
      const float mn = fmaxf(m_run, halves_max(mx)), corr = exp2f(m_run - mn);
      oacc *= corr;
      lsum *= corr;
      m_run = mn;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        f4 vv = *reinterpret_cast<const f4*>(vr + k0 + 8 * q);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if (k0 + 8 * q + 4 * hl + e >= N) vv[e] = 0.0f;
          const float p = exp2f(s[4 * q + e] - mn);
          lsum += p;
          oacc = __builtin_amdgcn_mfma_f32_32x32x2f32(vv[e], p, oacc, 0, 0, 0);
        }
      }
    }
  }
  const float ltot = halves_sum(lsum);
  if (jq >= N) return;
  const float inv = 1.0f / ltot;
  float* oq = out + ((int64_t)i * N + jq) * (int64_t)(H * C) + h * C;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int d0 = 8 * q + 4 * hl;
    const f4 gv = *reinterpret_cast<const f4*>(gp + (int64_t)jq * C + d0);
    f4 ov;
#pragma unroll
    for (int e = 0; e < 4; e++) ov[e] = oacc[4 * q + e] * inv * sigmoidf_(gv[e]);
    *reinterpret_cast<f4*>(oq + d0) = ov;
  }
}

}  // namespace

hipError_t launch_triattn_core_f32_x3(const void* qkg, const void* vt, const void* tb, const float* mask,
                                      int64_t mask_si, int64_t mask_sk, float inf, void* out, int64_t N, int64_t ldk,
                                      int H, hipStream_t st) {
  const int64_t units = (int64_t)H * N * ((N + 127) / 128);
  const int64_t per_xcd = (units + NXCD - 1) / NXCD;
  triattn_core_x3_k<<<dim3((unsigned)(per_xcd * NXCD)), 256, 0, st>>>(
      static_cast<const float*>(qkg), static_cast<const float*>(vt), static_cast<const float*>(tb), mask, mask_si,
      mask_sk, inf, static_cast<float*>(out), (int)N, (int)ldk, H, units, per_xcd);
  return hipGetLastError();
}

}  // namespace bzpf
