// The row-tile GEMM of bzpf_rowgemm.h for fp32 operands on the bf16 matrix cores: every operand value as three exact
// bf16 parts, a product as six part products (bzpf_x3.h), on v_mfma_f32_16x16x32_bf16. Fragment and accumulator layouts
// are those of the fp16 form (lane l = 16 g + r: row r, channels KIN / 4 g + 8 s + t of step s; accumulator rows or
// channels 4 g + e), six MFMAs of 16 cycles per 32 channels against the fp32 form's eight of 32.
// Weights sit in LDS as three planes of [rows][KIN + 8] bf16 (the padded pitch keeps the 16-byte fragment reads free of
// bank conflicts); they are split while they are staged, rows of x when a lane has loaded them.
#pragma once

#include "bzpf_rowgemm.h"
#include "bzpf_x3.h"

namespace bzpf {

template <int KIN> constexpr int ldx() { return KIN + 8; }

// Part fragments of one row (or weight row): p[part][step].
template <int KIN> struct X3Row {
  bf16x8 p[3][KIN / 32];
};

// Eight consecutive values -> one fragment per part.
__device__ __forceinline__ void split8(f4 a, f4 b, bf16x8& p0, bf16x8& p1, bf16x8& p2) {
  const Pair3 q0 = split3_pair(a[0], a[1]), q1 = split3_pair(a[2], a[3]), q2 = split3_pair(b[0], b[1]),
              q3 = split3_pair(b[2], b[3]);
  p0 = __builtin_bit_cast(bf16x8, uint4{q0.p[0], q1.p[0], q2.p[0], q3.p[0]});
  p1 = __builtin_bit_cast(bf16x8, uint4{q0.p[1], q1.p[1], q2.p[1], q3.p[1]});
  p2 = __builtin_bit_cast(bf16x8, uint4{q0.p[2], q1.p[2], q2.p[2], q3.p[2]});
}

template <int KIN> struct RawRow {
  f4 v[KIN / 16];
  __device__ __forceinline__ void load(const float* p, int g) {
#pragma unroll
    for (int j = 0; j < KIN / 16; j++) v[j] = *reinterpret_cast<const f4*>(p + KIN / 4 * g + 4 * j);
  }
};
template <int KIN>
__device__ __forceinline__ void split_row(X3Row<KIN>& x, const RawRow<KIN>& v) {
#pragma unroll
  for (int s = 0; s < KIN / 32; s++) split8(v.v[2 * s], v.v[2 * s + 1], x.p[0][s], x.p[1][s], x.p[2][s]);
}

template <bool ROWS>
__device__ __forceinline__ f4 mfma_x3(bf16x8 w, bf16x8 x, f4 c) {
  return ROWS ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, w, c, 0, 0, 0)
              : __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, c, 0, 0, 0);
}

// Part pairs (weight, row) of the six products, smallest first: each pair runs over all of K before the next, so the
// small products meet a small accumulator.
constexpr int X3_W[6] = {2, 1, 0, 1, 0, 0}, X3_X[6] = {0, 1, 2, 0, 1, 0};

// acc[rb] += W[0 .. 15][0 : KIN] . X[rb]^T (ROWS: transposed, as in mma_rows) for the 16 weight rows at Ws (plane 0;
// the planes are `plane` elements apart).
template <int RB, bool ROWS, int KIN>
__device__ __forceinline__ void mma_x3(f4 (&acc)[RB], const X3Row<KIN> (&x)[RB], const __bf16* Ws, int plane) {
  const int l = threadIdx.x & 63;
  const __bf16* wp = Ws + (l & 15) * ldx<KIN>() + KIN / 4 * (l >> 4);
  bf16x8 a[3][KIN / 32];
#pragma unroll
  for (int p = 0; p < 3; p++)
#pragma unroll
    for (int s = 0; s < KIN / 32; s++) a[p][s] = *reinterpret_cast<const bf16x8*>(wp + p * plane + 8 * s);
#pragma unroll
  for (int q = 0; q < 6; q++)
#pragma unroll
    for (int s = 0; s < KIN / 32; s++)
#pragma unroll
      for (int rb = 0; rb < RB; rb++) acc[rb] = mfma_x3<ROWS>(a[X3_W[q]][s], x[rb].p[X3_X[q]][s], acc[rb]);
}

// Values without parts. An infinity, and a finite value from 2^128 - 2^119 on (it rounds to a bf16 infinity), splits into
// an infinity and NaNs, and a product within 2^-8 of the largest fp32 value may pass it where its rounded parts meet.
// Each way the sum comes out not finite, so a wave that finds such a sum forms its block again on the fp32 matrix
// instructions, operands straight from memory, and gives what an fp32 product gives: the infinity, the NaN of inf - inf
// or 0 inf, or the finite value. Finite sums pay one v_fma each and a branch.
template <int NV>
__device__ __forceinline__ bool wave_nonfinite(const f4 (&v)[NV]) {
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < NV; i++)
#pragma unroll
    for (int e = 0; e < 4; e++) t = fmaf(v[i][e], 0.f, t);
  return __any(t != t);
}
// acc[rb] = W[0 .. 15][0 : KIN] . X[rb]^T (ROWS: transposed) in fp32: wrow and xrow[rb] are the lane's rows (l % 16) in
// memory.
template <int RB, bool ROWS, int KIN>
__device__ __forceinline__ void mma_f32(f4 (&acc)[RB], const float* wrow, const float* const (&xrow)[RB]) {
  const int c0 = KIN / 4 * ((threadIdx.x & 63) >> 4);
#pragma unroll
  for (int rb = 0; rb < RB; rb++) acc[rb] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int j = 0; j < KIN / 4; j += 4) {
    const f4 a = ld4(wrow + c0 + j);
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
      const f4 b = ld4(xrow[rb] + c0 + j);
#pragma unroll
      for (int t = 0; t < 4; t++)
        acc[rb] = ROWS ? __builtin_amdgcn_mfma_f32_16x16x4f32(b[t], a[t], acc[rb], 0, 0, 0)
                       : __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], b[t], acc[rb], 0, 0, 0);
    }
  }
}
// The same over a row in registers.
template <bool ROWS, int KIN>
__device__ __forceinline__ f4 mma_f32(const float* wrow, const RawRow<KIN>& x) {
  f4 acc = {};
#pragma unroll
  for (int j = 0; j < KIN / 16; j++) {
    const f4 a = ld4(wrow + KIN / 4 * ((threadIdx.x & 63) >> 4) + 4 * j);
#pragma unroll
    for (int t = 0; t < 4; t++)
      acc = ROWS ? __builtin_amdgcn_mfma_f32_16x16x4f32(x.v[j][t], a[t], acc, 0, 0, 0)
                 : __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], x.v[j][t], acc, 0, 0, 0);
  }
  return acc;
}

// Stage ROWS weight rows of KIN fp32 values, split, into LDS planes; row r comes from src(r) (nullptr: zeros). The
// loads of a batch are issued together (a weight block is cold in a CU's caches: one round trip, not one per vector).
template <int NROWS, int KIN, int THREADS, typename RowFn>
__device__ __forceinline__ void stage_x3(__bf16* dst, int plane, RowFn src) {
  constexpr int PER = KIN / 8, ITEMS = (NROWS * PER + THREADS - 1) / THREADS, BATCH = ITEMS < 4 ? ITEMS : 4;
  for (int i0 = 0; i0 < ITEMS; i0 += BATCH) {
    f4 v[BATCH][2];
#pragma unroll
    for (int i = 0; i < BATCH; i++) {
      const int e = (i0 + i) * THREADS + (int)threadIdx.x, r = min(e / PER, NROWS - 1), c = e % PER * 8;
      const float* s = src(r);
      v[i][0] = s != nullptr ? ld4(s + c) : f4{0.f, 0.f, 0.f, 0.f};
      v[i][1] = s != nullptr ? ld4(s + c + 4) : f4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < BATCH; i++) {
      const int e = (i0 + i) * THREADS + (int)threadIdx.x, r = e / PER, c = e % PER * 8;
      if (r >= NROWS) continue;
      bf16x8 p0, p1, p2;
      split8(v[i][0], v[i][1], p0, p1, p2);
      __bf16* d = dst + r * ldx<KIN>() + c;
      *reinterpret_cast<bf16x8*>(d) = p0;
      *reinterpret_cast<bf16x8*>(d + plane) = p1;
      *reinterpret_cast<bf16x8*>(d + 2 * plane) = p2;
    }
  }
}

}  // namespace bzpf
