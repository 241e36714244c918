// Triangle multiplication contraction: o[c, i, j] = sum_k a[c, i, k] * b[c, j, k], D independent N x N x N "NT"
// GEMMs on MFMA over the channel-major operands written by the projection (bzpf_pair_gemm.hip), which stores the
// incoming direction's operands transposed so that both directions contract the same way.
// Reference behaviour: boltz_mlx/layers/triangular_mult.py:90-93, 172-175 (per-channel matmul),
// kernels_nax2.py:315-407 (contraction kernel).
// Layout: ab is [2D][N][ld] and o is [D][N][ld] with ld = N rounded up to 64 and zero padding in k >= N, so the
// contraction's k loop and the 64-wide position tiles of proj/tail never straddle a row.
#include "bzpf_common.h"
#include "bzpf_kernels.h"
#include "bzpf_rowgemm.h"
#include "bzpf_x3.h"

namespace bzpf {

// ---------------------------------------------------------------- per-channel contraction, fp32
// o[c][i][j] = sum_{k < kl} a[c][i][k] * b[c][j][k], a = ab[c], b = ab[D + c] (k >= N is zero padding), as split operands
// on the bf16 matrix cores (bzpf_x3.h: three exact bf16 parts a value, six part products, fp32 sums).
// Workgroup: a (32 MB WM) x (32 NB WN) tile (i, j) of one channel, WM x WN waves of MB x NB blocks of 32 x 32. K advances
// KS = 16 per stage: the threads load the next stage's fp32 rows into registers while the current one computes, then
// split them into the three part planes of the other LDS buffer (one barrier a stage: a buffer is written two stages
// after it was last read). A block's lane holds one j and 16 i, so a store covers 128 contiguous bytes of two rows.
// Tiles are ordered (channel, tile) and dealt to the XCDs in contiguous ranges, so one channel's a and b stay in
// one XCD's L2.
// Bound by the matrix cores and the split beside them (a stage of a 64 x 64 wave tile is 768 MFMA cycles and 88 VALU
// instructions): N = 640 382 us (176 TFLOP/s, 0.42 of the bf16 peak in part products), N = 513 260, N = 400 164, against
// 622, 554 and 276 us for the fp32 MFMA kernel this replaces; error against float64 4.1e-7 -> 3.5e-7 (N = 513).
// The stages of bk columns to contract: `all` of them, or those up to the extent the device holds (rounded up to 64
// columns; 0 or >= N: all).
__device__ __forceinline__ int contract_stages(int all, int bk, const int* ext, int64_t N) {
  if (ext == nullptr) return all;
  const int e = __builtin_amdgcn_readfirstlane(*ext);
  return e <= 0 || e >= N ? all : min(all, (e + 63) / 64 * 64 / bk);
}

// ext[0] = 1 + the last column with a nonzero in any row of mask [N][N], ext[1] = 1 + the last row with a nonzero (both 0
// before the launch). A wave takes a row and scans it from its end, so a mask of leading real tokens is read for its
// padded part and one step more. The maxima go out once a workgroup, and only where they raise what is there (an atomic a
// row, all on two words, took 25 us at N = 1000; so 6.7).
__global__ __launch_bounds__(256) void key_extents_k(const float* __restrict__ mask, int64_t N, int* __restrict__ ext) {
  __shared__ int ks[4], rs[4];
  const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  const float* m = mask + min(row, N - 1) * N;
  int kx = 0;
  for (int64_t k0 = (N - 1) / 64 * 64; k0 >= 0 && kx == 0; k0 -= 64) {
    const uint64_t live = __ballot(k0 + l < N && m[min(k0 + l, N - 1)] != 0.0f);
    if (live != 0) kx = (int)(k0 + 64 - __clzll((long long)live));
  }
  if (l == 0) {
    ks[wave] = row < N ? kx : 0;
    rs[wave] = row < N && kx > 0 ? (int)(row + 1) : 0;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    const int* v = threadIdx.x == 0 ? ks : rs;
    const int top = max(max(v[0], v[1]), max(v[2], v[3]));
    if (top > __hip_atomic_load(ext + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(ext + threadIdx.x, top);
  }
}

// Element k of row r of a part plane: rows of KS = 16 values, their two 16-byte halves exchanged in every other group of
// eight rows, so the fragment reads (16 lanes on 16 rows at one half) meet 16 distinct bank groups without padding.
__device__ __forceinline__ int x3_at(int r, int k) { return r * KS + (k ^ (r & 8)); }

template <int WM, int WN, int MB, int NB>
__global__ __launch_bounds__(64 * WM * WN, 2) void trimul_contract_x3_k(const float* __restrict__ ab,
                                                                        float* __restrict__ o, int64_t N, int64_t ld,
                                                                        int D, int tiles_i, int tiles_j, int64_t units,
                                                                        int64_t per_xcd, int nst,
                                                                        const int* __restrict__ ext) {
  nst = contract_stages(nst, KS, ext, N);
  constexpr int BI = 32 * MB * WM, BJ = 32 * NB * WN, T = 64 * WM * WN;
  constexpr int LOADS = (BI + BJ) * (KS / 4) / T;  // 16-byte vectors per thread and stage
  constexpr int ROWS = T / (KS / 4);               // rows a pass of all threads covers
  static_assert((BI + BJ) * (KS / 4) % T == 0 && BI % ROWS == 0, "staging covers whole passes of a, then of b");
  constexpr int PL = (BI + BJ) * KS;               // one part plane: the a rows, then the b rows
  __shared__ LDS_ALIGN __bf16 P[2][3 * PL];

  const int64_t u = (int64_t)(blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (u >= units) return;  // whole workgroup
  const int tiles = tiles_i * tiles_j;
  const int64_t c = u / tiles;
  const int tt = (int)(u - c * tiles);
  const int i0 = (tt / tiles_j) * BI, j0 = (tt % tiles_j) * BJ;
  const float* a = ab + c * N * ld;
  const float* b = ab + ((int64_t)D + c) * N * ld;
  const int t = threadIdx.x, l = t & 63, r32 = l & 31, hl = l >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), wi = wave / WN, wj = wave % WN;

  // vector v of thread t: row v * ROWS + t / 4 of [a rows | b rows] (rows past N repeat the last one; their outputs are
  // not stored), k = 4 (t % 4) of the stage
  const float* src[LOADS];
#pragma unroll
  for (int v = 0; v < LOADS; v++) {
    const int row = v * ROWS + (t >> 2);
    const int64_t g = v * ROWS < BI ? min((int64_t)(i0 + row), N - 1) : min((int64_t)(j0 + row - BI), N - 1);
    src[v] = (v * ROWS < BI ? a : b) + g * ld + 4 * (t & 3);
  }
  f4 reg[LOADS];
  auto gload = [&](int st) {
#pragma unroll
    for (int v = 0; v < LOADS; v++) reg[v] = *reinterpret_cast<const f4*>(src[v] + st * KS);
  };
  f16x acc[MB][NB];
#pragma unroll
  for (int m = 0; m < MB; m++)
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[m][n][e] = 0.f;
  gload(0);
  for (int st = 0; st < nst; st++) {
    __bf16* pl = P[st & 1];
#pragma unroll
    for (int v = 0; v < LOADS; v++) {
      const Pair3 lo = split3_pair(reg[v][0], reg[v][1]), hi = split3_pair(reg[v][2], reg[v][3]);
#pragma unroll
      for (int q = 0; q < 3; q++)
        *reinterpret_cast<uint2*>(pl + q * PL + x3_at(v * ROWS + (t >> 2), 4 * (t & 3))) = uint2{lo.p[q], hi.p[q]};
    }
    __syncthreads();
    if (st + 1 < nst) gload(st + 1);
    bf16x8 fa[MB][3], fb[NB][3];
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
      for (int q = 0; q < 3; q++)
        fa[m][q] = *reinterpret_cast<const bf16x8*>(pl + q * PL + x3_at(32 * (MB * wi + m) + r32, 8 * hl));
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
      for (int q = 0; q < 3; q++)
        fb[n][q] = *reinterpret_cast<const bf16x8*>(pl + q * PL + x3_at(BI + 32 * (NB * wj + n) + r32, 8 * hl));
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
      for (int n = 0; n < NB; n++) acc[m][n] = mfma_parts6(fa[m], fb[n], acc[m][n]);
  }
  // sums that are not finite: the wave's blocks again on the fp32 matrix instructions, rows straight from memory
  // (bzpf_rowgemm_x3.h says which operands lead here)
  float t0 = 0.f;
#pragma unroll
  for (int m = 0; m < MB; m++)
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
      for (int e = 0; e < 16; e++) t0 = fmaf(acc[m][n][e], 0.f, t0);
  const bool again = __any(t0 != t0);
  // acc[m][n][4 q + e] = o[i0 + 32 MB wi + 32 m + 8 q + 4 hl + e][j0 + 32 NB wj + 32 n + r32]
  float* oc = o + c * N * ld;
#pragma unroll
  for (int m = 0; m < MB; m++)
#pragma unroll
    for (int n = 0; n < NB; n++) {
      const int64_t j = j0 + 32 * NB * wj + 32 * n + r32;
      if (again) {
        const float* ar = a + min((int64_t)(i0 + 32 * (MB * wi + m) + r32), N - 1) * ld + 4 * hl;
        const float* br = b + min(j, N - 1) * ld + 4 * hl;
#pragma unroll
        for (int e = 0; e < 16; e++) acc[m][n][e] = 0.f;
#pragma unroll 1
        for (int k0 = 0; k0 < nst * KS; k0 += 8) {
          const f4 va = ld4(ar + k0), vb = ld4(br + k0);
#pragma unroll
          for (int e = 0; e < 4; e++)
            acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[e], vb[e], acc[m][n], 0, 0, 0);
        }
      }
      if (j >= ld) continue;
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int64_t i = i0 + 32 * MB * wi + 32 * m + 8 * q + 4 * hl + e;
          if (i < N) oc[i * ld + j] = acc[m][n][4 * q + e];
        }
    }
}

// fp16 form, persistent and LDS-direct. One 512-thread workgroup per CU walks its tiles (256 x 256 of one channel) as
// one stream of K stages, so the next tile's first stages load while the current tile's last stages compute. A tile
// is 8 waves of 128 (j) x 64 (i) = 4 x 2 blocks of 32 x 32 on v_mfma_f32_32x32x16_f16 (128 accumulator registers per
// lane, 2 waves per SIMD). K stages of BK elements go from memory straight into LDS (buffer_load ... lds: no staging
// registers, no LDS store instructions), NS stages deep. A wave's load instruction fills 1 KB of LDS in lane order,
// so the LDS row layout is fixed; each lane picks its global 16-byte chunk so that LDS chunk p of row R holds the
// row's chunk p ^ swz(R), which makes the fragment reads (16 lanes on 16 rows at one logical chunk) hit distinct
// banks. The fragments of MFMA step g + 1 are read while step g computes (two register sets, across stage
// boundaries too) and the reads are interleaved with the MFMAs. The output tile leaves through a small LDS buffer so
// that each store instruction writes whole 128-byte row segments (scattered 8-byte stores took a third of the time).
// The lane-to-k assignment (lane half h takes k = 32 h + 8 s .. + 7 of a 64-element stage in step s) is the one the
// earlier register-staged kernel used, so the accumulation order, and the result, are unchanged.
// (ct_swz, in bzpf_layout.h: the swizzle of a row, checked on the host for bijectivity and bank conflicts)

template <int BK, int NS>
__global__ __launch_bounds__(512, 1) void trimul_contract_f16_k(const half_t* __restrict__ ab, half_t* __restrict__ o,
                                                                int64_t N, int64_t ld, int D, int64_t tiles1,
                                                                int64_t units, int64_t per_xcd, int wg_per_xcd,
                                                                int nst, const int* __restrict__ ext) {
  nst = contract_stages(nst, BK, ext, N);
  constexpr int BT = 256, NW = 8;
  constexpr int ROWB = BK * 2;               // bytes of a row per stage
  constexpr int CPR = ROWB / 16;             // 16-byte chunks per row
  constexpr int RPI = 1024 / ROWB;           // rows per load instruction
  constexpr int STAGE = 2 * BT * ROWB;       // a rows, then b rows
  constexpr int LPW = 2 * BT / RPI / NW;     // load instructions per wave per stage (first half a, second half b)
  constexpr int STEPS = BK / 16;
  // the stage slots, then one 4 KB output staging buffer per wave (160 KB)
  __shared__ __attribute__((aligned(1024))) char lds[NS * STAGE + NW * 4096];

  // this workgroup's tiles: u = first + wg_per_xcd * k, k < cnt, inside its XCD's contiguous range of units (the
  // XCD's CUs work on consecutive tiles, so one channel's a and b stay in its L2)
  const int xcd = blockIdx.x % 8;
  const int64_t first = (int64_t)xcd * per_xcd + blockIdx.x / 8;
  const int64_t end = min(units, (int64_t)(xcd + 1) * per_xcd);
  if (first >= end) return;
  const int cnt = (int)((end - first + wg_per_xcd - 1) / wg_per_xcd);
  const int total = cnt * nst;

  const int t = threadIdx.x, w = t >> 6, l = t & 63, r = l & 31, h = l >> 5;
  const int wj = w >> 2, wi = w & 3;  // wave tile: j = 128 wj .., i = 64 wi ..
  struct Tile { int64_t c, i0, j0; };
  auto tile = [&](int k) {
    const int64_t u = first + (int64_t)wg_per_xcd * k;
    const int64_t c = u / (tiles1 * tiles1);
    const int64_t tt = u - c * tiles1 * tiles1;
    return Tile{c, (tt / tiles1) * BT, (tt % tiles1) * BT};
  };

  constexpr int RSRC_CFG = 0x00020000;
  const int chan_bytes = (int)contract_extent(N, ld);
  // lane part of every load: row w * RPI + l / CPR of its 8-wave group, logical chunk (l % CPR) ^ swz(row)
  const int lrow = w * RPI + l / CPR;
  const int voff = (int)(((int64_t)lrow * ld + 8 * ((l % CPR) ^ ct_swz<BK>(lrow))) * 2);
  // The row part of the offset rides in the lane offset, which the buffer range check covers: rows past N read as
  // zeros (their outputs are not stored) and nothing is read past the end of a channel. The stage's k rides in the
  // scalar offset. Global stage gs = k * nst + stage; issues past the last one reload it (into a slot never read).
  auto issue = [&](int gs, int slot) {
    gs = min(gs, total - 1);
    const int k = gs / nst, stage = gs - k * nst;
    const Tile tl = tile(k);
    const __amdgpu_buffer_rsrc_t ars =
        __builtin_amdgcn_make_buffer_rsrc((void*)(ab + tl.c * N * ld), 0, chan_bytes, RSRC_CFG);
    const __amdgpu_buffer_rsrc_t brs =
        __builtin_amdgcn_make_buffer_rsrc((void*)(ab + ((int64_t)D + tl.c) * N * ld), 0, chan_bytes, RSRC_CFG);
    char* dst = lds + slot * STAGE + w * 1024;
#pragma unroll
    for (int v = 0; v < LPW; v++) {
      const bool isa = v < LPW / 2;
      const int64_t row0 = (isa ? tl.i0 : tl.j0) + (int64_t)(v % (LPW / 2)) * NW * RPI;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(isa ? ars : brs,
                                               (__attribute__((address_space(3))) void*)(dst + v * NW * 1024), 16,
                                               voff + (int)(row0 * ld * 2), stage * BK * 2, 0, 0);
    }
  };

  f16x acc[4][2];  // acc[jb][ib]: o^T block (j = 128 wj + 32 jb .., i = 64 wi + 32 ib ..)
  auto zero = [&]() {
#pragma unroll
    for (int jb = 0; jb < 4; jb++)
#pragma unroll
      for (int ib = 0; ib < 2; ib++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[jb][ib][e] = 0.0f;
  };
  // acc[jb][ib][4 q + e] = o[i = i0 + 64 wi + 32 ib + r][j = j0 + 128 wj + 32 jb + 8 q + 4 h + e]
  // Stores through a wave-private LDS buffer: each 32 (i) x 64 (j) piece of the wave's tile is written in the
  // accumulator layout (16-byte chunks XOR-swizzled by row) and read back as 16 bytes of one row per lane, so a
  // store instruction covers 8 rows x 128 contiguous bytes rather than 32 rows x 16 bytes.
  char* ob = lds + NS * STAGE + w * 4096;
  auto store = [&](int k) {
    const Tile tl = tile(k);
    half_t* oc = o + tl.c * N * ld;
#pragma unroll
    for (int ib = 0; ib < 2; ib++)
#pragma unroll
      for (int jp = 0; jp < 2; jp++) {
#pragma unroll
        for (int jj = 0; jj < 2; jj++)
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const f16x& v = acc[2 * jp + jj][ib];
            *reinterpret_cast<half4*>(ob + r * 128 + (((4 * jj + q) ^ (r & 7)) * 16) + 8 * h) =
                half4{(half_t)v[4 * q], (half_t)v[4 * q + 1], (half_t)v[4 * q + 2], (half_t)v[4 * q + 3]};
          }
#pragma unroll
        for (int rr = 0; rr < 4; rr++) {
          const int R = (l >> 3) + 8 * rr;
          const u32x4_t val = *reinterpret_cast<const u32x4_t*>(ob + R * 128 + (((l & 7) ^ (R & 7)) * 16));
          const int64_t i = tl.i0 + 64 * wi + 32 * ib + R;
          const int64_t j = tl.j0 + 128 * wj + 64 * jp + 8 * (l & 7);
          if (i < N && j < ld) *reinterpret_cast<u32x4_t*>(oc + i * ld + j) = val;
        }
      }
  };
  zero();
  const int sw = ct_swz<BK>(r);  // rows read by this lane: (block base, a multiple of 32) + r
  // fragment sets: the reads of MFMA step g + 1 are issued before the MFMAs of step g (two register sets), across
  // stage boundaries too, so each wave's own MFMAs cover its LDS latency and the barrier
  half8 fa[2][4], fb[2][2];
  auto read = [&](int set, int slot, int s) {
    const char* base = lds + slot * STAGE;
    const int chunk = (STEPS * h + s) ^ sw;
#pragma unroll
    for (int jb = 0; jb < 4; jb++)
      fa[set][jb] = *reinterpret_cast<const half8*>(base + (BT + 128 * wj + 32 * jb + r) * ROWB + 16 * chunk);
#pragma unroll
    for (int ib = 0; ib < 2; ib++)
      fb[set][ib] = *reinterpret_cast<const half8*>(base + (64 * wi + 32 * ib + r) * ROWB + 16 * chunk);
  };
  auto mfma = [&](int set) {
#pragma unroll
    for (int jb = 0; jb < 4; jb++)
#pragma unroll
      for (int ib = 0; ib < 2; ib++)
        acc[jb][ib] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[set][jb], fb[set][ib], acc[jb][ib], 0, 0, 0);
  };
  // stages gs + 1 .. gs + NS - 1 are in flight while stage gs computes, so every wave always has (NS - 2) * LPW
  // loads younger than the stage it waits for
  constexpr int YOUNGER = (NS - 2) * LPW;
  constexpr int WAIT = (YOUNGER & 15) | ((YOUNGER >> 4) << 14) | (0x7 << 4) | (0xF << 8);  // vmcnt only
#pragma unroll
  for (int p = 0; p < NS - 1; p++) issue(p, p);
  __builtin_amdgcn_s_waitcnt(WAIT);  // stage 0 has landed (this wave's part)
  __builtin_amdgcn_s_barrier();      // (everyone's)
  __builtin_amdgcn_sched_barrier(0);
  issue(NS - 1, NS - 1);
  read(0, 0, 0);
  int stage = 0, k = 0;
  for (int gs = 0; gs < total; gs++) {
    const int slot = gs % NS;
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
      const int cur = s & 1;  // STEPS is even: step 0 of every stage uses set 0
      if (s + 1 < STEPS) {
        read(cur ^ 1, slot, s + 1);
      } else if (gs + 1 < total) {
        // every read of this slot by this wave is done (the last set is in registers) and stage gs + 1 has landed;
        // after the barrier the slot takes stage gs + NS
        __builtin_amdgcn_s_waitcnt(WAIT & ~(0xF << 8));  // vmcnt as above, lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        issue(gs + NS, slot);
        read(cur ^ 1, (gs + 1) % NS, 0);
      }
      mfma(cur);
      // interleave: the next set's LDS reads between this set's MFMAs
#pragma unroll
      for (int q = 0; q < 6; q++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    }
    if (++stage == nst) {  // tile k done: its stores drain while the next tile computes
      store(k);
      zero();
      stage = 0;
      k++;
    }
  }
  __builtin_amdgcn_s_waitcnt(0);  // no LDS write of a trailing (unused) stage load outlives the workgroup
}

// kl: the k range contracted (a multiple of 64, <= ld); columns past it are zero in a and b.
static hipError_t contract_f16(const half_t* ab, half_t* o, int64_t N, int64_t ld, int64_t kl, const int* ext, int D,
                               hipStream_t st) {
  const int64_t tiles1 = (N + 255) / 256, units = (int64_t)D * tiles1 * tiles1, per_xcd = (units + 7) / 8;
  static int cache[kMaxDevices] = {};
  const int resident = resident_grid(trimul_contract_f16_k<64, 2>, 512, cache);
  if (resident < 8) return hipErrorInvalidConfiguration;
  const int wpx = (int)(resident / 8 < per_xcd ? resident / 8 : per_xcd);
  trimul_contract_f16_k<64, 2>
      <<<dim3(8 * wpx), 512, 0, st>>>(ab, o, N, ld, D, tiles1, units, per_xcd, wpx, (int)(kl / 64),
                                       ext);
  return hipGetLastError();
}

template <int WM, int WN, int MB, int NB>
static hipError_t contract_x3(const float* ab, float* o, int64_t N, int64_t ld, int64_t kl, const int* ext, int D,
                              hipStream_t st) {
  constexpr int BI = 32 * MB * WM, BJ = 32 * NB * WN;
  const int64_t ti = (N + BI - 1) / BI, tj = (N + BJ - 1) / BJ, units = (int64_t)D * ti * tj, per_xcd = (units + 7) / 8;
  trimul_contract_x3_k<WM, WN, MB, NB><<<dim3((unsigned)(per_xcd * 8)), 64 * WM * WN, 0, st>>>(
      ab, o, N, ld, D, (int)ti, (int)tj, units, per_xcd, (int)(kl / KS), ext);
  return hipGetLastError();
}

// 192 x 192 tiles (3 x 3 blocks a wave: half again the products per LDS read of 2 x 2) where their padded area is at most 8/7
// of that of 128 x 128 tiles: per padded output they take 0.85 to 0.96 of the time (us, 192 / 128 wide: N = 513 276 / 359 at
// 0.81 times the area; N = 333, equal areas, 79 / 93; N = 400, 1.27 times the area, 226 / 186; N = 640, 1.44 times, 502 / 402).
static hipError_t contract_f32(const float* ab, float* o, int64_t N, int64_t ld, int64_t kl, const int* ext, int D,
                               hipStream_t st) {
  const int64_t t128 = (N + 127) / 128 * 128, t192 = (N + 191) / 192 * 192;
  return 7 * t192 * t192 <= 8 * t128 * t128 ? contract_x3<2, 2, 3, 3>(ab, o, N, ld, kl, ext, D, st)
                                            : contract_x3<2, 2, 2, 2>(ab, o, N, ld, kl, ext, D, st);
}

hipError_t launch_trimul_contract(const void* ab, void* o, int dt, int64_t N, int64_t ld, int64_t k_len, const int* ext,
                                  int D, hipStream_t st) {
  if (dt == DT_F16 && !contract_shape_ok(N, ld)) return hipErrorInvalidValue;  // 32-bit buffer offsets per channel
  // contract over k < k_len rounded up to 64 (a whole number of stages of either kernel); 0 or >= N: every k
  const int64_t kl = k_len <= 0 || k_len >= N ? ld : (k_len + 63) / 64 * 64;
  return dt == DT_F16 ? contract_f16(static_cast<const half_t*>(ab), static_cast<half_t*>(o), N, ld, kl, ext, D, st)
                      : contract_f32(static_cast<const float*>(ab), static_cast<float*>(o), N, ld, kl, ext, D, st);
}

hipError_t launch_key_extents(const float* mask, int64_t N, int* ext, hipStream_t st) {
  if (N < 1 || (N + 3) / 4 > INT32_MAX) return hipErrorInvalidValue;
  key_extents_k<<<(unsigned)((N + 3) / 4), 256, 0, st>>>(mask, N, ext);
  return hipGetLastError();
}

}  // namespace bzpf
