// fp32 backward on gfx950: the recompute backward of elsa_bwd.hip with every fp32 product formed from
// three bf16 parts per operand on the bf16 MFMA (Split3 in elsa_mfma.h).
//
//   dq kernel     per 32-row wave tile, 32-key stages (attention_bwd.py:309-412), after the preprocess
//                 of its rows: D = rowsum(O * dO) and LSE2 (attention_bwd.py:188-224)
//   dk/dv kernel  per 32-key wave tile, 32-row stages (attention_bwd.py:415-527)
//
// The stage tiles are loaded through registers one stage ahead and split by the threads that load them.
// Bound: the matrix cores (72 and 96 MFMAs of 8 passes per 32 x 32 score tile at d64; 96 and 128 of 16
// passes on the fp32 MFMA before).  Whole backward ms, fp32 MFMA kernels -> these (B1 H8 d64 unless noted;
// largest relative gradient error against 64 bits): 16K 16.30 -> 9.08 (2.3e-6 -> 5.6e-7), 4K 1.065 -> 0.606
// (9.2e-7 -> 3.5e-7), 1K 0.102 -> 0.077, B8 H3 N1025 0.307 -> 0.169, B8 H3 N197 0.054 -> 0.040, causal 4K 1.068 ->
// 0.452 and N1025 0.133 -> 0.071 (their stages dealt out in turn, in causal_bwd_order), B1 H16 2K d32 0.318
// -> 0.194, 4K d128 2.237 -> 1.360.  The 4K backward executes 1.0 PFLOP/s of MFMA work.
// A pass that wrote the parts of q, k, v and dO to memory first, so that the kernels could load stages
// straight into LDS, took 0.618 at 4K and needs 24 B per element of workspace.
#include <algorithm>

#include "elsa_bwd_common.h"

namespace elsa {

__device__ inline void load8f(const float* src, bool ok, float (&x)[8]) {
  f32x4 a = f32x4{}, b = f32x4{};
  if (ok) {
    a = *reinterpret_cast<const f32x4*>(src);
    b = *reinterpret_cast<const f32x4*>(src + 4);
  }
#pragma unroll
  for (int t = 0; t < 8; ++t) x[t] = t < 4 ? a[t & 3] : b[t & 3];
}
__device__ inline Split3 split_row8(const float* src, bool ok) {
  float x[8];
  load8f(src, ok, x);
  return split3_any(x);
}

// Rows [t0, t0 + 32) of two operands (row strides sa, sb) on their way into stage tiles: chunk
// tid + i NT of the 2 * TCH 8-element chunks, the first operand's first; rows at or past `rows` and
// head dims at or past D are zeros.
template <int DP, int WAVES>
struct X3Loader {
  using S = X3Stage<DP>;
  static constexpr int NT = 64 * WAVES, TCH = S::TT * S::CPR, NCH = 2 * TCH / NT;
  static_assert((2 * TCH) % NT == 0 && TCH % 64 == 0, "whole chunks per thread, whole waves per operand");
  f32x4 reg[NCH][2];
  __device__ inline void load(const float* a, int64_t sa, const float* b, int64_t sb, int t0, int rows, int D, int tid,
                              int wave) {
    static_for<0, NCH>([&](auto I) {
      constexpr int i = decltype(I)::value;
      const bool second = wave * 64 + i * NT >= TCH;  // wave-uniform
      const int cj = (tid + i * NT) % TCH, r = cj / S::CPR, d0 = (cj % S::CPR) * 8;
      const int64_t st = second ? sb : sa;
      const float* base = (second ? b : a) + (int64_t)t0 * st;
      // row strides are below 2^25 elements: 31 of them fit 32 unsigned bits
      const float* src = base + ((uint32_t)r * (uint32_t)st + (uint32_t)d0);
      reg[i][0] = f32x4{};
      reg[i][1] = f32x4{};
      if (t0 + r < rows && d0 < D) {
        reg[i][0] = *reinterpret_cast<const f32x4*>(src);
        reg[i][1] = *reinterpret_cast<const f32x4*>(src + 4);
      }
    });
  }
  __device__ inline void store(bf16* ta, bf16* tb, int tid, int wave) const {
    split3_all<NCH>(
        [&](auto I, float(&x)[8]) __attribute__((always_inline)) {
          constexpr int i = decltype(I)::value;
#pragma unroll
          for (int t = 0; t < 8; ++t) x[t] = reg[i][t >> 2][t & 3];
        },
        [&](auto I, const Split3& s3) __attribute__((always_inline)) {
          constexpr int i = decltype(I)::value;
          const bool second = wave * 64 + i * NT >= TCH;
          const int cj = (tid + i * NT) % TCH;
          bf16* dst = (second ? tb : ta) + S::off(cj / S::CPR, (cj % S::CPR) * 8);
          *reinterpret_cast<bf16x8*>(dst) = s3.h;
          *reinterpret_cast<bf16x8*>(dst + S::PLANE) = s3.m;
          *reinterpret_cast<bf16x8*>(dst + 2 * S::PLANE) = s3.l;
        });
  }
};

// ------------------------------------------------------------------ dq
template <int DP, int WAVES, bool HAS_BIAS>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(DP >= 128 ? 1 : 2, 2)))
void bwd_dq_x3_kernel(const BwdParams p) {
  using S = X3Stage<DP>;
  constexpr int TT = S::TT, NKK = DP / 16, NDT = DP / 32, BM = 32 * WAVES;
  __shared__ __attribute__((aligned(16))) bf16 Ks[2][3 * S::PLANE], Vs[2][3 * S::PLANE];

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 31,
            g = lane >> 5;
  const WgCoord wg = p.causal ? causal_bwd_order(true, WAVES <= 4 && DP <= 64) : xcd_order();
  const int bh = wg.y;
  const int wg_row0 = wg.x * BM;
  const int wg_last = min(p.N, wg_row0 + BM) - 1;
  const int row0 = wg_row0 + wave * 32, my_row = row0 + c;
  const bool row_ok = my_row < p.N;
  const int bi = bh / p.H, hi = bh % p.H;
  const float* K = static_cast<const float*>(p.k) + bi * p.ks[0] + hi * p.ks[1];
  const float* V = static_cast<const float*>(p.v) + bi * p.vs[0] + hi * p.vs[1];
  const int k_end = p.causal ? wg_last + 1 : p.N;
  // split (bwd_splits; 1 otherwise): over grid z, work-group z takes the key stages z, z + split, ..., so
  // that the ranges differ by at most one stage, under a causal mask too; one without a stage writes zeros
  const int k_lo = wg.z * TT, k_step = p.split * TT;
  X3Loader<DP, WAVES> ld;
  if (k_lo < k_end) ld.load(K, p.ks[2], V, p.vs[2], k_lo, k_end, p.D, tid, wave);

  // this lane's row of Q and dO, and the preprocess of the row: chunk 2 kk + g of O * dO per lane, the
  // two lanes of a row added pairwise, then the chunk pairs.  The work-groups of the first key range store
  // D and LSE2 for the dk/dv kernel, so a whole backward launches no preprocess.
  const int64_t rsafe = row_ok ? my_row : 0;
  const float* Q = static_cast<const float*>(p.q) + bi * p.qs[0] + hi * p.qs[1] + rsafe * p.qs[2];
  const float* dO = static_cast<const float*>(p.dout) + bi * p.gs[0] + hi * p.gs[1] + rsafe * p.gs[2];
  const float* O = static_cast<const float*>(p.out) + bi * p.os[0] + hi * p.os[1] + rsafe * p.os[2];
  Split3 qf[NKK], gf[NKK];
  float pair[NKK];
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk) {
    const int d0 = 16 * kk + 8 * g;
    const bool ok = row_ok && d0 < p.D;
    qf[kk] = split_row8(Q + d0, ok);
    float x[8], o[8], a = 0.f;
    load8f(dO + d0, ok, x);
    load8f(O + d0, ok, o);
#pragma unroll
    for (int t = 0; t < 8; ++t) a = fmaf(o[t], x[t], a);
    pair[kk] = a + __shfl_xor(a, 32);
    gf[kk] = split3_any(x);
  }
#pragma unroll
  for (int w = 1; w < NKK; w <<= 1)
#pragma unroll
    for (int kk = 0; kk < NKK; kk += 2 * w) pair[kk] += pair[kk + w];
  const int64_t ri = (int64_t)bh * p.N + rsafe;
  float lhi, llo;
  lse2_split(p.row_m[ri], p.row_z[ri], lhi, llo);
  if (row_ok && g == 0 && wg.z == 0) {
    p.d_row[ri] = pair[0];
    p.lse_row[ri] = lhi;
    p.lse_lo[ri] = llo;
  }
  // rows without a valid key have LSE2 = +inf: their p is 0 (and so is that of rows past N)
  const float lse = row_ok ? lhi : __builtin_huge_valf();
  const float lse_lo = row_ok ? llo : 0.f;
  const float dd = row_ok ? pair[0] : 0.f;
  const TileLane<float, DP> ln(lane);

  const bool bias_vec = HAS_BIAS && bias_rows_vectorizable(p.bias);
  f32x16 acc[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) acc[dt] = f32x16{};

  auto stage = [&](int t0, const bf16* kt, const bf16* vt) __attribute__((always_inline)) {
    if (p.causal && t0 > row0 + 31) return;  // a causal wave whose rows all precede this stage
    f32x16 s = ln.dot(kt, qf);
    const bool full = (t0 + TT <= k_end) && (!p.causal || t0 + TT - 1 <= row0);
    float bv[HAS_BIAS ? 16 : 1];
    if constexpr (HAS_BIAS)
      bias_keys16(p.bias, bi * p.bias.sb + hi * p.bias.sh + rsafe * p.bias.sq, t0 + 8 * g, k_end, bias_vec, bv);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      // s*c - LSE2 with one rounding of the (small) difference, then LSE2's low part
      float x = fmaf(s[r], p.scale_log2, -lse) - lse_lo;
      if constexpr (HAS_BIAS) x = row_ok ? fmaf(bv[r], kLog2e, x) : x;
      s[r] = fast_exp2(x);
    }
    if (!full) {
      asm volatile("");  // keep this a branch: boundary tiles only
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = t0 + key_of_reg(r, g);
        if (!(key < k_end && (!p.causal || key <= my_row))) s[r] = 0.f;
      }
    }
    const f32x16 dp = ln.dot(vt, gf);
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] *= dp[r] - dd;
    Split3 w[2];
    ln.pack(s, w);
    ln.add_tr(kt, w, acc);
  };
  if (k_lo < k_end) ld.store(Ks[0], Vs[0], tid, wave);
  __syncthreads();
  for (int t0 = k_lo, buf = 0; t0 < k_end; t0 += k_step, buf ^= 1) {
    // buffer buf ^ 1 was last read by the previous stage, before the barrier that ended it
    const bool has_next = t0 + k_step < k_end;
    if (has_next) ld.load(K, p.ks[2], V, p.vs[2], t0 + k_step, k_end, p.D, tid, wave);
    stage(t0, Ks[buf], Vs[buf]);
    if (has_next) ld.store(Ks[buf ^ 1], Vs[buf ^ 1], tid, wave);
    __syncthreads();
  }
  if (!row_ok) return;
  // registers 4q .. 4q + 3 hold head dims dt * 32 + drow(4q, g) .. + 3: one 16-byte store each
  // (pointers are 16-byte aligned and strides multiples of 8 elements; D is a multiple of 8, so a
  // group starting below D ends below it)
  if (p.split > 1) {  // this key range's unscaled dQ: the combine sums the ranges and scales
    float* dst = p.part + (((int64_t)wg.z * p.BH + bh) * p.N + my_row) * p.dp;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        *reinterpret_cast<f32x4*>(dst + dt * 32 + drow(4 * q4, g)) =
            f32x4{acc[dt][4 * q4], acc[dt][4 * q4 + 1], acc[dt][4 * q4 + 2], acc[dt][4 * q4 + 3]};
    return;
  }
  float* out = static_cast<float*>(p.dq) + bi * p.dqs[0] + hi * p.dqs[1] + (int64_t)my_row * p.dqs[2];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int d = dt * 32 + drow(4 * q4, g);
      if (d < p.D)
        *reinterpret_cast<f32x4*>(out + d) = f32x4{acc[dt][4 * q4] * p.scale, acc[dt][4 * q4 + 1] * p.scale,
                                                   acc[dt][4 * q4 + 2] * p.scale, acc[dt][4 * q4 + 3] * p.scale};
    }
}

// ------------------------------------------------------------------ dk / dv
// VLDS: the wave's V parts (the operand of dP) live in LDS instead of registers, in lane order; with them
// in registers the 8-wave kernel at D = 64 spills.  D = 128 has room for one stage buffer beside them.
template <int DP, int WAVES, bool HAS_BIAS, bool VLDS>
__global__ __launch_bounds__(64 * WAVES)
__attribute__((amdgpu_waves_per_eu(DP >= 128 || (DP == 64 && WAVES <= 4) ? 1 : 2, 2)))
void bwd_dkdv_x3_kernel(const BwdParams p) {
  using S = X3Stage<DP>;
  constexpr int TT = S::TT, NKK = DP / 16, NDT = DP / 32, BN = 32 * WAVES;
  constexpr int NBUF = VLDS && DP == 128 ? 1 : 2;
  __shared__ __attribute__((aligned(16))) bf16 Qs[NBUF][3 * S::PLANE], Gs[NBUF][3 * S::PLANE];
  __shared__ __attribute__((aligned(16))) bf16x8 Vown[VLDS ? WAVES * NKK * 3 * 64 : 1];
  __shared__ __attribute__((aligned(16))) float st_s[2][3][TT];  // LSE2, its low part and D of the stage's rows

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 31,
            g = lane >> 5;
  const WgCoord wg = p.causal ? causal_bwd_order(false, WAVES <= 4 && DP == 32) : xcd_order();
  const int bh = wg.y;
  const int wg_key0 = wg.x * BN;
  const int key0 = wg_key0 + wave * 32, my_key = key0 + c;
  const bool key_ok = my_key < p.N;
  const int bi = bh / p.H, hi = bh % p.H;
  const float* Q = static_cast<const float*>(p.q) + bi * p.qs[0] + hi * p.qs[1];
  const float* dO = static_cast<const float*>(p.dout) + bi * p.gs[0] + hi * p.gs[1];
  // split, as in the dq kernel: the row stages z, z + split, ... from the causal key block's first one on
  const int r_lo = (p.causal ? wg_key0 : 0) + wg.z * TT, r_step = p.split * TT;

  float reg[3] = {0.f, 0.f, 0.f};
  auto row_load = [&](int t0) {
    if (tid < TT) {  // rows past N: LSE2 = +inf makes their p exactly 0
      const int64_t ra = (int64_t)bh * p.N + t0 + tid;
      const bool ok = t0 + tid < p.N;
      reg[0] = ok ? p.lse_row[ra] : __builtin_huge_valf();
      reg[1] = ok ? p.lse_lo[ra] : 0.f;
      reg[2] = ok ? p.d_row[ra] : 0.f;
    }
  };
  auto row_store = [&](int buf) {
    if (tid < TT) {
#pragma unroll
      for (int i = 0; i < 3; ++i) st_s[buf][i][tid] = reg[i];
    }
  };
  X3Loader<DP, WAVES> ld;
  if (r_lo < p.N) {
    ld.load(Q, p.qs[2], dO, p.gs[2], r_lo, p.N, p.D, tid, wave);
    row_load(r_lo);
  }

  const int64_t ksafe = key_ok ? my_key : 0;
  const float* K = static_cast<const float*>(p.k) + bi * p.ks[0] + hi * p.ks[1] + ksafe * p.ks[2];
  const float* V = static_cast<const float*>(p.v) + bi * p.vs[0] + hi * p.vs[1] + ksafe * p.vs[2];
  Split3 kf[NKK], vf[VLDS ? 1 : NKK];
  bf16x8* vown = Vown + (VLDS ? wave * NKK * 3 * 64 + lane : 0);
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk) {
    const int d0 = 16 * kk + 8 * g;
    kf[kk] = split_row8(K + d0, key_ok && d0 < p.D);
    const Split3 v3 = split_row8(V + d0, key_ok && d0 < p.D);
    if constexpr (VLDS) {
      vown[(kk * 3 + 0) * 64] = v3.h;
      vown[(kk * 3 + 1) * 64] = v3.m;
      vown[(kk * 3 + 2) * 64] = v3.l;
    } else {
      vf[kk] = v3;
    }
  }
  const TileLane<float, DP> ln(lane);
  f32x16 dk[NDT], dv[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) {
    dk[dt] = f32x16{};
    dv[dt] = f32x16{};
  }

  // four of the stage rows' values: those of this lane's registers 4 q .. 4 q + 3
  auto row_vals = [&](const float* v, int q) __attribute__((always_inline)) {
    return *reinterpret_cast<const f32x4*>(v + 16 * (q >> 1) + 8 * g + 4 * (q & 1));
  };
  auto stage = [&](int buf, int t0, const bf16* qt, const bf16* gt) __attribute__((always_inline)) {
    if (p.causal && t0 + TT - 1 < key0) return;  // a causal wave whose keys all follow this stage's rows
    f32x16 s = ln.dot(qt, kf);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 a = row_vals(st_s[buf][0], q), b = row_vals(st_s[buf][1], q);
      float bv[4];
      if constexpr (HAS_BIAS)
        bias_rows<4>(p.bias, bi * p.bias.sb + hi * p.bias.sh + ksafe * p.bias.sk, t0 + key_of_reg(4 * q, g), p.N, bv);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = 4 * q + t;
        // s*c - LSE2 with one rounding of the (small) difference, then LSE2's low part
        float x = fmaf(s[r], p.scale_log2, -a[t]) - b[t];
        if constexpr (HAS_BIAS) x = key_ok && t0 + key_of_reg(r, g) < p.N ? fmaf(bv[t], kLog2e, x) : x;
        s[r] = fast_exp2(x);
      }
    }
    // keys and rows past N (a row's LSE2 = +inf alone leaves a NaN where the key holds an infinity, times its zeros)
    // and, in a causal call, keys past the row
    if (key0 + 31 >= p.N || t0 + TT > p.N || (p.causal && t0 < key0 + 31)) {
      asm volatile("");  // keep this a branch: boundary tiles only
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = t0 + key_of_reg(r, g);
        if (!(key_ok && row < p.N && (!p.causal || row >= my_key))) s[r] = 0.f;
      }
    }
    Split3 w[2];
    ln.pack(s, w);
    ln.add_tr(gt, w, dv);
    f32x16 dp;
    if constexpr (VLDS) {
      dp = ln.dot_with(gt, [&](int kk) __attribute__((always_inline)) {
        return Split3{vown[(kk * 3 + 0) * 64], vown[(kk * 3 + 1) * 64], vown[(kk * 3 + 2) * 64]};
      });
    } else {
      dp = ln.dot(gt, vf);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 a = row_vals(st_s[buf][2], q);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = 4 * q + t;
        s[r] *= dp[r] - a[t];
        if constexpr (HAS_BIAS) {
          const int row = t0 + key_of_reg(r, g);
          if (p.ds_out != nullptr && key_ok && row < p.N) p.ds_out[((int64_t)bh * p.N + row) * p.N + my_key] = s[r];
        }
      }
    }
    ln.pack(s, w);
    ln.add_tr(qt, w, dk);
  };
  row_store(0);
  if (r_lo < p.N) ld.store(Qs[0], Gs[0], tid, wave);
  __syncthreads();
  for (int t0 = r_lo, buf = 0; t0 < p.N; t0 += r_step, buf ^= 1) {
    const bool has_next = t0 + r_step < p.N;
    if (has_next) {
      ld.load(Q, p.qs[2], dO, p.gs[2], t0 + r_step, p.N, p.D, tid, wave);
      row_load(t0 + r_step);
    }
    stage(buf, t0, Qs[NBUF == 2 ? buf : 0], Gs[NBUF == 2 ? buf : 0]);
    if constexpr (NBUF == 1) __syncthreads();  // every wave has read this stage
    if (has_next) {
      ld.store(Qs[NBUF == 2 ? buf ^ 1 : 0], Gs[NBUF == 2 ? buf ^ 1 : 0], tid, wave);
      row_store(buf ^ 1);
    }
    __syncthreads();
  }
  if (!key_ok) return;
  if (p.split > 1) {  // this row range's unscaled dK and dV: the combine sums the ranges and scales dK
    const int64_t o = (((int64_t)wg.z * p.BH + bh) * p.N + my_key) * p.dp;
    float* dkp = p.part + p.part_stride + o;
    float* dvp = p.part + 2 * p.part_stride + o;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int d = dt * 32 + drow(4 * q4, g);
        *reinterpret_cast<f32x4*>(dkp + d) =
            f32x4{dk[dt][4 * q4], dk[dt][4 * q4 + 1], dk[dt][4 * q4 + 2], dk[dt][4 * q4 + 3]};
        *reinterpret_cast<f32x4*>(dvp + d) =
            f32x4{dv[dt][4 * q4], dv[dt][4 * q4 + 1], dv[dt][4 * q4 + 2], dv[dt][4 * q4 + 3]};
      }
    return;
  }
  float* okp = static_cast<float*>(p.dk) + bi * p.dks[0] + hi * p.dks[1] + (int64_t)my_key * p.dks[2];
  float* ovp = static_cast<float*>(p.dv) + bi * p.dvs[0] + hi * p.dvs[1] + (int64_t)my_key * p.dvs[2];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int d = dt * 32 + drow(4 * q4, g);
      if (d < p.D) {
        *reinterpret_cast<f32x4*>(okp + d) = f32x4{dk[dt][4 * q4] * p.scale, dk[dt][4 * q4 + 1] * p.scale,
                                                   dk[dt][4 * q4 + 2] * p.scale, dk[dt][4 * q4 + 3] * p.scale};
        *reinterpret_cast<f32x4*>(ovp + d) =
            f32x4{dv[dt][4 * q4], dv[dt][4 * q4 + 1], dv[dt][4 * q4 + 2], dv[dt][4 * q4 + 3]};
      }
    }
}

// ------------------------------------------------------------------ launchers
// 8-wave work-groups (256 rows or keys, one per CU) at D = 64 against 4-wave ones: a stage loaded and split
// once serves twice the waves.  dq's 4-wave kernel runs two work-groups per CU (one alone on its CU takes
// about 0.645 of the time of two together), dk/dv's one (its registers); w4, w8: work-groups, the ranges
// of a split included.  dq ms, 4 -> 8 waves: 16K 3.92 -> 3.67, 4K 0.295 -> 0.284, B8 H3 N1025 0.0767 -> 0.0747;
// but N197 (B8 H3) 0.0196 -> 0.0247, B2 H8 N4097 0.73 -> 0.84, and every causal call (whose blocks it
// makes coarser: 4K 0.177 -> 0.209).  dk/dv: 16K 5.96 -> 5.11, 4K 0.428 -> 0.345, 1K 0.0503 -> 0.0428, causal
// N1025 0.0468 -> 0.0418; but N197 0.0232 -> 0.0300, B1 H8 N512 0.0252 -> 0.0301.
static bool dq_wide(const BwdParams& p, int64_t w4, int64_t w8) {
  if (p.causal) return false;
  const int64_t k4 = (w4 + 255) / 256, k8 = (w8 + 255) / 256;
  return 0.94 * (double)k8 < (double)(k4 / 2) + (k4 % 2 ? 0.645 : 0.0);
}
static bool dkdv_wide(const BwdParams& p, int64_t w4, int64_t w8) {
  if (p.causal) return std::max(1.0, (double)w8 / 256) < 0.645 * std::max(1.0, (double)w4 / 256);
  return (double)((w8 + 255) / 256) < 0.645 * (double)((w4 + 255) / 256);
}

template <int DP, bool B>
static hipError_t bwd_f32_b(const BwdParams& p, int stage, hipStream_t st) {
  hipError_t e = hipSuccess;
  const CombineOut all[3] = {
      {p.part, p.dq, {p.dqs[0], p.dqs[1], p.dqs[2]}, p.scale},
      {p.part + p.part_stride, p.dk, {p.dks[0], p.dks[1], p.dks[2]}, p.scale},
      {p.part + 2 * p.part_stride, p.dv, {p.dvs[0], p.dvs[1], p.dvs[2]}, 1.f}};
  // the key (dq) and row (dK/dV) loops split over grid z for under-filled grids
  const unsigned gz = p.split > 1 ? p.split : 1;
  const dim3 g2((p.N + 63) / 64, p.BH, gz), g4((p.N + 127) / 128, p.BH, gz), g8((p.N + 255) / 256, p.BH, gz);
  const int64_t w4 = (int64_t)g4.x * g4.y * g4.z, w8 = (int64_t)g8.x * g8.y * g8.z;
  if (stage < 0 || stage == 1) {
    bool done = false;
    if constexpr (DP == 64) {
      if ((done = p.N > 64 && dq_wide(p, w4, w8)))
        hipLaunchKernelGGL((bwd_dq_x3_kernel<DP, 8, B>), g8, dim3(512), 0, st, p);
    }
    if (!done) {
      if (p.N <= 64) {
        hipLaunchKernelGGL((bwd_dq_x3_kernel<DP, 2, B>), g2, dim3(128), 0, st, p);
      } else {
        hipLaunchKernelGGL((bwd_dq_x3_kernel<DP, 4, B>), g4, dim3(256), 0, st, p);
      }
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (p.split > 1 && stage == 1) return combine_launch_f32(p, all, 1, st);
  }
  if (stage < 0 || stage == 2) {
    bool done = false;
    if constexpr (DP == 64 && !B) {  // with a bias the 8-wave kernel spills
      if ((done = p.N > 64 && dkdv_wide(p, w4, w8)))
        hipLaunchKernelGGL((bwd_dkdv_x3_kernel<DP, 8, B, true>), g8, dim3(512), 0, st, p);
    }
    if (!done) {
      if (p.N <= 64) {
        hipLaunchKernelGGL((bwd_dkdv_x3_kernel<DP, 2, B, DP == 128>), g2, dim3(128), 0, st, p);
      } else {
        hipLaunchKernelGGL((bwd_dkdv_x3_kernel<DP, 4, B, DP == 128>), g4, dim3(256), 0, st, p);
      }
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (p.split > 1 && stage == 2) return combine_launch_f32(p, all + 1, 2, st);
  }
  if (p.split > 1 && stage < 0) e = combine_launch_f32(p, all, 3, st);
  return e;
}

// stages -1, 1 and 2 (the preprocess alone, stage 0, is bwd_pre_kernel)
hipError_t launch_bwd_f32(const BwdParams& p, int stage, hipStream_t st) {
  const bool b = p.bias.ptr != nullptr;
  switch (pad_head_dim(p.D)) {
    case 32: return b ? bwd_f32_b<32, true>(p, stage, st) : bwd_f32_b<32, false>(p, stage, st);
    case 64: return b ? bwd_f32_b<64, true>(p, stage, st) : bwd_f32_b<64, false>(p, stage, st);
    default: return b ? bwd_f32_b<128, true>(p, stage, st) : bwd_f32_b<128, false>(p, stage, st);
  }
}

}  // namespace elsa
