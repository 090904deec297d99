// Pieces of the backward that its 16-bit kernels (elsa_bwd.hip) and fp32 kernels (elsa_bwd_f32.hip) share.
#pragma once

#include "elsa_bias.h"

namespace elsa {

// LSE2 = m + log2(max(z, 1e-30)) (attention_bwd.py:224), formed in double and split into its fp32
// rounding hi and the remainder lo, so that the fp32 kernels' p = exp2(s*c - LSE2) does not carry
// the half-ulp of a ~15-magnitude LSE2 (3e-7 relative, the same for a whole row) into every
// gradient of that row.  A row with no valid key (z == 0) gets +inf instead of -inf, so that p is 0
// without a test.
__device__ inline void lse2_split(float m, float z, float& hi, float& lo) {
  if (z > 0.f) {
    const double l = (double)m + log2((double)fmaxf(z, 1.0e-30f));
    hi = (float)l;
    lo = (float)(l - (double)hi);
  } else {
    hi = __builtin_huge_valf();
    lo = 0.f;
  }
}

// Stage tile of 32 rows of one operand: three [32][DP] bf16 planes, each row's 16-byte chunks XOR-
// permuted so that row fragments (16 lanes: one chunk of 16 rows) and transposing reads (32 lanes: 64
// bytes of 4 consecutive rows) fall on distinct bank groups: a row is DP / 8 chunks of 4 banks.
template <int DP>
struct X3Stage {
  static constexpr int TT = 32, CPR = DP / 8, PLANE = TT * DP;
  __device__ __host__ static constexpr int swz(int r) {
    return DP == 32 ? (r >> 2) & 3 : (DP == 64 ? lds_swz(r) : ((r & 3) << 2) | ((r >> 2) & 3));
  }
  __device__ static inline int off(int r, int col) { return r * DP + ((((col >> 3) ^ swz(r)) << 3) | (col & 7)); }
};

// Products of this lane with 32-row stage tiles in LDS (X3Stage layout).  fp32 operands are three bf16
// planes (Split3), 16-bit ones a single plane.
template <typename T, int DP>
struct TileLane {
  using S = X3Stage<DP>;
  static constexpr bool F32 = sizeof(T) == 4;
  static constexpr int NP = F32 ? 3 : 1, NKK = DP / 16, NDT = DP / 32;
  typedef typename std::conditional<F32, bf16, T>::type E;            // element of a plane
  typedef typename Mfma<E>::frag F;
  typedef typename std::conditional<F32, Split3, F>::type Own;        // 8 elements of an own operand
  int o_row[NKK], o_tr[NDT][2];
  __device__ inline TileLane(int lane) {
    const int c = lane & 31, g = lane >> 5;
    const int tr_row = 8 * g + ((lane & 15) >> 2), tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) o_row[kk] = S::off(swap23(c), g * 8 + kk * 16);
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int h = 0; h < 2; ++h) o_tr[dt][h] = S::off(tr_row + 4 * h, dt * 32 + tr_col);
  }
  // rows 16 j + 8 g .. + 7 of column 32 dt + (lane % 32) of a plane
  __device__ inline F tr(const E* plane, int j, int dt) const {
    const i16x4 lo = lds_read_tr16(plane + 16 * j * DP + o_tr[dt][0]);
    const i16x4 hi = lds_read_tr16(plane + 16 * j * DP + o_tr[dt][1]);
    const i16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(F, both);
  }
  // (stage rows) x (own rows): D-layout register r of lane (c, g) = stage row key_of_reg(r, g) . own row c
  __device__ inline f32x16 dot(const E* tile, const Own (&own)[NKK]) const {
    f32x16 s = f32x16{};
    if constexpr (F32) {
      bf16x8 h[NKK];
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) {
        h[kk] = *reinterpret_cast<const bf16x8*>(tile + o_row[kk]);
        const bf16x8 m = *reinterpret_cast<const bf16x8*>(tile + S::PLANE + o_row[kk]);
        const bf16x8 l = *reinterpret_cast<const bf16x8*>(tile + 2 * S::PLANE + o_row[kk]);
        s = mma3_small(h[kk], m, l, own[kk], s);
      }
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) s = Mfma<bf16>::mma(h[kk], own[kk].h, s);
    } else {
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) s = Mfma<T>::mma(*reinterpret_cast<const F*>(tile + o_row[kk]), own[kk], s);
    }
    return s;
  }
  // the same with the own operand from own(kk)
  template <typename Get>
  __device__ inline f32x16 dot_with(const E* tile, Get&& own) const {
    f32x16 s = f32x16{};
    if constexpr (F32) {
      bf16x8 h[NKK], oh[NKK];
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) {
        h[kk] = *reinterpret_cast<const bf16x8*>(tile + o_row[kk]);
        const bf16x8 m = *reinterpret_cast<const bf16x8*>(tile + S::PLANE + o_row[kk]);
        const bf16x8 l = *reinterpret_cast<const bf16x8*>(tile + 2 * S::PLANE + o_row[kk]);
        const Split3 o = own(kk);
        oh[kk] = o.h;
        s = mma3_small(h[kk], m, l, o, s);
      }
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) s = Mfma<bf16>::mma(h[kk], oh[kk], s);
    } else {
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) s = Mfma<T>::mma(*reinterpret_cast<const F*>(tile + o_row[kk]), own(kk), s);
    }
    return s;
  }
  // acc[dt] += tile^T w over the stage's 32 rows.  fp32: each stage's product goes into a fresh
  // accumulator first, so that an output is a chain of N/32 adds.
  __device__ inline void add_tr(const E* tile, const Own (&w)[2], f32x16 (&acc)[NDT]) const {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
      if constexpr (F32) {
        f32x16 st = f32x16{};
        bf16x8 h[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          h[j] = tr(tile, j, dt);
          const bf16x8 m = tr(tile + S::PLANE, j, dt), l = tr(tile + 2 * S::PLANE, j, dt);
          st = mma3_small(h[j], m, l, w[j], st);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) st = Mfma<bf16>::mma(h[j], w[j].h, st);
        acc[dt] += st;
      } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[dt] = Mfma<T>::mma(tr(tile, j, dt), w[j], acc[dt]);
      }
    }
  }
  // a D-layout tile as the B operand of add_tr: rounded to T, or split
  __device__ static inline void pack(const f32x16& v, Own (&o)[2]) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if constexpr (F32) {
        float x[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) x[t] = v[j * 8 + t];
        o[j] = split3_reg(x);
      } else {
#pragma unroll
        for (int t = 0; t < 8; ++t) o[j][t] = static_cast<T>(v[j * 8 + t]);
      }
    }
  }
};

// acc of group 1 added into acc of group 0: head dim tiles dt in LDS buffer dt % 2
template <int NDT, int WAVES>
__device__ inline void add_groups(f32x16 (&acc)[NDT], float* b0, float* b1, int grp, int wave, int lane) {
  auto at = [&](int dt, int q4) {
    return reinterpret_cast<f32x4*>(dt & 1 ? b1 : b0) + (((dt >> 1) * 4 + q4) * WAVES + wave) * 64 + lane;
  };
  if (grp == 1) {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        *at(dt, q4) = f32x4{acc[dt][4 * q4], acc[dt][4 * q4 + 1], acc[dt][4 * q4 + 2], acc[dt][4 * q4 + 3]};
  }
  __syncthreads();
  if (grp == 0) {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const f32x4 v = *at(dt, q4);
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[dt][4 * q4 + t] += v[t];
      }
  }
}

// One sum of a split backward's partials (bwd_combine_kernel).
struct CombineOut {
  const float* part;
  void* out;
  int64_t os[3];
  float scale;
};
// one launch for up to three sums (n = 1, 2 or 3 of c[0..2]) into fp32 outputs
// dk/dv of fp16 / bf16 head dims above 64, unbiased (elsa_bwd_d128.hip)
hipError_t launch_dkdv_d128(const BwdParams& p, int dtype, hipStream_t st);
hipError_t combine_launch_f32(const BwdParams& p, const CombineOut* c, int n, hipStream_t st);

}  // namespace elsa
