// fp16 / bf16 dk and dv at head dims above 64, without a bias (attention_bwd.py:415-527).
//
// One workgroup = 128 keys of one head in two groups of 4 waves: wave w of both groups owns the keys 32 w ..
// + 31, and group g takes the 32-row stages g, g + 2, ...; group 1 hands its sums to group 0 through LDS at
// the end.  The keys' K and V fragments, 64 registers per lane, live in LDS, in lane order and once for both
// groups, so that the 128 accumulator registers leave room for two waves per SIMD.  Stage tiles go straight
// from global memory into LDS (buffer_load_dwordx4 ... lds, one stage ahead), 16-byte chunks permuted as in
// X3Stage.
// Bound: the matrix cores (32 MFMAs and 48 KB of LDS reads per 32 x 32 score tile).  The 4-wave kernel with the
// operands in registers (449 of them) ran one wave per SIMD, with nothing beside its MFMAs while it waited
// or formed p.  dk/dv ms, fp16 d128, that kernel -> this: B1 H8 16K 2.68 -> 2.06 (1.07 PFLOP/s), 4K 0.177 -> 0.141,
// B2 H8 2K 0.107 -> 0.083, B1 H4 N1000 0.056 -> 0.043, causal 8K 0.457 -> 0.280, d80 B8 H12 N577 0.074 -> 0.060.
#include "elsa_bwd_common.h"

namespace elsa {

template <typename T>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void bwd_dkdv_d128_kernel(const BwdParams p) {
  constexpr int DP = 128, WAVES = 4;
  using L = TileLane<T, DP>;
  using S = X3Stage<DP>;
  typedef typename L::F F;
  constexpr int TT = S::TT, NKK = L::NKK, NDT = L::NDT;
  // one array per buffer, so that the compiler sees the loads into one leave the other's reads alone
  __shared__ __attribute__((aligned(16))) T Qa[2][S::PLANE], Ga[2][S::PLANE], Qb[2][S::PLANE], Gb[2][S::PLANE];
  __shared__ __attribute__((aligned(16))) F Kown[WAVES * NKK * 64], Vown[WAVES * NKK * 64];
  __shared__ __attribute__((aligned(16))) float lse_s[2][2][TT], d_s[2][2][TT];  // [group][buffer]

  const int grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8), tid = threadIdx.x & 255;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 31, g = lane >> 5;
  const WgCoord wg = p.causal ? causal_bwd_order(false, false) : xcd_order();
  const int bh = wg.y;
  const int wg_key0 = wg.x * 32 * WAVES;
  const int key0 = wg_key0 + wave * 32, my_key = key0 + c;
  const bool key_ok = my_key < p.N;
  const int bi = bh / p.H, hi = bh % p.H;
  const T* Q = static_cast<const T*>(p.q) + bi * p.qs[0] + hi * p.qs[1];
  const T* dO = static_cast<const T*>(p.dout) + bi * p.gs[0] + hi * p.gs[1];

  // stage loads: load j of a wave fills 1 KB of each tile, rows 4 (wave + 4 j) .. + 3; lane l its row's slot
  // l % 16, which holds chunk (l % 16) ^ swz(row).  Rows past N (the buffer range ends there; the launcher
  // checks that it is below 2^31 bytes) and head dims past D read as zeros.
  const uint32_t qrb = (uint32_t)p.qs[2] * 2u, grb = (uint32_t)p.gs[2] * 2u;
  const auto rq = make_rsrc(Q, (uint32_t)p.N * qrb);
  const auto rg = make_rsrc(dO, (uint32_t)p.N * grb);
  uint32_t ldq[2], ldg[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = 4 * (wave + 4 * j) + (lane >> 4), ch = (lane & 15) ^ S::swz(r);
    ldq[j] = ch * 8 < p.D ? (uint32_t)r * qrb + (uint32_t)ch * 16u : kBufferOff;
    ldg[j] = ch * 8 < p.D ? (uint32_t)r * grb + (uint32_t)ch * 16u : kBufferOff;
  }
  float lreg = 0.f, dreg = 0.f;
  auto load = [&](int t0, T* qt, T* gt) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      buffer_load16_lds(rq, qt + 64 * (wave + 4 * j) * 8, ldq[j] + (uint32_t)t0 * qrb);
      buffer_load16_lds(rg, gt + 64 * (wave + 4 * j) * 8, ldg[j] + (uint32_t)t0 * grb);
    }
    if (tid < TT) {  // rows past N: LSE2 = +inf makes their p exactly 0
      const int ra = t0 + tid;
      lreg = ra < p.N ? p.lse_row[(int64_t)bh * p.N + ra] : __builtin_huge_valf();
      dreg = ra < p.N ? p.d_row[(int64_t)bh * p.N + ra] : 0.f;
    }
  };
  auto row_store = [&](int buf) __attribute__((always_inline)) {
    if (tid < TT) {
      lse_s[grp][buf][tid] = lreg;
      d_s[grp][buf][tid] = dreg;
    }
  };
  const int r0 = p.causal ? wg_key0 : 0, r_lo = r0 + grp * TT, step = 2 * TT;  // this group's stages
  if (r_lo < p.N) load(r_lo, Qa[grp], Ga[grp]);

  // the keys' operands: group 0 brings K, group 1 V
  F* kown = Kown + wave * NKK * 64 + lane;
  F* vown = Vown + wave * NKK * 64 + lane;
  {
    const T* src = grp == 0 ? static_cast<const T*>(p.k) + bi * p.ks[0] + hi * p.ks[1] + (int64_t)(key_ok ? my_key : 0) * p.ks[2]
                            : static_cast<const T*>(p.v) + bi * p.vs[0] + hi * p.vs[1] + (int64_t)(key_ok ? my_key : 0) * p.vs[2];
    F* dst = grp == 0 ? kown : vown;
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      const int d0 = kk * 16 + g * 8;
      dst[kk * 64] = load_frag<T>(src + d0, key_ok && d0 < p.D);
    }
  }
  const L ln(lane);
  f32x16 dk[NDT], dv[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) {
    dk[dt] = f32x16{};
    dv[dt] = f32x16{};
  }
  auto stage = [&](int buf, int t0, const T* qt, const T* gt) __attribute__((always_inline)) {
    if (p.causal && t0 + TT - 1 < key0) return;  // a causal wave whose keys all follow this stage's rows
    f32x16 s = ln.dot_with(qt, [&](int kk) __attribute__((always_inline)) { return kown[kk * 64]; });
#pragma unroll
    for (int q = 0; q < 4; ++q) {  // registers 4 q .. + 3: rows 16 (q / 2) + 8 g + 4 (q % 2) .. + 3
      const f32x4 l4 = *reinterpret_cast<const f32x4*>(&lse_s[grp][buf][16 * (q >> 1) + 8 * g + 4 * (q & 1)]);
#pragma unroll
      for (int t = 0; t < 4; ++t) s[4 * q + t] = fast_exp2(fmaf(s[4 * q + t], p.scale_log2, -l4[t]));
    }
    // rows past N too: their LSE2 = +inf alone leaves a NaN where the key holds an infinity, times their zeros
    if (key0 + 31 >= p.N || t0 + TT > p.N || (p.causal && t0 < key0 + 31)) {
      asm volatile("");  // keep this a branch: boundary tiles only
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = t0 + key_of_reg(r, g);
        if (!(key_ok && row < p.N && (!p.causal || row >= my_key))) s[r] = 0.f;
      }
    }
    F w[2];
    L::pack(s, w);
    ln.add_tr(gt, w, dv);
    const f32x16 dp = ln.dot_with(gt, [&](int kk) __attribute__((always_inline)) { return vown[kk * 64]; });
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 d4 = *reinterpret_cast<const f32x4*>(&d_s[grp][buf][16 * (q >> 1) + 8 * g + 4 * (q & 1)]);
#pragma unroll
      for (int t = 0; t < 4; ++t) s[4 * q + t] *= dp[4 * q + t] - d4[t];
    }
    L::pack(s, w);
    ln.add_tr(qt, w, dk);
  };
  row_store(0);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  // group 0's stages are the most: both groups run its count, so that every wave meets every barrier
  const int nloop = p.N > r0 ? (p.N - r0 + step - 1) / step : 0;
  for (int it = 0; it < nloop; it += 2) {
    const int t0 = r_lo + it * step, t1 = t0 + step, t2 = t1 + step;
    if (t1 < p.N) load(t1, Qb[grp], Gb[grp]);
    if (t0 < p.N) stage(0, t0, Qa[grp], Ga[grp]);
    if (t1 < p.N) row_store(1);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (it + 1 < nloop) {
      if (t2 < p.N) load(t2, Qa[grp], Ga[grp]);
      if (t1 < p.N) stage(1, t1, Qb[grp], Gb[grp]);
      if (t2 < p.N) row_store(0);
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
    }
  }
  // group 1's sums through the stage buffers (free after the last barrier): 64 KB, dk and then dv
  static_assert(sizeof(Qa) == 4 * WAVES * 64 * 16, "one head dim tile of 4 waves per buffer");
  float* red[4] = {reinterpret_cast<float*>(Qa), reinterpret_cast<float*>(Ga), reinterpret_cast<float*>(Qb),
                   reinterpret_cast<float*>(Gb)};
  auto exchange = [&](f32x16(&acc)[NDT]) __attribute__((always_inline)) {
    if (grp == 1) {
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4)
          reinterpret_cast<f32x4*>(red[dt])[(q4 * WAVES + wave) * 64 + lane] =
              f32x4{acc[dt][4 * q4], acc[dt][4 * q4 + 1], acc[dt][4 * q4 + 2], acc[dt][4 * q4 + 3]};
    }
    __syncthreads();
    if (grp == 0) {
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const f32x4 v = reinterpret_cast<const f32x4*>(red[dt])[(q4 * WAVES + wave) * 64 + lane];
#pragma unroll
          for (int t = 0; t < 4; ++t) acc[dt][4 * q4 + t] += v[t];
        }
    }
    __syncthreads();
  };
  exchange(dk);
  exchange(dv);
  if (grp == 1 || !key_ok) return;
  T* okp = static_cast<T*>(p.dk) + bi * p.dks[0] + hi * p.dks[1] + (int64_t)my_key * p.dks[2];
  T* ovp = static_cast<T*>(p.dv) + bi * p.dvs[0] + hi * p.dvs[1] + (int64_t)my_key * p.dvs[2];
  typedef T t4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int d = dt * 32 + drow(4 * q4, g);
      if (d < p.D) {
        *reinterpret_cast<t4*>(okp + d) =
            t4{static_cast<T>(dk[dt][4 * q4] * p.scale), static_cast<T>(dk[dt][4 * q4 + 1] * p.scale),
               static_cast<T>(dk[dt][4 * q4 + 2] * p.scale), static_cast<T>(dk[dt][4 * q4 + 3] * p.scale)};
        *reinterpret_cast<t4*>(ovp + d) = t4{static_cast<T>(dv[dt][4 * q4]), static_cast<T>(dv[dt][4 * q4 + 1]),
                                             static_cast<T>(dv[dt][4 * q4 + 2]), static_cast<T>(dv[dt][4 * q4 + 3])};
      }
    }
}

hipError_t launch_dkdv_d128(const BwdParams& p, int dtype, hipStream_t st) {
  const dim3 grid((p.N + 127) / 128, p.BH), block(512);
  if (dtype == ELSA_F16) {
    hipLaunchKernelGGL(bwd_dkdv_d128_kernel<f16>, grid, block, 0, st, p);
  } else {
    hipLaunchKernelGGL(bwd_dkdv_d128_kernel<bf16>, grid, block, 0, st, p);
  }
  return hipGetLastError();
}

}  // namespace elsa
