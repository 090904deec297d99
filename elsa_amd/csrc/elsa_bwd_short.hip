// The whole recompute backward of short sequences (at most 64 rows: attention windows) in one launch.
//
// One workgroup = one (batch, head) at a time: all of q, k, v and dO are staged into LDS once (fp32 as
// three bf16 planes, Split3), with D = rowsum(O * dO) and LSE2 formed on the way, and then waves 0-1
// compute dQ of 32 rows each while waves 2-3 compute dK and dV of 32 keys each.  The separate dq and
// dk/dv kernels read every operand twice and their preprocess dO and O once more; at 49 rows the launches
// and those passes, not the products, are the time.
// Whole fp32 backward, separate kernels -> this: 512 windows x 3 heads, N49 d32, [1, H, N, N] bias 0.068 ->
// 0.049 ms; B256 H12 N64 d64 0.292 -> 0.173; B8 H3 N49 d64 0.028 -> 0.013.
#include "elsa_bwd_common.h"

namespace elsa {

constexpr int kShortRows = 64;

template <typename T, int DP, bool HAS_BIAS, int DS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 && DP == 64 ? 1 : 2, 4)))
void bwd_short_kernel(const BwdParams p, int groups) {
  using L = TileLane<T, DP>;
  using S = X3Stage<DP>;
  typedef typename L::E E;
  typedef typename L::Own Own;
  constexpr int NKK = DP / 16, NDT = DP / 32, NP = L::NP, CPR = S::CPR;
  constexpr int TILE = NP * S::PLANE;                   // one 32-row tile
  constexpr int NCH = kShortRows * CPR / 256;           // 8-element chunks per thread and tensor
  constexpr int BS = kShortRows + 4;                    // bias row stride in LDS
  static_assert(kShortRows * CPR % 256 == 0, "whole chunks per thread");
  __shared__ __attribute__((aligned(16))) E tiles[4][2][TILE];  // q, k, v, dO; rows 0-31 and 32-63
  __shared__ __attribute__((aligned(16))) float rowv[3][kShortRows];  // LSE2, its low part, D
  __shared__ __attribute__((aligned(16))) float bias_s[HAS_BIAS ? kShortRows * BS : 1];

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 31,
            g = lane >> 5;
  const int N = p.N, hi = blockIdx.y, nsub = (N + 31) / 32;
  const L ln(lane);
  const bool keys = wave >= 2;          // waves 2-3: dK and dV
  const int own0 = (wave & 1) * 32;     // this wave's 32 rows or keys
  const bool own_ok = own0 + c < N;
  f32x16 dsum[DS == 2 ? 2 : 1];
#pragma unroll
  for (int i = 0; i < (DS == 2 ? 2 : 1); ++i) dsum[i] = f32x16{};

  for (int bi = blockIdx.x; bi < p.BH / p.H; bi += groups) {
    const int64_t bh = (int64_t)bi * p.H + hi;
    // ---- stage: 8 elements of a row per thread, chunk and tensor; the CPR lanes of a row sum O * dO
    float x[4][NCH][8], o[NCH][8];
    const int64_t* strides[4] = {p.qs, p.ks, p.vs, p.gs};
    const void* bases[4] = {p.q, p.k, p.v, p.dout};
    auto load8 = [&](const void* base, const int64_t* st, int row, int d0, float (&y)[8]) __attribute__((always_inline)) {
      if (row < N && d0 < p.D) {
        const T* src = static_cast<const T*>(base) + bi * st[0] + hi * st[1] + (int64_t)row * st[2] + d0;
        if constexpr (sizeof(T) == 4) {
          const f32x4 a = *reinterpret_cast<const f32x4*>(src), b = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
          for (int t = 0; t < 8; ++t) y[t] = t < 4 ? a[t & 3] : b[t & 3];
        } else {
          const typename Mfma<T>::frag a = *reinterpret_cast<const typename Mfma<T>::frag*>(src);
#pragma unroll
          for (int t = 0; t < 8; ++t) y[t] = static_cast<float>(a[t]);
        }
      } else {
#pragma unroll
        for (int t = 0; t < 8; ++t) y[t] = 0.f;
      }
    };
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int ci = tid + i * 256, row = ci / CPR, d0 = (ci % CPR) * 8;
#pragma unroll
      for (int w = 0; w < 4; ++w) load8(bases[w], strides[w], row, d0, x[w][i]);
      load8(p.out, p.os, row, d0, o[i]);
    }
    float rm = 0.f, rz = 0.f;
    if (tid < N) {
      rm = p.row_m[bh * N + tid];
      rz = p.row_z[bh * N + tid];
    }
    if constexpr (HAS_BIAS) {
      // the bias tile as fp32, a shared one only once
      if (p.bias.sb != 0 || bi == (int)blockIdx.x) {
        for (int i = tid; i < N * N; i += 256) {
          const int r = i / N, k = i - r * N;
          bias_s[r * BS + k] = load_bias_b(p.bias, bi, hi, r, k);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int ci = tid + i * 256, row = ci / CPR, d0 = (ci % CPR) * 8;
      const int lo = (row & 31) * DP + (((d0 >> 3) ^ S::swz(row & 31)) << 3);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        E* dst = tiles[w][row >> 5] + lo;
        if constexpr (sizeof(T) == 4) {
          const Split3 s3 = split3_any(x[w][i]);
          *reinterpret_cast<bf16x8*>(dst) = s3.h;
          *reinterpret_cast<bf16x8*>(dst + S::PLANE) = s3.m;
          *reinterpret_cast<bf16x8*>(dst + 2 * S::PLANE) = s3.l;
        } else {
          typename Mfma<T>::frag f;
#pragma unroll
          for (int t = 0; t < 8; ++t) f[t] = static_cast<T>(x[w][i][t]);
          *reinterpret_cast<typename Mfma<T>::frag*>(dst) = f;
        }
      }
      float acc = 0.f;
#pragma unroll
      for (int t = 0; t < 8; ++t) acc = fmaf(o[i][t], x[3][i][t], acc);
#pragma unroll
      for (int w = 1; w < CPR; w <<= 1) acc += __shfl_xor(acc, w);
      if (ci % CPR == 0) rowv[2][row] = acc;
    }
    if (tid < kShortRows) {  // rows past N: LSE2 = +inf makes their p exactly 0
      float lhi = __builtin_huge_valf(), llo = 0.f;
      if (tid < N) lse2_split(rm, rz, lhi, llo);
      rowv[0][tid] = lhi;
      rowv[1][tid] = sizeof(T) == 4 ? llo : 0.f;  // the 16-bit kernels use the fp32 LSE2 alone
    }
    __syncthreads();

    // own operands of S and dP: this lane's row (or key) own0 + c
    auto own = [&](const E* tile, Own (&f)[NKK]) __attribute__((always_inline)) {
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) {
        const E* src = tile + S::off(c, 16 * kk + 8 * g);
        if constexpr (sizeof(T) == 4) {
          f[kk].h = *reinterpret_cast<const bf16x8*>(src);
          f[kk].m = *reinterpret_cast<const bf16x8*>(src + S::PLANE);
          f[kk].l = *reinterpret_cast<const bf16x8*>(src + 2 * S::PLANE);
        } else {
          f[kk] = *reinterpret_cast<const typename L::F*>(src);
        }
      }
    };
    // store 4 consecutive head dims of this lane's row
    auto put = [&](void* base, const int64_t* st, const f32x16 (&acc)[NDT], float scale) __attribute__((always_inline)) {
      T* dst = static_cast<T*>(base) + bi * st[0] + hi * st[1] + (int64_t)(own0 + c) * st[2];
      typedef T t4 __attribute__((ext_vector_type(4)));
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const int d = dt * 32 + drow(4 * q4, g);
          if (own_ok && d < p.D)
            *reinterpret_cast<t4*>(dst + d) =
                t4{static_cast<T>(acc[dt][4 * q4] * scale), static_cast<T>(acc[dt][4 * q4 + 1] * scale),
                   static_cast<T>(acc[dt][4 * q4 + 2] * scale), static_cast<T>(acc[dt][4 * q4 + 3] * scale)};
        }
    };
    if (own0 < N) {
      Own af[NKK], bf[NKK];
      f32x16 acc0[NDT], acc1[NDT];
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        acc0[dt] = f32x16{};
        acc1[dt] = f32x16{};
      }
      if (!keys) {
        own(tiles[0][wave & 1], af);
        own(tiles[3][wave & 1], bf);
        const float lse = rowv[0][own0 + c], lo = rowv[1][own0 + c], dd = rowv[2][own0 + c];
#pragma unroll 1
        for (int sub = 0; sub < nsub; ++sub) {
          f32x16 s = ln.dot(tiles[1][sub], af);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = sub * 32 + key_of_reg(r, g);
            // s*c - LSE2 with one rounding of the (small) difference, then LSE2's low part
            float y = fmaf(s[r], p.scale_log2, -lse) - lo;
            const bool ok = key < N && (!p.causal || key <= own0 + c);
            if constexpr (HAS_BIAS) y = own_ok && key < N ? fmaf(bias_s[(own0 + c) * BS + key], kLog2e, y) : y;
            s[r] = ok ? fast_exp2(y) : 0.f;
          }
          const f32x16 dp = ln.dot(tiles[2][sub], bf);
#pragma unroll
          for (int r = 0; r < 16; ++r) s[r] *= dp[r] - dd;
          Own w[2];
          ln.pack(s, w);
          ln.add_tr(tiles[1][sub], w, acc0);
        }
        put(p.dq, p.dqs, acc0, p.scale);
      } else {
        own(tiles[1][wave & 1], af);
        own(tiles[2][wave & 1], bf);
        const int key = own0 + c;
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
          if (sub >= nsub) break;
          f32x16 s = ln.dot(tiles[0][sub], af);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int row = sub * 32 + key_of_reg(r, g);
            float y = fmaf(s[r], p.scale_log2, -rowv[0][row]) - rowv[1][row];
            if constexpr (HAS_BIAS) y = own_ok && row < N ? fmaf(bias_s[row * BS + key], kLog2e, y) : y;
            s[r] = own_ok && (!p.causal || row >= key) ? fast_exp2(y) : 0.f;
          }
          Own w[2];
          ln.pack(s, w);
          ln.add_tr(tiles[3][sub], w, acc1);
          const f32x16 dp = ln.dot(tiles[3][sub], bf);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int row = sub * 32 + key_of_reg(r, g);
            s[r] *= dp[r] - rowv[2][row];
            if constexpr (DS == 1) {
              if (own_ok && row < N) p.ds_out[(bh * N + row) * N + key] = s[r];
            }
          }
          if constexpr (DS == 2) dsum[sub] += s;
          ln.pack(s, w);
          ln.add_tr(tiles[0][sub], w, acc0);
        }
        put(p.dk, p.dks, acc0, p.scale);
        put(p.dv, p.dvs, acc1, 1.f);
      }
    }
    __syncthreads();  // the tiles are rewritten for the next (batch, head)
  }
  if constexpr (DS == 2) {
    if (keys && own_ok) {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = sub * 32 + key_of_reg(r, g);
          if (row < N) p.ds_out[(((int64_t)blockIdx.x * p.H + hi) * N + row) * N + own0 + c] = dsum[sub][r];
        }
    }
  }
}

// Head dims above 64 do not fit (fp32 tiles of 64 rows at D = 128: 196 KB of LDS).
bool bwd_short_takes(int dtype, int n, int dp) { return dtype == ELSA_F32 && n <= kShortRows && dp <= 64; }

// Groups of windows (ds_mode 2): 1024 work-groups fill the chip four deep, and no group takes more than
// one window more than another.
int bwd_short_groups(int batch, int heads) {
  const int64_t rounds = ((int64_t)batch * heads + 1023) / 1024;
  return (int)((batch + rounds - 1) / rounds);
}

template <typename T, int DP>
static hipError_t short_launch(const BwdParams& p, int ds_mode, hipStream_t st) {
  const int B = p.BH / p.H, groups = ds_mode == 2 ? bwd_short_groups(B, p.H) : B;
  const dim3 grid(groups, p.H), block(256);
  if (!p.bias.ptr) {
    hipLaunchKernelGGL((bwd_short_kernel<T, DP, false, 0>), grid, block, 0, st, p, groups);
  } else if (ds_mode == 0) {
    hipLaunchKernelGGL((bwd_short_kernel<T, DP, true, 0>), grid, block, 0, st, p, groups);
  } else if (ds_mode == 1) {
    hipLaunchKernelGGL((bwd_short_kernel<T, DP, true, 1>), grid, block, 0, st, p, groups);
  } else {
    hipLaunchKernelGGL((bwd_short_kernel<T, DP, true, 2>), grid, block, 0, st, p, groups);
  }
  return hipGetLastError();
}

template <typename T>
static hipError_t short_launch_d(const BwdParams& p, int ds_mode, hipStream_t st) {
  return pad_head_dim(p.D) == 32 ? short_launch<T, 32>(p, ds_mode, st) : short_launch<T, 64>(p, ds_mode, st);
}

hipError_t launch_bwd_short(const BwdParams& p, int dtype, int ds_mode, hipStream_t st) {
  if (dtype == ELSA_F16) return short_launch_d<f16>(p, ds_mode, st);
  if (dtype == ELSA_BF16) return short_launch_d<bf16>(p, ds_mode, st);
  return short_launch_d<float>(p, ds_mode, st);
}

}  // namespace elsa
