// The whole recompute backward of short sequences (at most 64 rows: attention windows) in one launch.
//
// One workgroup = one (batch, head) at a time: all of q, k, v and dO are staged into LDS once (fp32 as
// three bf16 planes, Split3), with D = rowsum(O * dO) and LSE2 formed on the way, and then waves 0-1
// compute dQ of 32 rows each while waves 2-3 compute dK and dV of 32 keys each.  The separate dq and
// dk/dv kernels read every operand twice and their preprocess dO and O once more; at 49 rows the launches
// and those passes, not the products, are the time.
// Bound: latency and memory (512 windows x 3 heads, N49 d32: 38 MB, 8 us of a large copy).  Whole backward
// ms, separate kernels -> this: fp16 512 windows x 3 heads, N49 d32, with the gradient of a [1, H, N, N] bias
// 0.0435 -> 0.0223, of a [B, H, N, N] one 0.0481 -> 0.0238, without bias 0.0271 -> 0.0138; B256 H12 N64 d64
// 0.186 -> 0.048, B8 H3 N49 d64 0.0126 -> 0.0076; fp32 the same windows 0.066 -> 0.045, 0.075 -> 0.046 and
// 0.054 -> 0.027, B256 H12 N64 d64 0.293 -> 0.169, B8 H3 N49 d64 0.028 -> 0.012.
#include "elsa_bwd_common.h"

namespace elsa {

constexpr int kShortRows = 64;

template <typename T, int DP, bool HAS_BIAS, int DS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? (DP == 64 ? 1 : 2) : (DP == 64 ? 2 : 3), 4)))
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

  const int N = p.N, hi = blockIdx.y, nsub = (N + 31) / 32;
  f32x16 dsum[DS == 2 ? 2 : 1];
#pragma unroll
  for (int i = 0; i < (DS == 2 ? 2 : 1); ++i) dsum[i] = f32x16{};

  for (int bi = blockIdx.x; bi < p.BH / p.H; bi += groups) {
    int tid = threadIdx.x;
    // nothing that depends on the lane is kept from one window to the next: those values filled 100
    // registers (217 VGPRs against 168 with them formed again, fp16 D = 32)
    if constexpr (DS == 2) asm volatile("" : "+v"(tid));
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 31, g = lane >> 5;
    const L ln(lane);
    const bool keys = wave >= 2;          // waves 2-3: dK and dV
    const int own0 = (wave & 1) * 32;     // this wave's 32 rows or keys
    const bool own_ok = own0 + c < N;
    const int64_t bh = (int64_t)bi * p.H + hi;
    // ---- stage: 8 elements of a row per thread, chunk and tensor; the CPR lanes of a row sum O * dO
    typedef typename Mfma<E>::frag F8;
    constexpr int NR = sizeof(T) == 4 ? 2 : 1;  // 16-byte loads per chunk
    Chunk16 x[5][NCH][NR];
    const int64_t* strides[5] = {p.qs, p.ks, p.vs, p.gs, p.os};
    const void* bases[5] = {p.q, p.k, p.v, p.dout, p.out};
#pragma unroll
    for (int w = 0; w < 5; ++w) {
      const T* base = static_cast<const T*>(bases[w]) + bi * strides[w][0] + hi * strides[w][1];
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const int ci = tid + i * 256, row = ci / CPR, d0 = (ci % CPR) * 8;
        // rows past N and head dims past D load an element in range and take zeros: no branch, so that all
        // loads are in flight together (row strides are below 2^25 elements: 63 of them fit 32 unsigned bits)
        const bool ok = row < N && d0 < p.D;
        const T* src = base + (ok ? (uint32_t)row * (uint32_t)strides[w][2] + (uint32_t)d0 : 0u);
#pragma unroll
        for (int u = 0; u < NR; ++u) {
          const Chunk16 v = reinterpret_cast<const Chunk16*>(src)[u];
          x[w][i][u] = ok ? v : Chunk16{};
        }
      }
    }
    float rm = 0.f, rz = 0.f;
    if (tid < N) {
      rm = p.row_m[bh * N + tid];
      rz = p.row_z[bh * N + tid];
    }
    if constexpr (HAS_BIAS) {
      // the bias tile as fp32, a shared one only once: a wave reads rows wave, wave + 4, ...
      if (p.bias.sb != 0 || bi == (int)blockIdx.x) {
#pragma unroll 8
        for (int r = wave; r < N; r += 4)
          if (lane < N) bias_s[r * BS + lane] = load_bias(p.bias, bi, hi, r, lane);
      }
    }
    // q, k, v and dO into their tiles
    auto tile_at = [&](int w, int i) __attribute__((always_inline)) -> E* {
      const int ci = tid + i * 256, row = ci / CPR, d0 = (ci % CPR) * 8;
      return tiles[w][row >> 5] + (row & 31) * DP + (((d0 >> 3) ^ S::swz(row & 31)) << 3);
    };
    if constexpr (sizeof(T) == 4) {
      split3_all<4 * NCH>(
          [&](auto I, float(&y)[8]) __attribute__((always_inline)) {
            constexpr int w = decltype(I)::value / NCH, i = decltype(I)::value % NCH;
#pragma unroll
            for (int t = 0; t < 8; ++t) y[t] = __uint_as_float(x[w][i][t >> 2][t & 3]);
          },
          [&](auto I, const Split3& s3) __attribute__((always_inline)) {
            E* dst = tile_at(decltype(I)::value / NCH, decltype(I)::value % NCH);
            *reinterpret_cast<bf16x8*>(dst) = s3.h;
            *reinterpret_cast<bf16x8*>(dst + S::PLANE) = s3.m;
            *reinterpret_cast<bf16x8*>(dst + 2 * S::PLANE) = s3.l;
          });
    } else {
#pragma unroll
      for (int i = 0; i < NCH; ++i)
#pragma unroll
        for (int w = 0; w < 4; ++w) *reinterpret_cast<Chunk16*>(tile_at(w, i)) = x[w][i][0];
    }
    // D of a row: O * dO over its CPR lanes
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int ci = tid + i * 256, row = ci / CPR;
      float acc = 0.f;
      if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int t = 0; t < 8; ++t)
          acc = fmaf(__uint_as_float(x[4][i][t >> 2][t & 3]), __uint_as_float(x[3][i][t >> 2][t & 3]), acc);
      } else {
        const F8 go = __builtin_bit_cast(F8, x[3][i][0]), oo = __builtin_bit_cast(F8, x[4][i][0]);
#pragma unroll
        for (int t = 0; t < 8; ++t) acc = fmaf(static_cast<float>(oo[t]), static_cast<float>(go[t]), acc);
      }
#pragma unroll
      for (int w = 1; w < CPR; w <<= 1) acc += __shfl_xor(acc, w);
      if (ci % CPR == 0) rowv[2][row] = acc;
    }
    if (tid < kShortRows) {  // rows past N: LSE2 = +inf makes their p exactly 0
      float lhi = __builtin_huge_valf(), llo = 0.f;
      if (tid < N) lse2_split(rm, rz, lhi, llo);
      rowv[0][tid] = lhi;
      if constexpr (sizeof(T) == 4) rowv[1][tid] = llo;  // the 16-bit kernels use the fp32 LSE2 alone
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
            float y = fmaf(s[r], p.scale_log2, -lse);
            if constexpr (sizeof(T) == 4) y -= lo;
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
        float* dso = DS == 1 ? p.ds_out + bh * N * N : nullptr;
#pragma unroll(DS == 2 ? 2 : 1)
        for (int sub = 0; sub < 2; ++sub) {
          if (sub >= nsub) break;
          f32x16 s = ln.dot(tiles[0][sub], af);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int row0 = sub * 32 + key_of_reg(4 * q, g);  // registers 4 q .. 4 q + 3: rows row0 .. + 3
            const f32x4 l4 = *reinterpret_cast<const f32x4*>(&rowv[0][row0]);
            f32x4 lo4 = f32x4{};
            if constexpr (sizeof(T) == 4) lo4 = *reinterpret_cast<const f32x4*>(&rowv[1][row0]);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const int row = row0 + t;
              float y = fmaf(s[4 * q + t], p.scale_log2, -l4[t]);
              if constexpr (sizeof(T) == 4) y -= lo4[t];
              if constexpr (HAS_BIAS) y = own_ok && row < N ? fmaf(bias_s[row * BS + key], kLog2e, y) : y;
              // (rows past N: LSE2 = +inf alone leaves a NaN where the key holds an infinity, times their zeros)
              s[4 * q + t] = own_ok && row < N && (!p.causal || row >= key) ? fast_exp2(y) : 0.f;
            }
          }
          Own w[2];
          ln.pack(s, w);
          ln.add_tr(tiles[3][sub], w, acc1);
          const f32x16 dp = ln.dot(tiles[3][sub], bf);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int row0 = sub * 32 + key_of_reg(4 * q, g);
            const f32x4 d4 = *reinterpret_cast<const f32x4*>(&rowv[2][row0]);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const int row = row0 + t;
              s[4 * q + t] *= dp[4 * q + t] - d4[t];
              if constexpr (DS == 1) {
                if (own_ok && row < N) dso[(uint32_t)(row * N + key)] = s[4 * q + t];
              }
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
    if constexpr (DS != 2) break;  // one (batch, head) per work-group
    __syncthreads();  // the tiles are rewritten for the next one
  }
  if constexpr (DS == 2) {
    const int wave = threadIdx.x >> 6, c = threadIdx.x & 31, g = (threadIdx.x >> 5) & 1, key = (wave & 1) * 32 + c;
    float* dst = p.ds_out + ((int64_t)blockIdx.x * p.H + hi) * N * N;
    if (wave >= 2 && key < N) {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = sub * 32 + key_of_reg(r, g);
          if (row < N) dst[(uint32_t)(row * N + key)] = dsum[sub][r];
        }
    }
  }
}

// Head dims above 64 do not fit (fp32 tiles of 64 rows at D = 128: 196 KB of LDS).
bool bwd_short_takes(int n, int dp) { return n <= kShortRows && dp <= 64; }

// Groups of windows (ds_mode 2): one round of the work-groups that run at once (by registers and LDS 3, 2,
// 2 and 1 per CU), and no group takes more than one window more than another.
int bwd_short_groups(int dtype, int dp, int batch, int heads) {
  const int64_t slots = dtype == ELSA_F32 ? (dp == 64 ? 256 : 512) : (dp == 64 ? 512 : 768);
  const int64_t rounds = ((int64_t)batch * heads + slots - 1) / slots;
  return (int)((batch + rounds - 1) / rounds);
}

template <typename T, int DP>
static hipError_t short_launch(const BwdParams& p, int dtype, int ds_mode, hipStream_t st) {
  const int B = p.BH / p.H, groups = ds_mode == 2 ? bwd_short_groups(dtype, DP, B, p.H) : B;
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
static hipError_t short_launch_d(const BwdParams& p, int dtype, int ds_mode, hipStream_t st) {
  return pad_head_dim(p.D) == 32 ? short_launch<T, 32>(p, dtype, ds_mode, st) : short_launch<T, 64>(p, dtype, ds_mode, st);
}

hipError_t launch_bwd_short(const BwdParams& p, int dtype, int ds_mode, hipStream_t st) {
  if (dtype == ELSA_F16) return short_launch_d<f16>(p, dtype, ds_mode, st);
  if (dtype == ELSA_BF16) return short_launch_d<bf16>(p, dtype, ds_mode, st);
  return short_launch_d<float>(p, dtype, ds_mode, st);
}

}  // namespace elsa
