// Additive bias loads of the forward and backward kernels.
#pragma once

#include "elsa_internal.h"
#include "elsa_mfma.h"

namespace elsa {

__device__ inline float load_bias(const BiasView& b, int bi, int hi, int row, int key) {
  const int64_t off = (int64_t)bi * b.sb + (int64_t)hi * b.sh + (int64_t)row * b.sq + (int64_t)key * b.sk;
  if (b.dtype == ELSA_F32) return static_cast<const float*>(b.ptr)[off];
  if (b.dtype == ELSA_F16) return static_cast<float>(static_cast<const f16*>(b.ptr)[off]);
  return static_cast<float>(static_cast<const bf16*>(b.ptr)[off]);
}

// Bias rows that 16-byte loads can read: 16-bit values, key stride 1, batch / head / row
// strides in multiples of 8 elements and a 16-byte aligned base.
__device__ inline bool bias_rows_vectorizable(const BiasView& b) {
  return b.dtype != ELSA_F32 && b.sk == 1 && b.sq % 8 == 0 && b.sb % 8 == 0 && b.sh % 8 == 0 &&
         reinterpret_cast<uintptr_t>(b.ptr) % 16 == 0;
}

// Bias of one query row (element offset row_off) at keys key0 + 16 j + t (j < 2, t < 8) into
// v[8 j + t]: the keys the D-layout registers of one 32-key sub-tile hold (key_of_reg).
// Keys at or past k_end read as 0 (the caller masks them).  vec: one 16-byte load per 8 keys.
template <typename B16>
__device__ inline void bias_keys16_vec(const BiasView& b, int64_t row_off, int key0, int k_end, float (&v)[16]) {
  typedef B16 b8 __attribute__((ext_vector_type(8)));
  const B16* base = static_cast<const B16*>(b.ptr) + row_off;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int k = key0 + 16 * j;
    if (k + 8 <= k_end) {
      const b8 c = *reinterpret_cast<const b8*>(base + k);
#pragma unroll
      for (int t = 0; t < 8; ++t) v[8 * j + t] = static_cast<float>(c[t]);
    } else {
#pragma unroll
      for (int t = 0; t < 8; ++t) v[8 * j + t] = k + t < k_end ? static_cast<float>(base[k + t]) : 0.f;
    }
  }
}

// Unit key stride, rows of any alignment: one address per lane and constant offsets.  Keys at or past k_end
// read the row's last key instead (in range: no branch, so that the 16 loads are in flight together).
template <typename BT>
__device__ inline void bias_keys16_row(const BiasView& b, int64_t row_off, int key0, int k_end, float (&v)[16]) {
  const BT* row = static_cast<const BT*>(b.ptr) + row_off;
  if (key0 + 24 <= k_end) {
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = static_cast<float>(row[key0 + 16 * (r >> 3) + (r & 7)]);
  } else {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = key0 + 16 * (r >> 3) + (r & 7);
      const float x = static_cast<float>(row[min(key, k_end - 1)]);
      v[r] = key < k_end ? x : 0.f;
    }
  }
}

__device__ inline void bias_keys16(const BiasView& b, int64_t row_off, int key0, int k_end, bool vec, float (&v)[16]) {
  if (vec) {
    if (b.dtype == ELSA_F16)
      bias_keys16_vec<f16>(b, row_off, key0, k_end, v);
    else
      bias_keys16_vec<bf16>(b, row_off, key0, k_end, v);
    return;
  }
  if (b.sk == 1) {
    if (b.dtype == ELSA_F16)
      bias_keys16_row<f16>(b, row_off, key0, k_end, v);
    else if (b.dtype == ELSA_BF16)
      bias_keys16_row<bf16>(b, row_off, key0, k_end, v);
    else
      bias_keys16_row<float>(b, row_off, key0, k_end, v);
    return;
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int key = key0 + 16 * (r >> 3) + (r & 7);
    float x = 0.f;
    if (key < k_end) {
      const int64_t off = row_off + (int64_t)key * b.sk;
      if (b.dtype == ELSA_F32)
        x = static_cast<const float*>(b.ptr)[off];
      else if (b.dtype == ELSA_F16)
        x = static_cast<float>(static_cast<const f16*>(b.ptr)[off]);
      else
        x = static_cast<float>(static_cast<const bf16*>(b.ptr)[off]);
    }
    v[r] = x;
  }
}

// CNT rows row0 .. of one key's column (element offset col_off): the rows a dk/dv lane's registers hold.
// Rows at or past n read row n - 1 (the caller masks them): no branch, one 64-bit product per call.
template <typename BT, int CNT>
__device__ inline void bias_rows_t(const BiasView& b, int64_t col_off, int row0, int n, float (&v)[CNT]) {
  const BT* col = static_cast<const BT*>(b.ptr) + col_off + (int64_t)min(row0, n - 1) * b.sq;
#pragma unroll
  for (int t = 0; t < CNT; ++t) {
    v[t] = static_cast<float>(*col);
    col += row0 + t + 1 < n ? b.sq : 0;
  }
}
template <int CNT>
__device__ inline void bias_rows(const BiasView& b, int64_t col_off, int row0, int n, float (&v)[CNT]) {
  if (b.dtype == ELSA_F16)
    bias_rows_t<f16, CNT>(b, col_off, row0, n, v);
  else if (b.dtype == ELSA_BF16)
    bias_rows_t<bf16, CNT>(b, col_off, row0, n, v);
  else
    bias_rows_t<float, CNT>(b, col_off, row0, n, v);
}

}  // namespace elsa
