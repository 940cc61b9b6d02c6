// Row arithmetic of the kernels around attention (dg_block.hip, dg_layer.hip):
// the row norm, the Block-AttnRes mixture on slices as stored, and SwiGLU.
#pragma once

#include <float.h>

#include "dg_common.h"

namespace dg {

constexpr int kMaxResSources = 32;

// RMSNorm of one row slice with rms_norm_kernel's arithmetic (squares summed
// by tree_sum inside the lane, then the butterfly over the G lanes of the row,
// here in registers: group_sum_dpp pairs the lanes as group_sum does, so the
// bits are the same)
template <int CH, int G>
__device__ __forceinline__ void row_rms(float (&x)[CH], int N) {
#pragma clang fp contract(off)
  float sq[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) sq[i] = x[i] * x[i];
  float ss = tree_sum<CH>(sq);
  ss = group_sum_dpp<G>(ss);
  const float mean = ss / (float)N;
  const float r = 1.0f / sqrtf(mean + FLT_EPSILON);
#pragma unroll
  for (int i = 0; i < CH; ++i) x[i] = x[i] * r;
}

template <typename T, int CH>
__device__ __forceinline__ void load_slice(const T* p, int c0, int N, bool vec, float (&x)[CH]) {
  if (vec && c0 + CH <= N) {
    load_vec<T, CH>(p, x);
  } else {
#pragma unroll
    for (int i = 0; i < CH; ++i) x[i] = (c0 + i < N) ? to_f32(p[i]) : 0.f;
  }
}

// The mixture's arithmetic on a lane's slices as they are stored, the same in
// its three kernels (so they agree bit for bit), each intermediate rounded to
// T where its torch tensor is.  16-bit types work on packed pairs: the squares
// and the products with w by v_dot2_f32_{bf16,f16} (exact products, fp32
// sums), each rounding by one conversion of a pair.  fp32 takes four chains and
// their tree: one chain over a wide row's slice (16 elements at C = 1024) leaves
// the result some 4 % further from float64 (8192 such rows: 9.94e-8 of the norm
// against 9.44e-8).

// sums of the products of two slices, and of a slice's squares
template <typename T, int CH>
__device__ __forceinline__ float slice_products(const RowRegs<T, CH>& x, const RowRegs<T, CH>& y) {
#pragma clang fp contract(off)
  if constexpr (sizeof(T) == 4) {
    constexpr int N = CH < 4 ? CH : 4;
    float v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = elem<T, CH>(x, i) * elem<T, CH>(y, i);
#pragma unroll
    for (int i = N; i < CH; ++i) v[i % N] = __builtin_fmaf(elem<T, CH>(x, i), elem<T, CH>(y, i), v[i % N]);
    return tree_sum<N>(v);
  } else {
    return slice_dot<T, CH>(x, y);
  }
}
template <typename T, int CH>
__device__ __forceinline__ float slice_squares(const RowRegs<T, CH>& x) {
  return slice_products<T, CH>(x, x);
}
// sum of rt(x r) w over the slice: the normalised row against the pseudo-query
template <typename T, int CH>
__device__ __forceinline__ float slice_score(const RowRegs<T, CH>& x, float r, const RowRegs<T, CH>& w) {
#pragma clang fp contract(off)
  float v[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) v[i] = elem<T, CH>(x, i) * r;
  RowRegs<T, CH> n;
  pack_row<T, CH>(n, v);
  return slice_products<T, CH>(n, w);
}
// h += rt(p x)
template <typename T, int CH>
__device__ __forceinline__ void slice_add(float (&h)[CH], float p, const RowRegs<T, CH>& x) {
#pragma clang fp contract(off)
  float v[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) v[i] = p * elem<T, CH>(x, i);
  RowRegs<T, CH> n;
  pack_row<T, CH>(n, v);
#pragma unroll
  for (int i = 0; i < CH; ++i) h[i] = h[i] + elem<T, CH>(n, i);
}
// the slice at p (elements c0 .. of a row of N), zeros past N
template <typename T, int CH>
__device__ __forceinline__ void load_packed(RowRegs<T, CH>& r, const T* p, int c0, int N, bool vec) {
  if (vec && c0 + CH <= N) {
    load_row<T, CH>(r, p);
  } else {
    float v[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) v[i] = (c0 + i < N) ? to_f32(p[i]) : 0.f;
    pack_row<T, CH>(r, v);
  }
}
// Sum over the G lanes of a row.  G = 64: halves and 16-lane rows first, in
// the order attn_res_norm_wave_kernel folds several sums at once.
__device__ __forceinline__ float row16_sum(float v) {
  v = v + dpp<kDppQuadXor1>(v);
  v = v + dpp<kDppQuadXor2>(v);
  v = v + dpp<kDppHalfMirror>(v);
  return v + dpp<kDppMirror>(v);
}
template <int G>
__device__ __forceinline__ float score_sum(float v) {
  if constexpr (G == 64) {
    float a, b;
    pair32(v, a, b);
    v = a + b;
    pair16(v, a, b);
    return row16_sum(a + b);
  } else {
    return group_sum_dpp<G>(v);
  }
}
__device__ __forceinline__ float row_factor(float ss, int N) {
#pragma clang fp contract(off)
  return 1.0f / sqrtf(ss / (float)N + FLT_EPSILON);
}

// One SwiGLU element with the torch sequence's roundings (swi_glu.py:15-19).
// clamp(max=limit) / clamp(-limit, limit) select existing values: exact.
template <typename T>
__device__ __forceinline__ float swiglu_value(float gate, float lin, float alpha, float limit) {
#pragma clang fp contract(off)
  gate = fminf(gate, limit);
  lin = fminf(fmaxf(lin, -limit), limit);
  const float s = sigmoid_rt<T>(rt<T>(alpha * gate));
  return rt<T>(gate * s) * rt<T>(lin + 1.0f);
}

// A logit from its fp32 sum: rounded to T (F.linear's output), then, with cap
// > 0, softcap_kernel's arithmetic and rounding.
template <typename T>
__device__ __forceinline__ float softcap_value(float v, float cap) {
#pragma clang fp contract(off)
  v = rt<T>(v);
  return cap > 0.f ? rt<T>(cap * rt<T>(tanhf(rt<T>(v / cap)))) : v;
}

// The first maximum over the four lanes (l & 15, g) of a row: larger value, or
// equal value and smaller entry.
__device__ __forceinline__ void first_max(float& best, int& entry) {
#pragma unroll
  for (int off = 16; off <= 32; off <<= 1) {
    const float ov = __shfl_xor(best, off, 64);
    const int oi = __shfl_xor(entry, off, 64);
    if (ov > best || (ov == best && oi < entry)) {
      best = ov;
      entry = oi;
    }
  }
}

}  // namespace dg
