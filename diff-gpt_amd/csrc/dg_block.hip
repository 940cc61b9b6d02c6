// Row kernels for the layers around attention in a decode step (the
// "neighbours" of the hot path), one launch each where torch issues several:
//
//   attn_res_norm_kernel  rms_norm(block_attn_res(V, w)) (block.py:10-44 then
//                         rms_norm.py:5-7): per row, the scores
//                         rms_norm(V_n) . w over the sources V_0 .. V_N, their
//                         softmax over n, the weighted sum h = sum_n p_n V_n,
//                         and the RMSNorm of h.  Torch runs stack, rms_norm,
//                         matmul, softmax, mul and sum, then rms_norm.
//   gate_kernel           y * sigmoid(g) (mha.py:84)
//   swiglu_kernel         clamped SwiGLU on interleaved (gate, linear) pairs
//                         (swi_glu.py:11-19)
//   softcap_kernel        cap * tanh(x / cap) (gpt.py:182-186)
//   lm_head_kernel        the tied lm_head GEMM, the softcap and, for greedy
//                         sampling, the argmax of each row (gpt.py:181-186,
//                         temperature.py:22-23) in one pass: the logits are
//                         written once and not read back
//
// Every intermediate is rounded to the storage dtype where the torch op
// sequence rounds it (each op returns a tensor of the input dtype; fp32
// arithmetic inside, as ATen's opmath does), so bf16 results follow the same
// rounding steps.  The RMSNorms of outputs use the lane mapping and
// reduction tree of rms_norm_kernel, so they produce its bits for the same row.
#include <type_traits>

#include "dg_rows.h"

namespace dg {

struct AttnResArgs {
  const void* src[kMaxResSources];
  int64_t ld[kMaxResSources];  // row strides (elements)
  const void* w;               // (C,) pseudo-query
  void* out;
  int64_t out_ld, M;
  int nsrc, N;
  int dup;  // 1 when source 1 is source 0 (same rows): read once
};

// Sources a lane loads into registers together, up front, to serve both
// passes of the mixture (one round trip to memory for them, instead of one
// per source and pass): about 64 registers of slices.
template <int CH>
constexpr int res_held_norm() {
  return CH <= 4 ? 16 : CH <= 8 ? 8 : CH <= 16 ? 4 : CH <= 32 ? 2 : 1;
}

// NS: the most sources of the instance (the launch's fit).
template <typename T, int NPAD, int CH, int NS>
__global__ __launch_bounds__(256) void attn_res_norm_kernel(const AttnResArgs a, const int vec) {
#pragma clang fp contract(off)
  constexpr int G = NPAD / CH;
  constexpr int HELD = res_held_norm<CH>() < NS ? res_held_norm<CH>() : NS;
  static_assert(G >= 1 && G <= 64, "row mapping");
  constexpr int ROWS_PER_BLOCK = 256 / G;
  const int sub = threadIdx.x % G;
  const int64_t row = (int64_t)blockIdx.x * ROWS_PER_BLOCK + threadIdx.x / G;
  if (row >= a.M) return;  // whole lane groups leave together; no barriers
  const int c0 = sub * CH;
  auto load = [&](int n, RowRegs<T, CH>& x) __attribute__((always_inline)) {
    load_packed<T, CH>(x, static_cast<const T*>(a.src[n]) + row * a.ld[n] + c0, c0, a.N, vec);
  };
  RowRegs<T, CH> held[HELD], w;
#pragma unroll
  for (int n = 0; n < HELD; ++n)
    if (n < a.nsrc) load(n, held[n]);  // uniform; no use before all are issued
  auto get = [&](int n, RowRegs<T, CH>& x) __attribute__((always_inline)) {
    if (n < HELD) x = held[n];
    else load(n, x);
  };
  load_packed<T, CH>(w, static_cast<const T*>(a.w) + c0, c0, a.N, vec);

  // pass 1: score_n = rms_norm(V_n) . w, each rounded as its tensor is
  float score[NS];
  float mx = -INFINITY;
#pragma unroll
  for (int n = 0; n < NS; ++n) {
    score[n] = -INFINITY;
    if (n >= a.nsrc) continue;  // uniform
    RowRegs<T, CH> x;
    get(n, x);
    const float r = row_factor(score_sum<G>(slice_squares<T, CH>(x)), a.N);
    score[n] = rt<T>(score_sum<G>(slice_score<T, CH>(x, r, w)));
    mx = fmaxf(mx, score[n]);
  }
  // softmax over the sources (fp32 inside, rounded output)
  float sum = 0.f;
#pragma unroll
  for (int n = 0; n < NS; ++n) {
    if (n >= a.nsrc) continue;
    score[n] = expf(score[n] - mx);
    sum += score[n];
  }
  // pass 2: h = sum_n rt(p_n V_n), fp32 sum in source order, rounded
  float h[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) h[i] = 0.f;
#pragma unroll
  for (int n = 0; n < NS; ++n) {
    if (n >= a.nsrc) continue;
    RowRegs<T, CH> x;
    get(n, x);
    slice_add<T, CH>(h, rt<T>(score[n] / sum), x);
  }
#pragma unroll
  for (int i = 0; i < CH; ++i) h[i] = rt<T>(h[i]);
  row_rms<CH, G>(h, a.N);
  T* os = static_cast<T*>(a.out) + row * a.out_ld + c0;
  if (vec && c0 + CH <= a.N) {
    store_vec<T, CH>(os, h);
  } else {
#pragma unroll
    for (int i = 0; i < CH; ++i)
      if (c0 + i < a.N) os[i] = from_f32<T>(h[i]);
  }
}

// attn_res_norm_kernel for rows that fill a wave (G = 64 lanes of CH elements,
// aligned) with at most NS sources, every one held in registers as loaded.
// A row's sums fold together: each step of the cross-lane
// reduction halves the number of registers (v_permlane32_swap hands the low
// half of the wave one sum and the high half another, v_permlane16_swap the
// same for rows of 16 lanes), so four sources cost the DPP steps of one, and
// the four 16-lane rows then take the square roots, exponentials and
// quotients of four sources at once.  Near HBM's rate at a prefill's sizes: 65536
// bf16 rows of 512 with 6 sources, 5 of them distinct (403 MB), take 101 us
// (4.0 TB/s), 28672 rows of 1024 with 4 (235 MB) 52 us (4.5 TB/s); one source at
// a time, with its own reductions and fp32 copies in registers, the former took
// 237.  NS = 4, 6, 8 or 12 sources and 96 registers of them: beyond either
// the general form's.
template <typename T, int CH, int NS>
__global__ __launch_bounds__(256) void attn_res_norm_wave_kernel(const AttnResArgs a) {
#pragma clang fp contract(off)
  constexpr int NG = (NS + 3) / 4;  // groups of four sources
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.M) return;  // whole waves leave; no barriers
  const int c0 = lane * CH;
  RowRegs<T, CH> v[NS], w;
#pragma unroll
  for (int n = 0; n < NS; ++n) {
    if (n >= a.nsrc) {  // uniform
#pragma unroll
      for (int i = 0; i < RowRegs<T, CH>::WORDS; ++i) v[n].w[i] = 0u;
    } else if (n == 1 && a.dup) {
      v[1] = v[0];
    } else {
      load_row<T, CH>(v[n], static_cast<const T*>(a.src[n]) + row * a.ld[n] + c0);
    }
  }
  load_row<T, CH>(w, static_cast<const T*>(a.w) + c0);
  // the sums of sources 4k .. 4k + 3 in 16-lane rows 0, 2, 1, 3 of one register
  auto fold4 = [](float s0, float s1, float s2, float s3) __attribute__((always_inline)) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(s0), __float_as_uint(s1), false, false);
    const float t0 = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(s2), __float_as_uint(s3), false, false);
    const float t1 = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = __builtin_amdgcn_permlane16_swap(__float_as_uint(t0), __float_as_uint(t1), false, false);
    return row16_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
  };
  auto of_source = [](const float (&x)[NG], int n) __attribute__((always_inline)) {
    const int lane0 = 16 * (((n & 1) << 1) | ((n >> 1) & 1));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x[n / 4]), lane0));
  };
  const int q = lane >> 4, in4 = ((q & 1) << 1) | (q >> 1);  // this 16-lane row's source of each four
  float part[4 * NG], sc[NG];
#pragma unroll
  for (int n = 0; n < 4 * NG; ++n) part[n] = n < NS ? slice_squares<T, CH>(v[n < NS ? n : 0]) : 0.f;
#pragma unroll
  for (int k = 0; k < NG; ++k)
    sc[k] = row_factor(fold4(part[4 * k], part[4 * k + 1], part[4 * k + 2], part[4 * k + 3]), a.N);
#pragma unroll
  for (int n = 0; n < NS; ++n) part[n] = slice_score<T, CH>(v[n], of_source(sc, n), w);
  float mx = -INFINITY;
#pragma unroll
  for (int k = 0; k < NG; ++k) {
    const float d = fold4(part[4 * k], part[4 * k + 1], part[4 * k + 2], part[4 * k + 3]);
    sc[k] = 4 * k + in4 < a.nsrc ? rt<T>(d) : -INFINITY;
    mx = fmaxf(mx, sc[k]);
  }
  {
    float x, y;
    pair16(mx, x, y);
    mx = fmaxf(x, y);
    pair32(mx, x, y);
    mx = fmaxf(x, y);
  }
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < NG; ++k) sc[k] = expf(sc[k] - mx);
#pragma unroll
  for (int n = 0; n < NS; ++n)
    if (n < a.nsrc) sum += of_source(sc, n);
#pragma unroll
  for (int k = 0; k < NG; ++k) sc[k] = rt<T>(sc[k] / sum);
  float h[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) h[i] = 0.f;
#pragma unroll
  for (int n = 0; n < NS; ++n)
    if (n < a.nsrc) slice_add<T, CH>(h, of_source(sc, n), v[n]);  // uniform
#pragma unroll
  for (int i = 0; i < CH; ++i) h[i] = rt<T>(h[i]);
  row_rms<CH, 64>(h, a.N);
  store_vec<T, CH>(static_cast<T*>(a.out) + row * a.out_ld + c0, h);
}

// attn_res_norm_kernel for few wide rows (one row per wave there, G = 64):
// a workgroup of 4 waves takes one row, so a decode step's few hundred rows
// keep four times the waves in flight and each wave's dependent chain of
// per-source reductions is a quarter as long.  Wave w scores sources w,
// w + 4, ... (each in the lane mapping, arithmetic and reduction order of
// attn_res_norm_kernel, so each score has its bits); the scores meet in LDS;
// every wave takes the softmax over them in source order; wave w forms the
// weighted sum for a quarter of the columns (each column summed over the
// sources in source order, as before) into LDS; wave 0 normalises the row in
// attn_res_norm_kernel's lane mapping and stores it.  Same bits throughout.
template <int CH>
constexpr int res_held_split() {
  return CH <= 8 ? 8 : 64 / CH;
}

template <typename T, int NPAD, int CH>
__global__ __launch_bounds__(256) void attn_res_norm_split_kernel(const AttnResArgs a, const int vec) {
#pragma clang fp contract(off)
  constexpr int G = NPAD / CH;
  static_assert(G == 64, "one row per wave in attn_res_norm_kernel's mapping");
  constexpr int HELD = res_held_split<CH>();  // sources a wave holds in registers
  constexpr int CQ = CH / 4;                  // columns per lane in the weighted sum
  static_assert(CQ >= 1 && CQ * 4 == CH, "column split");
  __shared__ float sc[kMaxResSources];
  __shared__ __attribute__((aligned(16))) float hrow[NPAD];
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int64_t row = blockIdx.x;  // the host launches one workgroup per row
  const int c0 = lane * CH;
  RowRegs<T, CH> w;
  load_packed<T, CH>(w, static_cast<const T*>(a.w) + c0, c0, a.N, vec);
  auto load = [&](int n, RowRegs<T, CH>& x) __attribute__((always_inline)) {
    load_packed<T, CH>(x, static_cast<const T*>(a.src[n]) + row * a.ld[n] + c0, c0, a.N, vec);
  };
  RowRegs<T, CH> held[HELD];
#pragma unroll
  for (int j = 0; j < HELD; ++j)
    if (wv + 4 * j < a.nsrc) load(wv + 4 * j, held[j]);  // wave-uniform; no use before all are issued
  // pass 1: this wave's scores
#pragma unroll
  for (int j = 0; j < kMaxResSources / 4; ++j) {
    const int n = wv + 4 * j;
    if (n >= a.nsrc) break;  // wave-uniform
    RowRegs<T, CH> x;
    if (j < HELD) x = held[j];
    else load(n, x);
    const float r = row_factor(score_sum<G>(slice_squares<T, CH>(x)), a.N);
    const float score = rt<T>(score_sum<G>(slice_score<T, CH>(x, r, w)));
    if (lane == 0) sc[n] = score;
  }
  __syncthreads();
  // softmax over the sources, in source order
  float mx = -INFINITY;
#pragma unroll
  for (int n = 0; n < kMaxResSources; ++n)
    if (n < a.nsrc) mx = fmaxf(mx, sc[n]);
  float e[kMaxResSources];
  float sum = 0.f;
#pragma unroll
  for (int n = 0; n < kMaxResSources; ++n) {
    e[n] = 0.f;
    if (n >= a.nsrc) continue;
    e[n] = expf(sc[n] - mx);
    sum += e[n];
  }
  // pass 2: columns [16 CH wv, 16 CH (wv + 1)) of the weighted sum, CQ per lane
  const int cq = 16 * CH * wv + lane * CQ;
  float h[CQ];
#pragma unroll
  for (int i = 0; i < CQ; ++i) h[i] = 0.f;
#pragma unroll
  for (int n = 0; n < kMaxResSources; ++n) {
    if (n >= a.nsrc) continue;
    const float p = rt<T>(e[n] / sum);
    float x[CQ];
    load_slice<T, CQ>(static_cast<const T*>(a.src[n]) + row * a.ld[n] + cq, cq, a.N, vec, x);
#pragma unroll
    for (int i = 0; i < CQ; ++i) h[i] = h[i] + rt<T>(p * x[i]);
  }
#pragma unroll
  for (int i = 0; i < CQ; ++i) hrow[cq + i] = (cq + i < a.N) ? rt<T>(h[i]) : 0.f;
  __syncthreads();
  if (wv != 0) return;  // no barrier follows
  float hn[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) hn[i] = hrow[c0 + i];
  row_rms<CH, G>(hn, a.N);
  T* os = static_cast<T*>(a.out) + row * a.out_ld + c0;
  if (vec && c0 + CH <= a.N) {
    store_vec<T, CH>(os, hn);
  } else {
#pragma unroll
    for (int i = 0; i < CH; ++i)
      if (c0 + i < a.N) os[i] = from_f32<T>(hn[i]);
  }
}

struct RowsArgs {
  const void* x;  // gate: y;  swiglu: interleaved input;  softcap: logits
  const void* g;  // gate: g
  void* out;
  int64_t x_ld, g_ld, out_ld, M;
  int N;          // output columns
  float p0, p1;   // swiglu: alpha, limit;  softcap: cap
  double d0, d1;  // the same in float64 (the float64 kernels)
};

template <typename T>
__global__ __launch_bounds__(256) void gate_kernel(const RowsArgs a) {
#pragma clang fp contract(off)
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= a.M * a.N) return;
  const int64_t r = idx / a.N;
  const int c = (int)(idx - r * a.N);
  const float y = to_f32(static_cast<const T*>(a.x)[r * a.x_ld + c]);
  const float s = sigmoid_rt<T>(to_f32(static_cast<const T*>(a.g)[r * a.g_ld + c]));
  static_cast<T*>(a.out)[r * a.out_ld + c] = from_f32<T>(y * s);
}

template <typename T>
__global__ __launch_bounds__(256) void swiglu_kernel(const RowsArgs a) {
#pragma clang fp contract(off)
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= a.M * a.N) return;
  const int64_t r = idx / a.N;
  const int j = (int)(idx - r * a.N);
  const T* xr = static_cast<const T*>(a.x) + r * a.x_ld;
  static_cast<T*>(a.out)[r * a.out_ld + j] =
      from_f32<T>(swiglu_value<T>(to_f32(xr[2 * j]), to_f32(xr[2 * j + 1]), a.p0, a.p1));
}

// gate_kernel and swiglu_kernel over rows of whole 16-byte vectors of their
// input (aligned; the host checks): same values, same bits.  A thread takes U
// vectors, 256 apart, all loaded before the first is used; the row and column
// of the first come from one 32-bit division, those of the next by adding the
// row and column steps of 256 vectors (drow, dcol).  One element per thread,
// with a 64-bit division each and 2-byte accesses, ran at 2.3 TB/s: the gate of
// 262144 bf16 rows of 512 (805 MB) took 348 us, here 172 (4.7 TB/s, a large copy's
// rate).
struct VecRowsArgs {
  RowsArgs a;
  uint32_t vectors, cols;  // vectors in all, and per row
  uint32_t drow, dcol;     // 256 / cols, 256 % cols
};

template <typename T, int U>
__global__ __launch_bounds__(256) void gate_vec_kernel(const VecRowsArgs v) {
#pragma clang fp contract(off)
  constexpr int E = 16 / (int)sizeof(T);
  const RowsArgs& a = v.a;
  const uint32_t idx = blockIdx.x * (256u * U) + threadIdx.x;
  uint32_t r = idx / v.cols, c = idx - r * v.cols;
  RowRegs<T, E> y[U], g[U];
  T* o[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    o[u] = nullptr;
    if (idx + 256u * u < v.vectors) {
      load_row<T, E>(y[u], static_cast<const T*>(a.x) + (int64_t)r * a.x_ld + c * E);
      load_row<T, E>(g[u], static_cast<const T*>(a.g) + (int64_t)r * a.g_ld + c * E);
      o[u] = static_cast<T*>(a.out) + (int64_t)r * a.out_ld + c * E;
    }
    r += v.drow;
    c += v.dcol;
    if (c >= v.cols) {
      c -= v.cols;
      ++r;
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (o[u] == nullptr) continue;
    store_row<T, E>(o[u], gate_row<T, E>(y[u], g[u]));
  }
}

template <typename T, int U>
__global__ __launch_bounds__(256) void swiglu_vec_kernel(const VecRowsArgs v) {
#pragma clang fp contract(off)
  constexpr int E = 16 / (int)sizeof(T);  // input elements: E / 2 outputs
  const RowsArgs& a = v.a;
  const uint32_t idx = blockIdx.x * (256u * U) + threadIdx.x;
  uint32_t r = idx / v.cols, c = idx - r * v.cols;
  RowRegs<T, E> x[U];
  T* o[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    o[u] = nullptr;
    if (idx + 256u * u < v.vectors) {
      load_row<T, E>(x[u], static_cast<const T*>(a.x) + (int64_t)r * a.x_ld + c * E);
      o[u] = static_cast<T*>(a.out) + (int64_t)r * a.out_ld + c * (E / 2);
    }
    r += v.drow;
    c += v.dcol;
    if (c >= v.cols) {
      c -= v.cols;
      ++r;
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (o[u] == nullptr) continue;
    float h[E / 2];
#pragma unroll
    for (int e = 0; e < E / 2; ++e)
      h[e] = swiglu_value<T>(elem<T, E>(x[u], 2 * e), elem<T, E>(x[u], 2 * e + 1), a.p0, a.p1);
    RowRegs<T, E / 2> p;
    pack_row<T, E / 2>(p, h);
    store_row<T, E / 2>(o[u], p);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void softcap_kernel(const RowsArgs a) {
#pragma clang fp contract(off)
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= a.M * a.N) return;
  const int64_t r = idx / a.N;
  const int c = (int)(idx - r * a.N);
  const float cap = a.p0;
  const float x = to_f32(static_cast<const T*>(a.x)[r * a.x_ld + c]);
  const float t = rt<T>(tanhf(rt<T>(x / cap)));
  static_cast<T*>(a.out)[r * a.out_ld + c] = from_f32<T>(cap * t);
}

// ---------------------------------------------------------------------------
// float64 rows (a GPT.double() model): the same ops in float64 arithmetic, as
// torch's float64 kernels evaluate them -- sigmoid 1 / (1 + exp(-x)), tanh,
// the RMSNorms with DBL_EPSILON, the source softmax with its maximum
// subtracted.  alpha, limit and cap are the ABI's float64 values.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double sigmoid_f64(double x) { return 1.0 / (1.0 + exp(-x)); }

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// rms_norm(block_attn_res(V, w)) for one row per wave, two passes over the
// sources (C <= 2048, lane l holding columns l, l + 64, ...): the scores
// rms_norm(V_n) . w, their softmax over n, h = sum_n p_n V_n written out, then
// h's RMSNorm in place (each lane rescales the columns it wrote).
__global__ __launch_bounds__(256) void attn_res_norm_f64_kernel(const AttnResArgs a) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.M) return;  // whole waves leave; no barriers follow
  const double* w = static_cast<const double*>(a.w);
  double score[kMaxResSources];
  double mx = -__builtin_huge_val();
  for (int n = 0; n < a.nsrc; ++n) {
    const double* x = static_cast<const double*>(a.src[n]) + row * a.ld[n];
    double ss = 0.0;
    for (int c = lane; c < a.N; c += 64) ss += x[c] * x[c];
    const double r = 1.0 / sqrt(wave_sum_f64(ss) / (double)a.N + DBL_EPSILON);
    double dot = 0.0;
    for (int c = lane; c < a.N; c += 64) dot += (x[c] * r) * w[c];
    score[n] = wave_sum_f64(dot);
    mx = fmax(mx, score[n]);
  }
  double sum = 0.0;
  for (int n = 0; n < a.nsrc; ++n) {
    score[n] = exp(score[n] - mx);
    sum += score[n];
  }
  double* o = static_cast<double*>(a.out) + row * a.out_ld;
  double ss = 0.0;
  for (int c = lane; c < a.N; c += 64) {
    double h = 0.0;
    for (int n = 0; n < a.nsrc; ++n) h += (score[n] / sum) * static_cast<const double*>(a.src[n])[row * a.ld[n] + c];
    o[c] = h;
    ss += h * h;
  }
  const double r = 1.0 / sqrt(wave_sum_f64(ss) / (double)a.N + DBL_EPSILON);
  for (int c = lane; c < a.N; c += 64) o[c] = o[c] * r;
}

__global__ __launch_bounds__(256) void gate_kernel_f64(const RowsArgs a) {
#pragma clang fp contract(off)
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= a.M * a.N) return;
  const int64_t r = idx / a.N;
  const int c = (int)(idx - r * a.N);
  const double y = static_cast<const double*>(a.x)[r * a.x_ld + c];
  const double s = sigmoid_f64(static_cast<const double*>(a.g)[r * a.g_ld + c]);
  static_cast<double*>(a.out)[r * a.out_ld + c] = y * s;
}

__global__ __launch_bounds__(256) void swiglu_kernel_f64(const RowsArgs a) {
#pragma clang fp contract(off)
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= a.M * a.N) return;
  const int64_t r = idx / a.N;
  const int j = (int)(idx - r * a.N);
  const double* xr = static_cast<const double*>(a.x) + r * a.x_ld;
  const double alpha = a.d0, limit = a.d1;
  const double gate = fmin(xr[2 * j], limit);
  const double lin = fmin(fmax(xr[2 * j + 1], -limit), limit);
  const double s = sigmoid_f64(alpha * gate);
  static_cast<double*>(a.out)[r * a.out_ld + j] = (gate * s) * (lin + 1.0);
}

__global__ __launch_bounds__(256) void softcap_kernel_f64(const RowsArgs a) {
#pragma clang fp contract(off)
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= a.M * a.N) return;
  const int64_t r = idx / a.N;
  const int c = (int)(idx - r * a.N);
  const double cap = a.d0;
  const double x = static_cast<const double*>(a.x)[r * a.x_ld + c];
  static_cast<double*>(a.out)[r * a.out_ld + c] = cap * tanh(x / cap);
}

namespace {

bool al(const void* p, int64_t bytes) { return (reinterpret_cast<uintptr_t>(p) % (uintptr_t)bytes) == 0; }

int pow2_at_least(int x) {
  int p = 1;
  while (p < x) p <<= 1;
  return p;
}

// Rows up to which wide rows (G = 64) take attn_res_norm_split_kernel.  The line
// is the one against attn_res_norm_kernel, a row per wave with its sources one at
// a time, which the split form leads up to some 4096 rows (512 rows of 512 in bf16,
// 3 / 9 sources: 6.8 -> 5.3 / 10.2 -> 7.8 us).  attn_res_norm_wave_kernel, which takes
// aligned rows beyond the line, is ahead of the split form below it as well, where
// its registers hold every source; us, split -> wave, two of the sources the same:
//   bf16  512, 3 sources: 16 rows 4.7 -> 3.1, 400 5.2 -> 3.3, 4096 15.0 -> 5.9; 10 sources: 400 8.0 -> 5.1
//   bf16 1024, 3 sources: 16 rows 4.9 -> 3.5, 400 5.6 -> 3.8, 4096 17.1 -> 8.4; 10 sources: 400 9.2 -> 6.7
//   fp32  512, 6 sources: 16 rows 5.7 -> 3.7, 400 6.3 -> 3.9, 4096 27.5 -> 11.5
// and behind it where they do not and the row goes to attn_res_norm_kernel:
//   fp32 1024, 10 sources: 400 rows 9.7 -> 12.0;  fp32 2048, 6: 400 rows 11.8 -> 17.6, 2048 37.3 -> 37.3
constexpr int64_t kResSplitRows = 4096;

template <typename T, int NPAD>
int launch_res(const AttnResArgs& a, hipStream_t s) {
  // the lane mapping of rms_norm_kernel for the same row length
  constexpr int PREF = 16 / (int)sizeof(T);
  constexpr int CH0 = NPAD / 64 > PREF ? NPAD / 64 : PREF;
  constexpr int CH = CH0 < NPAD ? CH0 : NPAD;
  constexpr int G = NPAD / CH;
  constexpr int RPB = 256 / G;
  const int64_t blocks = (a.M + RPB - 1) / RPB;
  DG_REQUIRE(blocks <= 0x7fffffffLL, DG_EINVAL, "attn_res_norm: too many rows (%lld)", (long long)a.M);
  const int64_t vb = (int64_t)CH * (int64_t)sizeof(T);
  bool vec = (vb == 4 || vb == 8 || vb % 16 == 0) && (CH * (int)sizeof(T)) >= 4 && al(a.w, vb) &&
             al(a.out, vb) && (a.out_ld * (int64_t)sizeof(T)) % vb == 0;
  for (int n = 0; n < a.nsrc; ++n) vec = vec && al(a.src[n], vb) && (a.ld[n] * (int64_t)sizeof(T)) % vb == 0;
  if constexpr (G == 64 && CH % 4 == 0) {
    // few wide rows (a decode step's): one row per workgroup of four waves
    if (a.M <= kResSplitRows) {
      hipLaunchKernelGGL((attn_res_norm_split_kernel<T, NPAD, CH>), dim3((unsigned)a.M), dim3(256), 0, s, a,
                         vec ? 1 : 0);
      return check_launch("attn_res_norm_split_kernel");
    }
  }
  if constexpr (G == 64 && CH * (int)sizeof(T) >= 16) {
    // rows that fill a wave, every source in registers (at most 96 of them)
    if (vec && a.N == NPAD) {
      constexpr int WORDS = RowRegs<T, CH>::WORDS;
#define DG_RES_WAVE(NS)                                                                                         \
  if constexpr (WORDS * NS <= 96) {                                                                             \
    if (a.nsrc <= NS) {                                                                                         \
      hipLaunchKernelGGL((attn_res_norm_wave_kernel<T, CH, NS>), dim3((unsigned)blocks), dim3(256), 0, s, a);   \
      return check_launch("attn_res_norm_wave_kernel");                                                         \
    }                                                                                                           \
  }
      DG_RES_WAVE(4)
      DG_RES_WAVE(6)
      DG_RES_WAVE(8)
      DG_RES_WAVE(12)
#undef DG_RES_WAVE
    }
  }
  // the unrolled loops as long as the sources need (few in a shallow model)
  if (a.nsrc <= 4)
    hipLaunchKernelGGL((attn_res_norm_kernel<T, NPAD, CH, 4>), dim3((unsigned)blocks), dim3(256), 0, s, a,
                       vec ? 1 : 0);
  else
    hipLaunchKernelGGL((attn_res_norm_kernel<T, NPAD, CH, kMaxResSources>), dim3((unsigned)blocks), dim3(256), 0, s,
                       a, vec ? 1 : 0);
  return check_launch("attn_res_norm_kernel");
}

template <typename T>
int res_pick(int npad, const AttnResArgs& a, hipStream_t s) {
  switch (npad) {
    case 1:
    case 2: return launch_res<T, 2>(a, s);
    case 4: return launch_res<T, 4>(a, s);
    case 8: return launch_res<T, 8>(a, s);
    case 16: return launch_res<T, 16>(a, s);
    case 32: return launch_res<T, 32>(a, s);
    case 64: return launch_res<T, 64>(a, s);
    case 128: return launch_res<T, 128>(a, s);
    case 256: return launch_res<T, 256>(a, s);
    case 512: return launch_res<T, 512>(a, s);
    case 1024: return launch_res<T, 1024>(a, s);
    case 2048: return launch_res<T, 2048>(a, s);
  }
  set_error("attn_res_norm: C=%d unsupported (max 2048)", a.N);
  return DG_EUNSUPPORTED;
}

}  // namespace

// ---------------------------------------------------------------------------
// lm_head + softcap + greedy argmax.  Block = 4 waves = 16 rows of x; wave w
// takes the vocabulary entries [w V/4, (w+1) V/4) in NTW tiles of 16.  Per
// tile, logits^T (16 entries x 16 rows) = W_tile x^T on the matrix cores with
// qk_mfma's lane mapping: lane (c, g) feeds embedding row 16t + c and x row c,
// each with the contiguous quarter g of the contraction (chunks of 16
// elements), and gets back row c's logits for entries 16t + 4g .. 16t + 4g + 3.
// The logit is rounded to T (F.linear's output), then capped with
// softcap_kernel's arithmetic and rounding, stored, and compared: the first
// maximum wins (torch.argmax), across the lane's values in entry order, the
// four lanes of a row, then the four waves through LDS.
// ---------------------------------------------------------------------------
struct LmHeadArgs {
  const void* x;  // (M, C) rows, already normalised (gpt.py:181 rms_norm)
  const void* w;  // (V, C) tied embedding table
  void* logits;   // (M, V)
  int64_t* ids;   // (M,) or null
  int64_t x_ld, w_ld, l_ld, M;
  int C, V;
  float cap;  // 0: no softcap
};

template <typename T, int NTW>
__global__ __launch_bounds__(256) void lm_head_kernel(const LmHeadArgs a) {
#pragma clang fp contract(off)
  constexpr int KCH = 16;  // contraction elements per lane and chunk
  __shared__ float red_v[4][16];
  __shared__ int red_i[4][16];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int64_t row0 = (int64_t)blockIdx.x * 16;
  const bool row_ok = row0 + c < a.M;
  const int64_t row = row_ok ? row0 + c : a.M - 1;
  const int cq = a.C / 4;  // this lane's quarter of the contraction
  const int vbase = w * (a.V / 4);
  const T* xr = static_cast<const T*>(a.x) + row * a.x_ld + g * cq;
  const T* wr = static_cast<const T*>(a.w) + (int64_t)(vbase + c) * a.w_ld + g * cq;

  f32x4_t acc[NTW];
#pragma unroll
  for (int t = 0; t < NTW; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < cq; k0 += KCH) {
    RowRegs<T, KCH> xo;
    load_row<T, KCH>(xo, xr + k0);
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
      RowRegs<T, KCH> wo;
      load_row<T, KCH>(wo, wr + (int64_t)16 * t * a.w_ld + k0);
      acc[t] = qk_mfma<T, KCH>(wo, xo, acc[t]);
    }
  }

  float best = kNegInf;
  int bidx = 0x7fffffff;
  T* lrow = static_cast<T*>(a.logits) + row * a.l_ld + vbase + 4 * g;
#pragma unroll
  for (int t = 0; t < NTW; ++t) {
    float out[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = softcap_value<T>(acc[t][r], a.cap);
      out[r] = v;
      const int e = vbase + 16 * t + 4 * g + r;  // increasing within the lane
      if (v > best) {
        best = v;
        bidx = e;
      }
    }
    if (row_ok) store_vec<T, 4>(lrow + 16 * t, out);
  }
  if (a.ids == nullptr) return;  // uniform over the grid
  first_max(best, bidx);
  if (g == 0) {
    red_v[w][c] = best;
    red_i[w][c] = bidx;
  }
  __syncthreads();
  if (w != 0 || g != 0 || !row_ok) return;
  // waves in entry order: a strictly larger value replaces the earlier one
  float bv = red_v[0][c];
  int bi = red_i[0][c];
#pragma unroll
  for (int q = 1; q < 4; ++q) {
    if (red_v[q][c] > bv) {
      bv = red_v[q][c];
      bi = red_i[q][c];
    }
  }
  a.ids[row0 + c] = (int64_t)(bi == 0x7fffffff ? 0 : bi);
}

namespace {

template <typename T>
int launch_lm_head(const LmHeadArgs& a, hipStream_t s) {
  const int ntw = a.V / 64;
  const unsigned blocks = (unsigned)((a.M + 15) / 16);
  switch (ntw) {
    case 1: hipLaunchKernelGGL((lm_head_kernel<T, 1>), dim3(blocks), dim3(256), 0, s, a); break;
    case 2: hipLaunchKernelGGL((lm_head_kernel<T, 2>), dim3(blocks), dim3(256), 0, s, a); break;
    case 4: hipLaunchKernelGGL((lm_head_kernel<T, 4>), dim3(blocks), dim3(256), 0, s, a); break;
    case 8: hipLaunchKernelGGL((lm_head_kernel<T, 8>), dim3(blocks), dim3(256), 0, s, a); break;
    case 16: hipLaunchKernelGGL((lm_head_kernel<T, 16>), dim3(blocks), dim3(256), 0, s, a); break;
    default:
      set_error("lm_head: vocabulary %d unsupported (64, 128, 256, 512 or 1024)", a.V);
      return DG_EUNSUPPORTED;
  }
  return check_launch("lm_head_kernel");
}

// one thread per output element; K<T> for the dtype
#define DG_LAUNCH_ROWS(K, dtype, a, s)                                                        \
  do {                                                                                        \
    const int64_t n_ = (a).M * (int64_t)(a).N;                                                \
    if (n_ == 0) return DG_OK;                                                                \
    const int64_t blocks_ = (n_ + 255) / 256;                                                 \
    DG_REQUIRE(blocks_ <= 0x7fffffffLL, DG_EINVAL, #K ": too many elements (%lld)", (long long)n_); \
    if ((dtype) == DG_F64)                                                                    \
      hipLaunchKernelGGL(K##_f64, dim3((unsigned)blocks_), dim3(256), 0, (s), (a));           \
    else if ((dtype) == DG_F32)                                                               \
      hipLaunchKernelGGL(K<float>, dim3((unsigned)blocks_), dim3(256), 0, (s), (a));          \
    else if ((dtype) == DG_BF16)                                                              \
      hipLaunchKernelGGL(K<bf16_t>, dim3((unsigned)blocks_), dim3(256), 0, (s), (a));         \
    else                                                                                      \
      hipLaunchKernelGGL(K<f16_t>, dim3((unsigned)blocks_), dim3(256), 0, (s), (a));          \
    return check_launch(#K);                                                                  \
  } while (0)

// Vectors per thread of the vector row kernels: 4 (64 bytes in flight per
// input and lane) once the launch still fills the chip with them -- 1024
// workgroups, 4 per CU -- else 1, so that a decode step's few rows spread over
// as many CUs as they can.
constexpr int64_t kVecRowsDeep = 4 * 256 * 1024;

// The vector form of a row op whose input rows hold `in_cols` elements: K<T, U>
// when they are whole 16-byte vectors (fewer than 2^31 in all) and every row
// pointed to is aligned (out_align bytes for the output); false otherwise.
bool vec_rows(const RowsArgs& a, int dtype, int64_t in_cols, int64_t out_align, VecRowsArgs& v) {
  if (dtype == DG_F64) return false;
  const int64_t es = dtype_bytes(dtype);
  auto rows = [&](const void* p, int64_t ld, int64_t n) {
    return p == nullptr || ((reinterpret_cast<uintptr_t>(p) % (uintptr_t)n) == 0 && (ld * es) % n == 0);
  };
  const int64_t cols = in_cols * es / 16;
  if ((in_cols * es) % 16 != 0 || cols > 0x7fffffffLL || a.M > 0x7fffffffLL / cols) return false;
  if (!rows(a.x, a.x_ld, 16) || !rows(a.g, a.g_ld, 16) || !rows(a.out, a.out_ld, out_align)) return false;
  // the last workgroup counts past the end
  if (a.M * cols > 0x7fffffffLL - 4 * 256) return false;
  v.a = a;
  v.vectors = (uint32_t)(a.M * cols);
  v.cols = (uint32_t)cols;
  v.drow = 256u / v.cols;
  v.dcol = 256u % v.cols;
  return true;
}

#define DG_LAUNCH_VEC_ROWS(K, dtype, v, s)                                                        \
  do {                                                                                            \
    const bool deep_ = (int64_t)(v).vectors >= kVecRowsDeep;                                      \
    const unsigned blocks_ = ((v).vectors + (deep_ ? 1023u : 255u)) / (deep_ ? 1024u : 256u);     \
    if ((dtype) == DG_F32) {                                                                      \
      if (deep_) hipLaunchKernelGGL((K<float, 4>), dim3(blocks_), dim3(256), 0, (s), (v));        \
      else hipLaunchKernelGGL((K<float, 1>), dim3(blocks_), dim3(256), 0, (s), (v));              \
    } else if ((dtype) == DG_BF16) {                                                              \
      if (deep_) hipLaunchKernelGGL((K<bf16_t, 4>), dim3(blocks_), dim3(256), 0, (s), (v));       \
      else hipLaunchKernelGGL((K<bf16_t, 1>), dim3(blocks_), dim3(256), 0, (s), (v));             \
    } else {                                                                                      \
      if (deep_) hipLaunchKernelGGL((K<f16_t, 4>), dim3(blocks_), dim3(256), 0, (s), (v));        \
      else hipLaunchKernelGGL((K<f16_t, 1>), dim3(blocks_), dim3(256), 0, (s), (v));              \
    }                                                                                             \
    return check_launch(#K);                                                                      \
  } while (0)

bool dtype_ok(int dtype) { return dtype == DG_F32 || dtype == DG_BF16 || dtype == DG_F16; }
// the row kernels with float64 forms (dg_attn_res_norm, dg_gate, dg_swiglu, dg_softcap)
bool dtype_ok_f64(int dtype) { return dtype_ok(dtype) || dtype == DG_F64; }

}  // namespace
}  // namespace dg

using namespace dg;

extern "C" int dg_attn_res_norm(int64_t M, int C, int dtype, int nsrc, const void* const* src,
                                const int64_t* src_ld, const void* w, void* out, int64_t out_ld,
                                void* stream) {
  DG_REQUIRE(M >= 0 && C >= 1, DG_EINVAL, "attn_res_norm: bad sizes M=%lld C=%d", (long long)M, C);
  DG_REQUIRE(C <= 2048, DG_EUNSUPPORTED, "attn_res_norm: C=%d > 2048", C);
  DG_REQUIRE(dtype_ok_f64(dtype), DG_EUNSUPPORTED, "attn_res_norm: dtype %d unsupported", dtype);
  DG_REQUIRE(nsrc >= 1 && nsrc <= kMaxResSources, DG_EINVAL, "attn_res_norm: %d sources (1..%d)", nsrc,
             kMaxResSources);
  if (M == 0) return DG_OK;
  DG_REQUIRE(src != nullptr && src_ld != nullptr && w != nullptr && out != nullptr, DG_EINVAL,
             "attn_res_norm: NULL pointer");
  DG_REQUIRE(out_ld >= C, DG_EINVAL, "attn_res_norm: output row stride smaller than C");
  AttnResArgs a{};
  for (int n = 0; n < nsrc; ++n) {
    DG_REQUIRE(src[n] != nullptr && src_ld[n] >= C, DG_EINVAL,
               "attn_res_norm: source %d is NULL or its row stride is smaller than C", n);
    a.src[n] = src[n];
    a.ld[n] = src_ld[n];
  }
  a.w = w;
  a.out = out;
  a.out_ld = out_ld;
  a.M = M;
  a.nsrc = nsrc;
  a.N = C;
  a.dup = nsrc > 1 && src[1] == src[0] && src_ld[1] == src_ld[0] ? 1 : 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == DG_F64) {
    DG_REQUIRE((M + 3) / 4 <= 0x7fffffffLL, DG_EINVAL, "attn_res_norm: too many rows (%lld)", (long long)M);
    hipLaunchKernelGGL(attn_res_norm_f64_kernel, dim3((unsigned)((M + 3) / 4)), dim3(256), 0, s, a);
    return check_launch("attn_res_norm_f64_kernel");
  }
  const int npad = pow2_at_least(C);
  if (dtype == DG_F32) return res_pick<float>(npad, a, s);
  if (dtype == DG_BF16) return res_pick<bf16_t>(npad, a, s);
  return res_pick<f16_t>(npad, a, s);
}

extern "C" int dg_gate(int64_t M, int C, int dtype, const void* y, int64_t y_ld, const void* g,
                       int64_t g_ld, void* out, int64_t out_ld, void* stream) {
  DG_REQUIRE(M >= 0 && C >= 1, DG_EINVAL, "gate: bad sizes M=%lld C=%d", (long long)M, C);
  DG_REQUIRE(dtype_ok_f64(dtype), DG_EUNSUPPORTED, "gate: dtype %d unsupported", dtype);
  if (M == 0) return DG_OK;
  DG_REQUIRE(y != nullptr && g != nullptr && out != nullptr, DG_EINVAL, "gate: NULL pointer");
  DG_REQUIRE(y_ld >= C && g_ld >= C && out_ld >= C, DG_EINVAL, "gate: row stride smaller than C");
  RowsArgs a{};
  a.x = y; a.g = g; a.out = out;
  a.x_ld = y_ld; a.g_ld = g_ld; a.out_ld = out_ld; a.M = M; a.N = C;
  hipStream_t s = static_cast<hipStream_t>(stream);
  VecRowsArgs v;
  if (vec_rows(a, dtype, C, 16, v)) DG_LAUNCH_VEC_ROWS(gate_vec_kernel, dtype, v, s);
  DG_LAUNCH_ROWS(gate_kernel, dtype, a, s);
}

extern "C" int dg_swiglu(int64_t M, int N, int dtype, const void* x, int64_t x_ld, void* out,
                         int64_t out_ld, double alpha, double limit, void* stream) {
  DG_REQUIRE(M >= 0 && N >= 1, DG_EINVAL, "swiglu: bad sizes M=%lld N=%d", (long long)M, N);
  DG_REQUIRE(dtype_ok_f64(dtype), DG_EUNSUPPORTED, "swiglu: dtype %d unsupported", dtype);
  if (M == 0) return DG_OK;
  DG_REQUIRE(x != nullptr && out != nullptr, DG_EINVAL, "swiglu: NULL pointer");
  DG_REQUIRE(x_ld >= 2 * (int64_t)N && out_ld >= N, DG_EINVAL, "swiglu: row stride too small");
  RowsArgs a{};
  a.x = x; a.out = out;
  a.x_ld = x_ld; a.out_ld = out_ld; a.M = M; a.N = N;
  a.p0 = (float)alpha; a.p1 = (float)limit;
  a.d0 = alpha; a.d1 = limit;
  hipStream_t s = static_cast<hipStream_t>(stream);
  VecRowsArgs v;
  if (vec_rows(a, dtype, 2 * (int64_t)N, 8, v)) DG_LAUNCH_VEC_ROWS(swiglu_vec_kernel, dtype, v, s);
  DG_LAUNCH_ROWS(swiglu_kernel, dtype, a, s);
}

extern "C" int dg_softcap(int64_t M, int N, int dtype, const void* x, int64_t x_ld, void* out,
                          int64_t out_ld, double cap, void* stream) {
  DG_REQUIRE(M >= 0 && N >= 1, DG_EINVAL, "softcap: bad sizes M=%lld N=%d", (long long)M, N);
  DG_REQUIRE(dtype_ok_f64(dtype), DG_EUNSUPPORTED, "softcap: dtype %d unsupported", dtype);
  DG_REQUIRE(cap > 0.0, DG_EINVAL, "softcap: cap must be positive (got %g)", cap);
  if (M == 0) return DG_OK;
  DG_REQUIRE(x != nullptr && out != nullptr, DG_EINVAL, "softcap: NULL pointer");
  DG_REQUIRE(x_ld >= N && out_ld >= N, DG_EINVAL, "softcap: row stride smaller than N");
  RowsArgs a{};
  a.x = x; a.out = out;
  a.x_ld = x_ld; a.out_ld = out_ld; a.M = M; a.N = N;
  a.p0 = (float)cap;
  a.d0 = cap;
  DG_LAUNCH_ROWS(softcap_kernel, dtype, a, static_cast<hipStream_t>(stream));
}

extern "C" int dg_lm_head(int64_t M, int C, int V, int dtype, const void* x, int64_t x_ld, const void* w,
                          int64_t w_ld, float cap, void* logits, int64_t logits_ld, int64_t* ids, void* stream) {
  DG_REQUIRE(M >= 0 && C >= 1 && V >= 1, DG_EINVAL, "lm_head: bad sizes M=%lld C=%d V=%d", (long long)M, C, V);
  DG_REQUIRE(dtype_ok(dtype), DG_EUNSUPPORTED, "lm_head: dtype %d unsupported", dtype);
  DG_REQUIRE(cap >= 0.f, DG_EINVAL, "lm_head: cap must be >= 0 (got %g)", (double)cap);
  DG_REQUIRE(C % 64 == 0 && C <= 8192, DG_EUNSUPPORTED, "lm_head: n_embd %d unsupported (a multiple of 64)", C);
  DG_REQUIRE(V == 64 || V == 128 || V == 256 || V == 512 || V == 1024, DG_EUNSUPPORTED,
             "lm_head: vocabulary %d unsupported (64, 128, 256, 512 or 1024)", V);
  if (M == 0) return DG_OK;
  DG_REQUIRE(M <= (int64_t)16 * 0x7fffffffLL, DG_EINVAL, "lm_head: too many rows (%lld)", (long long)M);
  DG_REQUIRE(x != nullptr && w != nullptr && logits != nullptr, DG_EINVAL, "lm_head: NULL pointer");
  DG_REQUIRE(x_ld >= C && w_ld >= C && logits_ld >= V, DG_EINVAL, "lm_head: row stride smaller than the row");
  const int64_t es = dtype == DG_F32 ? 4 : 2;
  auto al = [](const void* p, int64_t n) { return (reinterpret_cast<uintptr_t>(p) % (uintptr_t)n) == 0; };
  DG_REQUIRE(al(x, 16) && al(w, 16) && al(logits, 4 * es) && (x_ld * es) % 16 == 0 && (w_ld * es) % 16 == 0 &&
                 (logits_ld * es) % (4 * es) == 0,
             DG_EUNSUPPORTED, "lm_head: rows must be 16-byte aligned");
  LmHeadArgs a{};
  a.x = x; a.w = w; a.logits = logits; a.ids = ids;
  a.x_ld = x_ld; a.w_ld = w_ld; a.l_ld = logits_ld; a.M = M;
  a.C = C; a.V = V; a.cap = cap;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == DG_F32) return launch_lm_head<float>(a, s);
  if (dtype == DG_BF16) return launch_lm_head<bf16_t>(a, s);
  return launch_lm_head<f16_t>(a, s);
}

// ---------------------------------------------------------------------------
// The sampler's draw (torch.multinomial's one-sample method, temperature.py:
// 24-25 after the softmax): ids[r] = the first maximum over j of
// probs[r, j] / q[r, j], with q the caller's Exp(1) variates.  The quotient
// is rounded to the storage dtype as torch's division returns it (fp32
// arithmetic, correctly rounded; fp64 for fp64 data), and compared as
// torch.argmax compares: a NaN is above every number, the first of equal
// values (or of NaNs) wins.  One wave per row; lane l takes entries l,
// l + 64, ... so each lane meets its entries in increasing order.
// ---------------------------------------------------------------------------
namespace dg {

template <typename C>
__device__ __forceinline__ bool draw_better(C v, int i, C bv, int bi) {
  const bool vn = v != v, bn = bv != bv;
  if (vn || bn) return vn && (!bn || i < bi);
  return v > bv || (v == bv && i < bi);
}

template <typename T>
__global__ __launch_bounds__(256) void draw_argmax_kernel(const T* probs, int64_t p_ld, const T* q, int64_t q_ld,
                                                          int64_t* ids, int64_t M, int V) {
  using C = typename std::conditional<sizeof(T) == 8, double, float>::type;
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;  // whole waves
  const T* pr = probs + row * p_ld;
  const T* qr = q + row * q_ld;
  C best = (C)0;
  int bi = 0x7fffffff;
  for (int j = lane; j < V; j += 64) {
    C v;
    if constexpr (sizeof(T) == 8) {
      v = (C)pr[j] / (C)qr[j];
    } else {
      v = (C)to_f32(from_f32<T>(to_f32(pr[j]) / to_f32(qr[j])));
    }
    if (bi == 0x7fffffff || draw_better<C>(v, j, best, bi)) {
      best = v;
      bi = j;
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const C ov = __shfl_xor(best, off, 64);
    const int oi = __shfl_xor(bi, off, 64);
    if (oi != 0x7fffffff && (bi == 0x7fffffff || draw_better<C>(ov, oi, best, bi))) {
      best = ov;
      bi = oi;
    }
  }
  if (lane == 0) ids[row] = bi;
}

}  // namespace dg

extern "C" int dg_draw_argmax(int64_t M, int V, int dtype, const void* probs, int64_t p_ld, const void* q,
                              int64_t q_ld, int64_t* ids, void* stream) {
  using namespace dg;
  DG_REQUIRE(M >= 0 && V >= 1, DG_EINVAL, "draw_argmax: bad sizes M=%lld V=%d", (long long)M, V);
  DG_REQUIRE(dtype_ok_f64(dtype), DG_EUNSUPPORTED, "draw_argmax: dtype %d unsupported", dtype);
  if (M == 0) return DG_OK;
  DG_REQUIRE(probs && q && ids, DG_EINVAL, "draw_argmax: NULL pointer");
  DG_REQUIRE(p_ld >= V && q_ld >= V, DG_EINVAL, "draw_argmax: a row stride is narrower than its row");
  DG_REQUIRE(M <= 4 * 0x7fffffffLL, DG_EINVAL, "draw_argmax: too many rows (%lld)", (long long)M);
  const dim3 grid((unsigned)((M + 3) / 4));
  hipStream_t s = static_cast<hipStream_t>(stream);
#define DG_DRAW(T)                                                                                 \
  hipLaunchKernelGGL((draw_argmax_kernel<T>), grid, dim3(256), 0, s, static_cast<const T*>(probs), p_ld, \
                     static_cast<const T*>(q), q_ld, ids, M, V)
  if (dtype == DG_F32) DG_DRAW(float);
  else if (dtype == DG_BF16) DG_DRAW(bf16_t);
  else if (dtype == DG_F16) DG_DRAW(f16_t);
  else DG_DRAW(double);
#undef DG_DRAW
  return check_launch("draw_argmax_kernel");
}
