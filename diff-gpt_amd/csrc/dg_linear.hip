// A decode step's products at n_embd 512 and up (bf16, fp16), each with the
// elementwise work on either side of it in one launch (dg_linear_rows):
//
//   out = epilogue(prologue(x) @ w^T)    prologue: x * sigmoid(g)  (mha.py:84)
//                                        epilogue: the clamped SwiGLU of the
//                                        interleaved pairs (swi_glu.py:15-19), or
//                                        the addition of a residual row
//
// At a few hundred rows a product is short of work for the chip, not of matrix
// cores (400 x 512 x 2048: 0.8 GFLOP), and the launches around it cost as much
// as it does.  A workgroup takes 32 rows and 32 (SwiGLU: 64) features and its
// waves split the contraction, so that a launch has hundreds of workgroups and a
// wave's chain is short: K / waves, in chunks of 128 whose fragments (16 bytes of
// a row per lane, straight from the caches: both operands are contiguous along
// the contraction) are all in flight before the chunk in hand is multiplied.
// Lane (c, g) = (l % 16, l / 16) feeds rows c of a tile of the weights and of the
// tokens with elements 32 s + 8 g .. + 7 of step s (v_mfma_f32_16x16x32) and gets
// back token c's features 4 g .. 4 g + 3.  The partial
// sums meet in LDS in fp32, added in the waves' order, rounded once as the library's
// product, and the epilogue follows on 4 (8) neighbouring features a thread.
// Workgroups that share weight rows run on one XCD.
//
// 400 rows at n_embd 512 in bf16, us (before: the library's product and the
// elementwise launches): gate and c_proj 9.0 -> 6.4, FFN up and SwiGLU 8.9 ->
// 8.2, FFN down and residual 7.7 -> 6.2.  Up to one workgroup per CU the time is
// the chain of one (launch, one round trip for all fragments, the sums' barrier);
// each further one per CU adds 3 - 4 us, its 96 - 128 KB of operands at some 8
// TB/s over all CUs, which is where the library's larger tiles take over.
#include "dg_rows.h"

namespace dg {

struct LinearArgs {
  const void* x;    // (M, K)
  const void* g;    // (M, K) gate logits, or null
  const void* w;    // (N, K)
  const void* res;  // (M, N) added to the product, or null
  void* out;        // (M, N), with SwiGLU (M, N / 2)
  int64_t x_ld, g_ld, w_ld, res_ld, out_ld;
  int M, N, K;
  float alpha, limit;
};

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 lbf16x8_t;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 lf16x8_t;

template <typename T>
__device__ __forceinline__ f32x4_t linear_mma(const RowRegs<T, 8>& a, const RowRegs<T, 8>& b, f32x4_t c) {
  if constexpr (__is_same(T, bf16_t))
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lbf16x8_t, a), __builtin_bit_cast(lbf16x8_t, b),
                                                   c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(lf16x8_t, a), __builtin_bit_cast(lf16x8_t, b), c,
                                                  0, 0, 0);
}

constexpr int kLinRows = 32;
constexpr int kLinChunk = 128;  // contraction elements in flight together
constexpr int kLinSteps = kLinChunk / 32;

template <typename T, bool GATE, bool SWIGLU, int NW>
__global__ __launch_bounds__(64 * NW, 2) void linear_rows_kernel(const LinearArgs a) {
  constexpr int TM = kLinRows / 16;
  constexpr int TN = SWIGLU ? 4 : 2;     // 16-feature tiles
  constexpr int LD = 16 * TN + 4;        // row stride of the partial sums (floats)
  __shared__ __attribute__((aligned(16))) float part[NW][kLinRows * LD];
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int mt = (a.M + kLinRows - 1) / kLinRows, nt = a.N / (16 * TN);
  const int q = blockIdx.x >> 3;
  const int n = (blockIdx.x & 7) + 8 * (q / mt), m = q % mt;  // consecutive workgroups: consecutive XCDs
  if (n >= nt) return;                                        // the whole workgroup, before any barrier
  const int m0 = m * kLinRows, n0 = n * 16 * TN;
  const int kw = a.K / NW, chunks = kw / kLinChunk;
  const int k0 = wv * kw + 8 * g;
  const T *xp[TM], *gp[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t row = min(m0 + 16 * i + c, a.M - 1);  // rows past M: a copy, never stored
    xp[i] = static_cast<const T*>(a.x) + row * a.x_ld + k0;
    gp[i] = GATE ? static_cast<const T*>(a.g) + row * a.g_ld + k0 : nullptr;
  }
  const T* wp = static_cast<const T*>(a.w) + (int64_t)(n0 + c) * a.w_ld + k0;

  struct Chunk {
    RowRegs<T, 8> x[TM][kLinSteps], g[GATE ? TM : 1][GATE ? kLinSteps : 1], w[TN][kLinSteps];
  };
  auto load = [&](Chunk& f, int k) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int s = 0; s < kLinSteps; ++s) {
        load_row<T, 8>(f.x[i][s], xp[i] + k + 32 * s);
        if constexpr (GATE) load_row<T, 8>(f.g[i][s], gp[i] + k + 32 * s);
      }
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int s = 0; s < kLinSteps; ++s) load_row<T, 8>(f.w[t][s], wp + (int64_t)16 * t * a.w_ld + k + 32 * s);
  };
  f32x4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int t = 0; t < TN; ++t) acc[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto mma = [&](const Chunk& f) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < kLinSteps; ++s)
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        RowRegs<T, 8> x = f.x[i][s];
        if constexpr (GATE) x = gate_row<T, 8>(x, f.g[i][s]);
#pragma unroll
        for (int t = 0; t < TN; ++t) acc[i][t] = linear_mma<T>(f.w[t][s], x, acc[i][t]);
      }
  };
  Chunk even, odd;
  load(even, 0);
#pragma unroll 1
  for (int i = 0; i < chunks; i += 2) {
    if (i + 1 < chunks) load(odd, (i + 1) * kLinChunk);
    __builtin_amdgcn_sched_barrier(0);  // loads stay ahead of the products
    mma(even);
    if (i + 1 < chunks) {
      if (i + 2 < chunks) load(even, (i + 2) * kLinChunk);
      __builtin_amdgcn_sched_barrier(0);
      mma(odd);
    }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    mfma_settle(acc[i]);
#pragma unroll
    for (int t = 0; t < TN; ++t)
      *reinterpret_cast<f32x4_t*>(&part[wv][(16 * i + c) * LD + 16 * t + 4 * g]) = acc[i][t];
  }
  __syncthreads();
  constexpr int F = kLinRows * 16 * TN / 256;  // features a thread, of 256
  if (threadIdx.x >= 256) return;
  const int tr = threadIdx.x / 8, f0 = (threadIdx.x % 8) * F;
  if (m0 + tr >= a.M) return;
  float v[F];
#pragma unroll
  for (int i = 0; i < F; i += 4) {
    f32x4_t s = *reinterpret_cast<const f32x4_t*>(&part[0][tr * LD + f0 + i]);
#pragma unroll
    for (int w = 1; w < NW; ++w) s += *reinterpret_cast<const f32x4_t*>(&part[w][tr * LD + f0 + i]);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[i + e] = rt<T>(s[e]);
  }
  if constexpr (SWIGLU) {
    float o[F / 2];
#pragma unroll
    for (int i = 0; i < F / 2; ++i) o[i] = swiglu_value<T>(v[2 * i], v[2 * i + 1], a.alpha, a.limit);
    store_vec<T, F / 2>(static_cast<T*>(a.out) + (int64_t)(m0 + tr) * a.out_ld + (n0 + f0) / 2, o);
  } else {
    if (a.res != nullptr) {  // uniform
      float x[F];
      load_vec<T, F>(static_cast<const T*>(a.res) + (int64_t)(m0 + tr) * a.res_ld + n0 + f0, x);
#pragma unroll
      for (int i = 0; i < F; ++i) v[i] += x[i];
    }
    store_vec<T, F>(static_cast<T*>(a.out) + (int64_t)(m0 + tr) * a.out_ld + n0 + f0, v);
  }
}

namespace {

template <typename T, bool GATE, bool SWIGLU>
void launch_linear(const LinearArgs& a, unsigned grid, hipStream_t s) {
  // eight waves share the contraction where four would leave CUs without work
  if (grid <= 256 && a.K % (8 * kLinChunk) == 0)
    hipLaunchKernelGGL((linear_rows_kernel<T, GATE, SWIGLU, 8>), dim3(grid), dim3(512), 0, s, a);
  else
    hipLaunchKernelGGL((linear_rows_kernel<T, GATE, SWIGLU, 4>), dim3(grid), dim3(256), 0, s, a);
}

template <typename T>
void launch_linear_t(const LinearArgs& a, bool swiglu, unsigned grid, hipStream_t s) {
  if (swiglu) launch_linear<T, false, true>(a, grid, s);
  else if (a.g != nullptr) launch_linear<T, true, false>(a, grid, s);
  else launch_linear<T, false, false>(a, grid, s);
}

}  // namespace
}  // namespace dg

using namespace dg;

extern "C" int dg_linear_rows(int64_t M, int N, int K, int dtype, const void* x, int64_t x_ld, const void* g,
                              int64_t g_ld, const void* w, int64_t w_ld, const void* residual, int64_t res_ld,
                              int swiglu, float alpha, float limit, void* out, int64_t out_ld, void* stream) {
  DG_REQUIRE(M >= 0 && N >= 1 && K >= 1, DG_EINVAL, "linear_rows: bad sizes M=%lld N=%d K=%d", (long long)M, N, K);
  DG_REQUIRE(dtype == DG_BF16 || dtype == DG_F16, DG_EUNSUPPORTED, "linear_rows: dtype %d unsupported", dtype);
  DG_REQUIRE(!swiglu || (g == nullptr && residual == nullptr), DG_EINVAL,
             "linear_rows: SwiGLU goes without a gate and a residual");
  const int tile = swiglu ? 64 : 32;
  DG_REQUIRE(N % tile == 0 && K % (4 * kLinChunk) == 0, DG_EUNSUPPORTED,
             "linear_rows: N=%d K=%d unsupported (multiples of %d and %d)", N, K, tile, 4 * kLinChunk);
  if (M == 0) return DG_OK;
  const int64_t grid = (M + kLinRows - 1) / kLinRows * ((N / tile + 7) / 8 * 8);
  DG_REQUIRE(M <= 0x7fffffffLL - kLinRows && grid <= 0x7fffffffLL, DG_EUNSUPPORTED, "linear_rows: too many rows (%lld)",
             (long long)M);
  DG_REQUIRE(x && w && out, DG_EINVAL, "linear_rows: NULL pointer");
  DG_REQUIRE(x_ld >= K && w_ld >= K && (g == nullptr || g_ld >= K) && (residual == nullptr || res_ld >= N) &&
                 out_ld >= (swiglu ? N / 2 : N),
             DG_EINVAL, "linear_rows: a row stride is narrower than its row");
  auto rows16 = [](const void* p, int64_t ld) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && ld % 8 == 0; };
  DG_REQUIRE(rows16(x, x_ld) && rows16(w, w_ld) && rows16(out, out_ld) && (g == nullptr || rows16(g, g_ld)) &&
                 (residual == nullptr || rows16(residual, res_ld)),
             DG_EUNSUPPORTED, "linear_rows: rows must be 16-byte aligned");
  LinearArgs a{};
  a.x = x; a.g = g; a.w = w; a.res = residual; a.out = out;
  a.x_ld = x_ld; a.g_ld = g_ld; a.w_ld = w_ld; a.res_ld = res_ld; a.out_ld = out_ld;
  a.M = (int)M; a.N = N; a.K = K; a.alpha = alpha; a.limit = limit;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == DG_BF16) launch_linear_t<bf16_t>(a, swiglu != 0, (unsigned)grid, s);
  else launch_linear_t<f16_t>(a, swiglu != 0, (unsigned)grid, s);
  return check_launch("linear_rows_kernel");
}
