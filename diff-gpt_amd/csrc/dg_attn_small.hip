// Prefill attention at head_dim 16 and 32 on the matrix cores (the causal and
// chunked branches of mha.py:61-81 for small models: 4 heads of 16 at n_embd
// 64, of 32 at n_embd 128), fp32, bf16 and fp16.
//
// Work unit = one wavefront = 16 queries of one (b, h), walking the visible
// keys in chunks of NT tiles of 16.  Per tile, lane (c, g) = (l & 15, l >> 4):
//   S^T (16 keys x 16 queries) = K Q^T with qk_mfma (fp32 products for fp32
//     data, exact products of 16-bit data, fp32 sums); lane (c, g) gets query
//     c's scores of keys 4g .. 4g + 3.
//   O^T (D x 16 queries) += V^T P^T on v_mfma_f32_16x16x4_f32, step s taking
//     key 4g + s in lane group g: its P^T operand is score register s itself,
//     its V^T operand the one value V[4g + s][c].  Probabilities and values
//     stay fp32 for every data type.
// A lane's statistics belong to one query and meet across the four lane
// groups by two permlane swaps; the running maximum is raised lazily as in the
// other kernels.  K, V and Q come straight from global memory (no LDS, no
// barrier): the waves of a head run on one XCD and re-read its few KB of keys
// from L1 and L2, and a chunk's loads are issued while the one before
// computes.  Bound by the memory it must read and write at many short rows:
// 1024 (b, h) of 138 tokens, D = 16, fp32 (36 MB of q, k, v, y) take 22 us;
// one query per wave on the vector ALU took 103 us.
#include "dg_prefill.h"

namespace dg {

template <typename T, int D>
struct SmallCfg {
  static constexpr int DQ = D / 4;   // contraction elements of a lane's quarter
  static constexpr int NB = D / 16;  // 16-dim blocks of O^T
  // tiles per chunk: two chunks of keys and values in registers (64 of them)
  static constexpr int NT = D == 16 ? 4 : 2;
};

template <typename T, int D>
__global__ __launch_bounds__(256) void prefill_small_kernel(const PrefillArgs a, const int units, const int nqt) {
  using C = SmallCfg<T, D>;
  constexpr int DQ = C::DQ, NB = C::NB, NT = C::NT;
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  // the host rounds the grid to a multiple of 8 workgroups: consecutive units
  // (the query tiles of one head) on one XCD
  const int blk = (blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
  const int unit = 4 * blk + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (unit >= units) return;  // whole waves leave; no barriers
  const int bh = unit / nqt;
  const int q0 = 16 * (nqt - 1 - (unit - bh * nqt));  // the longest tiles of a head first
  const int head = bh % a.H;
  const int64_t b = bh / a.H;
  const T* qp = static_cast<const T*>(a.q) + b * a.qb + (int64_t)head * a.qh;
  const T* kp = static_cast<const T*>(a.k) + b * a.kb + (int64_t)head * a.kh;
  const T* vp = static_cast<const T*>(a.v) + b * a.vb + (int64_t)head * a.vh;
  const int kt = (int)a.kt, vt = (int)a.vt;  // host: Tk * stride < 2^31 bytes
  const int qoff = a.q_offset;
  const int kend = min(a.Tk, q0 + 16 + qoff);  // keys some query of the tile sees

  RowRegs<T, DQ> qop;  // rows past Tq hold row Tq - 1 and are not stored
  load_row<T, DQ>(qop, qp + (int64_t)min(q0 + c, a.Tq - 1) * a.qt + g * DQ);

  struct Chunk {
    RowRegs<T, DQ> k[NT];
    T v[NT][NB][4];
  };
  auto load = [&](Chunk& ch, int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int k0 = t0 + 16 * u;
      if (k0 >= kend) continue;  // wave-uniform
      // keys past the last re-read it; their scores are masked
      load_row<T, DQ>(ch.k[u], kp + (uint32_t)(min(k0 + c, a.Tk - 1) * kt + g * DQ));
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const uint32_t row = (uint32_t)(min(k0 + 4 * g + s, a.Tk - 1) * vt + c);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) ch.v[u][nb][s] = vp[row + 16 * nb];
      }
    }
  };

  f32x4_t o[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) o[nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = kNegInf, l = 0.f;

  auto process = [&](const Chunk& ch, int t0) __attribute__((always_inline)) {
    f32x4_t s[NT];
    float mt = kNegInf;
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      s[u] = f32x4_t{kNegInf, kNegInf, kNegInf, kNegInf};
      if (t0 + 16 * u < kend) s[u] = qk_mfma<T, DQ>(ch.k[u], qop, f32x4_t{0.f, 0.f, 0.f, 0.f});
    }
    mfma_settle(s);
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int k0 = t0 + 16 * u;
      if (k0 >= kend) continue;
      if (k0 + 15 > q0 + qoff || k0 + 16 > a.Tk) {  // the tile crosses the diagonal or the end
        const int lim = min(q0 + c + qoff, a.Tk - 1) - k0 - 4 * g;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (r > lim) s[u][r] = kNegInf;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) mt = fmaxf(mt, s[u][r]);
    }
    float x, y;
    pair16(mt, x, y);
    mt = fmaxf(x, y);
    pair32(mt, x, y);
    mt = fmaxf(x, y);
    if (__builtin_amdgcn_ballot_w64(mt > m + a.lazy_raw) != 0) {
      // m == -inf only before the first chunk, whose key 0 every query sees
      const float mnew = fmaxf(m, mt);
      const float alpha = m == kNegInf ? 0.f : __builtin_amdgcn_exp2f((m - mnew) * a.scale_log2);
      m = mnew;
      l *= alpha;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[nb][r] *= alpha;
    }
    const float moff = m * a.scale_log2;
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int k0 = t0 + 16 * u;
      if (k0 >= kend) continue;
      float v[NB][4];
      bool finite = true;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[u][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][r], a.scale_log2, -moff));
        l += s[u][r];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          v[nb][r] = to_f32(ch.v[u][nb][r]);
          finite = finite && __builtin_fabsf(v[nb][r]) < __builtin_huge_valf();
        }
      }
      const bool crosses = k0 + 15 > q0 + qoff || k0 + 16 > a.Tk;
      if (crosses && __builtin_amdgcn_ballot_w64(!finite) != 0) {
        // A value that is not finite in a tile some queries see only part of:
        // as a product, its 0 * inf would reach the queries it is hidden from.
        // Key by key, visible keys only.
        const int lim = min(q0 + c + qoff, a.Tk - 1) - k0;
        for (int kg = 0; kg < 4; ++kg) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float p = __shfl(s[u][r], c + 16 * kg, 64);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
              for (int d = 0; d < 4; ++d) {
                const float vv = __shfl(v[nb][r], 4 * g + d + 16 * kg, 64);
                if (4 * kg + r <= lim) o[nb][d] = __builtin_fmaf(p, vv, o[nb][d]);
              }
          }
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            o[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[nb][r], s[u][r], o[nb], 0, 0, 0);
      }
    }
  };

  Chunk ca, cb;
  constexpr int STEP = 16 * NT;
  load(ca, 0);
  for (int t0 = 0; t0 < kend; t0 += 2 * STEP) {
    if (t0 + STEP < kend) load(cb, t0 + STEP);
    process(ca, t0);
    if (t0 + STEP >= kend) break;
    if (t0 + 2 * STEP < kend) load(ca, t0 + 2 * STEP);
    process(cb, t0 + STEP);
  }

  float x, y;
  pair16(l, x, y);
  l = x + y;
  pair32(l, x, y);
  l = x + y;
  if (q0 + c >= a.Tq) return;
  const float inv = 1.0f / l;
  T* yr = static_cast<T*>(a.y) + b * a.yb + (int64_t)(q0 + c) * a.yt + (int64_t)head * a.yh + 4 * g;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const float w[4] = {o[nb][0] * inv, o[nb][1] * inv, o[nb][2] * inv, o[nb][3] * inv};
    store_vec<T, 4>(yr + 16 * nb, w);
  }
}

// At least 16 queries, so that a tile is mostly full (below, the vector
// kernel's wave per query); rows aligned to the lane's loads and stores; a
// positive scale (the maximum is taken on raw scores); offsets inside a head's
// K and V within 2^31 bytes.
bool small_prefill_applicable(int B, int H, int Tq, int Tk, int D, int dtype, const void* q, const dg_stride3* q_st,
                              const void* k, const dg_stride3* k_st, const void* v, const dg_stride3* v_st,
                              const void* y, const dg_stride3* y_st, float scale) {
  if ((D != 16 && D != 32) || Tq < 16 || !(scale > 0.f)) return false;
  if (dtype != DG_F32 && dtype != DG_BF16 && dtype != DG_F16) return false;
  const int64_t es = dtype_bytes(dtype);
  if ((int64_t)B * H * ((Tq + 15) / 16) > 0x7fffffffLL - 64) return false;
  if (k_st->t < 0 || v_st->t < 0) return false;
  const int64_t span = (int64_t)Tk * (k_st->t > v_st->t ? k_st->t : v_st->t) + D;
  if (span * es >= (int64_t)1 << 31) return false;
  const int64_t ld = D / 4 * es < 16 ? D / 4 * es : 16;  // bytes of a lane's load of q and k
  auto rows = [&](const void* p, const dg_stride3* s, int64_t n) {
    return (reinterpret_cast<uintptr_t>(p) % (uintptr_t)n) == 0 && (s->b * es) % n == 0 && (s->t * es) % n == 0 &&
           (s->h * es) % n == 0;
  };
  return rows(q, q_st, ld) && rows(k, k_st, ld) && rows(v, v_st, es) && rows(y, y_st, 4 * es);
}

int small_prefill(int B, int H, int Tq, int Tk, int D, int dtype, const void* q, const dg_stride3* q_st,
                  const void* k, const dg_stride3* k_st, const void* v, const dg_stride3* v_st, void* y,
                  const dg_stride3* y_st, float scale, hipStream_t s) {
  PrefillArgs a{};
  a.q = q; a.k = k; a.v = v; a.y = y;
  a.qb = q_st->b; a.qt = q_st->t; a.qh = q_st->h;
  a.kb = k_st->b; a.kt = k_st->t; a.kh = k_st->h;
  a.vb = v_st->b; a.vt = v_st->t; a.vh = v_st->h;
  a.yb = y_st->b; a.yt = y_st->t; a.yh = y_st->h;
  a.H = H; a.Tq = Tq; a.Tk = Tk;
  a.q_offset = Tk - Tq;
  a.nbh = B * H;
  a.scale_log2 = scale * 1.44269504088896340736f;
  a.lazy_raw = kLazyLog2 / a.scale_log2;
  const int nqt = (Tq + 15) / 16;
  const int units = (int)((int64_t)B * H * nqt);
  const unsigned blocks = ((unsigned)(units + 3) / 4 + 7u) & ~7u;
#define DG_SMALL(T)                                                                                               \
  do {                                                                                                            \
    if (D == 16) hipLaunchKernelGGL((prefill_small_kernel<T, 16>), dim3(blocks), dim3(256), 0, s, a, units, nqt); \
    else hipLaunchKernelGGL((prefill_small_kernel<T, 32>), dim3(blocks), dim3(256), 0, s, a, units, nqt);         \
  } while (0)
  if (dtype == DG_F32) DG_SMALL(float);
  else if (dtype == DG_BF16) DG_SMALL(bf16_t);
  else DG_SMALL(f16_t);
#undef DG_SMALL
  return check_launch("prefill_small_kernel");
}

}  // namespace dg
