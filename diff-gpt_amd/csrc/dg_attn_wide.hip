// Fused decode step (dg_decode_step) at head_dim 64 and 128 in bf16 / fp16 for
// rows that come in groups of at least 16 sharing a prefix (an Engine call's
// trajectories of one prompt): RoPE, QK-norm, the K/V append, and attention
// over the group's prefix, the row's own cached keys and the new key.
//
// The vector kernel reads the prefix once per (row, head): 400 rows of 8 heads
// of 64 over a 1024-token prefix pull 840 MB through the L2s and the vector ALU,
// 61 us.  Here a workgroup takes 16 rows of a group and one head, and the
// prefix becomes matrix products shared by the 16 rows:
//
//   * 8 waves deal the prefix's keys out in chunks of KC (64 at D = 64, 32 at
//     D = 128).  S^T (16 keys x 16 rows) = K Q^T on v_mfma_f32_16x16x32, lane
//     (c, g) = (l & 15, l >> 4) getting row c's scores of keys 4g .. 4g + 3; then
//     O^T (16 dims x 16 rows) += V^T P^T, the lane's scores of two key tiles
//     being its operand as they stand.  P enters as three terms of the data type
//     (split_pair): all 24 bits of the fp32 probability (of fp16's, what lies above
//     2^-41), with exact products and fp32 sums, and an infinite V gives the
//     infinity that an fp32 probability would.  V goes to LDS by direct copies
//     (16-byte pieces XOR-swizzled by row, 8 KB per wave, no barrier) and comes
//     back transposed (ds_read_b64_tr_b16).
//   * each wave first takes the own keys of two of the 16 rows, half a wave per
//     row, as the vector kernel does (D / 8 lanes of 16 bytes per key), appends
//     their new key and value, and adds the new key from registers at the end.
//   * every part leaves (m, l, acc) in LDS; after one barrier 32 threads per row
//     merge the 8 prefix parts and the row's own part.
//
// All row tiles of one (group, head) run on one XCD, so its L2 holds their
// prefix once.  Those 400 rows with 40 own keys: 56 us in the vector kernel, 15.5
// here (15.0 with two terms of P, 19.2 with fp32 P and V on
// v_mfma_f32_16x16x4_f32).  What bounds it then is the latency of two chains in a
// workgroup, 64-key chunks of the prefix and 16-key trips over the own keys (48
// own keys after a 3000-token prefix: 21 us for 100 rows, 25 for 400); from some
// 6000 rows of 8 heads the rows' own K/V from HBM.  The error against float64 is
// the vector kernel's (400 rows, 1024 + 40 keys: 1.646443e-3 of the norm in bf16,
// 2.064455e-4 in fp16, either kernel).
#include "dg_prefill.h"
#include "dg_rope_math.h"

namespace dg {

struct WideArgs {
  const void* q;   // the step's projections (B, 1, H, D)
  const void* kn;
  const void* vn;
  void* kc;        // the rows' cache pages, indexed by absolute position
  void* vc;
  void* y;
  int64_t qb, qh, knb, knh, vnb, vnh;
  int64_t kb, kt, kh, vb, vt, vh;
  int64_t yb, yh;
  PrefixRef pre;
  const void* freqs;
  int64_t fpos;
  const int* pos_dev;
  int pos, max_pos, qknorm;
  int B, H, units, tiles;  // tiles of 16 rows per group
  float scale_log2, lazy_raw;
};

constexpr int kWideWaves = 8;
constexpr int kWideRows = 16;

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 wbf16x8_t;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 wf16x8_t;

template <typename T>
__device__ __forceinline__ f32x4_t wide_mma(const u32x4_t& a, const u32x4_t& b, f32x4_t c) {
  if constexpr (__is_same(T, bf16_t))
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(wbf16x8_t, a), __builtin_bit_cast(wbf16x8_t, b),
                                                   c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(wf16x8_t, a), __builtin_bit_cast(wf16x8_t, b), c,
                                                  0, 0, 0);
}

// slot of 16-byte piece p of V row r in LDS: the 16 rows x 2 pieces of a
// transposing read fall on distinct banks
template <int D>
__device__ __forceinline__ int wide_slot(int p, int r) {
  if constexpr (D == 64) return p ^ (((r & 2) << 1) | ((r >> 2) & 3));
  else return p ^ (((r & 3) << 2) | ((r >> 2) & 3));
}

// maximum / sum over the half-wave's lanes of equal index in their group of LPK
template <int LPK>
__device__ __forceinline__ float half_sum_groups(float v) {
  if constexpr (LPK <= 8) v = v + dpp<kDppRowRor8>(v);
  float a, b;
  pair16(v, a, b);
  return a + b;
}

// A pair of probabilities as three terms of T whose sum they are, packed.
// bf16: the bits in three runs of eight, none negative, and the second and third
// at least 2^-126, so that no term of a probability above that makes a NaN of an
// infinite value and all three go into one sum (rounded terms, some of them
// negative, and a second sum for them took the registers of a wave's loads: 400
// rows over 1024 + 40 keys of 8 x 128 26.9 us, 25.0 so).
// fp16: each the rounding error of those before it, the second and third scaled by
// kRest, since the type's exponents end at 2^-24 (a first term's rounding error is
// at most 2^-12 of 2^kLazyLog2); they have a sum of their own.
constexpr float kRest = 65536.0f;
template <typename T>
__device__ __forceinline__ void split_pair(float p0, float p1, uint32_t (&term)[3]) {
#pragma clang fp contract(off)
  if constexpr (__is_same(T, bf16_t)) {
    typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
    auto top = [](float a, float b) __attribute__((always_inline)) {
      return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
    };
    auto rest = [](float a) __attribute__((always_inline)) {
      return a - __uint_as_float(__float_as_uint(a) & 0xffff0000u);
    };
    auto positive = [](uint32_t w) __attribute__((always_inline)) {
      const u16x2_t least = {0x0080, 0x0080};
      return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, w), least));
    };
    const float r0 = rest(p0), r1 = rest(p1);
    term[0] = top(p0, p1);
    term[1] = positive(top(r0, r1));
    term[2] = positive(top(rest(r0), rest(r1)));
  } else {
    RowRegs<T, 2> t0, t1;
    t0.w[0] = term[0] = pack_pair<T>(p0, p1);
    const float r0 = (p0 - elem<T, 2>(t0, 0)) * kRest, r1 = (p1 - elem<T, 2>(t0, 1)) * kRest;
    t1.w[0] = term[1] = pack_pair<T>(r0, r1);
    term[2] = pack_pair<T>(r0 - elem<T, 2>(t1, 0), r1 - elem<T, 2>(t1, 1));
  }
}

template <typename T, typename FT, int D>
__global__ __launch_bounds__(64 * kWideWaves, 4) void attn_wide_kernel(const WideArgs a) {
  constexpr int NC = D / 32;       // contraction steps of Q K^T
  constexpr int NB = D / 16;       // 16-dim blocks of O^T
  constexpr int KC = 4096 / D;     // keys of a chunk: 8 KB of V
  constexpr int NT = KC / 16;      // key tiles of a chunk
  constexpr int LPK = D / 8;       // lanes of a key row in the own-key part
  constexpr int KPH = 32 / LPK;    // keys per half-wave and slot
  constexpr int U = 4;             // slots per trip
  constexpr int PPR = D / 8;       // 16-byte pieces of a V row
  constexpr int kSums = __is_same(T, f16_t) ? 2 : 1;  // accumulators of a block of O^T
  constexpr int NR = kSums == 2 ? NB : 1;
  using Row = RowRegs<T, 8>;
  __shared__ __attribute__((aligned(16))) uint16_t stage[kWideWaves][4096];  // V, then the part's acc
  __shared__ __attribute__((aligned(16))) float own_acc[kWideRows][D];
  __shared__ float ml[kWideWaves + 1][kWideRows][2];

  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  // the host rounds the grid to a multiple of 8 workgroups: consecutive units
  // (the row tiles of one group and head) on one XCD
  const int unit = (blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
  if (unit >= a.units) return;  // the whole workgroup, before any barrier
  const int tile = unit % a.tiles;
  const int gh = unit / a.tiles;
  const int head = gh % a.H, grp = gh / a.H;
  const int b0 = grp * a.pre.group + tile * kWideRows;
  const int nrow = min(min(kWideRows, a.pre.group - tile * kWideRows), a.B - b0);  // rows of this tile
  if (nrow <= 0) return;  // a ragged last group's spare tiles

  const int pos = a.pos_dev != nullptr ? *a.pos_dev : a.pos;
  const bool pos_ok = pos >= a.pre.own_start && pos < a.max_pos;
  const int plen = min(a.pre.len, max(pos, 0));
  const int own0 = a.pre.len, own1 = min(pos, a.max_pos);  // cached own keys
  // a position outside the pages writes nothing and reads table row 0
  const FT* frow = static_cast<const FT*>(a.freqs) + (int64_t)(pos_ok ? pos : 0) * a.fpos;
  const float cl = a.scale_log2;

  // ---- this wave's rows 2 wv, 2 wv + 1: the new token and the own keys -------
  {
    const int half = lane >> 5, sub = lane % LPK, kg = (lane & 31) / LPK;
    const int r = 2 * wv + half, d0 = 8 * sub;
    const int64_t b = b0 + min(r, nrow - 1);  // spare rows re-read the last and store nothing
    float xq[8], xk[8], cs[8];
    Row qr, knew, vnew;
    load_vec<T, 8>(static_cast<const T*>(a.q) + b * a.qb + (int64_t)head * a.qh + d0, xq);
    load_vec<T, 8>(static_cast<const T*>(a.kn) + b * a.knb + (int64_t)head * a.knh + d0, xk);
    load_row<T, 8>(vnew, static_cast<const T*>(a.vn) + b * a.vnb + (int64_t)head * a.vnh + d0);
    load_vec<FT, 8>(frow + d0, cs);
    T* kp = static_cast<T*>(a.kc) + b * a.kb + (int64_t)head * a.kh + d0;
    T* vp = static_cast<T*>(a.vc) + b * a.vb + (int64_t)head * a.vh + d0;
    const int kt = (int)a.kt, vt = (int)a.vt;  // host: max_pos * stride < 2^31 bytes
    Row ka[U], va[U], kb[U], vb[U];
    auto load = [&](Row (&k)[U], Row (&v)[U], int t0) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (t0 + u * KPH >= own1) break;  // wave-uniform
        const int t = min(t0 + u * KPH + kg, own1 - 1);  // past the last key: it again, masked
        load_row<T, 8>(k[u], kp + t * kt);
        load_row<T, 8>(v[u], vp + t * vt);
      }
    };
    if (own0 < own1) load(ka, va, own0);
    // rope_qknorm_kernel's arithmetic (the cache's bits)
    rope_rotate<T, 8>(xq, cs);
    rope_rotate<T, 8>(xk, cs);
    if (a.qknorm) {
      qk_rms_norm<8, LPK, true>(xq, D);
      qk_rms_norm<8, LPK, true>(xk, D);
    }
    pack_row<T, 8>(qr, xq);
    pack_row<T, 8>(knew, xk);
    if (pos_ok && r < nrow && kg == 0) {
      store_row<T, 8>(kp + (int64_t)pos * kt, knew);
      store_row<T, 8>(vp + (int64_t)pos * vt, vnew);
    }
    float m = kNegInf, l = 0.f, acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
    auto raise = [&](float mt) __attribute__((always_inline)) {
      if (__builtin_amdgcn_ballot_w64(mt > m + a.lazy_raw) != 0) {
        const float mn = fmaxf(m, mt);
        const float alpha = m == kNegInf ? 0.f : __builtin_amdgcn_exp2f((m - mn) * cl);
        m = mn;
        l *= alpha;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] *= alpha;
      }
    };
    auto process = [&](Row (&k)[U], Row (&v)[U], int t0) __attribute__((always_inline)) {
      float s[U], mt = kNegInf;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        s[u] = kNegInf;
        if (t0 + u * KPH >= own1) continue;
        const float dot = group_sum_dpp<LPK>(slice_dot<T, 8>(qr, k[u]));
        s[u] = t0 + u * KPH + kg < own1 ? dot : kNegInf;
        mt = fmaxf(mt, s[u]);
      }
      // over the half-wave; a trip holds at least one key, so mt is finite
      mt = fmaxf(mt, dpp<kDppQuadXor1>(mt));
      mt = fmaxf(mt, dpp<kDppQuadXor2>(mt));
      mt = fmaxf(mt, dpp<kDppHalfMirror>(mt));
      mt = fmaxf(mt, dpp<kDppMirror>(mt));
      float x, y;
      pair16(mt, x, y);
      raise(fmaxf(x, y));
      const float moff = m * cl;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (t0 + u * KPH >= own1) continue;
        if (t0 + (u + 1) * KPH > own1) {  // wave-uniform: some lanes hold the last key again
          // its value weighs 0 there, and 0 times an infinity would be a NaN
          const bool own = t0 + u * KPH + kg < own1;
#pragma unroll
          for (int w = 0; w < Row::WORDS; ++w) v[u].w[w] = own ? v[u].w[w] : 0u;
        }
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u], cl, -moff));
        l += p;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = __builtin_fmaf(p, elem<T, 8>(v[u], e), acc[e]);
      }
    };
    constexpr int STEP = U * KPH;
    for (int t0 = own0; t0 < own1; t0 += 2 * STEP) {
      if (t0 + STEP < own1) load(kb, vb, t0 + STEP);
      process(ka, va, t0);
      if (t0 + STEP >= own1) break;
      if (t0 + 2 * STEP < own1) load(ka, va, t0 + 2 * STEP);
      process(kb, vb, t0 + STEP);
    }
    // the key groups share m; then the new key, once
    l = half_sum_groups<LPK>(l);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = half_sum_groups<LPK>(acc[e]);
    const float sn = group_sum_dpp<LPK>(slice_dot<T, 8>(qr, knew));
    raise(sn);
    const float pn = __builtin_amdgcn_exp2f(__builtin_fmaf(sn, cl, -(m * cl)));
    l += pn;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = __builtin_fmaf(pn, elem<T, 8>(vnew, e), acc[e]);
    if (kg == 0) {
      store_vec<float, 8>(&own_acc[r][d0], acc);
      if (sub == 0) {
        ml[kWideWaves][r][0] = m;
        ml[kWideWaves][r][1] = l;
      }
    }
  }

  // ---- the prefix: chunks wv, wv + 8, ... ------------------------------------
  u32x4_t qf[NC];  // Q^T operand: dims 32i + 8g .. of row c
  {
#pragma clang fp contract(off)
    const int64_t b = b0 + min(c, nrow - 1);
    const T* qrow = static_cast<const T*>(a.q) + b * a.qb + (int64_t)head * a.qh + 8 * g;
    float x[NC][8], s8[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      float cs[8], sq[8];
      load_vec<T, 8>(qrow + 32 * i, x[i]);
      load_vec<FT, 8>(frow + 32 * i + 8 * g, cs);
      rope_rotate<T, 8>(x[i], cs);
#pragma unroll
      for (int e = 0; e < 8; ++e) sq[e] = x[i][e] * x[i][e];
      // qk_rms_norm's pairwise tree over the row: the 8-element chunks of
      // lanes g ^ 1, then g ^ 2, then across i
      float u, v;
      pair16(tree_sum<8>(sq), u, v);
      pair32(u + v, u, v);
      s8[i] = u + v;
    }
    const float r = a.qknorm ? 1.0f / sqrtf(tree_sum<NC>(s8) / (float)D + FLT_EPSILON) : 1.0f;
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
      for (int w = 0; w < 4; ++w) qf[i][w] = pack_pair<T>(x[i][2 * w] * r, x[i][2 * w + 1] * r);
  }
  const T* kpre = static_cast<const T*>(a.pre.k) + (int64_t)grp * a.pre.kb + (int64_t)head * a.pre.kh;
  const T* vpre = static_cast<const T*>(a.pre.v) + (int64_t)grp * a.pre.vb + (int64_t)head * a.pre.vh;
  const int kt = (int)a.kt, vt = (int)a.vt;
  // rows past the prefix lie past the resource's range and read as zeros
  const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(vpre), 0, plen > 0 ? ((plen - 1) * vt + D) * 2 : 0, kBufferWord3);
  uint16_t* const st = stage[wv];
  const int vrow = lane / PPR, vslot = lane % PPR;
  const int t16 = lane & 15;

  float m = kNegInf, l = 0.f;
  f32x4_t o[NB], rest[NR];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) o[nb] = rest[nb % NR] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int k0 = wv * KC; k0 < plen; k0 += kWideWaves * KC) {
    // every lane is done reading the chunk before (its products waited for
    // the reads) when the copies of this one go out
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = i * (64 / PPR) + vrow;
      lds_copy16_buf(vrs, (row * vt + 8 * wide_slot<D>(vslot, row)) * 2, k0 * vt * 2, st + 512 * i);
    }
    f32x4_t s[NT];
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const T* krow = kpre + (int64_t)min(k0 + 16 * u + c, plen - 1) * kt + 8 * g;  // past the last: masked
      s[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < NC; ++i) s[u] = wide_mma<T>(*reinterpret_cast<const u32x4_t*>(krow + 32 * i), qf[i], s[u]);
    }
    mfma_settle(s);
    if (k0 + KC > plen) {
#pragma unroll
      for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (k0 + 16 * u + 4 * g + r >= plen) s[u][r] = kNegInf;
    }
    float mt = s[0][0];
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) mt = fmaxf(mt, s[u][r]);
    float x, y;
    pair16(mt, x, y);
    mt = fmaxf(x, y);
    pair32(mt, x, y);
    mt = fmaxf(x, y);
    if (__builtin_amdgcn_ballot_w64(mt > m + a.lazy_raw) != 0) {
      const float mn = fmaxf(m, mt);
      const float alpha = m == kNegInf ? 0.f : __builtin_amdgcn_exp2f((m - mn) * cl);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          o[nb][r] *= alpha;
          if constexpr (kSums == 2) rest[nb][r] *= alpha;
        }
    }
    const float moff = m * cl;
    u32x4_t p[NT / 2][3];  // P^T operands of 32 keys: the three terms
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][2 * w], cl, -moff));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][2 * w + 1], cl, -moff));
        l += p0;
        l += p1;
        uint32_t term[3];
        split_pair<T>(p0, p1, term);
#pragma unroll
        for (int k = 0; k < 3; ++k) p[u / 2][k][2 * (u & 1) + w] = term[k];
      }
    // this wave's V copies are in LDS
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int t = 0; t < NT / 2; ++t)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        // V^T: column 16nb + t16 of keys 32t + 4g .. and 32t + 16 + 4g ..
        uint2 vv[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int row = 32 * t + 16 * u + 4 * g + (t16 >> 2);
          const int col = 16 * nb + 4 * (t16 & 3);
          vv[u] = lds_read_tr16(st + row * D + 8 * wide_slot<D>(col >> 3, row) + (col & 7));
        }
        const u32x4_t vf = {vv[0].x, vv[0].y, vv[1].x, vv[1].y};
        o[nb] = wide_mma<T>(vf, p[t][0], o[nb]);
        f32x4_t& low = kSums == 2 ? rest[nb % NR] : o[nb];
        low = wide_mma<T>(vf, p[t][1], low);
        low = wide_mma<T>(vf, p[t][2], low);
      }
  }
  float x, y;
  pair16(l, x, y);
  l = x + y;
  pair32(l, x, y);
  l = x + y;
  // the part's acc over the wave's V (read for the last time), rows of D floats
  // with 16-byte units XORed by row
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  constexpr int UPR = D / 4;  // 16-byte units of a row
  float* part = reinterpret_cast<float*>(st);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    float w[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      // a value that is not finite has made the first terms' sum so, and a sum
      // of the others' own (zero or negative for some keys) a NaN
      const bool finite = __builtin_fabsf(o[nb][r]) < __builtin_huge_valf();
      w[r] = kSums == 2 && finite ? __builtin_fmaf(rest[nb % NR][r], 1.0f / kRest, o[nb][r]) : o[nb][r];
    }
    store_vec<float, 4>(part + c * D + 4 * ((4 * nb + g) ^ (c & (UPR - 1))), w);
  }
  if (g == 0) {
    ml[wv][c][0] = m;
    ml[wv][c][1] = l;
  }
  __syncthreads();

  // ---- merge: 32 threads per row, D / 32 dims each ----------------------------
  constexpr int DP = D / 32;
  const int r = threadIdx.x >> 5, d = DP * (threadIdx.x & 31);
  if (r >= nrow) return;  // no barrier follows
  float M = ml[kWideWaves][r][0];  // the new key: finite
#pragma unroll
  for (int w = 0; w < kWideWaves; ++w) M = fmaxf(M, ml[w][r][0]);
  float L = 0.f, out[DP];
#pragma unroll
  for (int i = 0; i < DP; ++i) out[i] = 0.f;
#pragma unroll
  for (int w = 0; w <= kWideWaves; ++w) {
    const float mw = ml[w][r][0];
    const float f = mw == kNegInf ? 0.f : __builtin_amdgcn_exp2f((mw - M) * cl);
    L += f * ml[w][r][1];
    const float* src = w < kWideWaves ? reinterpret_cast<const float*>(stage[w < kWideWaves ? w : 0]) + r * D +
                                            4 * ((d >> 2) ^ (r & (UPR - 1))) + (d & 3)
                                      : &own_acc[r][d];
#pragma unroll
    for (int i = 0; i < DP; ++i) out[i] += f * src[i];
  }
  const float inv = 1.0f / L;
#pragma unroll
  for (int i = 0; i < DP; ++i) out[i] *= inv;
  store_vec<T, DP>(static_cast<T*>(a.y) + (int64_t)(b0 + r) * a.yb + (int64_t)head * a.yh + d, out);
}

namespace {
bool w16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
}  // namespace

// Groups of at least 16 rows with a prefix, 16-bit data at head_dim 64 or 128,
// 16-byte aligned rows, and a prefix that pays.  The vector kernel splits every
// row's keys and reads the prefix per (row, head); this one walks a row's own keys
// with half a wave and the prefix with eight, a fixed chain that only what is
// saved, (rows * heads * P) key reads, can repay.  Both sides of the line, 8 heads
// of 64, us with the vector kernel -> here (D = 128 alike, both about twice):
//   rows * heads * P >= 3300 * own_max + 200000 (own_max: the own pages' room)
//     1 x 100 rows, P  200, own  48 of   96:   9.5 ->   9.1 below the line
//     1 x 100 rows, P 1024, own 250 of  256:  30.6 ->  24.4 just below
//     1 x  20 rows, P 1024, own 250 of  256:  11.4 ->  22.1 below
//    32 x  32 rows, P   64, own  48 of   96:  24.7 ->  21.8 just above
//     2 x  32 rows, P 1100, own  48 of   96:  14.8 ->  12.9 just above
//    32 x  32 rows, P 1024, own 1000 of 1024: 452 ->  389   above
//     4 x 100 rows, P 3000, own   8 of   96:   142 ->  21.7 above
//   rows * heads >= 320: 20 rows x 8, P 3000, own 48 of 96: 18.7 -> 20.9
//   2 P >= own_max: 64 x 100 rows, P 64, own 250 of 256: 564 -> 590
bool wide_step_applicable(int B, int H, int D, int dtype, const PrefixRef& pre, int max_pos, const void* q,
                          const dg_stride3* q_st, const void* k, const dg_stride3* k_st, const void* v,
                          const dg_stride3* v_st, const void* kc, const dg_stride3* kc_st, const void* vc,
                          const dg_stride3* vc_st, const void* freqs, int64_t fpos, int fdtype, const void* y,
                          const dg_stride3* y_st, float scale) {
  if ((dtype != DG_BF16 && dtype != DG_F16) || (D != 64 && D != 128)) return false;
  if (pre.group < kWideRows || pre.len < kWideRows || !(scale > 0.f)) return false;
  if (fdtype != dtype && fdtype != DG_F32) return false;
  const int64_t tiles = (pre.group + kWideRows - 1) / kWideRows;
  const int64_t units = ((int64_t)B + pre.group - 1) / pre.group * tiles * H;
  if (units > 0x7fffffffLL - 8) return false;
  const int64_t own_max = max_pos - pre.len, pairs = (int64_t)B * H;
  if (pairs < 320 || pairs * pre.len < 3300 * own_max + 200000 || 2LL * pre.len < own_max) return false;
  if (kc_st->t < 0 || vc_st->t < 0) return false;
  const int64_t span = (int64_t)max_pos * (kc_st->t > vc_st->t ? kc_st->t : vc_st->t) + D;
  if (span * 2 >= (int64_t)1 << 31) return false;
  auto st = [](const dg_stride3* s) { return s->b % 8 == 0 && s->h % 8 == 0 && s->t % 8 == 0; };
  const int64_t fes = fdtype == DG_F32 ? 4 : 2;
  return w16(q) && w16(k) && w16(v) && w16(kc) && w16(vc) && w16(pre.k) && w16(pre.v) && w16(freqs) && w16(y) &&
         st(q_st) && st(k_st) && st(v_st) && st(kc_st) && st(vc_st) && st(y_st) && pre.kb % 8 == 0 &&
         pre.kh % 8 == 0 && pre.vb % 8 == 0 && pre.vh % 8 == 0 && fpos >= 0 && (fpos * fes) % 16 == 0;
}

int wide_decode_step(int B, int H, int D, int dtype, const void* q, const dg_stride3* q_st, const void* k,
                     const dg_stride3* k_st, const void* v, const dg_stride3* v_st, void* kc, const dg_stride3* kc_st,
                     void* vc, const dg_stride3* vc_st, const void* freqs, int64_t fpos, int fdtype, int pos,
                     const int* pos_dev, int max_pos, void* y, const dg_stride3* y_st, float scale,
                     const PrefixRef& pre, int qknorm, hipStream_t s) {
  WideArgs a{};
  a.q = q; a.kn = k; a.vn = v; a.kc = kc; a.vc = vc; a.y = y;
  a.qb = q_st->b; a.qh = q_st->h;
  a.knb = k_st->b; a.knh = k_st->h;
  a.vnb = v_st->b; a.vnh = v_st->h;
  a.kb = kc_st->b; a.kt = kc_st->t; a.kh = kc_st->h;
  a.vb = vc_st->b; a.vt = vc_st->t; a.vh = vc_st->h;
  a.yb = y_st->b; a.yh = y_st->h;
  a.pre = pre;
  a.freqs = freqs; a.fpos = fpos;
  a.pos_dev = pos_dev; a.pos = pos; a.max_pos = max_pos; a.qknorm = qknorm;
  a.B = B; a.H = H;
  a.tiles = (pre.group + kWideRows - 1) / kWideRows;
  a.units = (int)(((int64_t)B + pre.group - 1) / pre.group * a.tiles * H);
  a.scale_log2 = scale * 1.44269504088896340736f;
  a.lazy_raw = kLazyLog2 / a.scale_log2;
  const dim3 grid(((unsigned)a.units + 7u) & ~7u), block(64 * kWideWaves);
#define DG_WIDE(T, FT)                                                                     \
  do {                                                                                     \
    if (D == 64) hipLaunchKernelGGL((attn_wide_kernel<T, FT, 64>), grid, block, 0, s, a);  \
    else hipLaunchKernelGGL((attn_wide_kernel<T, FT, 128>), grid, block, 0, s, a);         \
  } while (0)
  if (dtype == DG_BF16) {
    if (fdtype == DG_F32) DG_WIDE(bf16_t, float);
    else DG_WIDE(bf16_t, bf16_t);
  } else {
    if (fdtype == DG_F32) DG_WIDE(f16_t, float);
    else DG_WIDE(f16_t, f16_t);
  }
#undef DG_WIDE
  return check_launch("attn_wide_kernel");
}

}  // namespace dg
