// A small model's layer around its attention, in one launch to either side of
// it (n_embd 64 or 128; fp32, bf16, fp16):
//
//   block_in_kernel   the attention's Block-AttnRes mixture over the committed
//                     blocks and the partial sum with its RMSNorm (block.py:
//                     95-97), and the q/k/v/g projections of the result
//                     (mha.py:34-43)
//   block_out_kernel  a = y * sigmoid(g); attn_out = a @ W_proj^T (mha.py:84-85);
//                     the partial sum (attn_out, or partial_in + attn_out inside
//                     a block); the MLP's mixture over the committed blocks
//                     and that partial, its norm; the FFN (C -> 4C, clamped
//                     SwiGLU, 2C -> C) and the residual (block.py:98-106,
//                     feed_forward.py:10-14)
//
// A workgroup of 8 waves takes RT groups of 16 token rows at a time.  The
// stages meet in LDS (rows padded by 16 bytes, so the 16 rows of a matrix-core
// operand read fall on different banks); row work gives a row 16 lanes; every
// GEMM is a sequence of 16 x 16 output tiles on the matrix cores (qk_mfma's lane
// mapping: lane (c, g) feeds weight row 16t + c and token row c with the
// contiguous quarter g of the contraction, and gets back token row c's outputs
// 16t + 4g .. 16t + 4g + 3).  A wave's weight fragments are fetched once, with
// everything else the kernel reads, before the first stage, and stay in
// registers; at more rows than fill the chip a workgroup walks several groups
// with the same fragments, the next group's rows in flight under the current
// one's products.  fp32 at n_embd 128 fetches its FFN fragments as it goes (256
// registers would not hold them).  Instances for more than four committed blocks
// hold eight sources: after the attention some of them keep registers in scratch,
// with 32-row groups up to 39 of a lane's, at n_embd 64 in fp32 with the next
// layer's projections behind them up to 19.
//
// RT = 1 while every group of 16 has a workgroup of its own on the chip: the
// launch is bound by latency (one round trip to memory, the stages' chain), and
// half the waves sit out the row work.  RT = 2 beyond: all do, and the vector
// ALU's share (row work and SwiGLU, more than the products' in fp32) halves --
// but for the instances whose 32-row form loses by its scratch (both sides at
// launch_block_out_ns).
// Measured in captured graphs, us, 3 sources, two of them the same rows
// (before: the mixture's launch and a library GEMM; 4 waves per 16 rows after
// the attention):
//                         before the attention   after it
//   n_embd 64, fp32,    100 rows   17.7 ->  4.2    9.0 ->  7.5
//                      6400 rows   13.6 ->  8.8   13.0 -> 12.5
//                     35328 rows   39.8 -> 26.4   41.1 -> 44.0
//   n_embd 64, bf16,   1850 rows   10.4 ->  3.9    7.8 ->  5.9
//                      6400 rows   11.5 ->  5.8   10.9 ->  8.2
//                     35328 rows   23.6 -> 15.3   31.4 -> 24.7
//   n_embd 128, fp32,   100 rows   10.4 ->  5.7   22.5 -> 18.9
//                     35328 rows    105 -> 58.4    157 -> 126
//   n_embd 128, bf16,   100 rows   10.2 ->  4.2   12.6 -> 10.5
//                     35328 rows   46.8 -> 25.3   62.6 -> 41.3
// The products need 8.4 us of the fp32 matrix cores before the attention and
// 14.7 after it at 35328 rows of 64.
//
// Every intermediate is rounded to T where the torch sequence rounds it -- the
// gate as gate_kernel, each GEMM's fp32 sum once, the mixture as
// attn_res_norm_kernel, the SwiGLU as swiglu_kernel, the residual adds -- so
// 16-bit types follow the same rounding steps; only the GEMMs' summation order
// differs from hipBLASLt's.  A row's result does not depend on the number of
// rows.
#include "dg_rows.h"

namespace dg {

constexpr int kLayerRows = 16;  // rows of a matrix-core tile
constexpr int kLayerWaves = 8;
constexpr int kLayerThreads = 64 * kLayerWaves;
constexpr int kRowLanes = 16;   // lanes of a row

// LDS row stride (elements) of a K-wide operand matrix: 16 bytes of padding
template <typename T, int K>
constexpr int lds_ld() {
  return K + 16 / (int)sizeof(T);
}

// A lane's weight fragment of one 16 x 16 output tile over a K-long
// contraction: weight row 16t + c (c = lane & 15), the contiguous quarter
// g = lane >> 4 of the contraction, in chunks of 16 elements.
template <typename T, int K>
struct TileW {
  static constexpr int CQ = K / 4;  // contraction elements of a lane's quarter
  static constexpr int NCH = CQ / 16;
  static_assert(CQ % 16 == 0, "contraction chunking");
  RowRegs<T, 16> r[NCH];
};

template <typename T, int K>
__device__ __forceinline__ void load_tile_w(RowRegs<T, 16>* r, const T* __restrict__ w, int64_t w_ld, int t, int lane) {
  const int c = lane & 15, g = lane >> 4;
  const T* wr = w + (int64_t)(16 * t + c) * w_ld + g * TileW<T, K>::CQ;
#pragma unroll
  for (int i = 0; i < TileW<T, K>::NCH; ++i) load_row<T, 16>(r[i], wr + 16 * i);
}

// Products of NT tiles against the token rows of the LDS matrix x; the tiles'
// chains are interleaved, each in contraction order.
template <typename T, int K, int NT>
__device__ __forceinline__ void layer_tiles(f32x4_t (&acc)[NT], const RowRegs<T, 16>* const (&f)[NT], const T* x,
                                            int lane) {
  const T* xr = x + (lane & 15) * lds_ld<T, K>() + (lane >> 4) * TileW<T, K>::CQ;
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  constexpr int SW = sizeof(T) == 4 ? 1 : 2;  // words per step: one fp32, four 16-bit elements
  constexpr int LW = 4 * SW;                  // words of x read at a time: four steps
#pragma unroll
  for (int k = 0; k < TileW<T, K>::NCH * RowRegs<T, 16>::WORDS; k += LW) {
    RowRegs<T, LW * 4 / (int)sizeof(T)> xo;
    load_row(xo, xr + k * 4 / (int)sizeof(T));
#pragma unroll
    for (int s = 0; s < LW; s += SW) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        RowRegs<T, sizeof(T) == 4 ? 1 : 4> kw, qw;
#pragma unroll
        for (int w = 0; w < SW; ++w) {
          kw.w[w] = f[t][(k + s) / RowRegs<T, 16>::WORDS].w[(k + s) % RowRegs<T, 16>::WORDS + w];
          qw.w[w] = xo.w[s + w];
        }
        acc[t] = qk_mfma<T, sizeof(T) == 4 ? 1 : 4>(kw, qw, acc[t]);
      }
    }
  }
}

// Sources of a mixture held in registers: every one of an instance for up to 8
// (NS), the first 8 of the general instance.
template <int NS>
constexpr int layer_held() {
  return NS < 8 ? NS : 8;
}

// rms_norm(block_attn_res(V, w)) of a row spread over G = 16 lanes of CH
// elements, with attn_res_norm_kernel's roundings: the mixture over nmem
// sources of memory (held; from the ninth on read where used, src and ld at
// this lane's columns of the row) and, with LAST, the slice `last` after them.
// Held sources past nmem are zeros: their sums are taken with the others'
// (independent chains, no branch between them) and left out of the softmax.
// Lane n of the row keeps scores n and n + 16, so the row takes one
// exponential and one quotient for up to 16 sources.
template <typename T, int CH, int NS, bool LAST>
__device__ __forceinline__ void layer_mixture(const RowRegs<T, CH> (&held)[layer_held<NS>()], int nmem,
                                              const void* const* src, const int64_t* ld, int64_t row, int c0,
                                              const RowRegs<T, CH>& last, const RowRegs<T, CH>& w, int C,
                                              float (&h)[CH]) {
#pragma clang fp contract(off)
  constexpr int G = kRowLanes, HELD = layer_held<NS>();
  constexpr int NP = NS + (LAST ? 1 : 0) > G ? 2 : 1;  // scores a lane keeps
  const int sub = threadIdx.x & (G - 1);
  const int quarter = (threadIdx.x >> 4) & 3;  // the row's 16 lanes of the wave
  const int nsrc = nmem + (LAST ? 1 : 0);
  auto score = [&](const RowRegs<T, CH>& x) __attribute__((always_inline)) {
    const float r = row_factor(score_sum<G>(slice_squares<T, CH>(x)), C);
    return rt<T>(score_sum<G>(slice_score<T, CH>(x, r, w)));
  };
  auto get = [&](int n, RowRegs<T, CH>& x) __attribute__((always_inline)) {
    load_row<T, CH>(x, static_cast<const T*>(src[n]) + row * ld[n] + c0);
  };
  float sc[NP];
#pragma unroll
  for (int k = 0; k < NP; ++k) sc[k] = -INFINITY;
  auto keep = [&](int n, float v) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < NP; ++k) sc[k] = sub + G * k == n ? v : sc[k];
  };
#pragma unroll
  for (int n = 0; n < HELD; ++n) {
    const float v = score(held[n]);
    keep(n < nmem ? n : -1, v);
  }
  if constexpr (NS > HELD) {
#pragma unroll 1
    for (int n = HELD; n < nmem; ++n) {
      RowRegs<T, CH> x;
      get(n, x);
      keep(n, score(x));
    }
  }
  if constexpr (LAST) keep(nmem, score(last));
  float mx = sc[0];
#pragma unroll
  for (int k = 1; k < NP; ++k) mx = fmaxf(mx, sc[k]);
  mx = fmaxf(mx, dpp<kDppQuadXor1>(mx));
  mx = fmaxf(mx, dpp<kDppQuadXor2>(mx));
  mx = fmaxf(mx, dpp<kDppHalfMirror>(mx));
  mx = fmaxf(mx, dpp<kDppMirror>(mx));
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < NP; ++k) {
    // a NaN score makes the row NaN, as its exponential would
    sc[k] = sub + G * k < nsrc ? expf(sc[k] - mx) : 0.f;
    sum += sc[k];
  }
  sum = group_sum_dpp<G>(sum);
#pragma unroll
  for (int k = 0; k < NP; ++k) sc[k] = rt<T>(sc[k] / sum);
  auto weight = [&](int n) __attribute__((always_inline)) {
    const int p = __float_as_int(NP == 1 || n < G ? sc[0] : sc[NP - 1]);
    const int l = n & (G - 1);
    const float p0 = __int_as_float(__builtin_amdgcn_readlane(p, l));
    const float p1 = __int_as_float(__builtin_amdgcn_readlane(p, 16 + l));
    const float p2 = __int_as_float(__builtin_amdgcn_readlane(p, 32 + l));
    const float p3 = __int_as_float(__builtin_amdgcn_readlane(p, 48 + l));
    return quarter < 2 ? (quarter == 0 ? p0 : p1) : (quarter == 2 ? p2 : p3);
  };
#pragma unroll
  for (int i = 0; i < CH; ++i) h[i] = 0.f;
#pragma unroll
  for (int n = 0; n < HELD; ++n) {
    if (n >= nmem) continue;  // uniform
    slice_add<T, CH>(h, weight(n), held[n]);
  }
  if constexpr (NS > HELD) {
#pragma unroll 1
    for (int n = HELD; n < nmem; ++n) {
      RowRegs<T, CH> x;
      get(n, x);
      slice_add<T, CH>(h, weight(n), x);
    }
  }
  if constexpr (LAST) slice_add<T, CH>(h, weight(nmem), last);
#pragma unroll
  for (int i = 0; i < CH; ++i) h[i] = rt<T>(h[i]);
  row_rms<CH, G>(h, C);
}

template <typename T, int CH, int HELD>
__device__ __forceinline__ void load_held(RowRegs<T, CH> (&held)[HELD], const void* const* src, const int64_t* ld,
                                          int nmem, bool dup, int64_t row, int c0) {
#pragma unroll
  for (int n = 0; n < HELD; ++n) {
    if (n >= nmem) {  // uniform
#pragma unroll
      for (int i = 0; i < RowRegs<T, CH>::WORDS; ++i) held[n].w[i] = 0u;
    } else if (n == 1 && dup) {
      held[1] = held[0];
    } else {
      load_row<T, CH>(held[n], static_cast<const T*>(src[n]) + row * ld[n] + c0);
    }
  }
}

struct BlockInArgs {
  const void* src[kMaxResSources];  // the mixture's sources; with w_mix null one, the normalised rows
  int64_t ld[kMaxResSources];
  const void* w_mix;  // (C,), or null: src[0] goes into the projection as it is
  const void* w;      // (4C, C)
  void* out;          // (M, 4C)
  int64_t w_ld, out_ld, M;
  int nsrc, dup;      // dup: source 1 is source 0, read once
  // the embedding's form: row r of src[0] is row ids[r] of the table of V rows
  // (ids outside it give NaN rows); its norm goes to x (M, C), the norm of that
  // as stored into the projection
  const int64_t* ids;
  int64_t V;
  void* x;
  int64_t x_ld;
};

// SPLIT: the output columns are dealt to SPLIT workgroups (blockIdx.y), each
// with the mixture of its own, where a few groups would leave CUs idle.
// EMBED: the embedding's form.
template <typename T, int C, int NS, int RT, int SPLIT, bool EMBED>
__global__ __launch_bounds__(kLayerThreads, C == 64 ? 4 : 2) void block_in_kernel(const BlockInArgs a) {
#pragma clang fp contract(off)
  static_assert(!EMBED || RT == 1, "a workgroup gathers one group of rows");
  constexpr int LDC = lds_ld<T, C>();
  constexpr int CH = C / kRowLanes;
  constexpr int NT = 4 * C / 16 / kLayerWaves / SPLIT;  // output tiles per wave
  constexpr int HELD = layer_held<NS>();
  constexpr int ROWS = RT * kLayerRows;
  __shared__ __attribute__((aligned(16))) T xn[2][ROWS * LDC];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int gr = threadIdx.x / kRowLanes, gc0 = (threadIdx.x % kRowLanes) * CH;
  const bool rows_here = gr < ROWS;  // wave-uniform
  const int t0 = NT * (kLayerWaves * (SPLIT == 1 ? 0 : blockIdx.y) + wv);  // the wave's first tile
  const int ngroups = (int)((a.M + ROWS - 1) / ROWS);

  RowRegs<T, CH> held[HELD], wmix;
  auto load_rows = [&](int group) __attribute__((always_inline)) {
    // rows past M: a finite copy, never stored
    const int64_t row = min((int64_t)group * ROWS + gr, a.M - 1);
    load_held<T, CH, HELD>(held, a.src, a.ld, a.nsrc, a.dup != 0, row, gc0);
  };
  int group = blockIdx.x;
  bool bad_id = false;
  if constexpr (EMBED) {
    if (rows_here) {
      const int64_t id = a.ids[min((int64_t)group * ROWS + gr, a.M - 1)];
      bad_id = id < 0 || id >= a.V;
      load_row<T, CH>(held[0], static_cast<const T*>(a.src[0]) + (bad_id ? 0 : id) * a.ld[0] + gc0);
    }
  } else {
    if (rows_here) load_rows(group);
  }
#pragma unroll
  for (int i = 0; i < RowRegs<T, CH>::WORDS; ++i) wmix.w[i] = 0u;
  if (!EMBED && a.w_mix != nullptr) load_row<T, CH>(wmix, static_cast<const T*>(a.w_mix) + gc0);
  TileW<T, C> w[NT];
  const RowRegs<T, 16>* wf[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    load_tile_w<T, C>(w[j].r, static_cast<const T*>(a.w), a.w_ld, t0 + j, lane);
    wf[j] = w[j].r;
  }
  // keep the scheduler from sinking the loads toward their uses
  __builtin_amdgcn_sched_barrier(0);

  for (int buf = 0;; buf ^= 1) {
    // every wave left the products of the group before last at the last barrier
    if (EMBED && rows_here) {
      // rms_norm(table row), stored, and the norm of the stored row
      float x[CH];
#pragma unroll
      for (int i = 0; i < CH; ++i) x[i] = bad_id ? __builtin_nanf("") : elem<T, CH>(held[0], i);
      row_rms<CH, kRowLanes>(x, C);
      const int64_t row = (int64_t)group * ROWS + gr;
      if (row < a.M && (SPLIT == 1 || blockIdx.y == 0))
        store_vec<T, CH>(static_cast<T*>(a.x) + row * a.x_ld + gc0, x);
#pragma unroll
      for (int i = 0; i < CH; ++i) x[i] = rt<T>(x[i]);
      row_rms<CH, kRowLanes>(x, C);
      store_vec<T, CH>(xn[buf] + gr * LDC + gc0, x);
    } else if (rows_here) {
      if (a.w_mix != nullptr) {  // uniform
        float h[CH];
        const int64_t row = min((int64_t)group * ROWS + gr, a.M - 1);
        layer_mixture<T, CH, NS, false>(held, a.nsrc, a.src, a.ld, row, gc0, wmix, wmix, C, h);
        store_vec<T, CH>(xn[buf] + gr * LDC + gc0, h);
      } else {
        store_row<T, CH>(xn[buf] + gr * LDC + gc0, held[0]);
      }
    }
    __syncthreads();
    const int next = RT == 1 ? ngroups : group + (int)gridDim.x;  // RT = 1: a workgroup per group
    if (rows_here && next < ngroups) load_rows(next);
#pragma unroll
    for (int rt0 = 0; rt0 < RT; ++rt0) {
      f32x4_t acc[NT];
      layer_tiles<T, C, NT>(acc, wf, xn[buf] + rt0 * kLayerRows * LDC, lane);
      const int64_t row = (int64_t)group * ROWS + rt0 * kLayerRows + c;
      if (row < a.M) {
        T* o = static_cast<T*>(a.out) + row * a.out_ld + 16 * t0 + 4 * g;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const float v[4] = {acc[j][0], acc[j][1], acc[j][2], acc[j][3]};
          store_vec<T, 4>(o + 16 * j, v);
        }
      }
    }
    group = next;
    if (group >= ngroups) break;
  }
}

struct BlockOutArgs {
  const void* y;        // (M, C) attention output (before the gate)
  const void* g;        // (M, C) gate logits
  const void* w_proj;   // (C, C)
  const void* pin;      // (M, C) partial sum entering the layer; null when the layer commits it
  const void* blk[kMaxResSources];  // committed blocks (the MLP mixture's first sources)
  int64_t blk_ld[kMaxResSources];
  const void* w_mix;    // (C,)
  const void* w_up;     // (4C, C)
  const void* w_down;   // (C, 2C)
  void* out;            // (M, C) partial sum leaving the layer
  void* xn;             // (M, C) rms_norm(out) as stored, or null
  int64_t y_ld, g_ld, wp_ld, pin_ld, wu_ld, wd_ld, out_ld, xn_ld, M;
  int nblk, dup;        // dup: block 1 is block 0, read once
  float alpha, limit;
  // what follows the layer (its tail)
  const void* t_mix;    // (C,) the next layer's pseudo-query (kTailIn)
  const void* t_w;      // (t_n, C): the next layer's projections, or the lm_head's table (kTailHead)
  void* t_out;          // (M, t_n)
  int64_t* t_ids;       // (M,) first maximum of each logits row, or null
  int64_t t_wld, t_old;
  int t_n;
  float t_cap;          // logit soft cap, 0: none
  int* t_advance;       // device position to move on by one after the step, or null (kTailHead)
};

// What a launch adds after the layer.  At few rows every launch is a chain of
// latencies, and the next one's rows are the rows this workgroup holds: its
// weights are fetched under the FFN-down products instead.  n_embd 64 in fp32,
// 32 rows, us: the layer 7.5 and the next one's projections 4.1 in one launch
// 9.7, the head (5.7) 10.0; the embedding (4.1) and layer 0's projections 3.6.
enum LayerTail {
  kTailNone,
  kTailIn,    // block_in_kernel of the next layer, whose sources are the committed blocks and out
  kTailHead,  // lm_head_kernel over rms_norm(out)
};

// NS: the most committed blocks of the instance.
template <typename T, int C, int NS, int RT, LayerTail TAIL>
__global__ __launch_bounds__(kLayerThreads, C == 64 ? 4 : 2) void block_out_kernel(const BlockOutArgs a) {
#pragma clang fp contract(off)
  static_assert(TAIL == kTailNone || (RT == 1 && (C == 64 || sizeof(T) == 2)), "a tail follows one group of rows");
  constexpr int LDC = lds_ld<T, C>(), LDH = lds_ld<T, 2 * C>();
  constexpr int CH = C / kRowLanes;
  constexpr int ROWS = RT * kLayerRows;
  constexpr int NUP = 4 * C / 16 / kLayerWaves;  // FFN-up tiles per wave
  constexpr int NCT = C / 16;                    // c_proj tiles and FFN-down tiles: one for a wave at most
  constexpr int HELD = layer_held<NS>();
  // every fragment in registers, but for fp32 at n_embd 128
  constexpr bool kResident = C == 64 || sizeof(T) == 2;
  // fp32 at n_embd 64 fetches its FFN-down fragments behind the mixture, under
  // the FFN-up products: held through the mixture they spill (128 registers)
  constexpr bool kLateDown = C == 64 && sizeof(T) == 4;
  __shared__ __attribute__((aligned(16))) T ga[ROWS * LDC];  // gated attention output, then xn
  __shared__ __attribute__((aligned(16))) T pm[ROWS * LDC];  // the partial sum after the attention
  __shared__ __attribute__((aligned(16))) T hh[ROWS * LDH];  // SwiGLU output
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int gr = threadIdx.x / kRowLanes, gc0 = (threadIdx.x % kRowLanes) * CH;
  const bool rows_here = gr < ROWS;  // wave-uniform
  const int ngroups = (int)((a.M + ROWS - 1) / ROWS);
  const T* w_up = static_cast<const T*>(a.w_up);
  const T* w_down = static_cast<const T*>(a.w_down);
  // c_proj tiles go to the first waves, FFN-down tiles to the last (at n_embd
  // 64 a wave has one or the other)
  const int tp = wv, td = wv - (kLayerWaves - NCT);
  const bool has_p = tp < NCT, has_d = td >= 0;

  // The rows of a group, in the order the stages use them.
  RowRegs<T, CH> y, gl, held[HELD], wmix;
  RowRegs<T, 4> pin[RT];  // zeros when the layer commits its input
#pragma unroll
  for (int k = 0; k < RT; ++k)
#pragma unroll
    for (int i = 0; i < RowRegs<T, 4>::WORDS; ++i) pin[k].w[i] = 0u;
  auto load_rows = [&](int group) __attribute__((always_inline)) {
    // rows past M: a finite copy, never stored
    if (rows_here) {
      const int64_t row = min((int64_t)group * ROWS + gr, a.M - 1);
      load_row<T, CH>(y, static_cast<const T*>(a.y) + row * a.y_ld + gc0);
      load_row<T, CH>(gl, static_cast<const T*>(a.g) + row * a.g_ld + gc0);
      load_held<T, CH, HELD>(held, a.blk, a.blk_ld, a.nblk, a.dup != 0, row, gc0);
    }
    if (has_p && a.pin != nullptr) {  // uniform
#pragma unroll
      for (int k = 0; k < RT; ++k) {
        const int64_t crow = min((int64_t)group * ROWS + k * kLayerRows + c, a.M - 1);
        load_row<T, 4>(pin[k], static_cast<const T*>(a.pin) + crow * a.pin_ld + 16 * tp + 4 * g);
      }
    }
  };
  int group = blockIdx.x;
  load_rows(group);
  // one array for the c_proj and the FFN-down fragments where a wave has one
  // of them only
  constexpr int NPC = TileW<T, C>::NCH, NDC = TileW<T, 2 * C>::NCH;
  constexpr bool kShared = NCT < kLayerWaves;
  RowRegs<T, 16> wpd[kShared ? NDC : NPC], wd[kShared ? 1 : NDC];
  if (has_p) load_tile_w<T, C>(wpd, static_cast<const T*>(a.w_proj), a.wp_ld, tp, lane);
  load_row<T, CH>(wmix, static_cast<const T*>(a.w_mix) + gc0);
  TileW<T, C> wu[kResident ? NUP : 2];
  const RowRegs<T, 16>* wuf[NUP];
  if constexpr (kResident) {
#pragma unroll
    for (int j = 0; j < NUP; ++j) {
      load_tile_w<T, C>(wu[j].r, w_up, a.wu_ld, NUP * wv + j, lane);
      wuf[j] = wu[j].r;
    }
    if constexpr (kShared) {
      if (!kLateDown && has_d) load_tile_w<T, 2 * C>(wpd, w_down, a.wd_ld, td, lane);
    } else {
      load_tile_w<T, 2 * C>(wd, w_down, a.wd_ld, td, lane);
    }
  }
  // keep the scheduler from sinking the loads toward their uses
  __builtin_amdgcn_sched_barrier(0);

  while (true) {
    // fragments fetched inside the loop are fetched there: hoisted out of it
    // as invariant, they spill
    if constexpr (!kResident) asm volatile("" : "+s"(w_up), "+s"(w_down));
    // 1) gate (gate_kernel's arithmetic)
    if (rows_here) store_row<T, CH>(ga + gr * LDC + gc0, gate_row<T, CH>(y, gl));
    __syncthreads();
    // 2) c_proj, then the partial sum
    if constexpr (!kResident) load_tile_w<T, C>(wu[0].r, w_up, a.wu_ld, NUP * wv, lane);
    if (has_p) {
#pragma unroll
      for (int k = 0; k < RT; ++k) {
        f32x4_t acc[1];
        const RowRegs<T, 16>* const f[1] = {wpd};
        layer_tiles<T, C, 1>(acc, f, ga + k * kLayerRows * LDC, lane);
        // added in both cases: with a branch here, the compiler (ROCm 7.2)
        // stored the products' registers on the branch's far side without the
        // wait states that a matrix instruction's result needs
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = elem<T, 4>(pin[k], i) + rt<T>(acc[0][i]);
        store_vec<T, 4>(pm + (k * kLayerRows + c) * LDC + 16 * tp + 4 * g, p);
      }
    }
    __syncthreads();
    // 3) the MLP's mixture over the committed blocks and the new partial; its
    //    norm overwrites the gated rows (no longer read)
    if (rows_here) {
      RowRegs<T, CH> last;
      load_row<T, CH>(last, pm + gr * LDC + gc0);
      float h[CH];
      const int64_t row = min((int64_t)group * ROWS + gr, a.M - 1);
      layer_mixture<T, CH, NS, true>(held, a.nblk, a.blk, a.blk_ld, row, gc0, last, wmix, C, h);
      store_vec<T, CH>(ga + gr * LDC + gc0, h);
    }
    __syncthreads();
    if constexpr (kLateDown) {
      if (has_d) load_tile_w<T, 2 * C>(wpd, w_down, a.wd_ld, td, lane);
    }
    const int next = RT == 1 ? ngroups : group + (int)gridDim.x;  // RT = 1: a workgroup per group
    if (next < ngroups) load_rows(next);
    // 4) FFN up + SwiGLU (swiglu_kernel's arithmetic on the interleaved
    //    (gate, linear) pairs: features 2j, 2j + 1 -> hidden j)
    auto hidden = [&](const f32x4_t& acc, int k, int t) __attribute__((always_inline)) {
      float hv[2];
#pragma unroll
      for (int q = 0; q < 2; ++q)
        hv[q] = swiglu_value<T>(rt<T>(acc[2 * q]), rt<T>(acc[2 * q + 1]), a.alpha, a.limit);
      store_vec<T, 2>(hh + (k * kLayerRows + c) * LDH + 8 * t + 2 * g, hv);
    };
    if constexpr (kResident) {
#pragma unroll
      for (int k = 0; k < RT; ++k) {
        f32x4_t acc[NUP];
        layer_tiles<T, C, NUP>(acc, wuf, ga + k * kLayerRows * LDC, lane);
#pragma unroll
        for (int j = 0; j < NUP; ++j) hidden(acc[j], k, NUP * wv + j);
      }
    } else {
      // each tile's fragments fetched while the one before runs, the FFN-down
      // fragments behind the last
#pragma unroll
      for (int j = 0; j < NUP; ++j) {
        if (j + 1 < NUP) load_tile_w<T, C>(wu[(j + 1) & 1].r, w_up, a.wu_ld, NUP * wv + j + 1, lane);
        else load_tile_w<T, 2 * C>(wd, w_down, a.wd_ld, td, lane);
        const RowRegs<T, 16>* const f[1] = {wu[j & 1].r};
#pragma unroll
        for (int k = 0; k < RT; ++k) {
          f32x4_t acc[1];
          layer_tiles<T, C, 1>(acc, f, ga + k * kLayerRows * LDC, lane);
          hidden(acc[0], k, NUP * wv + j);
        }
      }
    }
    // the tail's operands, into the registers that the products above leave: its
    // tiles are dealt to the waves in runs of tail_n from tail_0 on
    constexpr int TB = NUP;  // tiles held at a time
    const T* t_w = static_cast<const T*>(a.t_w);
    const int tail_n = TAIL == kTailNone ? 0 : (a.t_n / 16 + kLayerWaves - 1) / kLayerWaves;
    const int tail_0 = tail_n * wv;
    const int tail_end = min(tail_0 + tail_n, a.t_n / 16);
    if constexpr (TAIL != kTailNone) {
#pragma unroll
      for (int b = 0; b < TB; ++b)
        if (tail_0 + b < tail_end) load_tile_w<T, C>(wu[b].r, t_w, a.t_wld, tail_0 + b, lane);
      if constexpr (TAIL == kTailIn) {
        if (rows_here) {
          const int64_t row = min((int64_t)group * ROWS + gr, a.M - 1);
          load_held<T, CH, HELD>(held, a.blk, a.blk_ld, a.nblk, a.dup != 0, row, gc0);
          load_row<T, CH>(wmix, static_cast<const T*>(a.t_mix) + gc0);
        }
      }
    }
    __syncthreads();
    // 5) FFN down + residual
    if (has_d) {
#pragma unroll
      for (int k = 0; k < RT; ++k) {
        f32x4_t acc[1];
        const RowRegs<T, 16>* const f[1] = {kShared ? wpd : wd};
        layer_tiles<T, 2 * C, 1>(acc, f, hh + k * kLayerRows * LDH, lane);
        const int64_t row = (int64_t)group * ROWS + k * kLayerRows + c;
        const int col = 16 * td + 4 * g;
        T* pr = pm + (k * kLayerRows + c) * LDC + col;
        float pmv[4], o[4];
        load_vec<T, 4>(pr, pmv);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = pmv[i] + rt<T>(acc[0][i]);
        if (row < a.M) store_vec<T, 4>(static_cast<T*>(a.out) + row * a.out_ld + col, o);
        // the same lane alone reads and writes this slice of pm
        if (TAIL != kTailNone || a.xn != nullptr) store_vec<T, 4>(pr, o);  // uniform
      }
    }
    // 6) the row work after the layer: dg_block_out_norm's and the head's
    //    RMSNorm of the stored output rows, or the next layer's mixture and norm
    if (TAIL != kTailNone || a.xn != nullptr) {  // uniform
      __syncthreads();
      if (rows_here) {
        float x[CH];
        const int64_t row = (int64_t)group * ROWS + gr;
        if constexpr (TAIL == kTailIn) {
          RowRegs<T, CH> last;
          load_row<T, CH>(last, pm + gr * LDC + gc0);
          layer_mixture<T, CH, NS, true>(held, a.nblk, a.blk, a.blk_ld, min(row, a.M - 1), gc0, last, wmix, C, x);
        } else {
          load_vec<T, CH>(pm + gr * LDC + gc0, x);
          row_rms<CH, kRowLanes>(x, C);
          if (a.xn != nullptr && row < a.M)
            store_vec<T, CH>(static_cast<T*>(a.xn) + row * a.xn_ld + gc0, x);
        }
        // the FFN-up products read ga last, before the barrier of stage 5
        if constexpr (TAIL != kTailNone) store_vec<T, CH>(ga + gr * LDC + gc0, x);
      }
    }
    // 7) the tail's products
    if constexpr (TAIL != kTailNone) {
      __syncthreads();
      // the step's readers of the position are launches before this one
      if (TAIL == kTailHead && a.t_advance != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *a.t_advance += 1;
      const int64_t row = (int64_t)group * ROWS + c;
      T* t_out = static_cast<T*>(a.t_out) + min(row, a.M - 1) * a.t_old + 4 * g;
      float best = kNegInf;
      int best_i = 0x7fffffff;
#pragma unroll 1
      for (int t0 = tail_0; t0 < tail_end; t0 += TB) {
#pragma unroll
        for (int b = 0; b < TB; ++b) {
          const int t = t0 + b;
          if (t >= tail_end) continue;  // wave-uniform
          f32x4_t acc[1];
          const RowRegs<T, 16>* const f[1] = {wu[b].r};
          layer_tiles<T, C, 1>(acc, f, ga, lane);
          mfma_settle(acc);
          if (t + TB < tail_end) load_tile_w<T, C>(wu[b].r, t_w, a.t_wld, t + TB, lane);
          float v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = acc[0][i];
          if constexpr (TAIL == kTailHead) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              v[i] = softcap_value<T>(v[i], a.t_cap);
              if (v[i] > best) {  // entries rise with t and i: the first maximum stays
                best = v[i];
                best_i = 16 * t + 4 * g + i;
              }
            }
          }
          if (row < a.M) store_vec<T, 4>(t_out + 16 * t, v);
        }
      }
      if (TAIL == kTailHead && a.t_ids != nullptr) {  // uniform
        // hh's last readers passed the barrier of stage 6
        float* red_v = reinterpret_cast<float*>(hh);
        int* red_i = reinterpret_cast<int*>(red_v + kLayerWaves * kLayerRows);
        first_max(best, best_i);
        if (g == 0) {
          red_v[wv * kLayerRows + c] = best;
          red_i[wv * kLayerRows + c] = best_i;
        }
        __syncthreads();
        if (threadIdx.x < kLayerRows && row < a.M) {
          for (int q = 1; q < kLayerWaves; ++q) {  // waves in entry order
            if (red_v[q * kLayerRows + c] > best) {
              best = red_v[q * kLayerRows + c];
              best_i = red_i[q * kLayerRows + c];
            }
          }
          a.t_ids[row] = (int64_t)(best_i == 0x7fffffff ? 0 : best_i);
        }
      }
    }
    // the next group's stages write ga, pm and hh again: every wave has passed
    // the barrier behind their last reads, but for pm, read here and written
    // past the barrier of the next stage 1
    group = next;
    if (group >= ngroups) break;
  }
}

namespace {

bool rows16(const void* p, int64_t ld, int64_t es) {
  return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && (ld * es) % 16 == 0;
}
bool layer_dtype_ok(int dtype) { return dtype == DG_F32 || dtype == DG_BF16 || dtype == DG_F16; }

// The workgroups that are resident at once: 2 per CU at n_embd 64, 1 at 128
// (512 threads of up to 128 or 256 registers).
int64_t layer_resident(int C) { return C == 64 ? 512 : 256; }

// Groups of 32 rows (RT = 2) once 16-row groups no longer all fit at once.
bool layer_deep(int64_t M, int C) { return M > layer_resident(C) * kLayerRows; }

// Workgroups of a launch over M rows: one per group of 16; with RT = 2 one per
// group of 32 while they all fit, beyond that as many as share them evenly.
unsigned layer_grid(int64_t M, bool deep, int C) {
  const int64_t rows = deep ? 2 * kLayerRows : kLayerRows;
  const int64_t groups = (M + rows - 1) / rows;
  if (!deep) return (unsigned)groups;
  const int64_t rounds = (groups + layer_resident(C) - 1) / layer_resident(C);
  return (unsigned)((groups + rounds - 1) / rounds);
}

template <typename T, int C, int NS>
void launch_block_in_ns(const BlockInArgs& a, hipStream_t s) {
  constexpr int SPLIT = 4 * C / 16 / kLayerWaves;  // one tile per wave
  const bool deep = layer_deep(a.M, C);
  const unsigned grid = layer_grid(a.M, deep, C);
  // n_embd 64: two workgroups per group up to 256 groups (100 rows in fp32: 4.2
  // us, 5.2 with one; 6400 rows, 400 groups: 9.1, 8.8 with one).  n_embd 128:
  // four (1850 rows in fp32: 8.9 us, 12.8 with one; bf16 6.1 and 7.1)
  if (deep) hipLaunchKernelGGL((block_in_kernel<T, C, NS, 2, 1, false>), dim3(grid), dim3(kLayerThreads), 0, s, a);
  else if (C == 64 && grid > 256)
    hipLaunchKernelGGL((block_in_kernel<T, C, NS, 1, 1, false>), dim3(grid), dim3(kLayerThreads), 0, s, a);
  else
    hipLaunchKernelGGL((block_in_kernel<T, C, NS, 1, SPLIT, false>), dim3(grid, SPLIT), dim3(kLayerThreads), 0, s,
                       a);
}

// The embedding's form: a workgroup per 16 rows at any size.
template <typename T, int C>
void launch_embed_in(const BlockInArgs& a, hipStream_t s) {
  constexpr int SPLIT = 4 * C / 16 / kLayerWaves;
  const unsigned grid = layer_grid(a.M, false, C);
  if (C == 64 && grid > 256)
    hipLaunchKernelGGL((block_in_kernel<T, C, 4, 1, 1, true>), dim3(grid), dim3(kLayerThreads), 0, s, a);
  else
    hipLaunchKernelGGL((block_in_kernel<T, C, 4, 1, SPLIT, true>), dim3(grid, SPLIT), dim3(kLayerThreads), 0, s, a);
}

template <typename T, int C>
void launch_block_in(const BlockInArgs& a, hipStream_t s) {
  if (a.nsrc <= 4) launch_block_in_ns<T, C, 4>(a, s);
  else if (a.nsrc <= 8) launch_block_in_ns<T, C, 8>(a, s);
  else launch_block_in_ns<T, C, kMaxResSources>(a, s);
}

// At n_embd 64 two kinds of instances keep a workgroup per 16 rows at any size,
// their 32-row forms needing more than the 128 registers of two workgroups per
// CU: fp32 (35328 rows: 54 us with the spills, 52 with one workgroup per CU, 44
// so), and 16-bit types for 5 to 8 blocks.  us after the attention, 16-row ->
// 32-row groups:
//                 blocks   8200 rows       16384          35328
//   n_embd  64 bf16    3    9.6 ->  9.7   12.4 -> 11.3   22.0 -> 25.3
//                      5   11.3 -> 13.1   15.3 -> 15.6   29.0 -> 33.8
//                      8   11.9 -> 13.6   15.8 -> 16.4   30.4 -> 36.1
//                      9   13.7 -> 15.8   18.1 -> 19.5   36.7 -> 41.8
//                     16   20.4 -> 21.1   28.8 -> 25.9   60.3 -> 61.1
//                     31   37.8 -> 33.6   51.2 -> 40.4    114 ->  104
//   n_embd 128 bf16    5   22.9 -> 19.6   43.3 -> 30.0   96.1 -> 56.6
//                     31   61.4 -> 44.2    107 -> 74.7    275 ->  196
//   n_embd 128 fp32    5   40.0 -> 36.5   78.6 -> 66.5    170 ->  149
template <typename T, int C, int NS>
void launch_block_out_ns(const BlockOutArgs& a, hipStream_t s) {
  constexpr bool kDeep = !(C == 64 && (sizeof(T) == 4 || NS == 8));
  const bool deep = kDeep && layer_deep(a.M, C);
  const unsigned grid = layer_grid(a.M, deep, C);
  if constexpr (kDeep) {
    if (deep) {
      hipLaunchKernelGGL((block_out_kernel<T, C, NS, 2, kTailNone>), dim3(grid), dim3(kLayerThreads), 0, s, a);
      return;
    }
  }
  hipLaunchKernelGGL((block_out_kernel<T, C, NS, 1, kTailNone>), dim3(grid), dim3(kLayerThreads), 0, s, a);
}

// With a tail: a workgroup per 16 rows at any size.
template <typename T, int C, int NS>
void launch_block_tail_ns(const BlockOutArgs& a, hipStream_t s) {
  const dim3 grid(layer_grid(a.M, false, C)), block(kLayerThreads);
  if (a.t_mix != nullptr) hipLaunchKernelGGL((block_out_kernel<T, C, NS, 1, kTailIn>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((block_out_kernel<T, C, NS, 1, kTailHead>), grid, block, 0, s, a);
}

// fp32 at n_embd 128 has none: 256 KB of weights a workgroup, fetched as they
// are used, take longer than the launch they save (3 layers, 100 rows: 100 us
// one by one, 106 joined).
template <typename T, int C>
int launch_block_tail(const BlockOutArgs& a, hipStream_t s) {
  if constexpr (C == 128 && sizeof(T) == 4) {
    set_error("block_out: n_embd 128 in fp32 is unsupported with what follows the layer");
    return DG_EUNSUPPORTED;
  } else {
    if (a.nblk <= 4) launch_block_tail_ns<T, C, 4>(a, s);
    else if (a.nblk <= 8) launch_block_tail_ns<T, C, 8>(a, s);
    else launch_block_tail_ns<T, C, kMaxResSources>(a, s);
    return check_launch("block_out_kernel");
  }
}

template <typename T, int C>
void launch_block_out(const BlockOutArgs& a, hipStream_t s) {
  if (a.nblk <= 4) launch_block_out_ns<T, C, 4>(a, s);
  else if (a.nblk <= 8) launch_block_out_ns<T, C, 8>(a, s);
  else launch_block_out_ns<T, C, kMaxResSources>(a, s);
}

#define DG_LAYER(launch)                                                   \
  do {                                                                     \
    if (dtype == DG_F32) C == 64 ? launch<float, 64>(a, s) : launch<float, 128>(a, s);         \
    else if (dtype == DG_BF16) C == 64 ? launch<bf16_t, 64>(a, s) : launch<bf16_t, 128>(a, s); \
    else C == 64 ? launch<f16_t, 64>(a, s) : launch<f16_t, 128>(a, s);                         \
  } while (0)

}  // namespace
}  // namespace dg

using namespace dg;

extern "C" int dg_block_in(int64_t M, int C, int dtype, int nsrc, const void* const* src, const int64_t* src_ld,
                           const void* w_mix, const void* w_qkvg, int64_t w_ld, void* out, int64_t out_ld,
                           void* stream) {
  DG_REQUIRE(M >= 0 && C >= 1, DG_EINVAL, "block_in: bad sizes M=%lld C=%d", (long long)M, C);
  DG_REQUIRE(layer_dtype_ok(dtype), DG_EUNSUPPORTED, "block_in: dtype %d unsupported", dtype);
  DG_REQUIRE(C == 64 || C == 128, DG_EUNSUPPORTED, "block_in: n_embd %d unsupported (64 or 128)", C);
  DG_REQUIRE(nsrc >= 1 && nsrc <= kMaxResSources && (w_mix != nullptr || nsrc == 1), DG_EINVAL,
             "block_in: %d sources (1..%d; 1 without a pseudo-query)", nsrc, kMaxResSources);
  if (M == 0) return DG_OK;
  DG_REQUIRE(src && src_ld && w_qkvg && out, DG_EINVAL, "block_in: NULL pointer");
  DG_REQUIRE(M <= (int64_t)kLayerRows * 0x7fffffffLL, DG_EINVAL, "block_in: too many rows (%lld)", (long long)M);
  DG_REQUIRE(w_ld >= C && out_ld >= 4 * (int64_t)C, DG_EINVAL, "block_in: a row stride is narrower than its row");
  const int64_t es = dtype_bytes(dtype);
  BlockInArgs a{};
  bool ok = rows16(w_mix, 0, es) && rows16(w_qkvg, w_ld, es) && rows16(out, out_ld, es);
  for (int n = 0; n < nsrc; ++n) {
    DG_REQUIRE(src[n] != nullptr && src_ld[n] >= C, DG_EINVAL, "block_in: source %d is NULL or narrower than C", n);
    ok = ok && rows16(src[n], src_ld[n], es);
    a.src[n] = src[n];
    a.ld[n] = src_ld[n];
  }
  DG_REQUIRE(ok, DG_EUNSUPPORTED, "block_in: rows must be 16-byte aligned");
  a.w_mix = w_mix; a.w = w_qkvg; a.out = out;
  a.w_ld = w_ld; a.out_ld = out_ld; a.M = M;
  a.nsrc = nsrc;
  a.dup = nsrc > 1 && src[1] == src[0] && src_ld[1] == src_ld[0] ? 1 : 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  DG_LAYER(launch_block_in);
  return check_launch("block_in_kernel");
}

extern "C" int dg_embed_in(int64_t M, int C, int dtype, const int64_t* ids, int64_t V, const void* table,
                           int64_t table_ld, void* x, int64_t x_ld, const void* w_qkvg, int64_t w_ld, void* out,
                           int64_t out_ld, void* stream) {
  DG_REQUIRE(M >= 0 && C >= 1 && V >= 1, DG_EINVAL, "embed_in: bad sizes M=%lld C=%d V=%lld", (long long)M, C,
             (long long)V);
  DG_REQUIRE(layer_dtype_ok(dtype), DG_EUNSUPPORTED, "embed_in: dtype %d unsupported", dtype);
  DG_REQUIRE(C == 64 || C == 128, DG_EUNSUPPORTED, "embed_in: n_embd %d unsupported (64 or 128)", C);
  if (M == 0) return DG_OK;
  DG_REQUIRE(ids && table && x && w_qkvg && out, DG_EINVAL, "embed_in: NULL pointer");
  DG_REQUIRE(M <= (int64_t)kLayerRows * 0x7fffffffLL, DG_EINVAL, "embed_in: too many rows (%lld)", (long long)M);
  DG_REQUIRE(table_ld >= C && x_ld >= C && w_ld >= C && out_ld >= 4 * (int64_t)C, DG_EINVAL,
             "embed_in: a row stride is narrower than its row");
  const int64_t es = dtype_bytes(dtype);
  DG_REQUIRE(rows16(table, table_ld, es) && rows16(x, x_ld, es) && rows16(w_qkvg, w_ld, es) && rows16(out, out_ld, es),
             DG_EUNSUPPORTED, "embed_in: rows must be 16-byte aligned");
  BlockInArgs a{};
  a.src[0] = table; a.ld[0] = table_ld; a.nsrc = 1;
  a.ids = ids; a.V = V; a.x = x; a.x_ld = x_ld;
  a.w = w_qkvg; a.out = out;
  a.w_ld = w_ld; a.out_ld = out_ld; a.M = M;
  hipStream_t s = static_cast<hipStream_t>(stream);
  DG_LAYER(launch_embed_in);
  return check_launch("block_in_kernel");
}

struct LayerTailArgs {
  const void* mix;  // the next layer's pseudo-query; null: the head
  const void* w;
  void* out;
  int64_t* ids;
  int64_t w_ld, out_ld;
  int n;
  float cap;
  int* advance;
};

static int block_out_impl(int64_t M, int C, int dtype, const void* y, int64_t y_ld, const void* g, int64_t g_ld,
                          const void* w_proj, int64_t wp_ld, const void* partial_in, int64_t pin_ld, int nblk,
                          const void* const* blocks, const int64_t* blocks_ld, const void* w_mix, const void* w_up,
                          int64_t wu_ld, const void* w_down, int64_t wd_ld, float alpha, float limit, void* out,
                          int64_t out_ld, void* xn, int64_t xn_ld, const LayerTailArgs* tail, void* stream) {
  DG_REQUIRE(M >= 0 && C >= 1, DG_EINVAL, "block_out: bad sizes M=%lld C=%d", (long long)M, C);
  DG_REQUIRE(layer_dtype_ok(dtype), DG_EUNSUPPORTED, "block_out: dtype %d unsupported", dtype);
  DG_REQUIRE(C == 64 || C == 128, DG_EUNSUPPORTED, "block_out: n_embd %d unsupported (64 or 128)", C);
  DG_REQUIRE(nblk >= 0 && nblk + 1 <= kMaxResSources, DG_EINVAL, "block_out: %d blocks (0..%d)", nblk,
             kMaxResSources - 1);
  if (M == 0) return DG_OK;
  DG_REQUIRE(y && g && w_proj && w_mix && w_up && w_down && out && (nblk == 0 || (blocks && blocks_ld)), DG_EINVAL,
             "block_out: NULL pointer");
  DG_REQUIRE(M <= (int64_t)kLayerRows * 0x7fffffffLL, DG_EINVAL, "block_out: too many rows (%lld)", (long long)M);
  const int64_t es = dtype_bytes(dtype);
  BlockOutArgs a{};
  bool ok = rows16(y, y_ld, es) && rows16(g, g_ld, es) && rows16(w_proj, wp_ld, es) && rows16(w_mix, 0, es) &&
            rows16(w_up, wu_ld, es) && rows16(w_down, wd_ld, es) && rows16(out, out_ld, es) &&
            (partial_in == nullptr || rows16(partial_in, pin_ld, es)) && (xn == nullptr || rows16(xn, xn_ld, es));
  DG_REQUIRE(y_ld >= C && g_ld >= C && wp_ld >= C && wu_ld >= C && wd_ld >= 2 * C && out_ld >= C &&
                 (partial_in == nullptr || pin_ld >= C) && (xn == nullptr || xn_ld >= C),
             DG_EINVAL, "block_out: a row stride is narrower than its row");
  for (int n = 0; n < nblk; ++n) {
    DG_REQUIRE(blocks[n] != nullptr && blocks_ld[n] >= C, DG_EINVAL, "block_out: block %d is NULL or narrower than C",
               n);
    ok = ok && rows16(blocks[n], blocks_ld[n], es);
    a.blk[n] = blocks[n];
    a.blk_ld[n] = blocks_ld[n];
  }
  DG_REQUIRE(ok, DG_EUNSUPPORTED, "block_out: rows must be 16-byte aligned");
  if (tail != nullptr) {
    DG_REQUIRE(tail->w && tail->out, DG_EINVAL, "block_out: NULL pointer");
    DG_REQUIRE(tail->w_ld >= C && tail->out_ld >= tail->n && tail->cap >= 0.f, DG_EINVAL,
               "block_out: bad strides or cap of what follows the layer");
    const int n = tail->n;
    DG_REQUIRE(n == 64 || n == 128 || n == 256 || n == 512 || n == 1024, DG_EUNSUPPORTED,
               "block_out: vocabulary %d unsupported (64, 128, 256, 512 or 1024)", n);
    DG_REQUIRE(rows16(tail->mix, 0, es) && rows16(tail->w, tail->w_ld, es) && rows16(tail->out, tail->out_ld, es),
               DG_EUNSUPPORTED, "block_out: rows must be 16-byte aligned");
    a.t_mix = tail->mix; a.t_w = tail->w; a.t_out = tail->out; a.t_ids = tail->ids;
    a.t_wld = tail->w_ld; a.t_old = tail->out_ld; a.t_n = tail->n; a.t_cap = tail->cap;
    a.t_advance = tail->advance;
  }
  a.y = y; a.g = g; a.w_proj = w_proj; a.pin = partial_in; a.w_mix = w_mix; a.w_up = w_up; a.w_down = w_down;
  a.out = out; a.xn = xn;
  a.y_ld = y_ld; a.g_ld = g_ld; a.wp_ld = wp_ld; a.pin_ld = pin_ld; a.wu_ld = wu_ld; a.wd_ld = wd_ld;
  a.out_ld = out_ld; a.xn_ld = xn_ld; a.M = M; a.nblk = nblk; a.alpha = alpha; a.limit = limit;
  a.dup = nblk > 1 && blocks[1] == blocks[0] && blocks_ld[1] == blocks_ld[0] ? 1 : 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (tail != nullptr) {
    if (dtype == DG_F32) return C == 64 ? launch_block_tail<float, 64>(a, s) : launch_block_tail<float, 128>(a, s);
    if (dtype == DG_BF16) return C == 64 ? launch_block_tail<bf16_t, 64>(a, s) : launch_block_tail<bf16_t, 128>(a, s);
    return C == 64 ? launch_block_tail<f16_t, 64>(a, s) : launch_block_tail<f16_t, 128>(a, s);
  }
  DG_LAYER(launch_block_out);
  return check_launch("block_out_kernel");
}

extern "C" int dg_block_out(int64_t M, int C, int dtype, const void* y, int64_t y_ld, const void* g, int64_t g_ld,
                            const void* w_proj, int64_t wp_ld, const void* partial_in, int64_t pin_ld, int nblk,
                            const void* const* blocks, const int64_t* blocks_ld, const void* w_mix,
                            const void* w_up, int64_t wu_ld, const void* w_down, int64_t wd_ld, float alpha,
                            float limit, void* out, int64_t out_ld, void* stream) {
  return block_out_impl(M, C, dtype, y, y_ld, g, g_ld, w_proj, wp_ld, partial_in, pin_ld, nblk, blocks, blocks_ld,
                        w_mix, w_up, wu_ld, w_down, wd_ld, alpha, limit, out, out_ld, nullptr, 0, nullptr, stream);
}

extern "C" int dg_block_out_norm(int64_t M, int C, int dtype, const void* y, int64_t y_ld, const void* g,
                                 int64_t g_ld, const void* w_proj, int64_t wp_ld, const void* partial_in,
                                 int64_t pin_ld, int nblk, const void* const* blocks, const int64_t* blocks_ld,
                                 const void* w_mix, const void* w_up, int64_t wu_ld, const void* w_down,
                                 int64_t wd_ld, float alpha, float limit, void* out, int64_t out_ld, void* xn,
                                 int64_t xn_ld, void* stream) {
  DG_REQUIRE(M == 0 || xn != nullptr, DG_EINVAL, "block_out_norm: NULL pointer");
  return block_out_impl(M, C, dtype, y, y_ld, g, g_ld, w_proj, wp_ld, partial_in, pin_ld, nblk, blocks, blocks_ld,
                        w_mix, w_up, wu_ld, w_down, wd_ld, alpha, limit, out, out_ld, xn, xn_ld, nullptr, stream);
}

extern "C" int dg_block_out_in(int64_t M, int C, int dtype, const void* y, int64_t y_ld, const void* g, int64_t g_ld,
                               const void* w_proj, int64_t wp_ld, const void* partial_in, int64_t pin_ld, int nblk,
                               const void* const* blocks, const int64_t* blocks_ld, const void* w_mix,
                               const void* w_up, int64_t wu_ld, const void* w_down, int64_t wd_ld, float alpha,
                               float limit, void* out, int64_t out_ld, const void* next_mix, const void* next_qkvg,
                               int64_t nq_ld, void* qkvg, int64_t qkvg_ld, void* stream) {
  DG_REQUIRE(M == 0 || next_mix != nullptr, DG_EINVAL, "block_out_in: NULL pointer");
  const LayerTailArgs tail{next_mix, next_qkvg, qkvg, nullptr, nq_ld, qkvg_ld, 4 * C, 0.f, nullptr};
  return block_out_impl(M, C, dtype, y, y_ld, g, g_ld, w_proj, wp_ld, partial_in, pin_ld, nblk, blocks, blocks_ld,
                        w_mix, w_up, wu_ld, w_down, wd_ld, alpha, limit, out, out_ld, nullptr, 0, &tail, stream);
}

extern "C" int dg_block_out_head(int64_t M, int C, int dtype, const void* y, int64_t y_ld, const void* g,
                                 int64_t g_ld, const void* w_proj, int64_t wp_ld, const void* partial_in,
                                 int64_t pin_ld, int nblk, const void* const* blocks, const int64_t* blocks_ld,
                                 const void* w_mix, const void* w_up, int64_t wu_ld, const void* w_down,
                                 int64_t wd_ld, float alpha, float limit, void* out, int64_t out_ld, void* xn,
                                 int64_t xn_ld, int V, const void* table, int64_t table_ld, float cap, void* logits,
                                 int64_t logits_ld, int64_t* ids, int32_t* advance, void* stream) {
  const LayerTailArgs tail{nullptr, table, logits, ids, table_ld, logits_ld, V, cap, advance};
  return block_out_impl(M, C, dtype, y, y_ld, g, g_ld, w_proj, wp_ld, partial_in, pin_ld, nblk, blocks, blocks_ld,
                        w_mix, w_up, wu_ld, w_down, wd_ld, alpha, limit, out, out_ld, xn, xn_ld, &tail, stream);
}
