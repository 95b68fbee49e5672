// The Dense chain over a block of rows, shared by the fused step kernels.
//
// A workgroup of four or eight waves (NW) owns a block of 16 * NT columns of MFMA tiles
// (one column per trajectory; a flow's block holds its rows twice, primal and
// tangent) and runs every layer with the activations in LDS.  Weights are the
// A operand (16 output features per tile), read straight from L2 into
// registers: they are packed in fragment order, one 16-byte vector per lane,
// so a wave reads 1 KB contiguous per fragment and each fragment is read by
// one wave of the workgroup only.  The activations are the B operand,
// [row][feature] in LDS, a 16-byte vector per lane as well.  An accumulator
// lane holds four consecutive features of one row, which is again one vector
// of the next layer's operand: no transposition between layers.
#pragma once
#include "chain.h"
#include "device_util.h"

namespace nodehip {

// Tsit5 tableau as compile-time constants of the step kernels (the same values
// as the GEMM epilogues' tables)
static __device__ const float chA[7][7] = {
    {0, 0, 0, 0, 0, 0, 0},
    {0.161, 0, 0, 0, 0, 0, 0},
    {-0.008480655492356989, 0.335480655492357, 0, 0, 0, 0, 0},
    {2.897153057105493, -6.359448489975075, 4.3622954328695815, 0, 0, 0, 0},
    {5.325864828439257, -11.748883564062828, 7.4955393428898365, -0.09249506636175525, 0, 0, 0},
    {5.86145544294642, -12.92096931784711, 8.159367898576159, -0.071584973281401,
     -0.028269050394068383, 0, 0},
    {0.09646076681806523, 0.01, 0.4798896504144996, 1.379008574103742, -3.290069515436081,
     2.324710524099774, 0}};
static __device__ const float chBT[7] = {-0.00178001105222577714, -0.0008164344596567469,
                                         0.007880878010261995,    -0.1447110071732629,
                                         0.5823571654525552,      -0.45808210592918697,
                                         0.015151515151515152};

// Feature order of FP32 blocks.  An FP32 MFMA adds its K products one after the
// other, so the order in which a dot product meets them is part of its
// rounding; the adaptive solves' first error estimates sit on that rounding
// (two terms of 1e-7 that cancel), and another order means other step sizes.
// Features are therefore stored (LDS, operand rows, fragments) in an order
// within each 16 that makes the four 16x16x4 steps take them as the GEMM path's
// eight 32x32x2 steps do: 0 4 1 5 2 6 3 7, 8 12 9 13 10 14 11 15.
__host__ __device__ __forceinline__ int chain_feat(int p) {  // position -> feature
  return (p & ~15) + ((p & 2) << 2) + ((p >> 3) & 1) + ((p & 1) << 1) + (((p >> 2) & 1) << 2);
}
__host__ __device__ __forceinline__ int chain_posn(int f) {  // feature -> position
  return (f & ~15) + ((f & 1) << 3) + (((f >> 2) & 1) << 2) + (((f >> 3) & 1) << 1) + ((f >> 1) & 1);
}
template <class PP> __device__ __forceinline__ int chain_pos(int f) {
  return sizeof(typename PP::T) == 4 ? chain_posn(f) : f;
}

// FP32 in blocks of few rows: tiles of 64 features x 4 rows (v_mfma_4x4x1, one
// K step of 16 four by four blocks) instead of 16 x 16.  The rate is the same,
// so a block of 8 rows spends half the matrix time of one of 16, and a batch
// that fills only some of the CUs with blocks of 16 spreads over twice as many.
struct PF32S : PF32 {};

// features per K tile, values per lane and K tile; rows (columns of the MFMA)
// and features of a tile.  An accumulator lane holds the features
// 4 (l / CW) .. + 3 of row l % CW in both shapes.
template <class PP> struct ChainK { static constexpr int KT = 32, V = 8, CW = 16, TF = 16; };
template <> struct ChainK<PF32> { static constexpr int KT = 16, V = 4, CW = 16, TF = 16; };
template <> struct ChainK<PF32S> { static constexpr int KT = 16, V = 4, CW = 4, TF = 64; };

// One MFMA K tile of a 16 x 16 block.  FP32: four 16x16x4 steps, lane l
// supplying k = 4 (l / 16) + j to step j for both operands.  Split BF16:
// hi*hi + lo*hi + hi*lo, as the GEMM path orders them.
template <class PP> struct ChainFrag {
  u32x4 p[PP::SPLIT ? 2 : 1];
};
template <class PP>
__device__ __forceinline__ void chain_mfma(f32x4v& c, const ChainFrag<PP>& a, const ChainFrag<PP>& b) {
  if constexpr (sizeof(typename PP::T) == 4) {
    const f32x4v fa = __builtin_bit_cast(f32x4v, a.p[0]), fb = __builtin_bit_cast(f32x4v, b.p[0]);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa.x, fb.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa.y, fb.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa.z, fb.z, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa.w, fb.w, c, 0, 0, 0);
  } else {
    auto m = [&](const u32x4& x, const u32x4& y) {
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x),
                                                  __builtin_bit_cast(bf16x8, y), c, 0, 0, 0);
    };
    m(a.p[0], b.p[0]);
    if constexpr (PP::SPLIT) {
      m(a.p[1], b.p[0]);
      m(a.p[0], b.p[1]);
    }
  }
}

// The workgroup's LDS.  Buffers are handed on as element offsets into it, not
// as pointers: through a pointer picked at run time the compiler loses the
// address space and emits FLAT accesses, which wait for every load in flight.
__device__ __forceinline__ unsigned char* chain_lds() {
  extern __shared__ __attribute__((aligned(16))) unsigned char ch_lds[];
  return ch_lds;
}
// Barrier that orders LDS only (__syncthreads also waits for every global
// access in flight).  Nothing that waves hand to each other here goes through
// global memory: entries stored there are read by the lane that wrote them, or
// by another launch.
__device__ __forceinline__ void chain_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
// What every stage reads, in LDS: tableau rows, stage times and (adjoint) the
// interpolation data of the stage times, and the hidden layers' biases.  As
// scalar loads these cost a stage several dependent trips to memory.
struct alignas(16) ChainShared {
  float A[7][8];               // tableau rows; column 7: the stage time
  float w[8][8];               // interpolation weights of a slot; column 7: its step
  int step[8], exact[8];
};
// A buffer of activations in LDS: [plane][row][pitch] elements at `off`
template <class PP> struct ChainBuf {
  int off, pitch, plane;
  __device__ __forceinline__ typename PP::T* at(int row, int f) const {
    return (typename PP::T*)chain_lds() + off + row * pitch + f;
  }
};

// chain_mma (below) on 64 x 4 tiles: a lane holds one feature's 16 K values
// (four vectors) and reads its row's, in the order that the 16 x 16 steps take
// them.
template <int NT, int MT, int PF>
__device__ __forceinline__ void chain_mma4(f32x4v (&acc)[MT][NT], const void* __restrict__ W, int t0,
                                           int tlast, int kt, int k0, int k1, const ChainBuf<PF32S>& in,
                                           int lane) {
  const f32x4v* w[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int t = t0 + m < tlast ? t0 + m : tlast;
    w[m] = (const f32x4v*)W + (int64_t)t * kt * 256 + lane;
  }
  const float* b = in.at(lane & 3, 0);
  f32x4v a[PF][MT][4];
  auto load = [&](f32x4v (&f)[4], int m, int k) {
    k = k < k1 ? k : k1 - 1;
#pragma unroll
    for (int v = 0; v < 4; ++v) f[v] = w[m][(k * 4 + v) * 64];
  };
  auto step = [&](f32x4v (&f)[MT][4], int k, bool refill) {
    f32x4v x[NT][4];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int v = 0; v < 4; ++v) x[n][v] = *(const f32x4v*)(b + n * 4 * in.pitch + k * 16 + 4 * v);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int n = 0; n < NT; ++n)
            acc[m][n] = __builtin_amdgcn_mfma_f32_4x4x1f32(f[m][v][j], x[n][v][j], acc[m][n], 0, 0, 0);
    if (refill)
#pragma unroll
      for (int m = 0; m < MT; ++m) load(f[m], m, k + PF);
  };
#pragma unroll
  for (int j = 0; j < PF; ++j)
#pragma unroll
    for (int m = 0; m < MT; ++m) load(a[j][m], m, k0 + j);
  int k = k0;
  for (; k + PF <= k1; k += PF)
#pragma unroll
    for (int j = 0; j < PF; ++j) step(a[j], k + j, true);
#pragma unroll
  for (int j = 0; j < PF - 1; ++j)
    if (k + j < k1) step(a[j], k + j, false);
}

// acc[m][n] += W tiles (first tile t0, MT of them, K tiles [k0, k1)) x columns.
// The fragments of PF K tiles are in flight (ring in registers, loads
// unconditional: the index is clamped instead).  side.step(): a piece of other
// work per K tile.
template <class PP, int NT, int MT, int PF, class Side>
__device__ __forceinline__ void chain_mma(f32x4v (&acc)[MT][NT], const void* __restrict__ W, int t0,
                                          int tlast, int kt, int k0, int k1, const ChainBuf<PP>& in,
                                          int lane, Side& side) {
  if constexpr (ChainK<PP>::CW == 4) {
    chain_mma4<NT, MT, (MT <= 2 ? 4 / MT : 2)>(acc, W, t0, tlast, kt, k0, k1, in, lane);
    return;
  } else {
  constexpr int P = PP::SPLIT ? 2 : 1;
  const u32x4* w[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int t = t0 + m < tlast ? t0 + m : tlast;
    w[m] = (const u32x4*)W + (int64_t)t * kt * P * 64 + lane;
  }
  const typename PP::T* b = in.at(lane & 15, ChainK<PP>::V * (lane >> 4));
  ChainFrag<PP> a[PF][MT];
  auto load = [&](ChainFrag<PP>& f, int m, int k) {
    k = k < k1 ? k : k1 - 1;
#pragma unroll
    for (int q = 0; q < P; ++q) f.p[q] = w[m][(k * P + q) * 64];
  };
  auto step = [&](ChainFrag<PP> (&f)[MT], int k, bool refill) {
    ChainFrag<PP> x[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int q = 0; q < P; ++q)
        x[n].p[q] = *(const u32x4*)(b + q * in.plane + n * 16 * in.pitch + k * ChainK<PP>::KT);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
      for (int n = 0; n < NT; ++n) chain_mfma<PP>(acc[m][n], f[m], x[n]);
      if (refill) load(f[m], m, k + PF);
    }
  };
#pragma unroll
  for (int j = 0; j < PF; ++j)
#pragma unroll
    for (int m = 0; m < MT; ++m) load(a[j][m], m, k0 + j);
  int k = k0;
  for (; k + PF <= k1; k += PF) {
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      step(a[j], k + j, true);
      side.step();
    }
  }
#pragma unroll
  for (int j = 0; j < PF - 1; ++j)
    if (k + j < k1) step(a[j], k + j, false);
  }
}

// FP32 blocks write their operand rows where they are produced (16 bytes per
// lane; the copy's index arithmetic below cost the small blocks 5-25%).  Split
// ones, at twice the values per row block and 8-byte pieces, copy:
//
// Copy of a block's activations (rows 0 .. rows of `buf`, all planes) from LDS
// to an operand matrix of the weight gradients, 16 bytes per lane along the
// rows.  Done a piece per K tile of the layer that reads the same buffer: as
// stores of the producing epilogue all workgroups' writes met in the same
// short phase (8-byte pieces of 16 rows each) while memory idled under the
// products.
struct ChainNoSide {
  __device__ __forceinline__ void step() {}
  __device__ __forceinline__ void finish() {}
};
template <class PP, int THREADS> struct ChainCopy {
  static constexpr int E = 16 / sizeof(typename PP::T);  // elements per piece
  ChainBuf<PP> buf;
  typename PP::T* dst;         // the block's first row
  int64_t plane;               // elements between the planes
  int w, cpr, n, pos;          // row width, pieces per row, pieces, next piece
  float rcpr;
  u32x4 held;
  typename PP::T* to;
  __device__ __forceinline__ ChainCopy(ChainBuf<PP> b, void* base, int64_t rows, int64_t row0, int w_,
                                       int used, int nrow)
      : buf(b), dst((typename PP::T*)base + row0 * w_), plane(rows * w_), w(w_), cpr(used / E),
        n((PP::SPLIT ? 2 : 1) * nrow * (used / E)), pos(threadIdx.x), rcpr(1.f / (used / E)),
        held{0, 0, 0, 0}, to(nullptr) {
    rows_ = nrow;
  }
  int rows_;
  __device__ __forceinline__ void flush() {
    if (to) *(u32x4*)to = held;
    to = nullptr;
  }
  __device__ __forceinline__ void step() {
    flush();
    if (pos < n) {
      int r = (int)(((float)pos + 0.5f) * rcpr);     // (exact: pos < 2^22)
      const int c = (pos - r * cpr) * E;
      int p = 0;
      if (PP::SPLIT && r >= rows_) { p = 1; r -= rows_; }
      held = *(const u32x4*)(buf.at(r, c) + p * buf.plane);
      to = dst + p * plane + r * w + c;
      pos += THREADS;
    }
  }
  __device__ __forceinline__ void finish() {
    while (pos < n) step();
    flush();
  }
};

// ring depth: enough K tiles in flight to cover an L2 read under load (~1000
// cycles) with two waves per SIMD at MT * NT * (128 FP32 / 48 split) MFMA
// cycles per tile, as far as the registers go
template <class PP, int NT, int MT> constexpr int chain_pf() {
  constexpr bool f32 = sizeof(typename PP::T) == 4;
  const int c = MT * NT * (f32 ? 128 : PP::SPLIT ? 48 : 16);
  if (f32) return c >= 512 ? 2 : 4;
  return c >= 768 ? 1 : c >= 192 ? 2 : 4;
}

// One chunk of MT tiles.  pro(tile, m): loads that the epilogue needs, issued
// before the products; epi(tile, m, acc[NT]).
template <class PP, int NT, int MT, class Side, class Pro, class Epi>
__device__ __forceinline__ void chain_chunk(const void* W, int t0, int tlast, int kt,
                                            const ChainBuf<PP>& in, int lane, bool sync, Side& side,
                                            Pro&& pro, Epi&& epi) {
  f32x4v acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m) pro(t0 + m < tlast ? t0 + m : tlast, m);
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = (f32x4v){0.f, 0.f, 0.f, 0.f};
  chain_mma<PP, NT, MT, chain_pf<PP, NT, MT>()>(acc, W, t0, tlast, kt, 0, kt, in, lane, side);
  if (sync) {  // in place: every wave has read the inputs
    side.finish();
    chain_barrier();
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
    if (t0 + m <= tlast) epi(t0 + m, m, acc[m]);
}

// Tiles of a wave in place: four-wave blocks have layers narrower than 128 (under
// 8 tiles), eight-wave ones up to 512 (32 tiles), by chain_plan's limits
template <int NW> constexpr int chain_inplace() { return NW == 4 ? 2 : 4; }

// One wide layer (mt output tiles over the waves): epi(tile, acc[NT]) for
// every tile.  INPLACE: the outputs may overwrite the inputs (a wave holds all
// its tiles' accumulators until the barrier: chain_inplace<NW> of them at most);
// else chunks of at most four tiles and the output goes to another buffer.  Ends
// with a barrier.
template <class PP, int NT, int NW, bool INPLACE, class Side, class Pro, class Epi>
__device__ __forceinline__ void chain_layer(const void* W, int mt, int kt, const ChainBuf<PP>& in,
                                            int wave, int lane, Side& side, Pro&& pro,
                                            Epi&& epi) {
  const int per = (mt + NW - 1) / NW;
  int t = wave * per;
  const int last = (t + per < mt ? t + per : mt) - 1;
  if constexpr (INPLACE) {
    // (a wave without tiles computes the last one again and drops it)
    const int tl = last < mt - 1 ? last : mt - 1;
    if (chain_inplace<NW>() > 2 && per > 2) chain_chunk<PP, NT, chain_inplace<NW>()>(W, t, tl, kt, in, lane, true, side, pro, epi);
    else if (per > 1) chain_chunk<PP, NT, 2>(W, t, tl, kt, in, lane, true, side, pro, epi);
    else chain_chunk<PP, NT, 1>(W, t, tl, kt, in, lane, true, side, pro, epi);
  } else {
    for (; t + 4 <= last + 1; t += 4) chain_chunk<PP, NT, 4>(W, t, last, kt, in, lane, false, side, pro, epi);
    if (t + 2 <= last + 1) { chain_chunk<PP, NT, 2>(W, t, last, kt, in, lane, false, side, pro, epi); t += 2; }
    if (t <= last) chain_chunk<PP, NT, 1>(W, t, last, kt, in, lane, false, side, pro, epi);
    side.finish();
  }
  chain_barrier();
}

// A narrow layer (state-sized output, mt <= 4 tiles): the K tiles are split
// over the waves; partial products go to LDS as FP32 [split][row][16 mt + 4],
// summed by the reader.  Up to 64 inputs in two splits of 32 features (FP32:
// the GEMM path's plan at these widths, see chain_feat), else four (the waves
// left over).  ALIAS: the partial products overwrite the activations.  Ends
// with a barrier.
template <int NW> __host__ __device__ __forceinline__ int chain_splits(int mt, int kt, int KT) {
  if (kt * KT <= 64) return 2;
  const int s = NW / mt;
  return s > 4 ? 4 : s;
}
template <class PP, int NT, int NW, bool ALIAS, class Side>
__device__ __forceinline__ void chain_narrow(const void* W, int mt, int kt, const ChainBuf<PP>& in,
                                             float* part, int wave, int lane, Side& side) {
  constexpr int KT = ChainK<PP>::KT;
  const int ks = chain_splits<NW>(mt, kt, KT);
  f32x4v acc[2][1][NT];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[u][0][n] = (f32x4v){0.f, 0.f, 0.f, 0.f};
  // (at most two units of work per wave: mt ks <= 2 NW)
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int w = wave + u * NW;
    if (w >= mt * ks) break;
    const int t = w % mt, s = w / mt;
    int k0 = kt * s / ks, k1 = kt * (s + 1) / ks;
    if (kt * KT <= 64) { k0 = s ? 32 / KT : 0; k1 = s ? kt : kt < 32 / KT ? kt : 32 / KT; }
    if (k0 < k1) chain_mma<PP, NT, 1, 4>(acc[u], W, t, t, kt, k0, k1, in, lane, side);
  }
  side.finish();
  if constexpr (ALIAS) chain_barrier();
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int w = wave + u * NW;
    if (w >= mt * ks) break;
    constexpr int CW = ChainK<PP>::CW, TF = ChainK<PP>::TF;
    const int t = w % mt, s = w / mt, pd = TF * mt + 4;
    float* o = part + s * (CW * NT) * pd + (lane & (CW - 1)) * pd + TF * t + 4 * (lane / CW);
#pragma unroll
    for (int n = 0; n < NT; ++n) *(f32x4v*)(o + n * CW * pd) = acc[u][0][n];
  }
  chain_barrier();
}
template <class PP, int NW, int NT>
__device__ __forceinline__ float chain_sum(const float* part, int mt, int kt, int row, int c) {
  const int ks = chain_splits<NW>(mt, kt, ChainK<PP>::KT), pd = ChainK<PP>::TF * mt + 4;
  float v = part[row * pd + c];
  for (int s = 1; s < ks; ++s) v += part[(s * ChainK<PP>::CW * NT + row) * pd + c];
  return v;
}

// FP32: zeros in the pre-activations of tile t, position f, whose features lie past
// the layer's n.  Their weights are zero, but 0 x inf is not: a hidden value that
// overflows would come back as NaN through the padding (the saturating layer
// behind it is finite).  Not needed for tangents and gradients, which an infinity
// leaves non-finite anyway, nor for split BF16, whose lo plane of it is NaN.
// Branchless: a branch around it cost the adjoint row pass 2-3.5%, this 0.5-2%
// (32-256-256-32, 4096 rows: 115.3 -> 115.9 us; 64-400-400-64, 1000 rows: 185 ->
// 188.5).
template <class PP> __device__ __forceinline__ f32x4v chain_keep(f32x4v v, int t, int f, int n) {
  if constexpr (sizeof(typename PP::T) == 4) {
    const int left = n - ChainK<PP>::TF * t - chain_feat(f - ChainK<PP>::TF * t);
    // (features of the four positions: +0, +2, +8, +10)
    v.x = left > 0 ? v.x : 0.f;
    v.y = left > 2 ? v.y : 0.f;
    v.z = left > 8 ? v.z : 0.f;
    v.w = left > 10 ? v.w : 0.f;
  }
  return v;
}

// Runge-Kutta stage values u + dt sum_j A[s][j] k_j: the latest stage first,
// the others in order, the first stage's product with dt * A (the GEMM path's
// stage kernels' order; fused multiply-adds in words, since the compiler moves
// sums across branches and then splits them).  The row is read once and the
// terms are selected, not branched on: a dozen branches per entry were a tenth
// of a small block's stage.  kl: the stage before s.
struct ChainRK {
  float w[5], wl, h;
  int s;
  __device__ __forceinline__ ChainRK(const ChainShared& sh, int s_, float dt) : s(s_) {
    const f32x4v a = *(const f32x4v*)sh.A[s_];
    w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w; w[4] = sh.A[s_][4];
    wl = sh.A[s_][s_ > 0 ? s_ - 1 : 0];
    h = s_ == 1 ? dt * wl : dt;
  }
  template <int NE>
  __device__ __forceinline__ float operator()(float u, const float (&k)[7][NE], float kl, int e) const {
    float sm = wl * kl;
#pragma unroll
    for (int j = 0; j < 5; ++j) {
      const float t = fmaf(w[j], k[j][e], sm);
      sm = j < s - 1 ? t : sm;
    }
    sm = s == 1 ? kl : sm;
    return fmaf(h, sm, u);
  }
};

// error estimate / dt, the same way (k7: the last stage, not in `k` yet)
template <int NE> __device__ __forceinline__ float chain_err(const float (&k)[7][NE], int e, float k7) {
  float v = fmaf(chBT[6], k7, chBT[0] * k[0][e]);
#pragma unroll
  for (int j = 1; j < 6; ++j) v = fmaf(chBT[j], k[j][e], v);
  return v;
}

// Fills ChainShared, the biases and the probe (rows [row0, row0 + R) of
// [B][dm], zero past B).  Ends with a barrier.
template <class PP, int THREADS, int R, bool CNF, bool ADJ>
__device__ __forceinline__ void chain_stage_init(const ChainModel& m, const Ctl* ctl, ChainShared& sh,
                                                 int mode, const float* probe, int row0) {
  const int tid = threadIdx.x;
  if (tid < 56) {
    const int s = tid >> 3, j = tid & 7;
    float v;
    if (j < 7) v = chA[s][j];
    else v = (float)(mode == SM_INIT_F1 ? ctl->t + ctl->tdir * ctl->dt0
                     : mode == SM_STEP ? ctl->t + dC[s] * ctl->dt : ctl->t);
    sh.A[s][j] = v;
  }
  if constexpr (ADJ) {
    const int i = tid - 64;
    if (i >= 0 && i < 64) {
      const int s = i >> 3, j = i & 7;
      sh.w[s][j] = j < 7 ? ctl->st_w[s][j] : ctl->st_dt[s];
      if (j == 0) { sh.step[s] = ctl->st_step[s]; sh.exact[s] = ctl->st_exact[s]; }
    }
  }
  float* lb = (float*)(chain_lds() + m.lds_bias);
  for (int l = 0; l < m.L - 1; ++l)
    for (int i = tid; i < ChainK<PP>::TF * m.mtf[l]; i += THREADS) lb[l * m.wmax + chain_pos<PP>(i)] = m.bias[l][i];
  if constexpr (CNF) {
    float* lp = (float*)(chain_lds() + m.lds_probe);
    for (int i = tid; i < R * m.dm; i += THREADS)
      lp[i] = row0 + i / m.dm < m.B ? probe[(int64_t)row0 * m.dm + i] : 0.f;
  }
  __syncthreads();
}

// activation of four values, chosen once
__device__ __forceinline__ f32x4v act_f4(int a, f32x4v z) {
  switch (a) {
    case 1: return (f32x4v){act_f(1, z.x), act_f(1, z.y), act_f(1, z.z), act_f(1, z.w)};
    case 2: return (f32x4v){act_f(2, z.x), act_f(2, z.y), act_f(2, z.z), act_f(2, z.w)};
    case 3: return (f32x4v){act_f(3, z.x), act_f(3, z.y), act_f(3, z.z), act_f(3, z.w)};
    case 4: return (f32x4v){act_f(4, z.x), act_f(4, z.y), act_f(4, z.z), act_f(4, z.w)};
    default: return z;
  }
}
__device__ __forceinline__ f32x4v act_d4(int a, f32x4v z, f32x4v y) {
  switch (a) {
    case 1: return (f32x4v){act_d(1, z.x, y.x), act_d(1, z.y, y.y), act_d(1, z.z, y.z), act_d(1, z.w, y.w)};
    case 2: return (f32x4v){act_d(2, z.x, y.x), act_d(2, z.y, y.y), act_d(2, z.z, y.z), act_d(2, z.w, y.w)};
    case 3: return (f32x4v){act_d(3, z.x, y.x), act_d(3, z.y, y.y), act_d(3, z.z, y.z), act_d(3, z.w, y.w)};
    case 4: return (f32x4v){act_d(4, z.x, y.x), act_d(4, z.y, y.y), act_d(4, z.z, y.z), act_d(4, z.w, y.w)};
    default: return (f32x4v){1.f, 1.f, 1.f, 1.f};
  }
}

// act' of four FP32 outputs
__device__ __forceinline__ f32x4v act_y4(int a, f32x4v y) {
  switch (a) {
    case 1: return (f32x4v){act_d(1, 0.f, y.x), act_d(1, 0.f, y.y), act_d(1, 0.f, y.z), act_d(1, 0.f, y.w)};
    case 2: return (f32x4v){act_d_y(2, y.x), act_d_y(2, y.y), act_d_y(2, y.z), act_d_y(2, y.w)};
    case 3: return (f32x4v){act_d_y(3, y.x), act_d_y(3, y.y), act_d_y(3, y.z), act_d_y(3, y.w)};
    case 4: return (f32x4v){act_d(4, 0.f, y.x), act_d(4, 0.f, y.y), act_d(4, 0.f, y.z), act_d(4, 0.f, y.w)};
    default: return (f32x4v){1.f, 1.f, 1.f, 1.f};
  }
}

// four features of one row into an LDS buffer
template <class PP>
__device__ __forceinline__ void chain_put4(const ChainBuf<PP>& o, int row, int f, f32x4v v) {
  const float x[4] = {v.x, v.y, v.z, v.w};
  put4<PP>(o.at(row, f), o.plane, x);
}

}  // namespace nodehip
