// Fused forward step of the Tsit5 solve: one launch per step attempt.
//
// Within an attempt a trajectory's stages depend on no other trajectory (the
// shared step size couples them only through the error norm), so a workgroup
// takes a block of rows through all six stages: stage input, the Dense chain
// (chain_common.h), k_s, the embedded error's partial sum.  Bound by the MFMA
// chain of the wide layers (FP32) or by the weights' way from L2 (split BF16);
// it replaces eight kernels per right-hand side whose launches and drains cost
// more than their work at these sizes.  Six stages in one launch:
//   32-256-256-32 FP32, 4096 rows 65 us, 333 or 1000 rows 52 us (16-row blocks
//   60; a 1000-row solve 2.69 -> 0.95 ms in all)
//   17-512-512-16 flow, split BF16, 8192 rows 215 us a step (36 us per
//   right-hand side against 135 us; the density solve 12.0 -> 3.0 ms)
//   2-50-2, one trajectory 17 us, of which half is instruction issue of the
//   stage inputs and epilogues: one wave per SIMD, nothing to overlap
#include <algorithm>

#include "chain_common.h"

namespace nodehip {

int chain_rows(const ChainModel& m, int nt, bool cnf) { return m.cw * nt / (cnf ? 2 : 1); }

// Pending saves of the last accepted step for the block's entries
template <int THREADS>
__device__ __forceinline__ void chain_saves(const ChainFwdArgs& a, int64_t e0, int n) {
  const Ctl* ctl = a.ctl;
  const int64_t lo = ctl->save_lo, hi = ctl->save_hi;
  if (lo >= hi) return;
  const float* ecur = a.tape + tape_slot(ctl, ctl->n) * a.ent;
  const float* es = a.tape + tape_slot(ctl, ctl->save_step) * a.ent;
  const double t = ctl->t, tprev = ctl->tprev, dts = ctl->dt_step;
  const int64_t nreal = (int64_t)a.m.B * a.m.D;
  for (int64_t si = lo; si < hi; ++si) {
    const double ts = a.save_times[si];
    float w[7];
    const bool exact = ts == t;
    if (!exact) interp_weights((ts - tprev) / dts, w);
    float* o = a.out + si * nreal;
    for (int i = threadIdx.x; i < n; i += THREADS) {
      const int64_t idx = e0 + i;
      if (idx >= nreal) break;
      float v;
      if (exact) v = ecur[idx];
      else {
        float sm = 0.f;
#pragma unroll
        for (int j = 0; j < 7; ++j) sm += w[j] * es[(1 + j) * a.sv + idx];
        v = es[idx] + (float)dts * sm;
      }
      o[idx] = v;
    }
  }
}

template <class PP, int NT, int NW, bool CNF>
__global__ void __launch_bounds__(64 * NW, NW == 8 ? 2 : 1) k_chain_fwd(ChainFwdArgs a) {
  using T = typename PP::T;
  constexpr int CH_THREADS = 64 * NW;
  constexpr int CW = ChainK<PP>::CW, TF = ChainK<PP>::TF;
  constexpr int COLS = CW * NT, R = CNF ? COLS / 2 : COLS;
  constexpr int NE = R * (CNF ? 32 : 64) / CH_THREADS;  // state entries per thread (D <= 64, flow 32)
  constexpr int P = PP::SPLIT ? 2 : 1;
  constexpr bool INPLACE = CNF;
  const ChainModel& m = a.m;
  const Ctl* ctl = a.ctl;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int D = m.D, L = m.L, mode = a.mode;
  const int row0 = blockIdx.x * R;
  const int64_t e0 = (int64_t)row0 * D;
  const int ne = R * D;                       // entries of the block
  if (mode == SM_STEP) {
    chain_saves<CH_THREADS>(a, e0, ne);
    if (ctl->done) return;
  }
  const int plane = COLS * m.pitch;
  const int other = INPLACE ? 0 : P * plane;  // offset of the second buffer
  const ChainBuf<PP> in0{0, m.pitch, plane};
  float* part = (float*)(chain_lds() + m.lds_part);
  const float* lbias = (const float*)(chain_lds() + m.lds_bias);
  const float* lprobe = (const float*)(chain_lds() + m.lds_probe);
  __shared__ ChainShared sh;
  chain_stage_init<PP, 64 * NW, R, CNF, false>(m, ctl, sh, mode, a.probe, row0);

  const int64_t n = mode == SM_STEP ? ctl->n : 0;
  // (the block's entries: uniform bases, 32-bit offsets)
  float* ent = a.tape + tape_slot(ctl, n) * a.ent + e0;
  float* nxt = a.tape + tape_slot(ctl, n + 1) * a.ent + e0;
  const float dt = (float)ctl->dt, h0 = (float)(ctl->tdir * ctl->dt0);
  const float atol = (float)ctl->abstol, rtol = (float)ctl->reltol;

  // this thread's state entries: row and column in the block
  int row[NE], col[NE];
  float u[NE], k[7][NE], kl[NE];               // kl: the last stage's k
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const int i = tid + e * CH_THREADS;
    row[e] = i / D;
    col[e] = i - row[e] * D;
    u[e] = 0.f;
#pragma unroll
    for (int s = 0; s < 7; ++s) k[s][e] = 0.f;
    if (i < ne) {
      u[e] = ent[i];
      if (mode == SM_STEP || mode == SM_INIT_F1) k[0][e] = (ent + a.sv)[i];
    }
    kl[e] = k[0][e];
  }
  double sum = 0.0, flag = 0.0;
  ChainNoSide none;
  const int s0 = mode == SM_STEP ? 1 : 0, s1 = mode == SM_STEP ? 7 : 1;
  float un[NE];
  for (int s = s0; s < s1; ++s) {
    // stage input
    const float ts = sh.A[s][7];
    const ChainRK rk(sh, s, dt);
    const int kin = m.ktf[0] * ChainK<PP>::KT;
    // columns past the state's: the time column, zeros
    for (int c = m.dm + tid / COLS; c < kin; c += CH_THREADS / COLS) {
      const int r = tid % COLS;
      put<PP>(in0.at(r, chain_pos<PP>(c)), plane, CNF && m.tcat && c == m.dm && r < R ? ts : 0.f);
    }
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      if (e * CH_THREADS >= ne) continue;   // (uniform: small states use the first entry only)
      if (tid + e * CH_THREADS >= ne) continue;
      float v = u[e];
      if (mode == SM_STEP) {
        v = rk(u[e], k, kl[e], e);
        un[e] = v;
      } else if (mode == SM_INIT_F1) {
        v = fmaf(h0, k[0][e], u[e]);
      }
      if (col[e] < m.dm) {
        const int cp = chain_pos<PP>(col[e]);
        put<PP>(in0.at(row[e], cp), plane, map_f(m.map, v));
        if constexpr (CNF)
          put<PP>(in0.at(R + row[e], cp), plane, lprobe[row[e] * m.dm + col[e]]);
      }
    }
    if (mode == SM_STEP && s == 6) {
#pragma unroll
      for (int e = 0; e < NE; ++e)
        if (tid + e * CH_THREADS < ne) nxt[tid + e * CH_THREADS] = un[e];
    }
    chain_barrier();
    int cur = 0;
    for (int l = 0; l < L - 1; ++l) {
      const ChainBuf<PP> in{cur, m.pitch, plane}, o{other - cur, m.pitch, plane};
      const float* bias = lbias + l * m.wmax;
      const int act = m.act[l], nout = m.out[l];
      auto epi = [&](int t, int, f32x4v (&acc)[NT]) {
        const int f = TF * t + 4 * (lane / CW), r = lane & (CW - 1);
        const f32x4v bv = *(const f32x4v*)(bias + f);
#pragma unroll
        for (int q = 0; q < (CNF ? NT / 2 : NT); ++q) {
          const f32x4v z = chain_keep<PP>(acc[q] + bv, t, f, nout), y = act_f4(act, z);
          chain_put4<PP>(o, CW * q + r, f, y);
          if constexpr (CNF)
            chain_put4<PP>(o, R + CW * q + r, f, acc[q + NT / 2] * act_d4(act, z, y));
        }
      };
      chain_layer<PP, NT, NW, INPLACE>(m.Wf[l], m.mtf[l], m.ktf[l], in, wave, lane, none,
                                       [](int, int) {}, epi);
      cur = other - cur;
    }
    const int ll = L - 1, mt = m.mtf[ll];
    chain_narrow<PP, NT, NW, INPLACE>(m.Wf[ll], mt, m.ktf[ll], ChainBuf<PP>{cur, m.pitch, plane}, part, wave, lane, none);
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      if (e * CH_THREADS >= ne) continue;
      const int i = tid + e * CH_THREADS;
      if (i >= ne) continue;
      float kv;
      if (!CNF || col[e] < m.dm) {
        kv = act_f(m.act[ll], chain_sum<PP, NW, NT>(part, mt, m.ktf[ll], row[e], col[e]) + m.bias[ll][col[e]]);
      } else {  // log p: minus the probe's directional derivative of f
        kv = 0.f;
        for (int c = 0; c < m.dm; ++c)
          kv -= lprobe[row[e] * m.dm + c] * chain_sum<PP, NW, NT>(part, mt, m.ktf[ll], R + row[e], c);
      }
      const bool live = row0 + row[e] < m.B;
      if (mode == SM_STEP) {
        (ent + (1 + s) * a.sv)[i] = kv;
        if (s == 6) {
          (nxt + a.sv)[i] = kv;  // FSAL
          const float ut = dt * chain_err(k, e, kv);
          const float sk = atol + fmaxf(fabsf(u[e]), fabsf(un[e])) * rtol;
          if (live) {
            const double q = (double)(ut / sk);
            sum += q * q;
            if (isnan(un[e])) flag = 1.0;
          }
        }
#pragma unroll
        for (int j = 1; j < 6; ++j) k[j][e] = j == s ? kv : k[j][e];
        kl[e] = kv;
      } else if (mode == SM_INIT_F0) {
        (ent + a.sv)[i] = kv;
        const float sk = atol + fabsf(u[e]) * rtol;
        if (live) {
          const double q = (double)(kv / sk);
          sum += q * q;
        }
      } else {
        const float sk = atol + fabsf(u[e]) * rtol, d = kv - k[0][e];
        if (live) {
          const double q = (double)(d / sk);
          sum += q * q;
          if (d != 0.f) flag = 1.0;
        }
      }
    }
    chain_barrier();  // (in place: the partial products lie over the next stage's inputs)
  }
  block_reduce_store(sum, flag, a.part, blockIdx.x);
}

void chain_layout(ChainModel& m, int nt, bool cnf) {
  // four bytes per activation: FP32, or two BF16 planes
  const int cols = m.cw * nt, act = (cnf ? 1 : 2) * cols * m.pitch * 4;
  int part = 0;
  m.wmax = 4;
  for (int i = 0; i < 2; ++i) {
    const int x = i ? m.mtb[0] : m.mtf[m.L - 1], k = i ? m.ktb[0] : m.ktf[m.L - 1];
    const int ks = m.nw == 8 ? chain_splits<8>(x, k, m.kt) : chain_splits<4>(x, k, m.kt);
    part = std::max(part, ks * cols * (m.tf * x + 4) * 4);
  }
  for (int l = 0; l < m.L - 1; ++l) m.wmax = std::max(m.wmax, m.tf * m.mtf[l]);
  m.lds_part = cnf ? 0 : act;
  m.lds_bias = cnf ? std::max(act, part) : act + part;
  m.lds_probe = m.lds_bias + (m.L - 1) * m.wmax * 4;
  m.lds_bytes = m.lds_probe + (cnf ? chain_rows(m, nt, true) * m.dm * 4 : 0);
}

void launch_chain_fwd(int prec, int nt, bool cnf, const ChainFwdArgs& a, int grid, hipStream_t s) {
  const size_t lds = a.m.lds_bytes;
  const int nw = a.m.nw;
  auto go = [&](auto kern) {
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, CHAIN_LDS_MAX);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * nw), lds, s, a);
  };
  if (prec == 0 && a.m.cw == 4) {
    if (nw == 8) go(k_chain_fwd<PF32S, 2, 8, false>);
    else go(k_chain_fwd<PF32S, 2, 4, false>);
  } else if (prec == 0) {
    if (cnf && nw == 8) go(k_chain_fwd<PF32, 2, 8, true>);
    else if (cnf) go(k_chain_fwd<PF32, 2, 4, true>);
    else if (nw == 8) go(k_chain_fwd<PF32, 1, 8, false>);
    else go(k_chain_fwd<PF32, 1, 4, false>);
  } else if (cnf) {
    if (nt == 4) go(k_chain_fwd<PBF16X3, 4, 8, true>);
    else if (nw == 8) go(k_chain_fwd<PBF16X3, 2, 8, true>);
    else go(k_chain_fwd<PBF16X3, 2, 4, true>);
  } else {
    if (nt == 2) go(k_chain_fwd<PBF16X3, 2, 8, false>);
    else if (nw == 8) go(k_chain_fwd<PBF16X3, 1, 8, false>);
    else go(k_chain_fwd<PBF16X3, 1, 4, false>);
  }
}

// Weights in fragment order.  One thread per lane of a fragment: V (4 FP32 or
// 8 BF16) consecutive K values of one output feature, zero past the layer's
// own size.  The forward fragments read the flat vector (W[o, i] at
// i * out + o) along o, the backward ones V consecutive values of a row.
template <class PP>
__global__ void __launch_bounds__(256) k_pack_chain(ChainPack a, const float* __restrict__ p) {
  using T = typename PP::T;
  constexpr int V = ChainK<PP>::V, KT = ChainK<PP>::KT, P = PP::SPLIT ? 2 : 1;
  constexpr int TF = ChainK<PP>::TF, NV = TF / 16;   // vectors of a K tile per lane (64 x 4 tiles: four)
  const int l = blockIdx.y >> 1;
  const bool bwd = blockIdx.y & 1;
  T* W = (T*)(bwd ? a.Wb[l] : a.Wf[l]);
  if (!W) return;
  const int mt = bwd ? a.mtb[l] : a.mtf[l], kt = bwd ? a.ktb[l] : a.ktf[l];
  const int in = a.in[l], out = a.out[l];
  const bool hid = bwd ? l > 0 : l < a.nl - 1;   // hidden features on the M side
  constexpr bool F32 = sizeof(T) == 4;           // (stored in chain_feat order)
  const float* w = p + a.w0[l];
  const int64_t nfl = (int64_t)mt * kt * NV * 64;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nfl;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int lane = (int)(i & 63);
    const int64_t f = i >> 6;                        // (fragment, vector)
    const int t = (int)(f / NV / kt), k = (int)(f / NV % kt);
    const int mr = TF * t + (lane & (TF - 1)), k0 = k * KT + V * (TF == 64 ? (int)(f & 3) : lane >> 4);
    const int mrow = F32 && hid ? chain_feat(mr) : mr;
    T* d = W + (f * P * 64 + lane) * V;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int kk = F32 ? chain_feat(k0 + j) : k0 + j;
      const int o = bwd ? kk : mrow, ii = bwd ? mrow : kk;
      const float v = o < out && ii < in ? w[(int64_t)ii * out + o] : 0.f;
      put<PP>(d + j, 64 * V, v);
    }
  }
}

void launch_pack_chain(int prec, const ChainPack& a, const float* p, hipStream_t s) {
  int64_t most = 1;
  for (int l = 0; l < a.nl; ++l) {
    const int64_t f = (int64_t)a.mtf[l] * a.ktf[l], b = (int64_t)a.mtb[l] * a.ktb[l];
    most = f > most ? f : most;
    most = b > most ? b : most;
  }
  const int grid = (int)((most + 3) / 4 < 1024 ? (most + 3) / 4 : 1024);
  if (prec == 0 && a.tf == 64)
    hipLaunchKernelGGL(k_pack_chain<PF32S>, dim3(grid, 2 * a.nl), dim3(256), 0, s, a, p);
  else if (prec == 0) hipLaunchKernelGGL(k_pack_chain<PF32>, dim3(grid, 2 * a.nl), dim3(256), 0, s, a, p);
  else hipLaunchKernelGGL(k_pack_chain<PBF16X3>, dim3(grid, 2 * a.nl), dim3(256), 0, s, a, p);
}

}  // namespace nodehip
