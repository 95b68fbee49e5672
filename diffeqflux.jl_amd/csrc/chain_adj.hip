// Fused adjoint step: three launches per step attempt besides the controller.
//
// k_chain_adj takes a block of rows through all stages of the adjoint's Tsit5
// step (step begin, u at the stage time, hidden recompute, data gradients,
// k^lambda): lambda's rows are independent within an attempt, as the forward's
// are.  It leaves each stage's layer inputs and output gradients behind, and
// k_chain_wgrad forms from them the two sums over stages that the parameter
// state needs (sum_s b_s G_s and sum_s bt_s G_s), one pass over the batch with
// both sums in registers; k_chain_mu adds the row ranges' partial sums, forms
// the speculative mu and its error norm.  Per-stage launches of one kernel per
// GEMM, stage, fold and norm (12 per VJP) spent most of their time in launches,
// drains and partial sums through memory.
//
// A step attempt of k_chain_adj (median of the launches with work), and the
// training step it belongs to before and now:
//   32-256-256-32 FP32, 4096 rows   135 us   17.6 -> 6.2 ms
//   the same, 333 rows              111 us   12.5 -> 4.3 ms
//   2-50-2 FP32, one trajectory      31 us   13.6 -> 3.8 ms (29 to 66 steps by
//                                            inputs: 2.5 to 5 ms)
//   17-512-512-16 flow, split BF16,
//   8192 rows                       568 us   38.8 -> 13.7 ms
// Bound by the matrix pipe and the phases around it: of a 16-row block's 43,000
// cycles per stage (256-wide layers) 20,000 are MFMA, the rest layer
// prologues, epilogues and barriers that two waves per SIMD only half hide; a
// 50-wide model's stage (9,800 cycles) is instruction issue throughout.
#include "chain_common.h"

namespace nodehip {

// Sum over the 16 lanes of a row of the wave (in every one of them)
__device__ __forceinline__ float row16_sum(float x) {
  auto ror = [](float v, auto n) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + n(),
                                                                 0xf, 0xf, true));
  };
  x += ror(x, std::integral_constant<int, 8>{});
  x += ror(x, std::integral_constant<int, 4>{});
  x += ror(x, std::integral_constant<int, 2>{});
  x += ror(x, std::integral_constant<int, 1>{});
  return x;
}

template <class PP, int NT, int NW, bool CNF>
__global__ void __launch_bounds__(64 * NW, NW == 8 ? 2 : 1) k_chain_adj(ChainAdjArgs a) {
  using T = typename PP::T;
  constexpr int THREADS = 64 * NW;
  constexpr int CW = ChainK<PP>::CW, TF = ChainK<PP>::TF;
  constexpr int COLS = CW * NT, R = CNF ? COLS / 2 : COLS;
  constexpr int NE = R * (CNF ? 32 : 64) / THREADS;
  constexpr int P = PP::SPLIT ? 2 : 1;
  constexpr bool INPLACE = CNF;
  constexpr bool F32 = sizeof(T) == 4;
  using Side = typename std::conditional<F32, ChainNoSide, ChainCopy<PP, THREADS>>::type;
  constexpr int NP = CNF ? NT / 2 : NT;        // column tiles of primal rows
  const ChainModel& m = a.m;
  const Ctl* ctl = a.ctl;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int D = m.D, L = m.L, mode = a.mode;
  const int row0 = blockIdx.x * R;             // first trajectory
  const int64_t orow0 = (int64_t)blockIdx.x * COLS;  // first operand row
  const int64_t e0 = (int64_t)row0 * D;
  const int ne = R * D;
  const int64_t nreal = (int64_t)m.B * D;
  const bool bs = !CNF && a.ubs != nullptr;
  const float dt = (float)ctl->dt;
  const float atol = (float)ctl->abstol, rtol = (float)ctl->reltol;
  const int gsel = ctl->gsel;

  int row[NE], col[NE];
  float ld[NE];                                // a flow's lambda_dlogp of the row (constant)
  float lam[NE], k[7][NE], kl[NE], ub[NE];     // kl: the last stage's k
  const int acc_ = mode == SM_STEP ? ctl->last_accept : 0;
  const int jidx = mode == SM_STEP ? ctl->jump_idx : -1;
  const bool re = mode == SM_STEP && ctl->fsal_reeval;
  // step begin: lambda (and u) of the accepted step, the cotangent jump, the
  // FSAL stage.  Idempotent: attempts enqueued past the end repeat it.
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const int i = tid + e * THREADS;
    row[e] = i / D;
    col[e] = i - row[e] * D;
    lam[e] = ub[e] = ld[e] = kl[e] = 0.f;
#pragma unroll
    for (int s = 0; s < 7; ++s) k[s][e] = 0.f;
    if (i >= ne) continue;
    const int64_t idx = e0 + i;
    float l = acc_ ? a.lam_new[idx] : a.lam[idx];
    if (acc_ && jidx >= 0 && idx < nreal) l += a.dLdout[(int64_t)jidx * nreal + idx];
    lam[e] = l;
    if (CNF && row0 + row[e] < m.B) ld[e] = a.lam[(int64_t)(row0 + row[e]) * D + m.dm];
    if (mode != SM_INIT_F0) k[0][e] = acc_ ? a.kl[6 * a.sv + idx] : a.kl[idx];
    kl[e] = k[0][e];
    if (acc_) { a.lam[idx] = l; a.kl[idx] = k[0][e]; }
    if (bs) {
      float u = acc_ ? a.ubs_new[idx] : a.ubs[idx];
      if (acc_ && jidx >= 0 && a.ckpt && idx < nreal) u = a.fsaved[(int64_t)jidx * nreal + idx];
      ub[e] = u;
      if (acc_) { a.ubs[idx] = u; a.ku[idx] = a.ku[6 * a.sv + idx]; }
    }
  }
  if (mode == SM_STEP && ctl->done) return;

  const int plane = COLS * m.pitch;
  const int other = INPLACE ? 0 : P * plane;
  const ChainBuf<PP> in0{0, m.pitch, plane};
  float* part = (float*)(chain_lds() + m.lds_part);
  const float* lbias = (const float*)(chain_lds() + m.lds_bias);
  const float* lprobe = (const float*)(chain_lds() + m.lds_probe);
  __shared__ ChainShared sh;
  chain_stage_init<PP, THREADS, R, CNF, true>(m, ctl, sh, mode, a.probe, row0);
  const float h0 = (float)(ctl->tdir * ctl->dt0);
  const int64_t orows = a.ops.rows;
  const int64_t sbase = (int64_t)blockIdx.x * (L - 1) * a.stiles;  // tiles of act' before the block
  // FP32: where layer l's inputs / output gradients of the block go; split:
  // the copy that takes them there from an LDS buffer
  auto rows_at = [&](char* ob, int64_t off, int w) { return (T*)(ob + off) + orow0 * w; };
  auto copy_of = [&](int buf, char* ob, int64_t off, int w, int used) {
    if constexpr (F32) return Side{};
    else return Side(ChainBuf<PP>{buf, m.pitch, plane}, ob + off, orows, orow0, w, used, COLS);
  };
  // u(t_s): the tape's entries are loaded a stage ahead
  float tv[8][NE];
  auto tape_load = [&](int is) {
    const float* te = a.tape + (int64_t)sh.step[is] * a.ent + e0;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      if (e * THREADS >= ne) continue;   // (uniform: small states use the first entry only)
      const int i = tid + e * THREADS < ne ? tid + e * THREADS : 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) tv[j][e] = (te + j * a.sv)[i];
    }
  };
  double sum = 0.0, flag = 0.0;
  const int s0 = mode == SM_STEP && !re ? 1 : 0, s1 = mode == SM_STEP ? 7 : 1;
  if (!bs) tape_load(mode == SM_INIT_F1 ? 7 : s0);
  for (int s = s0; s < s1; ++s) {
    const int slot = s == 0 ? (mode == SM_INIT_F1 ? 2 : gsel) : s == 6 ? (gsel ^ 1) : s + 1;
    char* ob = (char*)a.ops.base + (int64_t)slot * a.ops.slot;
    const int is = mode == SM_INIT_F1 ? 7 : s;   // interpolation slot
    const float ts = sh.A[s][7];
    const ChainRK rk(sh, s, dt);
    // stage inputs: x = map(u(t_s)) now, lambda_s after the hidden recompute
    const bool ex = sh.exact[is] != 0;
    const float tdt = sh.w[is][7];
    float ls[NE], us[NE];
    T* const x0r = rows_at(ob, a.ops.h[0], a.ops.w[0]);
    {
      const int kin = m.ktf[0] * ChainK<PP>::KT;
      for (int c = m.dm + tid / COLS; c < kin; c += THREADS / COLS) {
        const int r = tid % COLS;
        const bool tc = CNF && m.tcat && c == m.dm && r < R;
        const float v = tc && row0 + r < m.B ? ts : 0.f;
        const int cp = chain_pos<PP>(c);
        put<PP>(in0.at(r, cp), plane, v);
        if constexpr (F32) if (tc) x0r[r * a.ops.w[0] + cp] = v;
      }
    }
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      ls[e] = us[e] = 0.f;
      if (e * THREADS >= ne) continue;
      const int i = tid + e * THREADS;
      if (i >= ne) continue;
      const int64_t idx = e0 + i;
      float u;
      if (bs) {
        // (u's stage values stay in memory: each is read by its own thread)
        if (mode == SM_INIT_F1) u = fmaf(h0, a.ku[idx], ub[e]);
        else if (s == 0) u = ub[e];
        else {
          float ku[7][1];  // (entries past the stage before are read, not used)
#pragma unroll
          for (int j = 0; j < 5; ++j) ku[j][0] = a.ku[j * a.sv + idx];
          u = rk(ub[e], ku, a.ku[(s - 1) * a.sv + idx], 0);
        }
      } else {
        u = tv[0][e];
        if (!ex) {
          float sm = 0.f;
#pragma unroll
          for (int j = 0; j < 7; ++j) sm = fmaf(sh.w[is][j], tv[1 + j][e], sm);
          u = fmaf(tdt, sm, u);
        }
      }
      us[e] = u;
      if (mode == SM_INIT_F1) ls[e] = fmaf(h0, k[0][e], lam[e]);
      else if (s == 0) ls[e] = lam[e];
      else ls[e] = rk(lam[e], k, kl[e], e);
      if (col[e] < m.dm) {
        const float x = map_f(m.map, u);
        const int cp = chain_pos<PP>(col[e]);
        put<PP>(in0.at(row[e], cp), plane, x);
        if constexpr (F32) x0r[row[e] * a.ops.w[0] + cp] = x;
        if constexpr (CNF) {
          const float p = lprobe[row[e] * m.dm + col[e]];
          put<PP>(in0.at(R + row[e], cp), plane, p);
          if constexpr (F32) x0r[(R + row[e]) * a.ops.w[0] + cp] = p;
        }
      }
    }
    if (mode == SM_STEP && s == 6) {
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int i = tid + e * THREADS;
        if (i >= ne) continue;
        a.lam_new[e0 + i] = ls[e];
        if (bs) a.ubs_new[e0 + i] = us[e];
      }
    }
    if (!bs && s + 1 < s1) tape_load(s + 1);
    chain_barrier();
    // hidden recompute (a flow: with its tangent chain), act' and the
    // second-order factor act'' adot kept for the way back.  The lane that
    // writes an entry of them reads it again below: both sweeps deal a
    // layer's tiles to the waves alike.
    int cur = 0;
    for (int l = 0; l < L - 1; ++l) {
      const ChainBuf<PP> in{cur, m.pitch, plane}, o{other - cur, m.pitch, plane};
      const float* bias = lbias + l * m.wmax;
      const int act = m.act[l], nout = m.out[l];
      T* const hr = rows_at(ob, a.ops.h[l + 1], a.ops.w[l + 1]);
      const int hw = a.ops.w[l + 1];
      // act' (FP32 derives it from the stored output instead) and act'' adot in
      // the lanes' own order: whole lines per access
      f32x4v* sl = (f32x4v*)a.slope + (sbase + (int64_t)l * a.stiles) * NP * 64 + lane;
      f32x4v* cv = (f32x4v*)a.curve + (sbase + (int64_t)l * a.stiles) * NP * 64 + lane;
      auto epi = [&](int t, int, f32x4v (&acc)[NT]) {
        const int f = TF * t + 4 * (lane / CW);
        const f32x4v bv = *(const f32x4v*)(bias + f);
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          const int r = CW * q + (lane & (CW - 1));
          const f32x4v z = chain_keep<PP>(acc[q] + bv, t, f, nout), y = act_f4(act, z);
          chain_put4<PP>(o, r, f, y);
          if constexpr (F32) *(f32x4v*)(hr + r * hw + f) = y;
          else sl[(t * NP + q) * 64] = act_d4(act, z, y);
          if constexpr (CNF) {
            const f32x4v d = act_d4(act, z, y);
            const f32x4v tv = acc[q + NP] * d;
            chain_put4<PP>(o, R + r, f, tv);
            if constexpr (F32) *(f32x4v*)(hr + (R + r) * hw + f) = tv;
            // act'' adot in closed form (act' adot = t)
            f32x4v c2 = {0.f, 0.f, 0.f, 0.f};
            if (act == 1) c2 = -2.f * y * tv;
            else if (act == 2) c2 = tv * (1.f - d);
            else if (act == 4) c2 = tv * (1.f - 2.f * y);
            cv[(t * NP + q) * 64] = c2;
          }
        }
      };
      // (split: the layer's input leaves for the weight gradients meanwhile)
      Side copy = copy_of(cur, ob, a.ops.h[l], a.ops.w[l], m.ktf[l] * ChainK<PP>::KT);
      chain_layer<PP, NT, NW, INPLACE>(m.Wf[l], m.mtf[l], m.ktf[l], in, wave, lane, copy,
                                       [](int, int) {}, epi);
      cur = other - cur;
    }
    const int ll = L - 1;
    // the last layer's input: copied under its own products (backsolve), or
    // here
    Side lastc = copy_of(cur, ob, a.ops.h[ll], a.ops.w[ll], m.ktf[ll] * ChainK<PP>::KT);
    float fu[NE];
    if (bs) {  // f(u_s): u's own stage value
      const int mt = m.mtf[ll];
      chain_narrow<PP, NT, NW, INPLACE>(m.Wf[ll], mt, m.ktf[ll], ChainBuf<PP>{cur, m.pitch, plane}, part,
                                        wave, lane, lastc);
#pragma unroll
      for (int e = 0; e < NE; ++e)
        fu[e] = tid + e * THREADS < ne
                    ? chain_sum<PP, NW, NT>(part, mt, m.ktf[ll], row[e], col[e]) + m.bias[ll][col[e]] : 0.f;
      chain_barrier();
    }
    lastc.finish();
    if constexpr (INPLACE && !F32) chain_barrier();
    // seeds at the output: lambda_s (a flow's tangent rows: -lambda_dlogp e)
    cur = other - cur;
    {
      const ChainBuf<PP> o{cur, m.pitch, plane};
      const int kin = m.ktb[ll] * ChainK<PP>::KT;
      for (int c = m.dm + tid / COLS; c < kin; c += THREADS / COLS)
        put<PP>(o.at(tid % COLS, chain_pos<PP>(c)), plane, 0.f);
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int i = tid + e * THREADS;
        if (i >= ne || col[e] >= m.dm) continue;
        T* const dr = rows_at(ob, a.ops.d[ll], a.ops.w[L]);
        const int cp = chain_pos<PP>(col[e]);
        put<PP>(o.at(row[e], cp), plane, ls[e]);
        if constexpr (F32) dr[row[e] * a.ops.w[L] + cp] = ls[e];
        if constexpr (CNF) {
          const float p = -ld[e] * lprobe[row[e] * m.dm + col[e]];
          put<PP>(o.at(R + row[e], cp), plane, p);
          if constexpr (F32) dr[(R + row[e]) * a.ops.w[L] + cp] = p;
        }
      }
    }
    chain_barrier();
    for (int l = ll; l >= 1; --l) {
      const ChainBuf<PP> in{cur, m.pitch, plane}, o{other - cur, m.pitch, plane};
      T* const dr = rows_at(ob, a.ops.d[l - 1], a.ops.w[l]);
      const int dw = a.ops.w[l], act = m.act[l - 1];
      float* const bsr = a.bsum + (((int64_t)slot * gridDim.x + blockIdx.x) * (L - 1) + l - 1) * a.bw;
      const T* const hr = rows_at(ob, a.ops.h[l], dw);
      const f32x4v* sl = (const f32x4v*)a.slope + (sbase + (int64_t)(l - 1) * a.stiles) * NP * 64 + lane;
      const f32x4v* cv = (const f32x4v*)a.curve + (sbase + (int64_t)(l - 1) * a.stiles) * NP * 64 + lane;
      // FP32 blocks read act' ahead of the products, the split ones have no
      // registers left for it
      constexpr int ME = F32 ? (INPLACE ? chain_inplace<NW>() : 4) : 1;
      f32x4v sd[ME][NP], c2[CNF ? ME : 1][NP];
      auto read = [&](int t, int mi) {
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          if constexpr (F32)
            sd[mi][q] = *(const f32x4v*)(hr + (CW * q + (lane & (CW - 1))) * dw + TF * t + 4 * (lane / CW));
          else sd[mi][q] = sl[(t * NP + q) * 64];
          if constexpr (CNF) c2[mi][q] = cv[(t * NP + q) * 64];
        }
      };
      auto pro = [&](int t, int mi) { if constexpr (F32) read(t, mi); };
      auto epi = [&](int t, int mi, f32x4v (&acc)[NT]) {
        const int f = TF * t + 4 * (lane / CW);
        const int i = F32 ? mi : 0;
        if constexpr (!F32) read(t, 0);
        f32x4v bs4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          const int r = CW * q + (lane & (CW - 1));
          f32x4v d = sd[i][q];
          if constexpr (F32) d = act_y4(act, d);
          f32x4v v = acc[q] * d;
          if constexpr (CNF) {
            v += acc[q + NP] * c2[i][q];
            const f32x4v tv = acc[q + NP] * d;
            chain_put4<PP>(o, R + r, f, tv);
            if constexpr (F32) *(f32x4v*)(dr + (R + r) * dw + f) = tv;
          }
          chain_put4<PP>(o, r, f, v);
          if constexpr (F32) *(f32x4v*)(dr + r * dw + f) = v;
          else bs4 += v;
        }
        if constexpr (!F32) {  // (the 16 lanes of a row of the wave hold a row of the block each)
#pragma unroll
          for (int j = 0; j < 4; ++j) bs4[j] = row16_sum(bs4[j]);
          if ((lane & 15) == 0) *(f32x4v*)(bsr + f) = bs4;
        }
      };
      Side copy = copy_of(cur, ob, a.ops.d[l], a.ops.w[l + 1], m.ktb[l] * ChainK<PP>::KT);
      chain_layer<PP, NT, NW, INPLACE>(m.Wb[l], m.mtb[l], m.ktb[l], in, wave, lane, copy, pro, epi);
      cur = other - cur;
    }
    const int mt = m.mtb[0];
    Side copy0 = copy_of(cur, ob, a.ops.d[0], a.ops.w[1], m.ktb[0] * ChainK<PP>::KT);
    chain_narrow<PP, NT, NW, INPLACE>(m.Wb[0], mt, m.ktb[0], ChainBuf<PP>{cur, m.pitch, plane}, part,
                                      wave, lane, copy0);
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      if (e * THREADS >= ne) continue;
      const int i = tid + e * THREADS;
      if (i >= ne) continue;
      float kv = 0.f;                            // (log p column: lambda constant)
      if (!CNF || col[e] < m.dm) {
        float g = chain_sum<PP, NW, NT>(part, mt, m.ktb[0], row[e], col[e]);
        if (m.map == 1) g *= 3.f * us[e] * us[e];
        kv = -g;
      }
      const int64_t idx = e0 + i;
      const bool live = idx < nreal;
      auto add = [&](float d, float p, float q) {
        const float sk = atol + fmaxf(fabsf(p), fabsf(q)) * rtol;
        if (live) { const double v = (double)(d / sk); sum += v * v; }
      };
      if (mode == SM_STEP) {
        if (s == 0) a.kl[idx] = kv;
        if (bs) a.ku[s * a.sv + idx] = fu[e];
        if (s == 6) {
          a.kl[6 * a.sv + idx] = kv;
          const float ut = chain_err(k, e, kv);
          add(ut * dt, lam[e], ls[e]);
          if (live && isnan(ls[e])) flag = 1.0;
          if (bs) {
            float uu = fmaf(chBT[6], fu[e], chBT[0] * a.ku[idx]);
            for (int j = 1; j < 6; ++j) uu = fmaf(chBT[j], a.ku[j * a.sv + idx], uu);
            add(uu * dt, ub[e], us[e]);
            if (live && isnan(us[e])) flag = 1.0;
          }
        }
#pragma unroll
        for (int j = 0; j < 6; ++j) k[j][e] = j == s ? kv : k[j][e];
        kl[e] = kv;
      } else if (mode == SM_INIT_F0) {
        a.kl[idx] = kv;
        add(kv, lam[e], 0.f);
        if (bs) { a.ku[idx] = fu[e]; add(fu[e], ub[e], 0.f); }
      } else {
        add(kv - k[0][e], lam[e], 0.f);
        if (live && kv != k[0][e]) flag = 1.0;
        if (bs) {
          const float f0 = a.ku[idx];
          add(fu[e] - f0, ub[e], 0.f);
          if (live && fu[e] != f0) flag = 1.0;
        }
      }
    }
    // (the next stage's inputs go to buffer 0; `part` is written again only
    // after the barriers of its layers)
    chain_barrier();
  }
  block_reduce_store(sum, flag, a.part, blockIdx.x);
}

void launch_chain_adj(int prec, int nt, bool cnf, const ChainAdjArgs& a, int grid, hipStream_t s) {
  const size_t lds = a.m.lds_bytes;
  const int nw = a.m.nw;
  auto go = [&](auto kern) {
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, CHAIN_LDS_MAX);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * nw), lds, s, a);
  };
  if (prec == 0 && a.m.cw == 4) {
    if (nw == 8) go(k_chain_adj<PF32S, 2, 8, false>);
    else go(k_chain_adj<PF32S, 2, 4, false>);
  } else if (prec == 0) {
    if (cnf && nw == 8) go(k_chain_adj<PF32, 2, 8, true>);
    else if (cnf) go(k_chain_adj<PF32, 2, 4, true>);
    else if (nw == 8) go(k_chain_adj<PF32, 1, 8, false>);
    else go(k_chain_adj<PF32, 1, 4, false>);
  } else if (cnf) {
    if (nt == 4) go(k_chain_adj<PBF16X3, 4, 8, true>);
    else if (nw == 8) go(k_chain_adj<PBF16X3, 2, 8, true>);
    else go(k_chain_adj<PBF16X3, 2, 4, true>);
  } else {
    if (nw == 8) go(k_chain_adj<PBF16X3, 1, 8, false>);
    else go(k_chain_adj<PBF16X3, 1, 4, false>);
  }
}

// ---------------------------------------------------------------- weight gradients
// G_l[i][o] = sum over rows of h[row][i] d[row][o] per stage, K = rows, folded
// into acc_b = sum_s b_s G_s and acc_e = sum_s bt_s G_s in registers.
// Stage coefficients: the step's b and bt, or one stage alone (initial dt).
__device__ __forceinline__ int wg_slot(int mode, int s, int gsel) {
  if (mode == SM_INIT_F1) return 2;
  return s == 0 ? gsel : s == 6 ? (gsel ^ 1) : s + 1;
}

// Whether stage s has a weight in the quadrature (the last one has none; it is
// left out rather than multiplied by 0: its operands may have overflowed)
__device__ __forceinline__ bool wg_quad(int mode, int s) { return mode != SM_STEP || s < 6; }

// tile index -> layer, tile row (inputs) and column (outputs)
__device__ __forceinline__ int wg_tile(const ChainWgradArgs& a, int tile, int& it, int& ot) {
  int l = 0;
  while (l + 1 < a.m.L && tile >= a.tl[l + 1]) ++l;
  const int t = tile - a.tl[l];
  it = t / a.tw[l];
  ot = t % a.tw[l];
  return l;
}

// Block -> (tile, row range).  Blocks go to the eight XCDs in turn; each XCD
// gets a contiguous piece of the (range, tile) sequence, so that a range's rows
// are read into one L2 and serve all its tiles there (spread over the XCDs every
// L2 read every row).  False: no work.
__device__ __forceinline__ bool wg_block(const ChainWgradArgs& a, int& tile, int& chunk) {
  const int m = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  chunk = m / a.ntile;
  tile = m - chunk * a.ntile;
  return chunk < a.chunks;
}

// FP32.  A wave owns a 64 x 64 tile over its share of a row range: both
// operands come straight from memory, 16 bytes per lane (lane l: row l / 16 of
// a group of four, features 4 (l % 16) ..), and component v of the vectors is
// the operand of MFMA tile v, whose features are 4 (l % 16) + v.  32 B of
// operands per lane feed 16 MFMAs (512 cycles), so neither LDS nor a second
// read of the rows is needed; the four waves' sums meet in LDS at the end.
// 32-256-256-32, 4096 rows: 67 us for the 4.7 GFLOP of a step's seven stages,
// 70 TFLOP/s, or 84 with the 64-wide tiles' padding of the outer layers (a large
// FP32 product of the library: 129); one GEMM, one fold per stage before.
constexpr int GT = 64;
__global__ void __launch_bounds__(256, 2) k_chain_wgrad32(ChainWgradArgs a) {
  const Ctl* ctl = a.ctl;
  if (a.mode == SM_STEP && ctl->done) return;
  __shared__ float red[4][GT * GT / 2];
  __shared__ float redb[4][2][GT];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int it, ot, tile, chunk;
  if (!wg_block(a, tile, chunk)) return;
  const int l = wg_tile(a, tile, it, ot);
  const int64_t r0 = chunk * a.crows;
  const int64_t r1 = r0 + a.crows < a.ops.rows ? r0 + a.crows : a.ops.rows;
  const int wi = a.ops.w[l], wo = a.ops.w[l + 1];
  const int gsel = ctl->gsel;
  const int rblk = (int)a.rblk, rprim = (int)a.rprim;
  const int ns = a.mode == SM_STEP ? 7 : 1;
  f32x4v g[4][4], ab[4][4], ae[4][4];
  f32x4v gb, bb = {0.f, 0.f, 0.f, 0.f}, be = bb;
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) ab[x][y] = ae[x][y] = bb;
  const bool bias = it == 0;
  const int64_t rr = r0 + 4 * wave + (lane >> 4);
  for (int s = 0; s < ns; ++s) {
    const char* ob = (const char*)a.ops.base + (int64_t)wg_slot(a.mode, s, gsel) * a.ops.slot;
    const float* h = (const float*)(ob + a.ops.h[l]) + rr * wi + it * GT + 4 * (lane & 15);
    const float* d = (const float*)(ob + a.ops.d[l]) + rr * wo + ot * GT + 4 * (lane & 15);
    const f32x4v zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int y = 0; y < 4; ++y) g[x][y] = zero;
    gb = zero;
    const int n = (int)((r1 - r0) / 16);           // groups of 16 rows (4 per wave)
    constexpr int PF = 2;
    f32x4v hv[PF], dv[PF];
    auto load = [&](int j, int k) {
      k = k < n ? k : n - 1;
      hv[j] = *(const f32x4v*)(h + (int64_t)k * 16 * wi);
      dv[j] = *(const f32x4v*)(d + (int64_t)k * 16 * wo);
    };
    auto step = [&](int j, int k, bool refill) {
      const f32x4v x = hv[j], y = dv[j];
      if (refill) load(j, k + PF);
      // bias: primal rows only
      // (a block's rows: a power of two)
      if (bias && (((int)rr + k * 16) & (rblk - 1)) < rprim) gb += y;
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          g[p][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[p], y[q], g[p][q], 0, 0, 0);
    };
#pragma unroll
    for (int j = 0; j < PF; ++j) load(j, j);
    int k = 0;
    for (; k + PF <= n; k += PF)
#pragma unroll
      for (int j = 0; j < PF; ++j) step(j, k + j, true);
#pragma unroll
    for (int j = 0; j < PF - 1; ++j)
      if (k + j < n) step(j, k + j, false);
    const float cb = a.mode == SM_STEP ? (s < 6 ? chA[6][s] : 0.f) : 1.f;
    const float ce = a.mode == SM_STEP ? chBT[s] : 0.f;
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int y = 0; y < 4; ++y) ae[x][y] += ce * g[x][y];
    be += ce * gb;
    if (!wg_quad(a.mode, s)) break;                // (the last stage)
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int y = 0; y < 4; ++y) ab[x][y] += cb * g[x][y];
    bb += cb * gb;
  }
  // sum over the waves, two halves of the tile at a time; acc element (p, q, v)
  // of lane l is input 4 (4 (l / 16) + v) + p, output 4 (l % 16) + q
  const int64_t tsz = GT * (GT + 1);
  float* out = a.part + ((int64_t)chunk * 2 * a.ntile + tile) * tsz;
#pragma unroll
  for (int which = 0; which < 2; ++which) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      __syncthreads();
#pragma unroll
      for (int pp = 0; pp < 2; ++pp) {
        const int p = 2 * half + pp;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int ii = 4 * (lane >> 4) + v;    // input = 4 ii + p
          f32x4v o;
#pragma unroll
          for (int q = 0; q < 4; ++q) o[q] = which ? ae[p][q][v] : ab[p][q][v];
          *(f32x4v*)&red[wave][(pp * 16 + ii) * GT + 4 * (lane & 15)] = o;
        }
      }
      __syncthreads();
      for (int e = threadIdx.x; e < GT * GT / 2; e += 256) {
        const int rw = e / GT, c = e % GT;
        const int i = 4 * (rw & 15) + 2 * half + (rw >> 4);
        out[(int64_t)which * a.ntile * tsz + i * GT + c] =
            (red[0][e] + red[1][e]) + (red[2][e] + red[3][e]);
      }
    }
  }
  if (bias) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float x = bb[q], y = be[q];
      x += __shfl_xor(x, 16); x += __shfl_xor(x, 32);
      y += __shfl_xor(y, 16); y += __shfl_xor(y, 32);
      if (lane < 16) { redb[wave][0][4 * lane + q] = x; redb[wave][1][4 * lane + q] = y; }
    }
    __syncthreads();
    if (threadIdx.x < 2 * GT) {
      const int which = threadIdx.x / GT, c = threadIdx.x % GT;
      out[(int64_t)which * a.ntile * tsz + GT * GT + c] =
          (redb[0][which][c] + redb[1][which][c]) + (redb[2][which][c] + redb[3][which][c]);
    }
  }
}

// FP32, ranges of 16 rows (small batches).  With one group of rows per range
// the kernel above is a chain: a memory latency per stage and a sum over waves
// in four LDS rounds (12.7 us for one trajectory's 2 tiles, 21 us for 333 rows
// of 32-256-256-32; this one 6.5 and 13.9 us).
// Here all stages' operands are requested at once, and a wave takes all 16 rows
// of a quarter of the tile (inputs 4 i + wave), so nothing is summed across
// waves.
__global__ void __launch_bounds__(256, 2) k_chain_wgrad32s(ChainWgradArgs a) {
  const Ctl* ctl = a.ctl;
  if (a.mode == SM_STEP && ctl->done) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int it, ot, tile, chunk;
  if (!wg_block(a, tile, chunk)) return;
  const int l = wg_tile(a, tile, it, ot);
  const int wi = a.ops.w[l], wo = a.ops.w[l + 1];
  const int gsel = ctl->gsel;
  const bool bias = it == 0 && wave == 0;
  const int64_t rr = chunk * 16 + (lane >> 4);
  const int64_t ho = rr * wi + it * GT + 4 * (lane & 15) + wave, dof = rr * wo + ot * GT + 4 * (lane & 15);
  const f32x4v zero = {0.f, 0.f, 0.f, 0.f};
  f32x4v ab[4], ae[4], bb = zero, be = zero;
#pragma unroll
  for (int q = 0; q < 4; ++q) ab[q] = ae[q] = zero;
  // bias: primal rows only (a block's rows: a power of two, the primal first)
  bool keep[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) keep[j] = (((int)rr + 4 * j) & ((int)a.rblk - 1)) < (int)a.rprim;
  float hv[7][4];
  f32x4v dv[7][4];
  auto load = [&](int s) {
    const char* ob = (const char*)a.ops.base + (int64_t)wg_slot(a.mode, s, gsel) * a.ops.slot;
    const float* h = (const float*)(ob + a.ops.h[l]) + ho;
    const float* d = (const float*)(ob + a.ops.d[l]) + dof;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      hv[s][j] = h[4 * j * wi];
      dv[s][j] = *(const f32x4v*)(d + 4 * j * wo);
    }
  };
  auto fold = [&](int s, bool quad, float cb, float ce) {
    f32x4v gb = zero;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      gb += keep[j] ? dv[s][j] : zero;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f32x4v g = zero;
#pragma unroll
      for (int j = 0; j < 4; ++j) g = __builtin_amdgcn_mfma_f32_16x16x4f32(hv[s][j], dv[s][j][q], g, 0, 0, 0);
      if (quad) ab[q] += cb * g;
      ae[q] += ce * g;
    }
    if (quad) bb += cb * gb;
    be += ce * gb;
  };
  load(0);
  if (a.mode == SM_STEP) {
#pragma unroll
    for (int s = 1; s < 7; ++s) load(s);
#pragma unroll
    for (int s = 0; s < 7; ++s) fold(s, s < 6, chA[6][s < 6 ? s : 0], chBT[s]);
  } else {
    fold(0, true, 1.f, 0.f);
  }
  // acc element (q, v) of lane l: input 4 (4 (l / 16) + v) + wave, output 4 (l % 16) + q
  const int64_t tsz = GT * (GT + 1);
  float* out = a.part + ((int64_t)chunk * 2 * a.ntile + tile) * tsz;
#pragma unroll
  for (int which = 0; which < 2; ++which)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      f32x4v o;
#pragma unroll
      for (int q = 0; q < 4; ++q) o[q] = which ? ae[q][v] : ab[q][v];
      *(f32x4v*)(out + (int64_t)which * a.ntile * tsz + (4 * (4 * (lane >> 4) + v) + wave) * GT +
                 4 * (lane & 15)) = o;
    }
  if (bias) {
    f32x4v x, y;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      x[q] = bb[q] + __shfl_xor(bb[q], 16);
      x[q] += __shfl_xor(x[q], 32);
      y[q] = be[q] + __shfl_xor(be[q], 16);
      y[q] += __shfl_xor(y[q], 32);
    }
    if (lane < 16) {
      *(f32x4v*)(out + GT * GT + 4 * lane) = x;
      *(f32x4v*)(out + (int64_t)a.ntile * tsz + GT * GT + 4 * lane) = y;
    }
  }
}

// Split BF16.  K = rows must be contiguous per lane, the operands are
// row-major: a 128 x 128 tile stages 32 rows of both in LDS and reads them
// through the transposing LDS load (a group of 16 lanes reads four rows of 16
// features and gets each lane one feature of the four rows).  Row pitch 320 B:
// the four rows of a read fall on different banks.  Four waves, each 64 x 64
// (two 32 x 32 tiles each way, hi*hi + lo*hi + hi*lo) with both folded sums in
// registers, one wave per SIMD: nothing but the wave's own instructions hides a
// load, so three groups of 32 rows travel from memory at a time (a ring of
// registers; with one group, a read under load took four times the products it
// travelled under: 24% of the matrix rate) and LDS holds three: one written, one
// whose second half is read while its first half multiplies and the other way
// round with the next one (reading all of a group and then multiplying took as
// long again as the products).  Loads are unconditional: rows
// are padded to whole groups with zeros, columns past a layer's width repeat
// the last ones and end in tile entries nobody reads.  17-512-512-16 flow, 8192
// rows: 575 -> 384 us per step attempt, 39% of the matrix pipe (a large split
// product of the library's rate would be 52%), HBM reads 2.4 -> 0.65 GB.  The
// hidden layers' bias gradients are sums of the blocks' FP32 column sums, which
// the row pass leaves: the planes hold ~16 bits of a term (7.6e-6 off where the
// FP32 values are exact).
constexpr int GS = 128, GS_PITCH = 160, GS_K = 32;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* lds_s16x4;
__device__ __forceinline__ u32x4 wg_frag(const bf16* lds, int row, int col) {
  const s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(lds + row * GS_PITCH + col));
  const s16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(lds + (row + 4) * GS_PITCH + col));
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  const s16x8 v = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
  return __builtin_bit_cast(u32x4, v);
}
__global__ void __launch_bounds__(256, 1) k_chain_wgrad16(ChainWgradArgs a) {
  const Ctl* ctl = a.ctl;
  if (a.mode == SM_STEP && ctl->done) return;
  // [buffer][operand][plane][32 rows][pitch]
  __shared__ __attribute__((aligned(16))) bf16 lt[3 * 2 * 2 * GS_K * GS_PITCH];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  int it, ot, tile, chunk;
  if (!wg_block(a, tile, chunk)) return;
  const int l = wg_tile(a, tile, it, ot);
  const int64_t r0 = chunk * a.crows;
  const int64_t r1 = r0 + a.crows < a.ops.rows ? r0 + a.crows : a.ops.rows;
  const int wi = a.ops.w[l], wo = a.ops.w[l + 1];
  const int gsel = ctl->gsel;
  const int ns = a.mode == SM_STEP ? 7 : 1;
  const int n = (int)((r1 - r0) / GS_K);
  const int rblk = (int)a.rblk, rprim = (int)a.rprim;
  const bool bias = it == 0, lastb = bias && l == a.m.L - 1;
  // this thread's 16-byte pieces: 8 features (fc) of rows tr, tr + 16 of both
  // operands and planes
  const int fc = 8 * (tid & 15), tr = tid >> 4;
  const int hc = it * GS + fc < wi ? it * GS + fc : wi - 8, dc = ot * GS + fc < wo ? ot * GS + fc : wo - 8;
  const unsigned hoff = 2 * (tr * wi + hc), doff = 2 * (tr * wo + dc);
  f32x16 g[2][2], ab[2][2], ae[2][2];
  float gb[8], bb[8], be[8];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int v = 0; v < 16; ++v) ab[x][y][v] = ae[x][y][v] = 0.f;
#pragma unroll
  for (int v = 0; v < 8; ++v) bb[v] = be[v] = 0.f;
  // hidden biases: the blocks' sums (blocks that begin in this row range; 16
  // threads share a feature), all stages' loads in flight at once
  if (bias && !lastb) {
    const int hl = a.m.L - 1;
    const int64_t ss = (int64_t)a.nblk * hl * a.bw;
    for (int64_t b = (r0 + rblk - 1) / rblk + tr; b * rblk < r1 && b < a.nblk; b += 16) {
      const float* q = a.bsum + (b * hl + l) * a.bw + ot * GS + fc;
      f32x4v x[7][2];
#pragma unroll
      for (int s = 0; s < 7; ++s)
        if (s < ns)
#pragma unroll
          for (int j = 0; j < 2; ++j) x[s][j] = *(const f32x4v*)(q + wg_slot(a.mode, s, gsel) * ss + 4 * j);
#pragma unroll
      for (int s = 0; s < 7; ++s)
        if (s < ns) {
          const float cb = a.mode == SM_STEP ? (s < 6 ? chA[6][s] : 0.f) : 1.f;
          const float ce = a.mode == SM_STEP ? chBT[s] : 0.f;
#pragma unroll
          for (int v = 0; v < 8; ++v) {
            if (wg_quad(a.mode, s)) bb[v] += cb * x[s][v >> 2][v & 3];
            be[v] += ce * x[s][v >> 2][v & 3];
          }
        }
    }
  }
  const int wr = 64 * (wave >> 1), wc = 64 * (wave & 1);
  const int frow = 8 * (lane >> 5) + ((lane & 15) >> 2);          // first K row of this lane's reads
  const int fcol = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const int64_t hp = a.ops.rows * wi, dp = a.ops.rows * wo;
  constexpr int OPER = 2 * GS_K * GS_PITCH, BUF = 2 * OPER;       // LDS elements of an operand, a group
  for (int s = 0; s < ns; ++s) {
    const char* ob = (const char*)a.ops.base + (int64_t)wg_slot(a.mode, s, gsel) * a.ops.slot;
    const bf16* h = (const bf16*)(ob + a.ops.h[l]) + r0 * wi;       // (uniform; lane offsets apart)
    const bf16* d = (const bf16*)(ob + a.ops.d[l]) + r0 * wo;
    u32x4 hv[3][2][2], dv[3][2][2];                               // [ring][row half][plane]
    auto load = [&](int j, int k) {
      k = k < n ? k : n - 1;
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          hv[j][q][p] = *(const u32x4*)((const char*)(h + p * hp + (int64_t)(k * GS_K + 16 * q) * wi) + hoff);
          dv[j][q][p] = *(const u32x4*)((const char*)(d + p * dp + (int64_t)(k * GS_K + 16 * q) * wo) + doff);
        }
    };
    auto store = [&](int j, int k) {
      bf16* o = lt + j * BUF + tr * GS_PITCH + fc;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          *(u32x4*)(o + (p * GS_K + 16 * q) * GS_PITCH) = hv[j][q][p];
          *(u32x4*)(o + OPER + (p * GS_K + 16 * q) * GS_PITCH) = dv[j][q][p];
        }
        // last layer's bias: lambda, as the products read it (a block's rows: a
        // power of two, the primal ones first)
        if (lastb && k < n && (((int)r0 + k * GS_K + tr + 16 * q) & (rblk - 1)) < rprim) {
          const bf16x8 x = __builtin_bit_cast(bf16x8, dv[j][q][0]), y = __builtin_bit_cast(bf16x8, dv[j][q][1]);
#pragma unroll
          for (int v = 0; v < 8; ++v) gb[v] += (float)x[v] + (float)y[v];
        }
      }
    };
    struct Frags { u32x4 x[2][2], y[2][2]; };                     // [tile][plane] of 16 K rows
    auto read = [&](Frags& f, int j, int kk) {
      const bf16* in = lt + j * BUF;
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          f.x[t][p] = wg_frag(in + p * GS_K * GS_PITCH, 16 * kk + frow, wr + 32 * t + fcol);
          f.y[t][p] = wg_frag(in + OPER + p * GS_K * GS_PITCH, 16 * kk + frow, wc + 32 * t + fcol);
        }
    };
    auto mul = [&](const Frags& f) {
#pragma unroll
      for (int pq = 0; pq < 3; ++pq)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int u = 0; u < 2; ++u)
            g[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                __builtin_bit_cast(bf16x8, f.x[t][pq == 1]), __builtin_bit_cast(bf16x8, f.y[u][pq == 2]),
                g[t][u], 0, 0, 0);
    };
    Frags fa, fb;
    // group k (k % 3 = j; its first half is in fa): group k + 2 to LDS, group
    // k + 5 from memory, each half's products over the other's reads
    auto step = [&](int j, int k) {
      store((j + 2) % 3, k + 2);                                  // (past the last: not used)
      load((j + 2) % 3, k + 5);
      read(fb, j, 1);
      mul(fa);
      read(fa, (j + 1) % 3, 0);
      mul(fb);
      chain_barrier();
    };
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int v = 0; v < 16; ++v) g[x][y][v] = 0.f;
#pragma unroll
    for (int v = 0; v < 8; ++v) gb[v] = 0.f;
#pragma unroll
    for (int j = 0; j < 3; ++j) load(j, j);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      store(j, j);
      load(j, j + 3);
    }
    chain_barrier();
    read(fa, 0, 0);
    int k = 0;
    for (; k + 3 <= n; k += 3)
#pragma unroll
      for (int j = 0; j < 3; ++j) step(j, k + j);
    if (k < n) step(0, k);
    if (k + 1 < n) step(1, k + 1);
    const float cb = a.mode == SM_STEP ? (s < 6 ? chA[6][s] : 0.f) : 1.f;
    const float ce = a.mode == SM_STEP ? chBT[s] : 0.f;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) ae[x][y] += ce * g[x][y];
#pragma unroll
    for (int v = 0; v < 8; ++v) be[v] += ce * gb[v];
    if (!wg_quad(a.mode, s)) break;                // (the last stage)
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) ab[x][y] += cb * g[x][y];
#pragma unroll
    for (int v = 0; v < 8; ++v) bb[v] += cb * gb[v];
  }
  const int64_t tsz = GS * (GS + 1);
  float* out = a.part + ((int64_t)chunk * 2 * a.ntile + tile) * tsz;
#pragma unroll
  for (int which = 0; which < 2; ++which)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int i = wr + 32 * t + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
          out[(int64_t)which * a.ntile * tsz + i * GS + wc + 32 * u + (lane & 31)] =
              which ? ae[t][u][v] : ab[t][u][v];
        }
  if (bias) {
    float* red = (float*)lt;                                      // [2][16][GS]
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      red[tr * GS + fc + v] = bb[v];
      red[16 * GS + tr * GS + fc + v] = be[v];
    }
    __syncthreads();
    const int which = tid / GS, c = tid % GS;
    float x = 0.f;
    for (int r = 0; r < 16; ++r) x += red[which * 16 * GS + r * GS + c];
    out[(int64_t)which * a.ntile * tsz + GS * GS + c] = x;
  }
}

// ---------------------------------------------------------------- parameter state
// Adds the row ranges' partial sums in range order, forms the speculative mu in
// the other buffer and its error norm (modes: step, initial-dt norms).  The
// parameter equation is mu' = -lambda^T df/dp.
// Bound by latency (FP64 state, 2 x ranges floats per parameter in batches of
// eight independent loads): 4.5 us for 252 parameters and one range, 8 us for
// 99k parameters and 21 ranges, which is why small batches get at most 32
// ranges; four loads at a time took 10 us.
__global__ void __launch_bounds__(256) k_chain_mu(ChainMuArgs a) {
  const ChainWgradArgs& w = a.w;
  const Ctl* c = w.ctl;
  if (w.mode == SM_STEP && c->done) return;
  const double atol = c->abstol, rtol = c->reltol, dt = c->dt;
  const int ms = c->gsel_mu_;
  const double* mu = ms ? a.mu + a.P : a.mu;
  double* mo = ms ? a.mu : a.mu + a.P;
  const int E = a.edge;
  const int64_t tsz = (int64_t)E * (E + 1), half = (int64_t)w.ntile * tsz;
  double sum = 0.0, flag = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < a.P;
       i += (int64_t)gridDim.x * blockDim.x) {
    int l = 0;
    while (l + 1 < w.m.L && i >= a.w0[l + 1]) ++l;
    const int out = w.m.out[l];
    int64_t src;
    const bool f32 = E == 64;                      // (FP32 operand rows: chain_feat order)
    if (i < a.b0[l]) {
      const int q = (int)(i - a.w0[l]), qi = q / out, qo = q % out;
      const int in = f32 ? chain_posn(qi) : qi, o = f32 ? chain_posn(qo) : qo;
      src = (int64_t)(w.tl[l] + in / E * w.tw[l] + o / E) * tsz + (in % E) * E + o % E;
    } else {
      const int qo = (int)(i - a.b0[l]), o = f32 ? chain_posn(qo) : qo;
      src = (int64_t)(w.tl[l] + o / E) * tsz + (int64_t)E * E + o % E;
    }
    // (eight ranges' loads in flight: a chain of 20 otherwise)
    float b = 0.f, e = 0.f;
    const bool st = w.mode == SM_STEP;
    const float* p = w.part + src;
    int k = 0;
    for (; k + 8 <= w.chunks; k += 8, p += 16 * half) {
      float x[8], y[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        x[j] = p[2 * j * half];
        y[j] = st ? p[(2 * j + 1) * half] : 0.f;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) { b -= x[j]; e -= y[j]; }
    }
    for (; k < w.chunks; ++k, p += 2 * half) {
      b -= p[0];
      if (st) e -= p[half];
    }
    const double m = mu[i];
    double v;
    if (w.mode == SM_STEP) {
      const double mn = m + dt * (double)b;
      mo[i] = mn;
      v = dt * (double)e / (atol + fmax(fabs(m), fabs(mn)) * rtol);
    } else if (w.mode == SM_INIT_F0) {
      a.g0[i] = b;
      v = (double)b / (atol + fabs(m) * rtol);
    } else {
      v = ((double)b - (double)a.g0[i]) / (atol + fabs(m) * rtol);
      if (b != a.g0[i]) flag = 1.0;
    }
    sum += v * v;
  }
  block_reduce_store(sum, flag, a.part, blockIdx.x);
}

void launch_chain_wgrad(int prec, const ChainWgradArgs& a, hipStream_t s) {
  const dim3 grid(8 * ((a.ntile * a.chunks + 7) / 8));
  if (prec == 0 && a.crows == 16) hipLaunchKernelGGL(k_chain_wgrad32s, grid, dim3(256), 0, s, a);
  else if (prec == 0) hipLaunchKernelGGL(k_chain_wgrad32, grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL(k_chain_wgrad16, grid, dim3(256), 0, s, a);
}
void launch_chain_mu(const ChainMuArgs& a, int nblk, hipStream_t s) {
  hipLaunchKernelGGL(k_chain_mu, dim3(nblk), dim3(256), 0, s, a);
}

}  // namespace nodehip
