// Fused step kernels: interface between the host driver and chain_*.hip.
#pragma once
#include "node_internal.h"

namespace nodehip {

// ---- fused step kernels: the whole Dense chain of a block of rows per workgroup
// weights in MFMA fragment order: Wf (forward, M = outputs, K = inputs) and Wb
// (backward, M = inputs, K = outputs); mt 16-feature tiles, kt K tiles
struct ChainModel {
  int L, map, D, dm, tcat, B;
  int in[MAXL], out[MAXL], act[MAXL];
  int mtf[MAXL], ktf[MAXL], mtb[MAXL], ktb[MAXL];
  const void* Wf[MAXL]; const void* Wb[MAXL];
  const float* bias[MAXL];
  int pitch;                   // LDS row pitch (elements)
  int nw;                      // waves per workgroup (4 or 8)
  int cw, tf;                  // rows and features of an MFMA tile (16 x 16, or 4 x 64)
  int kt;                      // features per K tile
  // LDS byte offsets after the activation buffers: partial products of the
  // narrow layers (0: over the activations), hidden biases (rows of wmax), probe
  int lds_part, lds_bias, lds_probe, lds_bytes, wmax;
};
struct ChainPack {
  int nl;
  int in[MAXL], out[MAXL], mtf[MAXL], ktf[MAXL], mtb[MAXL], ktb[MAXL];
  int64_t w0[MAXL];
  void* Wf[MAXL]; void* Wb[MAXL];
  int tf;
};
void launch_pack_chain(int prec, const ChainPack& a, const float* p, hipStream_t s);
struct ChainFwdArgs {
  ChainModel m;
  float* tape; int64_t ent, sv;
  const float* probe;          // flow: [B][dm]
  const double* save_times; float* out;
  double* part;
  const Ctl* ctl;
  int mode;
};
// Operands of the weight gradients, kept per stage by the fused adjoint step:
// for layer l its inputs h ([row][inp]) and output gradients d ([row][outp]),
// T x planes (plane stride rows * width), rows = blocks * cw nt (a flow's block
// holds its primal rows first, then its tangent rows); widths padded to 64.
// Slot of stage s: 1..5 -> s + 1; stages 0 and 6 share slots 0 and 1 (the last
// stage of an accepted step is the next one's first: FSAL).
struct ChainOps {
  void* base;
  int64_t slot;                // bytes per stage slot
  int64_t h[MAXL], d[MAXL];    // byte offsets in a slot
  int w[MAXL + 1];             // inp of layer l; w[L] = outp of the last
  int64_t rows;
};
struct ChainAdjArgs {
  ChainModel m;
  ChainOps ops;
  const float* tape; int64_t ent, sv;
  float* lam; float* lam_new; float* kl;   // kl: slots 0 and 6 of 8 stage slots are used
  const float* dLdout;
  const float* probe;
  // act' (and act'' adot, flow) of the hidden layers: per block and layer
  // `stiles` feature tiles, each [primal column tile][lane][4]
  float* slope; float* curve;
  int stiles;
  // split BF16: sums of the hidden layers' output gradients over a block's
  // primal rows, [slot][block][hidden layer][bw] (the bias gradients come from
  // the FP32 values; the operand rows keep ~16 bits of them)
  float* bsum; int bw;
  // BacksolveAdjoint: u integrated with lambda (ubs != nullptr)
  float* ubs; float* ubs_new; float* ku; const float* fsaved; int ckpt;
  double* part;
  const Ctl* ctl;
  int mode;
};
struct ChainWgradArgs {
  ChainModel m;
  ChainOps ops;
  int64_t rblk;                // rows of a block
  int64_t rprim;               // of which primal (bias gradients sum these only)
  int ntile;                   // 64 x 64 (FP32) or 128 x 128 (split) tiles of all layers
  int tl[MAXL], tw[MAXL];      // first tile of a layer, its tiles along the outputs
  int chunks; int64_t crows;   // row ranges and rows per range
  const float* bsum; int bw, nblk;  // (split) bias sums per block, as in ChainAdjArgs
  float* part;                 // [chunk][2][ntile][65 x 64 or 129 x 128]
  const Ctl* ctl;
  int mode;
};
struct ChainMuArgs {
  ChainWgradArgs w;
  int64_t w0[MAXL], b0[MAXL], P;
  int edge;                    // tile edge (64 / 128)
  double* mu; float* g0;       // two mu buffers; gradient at the initial time
  double* part;
};
void launch_chain_adj(int prec, int nt, bool cnf, const ChainAdjArgs& a, int grid, hipStream_t s);
void launch_chain_wgrad(int prec, const ChainWgradArgs& a, hipStream_t s);
void launch_chain_mu(const ChainMuArgs& a, int nblk, hipStream_t s);

// Dynamic LDS of a step kernel at most (its static LDS comes on top).  Also what
// the launches set as the kernels' limit, whatever they need themselves: the
// limit belongs to the process, and handles of other sizes set it from other
// threads.
constexpr int CHAIN_LDS_MAX = 159 * 1024;

// nt: column tiles (of cw) per block (rows per block: cw nt, a flow half)
int chain_rows(const ChainModel& m, int nt, bool cnf);
// LDS layout of a model's step kernels (fills the lds_ fields)
void chain_layout(ChainModel& m, int nt, bool cnf);
void launch_chain_fwd(int prec, int nt, bool cnf, const ChainFwdArgs& a, int grid, hipStream_t s);

}  // namespace nodehip
