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
};
struct ChainPack {
  int nl;
  int in[MAXL], out[MAXL], mtf[MAXL], ktf[MAXL], mtb[MAXL], ktb[MAXL];
  int64_t w0[MAXL];
  void* Wf[MAXL]; void* Wb[MAXL];
};
void launch_pack_chain(int prec, const ChainPack& a, const float* p, hipStream_t s);
struct ChainFwdArgs {
  ChainModel m;
  float* tape; int64_t ent, sv;
  const float* probe;          // flow: [B][dm]
  const double* save_times; float* out;
  float* plain;                // SM_PLAIN: input state in tape[0..], output here
  double* part;
  const Ctl* ctl;
  int mode;
};
// nt: 16-column MFMA tiles per block (rows per block: 16 nt, a flow 8 nt)
int chain_rows(int nt, bool cnf);
size_t chain_fwd_lds(int prec, const ChainModel& m, int nt);
void launch_chain_fwd(int prec, int nt, bool cnf, const ChainFwdArgs& a, int grid, hipStream_t s);

}  // namespace nodehip
