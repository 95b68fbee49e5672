// Parameter packing: the flat Lux vector (per Dense layer W[o, i] at
// i * out + o, then the bias) to the operand layouts of the kernels.
#include "device_util.h"

namespace nodehip {

constexpr int PK = 32;         // tile edge
constexpr int PK_THREADS = 256;

// One 32 x 32 tile of one layer's weights (blockIdx.y) per workgroup, to
// Wr [outp][inp] and Wc [inp][outp], and the layer's bias by its first
// workgroup.  Bound by the launch for small models and by memory for wide ones
// (2.2M weights: 9 MB in, 18 MB of split-BF16 planes out): reads and both
// writes run along rows, the transposition goes through LDS (pitch 33: no
// bank conflicts).  The same layouts formed by host loops, with the parameters
// copied to the host and back, took 20 ms per call at 64-1024-1024-1024-64.
// Padded entries stay zero: they are never written.
template <class PP>
__global__ void __launch_bounds__(PK_THREADS) k_pack_params(PackArgs a, const float* __restrict__ p) {
  using T = typename PP::T;
  const int l = blockIdx.y;
  const int in = a.in[l], out = a.out[l], inp = a.inp[l], outp = a.outp[l];
  if (blockIdx.x == 0)
    for (int o = threadIdx.x; o < out; o += PK_THREADS) a.bias[l][o] = p[a.b0[l] + o];
  __shared__ float lt[PK][PK + 1];
  const int to = (out + PK - 1) / PK, ti = (in + PK - 1) / PK;
  const int64_t plane = (int64_t)inp * outp;
  T* Wr = (T*)a.Wr[l];
  T* Wc = (T*)a.Wc[l];
  const float* w = p + a.w0[l];
  const int x = threadIdx.x % PK, y = threadIdx.x / PK;
  for (int tile = blockIdx.x; tile < to * ti; tile += gridDim.x) {
    const int o0 = tile % to * PK, i0 = tile / to * PK;
    for (int j = y; j < PK; j += PK_THREADS / PK) {
      const int i = i0 + j, o = o0 + x;
      if (i < in && o < out) {
        const float v = w[(int64_t)i * out + o];
        lt[j][x] = v;
        put<PP>(Wc + (int64_t)i * outp + o, plane, v);
      }
    }
    __syncthreads();
    for (int j = y; j < PK; j += PK_THREADS / PK) {
      const int o = o0 + j, i = i0 + x;
      if (i < in && o < out) put<PP>(Wr + (int64_t)o * inp + i, plane, lt[x][j]);
    }
    __syncthreads();
  }
}

void launch_pack_params(int prec, const PackArgs& a, const float* p, hipStream_t s) {
  int tiles = 1;
  for (int l = 0; l < a.nl; ++l) {
    const int t = ((a.in[l] + PK - 1) / PK) * ((a.out[l] + PK - 1) / PK);
    tiles = t > tiles ? t : tiles;
  }
  tiles = tiles < 1024 ? tiles : 1024;
  DISPATCH_PREC(prec, hipLaunchKernelGGL(k_pack_params<PP>, dim3(tiles, a.nl), dim3(PK_THREADS), 0,
                                         s, a, p));
}

}  // namespace nodehip
