// Device helpers shared by the kernels' translation units: vector types,
// dense-output constants, activations, precision policies and the block
// reduction of the error partial sums.
#pragma once
#include <type_traits>

#include "node_internal.h"

namespace nodehip {

typedef __bf16 bf16;
typedef bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4v __attribute__((ext_vector_type(4)));
// native 16-byte vector (HIP's uint4 is a struct wrapper that blocks SROA of
// the register-staged tiles)
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

static __device__ const double dC[7] = {0.0, 0.161, 0.327, 0.9, 0.9800255409045097, 1.0, 1.0};
// free 4th-order dense output: b1(t) = t(r11 + t(r12 + t(r13 + t r14))),
// bi(t) = t^2 (ri2 + t(ri3 + t ri4))
static __device__ const double dR1[4] = {1.0, -2.763706197274826, 2.9132554618219126,
                                  -1.0530884977290216};
static __device__ const double dRI[6][3] = {
    {0.13169999999999998, -0.2234, 0.1017},
    {3.9302962368947516, -5.941033872131505, 2.490627285651253},
    {-12.411077166933676, 30.33818863028232, -16.548102889244902},
    {37.50931341651104, -88.1789048947664, 47.37952196281928},
    {-27.896526289197286, 65.09189467479366, -34.8706578614966},
    {1.5, -4.0, 2.5}};

// dense-output weights at theta of a step: state = u + dt sum_i w[i] k_{i+1}
__device__ __forceinline__ void interp_weights(double th, float* w) {
  const double th2 = th * th;
  w[0] = (float)(th * (dR1[0] + th * (dR1[1] + th * (dR1[2] + th * dR1[3]))));
#pragma unroll
  for (int i = 0; i < 6; ++i) w[i + 1] = (float)(th2 * (dRI[i][0] + th * (dRI[i][1] + th * dRI[i][2])));
}

// ---------------------------------------------------------------- helpers
__device__ __forceinline__ bool gate_ok(const Ctl* c, int gate) {
  if (gate == GATE_ALWAYS) return true;
  if (c->done) return false;
  if (gate == GATE_FSAL) return c->fsal_reeval != 0;
  return true;
}

// Tape entry of forward step n: the entries form a ring of c->tape_ring slots
// when that is set (a forward solve that keeps only checkpoints: the stage
// kernels touch entries n and n + 1, the pending saves n - 1 and n), else the
// record of every step.
__device__ __forceinline__ int64_t tape_slot(const Ctl* c, int64_t n) {
  const int64_t r = c->tape_ring;
  return r > 0 ? n % r : n;
}

// Activations from the hardware exp2 / log2 / reciprocal (v_exp_f32,
// v_log_f32, v_rcp_f32, ~1 ulp each): the epilogues run them once per output
// element at low occupancy, where the full-range library forms dominated the
// kernel time.  Absolute error stays at the FP32 rounding level of the result.
#define LOG2E_F 1.4426950408889634f
#define LN2_F 0.6931471805599453f
__device__ __forceinline__ float fast_sigmoid(float z) {
  return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-z * LOG2E_F));
}
__device__ __forceinline__ float act_f(int a, float z) {
  switch (a) {
    case 1: {  // tanh(z) = sign(z) (1 - t) / (1 + t), t = exp(-2|z|)
      const float t = __builtin_amdgcn_exp2f(-2.f * LOG2E_F * fabsf(z));
      return copysignf((1.f - t) * __builtin_amdgcn_rcpf(1.f + t), z);
    }
    case 2:  // softplus: log1p(exp(-|z|)) + max(z, 0)
      return fmaxf(z, 0.f) +
             LN2_F * __builtin_amdgcn_logf(1.f + __builtin_amdgcn_exp2f(-fabsf(z) * LOG2E_F));
    case 3: return fmaxf(z, 0.f);
    case 4: return fast_sigmoid(z);
    default: return z;
  }
}
__device__ __forceinline__ float act_d(int a, float z, float y) {
  switch (a) {
    case 1: return 1.f - y * y;
    case 2: return fast_sigmoid(z);
    case 3: return z > 0.f ? 1.f : 0.f;
    case 4: return y * (1.f - y);
    default: return 1.f;
  }
}
// act' from the activation's output y (identity, softplus, relu):
// softplus'(z) = sigmoid(z) = 1 - exp(-y) with y = softplus(z) > 0; below
// y = 1/4 its Taylor series to y^6 (relative truncation < 5e-8, no
// cancellation), above it the hardware exp2 (relative error < 1e-6)
__device__ __forceinline__ float act_d_y(int a, float y) {
  switch (a) {
    case 2: {
      if (y < 0.25f) {
        float t = 1.f - y * (1.f / 6.f);
        t = 1.f - y * (1.f / 5.f) * t;
        t = 1.f - y * 0.25f * t;
        t = 1.f - y * (1.f / 3.f) * t;
        t = 1.f - y * 0.5f * t;
        return y * t;
      }
      return 1.f - __builtin_amdgcn_exp2f(-y * LOG2E_F);
    }
    case 3: return y > 0.f ? 1.f : 0.f;
    default: return 1.f;
  }
}

// activations whose derivative the epilogues derive from the output
__device__ __forceinline__ bool act_from_output_d(int a) { return a == 0 || a == 2 || a == 3; }
__device__ __forceinline__ float map_f(int m, float u) { return m == 1 ? u * u * u : u; }

template <typename T> __device__ __forceinline__ T cvt(float x);
template <> __device__ __forceinline__ float cvt<float>(float x) { return x; }
template <> __device__ __forceinline__ bf16 cvt<bf16>(float x) { return (bf16)x; }
template <typename T> __device__ __forceinline__ float tof(T x);
template <> __device__ __forceinline__ float tof<float>(float x) { return x; }
template <> __device__ __forceinline__ float tof<bf16>(bf16 x) { return (float)x; }

// store 4 consecutive values (8 B for bf16, 16 B for fp32; caller guarantees alignment)
__device__ __forceinline__ void store4(float* p, const float v[4]) {
  *(float4*)p = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void store4(bf16* p, const float v[4]) {
  typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
  bf16x4 o = {(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]};
  *(bf16x4*)p = o;
}

// precision policy: operand type, split (hi/lo planes), act' storage type
template <typename T_, bool SPLIT_>
struct Prec {
  using T = T_;
  static constexpr bool SPLIT = SPLIT_;
  using ST = typename std::conditional<SPLIT_, float, T_>::type;
};
using PF32 = Prec<float, false>;
using PBF16 = Prec<bf16, false>;
using PBF16X3 = Prec<bf16, true>;

template <class PP>
__device__ __forceinline__ void put(typename PP::T* p, int64_t plane, float v) {
  if constexpr (PP::SPLIT) {
    const bf16 h = (bf16)v;
    p[0] = h;
    p[plane] = (bf16)(v - (float)h);
  } else {
    p[0] = cvt<typename PP::T>(v);
  }
}
template <class PP>
__device__ __forceinline__ float get(const typename PP::T* p, int64_t plane) {
  if constexpr (PP::SPLIT) return (float)p[0] + (float)p[plane];
  else return tof<typename PP::T>(p[0]);
}
template <class PP>
__device__ __forceinline__ void put4(typename PP::T* p, int64_t plane, const float v[4]) {
  if constexpr (PP::SPLIT) {
    float hi[4], lo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      hi[i] = (float)(bf16)v[i];
      lo[i] = v[i] - hi[i];
    }
    store4(p, hi);
    store4(p + plane, lo);
  } else {
    store4(p, v);
  }
}

#define DISPATCH_PREC(prec, ...)                   \
  do {                                             \
    if ((prec) == 1) { using PP = PBF16; __VA_ARGS__; }   \
    else if ((prec) == 2) { using PP = PBF16X3; __VA_ARGS__; } \
    else { using PP = PF32; __VA_ARGS__; }          \
  } while (0)

// Block-wide reduction of (sum, max-flag); thread 0 writes part[2*slot..].
__device__ __forceinline__ void block_reduce_store(double s, double f, double* part, int slot) {
  __shared__ double red[2][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nw = (blockDim.x + 63) >> 6;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    s += __shfl_xor(s, off);
    f = fmax(f, __shfl_xor(f, off));
  }
  if (lane == 0) { red[0][wave] = s; red[1][wave] = f; }
  __syncthreads();
  if (threadIdx.x == 0) {
    double ss = 0.0, ff = 0.0;
    for (int w = 0; w < nw; ++w) { ss += red[0][w]; ff = fmax(ff, red[1][w]); }
    part[2 * slot] = ss;
    part[2 * slot + 1] = ff;
  }
}

__device__ __forceinline__ double dspacing(double t) {
  double a = fabs(t);
  return nextafter(a, INFINITY) - a;
}

}  // namespace nodehip
