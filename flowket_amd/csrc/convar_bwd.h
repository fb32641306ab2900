// What the gradient kernels share: arguments, parameter offsets, the layout of
// a sample's workspace, activations and their derivatives.
#pragma once
#include "fk_common.h"
#include "convar_layout.h"

namespace fk {

template <int ACT>
__device__ __forceinline__ float bact(float x) {
  if constexpr (ACT == FK_ACT_RELU) return fmaxf(x, 0.0f);
  else return x > 0.0f ? x : expm1f(x);
}
template <int ACT>
__device__ __forceinline__ float bdact(float y) {  // derivative from the output
  if constexpr (ACT == FK_ACT_RELU) return y > 0.0f ? 1.0f : 0.0f;
  else return y > 0.0f ? 1.0f : y + 1.0f;
}

struct BwdArgs {
  const float* params;  // flat parameters (effective kernels), P floats
  int H, W, HW, C, nb;
  int64_t batch;
  const int8_t* spins;  // (batch, HW)
  float* work;          // per-workgroup activation store
  int64_t work_floats;  // floats per workgroup
  float* o_re;          // (batch, P)
  float* o_im;
  float* logpsi;        // (batch, 2) or null
  int64_t P;
  int64_t ld;           // row stride of o_re / o_im (>= P)
  const float* cot;     // GRAD_VJP: (batch, 2) cotangents of (Re, Im) log psi
  float* partial;       // GRAD_VJP: partial gradients, rows of P floats
  int64_t run;          // convar_grad.hip: samples of a workgroup that share a partial row
  const float* tangent; // JVP: direction, P floats
  float* jvp;           // JVP: (batch, 2) output
  const float* kt;      // the conv kernels transposed (transpose_kernels_kernel), P floats
  const float* tkt;     // JVP: the tangent's conv kernels transposed
  const float* kb;      // convar_grad.hip: the conv kernels packed for the data gradients (kt, tkt: packed too)
  int stage;            // LDS row stride (floats) of the two staging tiles, 0: no staging
};

// Offsets of layer parameters in the flat vector.
struct ParamOffsets {
  int64_t kv, bv, kh, bh, kx, bx, ky, by, kc, bc;
};
__device__ __forceinline__ ParamOffsets param_offsets(int blk, int C) {
  // block 0 has cin = 1; blocks >= 1 have cin = C
  const int64_t blk0 = 9LL * C + C + 3LL * C + C + (int64_t)C * (C / 2) * 2 + C + 9LL * C * C + C;
  const int64_t blkn = 9LL * C * C + C + 3LL * C * C + C + (int64_t)C * (C / 2) * 2 + C + 9LL * C * C + C;
  const int64_t base = blk == 0 ? 0 : blk0 + (int64_t)(blk - 1) * blkn;
  const int cin = blk == 0 ? 1 : C;
  ParamOffsets o;
  o.kv = base;
  o.bv = o.kv + 9LL * cin * C;
  o.kh = o.bv + C;
  o.bh = o.kh + 3LL * cin * C;
  o.kx = o.bh + C;
  o.bx = o.kx + (int64_t)C * (C / 2);
  o.ky = o.bx + C / 2;
  o.by = o.ky + (int64_t)C * (C / 2);
  o.kc = o.by + C / 2;
  o.bc = o.kc + 9LL * C * C;
  return o;
}
__device__ __forceinline__ int64_t head_offset(int nb, int C) {
  const ParamOffsets o = param_offsets(nb - 1, C);
  return o.bc + C;
}

// Tap offsets: vertical kxk rows -2..0 cols -1..1; horizontal 1xk cols -2..0;
// h3 kxk rows -2..0 cols -2..0.
__device__ __forceinline__ void tap_rc(int kind, int t, int& dr, int& dc) {
  if (kind == 0) {
    dr = t / 3 - 2;
    dc = t % 3 - 1;
  } else if (kind == 1) {
    dr = 0;
    dc = t - 2;
  } else {
    dr = t / 3 - 2;
    dc = t % 3 - 2;
  }
}

// Per-sample workspace layout (floats): spins HW, then per block
// VA (act(v')), XA (act(hx)), CAT (x2|y2), VO (vertical output), HO
// (horizontal output), each HW*C.
// (the spins region is padded to 4 floats so that every tensor is 16-byte
// aligned)
__device__ __forceinline__ float* ws_tensor(float* ws, int HW, int C, int blk, int which) {
  return ws + ((HW + 3) & ~3) + ((int64_t)blk * 5 + which) * HW * C;
}
enum { T_VA = 0, T_XA = 1, T_CAT = 2, T_VO = 3, T_HO = 4 };

// source-table rows: vertical taps 0-8, horizontal 9-11, h3 12-20, x1x1 21,
// x1x1 behind the RightShift (final block) 22, y1x1 behind the DownShift 23
constexpr int GT_V = 0, GT_H = 9, GT_C = 12, GT_X = 21, GT_XF = 22, GT_Y = 23, GT_N = 24;

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Elementwise passes over HW x C tensors (C a multiple of 4) in 16-byte
// vectors: element i of a tensor as a quad, the activation and its
// derivative per component.
__device__ __forceinline__ f32x4 L4(const float* p, int i) { return *reinterpret_cast<const f32x4*>(p + 4 * i); }
__device__ __forceinline__ f32x4& S4(float* p, int i) { return *reinterpret_cast<f32x4*>(p + 4 * i); }
template <int ACT>
__device__ __forceinline__ f32x4 bact4(f32x4 x) {
  return f32x4{bact<ACT>(x[0]), bact<ACT>(x[1]), bact<ACT>(x[2]), bact<ACT>(x[3])};
}
template <int ACT>
__device__ __forceinline__ f32x4 bdact4(f32x4 y) {
  return f32x4{bdact<ACT>(y[0]), bdact<ACT>(y[1]), bdact<ACT>(y[2]), bdact<ACT>(y[3])};
}

// Per-sample workspace of the MFMA kernel: the scalar kernel's layout plus six
// gradient tensors (dV, dH, dVr, dHr, t0, t1) of HW*C floats.
__device__ __forceinline__ float* ws_grad(float* ws, int HW, int C, int nb, int which) {
  return ws + ((HW + 3) & ~3) + ((int64_t)nb * 5 + which) * HW * C;
}

// Head logits z[k] (k = 0, 1: Re for spin +1 / -1; 2, 3: Im) of pixel p.
__device__ __forceinline__ void head_logits(const float* prm, int64_t ho, const float* HF, int C, int p, float z[4]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float acc = prm[ho + 4 * C + k];
#pragma unroll 8
    for (int ci = 0; ci < C; ++ci) acc += prm[ho + ci * 4 + k] * HF[p * C + ci];
    z[k] = acc;
  }
}

enum { GRAD_O = 0, GRAD_VJP = 1, GRAD_JVP = 2 };

// The kernel of convar_grad.hip (32 and 64 channels): how a launch runs, or
// threads = 0 where it does not take the shape or the operands (16-byte
// accesses), and the launch.
struct GradPlan {
  int threads, per_cu;
  bool resident;
  int64_t grid;
  size_t lds;
};
GradPlan grad_plan(const BwdArgs& a, int mode);
int launch_grad_plan(const GradPlan& p, const BwdArgs& a, int act, int mode, hipStream_t s);

}  // namespace fk
