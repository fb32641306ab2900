// What the two fast-sampler kernels share (fast_sampler.hip: one wave per 16
// samples; fast_sampler_mw.hip: a workgroup per 16 samples).
#pragma once
#include "fk_common.h"
#include "convar_layout.h"
#include "convar_dev.h"

namespace fk {

// Per-lane data of one pixel of a C-channel tensor for 16 samples: MT quads
// of 4 channels (channels 16*mt + 4*g + r for lane group g) in M-tile order.
template <int PREC, int C>
struct LaneData;

// 16-bit precisions (bf16, fp16): 8 bytes per quad
template <int PREC, int C>
struct LaneData {
  static constexpr int MT = C / 16;
  static constexpr int LB = MT * 8;  // bytes per lane
  uint2 q[MT];
  __device__ __forceinline__ void load(const uint8_t* p) {
#pragma unroll
    for (int k = 0; k < MT / 2; ++k) {
      const uint4 v = *reinterpret_cast<const uint4*>(p + 16 * k);
      q[2 * k] = make_uint2(v.x, v.y);
      q[2 * k + 1] = make_uint2(v.z, v.w);
    }
  }
  __device__ __forceinline__ void load_quads(const uint8_t* p, int m0, int m1) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (m >= m0 && m < m1) q[m] = *reinterpret_cast<const uint2*>(p + 8 * m);
  }
  // the same loads through a buffer resource: per-lane offset voff, uniform
  // offset soff (bytes)
  __device__ __forceinline__ void bload(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff) {
#pragma unroll
    for (int k = 0; k < MT / 2; ++k) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, voff + 16 * k, soff, 0);
      q[2 * k] = make_uint2(v.x, v.y);
      q[2 * k + 1] = make_uint2(v.z, v.w);
    }
  }
  __device__ __forceinline__ void bload_quads(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff, int m0, int m1) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (m >= m0 && m < m1) {
        const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, voff + 8 * m, soff, 0);
        q[m] = make_uint2(v.x, v.y);
      }
  }
  __device__ __forceinline__ void store_quads(uint8_t* p, int m0, int m1) const {
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (m >= m0 && m < m1) *reinterpret_cast<uint2*>(p + 8 * m) = q[m];
  }
  __device__ __forceinline__ void store(uint8_t* p) const {
#pragma unroll
    for (int k = 0; k < MT / 2; ++k)
      *reinterpret_cast<uint4*>(p + 16 * k) = make_uint4(q[2 * k].x, q[2 * k].y, q[2 * k + 1].x, q[2 * k + 1].y);
  }
  __device__ __forceinline__ void bstore_quads(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff, int m0,
                                               int m1) const {
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (m >= m0 && m < m1) __builtin_amdgcn_raw_buffer_store_b64(u32x2{q[m].x, q[m].y}, r, voff + 8 * m, soff, 0);
  }
  __device__ __forceinline__ void bstore(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff) const {
#pragma unroll
    for (int k = 0; k < MT / 2; ++k)
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{q[2 * k].x, q[2 * k].y, q[2 * k + 1].x, q[2 * k + 1].y}, r,
                                             voff + 16 * k, soff, 0);
  }
  __device__ __forceinline__ void set(int m, f32x4 v) {
    typename Prec<PREC>::quad h = to_quad<PREC>(v);
    q[m] = *reinterpret_cast<uint2*>(&h);
  }
  __device__ __forceinline__ f32x4 get(int m) const {
    return from_quad<PREC>(*reinterpret_cast<const typename Prec<PREC>::quad*>(&q[m]));
  }
  template <int KS>
  __device__ __forceinline__ void frags(typename Prec<PREC>::frag (&b)[KS]) const {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint4 v = make_uint4(q[2 * ks].x, q[2 * ks].y, q[2 * ks + 1].x, q[2 * ks + 1].y);
      b[ks] = *reinterpret_cast<typename Prec<PREC>::frag*>(&v);
    }
  }
};

template <int C>
struct LaneData<FK_PREC_FP32, C> {
  static constexpr int MT = C / 16;
  static constexpr int LB = MT * 16;
  f32x4 q[MT];
  __device__ __forceinline__ void load(const uint8_t* p) {
#pragma unroll
    for (int m = 0; m < MT; ++m) q[m] = *reinterpret_cast<const f32x4*>(p + 16 * m);
  }
  __device__ __forceinline__ void load_quads(const uint8_t* p, int m0, int m1) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (m >= m0 && m < m1) q[m] = *reinterpret_cast<const f32x4*>(p + 16 * m);
  }
  __device__ __forceinline__ void store_quads(uint8_t* p, int m0, int m1) const {
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (m >= m0 && m < m1) *reinterpret_cast<f32x4*>(p + 16 * m) = q[m];
  }
  __device__ __forceinline__ void store(uint8_t* p) const { store_quads(p, 0, MT); }
  __device__ __forceinline__ void bload_quads(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff, int m0, int m1) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (m >= m0 && m < m1)
        q[m] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff + 16 * m, soff, 0));
  }
  __device__ __forceinline__ void bload(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff) {
    bload_quads(r, voff, soff, 0, MT);
  }
  __device__ __forceinline__ void bstore_quads(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff, int m0,
                                               int m1) const {
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (m >= m0 && m < m1)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, q[m]), r, voff + 16 * m, soff, 0);
  }
  __device__ __forceinline__ void bstore(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff) const {
    bstore_quads(r, voff, soff, 0, MT);
  }
  __device__ __forceinline__ void set(int m, f32x4 v) { q[m] = v; }
  __device__ __forceinline__ f32x4 get(int m) const { return q[m]; }
  template <int KS>
  __device__ __forceinline__ void frags(float (&b)[KS]) const {
#pragma unroll
    for (int t = 0; t < KS; ++t) b[t] = q[t >> 2][t & 3];
  }
};

struct SampArgs {
  const void* w;
  const float* aux;
  int H, W, HW, nb;
  int64_t batch;
  const double* uniforms;
  int8_t* out;
  float* cond;
  uint8_t* cache;
  int64_t tile_bytes;
};

template <int PREC, int C>
constexpr int fast_lb() {
  return PREC == FK_PREC_FP32 ? (C / 16) * 16 : (C / 16) * 8;
}

// Four consecutive biases of one lane group (16-byte aligned: every bias
// offset of the aux buffer is a multiple of 4 floats, and channels 16 m + 4 g
// .. + 3 stay inside the C or C/2 biases of the M-tiles that read them).
__device__ __forceinline__ f32x4 ldq4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

// The workgroup-per-tile kernel: the cache bytes of a tile, whether it can take
// a network (channels: the kernel width), whether it takes a batch of it, and
// its launch.
int64_t fast_mw_tile_bytes(int H, int W, int nb, int channels, int precision);
bool fast_mw_supported(int H, int W, int nb, int channels, int precision);
bool fast_mw_takes(int H, int W, int nb, int channels, int precision, int64_t tiles);
int launch_fast_mw(const SampArgs& a, int channels, int precision, int act, int64_t tiles, hipStream_t s);

}  // namespace fk
