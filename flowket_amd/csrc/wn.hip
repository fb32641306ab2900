// Chain rule of weight normalisation (deepar/layers/wrappers.py:123-135):
// a wrapped layer's kernel is k = v / n * s per output channel c, with
// n = sqrt(max(sum_i v_i^2, 1e-12)) over the channel's kh*kw*cin values
// (tf.nn.l2_normalize) and s = exp(g) (exponential_norm) or g.  The gradient
// kernels of this library differentiate with respect to k; these kernels map
// such derivatives onto the trainable (v, g), and parameter directions
// (v', g') onto directions in k; fk_wn_effective forms the kernels k
// themselves.
#include "fk_common.h"

namespace fk {

// Layer table: 4 int64 per weight-normalised layer (kernel offset in the flat
// parameters, kh*kw*cin, cout, offset of its g in the g vector).
struct WnLayer {
  int64_t koff, nin, cout, goff;
};

__device__ __forceinline__ WnLayer wn_layer(const int64_t* t, int l) {
  return WnLayer{t[4 * l], t[4 * l + 1], t[4 * l + 2], t[4 * l + 3]};
}

// Threads of a workgroup over one (layer, tile of CT channels): channel
// c = tile * CT + tid % CT, and the channel's nin values dealt to G groups of
// threads.  Neighbouring threads then read neighbouring channels, so a wave's
// loads are contiguous (kernels are (..., cin, cout)).  What bounds these
// kernels is the chain of loads of one channel: with a thread per channel it
// was nin (up to 576) dependent iterations, 240 us for 64 rows of the 4x4
// depth-5 32-channel network and 520 us for 256 rows of the 12x12 depth-10 one;
// dealt to the groups, 32 and 283.
// Networks of fewer than 16 channels have too few values for the threads, and
// many rows would be as many nearly empty workgroups: there a group has four
// values or more and the threads take several rows at a time (8192 rows, depth 3,
// 2 channels: 24 us with a thread per channel, 593 with a row a workgroup, 26
// so; depth 5, 8 channels 407, 658 and 349; 12 channels 831, 878 and 834; at
// 16 channels one row a workgroup is the faster one, depth 6, 4096 rows: 733).
constexpr int WN_THREADS = 256;

struct WnTile {
  int CT, G, rows;  // channels; groups; rows at a time
  int col, grp, row;
  int64_t c;
  bool live;
};

__device__ __forceinline__ int wn_tile_channels(const WnLayer& L) { return L.cout < 64 ? (int)L.cout : 64; }

// Groups of a row (1 .. WN_THREADS / CT): of four values or more, and as many
// rows as come nearest to using all threads.
__host__ __device__ inline int wn_row_groups(int CT, int64_t nin) {
  const int all = WN_THREADS / CT;
  const int most = nin < 8 ? 1 : nin / 4 < all ? (int)(nin / 4) : all;
  const int rows = (2 * WN_THREADS / (CT * most) + 1) / 2;
  const int even = WN_THREADS / (CT * rows);  // 0 where rounding up left no thread for a row
  return even < 1 ? 1 : even < most ? even : most;
}

template <bool MULTI>
__device__ __forceinline__ WnTile wn_tile(const WnLayer& L, int64_t tile) {
  WnTile t;
  t.CT = wn_tile_channels(L);
  t.G = WN_THREADS / t.CT;
  t.rows = 1;
  t.grp = (int)threadIdx.x / t.CT;
  t.row = 0;
  t.col = (int)threadIdx.x % t.CT;
  t.c = tile * t.CT + t.col;
  if constexpr (MULTI) {
    t.G = wn_row_groups(t.CT, L.nin);
    t.rows = WN_THREADS / (t.CT * t.G);
    t.row = t.grp / t.G;
    t.grp -= t.row * t.G;
    t.live = t.row < t.rows && t.c < L.cout;
  } else {
    t.live = t.grp < t.G && t.c < L.cout;
  }
  return t;
}

// Sum over the groups of a channel (and row), in group order (FP64,
// deterministic); every thread of the channel gets it.  red: WN_THREADS doubles.
__device__ __forceinline__ double wn_group_sum(double x, const WnTile& t, double* red) {
  __syncthreads();
  red[threadIdx.x] = x;
  __syncthreads();
  const int first = (t.row < t.rows ? t.row : 0) * t.G * t.CT + t.col;
  double s = 0.0;
  for (int k = 0; k < t.G; ++k) s += red[first + k * t.CT];
  return s;
}

// Norm and scale of the thread's channel.
__device__ __forceinline__ void wn_norm(const float* __restrict__ v, const WnLayer& L, const WnTile& t,
                                        const float* __restrict__ g, int exp_norm, double* red, float& n, float& s,
                                        bool& clamped) {
  double ss = 0.0;
  if (t.live) {
    const float* p = v + L.koff + t.c;
#pragma unroll 4
    for (int64_t i = t.grp; i < L.nin; i += t.G) {
      const double x = p[i * L.cout];
      ss += x * x;
    }
  }
  ss = wn_group_sum(ss, t, red);
  clamped = (float)ss < 1e-12f;
  n = clamped ? sqrtf(1e-12f) : (float)sqrt(ss);
  s = 0.0f;
  if (t.live) s = exp_norm ? expf(g[L.goff + t.c]) : g[L.goff + t.c];
}

// v . x over the thread's channel (x: a row of d/dk or a direction).
__device__ __forceinline__ float wn_dot(const float* __restrict__ v, const float* __restrict__ x, const WnLayer& L,
                                        const WnTile& t, double* red) {
  double dot = 0.0;
  if (t.live) {
    const int64_t q0 = L.koff + t.c;
#pragma unroll 4
    for (int64_t i = t.grp; i < L.nin; i += t.G) dot += (double)v[q0 + i * L.cout] * x[q0 + i * L.cout];
  }
  return (float)wn_group_sum(dot, t, red);
}

// The kernels of wrapped layers, k = v / n * s, one workgroup per (tile of
// channels, layer); every other entry is copied beforehand.
__global__ __launch_bounds__(WN_THREADS) void wn_effective_kernel(const float* __restrict__ v,
                                                                  const float* __restrict__ g,
                                                                  const int64_t* __restrict__ layers, int exp_norm,
                                                                  float* __restrict__ out) {
  __shared__ double red[WN_THREADS];
  const WnLayer L = wn_layer(layers, blockIdx.y);
  if ((int64_t)blockIdx.x * wn_tile_channels(L) >= L.cout) return;
  const WnTile t = wn_tile<false>(L, blockIdx.x);
  float n, s;
  bool clamped;
  wn_norm(v, L, t, g, exp_norm, red, n, s, clamped);
  if (!t.live) return;
#pragma unroll 4
  for (int64_t i = t.grp; i < L.nin; i += t.G) {
    const int64_t q = L.koff + i * L.cout + t.c;
    out[q] = v[q] / n * s;
  }
}

// In place on rows (nrows, ld): row[:P] holds d/dk on entry; on exit the
// kernel entries of every wrapped layer hold d/dv and row[P + goff + c] holds
// d/dg.  dv_i = s/n (dk_i - v_i (v.dk)/n^2) (s/n dk_i when the norm is
// clamped), dg = s/n (v.dk) for exponential_norm, (v.dk)/n otherwise.  A
// workgroup takes sets of t.rows rows, blockIdx.z, blockIdx.z + gridDim.z, ...,
// of one (tile, layer), so the norm is computed once for them.
template <bool MULTI>
__global__ __launch_bounds__(WN_THREADS) void wn_grad_rows_kernel(float* __restrict__ rows, int64_t nrows, int64_t ld,
                                                                  const float* __restrict__ v,
                                                                  const float* __restrict__ g,
                                                                  const int64_t* __restrict__ layers, int exp_norm,
                                                                  int64_t P) {
  __shared__ double red[WN_THREADS];
  const WnLayer L = wn_layer(layers, blockIdx.y);
  if ((int64_t)blockIdx.x * wn_tile_channels(L) >= L.cout) return;
  const WnTile t = wn_tile<MULTI>(L, blockIdx.x);
  float n, s;
  bool clamped;
  wn_norm(v, L, t, g, exp_norm, red, n, s, clamped);
  const float sn = s / n;
  for (int64_t r0 = (int64_t)blockIdx.z * t.rows; r0 < nrows; r0 += (int64_t)gridDim.z * t.rows) {
    bool live = t.live;
    float* row = rows + r0 * ld;
    if constexpr (MULTI) {
      live = live && r0 + t.row < nrows;
      if (live) row += t.row * ld;
    }
    const float dot = wn_dot(v, row, L, t, red);
    if (!live) continue;
    const float proj = clamped ? 0.0f : dot / (n * n);
#pragma unroll 4
    for (int64_t i = t.grp; i < L.nin; i += t.G) {
      const int64_t q = L.koff + i * L.cout + t.c;
      row[q] = sn * (row[q] - v[q] * proj);
    }
    if (t.grp == 0) row[P + L.goff + t.c] = exp_norm ? sn * dot : dot / n;
  }
}

// t_eff (P) from a direction t over (v, g): kernel entries
// s/n (t_i - v_i (v.t)/n^2) + dk/dg t_g with dk/dg = k (exponential_norm) or
// v/n; every other entry (biases, the head) is t itself.
__global__ void wn_copy_kernel(const float* __restrict__ t, float* __restrict__ out, int64_t P) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < P) out[q] = t[q];
}

__global__ __launch_bounds__(WN_THREADS) void wn_tangent_kernel(const float* __restrict__ v,
                                                                const float* __restrict__ g,
                                                                const int64_t* __restrict__ layers, int exp_norm,
                                                                const float* __restrict__ x, float* __restrict__ out,
                                                                int64_t P) {
  __shared__ double red[WN_THREADS];
  const WnLayer L = wn_layer(layers, blockIdx.y);
  if ((int64_t)blockIdx.x * wn_tile_channels(L) >= L.cout) return;
  const WnTile t = wn_tile<false>(L, blockIdx.x);
  float n, s;
  bool clamped;
  wn_norm(v, L, t, g, exp_norm, red, n, s, clamped);
  const float dot = wn_dot(v, x, L, t, red);
  if (!t.live) return;
  const float sn = s / n;
  const float proj = clamped ? 0.0f : dot / (n * n);
  const float tg = x[P + L.goff + t.c];
#pragma unroll 4
  for (int64_t i = t.grp; i < L.nin; i += t.G) {
    const int64_t q = L.koff + i * L.cout + t.c;
    const float dkdg = exp_norm ? v[q] * sn : v[q] / n;
    out[q] = sn * (x[q] - v[q] * proj) + dkdg * tg;
  }
}

}  // namespace fk

using namespace fk;

extern "C" {

int fk_wn_grad_rows(float* rows, int64_t nrows, int64_t ld, const float* params, const float* g,
                    const int64_t* layers, int32_t n_layers, int32_t max_cout, int32_t exp_norm, int64_t n_params,
                    void* stream) {
  FK_REQUIRE(nrows >= 0 && n_layers >= 0 && max_cout >= 1 && n_params >= 0, "fk_wn_grad_rows: bad sizes");
  if (nrows == 0 || n_layers == 0) return FK_OK;
  FK_REQUIRE(rows && params && g && layers, "fk_wn_grad_rows: null pointer");
  FK_REQUIRE(ld >= n_params, "fk_wn_grad_rows: row stride shorter than the parameters");
  FK_REQUIRE(n_layers <= 65535, "fk_wn_grad_rows: too many layers");
  // few rows: a workgroup per row; many: the rows dealt to as many workgroups
  // as keep 16 of them per CU, so that the norms are not recomputed per row
  const int64_t most = 1 + 16LL * device_cu_count() / n_layers;
  hipLaunchKernelGGL((max_cout < 16 ? wn_grad_rows_kernel<true> : wn_grad_rows_kernel<false>),
                     dim3((unsigned)div_up(max_cout, 64), (unsigned)n_layers, (unsigned)(nrows < most ? nrows : most)),
                     dim3(WN_THREADS), 0, (hipStream_t)stream, rows, nrows, ld, params, g, layers, exp_norm, n_params);
  FK_CHECK_LAUNCH();
  return FK_OK;
}

int fk_wn_tangent(const float* params, const float* g, const int64_t* layers, int32_t n_layers, int32_t max_cout,
                  int32_t exp_norm, const float* t, float* t_eff, int64_t n_params, void* stream) {
  FK_REQUIRE(n_layers >= 0 && max_cout >= 1 && n_params >= 0, "fk_wn_tangent: bad sizes");
  FK_REQUIRE(params && t && t_eff && (n_layers == 0 || (g && layers)), "fk_wn_tangent: null pointer");
  FK_REQUIRE(n_layers <= 65535, "fk_wn_tangent: too many layers");
  hipStream_t s = (hipStream_t)stream;
  if (n_params > 0) {
    hipLaunchKernelGGL(wn_copy_kernel, dim3(div_up(n_params, 256)), dim3(256), 0, s, t, t_eff, n_params);
    FK_CHECK_LAUNCH();
  }
  if (n_layers == 0) return FK_OK;
  hipLaunchKernelGGL(wn_tangent_kernel, dim3((unsigned)div_up(max_cout, 64), (unsigned)n_layers), dim3(WN_THREADS), 0,
                     s, params, g, layers, exp_norm, t, t_eff, n_params);
  FK_CHECK_LAUNCH();
  return FK_OK;
}

int fk_wn_effective(const float* params, const float* g, const int64_t* layers, int32_t n_layers, int32_t max_cout,
                    int32_t exp_norm, float* effective, int64_t n_params, void* stream) {
  FK_REQUIRE(n_layers >= 0 && max_cout >= 1 && n_params >= 0, "fk_wn_effective: bad sizes");
  FK_REQUIRE(params && effective && (n_layers == 0 || (g && layers)), "fk_wn_effective: null pointer");
  FK_REQUIRE(n_layers <= 65535, "fk_wn_effective: too many layers");
  hipStream_t s = (hipStream_t)stream;
  if (n_params > 0) {
    hipLaunchKernelGGL(wn_copy_kernel, dim3(div_up(n_params, 256)), dim3(256), 0, s, params, effective, n_params);
    FK_CHECK_LAUNCH();
  }
  if (n_layers == 0) return FK_OK;
  hipLaunchKernelGGL(wn_effective_kernel, dim3((unsigned)div_up(max_cout, 64), (unsigned)n_layers), dim3(WN_THREADS),
                     0, s, params, g, layers, exp_norm, effective);
  FK_CHECK_LAUNCH();
  return FK_OK;
}

}  // extern "C"
