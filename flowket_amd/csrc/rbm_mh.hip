// Complex RBM wave function and Metropolis-Hastings chains.
//
// RBM (machines/rbm.py:35-48, layers/complex/dense.py:11-50,
// layers/complex/tensorflow_ops.py:69-85):
//   log psi(s) = sum_j a_j s_j + sum_h lncosh(theta_h),  theta_h = b_h + sum_j W_jh s_j,
// complex parameters stored as (real, imag) pairs and used as real - 1j*imag
// (layers/complex/base_layer.py:30-35).  A wavefront evaluates one configuration
// or eight, the hidden units spread over the lanes.
//
// MH (samplers/metropolis_hastings.py:15-145): a workgroup of one to eight waves
// per chain keeps theta in registers and updates it for each accepted move
// (a flipped site s_j changes theta by -2 s_j W_j.), so a proposal costs
// O(M) instead of a full O(N M) evaluation.  Acceptance is the reference rule
// exp(min(2 Re(logpsi' - logpsi), 0)) > U.  Random numbers are either
// injected (draw-for-draw parity) or drawn from a counter-based hash keyed by
// (seed, chain, step).
#include "fk_common.h"

namespace fk {

struct RbmParams {
  const float *w_re, *w_im, *b_re, *b_im, *a_re, *a_im;
  int N, M;
};

// Re and Im of lncosh(x + iy) (tensorflow_ops.py:79-85): |x| - log 2 +
// log(e^{z-|x|} + e^{-z-|x|}); the real part is written in the overflow-free
// form |x| - log 2 + 0.5 log1p(e^{-4|x|} + 2 e^{-2|x|} cos 2y).
__device__ __forceinline__ float lncosh_re(float x, float y) {
  const float ax = fabsf(x);
  const float e2 = expf(-2.0f * ax);
  return ax - 0.69314718055994531f + 0.5f * log1pf(e2 * e2 + 2.0f * e2 * cosf(2.0f * y));
}

// Sum over the wave, the butterfly v[l] + v[l ^ 32], then ^ 16, 8, 4, 2, 1, in
// lane-permuting vector instructions: the halves and rows are exchanged by
// permlane swaps, and after each step the sums repeat with the step's period,
// so a rotation by 8 and by 4 within a row of 16 is the exchange with lane
// ^ 8 and ^ 4.  (Six shuffles through LDS are a chain of about 400 cycles that
// every Metropolis proposal waits for.)
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float wave_sum(float v) {
  const u32x2 h = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v),
                                                                             false, false));
  v = __uint_as_float(h[0]) + __uint_as_float(h[1]);
  const u32x2 r = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v),
                                                                             false, false));
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  v = dpp_add<0x128>(v);  // row_ror:8
  v = dpp_add<0x124>(v);  // row_ror:4
  v = dpp_add<0x4e>(v);   // quad_perm [2, 3, 0, 1]
  return dpp_add<0xb1>(v);  // quad_perm [1, 0, 3, 2]
}

// Both parts, the imaginary one as the argument of e^{z-|x|} + e^{-z-|x|}, with
// one exponential: of e^{x-|x|} and e^{-x-|x|} one is 1 and the other e^{-2|x|},
// the e2 of lncosh_re.
__device__ __forceinline__ void lncosh(float x, float y, float& re, float& im) {
  const float ax = fabsf(x);
  const float e = expf(-2.0f * ax);
  re = ax - 0.69314718055994531f + 0.5f * log1pf(e * e + 2.0f * e * cosf(2.0f * y));
  const float e1 = x >= 0.0f ? 1.0f : e, e2 = x >= 0.0f ? e : 1.0f;
  float sy, cy;
  sincosf(y, &sy, &cy);
  im = atan2f((e1 - e2) * sy, (e1 + e2) * cy);
}

// log psi of configurations: rows of `spins` or (sample, connection) pairs
// applied with the connection table (kind as fk_find_conn).
//
// A wave evaluates K consecutive configurations, hidden units over its lanes
// (HPL per lane at a time): a weight read once serves K of them.  With K = 1
// the 131 KB of weights of the 8x8 alpha-4 RBM came from L2 for every
// configuration (266k of them in 2671 us, 13 TB/s); eight per wave take
// 830 us, most of it the lncosh of 256 hidden units each.
// The spins of the K configurations sit in LDS as floats, in chunks of
// RBM_NJ sites, so four sites of one configuration are one broadcast read.
// theta is summed over the sites in order and log psi over a lane's hidden
// units in order, whatever K and HPL: results do not depend on them.
constexpr int RBM_NJ = 64, RBM_WAVES = 4;

template <int K, int HPL>
__global__ __launch_bounds__(64 * RBM_WAVES, 4) void rbm_log_psi_kernel(
    RbmParams p, const int8_t* __restrict__ spins, const int32_t* __restrict__ pairs,
    const int64_t* __restrict__ m_dev, int64_t m_count, int conn_kind, const int32_t* __restrict__ conn_a,
    const int32_t* __restrict__ conn_b, float* __restrict__ out) {
  __shared__ f32x4 s_spin[RBM_WAVES][K][RBM_NJ / 4];
  // (the wave index made uniform: its configurations' addresses stay scalar)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t m0 = ((int64_t)blockIdx.x * RBM_WAVES + wave) * K;
  int64_t M = m_dev ? *m_dev : m_count;
  if (M > m_count) M = m_count;
  if (m0 >= M) return;  // waves are independent: no barrier below
  const int8_t* row[K];
  int fa[K], fb[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int64_t m = m0 + k < M ? m0 + k : M - 1;  // the last wave repeats the last configuration
    int64_t b = m;
    int c = 0;
    if (pairs) {
      b = pairs[2 * m];
      c = pairs[2 * m + 1];
    }
    row[k] = spins + b * p.N;
    fa[k] = fb[k] = -1;
    if (c > 0) {
      fa[k] = conn_a[c];
      fb[k] = (conn_kind == FK_CONN_FLIP) ? -1 : conn_b[c];
    }
  }
  auto spin = [&](int k, int j) -> float {
    int8_t v = row[k][j];
    if (conn_kind == FK_CONN_FLIP) {
      if (j == fa[k]) v = (int8_t)-v;
    } else if (fa[k] >= 0) {
      if (j == fa[k]) v = row[k][fb[k]];
      else if (j == fb[k]) v = row[k][fa[k]];
    }
    return (float)v;
  };
  // sites j0 .. j0 + RBM_NJ - 1 of the K configurations into LDS (zeros
  // past the last site); only this wave reads them
  auto stage = [&](int j0) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < K; ++k)
      reinterpret_cast<float*>(s_spin[wave][k])[lane] = j0 + lane < p.N ? spin(k, j0 + lane) : 0.0f;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  float lr[K], li[K];
#pragma unroll
  for (int k = 0; k < K; ++k) lr[k] = li[k] = 0.0f;
  if (p.N <= RBM_NJ) stage(0);
  for (int h0 = 0; h0 < p.M; h0 += 64 * HPL) {
    float tr[HPL][K], ti[HPL][K];
    int h[HPL];
#pragma unroll
    for (int u = 0; u < HPL; ++u) {
      h[u] = h0 + 64 * u + lane;
      const int hc = h[u] < p.M ? h[u] : p.M - 1;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        tr[u][k] = p.b_re[hc];
        ti[u][k] = -p.b_im[hc];
      }
    }
    for (int j0 = 0; j0 < p.N; j0 += RBM_NJ) {
      if (p.N > RBM_NJ) stage(j0);
      const int jn = p.N - j0 < RBM_NJ ? p.N - j0 : RBM_NJ;
      for (int j = 0; j < jn; j += 4) {
        float wr[4][HPL], wi[4][HPL];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int64_t jj = j0 + (j + e < jn ? j + e : jn - 1);
#pragma unroll
          for (int u = 0; u < HPL; ++u) {
            const int hc = h[u] < p.M ? h[u] : p.M - 1;
            wr[e][u] = p.w_re[jj * p.M + hc];
            wi[e][u] = p.w_im[jj * p.M + hc];
          }
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const f32x4 s = s_spin[wave][k][j >> 2];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (j + e < jn) {
#pragma unroll
              for (int u = 0; u < HPL; ++u) {
                tr[u][k] += wr[e][u] * s[e];
                ti[u][k] -= wi[e][u] * s[e];
              }
            }
          }
        }
      }
    }
#pragma unroll
    for (int u = 0; u < HPL; ++u) {
      if (h[u] < p.M) {
#pragma unroll 1
        for (int k = 0; k < K; ++k) {
          float r, i;
          lncosh(tr[u][k], ti[u][k], r, i);
          lr[k] += r;
          li[k] += i;
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    for (int j = lane; j < p.N; j += 64) {
      const float s = spin(k, j);
      lr[k] += p.a_re[j] * s;
      li[k] -= p.a_im[j] * s;
    }
    const float sr = wave_sum(lr[k]), si = wave_sum(li[k]);
    if (lane == 0 && m0 + k < M) {
      out[2 * (m0 + k)] = sr;
      out[2 * (m0 + k) + 1] = si;
    }
  }
}

// counter-based uniform in [0, 1) (splitmix64 finaliser of the counter)
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ double u01(uint64_t seed, uint64_t chain, uint64_t step, uint64_t k) {
  const uint64_t r = mix64(seed ^ mix64(chain * 0x100000001B3ull ^ mix64(step * 4 + k)));
  return (double)(r >> 11) * (1.0 / 9007199254740992.0);
}

struct MhArgs {
  RbmParams p;
  int H, W;              // lattice (N = H*W)
  int kind;              // 0 local flip, 1 exchange
  int64_t chains;
  int64_t n_burn;        // sweeps before the first record
  int64_t n_record;      // recorded samples per chain
  int64_t unused;        // sweeps between records are unused + 1
  int8_t* state;         // (chains, N) in/out
  int8_t* out;           // (chains, n_record, N)
  int64_t* accepts;      // (chains) accepted proposals during the recorded sweeps
  float* logpsi;         // (chains, 2) final log psi
  // randomness: injected (sweeps, chains) arrays or hashed from seed
  const int32_t* r_site;   // local: flat site; exchange: flat site
  const int32_t* r_move;   // exchange: (dy+1)*3 + (dx+1)
  const double* r_u;       // acceptance uniforms
  uint64_t seed;
  int32_t* nonfinite;      // set to 1 when a proposal's log psi is not finite (or null)
};

// One workgroup of NW waves per chain, HPL hidden units a lane (M <= 64 NW HPL).
// A step is a serial chain -- theta', lncosh, the sum over the units, the
// decision -- so while the chip is not full it is latency that bounds a chain,
// and a wave per 64 units is the fastest (1024 chains x 319 exchange proposals
// of the 8x8 alpha-4 RBM: 921 us in one wave, 480 in four with the proposals
// drawn 64 at a time).  Once it is full every wave's own instructions count (the
// draws, the sum, the decision), and fewer waves with more units are: with 191
// exchange / local proposals 2048 chains take 554 / 715 us in four waves and 421
// / 591 in two, 16384 chains 3.56 / 4.72 ms in four and 1.90 / 3.00 in one.
// The waves exchange their units' terms through LDS (double-buffered, one
// barrier a step); every wave then adds a lane's terms in unit order and
// reduces over the lanes, so all reach the same decision, the one a single
// wave would: chains do not depend on NW and HPL.
template <int NW, int HPL>
__global__ __launch_bounds__(64 * NW, 4) void mh_rbm_kernel(MhArgs a) {
  constexpr int NU = NW * HPL;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  __shared__ float s_part[2][NW > 1 ? NU : 1][64];
  const int64_t ch = blockIdx.x;
  if (ch >= a.chains) return;
  const RbmParams& p = a.p;
  const int N = p.N, M = p.M;
  extern __shared__ int8_t s_state[];  // N spins of this chain
  for (int j = threadIdx.x; j < N; j += 64 * NW) s_state[j] = a.state[ch * N + j];
  __syncthreads();
  int h[HPL];
  bool unit[HPL];
#pragma unroll
  for (int u = 0; u < HPL; ++u) {
    h[u] = 64 * (wave * HPL + u) + lane;
    unit[u] = h[u] < M;
  }
  float tr[HPL], ti[HPL];
  auto theta = [&](int u) {  // from the state
    tr[u] = p.b_re[h[u]];
    ti[u] = -p.b_im[h[u]];
#pragma unroll 4
    for (int j = 0; j < N; ++j) {
      const float s = (float)s_state[j];
      tr[u] += p.w_re[(int64_t)j * M + h[u]] * s;
      ti[u] -= p.w_im[(int64_t)j * M + h[u]] * s;
    }
  };
  // Re lncosh(theta) of the current state, kept with theta (recomputed
  // only where theta changes)
  float lc[HPL];
#pragma unroll
  for (int u = 0; u < HPL; ++u) {
    tr[u] = ti[u] = 0.0f;
    if (unit[u]) theta(u);
    lc[u] = unit[u] ? lncosh_re(tr[u], ti[u]) : 0.0f;
  }
  const int64_t total = a.n_burn + a.n_record * (a.unused + 1);
  int64_t acc = 0;
  // The proposal of a step: sites (j2 = -1 for local moves) and uniform, from
  // the injected arrays or the counter hash.  It does not depend on earlier
  // acceptances, so lane l draws that of step base + l, 64 steps at once
  // (drawn by the whole wave for each step, the hash's 64-bit products were
  // a third of a step), and the next step's weight rows and visible biases
  // are requested while the current step computes.
  int dj1 = 0, dj2 = -1;
  double du = 0.0;
  auto draw = [&](int64_t base) {
    const int64_t st = base + lane;
    if (st >= total) return;
    int j1, mv = 0;
    if (a.r_u) {
      j1 = a.r_site[st * a.chains + ch];
      du = a.r_u[st * a.chains + ch];
      if (a.kind == 1) mv = a.r_move[st * a.chains + ch];
    } else {
      j1 = (int)(u01(a.seed, ch, st, 0) * N);
      if (j1 >= N) j1 = N - 1;
      du = u01(a.seed, ch, st, 1);
      if (a.kind == 1) {
        mv = (int)(u01(a.seed, ch, st, 2) * 9.0);
        if (mv > 8) mv = 8;
      }
    }
    dj1 = j1;
    if (a.kind == 1) {
      const int dy = mv / 3 - 1, dx = mv % 3 - 1;
      const int y = j1 / a.W, x = j1 - (j1 / a.W) * a.W;
      dj2 = ((y + dy + a.H) % a.H) * a.W + ((x + dx + a.W) % a.W);
    }
  };
  int cj1 = 0, cj2 = -1;
  double cu = 0.0;
  float pw1r[HPL] = {}, pw1i[HPL] = {}, pw2r[HPL] = {}, pw2i[HPL] = {};
  float pa1 = 0.0f, pa2 = 0.0f;
  auto prefetch = [&](int64_t st) {
    const int l = (int)(st & 63);
    if (l == 0) draw(st);
    cj1 = __builtin_amdgcn_readlane(dj1, l);
    cj2 = __builtin_amdgcn_readlane(dj2, l);
    cu = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(du), l),
                          __builtin_amdgcn_readlane(__double2loint(du), l));
    const int jb = cj2 >= 0 ? cj2 : cj1;
#pragma unroll
    for (int u = 0; u < HPL; ++u) {
      if (unit[u]) {
        pw1r[u] = p.w_re[(int64_t)cj1 * M + h[u]];
        pw1i[u] = p.w_im[(int64_t)cj1 * M + h[u]];
        pw2r[u] = p.w_re[(int64_t)jb * M + h[u]];
        pw2i[u] = p.w_im[(int64_t)jb * M + h[u]];
      }
    }
    pa1 = p.a_re[cj1];
    pa2 = p.a_re[jb];
  };
  if (total > 0) prefetch(0);
  int buf = 0;
  for (int64_t step = 0; step < total; ++step) {
    if (step > 0 && (step & 255) == 0) {
      // refresh theta from the state (bounds the drift of the FP32
      // incremental updates)
      auto refresh = [&](int u) {
        if (unit[u]) {
          theta(u);
          lc[u] = lncosh_re(tr[u], ti[u]);
        }
      };
      if constexpr (HPL == 1) {  // (a loop of one trip took 11 scalar registers more, spilled)
        refresh(0);
      } else {
#pragma unroll
        for (int u = 0; u < HPL; ++u) refresh(u);
      }
    }
    // ---- proposal: drawn (and its weight rows requested) one step ahead
    const int j1 = cj1, j2 = cj2;
    const double uniform = cu;
    float w1r[HPL], w1i[HPL], w2r[HPL], w2i[HPL];
#pragma unroll
    for (int u = 0; u < HPL; ++u) {
      w1r[u] = pw1r[u];
      w1i[u] = pw1i[u];
      w2r[u] = pw2r[u];
      w2i[u] = pw2i[u];
    }
    const float a1 = pa1, a2 = pa2;
    if (step + 1 < total) prefetch(step + 1);
    // sites that change: local -> j1; exchange -> j1 and j2 if they differ
    const float s1 = (float)s_state[j1];
    bool flip1 = true, flip2 = false;
    if (a.kind == 1) {
      const float s2 = (float)s_state[j2];
      flip1 = (j2 != j1) && (s1 != s2);
      flip2 = flip1;
    }
    float dre = 0.0f;
    float nr[HPL], ni[HPL], nl[HPL];
#pragma unroll
    for (int u = 0; u < HPL; ++u) {
      nr[u] = tr[u];
      ni[u] = ti[u];
      nl[u] = lc[u];
    }
    if (flip1) {  // uniform over the workgroup, as every branch of the step
      const float s2 = flip2 ? (float)s_state[j2] : 0.0f;
#pragma unroll
      for (int u = 0; u < HPL; ++u) {
        if (unit[u]) {
          nr[u] -= 2.0f * s1 * w1r[u];
          ni[u] += 2.0f * s1 * w1i[u];
          if (flip2) {
            nr[u] -= 2.0f * s2 * w2r[u];
            ni[u] += 2.0f * s2 * w2i[u];
          }
          nl[u] = lncosh_re(nr[u], ni[u]);
        }
      }
      if constexpr (NW > 1) {
        // (a wave writes a buffer again two exchanges later, after the barrier
        // of the one between, which every reader of this one has reached)
        float(*part)[64] = s_part[buf];
        buf ^= 1;
#pragma unroll
        for (int u = 0; u < HPL; ++u) part[wave * HPL + u][lane] = unit[u] ? nl[u] - lc[u] : 0.0f;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NU; ++k) dre += part[k][lane];
      } else {
#pragma unroll
        for (int u = 0; u < HPL; ++u) dre += unit[u] ? nl[u] - lc[u] : 0.0f;
      }
      dre = wave_sum(dre);
      dre += -2.0f * s1 * a1;
      if (flip2) dre += -2.0f * s2 * a2;
    }
    // ---- acceptance (samplers/metropolis_hastings.py:106-110); a
    // candidate whose log psi is not finite is reported (the reference
    // raises, :103-105) and never accepted
    const bool finite = isfinite(dre);
    if (!finite && a.nonfinite && threadIdx.x == 0) a.nonfinite[0] = 1;
    const float lr = fminf(2.0f * dre, 0.0f);
    const bool accept = finite && (double)expf(lr) > uniform;
    if (accept) {
      if (flip1) {
#pragma unroll
        for (int u = 0; u < HPL; ++u) {
          tr[u] = nr[u];
          ti[u] = ni[u];
          lc[u] = nl[u];
        }
        // every wave has read the state by the exchange's barrier above
        if (NW == 1) __syncthreads();
        if (threadIdx.x == 0) {
          if (flip2) {
            const int8_t t = s_state[j1];
            s_state[j1] = s_state[j2];
            s_state[j2] = t;
          } else {
            s_state[j1] = (int8_t)-s_state[j1];
          }
        }
        __syncthreads();
      }
      if (step >= a.n_burn) ++acc;
    }
    // ---- record
    if (step >= a.n_burn) {
      const int64_t rs = step - a.n_burn;
      if ((rs + 1) % (a.unused + 1) == 0) {
        const int64_t rec = rs / (a.unused + 1);
        for (int j = threadIdx.x; j < N; j += 64 * NW) a.out[(ch * a.n_record + rec) * N + j] = s_state[j];
      }
    }
  }
  for (int j = threadIdx.x; j < N; j += 64 * NW) a.state[ch * N + j] = s_state[j];
  if (threadIdx.x == 0) a.accepts[ch] = acc;
  if (!a.logpsi) return;
  // final log psi from theta, a lane's units in order
  __shared__ float s_fin[NU][2][64];
#pragma unroll
  for (int u = 0; u < HPL; ++u) {
    float r = 0.0f, i = 0.0f;
    if (unit[u]) lncosh(tr[u], ti[u], r, i);
    s_fin[wave * HPL + u][0][lane] = r;
    s_fin[wave * HPL + u][1][lane] = i;
  }
  __syncthreads();
  if (wave > 0) return;
  float lr = 0.0f, li = 0.0f;
#pragma unroll
  for (int k = 0; k < NU; ++k) {
    if (lane + 64 * k < M) {
      lr += s_fin[k][0][lane];
      li += s_fin[k][1][lane];
    }
  }
  for (int j = lane; j < N; j += 64) {
    const float s = (float)s_state[j];
    lr += p.a_re[j] * s;
    li -= p.a_im[j] * s;
  }
  lr = wave_sum(lr);
  li = wave_sum(li);
  if (lane == 0) {
    a.logpsi[2 * ch] = lr;
    a.logpsi[2 * ch + 1] = li;
  }
}

// ---- machine-agnostic MH pieces (any wave function evaluated elsewhere)
__global__ void mh_propose_kernel(const int8_t* __restrict__ state, int64_t chains, int H, int W, int kind,
                                  const int32_t* __restrict__ r_site, const int32_t* __restrict__ r_move,
                                  int8_t* __restrict__ cand) {
  const int64_t ch = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (ch >= chains) return;
  const int N = H * W;
  const int8_t* s = state + ch * N;
  int8_t* c = cand + ch * N;
  for (int j = 0; j < N; ++j) c[j] = s[j];
  const int j1 = r_site[ch];
  if (kind == 0) {
    c[j1] = (int8_t)-c[j1];
  } else {
    const int mv = r_move[ch];
    const int dy = mv / 3 - 1, dx = mv % 3 - 1;
    const int y = j1 / W, x = j1 - (j1 / W) * W;
    const int j2 = ((y + dy + H) % H) * W + ((x + dx + W) % W);
    const int8_t t = c[j1];
    c[j1] = c[j2];
    c[j2] = t;
  }
}

__global__ void mh_accept_kernel(int8_t* __restrict__ state, float* __restrict__ logpsi_cur,
                                 const int8_t* __restrict__ cand, const float* __restrict__ logpsi_cand,
                                 const double* __restrict__ u, int64_t chains, int N, int32_t* __restrict__ accepted,
                                 int32_t* __restrict__ nonfinite) {
  const int64_t ch = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (ch >= chains) return;
  const bool finite = isfinite(logpsi_cand[2 * ch]) && isfinite(logpsi_cand[2 * ch + 1]);
  if (!finite && nonfinite) nonfinite[0] = 1;
  const float lr = fminf(2.0f * (logpsi_cand[2 * ch] - logpsi_cur[2 * ch]), 0.0f);
  const bool acc = finite && (double)expf(lr) > u[ch];
  accepted[ch] = acc ? 1 : 0;
  if (acc) {
    for (int j = 0; j < N; ++j) state[ch * N + j] = cand[ch * N + j];
    logpsi_cur[2 * ch] = logpsi_cand[2 * ch];
    logpsi_cur[2 * ch + 1] = logpsi_cand[2 * ch + 1];
  }
}

// Independent proposal with the exact Metropolis-Hastings ratio:
// accept iff exp(min(2 Re(logpsi' - logpsi) + log q(x) - log q(x'), 0)) > U.
__global__ void mh_accept_independent_kernel(int8_t* __restrict__ state, float* __restrict__ logpsi_cur,
                                             float* __restrict__ logq_cur, const int8_t* __restrict__ cand,
                                             const float* __restrict__ logpsi_cand, const float* __restrict__ logq_cand,
                                             const double* __restrict__ u, int64_t chains, int N,
                                             int32_t* __restrict__ accepted, int32_t* __restrict__ nonfinite) {
  const int64_t ch = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (ch >= chains) return;
  const bool finite = isfinite(logpsi_cand[2 * ch]) && isfinite(logpsi_cand[2 * ch + 1]);
  if (!finite && nonfinite) nonfinite[0] = 1;
  const float lr = fminf(2.0f * (logpsi_cand[2 * ch] - logpsi_cur[2 * ch]) + (logq_cur[ch] - logq_cand[ch]), 0.0f);
  const bool acc = finite && (double)expf(lr) > u[ch];
  accepted[ch] = acc ? 1 : 0;
  if (acc) {
    for (int j = 0; j < N; ++j) state[ch * N + j] = cand[ch * N + j];
    logpsi_cur[2 * ch] = logpsi_cand[2 * ch];
    logpsi_cur[2 * ch + 1] = logpsi_cand[2 * ch + 1];
    logq_cur[ch] = logq_cand[ch];
  }
}

// Per-sample O = d log psi / d(parameter) of the RBM (the Jacobian the
// reference's ComplexValuesOptimizer takes of complex layers,
// optimizers/complex_values_optimizer.py:60-76, written over the stored real
// and imaginary parts): with theta_h = b_h + sum_j W_jh s_j and
// T_h = tanh(theta_h), d/dW_re[j,h] = s_j T_h, d/dW_im[j,h] = -i s_j T_h,
// d/db_re[h] = T_h, d/db_im[h] = -i T_h, d/da_re[j] = s_j, d/da_im[j] = -i s_j
// (every complex parameter is used as real - i*imag, base_layer.py:30-35).
// One workgroup per sample; rows in the flat order W_re, W_im, b_re, b_im,
// a_re, a_im.
__global__ __launch_bounds__(256) void rbm_grad_kernel(RbmParams p, const int8_t* __restrict__ spins, int64_t batch,
                                                       float* __restrict__ o_re, float* __restrict__ o_im,
                                                       int64_t ld) {
  extern __shared__ float s_t[];  // T_h (re, im), then the spins
  const int N = p.N, M = p.M;
  const int64_t b = blockIdx.x;
  if (b >= batch) return;
  float* tre = s_t;
  float* tim = s_t + M;
  float* sv = s_t + 2 * M;
  for (int j = threadIdx.x; j < N; j += blockDim.x) sv[j] = (float)spins[b * N + j];
  __syncthreads();
  for (int h = threadIdx.x; h < M; h += blockDim.x) {
    float x = p.b_re[h], y = -p.b_im[h];
    for (int j = 0; j < N; ++j) {
      x += p.w_re[(int64_t)j * M + h] * sv[j];
      y -= p.w_im[(int64_t)j * M + h] * sv[j];
    }
    // tanh(x + iy) = (sinh 2x + i sin 2y) / (cosh 2x + cos 2y), written with
    // e = exp(-2|x|) so that it cannot overflow
    const float e = expf(-2.0f * fabsf(x));
    float sn, cs;
    sincosf(2.0f * y, &sn, &cs);
    const float den = 1.0f + e * e + 2.0f * e * cs;
    tre[h] = copysignf((1.0f - e * e) / den, x);
    tim[h] = 2.0f * e * sn / den;
  }
  __syncthreads();
  float* ore = o_re + b * ld;
  float* oim = o_im + b * ld;
  const int64_t NM = (int64_t)N * M;
  for (int64_t q = threadIdx.x; q < NM; q += blockDim.x) {
    const int j = (int)(q / M), h = (int)(q - (q / M) * M);
    const float sj = sv[j];
    ore[q] = sj * tre[h];
    oim[q] = sj * tim[h];
    ore[NM + q] = sj * tim[h];
    oim[NM + q] = -sj * tre[h];
  }
  for (int h = threadIdx.x; h < M; h += blockDim.x) {
    ore[2 * NM + h] = tre[h];
    oim[2 * NM + h] = tim[h];
    ore[2 * NM + M + h] = tim[h];
    oim[2 * NM + M + h] = -tre[h];
  }
  for (int j = threadIdx.x; j < N; j += blockDim.x) {
    ore[2 * NM + 2 * M + j] = sv[j];
    oim[2 * NM + 2 * M + j] = 0.0f;
    ore[2 * NM + 2 * M + N + j] = 0.0f;
    oim[2 * NM + 2 * M + N + j] = -sv[j];
  }
}

}  // namespace fk

using namespace fk;

extern "C" {

int fk_rbm_log_psi(const float* w_re, const float* w_im, const float* b_re, const float* b_im, const float* a_re,
                   const float* a_im, int32_t n_visible, int32_t n_hidden, const int8_t* spins,
                   const int32_t* pairs, const int64_t* m_dev, int64_t m_count, int32_t conn_kind,
                   const int32_t* conn_a, const int32_t* conn_b, float* logpsi, void* stream) {
  FK_REQUIRE(n_visible > 0 && n_hidden > 0, "fk_rbm_log_psi: bad sizes");
  if (m_count <= 0) return FK_OK;
  FK_REQUIRE(w_re && w_im && b_re && b_im && a_re && a_im && spins && logpsi, "fk_rbm_log_psi: null pointer");
  FK_REQUIRE(!pairs || (conn_a && conn_b), "fk_rbm_log_psi: pairs need a connection table");
  RbmParams p{w_re, w_im, b_re, b_im, a_re, a_im, n_visible, n_hidden};
  // eight configurations a wave once that still gives every CU eight waves
  // (two per SIMD); fewer configurations go one to a wave.  Two hidden units
  // per lane at a time keep the eight-configuration form at four waves per
  // SIMD (four took 290 registers: one wave per SIMD).
  auto launch = [&](auto kern, int k) {
    hipLaunchKernelGGL(kern, dim3(div_up(m_count, (int64_t)k * RBM_WAVES)), dim3(64 * RBM_WAVES), 0,
                       (hipStream_t)stream, p, spins, pairs, m_dev, m_count, conn_kind, conn_a, conn_b, logpsi);
  };
  const bool one = n_hidden <= 64;
  if (m_count >= 64LL * device_cu_count()) {
    if (one) launch(rbm_log_psi_kernel<8, 1>, 8);
    else launch(rbm_log_psi_kernel<8, 2>, 8);
  } else {
    if (one) launch(rbm_log_psi_kernel<1, 1>, 1);
    else launch(rbm_log_psi_kernel<1, 4>, 1);
  }
  FK_CHECK_LAUNCH();
  return FK_OK;
}

int fk_mh_rbm(const float* w_re, const float* w_im, const float* b_re, const float* b_im, const float* a_re,
              const float* a_im, int32_t n_visible, int32_t n_hidden, int32_t H, int32_t W, int32_t kind,
              int64_t chains, int64_t n_burn, int64_t n_record, int64_t unused, int8_t* state, int8_t* out,
              int64_t* accepts, float* logpsi, const int32_t* r_site, const int32_t* r_move, const double* r_u,
              uint64_t seed, int32_t* nonfinite, void* stream) {
  FK_REQUIRE(n_visible == H * W && n_visible > 0 && n_hidden > 0, "fk_mh_rbm: bad sizes");
  FK_REQUIRE(kind == 0 || kind == 1, "fk_mh_rbm: kind must be 0 (local) or 1 (exchange)");
  FK_REQUIRE(chains >= 0 && n_burn >= 0 && n_record >= 0 && unused >= 0, "fk_mh_rbm: bad counts");
  if (chains == 0) return FK_OK;
  FK_REQUIRE(w_re && w_im && b_re && b_im && a_re && a_im && state && accepts, "fk_mh_rbm: null pointer");
  FK_REQUIRE(n_record == 0 || out, "fk_mh_rbm: null output");
  FK_REQUIRE(!r_u || (r_site && (kind == 0 || r_move)), "fk_mh_rbm: injected randomness incomplete");
  FK_REQUIRE(chains <= 0x7fffffff, "fk_mh_rbm: too many chains");
  MhArgs a;
  a.p = RbmParams{w_re, w_im, b_re, b_im, a_re, a_im, n_visible, n_hidden};
  a.H = H;
  a.W = W;
  a.kind = kind;
  a.chains = chains;
  a.n_burn = n_burn;
  a.n_record = n_record;
  a.unused = unused;
  a.state = state;
  a.out = out;
  a.accepts = accepts;
  a.logpsi = logpsi;
  a.r_site = r_site;
  a.r_move = r_move;
  a.r_u = r_u;
  a.seed = seed;
  a.nonfinite = nonfinite;
  if (n_hidden > 512) {
    set_error("fk_mh_rbm: at most 512 hidden units");
    return FK_ERR_UNSUPPORTED;
  }
  const size_t lds = (size_t)((n_visible + 15) & ~15);
  hipStream_t s = (hipStream_t)stream;
  const int units = n_hidden <= 64 ? 1 : n_hidden <= 128 ? 2 : n_hidden <= 256 ? 4 : 8;  // of 64
  // a wave per unit while that leaves at most four waves a SIMD, then fewer of up
  // to four units (128 units: the two forms cross at about 1200 chains and differ
  // by 6 % at 2048; 256 units: at 1000 and 2300; 400 to 512: at 450 and 1800;
  // eight units a lane are slower than four everywhere)
  int nw = units;
  while (nw > 1 && units / nw < 4 && chains * nw > 16LL * device_cu_count()) nw /= 2;
  auto launch = [&](auto kern) -> int {
    // the state and the waves' exchange buffers together may pass the 64 KB
    // that a launch gets unasked
    if (lds > 48 * 1024)
      FK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds));
    hipLaunchKernelGGL(kern, dim3((unsigned)chains), dim3(64 * nw), lds, s, a);
    FK_CHECK_LAUNCH();
    return FK_OK;
  };
  if (units == 1) return launch(mh_rbm_kernel<1, 1>);
  if (units == 2) return nw == 2 ? launch(mh_rbm_kernel<2, 1>) : launch(mh_rbm_kernel<1, 2>);
  if (units == 4)
    return nw == 4 ? launch(mh_rbm_kernel<4, 1>) : nw == 2 ? launch(mh_rbm_kernel<2, 2>) : launch(mh_rbm_kernel<1, 4>);
  return nw == 8 ? launch(mh_rbm_kernel<8, 1>) : nw == 4 ? launch(mh_rbm_kernel<4, 2>) : launch(mh_rbm_kernel<2, 4>);
}

int fk_rbm_grad(const float* w_re, const float* w_im, const float* b_re, const float* b_im, const float* a_re,
                const float* a_im, int32_t n_visible, int32_t n_hidden, const int8_t* spins, int64_t batch,
                float* o_re, float* o_im, int64_t row_stride, void* stream) {
  FK_REQUIRE(n_visible > 0 && n_hidden > 0 && batch >= 0, "fk_rbm_grad: bad sizes");
  if (batch == 0) return FK_OK;
  FK_REQUIRE(w_re && w_im && b_re && b_im && a_re && a_im && spins && o_re && o_im, "fk_rbm_grad: null pointer");
  const int64_t P = 2 * (int64_t)n_visible * n_hidden + 2 * (int64_t)n_hidden + 2 * (int64_t)n_visible;
  FK_REQUIRE(row_stride == 0 || row_stride >= P, "fk_rbm_grad: row stride shorter than the parameters");
  FK_REQUIRE(batch <= 0x7fffffff, "fk_rbm_grad: batch too large");
  const size_t lds = (size_t)(2 * n_hidden + n_visible) * sizeof(float);
  FK_REQUIRE(lds <= 64 * 1024, "fk_rbm_grad: too many units");
  RbmParams p{w_re, w_im, b_re, b_im, a_re, a_im, n_visible, n_hidden};
  hipLaunchKernelGGL(rbm_grad_kernel, dim3((unsigned)batch), dim3(256), lds, (hipStream_t)stream, p, spins, batch,
                     o_re, o_im, row_stride > 0 ? row_stride : P);
  FK_CHECK_LAUNCH();
  return FK_OK;
}

int fk_mh_propose(const int8_t* state, int64_t chains, int32_t H, int32_t W, int32_t kind, const int32_t* r_site,
                  const int32_t* r_move, int8_t* candidates, void* stream) {
  FK_REQUIRE(kind == 0 || kind == 1, "fk_mh_propose: bad kind");
  if (chains <= 0) return FK_OK;
  FK_REQUIRE(state && r_site && candidates && (kind == 0 || r_move), "fk_mh_propose: null pointer");
  hipLaunchKernelGGL(mh_propose_kernel, dim3(div_up(chains, 256)), dim3(256), 0, (hipStream_t)stream, state, chains,
                     H, W, kind, r_site, r_move, candidates);
  FK_CHECK_LAUNCH();
  return FK_OK;
}

int fk_mh_accept(int8_t* state, float* logpsi_cur, const int8_t* candidates, const float* logpsi_cand,
                 const double* uniforms, int64_t chains, int32_t n_sites, int32_t* accepted, int32_t* nonfinite,
                 void* stream) {
  if (chains <= 0) return FK_OK;
  FK_REQUIRE(state && logpsi_cur && candidates && logpsi_cand && uniforms && accepted, "fk_mh_accept: null pointer");
  hipLaunchKernelGGL(mh_accept_kernel, dim3(div_up(chains, 256)), dim3(256), 0, (hipStream_t)stream, state,
                     logpsi_cur, candidates, logpsi_cand, uniforms, chains, n_sites, accepted, nonfinite);
  FK_CHECK_LAUNCH();
  return FK_OK;
}

int fk_mh_accept_independent(int8_t* state, float* logpsi_cur, float* logq_cur, const int8_t* candidates,
                             const float* logpsi_cand, const float* logq_cand, const double* uniforms, int64_t chains,
                             int32_t n_sites, int32_t* accepted, int32_t* nonfinite, void* stream) {
  if (chains <= 0) return FK_OK;
  FK_REQUIRE(state && logpsi_cur && logq_cur && candidates && logpsi_cand && logq_cand && uniforms && accepted,
             "fk_mh_accept_independent: null pointer");
  hipLaunchKernelGGL(mh_accept_independent_kernel, dim3(div_up(chains, 256)), dim3(256), 0, (hipStream_t)stream,
                     state, logpsi_cur, logq_cur, candidates, logpsi_cand, logq_cand, uniforms, chains, n_sites,
                     accepted, nonfinite);
  FK_CHECK_LAUNCH();
  return FK_OK;
}

}  // extern "C"
