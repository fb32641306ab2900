// Fast autoregressive sampling, a workgroup per 16 samples
// (deepar/samplers/fast_autoregressive.py:13-76, as fast_sampler.hip, whose
// cache layout, arithmetic, accumulation order and roundings it shares, so
// the draws are the same bits).
//
// What bounds a draw is a serial chain: site by site, the masked final block
// gives the conditional, the spin is drawn, and every block's horizontal
// stack advances one site, each block on the output of the one before.  Of a
// block step's taps only one of the 1x3 convolution's three and one of the
// 3x3's nine read the value that the chain just made; the others read earlier
// sites.  So wave 0 walks the chain and nothing else -- tap 2, the 1x1, tap
// 8: three dependent MFMA groups, operands in LDS and registers -- and the
// other waves (helpers) run ahead of it, one block step each, making
//   ph = bias + taps 0, 1 of the 1x3 convolution
//   pc = bias + taps 0..7 of the 3x3 convolution
// which the chain continues: the sums keep their order.  Helpers also write
// the chain's outputs to the cache, so the chain waits on no store.  After a
// row all waves share the vertical stack's pixels, block by block, the row
// itself in LDS.
//
// Steps and synchronisation.  A row is W x nb steps: for each site the
// conditional (block F = nb - 1), then blocks 0..F-1.  G steps make a
// super-tick, ended by one barrier.  In super-tick K
//   the chain runs the steps of K on the ph / pc made in K - 1,
//   helper g makes those of step g of K + 1 (its operands were requested at
//   the end of K - 1), stores step g of K - 1's outputs, and requests the
//   operands of step g of K + 2;
// LDS entries alternate between two sets.  A helper waits for all its memory
// operations at the start of each super-tick, so a store issued in J is
// complete when barrier J + 1 has passed, and requests made at the end of K
// see the outputs that the chain made in K - 3 or before.  An operand of a
// step is at least nb steps older than it, so nb >= 5 G suffices; between 4 G
// and 5 G (G is at most nb / 4) the helpers also wait for their stores before
// the barrier, which saves one super-tick.  Networks of two blocks, FP32
// networks of 64 channels (their fragments are single floats: spills, 226
// against 144 ms for 64 10x10 samples), rows wider than the LDS and the calls
// that fast_mw_takes leaves take the one-wave kernel.
//
// Measured (one wave per 16 samples -> this kernel):
//   20x20 depth 24 C64 bf16, 512 samples    204.3 -> 26.6 ms
//   10x10 depth 20 C48 bf16, 1024 / 8192      42 -> 6.3, 59 -> 16.6 ms
//   10x10 depth 20 C32 fp16, 64 / 1024 / 8192  4.7 -> 2.2, 4.8 -> 2.5, 7.4 -> 6.7 ms
//   10x10 depth 20 C32 fp32, 1024 / 8192      43 -> 9.1, 54 -> 19 ms
//   10x10 depth 5 C32 fp16, 64 / 8192       0.96 -> 0.56, 1.67 -> 1.50 ms
// A chain step takes 334 ns (774 cycles) at 16-bit C32 and 793 ns (1907) at C64
// (16 samples of a single row, 60 and 34 sites, depth 20), the issue of one
// wave's instructions.  At two tiles per CU (8192 10x10 samples) the cache's
// traffic beyond L2 bounds it: 36 GB in 6.9 ms, 5.3 TB/s, a copy's rate.
#include "fast_sampler.h"

#include <type_traits>

namespace fk {

template <int PREC, int C>
struct Mw {
  static constexpr bool H16 = Prec<PREC>::H16;
  static constexpr int MT = C / 16, KS = C / Prec<PREC>::KW, MTH = MT / 2;
  static constexpr int LB = fast_lb<PREC, C>(), PB = 64 * LB;
  static constexpr int QB = H16 ? 8 : 16;  // bytes of a lane's quad
  // waves per workgroup, and per SIMD for the register budget
  static constexpr int NW = 4;
  static constexpr int WPE = H16 && C == 32 ? 2 : 1;
  // pixels of the vertical pass that a wave takes together (one read of the
  // weights serves them), and whether a block's vertical weights fit in
  // registers whole
  static constexpr int PV = H16 ? (C == 32 ? 3 : 5) : (C == 32 ? 3 : 2);
  static constexpr bool VW = H16 && C == 32;
  // the same for the row partials
  static constexpr int PP = C == 64 ? 2 : 3;
  // vertical weights: taps in registers at a time (a divisor of 9)
  static constexpr int VT = VW ? 9 : (H16 || C == 32) ? 3 : 1;
  // sets of the chain's weights in registers (requested NS - 1 steps ahead)
  static constexpr int NS = H16 && C == 32 ? 4 : 2;
  // LDS of one step in chunks of 16 bytes a lane: ph and pc (MT each) and the
  // y half for the chain; its outputs, x half and stack value
  static constexpr int YC = MTH * QB > 16 ? MTH * QB / 16 : 1, LC = LB / 16;
  static constexpr int IN = (2 * MT + YC) * 1024, OUT = (YC + LC) * 1024;
};

// Waits for this wave's LDS operations, then for the other waves.  Global
// loads and stores stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
__device__ __forceinline__ void wait_memory() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Pixels before the first buffer: taps reach two rows up and three columns
// left of a buffer's first pixel.
__host__ __device__ inline int mw_pad(int W) { return 2 * W + 3; }

template <int PREC, int C, int ACT>
__global__ __launch_bounds__((64 * Mw<PREC, C>::NW), (Mw<PREC, C>::WPE)) void fast_sample_mw_kernel(SampArgs a, int G, int early) {
  using P = Prec<PREC>;
  using frag = typename P::frag;
  using LD = LaneData<PREC, C>;
  using M = Mw<PREC, C>;
  constexpr int MT = M::MT, KS = M::KS, MTH = M::MTH, LB = M::LB, PB = M::PB, QB = M::QB, NW = M::NW, PV = M::PV;
  const ConvarLayout lay(C, PREC);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int H = a.H, W = a.W, HW = a.HW, nb = a.nb, F = nb - 1;

  // cache of the tile, as in fast_sampler.hip: HW pixels per buffer (two more
  // unused).  Taps outside the lattice are loaded like the others, from
  // whatever lies there (so a row of taps is one scalar offset and constants),
  // and replaced by zeros; mw_pad pixels before the first buffer keep those
  // loads inside the cache.
  uint8_t* base = a.cache + (int64_t)blockIdx.x * a.tile_bytes;
  const int BUF = (HW + 2) * PB;
  constexpr int BUF_FLAGS = 0x00020000;  // raw buffer, 32-bit elements (gfx9)
  const __amdgpu_buffer_rsrc_t rs_w =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.w), (short)0, 0x7fffffff, BUF_FLAGS);
  const __amdgpu_buffer_rsrc_t rs_a =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.aux), (short)0, 0x7fffffff, BUF_FLAGS);
  const __amdgpu_buffer_rsrc_t rs_t =
      __builtin_amdgcn_make_buffer_rsrc(base, (short)0, (int)a.tile_bytes, BUF_FLAGS);
  const uint32_t vl = lane * LB;
  const int pad = mw_pad(W) * PB;
  auto cat_off = [&](int l, int q) { return pad + l * BUF + q * PB; };
  auto ha_off = [&](int l, int q) { return pad + (nb + l - 1) * BUF + q * PB; };
  // the row partials: block l, column c, MT quads per lane (FP32)
  constexpr int RB = MT * 1024;
  auto r_off = [&](int l, int c) { return pad + (3 * nb - 2) * BUF + (l * W + c) * RB; };
  auto va_off = [&](int l, int q) { return pad + (2 * nb - 1 + l - 1) * BUF + q * PB; };
  // Fragment k (a constant) of the convolution that starts at fragment f
  // (uniform), and four values of this lane's group, aux[f + k + 4 g .. + 3].
  // The constant goes into the lane's offset, where it becomes the
  // instruction's immediate: a scalar offset per fragment spilled.
  auto wfrag = [&](int f, int k) {
    constexpr int FB = 64 * (int)sizeof(frag);
    if constexpr (M::H16)
      return __builtin_bit_cast(frag, __builtin_amdgcn_raw_buffer_load_b128(rs_w, lane * 16u + k * FB, f * FB, 0));
    else
      return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_w, lane * 4u + k * FB, f * FB, 0));
  };
  auto ldaux4 = [&](int f, int k) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_a, 16u * g + 4 * k, f * 4, 0));
  };

  // LDS: spins of three rows, block 0's horizontal kernel, uniforms and
  // conditionals of the row (the chain itself reads and writes no memory but
  // its weights), then the steps' entries or, in the vertical pass, two rows of W + 2 pixels
  extern __shared__ __align__(16) uint8_t smem[];
  float* const s_spin = reinterpret_cast<float*>(smem);
  float* const s_kh0 = s_spin + 3 * W * 16;
  double* const s_u = reinterpret_cast<double*>(s_kh0 + 3 * C);  // a row's uniforms,
  f32x2* const s_lp = reinterpret_cast<f32x2*>(s_u + W * 16);    // and log-probabilities
  uint8_t* const s_ring = reinterpret_cast<uint8_t*>(s_lp + W * 16);
  // chunk k of 16 bytes a lane, and the quads m0 .. m0 + MTH of a pixel as
  // one half (x or y) in YC chunks, all of its quads in LC chunks
  auto f4 = [&](uint8_t* p, int k) -> f32x4& { return *reinterpret_cast<f32x4*>(p + k * 1024 + lane * 16); };
  auto get_half = [&](LD& d, int m0, uint8_t* p) {
    if constexpr (M::H16) {
#pragma unroll
      for (int m = 0; m < MTH; ++m) d.q[m0 + m] = *reinterpret_cast<uint2*>(p + lane * 16 + 8 * m);
    } else {
#pragma unroll
      for (int m = 0; m < MTH; ++m) d.q[m0 + m] = f4(p, m);
    }
  };
  auto put_half = [&](const LD& d, int m0, uint8_t* p) {
    if constexpr (M::H16) {
#pragma unroll
      for (int m = 0; m < MTH; ++m) *reinterpret_cast<uint2*>(p + lane * 16 + 8 * m) = d.q[m0 + m];
    } else {
#pragma unroll
      for (int m = 0; m < MTH; ++m) f4(p, m) = d.q[m0 + m];
    }
  };
  auto get_all = [&](LD& d, uint8_t* p) {
    if constexpr (M::H16) {
#pragma unroll
      for (int k = 0; k < M::LC; ++k) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(p + k * 1024 + lane * 16);
        d.q[2 * k] = make_uint2(v.x, v.y);
        d.q[2 * k + 1] = make_uint2(v.z, v.w);
      }
    } else {
#pragma unroll
      for (int k = 0; k < M::LC; ++k) d.q[k] = f4(p, k);
    }
  };
  auto put_all = [&](const LD& d, uint8_t* p) {
    if constexpr (M::H16) {
#pragma unroll
      for (int k = 0; k < M::LC; ++k)
        *reinterpret_cast<u32x4*>(p + k * 1024 + lane * 16) =
            u32x4{d.q[2 * k].x, d.q[2 * k].y, d.q[2 * k + 1].x, d.q[2 * k + 1].y};
    } else {
#pragma unroll
      for (int k = 0; k < M::LC; ++k) f4(p, k) = d.q[k];
    }
  };
  // act(v), rounded as stored
  auto set_act = [&](LD& d, int m, f32x4 v) {
    if constexpr (M::H16) d.q[m] = __builtin_bit_cast(uint2, act_quad<PREC, ACT>(v));
    else d.q[m] = act4<ACT>(v);
  };

  // row 0 of every block's concatenation: y = act(1x1(0) + b) (DownShift
  // zeros)
  for (int l = wave; l <= F; l += NW) {
    LD d{};
#pragma unroll
    for (int m = 0; m < MTH; ++m) set_act(d, MTH + m, ldaux4((int)lay.aux_bias(l), 2 * C + C / 2 + 16 * m));
    for (int j = 0; j < W; ++j) d.bstore_quads(rs_t, vl, cat_off(l, j), MTH, MT);
  }
  for (int k = threadIdx.x; k < 3 * C; k += 64 * NW) s_kh0[k] = a.aux[lay.aux_kh0(nb) + k];
  wait_memory();
  lds_barrier();

  const int S = W * nb;             // steps of a row (even: nb is)
  const int NK = (S + G - 1) / G;   // super-ticks of a row

  // ---- the chain (wave 0)
  // One wave issues an instruction in about 4.6 cycles whatever it is, and
  // with its operands at hand a step is bound by their number: the block kind
  // is the parity of the step, values pass between steps as packed fragments,
  // offsets advance by additions.
  struct CW {  // the chain's weights of one step: tap 2, the 1x1, tap 8
    frag wh[MT][KS], wx[MTH][KS], wc[MT][KS];
    f32x4 xb[MTH];
  };
  constexpr int NS = M::NS;
  const int64_t sample0 = (int64_t)blockIdx.x * 16;
  const bool live = sample0 + n < a.batch;
  const int BLK = (int)lay.blkN, NH = (int)lay.nH, NX = (int)lay.nX;  // fragments
  auto chain_row = [&](int i) {
    // the weights requested next: block wl, whose x1x1 kernel is at fragment
    // wl * BLK; the order is F, 0, 1, .. F - 1, F, ..
    int wl = F, wx = F * BLK;
    auto cw_load = [&](CW& w) {
      const int oh = wx > NH ? wx - NH : 0;  // (block 0 uses none)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) w.wh[m][ks] = wfrag(oh, (2 * MT + m) * KS + ks);
#pragma unroll
      for (int m = 0; m < MTH; ++m) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) w.wx[m][ks] = wfrag(wx, m * KS + ks);
        w.xb[m] = ldaux4(wl * 4 * C, 2 * C + 16 * m);
      }
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) w.wc[m][ks] = wfrag(wx, 2 * NX + (8 * MT + m) * KS + ks);
      const bool wrap = wl == F;
      wx = wrap ? 0 : wx + BLK;
      wl = wrap ? 0 : wl + 1;
    };
    frag wz[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) wz[ks] = wfrag((int)lay.head_base(nb), ks);
    const f32x4 hb = ldq4(a.aux + lay.aux_head_bias(nb));
    const f32x4 zb = g == 0 ? hb : f32x4{0.f, 0.f, 0.f, 0.f};
    LD hcur{}, hres{};  // the stack value after the block before, and two before
    float sv0 = 0.0f, sv1 = 0.0f, sv2 = 0.0f;  // spins of columns j-2, j-1, j
    uint8_t *in = s_ring, *out = s_ring + 2 * G * M::IN;
    int left = G, set = 0, j = 0, l = F;
    auto tick = [&]() {
      in += M::IN;
      out += M::OUT;
      if (--left == 0) {
        left = G;
        set ^= 1;
        if (set == 0) {
          in -= 2 * G * M::IN;
          out -= 2 * G * M::OUT;
        }
        lds_barrier();
      }
    };
    // the part that every step shares: cacc = the 3x3 sums of block l
    auto sums = [&](const CW& w, f32x4 (&hacc)[MT], f32x4 (&cacc)[MT], LD& cur, bool x1x1) {
      LD ax;
#pragma unroll
      for (int m = 0; m < MT; ++m) set_act(ax, m, hacc[m]);
      frag b[KS];
      ax.template frags<KS>(b);
#pragma unroll
      for (int m = 0; m < MTH; ++m) {
        f32x4 x = w.xb[m];
        if (x1x1) {
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) x = P::mfma(w.wx[m][ks], b[ks], x);
        }
        set_act(cur, m, x);
      }
      cur.template frags<KS>(b);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) cacc[m] = P::mfma(w.wc[m][ks], b[ks], cacc[m]);
      put_half(cur, 0, out);
    };
    // a step: ODD ones are block 0 and the second blocks of the residual
    // pairs, the others the conditional (block F) and the first blocks
    auto step = [&](auto odd, const CW& w, CW& wn) {
      constexpr bool ODD = decltype(odd)::value;
      f32x4 hacc[MT], cacc[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) hacc[m] = f4(in, m);
#pragma unroll
      for (int m = 0; m < MT; ++m) cacc[m] = f4(in, MT + m);
      LD cur;
      get_half(cur, MTH, in + 2 * MT * 1024);
      cw_load(wn);
      __builtin_amdgcn_sched_barrier(0);
      if (ODD && l == 0) {
        const float sv[3] = {sv0, sv1, sv2};
#pragma unroll
        for (int t = 0; t < 3; ++t)
#pragma unroll
          for (int m = 0; m < MT; ++m)
            hacc[m] += *reinterpret_cast<const f32x4*>(s_kh0 + t * C + 16 * m + 4 * g) * sv[t];
      } else {
        frag b[KS];
        hcur.template frags<KS>(b);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) hacc[m] = P::mfma(w.wh[m][ks], b[ks], hacc[m]);
      }
      if (!ODD && l == F) {
        // the conditional of site j (a row's first site has nothing to its left)
        sums(w, hacc, cacc, cur, j > 0);
        LD ah;
#pragma unroll
        for (int m = 0; m < MT; ++m) set_act(ah, m, cacc[m]);
        frag b[KS];
        ah.template frags<KS>(b);
        f32x4 z = zb;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) z = P::mfma(wz[ks], b[ks], z);
        float s = 1.0f;
        if (g == 0) {
          const float mx = fmaxf(z.x, z.y);
          const float lse = mx + 0.5f * log1pf(expf(-2.0f * fabsf(z.x - z.y)));
          const float lp0 = 2.0f * (z.x - lse);
          if (live) s = ((double)expf(lp0) > s_u[j * 16 + n]) ? 1.0f : -1.0f;
          s_spin[((i % 3) * W + j) * 16 + n] = s;
          s_lp[j * 16 + n] = f32x2{lp0, 2.0f * (z.y - lse)};
        }
        sv0 = sv1;
        sv1 = sv2;
        sv2 = __shfl(s, n, 64);
        l = 0;
      } else {
        sums(w, hacc, cacc, cur, true);
        // the value the next block sees is the stored (rounded) one
        if (ODD && l > 0) {
#pragma unroll
          for (int m = 0; m < MT; ++m) set_act(hcur, m, hres.get(m) + cacc[m]);
        } else {
          if (!ODD) hres = hcur;
#pragma unroll
          for (int m = 0; m < MT; ++m) set_act(hcur, m, cacc[m]);
        }
        put_all(hcur, out + M::YC * 1024);
        if (++l == F) ++j;
      }
      tick();
    };
    const std::false_type even{};
    const std::true_type odd{};
    CW ws[NS];
#pragma unroll
    for (int k = 0; k < NS - 1; ++k) cw_load(ws[k]);
    lds_barrier();  // super-tick -1
    // (whole turns of the sets, then the rest: a step that may be skipped
    // would make every wait count on its loads not being there)
    int k = 0;
    for (; k + NS <= S; k += NS) {
#pragma unroll
      for (int u = 0; u < NS; u += 2) {
        step(even, ws[u], ws[(u + NS - 1) % NS]);
        step(odd, ws[u + 1], ws[u]);
      }
    }
    if (k < S) {  // (S is even)
      step(even, ws[0], ws[NS - 1]);
      step(odd, ws[1], ws[0]);
    }
    if (left < G) lds_barrier();  // the last, partial super-tick
    lds_barrier();                // super-tick NK
  };

  // ---- helpers (waves 1 .. G)
  struct HItem {  // operands of one step's ph and pc: taps 0, 1 of the 1x3
                  // convolution and 6, 7 of the 3x3, the row partial
    LD px[4], y;
    f32x4 bh[MT], r[MT];
    frag w[4][MT][KS];
  };
  auto load_tap4 = [&](frag (&w)[MT][KS], int l, int k) {  // tap k of the four
    const int o = k >= 2 ? (int)lay.off_c(l) : l > 0 ? (int)lay.off_h(l) : 0;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) w[m][ks] = wfrag(o, ((k < 2 ? k : k + 4) * MT + m) * KS + ks);
  };
  auto helper_row = [&](int i) {
    const int h = wave - 1;  // this helper's step of each super-tick
    for (int k = h * 64 + lane; k < W * 16; k += 64 * (NW - 1)) {
      const int64_t b = sample0 + k % 16;
      s_u[k] = b < a.batch ? a.uniforms[b * HW + i * W + k / 16] : 0.0;
    }
    if (h >= G) {
      for (int K = -1; K <= NK; ++K) lds_barrier();
      return;
    }
    // A step of this helper: site j, r-th of its nb steps (r = 0: block F,
    // else block r - 1); advanced by G steps a super-tick.
    struct Step {
      int j, r;
    };
    auto advance = [&](Step& t) {
      t.r += G;
      if (t.r >= nb) {
        t.r -= nb;
        ++t.j;
      }
    };
    auto block = [&](const Step& t) { return t.r == 0 ? F : t.r - 1; };
    auto request = [&](HItem& x, const Step& t) {  // all but the weights
      const int j = t.j, l = block(t);
      const int ab = (int)lay.aux_bias(l), rs = r_off(l, j);
#pragma unroll
      for (int m = 0; m < MT; ++m) x.bh[m] = ldaux4(ab, C + 16 * m);
      if (i > 0) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
          x.r[m] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_t, lane * 16u + 1024 * m, rs, 0));
      } else {  // nothing above: the bias
#pragma unroll
        for (int m = 0; m < MT; ++m) x.r[m] = ldaux4(ab, 3 * C + 16 * m);
      }
      // the masked final block's 1x3 taps end one column to the left
      const int hs = l > 0 ? ha_off(l, i * W + (l == F ? j - 3 : j - 2)) : pad, cs = cat_off(l, i * W + j - 2);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        x.px[k].bload(rs_t, vl + k * PB, hs);
        x.px[2 + k].bload(rs_t, vl + k * PB, cs);
      }
      x.y.bload_quads(rs_t, vl + 2 * PB, cs, MTH, MT);
    };
    // (ln: the block whose weights are requested as this one's are used)
    auto make = [&](HItem& x, const Step& t, int ln, uint8_t* in) {
      const int j = t.j, l = block(t);
      if (j < 3) {  // taps to the left of the lattice
        const int h0 = l == F ? j - 3 : j - 2;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          if (h0 + k < 0) x.px[k] = LD{};
          if (j - 2 + k < 0) x.px[2 + k] = LD{};
        }
      }
      f32x4 acc[2][MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        acc[0][m] = x.bh[m];
        acc[1][m] = x.r[m];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (k >= 2 || l > 0) {  // (block 0: the chain adds the spins' taps)
          frag b[KS];
          x.px[k].template frags<KS>(b);
#pragma unroll
          for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) acc[k >= 2][m] = P::mfma(x.w[k][m][ks], b[ks], acc[k >= 2][m]);
        }
        load_tap4(x.w[k], ln, k);
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        f4(in, m) = acc[0][m];
        f4(in, MT + m) = acc[1][m];
      }
      put_half(x.y, MTH, in + 2 * MT * 1024);
    };
    auto flush = [&](const Step& t, uint8_t* out) {
      const int l = block(t), q = i * W + t.j;
      LD d;
      get_half(d, 0, out);
      d.bstore_quads(rs_t, vl, cat_off(l, q), 0, MTH);
      if (l < F) {
        get_all(d, out + M::YC * 1024);
        d.bstore(rs_t, vl, ha_off(l + 1, q));
      }
    };
    HItem x;
    Step tr{0, h}, tm{0, h}, tf{0, h};  // requested next, made next, stored next
    if (h < S) {
#pragma unroll
      for (int k = 0; k < 4; ++k) load_tap4(x.w[k], block(tr), k);
      request(x, tr);
    }
    for (int K = -1; K <= NK; ++K) {
      wait_memory();
      const int set = (K + 1) & 1;
      if (K >= 1) {
        if (tf.j < W) flush(tf, s_ring + 2 * G * M::IN + (set * G + h) * M::OUT);
        advance(tf);
      }
      advance(tr);
      if (tm.j < W) make(x, tm, block(tr), s_ring + (set * G + h) * M::IN);
      advance(tm);
      if (early) wait_memory();
      if (tr.j < W) request(x, tr);
      lds_barrier();
    }
  };

  // ---- row partials of row i + 1 (all waves): bias + taps 0..5 of every
  // block's 3x3 convolution, the taps that read rows i - 1 and i.  A wave
  // takes whole blocks, so a block's weights are read once a row, not once a
  // site; per step the helpers then read four taps' weights instead of ten
  // (per CU 64 B a cycle of them come through L1, which bounds a step).
  auto partials_row = [&](int i) {
    constexpr int PP = M::PP;
    struct Px {  // pixels of a group: rows i - 1, i, columns c0 - 2 .. c0 + PP - 1
      LD p[2][PP + 2];
    };
    frag w[6][MT][KS];
    f32x4 bc[MT];
    auto load_px = [&](Px& x, int l, int c0, int r) {
      const int cs = cat_off(l, (i - 1 + r) * W + c0 - 2);
#pragma unroll
      for (int k = 0; k < PP + 2; ++k) x.p[r][k].bload(rs_t, vl + k * PB, cs);
    };
    auto load_tap = [&](int l, int t) {
      const int oc = l * BLK;
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) w[t][m][ks] = wfrag(oc, 2 * NX + (t * MT + m) * KS + ks);
    };
    auto load_bias = [&](int l) {
#pragma unroll
      for (int m = 0; m < MT; ++m) bc[m] = ldaux4(l * 4 * C, 3 * C + 16 * m);
    };
    // groups in the order (block, column); the requests run two groups ahead
    int ql = wave, qc = 0;  // requested next
    auto next = [&](int& l, int& c0) {
      c0 += PP;
      if (c0 >= W) {
        c0 = 0;
        l = l + NW <= F ? l + NW : l;  // (past the last block: its first group again)
      }
    };
    int l = wave, c0 = 0;
    auto group = [&](Px& x) {
      const bool more = c0 + PP < W;
      if (i < 1 || c0 < 2) {  // taps outside the lattice
#pragma unroll
        for (int k = 0; k < PP + 2; ++k) {
          if (i < 1 || c0 - 2 + k < 0) x.p[0][k] = LD{};
          if (c0 - 2 + k < 0) x.p[1][k] = LD{};
        }
      }
      f32x4 acc[PP][MT];
#pragma unroll
      for (int u = 0; u < PP; ++u)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[u][m] = bc[m];
      const int ln = more || l + NW > F ? l : l + NW;
#pragma unroll
      for (int t = 0; t < 6; ++t) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int u = 0; u < PP; ++u) {
            frag b[KS];
            x.p[t / 3][u + t % 3].template frags<KS>(b);
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[u][m] = P::mfma(w[t][m][ks], b[ks], acc[u][m]);
          }
        if (!more) load_tap(ln, t);
        if (t % 3 == 2) load_px(x, ql, qc, t / 3);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (!more) load_bias(ln);
      next(ql, qc);
      const int rs = r_off(l, c0);
#pragma unroll
      for (int u = 0; u < PP; ++u) {
        if (c0 + u >= W) break;
#pragma unroll
        for (int m = 0; m < MT; ++m)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[u][m]), rs_t,
                                                 lane * 16u + 1024 * m + RB * u, rs, 0);
      }
      c0 += PP;
      if (c0 >= W) {
        c0 = 0;
        l += NW;
      }
    };
    if (wave > F) return;
    Px A, B;
    load_px(A, ql, qc, 0);
    load_px(A, ql, qc, 1);
    next(ql, qc);
    load_px(B, ql, qc, 0);
    load_px(B, ql, qc, 1);
    next(ql, qc);
#pragma unroll
    for (int t = 0; t < 6; ++t) load_tap(wave, t);
    load_bias(wave);
    const int groups = ((F - wave) / NW + 1) * ((W + PP - 1) / PP);
    for (int k = 0; k + 2 <= groups; k += 2) {
      group(A);
      group(B);
    }
    if (groups & 1) group(A);
  };

  // ---- vertical stack of row i (all waves): every block's row, pixels in
  // groups of PV over the waves
  auto vertical_row = [&](int i) {
    auto vbuf = [&](int which, int c) { return s_ring + (which * (W + 2) + c + 1) * PB; };  // column c, -1 .. W
    if (wave < 2) {
      put_all(LD{}, vbuf(wave, -1));
      put_all(LD{}, vbuf(wave, W));
    }
    struct VPre {  // operands of a block that do not come from this row
      LD up[2][PV + 2];
      frag w[M::VT][MT][KS], wy[MTH][KS];
      f32x4 bv[MT], by[MTH];
    };
    auto load_up = [&](VPre& v, int l, int c0, int r) {  // row i - 2 + r
      const int vs = va_off(l, (i - 2 + r) * W + c0 - 1);
#pragma unroll
      for (int k = 0; k < PV + 2; ++k) v.up[r][k].bload(rs_t, vl + k * PB, vs);
    };
    auto load_tap = [&](frag (&w)[MT][KS], int l, int t) {
      const int ov = (int)lay.off_v(l);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) w[m][ks] = wfrag(ov, (t * MT + m) * KS + ks);
    };
    auto load_rest = [&](VPre& v, int l) {
      const int ab = (int)lay.aux_bias(l), oy = (int)lay.off_y(l);
#pragma unroll
      for (int m = 0; m < MT; ++m) v.bv[m] = ldaux4(ab, 16 * m);
#pragma unroll
      for (int m = 0; m < MTH; ++m) {
        v.by[m] = ldaux4(ab, 2 * C + C / 2 + 16 * m);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) v.wy[m][ks] = wfrag(oy, m * KS + ks);
      }
    };
    // the epilogue of a group: pixels c0 .. of block l from their sums
    auto finish = [&](const VPre& v, const f32x4 (&acc)[PV][MT], int l, int c0) {
      const int kind = block_kind(l, nb);
      const int vs = l < F ? va_off(l + 1, i * W + c0) : 0, ys = cat_off(l, (i + 1) * W + c0);
#pragma unroll
      for (int u = 0; u < PV; ++u) {
        const int c = c0 + u;
        if (c >= W) break;
        LD av;
#pragma unroll
        for (int m = 0; m < MT; ++m) set_act(av, m, acc[u][m]);
        if (l < F) {
          uint8_t* const o = vbuf((l + 1) & 1, c);
          LD vn = av;
          if (kind == BK_B) {
            LD vr;  // the input of the block before, which this pixel's output replaces
            get_all(vr, o);
#pragma unroll
            for (int m = 0; m < MT; ++m) set_act(vn, m, vr.get(m) + acc[u][m]);
          }
          put_all(vn, o);
          vn.bstore(rs_t, vl + u * PB, vs);
        }
        frag b[KS];
        av.template frags<KS>(b);
        LD yd;
#pragma unroll
        for (int m = 0; m < MTH; ++m) {
          f32x4 y = v.by[m];
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) y = P::mfma(v.wy[m][ks], b[ks], y);
          set_act(yd, MTH + m, y);
        }
        yd.bstore_quads(rs_t, vl + u * PB, ys, MTH, MT);
      }
    };
    const int first = wave * PV;
    VPre v;
    // block 0: its input is the spins
    load_rest(v, 0);
    for (int c0 = first; c0 < W; c0 += NW * PV) {
      f32x4 acc[PV][MT];
#pragma unroll
      for (int u = 0; u < PV; ++u)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[u][m] = v.bv[m];
#pragma unroll 1
      for (int t = 0; t < 9; ++t) {
        const int r = i + t / 3 - 2;
        f32x4 k[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) k[m] = ldaux4((int)lay.aux_kv0(nb) + t * C, 16 * m);
#pragma unroll
        for (int u = 0; u < PV; ++u) {
          const int c = c0 + u + t % 3 - 1;
          const float sv = r >= 0 && c >= 0 && c < W ? s_spin[((r % 3) * W + c) * 16 + n] : 0.0f;
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[u][m] += k[m] * sv;
        }
      }
      finish(v, acc, 0, c0);
    }
    // Blocks 1 .. F as one sequence of groups (l, c0).  The next group's
    // operands are requested as this one's registers become free: a tap's
    // weights after its products, a row's pixels after its last tap.
    if (first < W) {
#pragma unroll
      for (int t = 0; t < M::VT; ++t) load_tap(v.w[t], 1, t);
      load_up(v, 1, first, 0);
      load_up(v, 1, first, 1);
      load_rest(v, 1);
    }
    lds_barrier();
    for (int l = 1; l <= F; ++l) {
      for (int c0 = first; c0 < W; c0 += NW * PV) {
        const bool more = c0 + NW * PV < W;
        const int ln = more || l == F ? l : l + 1, cn = more ? c0 + NW * PV : first;
        if (i < 2 || c0 == 0 || c0 + PV >= W) {  // taps outside the lattice
#pragma unroll
          for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int k = 0; k < PV + 2; ++k)
              if (i - 2 + r < 0 || c0 - 1 + k < 0 || c0 - 1 + k >= W) v.up[r][k] = LD{};
        }
        f32x4 acc[PV][MT];
#pragma unroll
        for (int u = 0; u < PV; ++u)
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[u][m] = v.bv[m];
        LD row[PV + 2];
#pragma unroll
        for (int t = 0; t < 9; ++t) {
          if (t == 6) {
#pragma unroll
            for (int k = 0; k < PV + 2; ++k) get_all(row[k], vbuf(l & 1, c0 - 1 + k < W ? c0 - 1 + k : W));
          }
          frag(&w)[MT][KS] = v.w[t % M::VT];
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int u = 0; u < PV; ++u) {
              frag b[KS];
              (t / 3 == 2 ? row[u + t % 3] : v.up[t / 3 == 2 ? 0 : t / 3][u + t % 3]).template frags<KS>(b);
#pragma unroll
              for (int m = 0; m < MT; ++m) acc[u][m] = P::mfma(w[m][ks], b[ks], acc[u][m]);
            }
          load_tap(w, t + M::VT < 9 ? l : ln, (t + M::VT) % 9);
          // (the row's own pixels take the registers of row i - 1's)
          if (t == 2 || t == 8) load_up(v, ln, cn, t / 6);
          __builtin_amdgcn_sched_barrier(0);
        }
        finish(v, acc, l, c0);
        load_rest(v, ln);
      }
      lds_barrier();
    }
    wait_memory();
    lds_barrier();
  };

  for (int i = 0; i < H; ++i) {
    if (wave == 0) chain_row(i);
    else helper_row(i);
    for (int k = threadIdx.x; k < W * 16; k += 64 * NW) {
      const int64_t b = sample0 + k / W;
      const int j = k % W;
      if (b < a.batch) {
        a.out[b * HW + i * W + j] = (int8_t)s_spin[((i % 3) * W + j) * 16 + k / W];
        if (a.cond) *reinterpret_cast<f32x2*>(a.cond + (b * HW + i * W + j) * 2) = s_lp[j * 16 + k / W];
      }
    }
    // (after the last row nothing reads what these make)
    if (i + 1 < H) {
      wait_memory();
      lds_barrier();
      partials_row(i);
      vertical_row(i);
    }
  }
}

// Steps per super-tick: one per helper, a quarter of the blocks at most, and
// what the LDS holds.
constexpr int MW_LDS = 160 * 1024;

template <int PREC, int C>
static int mw_lds(int W, int G) {
  using M = Mw<PREC, C>;
  const int ring = 2 * G * (M::IN + M::OUT), rows = 2 * (W + 2) * M::PB;
  return W * 16 * (3 * 4 + 8 + 8) + 3 * C * 4 + (ring > rows ? ring : rows);
}
template <int PREC, int C>
static int mw_steps(int W, int nb) {
  int G = Mw<PREC, C>::NW - 1;
  if (G > nb / 4) G = nb / 4;
  while (G > 0 && mw_lds<PREC, C>(W, G) > MW_LDS) --G;
  return G;
}

template <int PREC>
static int mw_steps_c(int W, int nb, int channels) {
  if (channels == 32) return mw_steps<PREC, 32>(W, nb);
  // (FP32 at 64 channels: its fragments are single floats, which spill)
  if constexpr (PREC != FK_PREC_FP32)
    if (channels == 64) return mw_steps<PREC, 64>(W, nb);
  return 0;
}

int64_t fast_mw_tile_bytes(int H, int W, int nb, int channels, int precision) {
  const int64_t pb = 16LL * channels * (precision == FK_PREC_FP32 ? 4 : 2);
  return ((int64_t)(3 * nb - 2) * ((int64_t)H * W + 2) + mw_pad(W)) * pb + (int64_t)nb * W * channels * 64;
}

// Steps per super-tick of a network that the kernel can take, or 0.
static int mw_steps_of(int H, int W, int nb, int channels, int precision) {
  // (the cache of a tile is addressed by 32-bit offsets)
  if (fast_mw_tile_bytes(H, W, nb, channels, precision) >= 0x7fffffff) return 0;
  return precision == FK_PREC_FP32   ? mw_steps_c<FK_PREC_FP32>(W, nb, channels)
         : precision == FK_PREC_BF16 ? mw_steps_c<FK_PREC_BF16>(W, nb, channels)
                                     : mw_steps_c<FK_PREC_FP16>(W, nb, channels);
}

bool fast_mw_supported(int H, int W, int nb, int channels, int precision) {
  return mw_steps_of(H, W, nb, channels, precision) > 0;
}

// Rounds of workgroups over the chip (one per CU) up to which this kernel is
// the faster one at 16-bit 64 channels and FP32.  Its waves share a tile, so it
// needs rows that they can divide and blocks for its helpers (steps: helpers
// that run; one of three for networks of four and six blocks); the one-wave
// kernel runs several tiles a CU instead, as soon as there are as many.  Time of
// this kernel over the other's, six rows, by rounds 1 / 2 / 4 / 8, depth 3 (one
// step) and depth 5 (two):
//   64 channels, W = 1   1.57 / 2.4 / 4.0 / 5.7    1.36 / 1.8 / 3.4 / 4.0
//                W = 3   0.66 / 0.86 / 1.6 / 2.0   0.45 / 0.66 / 0.96 / 1.3
//                W = 5   -    / 0.64 / 1.1 / 1.3   -    / 0.45 / 0.71 / 0.93
//                W = 10  -    / 0.49 / 0.81 / 1.0  -    / 0.36 / 0.61 / 0.72
//   FP32, 32     W = 1   2.0 / 3.4 / 5.4 / 7.8     1.9 / 2.7 / 5.2 / 6.1
//                W = 3   0.73 / 1.1 / 2.1 / 2.4    0.57 / 0.86 / 1.4 / 1.7
//                W = 5   -    / 0.86 / 1.4 / 1.7   -    / 0.60 / 0.98 / 1.2
//                W = 10  -    / 0.68 / 1.1 / 1.3   -    / 0.45 / 0.74 / 0.88
// (A single row has no vertical stack to divide; two rows have little of it.)
static int mw_rounds(int H, int W, int steps, int precision) {
  constexpr int ANY = 0x7fffffff;
  if (H == 1) W = 7;
  if (precision == FK_PREC_FP32) {
    if (steps == 1) return W <= 2 ? 0 : W == 3 ? 1 : W < 8 ? 2 : 3;
    return W < 5 ? W - 1 : W < 7 ? 4 : ANY;
  }
  if (steps == 1) return W <= 2 ? W - 1 : W < 5 ? 2 : W == 5 || H < 3 ? 3 : W < 10 || H < 6 ? 4 : ANY;
  return W <= 2 ? 2 * (W - 1) : W < 5 ? 4 : ANY;
}

bool fast_mw_takes(int H, int W, int nb, int channels, int precision, int64_t tiles) {
  const int steps = mw_steps_of(H, W, nb, channels, precision);
  if (steps == 0) return false;
  const int64_t cu = device_cu_count();
  // 16-bit 32 channels (two workgroups a CU): all but four-block networks on
  // narrow or two rows, which one wave draws faster once there is a second round,
  // or a third (4x4, 6x6, 8x8, 32768 samples: 544 against 449 us, 1101 and 992,
  // 1937 and 1838; 8x8, 16384: 977 and 1145; not 3x3, 282 and 315)
  if (precision != FK_PREC_FP32 && channels == 32) {
    const bool narrow = W <= 6 || H == 2;
    return !(nb == 4 && H > 1 && H * W >= 12 && (narrow || W <= 8) && tiles > (narrow ? 2 : 4) * cu);
  }
  return (tiles + cu - 1) / cu <= mw_rounds(H, W, steps, precision);
}

template <int PREC, int C>
static int launch_mw(const SampArgs& a, int act, int64_t tiles, hipStream_t s) {
  const int G = mw_steps<PREC, C>(a.W, a.nb);
  const int lds = mw_lds<PREC, C>(a.W, G);
  auto k = act == FK_ACT_ELU ? fast_sample_mw_kernel<PREC, C, FK_ACT_ELU> : fast_sample_mw_kernel<PREC, C, FK_ACT_RELU>;
  FK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  hipLaunchKernelGGL(k, dim3((unsigned)tiles), dim3(64 * Mw<PREC, C>::NW), lds, s, a, G, a.nb < 5 * G ? 1 : 0);
  FK_CHECK_LAUNCH();
  return FK_OK;
}

int launch_fast_mw(const SampArgs& a, int channels, int precision, int act, int64_t tiles, hipStream_t s) {
  if (precision == FK_PREC_BF16)
    return channels == 32 ? launch_mw<FK_PREC_BF16, 32>(a, act, tiles, s) : launch_mw<FK_PREC_BF16, 64>(a, act, tiles, s);
  if (precision == FK_PREC_FP16)
    return channels == 32 ? launch_mw<FK_PREC_FP16, 32>(a, act, tiles, s) : launch_mw<FK_PREC_FP16, 64>(a, act, tiles, s);
  return launch_mw<FK_PREC_FP32, 32>(a, act, tiles, s);
}

}  // namespace fk
