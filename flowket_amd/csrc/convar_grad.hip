// Gradients of log psi of ConvNetAutoregressive2D (32 and 64 channels): the
// per-sample rows O_k, their batched adjoint product (VJP) and forward mode
// (JVP), FP32 MFMA.  Same quantities as convar_bwd.hip, which keeps the other
// channel counts and what grad_plan leaves it.
//
// One workgroup per sample at a time, its waves sharing every phase.  A block
// of the network is two phases, forward and backward, with one barrier each:
//   forward  VH: the vertical and horizontal convolutions; the 1x1s continue
//                in registers (a D fragment of 16 pixels is the B operand of
//                the next contraction) and write the concatenation
//            C:  the 3x3 over it
//   backward C:  its weight and data gradients; the 1x1s' data gradients
//                continue in registers
//            VH: the weight gradients of the 1x1s and of the V and H
//                convolutions, and their data gradients
// The activations' derivatives, biases and residuals run in the epilogues.
// Five tensors of the sample (HW x C, FP32) are live in either direction, eight
// in the JVP; when they fit they stay in LDS (RES: up to 192 pixels at C 32, 108
// at C 64; JVP 127 and 67), with rows of C + 4 floats (the 16 pixels of a tile
// then start 36 or 68 banks apart) and a zero pixel that taps outside the lattice
// read.  The activations that the backward needs go to the
// workgroup's workspace.  Larger lattices keep all tensors there (L2).
//
// The bound is the matrix cores (FP32 MFMA, 32 cycles each), of which a phase
// keeps about half busy: the rest is the operands' and the epilogues' latency
// at its ends and units that do not divide evenly over the waves.  Hence few
// phases, epilogues that request everything before they store anything, packed
// weights, and requests between the MFMAs of the step before.  With a phase
// per convolution and one elementwise pass per derivative (13 barriers a
// block, four waves) the matrix cores were busy a quarter of the time.
// Measured, VJP / JVP / O in ms, convar_bwd.hip -> here: 10x10 depth 20 C 32, 64
// samples 5.86 / 3.81 / 9.21 -> 1.87 / 1.43 / 3.06, 2048 samples 25.2 / 19.6 /
// 36.1 -> 15.7 / 11.4 / 24.8; 20x20 depth 24 C 64, 128 samples 88.6 / 56.3 /
// 155.9 -> 27.6 / 22.5 / 45.2, 512 samples 141 / 100 / 238 -> 56.6 / 45.5 / 92.2;
// 4x4 depth 5 C 32, 1024 samples 1.55 / 0.64 / 1.23 -> 0.72 / 0.20 / 0.72.
#include "convar_bwd.h"

namespace fk {

namespace {

struct Lane {
  int l16, kk;  // this lane's column and contraction group (lane l16 + 16 kk)
  // (opaque: what follows from it is computed where it is used, not kept in
  // registers over the whole kernel)
  __device__ __forceinline__ Lane() : l16(threadIdx.x & 15), kk((threadIdx.x >> 4) & 3) {
    asm volatile("" : "+v"(l16), "+v"(kk));
  }
};

// The units of a phase are one list, taken by the waves from a counter in LDS:
// a wave's first unit is its number, the next come from the counter, so waves
// that drew short units take more.  Which wave computes a unit does not change
// it: results are deterministic.
struct Work {
  int* q;  // 4 counters, one per phase (modulo 4)
  int phase, cur;
  __device__ __forceinline__ void begin() {  // after a barrier
    ++phase;
    if (threadIdx.x == 0) q[(phase + 2) & 3] = 0;  // (last used two barriers ago)
    cur = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  }
  __device__ __forceinline__ void next() {
    int v = 0;
    if ((threadIdx.x & 63) == 0) v = atomicAdd(q + (phase & 3), 1);
    cur = (int)(blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(v);
  }
};

// The kernels are read packed (pack_kernels_kernel): the A operand of a
// (tap, tile, quad) is 1 KB in the order of the lanes.  The vector cache moves
// a line of adjacent lanes a cycle; read from rows of C floats, where adjacent
// lanes lie in different rows, a 16-byte load took 64 cycles instead of 16,
// and the cache's pipe was full (VJP of 2048 10x10 samples 18.3 ms, packed
// 16.8).  The tensors in the workspace are [C/4][HW][4] for the same reason.
//
// acc[n][m] += sum over taps and input channels of A[16 (m0 + m) + ..][k]
// B[k][pixel of tile n]: ka is tile m0's first packed weight, ts the floats of
// a tap, LDK the contraction's length.  The contraction runs in quads (quad j
// of lane group kk: indices 16 j + 4 kk + r, feeding four MFMAs); a step is QS
// quads of one tap, and a step's operands are requested a step ahead, a tap's
// source pixels (fp) two steps ahead.  TAN: the derivative along (tangent
// weights kt, tangent input fbt) goes to tac.
// The requests are dealt out between the MFMAs of the step before: a wave
// issues them in the 32 cycles that the matrix core needs for each.
template <int VM, int DS, int MF>
__device__ __forceinline__ void interleave() {
  constexpr int N = VM + DS, PER = MF / (N + 1) > 0 ? MF / (N + 1) : 1;
#pragma unroll
  for (int i = 0; i < N && i * PER < MF; ++i) {
    if (i < VM) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    else __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
}
template <int LDK, int MG, int NN, int QS, bool RES, bool TAN, class FP, class FB, class FBT, class FH>
__device__ __forceinline__ void conv_acc(f32x4 (&acc)[NN][MG], f32x4 (&tac)[TAN ? NN : 1][TAN ? MG : 1],
                                         const float* ka, const float* kt, int ntap, int ts, FP fp, FB fb, FBT fbt,
                                         FH has) {
  constexpr int KQ = LDK / 16, PT = KQ / QS;
  const unsigned lo = 4 * (threadIdx.x & 63);
  struct Ops {
    f32x4 a[QS][MG], b[QS][NN];
    f32x4 at[TAN ? QS : 1][TAN ? MG : 1], bt[TAN ? QS : 1][TAN ? NN : 1];
    bool ok[NN];  // (applied at the use: nothing waits for a load where it is requested)
  };
  int tap = 0, part = 0;
  int src[NN];
#pragma unroll
  for (int n = 0; n < NN; ++n) src[n] = fp(n, 0);
  auto request = [&](Ops& o) {
    const int ko = tap * ts + part * (256 * QS);
#pragma unroll
    for (int n = 0; n < NN; ++n) o.ok[n] = has(src[n]);
#pragma unroll
    for (int q = 0; q < QS; ++q) {
#pragma unroll
      for (int m = 0; m < MG; ++m) {
        o.a[q][m] = *reinterpret_cast<const f32x4*>(ka + ko + (m * KQ + q) * 256 + lo);
        if constexpr (TAN) o.at[q][m] = *reinterpret_cast<const f32x4*>(kt + ko + (m * KQ + q) * 256 + lo);
      }
#pragma unroll
      for (int n = 0; n < NN; ++n) {
        o.b[q][n] = fb(src[n], part * QS + q);
        if constexpr (TAN) o.bt[q][n] = fbt(src[n], part * QS + q);
      }
    }
    if (++part == PT) {
      part = 0;
      if (tap + 1 < ntap) ++tap;  // (past the last step: it again, unused)
#pragma unroll
      for (int n = 0; n < NN; ++n) src[n] = fp(n, tap);
    }
  };
  auto compute = [&](const Ops& o) {
#pragma unroll
    for (int q = 0; q < QS; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int n = 0; n < NN; ++n) {
          const float b = o.ok[n] ? o.b[q][n][r] : 0.0f;
          float bt = 0.0f;
          if constexpr (TAN) bt = o.ok[n] ? o.bt[q][n][r] : 0.0f;
#pragma unroll
          for (int m = 0; m < MG; ++m) {
            acc[n][m] = mfma4(o.a[q][m][r], b, acc[n][m]);
            if constexpr (TAN) {
              tac[n][m] = mfma4(o.a[q][m][r], bt, tac[n][m]);
              tac[n][m] = mfma4(o.at[q][m][r], b, tac[n][m]);
            }
          }
        }
  };
  Ops A, B;
  request(A);
  constexpr int T = TAN ? 2 : 1, VM = QS * T * (MG + (RES ? 0 : NN)), DS = NN + (RES ? QS * T * NN : 0),
                MF = 4 * QS * NN * MG * (TAN ? 3 : 1);
  int steps = ntap * PT, k = 0;
  asm volatile("" : "+s"(steps));  // (one copy of the loop)
#pragma unroll 1
  for (; k + 2 <= steps; k += 2) {
    __builtin_amdgcn_sched_barrier(0);
    request(B);
    compute(A);
    interleave<VM, DS, MF>();
    request(A);
    compute(B);
    interleave<VM, DS, MF>();
  }
  if (k < steps) compute(A);
}

template <int C_, bool RES_, int NT_>
struct Shape {
  static constexpr int C = C_, NT = NT_, MT = C / 16;
  static constexpr bool RES = RES_;
  static constexpr int SG = RES ? C + 4 : C;               // floats between pixels of the live tensors
  // pixel tiles of a unit: as many as the registers hold (128 a lane with 1024
  // threads, 256 else), and one where a lattice may have no more
  static constexpr int NN = NT == 128 || NT == 1024 ? 1 : RES || C == 32 ? 2 : 4;
  static constexpr int QS = C == 32 ? 2 : 1;
  static constexpr int WM = NT == 1024 ? 2 : MT;  // tiles of a weight gradient's unit, each way
};

__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ void st4(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }

// Taps' source pixels of every pixel, forward rows (GT_N) then the inverse of
// the first GT_X; HW where there is none, and for the pixels that fill the
// last tiles (a row has table_row entries).
__host__ __device__ inline int table_row(int HW) { return (HW + 63) / 64 * 64; }
__device__ void build_tables(int16_t* ftab, int16_t* itab, int H, int W) {
  const int HW = H * W, HP = table_row(HW);
  for (int idx = threadIdx.x; idx < GT_N * HP; idx += blockDim.x) {
    const int row = idx / HP, p = idx - row * HP;
    const int i = p / W, j = p - (p / W) * W;
    int dr = 0, dc = 0;
    if (row < GT_H) tap_rc(0, row - GT_V, dr, dc);
    else if (row < GT_C) tap_rc(1, row - GT_H, dr, dc);
    else if (row < GT_X) tap_rc(2, row - GT_C, dr, dc);
    else if (row == GT_XF) dc = -1;
    else if (row == GT_Y) dr = -1;
    const int r = i + dr, c = j + dc;
    ftab[idx] = (p < HW && r >= 0 && r < H && c >= 0 && c < W) ? (int16_t)(r * W + c) : (int16_t)HW;
    if (row < GT_X) {
      const int ri = i - dr, ci = j - dc;
      itab[idx] = (p < HW && ri >= 0 && ri < H && ci >= 0 && ci < W) ? (int16_t)(ri * W + ci) : (int16_t)HW;
    }
  }
  __syncthreads();
}

// Everything a sample's passes share.
template <class S>
struct Ctx {
  static constexpr int C = S::C;
  static constexpr bool RES = S::RES;
  const float *prm, *kt, *kb, *tan, *tkt;  // parameters; packed for the forward, the backward; tangents
  float *ws, *wt;        // workspace, and its tangent half
  const float* spins;    // HW, in the workspace
  const int16_t *ftab, *itab;
  float* lds;            // RES: the tiles
  int H, W, HW, HP, nb;
  __device__ __forceinline__ float* tile(int k) const { return lds + k * (HW + 1) * S::SG; }
  // source pixel of this lane's pixel p through a table row
  __device__ __forceinline__ int src(const int16_t* tab, int row, int p) const {
    return tab[row * HP + p];
  }
  // channel c of pixel p in the workspace's tensors and in the live ones
  __device__ __forceinline__ unsigned gat(int p, int c) const { return ((c >> 2) * HW + p) * 4 + (c & 3); }
  __device__ __forceinline__ unsigned at(int p, int c) const { return RES ? p * S::SG + c : gat(p, c); }
  // 16 bytes of pixel s of a live tensor; for s == HW the zeros of the zero
  // pixel (RES), or anything
  __device__ __forceinline__ f32x4 px(const float* t, int s, int off) const {
    if constexpr (RES) return ld4(t + s * S::SG + off);
    return ld4(t + gat(s < HW ? s : 0, off));
  }
  __device__ __forceinline__ bool has(int s) const { return RES || s < HW; }
};

// Forward of one sample; TAN: with the tangent of every tensor.  The live
// tensors: V (ping-pong with the dead V's place taken by the concatenation),
// H.  RES: tiles 0, 1 (V, V' / CAT), 2 (CAT / V), 3 (H), tangents 4..7.  Not
// RES: the workspace's own tensors.  Without TAN every block's VA, XA, CAT,
// VO, HO are stored for the backward.
template <class S, int ACT, bool TAN>
__device__ __forceinline__ void forward(Work& wk, const Ctx<S>& x) {
  constexpr int C = S::C, MT = S::MT, SG = S::SG, NN = TAN ? 1 : S::NN, QS = TAN ? 1 : S::QS;
  constexpr bool RES = S::RES;
  constexpr int MG = RES ? MT / 2 : MT;  // tiles per unit of the 3x3 (no chain follows it)
  const int HW = x.HW, W = x.W, F = x.nb - 1;
  const int ntl = (HW + 15) / 16, NU = (ntl + NN - 1) / NN;
  auto tens = [&](int blk, int which) { return ws_tensor(x.ws, HW, C, blk, which); };
  auto ttens = [&](int blk, int which) { return ws_tensor(x.wt, HW, C, blk, which); };
  for (int blk = 0; blk <= F; ++blk) {
    const ParamOffsets o = param_offsets(blk, C);
    const bool first = blk == 0, fin = blk == F;
    const bool kb = !first && !fin && ((blk & 1) == 0);
    // RES: V of block blk in tile (blk & 1) * 2, its output and the
    // concatenation in the other two of 0, 1, 2
    const int tv = (blk & 1) ? 1 : 0, to = (blk & 1) ? 0 : 1;
    const float* V = RES ? x.tile(tv) : first ? nullptr : tens(blk - 1, T_VO);
    const float* Hh = RES ? x.tile(3) : first ? nullptr : tens(blk - 1, T_HO);
    const float* Vd = !TAN ? nullptr : RES ? x.tile(4 + tv) : first ? nullptr : ttens(blk - 1, T_VO);
    const float* Hd = !TAN ? nullptr : RES ? x.tile(7) : first ? nullptr : ttens(blk - 1, T_HO);
    float* cat = RES ? x.tile(2) : tens(blk, T_CAT);
    float* catd = !TAN ? nullptr : RES ? x.tile(6) : ttens(blk, T_CAT);
    float* gCAT = tens(blk, T_CAT);
    // the concatenation's channels off .. off + C/2 of pixel p
    auto put_cat = [&](int p, int co, f32x4 v) {
      st4(cat + x.at(p, co), v);
      if constexpr (RES && !TAN) st4(gCAT + x.gat(p, co), v);
    };
    wk.begin();
    for (; wk.cur < 2 * NU; wk.next()) {
      const auto [l16, kk] = Lane();
      const bool isH = wk.cur >= NU;
      const int n0 = (isH ? wk.cur - NU : wk.cur) * NN;
      int p[NN];
#pragma unroll
      for (int n = 0; n < NN; ++n) p[n] = 16 * (n0 + n) + l16;
      f32x4 acc[NN][MT], tac[TAN ? NN : 1][TAN ? MT : 1];
#pragma unroll
      for (int n = 0; n < NN; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
          if constexpr (TAN) tac[n][m] = acc[n][m];
        }
      // the epilogue's operands (PRE: held over the contraction)
      constexpr bool PRE = !TAN && (RES || C == 32);  // (registers)
      const int64_t bx = isH ? o.bx : o.by;
      const float* k1p = x.kt + (isH ? o.kx : o.ky);
      const float* k1d = TAN ? x.tkt + (isH ? o.kx : o.ky) : nullptr;
      const float* bp = x.prm + (isH ? o.bh : o.bv);
      f32x4 bias[MT], b1[MT / 2], k1[PRE ? MT / 2 : 1][PRE ? MT : 1];
#pragma unroll
      for (int m = 0; m < MT; ++m) bias[m] = ld4(bp + 16 * m + (unsigned)(4 * kk));
#pragma unroll
      for (int m = 0; m < MT / 2; ++m) {
        b1[m] = ld4(x.prm + bx + 16 * m + (unsigned)(4 * kk));
        if constexpr (PRE) {
#pragma unroll
          for (int jq = 0; jq < MT; ++jq) k1[m][jq] = ld4(k1p + (m * MT + jq) * 256 + (unsigned)(4 * l16 + 64 * kk));
        }
      }
      const int ntap = isH ? 3 : 9, row0 = isH ? GT_H : GT_V;
      if (first) {  // the spins: one channel
        const float* k = x.prm + (isH ? o.kh : o.kv) + 4 * kk;
        const float* kd = TAN ? x.tan + (isH ? o.kh : o.kv) + 4 * kk : nullptr;
#pragma unroll
        for (int n = 0; n < NN; ++n)
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            acc[n][m] = bias[m];
            if constexpr (TAN) tac[n][m] = ld4(x.tan + (isH ? o.bh : o.bv) + 4 * kk + 16 * m);
          }
        for (int t = 0; t < ntap; ++t)
#pragma unroll
          for (int n = 0; n < NN; ++n) {
            const int s = x.src(x.ftab, row0 + t, p[n]);
            const float sv = s < HW ? x.spins[s] : 0.0f;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
              acc[n][m] += ld4(k + t * C + 16 * m) * sv;
              if constexpr (TAN) tac[n][m] += ld4(kd + t * C + 16 * m) * sv;
            }
          }
      } else {
        const int64_t ko = isH ? o.kh : o.kv;
        const float* in = isH ? Hh : V;
        const float* ind = isH ? Hd : Vd;
        conv_acc<C, MT, NN, QS, RES, TAN>(
            acc, tac, x.kt + ko, TAN ? x.tkt + ko : nullptr, ntap, C * C,
            [&](int n, int t) { return x.src(x.ftab, row0 + t, p[n]); },
            [&](int s, int j) { return x.px(in, s, 16 * j + 4 * kk); },
            [&](int s, int j) { return x.px(ind, s, 16 * j + 4 * kk); }, [&](int s) { return x.has(s); });
#pragma unroll
        for (int n = 0; n < NN; ++n)
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            acc[n][m] += bias[m];
            if constexpr (TAN) tac[n][m] += ld4(x.tan + (isH ? o.bh : o.bv) + 4 * kk + 16 * m);
          }
      }
      // What the epilogue reads is requested before it stores anything, and
      // outside of its branches: a load behind a store waits for the store too.
      const bool kr = kb && !isH;
      const float* rp = kr ? tens(blk - 2, T_VO) : x.ws;
      const float* rpd = TAN && kr ? ttens(blk - 2, T_VO) : x.ws;
      f32x4 rv[NN][MT], rd[TAN ? NN : 1][TAN ? MT : 1];
      auto residuals = [&]() {
#pragma unroll
        for (int n = 0; n < NN; ++n)
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const unsigned e = kr && p[n] < HW ? x.gat(p[n], 16 * m + 4 * kk) : 0;
            rv[n][m] = ld4(rp + e);
            if constexpr (TAN) rd[n][m] = ld4(rpd + e);
          }
      };
      constexpr bool LATE = C == 64 && !RES;  // (registers)
      if constexpr (!LATE) residuals();
      // the 1x1 on these pixels, in registers
      f32x4 a[NN][MT], ad[TAN ? NN : 1][TAN ? MT : 1];
#pragma unroll
      for (int n = 0; n < NN; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          a[n][m] = bact4<ACT>(acc[n][m]);
          if constexpr (TAN) ad[n][m] = bdact4<ACT>(a[n][m]) * tac[n][m];
        }
      const int off = (isH ? 0 : C / 2) + 4 * kk;
      f32x4 cv[NN][MT / 2], cd[TAN ? NN : 1][TAN ? MT / 2 : 1], c0[MT / 2], d0[TAN ? MT / 2 : 1];
#pragma unroll
      for (int m = 0; m < MT / 2; ++m) {
#pragma unroll
        for (int n = 0; n < NN; ++n) {
          cv[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
          if constexpr (TAN) cd[n][m] = cv[n][m];
        }
#pragma unroll
        for (int jq = 0; jq < MT; ++jq) {
          const f32x4 w = PRE ? k1[m][jq] : ld4(k1p + (m * MT + jq) * 256 + (unsigned)(4 * l16 + 64 * kk));
          f32x4 wd = {0.f, 0.f, 0.f, 0.f};
          if constexpr (TAN) wd = ld4(k1d + (m * MT + jq) * 256 + (unsigned)(4 * l16 + 64 * kk));
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int n = 0; n < NN; ++n) {
              cv[n][m] = mfma4(w[r], a[n][jq][r], cv[n][m]);
              if constexpr (TAN) {
                cd[n][m] = mfma4(w[r], ad[n][jq][r], cd[n][m]);
                cd[n][m] = mfma4(wd[r], a[n][jq][r], cd[n][m]);
              }
            }
        }
        c0[m] = bact4<ACT>(b1[m]);
        f32x4 bd = {0.f, 0.f, 0.f, 0.f};
        if constexpr (TAN) {
          bd = ld4(x.tan + bx + 16 * m + 4 * kk);
          d0[m] = bdact4<ACT>(c0[m]) * bd;
        }
#pragma unroll
        for (int n = 0; n < NN; ++n) {
          cv[n][m] = bact4<ACT>(cv[n][m] + b1[m]);
          if constexpr (TAN) cd[n][m] = bdact4<ACT>(cv[n][m]) * (cd[n][m] + bd);
        }
      }
      if constexpr (LATE) {
        __builtin_amdgcn_sched_barrier(0);
        residuals();
      }
#pragma unroll
      for (int n = 0; n < NN; ++n) {
        const int q = p[n];
        if (q >= HW) continue;
        if constexpr (!TAN) {
          float* act = tens(blk, isH ? T_XA : T_VA);
#pragma unroll
          for (int m = 0; m < MT; ++m) st4(act + x.gat(q, 16 * m + 4 * kk), a[n][m]);
        }
        if (!isH && !fin) {
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const int e = 16 * m + 4 * kk;
            f32x4 vo = a[n][m], vd = vo;
            if constexpr (TAN) vd = ad[n][m];
            if (kb) {
              vo = bact4<ACT>(rv[n][m] + acc[n][m]);
              if constexpr (TAN) vd = bdact4<ACT>(vo) * (rd[n][m] + tac[n][m]);
            }
            st4(tens(blk, T_VO) + x.gat(q, e), vo);
            if constexpr (RES) st4(x.tile(to) + x.at(q, e), vo);
            if constexpr (TAN) {
              st4(ttens(blk, T_VO) + x.gat(q, e), vd);
              if constexpr (RES) st4(x.tile(4 + to) + x.at(q, e), vd);
            }
          }
        }
        // target pixel: the DownShift, or the RightShift of the final block
        const int i = q / W, j = q - (q / W) * W;
        const bool to_ok = isH ? (!fin || j + 1 < W) : i + 1 < x.H;
        const bool edge = isH ? (fin && j == 0) : i == 0;  // the target that nothing reaches
        const int tp = isH ? (fin ? q + 1 : q) : q + W;
#pragma unroll
        for (int m = 0; m < MT / 2; ++m) {
          if (to_ok) put_cat(tp, off + 16 * m, cv[n][m]);
          if (edge) put_cat(q, off + 16 * m, c0[m]);
          if constexpr (TAN) {
            if (to_ok) st4(catd + x.at(tp, off + 16 * m), cd[n][m]);
            if (edge) st4(catd + x.at(q, off + 16 * m), d0[m]);
          }
        }
      }
    }
    __syncthreads();
    // ---- the 3x3 over the concatenation
    wk.begin();
    const int mgs = MT / MG;
    for (; wk.cur < mgs * NU; wk.next()) {
      const auto [l16, kk] = Lane();
      const int m0 = (wk.cur % mgs) * MG, n0 = (wk.cur / mgs) * NN;
      int p[NN];
#pragma unroll
      for (int n = 0; n < NN; ++n) p[n] = 16 * (n0 + n) + l16;
      f32x4 acc[NN][MG], tac[TAN ? NN : 1][TAN ? MG : 1];
#pragma unroll
      for (int n = 0; n < NN; ++n)
#pragma unroll
        for (int m = 0; m < MG; ++m) {
          acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
          if constexpr (TAN) tac[n][m] = acc[n][m];
        }
      f32x4 bias[MG];
#pragma unroll
      for (int m = 0; m < MG; ++m) bias[m] = ld4(x.prm + o.bc + 16 * (m0 + m) + (unsigned)(4 * kk));
      const int64_t ko = o.kc + 16 * m0 * C;
      conv_acc<C, MG, NN, QS, RES, TAN>(
          acc, tac, x.kt + ko, TAN ? x.tkt + ko : nullptr, 9, C * C,
          [&](int n, int t) { return x.src(x.ftab, GT_C + t, p[n]); },
          [&](int s, int j) { return x.px(cat, s, 16 * j + 4 * kk); },
          [&](int s, int j) { return x.px(catd, s, 16 * j + 4 * kk); }, [&](int s) { return x.has(s); });
      const float* rp = kb ? tens(blk - 2, T_HO) : x.ws;
      const float* rpd = TAN && kb ? ttens(blk - 2, T_HO) : x.ws;
      f32x4 rv[NN][MG], rd[TAN ? NN : 1][TAN ? MG : 1], bd[TAN ? MG : 1];
#pragma unroll
      for (int m = 0; m < MG; ++m) {
        if constexpr (TAN) bd[m] = ld4(x.tan + o.bc + 16 * (m0 + m) + 4 * kk);
#pragma unroll
        for (int n = 0; n < NN; ++n) {
          const unsigned e = kb && p[n] < HW ? x.gat(p[n], 16 * (m0 + m) + 4 * kk) : 0;
          rv[n][m] = ld4(rp + e);
          if constexpr (TAN) rd[n][m] = ld4(rpd + e);
        }
      }
#pragma unroll
      for (int n = 0; n < NN; ++n) {
        const int q = p[n];
        if (q >= HW) continue;
#pragma unroll
        for (int m = 0; m < MG; ++m) {
          const int e = 16 * (m0 + m) + 4 * kk;
          f32x4 h = acc[n][m] + bias[m];
          f32x4 hd = h;
          if constexpr (TAN) hd = tac[n][m] + bd[m];
          if (kb) {
            h = rv[n][m] + h;
            if constexpr (TAN) hd += rd[n][m];
          }
          const f32x4 ho = bact4<ACT>(h);
          st4(tens(blk, T_HO) + x.gat(q, e), ho);
          if constexpr (RES) st4(x.tile(3) + x.at(q, e), ho);
          if constexpr (TAN) {
            const f32x4 v = bdact4<ACT>(ho) * hd;
            st4(ttens(blk, T_HO) + x.gat(q, e), v);
            if constexpr (RES) st4(x.tile(7) + x.at(q, e), v);
          }
        }
      }
    }
    __syncthreads();
  }
}

// A weight gradient: dK[tap][ci][co] = sum_p in[src(tap, p)][ci] dout[p][co],
// db[co] = sum_p dout[p][co].
struct WGrad {
  const float* in;    // in the workspace
  const float* dout;  // a live tensor, from channel dc
  int dc;
  float *dk, *db;
  int row, ntap, cout;
  bool add;  // to dk and db (ACC)
};

// One unit of it: WM x WM 16x16 tiles (inputs x outputs) of one tap.  The
// outputs are the columns, so that 16 lanes store 64 adjacent bytes of a row.
template <class S, bool ACC>
__device__ __forceinline__ void wgrad_unit(const Ctx<S>& x, const WGrad& g, int unit) {
  constexpr int C = S::C, SG = S::SG, WM = S::WM, B = 16 * WM, NB = C / B;
  constexpr bool RES = S::RES;
  const auto [l16, kk] = Lane();
  const int HW = x.HW;
  const int mb = (g.cout + B - 1) / B;
  const int t = unit / (mb * NB), r = unit - t * (mb * NB);
  const int co0 = B * (r / NB), ci0 = B * (r % NB);
  const int nn = min(WM, (g.cout - co0) / 16);  // tiles of outputs (WM, or WM / 2)
  const int16_t* tt = x.ftab + (g.row + t) * x.HP + kk;
  const float* da = g.dout + (RES ? co0 + g.dc : (co0 + g.dc) * HW);
  const float* ia = g.in + ci0 * HW;
  const unsigned lb = (l16 >> 2) * (4 * HW) + (l16 & 3);  // this lane's channel in the workspace's layout
  float* dst = g.dk + ((int64_t)t * C + ci0) * g.cout + co0 + (unsigned)(4 * kk * g.cout + l16);
  const f32x4 z = {0.f, 0.f, 0.f, 0.f};
  f32x4 c[WM][WM], bs[WM];
#pragma unroll
  for (int m = 0; m < WM; ++m) {
    bs[m] = z;
#pragma unroll
    for (int n = 0; n < WM; ++n) c[m][n] = z;
  }
  const bool bias = t == 0 && ci0 == 0;
  // KB contraction steps (4 pixels each) at a time, the next ones' operands
  // requested before these are used and their source pixels before that
  constexpr int KB = WM == 4 ? 2 : 4;
  struct Ops {
    float a[KB][WM], b[KB][WM];
    bool iok[KB], pok[KB];  // (applied at the use)
  };
  int src[KB];
  auto sources = [&](int k) {
#pragma unroll
    for (int e = 0; e < KB; ++e) src[e] = tt[4 * (k + e)];
  };
  auto request = [&](Ops& o, int k) {
#pragma unroll
    for (int e = 0; e < KB; ++e) {
      const int p = 4 * (k + e) + kk;
      o.iok[e] = src[e] < HW;
      o.pok[e] = RES || p < HW;
      const unsigned ip = 4 * (src[e] < HW ? src[e] : 0) + lb;
#pragma unroll
      for (int m = 0; m < WM; ++m) o.a[e][m] = ia[ip + 16 * m * HW];
      const unsigned dp = RES ? (p < HW ? p : HW) * SG + l16 : 4 * (p < HW ? p : 0) + lb;  // (RES: the zero pixel)
#pragma unroll
      for (int n = 0; n < WM; ++n) o.b[e][n] = da[dp + (n < nn ? 16 * n * (RES ? 1 : HW) : 0)];
    }
    sources(k + KB);
  };
  auto compute = [&](const Ops& o) {
#pragma unroll
    for (int e = 0; e < KB; ++e) {
      float a[WM], b[WM];
#pragma unroll
      for (int m = 0; m < WM; ++m) {
        a[m] = o.iok[e] ? o.a[e][m] : 0.0f;
        b[m] = o.pok[e] ? o.b[e][m] : 0.0f;
      }
#pragma unroll
      for (int n = 0; n < WM; ++n)
        if (n < (WM + 1) / 2 || n < nn) {  // (uniform)
#pragma unroll
          for (int m = 0; m < WM; ++m) c[m][n] = mfma4(a[m], b[n], c[m][n]);
        }
      if (bias) {  // (uniform)
#pragma unroll
        for (int n = 0; n < WM; ++n) bs[n] = mfma4(1.0f, b[n], bs[n]);
      }
    }
  };
  Ops A, Bo;
  sources(0);
  request(A, 0);
  const int ks = (HW + 3) / 4;
  int k = 0;
#pragma unroll 1
  for (; k + KB < ks; k += 2 * KB) {
    __builtin_amdgcn_sched_barrier(0);
    request(Bo, k + KB);
    compute(A);
    interleave<KB * WM * (RES ? 1 : 2), KB + (RES ? KB * WM : 0), KB * WM * WM>();
    request(A, k + 2 * KB);
    compute(Bo);
    interleave<KB * WM * (RES ? 1 : 2), KB + (RES ? KB * WM : 0), KB * WM * WM>();
  }
  float old[ACC ? WM : 1][ACC ? WM : 1][4];
  if constexpr (ACC) {  // the sums so far
#pragma unroll
    for (int m = 0; m < WM; ++m)
#pragma unroll
      for (int n = 0; n < WM; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          old[m][n][e] = g.add ? dst[(16 * m + e) * g.cout + (n < nn ? 16 * n : 0)] : 0.0f;
  }
  if (k < ks) compute(A);
#pragma unroll
  for (int n = 0; n < WM; ++n)
    if (n < nn) {
#pragma unroll
      for (int m = 0; m < WM; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          dst[(16 * m + e) * g.cout + 16 * n] = ACC ? old[m][n][e] + c[m][n][e] : c[m][n][e];
      if (bias && kk == 0) {
        float* db = g.db + co0 + 16 * n + l16;
        *db = ACC && g.add ? *db + bs[n][0] : bs[n][0];
      }
    }
}

// Block 0's V and H weight gradients: one input channel.
template <class S, bool ACC>
__device__ __forceinline__ void wgrad_spins(const Ctx<S>& x, const WGrad& g) {
  constexpr int C = S::C;
  for (int idx = threadIdx.x; idx < (g.ntap + 1) * C; idx += blockDim.x) {
    const int t = idx / C, co = idx - (idx / C) * C;
    float acc = 0.0f;
#pragma unroll 4
    for (int p = 0; p < x.HW; ++p) {
      const int s = t < g.ntap ? (int)x.ftab[(g.row + t) * x.HP + p] : 0;
      const float v = t < g.ntap ? (s < x.HW ? x.spins[s] : 0.0f) : 1.0f;
      acc += v * g.dout[x.at(p, co)];
    }
    float* dst = t < g.ntap ? g.dk + t * C + co : g.db + co;
    *dst = ACC && g.add ? *dst + acc : acc;
  }
}

// Backward of one sample from the head's cotangent dz (HW x 4): d / d theta
// into O (overwritten; ACC: added to when add).  Live tensors (RES: tiles):
// gh 0, gv 1 and 2 in turn, dcat 3, dxa 4.
template <class S, int ACT, bool ACC>
__device__ __forceinline__ void backward(Work& wk, const Ctx<S>& x, const float* dz, float* O, bool add) {
  constexpr int C = S::C, MT = S::MT, NN = S::NN, QS = S::QS, SG = S::SG, NB = C / (16 * S::WM);
  constexpr bool RES = S::RES;
  constexpr int MG = RES ? MT / 2 : MT;
  const int HW = x.HW, W = x.W, F = x.nb - 1;
  const int ntl = (HW + 15) / 16, NU = (ntl + NN - 1) / NN;
  auto tens = [&](int blk, int which) -> const float* { return ws_tensor(x.ws, HW, C, blk, which); };
  auto live = [&](int k) { return RES ? x.tile(k) : ws_grad(x.ws, HW, C, x.nb, k); };
  float* gh = live(0);
  float* dcat = live(3);
  float* dxa = live(4);
  float* dVr = ws_grad(x.ws, HW, C, x.nb, 5);  // the residuals' gradients
  float* dHr = ws_tensor(x.ws, HW, C, F, T_VO);  // (the final block has no vertical output)
  const int64_t ho = head_offset(x.nb, C);
  const float* HF = tens(F, T_HO);
  // the head: weights (four partial sums over the pixels each), then gh
  for (int idx = threadIdx.x >> 2; idx < 4 * C + 4; idx += blockDim.x >> 2) {
    const int part = threadIdx.x & 3;
    float acc = 0.0f;
    if (idx < 4 * C) {
      const int ci = idx / 4, k = idx & 3;
#pragma unroll 4
      for (int p = part; p < HW; p += 4) acc += HF[x.gat(p, ci)] * dz[p * 4 + k];
    } else {
#pragma unroll 4
      for (int p = part; p < HW; p += 4) acc += dz[p * 4 + idx - 4 * C];
    }
    acc += __shfl_xor(acc, 1, 64);
    acc += __shfl_xor(acc, 2, 64);
    if (part == 0) O[ho + idx] = ACC && add ? O[ho + idx] + acc : acc;
  }
  {
    float* gv = live(1);
    for (int idx = threadIdx.x; idx < HW * (C / 4); idx += blockDim.x) {
      const int p = idx % HW, c = 4 * (idx / HW);
      const f32x4 d = ld4(dz + 4 * p);
      f32x4 g;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f32x4 k = ld4(x.prm + ho + (c + e) * 4);
        g[e] = 0.0f;
#pragma unroll
        for (int u = 0; u < 4; ++u) g[e] += k[u] * d[u];
      }
      st4(gh + x.at(p, c), g * bdact4<ACT>(ld4(HF + x.gat(p, c))));
      st4(gv + x.at(p, c), f32x4{0.f, 0.f, 0.f, 0.f});
    }
  }
  __syncthreads();
  for (int blk = F; blk >= 0; --blk) {
    const ParamOffsets o = param_offsets(blk, C);
    const bool first = blk == 0, fin = blk == F;
    const bool ka = !first && !fin && ((blk & 1) == 1);
    const bool kb_next = blk - 1 > 0 && ((blk - 1) & 1) == 0;  // the next block's gradients are its residual's too
    float* gv = live(1 + ((F - blk) & 1));
    float* gvn = live(1 + ((F - blk + 1) & 1));
    const float* CAT = tens(blk, T_CAT);
    const float* XA = tens(blk, T_XA);
    const float* VA = tens(blk, T_VA);
    const float* Vin = first ? x.spins : tens(blk - 1, T_VO);
    const float* Hin = first ? x.spins : tens(blk - 1, T_HO);
    // ---- phase C
    wk.begin();
    {
      const WGrad wc{CAT, gh, 0, O + o.kc, O + o.bc, GT_C, 9, C, add};
      const int nw = 9 * NB * NB;
      for (; wk.cur < NU + nw; wk.next()) {
        if (wk.cur >= NU) {
          wgrad_unit<S, ACC>(x, wc, wk.cur - NU);
          continue;
        }
        const auto [l16, kk] = Lane();
        // data gradient of NN pixel tiles, all channels; the 1x1s' follow
        int p[NN];
#pragma unroll
        for (int n = 0; n < NN; ++n) p[n] = 16 * (wk.cur * NN + n) + l16;
        f32x4 acc[NN][MT], none[1][1];
#pragma unroll
        for (int n = 0; n < NN; ++n)
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
        conv_acc<C, MT, NN, QS, RES, false>(
            acc, none, x.kb + o.kc, nullptr, 9, C * C,
            [&](int n, int t) { return x.src(x.itab, GT_C + t, p[n]); },
            [&](int s, int j) { return x.px(gh, s, 16 * j + 4 * kk); }, [&](int, int) { return f32x4{}; },
            [&](int s) { return x.has(s); });
        // (loads before stores and outside of branches, as in the forward)
#pragma unroll
        for (int n = 0; n < NN; ++n) {
          const int q = p[n];
          const bool in = q < HW;
          const int qc = in ? q : 0;
          const int i = qc / W, j = qc - (qc / W) * W;
          const bool xok = in && (!fin || j >= 1), yok = in && i >= 1;
          const int xp = xok ? (fin ? q - 1 : q) : 0, yp = yok ? q - W : 0;
          f32x4 d[MT], xa[MT], va[MT], g[MT];
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const int e = 16 * m + 4 * kk;
            d[m] = ld4(CAT + x.gat(qc, e));
            xa[m] = ld4(XA + x.gat(xp, e));
            va[m] = ld4(VA + x.gat(yp, e));
            g[m] = ld4(gv + x.at(yp, e));
          }
#pragma unroll
          for (int m = 0; m < MT; ++m) d[m] = acc[n][m] * bdact4<ACT>(d[m]);
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            f32x4 cx = {0.f, 0.f, 0.f, 0.f}, cy = cx;
#pragma unroll
            for (int jq = 0; jq < MT / 2; ++jq) {
              const int ko = (m * (MT / 2) + jq) * 256;
              const unsigned lo = 4 * l16 + 64 * kk;
              const f32x4 wx = ld4(x.kb + o.kx + ko + lo), wy = ld4(x.kb + o.ky + ko + lo);
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                cx = mfma4(wx[r], d[jq][r], cx);
                cy = mfma4(wy[r], d[MT / 2 + jq][r], cy);
              }
            }
            xa[m] = cx * bdact4<ACT>(xa[m]);
            g[m] += cy * bdact4<ACT>(va[m]);
          }
          if (in) {
#pragma unroll
            for (int m = 0; m < MT; ++m) {
              const int e = 16 * m + 4 * kk;
              st4(dcat + x.at(q, e), d[m]);
              if (xok) st4(dxa + x.at(xp, e), xa[m]);
              if (fin && j == W - 1) st4(dxa + x.at(q, e), f32x4{0.f, 0.f, 0.f, 0.f});
              if (yok) st4(gv + x.at(yp, e), g[m]);
            }
          }
        }
      }
    }
    __syncthreads();
    // ---- phase VH
    wk.begin();
    {
      const WGrad wv{Vin, gv, 0, O + o.kv, O + o.bv, GT_V, 9, C, add}, wh{Hin, dxa, 0, O + o.kh, O + o.bh, GT_H, 3, C, add};
      const WGrad wx{XA, dcat, 0, O + o.kx, O + o.bx, fin ? GT_XF : GT_X, 1, C / 2, add};
      const WGrad wy{VA, dcat, C / 2, O + o.ky, O + o.by, GT_Y, 1, C / 2, add};
      // the list: V's data gradient, its weights, H's, the 1x1s' weights
      const int mgs = MT / MG, nd = first ? 0 : mgs * NU, nv = first ? 0 : 9 * NB * NB, nh = first ? 0 : 3 * NB * NB;
      const int n1 = NB * ((C / 2 + 16 * S::WM - 1) / (16 * S::WM));
      for (; wk.cur < 2 * nd + nv + nh + 2 * n1; wk.next()) {
        int u = wk.cur;
        const bool isV = u < nd;
        if (!isV) {
          u -= nd;
          if (u >= nd) {
            u -= nd;
            WGrad w = wv;
            if (u >= nv) {
              u -= nv;
              w = wh;
              if (u >= nh) {
                u -= nh;
                w = wx;
                if (u >= n1) {
                  u -= n1;
                  w = wy;
                }
              }
            }
            wgrad_unit<S, ACC>(x, w, u);
            continue;
          }
        }
        const auto [l16, kk] = Lane();
        const int m0 = (u % mgs) * MG, n0 = (u / mgs) * NN;
        int p[NN];
#pragma unroll
        for (int n = 0; n < NN; ++n) p[n] = 16 * (n0 + n) + l16;
        f32x4 acc[NN][MG], none[1][1];
#pragma unroll
        for (int n = 0; n < NN; ++n)
#pragma unroll
          for (int m = 0; m < MG; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
        const float* dout = isV ? gv : dxa;
        const int row0 = isV ? GT_V : GT_H;
        conv_acc<C, MG, NN, QS, RES, false>(
            acc, none, x.kb + (isV ? o.kv : o.kh) + 16 * m0 * C, nullptr,
            isV ? 9 : 3, C * C,
            [&](int n, int t) { return x.src(x.itab, row0 + t, p[n]); },
            [&](int s, int j) { return x.px(dout, s, 16 * j + 4 * kk); }, [&](int, int) { return f32x4{}; },
            [&](int s) { return x.has(s); });
        const float* inp = isV ? Vin : Hin;
        float* dst = isV ? gvn : gh;
        float* res = isV ? dVr : dHr;
        f32x4 iv[NN][MG], rv[NN][MG];
#pragma unroll
        for (int n = 0; n < NN; ++n)
#pragma unroll
          for (int m = 0; m < MG; ++m) {
            const unsigned e = x.gat(p[n] < HW ? p[n] : 0, 16 * (m0 + m) + 4 * kk);
            iv[n][m] = ld4(inp + e);
            rv[n][m] = ld4(res + (ka ? e : 0));
          }
#pragma unroll
        for (int n = 0; n < NN; ++n) {
          const int q = p[n];
          if (q >= HW) continue;
#pragma unroll
          for (int m = 0; m < MG; ++m) {
            const int e = 16 * (m0 + m) + 4 * kk;
            f32x4 g = acc[n][m];
            if (ka) g += rv[n][m];
            g *= bdact4<ACT>(iv[n][m]);
            st4(dst + x.at(q, e), g);
            if (kb_next) st4(res + x.gat(q, e), g);
          }
        }
      }
      if (first) {
        wgrad_spins<S, ACC>(x, wv);
        wgrad_spins<S, ACC>(x, wh);
      }
    }
    __syncthreads();
  }
}

// Sums of NV values over the workgroup, in a fixed order; thread 0 gets them.
template <int NV>
__device__ __forceinline__ void block_sums(float (&v)[NV], float* red) {  // red: NV x waves
  const int wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    for (int s = 32; s > 0; s >>= 1) v[k] += __shfl_xor(v[k], s, 64);
    if ((threadIdx.x & 63) == 0) red[k * nw + wave] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    float s = 0.0f;
    for (int w = 0; w < nw; ++w) s += red[k * nw + w];
    v[k] = s;
  }
}

// MODE GRAD_O: one workgroup per sample, two backward passes (the cotangents
// of Re and Im log psi) into its rows of O_re and O_im.  GRAD_VJP: a
// persistent grid; cot_re d Re log psi + cot_im d Im log psi of a workgroup's
// samples, run by run (a.run samples), is summed in partial rows of its own: run
// r of workgroup w in row r gridDim.x + w.  GRAD_JVP: forward mode.
template <int C_, int ACT, int MODE, bool RES_, int NT>
__global__ __launch_bounds__(NT, NT == 1024 ? 4 : 2) void convar_grad_kernel3(BwdArgs a) {
  constexpr bool TAN = MODE == GRAD_JVP;
  using S = Shape<C_, RES_, NT>;
  constexpr int C = C_;
  constexpr bool RES = RES_;
  extern __shared__ __align__(16) uint8_t smem[];
  __shared__ int s_q[4];
  __shared__ float s_red[4 * (NT / 64)];
  const int HW = a.HW, nb = a.nb, F = nb - 1;
  Ctx<S> x;
  x.prm = a.params;
  x.kt = a.kt;
  x.kb = a.kb;
  x.tan = a.tangent;
  x.tkt = a.tkt;
  x.ws = a.work + (int64_t)blockIdx.x * a.work_floats;
  x.wt = TAN ? x.ws + a.work_floats / 2 : nullptr;
  x.spins = x.ws;
  x.H = a.H;
  x.W = a.W;
  x.HW = HW;
  x.HP = table_row(HW);
  x.nb = nb;
  float* dz = reinterpret_cast<float*>(smem);  // HW x 4
  x.lds = dz + 4 * HW;
  int16_t* ftab = reinterpret_cast<int16_t*>(x.lds + (RES ? (TAN ? 8 : 5) * (HW + 1) * S::SG : 0));
  int16_t* itab = ftab + GT_N * x.HP;
  x.ftab = ftab;
  x.itab = itab;
  if (threadIdx.x < 4) s_q[threadIdx.x] = 0;
  if constexpr (RES) {  // the tiles' zero pixels
    for (int k = threadIdx.x; k < (TAN ? 8 : 5) * S::SG; k += NT)
      x.tile(k / S::SG)[HW * S::SG + k % S::SG] = 0.0f;
  }
  build_tables(ftab, itab, a.H, a.W);
  Work wk{s_q, 0, 0};
  float* part = MODE == GRAD_VJP ? a.partial + (int64_t)blockIdx.x * a.P : nullptr;
  int64_t k = 0;  // the sample's number in its run
  const int64_t ho = head_offset(nb, C);
  for (int64_t b = blockIdx.x; b < a.batch; b += gridDim.x) {
    for (int q = threadIdx.x; q < HW; q += NT) x.ws[q] = (float)a.spins[b * HW + q];
    __syncthreads();
    forward<S, ACT, TAN>(wk, x);
    const float* HF = ws_tensor(x.ws, HW, C, F, T_HO);
    float sums[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int PASSES = MODE == GRAD_O ? 2 : 1;
    for (int pass = 0; pass < PASSES; ++pass) {
      const float wr = MODE == GRAD_VJP ? a.cot[2 * b] : pass == 0 ? 1.0f : 0.0f;
      const float wi = MODE == GRAD_VJP ? a.cot[2 * b + 1] : pass == 1 ? 1.0f : 0.0f;
      for (int p = threadIdx.x; p < HW; p += NT) {
        float z[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) z[k] = x.prm[ho + 4 * C + k];
#pragma unroll 4
        for (int c = 0; c < C; c += 4) {
          const f32x4 h = ld4(HF + x.gat(p, c));
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int k = 0; k < 4; ++k) z[k] += x.prm[ho + (c + e) * 4 + k] * h[e];
        }
        const float mx = fmaxf(z[0], z[1]);
        const float e0 = expf(2.0f * (z[0] - mx)), e1 = expf(2.0f * (z[1] - mx));
        const float p0 = e0 / (e0 + e1), p1 = e1 / (e0 + e1);
        const bool up = x.spins[p] > 0.0f;
        if (pass == 0) {
          const float lse = mx + 0.5f * logf(e0 + e1);
          sums[0] += (up ? z[0] : z[1]) - lse;
          sums[1] += up ? z[2] : z[3];
        }
        if constexpr (TAN) {
          const float* HFd = ws_tensor(x.wt, HW, C, F, T_HO);
          float zd[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            float acc = x.tan[ho + 4 * C + k];
#pragma unroll 4
            for (int ci = 0; ci < C; ++ci)
              acc += x.prm[ho + ci * 4 + k] * HFd[x.gat(p, ci)] + x.tan[ho + ci * 4 + k] * HF[x.gat(p, ci)];
            zd[k] = acc;
          }
          // d/dz of z_s - 0.5 log(e^{2 z0} + e^{2 z1}) is delta_s - p
          sums[2] += (up ? zd[0] : zd[1]) - (p0 * zd[0] + p1 * zd[1]);
          sums[3] += up ? zd[2] : zd[3];
        } else {
          dz[p * 4 + 0] = wr * ((up ? 1.0f : 0.0f) - p0);
          dz[p * 4 + 1] = wr * ((up ? 0.0f : 1.0f) - p1);
          dz[p * 4 + 2] = wi * (up ? 1.0f : 0.0f);
          dz[p * 4 + 3] = wi * (up ? 0.0f : 1.0f);
        }
      }
      if (pass == 0) block_sums(sums, s_red);  // (with a barrier: dz is complete)
      else __syncthreads();
      if constexpr (!TAN) {
        float* O = MODE == GRAD_VJP ? part : (pass == 0 ? a.o_re : a.o_im) + b * a.ld;
        backward<S, ACT, MODE == GRAD_VJP>(wk, x, dz, O, k > 0);
      }
    }
    if (threadIdx.x == 0) {
      if (a.logpsi) {
        a.logpsi[2 * b] = sums[0];
        a.logpsi[2 * b + 1] = sums[1];
      }
      if constexpr (TAN) {
        a.jvp[2 * b] = sums[2];
        a.jvp[2 * b + 1] = sums[3];
      }
    }
    if constexpr (MODE == GRAD_VJP) {
      if (++k == a.run) {
        k = 0;
        part += gridDim.x * a.P;
      }
    }
    __syncthreads();
  }
}

// The conv kernels with C input channels in the order of the MFMA operands,
// each at its own offset of the flat vector: [tap][tile][quad][lane][4], lane
// l16 + 16 kk holding row 16 tile + l16, contraction 16 quad + 4 kk + 0..3.
// Rows are outputs and the contraction inputs for the forward (fwd), the other
// way round for the data gradients (bwd; or null).  Block 0's V and H kernels
// (one input channel) are read as they are.  Grid: (entries, 5 nb, 1 or 2).
template <int C>
__global__ void pack_kernels_kernel(const float* __restrict__ prm, float* __restrict__ fwd, float* __restrict__ bwd) {
  const int blk = blockIdx.y / 5, which = blockIdx.y % 5;
  if (blk == 0 && which < 2) return;
  const ParamOffsets o = param_offsets(blk, C);
  const int64_t off = which == 0 ? o.kv : which == 1 ? o.kh : which == 2 ? o.kx : which == 3 ? o.ky : o.kc;
  const int ntap = which == 1 ? 3 : (which == 2 || which == 3) ? 1 : 9;
  const int cout = (which == 2 || which == 3) ? C / 2 : C;
  const bool back = blockIdx.z == 1;
  const int mt = (back ? C : cout) / 16, kq = (back ? cout : C) / 16;
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= ntap * C * cout / 4) return;
  const int lane = q & 63, frag = q >> 6;
  const int t = frag / (mt * kq), m = frag / kq % mt, j = frag % kq;
  const int row = 16 * m + (lane & 15), col = 16 * j + 4 * (lane >> 4);
  const float* k = prm + off + (int64_t)t * C * cout;
  f32x4 v;
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = back ? k[row * cout + col + r] : k[(col + r) * cout + row];
  st4((back ? bwd : fwd) + off + 4 * (int64_t)q, v);
}

size_t plan_lds(int HW, int C, int tiles) {
  return (size_t)16 * HW + (size_t)tiles * (HW + 1) * (C + 4) * 4 + (size_t)(GT_N + GT_X) * table_row(HW) * 2 + 128;
}

template <class K>
int launch_plan(K kern, const GradPlan& p, hipStream_t s, const BwdArgs& a) {
  FK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)p.lds));
  hipLaunchKernelGGL(kern, dim3((unsigned)p.grid), dim3(p.threads), p.lds, s, a);
  FK_CHECK_LAUNCH();
  return FK_OK;
}

// threads of a workgroup that has a CU to itself, tensors in LDS (grad_plan)
constexpr int resident_threads(int C, int mode) { return C == 32 && mode != GRAD_JVP ? 1024 : 512; }

template <int C, int ACT, int MODE>
int launch_mode(const GradPlan& p, const BwdArgs& a, hipStream_t s) {
  if (!p.resident) return launch_plan(convar_grad_kernel3<C, ACT, MODE, false, 512>, p, s, a);
  if constexpr (MODE != GRAD_VJP) {
    if (p.threads == 128) return launch_plan(convar_grad_kernel3<C, ACT, MODE, true, 128>, p, s, a);
    if (p.threads == 256) return launch_plan(convar_grad_kernel3<C, ACT, MODE, true, 256>, p, s, a);
  }
  return launch_plan(convar_grad_kernel3<C, ACT, MODE, true, resident_threads(C, MODE)>, p, s, a);
}
template <int C, int ACT>
int launch_act(const GradPlan& p, const BwdArgs& a, int mode, hipStream_t s) {
  if (mode == GRAD_O) return launch_mode<C, ACT, GRAD_O>(p, a, s);
  if (mode == GRAD_VJP) return launch_mode<C, ACT, GRAD_VJP>(p, a, s);
  return launch_mode<C, ACT, GRAD_JVP>(p, a, s);
}

}  // namespace

GradPlan grad_plan(const BwdArgs& a, int mode) {
  GradPlan p{};
  const int HW = a.HW, C = a.C;
  const int64_t batch = a.batch;
  if (C != 32 && C != 64) return p;
  if ((reinterpret_cast<uintptr_t>(a.params) | reinterpret_cast<uintptr_t>(a.kt) |
       reinterpret_cast<uintptr_t>(a.tangent)) & 15)
    return p;
  const int64_t cu = device_cu_count();
  // Lattices of one pixel tile at 64 channels: a sample is little but its weight
  // gradients' way through the partial rows, for which four workgroups of the
  // other kernel take turns better than one, once each has several samples (VJP,
  // ms, this kernel and the other: 2x2 depth 3, 2048 samples 3.08 and 3.24, 4096
  // 5.90 and 5.57, 16384 22.8 and 19.3; 4x4 depth 3, 4096 samples 6.06 and 6.24,
  // 16384 23.5 and 22.3; two blocks, 3x3, 16384: 8.99 and 9.43).
  if (mode == GRAD_VJP && C == 64 && HW <= 16 && a.nb > 2 && batch > (HW <= 6 ? 12 : 24) * cu) return p;
  const int tiles = mode == GRAD_JVP ? 8 : 5;
  p.resident = plan_lds(HW, C, tiles) <= 158 * 1024;
  p.lds = plan_lds(HW, C, p.resident ? tiles : 0);
  if (p.lds > 158 * 1024) return p;
  // One workgroup per CU of as many waves as the registers allow, except that
  // small lattices, with fewer units in a phase than waves, run two or four to
  // a CU once the batch has a sample for each.  Not the VJP: every workgroup
  // adds a row of partial sums for the reduction.  1024 samples, ms: 4x4 C 32
  // O 0.94 at one, 0.74 at four, JVP 0.48 and 0.22, but VJP (a row a workgroup)
  // 0.70 and 1.15; 8x8 C 32 O 2.20 at one, 2.06 at two.  1024 threads (one pixel
  // tile a unit) against 512 (two): 10x10 C 32, 2048 samples, VJP 15.6 and 16.6, O
  // 24.7 and 26.6, JVP 11.4 both; C 64 has no registers for 1024 (10x10, 1024
  // samples, VJP 14.4 and 13.0).
  p.threads = p.resident ? resident_threads(C, mode) : 512;
  p.per_cu = 1;
  if (p.resident && mode != GRAD_VJP) {
    if (4 * p.lds <= 156 * 1024 && batch > 2 * cu) {
      p.threads = 128;
      p.per_cu = 4;
    } else if (2 * p.lds <= 156 * 1024 && batch > cu) {
      p.threads = 256;
      p.per_cu = 2;
    }
  }
  p.grid = batch < p.per_cu * cu ? (batch > 0 ? batch : 1) : p.per_cu * cu;
  return p;
}

int launch_grad_pack(const BwdArgs& a, const float* prm, float* fwd, float* bwd, hipStream_t s) {
  const dim3 grid((unsigned)((9 * a.C * a.C / 4 + 255) / 256), (unsigned)(a.nb * 5), bwd ? 2 : 1);
  if (a.C == 32) hipLaunchKernelGGL(pack_kernels_kernel<32>, grid, dim3(256), 0, s, prm, fwd, bwd);
  else hipLaunchKernelGGL(pack_kernels_kernel<64>, grid, dim3(256), 0, s, prm, fwd, bwd);
  FK_CHECK_LAUNCH();
  return FK_OK;
}

int launch_grad_plan(const GradPlan& p, const BwdArgs& a, int act, int mode, hipStream_t s) {
  int rc = launch_grad_pack(a, a.params, const_cast<float*>(a.kt), const_cast<float*>(a.kb), s);
  if (rc == FK_OK && mode == GRAD_JVP) rc = launch_grad_pack(a, a.tangent, const_cast<float*>(a.tkt), nullptr, s);
  if (rc != FK_OK) return rc;
  if (a.C == 32)
    return act == FK_ACT_ELU ? launch_act<32, FK_ACT_ELU>(p, a, mode, s) : launch_act<32, FK_ACT_RELU>(p, a, mode, s);
  return act == FK_ACT_ELU ? launch_act<64, FK_ACT_ELU>(p, a, mode, s) : launch_act<64, FK_ACT_RELU>(p, a, mode, s);
}

}  // namespace fk
