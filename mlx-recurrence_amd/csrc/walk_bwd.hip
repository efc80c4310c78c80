// walk_bwd.hip — backward of long heads (SSD with one decay rate per head, GLA;
// bf16 inputs, Dh and N in {64, 128}): one workgroup walks a segment of a
// head's 32-step chunks from the last to the first with the adjoint in
// registers, so no adjoint ever passes through memory.
//
// Per chunk the products are those of chunked_bwd.hip (derivation there):
//   CB = C B^T, G2 = dY U^T, GH = dY h_in, UL = U lam, P = M o CB, MG = M o G2
//   du = diag(w) (P^T dY + diag(m31) B lam^T)
//   Z  = MG^T C + diag(m31) UL,  dB = diag(w) Z,  dC = diag(gam) GH + (MG o w_s) B
//   SSD: dA[n] = sum_t C (K B) + sum_t gam cd C GH + sum_t m31 (cd_31 - cd) w B UL
//                + gam_31 cd_31 sum_d lam h_in,   K = MG o w_s o (cd_t - cd_s)
//        d(delta)_t = a T_t + (1 - a delta_t) sum_n B_t Z_t
//   GLA: dg_t = sum_{t'} M[t', t] ((CB o G2) Mh + X gam_{t-1})[t', t]
//               + m31_t (sum_s Mh[s, t] Y_s + gam_{t-1} tr),  Mh[s, t] = M[t-1, s]
//   lam <- gam_31 lam + (gam o dY)^T C
// formed transposed (rows n or d, columns t), which makes every fp32 factor an
// accumulator that is itself the next operand (contracting over its rows, k
// in the accumulators' order pi(g, e), see final_fwd.hip), and every bf16
// gradient four consecutive values of a lane: 8-byte stores.
//
// Work split: wave w owns CPW column blocks n of the state (GH, UL, Z, dB, dC,
// dA of those columns; its h_in and lam columns are registers) and DPW row
// blocks d (du of those rows; a second copy of lam, rows n, kept by the same
// update): no reduction across waves but the row sums over n.  The masked 32x32
// products are formed once per chunk, their three nonzero 16x16 blocks by
// waves 0-2 in both orientations, and shared as operand fragments; wave 3
// forms the next chunk's step scalars and the previous chunk's step gradient
// meanwhile.  Three LDS-only barriers per chunk: rows staged; fragments and row
// sums written; all read.  The chunk before is loaded while this one runs.
// fp32 factors are split into bf16 hi + lo as in the per-chunk kernels.
//
// Heads alone may not fill the GPU: a head's chunks are cut into S segments; a
// first launch forms every later segment's adjoint map (from a zero adjoint,
// and its decay), and segment j starts from dfinal carried through the maps
// of segments S - 1 .. j + 1.
//
// What bounds it: per wave and chunk about 1300 VALU instructions (the splits of
// h_in and of both copies of lam are a fifth) beside 127 MFMAs (Dh 64, N 128) on
// two waves per SIMD, and the traffic of inputs, checkpoints and gradients.
// SSD B8 L4096 H80 Dh64 N128: 1.60 + 0.19 ms, the walk 4.3 TB/s of 6.9 GB (adjoint
// scan + pair kernel 2.7 ms, 12.6 GB); GLA B8 L2048 H12 Dh128: 254 + 69 us profiled
// (348 + 102 + 156 us).  No register may spill: a spilled load waits for its data at
// once, and a reload for every load in flight (8 % more with 4 spills).
#include "rr_chunked.h"
#include "rr_frag.h"

namespace {

using rr::bf4;
using rr::col_frag;
using rr::f32x4_t;
using rr::join;
using rr::lds_barrier;
using rr::mfma16;
using rr::pack4;
using rr::piece;
using rr::row_frag;
using rr::split_pair;
using rr::u16x4_t;
using rr::u16x8_t;

constexpr int Q = 32;

template <int DH, int NS>
struct Shape {
  static constexpr int NW = DH == 128 && NS == 128 ? 8 : 4, T = 64 * NW;
  static constexpr int NBN = NS / 16, NBD = DH / 16, NK = NS / 32, DK = DH / 32;
  static constexpr int CPW = NBN / NW, DPW = NBD / NW;
};

struct WalkArgs {
  rr::ChunkArgs p;
  float4* mapL;    // [B*H][S-1] adjoint maps of segments 1 .. S-1 (both layouts, fragment order)
  float2* mapP;    // [B*H][S-1] their decays, each as two factors (see scaled)
  int S, cps;      // segments, chunks per segment
};

enum { kP = 0, kMG = 1, kMGw = 2, kK = 3 };   // shared fragments (kK: SSD K, GLA CB o G2)
template <int DH, int NS, bool GLA>
struct alignas(16) WalkSm {
  using S = Shape<DH, NS>;
  uint16_t B[Q * NS], C[Q * NS], U[Q * DH], Yh[Q * DH], Yl[Q * DH], Gh[Q * DH], Gl[Q * DH];
  uint2 F[3][3][2][64];         // P, MG (rows t, columns s), MG o w (rows s, columns t); [block][hi, lo][lane]
  uint2 FK[2][3][2][64];        // K (rows s, columns t); GLA: CB o G2, read a chunk later
  float sc[3][4][Q];            // step scalars: gam, m31, cd (GLA: gates), w
  float X[2][S::NW][Q], Y[2][S::NW][Q], BZ[2][S::NW][Q], tr[2][S::NW];   // row sums by wave
  float R[2][4][16];            // SSD: blocks of R_t: [0] t < 16 own, [1] t < 16 from rows >= 16, [2] t >= 16 own,
                                // [3] row sums of the lower left block
};

// m 2^e as two factors: a segment's decay may overflow (gates above 1) where its
// product with a small or zero adjoint does not.  The second one is 1 within
// fp32's range.
__device__ __forceinline__ float2 scaled(float m, int e) {
  const int e1 = min(max(e, -100), 100), e2 = min(max(e - e1, -126), 126);
  return make_float2(ldexpf(m, e1), ldexpf(1.f, e2));
}

// The decays M[t][s] of 16x16 block blk (0: t, s < 16; 1: t >= 16, s < 16; 2:
// both >= 16): ROWS_T: t = 4 g + r, s = l15; else s = 4 g + r, t = l15.  Zero for
// s > t.  STRICT (GLA): M[t - 1][s], zero for s >= t.
template <bool GLA, bool ROWS_T, bool STRICT = false>
__device__ __forceinline__ void decays(const float* st, float a, int blk, int l15, int g, float (&m)[4]) {
  const int s0 = blk == 2 ? 16 : 0, t0 = blk > 0 ? 16 : 0;
  const float4 rq = *reinterpret_cast<const float4*>(&st[(ROWS_T ? t0 : s0) + 4 * g]);
  const float rv[4] = {rq.x, rq.y, rq.z, rq.w};
  if constexpr (!GLA) {
    const float cv = st[(ROWS_T ? s0 : t0) + l15];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      m[r] = rr::chunked::masked_exp(blk == 1 || (ROWS_T ? l15 <= 4 * g + r : 4 * g + r <= l15),
                                     a * (ROWS_T ? rv[r] - cv : cv - rv[r]));
  } else {
    // products of the gates of steps s + 1 .. t (STRICT: t - 1), by quads of
    // steps: the rest of s's quad, whole quads between, t's quad up to t
    const int qc = l15 >> 2, pc = l15 & 3;   // the lane's quad and position (ROWS_T: s, else t)
    const float4 cq = *reinterpret_cast<const float4*>(&st[(ROWS_T ? s0 : t0) + 4 * qc]);
    const float c01 = cq.x * cq.y, c012 = c01 * cq.z, c0123 = c012 * cq.w, c23 = cq.z * cq.w;
    auto quad = [&](int j) {
      const float4 q = *reinterpret_cast<const float4*>(&st[4 * j]);
      return (q.x * q.y) * (q.z * q.w);
    };
    const int qs = ROWS_T ? qc : g, qt = ROWS_T ? g : qc;   // quads of s and t within their 16 steps
    float mid;
    if (blk == 1) {
      const float q1 = quad(1), q2 = quad(2), q3 = quad(3), q4 = quad(4), q5 = quad(5), q6 = quad(6);
      mid = ((qs < 1 ? q1 : 1.f) * (qs < 2 ? q2 : 1.f)) * (qs < 3 ? q3 : 1.f);
      mid *= ((qt > 0 ? q4 : 1.f) * (qt > 1 ? q5 : 1.f)) * (qt > 2 ? q6 : 1.f);
    } else {
      const float q1 = quad(s0 / 4 + 1), q2 = quad(s0 / 4 + 2);
      mid = (qs < 1 && qt > 1 ? q1 : 1.f) * (qs < 2 && qt > 2 ? q2 : 1.f);
    }
    const bool same = blk != 1 && qs == qt;
    if constexpr (ROWS_T) {
      // s fixed: rest of its quad, then t's quad (rows) up to r
      const float rest = pc == 0 ? cq.y * c23 : pc == 1 ? c23 : pc == 2 ? cq.w : 1.f;
      const float base = rest * mid;
      const float u1 = rv[0] * rv[1], u2 = u1 * rv[2], u3 = u2 * rv[3];
      const float up[4] = {rv[0], u1, u2, u3};
      // own quad: positions pc + 1 .. r
      const float in1 = pc == 0 ? rv[1] : 1.f, in2 = pc == 0 ? rv[1] * rv[2] : pc == 1 ? rv[2] : 1.f;
      const float in3 = in2 * (pc < 3 ? rv[3] : 1.f);
      const float inq[4] = {1.f, in1, in2, in3};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float v = same ? inq[r] : base * up[r];
        m[r] = blk == 1 || l15 <= 4 * g + r ? v : 0.f;
      }
    } else {
      // t fixed: its quad up to t (STRICT: t - 1), rest of s's quad (rows) after r
      const float up = STRICT ? (pc == 0 ? 1.f : pc == 1 ? cq.x : pc == 2 ? c01 : c012)
                              : (pc == 0 ? cq.x : pc == 1 ? c01 : pc == 2 ? c012 : c0123);
      const float base = mid * up;
      const float r2 = rv[3], r1 = rv[2] * r2, r0 = rv[1] * r1;
      const float rest[4] = {r0, r1, r2, 1.f};
      // own quad: positions r + 1 .. pc (STRICT: pc - 1)
      const int pe = STRICT ? pc - 1 : pc;
      const float yz = rv[1] * rv[2];
      const float in0 = pe < 1 ? 1.f : pe == 1 ? rv[1] : pe == 2 ? yz : yz * rv[3];
      const float in1 = pe < 2 ? 1.f : pe == 2 ? rv[2] : rv[2] * rv[3];
      const float in2 = pe < 3 ? 1.f : rv[3];
      const float inq[4] = {in0, in1, in2, 1.f};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float v = same ? inq[r] : rest[r] * base;
        m[r] = blk == 1 || (STRICT ? 4 * g + r < l15 : 4 * g + r <= l15) ? v : 0.f;
      }
    }
  }
}

template <int DH, int NS, bool GLA, bool MAP>
__global__ __launch_bounds__((Shape<DH, NS>::T), 2) void walk_bwd_kernel(WalkArgs q) {
  using S = Shape<DH, NS>;
  constexpr int NW = S::NW, T = S::T, NBN = S::NBN, NBD = S::NBD, NK = S::NK, DK = S::DK, CPW = S::CPW, DPW = S::DPW;
  constexpr int UV = Q * DH / 8 / T, BV = Q * NS / 8 / T, GV = Q * DH / 4 / T;
  static_assert(UV * T * 8 == Q * DH && BV * T * 8 == Q * NS, "whole pieces per thread");
  const rr::ChunkArgs& p = q.p;
  __shared__ WalkSm<DH, NS, GLA> sm;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int tid = threadIdx.x, lane = tid & 63, l15 = lane & 15, g = lane >> 4;   // refreshed per chunk, see the loop
  const int bh = blockIdx.x, seg = MAP ? blockIdx.y + 1 : blockIdx.y, h = bh % p.H, b = bh / p.H;
  const int c0 = seg * q.cps, c1 = min(c0 + q.cps, p.nC);
  const float a = rr::chunked::head_rate<GLA>(p, h);
  const uint32_t rsN = (uint32_t)p.H * NS, rsD = (uint32_t)p.H * DH;

  u16x8_t uv[UV], bv[BV], cv[BV];
  float4 gv[GV];
  float xv;                 // step input of the chunk whose scalars come next
  f32x4_t hin[CPW][NBD];    // h_in[16 db + 4 g + r][16 nb + l15], nb = w CPW + cc
  auto load = [&](int c) {
    const int64_t row0 = (int64_t)b * p.L + (int64_t)max(c, 0) * Q;
    const uint16_t* Bp = p.Bm + (row0 * p.H + h) * NS;
    const uint16_t* Cp = p.Cm + (row0 * p.H + h) * NS;
    const uint16_t* Up = p.u + (row0 * p.H + h) * DH;
    const float* Yp = p.dy + (row0 * p.H + h) * DH;
#pragma unroll
    for (int v = 0; v < BV; ++v) {
      const int i = tid + T * v;
      const uint32_t o = (uint32_t)(i / (NS / 8)) * rsN + 8 * (i % (NS / 8));
      cv[v] = rr::ld32<u16x8_t>(Cp, o);
      if constexpr (!MAP) bv[v] = rr::ld32<u16x8_t>(Bp, o);
    }
#pragma unroll
    for (int v = 0; v < GV; ++v) {
      const int i = tid + T * v;
      gv[v] = rr::ld32<float4>(Yp, (uint32_t)(i / (DH / 4)) * rsD + 4 * (i % (DH / 4)));
    }
    if constexpr (!MAP) {
#pragma unroll
      for (int v = 0; v < UV; ++v) {
        const int i = tid + T * v;
        uv[v] = rr::ld32<u16x8_t>(Up, (uint32_t)(i / (DH / 8)) * rsD + 8 * (i % (DH / 8)));
      }
    }
  };
  auto load_step = [&](int c) {
    xv = rr::bf_val(p.delta[((int64_t)b * p.L + (int64_t)max(c, 0) * Q + (lane & (Q - 1))) * p.H + h]);
  };
  // the state entering chunk c: checkpoint c - 1, h0, or zero (a valid read, dropped)
  auto load_h = [&](int c) {
    const bool ck = c > 0;
    const float* src = ck ? p.ckpt + ((int64_t)bh * p.nC + c - 1) * DH * NS
                          : (p.h0 != nullptr ? p.h0 + (int64_t)bh * DH * NS : p.ckpt);
    const auto hs = rr::as_global(src);
    const int sd = GLA && !ck ? 1 : NS, sn = GLA && !ck ? DH : 1;   // element strides of d and n
#pragma unroll
    for (int cc = 0; cc < CPW; ++cc) {
      const uint32_t o = (uint32_t)((16 * (w * CPW + cc) + l15) * sn + 4 * g * sd);
#pragma unroll
      for (int db = 0; db < NBD; ++db)
#pragma unroll
        for (int r = 0; r < 4; ++r) hin[cc][db][r] = rr::ld32<float>(hs + (16 * db + r) * sd, o);
    }
  };
  auto scalars = [&](int c) {   // one wave
    const rr::chunked::StepScalars st = rr::chunked::step_scalars<GLA>(lane < Q ? xv : (GLA ? 1.f : 0.f), a, lane);
    float(*sc)[Q] = sm.sc[c % 3];
    if (lane < Q) {
      sc[0][lane] = st.gam;
      sc[1][lane] = st.m31;
      sc[2][lane] = GLA ? xv : st.cd;
      sc[3][lane] = st.w;
    }
  };
  auto stage = [&](int c) {
    const float* gam = sm.sc[c % 3][0];
    auto put16 = [&](uint16_t* img, auto len, int t, int m, const u16x8_t& v) {
      const uint4 x = __builtin_bit_cast(uint4, v);
      *reinterpret_cast<uint2*>(img + piece<decltype(len)::value>(t, 2 * m)) = make_uint2(x.x, x.y);
      *reinterpret_cast<uint2*>(img + piece<decltype(len)::value>(t, 2 * m + 1)) = make_uint2(x.z, x.w);
    };
#pragma unroll
    for (int v = 0; v < BV; ++v) {
      const int i = tid + T * v, t = i / (NS / 8), m = i % (NS / 8);
      put16(sm.C, std::integral_constant<int, NS>{}, t, m, cv[v]);
      if constexpr (!MAP) put16(sm.B, std::integral_constant<int, NS>{}, t, m, bv[v]);
    }
    if constexpr (!MAP) {
#pragma unroll
      for (int v = 0; v < UV; ++v) {
        const int i = tid + T * v;
        put16(sm.U, std::integral_constant<int, DH>{}, i / (DH / 8), i % (DH / 8), uv[v]);
      }
    }
#pragma unroll
    for (int v = 0; v < GV; ++v) {
      const int i = tid + T * v, t = i / (DH / 4), o = piece<DH>(t, i % (DH / 4));
      const float gt = gam[t];
      u16x4_t hi, lo;
      if constexpr (!MAP) {
        rr::bf_split4(f32x4_t{gv[v].x, gv[v].y, gv[v].z, gv[v].w}, hi, lo);
        *reinterpret_cast<u16x4_t*>(sm.Yh + o) = hi;
        *reinterpret_cast<u16x4_t*>(sm.Yl + o) = lo;
      }
      rr::bf_split4(f32x4_t{gt * gv[v].x, gt * gv[v].y, gt * gv[v].z, gt * gv[v].w}, hi, lo);
      *reinterpret_cast<u16x4_t*>(sm.Gh + o) = hi;
      *reinterpret_cast<u16x4_t*>(sm.Gl + o) = lo;
    }
  };

  f32x4_t lc[CPW][NBD];    // lam[16 db + 4 g + r][16 nb + l15]
  f32x4_t lr[DPW][NBN];    // lam[16 (w DPW + dd) + l15][16 nb + 4 g + r]
#pragma unroll
  for (int cc = 0; cc < CPW; ++cc)
#pragma unroll
    for (int db = 0; db < NBD; ++db) lc[cc][db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int dd = 0; dd < DPW; ++dd)
#pragma unroll
    for (int nb = 0; nb < NBN; ++nb) lr[dd][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float decay = 1.f;   // MAP: the segment's decay is decay 2^decay_e
  int decay_e = 0;
  load(c1 - 1);
  load_step(c1 - 1);
  constexpr int MF = CPW * NBD + DPW * NBN;   // float4 per thread of a map
  if constexpr (!MAP) {
    if (p.dfinal != nullptr) {
      const float* dp = p.dfinal + (int64_t)bh * DH * NS;
#pragma unroll
      for (int cc = 0; cc < CPW; ++cc)
#pragma unroll
        for (int db = 0; db < NBD; ++db)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            lc[cc][db][r] = dp[rr::chunked::state_off<GLA, DH, NS>(16 * db + 4 * g + r, 16 * (w * CPW + cc) + l15)];
#pragma unroll
      for (int dd = 0; dd < DPW; ++dd)
#pragma unroll
        for (int nb = 0; nb < NBN; ++nb)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            lr[dd][nb][r] = dp[rr::chunked::state_off<GLA, DH, NS>(16 * (w * DPW + dd) + l15, 16 * nb + 4 * g + r)];
    }
    const float4* E = q.mapL + rr::chunked::map_slot(bh, q.S, 0) * (MF * T) + tid;
    for (int j = q.S - 1; j > seg; --j) {
      const float2 P = q.mapP[rr::chunked::map_slot(bh, q.S, j - 1)];
      const float4* e = E + (int64_t)(j - 1) * MF * T;
#pragma unroll
      for (int cc = 0; cc < CPW; ++cc)
#pragma unroll
        for (int db = 0; db < NBD; ++db) {
          const float4 v = e[(cc * NBD + db) * T];
          lc[cc][db] = f32x4_t{v.x, v.y, v.z, v.w} + P.x * (P.y * lc[cc][db]);
        }
#pragma unroll
      for (int dd = 0; dd < DPW; ++dd)
#pragma unroll
        for (int nb = 0; nb < NBN; ++nb) {
          const float4 v = e[(CPW * NBD + dd * NBN + nb) * T];
          lr[dd][nb] = f32x4_t{v.x, v.y, v.z, v.w} + P.x * (P.y * lr[dd][nb]);
        }
    }
  }
  float dAt[CPW][4], dAh[CPW];   // SSD dA: terms summed over t (lanes l15; n = 4 g + r), over d (n = l15)
#pragma unroll
  for (int cc = 0; cc < CPW; ++cc) {
    dAh[cc] = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) dAt[cc][r] = 0.f;
  }

  // the step gradient of chunk c from its row sums (one wave, a chunk later)
  auto step_grad = [&](int c) {
    const int par = c & 1, t = lane & 31;
    const float(*sc)[Q] = sm.sc[c % 3];
    float X = 0.f, Y = 0.f, tr = 0.f;
#pragma unroll
    for (int k = 0; k < NW; ++k) {
      X += sm.X[par][k][t];
      Y += sm.Y[par][k][t];
      tr += sm.tr[par][k];
    }
    const int64_t row0 = (int64_t)b * p.L + (int64_t)c * Q;
    if constexpr (!GLA) {
      float bz = 0.f;
#pragma unroll
      for (int k = 0; k < NW; ++k) bz += sm.BZ[par][k][t];
      // lanes 0-31, step 31 - lane: suffix sums of gam X and of the lower left
      // block's row sums; lanes 32-63: prefix of m31 w Y
      const float gx = sc[0][t] * X, wy = sc[1][t] * sc[3][t] * Y;
      const float gxr = __shfl(gx, 31 - t);
      const float pre = rr::prefix32_sum(lane < Q ? gxr : wy);
      const float sx = __shfl(pre, 31 - t), py = __shfl(pre, 32 + t);
      const float rt = sm.R[par][3][15 - (t & 15)];
      const float rsum = rr::prefix32_sum(t < 16 ? rt : 0.f);   // lane 31 - t: rows t .. 31
      const float rsx = __shfl(rsum, 31 - t);
      const float R = t < 16 ? sm.R[par][0][t] + sm.R[par][1][t] : sm.R[par][2][t - 16] + rsx;
      const float Tt = R + sx + py + sc[1][t] * sc[0][t] * tr;
      if (lane < Q) rr::st_bf16(p.ddelta, (row0 + t) * p.H + h, a * Tt + (1.f - a * sc[3][t]) * bz);
    } else {
      // D[t'][t] = ((CB o G2) Mh)[t'][t] by blocks (t' >= t), t = column
      const float* st = sc[2];
      float m00[4], m01[4], m11[4];
      decays<true, false, true>(st, 0.f, 0, l15, g, m00);
      decays<true, false, true>(st, 0.f, 1, l15, g, m01);
      decays<true, false, true>(st, 0.f, 2, l15, g, m11);
      const f32x4_t z4 = {0.f, 0.f, 0.f, 0.f};
      u16x8_t b0h, b0l, b1h, b1l;
      split_pair(f32x4_t{m00[0], m00[1], m00[2], m00[3]}, z4, b0h, b0l);
      split_pair(f32x4_t{m01[0], m01[1], m01[2], m01[3]}, f32x4_t{m11[0], m11[1], m11[2], m11[3]}, b1h, b1l);
      const uint2 zz = make_uint2(0, 0);
      const uint2(*FK)[2][64] = sm.FK[par];
      const u16x8_t e0h = join(FK[0][0][lane], zz), e0l = join(FK[0][1][lane], zz);
      const u16x8_t e1h = join(FK[1][0][lane], FK[2][0][lane]), e1l = join(FK[1][1][lane], FK[2][1][lane]);
      auto mm = [&](const u16x8_t& ah, const u16x8_t& al, const u16x8_t& bh_, const u16x8_t& bl) {
        f32x4_t x = mfma16(al, bh_, z4);
        x = mfma16(ah, bl, x);
        return mfma16(ah, bh_, x);
      };
      const f32x4_t d00 = mm(e0h, e0l, b0h, b0l), d10 = mm(e1h, e1l, b0h, b0l), d11 = mm(e1h, e1l, b1h, b1l);
      float n00[4], n10[4], n11[4];   // M[t'][t], rows t'
      decays<true, true>(st, 0.f, 0, l15, g, n00);
      decays<true, true>(st, 0.f, 1, l15, g, n10);
      decays<true, true>(st, 0.f, 2, l15, g, n11);
      // row sums X, Y at rows 4 g + r
      float x0[4], x1[4], y0[4], y1[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x0[r] = __shfl(X, 4 * g + r);
        x1[r] = __shfl(X, 16 + 4 * g + r);
        y0[r] = __shfl(Y, 4 * g + r);
        y1[r] = __shfl(Y, 16 + 4 * g + r);
      }
      const float gp0 = l15 > 0 ? sc[0][(l15 + Q - 1) & (Q - 1)] : 1.f, gp1 = sc[0][15 + l15];
      float s0 = 0.f, s1 = 0.f, p0 = 0.f, p1 = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s0 += n00[r] * (d00[r] + x0[r] * gp0) + n10[r] * (d10[r] + x1[r] * gp0);
        s1 += n11[r] * (d11[r] + x1[r] * gp1);
        p0 += m00[r] * y0[r];
        p1 += m01[r] * y0[r] + m11[r] * y1[r];
      }
      s0 = rr::rows4_sum(s0), s1 = rr::rows4_sum(s1), p0 = rr::rows4_sum(p0), p1 = rr::rows4_sum(p1);
      const float v0 = s0 + sc[1][l15] * (p0 + gp0 * tr), v1 = s1 + sc[1][16 + l15] * (p1 + gp1 * tr);
      if (g == 0) rr::st_bf16(p.ddelta, (row0 + l15) * p.H + h, v0);
      if (g == 1) rr::st_bf16(p.ddelta, (row0 + 16 + l15) * p.H + h, v1);
    }
  };

  // masked products of 16x16 block blk, both orientations
  auto masked = [&](int c, int blk) {
    const float(*sc)[Q] = sm.sc[c % 3];
    const int tr0 = blk > 0 ? 16 : 0, sr0 = blk == 2 ? 16 : 0, par = c & 1;
    f32x4_t cb = {0.f, 0.f, 0.f, 0.f}, cbt = cb, g2 = cb, g2t = cb;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      const u16x8_t cf = row_frag<NS>(sm.C, tr0 + l15, kk, g), bf = row_frag<NS>(sm.B, sr0 + l15, kk, g);
      cb = mfma16(cf, bf, cb);                          // rows t, columns s
      if constexpr (GLA) cbt = mfma16(bf, cf, cbt);     // rows s, columns t
    }
#pragma unroll
    for (int kk = 0; kk < DK; ++kk) {
      const u16x8_t yh = row_frag<DH>(sm.Yh, tr0 + l15, kk, g), yl = row_frag<DH>(sm.Yl, tr0 + l15, kk, g);
      const u16x8_t uf = row_frag<DH>(sm.U, sr0 + l15, kk, g);
      g2 = mfma16(yl, uf, g2);
      g2 = mfma16(yh, uf, g2);
      g2t = mfma16(uf, yl, g2t);
      g2t = mfma16(uf, yh, g2t);
    }
    auto put = [&](uint2(*dst)[64], const float (&v)[4]) {
      u16x4_t hi, lo;
      rr::bf_split4(f32x4_t{v[0], v[1], v[2], v[3]}, hi, lo);
      dst[0][lane] = __builtin_bit_cast(uint2, hi);
      dst[1][lane] = __builtin_bit_cast(uint2, lo);
    };
    float m[4], v[4], x[4];
    decays<GLA, true>(sc[2], a, blk, l15, g, m);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[r] = m[r] * cb[r];
      x[r] = m[r] * g2[r];
    }
    put(sm.F[kP][blk], v);
    put(sm.F[kMG][blk], x);
    if constexpr (!GLA) {
      // R_t = sum_{t' >= t, s <= t} (M o w_s o G2 o CB)[t'][s]: prefix over s
      // along the 16 lanes of a row, then the rows t' of column s = t
      const float ws = sc[3][sr0 + l15];
      float rs = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float k = x[r] * ws * cb[r];
        k += rr::dpp_in<0x111, 0xF>(k);
        k += rr::dpp_in<0x112, 0xF>(k);
        k += rr::dpp_in<0x114, 0xF>(k);
        k += rr::dpp_in<0x118, 0xF>(k);
        rs += blk == 1 || 4 * g + r >= l15 ? k : 0.f;
        if (blk == 1 && l15 == 15) sm.R[par][3][4 * g + r] = k;
      }
      rs = rr::rows4_sum(rs);
      if (g == 0) sm.R[par][blk][l15] = rs;
    }
    decays<GLA, false>(sc[2], a, blk, l15, g, m);
    const float4 w4 = *reinterpret_cast<const float4*>(&sc[3][sr0 + 4 * g]);
    const float wv[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = m[r] * g2t[r] * wv[r];
    put(sm.F[kMGw][blk], v);
    if constexpr (!GLA) {
      const float4 c4 = *reinterpret_cast<const float4*>(&sc[2][sr0 + 4 * g]);
      const float cs[4] = {c4.x, c4.y, c4.z, c4.w}, ct = sc[2][tr0 + l15];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] *= ct - cs[r];
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = blk == 1 || 4 * g + r <= l15 ? cbt[r] * g2t[r] : 0.f;
    }
    put(sm.FK[par][blk], v);
  };

  if (w == NW - 1) scalars(c1 - 1);
  load_step(c1 - 2);
  if constexpr (!MAP) load_h(c1 - 1);   // (last, as in the loop: waits for older loads count past it)
  lds_barrier();

  for (int c = c1 - 1; c >= c0; --c) {
    // opaque copies per chunk keep the compiler from holding every lane address
    // of the body in a register across the loop
    asm volatile("" : "+v"(tid), "+v"(lane), "+v"(l15), "+v"(g));
    const int par = c & 1;
    const float(*sc)[Q] = sm.sc[c % 3];
    stage(c);
    if constexpr (MAP) load(c - 1);
    lds_barrier();   // rows staged
    const float g31 = sc[0][Q - 1];
    // ---- wave 3 (MAP: the last): the next chunk's scalars, the last chunk's step gradient
    if (w == (MAP ? NW - 1 : 3)) {
      if (c > c0) scalars(c - 1);
      if constexpr (!MAP) {
        if (c + 1 < c1) step_grad(c + 1);
      }
    }
    load_step(c - 2);
    f32x4_t gh[MAP ? 1 : CPW][2], ul[MAP ? 1 : CPW][2];   // GH^T[n][t], UL^T[n][s]
    if constexpr (!MAP) {
      if (w < 3) masked(c, w);
      if (c == 0 && p.h0 == nullptr) {   // a zero start (load_h read the last row it may)
#pragma unroll
        for (int cc = 0; cc < CPW; ++cc)
#pragma unroll
          for (int db = 0; db < NBD; ++db) hin[cc][db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
      // ---- GH, UL of this wave's columns, their row sums, lam o h_in
      float xs[2] = {0.f, 0.f}, ys[2] = {0.f, 0.f}, trp = 0.f;
#pragma unroll
      for (int cc = 0; cc < CPW; ++cc) {
        float s = 0.f;
#pragma unroll
        for (int db = 0; db < NBD; ++db)
#pragma unroll
          for (int r = 0; r < 4; ++r) s += lc[cc][db][r] * hin[cc][db][r];
        trp += s;
        if constexpr (!GLA) dAh[cc] += g31 * sc[2][Q - 1] * s;
#pragma unroll
        for (int k = 0; k < 2; ++k) gh[cc][k] = ul[cc][k] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int kk = 0; kk < DK; ++kk) {
        u16x8_t hh[CPW], hl[CPW], lh[CPW], ll[CPW];
#pragma unroll
        for (int cc = 0; cc < CPW; ++cc) {
          split_pair(hin[cc][2 * kk], hin[cc][2 * kk + 1], hh[cc], hl[cc]);
          split_pair(lc[cc][2 * kk], lc[cc][2 * kk + 1], lh[cc], ll[cc]);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const u16x8_t yh = row_frag<DH>(sm.Yh, 16 * k + l15, kk, g), yl = row_frag<DH>(sm.Yl, 16 * k + l15, kk, g);
          const u16x8_t uf = row_frag<DH>(sm.U, 16 * k + l15, kk, g);
#pragma unroll
          for (int cc = 0; cc < CPW; ++cc) {
            gh[cc][k] = mfma16(hl[cc], yh, gh[cc][k]);
            ul[cc][k] = mfma16(ll[cc], uf, ul[cc][k]);
            gh[cc][k] = mfma16(hh[cc], yl, gh[cc][k]);
            ul[cc][k] = mfma16(lh[cc], uf, ul[cc][k]);
            gh[cc][k] = mfma16(hh[cc], yh, gh[cc][k]);
          }
        }
      }
      load_h(c - 1 >= c0 ? c - 1 : c);   // (the segment's first chunk repeats itself)
#pragma unroll
      for (int cc = 0; cc < CPW; ++cc)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int pc = 4 * (w * CPW + cc) + g;
          const uint2 c4 = *reinterpret_cast<const uint2*>(sm.C + piece<NS>(16 * k + l15, pc));
          const uint2 b4 = *reinterpret_cast<const uint2*>(sm.B + piece<NS>(16 * k + l15, pc));
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            xs[k] += gh[cc][k][r] * bf4(c4, r);
            ys[k] += ul[cc][k][r] * bf4(b4, r);
          }
        }
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const float x = rr::rows4_sum(xs[k]), y = rr::rows4_sum(ys[k]);
        if (g == 0) {
          sm.X[par][w][16 * k + l15] = x;
          sm.Y[par][w][16 * k + l15] = y;
        }
      }
      trp = rr::wave_sum(trp);
      if (lane == 0) sm.tr[par][w] = trp;
      lds_barrier();   // fragments and row sums
      // ---- dB, dC (dA terms) of this wave's columns
      const uint2 zz = make_uint2(0, 0);
      const int64_t row0 = (int64_t)b * p.L + (int64_t)c * Q;
      {
        const float cd31 = GLA ? 0.f : sc[2][Q - 1];
        uint16_t* const dBp = p.dB + (row0 * p.H + h) * NS;
        uint16_t* const dCp = p.dC + (row0 * p.H + h) * NS;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          // k = 0: columns (s or t) 0-15, rows of the other index 0-31 resp. 0-15; k = 1: columns 16-31
          u16x8_t mg[2], mw[2], km[2];
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            mg[x] = k == 0 ? join(sm.F[kMG][0][x][lane], sm.F[kMG][1][x][lane]) : join(zz, sm.F[kMG][2][x][lane]);
            mw[x] = k == 0 ? join(sm.F[kMGw][0][x][lane], zz)
                           : join(sm.F[kMGw][1][x][lane], sm.F[kMGw][2][x][lane]);
            if constexpr (!GLA)
              km[x] = k == 0 ? join(sm.FK[par][0][x][lane], zz) : join(sm.FK[par][1][x][lane], sm.FK[par][2][x][lane]);
          }
          const int t = 16 * k + l15;
          const float gt = sc[0][t], m31 = sc[1][t], wt = sc[3][t], cdt = GLA ? 0.f : sc[2][t];
          float bz = 0.f;
#pragma unroll
          for (int cc = 0; cc < CPW; ++cc) {
            const int nb = w * CPW + cc;
            const u16x8_t ct = col_frag<NS>(sm.C, nb, l15, g), bt = col_frag<NS>(sm.B, nb, l15, g);
            f32x4_t z = {0.f, 0.f, 0.f, 0.f}, dc = z, kb = z;
            z = mfma16(ct, mg[1], z);
            dc = mfma16(bt, mw[1], dc);
            z = mfma16(ct, mg[0], z);
            dc = mfma16(bt, mw[0], dc);
            if constexpr (!GLA) {
              kb = mfma16(bt, km[1], kb);
              kb = mfma16(bt, km[0], kb);
            }
            const uint2 b4 = *reinterpret_cast<const uint2*>(sm.B + piece<NS>(t, 4 * nb + g));
            const uint2 c4 = *reinterpret_cast<const uint2*>(sm.C + piece<NS>(t, 4 * nb + g));
            float db4[4], dc4[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float u = m31 * ul[cc][k][r], zt = z[r] + u, gg = gt * gh[cc][k][r];
              db4[r] = wt * zt;
              dc4[r] = gg + dc[r];
              if constexpr (!GLA) {
                const float bb = bf4(b4, r);
                bz += bb * zt;
                dAt[cc][r] += bf4(c4, r) * (kb[r] + cdt * gg) + (cd31 - cdt) * wt * bb * u;
              }
            }
            const uint32_t o = (uint32_t)t * rsN + 16 * nb + 4 * g;
            *reinterpret_cast<uint2*>(reinterpret_cast<char*>(dBp) + 2 * o) = pack4(db4);
            *reinterpret_cast<uint2*>(reinterpret_cast<char*>(dCp) + 2 * o) = pack4(dc4);
          }
          if constexpr (!GLA) {
            bz = rr::rows4_sum(bz);
            if (g == 0) sm.BZ[par][w][t] = bz;
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);   // keeps the phases' operands from living at once
      // (here, not before: the registers of GH and UL are free now; a spilled
      // address or step input would make the wave wait for all of these at once)
      load(c - 1);
      // ---- du of this wave's rows
      uint16_t* const duP = p.du + (row0 * p.H + h) * DH;
#pragma unroll
      for (int dd = 0; dd < DPW; ++dd) {
        const int db = w * DPW + dd;
        const u16x8_t yh = col_frag<DH>(sm.Yh, db, l15, g), yl = col_frag<DH>(sm.Yl, db, l15, g);   // dY[pi][d]
        f32x4_t a1[2], a2[2];
        a1[0] = a1[1] = a2[0] = a2[1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) {
          u16x8_t lh, ll;
          split_pair(lr[dd][2 * kk], lr[dd][2 * kk + 1], lh, ll);
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const u16x8_t bf = row_frag<NS>(sm.B, 16 * k + l15, kk, g);
            a2[k] = mfma16(ll, bf, a2[k]);
            a2[k] = mfma16(lh, bf, a2[k]);
          }
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const u16x8_t ph = k == 0 ? join(sm.F[kP][0][0][lane], sm.F[kP][1][0][lane]) : join(zz, sm.F[kP][2][0][lane]);
          const u16x8_t pl = k == 0 ? join(sm.F[kP][0][1][lane], sm.F[kP][1][1][lane]) : join(zz, sm.F[kP][2][1][lane]);
          a1[k] = mfma16(yl, ph, a1[k]);
          a1[k] = mfma16(yh, pl, a1[k]);
          a1[k] = mfma16(yh, ph, a1[k]);
          const int s = 16 * k + l15;
          const float ws = sc[3][s], m31 = sc[1][s];
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = ws * (a1[k][r] + m31 * a2[k][r]);
          *reinterpret_cast<uint2*>(reinterpret_cast<char*>(duP) + 2 * ((uint32_t)s * rsD + 16 * db + 4 * g)) = pack4(v);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- lam <- gam_31 lam + (gam o dY)^T C, both copies
    {
      u16x8_t own[DPW][2];   // gam o dY of this wave's rows d
#pragma unroll
      for (int dd = 0; dd < DPW; ++dd) {
        own[dd][0] = col_frag<DH>(sm.Gh, w * DPW + dd, l15, g);
        own[dd][1] = col_frag<DH>(sm.Gl, w * DPW + dd, l15, g);
      }
      u16x8_t cf[CPW];
#pragma unroll
      for (int cc = 0; cc < CPW; ++cc) cf[cc] = col_frag<NS>(sm.C, w * CPW + cc, l15, g);
#pragma unroll
      for (int db = 0; db < NBD; ++db) {
        const u16x8_t gh_ = col_frag<DH>(sm.Gh, db, l15, g), gl_ = col_frag<DH>(sm.Gl, db, l15, g);
#pragma unroll
        for (int cc = 0; cc < CPW; ++cc) {
          f32x4_t z = {0.f, 0.f, 0.f, 0.f};
          z = mfma16(gl_, cf[cc], z);
          z = mfma16(gh_, cf[cc], z);
          lc[cc][db] = z + g31 * lc[cc][db];
        }
      }
#pragma unroll
      for (int nb = 0; nb < NBN; ++nb) {
        const u16x8_t ct = col_frag<NS>(sm.C, nb, l15, g);
#pragma unroll
        for (int dd = 0; dd < DPW; ++dd) {
          f32x4_t z = {0.f, 0.f, 0.f, 0.f};
          z = mfma16(ct, own[dd][1], z);
          z = mfma16(ct, own[dd][0], z);
          lr[dd][nb] = z + g31 * lr[dd][nb];
        }
      }
    }
    if constexpr (MAP) {
      decay *= g31;
      decay_e += __builtin_amdgcn_frexp_expf(decay);
      decay = __builtin_amdgcn_frexp_mantf(decay);
    }
    lds_barrier();   // every row image and fragment read
  }

  if constexpr (MAP) {
    float4* E = q.mapL + rr::chunked::map_slot(bh, q.S, seg - 1) * (MF * T) + tid;
#pragma unroll
    for (int cc = 0; cc < CPW; ++cc)
#pragma unroll
      for (int db = 0; db < NBD; ++db)
        E[(cc * NBD + db) * T] = make_float4(lc[cc][db][0], lc[cc][db][1], lc[cc][db][2], lc[cc][db][3]);
#pragma unroll
    for (int dd = 0; dd < DPW; ++dd)
#pragma unroll
      for (int nb = 0; nb < NBN; ++nb)
        E[(CPW * NBD + dd * NBN + nb) * T] =
            make_float4(lr[dd][nb][0], lr[dd][nb][1], lr[dd][nb][2], lr[dd][nb][3]);
    if (tid == 0) q.mapP[rr::chunked::map_slot(bh, q.S, seg - 1)] = scaled(decay, decay_e);
  } else {
    if (w == 3) step_grad(c0);
    if constexpr (!GLA) {
      // dA partial of the segment: terms over t by lane, over d by lane group
      float* red = sm.X[(c0 + 1) & 1][0];   // NS <= 32 NW floats, the row sums no one reads any more
      static_assert(NS <= Q * NW, "dA reduction space");
#pragma unroll
      for (int cc = 0; cc < CPW; ++cc)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = rr::row16_sum(dAt[cc][r]);
          if (l15 == 0) red[16 * (w * CPW + cc) + 4 * g + r] = v;
        }
      rr::wave_lds_sync();
#pragma unroll
      for (int cc = 0; cc < CPW; ++cc) {
        const float v = rr::rows4_sum(dAh[cc]);
        const int n = 16 * (w * CPW + cc) + l15;
        if (g == 0) p.ws[rr::chunked::dA_slot(bh, q.S, seg) * NS + n] = red[n] + v;
      }
    }
    if (seg == 0 && p.dh0 != nullptr) {
#pragma unroll
      for (int cc = 0; cc < CPW; ++cc)
#pragma unroll
        for (int db = 0; db < NBD; ++db)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            p.dh0[(int64_t)bh * DH * NS +
                  rr::chunked::state_off<GLA, DH, NS>(16 * db + 4 * g + r, 16 * (w * CPW + cc) + l15)] = lc[cc][db][r];
    }
  }
}

// ------------------------------------------------------------------ host
// Segments of a head: the count with the least estimated time, in chunks walked
// one after another.  The CUs hold `slots` workgroups (by registers and LDS); a
// round of them walks cps chunks plus about two for its start, a last round
// that fills at most half of the slots runs faster; the maps of all but one
// segment cost a quarter of a walk, and reading them 0.3 each.  At least four
// chunks a segment.  (Measured: SSD B8 L4096 H80 Dh64 N128 3411 us with 1
// segment, 3232 with 2, 3317 with 3, 3287 with 4; GLA B8 L2048 H12 Dh128 672,
// 523, 556, 529 and 489 with 5.)
void segments(int64_t BH, int64_t nC, int64_t Dh, int64_t N, int& S, int& cps) {
  const int per_cu = Dh == 64 && N == 64 ? 3 : Dh == 128 && N == 128 ? 1 : 2;
  const double slots = 256.0 * per_cu;
  double best = 0;
  S = 0;
  for (int64_t want = 1; want <= std::max<int64_t>(1, std::min<int64_t>(nC / 4, 64)); ++want) {
    const int64_t c = (nC + want - 1) / want, s = (nC + c - 1) / c;
    const double r = (double)(BH * s) / slots, full = (double)(int64_t)r, part = r - full;
    const double rounds = full + (part == 0 ? 0 : part <= 0.5 && per_cu > 1 && full > 0 ? 0.65 : 1);
    const double t = rounds * (double)(c + 2) * (1 + 0.24 * (double)(s - 1) / (double)s) + 0.3 * (double)(s - 1);
    if (S == 0 || t < best) best = t, S = (int)s, cps = (int)c;
  }
}

// Workspace floats: both layouts of every map, then the decays (two floats each).
size_t decay_offset(int64_t BH, int64_t Dh, int64_t N, int S) { return (size_t)BH * (S - 1) * 2 * Dh * N; }

template <int DH, int NS, bool GLA>
int launch(const WalkArgs& a, int64_t BH, hipStream_t s) {
  constexpr int T = Shape<DH, NS>::T;
  if (a.S > 1) {
    hipLaunchKernelGGL((walk_bwd_kernel<DH, NS, GLA, true>), dim3((unsigned)BH, a.S - 1), dim3(T), 0, s, a);
    if (int rc = rr::check_launch("walking backward (segment maps)")) return rc;
  }
  hipLaunchKernelGGL((walk_bwd_kernel<DH, NS, GLA, false>), dim3((unsigned)BH, a.S), dim3(T), 0, s, a);
  return rr::check_launch("walking backward");
}

}  // namespace

namespace rr {

// Where it measured no slower than the per-chunk kernels with their adjoint scan
// or pass (forward + backward, us): from 1100 chunks in all.  768 chunks 0.77x
// (GLA 96 heads Dh 64, 36.5 -> 47.7) to 1.29x; 1152 chunks 1.02x to 1.39x; 1280
// 1.0x (GLA 320 heads Dh 64, 4 chunks) to 1.6x; 6144 1.36x to 1.6x (GLA B8 L2048 H12
// Dh128 810 -> 450).  Fewer than 12 heads serialise too long segments (8
// heads, 128 chunks: 0.9x).
bool walk_bwd_preferred(int64_t BH, int64_t nC, int64_t Dh, int64_t N) {
  if (!grid_ok(BH, 512)) return false;   // the most threads a workgroup has
  return (Dh == 64 || Dh == 128) && (N == 64 || N == 128) && BH >= 12 && BH * nC >= 1100;
}

int walk_bwd_chunks(int64_t BH, int64_t nC, int64_t Dh, int64_t N) {
  int S, cps;
  segments(BH, nC, Dh, N, S, cps);
  return cps;
}

int64_t walk_bwd_extent_floats(int64_t BH, int64_t nC, int64_t Dh, int64_t N, int& S) {
  int cps;
  segments(BH, nC, Dh, N, S, cps);
  const int64_t NW = Dh == 128 && N == 128 ? 8 : 4, T = 64 * NW;   // Shape's
  const int64_t frags = N / 16 / NW * (Dh / 16) + Dh / 16 / NW * (N / 16);
  const int64_t decays = S > 1 ? (int64_t)decay_offset(BH, Dh, N, S) : 0;
  int64_t ext = 0;
  for (int64_t bh = 0; bh < BH; ++bh)
    for (int seg = 1; seg < S; ++seg) {
      const int64_t slot = chunked::map_slot(bh, S, seg - 1);
      if ((slot * frags * T + (frags - 1) * T + T) * 4 > decays) return INT64_MAX;   // into the decays
      ext = std::max(ext, decays + (slot + 1) * 2);
    }
  return ext;
}

size_t walk_bwd_ws_floats(int64_t BH, int64_t nC, int64_t Dh, int64_t N) {
  int S, cps;
  segments(BH, nC, Dh, N, S, cps);
  if (S <= 1) return 0;
  return decay_offset(BH, Dh, N, S) + (size_t)BH * (S - 1) * 2;
}

int walk_bwd(const ChunkArgs& p, int64_t B, hipStream_t s, bool gla) {
  const int64_t BH = B * p.H;
  WalkArgs a{};
  a.p = p;
  segments(BH, p.nC, p.DH, p.NS, a.S, a.cps);
  a.mapL = reinterpret_cast<float4*>(p.agg);
  a.mapP = p.agg == nullptr ? nullptr : reinterpret_cast<float2*>(p.agg + decay_offset(BH, p.DH, p.NS, a.S));
  switch (p.DH * 1000 + p.NS) {
    case 64064: return gla ? launch<64, 64, true>(a, BH, s) : launch<64, 64, false>(a, BH, s);
    case 64128: return launch<64, 128, false>(a, BH, s);
    case 128064: return launch<128, 64, false>(a, BH, s);
    case 128128: return gla ? launch<128, 128, true>(a, BH, s) : launch<128, 128, false>(a, BH, s);
    default: return fail(RR_EUNSUPPORTED, "walking backward: sizes not covered");
  }
}

}  // namespace rr
