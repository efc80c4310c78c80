// final_fwd.hip — SSD (one decay rate per head) and GLA forward, bf16 inputs, a
// head's chunks walked in order by one workgroup: for calls that need y and
// the final state only (no gradient, so no checkpoints; any length L >= 1),
// and, writing the state after every chunk, for the training forward.
//
// Per (batch, head) the recurrence and its 32-step chunk form are those of
// rr_chunked.h,
//     Y     = (M o C B^T o w_s) U + diag(gam) C h_in^T
//     h_end = gam_31 h_in + (diag(m31 o w) U)^T B,
// with the last chunk's missing steps taken as identity steps (zero rows, no
// decay).  A workgroup owns a head and walks its chunks; each wave owns 16 DB
// rows d of the state for all n and never exchanges anything with the others:
// the state lives in accumulators as h^T[n][d] (rows n), which are, element
// for element, the B operand of C h^T, and (C B^T)^T's accumulators (rows s)
// are the A operand of W U, so neither passes through LDS.  The k index of
// those products runs in the accumulators' order pi(g, e) = 4 g + e (e < 4),
// 16 + 4 g + e - 4 (e >= 4); B and C are staged in LDS with their n index in
// that order, and read back as row fragments (16 bytes) or transposed.
//
// fp32 factors (the state, W, the weighted U) are split into three bf16 terms,
// hi + mid + lo = all 24 bits, each multiplied with an exact bf16 operand, and
// the small terms are summed first: the error against float64 stays that of
// fp32 arithmetic (1e-7; the two-term split of the training kernels has
// 2.5e-6).
//
// Heads alone may not fill the GPU: the chunks are then cut into S segments.
// A first launch forms every segment's map (its state from a zero start and
// its decay), and the walk of segment j starts from h0 carried through the
// maps of segments 0 .. j - 1.
//
// W is formed once per chunk: its three nonzero 16x16 blocks are dealt to the
// waves, a chunk ahead, and the last wave forms the step scalars two ahead, so a
// chunk has two barriers (LDS only: loads and stores stay in flight across them).
//
// What bounds it: without checkpoints the instructions of a chunk (per wave
// about 500 VALU, a third of them the state's three-term split, beside 50
// MFMAs at N = 128) on two waves per SIMD; B4 L1000 H80 Dh64 N128 takes 95 us,
// 3.2 TB/s of the 0.31 GB it cannot do without (6.1 ms on the VALU engine,
// which forms and stores a state every 8 steps there; 132 us with W and the
// scalars formed by every wave for itself).  Three waves per SIMD (168 VGPRs)
// spill 18 and take 178 us.  With checkpoints the traffic: B8 L4096 H80 Dh64
// N128 1114 us, 4.6 TB/s of the 5.1 GB counted; B8 L2048 H12 GLA Dh128 448 -> 195 us.
#include "rr_chunked.h"
#include "rr_frag.h"

namespace {

using rr::f32x4_t;
using rr::lds_barrier;
using rr::u16x4_t;
using rr::u16x8_t;

constexpr int Q = 32;

// 16-row blocks of the state a wave owns.  One: two leave half the waves.  The
// kernel stays written for any number, since the compiler's schedule of the same
// code without the loops over blocks is slower (1 to 2 % in prompts of two chunks).
constexpr int DB = 1;

struct FinalArgs {
  const uint16_t* u;      // [B,L,H,DH] (GLA: v)
  const uint16_t* step;   // [B,L,H] delta (GLA: gates)
  const uint16_t* Bm;     // [B,L,H,N] (GLA: k)
  const uint16_t* Cm;     // [B,L,H,N] (GLA: q)
  const float* A;         // [H] (SSD)
  const float* h0;        // [B,H,DH,N] as d, n (GLA [B,H,N,DH] as n, d), or null
  float* y;               // [B,L,H,DH]
  float* fin;             // final state, layout of h0 (kCkpt: the checkpoints [B*H][nC][DH][N])
  float4* segE;           // [B*H][S-1] segment states in fragment order
  float* segP;            // [B*H][S-1] segment decays
  int L, H, nC, S, cps;   // chunks, segments, chunks per segment
};

// fp32 -> bf16 hi + mid + lo of eight values
__device__ __forceinline__ void split3(const float (&x)[8], u16x8_t& hi, u16x8_t& mid, u16x8_t& lo) {
  uint32_t h[4], m[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    h[i] = rr::bf_pack2(x[2 * i], x[2 * i + 1]);
    const float a = x[2 * i] - __uint_as_float(h[i] << 16), b = x[2 * i + 1] - __uint_as_float(h[i] & 0xffff0000u);
    m[i] = rr::bf_pack2(a, b);
    l[i] = rr::bf_pack2(a - __uint_as_float(m[i] << 16), b - __uint_as_float(m[i] & 0xffff0000u));
  }
  hi = __builtin_bit_cast(u16x8_t, make_uint4(h[0], h[1], h[2], h[3]));
  mid = __builtin_bit_cast(u16x8_t, make_uint4(m[0], m[1], m[2], m[3]));
  lo = __builtin_bit_cast(u16x8_t, make_uint4(l[0], l[1], l[2], l[3]));
}

// LDS images of one chunk.  16-byte units of a row are permuted by row (xor)
// so that both the row fragments (16 rows, one unit) and the transposing reads
// (4 rows x 4 units) of a 16-lane group hit distinct banks.
// (B and C: the images of rr_frag.h, written out here; through its helpers the
// kernel measured 0 to 1 % slower.)
template <int NSP>
__device__ __forceinline__ int swz_n(int row) {
  return NSP == 128 ? ((row & 3) << 2) | ((row >> 2) & 3)
         : NSP == 64 ? (((row >> 1) & 1) << 2) | ((row >> 2) & 3)
                     : (row >> 2) & 3;
}
template <int DH>
__device__ __forceinline__ int swz_d(int row) {
  return DH == 128 ? 2 * (row & 7) : DH == 64 ? 2 * ((row >> 1) & 3) : 2 * ((row >> 2) & 1);
}

template <int DH, int NS>
struct alignas(16) FinalSm {
  static constexpr int NSP = NS < 32 ? 32 : NS, NW = DH / (16 * DB);
  uint16_t B[2][Q * NSP], C[2][Q * NSP], U[2][Q * DH];
  uint2 W[2][3][3][64];    // a chunk's W: [16x16 block][hi, mid, lo][lane], see w_block
  float sc[3][4][Q];       // a chunk's step scalars: gam, m31 w, cd (GLA: gates), w
};

// The four decays M[t][s] a lane holds of 16x16 block blk of (C B^T)^T:
// blk 0: s = 4 g + e, t = l15; blk 1: s = 4 g + e, t = 16 + l15; blk 2: both
// plus 16.  Zero for s > t.
template <bool GLA>
__device__ __forceinline__ void decays(const float* st, float a, int blk, int l15, int g, float (&m)[4]) {
  const int s0 = blk == 2 ? 16 : 0, t0 = blk > 0 ? 16 : 0;
  const float4 sq = *reinterpret_cast<const float4*>(&st[s0 + 4 * g]);
  const float sv[4] = {sq.x, sq.y, sq.z, sq.w};
  if constexpr (!GLA) {
    const float ct = st[t0 + l15];
#pragma unroll
    for (int e = 0; e < 4; ++e) m[e] = rr::chunked::masked_exp(blk == 1 || 4 * g + e <= l15, a * (ct - sv[e]));
  } else {
    // products of the gates of steps s + 1 .. t, by quads of steps: the rest
    // of s's quad, whole quads between, t's quad up to t (any sign, zeros exact)
    const int qt = l15 >> 2, pt = l15 & 3;   // t's quad within its 16 steps, position in it
    const float4 tq = *reinterpret_cast<const float4*>(&st[t0 + 4 * qt]);
    const float p1 = tq.x * tq.y, p2 = p1 * tq.z, p3 = p2 * tq.w;
    float far = pt == 0 ? tq.x : pt == 1 ? p1 : pt == 2 ? p2 : p3;
    auto quad = [&](int j) {
      const float4 q = *reinterpret_cast<const float4*>(&st[4 * j]);
      return (q.x * q.y) * (q.z * q.w);
    };
    const float r2 = sv[3], r1 = sv[2] * r2, r0 = sv[1] * r1;   // rest of s's quad after s
    const float rest[4] = {r0, r1, r2, 1.f};
    if (blk == 1) {   // quads g + 1 .. 3 and 4 .. 3 + qt
      const float q1 = quad(1), q2 = quad(2), q3 = quad(3), q4 = quad(4), q5 = quad(5), q6 = quad(6);
      far *= (g < 1 ? q1 : 1.f) * (g < 2 ? q2 : 1.f) * (g < 3 ? q3 : 1.f);
      far *= (qt > 0 ? q4 : 1.f) * (qt > 1 ? q5 : 1.f) * (qt > 2 ? q6 : 1.f);
#pragma unroll
      for (int e = 0; e < 4; ++e) m[e] = rest[e] * far;
    } else {
      // whole quads strictly between g and qt (both in 0 .. 3: quads 1 and 2)
      const float q1 = quad(s0 / 4 + 1), q2 = quad(s0 / 4 + 2);
      far *= (g < 1 && qt > 1 ? q1 : 1.f) * (g < 2 && qt > 2 ? q2 : 1.f);
      // t in s's own quad: product of positions e + 1 .. pt
      const float yz = sv[1] * sv[2];
      const float in0 = pt == 0 ? 1.f : pt == 1 ? sv[1] : pt == 2 ? yz : yz * sv[3];
      const float in1 = pt == 1 ? 1.f : pt == 2 ? sv[2] : sv[2] * sv[3];
      const float in2 = pt == 2 ? 1.f : sv[3];
      const float inq[4] = {in0, in1, in2, 1.f};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = qt == g ? inq[e] : rest[e] * far;
        m[e] = 4 * g + e <= l15 ? v : 0.f;
      }
    }
  }
}

// OUT: kMap only the segment's state from a zero start and its decay (segE,
// segP); kFinal y and the final state; kCkpt y and the state after every chunk
// (L a multiple of 32).
enum Out { kMap = 0, kFinal = 1, kCkpt = 2 };
__device__ __forceinline__ bool finite(float x) { return fabsf(x) < __builtin_inff(); }

// The steps of chunks c0 .. c1 - 1 one after another, for a wave whose results of
// them are not all finite: the splits make NaN of an infinite factor (inf - inf),
// and so does a decay that overflows over a segment or a chunk before it meets a
// zero.  Starts from the head's first step (the maps of the segments before may
// have overflown) and replaces only the results that are not finite, so all
// others keep their bits.  The state left in hs is finite where it can be.
template <int DH, int NS, bool GLA, int OUT, int NBN>
__device__ __forceinline__ void by_steps(const FinalArgs& p, int bh, int c0, int c1, int d, int g, f32x4_t (&hs)[NBN]) {
  const int h = bh % p.H;
  const int64_t rows = (int64_t)(bh / p.H) * p.L;
  const float a = GLA ? 0.f : p.A[h];
  f32x4_t x[NS / 16];   // h^T[16 nb + 4 g + r][d]
#pragma unroll
  for (int nb = 0; nb < NS / 16; ++nb)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      x[nb][r] = p.h0 == nullptr ? 0.f
                                 : p.h0[(int64_t)bh * DH * NS +
                                        rr::chunked::state_off<GLA, DH, NS>(d, 16 * nb + 4 * g + r)];
  const int end = min(c1 * Q, p.L);
  for (int t = 0; t < end; ++t) {
    const int64_t i = (rows + t) * p.H + h;
    const float in = rr::bf_val(p.step[i]), decay = GLA ? in : __expf(a * in);
    const float wu = (GLA ? 1.f : in) * rr::bf_val(p.u[i * DH + d]);
    float y = 0.f;
#pragma unroll
    for (int nb = 0; nb < NS / 16; ++nb) {
      const uint2 b4 = *reinterpret_cast<const uint2*>(p.Bm + i * NS + 16 * nb + 4 * g);
      const uint2 c4 = *reinterpret_cast<const uint2*>(p.Cm + i * NS + 16 * nb + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x[nb][r] = decay * x[nb][r] + wu * rr::bf4(b4, r);
        y += rr::bf4(c4, r) * x[nb][r];
      }
    }
    y = rr::rows4_sum(y);
    if (t < c0 * Q) continue;
    if (g == 0 && !finite(p.y[i * DH + d])) p.y[i * DH + d] = y;
    if constexpr (OUT == kCkpt) {
      if (t % Q != Q - 1) continue;
      float* ck = p.fin + ((int64_t)bh * p.nC + t / Q) * DH * NS + d * NS + 4 * g;
#pragma unroll
      for (int nb = 0; nb < NS / 16; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (!finite(ck[16 * nb + r])) ck[16 * nb + r] = x[nb][r];
    }
  }
#pragma unroll
  for (int nb = 0; nb < NS / 16; ++nb)
#pragma unroll
    for (int r = 0; r < 4; ++r) hs[nb][r] = finite(hs[nb][r]) ? hs[nb][r] : x[nb][r];
}

template <int DH, int NS, bool GLA, int OUT>
__global__ __launch_bounds__(4 * DH / DB, 2) void final_fwd_kernel(FinalArgs p) {
  using S = FinalSm<DH, NS>;
  constexpr int NSP = S::NSP, NW = S::NW, T = 64 * NW, NK = NSP / 32, NBN = NSP / 16;
  constexpr bool AGG = OUT == kMap;
  constexpr int BV = (Q * NS / 8 + T - 1) / T, UV = (Q * DH / 8 + T - 1) / T;
  __shared__ S sm;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, g = lane >> 4;
  const int bh = blockIdx.x, seg = blockIdx.y, h = bh % p.H, b = bh / p.H;
  const int c0 = seg * p.cps, c1 = min(c0 + p.cps, p.nC);
  const float a = GLA ? 0.f : p.A[h];
  const int64_t rows = (int64_t)b * p.L;
  const uint32_t rsN = (uint32_t)p.H * NS, rsD = (uint32_t)p.H * DH;

  if constexpr (NS < 32) {   // n 16 .. 31 of both images stay zero
    for (int i = tid; i < 2 * Q * NSP / 2; i += T) {
      reinterpret_cast<uint32_t*>(&sm.B[0][0])[i] = 0;
      reinterpret_cast<uint32_t*>(&sm.C[0][0])[i] = 0;
    }
    lds_barrier();
  }

  u16x8_t bv[BV], cv[BV], uv[UV];
  float xv;   // this lane's step input of the chunk whose scalars come next
  // chunk c's pieces into registers: unconditional loads, offsets past the
  // sequence clamped to its last piece (those rows become zero, or the neutral
  // step, when staged)
  auto load = [&](int c) {
    const int t0 = min(c, p.nC - 1) * Q, last = p.L - 1 - t0;
    const uint32_t lastN = (uint32_t)min(last, Q) * rsN + NS - 8, lastD = (uint32_t)min(last, Q) * rsD + DH - 8;
    const uint16_t* Bp = p.Bm + ((rows + t0) * p.H + h) * NS;
    const uint16_t* Cp = p.Cm + ((rows + t0) * p.H + h) * NS;
    const uint16_t* Up = p.u + ((rows + t0) * p.H + h) * DH;
#pragma unroll
    for (int v = 0; v < BV; ++v) {
      const int i = min(tid + T * v, Q * NS / 8 - 1);
      const uint32_t o = min((uint32_t)(i / (NS / 8)) * rsN + 8 * (i % (NS / 8)), lastN);
      bv[v] = rr::ld32<u16x8_t>(Bp, o);
      if constexpr (!AGG) cv[v] = rr::ld32<u16x8_t>(Cp, o);
    }
#pragma unroll
    for (int v = 0; v < UV; ++v) {
      const int i = min(tid + T * v, Q * DH / 8 - 1);
      uv[v] = rr::ld32<u16x8_t>(Up, min((uint32_t)(i / (DH / 8)) * rsD + 8 * (i % (DH / 8)), lastD));
    }
  };
  auto load_step = [&](int c) {
    const int t0 = min(c, p.nC - 1) * Q;
    xv = rr::bf_val(p.step[(rows + t0 + min(lane & (Q - 1), p.L - 1 - t0)) * p.H + h]);
  };
  // step scalars of chunk c (one wave)
  auto scalars = [&](int c) {
    const bool live = lane < Q && lane < p.L - c * Q;
    const float x = live ? xv : (GLA ? 1.f : 0.f);
    const rr::chunked::StepScalars st = rr::chunked::step_scalars<GLA>(x, a, lane);
    float(*sc)[Q] = sm.sc[c % 3];
    if (lane < Q) {
      sc[0][lane] = st.gam;
      sc[1][lane] = st.m31 * st.w;
      sc[2][lane] = GLA ? x : st.cd;
      sc[3][lane] = st.w;
    }
  };
  // W[t][s] = M[t][s] (C B^T)[t][s] w_s of chunk c from its staged B and C, by
  // 16x16 blocks (three: the upper right one is zero) dealt to the waves; the
  // accumulators of (C B^T)^T are W's A operand, kept as lane fragments
  auto w_blocks = [&](int c, int buf) {
    const float(*sc)[Q] = sm.sc[c % 3];
    for (int blk = w; blk < 3; blk += NW) {
      const int ro = (blk == 2 ? 16 * NSP : 0), co = (blk > 0 ? 16 * NSP : 0);
      f32x4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) {
        const int off = l15 * NSP + 8 * ((4 * kk + g) ^ swz_n<NSP>(l15));
        d = rr::mfma16(rr::frag(&sm.B[buf][off + ro]), rr::frag(&sm.C[buf][off + co]), d);
      }
      float m[4];
      decays<GLA>(sc[2], a, blk, l15, g, m);
      const float4 x = *reinterpret_cast<const float4*>(&sc[3][(blk == 2 ? 16 : 0) + 4 * g]);
      const float wl[4] = {x.x, x.y, x.z, x.w};
      float v[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {   // a select, so that a non-finite B row stays out of earlier steps
        v[e] = blk == 1 || 4 * g + e <= l15 ? m[e] * (d[e] * wl[e]) : 0.f;
        v[4 + e] = 0.f;
      }
      u16x8_t f[3];
      split3(v, f[0], f[1], f[2]);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const uint4 u4 = __builtin_bit_cast(uint4, f[k]);
        sm.W[buf][blk][k][lane] = make_uint2(u4.x, u4.y);
      }
    }
  };
  auto stage_rows = [&](int V, int buf, auto full) {   // full: all 32 steps present
#pragma unroll
    for (int v = 0; v < BV; ++v) {
      const int i = tid + T * v, t = i / (NS / 8), m = i % (NS / 8);
      if (Q * NS / 8 % T != 0 && i >= Q * NS / 8) break;
      const bool in = decltype(full)::value || t < V;
      const int f = swz_n<NSP>(t), un = 4 * (m >> 2) + 2 * (m & 1), hf = 4 * ((m >> 1) & 1);
      const uint4 x = __builtin_bit_cast(uint4, bv[v]);
      uint16_t* d = &sm.B[buf][t * NSP + hf];
      *reinterpret_cast<uint2*>(d + 8 * (un ^ f)) = in ? make_uint2(x.x, x.y) : make_uint2(0, 0);
      *reinterpret_cast<uint2*>(d + 8 * ((un + 1) ^ f)) = in ? make_uint2(x.z, x.w) : make_uint2(0, 0);
      if constexpr (!AGG) {
        const uint4 z = __builtin_bit_cast(uint4, cv[v]);
        d = &sm.C[buf][t * NSP + hf];
        *reinterpret_cast<uint2*>(d + 8 * (un ^ f)) = in ? make_uint2(z.x, z.y) : make_uint2(0, 0);
        *reinterpret_cast<uint2*>(d + 8 * ((un + 1) ^ f)) = in ? make_uint2(z.z, z.w) : make_uint2(0, 0);
      }
    }
#pragma unroll
    for (int v = 0; v < UV; ++v) {
      const int i = tid + T * v, t = i / (DH / 8), m = i % (DH / 8);
      if (Q * DH / 8 % T != 0 && i >= Q * DH / 8) break;
      *reinterpret_cast<u16x8_t*>(&sm.U[buf][t * DH + 8 * (m ^ swz_d<DH>(t))]) =
          decltype(full)::value || t < V ? uv[v] : u16x8_t{};
    }
  };
  auto stage = [&](int c, int buf) {
    const int V = p.L - c * Q;   // steps present
    if (V >= Q) stage_rows(V, buf, std::true_type{});
    else stage_rows(V, buf, std::false_type{});
  };

  f32x4_t hs[DB][NBN];   // h^T[16 nb + 4 g + r][d = 16 (w DB + i) + l15]
  float decay = 1.f;     // AGG: the segment's decay
  float odd = 0.f;       // NaN once a result was not finite
#pragma unroll
  for (int i = 0; i < DB; ++i)
#pragma unroll
    for (int nb = 0; nb < NBN; ++nb) hs[i][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  load(c0);
  if constexpr (!AGG) {
    if (p.h0 != nullptr) {
      const float* hp = p.h0 + (int64_t)bh * DH * NS;
#pragma unroll
      for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int nb = 0; nb < NS / 16; ++nb)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            hs[i][nb][r] = hp[rr::chunked::state_off<GLA, DH, NS>(16 * (w * DB + i) + l15, 16 * nb + 4 * g + r)];
    }
    const float4* E = p.segE + rr::chunked::map_slot(bh, p.S, 0) * (DB * NBN * T) + tid;
#pragma unroll 2
    for (int j = 0; j < seg; ++j) {
      const float P = p.segP[rr::chunked::map_slot(bh, p.S, j)];
#pragma unroll
      for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int nb = 0; nb < NBN; ++nb) {
          const float4 e = E[(j * DB * NBN + i * NBN + nb) * T];
          hs[i][nb] = f32x4_t{P * hs[i][nb][0] + e.x, P * hs[i][nb][1] + e.y, P * hs[i][nb][2] + e.z,
                              P * hs[i][nb][3] + e.w};
        }
    }
  }
  load_step(c0);
  stage(c0, 0);
  load(c0 + 1);
  if (w == NW - 1) {
    scalars(c0);
    load_step(c0 + 1);
    scalars(min(c0 + 1, p.nC - 1));
  }
  load_step(c0 + 2);
  // the rows of y of chunk c, from this head's first column: a store past the
  // last row of V is dropped
  auto y_rows = [&](int c, int V) {
    float* yp = p.y + ((rows + (int64_t)c * Q) * p.H + h) * DH;
    return __builtin_amdgcn_make_buffer_rsrc(yp, 0, (int)((uint32_t)V * rsD * 4u), 0x00027000);
  };
  if constexpr (!AGG) {
    // as many dropped stores as a chunk makes after its loads: the waits for
    // those loads at the loop's head then count past a chunk's stores (without
    // them they cover the stores: 99.5 -> 96.6 us at the first size above)
    const auto none = y_rows(c0, 0);
#pragma unroll
    for (int j = 0; j < 8 * DB + (OUT == kCkpt ? DB * (NS / 16) : 0); ++j)
      __builtin_amdgcn_raw_buffer_store_b32(0u, none, 4 * lane + 256 * j, 0, 0);
  }
  lds_barrier();
  if constexpr (!AGG) w_blocks(c0, 0);

  for (int c = c0; c < c1; ++c) {
    const int buf = (c - c0) & 1;
    if (c + 1 < c1) stage(c + 1, buf ^ 1);
    load(c + 2);   // (unconditional: under the branch, the scalar wave's wait for its step input would cover these too)
    lds_barrier();   // this chunk's W, the next one's rows
    if constexpr (!AGG) {
      if (c + 1 < c1) w_blocks(c + 1, buf ^ 1);
    }
    if (w == NW - 1 && c + 2 < c1) scalars(c + 2);
    load_step(c + 3);
    const uint16_t *Bs = sm.B[buf], *Cs = sm.C[buf], *Us = sm.U[buf];
    const float(*sc)[Q] = sm.sc[c % 3];
    const float tot = sc[0][Q - 1];
    // U as B operand: U[pi(g, e)][d]
    u16x8_t uf[DB];
    {
      const int r0 = 4 * g + (l15 >> 2), q = l15 & 3;
#pragma unroll
      for (int i = 0; i < DB; ++i) {
        const uint16_t* up = Us + r0 * DH + 8 * ((2 * (w * DB + i) + (q >> 1)) ^ swz_d<DH>(r0)) + 4 * (q & 1);
        const u16x4_t lo = rr::tr_read4(up), hi = rr::tr_read4(up + 16 * DH);
        uf[i] = u16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    }
    if constexpr (!AGG) {
      u16x8_t cf[2][NK];   // C[16 tb + l15][32 kk + pi]
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) {
        const int off = l15 * NSP + 8 * ((4 * kk + g) ^ swz_n<NSP>(l15));
        cf[0][kk] = rr::frag(Cs + off);
        cf[1][kk] = rr::frag(Cs + off + 16 * NSP);
      }
      u16x8_t wf[2][3];   // W[16 tb + l15][pi]
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const uint2 x0 = sm.W[buf][0][k][lane], x1 = sm.W[buf][1][k][lane], x2 = sm.W[buf][2][k][lane];
        wf[0][k] = __builtin_bit_cast(u16x8_t, make_uint4(x0.x, x0.y, 0, 0));
        wf[1][k] = __builtin_bit_cast(u16x8_t, make_uint4(x1.x, x1.y, x2.x, x2.y));
      }
#pragma unroll
      for (int i = 0; i < DB; ++i) {
        f32x4_t ab[2], as[2];   // C h^T: hi terms, mid + lo terms
        ab[0] = ab[1] = as[0] = as[1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) {
          const float x[8] = {hs[i][2 * kk][0],     hs[i][2 * kk][1],     hs[i][2 * kk][2],     hs[i][2 * kk][3],
                              hs[i][2 * kk + 1][0], hs[i][2 * kk + 1][1], hs[i][2 * kk + 1][2], hs[i][2 * kk + 1][3]};
          u16x8_t hh, hm, hl;
          split3(x, hh, hm, hl);
#pragma unroll
          for (int tb = 0; tb < 2; ++tb) {
            as[tb] = rr::mfma16(cf[tb][kk], hl, as[tb]);
            ab[tb] = rr::mfma16(cf[tb][kk], hh, ab[tb]);
            as[tb] = rr::mfma16(cf[tb][kk], hm, as[tb]);
          }
        }
        // a non-finite u must not reach the steps before it through W's zeros:
        // such elements leave the product and are added step by step below
        u16x8_t ui = uf[i];
        bool inf_u = false;
        {
          uint4 x = __builtin_bit_cast(uint4, ui);
          auto over = [](uint32_t v) { return ((v & 0x7f807f80u) + 0x00800080u) & 0x80008000u; };
          inf_u = (over(x.x) | over(x.y) | over(x.z) | over(x.w)) != 0;
        }
        const bool any_odd = __any(inf_u);
        if (__builtin_expect(any_odd, 0)) {
#pragma unroll
          for (int e = 0; e < 8; ++e) ui[e] = (ui[e] & 0x7f80) == 0x7f80 ? 0 : ui[e];
        }
        f32x4_t o[2];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
          f32x4_t z = {0.f, 0.f, 0.f, 0.f};
          z = rr::mfma16(wf[tb][2], ui, z);
          z = rr::mfma16(wf[tb][1], ui, z);
          const float4 gm = *reinterpret_cast<const float4*>(&sc[0][16 * tb + 4 * g]);
          z = f32x4_t{gm.x * (ab[tb][0] + as[tb][0]) + z[0], gm.y * (ab[tb][1] + as[tb][1]) + z[1],
                      gm.z * (ab[tb][2] + as[tb][2]) + z[2], gm.w * (ab[tb][3] + as[tb][3]) + z[3]};
          o[tb] = rr::mfma16(wf[tb][0], ui, z);
        }
        if (__builtin_expect(any_odd, 0)) {
          for (int s = 0; s < Q; ++s) {
            const int src = 16 * ((s >> 2) & 3), e = (s & 3) + 4 * (s >> 4);
            float us = 0.f, ws0 = 0.f, ws1 = 0.f;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
              us = k == e ? rr::bf_val(uf[i][k]) : us;
              ws0 = k == e ? rr::bf_val(wf[0][0][k]) + rr::bf_val(wf[0][1][k]) : ws0;
              ws1 = k == e ? rr::bf_val(wf[1][0][k]) + rr::bf_val(wf[1][1][k]) : ws1;
            }
            us = __shfl(us, src + l15);
            const bool add = !(fabsf(us) < __builtin_inff());   // the elements left out above
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float v0 = __shfl(ws0, src + 4 * g + r), v1 = __shfl(ws1, src + 4 * g + r);
              if (add && s <= 4 * g + r) o[0][r] += v0 * us;
              if (add && s <= 16 + 4 * g + r) o[1][r] += v1 * us;
            }
          }
        }
        const auto yr = y_rows(c, min(p.L - c * Q, Q));
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float v = o[j >> 2][j & 3];   // (a copy: a bit cast of a vector's element takes the first one)
          odd = fmaf(v, 0.f, odd);
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), yr,
                                                (int)(4u * ((uint32_t)(16 * (j >> 2) + 4 * g + (j & 3)) * rsD + l15)),
                                                64 * (w * DB + i), 0);
        }
      }
    }
    // h^T <- gam_31 h^T + B^T (m31 w o U): B^T transposed reads are the exact A operand
    u16x8_t us[DB][3];
    {
      const float4 x0 = *reinterpret_cast<const float4*>(&sc[1][4 * g]);
      const float4 x1 = *reinterpret_cast<const float4*>(&sc[1][16 + 4 * g]);
      const float mw[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
      for (int i = 0; i < DB; ++i) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = mw[e] * rr::bf_val(uf[i][e]);
        split3(x, us[i][0], us[i][1], us[i][2]);
      }
    }
    {
      const int r0 = 4 * g + (l15 >> 2), f = swz_n<NSP>(r0);
#pragma unroll
      for (int nb = 0; nb < NBN; ++nb) {
        const uint16_t* bp = Bs + r0 * NSP + 8 * ((4 * (nb >> 1) + (l15 & 3)) ^ f) + 4 * (nb & 1);
        const u16x4_t lo = rr::tr_read4(bp), hi = rr::tr_read4(bp + 16 * NSP);
        const u16x8_t bt = u16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int i = 0; i < DB; ++i) {
          f32x4_t z = {0.f, 0.f, 0.f, 0.f};
          z = rr::mfma16(bt, us[i][2], z);
          z = rr::mfma16(bt, us[i][1], z);
          z = rr::mfma16(bt, us[i][0], z);
          hs[i][nb] = f32x4_t{tot * hs[i][nb][0] + z[0], tot * hs[i][nb][1] + z[1], tot * hs[i][nb][2] + z[2],
                              tot * hs[i][nb][3] + z[3]};
        }
      }
    }
    if constexpr (AGG) decay *= tot;
    if constexpr (OUT == kCkpt) {
      float* ck = p.fin + ((int64_t)bh * p.nC + c) * DH * NS;
#pragma unroll
      for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int nb = 0; nb < NS / 16; ++nb)
          *reinterpret_cast<float4*>(ck + (16 * (w * DB + i) + l15) * NS + 16 * nb + 4 * g) =
              make_float4(hs[i][nb][0], hs[i][nb][1], hs[i][nb][2], hs[i][nb][3]);
    }
    lds_barrier();
  }

  if constexpr (!AGG) {
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
      for (int nb = 0; nb < NBN; ++nb)   // (a state once not finite stays so)
#pragma unroll
        for (int r = 0; r < 4; ++r) odd = fmaf(hs[i][nb][r], 0.f, odd);
    if (__builtin_expect(__any(odd != 0.f), 0)) {
      __threadfence_block();   // the wave reads its own stores back
#pragma unroll
      for (int i = 0; i < DB; ++i)
        by_steps<DH, NS, GLA, OUT>(p, bh, c0, c1, 16 * (w * DB + i) + l15, g, hs[i]);
    }
  }
  if constexpr (AGG) {
    float4* E = p.segE + rr::chunked::map_slot(bh, p.S, seg) * (DB * NBN * T) + tid;
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
      for (int nb = 0; nb < NBN; ++nb)
        E[(i * NBN + nb) * T] = make_float4(hs[i][nb][0], hs[i][nb][1], hs[i][nb][2], hs[i][nb][3]);
    if (tid == 0) p.segP[rr::chunked::map_slot(bh, p.S, seg)] = decay;
  } else if (OUT == kFinal && seg == p.S - 1) {
    float* fp = p.fin + (int64_t)bh * DH * NS;
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
      for (int nb = 0; nb < NS / 16; ++nb) {
        const int d = 16 * (w * DB + i) + l15, n = 16 * nb + 4 * g;
        if constexpr (GLA) {
#pragma unroll
          for (int r = 0; r < 4; ++r) fp[(n + r) * DH + d] = hs[i][nb][r];
        } else {
          *reinterpret_cast<float4*>(fp + d * NS + n) =
              make_float4(hs[i][nb][0], hs[i][nb][1], hs[i][nb][2], hs[i][nb][3]);
        }
      }
  }
}

// ------------------------------------------------------------------ host
bool covered(int64_t Dh, int64_t N, bool gla) {
  if (gla) return Dh == N && (Dh == 32 || Dh == 64 || Dh == 128);
  return (Dh == 32 || Dh == 64 || Dh == 128) && (N == 16 || N == 32 || N == 64 || N == 128);
}

// Segments: enough workgroups for two waves per SIMD, at least two chunks each,
// and at most sqrt(8 nC): each segment before a walk costs it the reading of a
// map, each chunk of a segment its map and its output (SSD 8 heads, 32 chunks,
// Dh 64 N 128: 23.0 us with 8 segments, 22.8 with 10, 18.7 with 16).
void segments(int64_t BH, int64_t nC, int64_t Dh, int& S, int& cps) {
  const int64_t waves = BH * (Dh / 16), want = std::max<int64_t>(1, 2048 / std::max<int64_t>(waves, 1));
  int64_t s = std::max<int64_t>(1, std::min(want, nC / 2));
  while (s * s > 8 * nC) --s;
  cps = (int)((nC + s - 1) / s);
  S = (int)((nC + cps - 1) / cps);
}

// Workspace: the segments' states, then their decays.
size_t map_bytes(int64_t Dh, int64_t N) { return (size_t)Dh * (size_t)std::max<int64_t>(N, 32) * 4; }
size_t decay_offset(int64_t BH, int64_t Dh, int64_t N, int S) { return (size_t)BH * (S - 1) * map_bytes(Dh, N); }
size_t ws_bytes(int64_t BH, int64_t Dh, int64_t N, int S) {
  return S <= 1 ? 0 : decay_offset(BH, Dh, N, S) + (size_t)BH * (S - 1) * 4 + 256;
}

template <int DH, int NS, bool GLA, int OUT>
int launch(const FinalArgs& p, int64_t BH, hipStream_t s) {
  constexpr int T = 4 * DH;
  if (p.S > 1) {
    hipLaunchKernelGGL((final_fwd_kernel<DH, NS, GLA, kMap>), dim3((unsigned)BH, p.S - 1), dim3(T), 0, s, p);
    if (int rc = rr::check_launch("final-state forward (segment maps)")) return rc;
  }
  hipLaunchKernelGGL((final_fwd_kernel<DH, NS, GLA, OUT>), dim3((unsigned)BH, p.S), dim3(T), 0, s, p);
  return rr::check_launch("final-state forward");
}

template <bool GLA, int OUT>
int run(FinalArgs& p, int64_t B, int64_t H, int64_t Dh, int64_t N, void* ws, size_t wsb, hipStream_t s) {
  const int64_t BH = B * H;
  segments(BH, p.nC, Dh, p.S, p.cps);
  const size_t need = ws_bytes(BH, Dh, N, p.S);
  if (need > 0) {
    if (ws == nullptr || wsb < need) return rr::fail(RR_EWORKSPACE, "final-state forward: workspace too small");
    p.segE = static_cast<float4*>(ws);
    p.segP = reinterpret_cast<float*>(static_cast<char*>(ws) + decay_offset(BH, Dh, N, p.S));
  }
#define RR_CASE(D, NN) \
  if (Dh == D && N == NN) return launch<D, NN, GLA, OUT>(p, BH, s)
  if constexpr (GLA) {
    RR_CASE(32, 32);
    RR_CASE(64, 64);
    RR_CASE(128, 128);
  } else {
    RR_CASE(32, 16); RR_CASE(32, 32); RR_CASE(32, 64); RR_CASE(32, 128);
    RR_CASE(64, 16); RR_CASE(64, 32); RR_CASE(64, 64); RR_CASE(64, 128);
    RR_CASE(128, 16); RR_CASE(128, 32); RR_CASE(128, 64); RR_CASE(128, 128);
  }
#undef RR_CASE
  return rr::fail(RR_EUNSUPPORTED, "final-state forward: sizes not covered");
}

bool sizes_ok(int64_t B, int64_t L, int64_t H, int64_t Dh, int64_t N) {
  if (B <= 0 || L <= 0 || H <= 0 || Dh <= 0 || N <= 0) return false;
  // what the entry points take at all; a grid of heads; 32-bit byte offsets
  // within a chunk; int step counts
  return rr::scan_dims_ok(B, L, H) && rr::grid_ok(B * H, 4 * Dh) && L < (int64_t(1) << 30) &&
         H * std::max(Dh, N) * Q * 4 < (int64_t(1) << 31);
}

// Calls without a gradient: where seg leaves a checkpoint interval T below 32
// the other forward is the VALU engine, so every covered size runs here (bf16
// prompts of odd length: 2.8x at B1 L40 H8, 57x at B4 L1000 H80 Dh64 N128); at
// T = 32 the sizes for which the training forward walks too, and N = 32 from 24
// chunks (no checkpoints to write: SSD 36 heads Dh 32, 24 chunks 17.2 -> 14.3).
int64_t query(int64_t B, int64_t L, int64_t H, int64_t Dh, int64_t N, int64_t seg, int dtype, bool gla) {
  if (dtype != RR_BF16 || !sizes_ok(B, L, H, Dh, N) || !covered(Dh, N, gla)) return -1;
  const int64_t nC = (L + Q - 1) / Q;
  if (rr::chunk_len(L, seg) == Q && !(rr::walk_preferred(B * H, nC, Dh, N, gla) || (N == 32 && nC >= 24 && B * H >= 24)))
    return -1;
  int S, cps;
  segments(B * H, nC, Dh, S, cps);
  return (int64_t)ws_bytes(B * H, Dh, N, S);
}

}  // namespace

namespace rr {

// Measured at T = 32 with checkpoints, the walk against the other forwards
// (resident, direct, whole-head, scan + chunk kernels), us at (heads, chunks):
// - from 17 chunks with N >= 64 it never lost (1.0x at SSD B8 L4096 H80 Dh64
//   N128, 1233 -> 1224, bound by its traffic; 456 -> 215 at GLA 96 heads Dh
//   128; 1.02x to 2.24x between); with N = 32 it wins from 32 chunks (below,
//   14.8 -> 17.5 at 36 heads); with N = 16 its chunk costs as much as with 32,
//   so only where the others leave the GPU idle (up to 256 heads; 233 -> 254
//   at 640);
// - fewer than 24 heads: the chunk-parallel kernels (SSD 2 heads, 32 chunks,
//   Dh 64 N 128: 15.9 against 19.7; at 24 heads, 17 chunks 22.3 against 20.8);
// - in shorter heads the resident and direct kernels are more parallel
//   (SSD 36 heads, 16 chunks, Dh 64 N 16: 9.5 against 16.3) except
//   N = 64 from 256 heads (66 -> 44 at 320 heads, 16 chunks; 8.8 -> 6.5 at 256
//   heads, 1 chunk) unless the whole-head kernel, from 512 heads, has but one
//   or two chunks to carry (1 chunk: 8.3 against 8.8 at 512 heads, 26.6 against
//   31.6 at 2560; 2 chunks: 17.0 -> 15.9 at 640, 19.3 against 20.7 at 800; 3
//   chunks: even from 960), and
//   N = 128, which the resident kernel does not cover, below 512 heads (16
//   chunks: 123 -> 94; 8: 46 -> 36 at 256 heads; 1: 10.2 -> 6.4 at 24), unless
//   GLA's wide direct mode takes it (BH nC <= 768: 23 against 31) or Dh is 32
//   with 4 or 5 chunks of few heads, where a second segment's launch costs more
//   than the direct or pipelined kernels (4 chunks: 12.5 against 13.9 at 64
//   heads, 19.2 -> 14.0 at 72; 5: 15.1 against 16.2 at 48, 17.0 -> 16.5 at 56).
bool walk_preferred(int64_t BH, int64_t nC, int64_t Dh, int64_t N, bool gla) {
  if (BH < 24 || !grid_ok(BH, 4 * Dh)) return false;
  if (nC > 16) return N >= 64 || (nC >= 32 && (N == 32 || BH <= 256));
  if (N == 128) {
    if (Dh == 32 && ((nC == 4 && BH <= 64) || (nC == 5 && BH <= 48))) return false;
    return BH < 512 && !(gla && BH * nC <= 768);
  }
  return N == 64 && Dh == 64 && BH >= 256 && (nC >= 3 || BH < 256 * (nC + 1));
}

size_t walk_ws_bytes(int64_t B, int64_t H, int64_t nC, int64_t Dh, int64_t N) {
  int S, cps;
  segments(B * H, nC, Dh, S, cps);
  return ws_bytes(B * H, Dh, N, S);
}

int64_t walk_ws_extent(int64_t B, int64_t H, int64_t nC, int64_t Dh, int64_t N) {
  int S, cps;
  segments(B * H, nC, Dh, S, cps);
  const int64_t T = 4 * Dh, frags = std::max<int64_t>(N, 32) / 16;   // threads, float4 a thread keeps of a map
  const int64_t decays = S > 1 ? (int64_t)decay_offset(B * H, Dh, N, S) : 0;
  int64_t ext = 0;
  for (int64_t bh = 0; bh < B * H; ++bh)
    for (int j = 0; j + 1 < S; ++j) {
      const int64_t slot = chunked::map_slot(bh, S, j);
      if ((slot * frags * T + (frags - 1) * T + T) * 16 > decays) return INT64_MAX;   // into the decays
      ext = std::max(ext, decays + (slot + 1) * 4);
    }
  return ext;
}

int walk_fwd(const ChunkArgs& a, int64_t B, hipStream_t s, bool gla) {
  FinalArgs p{};
  p.u = a.u;
  p.step = a.delta;
  p.Bm = a.Bm;
  p.Cm = a.Cm;
  p.A = a.A;
  p.h0 = a.h0;
  p.y = a.y;
  p.fin = a.ckpt;
  p.L = a.L; p.H = a.H; p.nC = a.nC;
  const size_t wsb = walk_ws_bytes(B, a.H, a.nC, a.DH, a.NS);
  if (gla) return run<true, kCkpt>(p, B, a.H, a.DH, a.NS, a.ws, wsb, s);
  return run<false, kCkpt>(p, B, a.H, a.DH, a.NS, a.ws, wsb, s);
}

}  // namespace rr

extern "C" int64_t rr_ssd_final_workspace_bytes(int64_t B, int64_t L, int64_t H, int64_t Dh, int64_t N, int64_t seg,
                                                int64_t A_stride_n, int dtype) {
  if (rr::chunk_len(L, seg) == 0 || A_stride_n != 0) return -1;
  return query(B, L, H, Dh, N, seg, dtype, false);
}

extern "C" int rr_ssd_final_fwd(const void* u, const void* delta, const void* Bm, const void* Cm, const float* A_neg,
                                int64_t A_stride_n, int dtype, int64_t B, int64_t L, int64_t H, int64_t Dh, int64_t N,
                                int64_t seg, const float* h0, float* y, float* fin, void* workspace,
                                size_t workspace_bytes, void* stream) {
  if (int rc = rr::check_scan_dims("ssd_final_fwd", B, L, H, Dh, N, seg, dtype, "Dh")) return rc;
  if (!u || !delta || !Bm || !Cm || !A_neg || !y || !fin)
    return rr::fail(RR_EINVAL, "ssd_final_fwd: null pointer argument");
  if (rr_ssd_final_workspace_bytes(B, L, H, Dh, N, seg, A_stride_n, dtype) < 0)
    return rr::fail(RR_EUNSUPPORTED, "ssd_final_fwd: call not covered (rr_ssd_final_workspace_bytes is -1)");
  FinalArgs p{};
  p.u = static_cast<const uint16_t*>(u);
  p.step = static_cast<const uint16_t*>(delta);
  p.Bm = static_cast<const uint16_t*>(Bm);
  p.Cm = static_cast<const uint16_t*>(Cm);
  p.A = A_neg;
  p.h0 = h0;
  p.y = y;
  p.fin = fin;
  p.L = (int)L; p.H = (int)H; p.nC = (int)((L + Q - 1) / Q);
  return run<false, kFinal>(p, B, H, Dh, N, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}

extern "C" int64_t rr_gla_final_workspace_bytes(int64_t B, int64_t L, int64_t H, int64_t Dh, int64_t seg, int dtype) {
  if (rr::chunk_len(L, seg) == 0) return -1;
  return query(B, L, H, Dh, Dh, seg, dtype, true);
}

extern "C" int rr_gla_final_fwd(const void* q, const void* k, const void* v, const void* gates, int dtype, int64_t B,
                                int64_t L, int64_t H, int64_t Dh, int64_t seg, const float* h0, float* y, float* fin,
                                void* workspace, size_t workspace_bytes, void* stream) {
  if (int rc = rr::check_scan_dims("gla_final_fwd", B, L, H, Dh, Dh, seg, dtype, "Dh")) return rc;
  if (!q || !k || !v || !gates || !y || !fin) return rr::fail(RR_EINVAL, "gla_final_fwd: null pointer argument");
  if (rr_gla_final_workspace_bytes(B, L, H, Dh, seg, dtype) < 0)
    return rr::fail(RR_EUNSUPPORTED, "gla_final_fwd: call not covered (rr_gla_final_workspace_bytes is -1)");
  FinalArgs p{};
  p.u = static_cast<const uint16_t*>(v);
  p.step = static_cast<const uint16_t*>(gates);
  p.Bm = static_cast<const uint16_t*>(k);
  p.Cm = static_cast<const uint16_t*>(q);
  p.h0 = h0;
  p.y = y;
  p.fin = fin;
  p.L = (int)L; p.H = (int)H; p.nC = (int)((L + Q - 1) / Q);
  return run<true, kFinal>(p, B, H, Dh, Dh, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}
