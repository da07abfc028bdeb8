// Delta rule, backward for per-row beta or decay (and float32, or a head_dim that the chunked kernels
// do not take), from what the row-scan forward keeps (err and states; delta_rule_row.hip).
// Without a decay (DeltaNet), two kernels:
//
// 1. The reverse scan, 16 steps at a time in the form of the forward: with dS the gradient of the state
//    after a step, x_t = do_t,
//      du_t = (dS + do_t q_t^T) k_t;  w_t = beta_t du_t;  dS <- dS + do_t q_t^T - w_t k_t^T
//    is a row-wise recurrence that sees q and k only through dot products.  It writes du (float32) and dS
//    every 64 steps.  Roles of the waves as in the forward; the do terms of a chunk, which wait for
//    nothing, are the gram wave's.
// 2. The gradients of 64 steps, all chunks at once: with S0 the state before them and dS1 its gradient after
//    them, u_t = beta_t err_t,
//      dq_t = S0^T do_t + sum_{s <= t} (do_t . u_s) k_s
//      dk_t = dS1^T u_t - S0^T w_t + sum_{s >= t} (do_s . u_t) q_s
//             - sum_{s > t} (u_t . w_s) k_s - sum_{s < t} (w_t . u_s) k_s
//    (expand S_t and dS_t over the chunk in dq_t = S_t^T do_t and dk_t = dS_t^T u_t - S_{t-1}^T w_t:
//    lib/edifice/cuda/fused_scan.ex:1257-1431), dv = w, dbeta = err du: contractions over the rows
//    and over the steps, in float32 on v_mfma_f32_32x32x2_f32.  The sums over all rows of a head are inside
//    one workgroup, so there are no per-row-block partials to write and add.
// With a decay (GatedDeltaNet, KDA) the same two passes, the gradients per 16 steps: decays per row do not
// factor out of M and N over more steps than a short product per pair, so those sums over the rows, and
// the decay's gradient <dS_t - w_t k_t^T, S_{t-1}>, are formed one row per lane (dr_row_decay_grad_kernel).
// Forward and backward, against one workgroup per 16 rows stepping through the sequence with partial dq and
// dk per row block (its time is the chain of T steps): KDA 4x1000x8x128 bf16 875 -> 344 us,
// GatedDeltaNet 2x777x8x64 float32 470 -> 236 (213 before its float32 sums were split, see gram).
#include "edf_abi.hpp"
#include "edf_common.hpp"
#include "edf_row_scan.hpp"

namespace edf {
int dr_row_run(void* stream, const void* q, const void* k, const void* v, const void* beta, const void* alpha,
               void* out, int batch, int seq, int heads, int d, int dtype, int beta_per_head, int alpha_per_row,
               float* ckpt, float* err, int cw);
namespace {
using namespace rowscan;

template <typename TT, int DP, bool DECAY>
struct RevShared {
  static constexpr int LD = tile_ld<TT, DP>();
  static constexpr int SW = DP >= 64 ? 2 : 1;  // state waves
  TT k[4][CH * LD], q[4][CH * LD];              // the j-th chunk from the end in slot j % 4
  f32x4 w[2][64];                               // w of the chunk's steps
  f32x4 pk[2][SW][64];                          // state products of k
  f32x4 x[2][64];                               // do terms of a chunk and of the one after it
  f32x4 g[2][64], gx[2][64];                    // Gram tiles of a chunk, and of the one after with it
  f32x4 h[DECAY ? 2 : 1][DECAY ? 64 : 1], hx[DECAY ? 2 : 1][DECAY ? 64 : 1];  // the q . k tiles of the same
  float gs[2][32];                              // solve scalars
};

// p.v is do; du [B, T, H, d], p.ckpt the gradients of the states [BH][ceil(T / CPS) - 1][cw][cw] after
// each CPS steps but the last.
// With a decay (DECAY), the state gradient runs back as dS <- a_t (dS + do_t q_t^T - w_t k_t^T), and p.ckpt
// takes it after every chunk but the last, [BH][chunks][cw][cw]; the do terms of the chunk and of the
// one after it then decay with the others in the chain, and x holds only those inside a block of four.
template <typename TT, int DP, bool DECAY, bool VEC>
__global__ __launch_bounds__(64 * (2 + (DP >= 64 ? 2 : 1))) void dr_row_rev_kernel(const RowArgs p, float* du) {
  typedef RevShared<TT, DP, DECAY> Sh;
  constexpr int LD = Sh::LD, SW = Sh::SW, W = DP / SW;
  constexpr bool F32 = sizeof(TT) == 4;    // sums apart, as in the forward
  constexpr bool LAST = DECAY && F32;
  __shared__ __attribute__((aligned(16))) Sh sh;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, li = l & 15, grp = l >> 4;
  const RowIO<TT> io(p, li);
  const int nch = (p.T + CH - 1) / CH, tl = (nch - 1) * CH;

  if (wave == 0) {  // chain
    GateRegs<TT> nb, na, nd;
    nb.at(io.bbase, io.bstep, tl, grp);
    if (DECAY) na.at(io.abase, io.astep, tl, grp), nd.at(io.row0, io.step, tl, grp);
    auto load = [&]() {
      nb.load(io.rB, io.bstep, -CH);
      if (DECAY) na.load(io.rA, io.astep, -CH), nd.load(io.rV, io.step, -CH);
    };
    load();
    const long rowel = (long)p.T * p.H * p.d;
    const rsrc_t rU = make_rsrc(du + io.bh / p.H * rowel, (unsigned)(rowel * 4));
    const unsigned ustep = (unsigned)p.H * p.d * 4;
    unsigned uoff = (io.in ? ((unsigned)(io.bh % p.H) * p.d + io.i) * 4 : OOB_OFF) + (unsigned)(tl + grp) * ustep;
    f32x4 Wn = {0, 0, 0, 0}, Dn = {0, 0, 0, 0};  // -w and do of the chunk after, decayed to its start
    float dtot = 1.0f;                           // its decay
    lds_barrier();
    for (int j = 0; j < nch; ++j) {
      const int b = j & 1, t0 = (nch - 1 - j) * CH;
      const f32x4 x = sh.x[b][l];
      f32x4 e = {0, 0, 0, 0};
      if (j > 0) {
        e = sh.pk[b][0][l];
        if (SW == 2) e += sh.pk[b][SW - 1][l];
      }
      e = DECAY ? e * dtot : e + x;
      const f32x4 G = sh.g[b][l], Gx = sh.gx[b][l];
      f32x4 H, Hx;
      if (DECAY) H = sh.h[b][l], Hx = sh.hx[b][l];
      f32x4 gs[4][2];
#pragma unroll
      for (int r = 0; r < 4; ++r) gs[r][0] = *(const f32x4*)&sh.gs[b][8 * r], gs[r][1] = *(const f32x4*)&sh.gs[b][8 * r + 4];
      float bb[4][4], aa[4][4], dc[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        gather4(bits_f32(nb.v[r]), bb[r]);
        if (DECAY) {
          gather4(decay_of<TT>(na.v[r], t0 + 4 * r + grp < p.T && io.in, p.alpha_per_row), aa[r]);
          dc[r] = bits_f32(nd.v[r]);
        } else {
          aa[r][0] = aa[r][1] = aa[r][2] = aa[r][3] = 1.0f;
        }
      }
      load();
      e = tile_dot<F32>(Gx, Wn, e);
      if (DECAY) e = tile_dot<F32>(Hx, Dn, e);
      dtot = 1.0f;
      f32x4 raw, in = {0, 0, 0, 0};  // in: the part of e from the chunk's own steps (bf16: in e)
#pragma unroll
      for (int r = 3; r >= 0; --r) {
        auto g = [&](int m, int n) { return gs[r][pair(m, n) >> 2][pair(m, n) & 3]; };
        const BlockDecay D(aa[r], grp);
        float y[4], w[4];
        // what the chunk's do give within the block enters last (float32), as v in the forward
        const float er = F32 ? e[r] + in[r] : e[r];
        if constexpr (LAST)
          gather4(D.end * er, y);
        else
          gather4(DECAY ? fmaf(D.end, er, x[r]) : er, y);
        float xx[4] = {};
        if constexpr (LAST) gather4(x[r], xx);
        auto last = [&](float v, int m) { return LAST ? v + xx[m] : v; };
        y[3] = last(y[3], 3);
        w[3] = bb[r][3] * y[3];
        y[2] = last(fmaf(-(DECAY ? g(2, 3) * D.r32 : g(2, 3)), w[3], y[2]), 2);
        w[2] = bb[r][2] * y[2];
        y[1] = last(fmaf(-(DECAY ? g(1, 2) * D.r21 : g(1, 2)), w[2],
                         fmaf(-(DECAY ? g(1, 3) * D.r31 : g(1, 3)), w[3], y[1])), 1);
        w[1] = bb[r][1] * y[1];
        y[0] = last(fmaf(-(DECAY ? g(0, 1) * D.r10 : g(0, 1)), w[1],
                         fmaf(-(DECAY ? g(0, 2) * D.r20 : g(0, 2)), w[2],
                              fmaf(-(DECAY ? g(0, 3) * D.r30 : g(0, 3)), w[3], y[0]))), 0);
        w[0] = bb[r][0] * y[0];
        const float wo = -pick4(w[0], w[1], w[2], w[3], grp), wn = DECAY ? wo * D.pre : wo;
        raw[r] = wo;
        f32x4& own = F32 ? in : e;
        if (r > 0) own = mfma4(G[r], wn, DECAY ? own * D.all : own);
        if (DECAY) {
          const float dn = dc[r] * D.pre;
          if (r > 0) own = mfma4(H[r], dn, own);
          if (F32) e *= D.all;
#pragma unroll
          for (int n = r + 1; n < 4; ++n) Wn[n] *= D.all, Dn[n] *= D.all;
          Dn[r] = dn;
          dtot *= D.all;
        }
        Wn[r] = wn;
        bstore<float>(rU, uoff + 4 * r * ustep, pick4(y[0], y[1], y[2], y[3], grp));
      }
      uoff -= CH * ustep;
      sh.w[b][l] = -raw;
      lds_barrier();
    }
  } else if (wave <= SW) {  // state gradient, W columns
    const int half = wave - 1;
    f32x4 S[W / 16];
#pragma unroll
    for (int jt = 0; jt < W / 16; ++jt) S[jt] = f32x4{0, 0, 0, 0};
    GateRegs<TT> nd, na;
    nd.at(io.row0, io.step, tl, grp);
    nd.load(io.rV, io.step, -CH);
    if (DECAY) na.at(io.abase, io.astep, tl, grp), na.load(io.rA, io.astep, -CH);
    lds_barrier();
    for (int j = 0; j < nch; ++j) {
      const int c = nch - 1 - j;
      RowFrag<TT, W> kf;
      kf.template load<LD>(sh.k[(j + 1) & 3] + W * half, li, grp);
      if (j > 0) {
        ColFrag<TT, W> kc, qc;
        kc.template load<LD>(sh.k[(j - 1) & 3] + W * half, li, grp);
        qc.template load<LD>(sh.q[(j - 1) & 3] + W * half, li, grp);
        if (DECAY) {
          f32x4 x, wn = -sh.w[(j - 1) & 1][l];  // decayed to the start of chunk c + 1
          float dt = 1.0f;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float aa[4];
            gather4(decay_of<TT>(na.v[r], (c + 1) * CH + 4 * r + grp < p.T && io.in, p.alpha_per_row), aa);
            const BlockDecay D(aa, grp);
            x[r] = bits_f32(nd.v[r]) * (D.pre * dt);
            wn[r] *= D.pre * dt;
            dt *= D.all;
          }
          na.load(io.rA, io.astep, -CH);
#pragma unroll
          for (int jt = 0; jt < W / 16; ++jt) S[jt] *= dt;
          state_add<W>(S, qc, x);
          state_add<W>(S, kc, wn);
        } else {
          state_add2<W>(S, qc, nd.v, kc, sh.w[(j - 1) & 1][l]);
        }
        nd.load(io.rV, io.step, -CH);
        if ((DECAY || (c + 1) % (CPS / CH) == 0) && io.i < p.cw) {
          const long slot = DECAY ? io.bh * nch + c : io.bh * ((p.T + CPS - 1) / CPS - 1) + c / (CPS / CH);
          float* cp = p.ckpt + (slot * p.cw + io.i) * p.cw + W * half + 4 * grp;
#pragma unroll
          for (int jt = 0; jt < W / 16; ++jt)
            if (W * half + 16 * jt < p.cw) *(f32x4*)(cp + 16 * jt) = S[jt];
        }
      }
      sh.pk[(j + 1) & 1][half][l] = state_dot<W>(kf, S);
      lds_barrier();
    }
  } else {  // gram, do terms, staging
    TileRegs<TT, DP, VEC> nk, nq;
    GateRegs<TT> nd, na;
    if (DECAY) na.at(io.abase, io.astep, tl, grp);
    nk.at(io.base, io.step, tl, p.d, l);
    nq.at(io.base, io.step, tl, p.d, l);
    nd.at(io.row0, io.step, tl, grp);
    RowFrag<TT, DP> kp = {}, qp = {};  // rows of the chunk after the one whose tiles are formed
    f32x4 dp = {0, 0, 0, 0};           // and its do
    const int t = sigma(li);
    const int gm = grp, gn = li >> 2, gr = li & 3;  // the solve scalar this lane holds
    auto grams = [&](int j) {
      RowFrag<TT, DP> kf, qf;
      kf.template load<LD>(sh.k[j & 3], li, grp);
      qf.template load<LD>(sh.q[j & 3], li, grp);
      const f32x4 dc = {bits_f32(nd.v[0]), bits_f32(nd.v[1]), bits_f32(nd.v[2]), bits_f32(nd.v[3])};
      nd.load(io.rV, io.step, -CH);
      const f32x4 G = gram<DECAY, DP>(kf, kf), H = gram<DECAY, DP>(qf, kf), Hx = gram<DECAY, DP>(qp, kf);
      sh.g[j & 1][l] = G;
      sh.gx[j & 1][l] = gram<DECAY, DP>(kp, kf);
      const float gv = gr == 0 ? G[0] : gr == 1 ? G[1] : gr == 2 ? G[2] : G[3];
      if (gm < gn) sh.gs[j & 1][8 * gr + pair(gm, gn)] = gv;
      f32x4 x = {0, 0, 0, 0};
      if constexpr (DECAY) {
        sh.h[j & 1][l] = H;
        sh.hx[j & 1][l] = Hx;
        const int t0 = (nch - 1 - j) * CH;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float aa[4], dd[4];
          gather4(decay_of<TT>(na.v[r], t0 + 4 * r + grp < p.T && io.in, p.alpha_per_row), aa);
          gather4(dc[r], dd);
          const BlockDecay D(aa, grp);
#pragma unroll
          for (int n = 0; n < 4; ++n) {
            const int s = F32 ? 3 - n : n;  // (float32: the lane's own step, whose term is the largest, last)
            // decay from after the lane's step to step s; q_s . k of the lane's step
            const float rs = s == 3   ? pick4(D.r30, D.r31, D.r32, 1.0f, grp)
                             : s == 2 ? pick4(D.r20, D.r21, 1.0f, 1.0f, grp)
                             : s == 1 ? (grp == 0 ? D.r10 : 1.0f)
                                      : 1.0f;
            const float hs = __shfl(H[r], 16 * s + 4 * grp + r);
            x[r] = s >= grp ? fmaf(dd[s] * rs, hs, x[r]) : x[r];
          }
        }
        na.load(io.rA, io.astep, -CH);
        sh.x[j & 1][l] = x;
        kp = kf, qp = qf;
        return;
      }
      x = tile_dot<F32>(Hx, dp, x);
      const bool finite = fabsf(dc[0]) < INFINITY && fabsf(dc[1]) < INFINITY && fabsf(dc[2]) < INFINITY &&
                          fabsf(dc[3]) < INFINITY;
      if (!__any(!finite)) {
        // do_s (q_s . k_t) over the steps s >= t of the chunk (an earlier step's do enters with 0)
        f32x4 h;
#pragma unroll
        for (int r = 0; r < 4; ++r) h[r] = 4 * r + grp >= t ? H[r] : 0.0f;
        x = tile_dot<F32>(h, dc, x);
      } else {
#pragma unroll
        for (int s = 0; s < CH; ++s) {
          const float ds = __shfl(dc[s >> 2], 16 * (s & 3) + li);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float h = __shfl(H[s >> 2], 16 * (s & 3) + 4 * grp + r);  // q_s . k of step 4 r + grp
            x[r] = s >= 4 * r + grp ? fmaf(ds, h, x[r]) : x[r];
          }
        }
      }
      sh.x[j & 1][l] = x;
      kp = kf, qp = qf, dp = dc;
    };
    auto stage = [&](int j) {
      nk.store(sh.k[j & 3], l);
      nq.store(sh.q[j & 3], l);
      nk.load(io.rK, io.step, -CH);
      nq.load(io.rQ, io.step, -CH);
    };
    nk.load(io.rK, io.step, -CH);
    nq.load(io.rQ, io.step, -CH);
    nd.load(io.rV, io.step, -CH);
    if (DECAY) na.load(io.rA, io.astep, -CH);
    stage(0);
    stage(1);
    grams(0);
    lds_barrier();
    for (int j = 0; j < nch; ++j) {
      stage(j + 2);
      if (j + 1 < nch) grams(j + 1);
      lds_barrier();
    }
  }
}

struct GradArgs {
  const void *q, *k, *dout, *beta;
  const float *err, *du, *ckpt, *dckpt;
  void *dq, *dk, *dv, *dbeta;
  int H, T, d, beta_per_head;
  bool vec;  // d a multiple of 8, tensors 4-byte aligned
};

EDF_DEVICE f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// One workgroup per 64 steps of a head.  Wave (ct, rt) forms the 32 x 32 tile of dq and of dk at steps
// 32 rt .., columns 32 ct ..; the row factors do, u and -w are in LDS as float32, and so are the
// 64 x 64 tiles M = do u^T (s <= t) and N = -(u w^T, its strict upper part, mirrored).
// One workgroup per CU (136 KB of LDS at head_dim 128), so nothing else covers its waits: the row factors move in
// 16-byte pieces (element by element 23k cycles of a workgroup's 93k at 8x2048x8x128 bf16, 10k so), and the states
// arrive two stages of 32 rows ahead of their products (51k -> 42k, of which the f32 MFMAs take 32k).
template <typename TT, int DP>
__global__ __launch_bounds__(4 * DP) void dr_row_grad_kernel(const GradArgs p) {
  constexpr int LD = DP + 4, LM = CPS + 4, CT = DP / 32, NTH = 4 * DP, PER = DP / 4;
  constexpr int NA = sizeof(TT) == 4 ? 2 : 1;  // accumulators per sum (see below)
  __shared__ __attribute__((aligned(16))) float sD[CPS * LD], sU[CPS * LD], sW[CPS * LD];
  __shared__ __attribute__((aligned(16))) float sM[CPS * LM], sN[CPS * LM];
  const int n64 = (p.T + CPS - 1) / CPS;
  const long bh = blockIdx.x / n64;
  const int C = blockIdx.x % n64, t0 = C * CPS, d = p.d;
  const int b = (int)(bh / p.H), h = (int)(bh % p.H);
  const long rowel = (long)p.T * p.H * d, headel = (long)p.T * p.H;
  const unsigned rowb = (unsigned)(rowel * sizeof(TT)), rowf = (unsigned)(rowel * 4);
  const rsrc_t rQ = make_rsrc((const TT*)p.q + b * rowel, rowb), rK = make_rsrc((const TT*)p.k + b * rowel, rowb);
  const rsrc_t rG = make_rsrc((const TT*)p.dout + b * rowel, rowb);
  const rsrc_t rB = p.beta_per_head
                        ? make_rsrc((const TT*)p.beta + b * headel, (unsigned)(headel * sizeof(TT)))
                        : make_rsrc((const TT*)p.beta + b * rowel, rowb);
  const rsrc_t rE = make_rsrc(p.err + b * rowel, rowf), rU = make_rsrc(p.du + b * rowel, rowf);
  const rsrc_t rDQ = make_rsrc((TT*)p.dq + b * rowel, rowb), rDK = make_rsrc((TT*)p.dk + b * rowel, rowb);
  const rsrc_t rDV = make_rsrc((TT*)p.dv + b * rowel, rowb);
  const rsrc_t rDB = p.beta_per_head ? make_rsrc((TT*)p.dbeta + b * headel, (unsigned)(headel * sizeof(TT)))
                                     : make_rsrc((TT*)p.dbeta + b * rowel, rowb);
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, g = l >> 5, li = l & 31;
  const int ct = w % CT, rt = w / CT, j = 32 * ct + li;

  const unsigned hd = (unsigned)(p.H * d);
  // S0 and dS1 in stages of 32 rows (an empty buffer reads zero), two stages ahead
  const bool has0 = C > 0, has1 = C < n64 - 1;
  const rsrc_t rS0 = make_rsrc(p.ckpt + (has0 ? (bh * (n64 - 1) + C - 1) * DP * DP : 0), has0 ? DP * DP * 4u : 0u);
  const rsrc_t rS1 = make_rsrc(p.dckpt + (has1 ? (bh * (n64 - 1) + C) * DP * DP : 0), has1 ? DP * DP * 4u : 0u);
  constexpr int ST = DP / 32;
  float sv[2][16];
  auto load_stage = [&](int st, float (&v)[16]) {
#pragma unroll
    for (int x = 0; x < 16; ++x)
      v[x] = bits_f32(__builtin_amdgcn_raw_buffer_load_b32(st < ST ? rS0 : rS1, (int)(((4 * g + (x & 3)) * DP + j) * 4),
                                                           (32 * (st % ST) + 8 * (x >> 2)) * DP * 4, 0));
  };

  // row factors, dv and dbeta
  if (p.vec) {  // eight columns at a time (a piece is inside the head or past it)
    constexpr int P8 = DP / 8, NV = 4 * sizeof(TT) / 8;  // 16-byte pieces of 8 elements of TT
    auto load8 = [](rsrc_t r, unsigned off, float (&v)[8]) {
      if constexpr (sizeof(TT) == 4) {
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(off + 16 * y), 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[4 * y + e] = bits_f32(x[e]);
        }
      } else {
        const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[2 * e] = bits_f32(x[e] << 16);
          v[2 * e + 1] = bits_f32(x[e] & 0xffff0000u);
        }
      }
    };
    auto load8f = [](rsrc_t r, unsigned off, float (&v)[8]) {
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(off + 16 * y), 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * y + e] = bits_f32(x[e]);
      }
    };
    auto store8 = [](rsrc_t r, unsigned off, const float (&v)[8]) {
#pragma unroll
      for (int y = 0; y < NV; ++y) {
        u32x4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (sizeof(TT) == 4) {
            x[e] = __builtin_bit_cast(unsigned, v[4 * y + e]);
          } else {
            typedef __attribute__((ext_vector_type(2))) bf16 bf16x2;
            x[e] = __builtin_bit_cast(unsigned, bf16x2{(bf16)v[2 * e], (bf16)v[2 * e + 1]});
          }
        }
        __builtin_amdgcn_raw_buffer_store_b128(x, r, (int)(off + 16 * y), 0, 0);
      }
    };
    constexpr int NI = CPS * P8 / NTH;
    float er[NI][8], du[NI][8], go[NI][8], be[NI][8];
#pragma unroll
    for (int n = 0; n < NI; ++n) {
      const int e = tid + NTH * n, i0 = 8 * (e % P8);
      const unsigned t = t0 + e / P8, el = t * hd + h * d + i0, o = i0 < d ? el * (unsigned)sizeof(TT) : OOB_OFF;
      load8f(rE, i0 < d ? el * 4u : OOB_OFF, er[n]);
      load8f(rU, i0 < d ? el * 4u : OOB_OFF, du[n]);
      load8(rG, o, go[n]);
      if (p.beta_per_head) {
        be[n][0] = bits_f32(bload<TT>(rB, (t * p.H + h) * (unsigned)sizeof(TT)));
#pragma unroll
        for (int x = 1; x < 8; ++x) be[n][x] = be[n][0];
      } else {
        load8(rB, o, be[n]);
      }
    }
    load_stage(0, sv[0]);
#pragma unroll
    for (int n = 0; n < NI; ++n) {
      const int e = tid + NTH * n, row = e / P8, i0 = 8 * (e % P8);
      const unsigned t = t0 + row, o = i0 < d ? (t * hd + h * d + i0) * (unsigned)sizeof(TT) : OOB_OFF;
      float wv[8], db[8];
#pragma unroll
      for (int x = 0; x < 8; ++x) {
        wv[x] = be[n][x] * du[n][x];
        db[x] = er[n][x] * du[n][x];
        sD[row * LD + i0 + x] = go[n][x];
        sU[row * LD + i0 + x] = be[n][x] * er[n][x];
        sW[row * LD + i0 + x] = -wv[x];
      }
      store8(rDV, o, wv);
      if (!p.beta_per_head) {
        store8(rDB, o, db);
      } else {  // summed over the rows: the P8 lanes of this step
        float v = ((db[0] + db[1]) + (db[2] + db[3])) + ((db[4] + db[5]) + (db[6] + db[7]));
#pragma unroll
        for (int m = 1; m < P8; m *= 2) v += __shfl_xor(v, m);
        bstore<TT>(rDB, i0 == 0 ? (t * p.H + h) * (unsigned)sizeof(TT) : OOB_OFF, v);
      }
    }
  } else {
#pragma unroll
    for (int n = 0; n < CPS * PER / NTH; ++n) {
      const int e = tid + NTH * n, row = e / PER, i0 = 4 * (e % PER);
      const unsigned t = t0 + row, el = t * hd + h * d + i0;
      f32x4 er, du, be, go;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const bool in = i0 + x < d;
        const unsigned o = in ? (el + x) * (unsigned)sizeof(TT) : OOB_OFF;
        er[x] = bits_f32(bload<float>(rE, in ? (el + x) * 4u : OOB_OFF));
        du[x] = bits_f32(bload<float>(rU, in ? (el + x) * 4u : OOB_OFF));
        go[x] = bits_f32(bload<TT>(rG, o));
        be[x] = bits_f32(bload<TT>(rB, p.beta_per_head ? (t * p.H + h) * (unsigned)sizeof(TT) : o));
      }
      const f32x4 wv = be * du, db = er * du;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const unsigned o = i0 + x < d ? (el + x) * (unsigned)sizeof(TT) : OOB_OFF;
        bstore<TT>(rDV, o, wv[x]);
        if (!p.beta_per_head) bstore<TT>(rDB, o, db[x]);
      }
      if (p.beta_per_head) {  // summed over the rows: the PER lanes of this step
        float s = (db[0] + db[1]) + (db[2] + db[3]);
#pragma unroll
        for (int m = 1; m < PER; m *= 2) s += __shfl_xor(s, m);
        bstore<TT>(rDB, i0 == 0 ? (t * p.H + h) * (unsigned)sizeof(TT) : OOB_OFF, s);
      }
      *(f32x4*)(sD + row * LD + i0) = go;
      *(f32x4*)(sU + row * LD + i0) = be * er;
      *(f32x4*)(sW + row * LD + i0) = -wv;
    }
    load_stage(0, sv[0]);
  }
  __syncthreads();
  load_stage(1, sv[1]);

  // this lane's k and q values of the 64 steps (column j, steps 8 kk + 4 g + e), used last
  typename Bits<TT>::type kr[CPS / 2], qr[CPS / 2];
#pragma unroll
  for (int i = 0; i < CPS / 2; ++i) {
    const unsigned t = t0 + 8 * (i >> 2) + 4 * g + (i & 3);
    const unsigned off = j < d ? (t * hd + h * d + j) * (unsigned)sizeof(TT) : OOB_OFF;
    kr[i] = bload<TT>(rK, off);
    qr[i] = bload<TT>(rQ, off);
  }

  // the Gram tiles over the rows: M (0,0) (1,0) (1,1), N (0,0) (0,1) (1,1)
  for (int job = w; job < 6; job += 2 * CT) {
    const bool isM = job < 3;
    const int jj = isM ? job : job - 3;
    const int tr = isM ? (jj > 0) : (jj > 1), tc = isM ? (jj > 1) : (jj > 0);
    const float* A = (isM ? sD : sU) + (32 * tr + li) * LD + 4 * g;
    const float* B = (isM ? sU : sW) + (32 * tc + li) * LD + 4 * g;
    f32x16 acc[NA];
#pragma unroll
    for (int n = 0; n < NA; ++n) acc[n] = zero16();
#pragma unroll 4
    for (int kk = 0; kk < DP / 8; ++kk) {
      const f32x4 av = *(const f32x4*)(A + 8 * kk), bv = *(const f32x4*)(B + 8 * kk);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e % NA] = mfma_f32(av[e], bv[e], acc[e % NA]);
    }
#pragma unroll
    for (int n = 1; n < NA; ++n) acc[0] += acc[n];
    const int col = 32 * tc + li;
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const int row = 32 * tr + d_row(x, g);
      if (isM) {
        sM[row * LM + col] = col <= row ? acc[0][x] : 0.0f;
      } else if (row <= col) {
        const float v = row < col ? acc[0][x] : 0.0f;
        sN[row * LM + col] = v;
        sN[col * LM + row] = v;
      }
    }
  }

  // float32: the terms of S0, dS1 and the chunk's own steps in accumulators of their own
  f32x16 dqs[NA], dks[2 * NA - 1];
#pragma unroll
  for (int n = 0; n < NA; ++n) dqs[n] = zero16();
#pragma unroll
  for (int n = 0; n < 2 * NA - 1; ++n) dks[n] = zero16();
  f32x16 &dq = dqs[0], &dk = dks[0], &dk1 = dks[NA - 1], &dqc = dqs[NA - 1], &dkc = dks[2 * NA - 2];
  const float* aD = sD + (32 * rt + li) * LD + 4 * g;
  const float* aU = sU + (32 * rt + li) * LD + 4 * g;
  const float* aW = sW + (32 * rt + li) * LD + 4 * g;
  static_for<2 * ST>([&](auto sti) {
    constexpr int st = decltype(sti)::value;
    float(&v)[16] = sv[st & 1];
    if (st < ST ? has0 : has1) {
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int at = 32 * (st % ST) + 8 * x;
        if constexpr (st < ST) {
          const f32x4 dv = *(const f32x4*)(aD + at), wv = *(const f32x4*)(aW + at);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            dq = mfma_f32(dv[e], v[4 * x + e], dq);
            dk = mfma_f32(wv[e], v[4 * x + e], dk);
          }
        } else {
          const f32x4 uv = *(const f32x4*)(aU + at);
#pragma unroll
          for (int e = 0; e < 4; ++e) dk1 = mfma_f32(uv[e], v[4 * x + e], dk1);
        }
      }
    }
    if constexpr (st + 2 < 2 * ST) load_stage(st + 2, v);
  });
  __syncthreads();  // M and N

  bool finite = true;
#pragma unroll
  for (int i = 0; i < CPS / 2; ++i)
    finite = finite && fabsf(bits_f32(kr[i])) < INFINITY && fabsf(bits_f32(qr[i])) < INFINITY;
  const float* aM = sM + (32 * rt + li) * LM + 4 * g;
  const float* aN = sN + (32 * rt + li) * LM + 4 * g;
  const float* aT = sM + 4 * g * LM + 32 * rt + li;  // column of M
  if (!__any(!finite)) {
#pragma unroll
    for (int kk = 0; kk < CPS / 8; ++kk) {
      const bool useM = rt == 1 || kk < 4, useT = rt == 0 || kk >= 4;
      const f32x4 nv = *(const f32x4*)(aN + 8 * kk);
#pragma unroll
      for (int e = 0; e < 4; ++e) dkc = mfma_f32(nv[e], bits_f32(kr[4 * kk + e]), dkc);
      if (useM) {
        const f32x4 mv = *(const f32x4*)(aM + 8 * kk);
#pragma unroll
        for (int e = 0; e < 4; ++e) dqc = mfma_f32(mv[e], bits_f32(kr[4 * kk + e]), dqc);
      }
      if (useT) {
#pragma unroll
        for (int e = 0; e < 4; ++e) dkc = mfma_f32(aT[(8 * kk + e) * LM], bits_f32(qr[4 * kk + e]), dkc);
      }
    }
    if constexpr (NA > 1) dq += dqc, dk += dk1 + dkc;
  } else {  // a step outside a sum must not enter it even with 0: the pairs one by one
#pragma unroll 1
    for (int s = 0; s < CPS; ++s) {
      const unsigned off = j < d ? ((t0 + s) * hd + h * d + j) * (unsigned)sizeof(TT) : OOB_OFF;
      const float ks = bits_f32(bload<TT>(rK, off)), qs = bits_f32(bload<TT>(rQ, off));
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        const int t = 32 * rt + d_row(x, g);
        if (s <= t) dq[x] = fmaf(sM[t * LM + s], ks, dq[x]);
        if (s >= t) dk[x] = fmaf(sM[s * LM + t], qs, dk[x]);
        if (s != t) dk[x] = fmaf(sN[t * LM + s], ks, dk[x]);
      }
    }
    if constexpr (NA > 1) dk += dk1;
  }
#pragma unroll
  for (int x = 0; x < 16; ++x) {
    const unsigned t = t0 + 32 * rt + d_row(x, g);
    const unsigned off = j < d ? (t * hd + h * d + j) * (unsigned)sizeof(TT) : OOB_OFF;
    bstore<TT>(rDQ, off, dq[x]);
    bstore<TT>(rDK, off, dk[x]);
  }
}

// ---- with a decay: the gradients of 16 steps ------------------------------------------------------
struct DecayArgs {
  const void *q, *k, *dout, *beta, *alpha;
  const float *err, *du, *ckpt, *dckpt;  // states after each chunk, and their gradients (all but the last chunk's)
  void *dq, *dk, *dv, *dbeta, *dalpha;
  int H, T, d, beta_per_head, alpha_per_row;
};

// Sums over the wave's lanes: lane n receives the sum of buf[n].  A reduce-scatter without LDS: halves of the wave
// and of each half exchange by swaps (of buf[k] and buf[k + n], whose sum then has either index where it belongs),
// the last 16 lanes by DPP mirrors and quad permutes (pairings of lanes that agree in the bits already settled).
EDF_DEVICE float scatter16(float* buf, int lane) {  // within each 16 lanes: lane n receives the sum of buf[n & 15]
  static_for<4>([&](auto step) {
    constexpr int n = 8 >> decltype(step)::value, ctrl[4] = {0x140, 0x141, 0x4E, 0xB1};  // ^ 15, ^ 7, ^ 2, ^ 1
    const bool up = (lane & n) != 0;
#pragma unroll
    for (int k = 0; k < n; ++k) {
      const float send = up ? buf[k] : buf[k + n], keep = up ? buf[k + n] : buf[k];
      buf[k] = keep + dpp_f32<ctrl[decltype(step)::value]>(send);
    }
  });
  return buf[0];
}
EDF_DEVICE float scatter64(float (&buf)[64], int lane) {
#pragma unroll
  for (int k = 0; k < 32; ++k) {
    swap32(buf[k], buf[k + 32]);
    buf[k] += buf[k + 32];
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    swap16(buf[k], buf[k + 16]);
    buf[k] += buf[k + 16];
  }
  return scatter16(buf, lane);
}

// One workgroup per chunk of 16 steps of a head.  With A_t the decay from the chunk's start through step t,
// B_t that after it to the end, R(t, s) from after s through t, S0 the state before the chunk, dS1 its
// gradient after it (all per row i, sums over i):
//   dq_t = (do_t A_t) S0 + sum_{s <= t} M(t, s) k_s,          M(t, s) = sum do_t R(t, s) u_s
//   dk_t = (u_t B_t) dS1 - (w_t A_t) S0 + sum_{s >= t} M(s, t) q_s - sum_{s != t} N(t, s) k_s,
//                                                              N(t, s) = sum u_t R(s, t) w_s, t < s, mirrored
//   dalpha_t = sum <D_t, S_{t-1}>,  D_t = dS_t - w_t k_t^T: with z = <D_t, S0> and e_s = D_t k_s carried back over
//   the steps, <D_t, S_{t-1}> is Horner's rule z, then v <- a_s v + u_s e_s for s < t (no division by a decay)
// Phases: products of k, q with S0 and dS1 (f32 MFMA); one row per lane: z, e, dalpha and the decayed factors
// (waves 0 and 1), M and N (waves 2 and 3); products of those with S0, dS1, k and q, each wave 16 columns of four
// in a lane (whole 256-byte rows of S per load) and a part of the rows, the parts added in LDS.
// The states before the first chunk and the gradients after the last are zero: an empty buffer reads so, and the
// loads stay unconditional, in flight together (each behind a branch was waited for by itself: with the row phase on
// two of the four waves, 159k cycles a workgroup at KDA 4x1000x8x128 bf16, 74k now).  At 128 columns it spills 13
// registers in bf16 and 34 in float32, whose sums take more of them.
template <typename TT, int DP>
__global__ __launch_bounds__(256, 2) void dr_row_decay_grad_kernel(const DecayArgs p) {
  constexpr int LD = DP + 4, NT = DP / 16, LM = CH + 4, NP = 136 + 120;
  constexpr int VC = DP >= 64 ? 4 : 2, NC = DP >= 64 ? DP / 64 : 1;  // last phase: columns of a lane, groups of 16 VC
  constexpr int KS = 4 / NC < NT ? 4 / NC : NT, KX = NT / KS;        // parts of the rows, 16-row blocks of a part
  typedef f32x4 Part[NC][VC][64];
  struct Products {
    float P[CH * LD], O[CH * LD], E[CH * LD];
  };
  union Shared {
    Products f;
    Part part[2][KS > 1 ? KS - 1 : 1];  // dq, dk
  };
  __shared__ __attribute__((aligned(16))) float sK[CH * LD], sQ[CH * LD], sD[CH * LD], sU[CH * LD], sW[CH * LD];
  __shared__ __attribute__((aligned(16))) Shared sh;
  __shared__ __attribute__((aligned(16))) float sG[CH * CH], sH[CH * CH], sM[CH * LM], sN[CH * LM];
  __shared__ float sZ[DP], red[DP == 128 ? 2 : 1][NP + 2 * CH];
  __shared__ int sBad[4];
  float *const sP = sh.f.P, *const sO = sh.f.O, *const sE = sh.f.E;
  const int nch = (p.T + CH - 1) / CH;
  const long bh = blockIdx.x / nch;
  const int c = blockIdx.x % nch, t0 = c * CH, d = p.d;
  const int b = (int)(bh / p.H), h = (int)(bh % p.H);
  const long rowel = (long)p.T * p.H * d, headel = (long)p.T * p.H;
  const unsigned rowb = (unsigned)(rowel * sizeof(TT)), rowf = (unsigned)(rowel * 4);
  const unsigned headb = (unsigned)(headel * sizeof(TT));
  auto row_rsrc = [&](const void* t) { return make_rsrc((const TT*)t + b * rowel, rowb); };
  auto head_rsrc = [&](const void* t) { return make_rsrc((const TT*)t + b * headel, headb); };
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, li = l & 15, grp = l >> 4;
  const unsigned hd = (unsigned)(p.H * d);
  const bool has0 = c > 0, has1 = c < nch - 1;
  const rsrc_t rS0 = make_rsrc(p.ckpt + (has0 ? (bh * nch + c - 1) * DP * DP : 0), has0 ? DP * DP * 4u : 0u);
  const rsrc_t rS1 = make_rsrc(p.dckpt + (has1 ? (bh * nch + c) * DP * DP : 0), has1 ? DP * DP * 4u : 0u);
  auto el_off = [&](int t, int i) {  // byte offset of (step t of the chunk, column i), out of bounds past d
    return i < d ? ((unsigned)(t0 + t) * hd + h * d + i) * (unsigned)sizeof(TT) : OOB_OFF;
  };
  auto head_off = [&](int t) { return ((unsigned)(t0 + t) * p.H + h) * (unsigned)sizeof(TT); };

  const rsrc_t rQ = row_rsrc(p.q), rK = row_rsrc(p.k);
  constexpr int NE = CH * DP / 256;
  float kv[NE], qv[NE];
#pragma unroll
  for (int n = 0; n < NE; ++n) {
    const int e = tid + 256 * n, t = e / DP, col = e % DP;
    kv[n] = bits_f32(bload<TT>(rK, el_off(t, col)));
    qv[n] = bits_f32(bload<TT>(rQ, el_off(t, col)));
  }
  // one row per lane, in either pair of waves: this chunk's gates and factors
  const bool first = w < 2;
  const int i = tid & 127, ic = min(i, DP - 1);  // (head_dim 32: half the lanes of the wave idle)
  const bool rows = (w & 1) < (DP + 63) / 64, mine = i < DP;
  float u[CH], wv[CH], go[CH], a[CH];
  // sums over all rows, one step a lane, of a value per row that is 0 past d (per-head dbeta and dalpha)
  auto put_sums = [&](float (&x)[CH], int at) {
#pragma unroll
    for (int t = 0; t < CH; ++t) x[t] = i < d ? x[t] : 0.0f;
    float v = scatter16(x, l);
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    if (l < CH) red[w & 1][at + l] = v;
  };
  if (rows) {
    const rsrc_t rG = row_rsrc(p.dout), rB = p.beta_per_head ? head_rsrc(p.beta) : row_rsrc(p.beta);
    const rsrc_t rA = p.alpha_per_row ? row_rsrc(p.alpha) : head_rsrc(p.alpha);
    const rsrc_t rE = make_rsrc(p.err + b * rowel, rowf), rU = make_rsrc(p.du + b * rowel, rowf);
    float db[CH];
#pragma unroll
    for (int t = 0; t < CH; ++t) {
      const unsigned fo = i < d ? ((unsigned)(t0 + t) * hd + h * d + i) * 4u : OOB_OFF;
      const float er = bits_f32(bload<float>(rE, fo)), du = bits_f32(bload<float>(rU, fo));
      const float be = bits_f32(bload<TT>(rB, p.beta_per_head ? head_off(t) : el_off(t, i)));
      go[t] = bits_f32(bload<TT>(rG, el_off(t, i)));
      a[t] = decay_of<TT>(bload<TT>(rA, p.alpha_per_row ? el_off(t, i) : head_off(t)), t0 + t < p.T && i < d,
                          p.alpha_per_row);
      u[t] = be * er;
      wv[t] = be * du;
      db[t] = er * du;
    }
    if (first) {
      const rsrc_t rDV = row_rsrc(p.dv), rDB = p.beta_per_head ? head_rsrc(p.dbeta) : row_rsrc(p.dbeta);
#pragma unroll
      for (int t = 0; t < CH; ++t) {
        bstore<TT>(rDV, el_off(t, i), wv[t]);
        if (!p.beta_per_head) bstore<TT>(rDB, el_off(t, i), db[t]);
      }
      if (p.beta_per_head) put_sums(db, NP);
    }
  }
  for (int n = tid; n < CH * LM; n += 256) sM[n] = sN[n] = 0.0f;
  bool bad = false;
#pragma unroll
  for (int n = 0; n < NE; ++n) {
    const int e = tid + 256 * n, t = e / DP, col = e % DP;
    sK[t * LD + col] = kv[n];
    sQ[t * LD + col] = qv[n];
    bad = bad || !(fabsf(kv[n]) < INFINITY) || !(fabsf(qv[n]) < INFINITY);
  }
  bad = __any(bad);
  if (l == 0) sBad[w] = bad;
  __syncthreads();

  // S0 k, S0 q, dS1 k and <dS1, S0> per row; the Gram tiles
  const f32x4 zero = {0, 0, 0, 0};
#pragma unroll 1
  for (int it = w; it < NT; it += 4) {
    u32x4 s0[NT], s1[NT];
#pragma unroll
    for (int jt = 0; jt < NT; ++jt) {
      const int at = (li * DP + 16 * jt + 4 * grp) * 4, blk = 16 * it * DP * 4;
      s0[jt] = __builtin_amdgcn_raw_buffer_load_b128(rS0, at, blk, 0);
      s1[jt] = __builtin_amdgcn_raw_buffer_load_b128(rS1, at, blk, 0);
    }
    // float32: several chains, added as a tree (four at 128 columns spill: 768 -> 864 us, KDA 8x777x8x128; at 32 they
    // cost the occupancy)
    constexpr int NA = sizeof(TT) == 4 ? (DP == 64 ? 4 : 2) : 1;
    f32x4 pk[NA] = {}, pq[NA] = {}, ek[NA] = {};
    float zs[NA] = {};
#pragma unroll
    for (int jt = 0; jt < NT; ++jt) {
      const f32x4 kf = *(const f32x4*)(sK + li * LD + 16 * jt + 4 * grp);
      const f32x4 qf = *(const f32x4*)(sQ + li * LD + 16 * jt + 4 * grp);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x0 = bits_f32(s0[jt][e]), x1 = bits_f32(s1[jt][e]);
        pk[e % NA] = mfma4(kf[e], x0, pk[e % NA]);
        pq[e % NA] = mfma4(qf[e], x0, pq[e % NA]);
        ek[e % NA] = mfma4(kf[e], x1, ek[e % NA]);
        zs[e % NA] = fmaf(x0, x1, zs[e % NA]);
      }
    }
    auto sum = [&](auto at) {  // at(n), n < NA, as a tree
      if constexpr (NA == 4) return (at(0) + at(1)) + (at(2) + at(3));
      else if constexpr (NA == 2) return at(0) + at(1);
      else return at(0);
    };
    float z = sum([&](int n) { return zs[n]; });
    z += __shfl_xor(z, 16);
    z += __shfl_xor(z, 32);
    if (grp == 0) sZ[16 * it + li] = z;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int at = (4 * grp + r) * LD + 16 * it + li;
      sP[at] = sum([&](int n) { return pk[n][r]; });
      sO[at] = sum([&](int n) { return pq[n][r]; });
      sE[at] = sum([&](int n) { return ek[n][r]; });
    }
  }
  if (w >= 2) {  // G(t, s) = k_t . k_s, H(t, s) = q_t . k_s
    constexpr int NG = sizeof(TT) == 4 ? (DP == 32 ? 4 : 8) : 1;  // chains, as in gram
    f32x4 acc[NG] = {};
    const float* A = w == 2 ? sK : sQ;
#pragma unroll
    for (int jt = 0; jt < NT; ++jt) {
      const int at = li * LD + 16 * jt + 4 * grp;
      const f32x4 av = *(const f32x4*)(A + at), bv = *(const f32x4*)(sK + at);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[(4 * jt + e) % NG] = mfma4(av[e], bv[e], acc[(4 * jt + e) % NG]);
    }
#pragma unroll
    for (int n = NG / 2; n > 0; n /= 2)
#pragma unroll
      for (int m = 0; m < n; ++m) acc[m] += acc[m + n];
#pragma unroll
    for (int r = 0; r < 4; ++r) (w == 2 ? sG : sH)[(4 * grp + r) * CH + li] = acc[0][r];
  }
  __syncthreads();

  if (rows && first) {
    float dec = 1.0f;
#pragma unroll
    for (int t = 0; t < CH; ++t) {
      dec *= a[t];
      if (mine) sD[t * LD + i] = go[t] * dec;
      if (mine) sW[t * LD + i] = -wv[t] * dec;
    }
    dec = 1.0f;
#pragma unroll
    for (int t = CH - 1; t >= 0; --t) {
      if (mine) sU[t * LD + i] = u[t] * dec;
      dec *= a[t];
    }
    // the decay's gradient
    int io = i;
    asm volatile("" : "+v"(io));  // (the offsets of its stores formed here, not kept since the loads)
    const rsrc_t rDA = p.alpha_per_row ? row_rsrc(p.dalpha) : head_rsrc(p.dalpha);
    float da[CH];
    {
      float e[CH], z = sZ[ic];
#pragma unroll
      for (int s = 0; s < CH; ++s) e[s] = sE[s * LD + ic];
#pragma unroll
      for (int t = CH - 1; t >= 0; --t) {
        z = fmaf(go[t], sO[t * LD + ic], fmaf(-wv[t], sP[t * LD + ic], z));
        float v = z;
#pragma unroll
        for (int s = 0; s < t; ++s) {
          e[s] = fmaf(go[t], sH[t * CH + s], fmaf(-wv[t], sG[t * CH + s], e[s]));
          v = fmaf(a[s], v, u[s] * e[s]);
          e[s] *= a[t];
        }
        z *= a[t];
        da[t] = v;
        if (p.alpha_per_row) bstore<TT>(rDA, el_off(t, io), v * a[t]);  // log space
      }
    }
    if (!p.alpha_per_row) put_sums(da, NP + CH);
  } else if (rows) {
    // sums over the rows: M(t, s) at t (t + 1) / 2 + t - s, N(t, s) at 136 + s (s - 1) / 2 + s - 1 - t, 64 at a time
    float buf[64];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int t = 0; t < CH; ++t) {
        float x = go[t];
#pragma unroll
        for (int s = t; s >= 0; --s) {
          const int n = t * (t + 1) / 2 + t - s;
          if (n / 64 == q) buf[n % 64] = x * u[s];
          x *= a[s];
        }
      }
#pragma unroll
      for (int s = 1; s < CH; ++s) {
        float y = -wv[s] * a[s];
#pragma unroll
        for (int t = s - 1; t >= 0; --t) {
          const int n = 136 + s * (s - 1) / 2 + s - 1 - t;
          if (n / 64 == q) buf[n % 64] = y * u[t];
          y *= a[t];
        }
      }
      red[w & 1][64 * q + l] = scatter64(buf, l);
    }
  }
  __syncthreads();

  const int cg = w % NC, ks = w / NC, j0 = 16 * VC * cg + VC * li;  // this lane's columns j0 .. j0 + VC - 1
  u32x4 s0[KX][4], s1[KX][4];
  if (ks < KS) {
#pragma unroll
    for (int x = 0; x < KX; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int at = ((4 * grp + e) * DP + j0) * 4, blk = 16 * (KX * ks + x) * DP * 4;
        if constexpr (VC == 4) {
          s0[x][e] = __builtin_amdgcn_raw_buffer_load_b128(rS0, at, blk, 0);
          s1[x][e] = __builtin_amdgcn_raw_buffer_load_b128(rS1, at, blk, 0);
        } else {
#pragma unroll
          for (int n = 0; n < VC; ++n) {
            s0[x][e][n] = __builtin_amdgcn_raw_buffer_load_b32(rS0, at + 4 * n, blk, 0);
            s1[x][e][n] = __builtin_amdgcn_raw_buffer_load_b32(rS1, at + 4 * n, blk, 0);
          }
        }
      }
  }
  {
    float v = red[0][tid];
    if (DP == 128) v += red[DP == 128 ? 1 : 0][tid];
    int n = tid < 136 ? tid : tid - 136, t = 0;
    if (tid < 136) {
      while ((t + 1) * (t + 2) / 2 <= n) ++t;
      sM[t * LM + t - (n - t * (t + 1) / 2)] = v;
    } else {
      t = 1;
      while (t * (t + 1) / 2 <= n) ++t;
      const int s = t - 1 - (n - t * (t - 1) / 2);
      sN[t * LM + s] = v;
      sN[s * LM + t] = v;
    }
    if (tid < 2 * CH && (tid < CH ? p.beta_per_head : !p.alpha_per_row)) {
      float sum = red[0][NP + tid];
      if (DP == 128) sum += red[DP == 128 ? 1 : 0][NP + tid];
      if (tid < CH) bstore<TT>(head_rsrc(p.dbeta), head_off(tid), sum);
      else bstore<TT>(head_rsrc(p.dalpha), head_off(tid - CH), sum);
    }
  }

  // dq, dk: wave (cg, ks) forms the products of its rows; part 0 then finishes dq, part 1 dk
  f32x4 dq[VC], dk[VC], dk1[VC];  // (float32: the terms of dS1 by themselves)
#pragma unroll
  for (int n = 0; n < VC; ++n) dq[n] = dk[n] = dk1[n] = zero;
  if (ks < KS) {
#pragma unroll
    for (int x = 0; x < KX; ++x) {
      const int at = li * LD + 16 * (KX * ks + x) + 4 * grp;
      const f32x4 dv = *(const f32x4*)(sD + at), wn = *(const f32x4*)(sW + at), uv = *(const f32x4*)(sU + at);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int n = 0; n < VC; ++n) {
          dq[n] = mfma4(dv[e], bits_f32(s0[x][e][n]), dq[n]);
          dk[n] = mfma4(wn[e], bits_f32(s0[x][e][n]), dk[n]);
          f32x4& to = sizeof(TT) == 4 ? dk1[n] : dk[n];
          to = mfma4(uv[e], bits_f32(s1[x][e][n]), to);
        }
    }
    if constexpr (sizeof(TT) == 4) {
#pragma unroll
      for (int n = 0; n < VC; ++n) dk[n] += dk1[n];
    }
#pragma unroll
    for (int n = 0; n < VC; ++n) {
      if (ks != 0) sh.part[0][ks - 1][cg][n][l] = dq[n];
      if (ks != 1) sh.part[1][ks == 0 ? 0 : ks - 1][cg][n][l] = dk[n];
    }
  }
  __syncthreads();
  if (ks > 1) return;
  const bool isq = ks == 0;
  f32x4 acc[VC];
#pragma unroll
  for (int n = 0; n < VC; ++n) {
    acc[n] = isq ? dq[n] : dk[n];
#pragma unroll
    for (int m = 0; m < KS - 1; ++m) acc[n] += sh.part[isq ? 0 : 1][m][cg][n][l];
  }
  if (!(sBad[0] | sBad[1] | sBad[2] | sBad[3])) {
    const f32x4 av = *(const f32x4*)((isq ? sM : sN) + li * LM + 4 * grp);
    // the chunk's own steps; float32: four steps at a time, added as a tree (one chain through all of them would
    // round the largest term again with every other)
    constexpr int NC4 = sizeof(TT) == 4 ? 4 : 1;
#pragma unroll
    for (int n = 0; n < VC; ++n) {
      f32x4 ck[NC4] = {}, cq[NC4] = {};
      if constexpr (NC4 == 1) ck[0] = acc[n];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int s = 4 * grp + e;
        ck[e % NC4] = mfma4(av[e], sK[s * LD + j0 + n], ck[e % NC4]);
        f32x4& to = NC4 == 1 ? ck[0] : cq[e % NC4];
        if (!isq) to = mfma4(sM[s * LM + li], sQ[s * LD + j0 + n], to);
      }
      if constexpr (NC4 == 1)
        acc[n] = ck[0];
      else
        acc[n] += ((ck[0] + ck[1]) + (ck[2] + ck[3])) + ((cq[0] + cq[1]) + (cq[2] + cq[3]));
    }
  } else {  // a step outside a sum must not enter it even with 0
    for (int s = 0; s < CH; ++s)
#pragma unroll
      for (int n = 0; n < VC; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = 4 * grp + r;
          const float ks_ = sK[s * LD + j0 + n];
          if (isq) {
            if (s <= t) acc[n][r] = fmaf(sM[t * LM + s], ks_, acc[n][r]);
          } else {
            if (s >= t) acc[n][r] = fmaf(sM[s * LM + t], sQ[s * LD + j0 + n], acc[n][r]);
            if (s != t) acc[n][r] = fmaf(sN[t * LM + s], ks_, acc[n][r]);
          }
        }
  }
  const rsrc_t rDst = row_rsrc(isq ? p.dq : p.dk);
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int n = 0; n < VC; ++n) bstore<TT>(rDst, el_off(4 * grp + r, j0 + n), acc[n][r]);
}

template <typename TT, int DP>
void launch_bwd(hipStream_t s, const RowArgs& r, float* du, const GradArgs& a, const DecayArgs& da, int bh) {
  const unsigned grid = (unsigned)((long)bh * r.nrb), threads = 64 * (2 + (DP >= 64 ? 2 : 1));
  const uintptr_t at = (uintptr_t)r.q | (uintptr_t)r.k;
  const bool vec = r.d % (16 / (int)sizeof(TT)) == 0 && at % 4 == 0;
  if (r.alpha != nullptr) {
    vec ? dr_row_rev_kernel<TT, DP, true, true><<<grid, threads, 0, s>>>(r, du)
        : dr_row_rev_kernel<TT, DP, true, false><<<grid, threads, 0, s>>>(r, du);
    dr_row_decay_grad_kernel<TT, DP><<<(unsigned)((long)bh * ((r.T + CH - 1) / CH)), 256, 0, s>>>(da);
    return;
  }
  vec ? dr_row_rev_kernel<TT, DP, false, true><<<grid, threads, 0, s>>>(r, du)
      : dr_row_rev_kernel<TT, DP, false, false><<<grid, threads, 0, s>>>(r, du);
  GradArgs g = a;
  g.vec = r.d % 8 == 0 && (((uintptr_t)a.dout | (uintptr_t)a.beta | (uintptr_t)a.dv | (uintptr_t)a.dbeta) % 4 == 0);
  dr_row_grad_kernel<TT, DP><<<(unsigned)((long)bh * ((r.T + CPS - 1) / CPS)), 4 * DP, 0, s>>>(g);
}

template <typename TT>
void by_width(hipStream_t s, const RowArgs& r, float* du, const GradArgs& a, const DecayArgs& da, int bh) {
  if (r.cw == 32)
    launch_bwd<TT, 32>(s, r, du, a, da, bh);
  else if (r.cw == 64)
    launch_bwd<TT, 64>(s, r, du, a, da, bh);
  else
    launch_bwd<TT, 128>(s, r, du, a, da, bh);
}

inline size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }
inline int state_width(int d) { return d <= 32 ? 32 : d <= 64 ? 64 : 128; }
// States kept: with a decay after every chunk, without before every CPS steps but the first.
inline size_t states_bytes(int batch, int heads, int seq, int d, bool decay) {
  const size_t w = state_width(d), n = decay ? (seq + CH - 1) / CH : (seq + CPS - 1) / CPS - 1;
  return align256((size_t)batch * heads * n * w * w * 4);
}
inline size_t rows_bytes(int batch, int heads, int seq, int d) {
  return align256((size_t)batch * seq * heads * d * 4);
}

}  // namespace

// The forward's record for this backward: states, then err.
size_t dr_row_context_bytes(int batch, int heads, int seq, int d, bool decay) {
  return states_bytes(batch, heads, seq, d, decay) + rows_bytes(batch, heads, seq, d);
}

int dr_row_record_run(void* stream, const void* q, const void* k, const void* v, const void* beta, const void* alpha,
                      void* out, int batch, int seq, int heads, int d, int dtype, int beta_per_head,
                      int alpha_per_row, void* context) {
  return dr_row_run(stream, q, k, v, beta, alpha, out, batch, seq, heads, d, dtype, beta_per_head, alpha_per_row,
                    (float*)context, (float*)((char*)context + states_bytes(batch, heads, seq, d, alpha != nullptr)),
                    state_width(d));
}

// Workspace: state gradients and du; without the forward's record (saved) one of its own behind them.
size_t dr_row_backward_workspace_bytes(int batch, int heads, int seq, int d, bool decay, bool saved) {
  return (saved ? 1 : 2) * dr_row_context_bytes(batch, heads, seq, d, decay);
}

int dr_row_backward_run(void* stream, const void* q, const void* k, const void* v, const void* beta,
                        const void* alpha, const void* grad_out, void* dq, void* dk, void* dv, void* dbeta,
                        void* dalpha, void* workspace, int batch, int seq, int heads, int d, int dtype,
                        int beta_per_head, int alpha_per_row, const void* context) {
  const bool decay = alpha != nullptr;
  const size_t sb = states_bytes(batch, heads, seq, d, decay), ctx = dr_row_context_bytes(batch, heads, seq, d, decay);
  char* ws = (char*)workspace;
  if (context == nullptr) {
    context = ws + ctx;
    const int rc = dr_row_record_run(stream, q, k, v, beta, alpha, nullptr, batch, seq, heads, d, dtype,
                                     beta_per_head, alpha_per_row, ws + ctx);
    if (rc) return rc;
  }
  RowArgs r{};
  r.q = q, r.k = k, r.v = grad_out, r.beta = beta, r.alpha = alpha, r.ckpt = (float*)ws;
  r.H = heads, r.T = seq, r.d = d, r.cw = state_width(d), r.nrb = r.cw / RW;
  r.beta_per_head = beta_per_head, r.alpha_per_row = alpha_per_row;
  float* du = (float*)(ws + sb);
  GradArgs a{};
  a.q = q, a.k = k, a.dout = grad_out, a.beta = beta, a.dq = dq, a.dk = dk, a.dv = dv, a.dbeta = dbeta;
  a.ckpt = (const float*)context, a.err = (const float*)((const char*)context + sb), a.dckpt = r.ckpt, a.du = du;
  a.H = heads, a.T = seq, a.d = d, a.beta_per_head = beta_per_head;
  DecayArgs da{};
  da.q = q, da.k = k, da.dout = grad_out, da.beta = beta, da.alpha = alpha;
  da.dq = dq, da.dk = dk, da.dv = dv, da.dbeta = dbeta, da.dalpha = dalpha;
  da.ckpt = a.ckpt, da.err = a.err, da.dckpt = a.dckpt, da.du = du;
  da.H = heads, da.T = seq, da.d = d, da.beta_per_head = beta_per_head, da.alpha_per_row = alpha_per_row;
  hipStream_t s = as_stream(stream);
  if (dtype == EDF_BF16)
    by_width<bf16>(s, r, du, a, da, batch * heads);
  else
    by_width<float>(s, r, du, a, da, batch * heads);
  return check_launch("delta rule backward (row scan)");
}

}  // namespace edf
