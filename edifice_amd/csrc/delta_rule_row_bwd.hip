// Delta rule without decay (DeltaNet), backward for per-row beta (and float32, or a head_dim that the
// chunked kernels do not take), from what the row-scan forward keeps (err and the state every 64 steps;
// delta_rule_row.hip).  Two kernels:
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
#include "edf_abi.hpp"
#include "edf_common.hpp"
#include "edf_row_scan.hpp"

namespace edf {
int dr_row_run(void* stream, const void* q, const void* k, const void* v, const void* beta, const void* alpha,
               void* out, int batch, int seq, int heads, int d, int dtype, int beta_per_head, int alpha_per_row,
               float* ckpt, float* err, int cw);
namespace {
using namespace rowscan;

template <typename TT, int DP>
struct RevShared {
  static constexpr int LD = tile_ld<TT, DP>();
  static constexpr int SW = DP >= 64 ? 2 : 1;  // state waves
  TT k[4][CH * LD], q[4][CH * LD];              // the j-th chunk from the end in slot j % 4
  f32x4 w[2][64];                               // w of the chunk's steps
  f32x4 pk[2][SW][64];                          // state products of k
  f32x4 x[2][64];                               // do terms of a chunk and of the one after it
  f32x4 g[2][64], gx[2][64];                    // Gram tiles of a chunk, and of the one after with it
  float gs[2][32];                              // solve scalars
};

// p.v is do; du [B, T, H, d], p.ckpt the gradients of the states [BH][ceil(T / CPS) - 1][cw][cw] after
// each CPS steps but the last.
template <typename TT, int DP, bool VEC>
__global__ __launch_bounds__(64 * (2 + (DP >= 64 ? 2 : 1))) void dr_row_rev_kernel(const RowArgs p, float* du) {
  typedef RevShared<TT, DP> Sh;
  constexpr int LD = Sh::LD, SW = Sh::SW, W = DP / SW;
  __shared__ __attribute__((aligned(16))) Sh sh;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, li = l & 15, grp = l >> 4;
  const RowIO<TT> io(p, li);
  const int nch = (p.T + CH - 1) / CH, tl = (nch - 1) * CH;

  if (wave == 0) {  // chain
    GateRegs<TT> nb;
    nb.at(io.bbase, io.bstep, tl, grp);
    nb.load(io.rB, io.bstep, -CH);
    const long rowel = (long)p.T * p.H * p.d;
    const rsrc_t rU = make_rsrc(du + io.bh / p.H * rowel, (unsigned)(rowel * 4));
    const unsigned ustep = (unsigned)p.H * p.d * 4;
    unsigned uoff = (io.in ? ((unsigned)(io.bh % p.H) * p.d + io.i) * 4 : OOB_OFF) + (unsigned)(tl + grp) * ustep;
    f32x4 Wn = {0, 0, 0, 0};  // w of the chunk after, negated
    lds_barrier();
    for (int j = 0; j < nch; ++j) {
      const int b = j & 1;
      f32x4 e = sh.x[b][l];
      if (j > 0) {
        e += sh.pk[b][0][l];
        if (SW == 2) e += sh.pk[b][SW - 1][l];
      }
      const f32x4 G = sh.g[b][l], Gx = sh.gx[b][l];
      f32x4 gs[4][2];
#pragma unroll
      for (int r = 0; r < 4; ++r) gs[r][0] = *(const f32x4*)&sh.gs[b][8 * r], gs[r][1] = *(const f32x4*)&sh.gs[b][8 * r + 4];
      float bb[4][4];
#pragma unroll
      for (int r = 0; r < 4; ++r) gather4(bits_f32(nb.v[r]), bb[r]);
      nb.load(io.rB, io.bstep, -CH);
#pragma unroll
      for (int r = 0; r < 4; ++r) e = mfma4(Gx[r], Wn[r], e);
#pragma unroll
      for (int r = 3; r >= 0; --r) {
        auto g = [&](int m, int n) { return gs[r][pair(m, n) >> 2][pair(m, n) & 3]; };
        float y[4], w[4];
        gather4(e[r], y);
        w[3] = bb[r][3] * y[3];
        y[2] = fmaf(-g(2, 3), w[3], y[2]);
        w[2] = bb[r][2] * y[2];
        y[1] = fmaf(-g(1, 2), w[2], fmaf(-g(1, 3), w[3], y[1]));
        w[1] = bb[r][1] * y[1];
        y[0] = fmaf(-g(0, 1), w[1], fmaf(-g(0, 2), w[2], fmaf(-g(0, 3), w[3], y[0])));
        w[0] = bb[r][0] * y[0];
        const float wn = -pick4(w[0], w[1], w[2], w[3], grp);
        if (r > 0) e = mfma4(G[r], wn, e);
        Wn[r] = wn;
        bstore<float>(rU, uoff + 4 * r * ustep, pick4(y[0], y[1], y[2], y[3], grp));
      }
      uoff -= CH * ustep;
      sh.w[b][l] = -Wn;
      lds_barrier();
    }
  } else if (wave <= SW) {  // state gradient, W columns
    const int half = wave - 1;
    f32x4 S[W / 16];
#pragma unroll
    for (int jt = 0; jt < W / 16; ++jt) S[jt] = f32x4{0, 0, 0, 0};
    GateRegs<TT> nd;
    nd.at(io.row0, io.step, tl, grp);
    nd.load(io.rV, io.step, -CH);
    lds_barrier();
    for (int j = 0; j < nch; ++j) {
      const int c = nch - 1 - j;
      RowFrag<TT, W> kf;
      kf.template load<LD>(sh.k[(j + 1) & 3] + W * half, li, grp);
      if (j > 0) {
        ColFrag<TT, W> kc, qc;
        kc.template load<LD>(sh.k[(j - 1) & 3] + W * half, li, grp);
        qc.template load<LD>(sh.q[(j - 1) & 3] + W * half, li, grp);
        state_add2<W>(S, qc, nd.v, kc, sh.w[(j - 1) & 1][l]);
        nd.load(io.rV, io.step, -CH);
        if ((c + 1) % (CPS / CH) == 0 && io.i < p.cw) {
          const long slot = io.bh * ((p.T + CPS - 1) / CPS - 1) + c / (CPS / CH);
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
    GateRegs<TT> nd;
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
      const f32x4 G = gram<DP>(kf, kf), H = gram<DP>(qf, kf), Hx = gram<DP>(qp, kf);
      sh.g[j & 1][l] = G;
      sh.gx[j & 1][l] = gram<DP>(kp, kf);
      const float gv = gr == 0 ? G[0] : gr == 1 ? G[1] : gr == 2 ? G[2] : G[3];
      if (gm < gn) sh.gs[j & 1][8 * gr + pair(gm, gn)] = gv;
      f32x4 x = {0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < 4; ++r) x = mfma4(Hx[r], dp[r], x);
      const bool finite = fabsf(dc[0]) < INFINITY && fabsf(dc[1]) < INFINITY && fabsf(dc[2]) < INFINITY &&
                          fabsf(dc[3]) < INFINITY;
      if (!__any(!finite)) {
        // do_s (q_s . k_t) over the steps s >= t of the chunk (an earlier step's do enters with 0)
#pragma unroll
        for (int r = 0; r < 4; ++r) x = mfma4(4 * r + grp >= t ? H[r] : 0.0f, dc[r], x);
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
};

EDF_DEVICE f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// One workgroup per 64 steps of a head.  Wave (ct, rt) forms the 32 x 32 tile of dq and of dk at steps
// 32 rt .., columns 32 ct ..; the row factors do, u and -w are in LDS as float32, and so are the
// 64 x 64 tiles M = do u^T (s <= t) and N = -(u w^T, its strict upper part, mirrored).
template <typename TT, int DP>
__global__ __launch_bounds__(4 * DP) void dr_row_grad_kernel(const GradArgs p) {
  constexpr int LD = DP + 4, LM = CPS + 4, CT = DP / 32, NTH = 4 * DP, PER = DP / 4;
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

  // this lane's k and q values of the 64 steps (column j, steps 8 kk + 4 g + e), used last
  typename Bits<TT>::type kr[CPS / 2], qr[CPS / 2];
  const unsigned hd = (unsigned)(p.H * d);
#pragma unroll
  for (int i = 0; i < CPS / 2; ++i) {
    const unsigned t = t0 + 8 * (i >> 2) + 4 * g + (i & 3);
    const unsigned off = j < d ? (t * hd + h * d + j) * (unsigned)sizeof(TT) : OOB_OFF;
    kr[i] = bload<TT>(rK, off);
    qr[i] = bload<TT>(rQ, off);
  }

  // row factors, dv and dbeta
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
  __syncthreads();

  // the Gram tiles over the rows: M (0,0) (1,0) (1,1), N (0,0) (0,1) (1,1)
  for (int job = w; job < 6; job += 2 * CT) {
    const bool isM = job < 3;
    const int jj = isM ? job : job - 3;
    const int tr = isM ? (jj > 0) : (jj > 1), tc = isM ? (jj > 1) : (jj > 0);
    const float* A = (isM ? sD : sU) + (32 * tr + li) * LD + 4 * g;
    const float* B = (isM ? sU : sW) + (32 * tc + li) * LD + 4 * g;
    f32x16 acc = zero16();
#pragma unroll 4
    for (int kk = 0; kk < DP / 8; ++kk) {
      const f32x4 av = *(const f32x4*)(A + 8 * kk), bv = *(const f32x4*)(B + 8 * kk);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = mfma_f32(av[e], bv[e], acc);
    }
    const int col = 32 * tc + li;
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const int row = 32 * tr + d_row(x, g);
      if (isM) {
        sM[row * LM + col] = col <= row ? acc[x] : 0.0f;
      } else if (row <= col) {
        const float v = row < col ? acc[x] : 0.0f;
        sN[row * LM + col] = v;
        sN[col * LM + row] = v;
      }
    }
  }

  f32x16 dq = zero16(), dk = zero16();
  const float* aD = sD + (32 * rt + li) * LD + 4 * g;
  const float* aU = sU + (32 * rt + li) * LD + 4 * g;
  const float* aW = sW + (32 * rt + li) * LD + 4 * g;
  if (C > 0) {
    const float* S0 = p.ckpt + ((bh * (n64 - 1) + C - 1) * DP + 4 * g) * DP + j;
#pragma unroll 4
    for (int kk = 0; kk < DP / 8; ++kk) {
      const f32x4 dv = *(const f32x4*)(aD + 8 * kk), wv = *(const f32x4*)(aW + 8 * kk);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float s = S0[(8 * kk + e) * DP];
        dq = mfma_f32(dv[e], s, dq);
        dk = mfma_f32(wv[e], s, dk);
      }
    }
  }
  if (C < n64 - 1) {
    const float* S1 = p.dckpt + ((bh * (n64 - 1) + C) * DP + 4 * g) * DP + j;
#pragma unroll 4
    for (int kk = 0; kk < DP / 8; ++kk) {
      const f32x4 uv = *(const f32x4*)(aU + 8 * kk);
#pragma unroll
      for (int e = 0; e < 4; ++e) dk = mfma_f32(uv[e], S1[(8 * kk + e) * DP], dk);
    }
  }
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
      for (int e = 0; e < 4; ++e) dk = mfma_f32(nv[e], bits_f32(kr[4 * kk + e]), dk);
      if (useM) {
        const f32x4 mv = *(const f32x4*)(aM + 8 * kk);
#pragma unroll
        for (int e = 0; e < 4; ++e) dq = mfma_f32(mv[e], bits_f32(kr[4 * kk + e]), dq);
      }
      if (useT) {
#pragma unroll
        for (int e = 0; e < 4; ++e) dk = mfma_f32(aT[(8 * kk + e) * LM], bits_f32(qr[4 * kk + e]), dk);
      }
    }
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
  }
#pragma unroll
  for (int x = 0; x < 16; ++x) {
    const unsigned t = t0 + 32 * rt + d_row(x, g);
    const unsigned off = j < d ? (t * hd + h * d + j) * (unsigned)sizeof(TT) : OOB_OFF;
    bstore<TT>(rDQ, off, dq[x]);
    bstore<TT>(rDK, off, dk[x]);
  }
}

template <typename TT, int DP>
void launch_bwd(hipStream_t s, const RowArgs& r, float* du, const GradArgs& a, int bh) {
  const unsigned grid = (unsigned)((long)bh * r.nrb), threads = 64 * (2 + RevShared<TT, DP>::SW);
  const uintptr_t at = (uintptr_t)r.q | (uintptr_t)r.k;
  if (r.d % (16 / (int)sizeof(TT)) == 0 && at % 4 == 0)
    dr_row_rev_kernel<TT, DP, true><<<grid, threads, 0, s>>>(r, du);
  else
    dr_row_rev_kernel<TT, DP, false><<<grid, threads, 0, s>>>(r, du);
  dr_row_grad_kernel<TT, DP><<<(unsigned)((long)bh * ((r.T + CPS - 1) / CPS)), 4 * DP, 0, s>>>(a);
}

template <typename TT>
void by_width(hipStream_t s, const RowArgs& r, float* du, const GradArgs& a, int bh) {
  if (r.cw == 32)
    launch_bwd<TT, 32>(s, r, du, a, bh);
  else if (r.cw == 64)
    launch_bwd<TT, 64>(s, r, du, a, bh);
  else
    launch_bwd<TT, 128>(s, r, du, a, bh);
}

inline size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }
inline int state_width(int d) { return d <= 32 ? 32 : d <= 64 ? 64 : 128; }
inline size_t states_bytes(int batch, int heads, int seq, int d) {
  const size_t w = state_width(d);
  return align256((size_t)batch * heads * ((seq + CPS - 1) / CPS - 1) * w * w * 4);
}
inline size_t rows_bytes(int batch, int heads, int seq, int d) {
  return align256((size_t)batch * seq * heads * d * 4);
}

}  // namespace

// The forward's record for this backward: states, then err.
size_t dr_row_context_bytes(int batch, int heads, int seq, int d) {
  return states_bytes(batch, heads, seq, d) + rows_bytes(batch, heads, seq, d);
}

int dr_row_record_run(void* stream, const void* q, const void* k, const void* v, const void* beta, void* out,
                      int batch, int seq, int heads, int d, int dtype, int beta_per_head, void* context) {
  return dr_row_run(stream, q, k, v, beta, nullptr, out, batch, seq, heads, d, dtype, beta_per_head, 0,
                    (float*)context, (float*)((char*)context + states_bytes(batch, heads, seq, d)), state_width(d));
}

// Workspace: state gradients, du, and a record of its own for a caller without the forward's.
size_t dr_row_backward_workspace_bytes(int batch, int heads, int seq, int d) {
  return 2 * dr_row_context_bytes(batch, heads, seq, d);
}

int dr_row_backward_run(void* stream, const void* q, const void* k, const void* v, const void* beta,
                        const void* grad_out, void* dq, void* dk, void* dv, void* dbeta, void* workspace, int batch,
                        int seq, int heads, int d, int dtype, int beta_per_head, const void* context) {
  const size_t sb = states_bytes(batch, heads, seq, d), ctx = dr_row_context_bytes(batch, heads, seq, d);
  char* ws = (char*)workspace;
  if (context == nullptr) {
    context = ws + ctx;
    const int rc = dr_row_record_run(stream, q, k, v, beta, nullptr, batch, seq, heads, d, dtype, beta_per_head,
                                     ws + ctx);
    if (rc) return rc;
  }
  RowArgs r{};
  r.q = q, r.k = k, r.v = grad_out, r.beta = beta, r.ckpt = (float*)ws;
  r.H = heads, r.T = seq, r.d = d, r.cw = state_width(d), r.nrb = r.cw / RW, r.beta_per_head = beta_per_head;
  float* du = (float*)(ws + sb);
  GradArgs a{};
  a.q = q, a.k = k, a.dout = grad_out, a.beta = beta, a.dq = dq, a.dk = dk, a.dv = dv, a.dbeta = dbeta;
  a.ckpt = (const float*)context, a.err = (const float*)((const char*)context + sb), a.dckpt = r.ckpt, a.du = du;
  a.H = heads, a.T = seq, a.d = d, a.beta_per_head = beta_per_head;
  hipStream_t s = as_stream(stream);
  if (dtype == EDF_BF16)
    by_width<bf16>(s, r, du, a, batch * heads);
  else
    by_width<float>(s, r, du, a, batch * heads);
  return check_launch("delta rule backward (row scan)");
}

}  // namespace edf
