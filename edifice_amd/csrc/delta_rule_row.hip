// Delta rule with a gate per value row, 16 steps at a time on the matrix cores: the forward of
// DeltaNet and GatedDeltaNet with a beta per row (or float32, or a head_dim that the chunked
// kernels do not take) and of KDA (a decay per row).
//
//   S_g = a_t S;  err = v_t - S_g k_t;  u = beta_t err;  S = S_g + u k_t^T;  o_t = S q_t
// with a_t and beta_t per (step, row) (lib/edifice/recurrent/delta_net.ex:231-273,
// gated_delta_net.ex:300-353, native/cuda/fused_kda_scan.cu:1-24).
//
// A beta (or decay) per row leaves no triangular inverse to share between the rows, but the rows'
// recurrences see k and q only through dot products: with p_t = S k_t and w_t = S q_t for the
// steps still to come, one step is
//   err = v_t - a_t p_t;  u = beta_t err;  p_s <- a_t p_s + u (k_t . k_s),  w_s <- a_t w_s + u (k_t . q_s)
// so a chunk of 16 steps needs the products S k, S q (against the state that the chunk starts from), the
// 16 x 16 Gram tiles K K^T and K Q^T (shared by all rows), a short recurrence per row on these, and
// one rank-16 update of S: three contractions on the matrix cores.  The recurrence goes in blocks of four
// steps: the four p of a row are gathered in every lane, the block's 4 x 4 triangular system is solved
// there, and one 16x16x4 f32 MFMA takes the four u into the p of all later steps.  It is the
// per-step recurrence term by term (no division by a decay, no exponential of a difference).
//
// The chunks are a chain and one wave issues in order, so the scan is bound by the instructions that the
// chain's wave issues per chunk.  Each 16-row block has up to four waves, on four SIMDs, and one barrier per
// chunk; in iteration c
//   chain   solves chunk c and leaves its u in LDS; it holds no state: p of chunk c is the product with
//           the state before chunk c - 1, which came from the state waves, plus the u of chunk c - 1 through
//           the Gram tile between the two chunks;
//   state   (one wave per half of the columns) adds chunk c - 1 to the state and takes its products with
//           k of chunk c + 1 and q of chunk c;
//   gram    forms the Gram tiles of chunk c + 1, the outputs of chunk c - 1, and stages k and q.
// Forward without states, per call, against the per-step kernel it replaces (one lane per 8 state entries,
// 574 cycles a step): 8 x 2048 x 8 x 128 bf16 529 -> 143 us, 4 x 1000 x 8 x 128 KDA 247 -> 94 us,
// 2 x 777 x 8 x 64 f32 gated 129 -> 104 us.  One wave per block doing everything took 246 us for the first,
// a chain wave that also held the state 235 us.
#include "edf_abi.hpp"
#include "edf_common.hpp"
#include "edf_row_scan.hpp"

namespace edf {
namespace {
using namespace rowscan;


template <typename TT, int DP>
struct RowShared {
  static constexpr int LD = tile_ld<TT, DP>();
  static constexpr int SW = DP >= 64 ? 2 : 1;  // state waves
  TT k[4][CH * LD], q[3][CH * LD];              // chunk c in slot c % 4 of k, c % 3 of q
  f32x4 u[2][64];                               // u of the chunk's steps, undecayed
  f32x4 pk[2][SW][64], pq[2][SW][64];           // state products of k (chunk c + 1) and q (chunk c)
  f32x4 g[2][64], gx[2][64];                    // Gram tiles of a chunk, and of the chunk before with it
  float gs[2][32];                              // solve scalars
};

template <typename TT, int DP, bool DECAY, bool VEC>
__global__ __launch_bounds__(64 * (2 + (DP >= 64 ? 2 : 1))) void dr_row_fwd_kernel(const RowArgs p) {
  typedef RowShared<TT, DP> Sh;
  constexpr int LD = Sh::LD, SW = Sh::SW, W = DP / SW;
  // float32 sums the chunk's own terms apart from the state's and takes v last (edf_row_scan.hpp); bf16 values carry
  // their rounding anyway and save the instructions
  constexpr bool F32 = sizeof(TT) == 4;
  __shared__ __attribute__((aligned(16))) Sh sh;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, li = l & 15, grp = l >> 4;
  const RowIO<TT> io(p, li);
  const int nch = (p.T + CH - 1) / CH;

  if (wave == 0) {  // chain
    GateRegs<TT> nv, nb, na;
    nv.at(io.row0, io.step, 0, grp);
    nb.at(io.bbase, io.bstep, 0, grp);
    if (DECAY) na.at(io.abase, io.astep, 0, grp);
    auto load = [&]() {
      nv.load(io.rV, io.step, CH);
      nb.load(io.rB, io.bstep, CH);
      if (DECAY) na.load(io.rA, io.astep, CH);
    };
    load();
    const long rowel = (long)p.T * p.H * p.d;
    const bool keep = p.err != nullptr;
    const rsrc_t rE = make_rsrc(keep ? (const void*)(p.err + io.bh / p.H * rowel) : p.k, keep ? (unsigned)(rowel * 4) : 0u);
    const unsigned estep = (unsigned)p.H * p.d * 4;
    unsigned eoff = io.in ? ((unsigned)(io.bh % p.H) * p.d + io.i) * 4 + (unsigned)grp * estep : OOB_OFF;
    f32x4 U = {0, 0, 0, 0};  // u of the chunk before, decayed to its end
    float dtot = 1.0f;       // decay of the chunk before
    lds_barrier();
    for (int c = 0; c < nch; ++c) {
      const int t0 = c * CH, b = c & 1;
      f32x4 pk = {0, 0, 0, 0};
      if (c > 0) {
        pk = sh.pk[b][0][l];
        if (SW == 2) pk += sh.pk[b][SW - 1][l];
      }
      const f32x4 G = sh.g[b][l], Gx = sh.gx[b][l];
      f32x4 gs[4][2];
#pragma unroll
      for (int r = 0; r < 4; ++r) gs[r][0] = *(const f32x4*)&sh.gs[b][8 * r], gs[r][1] = *(const f32x4*)&sh.gs[b][8 * r + 4];
      float vv[4][4], bb[4][4], aa[4][4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if constexpr (F32)
          gather4(bits_f32(nv.v[r]), vv[r]);
        else
          vv[r][0] = bits_f32(nv.v[r]);  // this lane's step
        gather4(bits_f32(nb.v[r]), bb[r]);
        if (DECAY)
          gather4(decay_of<TT>(na.v[r], t0 + 4 * r + grp < p.T && io.in, p.alpha_per_row), aa[r]);
        else
          aa[r][0] = aa[r][1] = aa[r][2] = aa[r][3] = 1.0f;
      }
      load();  // the next chunk's, under this chunk's work
      pk = tile_dot<F32>(Gx, U, DECAY ? pk * dtot : pk);
      f32x4 raw, in = {0, 0, 0, 0};  // in: the part of p from the chunk's own steps (bf16: in pk)
      dtot = 1.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        auto g = [&](int m, int n) { return gs[r][pair(m, n) >> 2][pair(m, n) & 3]; };
        const BlockDecay D(aa[r], grp);
        float y[4], u[4];
        const float pr = F32 ? pk[r] + in[r] : pk[r];
        if constexpr (F32)
          gather4(DECAY ? D.pre * pr : pr, y);
        else
          gather4(DECAY ? fmaf(D.pre, pr, -vv[r][0]) : pr - vv[r][0], y);
        auto last = [&](float t, int m) { return F32 ? vv[r][m] - t : -t; };
        y[0] = last(y[0], 0);
        u[0] = bb[r][0] * y[0];
        y[1] = last(fmaf(DECAY ? g(0, 1) * D.r10 : g(0, 1), u[0], y[1]), 1);
        u[1] = bb[r][1] * y[1];
        y[2] = last(fmaf(DECAY ? g(1, 2) * D.r21 : g(1, 2), u[1],
                         fmaf(DECAY ? g(0, 2) * D.r20 : g(0, 2), u[0], y[2])), 2);
        u[2] = bb[r][2] * y[2];
        y[3] = last(fmaf(DECAY ? g(2, 3) * D.r32 : g(2, 3), u[2],
                         fmaf(DECAY ? g(1, 3) * D.r31 : g(1, 3), u[1],
                              fmaf(DECAY ? g(0, 3) * D.r30 : g(0, 3), u[0], y[3]))), 3);
        u[3] = bb[r][3] * y[3];
        if (keep) bstore<float>(rE, eoff + 4 * r * estep, pick4(y[0], y[1], y[2], y[3], grp));
        const float uo = pick4(u[0], u[1], u[2], u[3], grp);
        const float ue = DECAY ? uo * D.end : uo;
        f32x4& own = F32 ? in : pk;
        if (r < 3) own = mfma4(G[r], ue, DECAY ? own * D.all : own);
        if (DECAY) {
          if (F32) pk *= D.all;
#pragma unroll
          for (int e = 0; e < r; ++e) U[e] *= D.all;
          dtot *= D.all;
        }
        U[r] = ue;
        raw[r] = uo;
      }
      eoff += CH * estep;
      sh.u[b][l] = raw;
      lds_barrier();
    }
  } else if (wave <= SW) {  // state, W columns
    const int half = wave - 1;
    f32x4 S[W / 16];
#pragma unroll
    for (int jt = 0; jt < W / 16; ++jt) S[jt] = f32x4{0, 0, 0, 0};
    GateRegs<TT> na;
    if (DECAY) {
      na.at(io.abase, io.astep, 0, grp);
      na.load(io.rA, io.astep, CH);
    }
    lds_barrier();
    for (int c = 0; c <= nch; ++c) {
      RowFrag<TT, W> kf, qf;
      kf.template load<LD>(sh.k[(c + 1) & 3] + W * half, li, grp);
      qf.template load<LD>(sh.q[c % 3] + W * half, li, grp);
      if (c > 0) {
        ColFrag<TT, W> kc;
        kc.template load<LD>(sh.k[(c - 1) & 3] + W * half, li, grp);
        f32x4 U = sh.u[(c - 1) & 1][l];
        if (DECAY) {
          float dtot = 1.0f;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float aa[4];
            gather4(decay_of<TT>(na.v[r], (c - 1) * CH + 4 * r + grp < p.T && io.in, p.alpha_per_row), aa);
            const BlockDecay D(aa, grp);
#pragma unroll
            for (int e = 0; e < r; ++e) U[e] *= D.all;
            dtot *= D.all;
            U[r] *= D.end;
          }
          na.load(io.rA, io.astep, CH);
#pragma unroll
          for (int jt = 0; jt < W / 16; ++jt) S[jt] *= dtot;
        }
        state_add<W>(S, kc, U);
        if (p.ckpt != nullptr && io.i < p.cw && (DECAY || (c % (CPS / CH) == 0 && c < nch))) {
          const long slot = DECAY ? io.bh * nch + c - 1 : io.bh * ((p.T + CPS - 1) / CPS - 1) + c / (CPS / CH) - 1;
          float* cp = p.ckpt + (slot * p.cw + io.i) * p.cw + W * half + 4 * grp;
#pragma unroll
          for (int jt = 0; jt < W / 16; ++jt)
            if (W * half + 16 * jt < p.cw) *(f32x4*)(cp + 16 * jt) = S[jt];
        }
      }
      if (c < nch) {
        f32x4 pk, pq;
        state_dots<W>(kf, qf, S, pk, pq);
        sh.pk[(c + 1) & 1][half][l] = pk;
        sh.pq[c & 1][half][l] = pq;
        lds_barrier();
      }
    }
  } else {  // gram, outputs, staging
    TileRegs<TT, DP, VEC> nk, nq;
    GateRegs<TT> na;
    nk.at(io.base, io.step, 0, p.d, l);
    nq.at(io.base, io.step, 0, p.d, l);
    if (DECAY) na.at(io.abase, io.astep, 0, grp);
    RowFrag<TT, DP> kp = {};  // k rows of the chunk before the one whose Gram tiles are formed
    f32x4 Hq, Hn, Hp;    // k . q tiles of chunks c, c + 1 and c - 1
    const int t = sigma(li);
    // the solve scalar this lane holds: register r of lane (4 n + r, m) is k_m . k_n of block r
    const int gm = grp, gn = li >> 2, gr = li & 3;
    auto grams = [&](int c) {  // tiles of chunk c, which is staged
      RowFrag<TT, DP> kf, qf;
      kf.template load<LD>(sh.k[c & 3], li, grp);
      qf.template load<LD>(sh.q[c % 3], li, grp);
      const f32x4 G = gram<DECAY, DP>(kf, kf);
      sh.g[c & 1][l] = G;
      const float gv = gr == 0 ? G[0] : gr == 1 ? G[1] : gr == 2 ? G[2] : G[3];
      if (gm < gn) sh.gs[c & 1][8 * gr + pair(gm, gn)] = gv;
      sh.gx[c & 1][l] = gram<DECAY, DP>(kp, kf);
      kp = kf;
      return gram<DECAY, DP>(kf, qf);
    };
    auto stage = [&](int c) {  // chunk c into its slot, chunk c + 1 on its way
      nk.store(sh.k[c & 3], l);
      nq.store(sh.q[c % 3], l);
      nk.load(io.rK, io.step, CH);
      nq.load(io.rQ, io.step, CH);
    };
    nk.load(io.rK, io.step, CH);
    nq.load(io.rQ, io.step, CH);
    stage(0);
    stage(1);
    if (DECAY) na.load(io.rA, io.astep, CH);
    Hq = Hp = grams(0);
    unsigned ooff = io.row0 + (unsigned)grp * io.step;
    lds_barrier();
    for (int c = 0; c <= nch; ++c) {
      if (c < nch) {
        stage(c + 2);
        Hn = grams(c + 1);
      }
      if (c > 0) {  // outputs of chunk c - 1
        f32x4 U = sh.u[(c - 1) & 1][l];
        f32x4 pq = sh.pq[(c - 1) & 1][0][l];
        if (SW == 2) pq += sh.pq[(c - 1) & 1][SW - 1][l];
        const bool finite = fabsf(U[0]) < INFINITY && fabsf(U[1]) < INFINITY && fabsf(U[2]) < INFINITY &&
                            fabsf(U[3]) < INFINITY;
        if (!DECAY && !__any(!finite)) {
          // o = S q of the state before, plus u_s (k_s . q_t) over the steps s <= t of the chunk (a later
          // step's u enters with 0, so all must be finite)
          f32x4 h;
#pragma unroll
          for (int r = 0; r < 4; ++r) h[r] = 4 * r + grp <= t ? Hp[r] : 0.0f;
          pq = tile_dot<F32>(h, U, pq);
#pragma unroll
          for (int r = 0; r < 4; ++r) bstore<TT>(io.rO, ooff + 4 * r * io.step, pq[r]);
        } else {
          f32x4 in = {0, 0, 0, 0};  // the part of o from the chunk's blocks before
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float aa[4] = {1.0f, 1.0f, 1.0f, 1.0f}, u[4];
            if (DECAY)
              gather4(decay_of<TT>(na.v[r], (c - 1) * CH + 4 * r + grp < p.T && io.in, p.alpha_per_row), aa);
            const BlockDecay D(aa, grp);
            gather4(U[r], u);
            float o = F32 ? 0.0f : D.pre * pq[r];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
              // decay from after step m to the lane's step; k_m . q of the lane's step
              const float rm = m == 0   ? pick4(1.0f, D.r10, D.r20, D.r30, grp)
                               : m == 1 ? pick4(1.0f, 1.0f, D.r21, D.r31, grp)
                               : m == 2 ? (grp == 3 ? D.r32 : 1.0f)
                                        : 1.0f;
              const float hm = __shfl(Hp[r], 16 * m + 4 * grp + r);
              o = m <= grp ? fmaf(u[m] * rm, hm, o) : o;
            }
            if (F32) o = fmaf(D.pre, pq[r] + in[r], o);
            bstore<TT>(io.rO, ooff + 4 * r * io.step, o);
            f32x4& own = F32 ? in : pq;
            if (r < 3) own = mfma4(Hp[r], U[r] * D.end, own * D.all);
            if (F32) pq *= D.all;
          }
          if (DECAY) na.load(io.rA, io.astep, CH);
        }
        ooff += CH * io.step;
      }
      Hp = Hq;
      Hq = Hn;
      if (c < nch) lds_barrier();
    }
  }
}

template <typename TT, int DP>
void launch_fwd(hipStream_t s, const RowArgs& a, unsigned grid) {
  const uintptr_t at = (uintptr_t)a.q | (uintptr_t)a.k;
  const bool vec = a.d % (16 / (int)sizeof(TT)) == 0 && at % 4 == 0;
  const unsigned threads = 64 * (2 + RowShared<TT, DP>::SW);
  if (a.alpha != nullptr)
    vec ? dr_row_fwd_kernel<TT, DP, true, true><<<grid, threads, 0, s>>>(a)
        : dr_row_fwd_kernel<TT, DP, true, false><<<grid, threads, 0, s>>>(a);
  else
    vec ? dr_row_fwd_kernel<TT, DP, false, true><<<grid, threads, 0, s>>>(a)
        : dr_row_fwd_kernel<TT, DP, false, false><<<grid, threads, 0, s>>>(a);
}

template <typename TT>
void by_width(hipStream_t s, const RowArgs& a, unsigned grid) {
  if (a.d <= 32)
    launch_fwd<TT, 32>(s, a, grid);
  else if (a.d <= 64)
    launch_fwd<TT, 64>(s, a, grid);
  else
    launch_fwd<TT, 128>(s, a, grid);
}

}  // namespace

// Whether the row-wise kernels take a call: a batch row, of float32 too (err), addressed by 31-bit
// byte offsets.
bool dr_row_takes(int batch, int heads, int seq, int d) {
  const long bytes = (long)(seq + 6 * CH) * heads * d * 4;
  return d <= 128 && bytes < (1L << 31) && (long)batch * heads * ((d + RW - 1) / RW) < (1L << 31);
}

// ckpt, err, cw: see RowArgs (null: no backward follows)
int dr_row_run(void* stream, const void* q, const void* k, const void* v, const void* beta, const void* alpha,
               void* out, int batch, int seq, int heads, int d, int dtype, int beta_per_head, int alpha_per_row,
               float* ckpt, float* err, int cw) {
  RowArgs a{};
  a.q = q, a.k = k, a.v = v, a.beta = beta, a.alpha = alpha, a.out = out, a.ckpt = ckpt, a.err = err;
  a.H = heads, a.T = seq, a.d = d, a.cw = cw;
  a.nrb = ((ckpt != nullptr ? cw : d) + RW - 1) / RW;  // with states kept, the padding rows (zero) too
  a.beta_per_head = beta_per_head, a.alpha_per_row = alpha_per_row;
  const unsigned grid = (unsigned)((long)batch * heads * a.nrb);
  hipStream_t s = as_stream(stream);
  if (dtype == EDF_BF16)
    by_width<bf16>(s, a, grid);
  else
    by_width<float>(s, a, grid);
  return check_launch("delta rule (row scan)");
}

}  // namespace edf
