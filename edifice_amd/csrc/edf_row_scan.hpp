// Building blocks of the row-wise delta-rule scans (delta_rule_row.hip): one wave holds 16 rows of
// a head's state over all its columns and takes 16 steps at a time on the matrix cores.
//
// Layout.  Lane l of the wave is (li = l % 16, grp = l / 16).  The state S of the wave's rows is held
// transposed in 16 x 16 accumulator tiles: register r of tile jt is S[row li][column 16 jt + 4 grp + r].
// Quantities per (step, row) of the 16-step chunk are accumulator tiles too, with the steps in the
// order that makes register r of group grp step 4 r + grp: a register then is one block of four
// consecutive steps, spread over the groups as the B operand of v_mfma_f32_16x16x4_f32 wants it, and
// four registers are the B operand of the 16-deep bf16 product.  Row operands of the chunk's k and q
// read row sigma(li) of the staged tile for the same reason.
//
// bf16 inputs use bf16 products: k and q are exact, and the float32 factor (state, update) is split
// into three bf16 parts that add up to it exactly (8 + 8 + 8 mantissa bits, by truncation), so a
// product carries float32 accuracy at three bf16 products.  float32 inputs use the f32 MFMA.
#pragma once

#include "edf_common.hpp"
#include "edf_mfma.hpp"

namespace edf {
namespace rowscan {

typedef __attribute__((ext_vector_type(4))) float f32x4;
constexpr int CH = 16;  // steps per chunk
constexpr int RW = 16;  // state rows per wave
constexpr int CPS = 64; // steps between the states kept for a backward without decay

EDF_DEVICE int sigma(int x) { return 4 * (x & 3) + (x >> 2); }

EDF_DEVICE f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
EDF_DEVICE f32x4 mfma32k(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// x = hi + mid + lo, each a bf16, by truncation (exact for finite x)
EDF_DEVICE unsigned hi_bits(float x) { return __builtin_bit_cast(unsigned, x) & 0xffff0000u; }
EDF_DEVICE float bits_to_f32(unsigned v) { return __builtin_bit_cast(float, v); }
EDF_DEVICE unsigned pack_hi(float lo, float hi) {  // the upper halves of two floats, as two bf16
  return __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, hi), __builtin_bit_cast(unsigned, lo), 0x07060302u);
}
struct Split4 {
  bf16x4 part[3];
};
EDF_DEVICE Split4 split4(f32x4 x) {
  typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
  Split4 s;
#pragma unroll
  for (int n = 0; n < 3; ++n) {
    u32x2 w = {pack_hi(x[0], x[1]), pack_hi(x[2], x[3])};
    s.part[n] = __builtin_bit_cast(bf16x4, w);
    if (n < 2) {
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] -= bits_to_f32(hi_bits(x[e]));
    }
  }
  return s;
}

// ---- a staged 16-step tile of k or q and its operands ------------------------------------------
template <typename TT, int DP>
constexpr int tile_ld() {
  return DP + (sizeof(TT) == 2 ? 8 : 4);
}

// Row fragments over W columns (tile: stride LD, from the first of them): for bf16, columns
// 32 kk + 4 grp .. + 3 and 32 kk + 16 + 4 grp .. + 3 of row sigma(li); for float, columns 16 jt + 4 grp .. + 3.
template <typename TT, int W> struct RowFrag;
template <int W> struct RowFrag<bf16, W> {
  bf16x8 f[W / 32];
  template <int LD> EDF_DEVICE void load(const bf16* tile, int li, int grp) {
    const bf16* row = tile + sigma(li) * LD + 4 * grp;
#pragma unroll
    for (int kk = 0; kk < W / 32; ++kk)
      f[kk] = cat4(*(const bf16x4*)(row + 32 * kk), *(const bf16x4*)(row + 32 * kk + 16));
  }
};
template <int W> struct RowFrag<float, W> {
  f32x4 f[W / 16];
  template <int LD> EDF_DEVICE void load(const float* tile, int li, int grp) {
    const float* row = tile + sigma(li) * LD + 4 * grp;
#pragma unroll
    for (int jt = 0; jt < W / 16; ++jt) f[jt] = *(const f32x4*)(row + 16 * jt);
  }
};

// The chunk's Gram tile a b^T: register r of (li, grp) = a[step 4 r + grp] . b[step sigma(li)], the A
// operand of block r in a sum over a's steps.
template <bool DECAY, int DP>
EDF_DEVICE f32x4 gram(const RowFrag<bf16, DP>& a, const RowFrag<bf16, DP>& b) {
  f32x4 c = {0, 0, 0, 0};
#pragma unroll
  for (int kk = 0; kk < DP / 32; ++kk) c = mfma32k(a.f[kk], b.f[kk], c);
  return c;
}
// float32 with a decay: the tile's rounding is most of a call's error (the steps next to each other carry the
// result, so it is not averaged over a long state), so it is summed in eight chains (32 columns: four), added as a
// tree; without a decay one chain is enough.  Error against float64 at 2 x 1500 x 4 x 64, decay per head: out 1.6e-7 with one chain, 0.9e-7
// with eight (the per-step kernel 0.8e-7); the gram wave's additions cost 9% of a call.
template <bool DECAY, int DP>
EDF_DEVICE f32x4 gram(const RowFrag<float, DP>& a, const RowFrag<float, DP>& b) {
  constexpr int N = DECAY ? (DP == 32 ? 4 : 8) : 1;
  f32x4 c[N] = {};
#pragma unroll
  for (int jt = 0; jt < DP / 16; ++jt)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int n = (4 * jt + e) % N;
      c[n] = mfma4(a.f[jt][e], b.f[jt][e], c[n]);
    }
#pragma unroll
  for (int n = N / 2; n > 0; n /= 2)
#pragma unroll
    for (int i = 0; i < n; ++i) c[i] += c[i + n];
  return c[0];
}

// pa, pb: the [step][row] tiles of a[step] . S[row] and b[step] . S[row] over W columns (one split of
// S serves both).  The parts of S have accumulators of their own: more chains of products, and the
// small terms are added up before they meet the large ones.
template <int W>
EDF_DEVICE void state_dots(const RowFrag<bf16, W>& a, const RowFrag<bf16, W>& b, const f32x4 (&S)[W / 16], f32x4& pa,
                           f32x4& pb) {
  f32x4 ca[3] = {}, cb[3] = {};
#pragma unroll
  for (int kk = 0; kk < W / 32; ++kk) {
    const Split4 s0 = split4(S[2 * kk]), s1 = split4(S[2 * kk + 1]);
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      const bf16x8 s = cat4(s0.part[n], s1.part[n]);
      ca[n] = mfma32k(a.f[kk], s, ca[n]);
      cb[n] = mfma32k(b.f[kk], s, cb[n]);
    }
  }
  pa = (ca[2] + ca[1]) + ca[0];
  pb = (cb[2] + cb[1]) + cb[0];
}
template <int W>
EDF_DEVICE void state_dots(const RowFrag<float, W>& a, const RowFrag<float, W>& b, const f32x4 (&S)[W / 16], f32x4& pa,
                           f32x4& pb) {
  f32x4 ca[4] = {}, cb[4] = {};
#pragma unroll
  for (int jt = 0; jt < W / 16; ++jt)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      ca[e] = mfma4(a.f[jt][e], S[jt][e], ca[e]);
      cb[e] = mfma4(b.f[jt][e], S[jt][e], cb[e]);
    }
  pa = (ca[0] + ca[1]) + (ca[2] + ca[3]);
  pb = (cb[0] + cb[1]) + (cb[2] + cb[3]);
}

template <int W>
EDF_DEVICE f32x4 state_dot(const RowFrag<bf16, W>& a, const f32x4 (&S)[W / 16]) {
  f32x4 c[3] = {};
#pragma unroll
  for (int kk = 0; kk < W / 32; ++kk) {
    const Split4 s0 = split4(S[2 * kk]), s1 = split4(S[2 * kk + 1]);
#pragma unroll
    for (int n = 0; n < 3; ++n) c[n] = mfma32k(a.f[kk], cat4(s0.part[n], s1.part[n]), c[n]);
  }
  return (c[2] + c[1]) + c[0];
}
template <int W>
EDF_DEVICE f32x4 state_dot(const RowFrag<float, W>& a, const f32x4 (&S)[W / 16]) {
  f32x4 c[4] = {};
#pragma unroll
  for (int jt = 0; jt < W / 16; ++jt)
#pragma unroll
    for (int e = 0; e < 4; ++e) c[e] = mfma4(a.f[jt][e], S[jt][e], c[e]);
  return (c[0] + c[1]) + (c[2] + c[3]);
}

// The A operands of S += u^T tile over W columns: for bf16 element r of f[jt] is step 4 r + grp, column
// 16 jt + li; for float f[jt][r].
template <typename TT, int W> struct ColFrag;
template <int W> struct ColFrag<bf16, W> {
  bf16x4 f[W / 16];
  template <int LD> EDF_DEVICE void load(const bf16* tile, int li, int grp) {
    const bf16* at = tile + (4 * (li >> 2) + grp) * LD + 4 * (li & 3);
#pragma unroll
    for (int jt = 0; jt < W / 16; ++jt) f[jt] = lds_read_tr16(at + 16 * jt);
  }
};
template <int W> struct ColFrag<float, W> {
  f32x4 f[W / 16];
  template <int LD> EDF_DEVICE void load(const float* tile, int li, int grp) {
    const float* at = tile + grp * LD + li;
#pragma unroll
    for (int jt = 0; jt < W / 16; ++jt)
#pragma unroll
      for (int r = 0; r < 4; ++r) f[jt][r] = at[4 * r * LD + 16 * jt];
  }
};

// S[row][column] += sum over the chunk's steps of u[step][row] tile[step][column].  Both products of
// a tile are 32 deep (the second half of the small one zero).  A first form with a 16-deep product for the small
// part gave states 1e-6 off this one, for a cause that was not found: alone, a 16-deep product with a 32-deep one
// right behind it on the same accumulator gives bit for bit what it gives with waits between (both register forms of
// the accumulators), and differs from two 32-deep ones by an ulp in an element of eight.  So one shape is kept.
template <int W>
EDF_DEVICE void state_add(f32x4 (&S)[W / 16], const ColFrag<bf16, W>& k, f32x4 u) {
  const Split4 s = split4(u);
  const bf16x8 hm = cat4(s.part[0], s.part[1]), lo = cat4(s.part[2], bf16x4{});
#pragma unroll
  for (int jt = 0; jt < W / 16; ++jt) S[jt] = mfma32k(cat4(k.f[jt], k.f[jt]), lo, S[jt]);
#pragma unroll
  for (int jt = 0; jt < W / 16; ++jt) S[jt] = mfma32k(cat4(k.f[jt], k.f[jt]), hm, S[jt]);
}
template <int W>
EDF_DEVICE void state_add(f32x4 (&S)[W / 16], const ColFrag<float, W>& k, f32x4 u) {
  f32x4 c[W / 16] = {};  // the chunk's steps summed by themselves: one rounding of S per chunk
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int jt = 0; jt < W / 16; ++jt) c[jt] = mfma4(k.f[jt][r], u[r], c[jt]);
#pragma unroll
  for (int jt = 0; jt < W / 16; ++jt) S[jt] += c[jt];
}

// S[row][column] += sum over the chunk's steps of x[step][row] q[step][column] - w[step][row] k[step][column],
// x given as stored (bf16: exact, so it shares a product with the first part of w).
template <int W>
EDF_DEVICE void state_add2(f32x4 (&S)[W / 16], const ColFrag<bf16, W>& q, const unsigned short (&x)[4],
                           const ColFrag<bf16, W>& k, f32x4 w) {
  typedef __attribute__((ext_vector_type(4))) unsigned short u16x4;
  const Split4 s = split4(-w);
  const u16x4 xv = {x[0], x[1], x[2], x[3]};
  const bf16x8 xh = cat4(__builtin_bit_cast(bf16x4, xv), s.part[0]), ml = cat4(s.part[1], s.part[2]);
#pragma unroll
  for (int jt = 0; jt < W / 16; ++jt) S[jt] = mfma32k(cat4(k.f[jt], k.f[jt]), ml, S[jt]);
#pragma unroll
  for (int jt = 0; jt < W / 16; ++jt) S[jt] = mfma32k(cat4(q.f[jt], k.f[jt]), xh, S[jt]);
}
template <int W>
EDF_DEVICE void state_add2(f32x4 (&S)[W / 16], const ColFrag<float, W>& q, const unsigned (&x)[4],
                           const ColFrag<float, W>& k, f32x4 w) {
  f32x4 c[W / 16] = {};
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int jt = 0; jt < W / 16; ++jt) {
      c[jt] = mfma4(q.f[jt][r], bits_f32(x[r]), c[jt]);
      c[jt] = mfma4(k.f[jt][r], -w[r], c[jt]);
    }
#pragma unroll
  for (int jt = 0; jt < W / 16; ++jt) S[jt] += c[jt];
}

// acc plus the sum over the 16 steps of tile[step][.] x[step][row].  APART (float32): the four blocks side by side and
// acc last, which rounds at the size of acc once, not 16 times.
template <bool APART>
EDF_DEVICE f32x4 tile_dot(f32x4 tile, f32x4 x, f32x4 acc) {
  if constexpr (APART) {
    f32x4 c[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) c[r] = mfma4(tile[r], x[r], f32x4{0, 0, 0, 0});
    return acc + ((c[0] + c[1]) + (c[2] + c[3]));
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) acc = mfma4(tile[r], x[r], acc);
    return acc;
  }
}

// Value of each of the four groups, in every lane of the same li.  The swaps are not volatile (unlike
// swap16 / swap32): a gather is a function of its input, free to move among the chunk's other work.
EDF_DEVICE void gather4(float x, float (&v)[4]) {
  float a = x, b = x;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));  // a: groups 0 0 2 2, b: groups 1 1 3 3
  float c = a, d = b;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_permlane32_swap_b32 %2, %3" : "+v"(a), "+v"(c), "+v"(b), "+v"(d));
  v[0] = a, v[1] = b, v[2] = c, v[3] = d;
}
EDF_DEVICE float pick4(float v0, float v1, float v2, float v3, int grp) {
  const float lo = (grp & 1) ? v1 : v0, hi = (grp & 1) ? v3 : v2;
  return (grp & 2) ? hi : lo;
}
EDF_DEVICE float lane_value(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// ---- 16 steps of [B, T, H, d] rows: memory -> registers (a chunk ahead) -> LDS -------------------
// A lane's byte offset moves by 16 steps per load, forward or back.  Steps outside 0 .. T - 1 and
// columns past d read as zero (their offsets lie past the batch row, modulo 2^32; the caller keeps
// the steps it runs ahead below 2^31 bytes; a padding column of a step before 0 may read something).
// VEC: d is a multiple of 8 (bf16) or 4 (float) and rows start on 4-byte boundaries, so a row's
// 16-byte pieces lie whole inside or outside it.
template <typename TT, int DP, bool VEC> struct TileRegs;
template <typename TT, int DP> struct TileRegs<TT, DP, true> {
  static constexpr int EPV = 16 / (int)sizeof(TT);   // elements per 16 bytes
  static constexpr int PPR = DP / EPV;               // pieces per row
  static constexpr int N = CH * PPR / 64;            // pieces per lane, 64 / PPR steps apart
  static_assert(N >= 1 && 64 % PPR == 0, "a wave-wide load takes whole rows");
  u32x4 v[N];
  unsigned off;
  EDF_DEVICE void at(unsigned base, unsigned stepb, int t0, int d, int l) {
    const int col = (l % PPR) * EPV;
    off = (col < d ? base + col * (unsigned)sizeof(TT) : OOB_OFF) + (unsigned)(t0 + l / PPR) * stepb;
  }
  EDF_DEVICE void load(rsrc_t r, unsigned stepb, int advance) {
#pragma unroll
    for (int n = 0; n < N; ++n)
      v[n] = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(off + n * (64 / PPR) * stepb), 0, 0));
    off += (unsigned)advance * stepb;
  }
  EDF_DEVICE void store(TT* tile, int l) const {
#pragma unroll
    for (int n = 0; n < N; ++n)
      *(u32x4*)(tile + (l / PPR + n * (64 / PPR)) * tile_ld<TT, DP>() + (l % PPR) * EPV) = v[n];
  }
};
template <typename TT, int DP> struct TileRegs<TT, DP, false> {
  static constexpr int N = CH * DP / 64;
  typename Bits<TT>::type v[N];
  unsigned base, t;
  int d, l;
  EDF_DEVICE void at(unsigned base_, unsigned, int t0, int d_, int l_) { base = base_, t = t0, d = d_, l = l_; }
  EDF_DEVICE void load(rsrc_t r, unsigned stepb, int advance) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int e = l + 64 * n, col = e % DP;
      v[n] = bload<TT>(r, col < d ? base + (t + e / DP) * stepb + col * (unsigned)sizeof(TT) : OOB_OFF);
    }
    t += advance;
  }
  EDF_DEVICE void store(TT* tile, int l_) const {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int e = l_ + 64 * n;
      tile[e / DP * tile_ld<TT, DP>() + e % DP] = __builtin_bit_cast(TT, v[n]);
    }
  }
};

// This lane's four values (steps t0 + 4 r + grp, a byte offset running ahead) of a per-row or
// per-head tensor.
template <typename TT> struct GateRegs {
  typename Bits<TT>::type v[4];
  unsigned off;
  EDF_DEVICE void at(unsigned base, unsigned stepb, int t0, int grp) { off = base + (unsigned)(t0 + grp) * stepb; }
  EDF_DEVICE void load(rsrc_t r, unsigned stepb, int advance) {
#pragma unroll
    for (int n = 0; n < 4; ++n) v[n] = bload<TT>(r, off + 4 * n * stepb);
    off += (unsigned)advance * stepb;
  }
};

// LDS traffic of the workgroup's waves ordered around a barrier; global loads and stores stay in flight.
EDF_DEVICE void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

struct RowArgs {
  const void *q, *k, *v, *beta, *alpha;
  void* out;
  // what a backward (delta_rule_row_bwd.hip) reads, or null: err, [B, T, H, d], and states.  With a
  // decay the state after each chunk, [BH][chunks][cw][cw]; without, the state before every CPS steps
  // but the first, [BH][ceil(T / CPS) - 1][cw][cw].
  float *ckpt, *err;
  int H, T, d, nrb, cw;
  int beta_per_head, alpha_per_row;
};

// What a block's waves address: buffer resources over the batch row and the lane's byte offsets at
// step 0 and per step (lanes past d at an offset that reads zero and drops stores).
template <typename TT> struct RowIO {
  rsrc_t rQ, rK, rV, rO, rB, rA;
  unsigned step, base, row0, bbase, bstep, abase, astep;
  long bh;
  int i;
  bool in;
  EDF_DEVICE RowIO(const RowArgs& p, int li) {
    const int id = remap_xcd((int)blockIdx.x, (int)gridDim.x);  // a head's row blocks on one XCD
    bh = id / p.nrb;
    i = (id % p.nrb) * RW + li;
    in = i < p.d;
    const int b = (int)(bh / p.H), h = (int)(bh % p.H);
    const long rowel = (long)p.T * p.H * p.d, headel = (long)p.T * p.H;
    const unsigned rowb = (unsigned)(rowel * sizeof(TT)), headb = (unsigned)(headel * sizeof(TT));
    rQ = make_rsrc((const TT*)p.q + b * rowel, rowb), rK = make_rsrc((const TT*)p.k + b * rowel, rowb);
    rV = make_rsrc((const TT*)p.v + b * rowel, rowb);
    rO = make_rsrc(p.out != nullptr ? (const TT*)p.out + b * rowel : (const TT*)p.k, p.out != nullptr ? rowb : 0u);
    rB = p.beta_per_head ? make_rsrc((const TT*)p.beta + b * headel, headb)
                         : make_rsrc((const TT*)p.beta + b * rowel, rowb);
    rA = p.alpha == nullptr ? rB
         : p.alpha_per_row  ? make_rsrc((const TT*)p.alpha + b * rowel, rowb)
                            : make_rsrc((const TT*)p.alpha + b * headel, headb);
    step = (unsigned)((long)p.H * p.d * sizeof(TT));
    base = (unsigned)((long)h * p.d * sizeof(TT));
    row0 = in ? base + i * (unsigned)sizeof(TT) : OOB_OFF;
    const unsigned hstep = (unsigned)(p.H * sizeof(TT)), head0 = in ? h * (unsigned)sizeof(TT) : OOB_OFF;
    bbase = p.beta_per_head ? head0 : row0, bstep = p.beta_per_head ? hstep : step;
    abase = p.alpha_per_row ? row0 : head0, astep = p.alpha_per_row ? step : hstep;
  }
};

// The decay of the lane's steps; a step past T and a row past d are identities (a = 1; beta = v = 0).
template <typename TT>
EDF_DEVICE float decay_of(typename Bits<TT>::type raw, bool live, int alpha_per_row) {
  const float v = bits_f32(raw);
  return live ? (alpha_per_row ? __expf(v) : v) : 1.0f;
}

// Decays within a block of four steps: rMN from after step n to step m, a0 of the first step, all of
// the block, pre from the block's start to the lane's step, end from after the lane's step.
struct BlockDecay {
  float a0, r10, r20, r30, r21, r31, r32, all, pre, end;
  EDF_DEVICE BlockDecay(const float (&a)[4], int grp) {
    a0 = a[0], r10 = a[1], r21 = a[2], r32 = a[3];
    r31 = r32 * r21, r20 = r21 * r10, r30 = r32 * r20;
    all = r30 * a0;
    pre = pick4(a0, r10 * a0, r20 * a0, all, grp);
    end = pick4(r30, r31, r32, 1.0f, grp);
  }
};

// Scalars of the block solves: k_m . k_n of the four steps of block r, m < n, at r * 8 + pair(m, n).
EDF_DEVICE constexpr int pair(int m, int n) { return n * (n - 1) / 2 + m; }

}  // namespace rowscan
}  // namespace edf
