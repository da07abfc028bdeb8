// Flash attention with float32 scores, probabilities and accumulation on the f32 matrix cores
// (v_mfma_f32_32x32x2_f32), forward and backward: float32 tensors of any head_dim <= 128, and
// bfloat16 ones of the head_dims that the bf16 kernels (flash_attn.hip) do not take.
//
// A workgroup of four waves owns 32 queries (dK/dV: 32 keys) of one head and each wave takes
// every fourth 32-row tile of the other side; the four partial results are combined through
// LDS in wave order.  Splitting the other side over the waves, not the 32 rows, makes
// T / 32 x B x H workgroups, so a short sequence still fills the chip, and a causal block's work
// is even over its waves.
//
// Operands.  The scores are formed transposed, S^T = K Q^T, so a lane owns one query (column
// lane % 32): the softmax is lane-local plus one exchange between the wave's halves, and each
// accumulator register of S^T is, as it stands, the B operand of O^T += V^T P^T (register r of
// half g holds key d_row(r, g): the two halves give the two k of a 32x32x2 product, the A
// operand supplying V of the same two keys).  The contraction over head_dim takes four columns
// at a time per half, 8 j + 4 g .. + 3, so a row operand is one 16-byte read for four products.
// The workgroup's own rows (Q; Q and dO; K and V) are in LDS; the other side's tiles go straight
// from memory to registers, a tile ahead, through per-head buffer resources (rows past T and
// columns past head_dim read as zero): a 32 x 32 tile is 64 cycles x head_dim of MFMA against
// 8 x head_dim bytes per row of loads, so staging them through LDS would only add its round trip.
//
// Masked products.  A masked pair has probability 0, but 0 x inf = NaN: where the diagonal tile's
// V (backward: K, Q, dO) holds non-finite values, that tile goes through masked_fma, which takes
// only the visible pairs.
//
// Bound: the f32 MFMA rate (154 TFLOP/s for a large float32 product on this card); short sequences by
// the longest wave.  Measured against one wave per query walking the keys, which this replaces (forward
// and backward, 2 x 8 x 1000 float32 causal: 64 columns 3883 -> 163 us, 96 5290 -> 206, 128 5366 -> 373; bf16, 80
// columns 4377 -> 200; 4 x 16 x 2048 x 64 float32: 120 TFLOP/s forward, 86 backward).  At 128 columns dK/dV holds
// the row and column fragments of Q and dO at once, past its registers: 101 are spilled in float32, 90 in bf16 (FoX
// 308 and 637), which is why that width falls behind.
#include "edf_abi.hpp"
#include "edf_common.hpp"
#include "edf_mfma.hpp"

#include <type_traits>

namespace edf {
namespace {

constexpr float LN2 = 0.6931471805599453f;
constexpr int RB = 32;   // rows a workgroup owns, and rows of a tile
constexpr int NW = 4;    // waves per workgroup, splitting the tiles
typedef __attribute__((ext_vector_type(4))) float f32x4;

EDF_DEVICE f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

template <typename TT> EDF_DEVICE float bld(rsrc_t r, unsigned off) { return bits_f32(bload<TT>(r, off)); }

// Four consecutive elements at byte offset off of a row; left = columns from there to head_dim
// (VEC: head_dim is a multiple of 4, so the four are all inside or all outside).
template <typename TT, bool VEC>
EDF_DEVICE f32x4 load4(rsrc_t r, unsigned off, int left) {
  f32x4 v;
  if constexpr (VEC) {
    off = left > 0 ? off : OOB_OFF;
    if constexpr (sizeof(TT) == 4) {
      v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
    } else {
      const unsigned lo = __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
      const unsigned hi = __builtin_amdgcn_raw_buffer_load_b32(r, (int)(off + 4), 0, 0);
      v[0] = bits_f32(lo << 16), v[1] = bits_f32(lo & 0xffff0000u);
      v[2] = bits_f32(hi << 16), v[3] = bits_f32(hi & 0xffff0000u);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = bld<TT>(r, e < left ? off + e * (unsigned)sizeof(TT) : OOB_OFF);
  }
  return v;
}

// Row fragments of a 32-row tile: lane (li, g) holds columns 8 j + 4 g .. + 3 of row row0 + li.
template <typename TT, int DP, bool VEC>
EDF_DEVICE void load_rows(f32x4 (&f)[DP / 8], rsrc_t r, int row0, int HD, int li, int g) {
  const unsigned base = ((unsigned)(row0 + li) * HD + 4 * g) * (unsigned)sizeof(TT);
#pragma unroll
  for (int j = 0; j < DP / 8; ++j)
    f[j] = load4<TT, VEC>(r, base + 8 * j * (unsigned)sizeof(TT), HD - 8 * j - 4 * g);
}

// Column fragments: register r of c[dt] holds column 32 dt + li of row row0 + d_row(r, g).
template <typename TT, int DP>
EDF_DEVICE void load_cols(float (&c)[DP / 32][16], rsrc_t r, int row0, int HD, int li, int g) {
  const unsigned rowb = (unsigned)HD * (unsigned)sizeof(TT);
#pragma unroll
  for (int dt = 0; dt < DP / 32; ++dt) {
    const int col = 32 * dt + li;
    const unsigned base = col < HD ? (unsigned)(row0 + 4 * g) * rowb + col * (unsigned)sizeof(TT) : OOB_OFF;
#pragma unroll
    for (int x = 0; x < 16; ++x) c[dt][x] = bld<TT>(r, base + (unsigned)(8 * (x >> 2) + (x & 3)) * rowb);
  }
}

template <int DP>
EDF_DEVICE bool finite_cols(const float (&c)[DP / 32][16]) {
  bool ok = true;
#pragma unroll
  for (int dt = 0; dt < DP / 32; ++dt)
#pragma unroll
    for (int x = 0; x < 16; ++x) ok = ok && fabsf(c[dt][x]) < INFINITY;
  return ok;
}

// acc += a * b^T over head_dim: a this lane's row fragments, b rows in LDS (row li, stride LD).
template <int DP>
EDF_DEVICE f32x16 rows_mma(const f32x4 (&a)[DP / 8], const float* b) {
  f32x16 acc = zero16();
#pragma unroll
  for (int j = 0; j < DP / 8; ++j) {
    const f32x4 bv = *(const f32x4*)(b + 8 * j);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = mfma_f32(a[j][e], bv[e], acc);
  }
  return acc;
}

// acc^T[d][col] += sum over the tile's rows of c[row][d] p[row][col]
template <int DP>
EDF_DEVICE void cols_mma(f32x16 (&acc)[DP / 32], const float (&c)[DP / 32][16], const f32x16& p) {
#pragma unroll
  for (int x = 0; x < 16; ++x)
#pragma unroll
    for (int dt = 0; dt < DP / 32; ++dt) acc[dt] = mfma_f32(c[dt][x], p[x], acc[dt]);
}

// The same sum over the rows [lo, hi) only, by vector arithmetic: rows outside take no part, so
// their values (which may be infinite) do not matter.  tp: this wave's 32 x 33 floats of LDS.
template <typename TT, int DP>
EDF_DEVICE void masked_fma(f32x16 (&acc)[DP / 32], const f32x16& p, float* tp, rsrc_t r, int row0, int lo, int hi,
                           int HD, int li, int g) {
#pragma unroll
  for (int x = 0; x < 16; ++x) tp[li * 33 + d_row(x, g)] = p[x];
  __builtin_amdgcn_wave_barrier();
#pragma unroll 1
  for (int k = 0; k < RB; ++k) {
    const float pk = tp[li * 33 + k];
    const bool in = k >= lo && k < hi;
#pragma unroll
    for (int dt = 0; dt < DP / 32; ++dt)
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        const int col = 32 * dt + d_row(x, g);
        const float v =
            bld<TT>(r, in && col < HD ? ((unsigned)(row0 + k) * HD + col) * (unsigned)sizeof(TT) : OOB_OFF);
        acc[dt][x] = in ? fmaf(pk, v, acc[dt][x]) : acc[dt][x];
      }
  }
  __builtin_amdgcn_wave_barrier();
}

// LDS floats: N staged row tiles and each wave's masked_fma tile during the loop, then the four
// partials over them.
template <int DP, int N>
constexpr int lds_floats() {
  constexpr int loop = N * RB * (DP + 4) + NW * 32 * 33, part = NW * RB * (DP + 4);
  return loop > part ? loop : part;
}

// The workgroup's own 32 rows into LDS as float32, zero past T and past head_dim.
template <typename TT, int DP>
EDF_DEVICE void stage_rows(float* s, rsrc_t r, int row0, int HD) {
  constexpr int LD = DP + 4;
#pragma unroll
  for (int i = 0; i < RB * DP / 256; ++i) {
    const int e = threadIdx.x + 256 * i, row = e / DP, col = e % DP;
    s[row * LD + col] = bld<TT>(r, col < HD ? ((unsigned)(row0 + row) * HD + col) * (unsigned)sizeof(TT) : OOB_OFF);
  }
}

// One wave's accumulator tile (column = own row li) as rows of its LDS partial.
template <int DP>
EDF_DEVICE void store_partial(float* s, const f32x16 (&acc)[DP / 32], float f, int li, int g) {
  constexpr int LD = DP + 4;
#pragma unroll
  for (int dt = 0; dt < DP / 32; ++dt)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = acc[dt][4 * q + e] * f;
      *(f32x4*)(s + li * LD + 32 * dt + 8 * q + 4 * g) = v;
    }
}

// The four waves' partials added in wave order, times the row's factor, to the 32 rows of dst.
template <typename TT, int DP, typename F>
EDF_DEVICE void write_rows(rsrc_t r, const float* part, int row0, int HD, F&& factor) {
  constexpr int LD = DP + 4;
#pragma unroll
  for (int i = 0; i < RB * DP / 256; ++i) {
    const int e = threadIdx.x + 256 * i, row = e / DP, col = e % DP;
    const float* p = part + row * LD + col;
    float v = p[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += p[w * RB * LD];
    bstore<TT>(r, col < HD ? ((unsigned)(row0 + row) * HD + col) * (unsigned)sizeof(TT) : OOB_OFF, v * factor(row));
  }
}

struct Args {
  const void *q, *k, *v, *o, *dout, *cs;
  void *out, *dq, *dk, *dv, *dcs;
  float *lse_out, *dcsk;
  const float *lse, *dd;
  int T, HD;
  float scale_log2, scale, sqd;
};

// (head, first own row) of this workgroup: blocks of one head on one XCD, the block with the
// most tiles first (causal forward and dQ: the last rows; dK/dV: the first).
EDF_DEVICE void own_block(int T, bool last_first, long& bh, int& row0) {
  const int nb = (T + RB - 1) / RB;
  const int id = remap_xcd((int)blockIdx.x, (int)gridDim.x);
  bh = id / nb;
  const int b = id % nb;
  row0 = (last_first ? nb - 1 - b : b) * RB;
}

template <typename TT, int DP, bool CAUSAL, bool FOX, bool VEC>
__global__ __launch_bounds__(256, DP <= 64 ? 2 : 1) void fa32_fwd_kernel(const Args a) {
  constexpr int LD = DP + 4, NDT = DP / 32;
  __shared__ __attribute__((aligned(16))) float sP[lds_floats<DP, 1>()];
  __shared__ float sM[NW][RB], sL[NW][RB];
  float* const sQ = sP;
  float* const sT = sP + RB * LD + (threadIdx.x >> 6) * 32 * 33;
  const int T = a.T, HD = a.HD;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 5, li = l & 31;
  long bh;
  int q0;
  own_block(T, CAUSAL, bh, q0);
  const long head = bh * T * HD;
  const unsigned bytes = (unsigned)((long)T * HD * sizeof(TT));
  const rsrc_t rQ = make_rsrc((const TT*)a.q + head, bytes), rK = make_rsrc((const TT*)a.k + head, bytes);
  const rsrc_t rV = make_rsrc((const TT*)a.v + head, bytes);
  const rsrc_t rC = make_rsrc(FOX ? (const TT*)a.cs + bh * T : (const TT*)a.q, FOX ? T * (unsigned)sizeof(TT) : 0u);
  stage_rows<TT, DP>(sQ, rQ, q0, HD);
  __syncthreads();
  const float* myQ = sQ + li * LD + 4 * g;
  const int myq = q0 + li;
  const float csq = FOX ? bld<TT>(rC, (unsigned)myq * (unsigned)sizeof(TT)) * a.sqd : 0.0f;

  const int nt = CAUSAL ? q0 / RB + 1 : (T + RB - 1) / RB;
  f32x16 o[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) o[dt] = zero16();
  float m = -INFINITY, lsum = 0.0f;
  f32x4 kf[DP / 8];
  load_rows<TT, DP, VEC>(kf, rK, min(w, nt - 1) * RB, HD, li, g);
  for (int t = w; t < nt; t += NW) {
    const int k0 = t * RB;
    float vc[NDT][16];
    load_cols<TT, DP>(vc, rV, k0, HD, li, g);
    f32x16 s = rows_mma<DP>(kf, myQ);
    load_rows<TT, DP, VEC>(kf, rK, min(t + NW, nt - 1) * RB, HD, li, g);  // the next tile (at the end, a reload)
    if constexpr (FOX) {
#pragma unroll
      for (int x = 0; x < 16; ++x)
        s[x] += fmaf(-bld<TT>(rC, (unsigned)(k0 + d_row(x, g)) * (unsigned)sizeof(TT)), a.sqd, csq);
    }
    const bool edge = t == nt - 1;  // the diagonal tile, or the one that may pass T
    if (edge) {
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        const int key = k0 + d_row(x, g);
        s[x] = key < T && (!CAUSAL || key <= myq) ? s[x] : -INFINITY;
      }
    }
    float mt = s[0];
#pragma unroll
    for (int x = 1; x < 16; ++x) mt = fmaxf(mt, s[x]);
    mt = fmaxf(mt, __shfl_xor(mt, 32));
    const float mn = fmaxf(m, mt);
    const float c = mn == -INFINITY ? 0.0f : mn * a.scale_log2;  // (no finite score yet: every p is 0)
    const float al = m == -INFINITY ? 0.0f : fast_exp2(fmaf(m, a.scale_log2, -c));
    f32x16 p;
    float rs = 0.0f;
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      p[x] = fast_exp2(fmaf(s[x], a.scale_log2, -c));
      rs += p[x];
    }
    lsum = fmaf(lsum, al, rs);
    m = mn;
    if (__any(al != 1.0f)) {
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int x = 0; x < 16; ++x) o[dt][x] *= al;
    }
    if (CAUSAL && edge && __any(!finite_cols<DP>(vc)))
      masked_fma<TT, DP>(o, p, sT, rV, k0, 0, myq + 1 - k0, HD, li, g);
    else
      cols_mma<DP>(o, vc, p);
  }
  lsum += __shfl_xor(lsum, 32);
  if (g == 0) {
    sM[w][li] = m;
    sL[w][li] = lsum;
  }
  __syncthreads();
  float M = sM[0][li];
#pragma unroll
  for (int i = 1; i < NW; ++i) M = fmaxf(M, sM[i][li]);
  store_partial<DP>(sP + w * RB * LD, o, m == -INFINITY ? 0.0f : fast_exp2((m - M) * a.scale_log2), li, g);
  __syncthreads();
  auto total = [&](int row, float& mx) {
    mx = sM[0][row];
#pragma unroll
    for (int i = 1; i < NW; ++i) mx = fmaxf(mx, sM[i][row]);
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < NW; ++i)  // (a wave without a finite score has the sum 0, or NaN where a score was)
      sum += sM[i][row] == -INFINITY ? sL[i][row] : sL[i][row] * fast_exp2((sM[i][row] - mx) * a.scale_log2);
    return sum;
  };
  if (threadIdx.x < RB && q0 + threadIdx.x < T && a.lse_out != nullptr) {
    float mx;
    const float sum = total(threadIdx.x, mx);
    a.lse_out[bh * T + q0 + threadIdx.x] = (mx * a.scale_log2 + __log2f(sum)) * LN2;
  }
  const rsrc_t rO = make_rsrc((TT*)a.out + head, bytes);
  write_rows<TT, DP>(rO, sP, q0, HD, [&](int row) {
    float mx;
    return 1.0f / total(row, mx);
  });
}

// ---- bf16 tensors whose rows are whole 16-byte pieces (head_dim a multiple of 8): forward ----------
//
// The products of bf16 numbers are exact in float32, so the scores need no more than the bf16 MFMA with its
// float32 sums; the probabilities stay float32 by going into O^T += V^T P^T as three bf16 parts that
// add up to them exactly (8 + 8 + 8 mantissa bits, by truncation).  Four bf16 products take the place of two
// f32 ones at a sixteenth of the time each.  128 queries per workgroup (32 per wave), 64-key K and V tiles in
// a double LDS buffer, loaded a tile ahead through per-head buffer resources (rows past T and columns
// past head_dim read as zero); V^T operands by transposed LDS reads.
// 2 x 16 x 1500 x 96, not causal: 329 us on the f32 MFMA, 65 us here (424 TFLOP/s of the two products).

// hi, mid and low bf16 parts of eight probabilities
EDF_DEVICE void split8(const f32x16& p, int at, bf16x8 (&part)[3]) {
  float x[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = p[at + i];
#pragma unroll
  for (int n = 0; n < 3; ++n) {
    u32x4 w;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      w[i] = __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, x[2 * i + 1]), __builtin_bit_cast(unsigned, x[2 * i]),
                                   0x07060302u);
    part[n] = __builtin_bit_cast(bf16x8, w);
    if (n < 2) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        x[i] -= __builtin_bit_cast(float, __builtin_bit_cast(unsigned, x[i]) & 0xffff0000u);
    }
  }
}

EDF_DEVICE bool finite8(bf16x8 v) {
  const u32x4 b = __builtin_bit_cast(u32x4, v);
  bool ok = true;
#pragma unroll
  for (int i = 0; i < 4; ++i) ok = ok && (b[i] & 0x7f80u) != 0x7f80u && (b[i] & 0x7f800000u) != 0x7f800000u;
  return ok;
}

template <int DP, bool CAUSAL, bool FOX>
__global__ __launch_bounds__(256, CAUSAL && DP == 128 ? 1 : 2) void fa_split_fwd_kernel(const Args a) {
  constexpr int BM = 128, BN = 64, NKK = DP / 16, NDT = DP / 32, CPR = DP / 8, CPT = BN * CPR / 256;
  __shared__ __attribute__((aligned(16))) bf16 sK[2][lds_tile_elems<DP>(BN)];
  __shared__ __attribute__((aligned(16))) bf16 sV[2][lds_tile_elems<DP>(BN)];
  __shared__ __attribute__((aligned(16))) float sC[FOX ? 2 : 1][FOX ? BN : 4];
  const int T = a.T, HD = a.HD;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, g = l >> 5, li = l & 31;
  const int nb = (T + BM - 1) / BM, id = remap_xcd((int)blockIdx.x, (int)gridDim.x);
  const long bh = id / nb;
  const int q0 = (CAUSAL ? nb - 1 - id % nb : id % nb) * BM, qw = q0 + 32 * w, myq = qw + li;
  const long head = bh * T * HD;
  const unsigned bytes = (unsigned)((long)T * HD * 2);
  const rsrc_t rQ = make_rsrc((const bf16*)a.q + head, bytes), rK = make_rsrc((const bf16*)a.k + head, bytes);
  const rsrc_t rV = make_rsrc((const bf16*)a.v + head, bytes), rO = make_rsrc((bf16*)a.out + head, bytes);
  const rsrc_t rC = make_rsrc(FOX ? (const bf16*)a.cs + bh * T : (const bf16*)a.q, FOX ? T * 2u : 0u);
  auto piece = [&](rsrc_t r, int row, int col) {
    const unsigned off = col < HD ? ((unsigned)row * HD + col) * 2u : OOB_OFF;
    return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
  };

  bf16x8 qf[NKK];  // Q^T as MFMA B fragments
#pragma unroll
  for (int kk = 0; kk < NKK; ++kk) qf[kk] = piece(rQ, myq, kk * 16 + 8 * g);
  f32x16 o[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) o[dt] = zero16();
  float m = -INFINITY, lsum = 0.0f;
  bf16x8 rk[CPT], rv[CPT];
  float rcs = 0.0f;
  auto gload = [&](int k0) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = tid + 256 * i;
      rk[i] = piece(rK, k0 + c / CPR, (c % CPR) * 8);
      rv[i] = piece(rV, k0 + c / CPR, (c % CPR) * 8);
    }
    if (FOX && tid < BN) rcs = bld<bf16>(rC, (unsigned)(k0 + tid) * 2u);
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = tid + 256 * i, at = lds_off<DP>(c / CPR, (c % CPR) * 8);
      *(bf16x8*)(&sK[buf][at]) = rk[i];
      *(bf16x8*)(&sV[buf][at]) = rv[i];
    }
    if (FOX && tid < BN) sC[buf][tid] = rcs;
  };
  const float csq = FOX ? bld<bf16>(rC, (unsigned)myq * 2u) * a.sqd : 0.0f;
  // V^T fragment of keys 16 kc + 4 g + 0..3, 16 kc + 8 + 4 g + 0..3, columns 32 dt + li
  const int d0 = 16 * ((l >> 4) & 1) + 4 * (l & 3), kr = 4 * g + ((l & 15) >> 2);
  auto vfrag = [&](const bf16* sv, int dt, int kc) {
    return cat4(lds_read_tr16(sv + lds_off<DP>(16 * kc + kr, dt * 32 + d0)),
                lds_read_tr16(sv + lds_off<DP>(16 * kc + kr + 8, dt * 32 + d0)));
  };

  const int kend = CAUSAL ? min(T, q0 + BM) : T, nkt = (kend + BN - 1) / BN;
  gload(0);
  sstore(0);
  gload(BN);
  __syncthreads();
  auto tile = [&](int kt, auto masked) {
    constexpr bool MASK = decltype(masked)::value;
    const int k0 = kt * BN, buf = kt & 1;
    const bf16 *sk = sK[buf], *sv = sV[buf];
    f32x16 s[2];
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      s[h2] = zero16();
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk)
        s[h2] = mfma32(*(const bf16x8*)(sk + lds_off<DP>(h2 * 32 + li, kk * 16 + 8 * g)), qf[kk], s[h2]);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kl = h2 * 32 + d_row(r, g);
        if constexpr (FOX) s[h2][r] += fmaf(-sC[buf][kl], a.sqd, csq);
        if constexpr (MASK) s[h2][r] = (k0 + kl >= T || (CAUSAL && k0 + kl > myq)) ? -INFINITY : s[h2][r];
        mx = fmaxf(mx, s[h2][r]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float mnew = fmaxf(m, mx);
    const float mns = mnew == -INFINITY ? 0.0f : mnew * a.scale_log2;
    if (__any(mnew > m)) {  // rescale only when some row maximum grew
      const float alpha = fast_exp2(fmaf(m, a.scale_log2, -mns));
      lsum *= alpha;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
    }
    m = mnew;
    float rs = 0.0f;
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[h2][r] = fast_exp2(fmaf(s[h2][r], a.scale_log2, -mns));
        rs += s[h2][r];
      }
    lsum += rs;
    bool bad = false;  // a masked key's infinite or NaN value must not enter with probability 0
    if constexpr (MASK && CAUSAL) {
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) bad = bad || !finite8(vfrag(sv, dt, kc));
      bad = __any(bad);
    }
    if (MASK && CAUSAL && bad) {
      // the visible pairs one by one
#pragma unroll 1
      for (int k = 0; k < BN; ++k) {
        float pk = 0.0f;  // this lane's half of the keys; the key's half is (k / 4) % 2
#pragma unroll
        for (int r = 0; r < 32; ++r) pk = r == 16 * (k >> 5) + 4 * ((k >> 3) & 3) + (k & 3) ? s[r >> 4][r & 15] : pk;
        pk = __shfl(pk, li + 32 * ((k >> 2) & 1));
        const bool vis = k0 + k < T && k0 + k <= myq;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
#pragma unroll
          for (int rb = 0; rb < 4; ++rb) {
            const bf16x4 v = *(const bf16x4*)(sv + lds_off<DP>(k, dt * 32 + 8 * rb + 4 * g));
#pragma unroll
            for (int e = 0; e < 4; ++e) o[dt][4 * rb + e] = vis ? fmaf(pk, (float)v[e], o[dt][4 * rb + e]) : o[dt][4 * rb + e];
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      return;
    }
#pragma unroll
    for (int kc = 0; kc < 4; ++kc) {
      bf16x8 pf[3];
      split8(s[kc >> 1], 8 * (kc & 1), pf);
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        const bf16x8 vf = vfrag(sv, dt, kc);
#pragma unroll
        for (int n = 2; n >= 0; --n) o[dt] = mfma32(vf, pf[n], o[dt]);
      }
    }
  };
  auto advance = [&](int kt) {  // the next tile into the other buffer, the one after it into registers
    if (kt + 1 < nkt) {
      sstore((kt & 1) ^ 1);
      gload((kt + 2) * BN);
    }
    __syncthreads();
  };
  const int ksplit = min(min(T / BN, nkt), CAUSAL ? (qw + 1) / BN : nkt);  // tiles with nothing masked come first
  int kt = 0;
  for (; kt < ksplit; ++kt) {
    tile(kt, std::false_type{});
    advance(kt);
  }
  for (; kt < nkt; ++kt) {
    tile(kt, std::true_type{});
    advance(kt);
  }
  lsum += __shfl_xor(lsum, 32);
  // O as whole rows, each wave's 32 through the free K tiles
  static_assert(2 * lds_tile_elems<DP>(BN) >= lds_tile_elems<DP>(BM), "O staging");
  bf16* so = &sK[0][0];
  const float inv = 1.0f / lsum;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (bf16)(o[dt][rb * 4 + e] * inv);
      *(bf16x4*)(so + lds_off<DP>(32 * w + li, dt * 32 + 8 * rb + 4 * g)) = v;
    }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int i = 0; i < 32 * CPR / 64; ++i) {
    const int e = l + 64 * i, row = e / CPR, col = 8 * (e % CPR);
    const unsigned off = col < HD ? ((unsigned)(qw + row) * HD + col) * 2u : OOB_OFF;
    __builtin_amdgcn_raw_buffer_store_b128(*(const u32x4*)(so + lds_off<DP>(32 * w + row, col)), rO, (int)off, 0, 0);
  }
  if (myq < T && g == 0 && a.lse_out != nullptr) a.lse_out[bh * T + myq] = (m * a.scale_log2 + __log2f(lsum)) * LN2;
}

template <int DP>
void split_by_mask(hipStream_t s, const Args& a, unsigned grid, int causal) {
  if (a.cs != nullptr)
    fa_split_fwd_kernel<DP, true, true><<<grid, 256, 0, s>>>(a);
  else if (causal)
    fa_split_fwd_kernel<DP, true, false><<<grid, 256, 0, s>>>(a);
  else
    fa_split_fwd_kernel<DP, false, false><<<grid, 256, 0, s>>>(a);
}

// dQ of 32 queries: P and dP over the key tiles, dQ^T += K^T dS^T.  FOX: d cs of the query is
// the sum of its dS over the keys plus the key side that the dK/dV kernel wrote.
template <typename TT, int DP, bool CAUSAL, bool FOX, bool VEC>
__global__ __launch_bounds__(256, DP <= 64 ? 2 : 1) void fa32_dq_kernel(const Args a) {
  constexpr int LD = DP + 4, NDT = DP / 32;
  __shared__ __attribute__((aligned(16))) float sP[lds_floats<DP, 2>()];
  __shared__ float sR[NW][RB];
  float *const sQ = sP, *const sG = sP + RB * LD;
  float* const sT = sP + 2 * RB * LD + (threadIdx.x >> 6) * 32 * 33;
  const int T = a.T, HD = a.HD;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 5, li = l & 31;
  long bh;
  int q0;
  own_block(T, CAUSAL, bh, q0);
  const long head = bh * T * HD;
  const unsigned bytes = (unsigned)((long)T * HD * sizeof(TT));
  const rsrc_t rQ = make_rsrc((const TT*)a.q + head, bytes), rK = make_rsrc((const TT*)a.k + head, bytes);
  const rsrc_t rV = make_rsrc((const TT*)a.v + head, bytes), rG = make_rsrc((const TT*)a.dout + head, bytes);
  const rsrc_t rC = make_rsrc(FOX ? (const TT*)a.cs + bh * T : (const TT*)a.q, FOX ? T * (unsigned)sizeof(TT) : 0u);
  stage_rows<TT, DP>(sQ, rQ, q0, HD);
  stage_rows<TT, DP>(sG, rG, q0, HD);
  __syncthreads();
  const float *myQ = sQ + li * LD + 4 * g, *myG = sG + li * LD + 4 * g;
  const int myq = q0 + li;
  const float lse2 = myq < T ? a.lse[bh * T + myq] * LOG2E : 0.0f, D = myq < T ? a.dd[bh * T + myq] : 0.0f;
  const float csq = FOX ? bld<TT>(rC, (unsigned)myq * (unsigned)sizeof(TT)) * a.sqd : 0.0f;

  const int nt = CAUSAL ? q0 / RB + 1 : (T + RB - 1) / RB;
  f32x16 dq[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) dq[dt] = zero16();
  float rowacc = 0.0f;
  f32x4 kf[DP / 8];
  load_rows<TT, DP, VEC>(kf, rK, min(w, nt - 1) * RB, HD, li, g);
  for (int t = w; t < nt; t += NW) {
    const int k0 = t * RB;
    f32x4 vf[DP / 8];
    load_rows<TT, DP, VEC>(vf, rV, k0, HD, li, g);
    f32x16 s = rows_mma<DP>(kf, myQ);
    float kc[NDT][16];
    load_cols<TT, DP>(kc, rK, k0, HD, li, g);
    const f32x16 dp = rows_mma<DP>(vf, myG);
    load_rows<TT, DP, VEC>(kf, rK, min(t + NW, nt - 1) * RB, HD, li, g);
    if constexpr (FOX) {
#pragma unroll
      for (int x = 0; x < 16; ++x)
        s[x] += fmaf(-bld<TT>(rC, (unsigned)(k0 + d_row(x, g)) * (unsigned)sizeof(TT)), a.sqd, csq);
    }
    const bool edge = t == nt - 1;
    f32x16 ds;
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      ds[x] = fast_exp2(fmaf(s[x], a.scale_log2, -lse2)) * (dp[x] - D);
      if (edge) {
        const int key = k0 + d_row(x, g);
        ds[x] = key < T && (!CAUSAL || key <= myq) ? ds[x] : 0.0f;
      }
      if constexpr (FOX) rowacc += ds[x];
      ds[x] *= a.scale;
    }
    if (CAUSAL && edge && __any(!finite_cols<DP>(kc)))
      masked_fma<TT, DP>(dq, ds, sT, rK, k0, 0, myq + 1 - k0, HD, li, g);
    else
      cols_mma<DP>(dq, kc, ds);
  }
  __syncthreads();  // every wave is done with the staged rows, which the partials replace
  store_partial<DP>(sP + w * RB * LD, dq, 1.0f, li, g);
  if constexpr (FOX) {
    rowacc += __shfl_xor(rowacc, 32);
    if (g == 0) sR[w][li] = rowacc;
  }
  __syncthreads();
  write_rows<TT, DP>(make_rsrc((TT*)a.dq + head, bytes), sP, q0, HD, [](int) { return 1.0f; });
  if constexpr (FOX) {
    if (threadIdx.x < RB && q0 + threadIdx.x < T) {
      const int i = threadIdx.x;
      st((TT*)a.dcs, bh * T + q0 + i, ((sR[0][i] + sR[1][i]) + sR[2][i]) + sR[3][i] + a.dcsk[bh * T + q0 + i]);
    }
  }
}

// dK, dV of 32 keys: S = Q K^T, so a lane owns one key; dV^T += dO^T P, dK^T += Q^T dS over the
// query tiles.  FOX: the key side of d cs, minus the sum of dS over the queries, to dcsk.
template <typename TT, int DP, bool CAUSAL, bool FOX, bool VEC>
__global__ __launch_bounds__(256, 1) void fa32_dkdv_kernel(const Args a) {
  constexpr int LD = DP + 4, NDT = DP / 32;
  __shared__ __attribute__((aligned(16))) float sP[lds_floats<DP, 2>()];
  __shared__ float sR[NW][RB];
  float *const sK = sP, *const sV = sP + RB * LD;
  float* const sT = sP + 2 * RB * LD + (threadIdx.x >> 6) * 32 * 33;
  const int T = a.T, HD = a.HD;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 5, li = l & 31;
  long bh;
  int j0;
  own_block(T, false, bh, j0);
  const long head = bh * T * HD;
  const unsigned bytes = (unsigned)((long)T * HD * sizeof(TT));
  const rsrc_t rQ = make_rsrc((const TT*)a.q + head, bytes), rK = make_rsrc((const TT*)a.k + head, bytes);
  const rsrc_t rV = make_rsrc((const TT*)a.v + head, bytes), rG = make_rsrc((const TT*)a.dout + head, bytes);
  const rsrc_t rC = make_rsrc(FOX ? (const TT*)a.cs + bh * T : (const TT*)a.q, FOX ? T * (unsigned)sizeof(TT) : 0u);
  const rsrc_t rL = make_rsrc(a.lse + bh * T, T * 4u), rD = make_rsrc(a.dd + bh * T, T * 4u);
  stage_rows<TT, DP>(sK, rK, j0, HD);
  stage_rows<TT, DP>(sV, rV, j0, HD);
  __syncthreads();
  const float *myK = sK + li * LD + 4 * g, *myV = sV + li * LD + 4 * g;
  const int myk = j0 + li;
  const float csk = FOX ? bld<TT>(rC, (unsigned)myk * (unsigned)sizeof(TT)) * a.sqd : 0.0f;

  const int nt = (T + RB - 1) / RB, t0 = CAUSAL ? j0 / RB : 0;
  f32x16 dk[NDT], dv[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) dk[dt] = dv[dt] = zero16();
  float colacc = 0.0f;
  f32x4 qf[DP / 8];
  load_rows<TT, DP, VEC>(qf, rQ, min(t0 + w, nt - 1) * RB, HD, li, g);
  for (int t = t0 + w; t < nt; t += NW) {
    const int i0 = t * RB;
    f32x4 gf[DP / 8];
    load_rows<TT, DP, VEC>(gf, rG, i0, HD, li, g);
    float ls[16], dd[16];
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      ls[x] = bld<float>(rL, (unsigned)(i0 + d_row(x, g)) * 4u);
      dd[x] = bld<float>(rD, (unsigned)(i0 + d_row(x, g)) * 4u);
    }
    f32x16 s = rows_mma<DP>(qf, myK);
    float gc[NDT][16], qc[NDT][16];
    load_cols<TT, DP>(gc, rG, i0, HD, li, g);
    const f32x16 dp = rows_mma<DP>(gf, myV);
    load_cols<TT, DP>(qc, rQ, i0, HD, li, g);
    load_rows<TT, DP, VEC>(qf, rQ, min(t + NW, nt - 1) * RB, HD, li, g);
    if constexpr (FOX) {
#pragma unroll
      for (int x = 0; x < 16; ++x)
        s[x] += fmaf(bld<TT>(rC, (unsigned)(i0 + d_row(x, g)) * (unsigned)sizeof(TT)), a.sqd, -csk);
    }
    // the diagonal tile, and the last one, whose queries may pass T
    const bool edge = (CAUSAL && t == t0) || t == nt - 1;
    f32x16 p, ds;
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      p[x] = fast_exp2(fmaf(s[x], a.scale_log2, -ls[x] * LOG2E));
      ds[x] = p[x] * (dp[x] - dd[x]);
      if (edge) {
        const int qr = i0 + d_row(x, g);
        const bool in = qr < T && (!CAUSAL || qr >= myk);
        p[x] = in ? p[x] : 0.0f;
        ds[x] = in ? ds[x] : 0.0f;
      }
      if constexpr (FOX) colacc += ds[x];
      ds[x] *= a.scale;
    }
    if (CAUSAL && t == t0 && __any(!finite_cols<DP>(gc) || !finite_cols<DP>(qc))) {
      masked_fma<TT, DP>(dv, p, sT, rG, i0, myk - i0, RB, HD, li, g);
      masked_fma<TT, DP>(dk, ds, sT, rQ, i0, myk - i0, RB, HD, li, g);
    } else {
      cols_mma<DP>(dv, gc, p);
      cols_mma<DP>(dk, qc, ds);
    }
  }
  if constexpr (FOX) {
    colacc += __shfl_xor(colacc, 32);
    if (g == 0) sR[w][li] = colacc;
  }
  const auto one = [](int) { return 1.0f; };
  __syncthreads();  // every wave is done with the staged rows, which the partials replace
  store_partial<DP>(sP + w * RB * LD, dv, 1.0f, li, g);
  __syncthreads();
  write_rows<TT, DP>(make_rsrc((TT*)a.dv + head, bytes), sP, j0, HD, one);
  __syncthreads();
  store_partial<DP>(sP + w * RB * LD, dk, 1.0f, li, g);
  __syncthreads();
  write_rows<TT, DP>(make_rsrc((TT*)a.dk + head, bytes), sP, j0, HD, one);
  if constexpr (FOX) {
    if (threadIdx.x < RB && j0 + threadIdx.x < T) {
      const int i = threadIdx.x;
      a.dcsk[bh * T + j0 + i] = -(((sR[0][i] + sR[1][i]) + sR[2][i]) + sR[3][i]);
    }
  }
}

template <typename TT, int DP, bool CAUSAL, bool FOX, bool VEC>
void launch(hipStream_t s, const Args& a, unsigned grid, bool bwd) {
  if (!bwd) {
    fa32_fwd_kernel<TT, DP, CAUSAL, FOX, VEC><<<grid, 256, 0, s>>>(a);
    return;
  }
  fa32_dkdv_kernel<TT, DP, CAUSAL, FOX, VEC><<<grid, 256, 0, s>>>(a);  // first: dQ adds its key side of d cs
  fa32_dq_kernel<TT, DP, CAUSAL, FOX, VEC><<<grid, 256, 0, s>>>(a);
}

template <typename TT, int DP, bool VEC>
void by_mask(hipStream_t s, const Args& a, unsigned grid, int causal, bool bwd) {
  if (a.cs != nullptr)
    launch<TT, DP, true, true, VEC>(s, a, grid, bwd);  // FoX attention is causal
  else if (causal)
    launch<TT, DP, true, false, VEC>(s, a, grid, bwd);
  else
    launch<TT, DP, false, false, VEC>(s, a, grid, bwd);
}

template <typename TT>
void by_width(hipStream_t s, const Args& a, unsigned grid, int causal, bool bwd) {
  // 16-byte (bf16: two 4-byte) row loads need whole groups of four columns on 4-byte boundaries
  const uintptr_t at = (uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)(bwd ? a.dout : a.q);
  const bool vec = a.HD % 4 == 0 && at % 4 == 0;
#define EDF_FA32(DP) (vec ? by_mask<TT, DP, true>(s, a, grid, causal, bwd) : by_mask<TT, DP, false>(s, a, grid, causal, bwd))
  if (a.HD <= 32)
    EDF_FA32(32);
  else if (a.HD <= 64)
    EDF_FA32(64);
  else if (a.HD <= 96)
    EDF_FA32(96);
  else
    EDF_FA32(128);
#undef EDF_FA32
}

}  // namespace

// Whether these kernels take a call: rows of a head addressed by 31-bit byte offsets, and more than a few of them.
// A tile costs the same however many of its 32 rows are there, so the shortest sequences keep one wave per query
// (flash_attn.hip, flash_attn_bwd.hip); us with gradients, wave per query / tiles, 32 heads, causal:
//   float32 d 64:  seq 8 20 / 28, seq 16 31 / 28        d 96: seq 16 40 / 39, seq 24 56 / 39
//           d 128: seq 16 42 / 55, seq 24 57 / 55       FoX d 128: seq 24 61 / 81, seq 32 76 / 82, seq 48 112 / 84
bool fa32_takes(int batch_heads, int T, int HD, int dtype, bool fox) {
  if (T < (HD <= 64 ? 16 : HD <= 96 ? 17 : fox ? 33 : 25)) return false;
  const long nb = (long)((T + RB - 1) / RB) * batch_heads;
  return HD <= 128 && (long)(T + 256) * HD * (dtype == EDF_BF16 ? 2 : 4) < (1L << 31) && nb < (1L << 31);
}

int fa32_forward(hipStream_t s, const void* q, const void* k, const void* v, const void* cs, void* out, float* lse,
                 int BH, int T, int HD, int causal, int dtype) {
  Args a{};
  a.q = q, a.k = k, a.v = v, a.cs = cs, a.out = out, a.lse_out = lse;
  a.T = T, a.HD = HD;
  a.scale = 1.0f / sqrtf((float)HD), a.scale_log2 = LOG2E / sqrtf((float)HD), a.sqd = sqrtf((float)HD);
  const unsigned grid = (unsigned)(((T + RB - 1) / RB) * (long)BH);
  // the split kernel loads and stores rows in 16-byte pieces on 4-byte boundaries
  const uintptr_t at = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out;
  if (dtype == EDF_BF16 && HD % 8 == 0 && at % 4 == 0) {
    const unsigned gs = (unsigned)(((T + 127) / 128) * (long)BH);
    if (HD <= 32)
      split_by_mask<32>(s, a, gs, causal);
    else if (HD <= 64)
      split_by_mask<64>(s, a, gs, causal);
    else if (HD <= 96)
      split_by_mask<96>(s, a, gs, causal);
    else
      split_by_mask<128>(s, a, gs, causal);
  } else if (dtype == EDF_BF16) {
    by_width<bf16>(s, a, grid, causal, false);
  } else {
    by_width<float>(s, a, grid, causal, false);
  }
  return check_launch("flash attention (float32 probabilities)");
}

// dd: rowsum(dO o O) [BH][T], already written; cs, dcsk, dcs: FoX attention, else null
int fa32_backward(hipStream_t s, const void* q, const void* k, const void* v, const void* dout, const float* lse,
                  const float* dd, void* dq, void* dk, void* dv, const void* cs, float* dcsk, void* dcs, int BH, int T,
                  int HD, int causal, int dtype) {
  Args a{};
  a.q = q, a.k = k, a.v = v, a.dout = dout, a.cs = cs, a.lse = lse, a.dd = dd;
  a.dq = dq, a.dk = dk, a.dv = dv, a.dcsk = dcsk, a.dcs = dcs;
  a.T = T, a.HD = HD;
  a.scale = 1.0f / sqrtf((float)HD), a.scale_log2 = a.scale * LOG2E, a.sqd = sqrtf((float)HD);
  const unsigned grid = (unsigned)(((T + RB - 1) / RB) * (long)BH);
  if (dtype == EDF_BF16)
    by_width<bf16>(s, a, grid, causal, true);
  else
    by_width<float>(s, a, grid, causal, true);
  return check_launch("flash attention backward (f32 matrix cores)");
}

}  // namespace edf
