// The filters of the blocks after 0 on their radial tables, forward and
// reverse, shared by the v1 kernels (evaluator.hip) and the generic widths
// (generic.hip): 16 pairs of one bucket (spatial block and interval of r) per
// wavefront, F = 16 FT features in FT / 2 heads of 32.
//
// The pairs' node rows are what these kernels read most (8 KB a pair at
// F = 128), and a vector load takes one L1 access per quad of lanes and row:
// with the pairs on the lanes, a quad reads four rows and a 16-byte load takes
// 64 accesses; with 16 lanes along one row it takes 16.  So the rows are
// loaded and stored with lane j of a group of 16 on channels 2 j and 2 j + 1
// of a head and the pairs g + 4 r (r = 0..3) one after the other.  24,000
// atoms, 476,500 pairs (us, pairs on the lanes / this layout): forward 697 /
// 515, reverse 528 / 416; F = 256 1,887 / 1,208 and 1,396 / 1,035.  By the
// counters the L1's accesses alone were 0.93, 0.91, 0.69 and 0.91 of the time
// before and are 0.55, 0.59, 0.55 and 0.61 now.  No unit is busy all the time:
// the matrix pipe 0.44, 0.55, 0.57 and 0.70, the other vector instructions,
// none of which runs beside an MFMA, up to 0.18, 0.11, 0.14 and 0.08; the rest
// is waits, two wavefronts a SIMD not covering every operand from L2.
#pragma once

#include "node_chain.hpp"

namespace so3lr_amd {
namespace {

struct RowsArgs {
  const int *slots, *order, *pa;
  const double *pr, *qkv, *rtab;  // rtab: coefficient tiles (forward) or slope tiles (reverse)
  RadialDomain d;
  // the spherical layers: E0 and its bias; forward E1, its rows in head-pair
  // order (head_pairs); reverse E1^T and E0^T
  const double *e0[2], *eb0[2], *e1[2], *e0t[2];
  const double *exp2_256;
  double *ps;  // pair invariants (pair, slot): V1's forward writes them
  // forward
  const double *ev, *att_cg;  // V1
  double inv_avg;
  double *pf, *palpha;
  // reverse
  const double *psc, *dfc;
  double rc;
  double *ds, *dr;
};

// Pairs below which each filter and head of 16 slots has a wavefront of its
// own (SPLIT): one wavefront walks all their operands one after the other,
// and few pairs leave most SIMDs without one; with many, the hidden layers'
// copies and the reverse's sums cost more than the shorter walk gives.
// Whole evaluations without / with it (us, by pairs with the capacity's
// margin), shipped model: 22 atoms 317 / 286, 2,200 pairs 349 / 315, 4,700 371
// / 358, 6,200 370 / 362, 6,900 424 / 417, 10,300 392 / 410; F = 256: 22 atoms
// 691 / 623, 2,200 738 / 676, 4,700 772 / 792, 6,200 788 / 813.
template <int FT>
constexpr int kFewRows = FT == 8 ? 7500 : 3700;

// The sums of v[0..8) over the 16 lanes of a group: lane j ends with that of
// v[4 b3 + 2 b2 + b1], b its index's bits.  Half of the values go to the
// partner at each step: 8 exchanges where 8 separate sums take 32.
__device__ __forceinline__ double spread_sum8(const double (&v)[8], int j) {
  const bool b3 = j & 8, b2 = j & 4, b1 = j & 2;
  double u[4], w[2];
#pragma unroll
  for (int k = 0; k < 4; ++k) u[k] = (b3 ? v[k + 4] : v[k]) + dpp_f64<0x140, true>(b3 ? v[k] : v[k + 4]);
#pragma unroll
  for (int k = 0; k < 2; ++k) w[k] = (b2 ? u[k + 2] : u[k]) + dpp_f64<0x141, true>(b2 ? u[k] : u[k + 2]);
  const double x = (b1 ? w[1] : w[0]) + dpp_f64<0x4E, true>(b1 ? w[0] : w[1]);
  return x + dpp_f64<0xB1, true>(x);
}
// LDS values of one wavefront's lanes to its other lanes
__device__ __forceinline__ void wave_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// What both directions hold of their 16 slots: on the lanes (operands), pair
// p of lane j with its powers of t; on the accumulator rows, the pairs g + 4 r
// and their endpoints' rows at the lane's channels.
template <int FT, bool SPLIT>
struct RowsSlots {
  static constexpr int NH = FT / 2, F = 16 * FT, kWaves = SPLIT ? FT : 4;
  int lane, j, g, sub, wave, p, pp, ri;  // pp: p, or the bucket's first pair in the padding
  bool inside;
  v4d tp[2];
  int prow[4];  // -1: padding
  const double *ra[4], *rb[4];
  __device__ __forceinline__ bool init(const RowsArgs &A) {
    lane = threadIdx.x & 63;
    j = lane & 15;
    g = lane >> 4;
    sub = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    // consecutive slots on one XCD: a spatial block's buckets share its L2
    const int blk = xcd_block_active((*A.slots + (SPLIT ? 15 : 63)) / (SPLIT ? 16 : 64));
    wave = blk < 0 ? -1 : (SPLIT ? blk : blk * 4 + sub);
    if (!rint_slots(A.slots, A.order, A.pr, A.d, wave, j, g, p, ri, inside, tp)) return false;
    const int p0 = A.order[wave * 16];
    pp = p >= 0 ? p : p0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      prow[r] = A.order[wave * 16 + g + 4 * r];
      const int q = prow[r] >= 0 ? prow[r] : p0;
      ra[r] = A.qkv + std::size_t(A.pa[2 * q]) * 5 * F + 2 * j;
      rb[r] = A.qkv + std::size_t(A.pa[2 * q + 1]) * 5 * F + 2 * j;
    }
    return true;
  }
  // row item u of filter w and head hd: {q_a, k_b, q_b, k_a}[u % 4] of the
  // pairs g + 4 r, r = 2 (u / 4) and the next
  __device__ __forceinline__ v4d rows(int w, int hd, int u) const {
    const int t = u & 3, r = 2 * (u >> 2), off = (t & 1 ? (w ? 4 * F : F) : (w ? 3 * F : 0)) + 32 * hd;
    const bool at_a = t == 0 || t == 3;
    const v2d x = *reinterpret_cast<const v2d *>((at_a ? ra : rb)[r] + off);
    const v2d y = *reinterpret_cast<const v2d *>((at_a ? ra : rb)[r + 1] + off);
    return v4d{x[0], x[1], y[0], y[1]};
  }
};

// Pre-activations of hidden tile t (rows: features, columns: the 16 pairs)
template <int FT, bool V1>
__device__ __forceinline__ v4d rows_hidden(const double *e0, const double *eb0, int t, const double *s, int lane) {
  const v4d b = frag_load(eb0, t, lane);
  if constexpr (V1) {  // one operand per lane for both tiles
    const v4d e = frag_load(e0, 0, lane);
    return mfma(t ? e[1] : e[0], s[0], b);
  } else {
    const v4d e = frag_load(e0, t, lane);
    v4d h = mfma(e[0], s[0], b);
    if constexpr (FT > 8) h = mfma(e[1], s[1], h);
    return h;
  }
}

// Forward.  Per filter the hidden tiles silu(E0 s + e0), then per head its two
// output tiles (channels 2 j and 2 j + 1 on lane j, the pairs on the
// accumulator rows: the pairs' powers of t and their hidden tiles are the
// left operands, the interval's coefficient tile and E1 the right ones), and
// the endpoint rows against them to the logits of both directions, collected
// in LDS and written pair by pair.
template <int FT, bool SPLIT, bool V1>
__global__ __launch_bounds__(SPLIT ? 64 * FT : 256) __attribute__((amdgpu_waves_per_eu(SPLIT ? FT / 4 : 2))) void
k_rows_fwd(RowsArgs A) {
  using S_ = RowsSlots<FT, SPLIT>;
  constexpr int FHT = FT / 4, NH = S_::NH, F = S_::F, NT = 2 + FHT, NE = 2 * NT + 8, HEADS = SPLIT ? 1 : NH;
  constexpr bool SHARE = SPLIT && FHT > 2;  // hidden tiles formed once per 16 slots
  constexpr int kInv = 26;
  __shared__ double tab[256], logit[SPLIT ? 1 : 4][16][4 * NH + 2], inv[V1 ? S_::kWaves : 1][16][kInv];
  __shared__ v4d hid[2][SHARE ? FHT : 1][64];
  if (!SPLIT || threadIdx.x < 256) tab[threadIdx.x & 255] = A.exp2_256[threadIdx.x & 255];
  __syncthreads();
  S_ S;
  if (!S.init(A)) return;  // SPLIT: the whole block
  const int lane = S.lane, j = S.j, g = S.g, sub = S.sub;
  const int w0 = SPLIT ? sub / NH : 0, h0 = SPLIT ? sub % NH : 0;
  double s[V1 ? 1 : 4];
  if constexpr (V1) {
    // the equivariant invariants of degree slots 0..3: the endpoints' 24
    // channels two to a lane, then slot g of pair j from LDS
    const int a = A.pa[2 * S.pp], b = A.pa[2 * S.pp + 1];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int n = 64 * i + lane, q = n / 12, c = 2 * (n % 12);
      const v2d x = *reinterpret_cast<const v2d *>(A.ev + std::size_t(__shfl(a, q, 64)) * 24 + c);
      const v2d y = *reinterpret_cast<const v2d *>(A.ev + std::size_t(__shfl(b, q, 64)) * 24 + c);
      const v2d d = x - y, cg = *reinterpret_cast<const v2d *>(A.att_cg + c);
      *reinterpret_cast<v2d *>(&inv[sub][q][c]) = d * d * cg;
    }
    wave_lds();
    const SlotsV1 slot;
    s[0] = 0.0;
#pragma unroll
    for (int k = 0; k < 9; ++k)
      if (k < 2 * g + 3) s[0] += inv[sub][j][slot.off(g) + k];
    if (S.p >= 0 && (!SPLIT || sub == 0)) A.ps[4 * std::size_t(S.p) + g] = s[0];
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v) s[v] = g + 4 * v < NH ? A.ps[std::size_t(S.pp) * NH + g + 4 * v] : 0.0;
  }
  const v4d zero = v4d{0.0, 0.0, 0.0, 0.0};
  static_for<SPLIT ? 1 : 2>([&](auto wi) {
    const int w = w0 + decltype(wi)::value;
    const double *coef = A.rtab + (std::size_t(S.ri) * 2 + w) * FT * 2 * 256, *e1 = w ? A.e1[1] : A.e1[0];
    const double *e0 = w ? A.e0[1] : A.e0[0], *eb0 = w ? A.eb0[1] : A.eb0[0];
    auto ld = [&](auto si) -> v4d {
      constexpr int I = decltype(si)::value, u = I % NE;
      const int hd = h0 + I / NE;
      if constexpr (u < 2 * NT) {
        const int mt = 2 * hd + u / NT;
        if constexpr (u % NT < 2) return frag_load(coef, mt * 2 + u % NT, lane);
        else return frag_load(e1, mt * FHT + u % NT - 2, lane);
      } else {
        return S.rows(w, hd, u - 2 * NT);
      }
    };
    Stream<HEADS * NE, 8, decltype(ld)> st(ld);
    st.prime();
    v4d he[FHT];
    auto hidden = [&](int t) {
      v4d h = rows_hidden<FT, V1>(e0, eb0, t, s, lane);
#pragma unroll
      for (int r = 0; r < 4; ++r) h[r] = silu_tab_wide(h[r], tab);
      return h;
    };
    if constexpr (SHARE) {
      if (sub % NH < FHT) hid[w][sub % NH][lane] = hidden(sub % NH);
      __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < FHT; ++t) he[t] = SHARE ? hid[w][t][lane] : hidden(t);
    v4d o[2], hold;
    double sums[8];  // pairs g + 4 r: direction b -> a, then a -> b
    st.run([&](auto si, const v4d &v) {
      constexpr int I = decltype(si)::value, u = I % NE;
      const int hd = h0 + I / NE;
      if constexpr (u < 2 * NT) {
        constexpr int e = u / NT, c = u % NT;
        o[e] = mfma4(c < 2 ? S.tp[c & 1] : he[c < 2 ? 0 : c - 2], v, c == 0 ? zero : o[e]);
        if constexpr (u == 2 * NT - 1) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (S.prow[r] >= 0)
              __builtin_nontemporal_store(v2d{o[0][r], o[1][r]}, reinterpret_cast<v2d *>(
                  A.pf + std::size_t(S.prow[r]) * 2 * F + w * F + 32 * hd + 2 * j));
        }
      } else {
        constexpr int c = u - 2 * NT, t = c & 3, r = 2 * (c >> 2);
        if constexpr (t == 0 || t == 2) {
          hold = v;  // q_a: edge b -> a; q_b: edge a -> b
        } else {
          constexpr int k = (t == 3 ? 4 : 0) + r;
          const v4d qk = hold * v;
          sums[k] = qk[0] * o[0][r] + qk[1] * o[1][r];
          sums[k + 1] = qk[2] * o[0][r + 1] + qk[3] * o[1][r + 1];
        }
        if constexpr (c == 7) {
          const double x = spread_sum8(sums, j) * A.inv_avg;
          if (!(j & 1))
            logit[SPLIT ? 0 : sub][g + 2 * (j & 4) + 2 * (j & 2)][(j >> 3) * 2 * NH + w * NH + hd] = x;
        }
      }
    });
  });
  if constexpr (SPLIT) __syncthreads();
  else wave_lds();
  const double *l = &logit[SPLIT ? 0 : sub][0][0];
#pragma unroll
  for (int i = 0; i < (SPLIT ? 1 : 16 * 2 * NH / 64); ++i) {
    const int n = SPLIT ? int(threadIdx.x) : 64 * i + lane, q = n / (2 * NH), c = 2 * (n % (2 * NH));
    const int p = n < 16 * 2 * NH ? A.order[S.wave * 16 + q] : -1;
    if (p >= 0)
      *reinterpret_cast<v2d *>(A.palpha + std::size_t(p) * 4 * NH + c) =
          *reinterpret_cast<const v2d *>(l + q * (4 * NH + 2) + c);
  }
}

// Reverse.  Per filter and head df = s_in q_a k_b + s_out q_b k_a on the
// rows' lanes (the scalars from the node-major reverse's record), through LDS
// to the operand's layout (pairs on the lanes), then against E1^T (the
// spherical hidden layer's adjoint, on through silu' and E0^T to dE/ds) and
// the interval's slope tiles, whose sum over the powers of t is the radial
// branches' dE/dr.  A head's rows are taken in and its df stored while the
// MFMAs of the head before run.
template <int FT, bool SPLIT, bool V1>
__global__ __launch_bounds__(SPLIT ? 64 * FT : 256) __attribute__((amdgpu_waves_per_eu(SPLIT ? FT / 4 : 2))) void
k_rows_bwd(RowsArgs A) {
  using S_ = RowsSlots<FT, SPLIT>;
  constexpr int FHT = FT / 4, NH = S_::NH, NR = (NH + 3) / 4, HEADS = SPLIT ? 1 : NH;
  constexpr int M = 2 * (FHT + 2), PER = 8 + M, NS = HEADS * PER;  // stream: rows of head 0; rows of h + 1, MFMAs of h
  constexpr bool SHARE = SPLIT && FHT > 2;
  constexpr int kDf = 34, kSc = 4 * NH + 2;
  __shared__ double tab[256], dfl[S_::kWaves][16][kDf], scal[SPLIT ? 1 : 4][16][kSc];
  __shared__ double share[SPLIT ? FT : 1][NR + 1][64];
  __shared__ v4d prime[2][SHARE ? FHT : 1][64];
  if (!SPLIT || threadIdx.x < 256) tab[threadIdx.x & 255] = A.exp2_256[threadIdx.x & 255];
  __syncthreads();
  S_ S;
  if (!S.init(A)) return;  // SPLIT: the whole block
  const int lane = S.lane, j = S.j, g = S.g, sub = S.sub;
  const int w0 = SPLIT ? sub / NH : 0, h0 = SPLIT ? sub % NH : 0;
  // the record's scalars of filter w and head hd: the two directions'
  auto at_in = [](int w, int hd) { return V1 ? 4 * hd + 2 * w : w * NH + hd; };
  auto at_out = [](int w, int hd) { return V1 ? 4 * hd + 2 * w + 1 : 2 * NH + w * NH + hd; };
  double sc_in[4], sc_out[4];
  if constexpr (SPLIT) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const double *rec = A.psc + std::size_t(S.prow[r] >= 0 ? S.prow[r] : S.pp) * 4 * NH;
      sc_in[r] = rec[at_in(w0, h0)];
      sc_out[r] = rec[at_out(w0, h0)];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16 * 2 * NH / 64; ++i) {
      const int n = 64 * i + lane, q = n / (2 * NH), c = 2 * (n % (2 * NH));
      const int p = A.order[S.wave * 16 + q];
      v2d v = v2d{0.0, 0.0};
      if (p >= 0) v = *reinterpret_cast<const v2d *>(A.psc + std::size_t(p) * 4 * NH + c);
      *reinterpret_cast<v2d *>(&scal[sub][q][c]) = v;
    }
    wave_lds();
  }
  double s[V1 ? 1 : 4];
#pragma unroll
  for (int v = 0; v < (V1 ? 1 : 4); ++v) s[v] = g + 4 * v < NH ? A.ps[std::size_t(S.pp) * NH + g + 4 * v] : 0.0;
  const v4d zero = v4d{0.0, 0.0, 0.0, 0.0};
  v4d dsa = zero, accdr[2] = {zero, zero};
  static_for<SPLIT ? 1 : 2>([&](auto wi) {
    const int w = w0 + decltype(wi)::value;
    const double *slope = A.rtab + (std::size_t(S.ri) * 2 + w) * 2 * FT * 256, *e1t = w ? A.e1[1] : A.e1[0];
    const double *e0 = w ? A.e0[1] : A.e0[0], *eb0 = w ? A.eb0[1] : A.eb0[0], *e0t = w ? A.e0t[1] : A.e0t[0];
    v4d dh[FHT];
#pragma unroll
    for (int t = 0; t < FHT; ++t) dh[t] = zero;
    // entry I: head I / PER's MFMA operand (u >= 8), or a row item
    auto ld = [&](auto si) -> v4d {
      constexpr int I = decltype(si)::value, K = I - 8, H = K < 0 ? 0 : K / PER;
      constexpr int u = K < 0 ? I : (H == HEADS - 1 ? 8 + K % PER : K % PER);
      if constexpr (K < 0 || u < 8) {
        return S.rows(w, h0 + (K < 0 ? 0 : H + 1), u);
      } else {
        constexpr int q = (u - 8) % (FHT + 2);
        const int mt = 2 * (h0 + H) + (u - 8) / (FHT + 2);
        if constexpr (q < FHT) return frag_load(e1t, q * FT + mt, lane);
        else return frag_load(slope, (q - FHT) * FT + mt, lane);
      }
    };
    Stream<NS, 8, decltype(ld)> st(ld);
    st.prime();
    auto slope_of = [&](int t) {
      v4d pre = rows_hidden<FT, V1>(e0, eb0, t, s, lane);
#pragma unroll
      for (int r = 0; r < 4; ++r) pre[r] = silu_prime_tab_wide(pre[r], tab);
      return pre;
    };
    if constexpr (SHARE) {
      if (sub % NH < FHT) prime[w][sub % NH][lane] = slope_of(sub % NH);
    }
    v4d hold, df, next[2], bT[2];
    st.run([&](auto si, const v4d &v) {
      constexpr int I = decltype(si)::value, K = I - 8, H = K < 0 ? 0 : K / PER;
      constexpr int u = K < 0 ? I : (H == HEADS - 1 ? 8 + K % PER : K % PER);
      if constexpr (K < 0 || u < 8) {
        constexpr int t = u & 3, r = 2 * (u >> 2), hr = K < 0 ? 0 : H + 1;
        if constexpr (u == 0 && !SPLIT) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            sc_in[q] = scal[sub][g + 4 * q][at_in(w, hr)];
            sc_out[q] = scal[sub][g + 4 * q][at_out(w, hr)];
          }
        }
        if constexpr (t == 0 || t == 2) {
          hold = v;
        } else if constexpr (t == 1) {
          df = v4d{sc_in[r], sc_in[r], sc_in[r + 1], sc_in[r + 1]} * (hold * v);
        } else {
          df += v4d{sc_out[r], sc_out[r], sc_out[r + 1], sc_out[r + 1]} * (hold * v);
          *reinterpret_cast<v2d *>(&dfl[sub][g + 4 * r][2 * j]) = v2d{df[0], df[1]};
          *reinterpret_cast<v2d *>(&dfl[sub][g + 4 * r + 4][2 * j]) = v2d{df[2], df[3]};
        }
        if constexpr (u == 7) {
          wave_lds();
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const v2d x = *reinterpret_cast<const v2d *>(&dfl[sub][j][16 * q + 4 * g]);
            const v2d y = *reinterpret_cast<const v2d *>(&dfl[sub][j][16 * q + 4 * g + 2]);
            next[q] = v4d{x[0], x[1], y[0], y[1]};
          }
          wave_lds();
          if constexpr (K < 0) {
            bT[0] = next[0];
            bT[1] = next[1];
          }
        }
      } else {
        constexpr int q = (u - 8) % (FHT + 2), e = (u - 8) / (FHT + 2);
        if constexpr (q < FHT) dh[q] = mfma4(v, bT[e], dh[q]);
        else accdr[q - FHT] = mfma4(v, bT[e], accdr[q - FHT]);
        if constexpr (u == PER - 1) {
          bT[0] = next[0];
          bT[1] = next[1];
        }
      }
    });
    if constexpr (SHARE) __syncthreads();
#pragma unroll
    for (int t = 0; t < FHT; ++t) {
      dh[t] *= SHARE ? prime[w][t][lane] : slope_of(t);
      dsa = mfma4(frag_load(e0t, t, lane), dh[t], dsa);
    }
  });
  // dE/dr: sum over the powers of t (tile m, row g + 4 r: power 16 m + g + 4 r)
  double part = 0.0;
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) part += accdr[m][r] * S.tp[m][r];
  if constexpr (SPLIT) {  // the filters' and heads' shares, summed in wavefront order
#pragma unroll
    for (int r = 0; r < NR; ++r) share[sub][r][lane] = dsa[r];
    share[sub][NR][lane] = part;
    __syncthreads();
    if (sub != 0) return;
#pragma unroll
    for (int q = 1; q < FT; ++q) {
#pragma unroll
      for (int r = 0; r < NR; ++r) dsa[r] += share[q][r][lane];
      part += share[q][NR][lane];
    }
  }
  if (!S.inside) part = 0.0;
  part += __shfl_xor(part, 16, 64);
  part += __shfl_xor(part, 32, 64);
  if (S.p >= 0) {
#pragma unroll
    for (int r = 0; r < NR; ++r)
      if (g + 4 * r < NH) A.ds[std::size_t(S.p) * NH + g + 4 * r] = dsa[r];
    if (g == 0) {
      const double r = A.pr[S.p];
      double grad = part;
      if (r < A.rc) {
        const double t = r / A.rc;
        grad += A.dfc[S.p] * (-30.0 * t * t * (1.0 - t) * (1.0 - t) / A.rc);
      }
      A.dr[S.p] += grad;
    }
  }
}

// k_rows_fwd / k_rows_bwd over at most `slots_max` slots of fewer than `pairs`
// pairs
template <int FT, bool V1, bool FWD>
void launch_rows(hipStream_t s, int slots_max, int pairs, const RowsArgs &A) {
  auto go = [&](auto split) {
    constexpr bool SPLIT = decltype(split)::value;
    const dim3 grid(unsigned((slots_max + (SPLIT ? 15 : 63)) / (SPLIT ? 16 : 64))), block(SPLIT ? 64 * FT : 256);
    if constexpr (FWD) hipLaunchKernelGGL((k_rows_fwd<FT, SPLIT, V1>), grid, block, 0, s, A);
    else hipLaunchKernelGGL((k_rows_bwd<FT, SPLIT, V1>), grid, block, 0, s, A);
  };
  if (pairs < kFewRows<FT>) go(std::true_type{});
  else go(std::false_type{});
}

}  // namespace
}  // namespace so3lr_amd
