// The node side of an interaction block as fused fp64 MFMA kernels, shared by
// the v1 kernels (evaluator.hip) and the generic widths (generic.hip): the
// per-head projections, the post-attention chain with what follows it, and its
// reverse.  F = 16 NT features (NT = 8 or 16), NT / 2 heads and degree slots.
#pragma once

#include <type_traits>

#include "device_math.hpp"
#include "mfma_ops.hpp"
#include "model.hpp"

namespace so3lr_amd {
namespace {

// A lane's four channels 16 t + g + 4 r (r = 0..3, lane group g) of tile t of a
// node row: one 32-byte vector in the tile-transposed order (TO: fpos in
// evaluator.hip), four values in natural order.
template <bool TO>
__device__ __forceinline__ v4d row_load(const double *row, int t, int g) {
  if constexpr (TO) return *reinterpret_cast<const v4d *>(row + 16 * t + 4 * g);
  const double *r = row + 16 * t + g;
  return v4d{r[0], r[4], r[8], r[12]};
}
template <bool TO>
__device__ __forceinline__ void row_store(double *row, int t, int g, const v4d &v) {
  if constexpr (TO) {
    *reinterpret_cast<v4d *>(row + 16 * t + 4 * g) = v;
  } else {
    double *r = row + 16 * t + g;
    r[0] = v[0];
    r[4] = v[1];
    r[8] = v[2];
    r[12] = v[3];
  }
}

// Workgroups go to the 8 XCDs round-robin (block b on XCD b % 8).  Remapped
// so that each XCD walks one contiguous range of logical blocks: with nodes
// in spatial order, the neighbour rows a range gathers stay in its XCD's L2.
// A bijection of [0, gridDim.x) whatever the grid size.
__device__ __forceinline__ int xcd_block() {
#ifdef SO3LR_NO_XCD_MAP
  return blockIdx.x;
#endif
  const int G = gridDim.x, b = blockIdx.x;
  const int per = G >> 3, rem = G & 7, xcd = b & 7, i = b >> 3;
  return xcd * per + (xcd < rem ? xcd : rem) + i;
}
// xcd_block for a grid sized for an upper bound of the work: only the first A
// logical blocks have work (A <= gridDim.x, known on the device only), and
// they are spread evenly over the XCDs; -1 for a block with none.
__device__ __forceinline__ int xcd_block_active(int A) {
  const int b = blockIdx.x;
  const int per = A >> 3, rem = A & 7, xcd = b & 7, i = b >> 3;
  if (i >= per + (xcd < rem ? 1 : 0)) return -1;
  return xcd * per + (xcd < rem ? xcd : rem) + i;
}

// A node's wavefronts in the node-major kernels: W wavefronts share a node's
// incidence list in W runs, and the first adds the others' sums in run order.
// One wavefront per node reads its list serially (about 1 us per pair of
// partners, latency alone); with few nodes the chip is idle beside it, so the
// list is cut in 8 below kShare8 nodes and in 4 below kShare4.  Measured (us
// per evaluation at 1 / 2 / 4 / 8 wavefronts): 99 atoms 515 / 439 / 391 / 373,
// 375 atoms 502 / 438 / 409 / 397, 750 atoms 571 / 503 / 462 / 468, 1,764
// atoms 769 / 727 / 717 / 732, 3,000 atoms 929 / 958 / 931 / 961.
constexpr int kShare8 = 500, kShare4 = 2400;
template <class Launch>
void by_node_share(int N, Launch &&launch) {
  if (N < kShare8) launch(std::integral_constant<int, 8>{});
  else if (N < kShare4) launch(std::integral_constant<int, 4>{});
  else launch(std::integral_constant<int, 1>{});
}
template <int W>
struct NodeShare {
  static constexpr int kBlock = W > 4 ? 64 * W : 256, kNodes = kBlock / 64 / W;
  int n, c, beg, end;
  bool on, first;  // n < N; this wavefront writes the node's results
  // `cut`: a node's channels in that many slices, each with W wavefronts of
  // its own (c: this wavefront's slice; kNodes slices per block)
  __device__ __forceinline__ NodeShare(int N, const int *__restrict__ off, int cut = 1) {
    // the same in every lane: the node's offsets and rows are addressed by scalars
    const int wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), part = wv % W, u = xcd_block() * kNodes + wv / W;
    n = u / cut;
    c = u % cut;
    on = n < N;
    first = part == 0;
    if (on) {
      const int b = off[n], len = off[n + 1] - b;
      beg = b + len * part / W;
      end = b + len * (part + 1) / W;
    } else {
      beg = end = n = 0;
    }
  }
};
// v[0..M) summed over the node's wavefronts, in the first of them (every
// wavefront of the block calls this; lds: kBlock * M doubles)
template <int W, int M>
__device__ __forceinline__ void share_sum(double *lds, double (&v)[M]) {
  if constexpr (W > 1) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < M; ++k) lds[(wv * M + k) * 64 + lane] = v[k];
    __syncthreads();
    if (wv % W == 0) {
#pragma unroll
      for (int q = 1; q < W; ++q)
#pragma unroll
        for (int k = 0; k < M; ++k) v[k] += lds[((wv + q) * M + k) * 64 + lane];
    }
  }
}

// The degree slots of the v1 widths: degrees 1, 2, 3, 4, 24 channels.
struct SlotsV1 {
  __device__ __forceinline__ int E() const { return 24; }
  __device__ __forceinline__ int off(int s) const { return s == 0 ? 0 : (s == 1 ? 3 : (s == 2 ? 8 : (s == 3 ? 15 : 24))); }
  __device__ __forceinline__ int slot(int m) const { return degree_slot(m); }
};

// Block-diagonal projections: per head h, the 160 outputs (q k v q_ev k_ev,
// 32 each) depend on x[h*32 .. h*32+32).  Wp holds, per head, the permuted
// (160 x 32) matrix; out[n][w*F + h*32 + o].  One wavefront per 16 rows and
// head (blockIdx.y); stream: the two input chunks, then the 10 x 2 weight
// fragments (tile-major).
template <bool TO>
__global__ __launch_bounds__(256) void k_qkv_mfma(int rows, int F, const double *__restrict__ X,
                                                  const double *__restrict__ Wp, double *__restrict__ out) {
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
  const int w = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w * 16 >= rows) return;
  const int n = w * 16 + j;
  const bool valid = n < rows;
  const double *xr = X + std::size_t(valid ? n : rows - 1) * F;
  const int h = blockIdx.y;
  constexpr int PER_H = 2 + 20;
  auto load = [&](auto si) -> v4d {
    constexpr int s = decltype(si)::value;
    if constexpr (s < 2) return row_load<TO>(xr, 2 * h + s, g);
    else return wload(Wp + std::size_t(h) * 160 * 32, 2, (s - 2) / 2, (s - 2) % 2, lane);
  };
  Stream<PER_H, 4, decltype(load)> st(load);
  st.prime();
  const v4d zero = v4d{0, 0, 0, 0};
  v4d b[2] = {zero, zero}, acc;
  st.run([&](auto si, const v4d &wv) {
    constexpr int s = decltype(si)::value;
    if constexpr (s < 2) {
      b[s] = wv;
    } else {
      constexpr int mt = (s - 2) / 2, T = (s - 2) % 2;
      acc = mfma4(wv, b[T], T == 0 ? zero : acc);
      // tile mt is projection mt / 2, channels 32 h + 16 (mt % 2) + [0, 16)
      if constexpr (T == 1)
        if (valid) row_store<TO>(out + std::size_t(n) * 5 * F + (mt >> 1) * F, 2 * h + (mt & 1), g, acc);
    }
  });
}

// The post-attention node chain of one block with every activation in MFMA
// registers (kokkos_post_attention_block0.cpp:302-333):
//   n1 = LN1 row (its normalised values n1hat times the affine weights),
//   hpre = W1 silu(n1) + b1 (kept for the reverse), hid = silu(hpre),
//   p = n1 + W2 hid + b2,
//   t = Wint [p, inv(aev)] + bint, inv_s = sum_{m in s} aev_m^2 cg_m,
//   x' = LN2(p + t[0:F]) (statistics kept), ev' = aev (1 + gate[slot]),
//   gate s = t[F + s] (kept),
// then what reads x' next: the following block's q k v q_ev k_ev rows (TAIL
// 1), or the heads (TAIL 2): their hidden layer (HTC tiles; 0: H.HT) and the
// per-atom energy, raw charge and ratios.
//
// One workgroup of NT wavefronts per 16 atoms: wavefront w owns output tile
// w (16 of the F features) of every layer, and the layer inputs are
// exchanged through LDS in MFMA operand order (chunk T of lane l at
// buf[T][l]).  A tile of the chain is bound by its length (three dependent
// layers and two row normalisations, each wavefront streaming its own weight
// fragments from L2), so it is cut as short as the 16 x 16 tiles allow,
// kNodePF fragments in flight per wavefront.  The gate tile (one per slot: 4
// or 8 of 16 rows used) is formed from partial products, each wavefront
// taking its own chunk of p, summed through LDS in wavefront order.
// v1 widths: two wavefronts per tile, four output tiles each, and the
// projections, heads and row sums as launches of their own took 570 us per
// evaluation at 22 atoms, 716 at 99, 1,216 at 3,000, 2,326 for 512 packed
// molecules and 6.64 ms at 24,000; this form 443, 570, 1,046, 2,126 and 6.50.
// F = 256: one 64 x 128-tile GEMM per layer with row kernels between (19
// launches per block, 30-40 us each below a few thousand atoms) took 1,386 us
// at 22 atoms, 3,326 at 3,000 and 18.2 ms at 24,000; this form 783, 2,479 and
// 17.4.
struct NodeChainArgs {
  const double *m1p, *m1bp, *m2p, *m2bp, *intp, *intbp;  // MFMA operand order
  const double *int_cg, *ln1w, *ln1b, *ln2w, *ln2b;      // F-wide vectors in the rows' order
  double eps;
  int mode2;  // NormMode of the second position (RMSNorm, none: w = 1, b = 0 given)
};
// The heads: energy and charge units padded to HKT tiles each, Hirshfeld 4
// tiles (and the C6 ratio head 4).
struct HeadArgs {
  int HT, HKT;
  const double *w1p, *w1tp, *b1p;  // hidden layer (16 HT x F), its transpose and bias, MFMA operand order
  const double *ew2, *qw2, *hkey, *ckey;  // output rows (16 HKT, 16 HKT, 64 per element, 64), tile-transposed order
  const double *escale, *eshift, *qemb, *hvshift, *hkey_c, *ckey_c, *cvshift;  // per element
  double eb2, qb2;
  // the output row of tile t at the lane group's channels, for element z, and
  // the output it belongs to (0 energy, 1 charge, 2 Hirshfeld, 3 C6)
  __device__ __forceinline__ int output(int t) const {
    return t < HKT ? 0 : (t < 2 * HKT ? 1 : (t < 2 * HKT + 4 ? 2 : 3));
  }
  __device__ __forceinline__ v4d out_row(int t, int z, int g) const {
    const double *r = t < HKT ? ew2 + 16 * t
                              : (t < 2 * HKT ? qw2 + 16 * (t - HKT)
                                             : (t < 2 * HKT + 4 ? hkey + z * 64 + 16 * (t - 2 * HKT)
                                                                : ckey + z * 64 + 16 * (t - 2 * HKT - 4)));
    return *reinterpret_cast<const v4d *>(r + 4 * g);
  }
};
struct HeadOut {
  double *hhead;  // hidden pre-activations [N][16 HT], tile-transposed order
  double *eatom, *qraw, *heff, *hir, *c6eff, *c6r;
};
// Fragments in flight per wavefront, and wavefronts per SIMD (at NT = 8 two
// workgroups per CU): 6 and 4 measured best over sizes (4 and 4 within 0.3%;
// 8 and 4 spills; 8 or 12 and 2 cost 2% at 12,000 atoms and up).
constexpr int kNodePF = 6;

// sum over the four lane groups (every lane of a column ends with the total)
__device__ __forceinline__ double column_sum(double v) {
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}
// the NT wavefronts' values at one place, in wavefront order
template <int NT, int W>
__device__ __forceinline__ double wave_order_sum(const double (*part)[W], int at) {
  double s = part[0][at];
#pragma unroll
  for (int w = 1; w < NT; ++w) s += part[w][at];
  return s;
}
// sum over the channels of degree slot s: a_m b_m (cg_m)
template <class Slots>
__device__ __forceinline__ double slot_sum(const Slots &sl, int s, const double *a, const double *b, const double *cg) {
  const int lo = sl.off(s), hi = sl.off(s + 1);
  double v = 0.0;
  for (int m = lo; m < hi; ++m) v += cg ? a[m] * b[m] * cg[m] : a[m] * b[m];
  return v;
}

struct NodeFwdArgs {
  int N;
  const double *n1hat, *aev;
  NodeChainArgs A;
  HeadArgs H;
  const double *qkvp;  // TAIL 1: the next block's projections
  const int *z;
  double *hpre, *gates, *xout, *evout, *pre2hat, *pre2is, *qkv;
  HeadOut O;
};
template <int NT, bool TO, int TAIL, int HTC, class Slots>
__global__ __launch_bounds__(64 * NT, 4) void k_node_fwd(NodeFwdArgs P, Slots sl) {
  constexpr int F = 16 * NT, NH = NT / 2, NS = NH / 4;  // NS slots per lane group
  constexpr int NU = (HTC + NT - 1) / NT;               // heads' tiles per wavefront
  const NodeChainArgs &A = P.A;
  const HeadArgs &H = P.H;
  __shared__ v4d bufA[NT][64], bufB[NT][64];
  __shared__ double gpart[NT][64 * NS], st1[NT][16], st2[NT][16];
  __shared__ double hsum[TAIL == 2 ? NT : 1][64];
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4, w = threadIdx.x >> 6;
  // every wavefront runs to the end (the barriers); rows beyond N are clamped
  const int n = blockIdx.x * 16 + j;
  const bool valid = n < P.N;
  const std::size_t nn = std::size_t(valid ? n : P.N - 1);
  const int E = sl.E();
  const double *aer = P.aev + nn * E;
  // the stream of this wavefront
  constexpr int L1 = 3, L2 = L1 + 1 + NT, G = L2 + 1 + NT, L3 = G + 3, LN = L3 + NT + 2, TL = LN + 2;
  constexpr int NE = TL + (TAIL == 1 ? 10 : TAIL == 2 ? NU * (NT + 1) : 0);
  const int head = w >> 1;  // TAIL 1: this wavefront's head and half of its ten projection tiles
  auto load = [&](auto si) -> v4d {
    constexpr int s = decltype(si)::value;
    if constexpr (s == 0) return row_load<TO>(P.n1hat + nn * F, w, g);
    else if constexpr (s == 1) return row_load<TO>(A.ln1w, w, g);
    else if constexpr (s == 2) return row_load<TO>(A.ln1b, w, g);
    else if constexpr (s == L1) return frag_load(A.m1bp, w, lane);
    else if constexpr (s < L2) return wload(A.m1p, NT, w, s - L1 - 1, lane);
    else if constexpr (s == L2) return frag_load(A.m2bp, w, lane);
    else if constexpr (s < G) return wload(A.m2p, NT, w, s - L2 - 1, lane);
    else if constexpr (s == G) return wload(A.intp, NT + 1, NT, w, lane);
    else if constexpr (s == G + 1) return wload(A.intp, NT + 1, NT, NT, lane);
    else if constexpr (s == G + 2) return frag_load(A.intbp, NT, lane);
    else if constexpr (s == L3) return frag_load(A.intbp, w, lane);
    else if constexpr (s < LN) return wload(A.intp, NT + 1, w, s - L3 - 1, lane);
    else if constexpr (s == LN) return row_load<TO>(A.ln2w, w, g);
    else if constexpr (s == LN + 1) return row_load<TO>(A.ln2b, w, g);
    else if constexpr (TAIL == 1) {
      constexpr int T = (s - TL) / 5, q = (s - TL) % 5;
      return wload(P.qkvp + std::size_t(head) * 160 * 32, 2, 5 * (w & 1) + q, T, lane);
    } else {
      constexpr int u = (s - TL) / (NT + 1), e = (s - TL) % (NT + 1);
      const int t = w + NT * u < HTC ? w + NT * u : w;  // past the last tile: a valid address, not used
      if constexpr (e == 0) return frag_load(H.b1p, t, lane);
      else return wload(H.w1p, NT, t, e - 1, lane);
    }
  };
  Stream<NE, kNodePF, decltype(load)> st(load);
  st.prime();
  double inv[NS];
#pragma unroll
  for (int v = 0; v < NS; ++v) inv[v] = slot_sum(sl, g + 4 * v, aer, aer, A.int_cg);
  const v4d zero = v4d{0.0, 0.0, 0.0, 0.0};
  v4d n1, lw, p, acc, gp, pb, hh, tacc[5];
  double mean = 0.0, hs[4] = {0.0, 0.0, 0.0, 0.0};
  // a finished hidden tile of the heads: kept, and its share of its output
  auto head_tile = [&](int t, const v4d &pre) {
    if (valid) row_store<true>(P.O.hhead + nn * (16 * H.HT), t, g, pre);
    const v4d r = H.out_row(t, P.z[nn], g);
    const double v = (r[0] * silu(pre[0]) + r[1] * silu(pre[1])) + (r[2] * silu(pre[2]) + r[3] * silu(pre[3]));
    const int o = H.output(t);
#pragma unroll
    for (int k = 0; k < 4; ++k) hs[k] += o == k ? v : 0.0;
  };
  st.run([&](auto si, const v4d &wv) {
    constexpr int s = decltype(si)::value;
    if constexpr (s == 0) {
      n1 = wv;
    } else if constexpr (s == 1) {
      lw = wv;
    } else if constexpr (s == 2) {
      v4d a;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        n1[r] = n1[r] * lw[r] + wv[r];
        a[r] = silu(n1[r]);
      }
      bufA[w][lane] = a;
      __syncthreads();
    } else if constexpr (s == L1 || s == L2 || s == L3) {
      acc = wv;
    } else if constexpr (s < L2) {
      acc = mfma4(wv, bufA[s - L1 - 1][lane], acc);
      if constexpr (s == L2 - 1) {
        if (valid) row_store<TO>(P.hpre + nn * F, w, g, acc);
        v4d a;
#pragma unroll
        for (int r = 0; r < 4; ++r) a[r] = silu(acc[r]);
        bufB[w][lane] = a;
        __syncthreads();
      }
    } else if constexpr (s < G) {
      acc = mfma4(wv, bufB[s - L2 - 1][lane], acc);
      if constexpr (s == G - 1) {
        p = n1 + acc;
        bufA[w][lane] = p;  // every wavefront has read the MLP input (the barrier above)
      }
    } else if constexpr (s == G) {
      gp = mfma4(wv, p, zero);
    } else if constexpr (s == G + 1) {
      if (w == 0) {
#pragma unroll
        for (int v = 0; v < NS; ++v) gp = mfma(wv[v], inv[v], gp);
      }
    } else if constexpr (s == G + 2) {
#pragma unroll
      for (int v = 0; v < NS; ++v) gpart[w][64 * v + lane] = w == 0 ? gp[v] + wv[v] : gp[v];
      __syncthreads();
    } else if constexpr (s < LN - 1) {
      acc = mfma4(wv, bufA[s - L3 - 1][lane], acc);
    } else if constexpr (s == LN - 1) {
      // the invariants: K rows F + slot, zero beyond
#pragma unroll
      for (int v = 0; v < NS; ++v) acc = mfma(wv[v], inv[v], acc);
      // LayerNorm 2 of p + t over the row, the tiles' sums combined in LDS
      pb = p + acc;
      const double sum = column_sum((pb[0] + pb[1]) + (pb[2] + pb[3]));
      if (g == 0) st1[w][j] = sum;
      __syncthreads();
      mean = A.mode2 == 0 ? wave_order_sum<NT>(st1, j) / F : 0.0;
      double var = 0.0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double d = pb[r] - mean;
        var += d * d;
      }
      var = column_sum(var);
      if (g == 0) st2[w][j] = var;
      __syncthreads();
      const double is = A.mode2 == 2 ? 1.0 : 1.0 / sqrt(wave_order_sum<NT>(st2, j) / F + A.eps);
#pragma unroll
      for (int r = 0; r < 4; ++r) hh[r] = (pb[r] - mean) * is;
      if (valid) {
        row_store<TO>(P.pre2hat + nn * F, w, g, hh);
        if (w == 0 && g == 0) P.pre2is[nn] = is;
        auto gate = [&](int slot) { return wave_order_sum<NT>(gpart, 64 * (slot >> 2) + 16 * (slot & 3) + j); };
        for (int m = g + 4 * w; m < E; m += 4 * NT)  // ev' = aev (1 + gate[slot])
          P.evout[nn * E + m] = aer[m] * (1.0 + gate(sl.slot(m)));
        if (w >= NT - NS) {
          const int slot = g + 4 * (w - (NT - NS));
          P.gates[nn * NH + slot] = gate(slot);
        }
      }
    } else if constexpr (s == LN) {
      lw = wv;
    } else if constexpr (s == LN + 1) {
      v4d x;
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = hh[r] * lw[r] + wv[r];
      if constexpr (TAIL < 2) {
        if (valid) row_store<TO>(P.xout + nn * F, w, g, x);
      }
      if constexpr (TAIL > 0) {
        bufB[w][lane] = x;  // every wavefront has read the MLP-2 input
        __syncthreads();
      }
    } else if constexpr (TAIL == 1) {
      constexpr int T = (s - TL) / 5, q = (s - TL) % 5;
      tacc[q] = mfma4(wv, bufB[2 * head + T][lane], T == 0 ? zero : tacc[q]);
      if constexpr (T == 1) {
        // tile mt = 5 (w & 1) + q is projection mt / 2, channels 32 head +
        // 16 (mt % 2) + [0, 16) of it
        const int mt = 5 * (w & 1) + q;
        if (valid) row_store<TO>(P.qkv + nn * 5 * F + (mt >> 1) * F, 2 * head + (mt & 1), g, tacc[q]);
      }
    } else {
      constexpr int u = (s - TL) / (NT + 1), e = (s - TL) % (NT + 1);
      if constexpr (e == 0) acc = wv;
      else acc = mfma4(wv, bufB[e - 1][lane], acc);
      if constexpr (e == NT)
        if (w + NT * u < HTC) head_tile(w + NT * u, acc);
    }
  });
  if constexpr (TAIL == 2) {
    if constexpr (HTC == 0) {
      for (int t = w; t < H.HT; t += NT) {
        auto frag = [&](auto si) -> v4d {
          constexpr int s = decltype(si)::value;
          if constexpr (s == 0) return frag_load(H.b1p, t, lane);
          else return wload(H.w1p, NT, t, s - 1, lane);
        };
        Stream<NT + 1, kNodePF, decltype(frag)> hst(frag);
        hst.prime();
        hst.run([&](auto si, const v4d &wv) {
          constexpr int s = decltype(si)::value;
          if constexpr (s == 0) acc = wv;
          else acc = mfma4(wv, bufB[s - 1][lane], acc);
        });
        head_tile(t, acc);
      }
    }
    // per-atom energy, raw charge, Hirshfeld (and C6) logit and ratio
    // (kokkos_output_heads.cpp:108-180,341-451)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double v = column_sum(hs[k]);
      if (g == k) hsum[w][lane] = v;
    }
    __syncthreads();
    if (w == 0 && valid) {
      const int zz = P.z[nn];
      const double v = wave_order_sum<NT>(hsum, lane);
      if (g == 0) {
        P.O.eatom[nn] = (v + H.eb2) * H.escale[zz - 1] + H.eshift[zz - 1];
      } else if (g == 1) {
        P.O.qraw[nn] = v + H.qb2 + H.qemb[zz];
      } else if (g == 2) {
        // logit q_emb[z] . (W2 a + b2), contracted through the element's row
        // u[z] = W2^T q_emb[z]; sqrt(64) = 8
        const double ef = H.hvshift[zz] + (H.hkey_c[zz] + v) / 8.0;
        P.O.heff[nn] = ef;
        P.O.hir[nn] = fabs(ef);
      } else if (H.ckey) {
        const double ce = H.cvshift[zz] + (H.ckey_c[zz] + v) / 8.0;
        P.O.c6eff[nn] = ce;
        P.O.c6r[nn] = fabs(ce);
      }
    }
  }
}

// Reverse of the node chain, the adjoints in MFMA registers
// (kokkos_post_attention_reverse.cpp:328-449), starting from the adjoint gx of
// the block's output x':
//   SRC 0 (the last block): the heads' reverse, seeds energy 1, charge dE/dq
//     - mean, Hirshfeld dE/dh (and C6 dE/dc) through the hidden layer
//     (kokkos_output_heads.cpp:493-581);
//   SRC 1: the projections' reverse of the block above, gx = scale (base +
//     sum_w W_w^T dqkv_w), base its attention-residual adjoint (gainv, which
//     this kernel then overwrites row by row with its own).
// Then
//   LayerNorm 2 reverse: d = LN2^T gx, the adjoint of p and of t[0:F];
//   t[F + s] (gates): sum_{m in s} gev_m aev_m; aev: gev (1 + gate);
//   interaction reverse: gcat = Wint^T gt; p += gcat[0:F];
//   aev += 2 aev cg gcat[F + slot];
//   MLP reverse: ghid = (W2^T p) silu'(hpre), gact = W1^T ghid;
//   LayerNorm 1 reverse of g = p + gact silu'(n1): the adjoint of the
//   attention residual, gainv.
// NT wavefronts per 16 atoms as in k_node_fwd.  gev null: zero (the last
// block's equivariant output is not read).  gainv and gqkv are in the
// tile-transposed order when TO.
struct NodeChainBwdArgs {
  const double *inttp, *m2tp, *m1tp;          // MFMA operand order (transposes)
  const double *int_cg, *ln1w, *ln1b, *ln2w;  // F-wide vectors in the rows' order
  int mode1, mode2;  // NormMode of the two positions: RMSNorm drops the mean term, none both
};
struct HeadSeeds {
  const double *hhead, *qseed, *dh, *heff, *dc, *c6eff;
};
struct NodeBwdArgs {
  int N;
  const double *gqkv, *qkvtp;
  double scale;
  HeadArgs H;
  HeadSeeds S;
  const int *z;
  const double *gev, *gates, *aev, *pre2hat, *pre2is, *hpre, *n1hat, *n1is;
  NodeChainBwdArgs A;
  double *gainv, *gaev;
};
template <int NT, bool TO, int SRC, int HTC, class Slots>
__global__ __launch_bounds__(64 * NT, 4) void k_node_bwd(NodeBwdArgs P, Slots sl) {
  constexpr int F = 16 * NT, NH = NT / 2, NS = NH / 4;
  const NodeChainBwdArgs &A = P.A;
  const HeadArgs &H = P.H;
  __shared__ v4d buf[HTC > 2 * NT ? HTC : 2 * NT][64];  // chunks 0.. and NT..: the two layer-input buffers
  __shared__ double gpart[NT][64 * NS], st[4][NT][16];
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4, w = threadIdx.x >> 6;
  const int n = blockIdx.x * 16 + j;
  const bool valid = n < P.N;
  const std::size_t nn = std::size_t(valid ? n : P.N - 1);
  const int E = sl.E();
  const int head = w >> 1;
  constexpr int X = SRC == 0 ? HTC : 21;  // entries of gx
  constexpr int G = X + 2, LB = G + 2, L2 = LB + NT + 1, L1 = L2 + NT + 1, LN = L1 + NT, NE = LN + 3;
  auto load = [&](auto si) -> v4d {
    constexpr int s = decltype(si)::value;
    if constexpr (s < X) {
      if constexpr (SRC == 0) return wload(H.w1tp, HTC, w, s, lane);
      else if constexpr (s == 20) return row_load<TO>(P.gainv + nn * F, w, g);
      else if constexpr ((s & 1) == 0) {
        // K entries of chunk T: projection T / 2, channels 32 head + 16 (T % 2) + [0, 16)
        constexpr int T = s / 2;
        return row_load<TO>(P.gqkv + nn * 5 * F + (T >> 1) * F, 2 * head + (T & 1), g);
      } else {
        return wload(P.qkvtp + std::size_t(head) * 32 * 160, 10, w & 1, s / 2, lane);
      }
    } else if constexpr (s == X) return row_load<TO>(A.ln2w, w, g);
    else if constexpr (s == X + 1) return row_load<TO>(P.pre2hat + nn * F, w, g);
    else if constexpr (s == G) return wload(A.inttp, NT + 1, NT, w, lane);
    else if constexpr (s == G + 1) return wload(A.inttp, NT + 1, NT, NT, lane);
    else if constexpr (s < L2) return wload(A.inttp, NT + 1, w, s - LB, lane);
    else if constexpr (s < L1 - 1) return wload(A.m2tp, NT, w, s - L2, lane);
    else if constexpr (s == L1 - 1) return row_load<TO>(P.hpre + nn * F, w, g);
    else if constexpr (s < LN) return wload(A.m1tp, NT, w, s - L1, lane);
    else if constexpr (s == LN) return row_load<TO>(P.n1hat + nn * F, w, g);
    else if constexpr (s == LN + 1) return row_load<TO>(A.ln1w, w, g);
    else return row_load<TO>(A.ln1b, w, g);
  };
  Stream<NE, kNodePF, decltype(load)> stream(load);
  stream.prime();

  const double *ger = P.gev ? P.gev + nn * E : nullptr, *aer = P.aev + nn * E;
  double gsum[NS];
#pragma unroll
  for (int v = 0; v < NS; ++v) gsum[v] = ger ? slot_sum(sl, g + 4 * v, ger, aer, nullptr) : 0.0;
  const double is2 = P.pre2is[nn], is1 = P.n1is[nn];
  const v4d zero = v4d{0.0, 0.0, 0.0, 0.0};
  v4d acc = zero, hold, d, hat, p, gp, n1;
  if constexpr (SRC == 0) {
    // the adjoints of the heads' hidden pre-activations, tile t
    const int zz = P.z[nn];
    const HeadSeeds &S = P.S;
    double seed[4] = {H.escale[zz - 1], S.qseed[nn], 0.0, 0.0};
    const double ef = S.heff[nn];
    seed[2] = S.dh[nn] * (ef > 0.0 ? 1.0 : (ef < 0.0 ? -1.0 : 0.0)) / 8.0;
    if (H.ckey) {
      const double ce = S.c6eff[nn];
      seed[3] = S.dc[nn] * (ce > 0.0 ? 1.0 : (ce < 0.0 ? -1.0 : 0.0)) / 8.0;
    }
    auto adjoint = [&](int t) {
      const int o = H.output(t);
      const double sd = o == 0 ? seed[0] : (o == 1 ? seed[1] : (o == 2 ? seed[2] : seed[3]));
      const v4d r = H.out_row(t, zz, g), pre = row_load<true>(S.hhead + nn * (16 * H.HT), t, g);
      v4d out;
#pragma unroll
      for (int q = 0; q < 4; ++q) out[q] = sd * r[q] * silu_prime(pre[q]);
      return out;
    };
    if constexpr (HTC > 0) {
#pragma unroll
      for (int u = 0; u < (HTC + NT - 1) / NT; ++u)
        if (w + NT * u < HTC) buf[w + NT * u][lane] = adjoint(w + NT * u);
      __syncthreads();
    } else {
      // NT tiles at a time through LDS
      for (int base = 0; base < H.HT; base += NT) {
        if (base + w < H.HT) buf[w][lane] = adjoint(base + w);
        __syncthreads();
        const int m = min(NT, H.HT - base);
        for (int i = 0; i < m; ++i) acc = mfma4(wload(H.w1tp, H.HT, w, base + i, lane), buf[i][lane], acc);
        __syncthreads();
      }
    }
  }
  stream.run([&](auto si, const v4d &wv) {
    constexpr int s = decltype(si)::value;
    if constexpr (s < X) {
      if constexpr (SRC == 0) {
        acc = mfma4(wv, buf[s][lane], acc);
      } else if constexpr (s == 20) {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = P.scale * (wv[r] + acc[r]);
      } else if constexpr ((s & 1) == 0) {
        hold = wv;
      } else {
        acc = mfma4(wv, hold, acc);
      }
    } else if constexpr (s == X) {
#pragma unroll
      for (int r = 0; r < 4; ++r) d[r] = acc[r] * wv[r];
    } else if constexpr (s == X + 1) {
      // LayerNorm 2 reverse; the adjoint of p and t[0:F] into LDS
      const double a = column_sum((d[0] + d[1]) + (d[2] + d[3]));
      const double b = column_sum((d[0] * wv[0] + d[1] * wv[1]) + (d[2] * wv[2] + d[3] * wv[3]));
      if (g == 0) {
        st[0][w][j] = a;
        st[1][w][j] = b;
      }
      __syncthreads();
      const double tm = A.mode2 == 0 ? wave_order_sum<NT>(st[0], j) / F : 0.0;
      const double tx = A.mode2 == 2 ? 0.0 : wave_order_sum<NT>(st[1], j) / F;
#pragma unroll
      for (int r = 0; r < 4; ++r) d[r] = is2 * (d[r] - tm - wv[r] * tx);
      buf[w][lane] = d;
    } else if constexpr (s == G) {
      gp = mfma4(wv, d, zero);  // this chunk's share of the gate rows of gcat
    } else if constexpr (s == G + 1) {
      if (w == 0) {
#pragma unroll
        for (int v = 0; v < NS; ++v) gp = mfma(wv[v], gsum[v], gp);
      }
#pragma unroll
      for (int v = 0; v < NS; ++v) gpart[w][64 * v + lane] = gp[v];
      __syncthreads();
    } else if constexpr (s < L2) {
      // gcat = Wint^T [d, gate adjoints]
      if constexpr (s - LB < NT) {
        acc = mfma4(wv, buf[s - LB][lane], s == LB ? zero : acc);
      } else {
#pragma unroll
        for (int v = 0; v < NS; ++v) acc = mfma(wv[v], gsum[v], acc);
        p = d + acc;
        buf[NT + w][lane] = p;
        __syncthreads();
      }
    } else if constexpr (s < L1 - 1) {
      acc = mfma4(wv, buf[NT + s - L2][lane], s == L2 ? zero : acc);  // W2^T p
    } else if constexpr (s == L1 - 1) {
      v4d a;
#pragma unroll
      for (int r = 0; r < 4; ++r) a[r] = acc[r] * silu_prime(wv[r]);
      buf[w][lane] = a;  // every wavefront has read d
      __syncthreads();
    } else if constexpr (s < LN) {
      acc = mfma4(wv, buf[s - L1][lane], s == L1 ? zero : acc);  // W1^T ghid
    } else if constexpr (s == LN) {
      hat = wv;
    } else if constexpr (s == LN + 1) {
      hold = wv;
    } else {
      // g = p + gact silu'(n1), then LayerNorm 1 reverse
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        n1[r] = hat[r] * hold[r] + wv[r];
        acc[r] = (p[r] + acc[r] * silu_prime(n1[r])) * hold[r];
      }
      const double a = column_sum((acc[0] + acc[1]) + (acc[2] + acc[3]));
      const double b = column_sum((acc[0] * hat[0] + acc[1] * hat[1]) + (acc[2] * hat[2] + acc[3] * hat[3]));
      if (g == 0) {
        st[2][w][j] = a;
        st[3][w][j] = b;
      }
      __syncthreads();
      const double tm = A.mode1 == 0 ? wave_order_sum<NT>(st[2], j) / F : 0.0;
      const double tx = A.mode1 == 2 ? 0.0 : wave_order_sum<NT>(st[3], j) / F;
      if (valid) {
        v4d out;
#pragma unroll
        for (int r = 0; r < 4; ++r) out[r] = is1 * (acc[r] - tm - hat[r] * tx);
        row_store<TO>(P.gainv + nn * F, w, g, out);
        for (int m = g + 4 * w; m < E; m += 4 * NT) {
          // aev: gev (1 + gate) + 2 aev cg gcat[F + slot]
          const int slot = sl.slot(m);
          const double gc = wave_order_sum<NT>(gpart, 64 * (slot >> 2) + 16 * (slot & 3) + j);
          const double e = ger ? ger[m] * (1.0 + P.gates[nn * NH + slot]) : 0.0;
          P.gaev[nn * E + m] = e + gc * 2.0 * aer[m] * A.int_cg[m];
        }
      }
    }
  });
}

}  // namespace
}  // namespace so3lr_amd
