// Jacobi-preconditioned CG of one system in two or three launches per
// iteration.
//
// An iteration of a system of up to a few hundred thousand nodes is bound by
// its launches and the dependent loads inside them, not by bytes: at 46^3
// nodes (FP64) the form of seven launches (direction, row dots, stencil, row
// scatter and alpha, update, rho) spent 28 us per iteration on 6 MB of
// vectors.  What is merged here:
//   * the one-workgroup reductions: every workgroup of the next launch sums
//     the few hundred partials itself, all in the same order, so all agree;
//   * the data term: nodes with data rows hold their row of G = A^T W^2 A
//     (k_pcg_gram_build), so it is one gather from the direction instead of a
//     gather, a kernel boundary and a scatter; its workgroups run beside the
//     direction's (k_pcg_dir) or the stencil's (k_pcg_tile), and the update
//     adds the compact result where a node's bit is set;
//   * on grids where it pays (see pcg_tiles), the direction itself: a
//     workgroup of k_pcg_tile forms it for its tile and halo in LDS and
//     applies the regulariser there.
// The direction alternates between two buffers, because its neighbours'
// old values are still being read while the new ones are written.
#pragma once

namespace lsamd {

constexpr int kGramCap = 32;       // most entries of a node's Gram row (27 for rows of one cell)
constexpr int kGramLanes = 8;      // threads per row, two or four entries each
// more data nodes keep the row form in any case: the node rows of this many take
// 192 MB in FP64, 128 MB in FP32 and 256 MB in both
constexpr int64_t kGramNodesMax = 500000;
constexpr int kPcgBlocks = 2048;   // partials of the vector kernels
constexpr int kPcgPartMax = 2048;  // operator partials that every workgroup sums itself

// workgroups of the vector kernels: 16 bytes of each vector per thread, more
// trips only beyond kPcgBlocks
inline int pcg_blocks(int64_t n, size_t elem) {
  const int64_t b = ceil_div(n, VB * (int64_t)(16 / elem));
  return (int)(b < kPcgBlocks ? b : kPcgBlocks);
}

// Data term by node: node[d] ascending; row d in entries [W d, W d + W), W = 16
// or 32, padded with zeros on the node itself, so that its threads need no
// length before they load.  mask[w]: which of the nodes 64 w .. 64 w + 63 are listed,
// base[w]: how many are listed before them.
struct GramDev {
  int64_t ndn;
  const int32_t* node;
  const int32_t* col;
  const void* val;  // T
  const uint64_t* mask;
  const int32_t* base;
};

// one thread per data node: its distinct columns in order of appearance and
// the sums of w^2 a_i a_j, in rows of `width` (col, v64 and v32: those given);
// over[0] when a row needs more than kGramCap, over[1] when one needs more than
// half of that
__global__ __launch_bounds__(64) void k_pcg_gram_build(RowsDev R, const double* __restrict__ coef,
                                                       const double* __restrict__ w2, int width,
                                                       int32_t* __restrict__ col,
                                                       double* __restrict__ v64,
                                                       float* __restrict__ v32, int* over) {
  __shared__ int32_t lc[kGramCap][64];
  __shared__ double lv[kGramCap][64];
  const int t = threadIdx.x;
  const int64_t d = (int64_t)blockIdx.x * 64 + t;
  if (d >= R.ndn) return;
  int m = 0;
  for (int64_t s = R.seg_ptr[d]; s < R.seg_ptr[d + 1]; ++s) {
    const int64_t r = R.seg_row[s];
    const double a = w2[r] * coef[R.seg_entry[s]];
    for (int64_t e = R.row_ptr[r]; e < R.row_ptr[r + 1]; ++e) {
      const int32_t c = R.cols[e];
      int k = 0;
      while (k < m && lc[k][t] != c) ++k;
      if (k == m) {
        if (m == kGramCap) {
          over[0] = 1;
          return;
        }
        lc[k][t] = c;
        lv[k][t] = 0.0;
        ++m;
      }
      lv[k][t] += a * coef[e];
    }
  }
  if (m > kGramCap / 2) over[1] = 1;
  const int32_t self = R.dnode[d];
  for (int k = 0; k < width; ++k) {
    const double v = k < m ? lv[k][t] : 0.0;
    if (col) col[d * width + k] = k < m ? lc[k][t] : self;
    if (v64) v64[d * width + k] = v;
    if (v32) v32[d * width + k] = (float)v;
  }
}

// mask and (where given) base of the words of 64 nodes (node ids ascending)
__global__ void k_pcg_gram_mask(const int32_t* __restrict__ node, int64_t ndn, int64_t nw,
                                uint64_t* __restrict__ mask, int32_t* __restrict__ base) {
  const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= nw) return;
  int64_t lo = 0, hi = ndn;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (node[mid] < 64 * w)
      lo = mid + 1;
    else
      hi = mid;
  }
  if (base) base[w] = (int32_t)lo;
  uint64_t b = 0;
  for (; lo < ndn && node[lo] < 64 * w + 64; ++lo) b |= 1ull << (node[lo] - 64 * w);
  mask[w] = b;
}

// sum of n partials in a fixed order, in every thread of the workgroup
__device__ inline double pcg_total(const double* __restrict__ part, int n, double* sh) {
  double v = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) v += part[i];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  v = wave_sum(v);
  if (lane == 0) sh[wid] = v;
  __syncthreads();
  double t = 0.0;
  const int nw = (int)(blockDim.x >> 6);
  for (int i = 0; i < nw; ++i) t += sh[i];
  __syncthreads();
  return t;
}

// Start of an iteration, in every workgroup of its first launch: rho from the
// previous update's partials, the stopping test, beta.  `par`, the parity of
// the iteration, picks the slots written here; the other ones hold the
// previous iteration's.  False: stop (workgroup 0 records it).  Callers load
// what they can before; a solve that is done finds out here, with the rest.
template <typename T>
__device__ inline bool pcg_begin(const double* __restrict__ part_r, int nr, CgCtl* ctl, int par,
                                 double* sh, int* first, T* beta) {
  const int done = ctl->done, it = ctl->its[1 - par], maxiter = ctl->maxiter;
  const double thr = ctl->thr, prev = ctl->rs[1 - par];
  const double rho = pcg_total(part_r, nr, sh);
  if (done) return false;
  const int conv = sqrt(rho) < thr;
  const bool stop = conv || it >= maxiter;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (stop) {
      ctl->rho = rho;
      ctl->iter = it;
      ctl->converged = conv;
      ctl->done = 1;
    } else {
      ctl->rs[par] = rho;
      ctl->its[par] = it + 1;
    }
  }
  *first = it == 0;
  *beta = *first ? (T)0 : (T)(rho / prev);
  return !stop;
}

// one node of the direction
template <typename T>
__device__ inline T pcg_p(T r, T minv, T po, int first, T beta) {
  const T z = minv * r;
  return first ? z : z + beta * po;
}

// Data term of one node by kGramLanes neighbouring threads, W / kGramLanes
// entries each; r, minv and the old direction gathered before beta is known (load),
// the row's product after it (value; the node's share of p.Gp).
template <typename T, int W>
struct PcgGram {
  static constexpr int kE = W / kGramLanes;
  typedef int32_t cols_t __attribute__((ext_vector_type(kE)));
  int64_t d;
  bool in;
  T v[kE], r[kE], m[kE], p[kE], rd, md, pd;
  __device__ inline void load(const GramDev& G, int64_t thread, const T* __restrict__ rr,
                              const T* __restrict__ minv, const T* __restrict__ po) {
    d = thread / kGramLanes;
    in = d < G.ndn;
    if (!in) return;
    const int64_t e = d * W + (thread % kGramLanes) * kE;
    const cols_t c = *(const cols_t*)(G.col + e);
    const T* val = (const T*)G.val + e;
    const int32_t self = G.node[d];
#pragma unroll
    for (int q = 0; q < kE; ++q) {
      v[q] = val[q];
      r[q] = rr[c[q]];
      m[q] = minv[c[q]];
      p[q] = po[c[q]];
    }
    rd = rr[self];
    md = minv[self];
    pd = po[self];
  }
  __device__ inline double value(int first, T beta, T* __restrict__ gq) {
    T acc = 0;
    if (in) {
#pragma unroll
      for (int q = 0; q < kE; ++q) acc += v[q] * pcg_p(r[q], m[q], p[q], first, beta);
    }
#pragma unroll
    for (int o = kGramLanes / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if (!in || (threadIdx.x % kGramLanes) != 0) return 0.0;
    gq[d] = acc;
    return (double)pcg_p(rd, md, pd, first, beta) * (double)acc;
  }
};

// V neighbouring values (16 bytes) of a vector; past its end: zeros
template <typename T, int V>
__device__ inline void pcg_ld(const T* __restrict__ a, int64_t i, int64_t n, T* v) {
  typedef T vec __attribute__((ext_vector_type(V)));
  if (i + V <= n) {
    const vec w = *(const vec*)(a + i);
#pragma unroll
    for (int k = 0; k < V; ++k) v[k] = w[k];
  } else {
#pragma unroll
    for (int k = 0; k < V; ++k) v[k] = i + k < n ? a[i + k] : (T)0;
  }
}
template <typename T, int V>
__device__ inline void pcg_st(T* __restrict__ a, int64_t i, int64_t n, const T* v) {
  typedef T vec __attribute__((ext_vector_type(V)));
  if (i + V <= n) {
    vec w;
#pragma unroll
    for (int k = 0; k < V; ++k) w[k] = v[k];
    *(vec*)(a + i) = w;
  } else {
#pragma unroll
    for (int k = 0; k < V; ++k)
      if (i + k < n) a[i + k] = v[k];
  }
}

// direction, and beside it the data term (workgroups [0, ng))
template <typename T, int W>
__global__ __launch_bounds__(VB) void k_pcg_dir(const T* __restrict__ r,
                                                const T* __restrict__ minv,
                                                const T* __restrict__ po, T* __restrict__ pn,
                                                int64_t n, GramDev G, int ng, T* __restrict__ gq,
                                                const double* __restrict__ part_r, int nr,
                                                double* __restrict__ part_g, CgCtl* ctl, int par) {
  __shared__ double sh[VB / 64];
  int first;
  T beta;
  if ((int)blockIdx.x < ng) {
    PcgGram<T, W> gr;
    gr.load(G, (int64_t)blockIdx.x * VB + threadIdx.x, r, minv, po);
    if (!pcg_begin<T>(part_r, nr, ctl, par, sh, &first, &beta)) return;
    const double bs = block_sum(gr.value(first, beta, gq), sh);
    if (threadIdx.x == 0) part_g[blockIdx.x] = bs;
    return;
  }
  constexpr int V = 16 / sizeof(T);
  const int64_t step = (int64_t)(gridDim.x - ng) * VB * V;
  int64_t i = ((int64_t)(blockIdx.x - ng) * VB + threadIdx.x) * V;
  T rv[V], mv[V], pv[V];
  auto load = [&]() {
    pcg_ld<T, V>(r, i, n, rv);
    pcg_ld<T, V>(minv, i, n, mv);
    pcg_ld<T, V>(po, i, n, pv);
  };
  load();
  if (!pcg_begin<T>(part_r, nr, ctl, par, sh, &first, &beta)) return;
  while (i < n) {
#pragma unroll
    for (int k = 0; k < V; ++k) pv[k] = pcg_p(rv[k], mv[k], pv[k], first, beta);
    pcg_st<T, V>(pn, i, n, pv);
    i += step;
    if (i < n) load();
  }
}

// direction, regulariser and data term in one launch.  A workgroup takes a
// 16 x 8 x 4 tile: it forms the direction on the tile and two nodes around it
// in LDS, then each thread applies its node's 25 taps.  Workgroups [0, ng):
// the data term.
constexpr int kTlX = 16, kTlY = 8, kTlZ = 4, kTlN = kTlX * kTlY * kTlZ;
constexpr int kTlPX = kTlX + 4, kTlPY = kTlY + 4, kTlPZ = kTlZ + 4;
template <typename T, int W>
__global__ __launch_bounds__(kTlN) void k_pcg_tile(const T* __restrict__ r,
                                                   const T* __restrict__ minv,
                                                   const T* __restrict__ po, T* __restrict__ pn,
                                                   T* __restrict__ y, GridDev g,
                                                   const T* __restrict__ tab, GramDev G, int ng,
                                                   T* __restrict__ gq,
                                                   const double* __restrict__ part_r, int nr,
                                                   double* __restrict__ part, CgCtl* ctl,
                                                   int par) {
  __shared__ double sh[kTlN / 64];
  __shared__ T tile[kTlPX * kTlPY * kTlPZ];
  const int t = threadIdx.x;
  const int ntx = (g.nx + kTlX - 1) / kTlX, nty = (g.ny + kTlY - 1) / kTlY;
  const int b = (int)blockIdx.x - ng;
  const int bx = b % ntx, by = b / ntx % nty, bz = b / ntx / nty;
  const int64_t nxy = (int64_t)g.nx * g.ny;
  // the node's coefficients and the tile's vectors travel while rho is summed
  const int lx = t % kTlX, ly = t / kTlX % kTlY, lz = t / (kTlX * kTlY);
  const int i = bx * kTlX + lx, j = by * kTlY + ly, k = bz * kTlZ + lz;
  const bool in = i < g.nx && j < g.ny && k < g.nz;
  T c[kTaps];
  constexpr int kLoads = (kTlPX * kTlPY * kTlPZ + kTlN - 1) / kTlN;
  T lr[kLoads], lm[kLoads], lp[kLoads];
  int first;
  T beta;
  if (b < 0) {
    PcgGram<T, W> gr;
    gr.load(G, (int64_t)blockIdx.x * kTlN + t, r, minv, po);
    if (!pcg_begin<T>(part_r, nr, ctl, par, sh, &first, &beta)) return;
    const double bs = block_sum(gr.value(first, beta, gq), sh);
    if (t == 0) part[blockIdx.x] = bs;
    return;
  }
  {
#pragma unroll
    for (int q = 0; q < kLoads; ++q) {
      const int e = t + q * kTlN;
      const int x = bx * kTlX - 2 + e % kTlPX, yy = by * kTlY - 2 + e / kTlPX % kTlPY;
      const int z = bz * kTlZ - 2 + e / (kTlPX * kTlPY);
      const bool ok = e < kTlPX * kTlPY * kTlPZ && x >= 0 && x < g.nx && yy >= 0 && yy < g.ny &&
                      z >= 0 && z < g.nz;
      const int64_t id = ok ? x + (int64_t)g.nx * yy + nxy * z : 0;
      lr[q] = ok ? r[id] : (T)0;
      lm[q] = minv[id];
      lp[q] = ok ? po[id] : (T)0;
    }
    const T* cr =
        tab + ((cls7(in ? k : 0, g.nz) * 7 + cls7(in ? j : 0, g.ny)) * 7 + cls7(in ? i : 0, g.nx)) *
                  kTaps;
#pragma unroll
    for (int q = 0; q < kTaps; ++q) c[q] = cr[q];
  }
  if (!pcg_begin<T>(part_r, nr, ctl, par, sh, &first, &beta)) return;
#pragma unroll
  for (int q = 0; q < kLoads; ++q) {
    const int e = t + q * kTlN;
    if (e < kTlPX * kTlPY * kTlPZ) tile[e] = pcg_p(lr[q], lm[q], lp[q], first, beta);
  }
  __syncthreads();
  const T* s = tile + ((lz + 2) * kTlPY + ly + 2) * kTlPX + lx + 2;
  constexpr int kPl = kTlPX * kTlPY;
  T acc = inplane<T, kTlPX>(c, s);
  acc += c[13] * s[-kPl] + c[14] * s[kPl];
  const T *dn = s - 2 * kPl, *up = s + 2 * kPl;
  acc += c[15] * dn[0] + c[16] * dn[2] + c[17] * dn[-2] + c[18] * dn[2 * kTlPX] +
         c[19] * dn[-2 * kTlPX];
  acc += c[20] * up[0] + c[21] * up[2] + c[22] * up[-2] + c[23] * up[2 * kTlPX] +
         c[24] * up[-2 * kTlPX];
  double dot = 0.0;
  if (in) {
    const int64_t id = i + (int64_t)g.nx * j + nxy * k;
    pn[id] = s[0];
    y[id] = acc;
    dot = (double)s[0] * (double)acc;
  }
  const double bs = block_sum(dot, sh);
  if (t == 0) part[blockIdx.x] = bs;
}

// x += alpha p ; r -= alpha (q + the data term) ; partials of r.(minv r).
// alpha = rho / p.q from the partials of the operator (part_q, and part_g of
// the data term), or from ctl where they are too many to sum here (nq < 0).
template <typename T>
__global__ __launch_bounds__(VB) void k_pcg_upd(T* __restrict__ x, T* __restrict__ r,
                                                const T* __restrict__ p, const T* __restrict__ q,
                                                const T* __restrict__ minv, int64_t n, GramDev G,
                                                const T* __restrict__ gq,
                                                const double* __restrict__ part_q, int nq,
                                                const double* __restrict__ part_g, int ng,
                                                double* __restrict__ part_r, const CgCtl* ctl,
                                                int par) {
  __shared__ double sh[VB / 64];
  constexpr int V = 16 / sizeof(T);
  const int64_t step = (int64_t)gridDim.x * VB * V;
  int64_t i = ((int64_t)blockIdx.x * VB + threadIdx.x) * V;
  T xv[V], rv[V], pv[V], qv[V], mv[V];
  uint64_t mask = 0;
  int32_t base = 0;
  auto load = [&]() {
    pcg_ld<T, V>(q, i, n, qv);
    pcg_ld<T, V>(p, i, n, pv);
    pcg_ld<T, V>(x, i, n, xv);
    pcg_ld<T, V>(r, i, n, rv);
    pcg_ld<T, V>(minv, i, n, mv);
    if (G.ndn > 0 && i < n) {
      mask = G.mask[i >> 6];
      base = G.base[i >> 6];
    }
  };
  // the data term's value of the thread's nodes that have one
  auto add_data = [&]() {
    const uint64_t mine = (mask >> (i & 63)) & ((1u << V) - 1);
    if (!mine) return;
    int32_t at = base + __popcll(mask & ((1ull << (i & 63)) - 1));
#pragma unroll
    for (int k = 0; k < V; ++k)
      if ((mine >> k) & 1) qv[k] += gq[at++];
  };
  load();
  const int done = ctl->done;
  const double rho = ctl->rs[par];
  if (G.ndn > 0 && i < n) add_data();
  T alpha;
  if (nq < 0) {
    alpha = (T)ctl->alpha;
  } else {
    double pq = pcg_total(part_q, nq, sh);
    if (ng > 0) pq += pcg_total(part_g, ng, sh);
    alpha = (T)(rho / pq);
  }
  if (done) return;
  double acc = 0.0;
  while (i < n) {
#pragma unroll
    for (int k = 0; k < V; ++k) {
      xv[k] += alpha * pv[k];
      rv[k] -= alpha * qv[k];
      acc += (double)rv[k] * (double)(mv[k] * rv[k]);
    }
    pcg_st<T, V>(x, i, n, xv);
    pcg_st<T, V>(r, i, n, rv);
    i += step;
    if (i < n) {
      load();
      if (G.ndn > 0) add_data();
    }
  }
  const double bs = block_sum(acc, sh);
  if (threadIdx.x == 0) part_r[blockIdx.x] = bs;
}

// one workgroup: alpha where the operator's partials are many
__global__ __launch_bounds__(VB) void k_pcg_alpha(const double* __restrict__ part_q, int nq,
                                                  const double* __restrict__ part_g, int ng,
                                                  CgCtl* ctl, int par) {
  if (ctl->done) return;
  __shared__ double sh[VB / 64];
  double pq = pcg_total(part_q, nq, sh);
  if (ng > 0) pq += pcg_total(part_g, ng, sh);
  if (threadIdx.x == 0) ctl->alpha = ctl->rs[par] / pq;
}

// one workgroup, after the last iteration of a chunk (an even number): the
// stopping test that the next iteration would begin with
__global__ __launch_bounds__(VB) void k_pcg_check(const double* __restrict__ part_r, int nr,
                                                  CgCtl* ctl) {
  if (ctl->done) return;
  __shared__ double sh[VB / 64];
  const double rho = pcg_total(part_r, nr, sh);
  if (threadIdx.x == 0) {
    const int it = ctl->its[1];
    const int conv = sqrt(rho) < ctl->thr;
    if (conv || it >= ctl->maxiter) {
      ctl->rho = rho;
      ctl->iter = it;
      ctl->converged = conv;
      ctl->done = 1;
    }
  }
}

}  // namespace lsamd
