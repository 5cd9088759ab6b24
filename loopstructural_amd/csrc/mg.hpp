// Geometric multigrid preconditioner and flexible PCG for one FD system.
//
// Hierarchy: level 0 is the system itself; level l+1 is the grid with every
// second node of level l (cells halved, rounded up, so the coarse grid may
// reach one fine cell beyond the fine one), step doubled.  Prolongation P is
// trilinear ([1/2, 1, 1/2] per axis), restriction is P^T.  Coarse operators:
// the data term is the exact Galerkin product (A_d P): each data row is
// mapped through P and its repeated coarse columns merged; the regulariser is
// re-discretised on the coarse grid, its interior rows with the fine level's
// squared weights and its border rows with theirs quartered per level.  Those
// are the weights that come closest to the Galerkin product: for linear
// interpolation P^T D^T D P = D^T D / 4 along the differenced axis (the
// interpolant bends only at the coarse nodes), and P^T P sums to 2 along each
// of the other two, which gives 1; a border layer has one row per face node
// (2 x 2 of them per coarse one) and lies on odd fine nodes, where the
// interpolant does not bend, on every face but the far one of an even axis.
// Weights that keep a smooth field's energy (halved per level, borders too)
// let the coarse grids overcorrect what they only resolve as kinks: at 128^3
// (5000 values, 1000 normals) 97 outer iterations against 63, at 97^3 107
// against 65, 72 x 69 x 109 with 367 values 85 against 62, 24 x 24 x 36 80
// against 63, over 48 systems of 32^3..96^3 at most 139 against 101.
// The ridge is no difference and is not scaled by this rule: it stays halved per
// level, where P^T P would multiply it by 8.  As it is (64^3 nodes, iterations
// with both halved, and now): 1e-8 78, 62; 0.01 103, 66; 0.05 113, 88; 0.2 28,
// 33; 1.0 25, 26.
// The coarsest level (<= 5 nodes per axis) is solved with a dense inverse.
// Smoother: Chebyshev polynomial (degree 2 on the fine level, 3 on the
// coarse ones) in M N on
// [lambda_max/30, 1.15 lambda_max], lambda_max by power iteration, with M
// additive Schwarz: the exact inverse of N on each block, summed over
// blocks, point Jacobi on the nodes no block covers.  Blocks are the 8 nodes
// of every cell that holds a data row, and the boundary layers: per axis the
// first three and the last three nodes form one group (a short axis of < 6
// nodes is one group: an axis of 6 gives two groups of 3, whose blocks of
// 27 invert in LDS where one block of 216 took 35 ms in global memory),
// every other index is its own group, and each product
// of groups with at least one boundary group is a block.  Point Jacobi alone
// leaves the modes that those strong local couplings (data rows of weight
// ~1 against regulariser rows of ~0.1; border rows of weight dx) do not see:
// they are oscillatory and of tiny Rayleigh quotient, so neither the
// smoother nor the coarse grid reduces them.  The V-cycle runs in FP32; the
// outer flexible CG (Polak-Ribiere beta) runs in FP64 with the same FP64
// stopping test as the Jacobi form.
#pragma once

namespace lsamd {

constexpr int kMgDegMax = 8;  // largest Chebyshev degree (LSAMD_MG_DEGREE)
constexpr int kMgCoarse = 5;  // stop coarsening at <= 5 nodes per axis

// --------------------------------------------------------------- kernels ----
__global__ void k_mg_to_f32(const double* __restrict__ a, float* __restrict__ b, int64_t n,
                            const CgCtl* ctl) {
  if (ctl->done) return;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = (float)a[i];
}
// Smoother preconditioner M applied to r = b - q (r = b when from_zero) at
// node i.  Tag sm[i]: >= 0, the Jacobi scale of an uncovered node; -1, a
// node covered by Schwarz blocks, whose row of summed block inverses is
// sval[sptr[i] .. sptr[i+1]) over the columns scol.
struct MgSm {
  const float* sm;
  const int64_t* sptr;
  const int32_t* scol;
  const float* sval;
};

__device__ inline float mg_r(const float* __restrict__ b, const float* __restrict__ q,
                             int64_t j, int from_zero) {
  return from_zero ? b[j] : b[j] - q[j];
}

__device__ inline float mg_precond(int64_t i, const MgSm& S, const float* __restrict__ b,
                                   const float* __restrict__ q, int from_zero) {
  const float t = S.sm[i];
  if (t >= 0.f) return t * mg_r(b, q, i, from_zero);
  // four entries per step: independent loads in flight hide the latency of
  // the column-indexed gathers
  float acc = 0.f;
  int64_t e = S.sptr[i];
  const int64_t e1 = S.sptr[i + 1];
  for (; e + 4 <= e1; e += 4) {
    const int32_t j0 = S.scol[e], j1 = S.scol[e + 1], j2 = S.scol[e + 2], j3 = S.scol[e + 3];
    acc += S.sval[e] * mg_r(b, q, j0, from_zero) + S.sval[e + 1] * mg_r(b, q, j1, from_zero) +
           S.sval[e + 2] * mg_r(b, q, j2, from_zero) + S.sval[e + 3] * mg_r(b, q, j3, from_zero);
  }
  for (; e < e1; ++e) acc += S.sval[e] * mg_r(b, q, S.scol[e], from_zero);
  return acc;
}

// Chebyshev step of a level that keeps q = N x: mode 0 first step from zero
// (d = c0 M b, x = d), 1 first step (d = c0 M (b - q), x += d), 2 later step
// (d = c1 d + c2 M (b - q), x += d); last: the smoothing's final step, whose
// d is dead and not stored.
//
// Workgroups [0, ncb): the covered nodes (compact list, where the level has
// one), kCovLanes threads per row of block inverses, whose gathers would
// otherwise stall every wavefront that holds one; the rest: the other nodes
// (every node on a level without a list).  One launch for both: at 128^3 the
// two took 10.4 and 15.4 us one after the other.
constexpr int kCovLanes = 4;
__global__ __launch_bounds__(256) void k_mg_cheb(const int32_t* __restrict__ cov, int64_t ncov,
                                                 int ncb, const float* __restrict__ b,
                                                 const float* __restrict__ q, MgSm S,
                                                 float* __restrict__ x, float* __restrict__ d,
                                                 int64_t n, int mode, float c0, float c1, float c2,
                                                 int last, const CgCtl* ctl) {
  const int done = ctl->done;
  int64_t i;
  float z;
  if ((int)blockIdx.x < ncb) {
    const int64_t th = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (th / kCovLanes >= ncov) return;  // whole groups
    i = cov[th / kCovLanes];
    const int64_t e1 = S.sptr[i + 1];
    z = 0.f;
    for (int64_t e = S.sptr[i] + th % kCovLanes; e < e1; e += 4 * kCovLanes) {
      int32_t c[4];
      float a[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bool ok = e + k * kCovLanes < e1;
        const int64_t at = ok ? e + k * kCovLanes : e;
        c[k] = S.scol[at];
        a[k] = ok ? S.sval[at] : 0.f;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) z += a[k] * mg_r(b, q, c[k], mode == 0);
    }
#pragma unroll
    for (int o = kCovLanes / 2; o > 0; o >>= 1) z += __shfl_xor(z, o, 64);
    if (th % kCovLanes != 0) return;
  } else {
    i = (int64_t)(blockIdx.x - ncb) * 256 + threadIdx.x;
    if (i >= n) return;
    if (ncb > 0) {
      const float t = S.sm[i];
      if (t < 0.f) return;
      z = t * mg_r(b, q, i, mode == 0);
    } else {
      z = mg_precond(i, S, b, q, mode == 0);
    }
  }
  if (done) return;
  const float dv = mode == 2 ? c1 * d[i] + c2 * z : c0 * z;
  if (!last) d[i] = dv;
  x[i] = mode == 0 ? dv : x[i] + dv;
}

__host__ __device__ inline void mg_ijk(int64_t id, int nx, int ny, int& i, int& j, int& k) {
  const int64_t nxy = (int64_t)nx * ny;
  k = (int)(id / nxy);
  const int64_t r = id - (int64_t)k * nxy;
  j = (int)(r / nx);
  i = (int)(r - (int64_t)j * nx);
}

// P^T r at coarse node id, r = bf - qf (qf == nullptr: r = bf): the fine
// nodes 2J-1, 2J, 2J+1 per axis with weights 1/2, 1, 1/2 (those inside the
// fine grid).  All 27 loads are issued at once, those outside the grid from
// the centre with weight 0: a load behind a branch waits for the one before.
__device__ inline float mg_restrict_node(const float* __restrict__ bf,
                                         const float* __restrict__ qf, const GridDev& gf,
                                         const GridDev& gc, int64_t id) {
  int I, J, K;
  mg_ijk(id, gc.nx, gc.ny, I, J, K);
  const int64_t fnxy = (int64_t)gf.nx * gf.ny;
  float v[27];
#pragma unroll
  for (int t = 0; t < 27; ++t) {
    const int di = t % 3 - 1, dj = t / 3 % 3 - 1, dk = t / 9 - 1;
    const int i = 2 * I + di, j = 2 * J + dj, k = 2 * K + dk;
    const bool ok = (unsigned)i < (unsigned)gf.nx && (unsigned)j < (unsigned)gf.ny &&
                    (unsigned)k < (unsigned)gf.nz;
    const int64_t f = ok ? (int64_t)i + (int64_t)j * gf.nx + (int64_t)k * fnxy : 0;
    const float r = qf ? bf[f] - qf[f] : bf[f];
    v[t] = ok ? r : 0.f;
  }
  float acc = 0.f;
#pragma unroll
  for (int t = 0; t < 27; ++t)
    acc += (t % 3 == 1 ? 1.f : 0.5f) * (t / 3 % 3 == 1 ? 1.f : 0.5f) * (t / 9 == 1 ? 1.f : 0.5f) *
           v[t];
  return acc;
}

// (P xc) at fine node id: trilinear, coarse node c = fine node 2c; eight
// loads at once, weight 0 where an even index needs one neighbour only
__device__ inline float mg_prolong_node(const float* __restrict__ xc, const GridDev& gc,
                                        const GridDev& gf, int64_t id) {
  int i, j, k;
  mg_ijk(id, gf.nx, gf.ny, i, j, k);
  const int oi = i & 1, oj = j & 1, ok = k & 1;
  const int64_t cnxy = (int64_t)gc.nx * gc.ny;
  const float* c = xc + (i >> 1) + (int64_t)(j >> 1) * gc.nx + (int64_t)(k >> 1) * cnxy;
  float v[8];
#pragma unroll
  for (int t = 0; t < 8; ++t)
    v[t] = c[(t & 1) * oi + (int64_t)((t >> 1) & 1) * oj * gc.nx + (int64_t)(t >> 2) * ok * cnxy];
  // an even index has both its neighbours at the same node, half each
  return 0.125f * (((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])));
}

__global__ void k_mg_restrict(const float* __restrict__ bf, const float* __restrict__ qf,
                              GridDev gf, float* __restrict__ bc, GridDev gc, const CgCtl* ctl) {
  const int64_t nc = (int64_t)gc.nx * gc.ny * gc.nz;
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= nc) return;
  const int done = ctl->done;
  const float v = mg_restrict_node(bf, qf, gf, gc, id);
  if (!done) bc[id] = v;
}
__global__ void k_mg_prolong(const float* __restrict__ xc, GridDev gc, float* __restrict__ xf,
                             GridDev gf, const CgCtl* ctl) {
  const int64_t nf = (int64_t)gf.nx * gf.ny * gf.nz;
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= nf) return;
  const int done = ctl->done;
  const float v = xf[id] + mg_prolong_node(xc, gc, gf, id);
  if (!done) xf[id] = v;
}

__global__ __launch_bounds__(64) void k_mg_dense(const float* __restrict__ cinv,
                                                 const float* __restrict__ b,
                                                 float* __restrict__ x, int n, const CgCtl* ctl) {
  if (ctl->done) return;
  const int r = blockIdx.x;
  float acc = 0.f;
  for (int c = threadIdx.x; c < n; c += 64) acc += cinv[(int64_t)r * n + c] * b[c];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (threadIdx.x == 0) x[r] = acc;
}

// Gram matrix of the data rows of a coarse level, G = A^T W^2 A, as sorted
// (row << 32 | col, value) pairs: every row of width wc emits wc^2 pairs.
__global__ void k_gram_pairs(const int32_t* __restrict__ cols, const double* __restrict__ coef,
                             const double* __restrict__ w2, int64_t nrows, int wc,
                             uint64_t* __restrict__ key, double* __restrict__ val) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  const int64_t e0 = r * wc;
  const double w = w2[r];
  for (int a = 0; a < wc; ++a)
    for (int b = 0; b < wc; ++b) {
      const int64_t o = e0 * wc + (int64_t)a * wc + b;
      key[o] = ((uint64_t)(uint32_t)cols[e0 + a] << 32) | (uint32_t)cols[e0 + b];
      val[o] = w * coef[e0 + a] * coef[e0 + b];
    }
}

// CSR row pointers of the reduced Gram entries (keys sorted): first entry of
// each node row by binary search
__global__ void k_gram_ptr(const uint64_t* __restrict__ ukey, int64_t m, int64_t n,
                           int64_t* __restrict__ ptr) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i > n) return;
  int64_t lo = 0, hi = m;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)(ukey[mid] >> 32) < i)
      lo = mid + 1;
    else
      hi = mid;
  }
  ptr[i] = lo;
}

__global__ void k_gram_cols(const uint64_t* __restrict__ ukey, const double* __restrict__ v,
                            int64_t m, int32_t* __restrict__ col, float* __restrict__ v32,
                            double* __restrict__ v64) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m) return;
  col[e] = (int32_t)(ukey[e] & 0xffffffffu);
  v32[e] = (float)v[e];
  v64[e] = v[e];
}

// diag += diagonal of G; then the Jacobi inverses
__global__ void k_gram_diag(const int64_t* __restrict__ ptr, const int32_t* __restrict__ col,
                            const double* __restrict__ val, double* __restrict__ diag,
                            double* __restrict__ m64, float* __restrict__ m32, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double d = diag[i];
  for (int64_t e = ptr[i]; e < ptr[i + 1]; ++e)
    if (col[e] == (int32_t)i) d += val[e];
  diag[i] = d;
  const double m = d > 0.0 ? 1.0 / d : 1.0;
  m64[i] = m;
  m32[i] = (float)m;
}

// Coarse data rows A P: row r of width wf (columns on grid gf) mapped through
// P onto grid gc, repeated coarse columns merged.  count_only: write the
// number of distinct coarse columns; else write them (padded to wc with zero
// coefficients on the first column).  General form: any columns (two distant
// points), in arrays that live in memory.
__global__ void k_mg_rows(const int64_t* __restrict__ row_ptr, const int32_t* __restrict__ cols,
                          const double* __restrict__ coef, int64_t nrows, GridDev gf, GridDev gc,
                          int count_only, int wc, int32_t* __restrict__ ccount,
                          int32_t* __restrict__ ccols, double* __restrict__ ccoef) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  constexpr int kMax = 64;
  int32_t uc[kMax];
  double ua[kMax];
  int nu = 0;
  bool overflow = false;
  const int64_t cnxy = (int64_t)gc.nx * gc.ny;
  for (int64_t e = row_ptr[r]; e < row_ptr[r + 1]; ++e) {
    int i, j, k;
    mg_ijk(cols[e], gf.nx, gf.ny, i, j, k);
    const int ni = (i & 1) ? 2 : 1, nj = (j & 1) ? 2 : 1, nk = (k & 1) ? 2 : 1;
    const double w = coef[e] * (ni == 2 ? 0.5 : 1.0) * (nj == 2 ? 0.5 : 1.0) * (nk == 2 ? 0.5 : 1.0);
    for (int c = 0; c < nk; ++c)
      for (int b = 0; b < nj; ++b)
        for (int a = 0; a < ni; ++a) {
          const int32_t col = (int32_t)((i >> 1) + a + (int64_t)((j >> 1) + b) * gc.nx +
                                        (int64_t)((k >> 1) + c) * cnxy);
          int u = 0;
          while (u < nu && uc[u] != col) ++u;
          if (u == nu) {
            if (nu == kMax) {
              overflow = true;
              continue;
            }
            uc[nu] = col;
            ua[nu++] = 0.0;
          }
          ua[u] += w;
        }
  }
  if (count_only) {
    ccount[r] = overflow ? kMax + 1 : nu;
    return;
  }
  for (int u = 0; u < wc; ++u) {
    ccols[r * wc + u] = u < nu ? uc[u] : uc[0];
    ccoef[r * wc + u] = u < nu ? ua[u] : 0.0;
  }
}

// The same for rows whose coarse columns lie in a box of 4 x 4 x 4 nodes (one
// point): a column's place in the box is its slot, so nothing is searched; the
// slots in use are a word of bits, the sums lie in LDS.  Columns come in the
// order of their slots.  Count: kMgRowFar for a row that does not fit.  The
// rows of 129^3 nodes, per level: 75 us for each of the two launches in the general
// form, 11 (count) and 14 us in this one.
constexpr int kMgRowFar = 65, kMgRowThreads = 64;
template <bool COUNT>
__global__ __launch_bounds__(kMgRowThreads) void k_mg_rows_box(
    const int64_t* __restrict__ row_ptr, const int32_t* __restrict__ cols,
    const double* __restrict__ coef, int64_t nrows, GridDev gf, GridDev gc, int wc,
    int32_t* __restrict__ ccount, int32_t* __restrict__ ccols, double* __restrict__ ccoef) {
  __shared__ double sums[COUNT ? 1 : 64 * kMgRowThreads];
  const int64_t r = (int64_t)blockIdx.x * kMgRowThreads + threadIdx.x;
  if (r >= nrows) return;
  const int64_t e0 = row_ptr[r], e1 = row_ptr[r + 1];
  int lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {0, 0, 0};
  for (int64_t e = e0; e < e1; ++e) {
    int p[3];
    mg_ijk(cols[e], gf.nx, gf.ny, p[0], p[1], p[2]);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      lo[a] = min(lo[a], p[a] >> 1);
      hi[a] = max(hi[a], (p[a] + 1) >> 1);
    }
  }
  bool far = false;
#pragma unroll
  for (int a = 0; a < 3; ++a) far = far || (e1 > e0 && hi[a] - lo[a] > 3);
  if (far) {  // the write never meets one
    if (COUNT) ccount[r] = kMgRowFar;
    return;
  }
  double* ua = sums + threadIdx.x;
  if (!COUNT)
    for (int u = 0; u < 64; ++u) ua[u * kMgRowThreads] = 0.0;
  uint64_t used = 0;
  int first = 0;
  for (int64_t e = e0; e < e1; ++e) {
    int i, j, k;
    mg_ijk(cols[e], gf.nx, gf.ny, i, j, k);
    const int ni = i & 1, nj = j & 1, nk = k & 1;
    const int s0 = ((i >> 1) - lo[0]) + 4 * (((j >> 1) - lo[1]) + 4 * ((k >> 1) - lo[2]));
    const double w = COUNT ? 0.0 : coef[e] * (ni ? 0.5 : 1.0) * (nj ? 0.5 : 1.0) * (nk ? 0.5 : 1.0);
    if (e == e0) first = s0;
    for (int c = 0; c <= nk; ++c)
      for (int b = 0; b <= nj; ++b)
        for (int a = 0; a <= ni; ++a) {
          const int u = s0 + a + 4 * b + 16 * c;
          used |= 1ull << u;
          if (!COUNT) ua[u * kMgRowThreads] += w;
        }
  }
  if (COUNT) {
    ccount[r] = __popcll(used);
    return;
  }
  auto column = [&](int u) {
    return (int32_t)(lo[0] + (u & 3) + (int64_t)(lo[1] + (u >> 2 & 3)) * gc.nx +
                     (int64_t)(lo[2] + (u >> 4)) * gc.nx * gc.ny);
  };
  const int32_t pad = e1 > e0 ? column(first) : 0;
  for (int q = 0; q < wc; ++q) {
    const bool on = used != 0;
    const int u = on ? __ffsll((unsigned long long)used) - 1 : 0;
    used &= used - 1;
    ccols[r * wc + q] = on ? column(u) : pad;
    ccoef[r * wc + q] = on ? ua[u * kMgRowThreads] : 0.0;
  }
}

// power iteration step w = M y (y = N v), G threads per node
template <int G>
__global__ __launch_bounds__(256) void k_mg_power(const double* __restrict__ y,
                                                  const double* __restrict__ minv,
                                                  const float* __restrict__ sm,
                                                  const int64_t* __restrict__ sptr,
                                                  const int32_t* __restrict__ scol,
                                                  const double* __restrict__ sval, int64_t n,
                                                  double* __restrict__ w) {
  const int64_t th = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t i = th / G;
  const int l = (int)(th % G);
  if (i >= n) return;  // whole groups
  const float t = sm[i];
  const double own = minv[i] * y[i];
  double z = 0.0;
  if (sptr) {
    const int64_t e1 = sptr[i + 1];
    for (int64_t e = sptr[i] + l; e < e1; e += 2 * G) {
      const bool two = e + G < e1;
      const int64_t f = two ? e + G : e;
      z += sval[e] * y[scol[e]] + (two ? sval[f] : 0.0) * y[scol[f]];
    }
  }
#pragma unroll
  for (int o = G / 2; o > 0; o >>= 1) z += __shfl_xor(z, o, 64);
  if (l == 0) w[i] = t >= 0.f ? own : z;
}

// partials of |v|^2, then those of |w|^2
__global__ __launch_bounds__(256) void k_mg_norms(const double* __restrict__ v,
                                                  const double* __restrict__ w, int64_t n,
                                                  double* __restrict__ part) {
  __shared__ double sh[4];
  double a = 0.0, b = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    a += v[i] * v[i];
    b += w[i] * w[i];
  }
  const double sa = block_sum(a, sh);
  const double sb = block_sum(b, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = sa;
    part[gridDim.x + blockIdx.x] = sb;
  }
}

// one block: scal[0] = |w| / |v| (the eigenvalue estimate)
__global__ __launch_bounds__(256) void k_mg_norm_fin(const double* __restrict__ part, int np,
                                                     double* __restrict__ scal) {
  __shared__ double sh[4];
  const double a = pcg_total(part, np, sh), b = pcg_total(part + np, np, sh);
  if (threadIdx.x == 0) scal[0] = a > 0.0 ? sqrt(b / a) : 0.0;
}

// deterministic positive start vector of the power iteration
__global__ void k_mg_start(double* __restrict__ v, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint64_t z = (uint64_t)i * 0x9E3779B97F4A7C15ULL + 0x632BE59BD9B4E019ULL;
  z ^= z >> 31;
  z *= 0xBF58476D1CE4E5B9ULL;
  z ^= z >> 29;
  v[i] = 0.5 + (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

// rptr[r] = r * wc: row pointers of fixed-width rows
__global__ void k_iota_rows(int64_t* __restrict__ rptr, int64_t n, int64_t wc) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r < n) rptr[r] = r * wc;
}

// ------------------------------------------------------ flexible PCG ----
// partials of z.r, then those of z.r_prev (z: the FP32 V-cycle output, widened)
__global__ __launch_bounds__(256) void k_fcg_dots(const float* __restrict__ z,
                                                  const double* __restrict__ r,
                                                  const double* __restrict__ rp, int64_t n,
                                                  double* __restrict__ part, const CgCtl* ctl) {
  if (ctl->done) return;
  __shared__ double sh[4];
  double a = 0.0, b = 0.0;
  for (int64_t i = 2 * ((int64_t)blockIdx.x * 256 + threadIdx.x); i < n;
       i += (int64_t)gridDim.x * 512) {
    float zv[2];
    double rv[2], pv[2];
    pcg_ld<float, 2>(z, i, n, zv);
    pcg_ld<double, 2>(r, i, n, rv);
    pcg_ld<double, 2>(rp, i, n, pv);
    a += (double)zv[0] * rv[0] + (double)zv[1] * rv[1];
    b += (double)zv[0] * pv[0] + (double)zv[1] * pv[1];
  }
  const double sa = block_sum(a, sh);
  const double sb = block_sum(b, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = sa;
    part[gridDim.x + blockIdx.x] = sb;
  }
}

// p = z + beta p, beta = (z.r - z.r_prev) / rho_prev (0 on the first step):
// every workgroup sums the np pairs of partials, workgroup 0 records rho = z.r
__global__ __launch_bounds__(256) void k_fcg_dir(const float* __restrict__ z,
                                                 double* __restrict__ p, int64_t n,
                                                 const double* __restrict__ part, int np,
                                                 CgCtl* ctl) {
  __shared__ double sh[4];
  const int done = ctl->done, first = ctl->iter == 0;
  const double prev = ctl->rho_prev;
  const double zr = pcg_total(part, np, sh);
  const double zp = pcg_total(part + np, np, sh);
  if (done) return;
  const double beta = first ? 0.0 : (zr - zp) / prev;
  if (blockIdx.x == 0 && threadIdx.x == 0) ctl->rho = zr;
  for (int64_t i = 2 * ((int64_t)blockIdx.x * 256 + threadIdx.x); i < n;
       i += (int64_t)gridDim.x * 512) {
    float zv[2];
    double pv[2];
    pcg_ld<float, 2>(z, i, n, zv);
    pcg_ld<double, 2>(p, i, n, pv);
#pragma unroll
    for (int k = 0; k < 2; ++k) pv[k] = first ? (double)zv[k] : (double)zv[k] + beta * pv[k];
    pcg_st<double, 2>(p, i, n, pv);
  }
}

// y += the data term of x (rows by node, see pcg.hpp); partials of x.Gx
// where part is given
template <typename T, int W>
__global__ __launch_bounds__(256) void k_gram_add(GramDev G, const T* __restrict__ x,
                                                  T* __restrict__ y, double* __restrict__ part,
                                                  const CgCtl* ctl) {
  __shared__ double sh[4];
  constexpr int kE = W / kGramLanes;
  typedef int32_t cols_t __attribute__((ext_vector_type(kE)));
  const int done = ctl->done;
  const int64_t th = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t d = th / kGramLanes;
  double dot = 0.0;
  if (d < G.ndn) {  // whole groups
    const int64_t e = d * W + (th % kGramLanes) * kE;
    const cols_t c = *(const cols_t*)(G.col + e);
    const T* val = (const T*)G.val + e;
    const int32_t i = G.node[d];
    const T xi = x[i], yi = y[i];
    T acc = 0;
#pragma unroll
    for (int k = 0; k < kE; ++k) acc += val[k] * x[c[k]];
#pragma unroll
    for (int o = kGramLanes / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if (th % kGramLanes == 0 && !done) {
      y[i] = yi + acc;
      dot = (double)xi * (double)acc;
    }
  }
  if (!part) return;
  const double bs = block_sum(dot, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = bs;
}

// x += alpha p ; r_prev = r ; r -= alpha q ; rf = (float) r, the next
// V-cycle's input ; partials of r.(minv r).  alpha = rho / p.q from the
// operator's partials, or from ctl (nq < 0).
__global__ __launch_bounds__(256) void k_fcg_upd(double* __restrict__ x, double* __restrict__ r,
                                                 double* __restrict__ rp,
                                                 const double* __restrict__ p,
                                                 const double* __restrict__ q,
                                                 const double* __restrict__ minv,
                                                 float* __restrict__ rf, int64_t n,
                                                 const double* __restrict__ part_q, int nq,
                                                 const double* __restrict__ part_g, int ng,
                                                 double* __restrict__ part, const CgCtl* ctl) {
  __shared__ double sh[4];
  const int done = ctl->done;
  const double rho = ctl->rho;
  double alpha;
  if (nq < 0) {
    alpha = ctl->alpha;
  } else {
    double pq = pcg_total(part_q, nq, sh);
    if (ng > 0) pq += pcg_total(part_g, ng, sh);
    alpha = rho / pq;
  }
  if (done) return;
  double acc = 0.0;
  for (int64_t i = 2 * ((int64_t)blockIdx.x * 256 + threadIdx.x); i < n;
       i += (int64_t)gridDim.x * 512) {
    double xv[2], rv[2], pv[2], qv[2], mv[2];
    float fv[2];
    pcg_ld<double, 2>(x, i, n, xv);
    pcg_ld<double, 2>(p, i, n, pv);
    pcg_ld<double, 2>(r, i, n, rv);
    pcg_ld<double, 2>(q, i, n, qv);
    pcg_ld<double, 2>(minv, i, n, mv);
    pcg_st<double, 2>(rp, i, n, rv);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      xv[k] += alpha * pv[k];
      rv[k] -= alpha * qv[k];
      fv[k] = (float)rv[k];
      acc += rv[k] * (mv[k] * rv[k]);
    }
    pcg_st<double, 2>(x, i, n, xv);
    pcg_st<double, 2>(r, i, n, rv);
    pcg_st<float, 2>(rf, i, n, fv);
  }
  const double bs = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = bs;
}

// one workgroup: alpha = rho / p.q where its partials are many
__global__ __launch_bounds__(256) void k_fcg_alpha(const double* __restrict__ part_q, int nq,
                                                   const double* __restrict__ part_g, int ng,
                                                   CgCtl* ctl) {
  if (ctl->done) return;
  __shared__ double sh[4];
  double pq = pcg_total(part_q, nq, sh);
  if (ng > 0) pq += pcg_total(part_g, ng, sh);
  if (threadIdx.x == 0) ctl->alpha = ctl->rho / pq;
}

// one block: rho_prev = rho ; iter++ ; stopping test on |S r|, which has to hold
// in two iterations running.  A V-cycle with three coarse steps leaves more of
// the smooth error at the same |S r| than one with four: stopped at once, the
// field was up to 1.4 times as far from the FP64 minimiser (geometric means over
// six inputs each, 97 x 89 x 81 nodes 1.66e-8 against 1.14e-8, 64^3 1.20e-8
// against 1.19e-8).  Mostly the iteration more fits the chunk that is launched.
__global__ __launch_bounds__(256) void k_fcg_upd_fin(const double* __restrict__ part, int np,
                                                     CgCtl* ctl) {
  if (ctl->done) return;
  __shared__ double sh[4];
  const double tot = reduce_partials(part, np, sh);
  if (threadIdx.x == 0) {
    ctl->rho_prev = ctl->rho;
    const int it = ctl->iter + 1;
    ctl->iter = it;
    ctl->res2 = tot;  // |S r|^2 of the current iterate
    const int conv = sqrt(tot) < ctl->thr;
    ctl->done = (conv && ctl->converged) || it >= ctl->maxiter;
    ctl->converged = conv;
  }
}


// ----------------------------------------------- coarse levels, fused ----
// Device view of one coarse level's operator: regulariser (class table, or
// the exact per-node formula when the table does not apply) + data Gram
// matrix.
template <typename T>
struct MgDevT {
  GridDev g;
  int64_t n;
  const T* tab;  // class table, nullptr: per-node formula with w
  RegW<T> w;
  const int64_t* gptr;
  const int32_t* gcol;
  const T* gval;
};
using MgDev = MgDevT<float>;

template <typename T>
__device__ inline T mg_apply_node(const MgDevT<T>& L, const T* __restrict__ x, int64_t id) {
  int i, j, k;
  mg_ijk(id, L.g.nx, L.g.ny, i, j, k);
  T acc;
  if (L.tab) {
    const int nx = L.g.nx, ny = L.g.ny, nz = L.g.nz;
    const int64_t nxy = (int64_t)nx * ny;
    const T* c = L.tab + ((cls7(k, nz) * 7 + cls7(j, ny)) * 7 + cls7(i, nx)) * kTaps;
    acc = c[0] * x[id];
#pragma unroll
    for (int t = 1; t < kTaps; ++t) {
      const int dx = kBTap[t][0], dy = kBTap[t][1], dz = kBTap[t][2];
      const bool ok = (unsigned)(i + dx) < (unsigned)nx && (unsigned)(j + dy) < (unsigned)ny &&
                      (unsigned)(k + dz) < (unsigned)nz;
      const T xv = x[ok ? id + dx + (int64_t)nx * dy + nxy * dz : id];
      acc += c[t] * (ok ? xv : (T)0);
    }
  } else {
    acc = general_node<T>(x, L.g, L.w, nullptr, i, j, k);
  }
  if (L.gptr) {
    int64_t e = L.gptr[id];
    const int64_t e1 = L.gptr[id + 1];
    for (; e + 4 <= e1; e += 4) {
      const int32_t c0 = L.gcol[e], c1 = L.gcol[e + 1], c2 = L.gcol[e + 2], c3 = L.gcol[e + 3];
      acc += L.gval[e] * x[c0] + L.gval[e + 1] * x[c1] + L.gval[e + 2] * x[c2] +
             L.gval[e + 3] * x[c3];
    }
    for (; e < e1; ++e) acc += L.gval[e] * x[L.gcol[e]];
  }
  return acc;
}

// y = N x of a coarse level in one launch (stencil and Gram row per node)
__global__ __launch_bounds__(256) void k_mg_apply(MgDev L, const float* __restrict__ x,
                                                  float* __restrict__ y, const CgCtl* ctl) {
  if (ctl->done) return;
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id < L.n) y[id] = mg_apply_node(L, x, id);
}

// Coarse levels, G neighbouring threads per node.  These levels are bound by
// the chain of dependent loads (row pointer, columns, gathers) and by a row's
// length, not by bytes: one thread per row took 8.9 us for the operator and 7
// us for a smoothing step on 9^3 nodes, hardly less than on 33^3.  With G
// threads a row's entries are loaded at once and contiguously, the pointer
// travels beside the stencil's loads, and the solve's state is looked at last.
// The operator leaves the residual r = b - N x, so that a smoothing step
// gathers one vector.

// taps 0..24 as kBTap, packed (dx + 2) | (dy + 2) << 4 | (dz + 2) << 8; the
// rest: no tap
__constant__ int kTapPack[32] = {
    0x222, 0x223, 0x221, 0x232, 0x212, 0x224, 0x220, 0x242, 0x202, 0x244, 0x240,
    0x204, 0x200, 0x122, 0x322, 0x022, 0x024, 0x020, 0x042, 0x002, 0x422, 0x424,
    0x420, 0x442, 0x402, -1,    -1,    -1,    -1,    -1,    -1,    -1};

// sum of val[e] v[col[e]] over a row's entries, this thread's share
template <int G, typename T>
__device__ inline T mg_row_share(const int64_t* __restrict__ ptr, const int32_t* __restrict__ col,
                                 const T* __restrict__ val, const T* __restrict__ v, int64_t i,
                                 int l) {
  const int64_t e1 = ptr[i + 1];
  T acc = 0;
  for (int64_t e = ptr[i] + l; e < e1; e += 4 * G) {
    int32_t c[4];
    T a[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bool ok = e + k * G < e1;
      const int64_t at = ok ? e + k * G : e;
      c[k] = col[at];
      a[k] = ok ? val[at] : (T)0;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) acc += a[k] * v[c[k]];
  }
  return acc;
}

template <int G, typename T>
__device__ inline T mg_lane_sum(T v) {
#pragma unroll
  for (int o = G / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// (N x)[id], summed over the G threads of the node
template <int G, typename T>
__device__ inline T mg_product(const MgDevT<T>& L, const T* __restrict__ x, int64_t id, int l) {
  if (!L.tab) return mg_lane_sum<G>(l == 0 ? mg_apply_node(L, x, id) : (T)0);
  int i, j, k;
  mg_ijk(id, L.g.nx, L.g.ny, i, j, k);
  const int nx = L.g.nx, ny = L.g.ny, nz = L.g.nz;
  const int64_t nxy = (int64_t)nx * ny;
  const T* c = L.tab + ((cls7(k, nz) * 7 + cls7(j, ny)) * 7 + cls7(i, nx)) * kTaps;
  constexpr int kT = (kTaps + G - 1) / G;
  T cv[kT], xv[kT];
#pragma unroll
  for (int q = 0; q < kT; ++q) {
    const int t = l + q * G;
    const int p = kTapPack[t < 32 ? t : 31];
    const int dx = (p & 15) - 2, dy = ((p >> 4) & 15) - 2, dz = ((p >> 8) & 15) - 2;
    const bool ok = t < kTaps && (unsigned)(i + dx) < (unsigned)nx &&
                    (unsigned)(j + dy) < (unsigned)ny && (unsigned)(k + dz) < (unsigned)nz;
    cv[q] = ok ? c[t] : (T)0;
    xv[q] = x[ok ? id + dx + (int64_t)nx * dy + nxy * dz : id];
  }
  T acc = L.gptr ? mg_row_share<G>(L.gptr, L.gcol, L.gval, x, id, l) : (T)0;
#pragma unroll
  for (int q = 0; q < kT; ++q) acc += cv[q] * xv[q];
  return mg_lane_sum<G>(acc);
}

// (M r)[i] of the smoother, summed over the G threads of the node
template <int G>
__device__ inline float mg_smoothed(const MgSm& S, const float* __restrict__ r, int64_t i, int l) {
  const float t = S.sm[i], rv = r[i];
  float z = 0.f;
  if (S.sptr) z = mg_row_share<G>(S.sptr, S.scol, S.sval, r, i, l);
  z = mg_lane_sum<G>(z);
  return t >= 0.f ? t * rv : z;
}

// r = b - N x
template <int G>
__global__ __launch_bounds__(256) void k_mg_resid(MgDev L, const float* __restrict__ b,
                                                  const float* __restrict__ x,
                                                  float* __restrict__ r, const CgCtl* ctl) {
  const int64_t th = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t id = th / G;
  const int l = (int)(th % G);
  if (id >= L.n) return;  // whole groups
  const int done = ctl->done;
  const float bv = b[id];
  const float v = mg_product<G>(L, x, id, l);
  if (l == 0 && !done) r[id] = bv - v;
}

// y = N x in FP64 (set-up)
template <int G>
__global__ __launch_bounds__(256) void k_mg_apply64(MgDevT<double> L, const double* __restrict__ x,
                                                    double* __restrict__ y) {
  const int64_t th = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t id = th / G;
  if (id >= L.n) return;
  const double v = mg_product<G>(L, x, id, (int)(th % G));
  if (th % G == 0) y[id] = v;
}

// smoothing step from the residual r: dv = c1 d + c2 M r (c1 = 0: d is not
// read); x = dv (from_zero) or x += dv; d = dv unless it is dead (last)
template <int G>
__global__ __launch_bounds__(256) void k_mg_smooth(const float* __restrict__ r, MgSm S,
                                                   float* __restrict__ x, float* __restrict__ d,
                                                   int64_t n, float c1, float c2, int from_zero,
                                                   int last, const CgCtl* ctl) {
  const int64_t th = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t i = th / G;
  const int l = (int)(th % G);
  if (i >= n) return;  // whole groups
  const int done = ctl->done;
  const float xv = from_zero ? 0.f : x[i], dv0 = c1 != 0.f ? d[i] : 0.f;
  const float dv = c1 * dv0 + c2 * mg_smoothed<G>(S, r, i, l);
  if (l != 0 || done) return;
  if (!last) d[i] = dv;
  x[i] = xv + dv;
}

// coarse levels this large keep the product N x in q, as level 0 does, and
// smooth their covered nodes apart; the smaller ones keep the residual
constexpr int64_t kSplitMin = 1 << 20;
// coarse levels this large have a compact list of their covered nodes (level 0
// always has); the multi-rhs smoother splits the levels of this size, level 0
// among them, and the single-system and batched ones level 0 at any size
constexpr int64_t kCovListMin = 1 << 17;

// ------------------------------------------------ Schwarz smoother blocks ----
// Entry N(a, b) of a level's operator: regulariser rows (from their
// definition, ridge included) plus the data Gram matrix G (CSR, columns
// sorted per row; may be absent).
__host__ __device__ inline double reg_entry(const GridDev& g, const RegW<double>& w, const double* scale2,
                                   int64_t ia, int64_t ib) {
  int ai, aj, ak, bi, bj, bk;
  mg_ijk(ia, g.nx, g.ny, ai, aj, ak);
  mg_ijk(ib, g.nx, g.ny, bi, bj, bk);
  double v = ia == ib ? w.ridge : 0.0;
  // axial masks [1, -2, 1] / sqrt6: product of two taps / 6
  auto m = [](int o) { return o == 0 ? -2.0 : 1.0; };
  if (aj == bj && ak == bk)
    for (int c = (ai > bi ? ai : bi) - 1; c <= (ai < bi ? ai : bi) + 1; ++c)
      v += row_weight(g, w, scale2, F_XX, c, aj, ak) * m(ai - c) * m(bi - c) / 6.0;
  if (ai == bi && ak == bk)
    for (int c = (aj > bj ? aj : bj) - 1; c <= (aj < bj ? aj : bj) + 1; ++c)
      v += row_weight(g, w, scale2, F_YY, ai, c, ak) * m(aj - c) * m(bj - c) / 6.0;
  if (ai == bi && aj == bj)
    for (int c = (ak > bk ? ak : bk) - 1; c <= (ak < bk ? ak : bk) + 1; ++c)
      v += row_weight(g, w, scale2, F_ZZ, ai, aj, c) * m(ak - c) * m(bk - c) / 6.0;
  // cross masks: tap -1/2 * du * dv at (du, dv) in {-1, 1}^2
  for (int du = -1; du <= 1; du += 2)
    for (int dv = -1; dv <= 1; dv += 2) {
      // a sits at centre + (du, dv); b at centre + (eu, ev)
      if (ak == bk) {
        const int cx = ai - du, cy = aj - dv, eu = bi - cx, ev = bj - cy;
        if ((eu == 1 || eu == -1) && (ev == 1 || ev == -1))
          v += row_weight(g, w, scale2, F_XY, cx, cy, ak) * 0.25 * du * dv * eu * ev;
      }
      if (aj == bj) {
        const int cx = ai - du, cz = ak - dv, eu = bi - cx, ev = bk - cz;
        if ((eu == 1 || eu == -1) && (ev == 1 || ev == -1))
          v += row_weight(g, w, scale2, F_XZ, cx, aj, cz) * 0.25 * du * dv * eu * ev;
      }
      if (ai == bi) {
        const int cy = aj - du, cz = ak - dv, eu = bj - cy, ev = bk - cz;
        if ((eu == 1 || eu == -1) && (ev == 1 || ev == -1))
          v += row_weight(g, w, scale2, F_YZ, ai, cy, cz) * 0.25 * du * dv * eu * ev;
      }
    }
  return v;
}

__device__ inline double gram_entry(const int64_t* __restrict__ gptr,
                                    const int32_t* __restrict__ gcol,
                                    const double* __restrict__ gval, int64_t a, int64_t b) {
  if (!gptr) return 0.0;
  int64_t lo = gptr[a], hi = gptr[a + 1];
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (gcol[mid] < (int32_t)b)
      lo = mid + 1;
    else
      hi = mid;
  }
  return (lo < gptr[a + 1] && gcol[lo] == (int32_t)b) ? gval[lo] : 0.0;
}

// dense N restricted to every block: entry e of block q is (a, c) of the
// block's s x s matrix, nodes bnodes[boff[q] + a], bnodes[boff[q] + c]
__global__ void k_blk_fill(const int64_t* __restrict__ boff, const int32_t* __restrict__ bnodes,
                           const int64_t* __restrict__ moff, int nb, int64_t ntot, GridDev g,
                           RegW<double> w, const double* scale2, const int64_t* gptr,
                           const int32_t* gcol, const double* gval, double* __restrict__ dense) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ntot) return;
  int lo = 0, hi = nb - 1;
  while (lo < hi) {  // last block with moff <= e
    const int mid = (lo + hi + 1) >> 1;
    if (moff[mid] <= e)
      lo = mid;
    else
      hi = mid - 1;
  }
  const int64_t s = boff[lo + 1] - boff[lo];
  const int64_t r = e - moff[lo];
  const int64_t ia = bnodes[boff[lo] + r / s], ib = bnodes[boff[lo] + r % s];
  dense[e] = reg_entry(g, w, scale2, ia, ib) + gram_entry(gptr, gcol, gval, ia, ib);
}

// in-place Gauss-Jordan inverse of every (symmetric positive definite)
// block, one workgroup of 64 per block (the matrix in LDS up to kBlkLds
// rows, in global memory beyond); *bad set when a pivot is not positive
constexpr int kBlkLds = 40;
__global__ __launch_bounds__(64) void k_blk_inv(const int64_t* __restrict__ boff,
                                                const int64_t* __restrict__ moff, int nb,
                                                double* __restrict__ dense,
                                                int* __restrict__ bad) {
  __shared__ double lds[kBlkLds * kBlkLds];
  __shared__ double fcol[kBlkLds];
  const int q = blockIdx.x;
  if (q >= nb) return;
  const int s = (int)(boff[q + 1] - boff[q]);
  double* G = dense + moff[q];
  const bool in_lds = s <= kBlkLds;
  double* A = in_lds ? lds : G;
  const int t = threadIdx.x;
  if (in_lds)
    for (int e = t; e < s * s; e += 64) lds[e] = G[e];
  __syncthreads();
  for (int k = 0; k < s; ++k) {
    const double p = A[k * s + k];
    if (!(p > 0.0)) {
      if (t == 0) *bad = 1;
      return;  // uniform: every thread read the same pivot
    }
    const double ip = 1.0 / p;
    __syncthreads();
    for (int j = t; j < s; j += 64) A[k * s + j] = (j == k) ? ip : A[k * s + j] * ip;
    for (int i = t; i < s; i += 64)
      if (i != k && in_lds) fcol[i] = A[i * s + k];
    __syncthreads();
    if (in_lds) {
      for (int e = t; e < s * s; e += 64) {
        const int i = e / s, j = e - (e / s) * s;
        if (i == k) continue;
        const double f = fcol[i];
        A[e] = (j == k) ? -f * ip : A[e] - f * A[k * s + j];
      }
    } else {
      // global path: one row per thread, the factor read before the row
      for (int i = t; i < s; i += 64) {
        if (i == k) continue;
        const double f = A[i * s + k];
        for (int j = 0; j < s; ++j)
          A[i * s + j] = (j == k) ? -f * ip : A[i * s + j] - f * A[k * s + j];
      }
    }
    __syncthreads();
  }
  if (in_lds)
    for (int e = t; e < s * s; e += 64) G[e] = lds[e];
}

// (row << 32 | col, value) pairs of every block inverse
__global__ void k_blk_pairs(const int64_t* __restrict__ boff, const int32_t* __restrict__ bnodes,
                            const int64_t* __restrict__ moff, int nb, int64_t ntot,
                            const double* __restrict__ dense, uint64_t* __restrict__ key,
                            double* __restrict__ val) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ntot) return;
  int lo = 0, hi = nb - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (moff[mid] <= e)
      lo = mid;
    else
      hi = mid - 1;
  }
  const int64_t s = boff[lo + 1] - boff[lo];
  const int64_t r = e - moff[lo];
  const int32_t ia = bnodes[boff[lo] + r / s], ib = bnodes[boff[lo] + r % s];
  key[e] = ((uint64_t)(uint32_t)ia << 32) | (uint32_t)ib;
  val[e] = dense[e];
}

// flags of the covered nodes (negative tags)
__global__ void k_blk_flags(const float* __restrict__ sm, uint8_t* __restrict__ flag, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) flag[i] = sm[i] < 0.f ? 1 : 0;
}

// smoother tags: -1 on nodes with a Schwarz row, the Jacobi scale elsewhere
__global__ void k_blk_tags(const int64_t* __restrict__ sptr, const float* __restrict__ minv,
                           float* __restrict__ sm, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  sm[i] = sptr[i + 1] > sptr[i] ? -1.f : minv[i];
}

// ------------------------------------------------- sliced rows (SELL-64) ----
// A sparse row set in slices of 64 rows, one wavefront each: entry k of the
// slice's row t at off[s] + 64 k + t (columns and values), slice width
// width[s] (the longest row of the slice, rounded up to a multiple of 4).
// The 64 threads of a wavefront read one entry index of their 64 rows as one
// contiguous 256-byte line, where CSR with a thread per row touches 64
// lines.  Padding entries point at the row's own node with value 0.  Row r
// is node node[r] (node == nullptr: node r).
struct Sell {
  const int64_t* off;
  const int32_t* width;
  const int32_t* col;
  const float* val;
  const int32_t* node;
  int64_t nrows;
};

// row r of a CSR (ptr, with tags sm when given: a row whose tag is >= 0 is
// the single entry (node, tag), the smoother's point-Jacobi nodes)
__device__ inline int64_t sell_src_len(const int64_t* __restrict__ ptr,
                                       const float* __restrict__ sm, int64_t i) {
  if (sm && sm[i] >= 0.f) return 1;
  return ptr[i + 1] - ptr[i];
}

__global__ void k_sell_width(const int64_t* __restrict__ ptr, const float* __restrict__ sm,
                             const int32_t* __restrict__ node, int64_t nrows,
                             int32_t* __restrict__ width) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s * 64 >= nrows) return;
  int64_t w = 0;
  const int64_t r1 = s * 64 + 64 < nrows ? s * 64 + 64 : nrows;
  for (int64_t r = s * 64; r < r1; ++r) {
    const int64_t l = sell_src_len(ptr, sm, node ? node[r] : r);
    w = l > w ? l : w;
  }
  width[s] = (int32_t)((w + 3) & ~(int64_t)3);
}

__global__ void k_sell_fill(const int64_t* __restrict__ ptr, const int32_t* __restrict__ col,
                            const float* __restrict__ val, const float* __restrict__ sm,
                            const int32_t* __restrict__ node, int64_t nrows,
                            const int64_t* __restrict__ off, const int32_t* __restrict__ width,
                            int32_t* __restrict__ ocol, float* __restrict__ oval) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t s = r >> 6;
  if (s * 64 >= nrows) return;
  const int t = (int)(r & 63);
  const int w = width[s];
  const int64_t o = off[s] + t;
  if (r >= nrows) {
    for (int k = 0; k < w; ++k) {
      ocol[o + 64 * (int64_t)k] = 0;
      oval[o + 64 * (int64_t)k] = 0.f;
    }
    return;
  }
  const int64_t i = node ? node[r] : r;
  int k = 0;
  if (sm && sm[i] >= 0.f) {
    if (w > 0) {
      ocol[o] = (int32_t)i;
      oval[o] = sm[i];
      k = 1;
    }
  } else {
    const int64_t e0 = ptr[i], len = ptr[i + 1] - e0;
    for (; k < len; ++k) {
      ocol[o + 64 * (int64_t)k] = col[e0 + k];
      oval[o + 64 * (int64_t)k] = val[e0 + k];
    }
  }
  for (; k < w; ++k) {
    ocol[o + 64 * (int64_t)k] = (int32_t)i;
    oval[o + 64 * (int64_t)k] = 0.f;
  }
}

// flags of the nodes with a nonempty CSR row
__global__ void k_rows_nonempty(const int64_t* __restrict__ ptr, uint8_t* __restrict__ flag,
                                int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) flag[i] = ptr[i + 1] > ptr[i] ? 1 : 0;
}

// pos[cov[t]] = t (pos initialised to -1)
__global__ void k_cov_pos(const int32_t* __restrict__ cov, int64_t ncov, int32_t* __restrict__ pos) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < ncov) pos[cov[t]] = (int32_t)t;
}
// sliced columns (node ids) to covered-list positions; *bad = 1 for a node
// outside the list
__global__ void k_sell_to_pos(int32_t* __restrict__ col, int64_t nent,
                              const int32_t* __restrict__ pos, int* __restrict__ bad) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nent) return;
  const int32_t p = pos[col[e]];
  if (p < 0) {
    *bad = 1;
    col[e] = 0;
  } else {
    col[e] = p;
  }
}

// data rows of level 0 in fixed width wc (repeated columns merged, padded
// with zero coefficients on the first column), for the level's Gram matrix
__global__ void k_rows_fixed(const int64_t* __restrict__ row_ptr, const int32_t* __restrict__ cols,
                             const double* __restrict__ coef, int64_t nrows, int wc,
                             int32_t* __restrict__ ccols, double* __restrict__ ccoef) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  int nu = 0;
  const int64_t o = r * wc;
  for (int64_t e = row_ptr[r]; e < row_ptr[r + 1]; ++e) {
    int u = 0;
    while (u < nu && ccols[o + u] != cols[e]) ++u;
    if (u == nu) {
      if (nu == wc) continue;  // cannot happen: wc >= row width
      ccols[o + nu] = cols[e];
      ccoef[o + nu++] = 0.0;
    }
    ccoef[o + u] += coef[e];
  }
  for (int u = nu; u < wc; ++u) {
    ccols[o + u] = nu > 0 ? ccols[o] : 0;
    ccoef[o + u] = 0.0;
  }
}

}  // namespace lsamd
