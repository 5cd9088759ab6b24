// LSMR (Fong & Saunders, SIAM J. Sci. Comput. 33 (2011), the algorithm of
// scipy.sparse.linalg.lsmr) on the rectangular FD least-squares operator,
// matrix-free.  The operator is A S with the reference's row blocks: data
// rows w_r a_r, regulariser rows sqrt(W_f(i)) d_f(i) (an interior row and the
// border rows of the same mask at one node are merged into one row of the
// summed squared weight, which leaves A^T A, A^T b and |b| unchanged and with
// them the LSMR iterates), ridge rows ridge * e_i; S = diag(A^T A)^-1/2 is
// the column scaling.  Chunks of iterations replay from a graph.
//
// Small systems are bound by launches, so an iteration is three of them:
//   k_ls_fwd   u = A S v - coef u;
//   k_ls_bwd   beta = |u|, v = S A^T u / beta - beta v; one workgroup more
//              makes the estimates and stopping tests of the step before;
//   k_ls_rot   alpha = |v|, the rotations that the vectors need, the vectors.
// The tests can come that late because u and v may run ahead of a finished
// solve: x and |x| move in k_ls_rot only.  They are some thirty dependent FP64
// divisions and roots: in k_ls_rot, in every workgroup, they took 6 us at
// 26^3 and 15 us at 51^3 nodes, beside the products they take none.
// Reductions are summed by every workgroup for itself (in the same order);
// one records the scalars.  State alternates between two slots, so that no
// launch writes what it reads, and the estimates of a step can be made again
// at the end of a chunk.  For the same reason the end of a solve, recorded by
// k_ls_bwd, stops k_ls_rot at once and k_ls_bwd only from the next k_ls_fwd on
// (`halt`): had k_ls_bwd looked at `done` itself, the wavefronts of a
// workgroup could have parted before a barrier.  The regulariser's part of u is kept as
// uw = sqrt(W) u: its recurrence needs W itself, and the transposed product
// neither weights nor roots at the 21 neighbours it gathers.
// Eleven launches took 45 us per iteration at 26^3 nodes and 1000 rows, 55 us
// at 51^3, 212 us at 129^3 (floor 115 us: 606 MB); these three take 16, 26
// and 144 us.
#pragma once

namespace lsamd {

// after a step: Golub-Kahan and rotation state, and what the estimates need
struct LsCtl {
  double alpha, beta, fwd_coef, alphabar, rho, rhobar, cbar, sbar, zeta, zetabar;
  double rhobarold, zetaold, thetabar, rhotemp, chat, cc, ss;
  int itn;
};

// after the estimates of a step
struct LsEst {
  double betadd, betad, rhodold, tautildeold, thetatilde, normA2, maxrbar, minrbar;
};

// beta of the step in progress; the options; the end of the solve, once reached
struct LsMid {
  double beta, inv_beta, normb, atol, btol, ctol;
  double normx, normr, normar, normA, condA;
  int skipv;  // beta == 0: v and alpha kept (as scipy's lsmr)
  int maxiter, itn, istop, done;
  int halt;  // done as k_ls_fwd found it, for k_ls_bwd
};

// (c, s, r) with c a + s b = r, -s a + c b = 0 (stable); no jumps
__device__ inline void sym_ortho(double a, double b, double& c, double& s, double& r) {
  const bool big = fabs(b) > fabs(a);
  const double den = big ? b : a, tau = (big ? a : b) / den;
  const double q = (den > 0.0 ? 1.0 : -1.0) / sqrt(1.0 + tau * tau), qt = q * tau;
  const double rq = den / q;
  const bool bz = b == 0.0, az = a == 0.0;
  c = bz ? (az ? 1.0 : (a > 0.0 ? 1.0 : -1.0)) : (az ? 0.0 : (big ? qt : q));
  s = bz ? 0.0 : (az ? (b > 0.0 ? 1.0 : -1.0) : (big ? q : qt));
  r = bz ? fabs(a) : (az ? fabs(b) : rq);
}

__device__ inline void ls_ijk(int64_t id, const GridDev& g, int& i, int& j, int& k) {
  const int64_t nxy = (int64_t)g.nx * g.ny;
  k = (int)(id / nxy);
  const int64_t r = id - (int64_t)k * nxy;
  j = (int)(r / g.nx);
  i = (int)(r - (int64_t)j * g.nx);
}

__device__ inline void ls_finish(LsMid* m, int itn, int istop, double normx, double normr,
                                 double normar, double normA, double condA) {
  m->normx = normx;
  m->normr = normr;
  m->normar = normar;
  m->normA = normA;
  m->condA = condA;
  m->itn = itn;
  m->istop = istop;
  m->done = 1;
}

// |r|, |A|, cond(A) after the step of `c` and the stopping tests, istop
// numbered as scipy's lsmr (`e`: the step before, `o`: this one)
__device__ inline void ls_estimate(const LsCtl& c, const LsEst& e, LsEst* o, double normx,
                                   LsMid* m) {
  LsEst n;
  const double betaacute = c.chat * e.betadd;
  const double betahat = c.cc * betaacute;
  n.betadd = -c.ss * betaacute;
  double ctildeold, stildeold, rhotildeold;
  sym_ortho(e.rhodold, c.thetabar, ctildeold, stildeold, rhotildeold);
  n.thetatilde = stildeold * c.rhobar;
  n.rhodold = ctildeold * c.rhobar;
  n.betad = -stildeold * e.betad + ctildeold * betahat;
  n.tautildeold = (c.zetaold - e.thetatilde * e.tautildeold) / rhotildeold;
  const double taud = (c.zeta - n.thetatilde * n.tautildeold) / n.rhodold;
  const double normr = sqrt((n.betad - taud) * (n.betad - taud) + n.betadd * n.betadd);
  const double normA2 = e.normA2 + c.beta * c.beta;
  const double normA = sqrt(normA2);
  n.normA2 = normA2 + c.alpha * c.alpha;
  n.maxrbar = fmax(e.maxrbar, c.rhobarold);
  n.minrbar = c.itn > 1 ? fmin(e.minrbar, c.rhobarold) : e.minrbar;
  const double condA = fmax(n.maxrbar, c.rhotemp) / fmin(n.minrbar, c.rhotemp);
  const double normar = fabs(c.zetabar);
  *o = n;

  const double normb = m->normb, atol = m->atol;
  const double test1 = normr / normb;
  const double test2 = (normA * normr) != 0.0 ? normar / (normA * normr) : __builtin_inf();
  const double test3 = 1.0 / condA;
  const double t1 = test1 / (1.0 + normA * normx / normb);
  const double rtol = m->btol + atol * normA * normx / normb;
  int istop = 0;
  if (c.itn >= m->maxiter) istop = 7;
  if (1.0 + test3 <= 1.0) istop = 6;
  if (1.0 + test2 <= 1.0) istop = 5;
  if (1.0 + t1 <= 1.0) istop = 4;
  if (test3 <= m->ctol) istop = 3;
  if (test2 <= atol) istop = 2;
  if (test1 <= rtol) istop = 1;
  if (istop) ls_finish(m, c.itn, istop, normx, normr, normar, normA, condA);
}

// Systems of more workgroups than this sum their partials in a launch of their
// own: past some thousands every workgroup reading all of them costs more than
// a launch (about 4 us).
constexpr int kLsPart = 2048;
__global__ __launch_bounds__(1024) void k_ls_fold(const double* __restrict__ part, int n,
                                                  double* __restrict__ out) {
  __shared__ double sh[16];
  const double t = pcg_total(part, n, sh);
  if (threadIdx.x == 0) *out = t;
}

// one workgroup, at the end of a chunk: what k_ls_bwd of the next step would do
__global__ __launch_bounds__(256) void k_ls_check(const LsCtl* c, const LsEst* ein, LsEst* eout,
                                                  const double* __restrict__ px, int nx,
                                                  LsMid* m) {
  __shared__ double sh[4];
  const double x2 = pcg_total(px, nx, sh);
  if (threadIdx.x == 0 && !m->done) ls_estimate(*c, *ein, eout, sqrt(x2), m);
}

// u = A xs - fwd_coef u: data rows in workgroups [0, ndb), 8 threads each,
// then the regulariser and ridge rows, one node per thread; partials of |u|^2.
// init: u = (w b, 0, 0), nothing is read.
__global__ __launch_bounds__(256) void k_ls_fwd(const double* __restrict__ xs, GridDev g,
                                                RegW<double> w, const double* scale2,
                                                double* __restrict__ uw, double* __restrict__ urid,
                                                int64_t n, RowsDev R,
                                                const double* __restrict__ wr,
                                                const double* __restrict__ b,
                                                double* __restrict__ ud, int ndb, int init,
                                                double* __restrict__ part, const LsCtl* c,
                                                LsMid* m) {
  __shared__ double sh[4];
  double acc = 0.0;
  const int done = init ? 0 : m->done;
  if (blockIdx.x == 0 && threadIdx.x == 0) m->halt = done;
  const double a = init ? 0.0 : c->fwd_coef;
  if ((int)blockIdx.x < ndb) {
    const double* coef = (const double*)R.coef;
    const int64_t r = (int64_t)blockIdx.x * 32 + threadIdx.x / 8;
    const int l = threadIdx.x % 8;
    double s = 0.0, uo = 0.0, wv = 0.0, bv = 0.0;
    if (r < R.nrows) {
      wv = wr[r];
      if (init) {
        bv = b[r];
      } else {
        uo = ud[r];
        const int64_t e1 = R.row_ptr[r + 1];
        for (int64_t e = R.row_ptr[r] + l; e < e1; e += 8) s += coef[e] * xs[R.cols[e]];
      }
    }
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (done) return;
    if (r < R.nrows && l == 0) {
      const double un = init ? wv * bv : wv * s - a * uo;
      ud[r] = un;
      acc = un * un;
    }
  } else {
    const int64_t id = (int64_t)(blockIdx.x - ndb) * 256 + threadIdx.x;
    const bool in = id < n;
    int i, j, k;
    ls_ijk(in ? id : 0, g, i, j, k);
    const int64_t nxy = (int64_t)g.nx * g.ny;
    // the node's 19 values; those outside the grid only enter rows of weight 0
    double v[19], uo[7];
    if (!init) {
      const int64_t base = in ? id : 0;
      auto ld = [&](int dx, int dy, int dz) {
        const bool ok = in_grid(g, i + dx, j + dy, k + dz);
        return xs[ok ? base + dx + (int64_t)g.nx * dy + nxy * dz : base];
      };
      v[0] = ld(0, 0, 0);
      v[1] = ld(-1, 0, 0);
      v[2] = ld(1, 0, 0);
      v[3] = ld(0, -1, 0);
      v[4] = ld(0, 1, 0);
      v[5] = ld(0, 0, -1);
      v[6] = ld(0, 0, 1);
      v[7] = ld(-1, -1, 0);
      v[8] = ld(1, -1, 0);
      v[9] = ld(-1, 1, 0);
      v[10] = ld(1, 1, 0);
      v[11] = ld(-1, 0, -1);
      v[12] = ld(1, 0, -1);
      v[13] = ld(-1, 0, 1);
      v[14] = ld(1, 0, 1);
      v[15] = ld(0, -1, -1);
      v[16] = ld(0, 1, -1);
      v[17] = ld(0, -1, 1);
      v[18] = ld(0, 1, 1);
#pragma unroll
      for (int f = 0; f < 6; ++f) uo[f] = uw[f * n + base];
      uo[6] = urid[base];
      if (done) return;
    }
    if (in) {
      const double is6 = 0.40824829046386301637;
      const double row[6] = {is6 * (v[1] - 2.0 * v[0] + v[2]), is6 * (v[3] - 2.0 * v[0] + v[4]),
                             is6 * (v[5] - 2.0 * v[0] + v[6]),
                             0.5 * (-v[7] + v[8] + v[9] - v[10]),
                             0.5 * (-v[11] + v[12] + v[13] - v[14]),
                             0.5 * (-v[15] + v[16] + v[17] - v[18])};
#pragma unroll
      for (int f = 0; f < 6; ++f) {
        const double W = row_weight(g, w, scale2, f, i, j, k);
        const double un = init || !(W > 0.0) ? 0.0 : W * row[f] - a * uo[f];
        uw[f * n + id] = un;
        if (W > 0.0) acc += un * (un / W);
      }
      const double un = init ? 0.0 : sqrt(w.ridge) * v[0] - a * uo[6];
      urid[id] = un;
      acc += un * un;
    }
  }
  const double bs = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = bs;
}

// tap t of 21 of the transposed regulariser at a node: family, offset, value
__device__ inline void ls_tap(int t, int& f, int& dx, int& dy, int& dz, double& co) {
  const bool ax = t < 9;
  const int q = ax ? t : t - 9, p = q % 3, m = q / 3;
  const int du = ax ? 1 - m : (m & 1 ? -1 : 1), dv = m & 2 ? -1 : 1;
  f = ax ? p : 3 + p;  // F_XX.., then F_XY, F_XZ, F_YZ
  dx = ax ? (p == 0 ? du : 0) : (p < 2 ? du : 0);
  dy = ax ? (p == 1 ? du : 0) : (p == 0 ? dv : (p == 2 ? du : 0));
  dz = ax ? (p == 2 ? du : 0) : (p > 0 ? dv : 0);
  const double is6 = 0.40824829046386301637;
  co = ax ? (m == 1 ? -2.0 * is6 : is6) : (du * dv > 0 ? -0.5 : 0.5);
}

// beta = |u|; v = S y - beta v with y = A^T u / beta (init: v = S y, the old v
// is not read); partials of |v|^2.  Workgroup 0: the estimates of the step
// before; the next ncb: nodes with data rows (`mask`), 4 threads each over
// the taps and the entries (a node in a cluster has hundreds: one thread each
// took 75 us at 26^3 nodes and 1e5 points, this 14 us); the rest: one thread
// per node.  cw: the entries' w_r a_r in the order of seg_row.
__global__ __launch_bounds__(256) void k_ls_bwd(
    const double* __restrict__ uw, const double* __restrict__ urid, GridDev g, double sridge,
    RowsDev R, const double* __restrict__ cw, const double* __restrict__ ud,
    const uint64_t* __restrict__ mask, const double* __restrict__ sv, double* __restrict__ v,
    int64_t n, int ncb, int init, const double* __restrict__ part_u, int nu,
    double* __restrict__ part, const LsCtl* c, const LsEst* ein, LsEst* eout,
    const double* __restrict__ px, int nx, LsMid* m) {
  __shared__ double sh[4];
  const int done = init ? 0 : m->halt;
  if (blockIdx.x == 0) {
    if (init || c->itn == 0) return;
    const double x2 = pcg_total(px, nx, sh);
    if (threadIdx.x == 0 && !done) ls_estimate(*c, *ein, eout, sqrt(x2), m);
    return;
  }
  const int blk = (int)blockIdx.x - 1;
  const int64_t nxy = (int64_t)g.nx * g.ny;
  int64_t at = 0;
  double y = 0.0;
  bool in;
  int i, j, k;
  if (blk < ncb) {
    const int64_t d = (int64_t)blk * 64 + threadIdx.x / 4;
    const int l = threadIdx.x % 4;
    in = d < R.ndn;
    const int64_t dd = in ? d : 0;
    at = R.dnode[dd];
    const int64_t q0 = R.seg_ptr[dd], q1 = R.seg_ptr[dd + 1];
    ls_ijk(at, g, i, j, k);
#pragma unroll
    for (int t0 = 0; t0 < 24; t0 += 4) {
      int f, dx, dy, dz;
      double co;
      const int t = t0 + l;
      ls_tap(t < 21 ? t : 0, f, dx, dy, dz, co);
      const bool ok = t < 21 && in_grid(g, i + dx, j + dy, k + dz);
      const double x = uw[f * n + (ok ? at + dx + (int64_t)g.nx * dy + nxy * dz : at)];
      y += ok ? co * x : 0.0;
    }
    if (in)
      for (int64_t q = q0 + l; q < q1; q += 4) y += cw[q] * ud[R.seg_row[q]];
    y += __shfl_xor(y, 1, 64);
    y += __shfl_xor(y, 2, 64);
    y += sridge * urid[at];
    in = in && l == 0;
  } else {
    const int64_t id = (int64_t)(blk - ncb) * 256 + threadIdx.x;
    in = id < n;
    at = in ? id : 0;
    ls_ijk(at, g, i, j, k);
    const uint64_t mk = ncb > 0 ? mask[at >> 6] : 0;
    double u[21];
    const double ur = urid[at];
#pragma unroll
    for (int t = 0; t < 21; ++t) {
      int f, dx, dy, dz;
      double co;
      ls_tap(t, f, dx, dy, dz, co);
      const bool ok = in_grid(g, i + dx, j + dy, k + dz);
      const double x = uw[f * n + (ok ? at + dx + (int64_t)g.nx * dy + nxy * dz : at)];
      u[t] = ok ? co * x : 0.0;
    }
    y = sridge * ur;
#pragma unroll
    for (int t = 0; t < 21; ++t) y += u[t];
    in = in && !(mk >> (at & 63) & 1);
  }
  const double vo = init ? 0.0 : v[at], sc = sv[at];
  const double beta = sqrt(pcg_total(part_u, nu, sh));
  if (done) return;
  const double ib = beta > 0.0 ? 1.0 / beta : 0.0;
  if (blk == 0 && threadIdx.x == 0) {
    m->beta = beta;
    m->inv_beta = ib;
    m->skipv = !init && !(beta > 0.0);
    if (init) {
      m->done = 0;
      m->normb = beta;
    }
  }
  if (!init && !(beta > 0.0)) return;
  double acc = 0.0;
  if (in) {
    const double vn = init ? sc * (y * ib) : sc * (y * ib) - beta * vo;
    v[at] = vn;
    acc = vn * vn;
  }
  const double bs = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blk] = bs;
}

// alpha = |v| and the rotations (every thread; workgroup 0 records them in
// `out`), then v /= alpha ; hbar = h - c_hbar hbar ; x += c_x hbar ;
// h = v - c_h h ; xs = S v, the next product's operand ; partials of |x|^2
// (init: v /= alpha ; h = v ; hbar = 0 ; x = 0)
__global__ __launch_bounds__(256) void k_ls_rot(double* __restrict__ v, double* __restrict__ h,
                                                double* __restrict__ hbar,
                                                double* __restrict__ x, double* __restrict__ xs,
                                                const double* __restrict__ sv, int64_t n, int init,
                                                const double* __restrict__ part_v, int nv,
                                                double* __restrict__ part, const LsCtl* in,
                                                LsCtl* out, LsEst* est, LsMid* m) {
  __shared__ double sh[4];
  const int done = init ? 0 : m->done, skip = m->skipv;
  const double beta = m->beta, ib = m->inv_beta;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t at = i < n ? i : 0;
  const double vv = v[at], sc = sv[at];
  double hv = 0.0, hb = 0.0, xv = 0.0;
  LsCtl o = {};
  double c_hbar = 0.0;
  if (!init) {
    hv = h[at];
    hb = hbar[at];
    xv = x[at];
    const LsCtl c = *in;
    // Qhat (damp = 0): chat = sign of alphabar, alphahat = |alphabar|
    o.chat = c.alphabar < 0.0 ? -1.0 : 1.0;
    sym_ortho(fabs(c.alphabar), beta, o.cc, o.ss, o.rho);
    o.thetabar = c.sbar * o.rho;
    o.rhotemp = c.cbar * o.rho;
    o.rhobarold = c.rhobar;
    o.zetaold = c.zeta;
    o.zetabar = c.zetabar;
    o.alpha = c.alpha;
    o.itn = c.itn + 1;
    c_hbar = o.thetabar * o.rho / (c.rho * c.rhobar);
  }
  const double v2 = pcg_total(part_v, nv, sh);
  if (done) return;
  const bool zero = init && !(beta > 0.0);  // b = 0: x = 0
  const double alpha = skip ? o.alpha : (zero ? 0.0 : sqrt(v2));
  const double ia = skip ? 1.0 : (alpha > 0.0 ? 1.0 / alpha : 0.0);
  double c_x = 0.0, c_h = 0.0;
  o.alpha = alpha;
  o.beta = beta;
  o.fwd_coef = alpha * ib;  // the next product subtracts alpha (u / beta)
  if (init) {
    o.zetabar = alpha * beta;
    o.alphabar = alpha;
    o.rho = o.rhobar = o.cbar = 1.0;
  } else {
    const double thetanew = o.ss * alpha;
    o.alphabar = o.cc * alpha;
    sym_ortho(o.rhotemp, thetanew, o.cbar, o.sbar, o.rhobar);
    o.zeta = o.cbar * o.zetabar;
    o.zetabar = -o.sbar * o.zetabar;
    c_x = o.zeta / (o.rho * o.rhobar);
    c_h = thetanew / o.rho;
  }
  double acc = 0.0;
  if (i < n) {
    const double vn = vv * ia;
    v[i] = vn;
    xs[i] = sc * vn;
    hb = hv - c_hbar * hb;  // init: zeros
    hbar[i] = hb;
    xv += c_x * hb;
    x[i] = xv;
    acc = xv * xv;
    h[i] = vn - c_h * hv;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *out = o;
    if (init) {
      *est = LsEst{beta, 0.0, 1.0, 0.0, 0.0, alpha * alpha, 0.0, 1e100};
      const double normar = alpha * beta;
      if (zero || normar == 0.0)  // also A^T b = 0
        ls_finish(m, 0, 0, 0.0, beta, normar, alpha, zero ? 0.0 : 1.0);
    }
  }
  const double bs = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = bs;
}

// cw = w_r a_r of the entries sorted by node
__global__ void k_ls_coef(RowsDev R, const double* __restrict__ wr, double* __restrict__ cw,
                          int64_t nnz) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < nnz) cw[q] = ((const double*)R.coef)[R.seg_entry[q]] * wr[R.seg_row[q]];
}

__global__ void k_ls_sqrt(const double* __restrict__ minv, double* __restrict__ sv, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) sv[i] = sqrt(minv[i]);
}

// c = S x
__global__ void k_ls_out(const double* __restrict__ x, const double* __restrict__ sv,
                         double* __restrict__ out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = sv[i] * x[i];
}

}  // namespace lsamd
