// Point location, least-squares row builders and evaluation on a structured
// grid.  This translation unit is compiled with -ffp-contract=off (and the
// pragma below) so that every product, quotient and sum rounds exactly like
// the reference's numpy expressions: cell ids, trilinear weights, shape
// gradients, row norms and evaluated values are bit-identical.
//
// Reference: LC/supports/_3d_base_structured.py:251-293 (cell lookup,
// inside test), :386-412 (corner ids), LC/supports/_3d_structured_grid.py:
// 90-146 (trilinear, local coordinates), :295-391 (evaluation), :393-454
// (shape gradients); LI/_discrete_interpolator.py:361-366 (row
// normalisation); LI/_finite_difference_interpolator.py:236-269 (value),
// :342-401 (gradient), :403-476 (normal), :478-539 (gradient orthogonal);
// LC/math/_maths.py:126-160,276-332 (strike/dip basis).
#pragma clang fp contract(off)

#include <math.h>

#include "exact_div.hpp"
#include "lsamd_common.hpp"

namespace lsamd {
namespace {

constexpr double kEps32 = 2.220446049250313e-16 * 32.0;  // np.finfo(float).eps * 32

// numpy's np.clip(v, 0, 1): keeps -0.0 and NaN.
__device__ inline double clip01(double v) { return v < 0.0 ? 0.0 : (v > 1.0 ? 1.0 : v); }

// numpy pairwise order for a contiguous 8-term sum.
__device__ inline double sum8(const double* a) {
  return ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
}

struct Located {
  bool inside;
  int cx, cy, cz;
  double lx, ly, lz;
  double hx, hy, hz;  // size of the cell along each axis
};

__device__ inline bool inside_axis(double p, double o, double h, int nn) {
  const double mx = o + (double)(nn - 1) * h;
  double ext = fabs(mx - o);
  ext = ext > 1.0 ? ext : 1.0;  // np.maximum(|max-origin|, 1.0)
  const double tol = kEps32 * ext;
  return (p >= (o - tol)) && (p <= (mx + tol));
}

__device__ inline int cell_axis(double p, double o, double h, int nn) {
  const double x = p - o;
  long long c = (long long)floor(x / h);
  const long long hi = nn - 2;  // ncells - 1
  if (c < 0) c = 0;
  if (c > hi) c = hi;
  return (int)c;
}

// Rectilinear axis (LC/supports/_3d_rectilinear_grid.py:115-159): cell =
// clip(searchsorted(nodes, p, 'right') - 1, 0, ncells - 1), local coordinate
// (p - x0) / h unclipped with h = x1 - x0 (1 where 0), inside strictly
// between the first and last node.
__device__ inline bool rect_axis(const double* nodes, int nn, double p, int* cell, double* loc,
                                 double* h) {
  int lo = 0, hi = nn;
  while (lo < hi) {  // number of nodes <= p
    const int mid = (lo + hi) >> 1;
    if (nodes[mid] <= p)
      lo = mid + 1;
    else
      hi = mid;
  }
  int c = lo - 1;
  if (c < 0) c = 0;
  if (c > nn - 2) c = nn - 2;
  const double x0 = nodes[c];
  const double x1 = nodes[c + 1 < nn ? c + 1 : nn - 1];
  double w = x1 - x0;
  if (w == 0.0) w = 1.0;
  *cell = c;
  *loc = (p - x0) / w;
  *h = w;
  return (p > nodes[0]) && (p < nodes[nn - 1]);
}

__device__ inline Located locate(const GridDev& g, double px, double py, double pz) {
  Located L;
  if (g.xn) {
    const bool ix = rect_axis(g.xn, g.nx, px, &L.cx, &L.lx, &L.hx);
    const bool iy = rect_axis(g.yn, g.ny, py, &L.cy, &L.ly, &L.hy);
    const bool iz = rect_axis(g.zn, g.nz, pz, &L.cz, &L.lz, &L.hz);
    L.inside = ix && iy && iz;
    return L;
  }
  L.hx = g.hx;
  L.hy = g.hy;
  L.hz = g.hz;
  L.inside = inside_axis(px, g.ox, g.hx, g.nx) && inside_axis(py, g.oy, g.hy, g.ny) &&
             inside_axis(pz, g.oz, g.hz, g.nz);
  L.cx = L.cy = L.cz = 0;
  if (L.inside) {
    L.cx = cell_axis(px, g.ox, g.hx, g.nx);
    L.cy = cell_axis(py, g.oy, g.hy, g.ny);
    L.cz = cell_axis(pz, g.oz, g.hz, g.nz);
  }
  // local coordinates: clip((p - (o + h*cell)) / h, 0, 1)
  L.lx = clip01((px - (g.ox + g.hx * (double)L.cx)) / g.hx);
  L.ly = clip01((py - (g.oy + g.hy * (double)L.cy)) / g.hy);
  L.lz = clip01((pz - (g.oz + g.hz * (double)L.cz)) / g.hz);
  return L;
}

__device__ inline void corner_ids(const GridDev& g, const Located& L, int64_t* id) {
  const int64_t nx = g.nx, nxy = (int64_t)g.nx * g.ny;
  const int64_t g0 = (int64_t)L.cx + nx * L.cy + nxy * L.cz;
  id[0] = g0;
  id[1] = g0 + 1;
  id[2] = g0 + nx;
  id[3] = g0 + nx + 1;
  id[4] = g0 + nxy;
  id[5] = g0 + nxy + 1;
  id[6] = g0 + nxy + nx;
  id[7] = g0 + nxy + nx + 1;
}

// _3d_structured_grid.py:114-123 (same association: left to right)
__device__ inline void trilinear(double x, double y, double z, double* w) {
  w[0] = (1 - x) * (1 - y) * (1 - z);
  w[1] = x * (1 - y) * (1 - z);
  w[2] = (1 - x) * y * (1 - z);
  w[4] = (1 - x) * (1 - y) * z;
  w[5] = x * (1 - y) * z;
  w[6] = (1 - x) * y * z;
  w[3] = x * y * (1 - z);
  w[7] = x * y * z;
}

// _3d_structured_grid.py:425-453, T[d*8 + k]
__device__ inline void shape_grad(double x, double y, double z, double hx, double hy, double hz,
                                  double* T) {
  T[0] = (1 - z) * (y - 1);
  T[1] = (1 - y) * (1 - z);
  T[2] = -y * (1 - z);
  T[4] = -(1 - y) * z;
  T[5] = (1 - y) * z;
  T[6] = -y * z;
  T[3] = y * (1 - z);
  T[7] = y * z;
  T[8 + 0] = (x - 1) * (1 - z);
  T[8 + 1] = -x * (1 - z);
  T[8 + 2] = (1 - x) * (1 - z);
  T[8 + 4] = -(1 - x) * z;
  T[8 + 5] = -x * z;
  T[8 + 6] = (1 - x) * z;
  T[8 + 3] = x * (1 - z);
  T[8 + 7] = x * z;
  T[16 + 0] = -(1 - x) * (1 - y);
  T[16 + 1] = -x * (1 - y);
  T[16 + 2] = -(1 - x) * y;
  T[16 + 4] = (1 - x) * (1 - y);
  T[16 + 5] = x * (1 - y);
  T[16 + 6] = (1 - x) * y;
  T[16 + 3] = -x * y;
  T[16 + 7] = x * y;
#pragma unroll
  for (int k = 0; k < 8; ++k) T[k] /= hx;
#pragma unroll
  for (int k = 0; k < 8; ++k) T[8 + k] /= hy;
#pragma unroll
  for (int k = 0; k < 8; ++k) T[16 + k] /= hz;
}

__global__ void k_locate(GridDev g, const double* __restrict__ pts, int64_t n,
                         int64_t* __restrict__ idc, double* __restrict__ w, double* __restrict__ T,
                         uint8_t* __restrict__ ins) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double px = pts[3 * i], py = pts[3 * i + 1], pz = pts[3 * i + 2];
  Located L = locate(g, px, py, pz);
  if (idc) {
    int64_t id[8];
    corner_ids(g, L, id);
#pragma unroll
    for (int k = 0; k < 8; ++k) idc[8 * i + k] = L.inside ? id[k] : -1;
  }
  if (w) {
    double a[8];
    trilinear(L.lx, L.ly, L.lz, a);
#pragma unroll
    for (int k = 0; k < 8; ++k) w[8 * i + k] = L.inside ? a[k] : 0.0;
  }
  if (T) {
    double t[24];
    shape_grad(L.lx, L.ly, L.lz, L.hx, L.hy, L.hz, t);
#pragma unroll
    for (int k = 0; k < 24; ++k) T[24 * i + k] = L.inside ? t[k] : 0.0;
  }
  if (ins) ins[i] = L.inside ? 1 : 0;
}

// np.linalg.norm of a 3-vector: sequential sum of squares (n < 8).
__device__ inline double norm3(double a, double b, double c) {
  return sqrt((a * a + b * b) + c * c);
}

// Row normalisation, LI/_discrete_interpolator.py:361-366.
__device__ inline double normalise8(double* a, double* b) {
  double sq[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) sq[k] = a[k] * a[k];
  const double len = sqrt(sum8(sq));
  if (len > 0) {
    *b /= len;
#pragma unroll
    for (int k = 0; k < 8; ++k) a[k] /= len;
  }
  return len;
}

__device__ inline void emit_row(int64_t row, const int32_t* id, const double* a, double bv,
                                double wv, double len, int32_t* cols, double* coef, double* b,
                                double* w, double* norm) {
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    cols[8 * row + k] = id[k];
    coef[8 * row + k] = a[k];
  }
  b[row] = bv;
  w[row] = wv;
  if (norm) norm[row] = len;
}

// get_vectors (LC/math/_maths.py:276-298) for an already unit vector v:
// strike = [sin(-s), -cos(-s), 0] with s = deg2rad(rad2deg(-atan2(ny, nx))),
// dip = strike x v; both normalised, then scaled by |v|.
__device__ inline void strike_dip(double* v, double* s, double* d) {
  const double len = norm3(v[0], v[1], v[2]);
  v[0] /= len;
  v[1] /= len;
  v[2] /= len;
  double nv0 = v[0], nv1 = v[1], nv2 = v[2];
  const double l2 = norm3(nv0, nv1, nv2);
  nv0 /= l2;
  nv1 /= l2;
  nv2 /= l2;
  (void)nv2;
  const double strike_deg = (-atan2(nv1, nv0)) * (180.0 / M_PI);
  const double st = strike_deg * (M_PI / 180.0);
  s[0] = sin(-st);
  s[1] = -cos(-st);
  s[2] = 0.0;
  const double ls = norm3(s[0], s[1], s[2]);
  s[0] /= ls;
  s[1] /= ls;
  s[2] /= ls;
  d[0] = s[1] * v[2] - s[2] * v[1];
  d[1] = s[2] * v[0] - s[0] * v[2];
  d[2] = s[0] * v[1] - s[1] * v[0];
  const double ld = norm3(d[0], d[1], d[2]);
  d[0] /= ld;
  d[1] /= ld;
  d[2] /= ld;
  for (int k = 0; k < 3; ++k) {
    s[k] *= len;
    d[k] *= len;
  }
}

__global__ void k_build_rows(GridDev g, int kind, double* __restrict__ pts, int64_t n, int64_t ld,
                             int wcol, double wscale, int32_t* __restrict__ cols,
                             double* __restrict__ coef, double* __restrict__ b,
                             double* __restrict__ w, double* __restrict__ norm) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double* P = pts + i * ld;
  const Located L = locate(g, P[0], P[1], P[2]);
  int64_t id64[8];
  corner_ids(g, L, id64);
  int32_t id[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) id[k] = (int32_t)id64[k];
  const double pw = wcol >= 0 ? P[wcol] : 1.0;
  if (kind == LSAMD_ROWS_VALUE) {
    double a[8];
    trilinear(L.lx, L.ly, L.lz, a);
    double bv = P[3];
    const double len = normalise8(a, &bv);
    emit_row(i, id, a, bv, wscale * pw, len, cols, coef, b, w, norm);
    return;
  }
  double T[24];
  shape_grad(L.lx, L.ly, L.lz, L.hx, L.hy, L.hz, T);
  if (kind == LSAMD_ROWS_NORMAL) {
    for (int d = 0; d < 3; ++d) {
      double a[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) a[k] = T[8 * d + k];
      double bv = P[3 + d];
      const double len = normalise8(a, &bv);
      emit_row((int64_t)d * n + i, id, a, bv, wscale * pw, len, cols, coef, b, w, norm);
    }
    return;
  }
  // gradient / tangent: normalise the stored vector in place, scale T by 1/|v|
  double v[3] = {P[3], P[4], P[5]};
  const double vn = norm3(v[0], v[1], v[2]);
  if (kind == LSAMD_ROWS_GRADIENT || vn > 0) {
    for (int k = 0; k < 3; ++k) v[k] /= vn;
    for (int k = 0; k < 24; ++k) T[k] /= vn;
  }
  P[3] = v[0];
  P[4] = v[1];
  P[5] = v[2];
  if (kind == LSAMD_ROWS_TANGENT) {
    double a[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) a[k] = (v[0] * T[k] + v[1] * T[8 + k]) + v[2] * T[16 + k];
    double bv = 0.0;
    const double len = normalise8(a, &bv);
    emit_row(i, id, a, bv, wscale, len, cols, coef, b, w, norm);
    return;
  }
  double s[3], dv[3];
  double vv[3] = {v[0], v[1], v[2]};
  strike_dip(vv, s, dv);
  double a[8], c2[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    a[k] = (s[0] * T[k] + s[1] * T[8 + k]) + s[2] * T[16 + k];
    c2[k] = (dv[0] * T[k] + dv[1] * T[8 + k]) + dv[2] * T[16 + k];
  }
  double b0 = 0.0, b1 = 0.0;
  const double l0 = normalise8(a, &b0);
  const double l1 = normalise8(c2, &b1);
  emit_row(i, id, a, b0, wscale, l0, cols, coef, b, w, norm);
  emit_row(n + i, id, c2, b1, wscale, l1, cols, coef, b, w, norm);
}

// values[i] and gradient of one point from its located cell and the cell's
// corner coefficients, as numpy evaluates them
__device__ inline void eval_point(const GridDev& g, const double* __restrict__ c, double px,
                                  double py, double pz, double* val, double* gr) {
  const Located L = locate(g, px, py, pz);
  *val = isnan(px) || isnan(py) || isnan(pz) ? 0.0 : __builtin_nan("");
  gr[0] = gr[1] = gr[2] = 0.0;
  if (!L.inside) return;
  int64_t id[8];
  corner_ids(g, L, id);
  double a[8], T[24];
  trilinear(L.lx, L.ly, L.lz, a);
  shape_grad(L.lx, L.ly, L.lz, L.hx, L.hy, L.hz, T);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const double cv = c[id[k]];
    a[k] *= cv;
    T[k] *= cv;
    T[8 + k] *= cv;
    T[16 + k] *= cv;
  }
  *val = sum8(a);
  gr[0] = sum8(T);
  gr[1] = sum8(T + 8);
  gr[2] = sum8(T + 16);
}

// What an evaluation on a uniform grid computes once: the bounds of the
// inside test and the rounded reciprocal of each step.
struct EvalGrid {
  double lo[3], hi[3], y[3];
};

inline EvalGrid to_eval(const lsamd_grid& g) {
  EvalGrid e;
  for (int a = 0; a < 3; ++a) {
    const double o = g.origin[a], mx = o + (double)(g.nnodes[a] - 1) * g.step[a];
    double ext = fabs(mx - o);
    ext = ext > 1.0 ? ext : 1.0;
    e.lo[a] = o - kEps32 * ext;
    e.hi[a] = mx + kEps32 * ext;
    e.y[a] = 1.0 / g.step[a];
  }
  return e;
}

typedef double pair_t __attribute__((ext_vector_type(2), aligned(8)));

// eval_point on a uniform grid whose steps are known divisors, bit for bit
// the same: the steps' reciprocals replace the divisions (div_known), and the
// 24 gradient weights come from the 12 that differ in more than their sign
// (1 - y is -(y - 1) exactly, and a product's sign does not change its
// rounding).  False where a dividend is out of range (the caller takes
// eval_point); cells past int32 node ids stay with 64-bit offsets.
// QUAD: c is the corners' copy (k_eval_quad).
template <bool QUAD>
__device__ inline bool eval_point_known(const GridDev& g, const EvalGrid& e,
                                        const double* __restrict__ c, double px, double py,
                                        double pz, double* val, double* gr) {
  *val = isnan(px) || isnan(py) || isnan(pz) ? 0.0 : __builtin_nan("");
  gr[0] = gr[1] = gr[2] = 0.0;
  if (!(px >= e.lo[0] && px <= e.hi[0] && py >= e.lo[1] && py <= e.hi[1] && pz >= e.lo[2] &&
        pz <= e.hi[2]))
    return true;
  auto cell = [](double d, double h, double y, int nn) {
    const int k = (int)floor(div_known(d, h, y));
    return k < 0 ? 0 : (k > nn - 2 ? nn - 2 : k);
  };
  const double dx = px - g.ox, dy = py - g.oy, dz = pz - g.oz;
  bool ok = div_known_dividend(dx) && div_known_dividend(dy) && div_known_dividend(dz);
  const int cx = cell(dx, g.hx, e.y[0], g.nx);
  const int cy = cell(dy, g.hy, e.y[1], g.ny);
  const int cz = cell(dz, g.hz, e.y[2], g.nz);
  const int64_t nx = g.nx, nxy = nx * g.ny;
  const int64_t at = cx + nx * cy + nxy * cz;
  double cv[8];
  auto ld = [](const double* p, double& a, double& b) {
    const pair_t v = *(const pair_t*)p;
    a = v.x;
    b = v.y;
  };
  if constexpr (QUAD) {
    const double* c0 = c + 4 * at;
    ld(c0, cv[0], cv[2]);
    ld(c0 + 2, cv[4], cv[6]);
    ld(c0 + 4, cv[1], cv[3]);
    ld(c0 + 6, cv[5], cv[7]);
  } else {
    const double* c0 = c + at;
    ld(c0, cv[0], cv[1]);
    ld(c0 + nx, cv[2], cv[3]);
    ld(c0 + nxy, cv[4], cv[5]);
    ld(c0 + nxy + nx, cv[6], cv[7]);
  }
  const double ax = px - (g.ox + g.hx * (double)cx), ay = py - (g.oy + g.hy * (double)cy);
  const double az = pz - (g.oz + g.hz * (double)cz);
  ok = ok && div_known_dividend(ax) && div_known_dividend(ay) && div_known_dividend(az);
  const double x = clip01(div_known(ax, g.hx, e.y[0]));
  const double y = clip01(div_known(ay, g.hy, e.y[1]));
  const double z = clip01(div_known(az, g.hz, e.y[2]));
  const double x1 = 1 - x, y1 = 1 - y, z1 = 1 - z;
  // products of two factors, shared by the weights and the gradients
  const double yz00 = y1 * z1, yz10 = y * z1, yz01 = y1 * z, yz11 = y * z;
  const double xz00 = x1 * z1, xz10 = x * z1, xz01 = x1 * z, xz11 = x * z;
  const double xy00 = x1 * y1, xy10 = x * y1, xy01 = x1 * y, xy11 = x * y;
  for (const double d : {yz00, yz10, yz01, yz11, xz00, xz10, xz01, xz11, xy00, xy10, xy01, xy11})
    ok = ok && div_known_dividend(d);
  if (!ok) return false;
  const double w[8] = {xy00 * z1, xy10 * z1, xy01 * z1, xy11 * z1,
                       xy00 * z,  xy10 * z,  xy01 * z,  xy11 * z};
  double a[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) a[k] = w[k] * cv[k];
  *val = sum8(a);
  // gradient weights of the corner pairs along each axis
  const double p0 = div_known(yz00, g.hx, e.y[0]), p1 = div_known(yz10, g.hx, e.y[0]);
  const double p2 = div_known(yz01, g.hx, e.y[0]), p3 = div_known(yz11, g.hx, e.y[0]);
  const double tx[8] = {-p0 * cv[0], p0 * cv[1], -p1 * cv[2], p1 * cv[3],
                        -p2 * cv[4], p2 * cv[5], -p3 * cv[6], p3 * cv[7]};
  gr[0] = sum8(tx);
  const double q0 = div_known(xz00, g.hy, e.y[1]), q1 = div_known(xz10, g.hy, e.y[1]);
  const double q2 = div_known(xz01, g.hy, e.y[1]), q3 = div_known(xz11, g.hy, e.y[1]);
  const double ty[8] = {-q0 * cv[0], -q1 * cv[1], q0 * cv[2], q1 * cv[3],
                        -q2 * cv[4], -q3 * cv[5], q2 * cv[6], q3 * cv[7]};
  gr[1] = sum8(ty);
  const double r0 = div_known(xy00, g.hz, e.y[2]), r1 = div_known(xy10, g.hz, e.y[2]);
  const double r2 = div_known(xy01, g.hz, e.y[2]), r3 = div_known(xy11, g.hz, e.y[2]);
  const double tz[8] = {-r0 * cv[0], -r1 * cv[1], -r2 * cv[2], -r3 * cv[3],
                        r0 * cv[4],  r1 * cv[5],  r2 * cv[6],  r3 * cv[7]};
  gr[2] = sum8(tz);
  return true;
}

// Scattered points read four pieces of c each, from lines that no neighbour
// shares: past the L2 that is what an evaluation waits for.  The table holds
// for each node the four values c(i, j..j+1, k..k+1) side by side, so that a
// point's eight corners are 64 bytes in one place: 1e7 random points on 128^3
// nodes 598 -> 306 us, of which 25 us make the table.
// Points in some order share their lines and would only pay for the table: 252
// pairs of neighbours in four places of the list are looked at, and the
// table is filled (ws[0] = 1) where fewer than half of them are within two
// cells of each other.
constexpr int kQuadHead = 16;      // doubles before the table
constexpr int kQuadBlocks = 1024;  // every workgroup looks at the points: few
__global__ __launch_bounds__(256) void k_eval_quad(GridDev g, EvalGrid e,
                                                   const double* __restrict__ c,
                                                   const double* __restrict__ pts, int64_t n,
                                                   double* __restrict__ ws) {
  __shared__ int sh[4];
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int64_t s = (n - 64) / 4 * wave + lane;  // n >= 64
  float q[3];
  const double o[3] = {g.ox, g.oy, g.oz};
  int near = lane < 63;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    q[a] = (float)((pts[3 * s + a] - o[a]) * e.y[a]);
    near = near && fabsf(q[a] - __shfl_down(q[a], 1, 64)) <= 2.f;
  }
  const int cnt = __popcll(__ballot(near));
  if (lane == 0) sh[wave] = cnt;
  __syncthreads();
  const bool fill = sh[0] + sh[1] + sh[2] + sh[3] < 126;
  if (blockIdx.x == 0 && t == 0) ws[0] = fill ? 1.0 : 0.0;
  if (!fill) return;
  const int64_t nx = g.nx, nxy = nx * g.ny, nn = nxy * g.nz;
  typedef double quad_t __attribute__((ext_vector_type(4)));
  for (int64_t i = (int64_t)blockIdx.x * 256 + t; i < nn; i += (int64_t)gridDim.x * 256) {
    // past the last row or plane: any value, no cell has its corners there
    const int64_t a = i + nx < nn ? i + nx : i, b = i + nxy < nn ? i + nxy : i;
    const int64_t d = i + nx + nxy < nn ? i + nx + nxy : i;
    *(quad_t*)(ws + kQuadHead + 4 * i) = quad_t{c[i], c[a], c[b], c[d]};
  }
}

// Values and gradients at n points.  A workgroup's points come in, and its
// gradients leave, through LDS in whole lines (a thread's own three doubles
// lie 24 bytes from its neighbour's).  KNOWN: uniform grid with steps that
// div_known takes.  QUAD: corners from the table of k_eval_quad, where that has
// been filled.  STREAM: points are read past the caches (see eval_streams).
constexpr int kEvalBlock = 256;
template <bool KNOWN, bool QUAD, bool STREAM>
__global__ __launch_bounds__(kEvalBlock) void k_evaluate(GridDev g, EvalGrid e,
                                                         const double* __restrict__ c,
                                                         const double* __restrict__ ws,
                                                         const double* __restrict__ pts,
                                                         int64_t n, double* __restrict__ vals,
                                                         double* __restrict__ grads) {
  __shared__ double sh[3 * kEvalBlock];
  const int t = threadIdx.x;
  const int64_t b = (int64_t)blockIdx.x * kEvalBlock;
  const int m = (int)(n - b < kEvalBlock ? n - b : kEvalBlock);
  const bool quad = QUAD && ws[0] != 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (t + k * kEvalBlock < 3 * m)
      sh[t + k * kEvalBlock] = eval_ld<STREAM>(pts + 3 * b + t + k * kEvalBlock);
  __syncthreads();
  double val = 0.0, gr[3] = {0.0, 0.0, 0.0};
  if (t < m) {
    const double px = sh[3 * t], py = sh[3 * t + 1], pz = sh[3 * t + 2];
    bool ok = false;
    if constexpr (KNOWN)
      ok = quad ? eval_point_known<true>(g, e, ws + kQuadHead, px, py, pz, &val, gr)
                : eval_point_known<false>(g, e, c, px, py, pz, &val, gr);
    if (!ok) eval_point(g, c, px, py, pz, &val, gr);
    if (vals) __builtin_nontemporal_store(val, vals + b + t);
  }
  if (!grads) return;
  // a thread overwrites only the three entries that it alone has read
  if (t < m) {
    sh[3 * t] = gr[0];
    sh[3 * t + 1] = gr[1];
    sh[3 * t + 2] = gr[2];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (t + k * kEvalBlock < 3 * m)
      __builtin_nontemporal_store(sh[t + k * kEvalBlock], grads + 3 * b + t + k * kEvalBlock);
}

// numpy's pairwise summation of a contiguous run of n <= 128 doubles
// (n < 8: sequential from 0; else eight interleaved accumulators).
__device__ inline double np_sum(const double* a, int n) {
  if (n < 8) {
    double r = 0.0;
    for (int i = 0; i < n; ++i) r += a[i];
    return r;
  }
  double r[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = a[j];
  int i = 8;
  for (; i < n - (n % 8); i += 8)
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] += a[i + j];
  double res = ((r[0] + r[1]) + (r[2] + r[3])) + ((r[4] + r[5]) + (r[6] + r[7]));
  for (; i < n; ++i) res += a[i];
  return res;
}

__global__ void k_rows_normalise(int64_t nrows, int k, double* __restrict__ coef,
                                 double* __restrict__ b, double* __restrict__ norm) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  double sq[128];
  double* a = coef + r * k;
  for (int j = 0; j < k; ++j) sq[j] = a[j] * a[j];
  const double len = sqrt(np_sum(sq, k));
  if (len > 0) {
    b[r] /= len;
    for (int j = 0; j < k; ++j) a[j] /= len;
  }
  if (norm) norm[r] = len;
}

// (node, point entry, w_k * gv) for the 8 corners of every point; outside
// points give zero contributions to node 0.
__global__ void k_eval_entries(GridDev g, const double* __restrict__ pts,
                               const double* __restrict__ gv, int64_t n,
                               int32_t* __restrict__ key, int32_t* __restrict__ idx,
                               double* __restrict__ val) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const Located L = locate(g, pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]);
  int64_t id[8];
  corner_ids(g, L, id);
  double a[8];
  trilinear(L.lx, L.ly, L.lz, a);
  for (int k = 0; k < 8; ++k) {
    const int64_t e = 8 * i + k;
    key[e] = L.inside ? (int32_t)id[k] : 0;
    idx[e] = (int32_t)e;
    val[e] = L.inside ? a[k] * gv[i] : 0.0;
  }
}

}  // namespace

void launch_eval_entries(const GridDev& g, const double* pts, const double* gv, int64_t n,
                         int32_t* key, int32_t* idx, double* val, hipStream_t st) {
  hipLaunchKernelGGL(k_eval_entries, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, st, g, pts,
                     gv, n, key, idx, val);
}

}  // namespace lsamd

using namespace lsamd;

extern "C" int lsamd_rows_normalise(int64_t nrows, int32_t k, double* coef, double* b,
                                    double* norm, void* stream) {
  if (int rc = injected("rows_normalise")) return rc;
  if (nrows < 0 || k < 1 || k > 128)
    return fail(LSAMD_ERR_ARG, "lsamd_rows_normalise: need nrows >= 0 and 1 <= k <= 128");
  if (nrows == 0) return LSAMD_OK;
  if (!coef || !b) return fail(LSAMD_ERR_ARG, "lsamd_rows_normalise: NULL input");
  const int bs = 64;
  hipLaunchKernelGGL(k_rows_normalise, dim3((unsigned)ceil_div(nrows, bs)), dim3(bs), 0,
                     (hipStream_t)stream, nrows, (int)k, coef, b, norm);
  LSAMD_CHECK_LAUNCH("k_rows_normalise");
  return LSAMD_OK;
}

extern "C" int lsamd_fd_locate(const lsamd_grid* g, const double* pts, int64_t n, int64_t* idc,
                               double* w, double* T, uint8_t* inside, void* stream) {
  if (int rc = injected("locate")) return rc;
  if (int rc = check_grid(g)) return rc;
  if (n < 0) return fail(LSAMD_ERR_ARG, "lsamd_fd_locate: n < 0");
  if (n == 0) return LSAMD_OK;
  if (!pts) return fail(LSAMD_ERR_ARG, "lsamd_fd_locate: pts is NULL");
  const int bs = 256;
  hipLaunchKernelGGL(k_locate, dim3((unsigned)ceil_div(n, bs)), dim3(bs), 0, (hipStream_t)stream,
                     to_dev(*g), pts, n, idc, w, T, inside);
  LSAMD_CHECK_LAUNCH("k_locate");
  return LSAMD_OK;
}

extern "C" int lsamd_fd_build_rows(const lsamd_grid* g, int32_t kind, double* pts, int64_t n,
                                   int64_t ld, int32_t weight_col, double wscale, int32_t* cols,
                                   double* coef, double* b, double* w, double* norm,
                                   void* stream) {
  if (int rc = injected("build_rows")) return rc;
  if (int rc = check_grid(g)) return rc;
  if (kind < LSAMD_ROWS_VALUE || kind > LSAMD_ROWS_TANGENT)
    return fail(LSAMD_ERR_ARG, "lsamd_fd_build_rows: unknown row kind");
  const int need = (kind == LSAMD_ROWS_VALUE) ? 4 : 6;
  if (ld < need) return fail(LSAMD_ERR_ARG, "lsamd_fd_build_rows: ld too small for row kind");
  if (weight_col >= ld) return fail(LSAMD_ERR_ARG, "lsamd_fd_build_rows: weight_col >= ld");
  if (n < 0) return fail(LSAMD_ERR_ARG, "lsamd_fd_build_rows: n < 0");
  if (n == 0) return LSAMD_OK;
  if (!pts || !cols || !coef || !b || !w)
    return fail(LSAMD_ERR_ARG, "lsamd_fd_build_rows: NULL output");
  const int64_t nn = g->nnodes[0] * g->nnodes[1] * g->nnodes[2];
  if (nn > 2147483647LL)
    return fail(LSAMD_ERR_ARG, "lsamd_fd_build_rows: grid exceeds int32 node ids");
  const int bs = 128;
  hipLaunchKernelGGL(k_build_rows, dim3((unsigned)ceil_div(n, bs)), dim3(bs), 0,
                     (hipStream_t)stream, to_dev(*g), (int)kind, pts, n, ld, (int)weight_col,
                     wscale, cols, coef, b, w, norm);
  LSAMD_CHECK_LAUNCH("k_build_rows");
  return LSAMD_OK;
}

// Where the table of k_eval_quad is worth a look at the points: c well past an
// L2 (scattered points on 80^3 nodes, 1e6 of them: 32 us without, 42 with the
// table), no more nodes than points (200^3 nodes, scattered: 1e6 points 82, 131;
// 2e6 160, 168; 3e6 238, 196), and so many points that the look, 2.2 us, is
// little beside them.  The last is a trade: scattered points would gain from
// 1e6 on, points in order pay the look and gain nothing.  On 128^3 nodes,
// scattered without and with the table, and in order: 1e6 64, 51 and 32 us; 2e6
// 123, 79 and 45; 3e6 183, 107 and 57; 4e6 242, 136 and 70, where the look is 3%.
// (The package's _SCRATCH_POINTS saves fewer points than this the call that
// asks.)
constexpr int64_t kQuadNodesMin = 1 << 20, kQuadPointsMin = 1 << 22;
static bool eval_quad_takes(const lsamd_grid* g, int64_t n) {
  const int64_t nn = (int64_t)g->nnodes[0] * g->nnodes[1] * g->nnodes[2];
  return nn >= kQuadNodesMin && n >= kQuadPointsMin && n >= nn && !g->axis_nodes[0] &&
         div_known_divisor(g->step[0]) && div_known_divisor(g->step[1]) &&
         div_known_divisor(g->step[2]);
}

extern "C" int lsamd_fd_evaluate_scratch(const lsamd_grid* g, int64_t n, int64_t* bytes) {
  if (int rc = check_grid(g)) return rc;
  if (!bytes) return fail(LSAMD_ERR_ARG, "lsamd_fd_evaluate_scratch: NULL output");
  const int64_t nn = (int64_t)g->nnodes[0] * g->nnodes[1] * g->nnodes[2];
  *bytes = eval_quad_takes(g, n) ? (kQuadHead + 4 * nn) * 8 : 0;
  return LSAMD_OK;
}

extern "C" int lsamd_fd_evaluate_with(const lsamd_grid* g, const double* c, const double* pts,
                                      int64_t n, double* values, double* grads, void* scratch,
                                      void* stream) {
  if (int rc = injected("evaluate")) return rc;
  if (int rc = check_grid(g)) return rc;
  if (n < 0) return fail(LSAMD_ERR_ARG, "lsamd_fd_evaluate: n < 0");
  if (n == 0) return LSAMD_OK;
  if (!c || !pts) return fail(LSAMD_ERR_ARG, "lsamd_fd_evaluate: NULL input");
  if ((uintptr_t)scratch % 32) return fail(LSAMD_ERR_ARG, "lsamd_fd_evaluate: scratch alignment");
  const dim3 nb((unsigned)ceil_div(n, kEvalBlock)), bs(kEvalBlock);
  const EvalGrid e = to_eval(*g);
  const hipStream_t st = (hipStream_t)stream;
  double* ws = (double*)scratch;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, nb, bs, 0, st, to_dev(*g), e, c, (const double*)ws, pts, n, values,
                       grads);
  };
  const bool known = !g->axis_nodes[0] && div_known_divisor(g->step[0]) &&
                     div_known_divisor(g->step[1]) && div_known_divisor(g->step[2]);
  const bool past = eval_streams(n, values, grads);
  if (ws && eval_quad_takes(g, n)) {
    hipLaunchKernelGGL(k_eval_quad, dim3(kQuadBlocks), dim3(256), 0, st, to_dev(*g), e, c, pts, n,
                       ws);
    launch(past ? k_evaluate<true, true, true> : k_evaluate<true, true, false>);
  } else if (known) {
    launch(past ? k_evaluate<true, false, true> : k_evaluate<true, false, false>);
  } else {
    launch(past ? k_evaluate<false, false, true> : k_evaluate<false, false, false>);
  }
  LSAMD_CHECK_LAUNCH("k_evaluate");
  return LSAMD_OK;
}

extern "C" int lsamd_fd_evaluate(const lsamd_grid* g, const double* c, const double* pts,
                                 int64_t n, double* values, double* grads, void* stream) {
  return lsamd_fd_evaluate_with(g, c, pts, n, values, grads, nullptr, stream);
}
