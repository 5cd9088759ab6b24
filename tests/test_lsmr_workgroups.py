"""The LSMR kernels on the CPU, one workgroup at a time and its wavefronts one
after the other: what another workgroup of the same launch stores while a
workgroup runs must not split its wavefronts at a barrier."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "loopstructural_amd", "csrc")

HARNESS = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>
#include <vector>
#define __global__
#define __device__
#define __shared__ static
#define __launch_bounds__(...)

// ---- a workgroup: one fibre per thread ----
struct Idx { int x; };
enum { RUN, BARRIER, WAVE, END };
struct Fibre {
  ucontext_t ctx;
  int state;
  Idx tid;
  double shfl[2];
  int nsh;
};
static std::vector<Fibre> fib;
static Fibre* cur;
static ucontext_t sched;
static Idx blockIdx, blockDim, gridDim;
#define threadIdx (cur->tid)
static void yield_as(int s) {
  cur->state = s;
  swapcontext(&cur->ctx, &sched);
}
static void __syncthreads() { yield_as(BARRIER); }
static double __shfl_xor(double v, int o, int) {
  Fibre* me = cur;
  const int p = me->nsh++ & 1;
  me->shfl[p] = v;
  yield_as(WAVE);
  return fib[me->tid.x ^ o].shfl[p];
}

// ---- what lsmr.hpp takes from the other sources ----
namespace lsamd {
struct GridDev { int nx, ny, nz; };
template <typename T> struct RegW { T ridge; };
struct RowsDev {
  int64_t nrows;
  const int64_t* row_ptr;
  const int32_t* cols;
  const void *coef, *w2;
  int64_t ndn;
  const int64_t* seg_ptr;
  const int32_t *seg_entry, *seg_row, *dnode;
};
enum { F_XX, F_YY, F_ZZ, F_XY, F_XZ, F_YZ };
static bool in_grid(const GridDev& g, int i, int j, int k) {
  return i >= 0 && i < g.nx && j >= 0 && j < g.ny && k >= 0 && k < g.nz;
}
static double row_weight(const GridDev& g, const RegW<double>&, const double*, int, int i, int j,
                         int k) {
  return i > 0 && i < g.nx - 1 && j > 0 && j < g.ny - 1 && k > 0 && k < g.nz - 1 ? 0.01 : 0.0;
}
static double wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
static double pcg_total(const double* part, int n, double* sh) {
  double v = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) v += part[i];
  v = wave_sum(v);
  if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = v;
  __syncthreads();
  double t = 0.0;
  for (int i = 0; i < blockDim.x / 64; ++i) t += sh[i];
  __syncthreads();
  return t;
}
static double block_sum(double v, double* sh) {
  v = wave_sum(v);
  if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = v;
  __syncthreads();
  double t = 0.0;
  for (int i = 0; i < blockDim.x / 64; ++i) t += sh[i];
  return t;
}
}  // namespace lsamd
#include "lsmr.hpp"
using namespace lsamd;

// ---- the launches, on a grid of one workgroup of nodes and a few rows ----
static const int NX = 6, N = NX * NX * NX, ROWS = 3;
static double xs[N], uw[6 * N], urid[N], v[N], h[N], hbar[N], x[N], sv[N], ud[ROWS], wr[ROWS],
    b[ROWS], cw[8 * ROWS], coef[8 * ROWS], pu[8], pv[8], px[8];
static int64_t row_ptr[ROWS + 1], seg_ptr[8 * ROWS + 1];
static int32_t cols[8 * ROWS], seg_entry[8 * ROWS], seg_row[8 * ROWS], dnode[8 * ROWS];
static uint64_t mask[(N + 63) / 64];
static LsCtl ctl[2];
static LsEst est[2];
static LsMid mid;
static int kernel;

static void body() {
  const GridDev g = {NX, NX, NX};
  const RegW<double> w = {1e-16};
  const RowsDev R = {ROWS, row_ptr, cols, coef, wr, 8 * ROWS, seg_ptr, seg_entry, seg_row, dnode};
  if (kernel == 0)
    k_ls_fwd(xs, g, w, nullptr, uw, urid, N, R, wr, b, ud, 1, 0, pu, ctl, &mid);
  else if (kernel == 1)
    k_ls_bwd(uw, urid, g, 1e-8, R, cw, ud, mask, sv, v, N, 1, 0, pu, 2, pv, ctl, est + 1, est, px,
             1, &mid);
  else
    k_ls_rot(v, h, hbar, x, xs, sv, N, 0, pv, 2, px, ctl, ctl + 1, est, &mid);
  yield_as(END);
}

static int groups() { return kernel == 0 ? 2 : kernel == 1 ? 3 : 1; }

// Runs workgroup `blk`; after wavefront `at` has run up to its first barrier
// (-1: never) the bytes `next` replace those of mid.  1: some wavefronts of
// the workgroup ended while others waited at a barrier.
static int run(int blk, int at, const LsMid* next) {
  static std::vector<char> stacks;
  const int T = 256, SZ = 1 << 16;
  stacks.resize((size_t)T * SZ);
  fib.assign(T, Fibre());
  blockIdx.x = blk;
  blockDim.x = T;
  gridDim.x = groups();
  for (int t = 0; t < T; ++t) {
    Fibre& f = fib[t];
    f.tid.x = t;
    f.state = RUN;
    getcontext(&f.ctx);
    f.ctx.uc_stack.ss_sp = stacks.data() + (size_t)t * SZ;
    f.ctx.uc_stack.ss_size = SZ;
    f.ctx.uc_link = nullptr;
    makecontext(&f.ctx, body, 0);
  }
  for (int trip = 0;; ++trip) {
    for (int wv = 0; wv < T / 64; ++wv) {
      for (bool more = true; more;) {  // the wavefront, up to a barrier or its end
        more = false;
        for (int t = wv * 64; t < wv * 64 + 64; ++t)
          if (fib[t].state == RUN) {
            cur = &fib[t];
            swapcontext(&sched, &cur->ctx);
          }
        for (int t = wv * 64; t < wv * 64 + 64; ++t)
          if (fib[t].state == WAVE) fib[t].state = RUN, more = true;
      }
      if (trip == 0 && wv == at) mid = *next;
    }
    int nb = 0, ne = 0;
    for (auto& f : fib) nb += f.state == BARRIER, ne += f.state == END;
    if (nb && ne) return 1;
    if (!nb) return 0;
    for (auto& f : fib) f.state = RUN;
  }
}

int main() {
  for (int i = 0; i < N; ++i) {
    xs[i] = sin(i), v[i] = cos(i), h[i] = sin(2 * i), sv[i] = 1.0, urid[i] = 0.1;
    for (int f = 0; f < 6; ++f) uw[f * N + i] = cos(f + i);
  }
  for (int r = 0; r < ROWS; ++r) {
    row_ptr[r + 1] = 8 * (r + 1), wr[r] = 1.0, b[r] = 1.0, ud[r] = 0.5;
    for (int e = 8 * r; e < 8 * r + 8; ++e) {
      cols[e] = dnode[e] = 50 + e, coef[e] = cw[e] = 0.3, seg_entry[e] = e, seg_row[e] = r;
      seg_ptr[e + 1] = e + 1;
      mask[cols[e] / 64] |= 1ull << (cols[e] % 64);
    }
  }
  pu[0] = pu[1] = pv[0] = pv[1] = px[0] = 1.0;
  ctl[0].alpha = ctl[0].beta = ctl[0].alphabar = ctl[0].rho = ctl[0].rhobar = ctl[0].cbar = 1.0;
  ctl[0].zeta = ctl[0].zetabar = ctl[0].rhobarold = ctl[0].rhotemp = ctl[0].chat = 1.0;
  ctl[0].itn = 1;  // with maxiter 1: the tests of this step end the solve
  est[1] = LsEst{1.0, 0.0, 1.0, 0.0, 0.0, 1.0, 0.0, 1e100};
  mid.maxiter = 1;
  mid.normb = mid.beta = mid.inv_beta = 1.0;
  const LsMid start = mid;
  int ended = 0;
  for (kernel = 0; kernel < 3; ++kernel)
    for (int writer = 0; writer < groups(); ++writer) {
      mid = start;
      if (run(writer, -1, nullptr)) return printf("kernel %d splits by itself\n", kernel), 2;
      const LsMid after = mid;
      ended |= kernel == 1 && after.done;
      for (int blk = 0; blk < groups(); ++blk)
        for (int at = 0; blk != writer && at < 3; ++at) {
          mid = start;
          if (run(blk, at, &after))
            return printf("kernel %d: workgroup %d splits after wavefront %d on the stores of "
                          "workgroup %d\n", kernel, blk, at, writer), 1;
        }
    }
  if (!ended) return printf("the solve was to end\n"), 3;
  printf("ok\n");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a C++ compiler")
def test_lsmr_workgroups_stay_whole(tmp_path):
    src, exe = tmp_path / "lsmr_waves.cpp", tmp_path / "lsmr_waves"
    src.write_text(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", f"-I{CSRC}", str(src), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
