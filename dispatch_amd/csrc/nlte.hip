// Per-cell statistical equilibrium in FP64 for gfx950: the rate-matrix assembly of
// setup_transition_matrix (SRC/atom_mod.f90:740-851, line_rate_coefficients
// 862-884), the no-pivot LU of lineq_no_pivot (HOP/op_math_mod.f90:420-449) and
// the update of update_populations (SRC/atom_mod.f90:439-732): limiter,
// under-relaxation, particle conservation, population floor and the convergence
// measure.  Also the rate normalisation of normalize_profiles (377-431).
//
// Mapping.  Sixteen lanes per cell, four cells a wavefront (many cells of few levels: four
// lanes, rate_solve).  A workgroup of NT cells keeps every cell's nk x nk matrix,
// right-hand side and b*n* vector in LDS, one cell after another.  A cell's lanes share its
// elimination as a 4 x 4 (2 x 2) grid over the rows and columns left, and otherwise take its levels in turn; they lie in one wavefront, whose
// LDS accesses are in order, so no barrier is needed between the steps.  Every element
// sees the operations of the sequential algorithm in its order, so the results are
// those of one lane per cell.  What bounds it is the latency of the dependent steps
// (LDS, FP64): a cell's matrix (3.9 KB at 21 levels) allows 40 cells a CU, which with one
// lane each were a single wave.  432 000 cells of 21 levels: 12.7 -> 3.7 ms.
// The atom (levels, transitions, pairs) is uniform and read through the scalar
// cache.  The largest change and the per-level changes are reduced first per
// workgroup and then by one workgroup each, both keeping the first cell in the
// reference's loop order on ties, so the result is deterministic.
#include "m3drt_internal.hpp"
#include <cmath>
#include <algorithm>
#include <vector>

namespace m3drt {

namespace {

struct SeArgs {
  int nk, nrad, nline, npair, ncell, nt;
  const int32_t *ti, *tj, *active, *pi, *pj;
  const double *g, *ev, *Aji;
  const double *e_kT, *temp, *totn, *nstar, *cup;
  double *b;
  const float *gij, *gji;
  double max_update, min_pop_frac, conv_pop_floor, sor_w, cswitch, cut_x, bf_cut_rate, tmax_update;
  double *blk_err;       // (nblk) signed weighted change of the block's winner
  int32_t *blk_cell;     // (nblk) its cell, -1 for none
  int32_t *blk_lvl;      // (nblk) its level
  double *blk_lerr;      // (nblk, nk) per-level signed change
  int32_t *blk_lcell;    // (nblk, nk) its cell
  unsigned long long *nclamp;
  int32_t *status;       // smallest 1-based cell without a finite solution
};

// keep the larger |value|; on ties the smaller cell (earlier in the reference's loop)
__device__ __forceinline__ bool better(double va, int ca, double vb, int cb) {
  if (cb < 0) return ca >= 0;
  if (ca < 0) return false;
  const double a = fabs(va), b = fabs(vb);
  return a > b || (a == b && ca < cb);
}

// cells of a workgroup at most, with LANES lanes a cell
template <int LANES>
constexpr int se_cells() { return LANES == 16 ? 40 : 64; }

// doubles of a cell in LDS: matrix, right-hand side, b*n*; odd, so that the cells of a
// wavefront start on different banks
__host__ __device__ __forceinline__ int se_stride(int nk) { return (nk * nk + 2 * nk) | 1; }

template <int LANES>
__global__ void __launch_bounds__(LANES *se_cells<LANES>()) se_update_kernel(const SeArgs a) {
  extern __shared__ double sm[];
  const int nk = a.nk, NT = a.nt;
  const int t = threadIdx.x / LANES, p = threadIdx.x % LANES;
  const int c = blockIdx.x * NT + t;
  double *W = sm + (size_t)t * se_stride(nk);    // nk*nk
  double *E = W + (size_t)nk * nk;               // nk
  double *BN = E + nk;                           // nk (b*n*, then b_old)
  double *RV = sm + (size_t)NT * se_stride(nk);  // NT reduction values
  int *RC = reinterpret_cast<int *>(RV + NT);    // NT cells, NT levels
#define Wm(i, j) W[(i) * nk + (j)]
#define Ev(i) E[i]
#define Bv(i) BN[i]
  // orders a cell's LDS accesses between its lanes (one wavefront: no barrier needed)
  auto sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  const bool live = c < a.ncell && a.totn[c] > 0 && a.temp[c] < a.tmax_update;
  double my_err = 0.0;
  int my_lvl = -1;
  unsigned long long clamps = 0;
  if (live) {
    const double ekt = a.e_kT[c];
    auto NS = [&](int i) { return a.nstar[(size_t)i * a.ncell + c]; };
    for (int e = p; e < nk * nk; e += LANES) W[e] = 0.0;
    for (int i = p; i < nk; i += LANES) Ev(i) = 0.0;
    sync();
    // The rates of as many transitions at a time as lanes, one a lane, then added in their order:
    // lane 0 the upward rate to W(j, i), lane 1 the downward one to W(i, j).
    auto add = [&](int i, int j, double up, double down) {
      if (i == j) {
        if (p == 0) Wm(i, i) = (Wm(i, i) + up) + down;
      } else if (p < 2) {
        double *w = p ? &Wm(i, j) : &Wm(j, i);
        *w = *w + (p ? down : up);
      }
      sync();
    };
    for (int k0 = 0; k0 < a.nrad; k0 += LANES) {
      const int kr = k0 + p;
      double r_up = 0.0, r_down = 0.0;
      if (kr < a.nrad && a.active[kr]) {
        const int i = a.ti[kr] - 1, j = a.tj[kr] - 1;
        if ((a.ev[j] - a.ev[i]) * ekt > a.cut_x) {
          // a detailed-balance pair for a transition beyond cut_x kT
          const double cut = kr < a.nline ? a.Aji[kr] : a.bf_cut_rate;
          r_down = cut;
          r_up = cut * NS(j) / NS(i);
        } else if (kr < a.nline) {
          const double th = a.gij[(size_t)kr * a.ncell + c], dev = a.gji[(size_t)kr * a.ncell + c];
          const double g_ij = a.g[i] / a.g[j];
          if (NS(i) > 0 && NS(j) > 0) {
            const double beta = NS(j) * g_ij / NS(i);
            r_up = th * (beta / (1.0 - beta)) + dev;
            r_down = g_ij * (th / (1.0 - beta) + dev);
          }
        } else {
          r_up = a.gij[(size_t)kr * a.ncell + c];
          r_down = a.gji[(size_t)kr * a.ncell + c];
        }
      }
      for (int q = 0; q < LANES && k0 + q < a.nrad; ++q) {
        if (!a.active[k0 + q]) continue;
        add(a.ti[k0 + q] - 1, a.tj[k0 + q] - 1, __shfl(r_up, q, LANES), __shfl(r_down, q, LANES));
      }
    }
    if (a.cswitch > 0 && a.cup) {
      for (int q0 = 0; q0 < a.npair; q0 += LANES) {
        const int q = q0 + p;
        double up = 0.0, down = 0.0;
        if (q < a.npair) {
          const int i = a.pi[q] - 1, j = a.pj[q] - 1;
          const double cu = a.cup[(size_t)q * a.ncell + c];
          if (cu != 0) {
            up = cu * a.cswitch;
            down = cu * (NS(i) / NS(j)) * a.cswitch;
          }
        }
        for (int m = 0; m < LANES && q0 + m < a.npair; ++m)
          add(a.pi[q0 + m] - 1, a.pj[q0 + m] - 1, __shfl(up, m, LANES), __shfl(down, m, LANES));
      }
    }
    for (int i = p; i < nk; i += LANES) {
      double s = 0.0;
      for (int k = 0; k < nk; ++k) s += Wm(k, i);
      Wm(i, i) = -s;
      Bv(i) = a.b[(size_t)i * a.ncell + c] * NS(i);
    }
    sync();
    int pos = 0;
    for (int i = 0; i < nk; ++i)
      if (Bv(i) > Bv(pos)) pos = i;
    if (p == 0) Ev(pos) = a.totn[c];
    for (int j = p; j < nk; j += LANES) {
      const double bj = Bv(j);
      for (int i = 0; i < nk; ++i) Wm(i, j) = i == pos ? bj : Wm(i, j) * bj;
    }
    sync();

    // lineq_no_pivot: Doolittle without pivoting, zero upper entries skipped
    constexpr int G = LANES == 16 ? 4 : 2;
    static_assert(G * G == LANES, "a cell's lanes form a square");
    const int pi = p / G, pj = p % G;
    for (int k = 0; k < nk - 1; ++k) {
      const double akk = Wm(k, k);
      for (int i = k + 1 + p; i < nk; i += LANES) Wm(i, k) = Wm(i, k) / akk;
      sync();
      for (int j = k + 1 + pj; j < nk; j += G) {
        const double akj = Wm(k, j);
        if (akj != 0)
          for (int i = k + 1 + pi; i < nk; i += G) Wm(i, j) = Wm(i, j) - Wm(i, k) * akj;
      }
      sync();
    }
    // forward by columns (each Ev(i) takes its terms in the order of j), backward by rows
    // on every lane alike
    for (int j = 0; j < nk - 1; ++j) {
      const double ej = Ev(j);
      for (int i = j + 1 + p; i < nk; i += LANES) Ev(i) = Ev(i) - Wm(i, j) * ej;
      sync();
    }
    for (int i = nk - 1; i >= 0; --i) {
      double e = Ev(i);
      for (int j = i + 1; j < nk; ++j) e = e - Wm(i, j) * Ev(j);
      e = e / Wm(i, i);
      sync();
      if (p == 0) Ev(i) = e;
      sync();
    }
    bool finite = true;
    for (int i = 0; i < nk; ++i) finite = finite && (fabs(Ev(i)) <= 1.79769313486231570e308);
    if (!finite) {
      if (p == 0) atomicMin(a.status, c + 1);
    } else {
      const double eup = a.max_update > 1.0 ? a.max_update : 1.0, elo = 1.0 / eup;
      for (int i = p; i < nk; i += LANES) {
        double e = Ev(i);
        if (e < elo || e > eup) clamps++;
        if (e < elo)
          e = elo * exp(fmax(e, 0.0) / elo - 1.0);
        else if (e > eup)
          e = eup * (2.0 - eup / e);
        if (a.sor_w != 1.0) e = pow(e, a.sor_w);
        const double bo = a.b[(size_t)i * a.ncell + c];
        Bv(i) = bo;                       // b_old
        Ev(i) = bo * e;                   // b, before normalisation
      }
      sync();
      double sum = 0.0;
      for (int i = 0; i < nk; ++i) sum += Ev(i) * NS(i);
      const double norm = a.totn[c] / sum;
      sync();
      for (int i = p; i < nk; i += LANES) {
        const size_t o = (size_t)i * a.ncell + c;
        double bn = Ev(i) * norm;
        if (a.nstar[o] > 0) bn = fmax(bn, fmin(1.0, a.min_pop_frac * a.totn[c] / a.nstar[o]));
        a.b[o] = bn;
        const double e = Bv(i) > 0 ? bn / Bv(i) - 1.0 : 0.0;
        double ew = fabs(e);
        if (a.conv_pop_floor > 0) ew = fabs(e) * fmin(1.0, bn * a.nstar[o] / (a.conv_pop_floor * a.totn[c]));
        Ev(i) = e;                        // the change, for the per-level reduction
        Bv(i) = ew;
      }
      sync();
      double wmax = -1.0;
      for (int i = 0; i < nk; ++i)
        if (Bv(i) > wmax) {
          wmax = Bv(i);
          my_lvl = i;
        }
      // (my_lvl stays -1 where every change is NaN)
      if (my_lvl >= 0) my_err = copysign(wmax, Ev(my_lvl));
    }
  }
  if (clamps) atomicAdd(a.nclamp, clamps);

  // workgroup reduction: the largest weighted change, and every level's change, one
  // thread each
  if (p == 0) {
    RV[t] = my_err;
    RC[t] = (live && my_lvl >= 0) ? c : -1;
    RC[NT + t] = my_lvl;
  }
  __syncthreads();
  const int nblk = blockIdx.x;
  for (int q = threadIdx.x; q <= nk; q += blockDim.x) {
    double bv = 0.0;
    int bc = -1, bl = -1;
    for (int s = 0; s < NT; ++s) {
      const int cs = RC[s];
      const double v = q == nk ? RV[s] : cs >= 0 ? sm[(size_t)s * se_stride(nk) + nk * nk + q] : 0.0;
      if (better(v, cs, bv, bc)) {
        bv = v;
        bc = cs;
        bl = RC[NT + s];
      }
    }
    if (q == nk) {
      a.blk_err[nblk] = bv;
      a.blk_cell[nblk] = bc;
      a.blk_lvl[nblk] = bl;
    } else {
      a.blk_lerr[(size_t)nblk * nk + q] = bv;
      a.blk_lcell[(size_t)nblk * nk + q] = bc;
    }
  }
#undef Wm
#undef Ev
#undef Bv
}

// the blocks' winners, one workgroup per value: workgroup 0 maxerr (out[0], its cell
// iout[0] and level iout[1]), workgroup 1 + q level q (out[1 + q])
__global__ void __launch_bounds__(256) se_final_kernel(int nblk, int nk, const double *blk_err,
                                                       const int32_t *blk_cell, const int32_t *blk_lvl,
                                                       const double *blk_lerr, const int32_t *blk_lcell,
                                                       double *out, int32_t *iout) {
  __shared__ double rv[256];
  __shared__ int rc[256], rl[256];
  const int t = threadIdx.x, q = (int)blockIdx.x - 1;
  double bv = 0.0;
  int bc = -1, bl = -1;
  for (int s = t; s < nblk; s += blockDim.x) {
    const double v = q < 0 ? blk_err[s] : blk_lerr[(size_t)s * nk + q];
    const int cc = q < 0 ? blk_cell[s] : blk_lcell[(size_t)s * nk + q];
    if (better(v, cc, bv, bc)) {
      bv = v;
      bc = cc;
      bl = q < 0 ? blk_lvl[s] : q;
    }
  }
  rv[t] = bv;
  rc[t] = bc;
  rl[t] = bl;
  __syncthreads();
  for (int h = 128; h > 0; h /= 2) {
    if (t < h && better(rv[t + h], rc[t + h], rv[t], rc[t])) {
      rv[t] = rv[t + h];
      rc[t] = rc[t + h];
      rl[t] = rl[t + h];
    }
    __syncthreads();
  }
  if (t == 0) {
    out[1 + q] = rc[0] >= 0 ? rv[0] : 0.0;
    if (q < 0) {
      iout[0] = rc[0];
      iout[1] = rl[0];
    }
  }
}

__global__ void __launch_bounds__(256) normalize_kernel(int nrad, int nline, int ncell, const int32_t *active,
                                                        const int32_t *ti, const int32_t *tj,
                                                        const double *nstar, const float *wphi,
                                                        float *gij, float *gji) {
  const int64_t n = (int64_t)nrad * ncell;
  for (int64_t id = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; id < n;
       id += (int64_t)gridDim.x * blockDim.x) {
    const int kr = (int)(id / ncell), c = (int)(id % ncell);
    if (!active[kr]) continue;
    if (kr < nline) {
      if (wphi) {
        gij[id] = gij[id] * wphi[id];
        gji[id] = gji[id] * wphi[id];
      }
    } else {
      const int i = ti[kr] - 1, j = tj[kr] - 1;
      gji[id] = (float)((double)gji[id] * (nstar[(int64_t)i * ncell + c] / nstar[(int64_t)j * ncell + c]));
    }
  }
}

}  // namespace

int rate_solve(m3drt_ctx *ctx, const m3drt_rate_solve_args *r, m3drt_rate_solve_result *res) {
  const int nk = r->nk;
  const size_t per_cell = ((size_t)nk * nk + 2 * (size_t)nk + 2) * sizeof(double) + 2 * sizeof(int);
  // Few levels leave most of sixteen lanes idle, and more cells than the chip holds at
  // sixteen lanes then wait: four lanes.  Measured (4 lanes against 16, us): 432 000 cells
  // of 3 levels 214 / 592, 6 levels 322 / 928, 11 levels 1133 / 1829, 16 levels
  // 3442 / 3818, 21 levels 7780 / 5397; 30 000 cells of 3 levels 112 / 128, 9 levels
  // 141 / 181, 16 levels 326 / 348; 10 000 cells of 6 levels 124 / 111, 9 levels 133 / 120,
  // 16 levels 211 / 175.  (One lane: 171 us for 432 000 cells of 3 levels, 373 for 6.)
  const int lanes = nk <= 16 && r->ncell > 16384 ? 4 : 16;
  int nt = (int)std::min<size_t>(lanes == 4 ? se_cells<4>() : se_cells<16>(), (size_t)ctx->lds_max / per_cell);
  if (nt >= 4) nt -= nt % 4;
  if (nt < 1) return set_error(M3DRT_ELIMIT, "m3drt_rate_solve_f64: nk too large for the LDS");
  const int nblk = (r->ncell + nt - 1) / nt;
  const size_t lds = per_cell * nt;
  // scratch: per-block winners, then the final values
  const size_t bytes = (size_t)nblk * (sizeof(double) + 2 * sizeof(int32_t)) +
                       (size_t)nblk * nk * (sizeof(double) + sizeof(int32_t)) +
                       (nk + 1) * sizeof(double) + 4 * sizeof(int32_t) + sizeof(unsigned long long) + 64;
  int rc = ensure_scratch(ctx, bytes);
  if (rc) return rc;
  char *s = static_cast<char *>(ctx->scratch);
  double *blk_err = reinterpret_cast<double *>(s);
  double *blk_lerr = blk_err + nblk;
  double *out = blk_lerr + (size_t)nblk * nk;
  unsigned long long *nclamp = reinterpret_cast<unsigned long long *>(out + nk + 1);
  int32_t *blk_cell = reinterpret_cast<int32_t *>(nclamp + 1);
  int32_t *blk_lvl = blk_cell + nblk;
  int32_t *blk_lcell = blk_lvl + nblk;
  int32_t *iout = blk_lcell + (size_t)nblk * nk;
  int32_t *status = iout + 2;
  const int32_t big = 0x7fffffff;
  M3DRT_HIP(hipMemsetAsync(nclamp, 0, sizeof(unsigned long long), ctx->stream));
  M3DRT_HIP(hipMemcpyAsync(status, &big, sizeof(int32_t), hipMemcpyHostToDevice, ctx->stream));

  SeArgs a;
  a.nk = nk; a.nrad = r->nrad; a.nline = r->nline; a.npair = r->npair; a.ncell = r->ncell; a.nt = nt;
  a.ti = r->trans_i; a.tj = r->trans_j; a.active = r->trans_active; a.pi = r->pair_i; a.pj = r->pair_j;
  a.g = r->g; a.ev = r->ev; a.Aji = r->Aji;
  a.e_kT = r->e_kT; a.temp = r->temp; a.totn = r->totn; a.nstar = r->nstar; a.cup = r->cup;
  a.b = r->b; a.gij = r->gamma_ij; a.gji = r->gamma_ji;
  a.max_update = r->max_update; a.min_pop_frac = r->min_pop_frac; a.conv_pop_floor = r->conv_pop_floor;
  a.sor_w = r->sor_w; a.cswitch = r->cswitch; a.cut_x = r->cut_x; a.bf_cut_rate = r->bf_cut_rate;
  a.tmax_update = r->tmax_update;
  a.blk_err = blk_err; a.blk_cell = blk_cell; a.blk_lvl = blk_lvl; a.blk_lerr = blk_lerr;
  a.blk_lcell = blk_lcell; a.nclamp = nclamp; a.status = status;
  auto run = [&](auto kern) -> int {
    M3DRT_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3(nblk), dim3(nt * lanes), lds, ctx->stream, a);
    return M3DRT_OK;
  };
  rc = lanes == 4 ? run(se_update_kernel<4>) : run(se_update_kernel<16>);
  if (rc) return rc;
  M3DRT_HIP(hipGetLastError());
  hipLaunchKernelGGL(se_final_kernel, dim3(nk + 1), dim3(256), 0, ctx->stream, nblk, nk, blk_err, blk_cell, blk_lvl,
                     blk_lerr, blk_lcell, out, iout);
  M3DRT_HIP(hipGetLastError());
  if (!res) return M3DRT_OK;
  std::vector<double> hout(nk + 1);
  int32_t hi[3];
  unsigned long long hcl = 0;
  M3DRT_HIP(hipMemcpyAsync(hout.data(), out, (nk + 1) * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  M3DRT_HIP(hipMemcpyAsync(hi, iout, 3 * sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
  M3DRT_HIP(hipMemcpyAsync(&hcl, nclamp, sizeof(hcl), hipMemcpyDeviceToHost, ctx->stream));
  M3DRT_HIP(hipStreamSynchronize(ctx->stream));
  res->maxerr = hout[0];
  res->epos = hi[0];
  res->elvl = hi[1];
  res->nclamp = (int64_t)hcl;
  if (res->lvlerr)
    for (int i = 0; i < nk; ++i) res->lvlerr[i] = hout[1 + i];
  if (hi[2] != big) {
    char msg[160];
    snprintf(msg, sizeof msg,
             "m3drt_rate_solve_f64: statistical equilibrium has no finite solution at cell %d "
             "(0-based, x fastest); check the rate coefficients for overflow", hi[2] - 1);
    res->epos = hi[2] - 1;
    return set_error(M3DRT_EINVAL, msg);
  }
  return M3DRT_OK;
}

int normalize_rates(m3drt_ctx *ctx, const m3drt_rate_solve_args *r, const float *wphi) {
  const int64_t n = (int64_t)r->nrad * r->ncell;
  const int blocks = (int)std::min<int64_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(normalize_kernel, dim3(blocks), dim3(256), 0, ctx->stream, r->nrad, r->nline, r->ncell,
                     r->trans_active, r->trans_i, r->trans_j, r->nstar, wphi, r->gamma_ij, r->gamma_ji);
  M3DRT_HIP(hipGetLastError());
  return M3DRT_OK;
}

}  // namespace m3drt
