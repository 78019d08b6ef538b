// The short_char2 sweep (SRC/rt_solvers_mod.f90:224-507, with integrate_intensity,
// SRC/rt_patch_mod.f90:3399-3431, fused) for cubes whose frequencies are at unit
// stride, the host code's own order work(f,x,y,z), for gfx950.
//
// The kernels that give a workgroup one frequency (sc2_fast.hip, sweep_sc2.hip) read
// such a cube four bytes out of every cache line.  Here the lanes of a wavefront are
// consecutive frequencies of one column, so every access is one contiguous run, and
// the grid covers the whole plane: one launch advances one plane, and the plane
// before it (chi, S and the intensities, which alternate between two scratch planes)
// is read back from the caches.  The launches are in stream order, which is all the
// ordering the planes need.
//
// Threads.  A lane takes one (f, x) and a strip of L consecutive rows y, with the
// sliding 4-row window of the other kernels: each cell reads one new upwind row
// (4 I, 2 chi, 2 S) and reduces it in x at once.  A workgroup is 256 threads: FW
// frequencies (16, 32 or 64) of 256/FW adjacent columns, whose 4-column stencils
// overlap in the L1.
//
// Bound by: HBM for chi, S and J (16 B per update) and the last-level cache for the
// upwind plane's chi, S and I and the intensities written (16 B more): 360 us for a ray
// of the 120 x 120 x 23 slab at 128 frequencies (FP32, J), 1.9 TB/s of the 16 B, where
// the workgroup-per-frequency kernel took 2395 us.
#include "m3drt_internal.hpp"
#include "sweep_sc2.hpp"
#include <cstdio>
#include <cstdlib>
#include <cmath>
#include <algorithm>

namespace m3drt {
namespace {

template <typename T>
struct PlaneArgs {
  // this plane (z offset applied), the upwind plane, and the intensity planes
  const T *chi, *S;
  const T *uchi, *uS, *uI;
  const T *dt500, *rc, *urc;  // (x, y) of this plane and of the upwind one
  T *nI;                      // this plane's intensities, (f, x, y), f fastest
  T *J, *PsiJ, *Iout, *Psiout, *Irem, *esc, *exitI;
  uint32_t cs_x, cs_y, us_x, us_y, is_x, is_y, gs_x, gs_y;  // row strides in elements
  int nf, nx, ny, xo, yo, split;
  int nfc, nxb, per, total;   // frequency chunks, column groups, workgroups per XCD and in all
  T xk0, xk1, xk2, xk3, yk0, yk1, yk2, yk3, hx, hy, mdtau, imax, wj;
};

constexpr int kXcds = 8;

template <typename T, int L, bool PLAIN>
__global__ void __launch_bounds__(256) sc2_plane(const PlaneArgs<T> a, int fw) {
  using namespace dev;
  // Workgroups go to the XCDs in turn; each XCD takes a contiguous run of them
  // (columns fastest, then rows, then frequencies), so that neighbours, whose
  // stencils overlap, share an L2.
  const int b = (int)(blockIdx.x % kXcds) * a.per + (int)(blockIdx.x / kXcds);
  if (b >= a.total) return;
  const int fl = threadIdx.x & (fw - 1), xl = threadIdx.x / fw;
  const int xb = b % a.nxb, q = b / a.nxb;
  const int nyb = (a.ny + L - 1) / L;
  const int yb = (q % nyb) * L;
  const int f = (q / nyb) * fw + fl;
  const int x = xb * (256 / fw) + xl;
  if (f >= a.nf || x >= a.nx) return;
  const int nx = a.nx, ny = a.ny;

  const int xc0 = wrap(x + a.xo, nx), xc1 = wrap(x + a.xo + 1, nx);
  const int xc2 = wrap(x + a.xo + 2, nx), xc3 = wrap(x + a.xo + 3, nx);
  const uint32_t i0 = f + xc0 * a.is_x, i1 = f + xc1 * a.is_x, i2 = f + xc2 * a.is_x, i3 = f + xc3 * a.is_x;
  const uint32_t u1 = f + xc1 * a.us_x, u2 = f + xc2 * a.us_x;
  const T ohx = (T)1 - a.hx, ohy = (T)1 - a.hy;

  struct Row { T rI, rmin, rX, rS; };
  auto read_row = [&](int y) -> Row {
    const int yr = wrap_near(y, ny);
    const uint32_t io = yr * a.is_y, uo = yr * a.us_y;
    const T v0 = a.uI[i0 + io], v1 = a.uI[i1 + io], v2 = a.uI[i2 + io], v3 = a.uI[i3 + io];
    const T x1 = a.uchi[u1 + uo] * a.urc[yr * nx + xc1], x2 = a.uchi[u2 + uo] * a.urc[yr * nx + xc2];
    Row r;
    r.rI = a.xk0 * v0 + a.xk1 * v1 + a.xk2 * v2 + a.xk3 * v3;
    r.rmin = fmin(v1, v2);
    r.rX = ohx * x1 + a.hx * x2;
    r.rS = ohx * a.uS[u1 + uo] + a.hx * a.uS[u2 + uo];
    return r;
  };

  const int ylen = min(L, ny - yb);
  Row w0 = read_row(yb + a.yo), w1 = read_row(yb + a.yo + 1), w2 = read_row(yb + a.yo + 2);
#pragma unroll
  for (int k = 0; k < L; ++k) {
    if (k < ylen) {
      const int y = yb + k;
      const uint32_t o = f + x * a.cs_x + y * a.cs_y;
      const T chiv = a.chi[o], ss = a.S[o];
      const T dt500 = a.dt500[y * nx + x], rc = a.rc[y * nx + x];
      const T Jv = PLAIN || a.J ? a.J[o] : (T)0;
      const T PJv = !PLAIN && a.PsiJ ? a.PsiJ[o] : (T)0;
      const Row w3 = read_row(y + a.yo + 3);
      // upwind values, SRC/rt_solvers_mod.f90:379-394
      const T xxup = ohy * w1.rX + a.hy * w2.rX;
      const T ssup = ohy * w1.rS + a.hy * w2.rS;
      T Inuup = a.yk0 * w0.rI + a.yk1 * w1.rI + a.yk2 * w2.rI + a.yk3 * w3.rI;
      Inuup = fmax(Inuup, fmin(w1.rmin, w2.rmin));
      const T xx = chiv * rc;
      const T dt = fmax((T)0.5 * (xxup + xx) * dt500, a.mdtau);
      T E, W, Ps, Es;
      lin_weights(dt, E, W, Ps, Es);
      // the S step of a cell without eta flags (SRC/rt_solvers_mod.f90:419-440, 465-475)
      const T Ir = Inuup * E + W * ssup;
      T Inu = Ir + Ps * ss;
      if (!PLAIN) {
        const T sgnchi = copysign(fmax(fabs(chiv), (T)1.17549435e-38f), chiv);
        bool off = fmin(dt, chiv) <= (T)0;
        if (a.split) off = off || (a.imax - fabs(Inu)) <= (T)0;
        const T psiout = off ? (T)0 : Ps * rcp(sgnchi);
        Inu = fmax(-a.imax, fmin(a.imax, Inu));
        if (a.J) a.J[o] = Jv + a.wj * Inu;
        if (a.PsiJ) a.PsiJ[o] = PJv + a.wj * psiout;
        if (a.Iout) a.Iout[o] = Inu;
        if (a.Psiout) a.Psiout[o] = psiout;
        if (a.split) {
          a.Irem[o] = off ? Inu : Ir;
          a.esc[o] = off ? (T)1 : Es;
        }
      } else {
        Inu = fmax(-a.imax, fmin(a.imax, Inu));
        a.J[o] = Jv + a.wj * Inu;
      }
      a.nI[f + (uint32_t)(x + y * nx) * (uint32_t)a.nf] = Inu;
      if (a.exitI) a.exitI[f + x * a.gs_x + y * a.gs_y] = Inu;
      w0 = w1;
      w1 = w2;
      w2 = w3;
    }
  }
}

template <typename T, int L>
void launch_plane(hipStream_t st, const PlaneArgs<T> &a, int blocks, int fw, bool plain) {
  if (plain) hipLaunchKernelGGL((sc2_plane<T, L, true>), dim3(blocks), dim3(256), 0, st, a, fw);
  else hipLaunchKernelGGL((sc2_plane<T, L, false>), dim3(blocks), dim3(256), 0, st, a, fw);
}

}  // namespace

template <typename T>
int sweep_sc2_plane(m3drt_ctx *ctx, const m3drt_sweep_desc *d, const m3drt_sweep_bufs *b) {
  const int nf = d->nf, nx = d->nx, ny = d->ny, nz = d->nz;
  const int64_t nxy = (int64_t)nx * ny;
  if (d->cs_f != 1 || d->gs_f != 1 || b->eta_row || getenv("M3DRT_NO_PLANE")) return -1;
  // Where this form is the faster one.  A plane costs it at least a launch (3.5 us; the
  // workgroup-per-frequency kernels take 1.5 us for a plane of a few hundred cells),
  // and from there on its time follows the points, the others' the plane's cells
  // (every one of them a cache line per frequency).  Measured, 20 to 23 planes, J only
  // (FP32): 16 x 16 x 64 frequencies 70 us against 39, 24 x 24 x 64 71 against 64,
  // 24 x 24 x 256 85 against 104, 13 x 11 x 1024 87 against 111, 40 x 40 x 16 80
  // against 109, 120 x 120 x 16 111 against 1072, 120 x 120 x 250 770 against 2505;
  // FP64: 16 x 16 x 64 83 against 69, 24 x 24 x 64 84 against 159.
  const int64_t wide = sizeof(T) / 4;
  const bool pays = nxy * wide >= 1024 || (nxy >= 128 && nxy * nf * wide >= 131072);
  if (nf < 16 || !(pays || getenv("M3DRT_PLANE_ALWAYS"))) return -1;
  const uint64_t span = (uint64_t)(nx - 1) * d->cs_x + (uint64_t)(ny - 1) * d->cs_y + nf;
  const uint64_t gspan = (uint64_t)(nx - 1) * d->gs_x + (uint64_t)(ny - 1) * d->gs_y + nf;
  if (span >= (1ull << 31) || gspan >= (1ull << 31) || (uint64_t)nxy * nf >= (1ull << 31)) return -1;

  // An exit plane written over the ghost plane: safe while other launches lie between a
  // frequency's reads and its writes, so not with a single plane.
  if (nz == 1 && b->exit_I) {
    const char *e = static_cast<const char *>(b->exit_I);
    for (const void *p : {b->ghost_chi, b->ghost_S, b->ghost_I}) {
      const char *q = static_cast<const char *>(p);
      if (e < q + gspan * sizeof(T) && q < e + gspan * sizeof(T)) return -1;
    }
  }

  // The frequencies in runs whose two intensity planes the scratch holds: all of them
  // where it may grow (to 512 MiB of planes), the ones that fit beside the preparation
  // where it may not (m3drt_sc_sweep_noalloc's 32 MiB, a capture, no memory).  They are
  // independent, so the runs change no value: 1024 frequencies of the 120 x 120 x 23 slab
  // take four runs of 256 in the 32 MiB.
  const size_t nprep = (size_t)nxy * (nz + 1), prep = 2 * nprep * sizeof(T), per_f = 2 * (size_t)nxy * sizeof(T);
  const size_t most = std::min<size_t>(nf, std::max<size_t>(64, ((size_t)512 << 20) / per_f / 64 * 64));
  const size_t room = offer_scratch(ctx, prep + 16 * per_f, prep + most * per_f);
  if (!room) return -1;
  int run = (int)((room - prep) / per_f);
  if (run < nf) {
    run -= run % (run >= 64 ? 64 : 16);
    const int nrun = (nf + run - 1) / run;
    run = std::min(run, ((nf + nrun - 1) / nrun + 15) / 16 * 16);
  }
  const size_t nI = (size_t)nxy * run;
  T *dt500 = static_cast<T *>(ctx->scratch), *rc = dt500 + nprep, *I0 = rc + nprep, *I1 = I0 + nI;
  const Sc2Geom g = sc2_geometry(d);
  const int st = sc2_prep<T>(ctx, d, b->chi500, b->chi500_up, b->g500, dt500, rc);
  if (st) return st;

  PlaneArgs<T> a;
  const bool rates = (d->flags & M3DRT_GET_RATES) != 0;
  T *const J = static_cast<T *>(b->J), *const PsiJ = rates ? static_cast<T *>(b->PsiJ) : nullptr;
  T *const Iout = static_cast<T *>(b->I_out), *const Psiout = rates ? static_cast<T *>(b->Psi_out) : nullptr;
  a.split = (d->flags & M3DRT_SPLIT_RATES) ? 1 : 0;
  const bool plain = J && !PsiJ && !Iout && !Psiout && !a.split;
  a.nx = nx; a.ny = ny; a.xo = g.xo; a.yo = g.yo;
  a.cs_x = (uint32_t)d->cs_x; a.cs_y = (uint32_t)d->cs_y;
  a.gs_x = (uint32_t)d->gs_x; a.gs_y = (uint32_t)d->gs_y;
  // the stencil in FP32 as the reference casts it (FP64 sweep: in FP64)
  const bool f64 = sizeof(T) == 8;
  auto cast = [&](double v) { return f64 ? (T)v : (T)(float)v; };
  a.xk0 = cast(g.kx[0]); a.xk1 = cast(g.kx[1]); a.xk2 = cast(g.kx[2]); a.xk3 = cast(g.kx[3]);
  a.yk0 = cast(g.ky[0]); a.yk1 = cast(g.ky[1]); a.yk2 = cast(g.ky[2]); a.yk3 = cast(g.ky[3]);
  a.hx = -a.xk0 + a.xk2 + (T)2 * a.xk3;  // inner_fraction, SRC/rt_solvers_mod.f90:500-506
  a.hy = -a.yk0 + a.yk2 + (T)2 * a.yk3;
  a.mdtau = f64 ? -(T)d->maser_dtau_max : (T)(-(float)d->maser_dtau_max);
  a.imax = f64 ? (T)d->maser_Inu_max : (T)(float)d->maser_Inu_max;
  a.wj = (T)d->wj;

  // Rows a lane takes: one where the plane barely fills the chip (a lane's rows follow
  // one another, each a round trip to the cache), up to eight where the points keep
  // the memory busy and the three rows a strip re-reads count.  Measured (FP32, 20 to
  // 23 planes, L = 8 / 4 / 2 / 1): 24 x 24 x 256 frequencies 148 / 105 / 92 / 85 us,
  // 60 x 60 x 256 247 / 213 / 210 / 234, 120 x 120 x 250 772 / 768 / 806 / 901.
  const char *lenv = getenv("M3DRT_PLANE_L");
  const int64_t pb = nxy * nf * (int64_t)sizeof(T) >> 20;
  int L = lenv ? atoi(lenv) : pb >= 12 ? 8 : pb >= 4 ? 4 : pb >= 1 ? 2 : 1;
  L = L >= 8 ? 8 : L >= 4 ? 4 : L >= 2 ? 2 : 1;
  const int dir = d->dir > 0 ? 1 : -1;
  for (int f0 = 0; f0 < nf; f0 += run) {
    a.nf = std::min(run, nf - f0);
    // frequencies a wave takes: the widest of 64, 32, 16 that leaves no more lanes idle
    int fw = 64;
    auto lanes = [&](int w) { return (a.nf + w - 1) / w * w; };
    for (int w : {32, 16})
      if (lanes(w) * 9 <= lanes(fw) * 8) fw = w;
    a.nfc = (a.nf + fw - 1) / fw;
    a.nxb = (nx + 256 / fw - 1) / (256 / fw);
    a.total = a.nxb * ((ny + L - 1) / L) * a.nfc;
    a.per = (a.total + kXcds - 1) / kXcds;
    if (getenv("M3DRT_VERBOSE"))
      fprintf(stderr, "[m3drt] sc2 plane %s nf=%d+%d of %d plane=%dx%d nz=%d: %d workgroups a plane, %d frequencies a wave, strip %d\n",
              f64 ? "f64" : "f32", f0, a.nf, nf, nx, ny, nz, a.total, fw, L);
    for (int step = 0; step < nz; ++step) {
      const int z = dir > 0 ? step : nz - 1 - step;
      const int64_t zo = (int64_t)z * d->cs_z + f0, uo = (int64_t)(z - dir) * d->cs_z + f0;
      auto at = [&](void *p) { return p ? static_cast<T *>(p) + zo : nullptr; };
      a.chi = static_cast<const T *>(b->chi) + zo;
      a.S = static_cast<const T *>(b->S) + zo;
      a.dt500 = dt500 + (int64_t)z * nxy;
      a.rc = rc + (int64_t)z * nxy;
      if (step == 0) {
        a.uchi = static_cast<const T *>(b->ghost_chi) + f0;
        a.uS = static_cast<const T *>(b->ghost_S) + f0;
        a.uI = static_cast<const T *>(b->ghost_I) + f0;
        a.urc = rc + (int64_t)nz * nxy;
        a.us_x = a.is_x = a.gs_x;
        a.us_y = a.is_y = a.gs_y;
      } else {
        a.uchi = static_cast<const T *>(b->chi) + uo;
        a.uS = static_cast<const T *>(b->S) + uo;
        a.uI = step & 1 ? I0 : I1;
        a.urc = rc + (int64_t)(z - dir) * nxy;
        a.us_x = a.cs_x; a.us_y = a.cs_y;
        a.is_x = (uint32_t)a.nf; a.is_y = (uint32_t)a.nf * nx;
      }
      a.nI = step & 1 ? I1 : I0;
      a.J = at(J); a.PsiJ = at(PsiJ); a.Iout = at(Iout); a.Psiout = at(Psiout);
      a.Irem = a.split ? at(b->Irem_out) : nullptr;
      a.esc = a.split ? at(b->escape_out) : nullptr;
      a.exitI = step == nz - 1 && b->exit_I ? static_cast<T *>(b->exit_I) + f0 : nullptr;
      if (L == 8) launch_plane<T, 8>(ctx->stream, a, a.per * kXcds, fw, plain);
      else if (L == 4) launch_plane<T, 4>(ctx->stream, a, a.per * kXcds, fw, plain);
      else if (L == 2) launch_plane<T, 2>(ctx->stream, a, a.per * kXcds, fw, plain);
      else launch_plane<T, 1>(ctx->stream, a, a.per * kXcds, fw, plain);
      M3DRT_HIP(hipGetLastError());
    }
  }
  return M3DRT_OK;
}

template int sweep_sc2_plane<float>(m3drt_ctx *, const m3drt_sweep_desc *, const m3drt_sweep_bufs *);
template int sweep_sc2_plane<double>(m3drt_ctx *, const m3drt_sweep_desc *, const m3drt_sweep_bufs *);

}  // namespace m3drt
