// kz_sim_kernels.h — the step kernels that the reference's non-default
// options change, as templates over the option: the wavespeeds (the
// synchrotron bridge in the optical depth), the u2p pass (the b^2/rho floor
// frame), the face flux (reconstruction order per cell, floor frame) and the
// implicit ladder (the synchrotron bridge).  kz_step.hip
// instantiates the default of each, kz_options.hip the option variants, so
// that the default code object carries none of the variants' code.
#ifndef KZ_SIM_KERNELS_H
#define KZ_SIM_KERNELS_H

#include "kz_sim_dev.h"

// wavespeeds + CFL denominators (sim.zig:747-886)
__device__ __forceinline__ long long dbits(double x) { return __double_as_longlong(x); }
// one thread per cell of the domain and its one-cell ring; BR fixes the
// synchrotron bridge of the opacities on or off
template <bool BR>
__device__ __forceinline__ void wavespeeds_pass(const GridD &g, const Dev &d, const kz_physics &ph) {
  long t = TID;
  int act[3] = {g.nx > 1, g.ny > 1, g.nz > 1};
  long lx = act[0], ly = act[1], lz = act[2];
  long wx = g.nx + 2 * lx, wy = g.ny + 2 * ly, wz = g.nz + 2 * lz;
  if (t >= wx * wy * wz) return;
  long ix, iy, iz;
  split3(t, wx, wy, ix, iy, iz);
  ix -= lx;
  iy -= ly;
  iz -= lz;
  long n = g.ncell;
  long c = cidx(g, ix, iy, iz);
  double pp[NV];
  ld(d.p, n, c, pp);
  Geo gm;
  geo_c(g, d, ix, iy, iz, gm);
  double aaa[6], av[12], rad0[6], radl[6];
  gas_wavespeeds(pp, gm, ph.gam, act, aaa);
  double tau[3] = {0, 0, 0};
  if (ph.has_opac) {
    kz_opac_params op = ph.opac;
    op.synchrotron_bridge = BR;
    double chi = calc_chi_slim(pp, gm, ph.gam, op);
    long idx3[3] = {ix, iy, iz};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      double sg = kzm_sqrt(gm.g[k + 1][k + 1]);
      double dxp = kzm_fmax(csize(g, idx3[k], k) * sg, csize(g, idx3[k] + 1, k) * sg);
      tau[k] = chi * dxp;
    }
  }
  if (ph.dampradwavespeednearaxis > 0) {
    long nc = ph.dampradwavespeednearaxis;
    if (iy < nc || iy >= g.ny - nc) tau[0] = tau[1] = tau[2] = 0;
  }
  rad_wavespeeds(pp, gm, tau, act, av);
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    rad0[i] = av[i];
    radl[i] = av[6 + i];
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    if (radl[2 * k] > 0.0) radl[2 * k] = 0.0;
    if (radl[2 * k + 1] < 0.0) radl[2 * k + 1] = 0.0;
    if (rad0[2 * k] > 0.0) rad0[2 * k] = 0.0;
    if (rad0[2 * k + 1] < 0.0) rad0[2 * k + 1] = 0.0;
  }
  double ax = kzm_fmax(kzm_fabs(aaa[0]), kzm_fabs(aaa[1]));
  double ay = kzm_fmax(kzm_fabs(aaa[2]), kzm_fabs(aaa[3]));
  double az = kzm_fmax(kzm_fabs(aaa[4]), kzm_fabs(aaa[5]));
  d.scal[(SC_AHD + 0) * n + c] = ax;
  d.scal[(SC_AHD + 1) * n + c] = ay;
  d.scal[(SC_AHD + 2) * n + c] = az;
#pragma unroll
  for (int k = 0; k < 3; ++k)
    d.scal[(SC_ARAD + k) * n + c] = kzm_fmax(kzm_fabs(radl[2 * k]), kzm_fabs(radl[2 * k + 1]));
  double wsx = kzm_fmax(ax, kzm_fmax(kzm_fabs(rad0[0]), kzm_fabs(rad0[1])));
  double wsy = kzm_fmax(ay, kzm_fmax(kzm_fabs(rad0[2]), kzm_fabs(rad0[3])));
  double wsz = kzm_fmax(az, kzm_fmax(kzm_fabs(rad0[4]), kzm_fabs(rad0[5])));
  if (!(ix >= 0 && ix < g.nx && iy >= 0 && iy < g.ny && iz >= 0 && iz < g.nz)) return;
  double dx = csize(g, ix, 0), dy = csize(g, iy, 1), dz = csize(g, iz, 2);
  double tsd;
  if (g.nz > 1 && g.ny > 1) tsd = wsx / dx + wsy / dy + wsz / dz;
  else if (g.nz == 1 && g.ny > 1) tsd = wsx / dx + wsy / dy;
  else if (g.ny == 1 && g.nz > 1) tsd = wsx / dx + wsz / dz;
  else tsd = wsx / dx;
  tsd /= ph.tsteplim;
  d.scal[SC_TSTEPDEN * n + c] = tsd;
  if (tsd == tsd) {
    long long *b = (long long *)slot_of(d.tsd);
    atomicMax(&b[0], dbits(tsd));
    atomicMin(&b[1], dbits(tsd));
  }
}

// u2p pass (sim.zig:940-1000), one thread per domain cell; cells flagged for
// the u2p fixups (sim.zig:1001-1003) are listed for k_u2p_fixups.  ZAMO
// floors in the ZAMO frame (invert.zig:649-684).
template <bool ZAMO>
__device__ __forceinline__ void u2p_pass(const GridD &g, const Dev &d, const kz_physics &ph) {
  long t = TID;
  long nd = (long)g.nx * g.ny * g.nz;
  const bool fix_hd = ph.do_fixups, fix_rad = ph.do_fixups && ph.do_u2prad_fixups;
  if (t < nd) {
    long ix, iy, iz;
    split3(t, g.nx, g.ny, ix, iy, iz);
    long c = cidx(g, ix, iy, iz);
    long n = g.ncell;
    double uu[NV], pp[NV];
    ld(d.u, n, c, uu);
    ld(d.p, n, c, pp);
    d.flags[KZ_FLAG_ENTROPY * n + c] = 0;
    d.flags[KZ_FLAG_ENTROPY2 * n + c] = 0;
    Geo gm;
    geo_c(g, d, ix, iy, iz, gm);
    if (polar_row(ph, g, iy)) {
      double gi = 1.0 / gm.gdet;
      d.p[B1 * n + c] = uu[B1] * gi;
      d.p[B2 * n + c] = uu[B2] * gi;
      d.p[B3 * n + c] = uu[B3] * gi;
      d.flags[KZ_FLAG_HD_FIXUP * n + c] = 0;
      d.flags[KZ_FLAG_RAD_FIXUP * n + c] = 0;
    } else {
      int ent;
      int ret = u2p_mhd(uu, pp, gm, ph.gam, ph.floors, &ent);
      if (ent) d.flags[KZ_FLAG_ENTROPY * n + c] = 1;
      int corr;
      u2p_rad(uu, pp, gm, ph.rad, &corr);
      int guard = 0;
      check_floors_mhd<ZAMO>(pp, gm, ph.gam, ph.floors, &guard);
      check_floors_rad(pp, gm, ph.rad);
      st(d.p, n, c, pp);
      int fh = ret < -1 ? 1 : 0, fr = corr ? -1 : 0;
      d.flags[KZ_FLAG_HD_FIXUP * n + c] = fh;
      d.flags[KZ_FLAG_RAD_FIXUP * n + c] = fr;
      if (guard) atomicAdd(&slot_of(d.cnt)[3], (unsigned long long)guard);
      if ((fix_hd && fh) || (fix_rad && fr)) {
        unsigned k = atomicAdd(&d.sync[SY_NFIX], 1u);
        d.fix_list[k] = (int32_t)t;
      }
    }
  }
}
// ---------------------------------------------------------------------------
// fused face flux: PPM of the two adjacent cells, face floors, fFluxPrime,
// p2u, LAXF (sim.zig:1284-1503) for faces i in [0, n] of each active
// dimension, cross indices over [-1, n_c + 1) in the other active ones.

// rijvisc.zig:313-353 faceAvg + radvisc.zig:201-244 addRadViscFlux: row
// dim+1 of the face-averaged viscous R^i_j (rv), velocity-capped, added to
// the radiation rows of one face state's flux; uu is that state's p2u.  Of
// the reference's three capped velocities only the face-normal one is used.
template <int DIM>
__device__ __forceinline__ void add_visc_flux(const double rv[4], const double *uu, const Geo &gm, const GridD &g,
                                              const kz_physics &ph, double *ff) {
  const bool y_active = g.ny > 1, z_active = g.nz > 1;
  const double gdetu = gm.gdet;
  double vel = 0;
#pragma unroll
  for (int ii = 1; ii < 4; ++ii) {
    if (ii == 2 && !y_active) continue;
    if (ii == 3 && !z_active) continue;
    if (kzm_fabs(uu[EE + ii]) < 1.0e-10 * kzm_fabs(uu[EE])) continue;
    vel = rv[ii] / (uu[EE + ii] / gdetu) * kzm_sqrt(gm.g[DIM + 1][DIM + 1]);
  }
  const double maxv = kzm_fabs(vel);
  double dampfac = 1.0;
  if (maxv > ph.radvisc.maxvel) dampfac = ph.radvisc.maxvel / maxv;
#pragma unroll
  for (int nu = 0; nu < 4; ++nu) ff[EE + nu] += gdetu * dampfac * rv[nu];
}
// Face fluxes by tiles.  A block of 128 threads owns up to 64 faces of one
// dimension whose adjacent cells number at most 64:
//   x faces: a run of FaceTiles::fx consecutive faces of the x-fastest face
//   order (a run may continue on the next row);
//   y and z faces: FT_T consecutive x columns by FT_F consecutive faces
//   along the dimension.
// Phase 1: the block reconstructs each of its cells once, both face values
// of every slot, into LDS (the left state of face i is cell i-1's right
// value, the right state cell i's left one); the two waves share the slots.
// Phase 2: one thread per face side takes its state from LDS, applies the
// face floors and forms its flux fFluxPrime and conserved vector p2u (with
// the viscous flux when enabled).  Phase 3: the two sides of a face,
// neighbouring lanes, exchange flux and conserved vector and each writes the
// LAXF flux of half the slots.  Each side is exactly the reference's
// computation for that face state, so the fluxes and the floor guard count
// are the reference's.
#ifndef KZ_FT_T
#define KZ_FT_T 8
#endif
constexpr int FT_T = KZ_FT_T, FT_F = 64 / FT_T - 1;
struct FaceTiles {
  long nb[3];  // blocks of each dimension, launched in the order x, y, z
  int fx;      // x faces per block
};
struct FaceShared {
  double st[2][NV][64];  // [0] left, [1] right face value of each slot of each cell
};
// The faces and cells of block b of dimension DIM, numbered locally: face f
// lies between cells left(f) and right(f).  Coordinates are (ix, iy, iz)
// with the face index in component DIM.
template <int DIM>
struct FaceTile {
  static constexpr int c0d = DIM == 0 ? 1 : 0, c1d = DIM == 2 ? 1 : 2;
  long wf, w0, l0, l1;
  long t0, r0, p0;  // x runs: first face, its row and its place in the row
  long x0, i0, c1;  // y/z tiles: first column, first face along DIM, the other cross index
  int nface, ncell;
  __device__ FaceTile(const GridD &g, const FaceTiles &ft, long b) {
    const long n0 = c0d == 1 ? g.ny : g.nx, n1 = c1d == 1 ? g.ny : g.nz;
    l0 = n0 > 1 ? -1 : 0;
    w0 = n0 > 1 ? n0 + 2 : n0;
    l1 = n1 > 1 ? -1 : 0;
    const long w1 = n1 > 1 ? n1 + 2 : n1;
    wf = (DIM == 0 ? g.nx : (DIM == 1 ? g.ny : g.nz)) + 1;
    if (DIM == 0) {
      t0 = b * ft.fx;
      const long left = wf * w0 * w1 - t0;
      nface = (int)(left < ft.fx ? left : ft.fx);
      r0 = (unsigned)t0 / (unsigned)wf;
      p0 = t0 - r0 * wf;
      ncell = right(nface - 1) + 1;
    } else {
      const long ntx = (w0 + FT_T - 1) / FT_T, nti = (wf + FT_F - 1) / FT_F;
      split3(b, ntx, nti, x0, i0, c1);
      x0 *= FT_T;
      i0 *= FT_F;
      c1 += l1;
      nface = FT_T * FT_F;
      ncell = FT_T * (FT_F + 1);
    }
  }
  __device__ int left(int f) const { return DIM == 0 ? f + (int)((unsigned)(p0 + f) / (unsigned)wf) : f; }
  __device__ int right(int f) const { return DIM == 0 ? left(f) + 1 : f + FT_T; }
  __device__ bool face(int f, long cell[3]) const {
    if (f >= nface) return false;
    if (DIM == 0) {
      split3(t0 + f, wf, w0, cell[0], cell[1], cell[2]);
      cell[1] += l0;
      cell[2] += l1;
      return true;
    }
    const long x = x0 + f % FT_T, i = i0 + f / FT_T;
    if (x >= w0 || i >= wf) return false;
    cell[DIM] = i;
    cell[c0d] = x + l0;
    cell[c1d] = c1;
    return true;
  }
  __device__ bool cellk(int k, long cell[3]) const {
    if (k >= ncell) return false;
    if (DIM == 0) {
      split3(r0 * (wf + 1) + p0 + k, wf + 1, w0, cell[0], cell[1], cell[2]);
      cell[0] -= 1;
      cell[1] += l0;
      cell[2] += l1;
      return true;
    }
    const long x = x0 + k % FT_T, i = i0 - 1 + k / FT_T;
    if (x >= w0 || i >= wf) return false;
    cell[DIM] = i;
    cell[c0d] = x + l0;
    cell[c1d] = c1;
    return true;
  }
};
// sim.zig:1316-1337: the reconstruction order of a cell: PPM, one lower with
// REDUCEORDERATBH inside the horizon (radial index <= reduce_order_ix_max)
// or REDUCEORDERAFTERFIXUP on a cell that the last u2p or implicit pass
// flagged for a fixup (ghost cells carry no flag)
__device__ __forceinline__ int recon_order(const GridD &g, const Dev &d, const kz_physics &ph, const long cell[3]) {
  if (ph.reduceorderatbh && cell[0] <= ph.reduce_order_ix_max) return 1;
  if (ph.reduceorderafterfixup) {
    const long c = cidx(g, cell[0], cell[1], cell[2]), n = g.ncell;
    if (d.flags[KZ_FLAG_HD_FIXUP * n + c] != 0 || d.flags[KZ_FLAG_RAD_FIXUP * n + c] != 0 ||
        d.flags[KZ_FLAG_RADIMP_FIXUP * n + c] != 0)
      return 1;
  }
  return 2;
}
template <int DIM, bool VISC, bool OPTS>
__device__ __forceinline__ void face_tile(const GridD &g, const Dev &d, const kz_physics &ph, const FaceTiles &ft,
                                          long b, FaceShared &sh) {
  constexpr int dim = DIM;
  const FaceTile<DIM> tl(g, ft, b);
  const int j = threadIdx.x;
  const long n = g.ncell;
  const long stride = dim == 0 ? 1 : (dim == 1 ? g.sx : (long)g.sx * g.sy);
  long cell[3];
  // phase 1: both face values of cell j & 63 over the stencil along DIM;
  // the block's first wave takes slots [0, 7), the second [7, 13)
  const int kc = j & 63;
  if (tl.cellk(kc, cell)) {
    const long i = cell[dim];
    const long c = cidx(g, cell[0], cell[1], cell[2]);
    double dxs[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) dxs[k] = csize(g, i - 2 + k, dim);
    const int iv0 = j < 64 ? 0 : 7, iv1 = j < 64 ? 7 : NV;
    const int order = OPTS ? recon_order(g, d, ph, cell) : 2;
    for (int iv = iv0; iv < iv1; ++iv) {
      const double *f = d.p + iv * n;
      double s5[5];
#pragma unroll
      for (int k = 0; k < 5; ++k) s5[k] = f[c + (k - 2) * stride];
      double lo, ro;
      if (order == 2) ppm(s5, dxs, &lo, &ro);
      else reconstruct(order, ph.minmod_theta, s5, dxs, &lo, &ro);
      sh.st[0][iv][kc] = lo;
      sh.st[1][iv][kc] = ro;
    }
  }
  __syncthreads();
  // phase 2: face side j & 1 of face j >> 1
  const int slot = j >> 1, side = j & 1;
  const bool act = tl.face(slot, cell);
  double fl[NV], ul[NV], ag = 0, agr = 0;
  long fi = 0;
  if (act) {
    const int k = side == 0 ? tl.left(slot) : tl.right(slot);
    double ps[NV];
#pragma unroll
    for (int iv = 0; iv < NV; ++iv) ps[iv] = sh.st[side == 0 ? 1 : 0][iv][k];
    const long cf = cidx(g, cell[0], cell[1], cell[2]);
    const long cm = cf - stride;
    Geo gm;
    geo_f(g, d, dim, cell[0], cell[1], cell[2], gm);
    int guard = 0;
    if (OPTS && ph.floors.b2rhofloorframe == 1) check_floors_mhd<true>(ps, gm, ph.gam, ph.floors, &guard);
    else check_floors_mhd<false>(ps, gm, ph.gam, ph.floors, &guard);
    if (flux_prime_d<DIM>(ps, gm, ph.gam, fl)) set_err(d.err, E_NANFLUX);
    p2u(ps, ul, gm, ph.gam);
    if (VISC) {
      double rv[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        rv[q] = 0.5 * (d.rijvisc[((DIM + 1) * 4 + q) * n + cf] + d.rijvisc[((DIM + 1) * 4 + q) * n + cm]);
      add_visc_flux<DIM>(rv, ul, gm, g, ph, fl);
    }
    ag = kzm_fmax(d.scal[(SC_AHD + dim) * n + cf], d.scal[(SC_AHD + dim) * n + cm]);
    agr = kzm_fmax(d.scal[(SC_ARAD + dim) * n + cf], d.scal[(SC_ARAD + dim) * n + cm]);
    fi = fidx(g, dim, cell[0], cell[1], cell[2]);
    if (guard) atomicAdd(&slot_of(d.cnt)[3], (unsigned long long)guard);
  }
  // phase 3: the two sides of a face are neighbouring lanes; each takes the
  // other's flux and conserved vector and writes the LAXF flux of half the
  // slots (side 0: [0, 7), side 1: [7, 13))
  double fo[NV], uo[NV];
#pragma unroll
  for (int iv = 0; iv < NV; ++iv) {
    fo[iv] = __shfl_xor(fl[iv], 1);
    uo[iv] = __shfl_xor(ul[iv], 1);
  }
  if (!act) return;
  const long nfd = g.nface[dim];
  double *out = d.flb[dim];
#pragma unroll
  for (int iv = 0; iv < NV; ++iv) {
    if ((iv < 7) != (side == 0)) continue;
    const double fL = side == 0 ? fl[iv] : fo[iv], fR = side == 0 ? fo[iv] : fl[iv];
    const double uL = side == 0 ? ul[iv] : uo[iv], uR = side == 0 ? uo[iv] : ul[iv];
    out[iv * nfd + fi] = laxf(fL, fR, uL, uR, iv >= EE ? agr : ag);
  }
}
// One launch for the faces of every active dimension (faces of different
// dimensions are independent): blocks [0, nb[0]) are x tiles, then y, then
// z.  VISC adds the radiative-viscosity flux (sim.zig:1349-1364).  OPTS
// reads the reference options of this pass from the parameter block (the
// reconstruction order per cell, the b^2/rho floor frame); without it the
// kernel is compiled for PPM everywhere and the drift frame, so the default
// build carries none of their code.
template <bool VISC, bool OPTS>
__global__ void __launch_bounds__(128) KZ_WPE(KZ_WPE_FACE) k_face_flux(GridD g, Dev d, kz_physics ph, FaceTiles ft) {
  __shared__ FaceShared sh;
  long b = blockIdx.x;
  if (b < ft.nb[0]) face_tile<0, VISC, OPTS>(g, d, ph, ft, b, sh);
  else if (b < ft.nb[0] + ft.nb[1]) face_tile<1, VISC, OPTS>(g, d, ph, ft, b - ft.nb[0], sh);
  else face_tile<2, VISC, OPTS>(g, d, ph, ft, b - ft.nb[0] - ft.nb[1], sh);
}


// implicit four-force solve (sim.zig:1736-1776 -> implicit.zig:927-1004),
// split in three kernels so that each keeps its state in registers:
//   k_imp_prep     reference state, bisection warm start, starting block
//   k_imp_rung0    the first rung (energy equation, lab frame), one launch
//                  over both starting-block lists: the RAD-start cells (the
//                  longer solves) take the first blocks, so their waves are
//                  dispatched first and the MHD-start waves fill the SIMDs
//                  that remain and those freed as waves finish
//   k_imp_slow     rungs 1..5 (and damped-opacity levels) for the cells the
//                  first rung did not solve, gathered into a list
// Batches, whose cells need from one to forty iterations per rung, run the
// first rung and then the later rungs of level 0 as persistent work-stealing
// launches (k_imp_rung0_persist, k_imp_ladder_persist): every lane holds one
// cell's Newton state and takes the next entry of the queue when its Newton
// ends, so a wave's time is its lanes' total iterations, not 64 times its
// slowest cell's; k_imp_slow then takes the damped levels.
// The sequence of attempts per cell is the reference ladder's; inputs to
// every rung are the stored reference-state values, so results equal the
// single-pass ladder bit for bit.
// Scratch of the split solve, indexed by the solve's cell index t.
struct ImpWork {
  double *uu00;  // [13][n] conserved state of the incoming primitives
  double *pp0;   // [13][n] Newton start (after the bisection warm start)
  double *aux;   // [IMP_NAUX][n] reference-state scalars
  int32_t *slow;                  // cells that need rungs past the first
  int32_t *list;                  // [2][n] cells by starting block (MHD, RAD)
  unsigned long long *nslow;      // length of `slow`
  unsigned long long *ncnt;       // lengths of the two lists: MHD in the low 32 bits, RAD in the high ones
  // batches (null for grids): the cells the persistent first rung left,
  // rl = [2][n] by starting block (MHD, RAD) with lengths rc = [2], and the
  // queue claim positions qpos (first rung RAD, MHD; the later-rung ladder)
  int32_t *rl;
  unsigned long long *rc;
  unsigned long long *qpos;
  unsigned *st;  // [n] by cell: which rungs past the first have failed or solved it
};
// The cells of one run's domain (opImplicit, sim.zig:1736-1776): polar rows
// are skipped, dt is a step scalar, a solved cell stores u and p and clears
// its radimp flag (sim.zig:1762-1768), a failed one sets it to -1.
struct GridCells {
  static constexpr bool PERSIST_ONLY = false;
  GridD g;
  Dev d;
  int sslot;
  __device__ long count() const { return (long)g.nx * g.ny * g.nz; }
  __device__ void ijk(long t, long &ix, long &iy, long &iz) const {
    ix = t % g.nx;
    iy = (t / g.nx) % g.ny;
    iz = t / ((long)g.nx * g.ny);
  }
  __device__ bool skip(const kz_physics &ph, long t) const { return polar_row(ph, g, (t / g.nx) % g.ny); }
  __device__ void load_p(long t, double *pp) const {
    long ix, iy, iz;
    ijk(t, ix, iy, iz);
    ld(d.p, g.ncell, cidx(g, ix, iy, iz), pp);
  }
  __device__ void geo(long t, Geo &gm) const {
    long ix, iy, iz;
    ijk(t, ix, iy, iz);
    geo_c(g, d, ix, iy, iz, gm);
  }
  __device__ double dt(long) const { return d.ss[sslot]; }
  __device__ void solved(const kz_physics &ph, long t, const Geo &gm, const double *ppw, int iters, int, int, int,
                         int) const {
    long ix, iy, iz;
    ijk(t, ix, iy, iz);
    const long c = cidx(g, ix, iy, iz);
    double uu[NV];
    p2u(ppw, uu, gm, ph.gam);
    st(d.u, g.ncell, c, uu);
    st(d.p, g.ncell, c, ppw);
    d.flags[KZ_FLAG_RADIMP_FIXUP * g.ncell + c] = 0;
    unsigned long long *k = slot_of(d.cnt);
    atomicAdd(&k[1], (unsigned long long)iters);
    atomicAdd(&k[2], 1ULL);
  }
  __device__ void failed(long t) const {
    long ix, iy, iz;
    ijk(t, ix, iy, iz);
    d.flags[KZ_FLAG_RADIMP_FIXUP * g.ncell + cidx(g, ix, iy, iz)] = -1;
    atomicAdd(&slot_of(d.cnt)[0], 1ULL);
  }
};
// n independent cells (solveImplicitLab per record, implicit.zig:927-1009):
// geometry planes and dt per cell, the ladder's outcome recorded per cell.
struct BatchCells {
  static constexpr bool PERSIST_ONLY = true;
  long n;
  const double *gp;   // [GEO_NC + 1][n]: the geometry planes, then x1
  const double *dtv;  // [n]
  double *uu, *pp;    // [NV][n]
  kz_implicit_result *res;
  unsigned long long *cnt;  // [NSLOT][SLOT_W]: [0] failures [1] iterations [2] solves
  __device__ long count() const { return n; }
  __device__ bool skip(const kz_physics &, long) const { return false; }
  __device__ void load_p(long t, double *p) const { ld(pp, n, t, p); }
  __device__ void geo(long t, Geo &gm) const { load_geo(gp, n, t, gp[GEO_NC * n + t], gm); }
  __device__ double dt(long t) const { return dtv[t]; }
  __device__ void solved(const kz_physics &ph, long t, const Geo &gm, const double *ppw, int iters, int ir, int wp,
                         int we, int wf) const {
    double u[NV];
    p2u(ppw, u, gm, ph.gam);
    st(uu, n, t, u);
    st(pp, n, t, ppw);
    res[t] = kz_implicit_result{1, ir, iters, wp, we, wf};
    unsigned long long *k = slot_of(cnt);
    atomicAdd(&k[1], (unsigned long long)iters);
    atomicAdd(&k[2], 1ULL);
  }
  __device__ void failed(long t) const {
    res[t] = kz_implicit_result{0, -1, 0, WP_RAD, WE_ENERGY, WF_LAB};
    atomicAdd(&slot_of(cnt)[0], 1ULL);
  }
};
// The cells of several runs as one sequence (a run group's implicit pass):
// run k owns t in [off_k, off_k + ndom_k), each with its own grid, fields,
// metric, dt slot value and counters.
struct RunCells {
  GridD g;
  Dev d;
  long off;
};
struct MultiCells {
  static constexpr bool PERSIST_ONLY = false;
  const RunCells *r;  // [nr], off ascending, r[0].off == 0
  int nr;
  long n;
  int sslot;
  __device__ int run(long t) const {
    int lo = 0, hi = nr - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (r[mid].off <= t) lo = mid;
      else hi = mid - 1;
    }
    return lo;
  }
  __device__ GridCells at(long t, long &tl) const {
    const int k = run(t);
    tl = t - r[k].off;
    return GridCells{r[k].g, r[k].d, sslot};
  }
  __device__ long count() const { return n; }
  __device__ bool skip(const kz_physics &ph, long t) const {
    long tl;
    const GridCells c = at(t, tl);
    return c.skip(ph, tl);
  }
  __device__ void load_p(long t, double *pp) const {
    long tl;
    const GridCells c = at(t, tl);
    c.load_p(tl, pp);
  }
  __device__ void geo(long t, Geo &gm) const {
    long tl;
    const GridCells c = at(t, tl);
    c.geo(tl, gm);
  }
  __device__ double dt(long t) const {
    long tl;
    const GridCells c = at(t, tl);
    return c.dt(tl);
  }
  __device__ void solved(const kz_physics &ph, long t, const Geo &gm, const double *ppw, int iters, int ir, int wp,
                         int we, int wf) const {
    long tl;
    const GridCells c = at(t, tl);
    c.solved(ph, tl, gm, ppw, iters, ir, wp, we, wf);
  }
  __device__ void failed(long t) const {
    long tl;
    const GridCells c = at(t, tl);
    c.failed(tl);
  }
};
template <class S, bool BR>
__global__ void __launch_bounds__(64) KZ_WPE(KZ_WPE_PREP) k_imp_prep(S s, ImpWork w, kz_physics ph) {
  ph.opac.synchrotron_bridge = BR;
  long t = TID;
  if (t == 0) {  // no appends run concurrently with this kernel
    *w.nslow = 0;
    if (w.qpos) {
      w.rc[0] = w.rc[1] = 0;
      for (int k = 0; k < 3; ++k) w.qpos[k] = 0;
    }
  }
  const long nd = s.count();
  if (t >= nd) return;
  if (s.skip(ph, t)) return;
  double dt = s.dt(t);
  double pp00[NV], pp0[NV];
  s.load_p(t, pp00);
  Geo gm;
  s.geo(t, gm);
  // the reference state and the starting block are stored before the
  // bisection, so that only its three inputs stay live through it
  double st_ehat, st_ut, st_tgas;
  int sw;
  {
    double uu00[NV];
    p2u(pp00, uu00, gm, ph.gam);
    st(w.uu00, nd, t, uu00);
    const double ehat = -calc_ff_rtt(pp00, gm);
    RadState st00;
    fill_radstate(pp00, gm, ph.gam, ph.opac, true, st00);
    sw = (ehat < ph.implicit.threshold * pp00[UU]) ? WP_RAD : WP_MHD;
    double *a = w.aux;
    a[IA_EHAT * nd + t] = st00.ehat;
    a[IA_UINT * nd + t] = st00.uint;
    a[IA_SGAS * nd + t] = st00.sgas;
    a[IA_KES * nd + t] = st00.kappaes;
    a[IA_KGA * nd + t] = st00.op.gas_abs;
    a[IA_KRA * nd + t] = st00.op.rad_abs;
    a[IA_KRR * nd + t] = st00.op.rad_ross;
    a[IA_SW * nd + t] = (double)sw;
    st_ehat = st00.ehat;
    st_ut = st00.ucon[0];
    st_tgas = st00.tgas;
  }
  // gather the cell into the list of its starting block, so that each
  // first-rung kernel runs full waves of one Newton variant: the wave (a
  // block) asks for its places in both lists with one atomic, whose answer is
  // not looked at before the bisection is done, so that the wave does not
  // stand in the queue of one address (12 ns per atomic, 2160 waves at
  // 384x360, two lists before)
  const unsigned long long m_mhd = __ballot(sw == WP_MHD), m_rad = __ballot(sw != WP_MHD);
  const int leader = __ffsll(m_mhd | m_rad) - 1;
  unsigned long long base = 0;
  if ((int)threadIdx.x == leader)
    base = atomicAdd(w.ncnt, ((unsigned long long)__popcll(m_rad) << 32) | (unsigned long long)__popcll(m_mhd));
  ImpCtx cx{&gm, ph.gam, &ph.rad, &ph.opac, &ph.implicit, 1.0};
  if (ph.implicit.start_with_bisect) {
    solve_1d_prim(pp00, st_ehat, st_ut, st_tgas, dt, cx, pp0);
  } else {
#pragma unroll
    for (int i = 0; i < NV; ++i) pp0[i] = pp00[i];
  }
  st(w.pp0, nd, t, pp0);
  base = __shfl(base, leader);
  const unsigned long long below = (1ULL << threadIdx.x) - 1ULL;
  if (sw == WP_MHD) w.list[(long)(base & 0xffffffffULL) + __popcll(m_mhd & below)] = (int32_t)t;
  else w.list[nd + (long)(base >> 32) + __popcll(m_rad & below)] = (int32_t)t;
}
// lengths of the starting-block lists that k_imp_prep filled
__device__ __forceinline__ long n_mhd(const ImpWork &w) { return (long)(*w.ncnt & 0xffffffffULL); }
__device__ __forceinline__ long n_rad(const ImpWork &w) { return (long)(*w.ncnt >> 32); }
__device__ __forceinline__ void imp_load(const ImpWork &w, long nd, long t, double *uu00, double *pp0, State0 &s0,
                                         LagOpac &lag) {
  ld(w.uu00, nd, t, uu00);
  ld(w.pp0, nd, t, pp0);
  const double *a = w.aux;
  s0.ehat = a[IA_EHAT * nd + t];
  s0.uint = a[IA_UINT * nd + t];
  s0.sgas = a[IA_SGAS * nd + t];
  lag.kappaes = a[IA_KES * nd + t];
  lag.op.gas_abs = a[IA_KGA * nd + t];
  lag.op.rad_abs = a[IA_KRA * nd + t];
  lag.op.rad_ross = a[IA_KRR * nd + t];
}
template <class S, int WP>
__device__ __forceinline__ void rung0_cell(NewtonLds &l, const S &s, const ImpWork &w, const kz_physics &ph, long i) {
  constexpr int which = WP == WP_MHD ? 0 : 1;
  if (i >= (WP == WP_MHD ? n_mhd(w) : n_rad(w))) return;
  const long nd = s.count();
  long t = w.list[which * nd + i];
  double uu00[NV], pp0[NV], ppw[NV];
  State0 s0;
  LagOpac lag;
  imp_load(w, nd, t, uu00, pp0, s0, lag);
  Geo gm;
  s.geo(t, gm);
  double dt = s.dt(t);
  ImpCtx cx{&gm, ph.gam, &ph.rad, &ph.opac, &ph.implicit, 1.0};
  int iters = 0;
  bool ok = ph.implicit.opdamp_maxlevels >= 0 &&
            solve_4d_prim_core<WP>(l, uu00, lag, s0, pp0, dt, cx, WE_ENERGY, WF_LAB, ppw, &iters);
  if (ok) {
    s.solved(ph, t, gm, ppw, iters, 0, WP, WE_ENERGY, WF_LAB);
  } else {
    unsigned long long k = atomicAdd(w.nslow, 1ULL);
    w.slow[k] = (int32_t)t;
  }
}
// launched with nblk(n, 64) + 1 blocks: ceil(nrad/64) + ceil(nmhd/64) never
// exceeds that for nrad + nmhd <= n
// W: waves per SIMD it is compiled for (launch_implicit_br).
template <class S, bool BR, int W>
__global__ void __launch_bounds__(64) KZ_WPE(W) k_imp_rung0(S s, ImpWork w, kz_physics ph) {
  ph.opac.synchrotron_bridge = BR;
  __shared__ NewtonLds l;
  const long brad = (n_rad(w) + 63) / 64;
  const long b = blockIdx.x;
  if (b < brad) rung0_cell<S, WP_RAD>(l, s, w, ph, b * 64 + threadIdx.x);
  else rung0_cell<S, WP_MHD>(l, s, w, ph, (b - brad) * 64 + threadIdx.x);
}
// Where a cell of the persistent first-rung launch goes when its Newton
// ends: solved (recorded with the rung's attempt) or to the later rungs'
// list of its starting block.
template <class S>
struct RungDone {
  const S *s;
  const ImpWork *w;
  const kz_physics *ph;
  int ir, which, wp, we, wf;
  __device__ void operator()(long t, const Geo &gm, const NewtonState &n, bool ok) const {
    if (ok) {
      s->solved(*ph, t, gm, n.pp, n.iter, ir, wp, we, wf);
      return;
    }
    const long nd = s->count();
    unsigned long long k = atomicAdd(&w->rc[which], 1ULL);
    w->rl[which * nd + k] = (int32_t)t;
    w->st[t] = 0;
  }
};
// Lanes of a wave that take cells from a queue of qlen entries.  Where the
// entries do not fill the launch, they are spread over its waves rather than
// packed 64 to a wave: lanes at different depths of their solves run one
// after the other, and a wave of its own costs an idle SIMD nothing (4099
// cells: first rung 15 -> 7 ms per solve).
__device__ __forceinline__ int queue_lanes(long qlen) {
  const long per = (qlen + gridDim.x - 1) / gridDim.x;
  return per < 1 ? 1 : (per > 64 ? 64 : (int)per);
}
// Work stealing over one queue (cells list[0 .. qlen)) with Newton variant
// WP at opdamp level 0: each lane holds one cell; the lanes without one claim
// the next queue entries together (one atomic per wave and refill) until the
// queue is exhausted; the loop ends when no lane holds a cell.  Every Newton
// ends within maxiter + 1 steps and the queue is finite, so every wave exits.
template <class S, int WP>
__device__ __forceinline__ void drain_queue(NewtonLds &l, const S &s, const ImpWork &w, const kz_physics &ph, const int32_t *list,
                                            long qlen, unsigned long long *qpos, int we, int wf,
                                            const RungDone<S> &done) {
  const int lane = threadIdx.x & 63;
  const unsigned long long below = (1ULL << lane) - 1ULL;
  const long nd = s.count();
  bool has = false, exhausted = qlen <= 0 || lane >= queue_lanes(qlen);
  long t = 0;
  double dt = 0;
  NewtonState ns;
  Geo gm;
  for (;;) {
    const unsigned long long need = __ballot(!has && !exhausted);
    if (need) {
      const int leader = __ffsll((unsigned long long)need) - 1;
      const int cnt = __popcll(need);
      long base = 0;
      if (lane == leader) base = (long)atomicAdd(qpos, (unsigned long long)cnt);
      base = __shfl(base, leader);
      if (!has && !exhausted) {
        const long q = base + __popcll(need & below);
        if (q < qlen && ph.implicit.opdamp_maxlevels < 0) {
          done(list[q], gm, ns, false);  // the ladder has no level to run (implicit.zig:961)
        } else if (q < qlen) {
          t = list[q];
          double uu00[NV], pp0[NV];
          State0 s0;
          LagOpac lag;
          imp_load(w, nd, t, uu00, pp0, s0, lag);
          newton_keep(l, uu00, s0, lag);
          s.geo(t, gm);
          dt = s.dt(t);
          const ImpCtx cx{&gm, ph.gam, &ph.rad, &ph.opac, &ph.implicit, 1.0};
          newton_start(ns, uu00, pp0);
          has = true;
        }
      }
      if (base + cnt >= qlen) exhausted = true;
    }
    if (!__ballot(has)) {
      if (__ballot(!exhausted)) continue;
      break;
    }
    if (has) {
      const ImpCtx cx{&gm, ph.gam, &ph.rad, &ph.opac, &ph.implicit, 1.0};
      const int r = newton_pass<WP>(ns, l, dt, cx, we, wf);
      if (r != 0) {
        done(t, gm, ns, r > 0);
        has = false;
      }
    }
  }
}
// first rung over both starting-block lists, RAD-start queue first
template <class S, bool BR>
__global__ void __launch_bounds__(64) KZ_WPE(KZ_WPE_RUNG0) k_imp_rung0_persist(S s, ImpWork w, kz_physics ph) {
  ph.opac.synchrotron_bridge = BR;
  __shared__ NewtonLds l;
  const long nd = s.count();
  const RungDone<S> dr{&s, &w, &ph, 0, 1, WP_RAD, WE_ENERGY, WF_LAB};
  drain_queue<S, WP_RAD>(l, s, w, ph, w.list + nd, n_rad(w), &w.qpos[0], WE_ENERGY, WF_LAB, dr);
  const RungDone<S> dm{&s, &w, &ph, 0, 0, WP_MHD, WE_ENERGY, WF_LAB};
  drain_queue<S, WP_MHD>(l, s, w, ph, w.list, n_mhd(w), &w.qpos[1], WE_ENERGY, WF_LAB, dm);
}
// bits of ImpWork::st: RUNG_FAILED << r and RUNG_SOLVED << r for rung r = 1..5
constexpr unsigned RUNG_FAILED = 1u, RUNG_SOLVED = 1u << 8, RUNG_FAILED_MASK = 0x3eu;
// a cell's bits as the other waves have set them (past this die's caches)
__device__ __forceinline__ unsigned rung_state(const ImpWork &w, long t) {
  return __hip_atomic_load(&w.st[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool rung_solved_below(const ImpWork &w, long t, int ir) {
  return rung_state(w, t) & (((1u << ir) - 2u) * RUNG_SOLVED);
}
// Rungs 1..5 of level 0 (implicit.zig:961-968) over the m cells the first
// rung left (both starting-block lists, MHD start then RAD start), as one
// queue of 5 m attempts ordered by rung.  Every attempt starts from the stored
// reference state and knows nothing of the others, so the rungs of a cell may
// run at the same time; the cell takes the solution of the lowest rung that
// solves it, as the reference's ladder does.  w.st[cell] has a bit for each
// rung that failed and one for each that solved:
//   a lane whose attempt solved its cell stores the solution once every lower
//   rung has failed, waits while some are open, and drops it when one solves;
//   an attempt that is under way or about to start is dropped when a lower
//   rung has solved the cell;
//   the attempt that completes five failures sends the cell to the slow list.
// A lane waits only for attempts that were claimed before its own and that
// their lanes began at once, each at most maxiter + 1 iterations long, so
// every wave ends.  Attempts of one rung and starting block stand together in
// the queue, so a wave's lanes mostly run one primitive block.
//
// Bound by the serial chain of the longest ladder: run one after the other by
// one lane per cell, the five rungs of the slowest cell set the time of every
// batch.  This launch, with queue_lanes: 69 -> 8 ms at 4099 cells (480 of them
// here), 148 -> 40 ms at 2^19; the first rung is another 8 and 36 ms.  In the
// independent-cell batch rung 1 fails for 93 % of these cells and rung 2 then
// solves 96 %, so little is tried in vain.
template <class S, bool BR>
__global__ void __launch_bounds__(64) KZ_WPE(KZ_WPE_RUNG0) k_imp_ladder_persist(S s, ImpWork w, kz_physics ph) {
  ph.opac.synchrotron_bridge = BR;
  const int lane = threadIdx.x & 63;
  const unsigned long long below = (1ULL << lane) - 1ULL;
  const long nd = s.count();
  __shared__ NewtonLds l;
  const long n0 = (long)w.rc[0], m = n0 + (long)w.rc[1], qlen = 5 * m;
  // lanes for the two rungs that most of these cells need
  bool has = false, held = false, exhausted = qlen <= 0 || lane >= queue_lanes(2 * m);
  long t = 0;
  int ir = 1, wp = WP_MHD, we = WE_ENERGY, wf = WF_FF;
  double dt = 0;
  NewtonState ns;
  Geo gm;
  for (;;) {
    const unsigned long long need = __ballot(!has && !exhausted);
    if (need) {
      const int leader = __ffsll((unsigned long long)need) - 1;
      const int cnt = __popcll(need);
      long base = 0;
      if (lane == leader) base = (long)atomicAdd(&w.qpos[2], (unsigned long long)cnt);
      base = __shfl(base, leader);
      if (!has && !exhausted) {
        const long q = base + __popcll(need & below);
        if (q < qlen) {
          ir = 1 + (int)(q / m);
          const long i = q - (ir - 1) * m;
          const int sw = i < n0 ? WP_MHD : WP_RAD, ot = i < n0 ? WP_RAD : WP_MHD;
          t = i < n0 ? w.rl[i] : w.rl[nd + (i - n0)];
          if (ph.implicit.opdamp_maxlevels < 0) {  // no level to run (implicit.zig:961)
            if (ir == 1) {
              unsigned long long k = atomicAdd(w.nslow, 1ULL);
              w.slow[k] = (int32_t)t;
            }
          } else if (!rung_solved_below(w, t, ir)) {
            double uu00[NV], pp0[NV];
            State0 s0;
            LagOpac lag;
            imp_load(w, nd, t, uu00, pp0, s0, lag);
            newton_keep(l, uu00, s0, lag);
            s.geo(t, gm);
            dt = s.dt(t);
            wp = (ir == 1 || ir == 4) ? sw : ot;
            we = (ir >= 4) ? WE_ENTROPY : WE_ENERGY;
            wf = (ir == 2) ? WF_LAB : WF_FF;
            newton_start(ns, uu00, pp0);
            has = true;
          }
        }
      }
      if (base + cnt >= qlen) exhausted = true;
    }
    if (!__ballot(has)) {
      if (__ballot(!exhausted)) continue;  // only attempts that nobody needs any more were claimed
      break;
    }
    if (has && !held) {
      const ImpCtx cx{&gm, ph.gam, &ph.rad, &ph.opac, &ph.implicit, 1.0};
      int r = 0;
      if (wp == WP_MHD) r = newton_pass<WP_MHD>(ns, l, dt, cx, we, wf);
      if (wp == WP_RAD) r = newton_pass<WP_RAD>(ns, l, dt, cx, we, wf);
      if (r > 0) {
        atomicOr(&w.st[t], RUNG_SOLVED << ir);
        held = true;
      } else if (r < 0) {
        const unsigned now = atomicOr(&w.st[t], RUNG_FAILED << ir) | (RUNG_FAILED << ir);
        if ((now & RUNG_FAILED_MASK) == RUNG_FAILED_MASK) {
          unsigned long long k = atomicAdd(w.nslow, 1ULL);
          w.slow[k] = (int32_t)t;
        }
        has = false;
      }
    }
    if (has && (held || ns.at == AT_UPDATE)) {
      const unsigned now = rung_state(w, t);
      const unsigned low = (1u << ir) - 2u;  // the rungs 1 .. ir - 1
      if (now & (low * RUNG_SOLVED)) {
        has = held = false;
      } else if (held && (now & low) == low) {
        s.solved(ph, t, gm, ns.pp, ns.iter, ir, wp, we, wf);
        has = held = false;
      }
    }
    if (!__ballot(has && !held)) __builtin_amdgcn_s_sleep(8);
  }
}

// The rest of the ladder over `slow` from opdamp level `first_level` (0:
// rungs 1..5 of level 0 first; 1: after the persistent rung launches).
template <class S, bool BR>
__global__ void __launch_bounds__(64) k_imp_slow(S s, ImpWork w, kz_physics ph, int first_level) {
  ph.opac.synchrotron_bridge = BR;
  __shared__ NewtonLds l;
  long i = TID;
  // the first-rung lists have been consumed; clear them for the next pass
  if (i == 0) *w.ncnt = 0;
  if (i >= (long)*w.nslow) return;
  const long nd = s.count();
  long t = w.slow[i];
  double uu00[NV], pp0[NV];
  State0 s0;
  LagOpac lag;
  imp_load(w, nd, t, uu00, pp0, s0, lag);
  const int sw = (int)w.aux[IA_SW * nd + t];
  const int ot = (sw == WP_RAD) ? WP_MHD : WP_RAD;
  Geo gm;
  s.geo(t, gm);
  double dt = s.dt(t);
  const kz_implicit_params &ip = ph.implicit;
  ImpCtx cx{&gm, ph.gam, &ph.rad, &ph.opac, &ip, 1.0};
  for (int level = first_level; level <= ip.opdamp_maxlevels; ++level) {
    double od = 1.0;
    for (int k = 0; k < level; ++k) od /= ip.opdamp_factor;
    cx.opdamp = od;
    for (int ir = level == 0 ? 1 : 0; ir < 6; ++ir) {
      int wp = (ir == 0 || ir == 1 || ir == 4) ? sw : ot;
      int we = (ir >= 4) ? WE_ENTROPY : WE_ENERGY;
      int wf = (ir == 0 || ir == 2) ? WF_LAB : WF_FF;
      double ppw[NV];
      int iters = 0;
      bool ok = (wp == WP_MHD) ? solve_4d_prim_core<WP_MHD>(l, uu00, lag, s0, pp0, dt, cx, we, wf, ppw, &iters)
                               : solve_4d_prim_core<WP_RAD>(l, uu00, lag, s0, pp0, dt, cx, we, wf, ppw, &iters);
      if (ok) {
        s.solved(ph, t, gm, ppw, iters, ir, wp, we, wf);
        return;
      }
    }
  }
  s.failed(t);
}

// The implicit kernels over the n cells of a cell source, with the
// synchrotron bridge of the opacities (BR) fixed on or off at kernel entry:
// left to a runtime test, the bridge's branch costs the ladder's register
// allocation about 64 spilled registers.  w carries the queue arrays when
// `persist`.
template <class S, bool BR>
static void launch_implicit_br(const S &cells, const ImpWork &w, const kz_physics &ph, long n, bool persist,
                               unsigned ncu, hipStream_t st) {
  const unsigned nb = nblk(n, 64);
  k_imp_prep<S, BR><<<nb, 64, 0, st>>>(cells, w, ph);
  // batches know no other shape: their merged kernels would be reached by nothing
  if (persist || S::PERSIST_ONLY) {
    const unsigned width = KZ_PERSIST_PER_CU * ncu, np = width < (unsigned long)n ? width : (unsigned)n;
    k_imp_rung0_persist<S, BR><<<np, 64, 0, st>>>(cells, w, ph);
    k_imp_ladder_persist<S, BR><<<np, 64, 0, st>>>(cells, w, ph);
    k_imp_slow<S, BR><<<nb, 64, 0, st>>>(cells, w, ph, 1);
  } else if constexpr (!S::PERSIST_ONLY) {
    // Two waves per SIMD hide each other's latencies at the price of 167 spilled
    // vector registers (384 B of scratch per lane; 157 to 189 over the cell
    // sources and the bridge): where the cells fill the chip several times over
    // that wins, with fewer the chain of the longest solve sets the time and a
    // wave is better off alone.  Whole implicit pass, one and two
    // waves: 256x256 166 and 179 us, 384x360 288 and 299, 512x384 383 and 364,
    // 512x400 422 and 382, 128x128x16 528 and 463, 128x128x32 932 and 820.  With
    // the bridge 512x384 413 and 417, 512x400 461 and 450, 128x128x16 567 and
    // 535, 128x128x32 1005 and 960.  A step of a run group, without and with the
    // bridge: three 256x256 runs 1645 and 1646 us, 1735 and 1737; two 384x360
    // runs 1930 and 1892, 2026 and 1988.
    if (n >= wide_cells(ncu)) k_imp_rung0<S, BR, 2><<<nb + 1, 64, 0, st>>>(cells, w, ph);
    else k_imp_rung0<S, BR, KZ_WPE_RUNG0><<<nb + 1, 64, 0, st>>>(cells, w, ph);
    k_imp_slow<S, BR><<<nb, 64, 0, st>>>(cells, w, ph, 0);
  }
}
// The option variants (kz_options.hip).
void opt_launch_wavespeeds(const GridD &g, const Dev &d, const kz_physics &ph, unsigned nb, hipStream_t st);
void opt_launch_u2p_zamo(const GridD &g, const Dev &d, const kz_physics &ph, unsigned nb, hipStream_t st);
void opt_launch_face_flux(const GridD &g, const Dev &d, const kz_physics &ph, const FaceTiles &ft, unsigned nb,
                          hipStream_t st);
template <class S>
void opt_launch_implicit_bridge(const S &cells, const ImpWork &w, const kz_physics &ph, long n, bool persist,
                                unsigned ncu, hipStream_t st);

#endif
