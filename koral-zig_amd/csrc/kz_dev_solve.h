// kz_dev_solve.h — the per-cell inversions and the implicit four-force
// Newton of the koral step as gfx950 device code: koral/solve/invert.zig
// (u2p W-Newton, MHD floors), koral/solve/invert_rad.zig (closed-form M1
// u2p, radiation floors) and koral/solve/implicit.zig (6-rung ladder).
// One thread runs one cell's whole solve; branch decisions follow the
// reference exactly, so iteration counts and flags match the CPU path.
#pragma once

#include "kz_dev.h"

namespace kzd {

// ---- invert.zig ------------------------------------------------------------
struct Resid {
  double f, df, err;
};
struct Cons {
  double Qn, Qtsq, D, QdotBsq, Bsq, Sc;
};

KZDM Resid f_u2p(int etype, double Wp, const Cons &c, double pg) {
  double W = Wp + c.D;  // invert.zig:116-210 (both residuals share wKinematics)
  double x = c.Bsq + W;
  double wsq = W * W;
  double w3 = wsq * W;
  double x3 = x * x * x;
  double v2 = (wsq * c.Qtsq + c.QdotBsq * (c.Bsq + 2.0 * W)) / (wsq * (x * x));
  double gamma2 = 1.0 / (1.0 - v2);
  double gamma = kzm_sqrt(gamma2);
  double rho0 = c.D / gamma;
  double wmrho0 = Wp / gamma2 - c.D * v2 / (1.0 + gamma);
  double dvsq = -2.0 / x3 * (c.Qtsq + c.QdotBsq * (3.0 * W * x + c.Bsq * c.Bsq) / w3);
  double dwmrho0dvsq = c.D * (gamma * 0.5 - 1.0) - Wp;
  Resid r;
  if (etype == 0) {
    double u = wmrho0 / pg;
    double p = (pg - 1.0) * u;
    r.f = c.Qn + W - p + 0.5 * c.Bsq * (1.0 + v2) - c.QdotBsq / 2.0 / wsq;
    r.err = kzm_fabs(r.f) / (kzm_fabs(c.Qn) + kzm_fabs(W) + kzm_fabs(p) + kzm_fabs(0.5 * c.Bsq * (1.0 + v2)) +
                             kzm_fabs(c.QdotBsq / 2.0 / wsq));
    double dp1 = (pg - 1.0) * (1.0 - v2) / pg;
    double idw = (pg - 1.0) / pg;
    double dp2 = dwmrho0dvsq * idw;
    double dpdW = dp1 + dp2 * dvsq;
    r.df = 1.0 - dpdW + c.QdotBsq / (wsq * W) + 0.5 * c.Bsq * dvsq;
  } else {
    double pressure = (pg - 1.0) / pg * wmrho0;
    double indexn = 1.0 / (pg - 1.0);
    double ss = dm_log_entropy(pressure, rho0, indexn);
    r.f = -c.Sc + c.D * ss;
    r.err = kzm_fabs(r.f) / (kzm_fabs(c.Sc) + kzm_fabs(c.D * ss));
    double dssdrho = pg / ((1.0 - pg) * rho0);
    double dssdchi = 1.0 / ((pg - 1.0) * wmrho0);
    double dwmrho0dw = 1.0 / (gamma * gamma);
    double drho0dvsq = -c.D * gamma * 0.5;
    double dssdw = dwmrho0dw * dssdchi;
    double dssdvsq = drho0dvsq * dssdrho + dwmrho0dvsq * dssdchi;
    double dssdwp = dssdw + dssdvsq * dvsq;
    r.df = c.D * dssdwp;
  }
  return r;
}

// the two halves of invert.zig:221-224: W below the physical range, and a
// residual that is no number.  The first needs no residual, so it is asked
// first.
KZD bool w_below(double W, const Cons &c) {
  return (W * W * W * (W + 2.0 * c.Bsq) - c.QdotBsq * (2.0 * W + c.Bsq)) <= W * W * (c.Qtsq - c.Bsq * c.Bsq);
}
KZD bool r_bad(const Resid &r) { return !kzm_isfinite(r.f) || !kzm_isfinite(r.df); }

// invert.zig:235-404 u2pSolverW, from the energy equation (etype 0) or the
// entropy (1), and with `fallback` from the entropy where the energy equation
// fails (one cell in twenty of a 48x48x16 wedge), which is how its callers use
// it (invert.zig:441-451, implicit.zig:293-296).  pp in/out; returns the
// reference's code of the last attempt and in *etype which one that was.
//
// The reference evaluates the residual at every trial W and once more, at the
// same W, where it goes on from it; here the value of an accepted trial is
// kept for the next iteration (the same arguments, the same bits), so an
// iteration takes one evaluation instead of two, and a trial below the range
// (w_below) takes none.  Bracketing, damped trials, the step after a zero
// derivative and both equations share this one evaluation: a lane that has
// fallen back runs beside one that has not, and the code stands once.
KZDM int u2p_solver_w(const double *uu, double *pp, const Geo &gm, int *etype_io, bool fallback, double pg) {
  int etype = *etype_io;
  double gi = 1.0 / gm.gdet;
  double alpha = gm.alpha;
  Cons c;
  c.D = uu[RHO] * gi * alpha;
  c.Sc = uu[ENTR] * gi * alpha;
  double Qcov[4] = {(uu[UU] * gi - uu[RHO] * gi) * alpha, uu[VX] * gi * alpha, uu[VY] * gi * alpha,
                    uu[VZ] * gi * alpha};
  double Qcon[4];
  raise4(Qcov, gm, Qcon);
  double Bcon[4] = {0, uu[B1] * gi * alpha, uu[B2] * gi * alpha, uu[B3] * gi * alpha}, Bcov[4];
  lower4(Bcon, gm, Bcov);
  c.Bsq = dot4(Bcon, Bcov);
  double QdotB = dot4(Qcov, Bcon);
  c.QdotBsq = QdotB * QdotB;
  // n_mu = (-alpha, 0, 0, 0): the reference's full sums over it add only
  // zeros to these (a metric is finite), and to Qt what 0 * Qcon gives, zero
  // or NaN
  double Qt[4];
  {
    const double zero = 0.0 * Qcon[1] + 0.0 * Qcon[2] + 0.0 * Qcon[3];
    const double nc = -alpha;
    c.Qn = Qcon[0] * nc;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double ncon = 0.0 + nc * gm.G[i][0];
      const double s = 0.0 + ((i == 0 ? 1.0 : 0.0) + ncon * nc) * Qcon[0];
      Qt[i] = (i == 0 ? s : s + Qcon[i]) + zero;
    }
  }
  double Qtcov[4];
  lower4(Qt, gm, Qtcov);
  c.Qtsq = dot4(Qt, Qtcov);
  const double conv = 1.0e-10;

  enum { BRACKET, TRIAL, PLAIN };
  int mode = BRACKET, tries = 0, iter = 0;
  double W = 0, Wt = 0, f0 = 0, dfdW = 0, dumpfac = 1.0, errr = 0;
  bool start = true;
  for (;;) {
    if (start) {
      double qsq = 0;
#pragma unroll
      for (int i = 1; i < 4; ++i)
#pragma unroll
        for (int j = 1; j < 4; ++j) qsq += pp[VX - 1 + i] * pp[VX - 1 + j] * gm.g[i][j];
      Wt = (pp[RHO] + pg * pp[UU]) * (1.0 + qsq);
      mode = BRACKET;
      tries = iter = 0;
      start = false;
    }
    Resid r{};
    bool oob = mode != PLAIN && w_below(Wt, c);
    if (!oob) {
      r = f_u2p(etype, Wt - c.D, c, pg);
      oob = mode != PLAIN && r_bad(r);
    }
    int code = 0;
    bool ends = false;  // this attempt's iteration ends
    if (oob) {
      tries += 1;
      if (mode == BRACKET) {
        Wt *= 10.0;
        if (tries >= 50) code = -150;
      } else {
        dumpfac /= 2.0;
        Wt = W - dumpfac * f0 / dfdW;
        if (tries >= 100) code = -101;
      }
    } else {
      if (mode == TRIAL) {
        const double Wprev = W;
        W = Wt;
        if (kzm_fabs(W) > 1.0 / 1.0e-80) code = -103;
        else if (kzm_fabs((W - Wprev) / Wprev) < conv && errr < 1.0e-1) ends = true;
      } else {
        W = Wt;
      }
      if (code == 0 && !ends) {
        if (iter >= 50) {
          ends = true;
        } else {
          iter += 1;
          errr = r.err;
          if (errr < conv) {
            ends = true;
          } else if (r.df == 0.0) {
            Wt = W * 1.1;
            mode = PLAIN;
          } else {
            f0 = r.f;
            dfdW = r.df;
            dumpfac = 1.0;
            tries = 0;
            mode = TRIAL;
            Wt = W - f0 / dfdW;
          }
        }
      }
      if (ends) {
        if (iter >= 50) code = -102;
        else if (!kzm_isfinite(W)) code = -103;
        else {
          double wsq = W * W;
          double xsq = (c.Bsq + W) * (c.Bsq + W);
          double v2 = (wsq * c.Qtsq + c.QdotBsq * (c.Bsq + 2.0 * W)) / (wsq * xsq);
          double gamma2 = 1.0 / (1.0 - v2);
          double gamma = kzm_sqrt(gamma2);
          double rho = c.D / gamma;
          double entr = c.Sc / gamma;
          double uint = 1.0 / pg * (W / gamma2 - rho);
          double ut[4];
#pragma unroll
          for (int i = 1; i < 4; ++i) ut[i] = gamma / (W + c.Bsq) * (Qt[i] + QdotB * Bcon[i] / W);
          if (!kzm_isfinite(ut[1])) code = -120;
          else if (uint < 0.0 || gamma2 < 0.0 || W != W || !kzm_isfinite(W)) code = -104;
          else {
            pp[RHO] = rho;
            pp[UU] = uint;
            pp[VX] = ut[1];
            pp[VY] = ut[2];
            pp[VZ] = ut[3];
            if (rho < 0.0) code = -105;
            else {
              pp[ENTR] = entr;
              pp[B1] = uu[B1] * gi;
              pp[B2] = uu[B2] * gi;
              pp[B3] = uu[B3] * gi;
              *etype_io = etype;
              return 0;
            }
          }
        }
      }
    }
    if (code != 0) {
      if (etype != 0 || !fallback) {
        *etype_io = etype;
        return code;
      }
      etype = 1;
      start = true;
    }
  }
}

// invert.zig:422-467 u2pMhd; returns ret (0/-1/-2/-3), sets *entropy_used.
// A failed solve leaves pp as it came (the reference's ppbak), except that
// its guess fields are put back here.
KZDM int u2p_mhd(const double *uu_in, double *pp, const Geo &gm, double gam, const kz_floor_params &f,
                 int *entropy_used) {
  double uu[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) uu[i] = uu_in[i];
  double keep[5] = {pp[RHO], pp[UU], pp[VX], pp[VY], pp[VZ]};
  int ret = 0;
  if (uu[RHO] * gm.alpha / gm.gdet < 0.0) {
    pp[RHO] = f.rhofloor;
    uu[RHO] = f.rhofloor * gm.gdet / gm.alpha;
    ret = -2;
  }
  int etype = 0;
  const int r = u2p_solver_w(uu, pp, gm, &etype, true, gam);
  *entropy_used = etype;
  if (etype) ret = -1;
  if (r < 0) {
    ret = -3;  // pp keeps the incoming primitives
    pp[RHO] = keep[0];
    pp[UU] = keep[1];
    pp[VX] = keep[2];
    pp[VY] = keep[3];
    pp[VZ] = keep[4];
  }
  return ret;
}

// invert.zig:474-715 checkFloorsMhd; *guard counts the guard-ladder
// recoveries (n_guard_recoveries).  ZAMO selects the b^2/rho floor in the
// ZAMO frame (b2rhofloorframe 1) at compile time, so that the kernels of the
// default drift frame carry none of its code.
template <bool ZAMO = false>
KZD int check_floors_mhd(double *pp, const Geo &gm, double pg, const kz_floor_params &fp, int *guard) {
  int ret = 0;
  // invert.zig:485-492: the ZAMO floor adds its delta to the conserveds of
  // the primitives as they enter, before any floor
  double uu_entry[NV];
  if (ZAMO) p2u_mhd(pp, uu_entry, gm, pg);
  if (pp[RHO] < fp.rhofloor) {
    pp[RHO] = fp.rhofloor;
    ret = -1;
  }
  if (pp[UU] < fp.uurhoratiomin * pp[RHO]) {
    pp[UU] = fp.uurhoratiomin * pp[RHO];
    ret = -1;
  }
  if (pp[UU] > fp.uurhoratiomax * pp[RHO]) {
    pp[UU] = fp.uurhoratiomax * pp[RHO];
    ret = -1;
  }
  {
    double ucon[4], ucov[4];
    ucon_ucov(pp, gm, ucon, ucov);
    double bcon[4], bcov[4], bsq;
    bcon_bcov_bsq(pp[B1], pp[B2], pp[B3], ucon, ucov, gm, bcon, bcov, &bsq);
    double f = 1.0, fuu = 1.0;
    bool floored = false;
    if (bsq > fp.b2rhoratiomax * pp[RHO]) {
      f = bsq / (fp.b2rhoratiomax * pp[RHO]);
      floored = true;
    }
    if (!ZAMO && fp.b2rhofloorframe == 0 && fp.b2uufloor && bsq > fp.b2uuratiomax * pp[UU]) {
      fuu = bsq / (fp.b2uuratiomax * pp[UU]);
      floored = true;
    }
    if (ZAMO && floored) {
      // invert.zig:649-684: the new mass drho = rho (f - 1) moves with the
      // normal observer n^mu = -alpha g^{mu 0}; its conserved vector is added
      // to the entry conserveds through B3 and the primitives recovered by the
      // hot, then the entropy solver; if both fail the fluid-frame backup
      // scales rho and u by f
      double pporg[NV];
#pragma unroll
      for (int iv = 0; iv < NV; ++iv) pporg[iv] = pp[iv];
      const double drho = pp[RHO] * (f - 1.0);
      double etacon[4], etarel[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) etacon[i] = -gm.alpha * gm.G[i][0];
      vel4_to_velr(etacon, gm, true, etarel);
      double dpp[NV], duu[NV], uu[NV];
#pragma unroll
      for (int iv = 0; iv < NV; ++iv) dpp[iv] = 0.0;
      dpp[RHO] = drho;
      dpp[VX] = etarel[1];
      dpp[VY] = etarel[2];
      dpp[VZ] = etarel[3];
      p2u_mhd(dpp, duu, gm, pg);
#pragma unroll
      for (int iv = 0; iv < NV; ++iv) uu[iv] = iv <= B3 ? uu_entry[iv] + duu[iv] : 0.0;
      int etype = 0;
      if (u2p_solver_w(uu, pp, gm, &etype, true, pg) < 0) {
#pragma unroll
        for (int iv = 0; iv < NV; ++iv) pp[iv] = pporg[iv];
        pp[RHO] *= f;
        pp[UU] *= f;
      }
      ret = -1;
    } else if (floored) {
      double wold = pp[RHO] + pp[UU] * pg;
      pp[RHO] *= f;
      pp[UU] *= fp.isentropic_b2rhofloors ? f : fuu;
      double wnew = pp[RHO] + pp[UU] * pg;
      bool guarded = false;
      if (gm.x1 >= fp.horizon_x1) {
        do {
          double Bcon[4] = {0, pp[B1], pp[B2], pp[B3]}, Bcov[4];
          lower4(Bcon, gm, Bcov);
          double Bsq = dot4(Bcon, Bcov);
          double Bmag = kzm_sqrt(Bsq);
          if (!(bsq > 1.0e-10 * wnew && Bsq > 1.0e-10 * wnew)) {
            guarded = true;
            break;
          }
          double betapar = -bcon[0] / (bsq * ucon[0]);
          double betasq = betapar * betapar * bsq;
          double betasqmax = 1.0 - 1.0 / (fp.gammamaxhd * fp.gammamaxhd);
          if (betasq > betasqmax) betasq = betasqmax;
          double gammapar = 1.0 / kzm_sqrt(1.0 - betasq);
          double ucondr[4];
#pragma unroll
          for (int iv = 0; iv < 4; ++iv) ucondr[iv] = gammapar * (ucon[iv] + betapar * bcon[iv]);
          if (!kzm_isfinite(ucondr[0]) || kzm_fabs(ucondr[0]) < 1.0e-10) {
            guarded = true;
            break;
          }
          double udotB = dot4(ucon, Bcov);
          double QdotB = udotB * wold * ucon[0];
          double xx = 2.0 * QdotB / (Bmag * wnew * ucondr[0]);
          if (!(xx <= 1.0e10)) {
            xx = 1.0e10;
            guarded = true;
          }
          if (!(xx >= -1.0e10)) {
            xx = -1.0e10;
            guarded = true;
          }
          double vpar = xx / (ucondr[0] * (1.0 + kzm_sqrt(1.0 + xx * xx)));
          double vcon[4];
          vcon[0] = 1.0;
#pragma unroll
          for (int iv = 1; iv < 4; ++iv) vcon[iv] = vpar * Bcon[iv] / Bmag + ucondr[iv] / ucondr[0];
          for (int idamp = 0; idamp < 50; ++idamp) {
            double bv = 0.0, cv = 0.0;
#pragma unroll
            for (int iv = 1; iv < 4; ++iv) {
              bv += vcon[iv] * gm.g[0][iv];
#pragma unroll
              for (int jv = 1; jv < 4; ++jv) cv += vcon[iv] * vcon[jv] * gm.g[iv][jv];
            }
            if (gm.g[0][0] + 2.0 * bv + cv < -1.0 / (fp.gammamaxhd * fp.gammamaxhd)) break;
            guarded = true;
            vpar *= 0.5;
#pragma unroll
            for (int iv = 1; iv < 4; ++iv) vcon[iv] = vpar * Bcon[iv] / Bmag + ucondr[iv] / ucondr[0];
          }
          double ucont[4];
          if (vel3_to_velr(vcon, gm, ucont) != E_OK) {
            guarded = true;
            break;
          }
          pp[VX] = ucont[1];
          pp[VY] = ucont[2];
          pp[VZ] = ucont[3];
        } while (0);
      }
      if (guarded) *guard += 1;
      ret = -1;
    }
  }
  {
    double qsq = 0;
#pragma unroll
    for (int i = 1; i < 4; ++i)
#pragma unroll
      for (int j = 1; j < 4; ++j) qsq += pp[VX - 1 + i] * pp[VX - 1 + j] * gm.g[i][j];
    double gamma2 = 1.0 + qsq;
    if (gamma2 > fp.gammamaxhd * fp.gammamaxhd) {
      double qsqmax = fp.gammamaxhd * fp.gammamaxhd - 1.0;
      double a = kzm_sqrt(qsqmax / qsq);
#pragma unroll
      for (int j = 1; j < 4; ++j) pp[VX - 1 + j] *= a;
      ret = -1;
    }
  }
  if (ret < 0) pp[ENTR] = s_from_u(pp[RHO], pp[UU], pg);
  return ret;
}

// ---- invert_rad.zig ----------------------------------------------------------
constexpr double GSL = 1.0 - 1e-10;

KZD double m1_gammarel2(const Geo &gm, const double av[4]) {  // :66-124
  double gn11 = gm.G[0][0], gn12 = gm.G[0][1], gn13 = gm.G[0][2], gn14 = gm.G[0][3];
  double gn22 = gm.G[1][1], gn23 = gm.G[1][2], gn24 = gm.G[1][3], gn33 = gm.G[2][2], gn34 = gm.G[2][3],
         gn44 = gm.G[3][3];
  double rdtt = av[0], rdtx = av[1], rdty = av[2], rdtz = av[3];
  double mix = gn12 * rdtx + gn13 * rdty + gn14 * rdtz;
  double sq = kzm_sqrt(4.0 * (gn11 * gn11) * (rdtt * rdtt) + mix * mix +
                       gn11 * (8.0 * gn12 * rdtt * rdtx + 3.0 * gn22 * (rdtx * rdtx) + 8.0 * gn13 * rdtt * rdty +
                               6.0 * gn23 * rdtx * rdty + 3.0 * gn33 * (rdty * rdty) + 8.0 * gn14 * rdtt * rdtz +
                               6.0 * gn24 * rdtx * rdtz + 6.0 * gn34 * rdty * rdtz + 3.0 * gn44 * (rdtz * rdtz)));
  double den = gn11 * (rdtt * rdtt) + 2.0 * gn12 * rdtt * rdtx + gn22 * (rdtx * rdtx) + 2.0 * gn13 * rdtt * rdty +
               2.0 * gn23 * rdtx * rdty + gn33 * (rdty * rdty) + 2.0 * (gn14 * rdtt + gn24 * rdtx + gn34 * rdty) * rdtz +
               gn44 * (rdtz * rdtz);
  double g2a = (-0.25 * (2.0 * (gn11 * gn11) * (rdtt * rdtt) + mix * (mix + sq) +
                         gn11 * (4.0 * gn12 * rdtt * rdtx + gn22 * (rdtx * rdtx) + 2.0 * gn23 * rdtx * rdty +
                                 gn33 * (rdty * rdty) + 2.0 * gn24 * rdtx * rdtz + 2.0 * gn34 * rdty * rdtz +
                                 gn44 * (rdtz * rdtz) + rdtt * (4.0 * gn13 * rdty + 4.0 * gn14 * rdtz + sq)))) /
               den;
  double g2;
  if (g2a < GSL || !kzm_isfinite(g2a)) {
    g2 = (0.25 * (-2.0 * (gn11 * gn11) * (rdtt * rdtt) -
                  1.0 * gn11 * (4.0 * gn12 * rdtt * rdtx + gn22 * (rdtx * rdtx) +
                                rdty * (4.0 * gn13 * rdtt + 2.0 * gn23 * rdtx + gn33 * rdty) +
                                2.0 * (2.0 * gn14 * rdtt + gn24 * rdtx + gn34 * rdty) * rdtz + gn44 * (rdtz * rdtz)) +
                  gn11 * rdtt * sq + mix * (-1.0 * gn12 * rdtx - 1.0 * gn13 * rdty - 1.0 * gn14 * rdtz + sq))) /
         den;
  } else {
    g2 = g2a;
  }
  double gr2 = g2 * gm.alpha * gm.alpha;
  if (gr2 > GSL && gr2 < 1.0) gr2 = 1.0;
  return gr2;
}

KZD void m1_cold(const Geo &gm, const double in[4], double gr2, double av[4], double *erf_o, double ur[4]) {
  double gn11 = gm.G[0][0], gn12 = gm.G[0][1], gn13 = gm.G[0][2], gn14 = gm.G[0][3];  // :140-185
  double gn22 = gm.G[1][1], gn23 = gm.G[1][2], gn24 = gm.G[1][3], gn33 = gm.G[2][2], gn34 = gm.G[2][3],
         gn44 = gm.G[3][3];
  double alpha = gm.alpha, rdtx = in[1], rdty = in[2], rdtz = in[3];
  double utsq = gr2 / (alpha * alpha);
#pragma unroll
  for (int i = 0; i < 4; ++i) av[i] = in[i];
  double mix = gn13 * rdty + gn14 * rdtz;
  double disc = kzm_sqrt(((gn12 * gn12) * (rdtx * rdtx) + 2.0 * gn12 * rdtx * mix + mix * mix -
                          1.0 * gn11 * (gn22 * (rdtx * rdtx) + 2.0 * gn23 * rdtx * rdty + gn33 * (rdty * rdty) +
                                        2.0 * gn24 * rdtx * rdtz + 2.0 * gn34 * rdty * rdtz + gn44 * (rdtz * rdtz))) *
                         utsq * (gn11 + utsq) * ((gn11 + 4.0 * utsq) * (gn11 + 4.0 * utsq)));
  av[0] = (0.25 * (-4.0 * (gn12 * rdtx + gn13 * rdty + gn14 * rdtz) * utsq * (gn11 + utsq) + disc)) /
          (gn11 * utsq * (gn11 + utsq));
  double erf = (0.75 * disc) / (utsq * (gn11 + utsq) * (gn11 + 4.0 * utsq));
  double avc[4];
  raise4(av, gm, avc);
  double gr = kzm_sqrt(gr2);
#pragma unroll
  for (int i = 0; i < 4; ++i) ur[i] = 0;
  if (erf > 0.0) {
#pragma unroll
    for (int jj = 1; jj < 4; ++jj)
      ur[jj] = alpha * (avc[jj] + 1.0 / 3.0 * erf * gm.G[0][jj] * (4.0 * gr2 - 1.0)) / (4.0 / 3.0 * erf * gr);
  }
  *erf_o = erf;
}

// invert_rad.zig:189-261 u2pRad; returns ret, *corrected
KZD int u2p_rad(const double *uu, double *pp, const Geo &gm, const kz_rad_params &rp, int *corrected) {
  double av[4] = {uu[EE] / gm.gdet, uu[FX] / gm.gdet, uu[FY] / gm.gdet, uu[FZ] / gm.gdet}, avc[4];
  raise4(av, gm, avc);
  double gr2 = m1_gammarel2(gm, av);
  double erf = 3.0 * avc[0] * gm.alpha * gm.alpha / (4.0 * gr2 - 1.0);
  double gmax = rp.gammamaxrad;
  bool ok = gr2 >= 1.0 && erf > rp.eradfloor && gr2 <= gmax * gmax / GSL / GSL;
  double uc[4];
  *corrected = 0;
  if (ok) {
    double gr = kzm_sqrt(gr2);
#pragma unroll
    for (int ii = 0; ii < 4; ++ii)
      uc[ii] = gm.alpha * (avc[ii] + 1.0 / 3.0 * erf * gm.G[0][ii] * (4.0 * gr2 - 1.0)) / (4.0 / 3.0 * erf * gr);
  } else {
    const double one_eps = 1.0 + 10.0 * 2.220446049250313080847e-16;
    double sa[4], se, su[4], fa[4], fe, fu[4];
    m1_cold(gm, av, one_eps * one_eps, sa, &se, su);
    m1_cold(gm, av, gmax * gmax, fa, &fe, fu);
    if (kzm_fabs(sa[0] - av[0]) > kzm_fabs(fa[0] - av[0])) {
#pragma unroll
      for (int i = 0; i < 4; ++i) uc[i] = fu[i];
      gr2 = gmax * gmax;
      erf = fe;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) uc[i] = su[i];
      gr2 = one_eps * one_eps;
      erf = se;
    }
    *corrected = 1;
    if (!kzm_isfinite(erf) || !kzm_isfinite(gr2) || !kzm_isfinite(uc[1]) || !kzm_isfinite(uc[2]) ||
        !kzm_isfinite(uc[3]))
      return -1;
  }
  pp[EE] = erf;
  pp[FX] = uc[1];
  pp[FY] = uc[2];
  pp[FZ] = uc[3];
  return 0;
}

// invert_rad.zig:266-303 checkFloorsRad
KZD int check_floors_rad(double *pp, const Geo &gm, const kz_rad_params &rp) {
  int ret = 0;
  double ehat = -calc_ff_rtt(pp, gm);
  double eratio = pp[EE] / ehat;
  if (pp[EE] < rp.eradfloor) {
    pp[EE] = rp.eradfloor;
    ret = -1;
  }
  if (ehat < rp.eerhoratiomin * pp[RHO]) {
    pp[EE] = eratio * rp.eerhoratiomin * pp[RHO];
    ret = -1;
  }
  if (ehat > rp.eerhoratiomax * pp[RHO]) {
    pp[RHO] = 1.0 / rp.eerhoratiomax * ehat;
    ret = -1;
  }
  if (ehat < rp.eeuuratiomin * pp[UU]) {
    pp[EE] = eratio * rp.eeuuratiomin * pp[UU];
    ret = -1;
  }
  if (ehat > rp.eeuuratiomax * pp[UU]) {
    pp[UU] = 1.0 / rp.eeuuratiomax * ehat;
    ret = -1;
  }
  return ret;
}

// ---- implicit.zig --------------------------------------------------------------
KZD double my_sign(double x) { return x > 0.0 ? 1.0 : (x < 0.0 ? -1.0 : 1.0); }  // :167-172

KZD double abs_t(double x) { return kzm_fabs(x); }
KZD float abs_t(float x) { return __builtin_fabsf(x); }
// implicit.zig:176-224 invert4, on doubles (the reference) or on floats (the
// mixed-precision Newton's LU; same pivoting and elimination order)
template <class T>
KZD void invert4_t(const T a[4][4], T inv[4][4]) {
  T lu[4][4];
  int perm[4] = {0, 1, 2, 3};
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) lu[i][j] = a[i][j];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    int piv = k;
    T pmax = abs_t(lu[k][k]);
#pragma unroll
    for (int r = k + 1; r < 4; ++r)
      if (abs_t(lu[r][k]) > pmax) {
        pmax = abs_t(lu[r][k]);
        piv = r;
      }
    // row swap expressed as selects so the matrix stays in registers
#pragma unroll
    for (int r = k + 1; r < 4; ++r) {
      bool sw = piv == r;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        T tk = lu[k][j], tr = lu[r][j];
        lu[k][j] = sw ? tr : tk;
        lu[r][j] = sw ? tk : tr;
      }
      int pk = perm[k], pr = perm[r];
      perm[k] = sw ? pr : pk;
      perm[r] = sw ? pk : pr;
    }
#pragma unroll
    for (int r = k + 1; r < 4; ++r) {
      lu[r][k] /= lu[k][k];
#pragma unroll
      for (int cc = k + 1; cc < 4; ++cc) lu[r][cc] -= lu[r][k] * lu[k][cc];
    }
  }
#pragma unroll
  for (int col = 0; col < 4; ++col) {
    T y[4], x[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      y[r] = (perm[r] == col) ? T(1) : T(0);
#pragma unroll
      for (int cc = 0; cc < r; ++cc) y[r] -= lu[r][cc] * y[cc];
    }
#pragma unroll
    for (int r = 3; r >= 0; --r) {
      x[r] = y[r];
#pragma unroll
      for (int cc = r + 1; cc < 4; ++cc) x[r] -= lu[r][cc] * x[cc];
      x[r] /= lu[r][r];
    }
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) inv[rr][col] = x[rr];
  }
}
KZD void invert4(const double a[4][4], double inv[4][4]) { invert4_t<double>(a, inv); }

struct ImpCtx {
  const Geo *gm;
  double gam;
  const kz_rad_params *rp;
  const kz_opac_params *op;
  const kz_implicit_params *ip;
  double opdamp;
};

// implicit.zig:240-306 applyConstraints.  WP (the primitive block the
// Newton solves for) is a template parameter so that every state index is
// a compile-time constant and the 13-slot states stay in registers.
template <int WP, class Uu0>
KZDM int apply_constraints(double *pp, double *uu, const Uu0 &uu0, const ImpCtx &cx) {
  const Geo &gm = *cx.gm;
  double gdetu = gm.gdet, gi = 1.0 / gdetu;
  if (WP == WP_MHD) {
    double ucon[4], ucov[4];
    ucon_ucov(pp, gm, ucon, ucov);
    pp[RHO] = uu0[RHO] * gi / ucon[0];
    pp[ENTR] = s_from_u(pp[RHO], pp[UU], cx.gam);
    p2u_mhd(pp, uu, gm, cx.gam);
#pragma unroll
    for (int k = 0; k < 4; ++k) uu[EE + k] = uu0[EE + k] - (uu[UU + k] - uu0[UU + k]);
    int corr;
    int r = u2p_rad(uu, pp, gm, *cx.rp, &corr);
    if (corr) r = cx.ip->allow_rad_ceiling ? -1 : -2;
    return r;
  }
  p2u_rad(pp, uu, gm);
  uu[RHO] = uu0[RHO];
#pragma unroll
  for (int k = 0; k < 4; ++k) uu[UU + k] = uu0[UU + k] - (uu[EE + k] - uu0[EE + k]);
#pragma unroll
  for (int k = 0; k < 3; ++k) uu[B1 + k] = gdetu * pp[B1 + k];
  int etype = 0;
  int ret = u2p_solver_w(uu, pp, gm, &etype, cx.ip->allow_entr_in_4dprim != 0, cx.gam) < 0 ? -2 : 0;
  double ucon[4], ucov[4];
  ucon_ucov(pp, gm, ucon, ucov);
  pp[ENTR] = s_from_u(pp[RHO], pp[UU], cx.gam);
  uu[ENTR] = pp[ENTR] * gdetu * ucon[0];
  return ret;
}

// reference-state quantities the residual reads (implicit.zig:345-347,377,397)
struct State0 {
  double ehat, uint, sgas;
};
// the reference-state opacities lagOpac substitutes (implicit.zig:631-640)
struct LagOpac {
  double kappaes;
  Opac op;
};

// implicit.zig:337-427 residualG (scalar) on a filled state
template <int WP, bool ALL, class Uu0>
KZDM double residual(const double *uu, const double *pp, const RadState &st, const Uu0 &uu0, const State0 &s0,
                     double dt, const ImpCtx &cx, int we, int wf, double f[4]) {
  const Geo &gm = *cx.gm;
  double gdetu = gm.gdet;
  double dtau = dt / st.ucon[0];
  double giff0, gilab[4], gi[4];
  calc_gi<ALL>(st, *cx.op, cx.opdamp, &giff0, gilab);
  lower4(gilab, gm, gi);
  double err[4] = {0, 0, 0, 0};
  const double SMALLI = 1.0e-80;
  constexpr int base = (WP == WP_MHD) ? UU : EE;
#pragma unroll
  for (int k = 1; k < 4; ++k) {
    // MHD: uu - uu0 - dt*gdet*G;  RAD: uu - uu0 + dt*gdet*G
    f[k] = (WP == WP_MHD) ? uu[base + k] - uu0[base + k] - dt * gdetu * gi[k]
                          : uu[base + k] - uu0[base + k] + dt * gdetu * gi[k];
    const double e = kzm_fabs(f[k]) / (1.0e-20 * uu[base] + kzm_fabs(uu[base + k]) + kzm_fabs(uu0[base + k]) +
                                       kzm_fabs(dt * gdetu * gi[k]));
    err[k] = dm_sel(kzm_fabs(f[k]) > SMALLI, e, 0.0);
  }
  if (wf == WF_LAB) {
    if (WP == WP_RAD) {
      f[0] = uu[EE] - uu0[EE] + dt * gdetu * gi[0];
      const double e = kzm_fabs(f[0]) / (kzm_fabs(uu[EE]) + kzm_fabs(uu0[EE]) + kzm_fabs(dt * gdetu * gi[0]));
      err[0] = dm_sel(kzm_fabs(f[0]) > SMALLI, e, 0.0);
    } else {
      f[0] = uu[UU] - uu0[UU] - dt * gdetu * gi[0];
      const double e = kzm_fabs(f[0]) / (kzm_fabs(uu[UU]) + kzm_fabs(uu0[UU]) + kzm_fabs(dt * gdetu * gi[0]));
      err[0] = dm_sel(kzm_fabs(f[0]) > SMALLI, e, 0.0);
    }
  } else if (we == WE_ENERGY) {
    if (WP == WP_RAD) {
      f[0] = st.ehat - s0.ehat + dtau * giff0;
      err[0] = kzm_fabs(f[0]) / (kzm_fabs(st.ehat) + kzm_fabs(s0.ehat) + kzm_fabs(dtau * giff0));
    } else {
      f[0] = pp[UU] - s0.uint - dtau * giff0;
      err[0] = kzm_fabs(f[0]) / (kzm_fabs(pp[UU]) + kzm_fabs(s0.uint) + kzm_fabs(dtau * giff0));
    }
  } else {
    f[0] = st.tgas * (st.sgas - s0.sgas) - dtau * giff0;
    err[0] = kzm_fabs(f[0]) / (kzm_fabs(st.tgas * st.sgas) + kzm_fabs(st.tgas * s0.sgas) + kzm_fabs(dtau * giff0));
  }
  double e0 = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) e0 = err[k] > e0 ? err[k] : e0;
  return e0;
}

// The residual at pp: fill the radiation state (slim for the energy
// equations, full for entropy), apply lagOpac, evaluate.  The reference
// fills the state right after each applyConstraints and consumes it only
// here, with pp unchanged in between, so filling at the point of use gives
// the same values and keeps the state a temporary.
template <int WP, bool ALL, class Uu0>
KZDM double eval_residual_t(const double *uu, const double *pp, const LagOpac &lag, const Uu0 &uu0,
                            const State0 &s0, double dt, const ImpCtx &cx, int we, int wf, double f[4]) {
  RadState st;
  fill_radstate_t<ALL>(pp, *cx.gm, cx.gam, *cx.op, we == WE_ENTROPY, st);
  if (cx.ip->lag_opac) {
    st.kappaes = lag.kappaes;
    st.op = lag.op;
  }
  return residual<WP, ALL>(uu, pp, st, uu0, s0, dt, cx, we, wf, f);
}
template <int WP, class Uu0>
KZDM double eval_residual(const double *uu, const double *pp, const LagOpac &lag, const Uu0 &uu0,
                          const State0 &s0, double dt, const ImpCtx &cx, int we, int wf, double f[4]) {
  return all_channels(*cx.op) ? eval_residual_t<WP, true>(uu, pp, lag, uu0, s0, dt, cx, we, wf, f)
                              : eval_residual_t<WP, false>(uu, pp, lag, uu0, s0, dt, cx, we, wf, f);
}

// implicit.zig:431-467 f1dErr (energy equation, undamped opacities)
template <bool ALL>
KZDM double f1d_err_t(double xxx, const double *pp0, double dtau, const ImpCtx &cx, int wp, double totenergy,
                      double ratio) {
  const bool rad = wp == WP_RAD;
  const double xr = xxx * ratio;
  const double ehat = dm_sel(rad, xr, totenergy - xxx);
  const double ugas = dm_sel(rad, totenergy - xr, xxx);
  double pp[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) pp[i] = pp0[i];
  pp[UU] = ugas;
  pp[EE] = ehat / ratio;
  RadState st;
  fill_radstate_t<ALL>(pp, *cx.gm, cx.gam, *cx.op, false, st);
  double giff0, gilab[4];
  calc_gi<ALL>(st, *cx.op, cx.op->opdamp, &giff0, gilab);
  return dm_sel(rad, ehat - pp0[EE] / ratio + dtau * giff0, ugas - pp0[UU] - dtau * giff0);
}
KZDM double f1d_err(double xxx, const double *pp0, double dtau, const ImpCtx &cx, int wp, double totenergy,
                    double ratio) {
  return all_channels(*cx.op) ? f1d_err_t<true>(xxx, pp0, dtau, cx, wp, totenergy, ratio)
                              : f1d_err_t<false>(xxx, pp0, dtau, cx, wp, totenergy, ratio);
}

// implicit.zig:473-574 solve1dPrim: bisection warm start on the fluid-frame
// energy equation; reads Ehat, u^t and T_gas of the reference state.  The
// reference evaluates the equation in four places (both ends of the bracket,
// its growth, the midpoints); here they are one loop with one evaluation, so
// that its code stands once and the lanes of a wave share it wherever each of
// them is.
KZDM void solve_1d_prim(const double *pp00, double st_ehat, double st_ut, double st_tgas, double dt, const ImpCtx &cx,
                        double *pp0out) {
#pragma unroll
  for (int i = 0; i < NV; ++i) pp0out[i] = pp00[i];
  double ehat = st_ehat;
  double dtau = dt / st_ut;
  double tot = ehat + pp00[UU];
  int wp = (ehat < 1.0e-3 * pp00[UU]) ? WP_RAD : WP_MHD;
  double tgas = st_tgas;
  double ratio = ehat / pp00[EE];
  const double fac = 3.0, fac1 = fac + 1.0;
  double pu = pp00[UU], pe = pp00[EE];
  if (tgas > 1.0e14) {
    pu = pp00[UU] * 1.0e14 / tgas;
    pe = (tot - pu) / ratio;
  }
  double xlo, xhi;
  if (wp == WP_MHD) {
    xlo = pu / 1.05;
    xhi = kzm_fmin(pu * 1.05, (pu + fac * tot) / fac1);
  } else {
    xlo = pe / 1.05;
    xhi = kzm_fmin(pe * 1.05, (pe + fac * tot / ratio) / fac1);
  }
  enum { LOW, HIGH, GROW_LOW, GROW_HIGH, MID };
  int at = LOW, iter = 0;
  double elo = 0, ehi = 0, x = xlo;
  for (;;) {
    const double e = f1d_err(x, pp00, dtau, cx, wp, tot, ratio);
    if (at == LOW) {
      elo = e;
      x = xhi;
      at = HIGH;
      continue;
    }
    if (at == MID) {
      if (e * elo > 0.0) {
        xlo = x;
        elo = e;
      } else {
        xhi = x;
        ehi = e;
      }
      if (x != x || e != e) return;
      if (!(kzm_fabs((xhi - xlo) / x) > 1.0e-3)) break;
    } else {
      if (at == GROW_LOW) elo = e;
      else ehi = e;
      if (at != HIGH && (elo != elo || ehi != ehi)) iter = 50;
      if (iter >= 50) return;
      if (elo * ehi > 0.0) {
        iter += 1;
        if (elo > 0.0) {
          xhi = xlo;
          ehi = elo;
          xlo /= fac;
          x = xlo;
          at = GROW_LOW;
        } else {
          xlo = xhi;
          elo = ehi;
          if (wp == WP_RAD) xhi = kzm_fmin(xhi * fac, (xhi + fac * tot / ratio) / fac1);
          else xhi = kzm_fmin(xhi * fac, (xhi + fac * tot) / fac1);
          x = xhi;
          at = GROW_HIGH;
        }
        continue;
      }
    }
    at = MID;
    x = 0.5 * (xlo + xhi);
  }
  if (wp == WP_RAD) {
    pp0out[EE] = x;
    pp0out[UU] = tot - x * ratio;
  } else {
    pp0out[UU] = x;
    pp0out[EE] = (tot - x) / ratio;
  }
}

// Element j (0..3, not a compile-time constant) of a 4-block, by selects,
// so that register-resident arrays are never indexed dynamically.
// (the values are taken before the choice: a choice between addresses would
// keep the array, and the whole structure around it, in scratch memory)
KZDM double get4(const double *a, int j) {
  const double a0 = a[0], a1 = a[1], a2 = a[2], a3 = a[3];
  return j == 0 ? a0 : (j == 1 ? a1 : (j == 2 ? a2 : a3));
}
KZDM void set4(double *a, int j, double v) {
#pragma unroll
  for (int k = 0; k < 4; ++k) a[k] = j == k ? v : a[k];
}
KZDM double gdiag(const Geo &gm, int j) {
  const double g1 = gm.g[1][1], g2 = gm.g[2][2], g3 = gm.g[3][3];
  return j == 1 ? g1 : (j == 2 ? g2 : g3);
}

// implicit.zig:586-591 fdDel on the block b = ppp + sh
KZDM double fd_del(int j, double sign, const double *b, double eps, const Geo &gm) {
  if (j == 0) return sign * eps * b[0];
  double bj = get4(b, j);
  double veleps = eps * my_sign(bj) * kzm_fmax(1.0e-8 / kzm_sqrt(gdiag(gm, j)), kzm_fabs(bj));
  return bj >= 0.0 ? sign * veleps : -sign * veleps;
}

// implicit.zig:642-922 solve4dPrimCore (scalar Jacobian) as a start and a
// pass that evaluates one trial state: newton_pass applies the constraints to
// n.pp, judges them by what the state was tried for (n.at: the base of an
// iteration, one column of the Jacobian, or the update), takes the residual
// there and sets up the next trial state.  It returns 0 to go on, 1 when the
// reference's loop ends solved (n.pp and n.iter hold the result) and -1 when
// it ends failed; the sequence of trial states is the reference's.
//
// One pass per trial state, so that the constraints and the residual stand in
// the code once each.  Written out per use (three and two copies per
// primitive block) the first rung's code was 293 KB (142 KB now) against the
// 64 KB of instruction cache that two CUs share, with 400 B of scratch per
// lane (none now).  It also lets the lanes of a wave stand at different trial
// states.  First rung at 384x360, with kz_dev_math.h: 262 -> 194 us.
enum { AT_BASE = 0, AT_COL, AT_UPDATE };
// What a Newton keeps for its whole length but reads once or twice per pass
// lies in LDS, 40 doubles per lane (20 KB per wave, eight waves fill a CU's
// 160 KB): the incoming conserved state, the reference-state scalars, the
// residual at the base and the Jacobian.  With them in registers a lane
// needed 350 to 450, one wave per SIMD, and the part past 256 was moved to
// and fro between the two halves of the register file.
enum { NL_JAC = 0, NL_F1 = 16, NL_UU0 = 20, NL_S0 = 33, NL_LAG = 36, NL_N = 40 };
struct NewtonLds {
  double v[NL_N][64];
};
// n values of the wave's LDS block as one lane's array
struct LaneVec {
  double *p;
  __device__ __forceinline__ double operator[](int i) const { return p[i * 64]; }
  __device__ __forceinline__ void put(int i, double x) const { p[i * 64] = x; }
};
KZDM LaneVec lane_vec(NewtonLds &l, int first) { return LaneVec{&l.v[first][threadIdx.x & 63]}; }
struct NewtonState {
  double uu[NV], pp[NV];
  double b[4];        // the iteration's primitive block
  double rho0, en0;   // its density, and the energy density of the other block
  double errbase, del, xiapp;
  int iter, at, j;
  bool second;        // the column's second sign
};
KZDM void newton_start(NewtonState &n, const double *uu00, const double *pp0in) {
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    n.uu[i] = uu00[i];
    n.pp[i] = pp0in[i];
  }
  n.iter = 0;
  n.at = AT_BASE;
}
// puts a cell's incoming state and reference scalars into its lane's LDS
KZDM void newton_keep(NewtonLds &l, const double *uu00, const State0 &s0, const LagOpac &lag) {
  const LaneVec u = lane_vec(l, NL_UU0), s = lane_vec(l, NL_S0), o = lane_vec(l, NL_LAG);
#pragma unroll
  for (int i = 0; i < NV; ++i) u.put(i, uu00[i]);
  s.put(0, s0.ehat);
  s.put(1, s0.uint);
  s.put(2, s0.sgas);
  o.put(0, lag.kappaes);
  o.put(1, lag.op.gas_abs);
  o.put(2, lag.op.rad_abs);
  o.put(3, lag.op.rad_ross);
}
// the update's trial state ppp - xiapp * (inverse) * f1
KZDM void newton_update(NewtonState &n, NewtonLds &l, double *blk) {
  const LaneVec jac = lane_vec(l, NL_JAC), f1 = lane_vec(l, NL_F1);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    double x = n.b[i];
#pragma unroll
    for (int j = 0; j < 4; ++j) x -= n.xiapp * jac[i * 4 + j] * f1[j];
    blk[i] = x;
  }
}
template <int WP>
KZDM int newton_pass(NewtonState &n, NewtonLds &l, double dt, const ImpCtx &cx, int we, int wf) {
  const kz_implicit_params &ip = *cx.ip;
  const Geo &gm = *cx.gm;
  double *uu = n.uu, *pp = n.pp;
  constexpr int sh = (WP == WP_MHD) ? UU : EE;
  constexpr int other = (WP == WP_MHD) ? EE : UU;
  double *blk = pp + sh;
  const LaneVec uu0 = lane_vec(l, NL_UU0), jac = lane_vec(l, NL_JAC), f1 = lane_vec(l, NL_F1);
  const int fret = apply_constraints<WP>(pp, uu, uu0, cx);
  if (n.at == AT_UPDATE) {
    bool ok = false;
    double edenmin = n.b[0] / ip.max_en_change_down;
    double edenmax = n.b[0] * ip.max_en_change_up;
    if (blk[0] > edenmin && blk[0] < edenmax && fret >= -1) ok = true;
    double tgo = t_from_urho(*cx.op, WP == WP_MHD ? n.b[0] : n.en0, n.rho0, cx.gam);
    double tgn = t_from_urho(*cx.op, pp[UU], pp[RHO], cx.gam);
    if (ok && (tgn > tgo * ip.max_tgas_change || tgn < tgo / ip.max_tgas_change)) ok = false;
    double trn = lte_t_from_e(*cx.op, pp[EE]);
    double tro = lte_t_from_e(*cx.op, WP == WP_MHD ? n.en0 : n.b[0]);
    if (ok && (trn > tro * ip.max_trad_change || trn < tro / ip.max_trad_change)) ok = false;
    if (!ok) {
      if (blk[0] <= 0.0) {
        n.xiapp *= n.b[0] / (n.b[0] + kzm_fabs(blk[0]));
        n.xiapp *= 1.0e-1;
      } else {
        n.xiapp /= ip.damping_factor;
      }
      if (n.xiapp < ip.max_damping) return -1;
      newton_update(n, l, blk);
      return 0;
    }
    double f3[4];
    f3[0] = kzm_fabs((blk[0] - n.b[0]) / n.b[0]);
#pragma unroll
    for (int i = 1; i < 4; ++i) f3[i] = kzm_fabs((blk[i] - n.b[i]) / kzm_fmax(ip.eps, kzm_fabs(n.b[i])));
    double cr = (we == WE_ENTROPY) ? ip.convrelentr : ip.convrel;
    double cre = (we == WE_ENTROPY) ? ip.convrelentrerr : ip.convrelerr;
    bool cc = true;
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
      if (f3[ib] > cr) cc = false;
    if (cc || n.errbase <= cre) return n.iter > ip.maxiter ? -1 : 1;
    if (n.iter > ip.maxiter) return -1;
    n.at = AT_BASE;
  } else if (fret < -1) {
    if (n.at == AT_BASE || n.second) return -1;
    n.second = true;
    set4(blk, n.j, get4(n.b, n.j));
    n.del = fd_del(n.j, 1.0, n.b, ip.eps, gm);
    set4(blk, n.j, get4(n.b, n.j) + n.del);
    return 0;
  }
  double f[4], err;
  {
    asm volatile("" ::: "memory");  // read the LDS again rather than keep it through the constraints
    const LaneVec s = lane_vec(l, NL_S0), o = lane_vec(l, NL_LAG);
    const State0 s0{s[0], s[1], s[2]};
    LagOpac lag;
    lag.kappaes = o[0];
    lag.op = Opac{o[1], o[2], o[3]};
    err = eval_residual<WP>(uu, pp, lag, uu0, s0, dt, cx, we, wf, f);
  }
  if (n.at == AT_BASE) {
    n.iter += 1;
    const double conv = (we == WE_ENTROPY) ? ip.entrconv : ip.conv;
    if (err < conv) return n.iter > ip.maxiter ? -1 : 1;
    n.errbase = err;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      n.b[i] = blk[i];
      f1.put(i, f[i]);
    }
    n.rho0 = pp[RHO];
    n.en0 = pp[other];
    n.at = AT_COL;
    n.j = 0;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) jac.put(i * 4 + n.j, (f[i] - f1[i]) / n.del);
    set4(blk, n.j, get4(n.b, n.j));
    n.j += 1;
  }
  if (n.j < 4) {
    n.second = false;
    n.del = fd_del(n.j, -1.0, n.b, ip.eps, gm);
    set4(blk, n.j, get4(n.b, n.j) + n.del);
    return 0;
  }
  double sv[4] = {blk[0], 1.0, 1.0, 1.0}, isv[4];
  if (ip.scale_jacobian) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (sv[j] == 0.0) sv[j] = 1.0;
      isv[j] = 1.0 / sv[j];
    }
  }
  double ij[4][4], jm[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) jm[i][j] = jac[i * 4 + j];
  if (ip.jacobian_fp32) {
    // mixed precision: FP64 quotients rounded to FP32, scaled and
    // factored in FP32, the inverse applied in FP64
    float jf[4][4], ijf[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) jf[i][j] = (float)jm[i][j];
    if (ip.scale_jacobian) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (i != j) jf[i][j] = jf[i][j] * ((float)sv[j] * (float)isv[i]);
    }
    invert4_t<float>(jf, ijf);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) ij[i][j] = (double)ijf[i][j];
  } else {
    if (ip.scale_jacobian) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (i != j) jm[i][j] = jm[i][j] * (sv[j] * isv[i]);
    }
    invert4(jm, ij);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) jac.put(i * 4 + j, ip.scale_jacobian ? ij[i][j] * sv[i] * isv[j] : ij[i][j]);
  n.xiapp = 1.0;
  n.at = AT_UPDATE;
  newton_update(n, l, blk);
  return 0;
}
template <int WP>
KZDM bool solve_4d_prim_core(NewtonLds &l, const double *uu00, const LagOpac &lag, const State0 &s0,
                             const double *pp0in, double dt, const ImpCtx &cx, int we, int wf, double *pp_out,
                             int *iters_out) {
  NewtonState n;
  newton_keep(l, uu00, s0, lag);
  newton_start(n, uu00, pp0in);
  int r;
  do {
    r = newton_pass<WP>(n, l, dt, cx, we, wf);
  } while (r == 0);
  if (r < 0) return false;
#pragma unroll
  for (int i = 0; i < NV; ++i) pp_out[i] = n.pp[i];
  *iters_out = n.iter;
  return true;
}

// implicit.zig:927-1004 solveImplicitLab; returns kz_implicit_result
KZD kz_implicit_result solve_implicit_lab(NewtonLds &l, double *uu, double *pp, const Geo &gm, double dt, double gam,
                                          const kz_rad_params &rp, const kz_opac_params &op,
                                          const kz_implicit_params &ip) {
  kz_implicit_result fail = {0, -1, 0, WP_RAD, WE_ENERGY, WF_LAB};
  ImpCtx cx{&gm, gam, &rp, &op, &ip, 1.0};
  double pp00[NV], uu00[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) pp00[i] = pp[i];
  p2u(pp00, uu00, gm, gam);
  double ehat = -calc_ff_rtt(pp00, gm);
  State0 s0;
  LagOpac lag;
  double pp0[NV];
  {
    RadState st00;
    fill_radstate(pp00, gm, gam, op, true, st00);
    s0 = State0{st00.ehat, st00.uint, st00.sgas};
    lag.kappaes = st00.kappaes;
    lag.op = st00.op;
    if (ip.start_with_bisect) {
      solve_1d_prim(pp00, st00.ehat, st00.ucon[0], st00.tgas, dt, cx, pp0);
    } else {
#pragma unroll
      for (int i = 0; i < NV; ++i) pp0[i] = pp00[i];
    }
  }
  const int sw = (ehat < ip.threshold * pp00[UU]) ? WP_RAD : WP_MHD;
  const int ot = (sw == WP_RAD) ? WP_MHD : WP_RAD;
  for (int level = 0; level <= ip.opdamp_maxlevels; ++level) {
    double od = 1.0;
    for (int i = 0; i < level; ++i) od /= ip.opdamp_factor;
    cx.opdamp = od;
    for (int ir = 0; ir < 6; ++ir) {
      int wp = (ir == 0 || ir == 1 || ir == 4) ? sw : ot;
      int we = (ir >= 4) ? WE_ENTROPY : WE_ENERGY;
      int wf = (ir == 0 || ir == 2) ? WF_LAB : WF_FF;
      double ppw[NV];
      int iters = 0;
      bool ok = (wp == WP_MHD) ? solve_4d_prim_core<WP_MHD>(l, uu00, lag, s0, pp0, dt, cx, we, wf, ppw, &iters)
                               : solve_4d_prim_core<WP_RAD>(l, uu00, lag, s0, pp0, dt, cx, we, wf, ppw, &iters);
      if (ok) {
#pragma unroll
        for (int i = 0; i < NV; ++i) pp[i] = ppw[i];
        p2u(ppw, uu, gm, gam);
        kz_implicit_result r = {1, ir, iters, wp, we, wf};
        return r;
      }
    }
  }
  return fail;
}

}  // namespace kzd
