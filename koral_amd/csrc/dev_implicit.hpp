// Device implicit gas-radiation four-force solve: residual
// f_implicit_lab_4dprim (rad.c:110-351), damped Newton
// solve_implicit_lab_4dprim (rad.c:376-1218) by one lane or by one wave per
// cell, and the six-attempt fallback chain of solve_implicit_lab
// (rad.c:1225-1570).
#pragma once
#include "dev_cell.hpp"

namespace kd {

// inverse_44matrix (misc.c:502-605): adjugate inverse, fails on NaN entries
KD_INL int inverse44(const double *a, double *ia)
{
  double s0 = a[0] * a[5] - a[4] * a[1];
  double s1 = a[0] * a[6] - a[4] * a[2];
  double s2 = a[0] * a[7] - a[4] * a[3];
  double s3 = a[1] * a[6] - a[5] * a[2];
  double s4 = a[1] * a[7] - a[5] * a[3];
  double s5 = a[2] * a[7] - a[6] * a[3];
  double c5 = a[10] * a[15] - a[14] * a[11];
  double c4 = a[9] * a[15] - a[13] * a[11];
  double c3 = a[9] * a[14] - a[13] * a[10];
  double c2 = a[8] * a[15] - a[12] * a[11];
  double c1 = a[8] * a[14] - a[12] * a[10];
  double c0 = a[8] * a[13] - a[12] * a[9];
  double det = s0 * c5 - s1 * c4 + s2 * c3 + s3 * c2 - s4 * c1 + s5 * c0;
  double id = 1 / det;
  if (isnan(id)) return -1;
  double b[16];
  b[0] = (a[5] * c5 - a[6] * c4 + a[7] * c3);
  b[1] = (-a[1] * c5 + a[2] * c4 - a[3] * c3);
  b[2] = (a[13] * s5 - a[14] * s4 + a[15] * s3);
  b[3] = (-a[9] * s5 + a[10] * s4 - a[11] * s3);
  b[4] = (-a[4] * c5 + a[6] * c2 - a[7] * c1);
  b[5] = (a[0] * c5 - a[2] * c2 + a[3] * c1);
  b[6] = (-a[12] * s5 + a[14] * s2 - a[15] * s1);
  b[7] = (a[8] * s5 - a[10] * s2 + a[11] * s1);
  b[8] = (a[4] * c4 - a[5] * c2 + a[7] * c0);
  b[9] = (-a[0] * c4 + a[1] * c2 - a[3] * c0);
  b[10] = (a[12] * s4 - a[13] * s2 + a[15] * s0);
  b[11] = (-a[8] * s4 + a[9] * s2 - a[11] * s0);
  b[12] = (-a[4] * c3 + a[5] * c1 - a[6] * c0);
  b[13] = (a[0] * c3 - a[1] * c1 + a[2] * c0);
  b[14] = (-a[12] * s3 + a[13] * s1 - a[14] * s0);
  b[15] = (a[8] * s3 - a[9] * s1 + a[10] * s0);
  int bad = 0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    ia[i] = b[i] * id;
    bad |= isnan(ia[i]) ? 1 : 0;
  }
  return bad ? -1 : 0;
}

enum { IMP_FAIL = -1, IMP_CONT = 0, IMP_OK = 1 };

// One evaluation of an attempt's state machine: the residual (rad.c:110-351)
// and the completion of a state (rad.c:880-950) as one function, so a solver
// that runs it in a loop holds a single inlined copy.  mode EVAL: the residual
// f and its error at the state pp (pp is a work copy); returns < 0 where the
// residual fails.  TRIAL and FINAL: pp completed as a damped trial / as the
// converged state, the inversion's return value in cret; pp[5] is left alone (imp_finish sets it).  On the gas primitives with the
// energy equation the residual at a completed state is the next iteration's:
// both complete it with the same operations, so TRIAL evaluates it too
// (imp_trial_residual).  pp0_u and Ehat0 = -ff_Rtt, of the old state, enter
// the fluid-frame equation.  Template kind values < 0: the attempt's kind at
// run time (k), the same in all lanes that run together.  WG > 0: lanes of a
// group that share the W inversion's trials (the wave-per-cell solve, whose
// trials skip the residual: its next iterate is evaluated beside the columns).
enum { IMP_EVAL = 0, IMP_TRIAL = 1, IMP_FINAL = 2 };
struct ImpKind {
  int wp, we, wf;
};
KD_INL bool imp_trial_residual(int wp, int we) { return wp == P_MHD && we == ENERGYEQ; }
template <int MAG, int WG, int WP, int WE, int WF, class UT, class GT>
KD_INL int imp_eval(const koral_params &P, const ImpKind &k, int mode, double *pp, const UT &uu0, double pp0_u,
                    double Ehat0, double dt, const GT &g, double *f, double &err0, int &cret)
{
  constexpr int RAD = 1;
  constexpr int NV = Lay<MAG, RAD>::NV;
  constexpr int EE = Lay<MAG, RAD>::EE;
  const int whichprim = WP >= 0 ? WP : k.wp, whicheq = WE >= 0 ? WE : k.we, whichframe = WF >= 0 ? WF : k.wf;
  double uu[NV];
  int corr = 0, ret;
  // uu0 and g live in LDS: the fences keep the compiler from holding them in
  // registers from one part of the evaluation to the next
  compiler_fence();
  double gdetu = g.gdet;
  if (whichprim == P_MHD) {
    double ucon[4];
    relr_to_4vel(pp[2], pp[3], pp[4], ucon, nullptr, g);
    pp[0] = (uu0[0]) / gdetu / ucon[0];
  }
  p2u_mhd<MAG, RAD>(P, pp, uu, g);
  compiler_fence();
  // the gas primitives' energy equation reads none of the radiation's
  // conserved variables here
  if (whichprim == P_RAD || whicheq != ENERGYEQ) {
    p2u_rad<MAG, RAD>(pp, uu, g);
    compiler_fence();
    uu[5] = uu0[5] - (uu[EE] - uu0[EE]);
  }
  if (whichprim == P_RAD) {
    uu[0] = uu0[0];
    uu[1] = uu0[1] - (uu[EE] - uu0[EE]);
    uu[2] = uu0[2] - (uu[EE + 1] - uu0[EE + 1]);
    uu[3] = uu0[3] - (uu[EE + 2] - uu0[EE + 2]);
    uu[4] = uu0[4] - (uu[EE + 3] - uu0[EE + 3]);
    const int rt = u2p_solver_W<MAG, RAD, (WG > 0), (WG > 0 ? WG : WAVE_GROUP)>(P, uu, pp, g, 0, 0., nullptr, 0, false);
    ret = cret = (rt < 0) ? -2 : 0;
  } else {
    uu[EE] = uu0[EE] - (uu[1] - uu0[1]);
    uu[EE + 1] = uu0[EE + 1] - (uu[2] - uu0[2]);
    uu[EE + 2] = uu0[EE + 2] - (uu[3] - uu0[3]);
    uu[EE + 3] = uu0[EE + 3] - (uu[4] - uu0[4]);
    ret = u2p_rad<MAG, RAD>(P, uu, pp, g, corr);
    cret = corr > 0 ? (mode == IMP_FINAL ? -2 : -1) : ret;
  }
  // (a wave evaluates the next iterate beside its columns anyway)
  if (mode == IMP_FINAL || (mode == IMP_TRIAL && (WG > 0 || !imp_trial_residual(whichprim, whicheq)))) return 0;
  if (ret < -1) return -1;

  compiler_fence();
  double Gi[4], Gff = 0., Rtt = 0., ut = 1.;
  calc_Gi_ff<MAG, RAD, (WF != LAB)>(P, pp, g, Gi, whichframe == FF, Gff, Rtt, ut);
  compiler_fence();
  lower(Gi, Gi, g);
  double err[4];
#pragma unroll
  for (int i = 1; i < 4; i++) {
    const double u = whichprim == P_MHD ? uu[1 + i] : uu[EE + i], u0 = whichprim == P_MHD ? uu0[1 + i] : uu0[EE + i];
    if (whichprim == P_MHD)
      f[i] = u - u0 - dt * gdetu * Gi[i];
    else
      f[i] = u - u0 + dt * gdetu * Gi[i];
    err[i] = (fabs(f[i]) > SMALL) ? fabs(f[i]) / (fabs(u) + fabs(u0) + fabs(dt * gdetu * Gi[i])) : 0.;
  }
  if (whichframe == LAB) {
    const double u = whicheq != ENERGYEQ ? uu[5] : (whichprim == P_MHD ? uu[1] : uu[EE]);
    const double u0 = whicheq != ENERGYEQ ? uu0[5] : (whichprim == P_MHD ? uu0[1] : uu0[EE]);
    if (whichprim == P_RAD)
      f[0] = u - u0 + dt * gdetu * Gi[0];
    else
      f[0] = u - u0 - dt * gdetu * Gi[0];
    err[0] = (fabs(f[0]) > SMALL) ? fabs(f[0]) / (fabs(u) + fabs(u0) + fabs(dt * gdetu * Gi[0])) : 0.;
  } else {
    // the energy equation in the fluid frame (the chain asks for no other)
    const double Ehat = -Rtt;
    const double dtau = dt / ut;
    if (whichprim == P_RAD) {
      f[0] = Ehat - Ehat0 + dtau * Gff;
      err[0] = fabs(f[0]) / (fabs(Ehat) + fabs(Ehat0) + fabs(dtau * Gff));
    } else {
      f[0] = pp[1] - pp0_u - dtau * Gff;
      err[0] = fabs(f[0]) / (fabs(pp[1]) + fabs(pp0_u) + fabs(dtau * Gff));
    }
  }
  if (!isfinite(f[0]) || !isfinite(f[1]) || !isfinite(f[2]) || !isfinite(f[3])) return -1;
  err0 = mx(mx(err[0], err[1]), mx(err[2], err[3]));
  return corr != 0 ? 1 : 0;
}

// The entropy and the conserved variables of a solved cell, which the solvers
// leave to one pass over all cells at the end (the lanes of the persistent
// passes finish at different times, and three powers and a logarithm for one
// lane would hold its whole wave)
template <int MAG>
KD_INL void imp_finish(const koral_params &P, double *pp, double *uu, const Geom &g)
{
  pp[5] = Sfromu(P, pp[0], pp[1]);
  p2u<MAG, 1>(P, pp, uu, g);
}

// Step of variable j of the iterate for the Jacobian's one-sided difference
KD_INL double imp_delta(double EPS, int j, double sign, double xj, double gjj)
{
  if (j <= 0) return sign * EPS * xj;
  const double veleps = EPS * sgn(xj) * mx(1.e-6 / sqrt(gjj), fabs(xj));
  return (xj >= 0.) ? sign * veleps : -sign * veleps;
}

// Newton update of the iterated variables with damping xiapp
KD_INL void imp_update(const double *x0, const double *iJ, const double *f1, double xiapp, double *x)
{
#pragma unroll
  for (int i = 0; i < 4; i++) {
    x[i] = x0[i];
#pragma unroll
    for (int j = 0; j < 4; j++) x[i] -= xiapp * iJ[i * 4 + j] * f1[j];
  }
}

// Whether a damped trial is accepted; otherwise the next damping factor
KD_INL bool imp_accept(const koral_params &P, double x00, double xnew, int u2pret, double &xiapp)
{
  const double edenmin = x00 / P.maxenchangedown, edenmax = x00 * P.maxenchangeup;
  if (xnew > edenmin && xnew < edenmax && u2pret >= -1) return true;
  if (xnew <= 0.) {
    xiapp *= x00 / (x00 + fabs(xnew));
    xiapp *= 1.e-1;
  } else {
    xiapp /= P.dampingfactor;
  }
  return false;
}

// The relative-change convergence of an accepted step (rad.c: CONVREL)
KD_INL bool imp_conv_rel(const koral_params &P, int whicheq, double EPS, const double *x0, const double *x,
                         double errbase, double global_time)
{
  if (!(P.convrel_enabled && global_time < 100.)) return false;
  double f3[4];
  f3[0] = fabs((x[0] - x0[0]) / x0[0]);
#pragma unroll
  for (int i = 1; i < 4; i++) {
    f3[i] = x[i] - x0[i];
    f3[i] = fabs(f3[i] / mx(EPS, fabs(x0[i])));
  }
  const double CR = (whicheq == ENTROPYEQ) ? P.radimpconvrelentr : P.radimpconvrel;
  const double CRE = (whicheq == ENTROPYEQ) ? P.radimpconvrelentrerr : P.radimpconvrelerr;
  return f3[0] < CR && f3[1] < CR && f3[2] < CR && f3[3] < CR && errbase < CRE;
}

// One lane's attempt as a state machine that makes one evaluation per trip:
// the residual at the iterate (stage 0), the four Jacobian columns (1..4), a
// damped trial (5) and the completion of a converged iterate (6).  The lanes
// of a wave hold cells at different points of their iterations, so in
// nested loops over iterations, columns and trials a wave waits for the lane
// with the most damped trials (up to eleven) and repeated columns; here every lane advances
// by one evaluation per trip whatever the others do, and the kernel holds one
// inlined copy of the evaluation instead of four.  The operations on a cell
// are those of the nested loops, in the same order.
struct ImpLane {
  int stage, iter;
  double sign, xp, xj, xiapp, errbase;
  double x0[4], f1[4];
};
template <int WP, int EE>
KD_INL void imp_lane_start(ImpLane &s, const double *pp)
{
  constexpr int sh = (WP == P_MHD) ? 1 : EE;
  s.stage = 0;
  s.iter = 1;
  s.sign = -1.;
#pragma unroll
  for (int i = 0; i < 4; i++) s.x0[i] = pp[sh + i];
}
// J(i): the lane's 16 doubles of the Jacobian, then of its inverse
template <int MAG, int WP, int WE, int WF, class UT, class GT, class JF>
KD_INL int imp_lane_trip(const koral_params &P, ImpLane &s, double *pp, const UT &uu0, double pp0_u, double Ehat0,
                         double dt, const GT &g, double global_time, int maxiter, JF J)
{
  constexpr int NV = Lay<MAG, 1>::NV;
  constexpr int EE = Lay<MAG, 1>::EE;
  constexpr int sh = (WP == P_MHD) ? 1 : EE;
  const double EPS = P.radimpeps;
  const double CONV = (WE == ENTROPYEQ) ? P.radimpentrconv : P.radimpconv;
  const int st = s.stage, col = st - 1;
  const int mode = st < 5 ? IMP_EVAL : (st == 5 ? IMP_TRIAL : IMP_FINAL);
  double ppt[NV], f[4] = {0., 0., 0., 0.}, err = 0.;
#pragma unroll
  for (int i = 0; i < NV; i++) ppt[i] = pp[i];
  if (st >= 1 && st <= 4) {
    s.xj = s.x0[0];
    double gjj = g.g[1][1];
#pragma unroll
    for (int i = 1; i < 4; i++) {
      s.xj = (col == i) ? s.x0[i] : s.xj;
      gjj = (col == i) ? g.g[i][i] : gjj;
    }
    s.xp = s.xj + imp_delta(EPS, col, s.sign, s.xj, gjj);
#pragma unroll
    for (int i = 0; i < 4; i++) ppt[sh + i] = (col == i) ? s.xp : ppt[sh + i];
  }
  int cret = 0;
  const int eret = imp_eval<MAG, 0, WP, WE, WF>(P, ImpKind{WP, WE, WF}, mode, ppt, uu0, pp0_u, Ehat0, dt, g, f, err, cret);
  if (st >= 5)
#pragma unroll
    for (int i = 0; i < NV; i++) pp[i] = ppt[i];
  bool base = st == 0, update = false;
  if (st == 6) return cret < -1 ? IMP_FAIL : IMP_OK;
  if (st == 5) {
    if (imp_accept(P, s.x0[0], pp[sh], cret, s.xiapp)) {
      const bool conv = imp_conv_rel(P, WE, EPS, s.x0, pp + sh, s.errbase, global_time);
      if (s.iter > maxiter) return IMP_FAIL;
      if (conv) {
        s.stage = 6;
      } else {
        s.iter++;
        s.stage = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) s.x0[i] = pp[sh + i];
        base = imp_trial_residual(WP, WE);
      }
    } else {
      // a NaN factor ends the attempt too
      if (!(s.xiapp >= P.maxradimpdamping)) return IMP_FAIL;
      update = true;
    }
  }
  if (base) {
    if (eret < 0) return IMP_FAIL;
    s.errbase = err;
#pragma unroll
    for (int i = 0; i < 4; i++) s.f1[i] = f[i];
    s.sign = -1.;
    s.stage = 1;
    if (!(err >= CONV)) {
      if (s.iter > maxiter) return IMP_FAIL;
      s.stage = 6;
    }
  } else if (st >= 1 && st <= 4) {
    if (eret < 0) {
      // a column that fails on one side is taken on the other
      if (s.sign > 0.) return IMP_FAIL;
      s.sign = 1.;
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++) J(4 * i + col) = (f[i] - s.f1[i]) / (s.xp - s.xj);
      s.sign = -1.;
      s.stage = st + 1;
      if (st == 4) {
        double a[16], b[16];
#pragma unroll
        for (int i = 0; i < 16; i++) a[i] = J(i);
        if (inverse44(a, b) < 0) return IMP_FAIL;
#pragma unroll
        for (int i = 0; i < 16; i++) J(i) = b[i];
        s.xiapp = 1.;
        update = true;
      }
    }
  }
  if (update) {
    double iJ[16], x[4];
#pragma unroll
    for (int i = 0; i < 16; i++) iJ[i] = J(i);
    imp_update(s.x0, iJ, s.f1, s.xiapp, x);
#pragma unroll
    for (int i = 0; i < 4; i++) pp[sh + i] = x[i];
  }
  return IMP_CONT;
}

#if KD_WAVE_SOLVER
// One attempt of a cell by a whole wave (solve_implicit_lab_4dprim from the
// iterate pp, every argument the same in all lanes): the arithmetic and the
// outcome of the one-lane attempt, bit for bit.  The wave is eight groups
// of eight lanes.  Group 0 evaluates the residual at the iterate while groups
// 1..4 evaluate the four Jacobian columns (groups 5..7 repeat the iterate),
// so an iteration costs one residual and one trial in sequence instead of
// five and one, and within a group the W inversion of the radiation
// primitives tries eight bumps or step halvings at once.  The damped trials
// start from what the trial before left in pp and stay sequential.  The kind
// of the attempt is a run-time value and there is one call of the evaluation,
// so the kernel holds one inlined copy of it (six kinds with their own copies
// took 340 KB of code and spilled 850 registers).
// What the wave knows of its cell (one copy in LDS, read as broadcasts):
// inputs, the iterate pp, and of the current iteration the iterated variables
// x0, the residual f1 there and the inverse Jacobian.  Held in registers by
// every lane they would leave the evaluation too few.
template <int MAG>
struct WaveCell {
  double uu[Lay<MAG, 1>::NV], pp00[Lay<MAG, 1>::NV], pp[Lay<MAG, 1>::NV];
  double x0[4], f1[4], J[16], iJ[16];
  double dt, Ehat0;
  Geom g;
};
// orders the wave's LDS writes before its later reads by other lanes
KD_INL void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
template <int MAG>
KD_INL int imp_wave_attempt(const koral_params &P, ImpKind k, WaveCell<MAG> &w, double global_time, int maxiter,
                            int &iter)
{
  constexpr int NV = Lay<MAG, 1>::NV;
  constexpr int EE = Lay<MAG, 1>::EE;
  constexpr int WG = 8;
  const int sh = k.wp == P_MHD ? 1 : EE;
  const int grp = (threadIdx.x & 63) / WG;
  const int col = (grp >= 1 && grp <= 4) ? grp - 1 : -1;  // this lane's Jacobian column
  const double EPS = P.radimpeps;
  double xiapp = 1., errbase = 0.;
  double sign = -1., xp = 0., xj = 0., f[4] = {0., 0., 0., 0.}, err = 0.;
  int fret = 0, cret = 0, mode = IMP_EVAL;
  bool mine = true;  // this lane's group takes part in the next evaluation
  iter = 1;
#pragma unroll
  for (int i = 0; i < 4; i++) w.x0[i] = w.pp[sh + i];
  wave_sync();
  for (;;) {
    // the kind is opaque in the loop: specialised copies of it would not fit
    // the instruction cache
    asm volatile("" : "+s"(k.wp), "+s"(k.we), "+s"(k.wf));
    if (mine) {
      double ppt[NV];
#pragma unroll
      for (int i = 0; i < NV; i++) ppt[i] = w.pp[i];
      if (mode == IMP_EVAL) {
        xj = w.x0[col > 0 ? col : 0];
        xp = xj + imp_delta(EPS, col, sign, xj, w.g.g[col > 0 ? col : 1][col > 0 ? col : 1]);
#pragma unroll
        for (int i = 0; i < NV; i++)
          if (col >= 0 && i == sh + col) ppt[i] = xp;
      }
      fret = imp_eval<MAG, WG, -1, -1, -1>(P, k, mode, ppt, w.uu, w.pp00[1], w.Ehat0, w.dt, w.g, f, err, cret);
      if (mode != IMP_EVAL) {
        wave_sync();
#pragma unroll
        for (int i = 0; i < NV; i++) w.pp[i] = ppt[i];
        wave_sync();
      }
    }
    if (mode == IMP_FINAL) return cret < -1 ? IMP_FAIL : IMP_OK;
    if (mode == IMP_EVAL) {
      // a column that fails on one side is taken on the other
      mine = mine && col >= 0 && fret < 0 && sign < 0.;
      if (__ballot(mine)) {
        sign = mine ? 1. : sign;
        continue;
      }
      if (__shfl(fret, 0) < 0) return IMP_FAIL;
      errbase = __shfl(err, 0);
      mine = true;
      if (!(errbase >= ((k.we == ENTROPYEQ) ? P.radimpentrconv : P.radimpconv))) {
        if (iter > maxiter) return IMP_FAIL;
        mode = IMP_FINAL;
        continue;
      }
      if (__ballot(col >= 0 && fret < 0)) return IMP_FAIL;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const double f1 = __shfl(f[i], 0);
        w.f1[i] = f1;
        if (col >= 0) w.J[i * 4 + col] = (f[i] - f1) / (xp - xj);
      }
      wave_sync();
      double J[16], iJ[16];
#pragma unroll
      for (int i = 0; i < 16; i++) J[i] = w.J[i];
      if (inverse44(J, iJ) < 0) return IMP_FAIL;
#pragma unroll
      for (int i = 0; i < 16; i++) w.iJ[i] = iJ[i];
      xiapp = 1.;
      mode = IMP_TRIAL;
    } else {
      double x0[4], x[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        x0[i] = w.x0[i];
        x[i] = w.pp[sh + i];
      }
      if (imp_accept(P, x0[0], x[0], cret, xiapp)) {
        const bool conv = imp_conv_rel(P, k.we, EPS, x0, x, errbase, global_time);
        if (iter > maxiter) return IMP_FAIL;
        if (conv) {
          mode = IMP_FINAL;
          continue;
        }
        iter++;
        sign = -1.;
        mode = IMP_EVAL;
        wave_sync();
#pragma unroll
        for (int i = 0; i < 4; i++) w.x0[i] = x[i];
        wave_sync();
        continue;
      }
      // a NaN factor ends the attempt too
      if (!(xiapp >= P.maxradimpdamping)) return IMP_FAIL;
    }
    wave_sync();
    double x[4];
    imp_update(w.x0, w.iJ, w.f1, xiapp, x);
#pragma unroll
    for (int i = 0; i < 4; i++) w.pp[sh + i] = x[i];
    wave_sync();
  }
}
#endif

// solve_implicit_lab_4dprim, rad.c:376-1218: one attempt from pp00 by one
// lane; pp[5] and the conserved state are left to imp_finish
template <int MAG, int WP, int WE, int WF>
KD_INL int solve_4dprim_kind(const koral_params &P, const double *uu00, const double *pp00, double Ehat0,
                             const Geom &g, double dt, double *pp, double global_time, int &iters)
{
  constexpr int NV = Lay<MAG, 1>::NV;
  double Jm[16];
  ImpLane s;
#pragma unroll
  for (int i = 0; i < NV; i++) pp[i] = pp00[i];
  imp_lane_start<WP, Lay<MAG, 1>::EE>(s, pp);
  int st;
  do {
    st = imp_lane_trip<MAG, WP, WE, WF>(P, s, pp, uu00, pp00[1], Ehat0, dt, g, global_time, P.radimpmaxiter,
                                        [&](int i) -> double & { return Jm[i]; });
  } while (st == IMP_CONT);
  iters = s.iter;
  return st == IMP_OK ? 0 : -1;
}

// the six (primitives, equation, frame) kinds the fallback chain uses
template <int MAG>
KD_INL int solve_4dprim(const koral_params &P, const double *uu00, const double *pp00, double Ehat0, const Geom &g,
                        double dt, int wp, int we, int wf, double *pp, double global_time, int &iters)
{
#define KD_KIND(A, B, C) solve_4dprim_kind<MAG, A, B, C>(P, uu00, pp00, Ehat0, g, dt, pp, global_time, iters)
  if (wp == P_MHD) {
    if (we == ENERGYEQ) return wf == LAB ? KD_KIND(P_MHD, ENERGYEQ, LAB) : KD_KIND(P_MHD, ENERGYEQ, FF);
    if (wf == LAB) return KD_KIND(P_MHD, ENTROPYEQ, LAB);
  } else {
    if (we == ENERGYEQ) return wf == LAB ? KD_KIND(P_RAD, ENERGYEQ, LAB) : KD_KIND(P_RAD, ENERGYEQ, FF);
    if (wf == LAB) return KD_KIND(P_RAD, ENTROPYEQ, LAB);
  }
#undef KD_KIND
  return -1;  // the chain never asks for the fluid-frame entropy equation
}

// attempt a of the fallback chain (rad.c:1389-1464): energy LAB, energy FF,
// swapped LAB, swapped FF, entropy LAB, entropy swapped
KD_INL void imp_attempt(int a, int startwith, int &wp, int &we, int &wf)
{
  const int other = (startwith == P_RAD) ? P_MHD : P_RAD;
  wp = (a == 2 || a == 3 || a == 5) ? other : startwith;
  we = (a >= 4) ? ENTROPYEQ : ENERGYEQ;
  wf = (a == 1 || a == 3) ? FF : LAB;
}

// the fallback chain starts from RAD primitives when the fluid-frame
// radiation energy is small against the gas energy (rad.c:1340, 1381)
template <int MAG, int RAD>
KD_INL int imp_startwith(const koral_params &P, const double *pp00, const Geom &g)
{
  double Ehat = -ff_Rtt<MAG, RAD>(pp00, g, nullptr);
  return (Ehat < P.radimplicitthreshold * pp00[1]) ? P_RAD : P_MHD;
}

struct ImpInfo {
  int iters, attempt, whichprim, whicheq, whichframe, total;
};

// solve_implicit_lab + implicit_lab_rad_source_term (rad.c:1225-1570,
// rad.c:2758-2795).  Returns 0 on success with uu/pp updated.
template <int MAG, int RAD>
KD_FUN int solve_implicit_lab(const koral_params &P, double *uu, double *pp, const Geom &g, double dt,
                              double global_time, ImpInfo &info)
{
  constexpr int NV = Lay<MAG, RAD>::NV;
  double pp00[NV], ppn[NV];
#pragma unroll
  for (int i = 0; i < NV; i++) pp00[i] = pp[i];
  const double Ehat0 = -ff_Rtt<MAG, RAD>(pp00, g, nullptr);
  const int startwith = imp_startwith<MAG, RAD>(P, pp00, g);
  int ret = -1, total = 0, it = 0, a = 0;
  int wp = startwith, we = ENERGYEQ, wf = LAB;
  for (a = 0; a < 6; a++) {
    imp_attempt(a, startwith, wp, we, wf);
    ret = solve_4dprim<MAG>(P, uu, pp00, Ehat0, g, dt, wp, we, wf, ppn, global_time, it);
    total += it;
    if (ret == 0) break;
  }
  info.total = total;
  info.attempt = (ret == 0) ? a : -1;
  info.iters = (ret == 0) ? it : 0;
  info.whichprim = (ret == 0) ? wp : 0;
  info.whicheq = (ret == 0) ? we : 0;
  info.whichframe = (ret == 0) ? wf : 0;
  if (ret != 0) return -1;
  imp_finish<MAG>(P, ppn, uu, g);
#pragma unroll
  for (int i = 0; i < NV; i++) pp[i] = ppn[i];
  return 0;
}

}  // namespace kd
