// speedy_adjoint.hpp -- reverse mode (vector-Jacobian product) of the SPEEDY
// column physics of speedy_column.hpp, written by hand term by term.
//
// It replaces jax.vjp of SpeedyPhysics.compute_tendencies
// (jcm/physics/speedy/speedy_physics.py:88-127) with respect to the state
// fields T, q, u, v, ps and five parameters: convection.rhbl (params.py:24),
// convection.trcnv (:22), condensation.rhlsc (:60), a multiplier on the CO2
// longwave absorptivity (speedy/forcing.py:33) and a multiplier on the surface
// drag coefficients cdl, cds (params.py:191-192).
//
// Conventions follow JAX's differentiation of the reference expressions:
//   * discrete decisions (convective top, cloud top, the level set S, every
//     jnp.where condition) are held fixed; the gradient flows through the
//     selected branch only;
//   * max/min/clip give 1/2 to each operand at a tie (lax.max / lax.min);
//   * a reduction max (jnp.max over levels, clouds) splits the gradient evenly
//     over the tied entries.
// The forward and its reversal are interleaved (phase_b1_vjp, phase_b2_taped,
// phase_b2_vjp, phase_a_adj): the surface fluxes and the shortwave are reversed
// right after they ran, the longwave in the two sweeps that its forward makes, and
// phase A last, from a recompute of the convection and the clouds.
#pragma once

#include "speedy_column.hpp"

namespace speedy {

enum { VJP_RHBL = 0, VJP_TRCNV = 1, VJP_RHLSC = 2, VJP_CO2 = 3, VJP_DRAG = 4, VJP_NPARAM = 5 };

// Floats per column of the longwave tape: per level 1 .. KX-1 and band the flux
// entering the level from above and the adjoint of the flux leaving it upward.
template <int KX>
constexpr int vjp_tape_floats() { return 8 * (KX - 1); }

// Cotangents of one column's tendencies.  Only level KX-1 of the u and v
// tendencies is nonzero in the forward (surface stress), so only those matter.
template <typename R, int KX>
struct ColumnCt {
  R du1, dv1;
  R dt[KX], dq[KX];
};

// Adjoint accumulators: the state gradients, the parameter gradients and the
// adjoints of the intermediates that several terms share.
template <typename R, int KX>
struct ColumnAdj {
  R T[KX], Q[KX], ps, u1, v1;
  R prm[VJP_NPARAM];
  R qsat[KX], rh[KX], se[KX];
  R cloudc, clstr, qcloud, precnv, precls, rps;
};

// Materialize values at this point of the program: an empty asm that reads and
// writes them.  Computations feeding them cannot be sunk past it, so a term's
// (or a level's) reversal completes before the next one's recompute starts and
// its intermediates die there.
template <typename R>
SPD_HD void settle(R& x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(x));
#else
  (void)x;
#endif
}

// The accumulator fences are applied where the kernel fits in registers (up to
// eight levels).  At sixteen levels the accumulators alone are ~100 values, and
// forcing them into VGPRs at every fence makes the kernel spill around the fences.
template <int KX>
constexpr bool kSettle = KX <= 8;

template <typename R, int KX>
SPD_HD void settle_adj(ColumnAdj<R, KX>& g) {
  if constexpr (!kSettle<KX>) return;
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    settle(g.T[k]); settle(g.Q[k]); settle(g.qsat[k]); settle(g.rh[k]); settle(g.se[k]);
  }
  settle(g.ps); settle(g.u1); settle(g.v1);
#pragma unroll
  for (int i = 0; i < VJP_NPARAM; ++i) settle(g.prm[i]);
  settle(g.cloudc); settle(g.clstr); settle(g.qcloud); settle(g.precnv); settle(g.precls); settle(g.rps);
}

// The same after level k of the longwave's up sweep.
template <typename R, int KX>
SPD_HD void settle_lw(ColumnAdj<R, KX>& g, int k, R Fu[4], R aD[4], R& a_below) {
  settle(g.T[k]); settle(g.Q[k]); settle(g.ps); settle(g.cloudc); settle(g.rps); settle(a_below);
  if (k < KX - 1) settle(g.T[k + 1]);
#pragma unroll
  for (int bnd = 0; bnd < 4; ++bnd) { settle(Fu[bnd]); settle(aD[bnd]); }
}

template <typename R, int KX>
SPD_HD void adj_zero(ColumnAdj<R, KX>& g) {
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    g.T[k] = R(0.0); g.Q[k] = R(0.0); g.qsat[k] = R(0.0); g.rh[k] = R(0.0); g.se[k] = R(0.0);
  }
  g.ps = R(0.0); g.u1 = R(0.0); g.v1 = R(0.0);
#pragma unroll
  for (int i = 0; i < VJP_NPARAM; ++i) g.prm[i] = R(0.0);
  g.cloudc = R(0.0); g.clstr = R(0.0); g.qcloud = R(0.0); g.precnv = R(0.0); g.precls = R(0.0);
  g.rps = R(0.0);
}

// verify_tendencies (physics_interface.py:321-342) in reverse: where a level's
// q tendency was limited to -q/dt, its cotangent reaches the unclamped q as
// -1/dt and none of it reaches the physics.  g_qraw receives that part.
template <typename R, int KX>
SPD_HD void verify_ct(uint32_t flags, uint32_t limited, R dt, ColumnCt<R, KX>& ct, R g_qraw[KX]) {
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    g_qraw[k] = R(0.0);
    const bool lim = (flags & SPEEDY_FLAG_VERIFY_TENDENCIES) && ((limited >> k) & 1u);
    g_qraw[k] = sel(lim, -ct.dq[k] / dt, R(0.0));
    ct.dq[k] = sel(lim, R(0.0), ct.dq[k]);
  }
}

// verify_state in reverse: where(q < 0, 0, q) passes the gradient only where q >= 0.
template <typename R>
SPD_HD R verify_q_grad(R q_raw, R g) { return sel(q_raw < R(0.0), R(0.0), g); }

// Reciprocal for gradients of the fields alone: the hardware reciprocal and one
// Newton step (1 ulp), 3 instructions where a division takes 11.  The forward's
// values, which decisions depend on, and what the parameter gradients pass through
// keep mdiv: those are sums of many columns that nearly cancel.
SPD_HD float mrcp(float b) {
#if defined(__HIP_DEVICE_COMPILE__)
  const float r = __builtin_amdgcn_rcpf(b);
  return __builtin_fmaf(__builtin_fmaf(-b, r, 1.0f), r, r);
#else
  return 1.0f / b;
#endif
}
SPD_HD double mrcp(double b) { return 1.0 / b; }

// d q / d ta and ps * d q / d ps of q = qsat_f(ta, ps, sig) (humidity.py:95-102), from
// q itself.  With q = 622 e / D and D = sig ps - 0.378 e, sig ps / D = 1 + 0.378 q / 622, so
// dq/dta = q (sig ps / D) e'/e with e'/e = c (273.16 - tt) / (ta - tt)^2, and
// dq/dps = -q (sig ps / D) / ps: no exponential and one reciprocal.
template <typename R>
SPD_HD void qsat_grad(R ta, R q, R& dq_dt, R& ps_dq_dps) {
  const bool warm = ta >= R(273.16);
  const R c = warm ? R(17.269 * (273.16 - 35.86)) : R(21.875 * (273.16 - 7.66));
  const R tt = warm ? R(35.86) : R(7.66);
  const R gq = q + q * q * R(0.378 / 622.0);
  dq_dt = gq * c * mrcp(sq(ta - tt));
  ps_dq_dps = -gq;
}

// acc += a * b where `on`.  The choice is made on the sum and not on a factor: a term that
// is off adds nothing, whatever its other factor is (a level whose humidity is not finite
// must not reach the gradients of the levels beside it through terms that are off).
template <typename R>
SPD_HD void add_if(bool on, R& acc, R a, R b) { acc = sel(on, acc + a * b, acc); }

// Adjoint of radset4 (longwave_radiation.py:216-225): returns d/d temp of
// sum_b a_fb[b] * fb[b].  jnp.clip(temp, 200, 320) = min(max(temp, 200), 320).
template <typename R>
SPD_HD R radset4_adj(R temp, R omeps, const R a_fb[4]) {
  const R jlo = mmax(temp, R(200.0));
  const R jt = mmin(jlo, R(320.0));
  const R d1 = R(-2.0 * 3.0e-6) * (jt - R(247.0));
  const R d2 = R(-2.0 * 5.2e-6) * (jt - R(282.0));
  const R d3 = R(2.0 * 1.0e-5) * (jt - R(315.0));
  const R d0 = -((d1 + d2) + d3);
  const R a_jt = omeps * (a_fb[0] * d0 + a_fb[1] * d1 + a_fb[2] * d2 + a_fb[3] * d3);
  return a_jt * dmin_x(jlo, R(320.0)) * dmax_x(temp, R(200.0));
}

// Adjoint of level k's longwave transmissivities tauL[k][:] = exp(-ab * ps * dhs)
// (shortwave_radiation.py:177-200) and emissions st4a0[k], st4a1[k]
// (longwave_radiation.py:48-68), applied at once so that no per-level adjoint
// arrays stay live.  Gradients of the half-level temperatures above and below the
// level go to a_Th[0] and a_Th[1].
template <typename R, int KX>
SPD_HD void lw_level_adj(int k, const R a_tau[4], R a_s0, R a_s1, const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a,
                         const R tau[4], const SpeedyParams& p, const SpeedyVertical& v, const Uniforms<R>& u,
                         ColumnAdj<R, KX>& g, R a_Th[2]) {
  R ab[4];
  lw_absorptivity<R, KX>(k, c, a, p, u, ab);
#pragma unroll
  for (int bnd = 0; bnd < 4; ++bnd) {
    const R ax = a_tau[bnd] * tau[bnd];
    g.ps += ax * (-(ab[bnd] * v.dhs[k]));
    const R a_ab = ax * (-(c.ps * v.dhs[k]));
    if (bnd == 0) {
      if (k >= 2 && k <= KX - 2) g.cloudc += a_ab * sel(k > a.icltop, R(p.ablcl1), R(p.ablcl2));
    } else if (bnd >= 2 && k >= 1) {   // band 1 (CO2): the caller's

      const R wv = (bnd == 2) ? p.ablwv1 : p.ablwv2;
      if (k >= 2 && k <= KX - 2) {
        const R x = wv * c.Q[k], ac2 = a.cloudc * p.ablcl2;
        g.Q[k] += a_ab * dmax_x(x, ac2) * wv;
        g.cloudc += a_ab * dmax_x(ac2, x) * p.ablcl2;
      } else {
        g.Q[k] += a_ab * wv;
      }
    }
  }
  // emissions; Th[j] = T[j] + wvi1[j] * (T[j+1] - T[j]) as in lw_down
  auto Th = [&](int j) { return c.T[j] + u.wvi1[j] * (c.T[j + 1] - c.T[j]); };
  if (k >= 2) {
    const R T = c.T[k];
    const R st3a = R(SBC) * pow3(T);
    R grad;
    if (k < KX - 1) grad = R(0.5) * mmax(Th(k) - Th(k - 1), R(0.0));
    else grad = mmax(c.T[KX - 1] - Th(KX - 2), R(0.0));
    const R a_st3a = a_s0 * T + a_s1 * R(4.0) * grad;
    g.T[k] += a_s0 * st3a + a_st3a * R(3.0 * SBC) * T * T;
    const R a_grad = a_s1 * R(4.0) * st3a;
    if (k < KX - 1) {
      const R ax = a_grad * R(0.5) * dmax_x(Th(k) - Th(k - 1), R(0.0));
      a_Th[1] += ax;
      a_Th[0] += -ax;
    } else {
      const R ax = a_grad * dmax_x(c.T[KX - 1] - Th(KX - 2), R(0.0));
      g.T[KX - 1] += ax;
      a_Th[0] += -ax;
    }
  } else if (k == 0) {
    const R s0 = R(0.75) * c.T[0] + R(0.25) * Th(0);
    const R as = a_s0 * R(4.0 * SBC) * pow3(s0);
    g.T[0] += R(0.75) * as;
    a_Th[1] += R(0.25) * as;
  } else {
    const R s1 = R(0.50) * c.T[1] + R(0.25) * (Th(0) + Th(1));
    const R as = a_s0 * R(4.0 * SBC) * pow3(s1);
    g.T[1] += R(0.50) * as;
    a_Th[0] += R(0.25) * as;
    a_Th[1] += R(0.25) * as;
  }
}

// The column as level k's longwave recompute sees it: the values lw_level(k)
// reads (T at k-1..k+1, q at k, ps) are passed through an empty asm that also
// takes `dep`, the flux entering level k, so the recompute is neither merged with
// the downward sweep's (which would keep every level's transmissivities live in
// between) nor hoisted above the previous level.
template <typename R, int KX>
SPD_HD ColumnIn<R, KX> column_at_level(const ColumnIn<R, KX>& c, int k, R dep) {
  ColumnIn<R, KX> cc = c;
#if defined(__HIP_DEVICE_COMPILE__)
  for (int j = k - 1; j <= k + 1; ++j)
    if (j >= 0 && j < KX) asm volatile("" : "+v"(cc.T[j]) : "v"(dep));
  asm volatile("" : "+v"(cc.Q[k]) : "v"(dep));
  asm volatile("" : "+v"(cc.ps) : "v"(dep));
#else
  (void)k; (void)dep;
#endif
  return cc;
}

// ---------------------------------------------------------------- longwave
// Cotangent of level k's longwave flux divergence (tlw[k] = dfl[k] grdscp[k] / ps).
template <typename R, int KX>
SPD_HD R dfl_ct(const ColumnCt<R, KX>& ct, const SpeedyVertical& v, int k, R rps) {
  return ct.dt[k] * v.grdscp[k] * rps;
}

// Longwave down (longwave_radiation.py:13-117) runs from the top down, and so does
// the adjoint of longwave up; longwave up and the adjoint of longwave down run from
// the surface up.  So the forward and the reverse of the whole longwave take two
// sweeps.  The adjoint fluxes need only the cotangents and the transmissivities:
//   down sweep   Fd (forward) and aU, the adjoint of the upward fluxes; both are kept
//                per level and band on the tape;
//   up sweep     Fu (forward) and aD, the adjoint of the downward fluxes; each level
//                then has all four, and its transmissivities, emissions and band
//                fractions are reversed once for both directions.
// One recompute of a level's transmissivities remains (the up sweep's, which the
// forward kernels make too).  Reversing each direction by itself with a forward
// recompute before it took six evaluations of every level and 7700 VALU
// instructions a wave at 8 levels for the whole adjoint.
//
// Leaves aF, the adjoint of the flux leaving the surface, and b.dfl, b.rlds as
// lw_down does.
template <typename R, int KX, class Store>
SPD_HD void lw_down_vjp(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, const SpeedyParams& p,
                        const SpeedyVertical& v, const Uniforms<R>& u, const ColumnCt<R, KX>& ct, PhaseB<R, KX>& b,
                        Store& tape, R aF[4]) {
  const R rps = mdiv(R(1.0), c.ps);
  R Fd[4], Fprev = R(0.0);
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    const R a_dfl = dfl_ct<R, KX>(ct, v, k, rps);
    LwLevel<R> L;
    lw_level<R, KX>(k, c, a, p, v, u, L);
    if (k == 0) {
#pragma unroll
      for (int bnd = 0; bnd < 4; ++bnd) {
        const R em = R(1.0) - L.tau[bnd];
        Fd[bnd] = bnd < 2 ? em * (L.fb[bnd] * (L.st0 + em * L.st1)) : R(0.0);
        aF[bnd] = bnd < 2 ? a_dfl - a_dfl * L.tau[bnd] : R(0.0);
      }
    } else {
#pragma unroll
      for (int bnd = 0; bnd < 4; ++bnd) {
        const R au = aF[bnd] - a_dfl;              // dfl[k] += sum Fu[k+1] - sum Fu[k]
        tape.put((k - 1) * 8 + bnd, Fd[bnd]);
        tape.put((k - 1) * 8 + 4 + bnd, au);
        aF[bnd] = a_dfl + au * L.tau[bnd];
        const R em = R(1.0) - L.tau[bnd];
        Fd[bnd] = L.tau[bnd] * Fd[bnd] + em * (L.fb[bnd] * (L.st0 + em * L.st1));
      }
    }
    const R Fs = ((Fd[0] + Fd[1]) + Fd[2]) + Fd[3];
    b.dfl[k] = k == 0 ? -Fs : -(Fs - Fprev);
    Fprev = Fs;
    if (k == KX - 1) {
      R rlds = ((p.emisfc * Fd[0] + p.emisfc * Fd[1]) + p.emisfc * Fd[2]) + p.emisfc * Fd[3];
      const R corlw = u.corlw * L.st0;
      b.dfl[KX - 1] = b.dfl[KX - 1] + (-corlw);
      b.rlds = rlds + corlw;
    }
  }
}

// Cotangents of the longwave's surface inputs, from the down sweep's aF and the
// lowest level's a_dfl.
template <typename R, int KX>
SPD_HD void lw_surface_adj(const Uniforms<R>& u, const SpeedyParams& p, R tsfc, R a_dfl, const R aF[4], R& a_rlus2,
                           R a_flux_h[2]) {
  R fbt[4];
  radset4(tsfc, u.omeps, fbt);
  a_rlus2 = ((aF[0] * fbt[0] + aF[1] * fbt[1]) + (aF[2] * fbt[2] + aF[3] * fbt[3])) + a_dfl * p.epslw;
  a_flux_h[0] = aF[0] * u.refsfc;
  a_flux_h[1] = aF[1] * u.refsfc;
}

// The gradient of the CO2 multiplier is the one sum that cancels both between the
// directions and over the columns, so each direction's part is formed by itself (it
// waits on the tape, in the place of the level's band-1 fluxes) and added in the order
// of the levels, upward flux first.
//
// The up sweep: longwave up (longwave_radiation.py:119-202; b.dfl enters holding the
// longwave-down divergence, b.tlw leaves as lw_up leaves it) and every level's
// reversal.  b.rlus2, b.tsfc, b.flux_h: the hand-offs of the surface fluxes and the
// shortwave; a_rlds: cotangent of the downward flux at the surface.
template <typename R, int KX, class Store>
SPD_HD void lw_up_vjp(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, const SpeedyParams& p,
                      const SpeedyVertical& v, const Uniforms<R>& u, PhaseB<R, KX>& b, Store& tape,
                      const ColumnCt<R, KX>& ct, R a_rlds, ColumnAdj<R, KX>& g) {
  const R ps = c.ps;
  const R rps = mdiv(R(1.0), ps);
  const R stratc0 = c.stratz * ps, stratc1 = u.eps1 * ps;
  R Fu[4], aD[4];
  {
    R fbt[4];
    radset4(b.tsfc, u.omeps, fbt);
    const R flux_h[4] = {b.flux_h[0], b.flux_h[1], R(0.0), R(0.0)};
#pragma unroll
    for (int bnd = 0; bnd < 4; ++bnd) {
      Fu[bnd] = fbt[bnd] * b.rlus2 + u.refsfc * flux_h[bnd];
      aD[bnd] = a_rlds * p.emisfc;
    }
  }
  b.dfl[KX - 1] = b.dfl[KX - 1] + p.epslw * b.rlus2;
  R Gnext = ((Fu[0] + Fu[1]) + Fu[2]) + Fu[3];
  // a_below: cotangent of the half-level temperature under level k, complete once
  // level k is reversed, and then passed on to T
  R a_below = R(0.0), corlw2 = R(0.0), up0 = R(0.0), dn0 = R(0.0);
#pragma unroll
  for (int k = KX - 1; k >= 0; --k) {
    const ColumnIn<R, KX> ck = column_at_level<R, KX>(c, k, Fu[0]);
    auto&& tk = tape.after(Fu[0]);
    LwLevel<R> L;
    lw_level<R, KX>(k, ck, a, p, v, u, L);
    const R a_dfl = dfl_ct<R, KX>(ct, v, k, rps);
    R afb[4], atau[4], as0 = R(0.0), as1 = R(0.0);
    if (k == KX - 1) as0 = (a_rlds - a_dfl) * u.corlw;   // rlds += corlw, dfl[KX-1] -= corlw
    if (k <= 1) {   // dfl[k] -= dhs[k] stratc1 st4a0[k] (+ stratc0 at k = 0)
      as0 += -a_dfl * v.dhs[k] * stratc1;
      g.ps += -a_dfl * v.dhs[k] * L.st0 * u.eps1;
      if (k == 0) g.ps += -a_dfl * c.stratz;
    }
    if (k > 0) {
#pragma unroll
      for (int bnd = 0; bnd < 4; ++bnd) {
        const R tau = L.tau[bnd], em = R(1.0) - tau;
        const R au = tk.get((k - 1) * 8 + 4 + bnd), fd = tk.get((k - 1) * 8 + bnd);
        const R ad = aD[bnd] - a_dfl;             // dfl[k] = sum Fd[k-1] - sum Fd[k]
        aD[bnd] = a_dfl + ad * tau;
        // up: tau Fu + em fb (st0 - em st1); down: tau Fd + em fb (st0 + em st1).  The flux
        // and the emission nearly cancel: their difference is formed before the product
        const R sum = au + ad, dif = ad - au;
        const R es = em * L.st1;
        const R up = au * (Fu[bnd] - L.fb[bnd] * (L.st0 - R(2.0) * em * L.st1));
        const R dn = ad * (fd - L.fb[bnd] * (L.st0 + R(2.0) * em * L.st1));
        atau[bnd] = up + dn;
        if (bnd == 1) {
          tk.put((k - 1) * 8 + 5, up * tau * (-(ck.ps * v.dhs[k])));
          tk.put((k - 1) * 8 + 1, dn * tau * (-(ck.ps * v.dhs[k])));
        }
        afb[bnd] = em * (sum * L.st0 + dif * es);
        const R ef = em * L.fb[bnd];
        as0 += sum * ef;
        as1 += dif * ef * em;
        Fu[bnd] = L.tau[bnd] * Fu[bnd] + em * (L.fb[bnd] * (L.st0 - em * L.st1));
      }
      const R Gk = ((Fu[0] + Fu[1]) + Fu[2]) + Fu[3];
      b.dfl[k] = b.dfl[k] + (Gnext - Gk);
      Gnext = Gk;
      if (k == 1) {
        corlw2 = v.dhs[1] * stratc1 * L.st0;
        b.dfl[1] = b.dfl[1] + (-corlw2);
      }
    } else {   // the top level absorbs and emits in bands 0 and 1 only (st1 = 0 there)
      R ft[2];
#pragma unroll
      for (int bnd = 0; bnd < 2; ++bnd) {
        const R em = R(1.0) - L.tau[bnd];
        const R au = -a_dfl, ad = aD[bnd] - a_dfl;
        const R sum = au + ad;
        const R up = au * (Fu[bnd] - L.fb[bnd] * L.st0), dn = -ad * L.fb[bnd] * L.st0;
        atau[bnd] = up + dn;
        if (bnd == 1) {
          up0 = up * L.tau[1] * (-(ck.ps * v.dhs[0]));
          dn0 = dn * L.tau[1] * (-(ck.ps * v.dhs[0]));
        }
        afb[bnd] = sum * em * L.st0;
        as0 += sum * em * L.fb[bnd];
        ft[bnd] = L.tau[bnd] * Fu[bnd] + em * (L.fb[bnd] * (L.st0 - em * L.st1));
      }
      atau[2] = atau[3] = afb[2] = afb[3] = R(0.0);
      b.dfl[0] = b.dfl[0] + ((Fu[0] - ft[0]) + (Fu[1] - ft[1]));
      const R corlw1 = v.dhs[0] * stratc1 * L.st0 + stratc0;
      b.dfl[0] = b.dfl[0] + (-corlw1);
    }
    b.tlw[k] = b.dfl[k] * v.grdscp[k] * rps;
    g.rps += ct.dt[k] * b.dfl[k] * v.grdscp[k];
    g.T[k] += radset4_adj(ck.T[k], u.omeps, afb);
    R a_Th[2] = {R(0.0), a_below};   // the half levels above (k - 1) and below (k)
    lw_level_adj<R, KX>(k, atau, as0, as1, ck, a, L.tau, p, v, u, g, a_Th);
    if (k < KX - 1) {   // Th[k] = T[k] + wvi1[k] (T[k+1] - T[k])
      g.T[k] += a_Th[1] * (R(1.0) - u.wvi1[k]);
      g.T[k + 1] += a_Th[1] * u.wvi1[k];
    }
    a_below = a_Th[0];
    settle_lw<R, KX>(g, k, Fu, aD, a_below);
  }
  auto&& tc = tape.after(up0);
  g.prm[VJP_CO2] += up0 * u.ablco2_d;
#pragma unroll
  for (int k = 1; k < KX; ++k) g.prm[VJP_CO2] += tc.get((k - 1) * 8 + 5) * u.ablco2_d;
#pragma unroll
  for (int k = KX - 1; k >= 1; --k) g.prm[VJP_CO2] += tc.get((k - 1) * 8 + 1) * u.ablco2_d;
  g.prm[VJP_CO2] += dn0 * u.ablco2_d;
}

// ---------------------------------------------------------------- surface fluxes
template <typename R, int KX>
SPD_HD void surface_adj(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, const PhaseB<R, KX>& b,
                        const SpeedyParams& s, const SpeedyVertical& v, const Uniforms<R>& u, const SfcTape<R>& t,
                        const ColumnCt<R, KX>& ct, R a_rlus2, R& a_rsds, R& a_rlds, ColumnAdj<R, KX>& g) {
  if (!t.land) return;   // every surface output is zero without lfluxland (Q8)
  const R ps = c.ps;
  const R rps = mdiv(R(1.0), ps);
  const R fm = c.fmask;
  const R gs = v.grdsig[KX - 1], gc = v.grdscp[KX - 1];
  const R a_ustr2 = ct.du1 * rps * gs, a_vstr2 = ct.dv1 * rps * gs;
  const R a_shf2 = ct.dt[KX - 1] * rps * gc, a_evap2 = ct.dq[KX - 1] * rps * gs;
  g.rps += ((ct.du1 * t.ustr2 * gs + ct.dv1 * t.vstr2 * gs) + ct.dt[KX - 1] * t.shf2 * gc) + ct.dq[KX - 1] * t.evap2 * gs;
  const R om = R(1.0) - fm;
  R a_ustr0 = fm * a_ustr2, a_ustr1 = om * a_ustr2;
  R a_vstr0 = fm * a_vstr2, a_vstr1 = om * a_vstr2;
  R a_shf0 = fm * a_shf2, a_shf1 = om * a_shf2;
  R a_evap0 = fm * a_evap2, a_evap1 = om * a_evap2;
  R a_rlus0 = fm * a_rlus2;
  R a_Tb = R(0.0), a_Qb = R(0.0), a_t1_0 = R(0.0), a_t1_1 = R(0.0), a_t2_0 = R(0.0), a_t2_1 = R(0.0);
  R a_den0 = R(0.0), a_den1 = R(0.0), a_den2 = R(0.0), a_tskin = R(0.0), a_qsat00 = R(0.0);
  R dqt, dqp, a_psq = R(0.0);   // a_psq: sum of the qsat gradients times ps
  // sea
  a_den2 += a_evap1 * s.chs * (t.qsat01 - t.q1_1);
  const R a_qsat01 = a_evap1 * s.chs * t.den2;
  R a_q1_1 = -a_evap1 * s.chs * t.den2;
  qsat_grad(c.sst, t.qsat01, dqt, dqp);
  a_psq += a_qsat01 * dqp;
  a_den2 += a_shf1 * u.chscp * (c.sst - t.t1_1);
  a_t1_1 += -a_shf1 * u.chscp * t.den2;
  // land: sea-side stress and humidity
  {
    const R cdsdv = u.cds * t.den2;
    const R a_cdsdv = -(a_ustr1 * c.u1 + a_vstr1 * c.v1);
    g.u1 += -a_ustr1 * cdsdv;
    g.v1 += -a_vstr1 * cdsdv;
    a_den2 += a_cdsdv * u.cds;
    g.prm[VJP_DRAG] += a_cdsdv * t.den2 * s.cds;
  }
  if (s.fhum0 > R(0.0)) {
    const R qs = qsat_f(t.t1_1, ps, R(1.0));
    const R a_qs = a_q1_1 * s.fhum0 * a.rh[KX - 1];
    g.rh[KX - 1] += a_q1_1 * s.fhum0 * qs;
    qsat_grad(t.t1_1, qs, dqt, dqp);
    a_t1_1 += a_qs * dqt;
    a_psq += a_qs * dqp;
    a_Qb += a_q1_1 * u.ghum0;
  } else {
    a_Qb += a_q1_1;
  }
  a_den0 += a_den2 * (R(1.0) + t.dths * u.rdth);
  {
    const R a_dths = a_den2 * t.den0 * u.rdth;
    const R a_ds = sel(c.sst > t.t2_1, a_dths * dmin_x(t.ds, R(s.dtheta)),
                       a_dths * dmax_x(u.astab * t.ds, -R(s.dtheta)) * u.astab);
    a_t2_1 += -a_ds;
  }
  // skin-temperature energy-balance correction (surface_flux.py:189-221)
  R a_hfl0 = R(0.0), a_drls = R(0.0);
  if (s.lskineb) {
    R a_dtskin = a_shf0 * u.chlcp * t.den1;
    a_den1 += a_shf0 * u.chlcp * t.dtskin;
    a_den1 += a_evap0 * s.chl * t.qs1 * t.dtskin;
    R a_qs1 = a_evap0 * s.chl * t.den1 * t.dtskin;
    a_dtskin += a_evap0 * s.chl * t.den1 * t.qs1;
    a_drls += a_rlus0 * t.dtskin;
    a_dtskin += a_rlus0 * t.drls;
    const R Dn = t.clamb + t.drls + (s.chl * t.den1 * (R(CP) + (R(ALHC) * t.qs1)));
    const R a_hflc = mdiv(a_dtskin, Dn);
    const R a_Dn = -a_hflc * t.dtskin;
    a_drls += a_Dn;
    a_den1 += a_Dn * s.chl * (R(CP) + R(ALHC) * t.qs1);
    a_qs1 += a_Dn * s.chl * t.den1 * R(ALHC);
    {
      const bool wet = t.evap0a > R(0.0);
      const R a_qs1p = a_qs1 * c.soilw;
      a_qsat00 += sel(wet, -a_qs1p, R(0.0));
      qsat_grad(t.tskin0 + R(1.0), t.qs1p, dqt, dqp);
      add_if(wet, a_tskin, a_qs1p, dqt);
      add_if(wet, a_psq, a_qs1p, dqp);
    }
    a_hfl0 += a_hflc;
    a_tskin += -a_hflc * t.clamb;
  }
  // net surface heat flux hfl0 (surface_flux.py:185)
  a_rsds += a_hfl0 * (R(1.0) - b.alb_l);
  a_rlds += a_hfl0;
  a_rlus0 += -a_hfl0;
  a_shf0 += -a_hfl0;
  a_evap0 += -a_hfl0 * R(ALHC);
  {
    const R a_tsk3 = a_rlus0 * u.esbc * t.tskin0 + a_drls * R(4.0) * u.esbc;
    a_tskin += a_rlus0 * u.esbc * t.tsk3 + a_tsk3 * R(3.0) * t.tskin0 * t.tskin0;
  }
  {
    a_den1 += a_evap0 * s.chl * mmax(R(0.0), t.evx);
    const R a_evx = a_evap0 * s.chl * t.den1 * dmax_x(t.evx, R(0.0));
    a_qsat00 += a_evx * c.soilw;
    const R a_q1_0 = -a_evx;
    qsat_grad(t.tskin0, t.qsat00, dqt, dqp);
    a_tskin += a_qsat00 * dqt;
    a_psq += a_qsat00 * dqp;
    if (s.fhum0 > R(0.0)) {
      const R qs = qsat_f(t.t1_0, ps, R(1.0));
      const R a_qs = a_q1_0 * s.fhum0 * a.rh[KX - 1];
      g.rh[KX - 1] += a_q1_0 * s.fhum0 * qs;
      qsat_grad(t.t1_0, qs, dqt, dqp);
      a_t1_0 += a_qs * dqt;
      a_psq += a_qs * dqp;
      a_Qb += a_q1_0 * u.ghum0;
    } else {
      a_Qb += a_q1_0;
    }
  }
  a_den1 += a_shf0 * u.chlcp * (t.tskin0 - t.t1_0);
  a_tskin += a_shf0 * u.chlcp * t.den1;
  a_t1_0 += -a_shf0 * u.chlcp * t.den1;
  {
    const R a_cdldv = -(a_ustr0 * c.u1 + a_vstr0 * c.v1);
    g.u1 += -a_ustr0 * t.cdldv;
    g.v1 += -a_vstr0 * t.cdldv;
    a_den0 += a_cdldv * u.cdl * t.forog;
    g.prm[VJP_DRAG] += a_cdldv * s.cdl * t.den0 * t.forog;
  }
  a_den0 += a_den1 * (R(1.0) + t.dthl * u.rdth);
  {
    const R a_dthl = a_den1 * t.den0 * u.rdth;
    const R a_dd = sel(t.tskin0 > t.t2_0, a_dthl * dmin_x(t.dd, R(s.dtheta)),
                       a_dthl * dmax_x(u.astab * t.dd, -R(s.dtheta)) * u.astab);
    a_tskin += a_dd;
    a_t2_0 += -a_dd;
  }
  // tskin0 = stl + ctday * sqcoa * rsds * (1 - alb_l) * ps
  {
    const R k0 = s.ctday * c.sqcoa;
    a_rsds += a_tskin * k0 * (R(1.0) - b.alb_l) * ps;
    g.ps += a_tskin * k0 * b.rsds * (R(1.0) - b.alb_l);
  }
  // den0 = (p0 * ps / (rgas * t0)) * wind
  R a_t0;
  {
    const R rt0 = mrcp(t.t0);
    const R rho_ps = R(P0 / RGAS) * rt0;
    const R rho = rho_ps * ps;
    const R a_rho = a_den0 * t.wind;
    const R a_wind = a_den0 * rho;
    g.ps += a_rho * rho_ps;
    a_t0 = -a_rho * rho * rt0;
    const R aw = a_wind * mrcp(t.wind) * s.fwind0;
    g.u1 += aw * t.u0;
    g.v1 += aw * t.v0;
  }
  a_t1_0 += a_t0 * fm;
  a_t1_1 += a_t0 * om;
  const R aw0 = sel(t.warm, a_t1_0, R(0.0)), aw1 = sel(t.warm, a_t1_1, R(0.0));
  R a_t1_0a = aw0 * s.ftemp0;
  const R a_t1_1a = aw1 * s.ftemp0;
  a_t2_0 += aw0 * u.gtemp0;
  a_t2_1 += aw1 * u.gtemp0;
  a_Tb += sel(t.warm, R(0.0), a_t1_0 + a_t1_1);
  a_t2_1 += a_t2_0;
  a_Tb += a_t2_1;
  a_t1_0a += a_t1_1a;
  R a_dt1 = -a_t1_1a * t.phi0 * mrcp(R(RGAS288) * v.sigl[KX - 1]);
  a_Tb += a_t1_0a;
  a_dt1 += a_t1_0a;
  a_Tb += a_dt1 * v.wvi[KX - 1][1];
  g.ps += a_psq * rps;
  g.T[KX - 2] += -a_dt1 * v.wvi[KX - 1][1];
  g.T[KX - 1] += a_Tb;
  g.Q[KX - 1] += a_Qb;
}

// ---------------------------------------------------------------- shortwave
// Only the transmissivities are kept from the forward (and a few scalars): the
// fluxes are their products, 45 instructions to form again against 32 values held
// across the surface fluxes and their reversal.
template <typename R, int KX>
SPD_HD void shortwave_adj(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, const PhaseB<R, KX>& b, uint32_t S,
                          const SpeedyParams& p, const SpeedyVertical& v, const Uniforms<R>& u,
                          const SwTape<R, KX>& fwd, const ColumnCt<R, KX>& ct, const R a_flux_h[2], R a_rsds,
                          ColumnAdj<R, KX>& g) {
  const R ps = c.ps;
  const R rps = mdiv(R(1.0), ps);
  SwTape<R, KX> t;
  t.psaz = fwd.psaz;
  t.acloud = fwd.acloud;
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    t.tau0[k] = fwd.tau0[k];
    t.tau1[k] = fwd.tau1[k];
    settle(t.tau0[k]);   // not the forward's registers: its products are not kept for the ones below
    if (k > 0) settle(t.tau1[k]);
    t.t22[k] = k == KX - 1 ? p.albcls * a.clstr : sel(((S >> k) & 1u) != 0u, fwd.a_cl, R(0.0));
  }
  const R F0 = c.fsol * R(0.95);
  t.f1[0] = t.tau0[0] * (F0 - c.ozupp * ps);
  t.f1[1] = t.tau0[1] * (t.f1[0] - c.ozone * ps);
  t.f2[0] = c.fsol * R(0.05);
#pragma unroll
  for (int k = 1; k < KX; ++k) {
    if (k > 1) t.f1[k] = t.f1[k - 1] * t.tau0[k] * (R(1.0) - t.t22[k]);
    t.f2[k] = t.f2[k - 1] * t.tau1[k];
  }
  t.fu[KX - 1] = t.f1[KX - 1] * b.albsfc;
#pragma unroll
  for (int k = KX - 1; k >= 1; --k) t.fu[k - 1] = t.fu[k] * t.tau0[k] + (k > 1 ? t.t22[k] * t.f1[k - 1] : t.t22[k]);
  const bool csw = u.compute_sw != 0u;
  R a_dfabs[KX];
#pragma unroll
  for (int k = 0; k < KX; ++k) a_dfabs[k] = sel(csw, ct.dt[k] * v.grdscp[k] * rps, R(0.0));
  R a_tau0[KX], a_tau1[KX], a_f1[KX], a_f2[KX], a_Rf[KX], a_fu[KX], a_t22[KX];
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    a_tau0[k] = R(0.0); a_tau1[k] = R(0.0); a_f1[k] = R(0.0); a_f2[k] = R(0.0);
    a_Rf[k] = R(0.0); a_fu[k] = R(0.0); a_t22[k] = R(0.0);
  }
  // ftoa = tau0[0] * fu[0] + Rf[0]; flux_h = (ftoa, f2[KX-1])
  a_tau0[0] += a_flux_h[0] * t.fu[0];
  a_fu[0] += a_flux_h[0] * t.tau0[0];
  a_Rf[0] += a_flux_h[0];
  a_f2[KX - 1] += a_flux_h[1];
  // dfabs[k] += fu[k] * (1 - tau0[k])
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    a_fu[k] += a_dfabs[k] * (R(1.0) - t.tau0[k]);
    a_tau0[k] += -a_dfabs[k] * t.fu[k];
  }
  // upward scan fu[k-1] = fu[k] * tau0[k] + Rf[k]
#pragma unroll
  for (int k = 1; k < KX; ++k) {
    a_fu[k] += a_fu[k - 1] * t.tau0[k];
    a_tau0[k] += a_fu[k - 1] * t.fu[k];
    a_Rf[k] += a_fu[k - 1];
  }
  a_f1[KX - 1] += a_fu[KX - 1] * b.albsfc + a_rsds;
  a_f2[KX - 1] += a_rsds;
  // dfabs[k] += f2[k-1] * (1 - tau1[k]); f2[k] = f2[k-1] * tau1[k]
#pragma unroll
  for (int k = 1; k < KX; ++k) {
    a_f2[k - 1] += a_dfabs[k] * (R(1.0) - t.tau1[k]);
    a_tau1[k] += -a_dfabs[k] * t.f2[k - 1];
  }
#pragma unroll
  for (int k = KX - 1; k >= 1; --k) {
    a_f2[k - 1] += a_f2[k] * t.tau1[k];
    a_tau1[k] += a_f2[k] * t.f2[k - 1];
  }
  a_t22[0] += a_Rf[0];
  a_t22[1] += a_Rf[1];
  // downward scan, levels KX-1 .. 2
#pragma unroll
  for (int k = KX - 1; k >= 2; --k) {
    const R om22 = R(1.0) - t.t22[k], omt = R(1.0) - t.tau0[k];
    const R fp = t.f1[k - 1];
    a_f1[k - 1] += a_dfabs[k] * om22 * omt + a_Rf[k] * t.t22[k] + a_f1[k] * t.tau0[k] * om22;
    a_t22[k] += -a_dfabs[k] * fp * omt + a_Rf[k] * fp - a_f1[k] * fp * t.tau0[k];
    a_tau0[k] += -a_dfabs[k] * fp * om22 + a_f1[k] * fp * om22;
  }
  // levels 1 and 0 (ozone absorption)
  a_f1[0] += a_dfabs[1];
  a_f1[1] += -a_dfabs[1];
  a_tau0[1] += a_f1[1] * (t.f1[0] - c.ozone * ps);
  a_f1[0] += a_f1[1] * t.tau0[1];
  g.ps += -a_f1[1] * t.tau0[1] * c.ozone;
  a_f1[0] += -a_dfabs[0];
  a_tau0[0] += a_f1[0] * (F0 - c.ozupp * ps);
  g.ps += -a_f1[0] * t.tau0[0] * c.ozupp;
  // transmissivities
  R a_psaz = R(0.0), a_acloud = R(0.0);
  a_psaz += a_tau0[0] * t.tau0[0] * (-(v.dhs[0] * p.absdry));
#pragma unroll
  for (int k = 1; k < KX; ++k) {
    const bool cloudy = k <= KX - 2 && k >= a.icltop;
    const R cl = sel(cloudy, t.acloud, R(0.0));
    const R A = u.sw_abs1[k] + p.abswv1 * c.Q[k] + cl;
    const R ax = a_tau0[k] * t.tau0[k];
    a_psaz += ax * (-(v.dhs[k] * A));
    const R a_A = ax * (-(t.psaz * v.dhs[k]));
    g.Q[k] += a_A * p.abswv1;
    a_acloud += sel(cloudy, a_A, R(0.0));
    const R bx = a_tau1[k] * t.tau1[k];
    a_psaz += bx * (-(v.dhs[k] * p.abswv2 * c.Q[k]));
    g.Q[k] += bx * (-(t.psaz * v.dhs[k] * p.abswv2));
  }
  {
    const R x = p.abscl1 * a.qcloud;
    g.cloudc += a_acloud * mmin(x, R(p.abscl2));
    g.qcloud += a_acloud * a.cloudc * dmin_x(x, R(p.abscl2)) * p.abscl1;
  }
  g.ps += a_psaz * c.zenit;
  // cloud albedo at the levels of S (Q1) and stratiform albedo at KX-1
  R a_acl = R(0.0);
#pragma unroll
  for (int k = 0; k < KX - 1; ++k)
    a_acl += sel(((S >> k) & 1u) != 0u, a_t22[k], R(0.0));
  g.clstr += a_t22[KX - 1] * p.albcls;
  g.cloudc += sel(a.icltop < KX, a_acl * p.albcl, R(0.0));
}

// ---------------------------------------------------------------- vertical diffusion
template <typename R, int KX>
SPD_HD void vdiff_adj(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, const SpeedyParams& p, const Uniforms<R>& u,
                      const ColumnCt<R, KX>& ct, ColumnAdj<R, KX>& g) {
  constexpr int NL1 = KX - 1;
  const int icnv = KX - a.iptop - 1;
  // super-adiabatic damping: tt[k] += fse[k] * rsig[k]; tt[k+1] -= sum_{j<=k} fse[j] * rsig1[j]
  R suf = R(0.0);
#pragma unroll
  for (int k = NL1 - 1; k >= 0; --k) {
    suf = suf + ct.dt[k + 1];
    const R se0 = a.se[k + 1] - p.segrad * (c.PHI[k + 1] - c.PHI[k]);
    const R a_fse = ct.dt[k] * u.rsig[k] - suf * u.rsig1[k];
    const R a_x = sel(a.se[k] < se0, a_fse * u.fvdise, R(0.0));
    g.se[k + 1] += a_x;
    g.se[k] += -a_x;
  }
  // moisture diffusion above the PBL
#pragma unroll
  for (int k = 2; k < KX - 2; ++k) {
    const R d = a.rh[k + 1] - a.rh[k];
    const bool on = (d >= u.vd_drh0[k]) & (((u.vd_on >> k) & 1u) != 0u);
    const R a_fq = (ct.dq[k] * u.rsig[k] - ct.dq[k + 1] * u.rsig[k + 1]) * u.vd_fq[k];
    add_if(on, g.qsat[k], a_fq, d);
    const R a_d = sel(on, a_fq * a.qsat[k], R(0.0));
    g.rh[k + 1] += a_d;
    g.rh[k] += -a_d;
  }
  // shallow convection / PBL moisture exchange between the two lowest levels
  const R dmse = a.se[KX - 1] - a.se[NL1 - 1] + R(ALHC) * (c.Q[KX - 1] - a.qsat[NL1 - 1]);
  const R drh = a.rh[KX - 1] - a.rh[NL1 - 1];
  const bool up = dmse >= R(0.0);
  const R fcnv = sel((icnv > 0) & up, R(p.redshc), R(1.0));
  const R rsA = u.rsig[NL1 - 1], rsB = u.rsig[KX - 1];
  const R a_fq2 = ct.dq[NL1 - 1] * rsA - ct.dq[KX - 1] * rsB;
  const R a_dmse = sel(up, (ct.dt[NL1 - 1] * rsA - ct.dt[KX - 1] * rsB) * fcnv * u.fshcse, R(0.0));
  const bool mix_up = up & (drh >= R(0.0)), mix_dn = !up & (drh > u.drh0);
  const R a_up = a_fq2 * fcnv * u.fshcq, a_dn = a_fq2 * u.fvdiq2;
  add_if(mix_up, g.qsat[KX - 1], a_up, drh);
  add_if(mix_dn, g.qsat[NL1 - 1], a_dn, drh);
  const R a_drh = sel(mix_up, a_up * a.qsat[KX - 1], sel(mix_dn, a_dn * a.qsat[NL1 - 1], R(0.0)));
  g.se[KX - 1] += a_dmse;
  g.se[NL1 - 1] += -a_dmse;
  g.Q[KX - 1] += a_dmse * R(ALHC);
  g.qsat[NL1 - 1] += -a_dmse * R(ALHC);
  g.rh[KX - 1] += a_drh;
  g.rh[NL1 - 1] += -a_drh;
}

// ---------------------------------------------------------------- clouds
template <typename R, int KX>
SPD_HD void clouds_adj(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, const SpeedyParams& p,
                       const Uniforms<R>& u, const CloudTape<R, KX>& t, ColumnAdj<R, KX>& g) {
  const R fm = c.fmask;
  R a_cl0 = g.clstr * (R(1.0) - fm);
  const R a_cll = g.clstr * fm;
  g.rh[KX - 1] += a_cll * mmax(t.clstr0, R(p.clsminl));
  a_cl0 += a_cll * a.rh[KX - 1] * dmax_x(t.clstr0, R(p.clsminl));
  const R a_fstab = a_cl0 * mmax(t.clsx, R(0.0));
  const R a_clsx = a_cl0 * t.fstab * dmax_x(t.clsx, R(0.0));
  const R a_cc = g.cloudc - R(1.2) * a_clsx;
  const R a_fsa = a_fstab * dmin_x(mmax(t.fstab_arg, R(0.0)), R(1.0)) * dmax_x(t.fstab_arg, R(0.0));
  const R a_gse = a_fsa * u.rgse;
  const R rdphi = mdiv(R(1.0), c.PHI[KX - 2] - c.PHI[KX - 1]);
  g.se[KX - 2] += a_gse * rdphi;
  g.se[KX - 1] += -a_gse * rdphi;
  g.Q[KX - 2] += g.qcloud;
  const R a_raw = a_cc * dmin_x(t.ccraw, R(1.0));
  const R mx = mmax(R(EPS), t.pr1);
  const R a_pr1 = a_raw * p.wpcl * mdiv(R(0.5), msqrt_1ulp(mx)) * dmax_x(t.pr1, R(EPS));
  const R a_sum = a_pr1 * dmin_x(R(86.4) * (a.precnv + a.precls), R(p.pmaxcl)) * R(86.4);
  g.precnv += a_sum;
  g.precls += a_sum;
  const R a_cmax = a_raw * R(2.0) * t.cl2 * dmin_x(t.cmax * u.rrcl, R(1.0)) * u.rrcl;
  // jnp.max over levels 2..KX-3: the gradient is shared evenly by the tied entries
  int nt = 0;
#pragma unroll
  for (int k = 2; k <= KX - 3; ++k) nt += (t.cu[k] == t.cmax) ? 1 : 0;
  const R share = mdiv(a_cmax, R(nt > 0 ? nt : 1));
  R a_cc0 = R(0.0);
#pragma unroll
  for (int k = 2; k <= KX - 3; ++k) {
    const R part = sel(t.cu[k] == t.cmax, share, R(0.0));
    const bool own = ((t.mk >> k) & 1u) != 0u;
    g.rh[k] += sel(own, part, R(0.0));
    a_cc0 += sel(own, R(0.0), part);
  }
  g.rh[KX - 2] += sel(t.m0, a_cc0, R(0.0));
}

// ---------------------------------------------------------------- condensation
template <typename R, int KX>
SPD_HD void condensation_adj(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, const Uniforms<R>& u,
                             const ColumnCt<R, KX>& ct, ColumnAdj<R, KX>& g) {
  const R ps = c.ps;
  const R psa2 = ps * ps;
  R qlsc[KX];
#pragma unroll
  for (int k = 1; k < KX; ++k) {
    const R dqa = u.rhref[k] * a.qsat[k] - c.Q[k];
    qlsc[k] = sel(dqa < R(0.0), dqa * u.rtlsc, R(0.0));
  }
  R sum = R(0.0);
#pragma unroll
  for (int k = 1; k < KX; ++k) sum = (k == 1) ? u.pfact[k] * qlsc[k] : sum + u.pfact[k] * qlsc[k];
  g.ps += g.precls * (R(0.0) - sum);
  const R a_sum = -g.precls * ps;
  R a_psa2 = R(0.0);
#pragma unroll
  for (int k = 1; k < KX; ++k) {
    const R dqa = u.rhref[k] * a.qsat[k] - c.Q[k];
    const bool on = dqa < R(0.0);
    const R dq = qlsc[k];
    const R cap = u.dqmax[k] * psa2;
    const R a_m = ct.dt[k] * R(TFACT);
    const R a_dq = ct.dq[k] + a_sum * u.pfact[k] - a_m * dmin_x(-dq, cap);
    a_psa2 += sel(on, a_m * dmin_x(cap, -dq) * u.dqmax[k], R(0.0));
    const R a_dqa = sel(on, a_dq * u.rtlsc, R(0.0));
    g.qsat[k] += a_dqa * u.rhref[k];
    g.Q[k] += -a_dqa;
    add_if(on, g.prm[VJP_RHLSC], a_dqa * a.qsat[k], u.rhref_d[k]);
  }
  g.ps += a_psa2 * R(2.0) * ps;
}

// ---------------------------------------------------------------- convection
template <typename R, int KX>
SPD_HD void convection_adj(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, const SpeedyParams& p,
                           const SpeedyVertical& v, const Uniforms<R>& u, const ConvTape<R, KX>& t,
                           const ColumnCt<R, KX>& ct, ColumnAdj<R, KX>& g) {
  const int iptop = a.iptop_conv;
  const R ps = c.ps;
  const R rps = mdiv(R(1.0), ps);
  R a_dfse[KX], a_dfqa[KX];
  a_dfse[0] = ct.dt[0];
  a_dfqa[0] = ct.dq[0];
#pragma unroll
  for (int k = 1; k < KX; ++k) {
    a_dfse[k] = ct.dt[k] * rps * v.grdscp[k];
    a_dfqa[k] = ct.dq[k] * rps * v.grdsig[k];
    g.rps += ct.dt[k] * t.dfse[k] * v.grdscp[k] + ct.dq[k] * t.dfqa[k] * v.grdsig[k];
  }
  // top layer: dfse[iptop-1] = top_s, dfqa[iptop-1] = top_q overwrite the fluxes
  R a_top_s = R(0.0), a_top_q = R(0.0);
#pragma unroll
  for (int k = 0; k < KX; ++k)
  {
    const bool at = iptop - 1 == k;
    a_top_s = sel(at, a_dfse[k], a_top_s);
    a_top_q = sel(at, a_dfqa[k], a_top_q);
    a_dfse[k] = sel(at, R(0.0), a_dfse[k]);
    a_dfqa[k] = sel(at, R(0.0), a_dfqa[k]);
  }
  R a_fm_t = R(0.0), a_fus_t = a_top_s, a_fds_t = -a_top_s, a_fuq_t = a_top_q, a_fdq_t = -a_top_q;
  {
    const R a_pr = g.precnv + R(ALHC) * a_top_s - a_top_q;
    const R P = t.fuq_t - t.fm_t * t.qsatb;
    const R a_P = a_pr * dmax_x(P, R(0.0));
    a_fuq_t += a_P;
    a_fm_t += -a_P * t.qsatb;
    const R a_qsatb = -a_P * t.fm_t;
#pragma unroll
    for (int k = 0; k < KX - 1; ++k) {
      const R aq = sel(iptop - 1 == k, a_qsatb, R(0.0));
      g.qsat[k] += aq * (R(1.0) - u.wvi1[k]);
      g.qsat[k + 1] += aq * u.wvi1[k];
    }
  }
  R a_FM[KX], a_FUS[KX], a_FUQ[KX], a_FDS[KX], a_FDQ[KX];
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    const bool top = iptop == k;
    a_FM[k] = top ? a_fm_t : R(0.0);
    a_FUS[k] = top ? a_fus_t : R(0.0);
    a_FUQ[k] = top ? a_fuq_t : R(0.0);
    a_FDS[k] = top ? a_fds_t : R(0.0);
    a_FDQ[k] = top ? a_fdq_t : R(0.0);
  }
  // secondary moisture flux and the flux differences
  R a_cbmf = R(0.0);
#pragma unroll
  for (int k = 0; k < KX - 1; ++k) {
    const R a_fsq = a_dfqa[k] - a_dfqa[KX - 1];
    const bool dry = t.delq[k] > R(0.0);
    const R a_s = a_fsq * p.smf;
    add_if(dry, a_cbmf, a_s, t.delq[k]);
    const R a_delq = sel(dry, a_s * a.cbmf, R(0.0));
    g.qsat[k] += a_delq * p.rhil;
    g.Q[k] += -a_delq;
    const R as = sel(k >= iptop, a_dfse[k], R(0.0)), aq = sel(k >= iptop, a_dfqa[k], R(0.0));
    a_FUS[k + 1] += as; a_FDS[k + 1] += -as;
    a_FUS[k] += -as; a_FDS[k] += as;
    a_FUQ[k + 1] += aq; a_FDQ[k + 1] += -aq;
    a_FUQ[k] += -aq; a_FDQ[k] += aq;
  }
  R a_fds = a_dfse[KX - 1] + a_FDS[KX - 1], a_fus = -a_dfse[KX - 1];
  R a_fdq = a_dfqa[KX - 1] + a_FDQ[KX - 1], a_fuq = -a_dfqa[KX - 1];
  R a_sbh[KX], a_qbh[KX];
  R a_fmass = R(0.0);
  a_sbh[0] = R(0.0); a_qbh[0] = R(0.0);
#pragma unroll
  for (int k = 0; k < KX - 1; ++k) {
    a_FM[k] += a_FDS[k] * t.sbh[k] + a_FDQ[k] * t.qbh[k];
    a_sbh[k] = a_FDS[k] * t.FM[k];
    a_qbh[k] = a_FDQ[k] * t.FM[k];
  }
  a_sbh[KX - 1] = R(0.0); a_qbh[KX - 1] = R(0.0);
  // cumulative sums from the bottom: FM[k] = fmass + sum_{j>=k} en[j], ...
  {
    R pm = R(0.0), pS = R(0.0), pQ = R(0.0);
#pragma unroll
    for (int j = 0; j < KX; ++j) {
      pm = pm + a_FM[j];
      pS = pS + a_FUS[j];
      pQ = pQ + a_FUQ[j];
      const R a_en = pm + pS * a.se[j] + pQ * c.Q[j];
      g.se[j] += pS * t.en[j];
      g.Q[j] += pQ * t.en[j];
      if (j >= 1 && j <= KX - 2) {
        const R ae = a_en * u.entr[j];
        add_if(j >= iptop, g.ps, ae, a.cbmf);
        add_if(j >= iptop, a_cbmf, ae, ps);
      }
    }
    a_fmass += pm;
    a_fus += pS;
    a_fuq += pQ;
  }
  // fus = fmass*se[KX-1], fuq = fmass*qmax, fds = fmass*sb, fdq = fmass*qb
  a_fmass += ((a_fus * a.se[KX - 1] + a_fuq * t.qmax) + a_fds * t.sb) + a_fdq * t.qb;
  g.se[KX - 1] += a_fus * t.fmass;
  R a_qmax = a_fuq * t.fmass;
  const R a_sb = a_fds * t.fmass;
  R a_qb = a_fdq * t.fmass;
  a_fmass += sel(iptop < KX, a_cbmf, R(0.0));
  // fmass = fm0 * fpsa * min(5, qdif / (qmax - qb))
  R a_qdif;
  {
    const R den = t.qmax - t.qb;
    const R ratio = mdiv(t.qdif, den);
    const R m = mmin(R(5.0), ratio);
    const R a_fpsa = a_fmass * u.fm0 * m;
    const R a_fm0 = a_fmass * t.fpsa * m;
    const R a_ratio = a_fmass * u.fm0 * t.fpsa * dmin_x(ratio, R(5.0));
    a_qdif = mdiv(a_ratio, den);
    const R a_den = mdiv(-a_ratio * ratio, den);
    a_qmax += a_den;
    a_qb += -a_den;
    g.prm[VJP_TRCNV] += a_fm0 * (-mdiv(u.fm0, R(p.trcnv)));
    const R y = (ps - p.psmin) * u.rdps;
    g.ps += a_fpsa * mmin(R(1.0), y) + a_fpsa * ps * dmin_x(y, R(1.0)) * u.rdps;
  }
  // qb = min(qbh[KX-1], Q[KX-1]); sb = sbh[KX-1]
  a_qbh[KX - 1] += a_qb * dmin_x(t.qbh[KX - 1], c.Q[KX - 1]);
  g.Q[KX - 1] += a_qb * dmin_x(c.Q[KX - 1], t.qbh[KX - 1]);
  a_sbh[KX - 1] += a_sb;
#pragma unroll
  for (int k = 1; k < KX; ++k) {
    const R w = u.wvi1[k - 1];
    g.se[k - 1] += a_sbh[k] * (R(1.0) - w);
    g.se[k] += a_sbh[k] * w;
    g.Q[k - 1] += a_qbh[k] * (R(1.0) - w);
    g.Q[k] += a_qbh[k] * w;
  }
  // qmax = max(1.01 Q[KX-1], qsat[KX-1])
  {
    const R q1 = R(1.01) * c.Q[KX - 1];
    g.Q[KX - 1] += a_qmax * R(1.01) * dmax_x(q1, a.qsat[KX - 1]);
    g.qsat[KX - 1] += a_qmax * dmax_x(a.qsat[KX - 1], q1);
  }
  // qdif (diagnose_convection)
  const R A = c.Q[KX - 1] - t.qthr0;
  const R B = (t.mse0 - t.msthr) * R(RLHC);
  const R a_A = sel(t.case1, a_qdif * dmax_x(A, B), sel(t.case2, a_qdif, R(0.0)));
  const R a_B = sel(t.case1, a_qdif * dmax_x(B, A), R(0.0));
  g.Q[KX - 1] += a_A;
  const R a_qthr0 = -a_A, a_mse0 = a_B * R(RLHC), a_msthr = -a_B * R(RLHC);
  g.prm[VJP_RHBL] += a_qthr0 * a.qsat[KX - 1];
  g.qsat[KX - 1] += a_qthr0 * p.rhbl;
  g.se[KX - 1] += a_mse0;
  g.Q[KX - 1] += a_mse0 * R(ALHC);
#pragma unroll
  for (int k = 2; k <= KX - 4; ++k) {   // msthr = mss2[k] at k = ktop2 - 1, mss = se + alhc * qsat
    const R w = u.wvi1[k];
    const R am = sel(t.ktop2 == k + 1, a_msthr, R(0.0));
    const R am0 = am * (R(1.0) - w), am1 = am * w;
    g.se[k] += am0;
    g.qsat[k] += am0 * R(ALHC);
    g.se[k + 1] += am1;
    g.qsat[k + 1] += am1 * R(ALHC);
  }
}

// humidity, static energy and 1/ps back to the state.
template <typename R, int KX>
SPD_HD void humidity_adj(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, ColumnAdj<R, KX>& g) {
  const R rps = mrcp(c.ps);
  R a_psq = R(0.0);
#pragma unroll
  for (int k = 0; k < KX; ++k) {
    const R a_q = g.rh[k] * mrcp(a.qsat[k]);   // rh = Q / qsat
    g.Q[k] += a_q;
    const R a_qs = g.qsat[k] - a_q * a.rh[k];
    R dqt, dqp;
    qsat_grad(c.T[k], a.qsat[k], dqt, dqp);
    g.T[k] += a_qs * dqt + R(CP) * g.se[k];
    a_psq += a_qs * dqp;
  }
  g.ps += a_psq * rps - g.rps * rps * rps;
}

// Per-column storage for the longwave flux tapes between a term's recompute and
// its reversal: a plain array on the host; LDS on the GPU (speedy_kernels.hip).
template <typename R, int N>
struct ArrayStore {
  R v[N];
  SPD_HD void put(int i, R x) { v[i] = x; }
  SPD_HD R get(int i) const { return v[i]; }
  SPD_HD ArrayStore& after(R) { return *this; }
};

// What phase b2 hands from its forward to its reversal.
template <typename R, int KX>
struct VjpTapeB {
  SwTape<R, KX> sw;
  SfcTape<R> sf;
  R aF[4];       // adjoint of the upward longwave fluxes at the surface
};

// Forward + VJP of phase b1: the forward of phase_b1 (b.dfl, b.rlds, albedos, vertical
// diffusion) with the longwave's down sweep.  Clears g.
template <typename R, int KX, class Store>
SPD_HD void phase_b1_vjp(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, const SpeedyParams& p,
                         const SpeedyVertical& v, const Uniforms<R>& u, const ColumnCt<R, KX>& ct, PhaseB<R, KX>& b,
                         ColumnAdj<R, KX>& g, VjpTapeB<R, KX>& t, Store& tape) {
  adj_zero<R, KX>(g);
  albedos<R, KX>(c, p, b);
  lw_down_vjp<R, KX>(c, a, p, v, u, ct, b, tape, t.aF);
  vdiff<R, KX>(c, a, p, u, b);
}

// The forward of the shortwave and the surface fluxes, with their tapes.
template <typename R, int KX>
SPD_HD void phase_b2_taped(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, uint32_t S, const SpeedyParams& p,
                           const SpeedyVertical& v, const Uniforms<R>& u, uint32_t flags, const ColumnCt<R, KX>& ct,
                           PhaseB<R, KX>& b, ColumnAdj<R, KX>& g, VjpTapeB<R, KX>& t) {
  R flux_h[4];
  shortwave<R, KX, false>(c, a, S, p, v, u, b, flux_h, t.sw);
#pragma unroll
  for (int k = 0; k < KX; ++k)   // tsw[k] = dfabs[k] grdscp[k] / ps
    add_if(u.compute_sw != 0u, g.rps, ct.dt[k] * t.sw.dfabs[k], R(v.grdscp[k]));
  R tsfc;
  surface<R, KX, false>(c, a, p, v, u, flags, b, tsfc, t.sf);
  b.flux_h[0] = flux_h[0]; b.flux_h[1] = flux_h[1]; b.rlus2 = t.sf.rlus2; b.tsfc = tsfc;
}

// Reversal of the surface fluxes and the shortwave, then the longwave's up sweep
// (which also leaves the forward's b.tlw).  ct.dq as verify_ct left it.
template <typename R, int KX, class Store>
SPD_HD void phase_b2_vjp(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, uint32_t S, const SpeedyParams& p,
                         const SpeedyVertical& v, const Uniforms<R>& u, const ColumnCt<R, KX>& ct, PhaseB<R, KX>& b,
                         ColumnAdj<R, KX>& g, const VjpTapeB<R, KX>& t, Store& tape) {
  R a_rlus2, a_flux_h[2], a_rsds = R(0.0), a_rlds = R(0.0);
  lw_surface_adj<R, KX>(u, p, b.tsfc, dfl_ct<R, KX>(ct, v, KX - 1, mdiv(R(1.0), c.ps)), t.aF, a_rlus2, a_flux_h);
  surface_adj<R, KX>(c, a, b, p, v, u, t.sf, ct, a_rlus2, a_rsds, a_rlds, g);
  shortwave_adj<R, KX>(c, a, b, S, p, v, u, t.sw, ct, a_flux_h, a_rsds, g);
  lw_up_vjp<R, KX>(c, a, p, v, u, b, tape, ct, a_rlds, g);
}

// Reversal of vertical diffusion and phase A.  The cloud and convection
// intermediates are recomputed (376 of the forward's 2842 instructions; keeping them
// would hold about 70 values across phase B).
template <typename R, int KX>
SPD_HD void phase_a_adj(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, const SpeedyParams& p,
                        const SpeedyVertical& v, const Uniforms<R>& u, const ColumnCt<R, KX>& ct,
                        ColumnAdj<R, KX>& g) {
  vdiff_adj<R, KX>(c, a, p, u, ct, g);
  settle_adj<R, KX>(g);
  {
    PhaseA<R, KX> aa = a;
    CloudTape<R, KX> t;
    clouds<R, KX>(c, p, u, aa, t);
    clouds_adj<R, KX>(c, a, p, u, t, g);
    settle_adj<R, KX>(g);
  }
  condensation_adj<R, KX>(c, a, u, ct, g);
  settle_adj<R, KX>(g);
  {
    PhaseA<R, KX> aa = a;
    ConvTape<R, KX> t;
    convection<R, KX>(c, p, v, u, aa, t);
    convection_adj<R, KX>(c, a, p, v, u, t, ct, g);
  }
  humidity_adj<R, KX>(c, a, g);
}

// The whole column from the forward's phase A: the gradients into g (the forward of
// phase B is evaluated again; the kernels run the pieces above in place of it).
template <typename R, int KX, class Store>
SPD_HD void column_vjp(const ColumnIn<R, KX>& c, const PhaseA<R, KX>& a, const PhaseB<R, KX>&, uint32_t S,
                       const SpeedyParams& p, const SpeedyVertical& v, const Uniforms<R>& u, uint32_t flags,
                       const ColumnCt<R, KX>& ct, ColumnAdj<R, KX>& g, Store& tape) {
  PhaseB<R, KX> b;
  VjpTapeB<R, KX> t;
  phase_b1_vjp<R, KX>(c, a, p, v, u, ct, b, g, t, tape);
  phase_b2_taped<R, KX>(c, a, S, p, v, u, flags, ct, b, g, t);
  phase_b2_vjp<R, KX>(c, a, S, p, v, u, ct, b, g, t, tape);
  phase_a_adj<R, KX>(c, a, p, v, u, ct, g);
}

}  // namespace speedy
