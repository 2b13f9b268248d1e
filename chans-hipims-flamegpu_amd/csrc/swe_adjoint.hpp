// Reverse-mode derivatives of the step's physics (no counterpart in the
// reference).  Each function recomputes the forward expression of
// swe_physics.hpp with its branch decisions (minmod selections, wet/dry
// tests, clamps, HLLC region, friction limiter) and propagates cotangents
// back through the branch that was taken, so the result is the exact
// derivative of the forward map wherever that map is differentiable.
// Bed elevation is static and the time step is frozen, so neither gets a
// cotangent.
#pragma once

#include "swe_physics.hpp"

namespace hp {

template <class T> struct FrameAdj {
  T h, qn, qt;
};

template <class T> __host__ __device__ inline FrameAdj<T> zero_adj() {
  FrameAdj<T> a;
  a.h = T(0); a.qn = T(0); a.qt = T(0);
  return a;
}

// v where on, else 0 (a select; v may be anything where it is dropped).
template <class T> __host__ __device__ inline T only(bool on, T v) { return on ? v : T(0); }

// Cotangent of e = c + 0.5 * minmod(c - l, r - c) pushed to (c, l, r): half of
// it goes to the two cells of the difference that minmod returned, if any.
template <class T> __host__ __device__ inline void muscl_adj(T c, T l, T r, T a_e, T& a_c, T& a_l, T& a_r) {
  const T x = c - l, y = r - c, m = T(0.5) * a_e;
  const bool some = x * y > T(0), first = fabs(x) < fabs(y);
  const T mx = only(both(some, first), m), my = only(both(some, !first), m);
  a_c += a_e + (mx - my);
  a_l -= mx;
  a_r += my;
}

// VJP of solve_edge (swe_physics.hpp) with cotangents (v_fh, v_fn, v_ft,
// v_bc, v_br) of its five scaled outputs.  Accumulates into the cotangents of
// c, l, r, rr (h, qn, qt) and of the two water levels.  Returns whether the
// edge was active.
template <class T, int ORDER>
__host__ __device__ inline bool solve_edge_vjp(const FrameCell<T>& c, const FrameCell<T>& l, const FrameCell<T>& r,
                                               const FrameCell<T>& rr, bool r_is_ghost, T etaC, T etaR, T dx, T dt,
                                               T v_fh, T v_fn, T v_ft, T v_bc, T v_br, FrameAdj<T>& ac,
                                               FrameAdj<T>& al, FrameAdj<T>& ar, FrameAdj<T>& arr, T& a_etaC,
                                               T& a_etaR, bool frozen_slopes = false) {
  using P = Prec<T>;
  const T g = T(kG);
  if (lt_hs(c.h) && lt_hs(r.h)) return false;

  // ---- forward: edge states ----
  FrameCell<T> eL, eR;
  bool zeroL = false, zeroR = false;
  if (ORDER == 1 || r_is_ghost) {
    eL = c;
    eR = r;
    if (ORDER == 1 && !r_is_ghost) {
      const T zl = eL.z + T(0.5) * Prec<T>::limit(c.z - l.z, r.z - c.z);
      const T zr = eR.z + T(0.5) * Prec<T>::limit(r.z - rr.z, c.z - r.z);
      eL.z = gt_hs(r.h) ? zl : eL.z;
      eR.z = gt_hs(c.h) ? zr : eR.z;
    }
  } else {
    eL.h = c.h + T(0.5) * Prec<T>::limit(c.h - l.h, r.h - c.h);
    eL.z = c.z + T(0.5) * Prec<T>::limit(c.z - l.z, r.z - c.z);
    eR.h = r.h + T(0.5) * Prec<T>::limit(r.h - rr.h, c.h - r.h);
    eR.z = r.z + T(0.5) * Prec<T>::limit(r.z - rr.z, c.z - r.z);
    zeroL = lt_hs(c.h);
    zeroR = lt_hs(r.h);
    const T nL = c.qn + T(0.5) * Prec<T>::limit(c.qn - l.qn, r.qn - c.qn);
    const T tL = c.qt + T(0.5) * Prec<T>::limit(c.qt - l.qt, r.qt - c.qt);
    const T nR = r.qn + T(0.5) * Prec<T>::limit(r.qn - rr.qn, c.qn - r.qn);
    const T tR = r.qt + T(0.5) * Prec<T>::limit(r.qt - rr.qt, c.qt - r.qt);
    eL.qn = only(!zeroL, nL);
    eL.qt = only(!zeroL, tL);
    eR.qn = only(!zeroR, nR);
    eR.qt = only(!zeroR, tR);
  }
  // From here on straight-line code with selects, as in hllc_edge: the
  // branches of the forward step become masks on the cotangents, and what a
  // mask drops may hold anything.  (With the branches, a wave whose edges fell
  // in different regions ran each in turn and copied some twenty values at
  // every join: 62 -> 52.8 us per reverse step of 1024^2 cells, order 1, float.)
  // ---- forward: velocities and hydrostatic reconstruction ----
  const bool dryL0 = lt_hs(eL.h), dryR0 = lt_hs(eR.h);
  const T rhL = P::div(T(1), eL.h), rhR = P::div(T(1), eR.h);  // as hllc_edge forms them
  const T uL0 = dryL0 ? T(0) : mul_alone(eL.qn, rhL), vL0 = dryL0 ? T(0) : mul_alone(eL.qt, rhL);
  const T uR0 = dryR0 ? T(0) : mul_alone(eR.qn, rhR), vR0 = dryR0 ? T(0) : mul_alone(eR.qt, rhR);
  const T wL0 = eL.h + eL.z, wR0 = eR.h + eR.z;
  const bool maxC = etaC >= etaR;  // fmax(etaC, etaR) took etaC
  const bool minC = etaC <= etaR;  // fmin(etaC, etaR) took etaC
  const T emax = maxC ? etaC : etaR, emin = minC ? etaC : etaR;
  const bool L1a = wL0 <= emax, R1a = wR0 <= emax;
  const T wL1 = L1a ? wL0 : emax, wR1 = R1a ? wR0 : emax;
  const bool L2a = wL1 >= emin, R2a = wR1 >= emin;
  const T wL2 = L2a ? wL1 : emin, wR2 = R2a ? wR1 : emin;
  T wL3 = wL2, wR3 = wR2;
  bool avg = false, liftL = false, takeL = false;
  if (ORDER == 1) {
    avg = (etaC - etaR) * (wL2 - wR2) < T(0);
    const T m = (wL2 + wR2) / T(2);
    wL3 = avg ? m : wL2;
    wR3 = avg ? m : wR2;
  } else {
    liftL = etaC > etaR;
    takeL = wL2 >= wR2;
    const T m = takeL ? wL2 : wR2;
    wL3 = liftL ? m : wL2;
    wR3 = liftL ? wR2 : m;
  }
  const T zL0 = wL3 - eL.h, zR0 = wR3 - eR.h;
  const bool zbL = zL0 >= zR0;
  const T zbm = zbL ? zL0 : zR0;
  const T dL = wL3 - zbm, dR = wR3 - zbm;
  const bool posL = dL > T(0), posR = dR > T(0);
  const T hL = only(posL, dL), hR = only(posR, dR);
  const T zL = wL3 - hL, zR = wR3 - hR;
  const bool flux_on = !both(lt_hs(hL), lt_hs(hR));

  const T s = dt / dx;
  const T Gb = T(0.5) * g * s;
  // ---- reverse: bed terms ----
  T a_hL = v_bc * Gb * (zL - c.z), a_zL = v_bc * Gb * (hL + c.h);
  ac.h += v_bc * Gb * (zL - c.z);
  T a_hR = v_br * Gb * (zR - r.z), a_zR = v_br * Gb * (hR + r.h);
  ar.h += v_br * Gb * (zR - r.z);

  // ---- reverse: HLLC ----
  const T qnL = uL0 * hL, qtL = vL0 * hL, qnR = uR0 * hR, qtR = vR0 * hR;
  const T aL = P::sqrt_(g * hL), aR = P::sqrt_(g * hR);
  const T base = (aL + aR) / T(2) + (uL0 - uR0) / T(4);
  const T u_star = (uL0 + uR0) / T(2) + aL - aR;
  const T a_star = P::star_celerity(base, g);
  const bool sLdry = le_hs(hL), sRdry = le_hs(hR);
  const T x1 = uL0 - aL, x2 = u_star - a_star;
  const T y1 = uR0 + aR, y2 = u_star + a_star;
  const bool sLx1 = x1 <= x2, sRy1 = y1 >= y2;
  const T sLd = uR0 - T(2) * aR, sLw = sLx1 ? x1 : x2;
  const T sRd = uL0 + T(2) * aL, sRw = sRy1 ? y1 : y2;
  const T sL = sLdry ? sLd : sLw, sR = sRdry ? sRd : sRw;
  // the sign of the contact speed, as hllc_edge takes it
  const T num = sL * hR * (uR0 - sR) - sR * hL * (uL0 - sL), den = hR * (uR0 - sR) - hL * (uL0 - sL);
  const T sM = P::quotient_sign(num, den);
  const bool left = T(0) <= sL, useL = both(sL < T(0), T(0) <= sM);
  const bool star = both(!left, either(useL, both(sM < T(0), T(0) <= sR)));
  const bool inL = both(flux_on, left), inS = both(flux_on, star), inR = both(flux_on, !either(left, star));
  const T b_fh = v_fh * s, b_fn = v_fn * s, b_ft = v_ft * s;
  // the outer regions: the flux of one side
  const T lh = only(inL, b_fh), ln = only(inL, b_fn), lt = only(inL, b_ft);
  const T rh = only(inR, b_fh), rn = only(inR, b_fn), rt = only(inR, b_ft);
  T a_qnL = lh + ln * uL0, a_qtL = lt * uL0, a_uL0 = ln * qnL + lt * qtL;
  T a_qnR = rh + rn * uR0, a_qtR = rt * uR0, a_uR0 = rn * qnR + rt * qtR;
  a_hL += ln * g * hL;
  a_hR += rn * g * hR;
  // the star region
  const T sh = only(inS, b_fh), sn = only(inS, b_fn), st = only(inS, b_ft);
  const T D = inS ? sR - sL : T(1), rD = P::div(T(1), D);
  const T dh = hR - hL, dq = qnR - qnL, sLR = sL * sR;
  const T qnfL = uL0 * qnL + T(0.5) * g * hL * hL;
  const T qnfR = uR0 * qnR + T(0.5) * g * hR * hR;
  const T fh = (sR * qnL - sL * qnR + sLR * dh) * rD, fn = (sR * qnfL - sL * qnfR + sLR * dq) * rD;
  const T vstar = useL ? vL0 : vR0;
  const T tot = sh + st * vstar;
  const T a_D = -(tot * fh + sn * fn) * rD, a_Nh = tot * rD, a_Nn = sn * rD;
  T a_vL0 = only(useL, st * fh), a_vR0 = only(!useL, st * fh);
  const T a_sL = a_Nh * (sR * dh - qnR) + a_Nn * (sR * dq - qnfR) - a_D;
  const T a_sR = a_Nh * (qnL + sL * dh) + a_Nn * (qnfL + sL * dq) + a_D;
  const T a_qnfL = a_Nn * sR, a_qnfR = -a_Nn * sL;
  a_qnL += a_Nh * sR - a_Nn * sLR + a_qnfL * uL0;
  a_qnR += a_Nn * sLR - a_Nh * sL + a_qnfR * uR0;
  a_hL += a_qnfL * g * hL - a_Nh * sLR;
  a_hR += a_qnfR * g * hR + a_Nh * sLR;
  a_uL0 += a_qnfL * qnL;
  a_uR0 += a_qnfR * qnR;
  // wave speeds
  const T sl_d = only(sLdry, a_sL), sl_x = only(both(!sLdry, sLx1), a_sL), sl_s = only(!either(sLdry, sLx1), a_sL);
  const T sr_d = only(sRdry, a_sR), sr_y = only(both(!sRdry, sRy1), a_sR), sr_s = only(!either(sRdry, sRy1), a_sR);
  const T a_ustar = sl_s + sr_s, a_astar = sr_s - sl_s;
  const T a_base = P::star_celerity_adj(base, g, a_star, a_astar);
  const T a_aL = T(2) * sr_d - sl_x + a_ustar + a_base / T(2);
  const T a_aR = sr_y - T(2) * sl_d - a_ustar + a_base / T(2);
  a_uL0 += sl_x + sr_d + a_ustar / T(2) + a_base / T(4);
  a_uR0 += sl_d + sr_y + a_ustar / T(2) - a_base / T(4);
  const T c_aL = P::div(a_aL * g, T(2) * aL), c_aR = P::div(a_aR * g, T(2) * aR);
  a_hL += only(aL > T(0), c_aL);
  a_hR += only(aR > T(0), c_aR);
  a_uL0 += a_qnL * hL;
  a_vL0 += a_qtL * hL;
  a_hL += a_qnL * uL0 + a_qtL * vL0;
  a_uR0 += a_qnR * hR;
  a_vR0 += a_qtR * hR;
  a_hR += a_qnR * uR0 + a_qtR * vR0;

  // ---- reverse: hydrostatic reconstruction ----
  a_hL -= a_zL;
  a_hR -= a_zR;
  const T pL = only(posL, a_hL), pR = only(posR, a_hR);
  const T a_zbm = -(pL + pR);
  const T a_zL0 = only(zbL, a_zbm), a_zR0 = only(!zbL, a_zbm);
  const T a_wL3 = a_zL + pL + a_zL0, a_wR3 = a_zR + pR + a_zR0;
  T a_eLh = -a_zL0, a_eRh = -a_zR0;
  T a_wL2, a_wR2;
  if (ORDER == 1) {
    const T m = (a_wL3 + a_wR3) / T(2);
    a_wL2 = avg ? m : a_wL3;
    a_wR2 = avg ? m : a_wR3;
  } else {
    // the lifted side took the higher of the two levels
    const T a_m = liftL ? a_wL3 : a_wR3;
    a_wL2 = only(!liftL, a_wL3) + only(takeL, a_m);
    a_wR2 = only(liftL, a_wR3) + only(!takeL, a_m);
  }
  const T a_emin = only(!L2a, a_wL2) + only(!R2a, a_wR2);
  const T a_wL1 = only(L2a, a_wL2), a_wR1 = only(R2a, a_wR2);
  const T a_emax = only(!L1a, a_wL1) + only(!R1a, a_wR1);
  const T a_wL0 = only(L1a, a_wL1), a_wR0 = only(R1a, a_wR1);
  a_etaC += only(maxC, a_emax) + only(minC, a_emin);
  a_etaR += only(!maxC, a_emax) + only(!minC, a_emin);
  a_eLh += a_wL0;
  a_eRh += a_wR0;
  T a_eLqn = a_uL0 * rhL, a_eLqt = a_vL0 * rhL, a_eRqn = a_uR0 * rhR, a_eRqt = a_vR0 * rhR;
  const T c_hL = (a_uL0 * uL0 + a_vL0 * vL0) * rhL, c_hR = (a_uR0 * uR0 + a_vR0 * vR0) * rhR;
  a_eLqn = only(!dryL0, a_eLqn);
  a_eLqt = only(!dryL0, a_eLqt);
  a_eLh -= only(!dryL0, c_hL);
  a_eRqn = only(!dryR0, a_eRqn);
  a_eRqt = only(!dryR0, a_eRqt);
  a_eRh -= only(!dryR0, c_hR);

  // ---- reverse: edge states ----
  if (ORDER == 1 || r_is_ghost || frozen_slopes) {
    // (with frozen slopes the limited slope terms are constants)
    if (ORDER == 2 && !r_is_ghost) {
      a_eLqn = only(!zeroL, a_eLqn);
      a_eLqt = only(!zeroL, a_eLqt);
      a_eRqn = only(!zeroR, a_eRqn);
      a_eRqt = only(!zeroR, a_eRqt);
    }
    ac.h += a_eLh; ac.qn += a_eLqn; ac.qt += a_eLqt;
    ar.h += a_eRh; ar.qn += a_eRqn; ar.qt += a_eRqt;
  } else {
    muscl_adj<T>(c.h, l.h, r.h, a_eLh, ac.h, al.h, ar.h);
    muscl_adj<T>(r.h, rr.h, c.h, a_eRh, ar.h, arr.h, ac.h);
    muscl_adj<T>(c.qn, l.qn, r.qn, only(!zeroL, a_eLqn), ac.qn, al.qn, ar.qn);
    muscl_adj<T>(c.qt, l.qt, r.qt, only(!zeroL, a_eLqt), ac.qt, al.qt, ar.qt);
    muscl_adj<T>(r.qn, rr.qn, c.qn, only(!zeroR, a_eRqn), ar.qn, arr.qn, ac.qn);
    muscl_adj<T>(r.qt, rr.qt, c.qt, only(!zeroR, a_eRqt), ar.qt, arr.qt, ac.qt);
  }
  return true;
}

// Cotangent of a boundary ghost (bc_ghost) and of its water level pushed to
// the cell it mirrors.  Given values are constants.
template <class T, int ORDER>
__host__ __device__ inline void ghost_adj(int type, int d, const FrameAdj<T>& ag, T a_etaG, FrameAdj<T>& ac) {
  T gh = T(0), gn = T(0), gt = T(0);  // d ghost / d cell for h, qn, qt
  switch (type) {
    case 3:
      gh = T(1);
      gn = (d == 0 || d == 2) ? T(-1) : T(1);
      gt = gn;
      break;
    case 4: gh = T(1); gn = T(-1); gt = T(1); break;
    case 6: gh = T(0); gn = T(1); gt = T(1); break;
    case 7: gh = T(1); gn = T(0); gt = T(0); break;
    case 8: gh = T(0); gn = T(1); gt = T(1); break;
    case 9: gh = T(0); gn = T(0); gt = T(0); break;
    default: gh = T(1); gn = T(1); gt = T(1); break;
  }
  ac.h += gh * ag.h;
  ac.qn += gn * ag.qn;
  ac.qt += gt * ag.qt;
  // water level of the ghost
  if (ORDER == 1) {
    ac.h += gh * a_etaG;  // h_g + z_g
  } else {
    switch (type) {
      case 6: break;                         // z + given depth
      case 7: ac.h += a_etaG; break;         // z + h_c
      case 8: break;                         // given level
      default: ac.h += a_etaG; break;        // the cell's own wl
    }
  }
}

// VJP of implicit_friction for one wet cell, in its cancellation-free form
// q' = 2 q / (1 + sqrt(1 + x)), x = 4 dt C_f |q| / h^2, C_f = g n^2 h^(-1/3),
// with the Froude limiter branch.  (qx, qy) are the momenta the friction
// acts on; (a_ox, a_oy) the cotangents of its outputs.  Adds the cotangents
// of qx, qy, h and n.
template <class T>
__host__ __device__ inline void friction_vjp(T h, T n, T dt, T qx, T qy, T a_ox, T a_oy, T& a_qx, T& a_qy, T& a_h,
                                             T& a_n) {
  const T g = T(kG);
  using P = Prec<T>;
  const T h13 = P::rcbrt_friction(h);
  const T C_f = g * n * n * h13;
  const T qn2 = qx * qx + qy * qy;
  const T q_norm = P::sqrt_(qn2);
  const T lim = T(5) * h * P::sqrt_(h * g);
  const T coef = P::div(T(4) * dt, h * h);
  const T x = coef * C_f * q_norm;
  const T S = P::sqrt_(T(1) + x);
  const T k = P::div(T(2), T(1) + S);
  // per component: q' = k q, past the Froude limit the reflected 2 q' - q
  // (nothing once that changes sign); |q| <= 1e-10 passes unchanged
  T a_k = T(0), aq[2];
  const T qc[2] = {qx, qy};
  const T ac_[2] = {a_ox, a_oy};
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const T q = qc[m], tmp = k * q, out = T(2) * tmp - q;
    const bool moves = fabs(q) > T(1.0e-10), over = fabs(tmp) > lim, clipped = both(over, out * tmp <= T(0));
    const bool live = both(moves, !clipped);
    const T twice = T(2) * ac_[m];
    const T a_tmp = only(live, over ? twice : ac_[m]);
    const T direct = only(both(live, over), -ac_[m]);
    a_k += a_tmp * q;
    aq[m] = (moves ? direct : ac_[m]) + a_tmp * k;
  }
  const T dk_dx = P::div(-T(1), (T(1) + S) * (T(1) + S) * S);
  const T a_x = a_k * dk_dx;
  const T a_Cf = a_x * coef * q_norm;
  const T a_qnorm = a_x * coef * C_f;
  const T over_q = P::div(a_qnorm, q_norm);
  const bool flows = q_norm > T(0);
  const T ax = aq[0] + only(flows, over_q * qx), ay = aq[1] + only(flows, over_q * qy);
  const T hx = P::div(a_x * (T(-2) * x) + a_Cf * (T(-1.0 / 3.0)) * C_f, h);
  const T nx = P::div(a_Cf * T(2) * C_f, n);
  const bool rough = n > T(0);  // without friction the momenta pass through
  a_qx += rough ? ax : a_ox;
  a_qy += rough ? ay : a_oy;
  a_h += only(rough, hx);
  a_n += only(rough, nx);
}

}  // namespace hp
