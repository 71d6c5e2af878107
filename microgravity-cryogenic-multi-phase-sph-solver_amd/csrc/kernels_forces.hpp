// Forces pass on gfx950: transport velocity, momentum with wall loads, CSF or
// Akinci, continuity, conduction and the dt maxima in one walk of each fluid
// particle's neighbour list (SPH_kernels.cu:56-104,162-203,
// navier_stokes.cu:121-245, surface_tension.cu:120-213,
// phase_change.cu:31-75, sph_solver.cu:62-99).  Compiled once per tension
// model (kernels_forces_none / _csf / _akinci.hip).
#pragma once

#include <algorithm>
#include <stdexcept>

#include "pair_lanes.hpp"

namespace cryo {
namespace {

__host__ __device__ inline bool forces_need_vt(const SimParams& P, bool continuity) {
  return (P.tvf && P.tvf_stress) || (continuity && P.tvf);
}

struct Maxima {
  float v = 0.0f, a = 0.0f, tv = 0.0f, nu = 0.0f, sp = 0.0f;
};

// One neighbour's record in registers (t only where the pass needs it).
struct PairData {
  float4 x, q, v, t;
  V3 lo;  // KS: the position's low-order part
};

// What one pair adds to its target's sums, each term to be added once, in the
// order of the members (zero where the pair has no such term: a zero added to
// a running sum that starts at +0 never changes it).
template <bool KS>
struct PairTerms {
  V3 f1{0, 0, 0}, fs{0, 0, 0}, f2{0, 0, 0};  // force: pressure, transport stress, viscous
  V3 a1{0, 0, 0}, a2{0, 0, 0}, a3{0, 0, 0};  // acceleration: wall guard (two; KS only), artificial viscosity
  V3 t{0, 0, 0};                             // transport velocity
  V3 xj{0, 0, 0};                            // a wall's position
  V3 dF{0, 0, 0}, dM{0, 0, 0};               // KS: a wall's load and moment
  V3 G{0, 0, 0}, ak{0, 0, 0};                // balanced CSF, Akinci
  float num = 0.0f, den = 0.0f;              // curvature
  float div = 0.0f, diff = 0.0f, q = 0.0f;   // continuity, conduction
  bool wall = false, guard = false;
};

// Momentum, wall loads, transport velocity, CSF / Akinci, continuity and
// conduction rates of one fluid particle: its constants, one pair, the sums.
// ST: 0 no tension pass, 1 CSF with vapour present, 2 Akinci.
// OPT: any of the transport stress, balanced CSF and SPS is on (compiled out of
// the common instances: their terms would hold registers).
template <int ST, bool CONT, bool THERMAL, bool KS, bool OPT>
struct ForcesTarget {
  static constexpr bool kCsf = ST == 1, kAkinci = ST == 2;
  int i, pi_idx;
  uint8_t ph;
  V3 xi, li, vi, dvi, origin, ni, nak, vci;
  float dt_now, mi, rhoi, Ti, Vi, p_i, ci, Vt, etai, alpha_i, k_same, k_other;
  bool tvf_on, csf_on, ak_on;
  // what the fast pairs met: the smallest r2, the smallest non-zero numerator
  float r2_low;
  uint32_t x_low;
  // sums
  AccV3<KS> force, acc_av, sum_t, fwall, mwall, Gs, acc_ak;
  Acc<KS> num, den, div, diff, q;

  __device__ inline void reset() {
    r2_low = 1.0f;
    x_low = ~0u;
    force = acc_av = sum_t = fwall = mwall = Gs = acc_ak = AccV3<KS>{};
    num = den = div = diff = q = Acc<KS>{};
  }

  __device__ ForcesTarget(const PV& pv, const SimParams& P, const DevState* st, int i_) : i(i_) {
    const PairRec r = pv.t.rec[i];
    ph = static_cast<uint8_t>(__float_as_int(r.x.w));
    dt_now = uniform(st->dt);
    origin = V3{uniform(st->origin.x), uniform(st->origin.y), uniform(st->origin.z)};
    pi_idx = pidx(ph);
    xi = ld3(r.x);
    li = pos_lo<KS>(pv.s.xlo, i);
    vi = ld3(r.v);
    dvi = OPT ? ld3(r.t) - vi : V3{0, 0, 0};
    p_i = r.q.x;
    mi = r.q.y;
    rhoi = r.q.z;
    Ti = r.q.w;
    Vi = r.v.w;
    ci = sound_speed(P, ph, Ti);
    const float sigmai = pv.t.sigma[i];
    // transport velocity (SPH_kernels.cu:56-104)
    tvf_on = P.tvf && !(sigmai < P.tvf_sigma_min) && !(P.tvf_interface_only && !(pv.t.alpha[i] > 0.0f));
    Vt = r.t.w;
    // momentum (navier_stokes.cu:121-245)
    etai = sel2(P.mu, pi_idx) + (OPT && P.sps ? rhoi * pv.t.nu_t[i] : 0.0f);
    alpha_i = ph == kVapor ? P.alpha_av_vap : P.alpha_av;
    // CSF (surface_tension.cu:120-177)
    ni = kCsf ? ld3(pv.t.ns[i]) : V3{0, 0, 0};
    csf_on = kCsf && norm2(ni) > 0.25f;
    // Akinci (surface_tension.cu:179-213)
    ak_on = kAkinci && ph == kLiquid;
    nak = ak_on ? ld3(pv.s.nrm[i]) : V3{0, 0, 0};
    // continuity (SPH_kernels.cu:162-203)
    vci = CONT ? (P.tvf ? ld3(r.t) : vi) : V3{0, 0, 0};
    // conduction (phase_change.cu:31-75)
    k_same = pi_idx ? P.k_vv : P.k_ll;
    k_other = pi_idx ? P.k_vl : P.k_lv;
    reset();
  }

  // Numerator of a fast division, or a scaled one's quotient: too small a one
  // (remainders, or the scaling back, would leave the normal range) is seen by
  // unsafe().
  __device__ inline float noted(float x) {
    const uint32_t u = (__float_as_uint(x) << 1) - 1u;  // zero, which divides exactly, becomes the largest
    x_low = u < x_low ? u : x_low;
    return x;
  }
  // Whether some fast pair left the range its arithmetic is exact in (or met
  // an infinity or NaN): the target is then done again with IEEE operations.
  __device__ inline bool unsafe(const SimParams& P) const {
    const V3 f = force, a = acc_av, t = sum_t, k = acc_ak;
    const float sum = f.x + f.y + f.z + a.x + a.y + a.z + t.x + t.y + t.z + k.x + k.y + k.z + float(num) + float(den) +
                      float(div) + float(diff) + float(q);
    return !(r2_low >= P.r2_fast) || x_low < (kFastLow << 1) - 1u || !(sum - sum == 0.0f);
  }

  // The terms of pair (i, j); none for j == i (also used for a lane without a
  // neighbour).  FAST: correctly rounded division and square root without the
  // range handling of the IEEE sequences (the same bits within the range that
  // unsafe() checks).  DIRECT: the terms go straight to the sums (the cell sweep,
  // never FAST), else to o.
  // tvf_any / csf_any: some lane of the wave needs those terms.
  template <bool FAST, bool DIRECT>
  __device__ inline void pair(const PV& pv, const SimParams& P, int j, const PairData d, bool tvf_any, bool csf_any,
                              PairTerms<KS>& o) {
    static_assert(!(FAST && DIRECT), "the cell sweep uses IEEE operations");
    const float h = P.kernel.h;
    const float eta2 = 0.01f * h * h;
    const V3 xj = ld3(d.x);
    const int phj = __float_as_int(d.x.w);
    const V3 rij = KS ? df_diff3(xi, li, xj, d.lo) : xi - xj;
    const float r2 = norm2(rij);
    if (j == i || r2 >= P.support2) return;
    if (FAST) r2_low = r2 < r2_low ? r2 : r2_low;
    const float r = FAST ? sqrt_rn(r2) : sqrtf(r2);
    const Recip Rr = FAST ? recip_rn(r) : Recip{r, 0.0f};
    auto over = [](float x, const Recip& R) { return FAST ? div_rn(x, R) : x / R.y; };
    const float dW = kdW(P.kernel, r);
    const bool separated = FAST || r > 1e-12f * h;
    const float dWr = over(dW, Rr);
    const V3 gw = separated ? rij * dWr : V3{0, 0, 0};
    const float Tj = d.q.w;
    const bool tvf_stress = OPT && P.tvf && P.tvf_stress;
    const Recip Re = FAST ? recip_rn(r2 + eta2) : Recip{r2 + eta2, 0.0f};
    if (phj == kWall) {
      const float pj = d.q.x, pwv = d.q.y;
      V3 t{0, 0, 0};
      if (tvf_any && tvf_on) {
        float rho_w;
        if (ph == kVapor) {
          rho_w = (pwv - (P.p_bg - P.vapor_K)) / (P.gas_R * Ti);
        } else {
          rho_w = d.q.z;  // the wall pass stored rho0 * max(ratio, 0.5)^(1/gamma) here
        }
        const float Vj = rho_w > 0.0f ? Vt * rhoi / rho_w : Vt;
        t = gw * (Vt * Vt + Vj * Vj);
      }
      const float Vj = P.vol0;
      const float vsum = Vi * Vi + Vj * Vj;
      const float pw = ph == kVapor ? pwv : pj;
      const V3 f1 = -(gw * (vsum * 0.5f * (p_i + pw)));
      V3 fs{0, 0, 0}, f2{0, 0, 0}, a1{0, 0, 0}, a2{0, 0, 0}, a3{0, 0, 0};
      if (tvf_stress) fs = vi * (0.5f * vsum * rhoi * dot(dvi, gw));
      const bool guard = r < 0.6f * P.dx && separated;
      if ((DIRECT || KS) && guard) guard_terms(P, rij, r, a1, a2);
      if (P.no_slip) {
        const V3 vij = vi - ld3(d.v);
        if (separated) f2 = vij * over_scaled<FAST>(vsum * etai * dW, Rr);
        const float vr = dot(vij, rij);
        if (alpha_i > 0.0f && vr < 0.0f) {
          const float mu_ij = FAST ? div_rn(noted(h * vr), Re) : h * vr / Re.y;
          const float Pi = -alpha_i * ci * mu_ij / rhoi;
          a3 = -(gw * (rhoi * P.vol0 * Pi));
        }
      }
      V3 ak{0, 0, 0};
      if (kAkinci && ak_on && r2 > 0.0f) {
        const float psi = P.rho0[0] * P.vol0;
        const float arg = -4.0f * r * r / P.kernel.support + 6.0f * r - 2.0f * P.kernel.support;
        float adh = 0.0f;
        if (!(r >= P.kernel.support || 2.0f * r <= P.kernel.support) && arg > 0.0f)
          adh = P.ak_adh_scale * powf_cr(arg, 0.25f);
        ak = -((rij / r) * (P.ak_beta * psi * adh));
      }
      const float dv = CONT ? P.vol0 * dot(vci, gw) : 0.0f;
      float qq = 0.0f;
      const bool iso = THERMAL && P.wall_bc == 1;
      if (iso) {
        const float rgw = r * dW;
        qq = Vi * P.vol0 * (2.0f * sel2(P.k, pi_idx)) * (Ti - Tj) * rgw / (r2 + eta2);
      }
      V3 dF, df{0, 0, 0}, da{0, 0, 0};
      if constexpr (KS) {  // the pair's own terms, added once to each sum
        df += f1;
        if (tvf_stress) df += fs;
        df += f2;
        da += a1;
        da += a2;
        da += a3;
        dF = df + da * mi;
      }
      if constexpr (DIRECT) {
        if constexpr (KS) {
          force += df;
          acc_av += da;
        } else {  // the reference's wall load: what the pair changed
          const V3 f0 = force, a0 = acc_av;
          force += f1;
          if (tvf_stress) force += fs;
          force += f2;
          if (guard) {
            acc_av += a1;
            acc_av += a2;
          }
          acc_av += a3;
          dF = (V3(force) - f0) + (V3(acc_av) - a0) * mi;
        }
        fwall += dF;
        mwall += cross(xj - origin, dF);
        if (tvf_any) sum_t += t;
        if (kAkinci) acc_ak += ak;
        if (CONT) div += dv;
        if (iso) q += qq;
      } else {
        o.wall = true;
        o.guard = guard;
        o.xj = xj;
        if constexpr (KS) {
          o.f1 = df;
          o.a3 = da;
          o.dF = dF;
          o.dM = cross(xj - origin, dF);
        } else {
          o.f1 = f1;
          o.fs = fs;
          o.f2 = f2;
          o.a3 = a3;
        }
        o.t = t;
        o.ak = ak;
        o.div = dv;
        o.q = qq;
      }
      return;
    }
    // fluid neighbour
    const float pj = d.q.x, mj = d.q.y, rhoj = d.q.z;
    const float Vj = d.v.w;  // mj / rhoj, divided once per particle
    const float vsum = Vi * Vi + Vj * Vj;
    const float rsum = rhoi + rhoj;
    const Recip Rs = FAST ? recip_rn(rsum) : Recip{rsum, 0.0f};
    const float pt = FAST ? div_rn(noted(rhoj * p_i + rhoi * pj), Rs) : (rhoj * p_i + rhoi * pj) / rsum;
    const V3 f1 = -(gw * (vsum * pt));
    const V3 vj = ld3(d.v);
    V3 fs{0, 0, 0}, f2{0, 0, 0}, a3{0, 0, 0};
    if (tvf_stress) {
      const V3 Ag = vi * (rhoi * dot(dvi, gw)) + vj * (rhoj * dot(ld3(d.t) - vj, gw));
      fs = Ag * (0.5f * vsum);
    }
    const V3 vij = vi - vj;
    const bool same = phj == ph;
    if constexpr (OPT) {
      const float etaj = sel2(P.mu, pidx(phj)) + (P.sps ? rhoj * pv.t.nu_t[j] : 0.0f);
      const float eta_sum = etai + etaj;
      if (eta_sum > 0.0f && separated) {
        const float eta_ij = P.sps ? 2.0f * etai * etaj / eta_sum : (same ? (ph == kLiquid ? P.eta_ll : P.eta_vv) : P.eta_lv);
        f2 = vij * (vsum * eta_ij * dW / r);
      }
    } else {
      // no viscosity at all (eta_sum = 0): eta is 0 and so is the term
      const float eta_ij = same ? (ph == kLiquid ? P.eta_ll : P.eta_vv) : P.eta_lv;
      if (separated) f2 = vij * over_scaled<FAST>(vsum * eta_ij * dW, Rr);
    }
    if (same) {
      const float vr = dot(vij, rij);
      if (alpha_i > 0.0f && vr < 0.0f) {
        const float cj = ph == kVapor ? sqrtf(P.gas_R * (Tj > 0.0f ? Tj : 0.0f)) : P.c0;
        const float mu_ij = FAST ? div_rn(noted(h * vr), Re) : h * vr / Re.y;
        const float x = -alpha_i * 0.5f * (ci + cj) * mu_ij;
        const float Pi = FAST ? div_rn(noted(2.0f * x), Rs) : x / (0.5f * rsum);  // scaling by 2 is exact
        a3 = -(gw * (mj * Pi));
      }
    }
    if constexpr (DIRECT) {
      force += f1;
      if (tvf_stress) force += fs;
      force += f2;
      acc_av += a3;
    } else {
      o.f1 = f1;
      o.fs = fs;
      o.f2 = f2;
      o.a3 = a3;
    }
    if (tvf_any && tvf_on) {
      const float Vtj = d.t.w;  // 1 / sigma_j
      const V3 t = gw * (Vt * Vt + Vtj * Vtj);
      if constexpr (DIRECT) sum_t += t;
      else o.t = t;
    }
    if (kCsf && csf_any && csf_on && is_fluid(phj)) {
      const V3 gwc = rij * dWr;
      const V3 nj = ld3(pv.t.ns[j]);
      if (norm2(nj) > 0.25f) {
        const float nn = Vj * dot(ni - nj, gwc), dd = Vj * r * (-dW);
        if constexpr (DIRECT) num += nn, den += dd;
        else o.num = nn, o.den = dd;
      }
      if (OPT && P.csf_balanced) {
        const float cci = ph == kLiquid ? 1.0f : 0.0f;
        const float cj = phj == kLiquid ? 1.0f : 0.0f;
        const V3 g = gwc * ((Vi * Vi + Vj * Vj) * (rhoj * cci + rhoi * cj) / (rhoi + rhoj));
        if constexpr (DIRECT) Gs += g;
        else o.G = g;
      }
    }
    if (kAkinci && ak_on && r2 > 0.0f && phj == kLiquid) {
      const V3 rhat = rij / r;
      const float K = 2.0f * P.rho0[0] / (rhoi + rhoj);
      const V3 f_coh = rhat * (-P.ak_gamma * mi * mj * akinci_coh(r, P.kernel.support));
      const V3 f_curv = (nak - ld3(pv.s.nrm[j])) * (-P.ak_gamma * mi);
      const V3 ak = (f_coh + f_curv) * (K / mi);
      if constexpr (DIRECT) acc_ak += ak;
      else o.ak = ak;
    }
    if (CONT) {
      const float dv = Vj * dot(vci - (P.tvf ? ld3(d.t) : vj), gw);
      float df = 0.0f;
      if (same) {
        const float x = Vj * 2.0f * (rhoj - rhoi) * dot(-rij, gw);
        df = FAST ? div_rn(noted(x), Re) : x / Re.y;
      }
      if constexpr (DIRECT) div += dv, diff += df;
      else o.div = dv, o.diff = df;
    }
    if (THERMAL) {
      const float kij = pidx(phj) == pi_idx ? k_same : k_other;
      const float rgw = r * dW;
      const float x = Vi * Vj * kij * (Ti - Tj) * rgw;
      const float qq = over_scaled<FAST>(x, Re);
      if constexpr (DIRECT) q += qq;
      else o.q = qq;
    }
  }

  // x / R.y for an x that is often tiny (a pair near the support's edge):
  // scaled by 2^64 and back, exact while the quotient is normal.
  template <bool FAST>
  __device__ inline float over_scaled(float x, const Recip& R) {
    if constexpr (!FAST) return x / R.y;
    return noted(div_rn(x * 0x1p64f, R) * 0x1p-64f);
  }

  // Wall guard of a pair closer than 0.6 dx (navier_stokes.cu:121-245).
  __device__ inline void guard_terms(const SimParams& P, V3 rij, float r, V3& a1, V3& a2) const {
    const float r_guard = 0.6f * P.dx;
    const float qg = 1.0f - r / r_guard;
    const V3 nn = rij / r;
    a1 = nn * (4.0f * ci * ci * qg * qg / r_guard);
    const float vn = dot(vi, nn);
    if (vn < 0.0f && dt_now > 0.0f) a2 = -(nn * (qg * vn / dt_now));
  }

  // Adds the group's G pairs to the sums, lane 0's first.
  template <int G>
  __device__ inline void add(const SimParams& P, const PairTerms<KS>& o, bool tvf_any, bool csf_any) {
    using Ln = Lanes<G>;
    const unsigned long long walls = __ballot(o.wall), guards = __ballot(o.guard);
    const bool stress = OPT && P.tvf && P.tvf_stress;
    const float is_wall = o.wall ? 1.0f : 0.0f;
    V3 a1{0, 0, 0}, a2{0, 0, 0};
    if constexpr (!KS) {  // rare: evaluated here, so that pair() holds no registers for it
      if (guards && o.guard) {
        const V3 rij = xi - o.xj;
        guard_terms(P, rij, sqrtf(norm2(rij)), a1, a2);
      }
    }
    unrolled<G>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      const bool any_wall = (walls & Ln::mask(k)) != 0;
      V3 f0{0, 0, 0}, a0{0, 0, 0};
      if constexpr (!KS) f0 = force, a0 = acc_av;
      force += Ln::template from<k>(o.f1);
      if (stress) force += Ln::template from<k>(o.fs);
      force += Ln::template from<k>(o.f2);
      if constexpr (!KS) {
        if (guards & Ln::mask(k)) {
          acc_av += Ln::template from<k>(a1);
          acc_av += Ln::template from<k>(a2);
        }
      }
      acc_av += Ln::template from<k>(o.a3);
      if (any_wall) {
        const bool w = Ln::template from<k>(is_wall) != 0.0f;
        if constexpr (KS) {
          fwall += Ln::template from<k>(o.dF);
          mwall += Ln::template from<k>(o.dM);
        } else {  // the reference's wall load: what the pair changed
          const V3 dF = (V3(force) - f0) + (V3(acc_av) - a0) * mi;
          const V3 m = cross(Ln::template from<k>(o.xj) - origin, dF);
          fwall += w ? dF : V3{0, 0, 0};
          mwall += w ? m : V3{0, 0, 0};
        }
      }
      if (tvf_any) sum_t += Ln::template from<k>(o.t);
      if constexpr (kCsf) {
        if (csf_any) {
          num += Ln::template from<k>(o.num);
          den += Ln::template from<k>(o.den);
          if (OPT && P.csf_balanced) Gs += Ln::template from<k>(o.G);
        }
      }
      if constexpr (kAkinci) acc_ak += Ln::template from<k>(o.ak);
      if constexpr (CONT) {
        div += Ln::template from<k>(o.div);
        diff += Ln::template from<k>(o.diff);
      }
      if constexpr (THERMAL) q += Ln::template from<k>(o.q);
    });
  }

  __device__ void finish(const PV& pv, const SimParams& P, const DevState* st, bool store, Maxima& mx) {
    const float pb = P.tvf_factor * sel2(P.rho0, pi_idx) * ci * ci;
    const float mt = rhoi * Vt;
    const float h = P.kernel.h;
    const V3 ab = tvf_on ? V3(sum_t) * (-pb / mt) : V3{0, 0, 0};
    V3 acc = st->gravity + V3(force) / mi + V3(acc_av);
    if (st->frame_rot) {
      const V3 om = st->omega, omd = st->omega_dot;
      const V3 rr = xi - origin;
      acc -= cross(omd, rr) + cross(om, cross(om, rr)) + cross(om, vi) * 2.0f;
    }
    float kappa = 0.0f;
    if (kCsf && csf_on) {
      kappa = float(den) > 0.0f ? 3.0f * float(num) / float(den) : 0.0f;
      if (P.wetting != 0) acc += ld3(pv.t.vw[i]);
      if (OPT && P.csf_balanced) {
        acc += V3(Gs) * (P.sigma * kappa / mi);
      } else {
        const float coeff = 2.0f * P.sigma / (P.rho0[0] + P.rho0[1]);
        acc += ld3(pv.s.nrm[i]) * (coeff * kappa);
      }
    }
    if (ak_on) acc += V3(acc_ak);
    if (store) {
      pv.t.ab[i] = st3(ab);
      if (kCsf) pv.t.kappa[i] = kappa;
      pv.t.a[i] = st3(acc);
      pv.t.fw[i] = st3(V3(fwall));
      pv.t.mw[i] = st3(V3(mwall));
      if (CONT) pv.t.drho[i] = rhoi * float(div) + P.delta_sph * h * P.c0 * float(diff);
      if (THERMAL) {
        const float qt = float(q) + P.heat_power * pv.t.heat_w[i] * st->heat_inv_norm;
        pv.t.dTdt[i] = qt / (mi * sel2(P.cp, pi_idx));
      }
    }
    // evaluate_rates maxima (sph_solver.cu:62-99)
    mx.v = norm(vi);
    const float na = norm(acc), nb = norm(ab);
    mx.a = na > nb ? na : nb;
    if (ph == kVapor) mx.tv = Ti;
    if (OPT && P.sps) mx.nu = pv.t.nu_t[i];
    const float rm = pv.t.rmin[i] > 0.05f * P.dx ? pv.t.rmin[i] : 0.05f * P.dx;
    mx.sp = 0.5f * P.dx / rm;
  }
};

// The rates of a particle that is not fluid.
template <bool CONT, bool THERMAL>
__device__ inline void zero_rates(const PV& pv, int i) {
  pv.t.ab[i] = st3(V3{0, 0, 0});
  pv.t.a[i] = st3(V3{0, 0, 0});
  pv.t.fw[i] = st3(V3{0, 0, 0});
  pv.t.mw[i] = st3(V3{0, 0, 0});
  if (CONT) pv.t.drho[i] = 0.0f;
  if (THERMAL) pv.t.dTdt[i] = 0.0f;
}

// The block's maxima into the step's (every thread of the block calls it).
// One look at the step's present maximum per block, and an atomic only where
// the block raises it: five atomics of every wave to one cache line queue up
// (this pass over 2.2 M particles, 45 k waves: 4.2 ms with them, 0.84 without).
template <int NT>
__device__ inline void publish_maxima(DevState* st, Maxima mx) {
  __shared__ float s_max[NT / 64][5];
  const float v[5] = {wave_max(mx.v), wave_max(mx.a), wave_max(mx.tv), wave_max(mx.nu), wave_max(mx.sp)};
  if ((threadIdx.x & 63) == 0)
    for (int k = 0; k < 5; ++k) s_max[threadIdx.x >> 6][k] = v[k];
  __syncthreads();
  if (threadIdx.x < 5) {
    float m = 0.0f;
    for (int w = 0; w < NT / 64; ++w) m = s_max[w][threadIdx.x] > m ? s_max[w][threadIdx.x] : m;
    unsigned* at = &st->max_bits[threadIdx.x];
    if (__float_as_uint(m) > __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomic_max_nonneg(at, m);
  }
}

// One block: kBlock / G consecutive particles; its fluid ones with a complete
// list are packed onto consecutive groups of G lanes (a wall only writes
// zeros), so that no group idles for a wall.  Neighbour records are gathered
// from L2 one step ahead of their pair: 64 bytes of one line each, no LDS, so
// registers alone (<= 128, four waves per SIMD) set the occupancy, and any
// number of particles spreads evenly over the chip.  It replaced one thread
// per particle over LDS-staged cell tiles (159 KB, 1.35 waves per SIMD, five
// atomics a wave).  us a launch by kernel traces, before and now: 2.2 M-particle
// column in motion 2274 / 831, the benchmark's column in its first 24 launches
// 1907 / 1015 (nearly at rest: up to a quarter of its fluid targets meet tiny
// numerators and are swept twice), 1.2 M two-phase sphere 1828 / 661, 188 k tank
// 323 / 142, 26 k tank 203 / 48, precision form at 293 k 713 / 281.  Bound by the
// pair arithmetic (84 % of the VALU's issue at 3 cycles an instruction) and the
// gathers (a tag look-up per lane and 16 bytes).
template <int ST, bool CONT, bool THERMAL, bool KS, bool OPT, int G>
__global__ __launch_bounds__(kBlock, KS || ST == 2 ? 2 : (OPT || (ST == 1 && CONT) ? 3 : 4)) void k_forces(PV pv, SimParams P, NbrList L, DevState* st, Count nc) {
  constexpr int kSpan = kBlock / G;
  __shared__ int s_work[kSpan], s_tot[kBlock / 64];
  const int n = nc.get();
  const int base = xcd_span(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x)) * kSpan;
  if (base >= n) return;  // uniform over the block
  const int t = static_cast<int>(threadIdx.x);
  bool keep = false;
  if (t < kSpan && base + t < n) {
    const int i = base + t;
    if (L.count[i] >= 0) {
      if (is_fluid(pv.s.phase[i])) keep = true;
      else zero_rates<CONT, THERMAL>(pv, i);
    }
  }
  const unsigned long long kept = __ballot(keep);
  const int lane = t & 63, wave = t >> 6;
  if (lane == 0) s_tot[wave] = __popcll(kept);
  __syncthreads();
  int first = 0, total = 0;
  for (int w = 0; w < (kSpan + 63) / 64; ++w) {
    const int c = s_tot[w];
    first += w < wave ? c : 0;
    total += c;
  }
  if (keep) s_work[first + __popcll(kept & ((1ull << lane) - 1ull))] = base + t;
  __syncthreads();
  const int slot = t / G, sub = t % G;
  Maxima mx;
  if (slot < total) {
    const int i = s_work[slot];
    ForcesTarget<ST, CONT, THERMAL, KS, OPT> T(pv, P, st, i);
    const bool need_vt = forces_need_vt(P, CONT);
    const bool tvf_any = __any(T.tvf_on), csf_any = __any(T.csf_on);
    const bool need_t = need_vt || tvf_any;
    const int cnt = L.count[i];
    const int* lp = reinterpret_cast<const int*>(list_chunks(L, i));
    // entry e of the list; past the end the particle itself, which adds nothing
    auto entry = [&](int e) { return e < cnt ? lp[(e >> 2) * (4 * kListGroup) + (e & 3)] : i; };
    auto load = [&](int j) {
      const PairRec* r = pv.t.rec + j;
      float4 tq = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (need_t) tq = r->t;
      return PairData{r->x, r->q, r->v, tq, pos_lo<KS>(pv.s.xlo, j)};
    };
    auto sweep = [&](auto fast) {
      int j = entry(sub), jn = entry(sub + G);
      PairData d = load(j);
      for (int e = 0; e < cnt; e += G) {  // the next record and the entry after it are in flight
        PairData c;
        c.x = take(d.x);
        c.q = take(d.q);
        c.v = take(d.v);
        c.t = need_t ? take(d.t) : d.t;
        if (KS) c.lo = V3{take(d.lo.x), take(d.lo.y), take(d.lo.z)};
        const int jc = j;
        j = take(jn);
        d = load(j);
        jn = entry(e + sub + 2 * G);
        PairTerms<KS> o;
        T.template pair<decltype(fast)::value, false>(pv, P, jc, c, tvf_any, csf_any, o);
        T.template add<G>(P, o, tvf_any, csf_any);
      }
    };
    if (P.fast) sweep(std::true_type{});
    // (uniform over a group: its lanes hold the same sums; what each lane's own pairs met differs)
    bool again = !P.fast || T.unsafe(P);
    again = (__ballot(again) >> (lane & ~(G - 1)) & ((1ull << G) - 1)) != 0;
    if (again) {
      T.reset();
      sweep(std::false_type{});
    }
    T.finish(pv, P, st, sub == 0, mx);
  }
  publish_maxima<kBlock>(st, mx);
}

// The particles whose list overflowed (count < 0), by the cell sweep, which
// visits the same neighbours in the same order.
template <int ST, bool CONT, bool THERMAL, bool KS, bool OPT>
__global__ __launch_bounds__(kBlock) void k_forces_sweep(PV pv, GridDev g, SimParams P, NbrList L, DevState* st,
                                                        Count nc) {
  const int n = nc.get();
  const int i = gtid();
  const bool mine = i < n && L.count[i] < 0;
  if (!__syncthreads_or(mine)) return;
  Maxima mx;
  if (mine) {
    if (is_fluid(pv.s.phase[i])) {
      ForcesTarget<ST, CONT, THERMAL, KS, OPT> T(pv, P, st, i);
      const bool tvf_any = T.tvf_on, csf_any = T.csf_on;
      for_each_nbr(g, T.xi, [&](int j) {
        const PairRec* r = pv.t.rec + j;
        const PairData d{r->x, r->q, r->v, r->t, pos_lo<KS>(pv.s.xlo, j)};
        PairTerms<KS> o;
        T.template pair<false, true>(pv, P, j, d, tvf_any, csf_any, o);
      });
      T.finish(pv, P, st, true, mx);
    } else {
      zero_rates<CONT, THERMAL>(pv, i);
    }
  }
  publish_maxima<kBlock>(st, mx);
}

template <int ST, bool CONT, bool THERMAL, bool KS, bool OPT>
void forces_run(const PV& pv, const GridDev& g, const SimParams& P, const NbrList& L, DevState* st, Count n, int lanes,
                hipStream_t s) {
  const int m = std::max(n.ub, 1);
  if (lanes == 2) k_forces<ST, CONT, THERMAL, KS, OPT, 2><<<blocks_for(2ll * m), kBlock, 0, s>>>(pv, P, L, st, n);
  else k_forces<ST, CONT, THERMAL, KS, OPT, 4><<<blocks_for(4ll * m), kBlock, 0, s>>>(pv, P, L, st, n);
  k_forces_sweep<ST, CONT, THERMAL, KS, OPT><<<blocks_for(m), kBlock, 0, s>>>(pv, g, P, L, st, n);
}
template <int ST, bool CONT, bool THERMAL>
void forces_flags(const PV& pv, const GridDev& g, const SimParams& P, const NbrList& L, DevState* st, Count n,
                  int lanes, hipStream_t s) {
  const bool opt = (P.tvf && P.tvf_stress) || P.csf_balanced || P.sps;
  if (P.compensated) {
    if (opt) forces_run<ST, CONT, THERMAL, true, true>(pv, g, P, L, st, n, lanes, s);
    else forces_run<ST, CONT, THERMAL, true, false>(pv, g, P, L, st, n, lanes, s);
  } else {
    if (opt) forces_run<ST, CONT, THERMAL, false, true>(pv, g, P, L, st, n, lanes, s);
    else forces_run<ST, CONT, THERMAL, false, false>(pv, g, P, L, st, n, lanes, s);
  }
}

}  // namespace

template <int ST>
void launch_forces_model(const PV& pv, const GridDev& g, const SimParams& P, const NbrList& L, DevState* st, Count n,
                         bool continuity, bool thermal, int lanes, hipStream_t s) {
  if (!L.valid) throw std::logic_error("forces pass: neighbour lists not built");
  if (continuity) {
    if (thermal) forces_flags<ST, true, true>(pv, g, P, L, st, n, lanes, s);
    else forces_flags<ST, true, false>(pv, g, P, L, st, n, lanes, s);
  } else {
    if (thermal) forces_flags<ST, false, true>(pv, g, P, L, st, n, lanes, s);
    else forces_flags<ST, false, false>(pv, g, P, L, st, n, lanes, s);
  }
}

}  // namespace cryo
