// Multi-phase device functions: the per-cell aerosol state (phase mass,
// average molecular weight, number concentration of every bin), ZSR water
// uptake and its parameter Jacobian, and the SIMPOL phase-transfer and
// aqueous-equilibrium contributions to f(y) and J(y).
//
// Arithmetic follows the reference operation by operation: where it
// computes in double the same double operations are used, and where it
// uses long double (accumulators and rate products) double-double is used,
// which is at least as precise.  Sources restated:
//   aero_phase_solver.c:78-150           phase mass, average MW, volume
//   aero_rep_modal_binned_mass.c:183-266 bin number concentration (BINNED)
//   sub_model_ZSR_aerosol_water.c:216-440  water (JACOBSON pairs), Jacobian
//   rxn_SIMPOL_phase_transfer.c:220-740  environment, f, J
//   rxn_aqueous_equilibrium.c:244-548    environment, f, J
//   util.h:19-68                          transition-regime rate constants
#pragma once

#include "camp_aero.hpp"
#include "camp_device.hpp"

namespace camp {

constexpr int kAeroSlots = 8;           // per phase instance in LDS
constexpr int kSpScalars = 17;          // per SIMPOL instance
constexpr int kAqScalars = 6;           // per aqueous-equilibrium instance

// --- transition-regime condensation (util.h:19-68), all double -------------
__host__ __device__ __forceinline__ double mp_transition_corr(double mfp, double r, double alpha) {
  double kn = mfp / r;
  return (0.75 * alpha * (1.0 + kn)) / (kn * kn + (1.0 + 0.283 * alpha) * kn + 0.75 * alpha);
}
__host__ __device__ __forceinline__ double mp_cond_rate(double D, double mfp, double r, double alpha) {
  return 4.0 * kPi * r * D * mp_transition_corr(mfp, r, alpha);
}
__host__ __device__ __forceinline__ double mp_dcond_rate_dr(double D, double mfp, double r, double alpha) {
  double kn = mfp / r;
  double dcorr = (0.75 * alpha * mfp * (kn * kn + 2.0 * kn + 1.0 + (0.283 - 0.75) * alpha)) /
                 cr_powi(r * (kn * kn + (1.0 + 0.283 * alpha) * kn + 0.75 * alpha), 2);
  return 4.0 * kPi * D * (mp_transition_corr(mfp, r, alpha) + r * dcorr);
}

// --- aerosol state of one cell (aero_rep_update_state) ---------------------
// s_aero[i*8]: mass, average MW, number concentration (cached, as the
// representation caches them), then the mass and mole sums (dd) of the
// current state, which the MW partial derivatives use, and its volume
// The sums run over the counted species of each phase instance ("items",
// Program::pit_ptr).  A lane per phase, as the sums' order suggests, leaves 8
// of 64 lanes with 29 double-double divisions one after another; the quotients
// x / MW and x / density are formed by a lane per item into scratch and only
// the additions stay in order, the three sums of a phase on three lanes.
//
// The scratch (here, in the ZSR passes and for J's partial derivatives) is the
// LDS of f's contribution slots and of the per-term rates after them, which
// hold nothing yet: mp_scratch_doubles(P) of it.  What does not fit at once
// goes in chunks, each continuing the sums of the last.
__host__ __device__ inline size_t mp_slot_doubles(const DevProgram& P) {
  const size_t n = 2 * (size_t)P.n_slots;
  return n > 6 ? n : 6;  // (one item or ion pair at least)
}
__host__ __device__ inline int mp_scratch_doubles(const DevProgram& P) {
  return (int)(mp_slot_doubles(P) + 2 * (size_t)P.n_terms);
}

// mass, moles (dd) and volume of every phase into s_aero[3..7]
__device__ __forceinline__ void mp_phase_sums(const DevProgram& P, int lane, const double* s_state,
                                              double* s_aero, double* scratch) {
  const int cap = mp_scratch_doubles(P) / 4;
  int b = 0;
  do {
    const int end = min(b + cap, P.n_it);
    for (int it = b + lane; it < end; it += kWave) {
      double x = s_state[P.pit_state[it]];
      dd m = dd_div_d(dd_from(x), P.pit_mw[it]);
      double* q = scratch + 4 * (it - b);
      q[0] = x;
      q[1] = m.hi;
      q[2] = m.lo;
      q[3] = x / P.pit_dens[it];
    }
    wsync();
    for (int t = lane; t < 3 * P.n_pi; t += kWave) {
      const int i = t / 3, w = t - 3 * i;
      const int k0 = max(P.pit_ptr[i], b), k1 = min(P.pit_ptr[i + 1], end);
      double* a = s_aero + kAeroSlots * i + 3 + 2 * w;
      const double* q = scratch + 4 * (k0 - b) + (w == 0 ? 0 : w == 1 ? 1 : 3);
      dd s = w == 0 ? dd{P.min_mass_hi, P.min_mass_lo}
                    : w == 1 ? dd{P.min_moles_hi, P.min_moles_lo} : dd{P.min_volume, 0.0};
      if (b > 0) s = dd{a[0], w < 2 ? a[1] : 0.0};
      for (int k = k0; k < k1; ++k, q += 4) {
        dd v = {q[0], w == 1 ? q[1] : 0.0};
        const double plain = s.hi + v.hi;
        s = dd_add(s, v);
        if (w == 2) s = dd{plain, 0.0};
      }
      a[0] = s.hi;
      if (w < 2) a[1] = s.lo;
    }
    wsync();
    b += cap;
  } while (b < P.n_it);
}

// --- ZSR water of every (sub model, phase) item (:216-301) -----------------
// A lane per ion for the exponentials, a lane per ion pair for its molality and
// contribution, a lane per item to add the pairs in order; scratch holds 6
// doubles per pair (cation, anion, their exponentials, the contribution).
// (pairs x0 to x1, pair x's scratch at 6 (x - x0))
__device__ __forceinline__ void mp_zsr_ions(const DevProgram& P, int lane, int x0, int x1,
                                            const double* s_state, double* scratch) {
  for (int t = lane; t < 2 * (x1 - x0); t += kWave) {
    const bool an = t >= x1 - x0;
    const int x = x0 + (an ? t - (x1 - x0) : t);
    // ion concentrations are double expressions (state / int / MW / 1000)
    double c = s_state[an ? P.zp_an[x] : P.zp_cat[x]] / (double)(an ? P.zp_nan[x] : P.zp_ncat[x]) /
               (an ? P.zp_anmw[x] : P.zp_catmw[x]) / 1000.0;
    scratch[6 * (x - x0) + (an ? 1 : 0)] = c;
    scratch[6 * (x - x0) + (an ? 3 : 2)] = cr_exp(-100.0 * c);
  }
  wsync();
}

__device__ __forceinline__ void mp_zsr(const DevProgram& P, int lane, const double* s_sub_env,
                                       double* s_state, double* scratch) {
  const int cap = mp_scratch_doubles(P) / 6;
  int x0 = 0;
  do {
    const int x1 = min(x0 + cap, P.n_zp);
    mp_zsr_ions(P, lane, x0, x1, s_state, scratch);
    for (int x = x0 + lane; x < x1; x += kWave) {
      const int z = P.zp_zi[x];
      // a_w = PPM_TO_RH * state: a double product (both operands double)
      dd aw = dd_from(s_sub_env[P.zi_sub[z]] * s_state[P.zi_gw[z]]);
      double low = P.zp_lowrh[x];
      dd jaw = dd_gt(aw, low) ? aw : dd_from(low);
      double jaw_d = dd_round(jaw);
      // the powers of jaw (cr_powi) as one chain: each continues the last
      dd mol = dd_from(0.0);
      dd pw = dd_from(fabs(jaw_d));
      for (int k = 0; k < P.zp_ny[x]; ++k) {
        double pk = k == 0 ? 1.0 : dd_round(pw);
        if (jaw_d < 0.0 && (k & 1)) pk = -pk;
        if (k > 0) pw = dd_mul_d(pw, fabs(jaw_d));
        mol = dd_add(mol, dd_from(P.zp_y[8 * x + k] * pk));
      }
      mol = dd_mul(mol, mol);
      double* q = scratch + 6 * (x - x0);
      dd cat = dd_from(q[0]), an = dd_from(q[1]), e_ac = dd_from(q[2]), e_aa = dd_from(q[3]);
      dd conc = dd_div(dd_add(dd_mul(cat, e_ac), dd_mul(an, e_aa)), dd_add(e_ac, e_aa));
      dd v = dd_mul(dd_div(conc, mol), dd_from(1000.0));
      q[4] = v.hi;
      q[5] = v.lo;
    }
    wsync();
    for (int z = lane; z < P.n_zi; z += kWave) {
      double water = x0 > 0 ? s_state[P.zi_water[z]] : 1.0e-30;
      const int e = min(P.zi_pair_ptr[z + 1], x1);
      for (int x = max(P.zi_pair_ptr[z], x0); x < e; ++x) {
        const double* q = scratch + 6 * (x - x0);
        water = dd_round(dd_add(dd_from(water), dd{q[4], q[5]}));
      }
      s_state[P.zi_water[z]] = water;
    }
    wsync();
    x0 += cap;
  } while (x0 < P.n_zp);
}

// --- ZSR parameter Jacobian (:314-~440), added into s_jp: a lane per pair,
// then a lane per item adds its pairs in order ------------------------------
__device__ __forceinline__ void mp_zsr_jac(const DevProgram& P, int lane, const double* s_sub_env,
                                           const double* s_state, double* s_jp, double* scratch) {
  const int cap = mp_scratch_doubles(P) / 6;
  int x0 = 0;
  do {
    const int x1 = min(x0 + cap, P.n_zp);
    mp_zsr_ions(P, lane, x0, x1, s_state, scratch);
    for (int x = x0 + lane; x < x1; x += kWave) {
      const int z = P.zp_zi[x];
      double ppm = s_sub_env[P.zi_sub[z]];
      dd aw = dd_from(ppm * s_state[P.zi_gw[z]]);
      double low = P.zp_lowrh[x];
      bool above = dd_gt(aw, low);
      dd jaw = above ? aw : dd_from(low);
      double jaw_d = dd_round(jaw);
      dd djaw = above ? dd_from(ppm) : dd_from(0.0);
      const double* Y = P.zp_y + 8 * x;
      dd mol = dd_from(Y[0]), dmol = dd_from(0.0);
      for (int k = 1; k < P.zp_ny[x]; ++k) {
        mol = dd_add(mol, dd_from(Y[k] * cr_powi(jaw_d, k)));
        dmol = dd_add(dmol, dd_from(Y[k] * k * cr_powi(jaw_d, k - 1)));
      }
      dmol = dd_mul(dmol, djaw);
      double* q = scratch + 6 * (x - x0);
      dd cat = dd_from(q[0]), an = dd_from(q[1]), e_ac = dd_from(q[2]), e_aa = dd_from(q[3]);
      double dcat = 1.0 / (double)P.zp_ncat[x] / P.zp_catmw[x] / 1000.0;
      double dan = 1.0 / (double)P.zp_nan[x] / P.zp_anmw[x] / 1000.0;
      dd conc = dd_div(dd_add(dd_mul(cat, e_ac), dd_mul(an, e_aa)), dd_add(e_ac, e_aa));
      dd den = dd_mul(dd_add(e_ac, e_aa), dd_add(e_ac, e_aa));
      // (1 - ALPHA*anion + ALPHA*cation), ALPHA = -100
      dd kc = dd_add(dd_add(dd_from(1.0), dd_mul(dd_from(100.0), an)), dd_mul(dd_from(-100.0), cat));
      dd ka = dd_add(dd_add(dd_from(1.0), dd_mul(dd_from(100.0), cat)), dd_mul(dd_from(-100.0), an));
      dd dcdc = dd_div(dd_add(dd_mul(e_ac, e_ac), dd_mul(dd_mul(e_ac, e_aa), kc)), den);
      dd dcda = dd_div(dd_add(dd_mul(e_aa, e_aa), dd_mul(dd_mul(e_ac, e_aa), ka)), den);
      double mol_d = dd_round(mol);
      double p3 = cr_powi(mol_d, 3), p2 = cr_powi(mol_d, 2);
      // J[...] += value: each a double += (long double) rounded to double
      // -2.0 * conc / pow(m, 3) * 1000.0 * dm and 1.0 / pow(m, 2) * 1000.0 * dc * dion,
      // evaluated left to right as the reference does
      dd v_gw = dd_mul(dd_mul(dd_div_d(dd_mul(dd_from(-2.0), conc), p3), dd_from(1000.0)), dmol);
      double t2 = 1.0 / p2 * 1000.0;
      dd v_an = dd_mul(dd_mul(dd_from(t2), dcda), dd_from(dan));
      dd v_cat = dd_mul(dd_mul(dd_from(t2), dcdc), dd_from(dcat));
      q[0] = v_gw.hi;
      q[1] = v_gw.lo;
      q[2] = v_an.hi;
      q[3] = v_an.lo;
      q[4] = v_cat.hi;
      q[5] = v_cat.lo;
    }
    wsync();
    for (int z = lane; z < P.n_zi; z += kWave) {
      const int e = min(P.zi_pair_ptr[z + 1], x1);
      for (int x = max(P.zi_pair_ptr[z], x0); x < e; ++x) {
        const double* q = scratch + 6 * (x - x0);
        double* j = s_jp + P.zp_jgw[x];
        *j = dd_round(dd_add(dd_from(*j), dd{q[0], q[1]}));
        j = s_jp + P.zp_jan[x];
        *j = dd_round(dd_add(dd_from(*j), dd{q[2], q[3]}));
        j = s_jp + P.zp_jcat[x];
        *j = dd_round(dd_add(dd_from(*j), dd{q[4], q[5]}));
      }
    }
    wsync();
    x0 += cap;
  } while (x0 < P.n_zp);
}

// --- per-instance quantities shared by f and J ------------------------------
struct SpInst {
  double nconc, kp, kc, ev0;  // number conc., ppm per kg/m3, k_c(r), k_c*Keq*MW/mass
  dd cond, evap;              // k_c*gas and k_c*Keq*MW/mass*act*aero (long double in CAMP)
};

__host__ __device__ __forceinline__ SpInst mp_simpol_inst(const DevProgram& P, int i, const double* s_state,
                                                 const double* s_k, const double* s_aero) {
  const double* e = s_k + P.sp_env[i];
  const double* f = P.rx_float + P.sp_flt[i];
  const double* a = s_aero + kAeroSlots * P.sp_pi[i];
  SpInst s;
  s.nconc = a[2];
  s.kp = e[3];
  s.kc = mp_cond_rate(f[2], e[0], P.sp_radius[i], e[1]);
  // evap = cond_rate * (EQUIL_CONST * avg_MW / mass): the factor in double
  s.ev0 = e[2] * a[1] / a[0];
  dd evap = dd_mul(dd_from(s.kc), dd_from(s.ev0));
  s.cond = dd_mul(dd_from(s.kc), dd_from(s_state[P.sp_gas[i]]));
  s.evap = dd_mul(evap, dd_from(s_state[P.sp_aero[i]]));
  return s;
}

// f slots of one SIMPOL instance (rxn_SIMPOL_phase_transfer.c:355-399)
__host__ __device__ __forceinline__ void mp_simpol_f(const DevProgram& P, int i, const double* s_state,
                                            const double* s_k, const double* s_aero,
                                            double* s_slot) {
  SpInst s = mp_simpol_inst(P, i, s_state, s_k, s_aero);
  double* o = s_slot + 2 * P.sp_slot[i];
  dd ne = dd_mul(dd_from(s.nconc), s.evap), nc = dd_mul(dd_from(s.nconc), s.cond);
  dd v[4] = {ne, dd_neg(nc), dd_neg(dd_div_d(ne, s.kp)), dd_div_d(nc, s.kp)};
  for (int q = 0; q < 4; ++q) {
    o[2 * q] = v[q].hi;
    o[2 * q + 1] = v[q].lo;
  }
}

// aqueous equilibrium: forward and reverse rates of one instance, or
// skipped (water below the threshold) -- calc_standard_rate (:278-310)
struct AqRates {
  bool skip;
  dd rf, rr;
};
__host__ __device__ __forceinline__ AqRates mp_aqeq_rates(const DevProgram& P, int i,
                                                 const double* s_state, const double* s_k) {
  AqRates r;
  const double* f = P.rx_float + P.aq_flt[i];
  int nr = P.aq_nr[i], np = P.aq_np[i];
  const int* sp = P.aq_sp + 6 * i;
  double w = s_state[P.aq_water[i]];
  r.skip = w < 1.0e-4 * P.aq_small_water[i];
  dd water = dd_from(w);
  dd react = dd_mul(dd_from(s_state[sp[0]]), dd_from(f[5]));
  for (int q = 1; q < nr; ++q) react = dd_mul(react, dd_div(dd_from(s_state[sp[q]] * f[5 + q]), water));
  dd prod = dd_mul(dd_from(s_state[sp[3]]), dd_from(f[5 + nr]));
  for (int q = 1; q < np; ++q)
    prod = dd_mul(prod, dd_div(dd_from(s_state[sp[3 + q]] * f[5 + nr + q]), water));
  r.rf = dd_mul(dd_from(s_k[P.aq_env[i]]), react);
  r.rr = dd_mul(dd_from(f[2]), prod);
  return r;
}

__host__ __device__ __forceinline__ void mp_aqeq_f(const DevProgram& P, int i, const double* s_state,
                                          const double* s_k, double* s_slot) {
  int nr = P.aq_nr[i], np = P.aq_np[i];
  double* o = s_slot + 2 * P.aq_slot[i];
  AqRates r = mp_aqeq_rates(P, i, s_state, s_k);
  dd rate = dd_sub(r.rf, r.rr);
  bool zero = r.skip || (rate.hi == 0.0 && rate.lo == 0.0);
  const double* f = P.rx_float + P.aq_flt[i];
  for (int q = 0; q < nr + np; ++q) {
    double m = f[5 + q];
    dd a = dd_div_d(r.rf, m), b = dd_div_d(r.rr, m);
    if (q < nr) a = dd_neg(a);
    else b = dd_neg(b);
    o[4 * q] = zero ? 0.0 : a.hi;
    o[4 * q + 1] = zero ? 0.0 : a.lo;
    o[4 * q + 2] = zero ? 0.0 : b.hi;
    o[4 * q + 3] = zero ? 0.0 : b.lo;
  }
}


// --- Jacobian scalars of one SIMPOL instance (rxn_SIMPOL_phase_transfer.c:
// 415-~590), kSpScalars doubles: N, kp, kc, evap0 (dd), cond (dd), evap
// (dd), d_cond_d_radius, d_evap_d_radius, d_evap_d_mass, d_evap_d_MW, evap /
// kp (dd), cond / kp (dd).  evap0
// is k_c*Keq*MW/mass before the activity coefficient and the aerosol factor.
__host__ __device__ __forceinline__ void mp_simpol_jscalars(const DevProgram& P, int i,
                                                   const double* s_state, const double* s_k,
                                                   const double* s_aero, double* o) {
  const double* e = s_k + P.sp_env[i];
  const double* f = P.rx_float + P.sp_flt[i];
  const double* a = s_aero + kAeroSlots * P.sp_pi[i];
  double gas = s_state[P.sp_gas[i]], aero = s_state[P.sp_aero[i]];
  double kc = mp_cond_rate(f[2], e[0], P.sp_radius[i], e[1]);
  dd evap0 = dd_mul(dd_from(kc), dd_from(e[2] * a[1] / a[0]));
  dd cond = dd_mul(dd_from(kc), dd_from(gas));
  dd evap = dd_mul(evap0, dd_from(aero));
  double dcdr = mp_dcond_rate_dr(f[2], e[0], P.sp_radius[i], e[1]) * gas;
  double dedr = dcdr / gas * e[2] * a[1] / a[0] * aero;
  double dedm = dd_round(dd_div_d(dd_neg(evap), a[0]));
  double dedw = dd_round(dd_div_d(evap, a[1]));
  o[0] = a[2];
  o[1] = e[3];
  o[2] = kc;
  o[3] = evap0.hi;
  o[4] = evap0.lo;
  o[5] = cond.hi;
  o[6] = cond.lo;
  o[7] = evap.hi;
  o[8] = evap.lo;
  o[9] = dcdr;
  o[10] = dedr;
  o[11] = dedm;
  o[12] = dedw;
  dd ek = dd_div_d(evap, e[3]), ck = dd_div_d(cond, e[3]);
  o[13] = ek.hi;
  o[14] = ek.lo;
  o[15] = ck.hi;
  o[16] = ck.lo;
}

// --- Jacobian scalars of one aqueous-equilibrium instance (:403-~430):
// forward (dd), reverse (dd), water, skip flag
__host__ __device__ __forceinline__ void mp_aqeq_jscalars(const DevProgram& P, int i,
                                                 const double* s_state, const double* s_k,
                                                 double* o) {
  const double* f = P.rx_float + P.aq_flt[i];
  int nr = P.aq_nr[i], np = P.aq_np[i];
  const int* sp = P.aq_sp + 6 * i;
  double w = s_state[P.aq_water[i]];
  dd water = dd_from(w);
  dd fwd = dd_from(s_k[P.aq_env[i]]);
  for (int q = 0; q < nr; ++q) fwd = dd_mul(fwd, dd_div(dd_from(s_state[sp[q]] * f[5 + q]), water));
  dd rev = dd_from(f[2]);
  for (int q = 0; q < np; ++q)
    rev = dd_mul(rev, dd_div(dd_from(s_state[sp[3 + q]] * f[5 + nr + q]), water));
  o[0] = fwd.hi;
  o[1] = fwd.lo;
  o[2] = rev.hi;
  o[3] = rev.lo;
  o[4] = w;
  o[5] = w < 1.0e-4 * P.aq_small_water[i] ? 1.0 : 0.0;
}

// The partial derivatives of an item's phase's number concentration and average
// MW by the item's species (aero_phase_solver.c:78-150 and the representation's
// getters).
__host__ __device__ __forceinline__ void mp_item_partials(const DevProgram& P, int it,
                                                          const double* s_aero, double& numj,
                                                          double& mwj) {
  const int pi = P.pit_pi[it];
  const double* ag = s_aero + kAeroSlots * pi;
  double factor = 3.0 / (4.0 * kPi) / cr_powi(P.pi_dp[pi] / 2.0, 3);
  numj = 1.0 / P.pit_dens[it] * factor;
  dd lm = {ag[3], ag[4]}, mo = {ag[5], ag[6]};
  mwj = dd_round(dd_div(dd_sub(mo, dd_mul(dd_from(1.0 / P.pit_mw[it]), lm)), dd_mul(mo, mo)));
}

// --- one special Jacobian record {kind, instance, p1, p2}, c, added to D ----
// PRODUCTION contributions add, LOSS contributions subtract (Jacobian.c:
// 223-241 keeps them in separate long double sums and outputs prod - loss).
// s_part: the items' partials (mp_item_partials), or nullptr where they do not
// fit the scratch and are formed here.
__host__ __device__ __forceinline__ dd mp_jac_record(const DevProgram& P, int4 a, double c,
                                            const double* s_state, const double* s_part,
                                            const double* s_aero, const double* s_jsc, dd D) {
  const double* aq0 = s_jsc + kSpScalars * P.n_sp;
  if (a.x <= kJsSimpolAP) {
    const double* s = s_jsc + kSpScalars * a.y;
    double N = s[0], kp = s[1], kc = s[2];
    dd evap0 = {s[3], s[4]}, cond = {s[5], s[6]}, evap = {s[7], s[8]};
    double dcdr = s[9], dedr = s[10], dedm = s[11], dedw = s[12];
    switch (a.x) {
      case kJsSimpolGG:  // LOSS N * cond_rate
        D = dd_sub(D, dd_mul(dd_from(N), dd_from(kc)));
        break;
      case kJsSimpolAG:  // PRODUCTION N * cond_rate / kp
        D = dd_add(D, dd_div_d(dd_mul(dd_from(N), dd_from(kc)), kp));
        break;
      case kJsSimpolGA:  // PRODUCTION N * evap_rate * act
        D = dd_add(D, dd_mul(dd_from(N), evap0));
        break;
      case kJsSimpolAA:  // LOSS N * evap_rate * act / kp
        D = dd_sub(D, dd_div_d(dd_mul(dd_from(N), evap0), kp));
        break;
      default: {  // phase element: item a.w
        double numj, mwj;
        if (s_part) {
          numj = s_part[2 * a.w];
          mwj = s_part[2 * a.w + 1];
        } else {
          mp_item_partials(P, a.w, s_aero, numj, mwj);
        }
        double massj = 1.0;
        double radj = 0.0;
        // (a radius term is an exact zero unless its factor overflowed)
        auto term = [](dd d, double v) { return v == 0.0 ? d : dd_add(d, dd_from(v)); };
        if (a.x == kJsSimpolGP) {
          D = term(D, N * dedr * radj);
          D = term(D, -(N * dcdr * radj));
          D = dd_add(D, dd_mul(evap, dd_from(numj)));
          D = dd_sub(D, dd_mul(cond, dd_from(numj)));
          D = dd_add(D, dd_from(N * dedm * massj));
          D = dd_add(D, dd_from(N * dedw * mwj));
        } else {
          D = term(D, -(N * dedr / kp * radj));
          D = term(D, N * dcdr / kp * radj);
          D = dd_sub(D, dd_mul(dd{s[13], s[14]}, dd_from(numj)));
          D = dd_add(D, dd_mul(dd{s[15], s[16]}, dd_from(numj)));
          D = dd_sub(D, dd_from(N * dedm / kp * massj));
          D = dd_sub(D, dd_from(N * dedw / kp * mwj));
        }
      }
    }
    return D;
  }
  const double* s = aq0 + kAqScalars * a.y;
  if (s[5] != 0.0) return D;  // water below threshold: no contribution
  dd fwd = {s[0], s[1]}, rev = {s[2], s[3]};
  dd water = dd_from(s[4]);
  const int* sp = P.aq_sp + 6 * a.y;
  int nr = P.aq_nr[a.y], np = P.aq_np[a.y];
  switch (a.x) {
    case kJsAqRR:
      if (fwd.hi != 0.0) D = dd_sub(D, dd_mul(dd_div_d(dd_div_d(fwd, s_state[sp[a.z]]), c), water));
      break;
    case kJsAqRP:
      if (fwd.hi != 0.0) D = dd_add(D, dd_mul(dd_div_d(dd_div_d(fwd, s_state[sp[a.z]]), c), water));
      break;
    case kJsAqPR:
      if (rev.hi != 0.0) D = dd_add(D, dd_mul(dd_div_d(dd_div_d(rev, s_state[sp[a.z]]), c), water));
      break;
    case kJsAqPP:
      if (rev.hi != 0.0) D = dd_sub(D, dd_mul(dd_div_d(dd_div_d(rev, s_state[sp[a.z]]), c), water));
      break;
    case kJsAqRW:  // LOSS -fwd/m*(nr-1), PRODUCTION -rev/m*(np-1)
      D = dd_sub(D, dd_mul(dd_div_d(dd_neg(fwd), c), dd_from((double)(nr - 1))));
      D = dd_add(D, dd_mul(dd_div_d(dd_neg(rev), c), dd_from((double)(np - 1))));
      break;
    case kJsAqPW:  // PRODUCTION -fwd/m*(nr-1), LOSS -rev/m*(np-1)
      D = dd_add(D, dd_mul(dd_div_d(dd_neg(fwd), c), dd_from((double)(nr - 1))));
      D = dd_sub(D, dd_mul(dd_div_d(dd_neg(rev), c), dd_from((double)(np - 1))));
      break;
  }
  return D;
}

// --- per-cell LDS of the multi-phase extras ----------------------------------
struct MpLds {
  double *sub_env, *aero, *slot, *jsc, *jp;
};

// Per-cell extras kept in LDS (environment, aerosol state, f slots, the
// parameter Jacobian); the per-instance Jacobian scalars (used only while J
// is assembled) get their own mp_jsc_doubles(P) region, in LDS or in
// per-wavefront global scratch as the caller places it.
// The slots come last, before the per-term rates, so that both together serve
// as scratch (mp_scratch_doubles).  While J is assembled it holds the items'
// partials, where they fit.
__host__ __device__ inline bool mp_part(const DevProgram& P) {
  return 2 * (long)P.n_it <= (long)mp_scratch_doubles(P);
}
__host__ __device__ inline size_t mp_lds_doubles(const DevProgram& P) {
  if (!P.mp) return 0;
  return even_up((size_t)P.n_sub_env + kAeroSlots * (size_t)P.n_pi + P.pnnz) + mp_slot_doubles(P);
}
__host__ __device__ inline size_t mp_jsc_doubles(const DevProgram& P) {
  if (!P.mp) return 0;
  return kSpScalars * (size_t)P.n_sp + kAqScalars * (size_t)P.n_aq;
}

__device__ __forceinline__ MpLds mp_lds(const DevProgram& P, double* base, double* jsc) {
  MpLds L;
  L.sub_env = base;
  L.aero = L.sub_env + P.n_sub_env;
  L.jp = L.aero + kAeroSlots * P.n_pi;
  // (16-byte aligned: the f gather reads (hi, lo) pairs)
  L.slot = base + even_up((size_t)P.n_sub_env + kAeroSlots * (size_t)P.n_pi + P.pnnz);
  L.jsc = jsc;
  return L;
}

// sub_model_update_env_state for one cell: PPM_TO_RH of every ZSR model
__device__ __forceinline__ void mp_cell_env(const DevProgram& P, int lane, double T, double Pa,
                                            MpLds L) {
  for (int k = lane; k < P.n_sub_env; k += kWave) L.sub_env[k] = mp_ppm_to_rh(T, Pa);
  wsync();
}

// aero_rep_update_state then sub_model_calculate for one cell
// (camp_solver.c:913-917 in f(), 1065-1072 in Jac()): the representation
// caches mass, MW and number concentration from the water currently in the
// state, then ZSR writes the new water.  Jac() runs f() first, so its own
// update sees the water that f() left.
__device__ __forceinline__ void mp_refresh(const DevProgram& P, int lane, double* s_state, MpLds L) {
  lane = phase_lane(lane);
  mp_phase_sums(P, lane, s_state, L.aero, L.slot);
  for (int i = lane; i < P.n_pi; i += kWave) {
    double* a = L.aero + kAeroSlots * i;
    double mass_d = dd_round(dd{a[3], a[4]});
    a[0] = mass_d;
    a[1] = dd_round(dd_div(dd_from(mass_d), dd{a[5], a[6]}));
    double r = P.pi_dp[i] / 2.0;
    a[2] = a[7] * 3.0 / (4.0 * kPi) / cr_powi(r, 3);
  }
  wsync();
  mp_zsr(P, lane, L.sub_env, s_state, L.slot);
}

// The per-cell start of f(): refresh, then the contributions of the
// multi-phase reactions into their f slots.
__device__ __forceinline__ void mp_f_prologue(const DevProgram& P, int lane, double* s_state,
                                              const double* s_k, MpLds L) {
  lane = phase_lane(lane);
  mp_refresh(P, lane, s_state, L);
  for (int i = lane; i < P.n_sp; i += kWave) mp_simpol_f(P, i, s_state, s_k, L.aero, L.slot);
  for (int i = lane; i < P.n_aq; i += kWave) mp_aqeq_f(P, i, s_state, s_k, L.slot);
  wsync();
}

// After mp_f_prologue and the refresh of Jac(): the sums the partial derivatives use, the
// per-instance Jacobian scalars and the ZSR parameter Jacobian, whose
// element 0 is then set to 1 (the map's dummy, camp_solver.c:1099).
__device__ __forceinline__ void mp_j_prologue(const DevProgram& P, int lane, const double* s_state,
                                              const double* s_k, MpLds L) {
  lane = phase_lane(lane);
  mp_phase_sums(P, lane, s_state, L.aero, L.slot);
  for (int q = lane; q < P.pnnz; q += kWave) L.jp[q] = 0.0;
  wsync();
  mp_zsr_jac(P, lane, L.sub_env, s_state, L.jp, L.slot);
  // one division per item instead of one per record that uses it
  if (mp_part(P))
    for (int it = lane; it < P.n_it; it += kWave)
      mp_item_partials(P, it, L.aero, L.slot[2 * it], L.slot[2 * it + 1]);
  for (int i = lane; i < P.n_sp; i += kWave)
    mp_simpol_jscalars(P, i, s_state, s_k, L.aero, L.jsc + kSpScalars * i);
  for (int i = lane; i < P.n_aq; i += kWave)
    mp_aqeq_jscalars(P, i, s_state, s_k, L.jsc + kSpScalars * P.n_sp + kAqScalars * i);
  wsync();
  if (lane == 0) L.jp[0] = 1.0;
  wsync();
}

// One record of a J_rxn row stream (Program::mj_rec) added to D: a
// mass-action record as gj_acc adds it, a special record as mp_jac_record does,
// padding not at all.
__device__ __forceinline__ dd mp_jac_stream_record(const DevProgram& P, int4 a, int4 b,
                                                   const double* s_state, const double* s_k,
                                                   double h, const double* s_part,
                                                   const double* s_aero, const double* s_jsc,
                                                   dd D) {
  const double c = hilo_to_double(b.w, b.z);
  if (a.x == -1) {
    double v = s_k[a.y];
    if (a.z >= 0) v *= s_state[a.z];
    if (a.w >= 0) v *= s_state[a.w];
    if (c == -1.0) return dd_add(D, dd{-v, 0.0});
    const int g = b.y;
    if (g >= 0 && !(-v * s_state[b.x] * c * h <= s_state[g])) return D;
    return dd_add(D, dd{c * v, 0.0});
  }
  if (a.x == 0) return D;
  return mp_jac_record(P, a, c, s_state, s_part, s_aero, s_jsc, D);
}

// J of a multi-phase cell: the reaction Jacobian into Jr (global scratch,
// rnnz values), then J = J_rxn * J_params over the map (camp_solver.c:
// 1100-1106), one solver element per lane.
__device__ __forceinline__ void cell_jac_mp(const DevProgram& P, int lane, const double* s_state,
                                            const double* s_k, double h, MpLds L, double* Jr,
                                            double* J) {
  lane = phase_lane(lane);
  vm_drain();
  const double* part = mp_part(P) ? L.slot : nullptr;
  // elements in the program's order, whose rows share their record kinds;
  // each lane reads its element's records as a stream, the next record in
  // flight while the current one is added
  for (int r = 0; r < P.mj_rows; ++r) {
    const int e = P.mj_elist[r * kWave + lane];
    const int2 rh = ld_uniform(P.mj_rhdr, r);
    const int4* rec = P.mj_rec + 2 * ((size_t)rh.x * kWave + lane);
    dd D = {0.0, 0.0};
    int4 a = rec[0], b = rec[1];
    for (int k = 0; k < rh.y; ++k) {
      const int4 ca = a, cb = b;
      const int4* nx = rec + 2 * (size_t)(k + 1) * kWave;
      a = nx[0];
      b = nx[1];
      D = mp_jac_stream_record(P, ca, cb, s_state, s_k, h, part, L.aero, L.jsc, D);
    }
    if (e >= 0) Jr[e] = D.hi;
  }
  __threadfence_block();
  wsync();
  for (int e = lane; e < P.nnz; e += kWave) {
    double v = 0.0;
    for (int q = P.jm_ptr[e]; q < P.jm_ptr[e + 1]; ++q) v += Jr[P.jm_rxn[q]] * L.jp[P.jm_param[q]];
    J[e] = v;
  }
}
}  // namespace camp
