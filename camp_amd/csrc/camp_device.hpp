// Device-side building blocks shared by the plain-path kernels and the
// persistent per-cell BDF kernel.
//
// Execution model: one wavefront (64 lanes) owns one grid cell at a time.
// The cell's state, rate constants, BDF vectors and LU factors live in LDS;
// lanes split the work of each sparse phase (rate terms and species in
// f(y), Jacobian elements in J(y), entries of the LU factors in the
// factorisation, ready rows in the triangular solves).  Every decision that
// controls the cell's integration is made on wave-uniform values (lane 0's
// reduction result is broadcast), so a wavefront never diverges between
// cells and never needs a workgroup barrier.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "camp_dd.hpp"
#include "camp_model.hpp"

namespace camp {

constexpr int kWave = 64;
// doubles rounded up to whole 16-byte pairs
__host__ __device__ constexpr size_t even_up(size_t n) { return n + (n & 1); }

struct DevProgram {
  int ns, nv, nnz, n_env, n_terms, lu_nnz, n_rxn;
  const int* dep_state;
  const int *colptr, *rowval;  // solver pattern (dep ids, CSC)
  // lane-group f/J programs (gas-phase programs; Program::gf_rec), one per
  // group width (8, 16, 32 lanes per cell)
  int g_f_rows[3], g_j_rows[3], n_k, n_fzero;
  const int4 *gf_rec[3], *gj_rec[3];   // 2 int4 per record
  const int4* cj_rec;                  // per-cell J (Program::cj_rec), 2 int4 per record
  int cj_rows;
  const int *k_slot, *f_count, *f_zero;
  const int *r_ptr, *r_elem, *r_col;  // row view of the solver pattern
  int n_cs;                            // state variables that are not solver variables
  const int* cs_ids;
  const int *perm, *diag_pos;
  // LU factorisation (Program::lg_rec and following)
  int lu_d, lg_n;
  const int4* lg_rec;
  const int* lt_pos;
  // triangular solves (Program::tri_e and following)
  int tri_s, tri_d, tri_nf, tri_nb, tt_nf, tt_nb;
  const int4 *tri_e, *tt;
  const int2* tri_r;
  const int* fs_species;             // lane slot -> species of the f gather
  const int4* t_rec;                 // per term: {k index | flags << 28, reactants x3}
  int es_n;                          // f estimate (Program::es_hdr and following)
  const int4 *es_col, *es_fin;
  const int2* es_hdr;
  const int* es_src;
  int fb_rows, fb_nparts;            // balanced f gather: rows per lane, partials
  const int4* fb_rec;                // {index | target << 16, guard | flags << 24, coef}
  // rate-constant program (rxn_update_env_state)
  const int *rx_type, *rx_fidx, *rx_eidx, *rx_nreact;
  const double* rx_float;
  const double* abs_tol_dep;  // [nv]
  // multi-phase tables (mp == 0 for gas-phase programs); see Program in
  // camp_model.hpp for their meaning
  int mp, rnnz, pnnz, n_pi, n_zi, n_sp, n_aq, n_slots, n_sub_env;
  double min_mass_hi, min_mass_lo, min_moles_hi, min_moles_lo, min_volume;
  int n_it, n_zp;
  const int *pit_ptr, *pit_state, *pit_pi, *zp_zi;
  const double *pi_dp, *pit_mw, *pit_dens;
  const int *zi_water, *zi_gw, *zi_sub, *zi_pair_ptr, *zp_cat, *zp_an, *zp_ncat, *zp_nan, *zp_ny,
      *zp_jgw, *zp_jcat, *zp_jan;
  const double *zp_catmw, *zp_anmw, *zp_lowrh, *zp_y;
  const int *sp_gas, *sp_aero, *sp_dgas, *sp_daero, *sp_pi, *sp_env, *sp_flt, *sp_slot;
  const double* sp_radius;
  const int *aq_nr, *aq_np, *aq_sp, *aq_water, *aq_env, *aq_flt, *aq_slot;
  const double* aq_small_water;
  const int *jm_ptr, *jm_rxn, *jm_param;
  const int* mj_elist;  // J_rxn assembly order (Program::mj_elist)
  int mj_rows;
  const int4* mj_rec;   // the rows' record streams (Program::mj_rec), 2 int4 per record
  const int2* mj_rhdr;  // per row: first record row, records
};


// ---------------------------------------------------------------------
// Wavefront helpers
// ---------------------------------------------------------------------
// Orders the LDS (and global) accesses of one wavefront across lanes.  A
// wavefront's memory instructions are processed in program order, so a
// wavefront-scope fence needs no s_waitcnt: it only stops the compiler from
// moving memory operations across it, and outstanding global prefetches
// stay in flight.
__device__ __forceinline__ void wsync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
// Wait for every outstanding global load and store of the wavefront
// (s_waitcnt vmcnt(0); expcnt and lgkmcnt left open).  Placed in uniform
// control flow before a loop that keeps loads in flight across iterations:
// the compiler counts those loads exactly only when no store is pending on
// some path into the loop; with one pending (stores and loads complete in no
// fixed order) it waits for all loads at the top of every iteration, and
// the look-ahead hides nothing.
__device__ __forceinline__ void vm_drain() { __builtin_amdgcn_s_waitcnt(0x0F70); }
// The lane index made opaque to the compiler at the start of a phase (f, J,
// LU, solve): per-lane program addresses derived from it are then computed
// inside the phase instead of being hoisted to the kernel's start and held
// in registers through the whole solve (they raised the per-cell kernel's
// register use past the two-wavefront bound).
__host__ __device__ __forceinline__ int phase_lane(int lane) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(lane));
#endif
  return lane;
}
// A wave-uniform value made opaque the same way, in its scalar register.
__host__ __device__ __forceinline__ int phase_uniform(int v) {
#if defined(__HIP_DEVICE_COMPILE__)
  v = __builtin_amdgcn_readfirstlane(v);
  asm volatile("" : "+s"(v));
#endif
  return v;
}
// Read-only program data at a wave-uniform index through the scalar cache
// (the program is never written while a kernel runs): the value lands in
// scalar registers without a vector load and a wait on it.
// (Host builds of the shared routines read it directly.)
template <typename T>
__host__ __device__ __forceinline__ T ld_uniform(const T* p, int i) {
#if defined(__HIP_DEVICE_COMPILE__)
  return ((const __attribute__((address_space(4))) T*)p)[i];
#else
  return p[i];
#endif
}
// Wavefront reductions with DPP lane moves (no LDS round trip): quad
// butterflies, half-row and row mirrors give every lane its row's value,
// then row broadcasts of lanes 15 and 31 carry the rows into lane 63, whose
// value is read into a scalar register.  Rows a broadcast does not write
// keep the identity.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_i(int v, int id) {
  return __builtin_amdgcn_update_dpp(id, v, CTRL, ROWS, 0xF, false);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_d(double v, double id) {
  int lo = dpp_i<CTRL, ROWS>(__double2loint(v), __double2loint(id));
  int hi = dpp_i<CTRL, ROWS>(__double2hiint(v), __double2hiint(id));
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane63_d(double v) {
  int lo = __builtin_amdgcn_readlane(__double2loint(v), kWave - 1);
  int hi = __builtin_amdgcn_readlane(__double2hiint(v), kWave - 1);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sum(double v) {
  v += dpp_d<0xB1, 0xF>(v, 0.0);   // quad_perm [1,0,3,2]
  v += dpp_d<0x4E, 0xF>(v, 0.0);   // quad_perm [2,3,0,1]
  v += dpp_d<0x141, 0xF>(v, 0.0);  // row_half_mirror
  v += dpp_d<0x140, 0xF>(v, 0.0);  // row_mirror
  v += dpp_d<0x142, 0xA>(v, 0.0);  // row_bcast:15 into rows 1, 3
  v += dpp_d<0x143, 0xC>(v, 0.0);  // row_bcast:31 into rows 2, 3
  return lane63_d(v);
}
__device__ __forceinline__ double wave_min(double v) {
  const double inf = __builtin_huge_val();
  v = fmin(v, dpp_d<0xB1, 0xF>(v, inf));
  v = fmin(v, dpp_d<0x4E, 0xF>(v, inf));
  v = fmin(v, dpp_d<0x141, 0xF>(v, inf));
  v = fmin(v, dpp_d<0x140, 0xF>(v, inf));
  v = fmin(v, dpp_d<0x142, 0xA>(v, inf));
  v = fmin(v, dpp_d<0x143, 0xC>(v, inf));
  return lane63_d(v);
}
__device__ __forceinline__ int wave_or(int v) {
  v |= dpp_i<0xB1, 0xF>(v, 0);
  v |= dpp_i<0x4E, 0xF>(v, 0);
  v |= dpp_i<0x141, 0xF>(v, 0);
  v |= dpp_i<0x140, 0xF>(v, 0);
  v |= dpp_i<0x142, 0xA>(v, 0);
  v |= dpp_i<0x143, 0xC>(v, 0);
  return __builtin_amdgcn_readlane(v, kWave - 1);
}

constexpr double kPi = 3.14159265358979323846;
constexpr double kGasConst = 8.314472;  // util.h:17

// --- environment: SIMPOL and aqueous equilibrium (rxn env slots) ----------
// rxn_SIMPOL_phase_transfer_update_env_state (:220-266):
// e = [MFP_M, ALPHA, EQUIL_CONST, KGM3_TO_PPM]
__host__ __device__ __forceinline__ void mp_simpol_env(const double* f, double* e, double T, double Pa) {
  double alpha = 0.1;
  if (f[0] != 0.0 || f[1] != 0.0) {
    double del_g = f[0] - T * f[1];
    alpha = cr_exp(-del_g / (kGasConst * T));
    alpha = alpha / (1.0 + alpha);
  }
  e[1] = alpha;
  e[0] = 3.0 * f[2] / sqrt(8.0 * kGasConst * T / (kPi * f[9]));
  double vp = f[4] / T + f[5] + f[6] * T + f[7] * cr_log(T);
  vp = 101325.0 * cr_pow(10.0, vp);
  e[3] = f[8] * T / Pa;
  e[2] = vp / Pa / f[9] * 1.0e6;
}
// rxn_aqueous_equilibrium_update_env_state (:244-265): e = [k_forward]
__host__ __device__ __forceinline__ void mp_aqeq_env(const double* f, double* e, double T) {
  double k = f[1] == 0.0 ? f[0] : f[0] * cr_exp(f[1] * (1.0 / T - 1.0 / 298.0));
  e[0] = k * f[2];
}
// sub_model_ZSR_aerosol_water_update_env_state (:189-207): PPM_TO_RH
__host__ __device__ __forceinline__ double mp_ppm_to_rh(double T, double Pa) {
  double a = 1.0 - 373.15 / T;
  a = (((-0.1299 * a - 0.6445) * a - 1.976) * a + 13.3185) * a;
  return Pa / (101325.0 * cr_exp(a)) / 1.0e6;
}

// ---------------------------------------------------------------------
// Rate constants of one cell: rxn_update_env_state (rxn_solver.c:224-313)
// with rxn_arrhenius.c:103-118, rxn_troe.c:106-130, rxn_CMAQ_H2O2.c:
// 106-124, rxn_CMAQ_OH_HNO3.c:110-133, rxn_photolysis.c:137-147,
// rxn_emission.c:109-119, rxn_first_order_loss.c:119-129.
// env_cell points at the cell's rxn_env block (k slots written in place).
// ---------------------------------------------------------------------
__host__ __device__ __forceinline__ void rate_constant(const DevProgram& P, int r, double T, double Pa,
                                              double* env_cell) {
  const double* f = P.rx_float + P.rx_fidx[r];
  double* e = env_cell + P.rx_eidx[r];
  int t = P.rx_type[r];
  int nr = P.rx_nreact[r];
  if (t == 1) {  // ARRHENIUS
    e[0] = f[0] * cr_exp(f[2] / T) * (f[1] == 0.0 ? 1.0 : cr_pow(T / f[3], f[1])) *
           (f[4] == 0.0 ? 1.0 : (1.0 + f[4] * Pa)) * cr_pow(f[5] * Pa / T, (double)(nr - 1));
  } else if (t == 2) {  // TROE
    double conv = f[9] * Pa / T;
    double k0 = f[0] * (f[2] == 0.0 ? 1.0 : cr_exp(f[2] / T)) *
                (f[1] == 0.0 ? 1.0 : cr_pow(T / 300.0, f[1])) * conv;
    double kinf = k0 / (f[3] * (f[5] == 0.0 ? 1.0 : cr_exp(f[5] / T)) *
                        (f[4] == 0.0 ? 1.0 : cr_pow(T / 300.0, f[4])));
    double lg = cr_log10(kinf) / f[7];
    e[0] = (k0 / (1.0 + kinf)) * cr_pow(f[6], (1.0 / (1.0 + cr_pow(lg, 2.0)))) *
           cr_pow(conv, (double)(nr - 1)) * f[8];
  } else if (t == 3) {  // CMAQ_H2O2: (k1 + k2 [M]) conv^(nr-1), [M] in k2_A
    double conv = f[6] * Pa / T;
    e[0] = (f[0] * (f[2] == 0.0 ? 1.0 : cr_exp(f[2] / T)) *
                (f[1] == 0.0 ? 1.0 : cr_pow(T / 300.0, f[1])) +
            f[3] * (f[5] == 0.0 ? 1.0 : cr_exp(f[5] / T)) *
                (f[4] == 0.0 ? 1.0 : cr_pow(T / 300.0, f[4])) * conv) *
           cr_pow(conv, (double)(nr - 1));
  } else if (t == 4) {  // CMAQ_OH_HNO3: (k0 + k3 / (1 + k3 / k2)) conv^(nr-1) SCALING
    double conv = f[10] * Pa / T;
    double k2 = f[3] * (f[5] == 0.0 ? 1.0 : cr_exp(f[5] / T)) *
                (f[4] == 0.0 ? 1.0 : cr_pow(T / 300.0, f[4]));
    double k3 = f[6] * (f[8] == 0.0 ? 1.0 : cr_exp(f[8] / T)) *
                (f[7] == 0.0 ? 1.0 : cr_pow(T / 300.0, f[7])) * conv;
    e[0] = (f[0] * (f[2] == 0.0 ? 1.0 : cr_exp(f[2] / T)) *
                (f[1] == 0.0 ? 1.0 : cr_pow(T / 300.0, f[1])) +
            k3 / (1.0 + k3 / k2)) *
           cr_pow(conv, (double)(nr - 1)) * f[9];
  } else if (t == 10) {  // SIMPOL_PHASE_TRANSFER
    mp_simpol_env(f, e, T, Pa);
  } else if (t == 7) {  // AQUEOUS_EQUILIBRIUM
    mp_aqeq_env(f, e, T);
  } else {  // PHOTOLYSIS, EMISSION, FIRST_ORDER_LOSS: SCALING * BASE_RATE
    e[0] = f[0] * e[1];
  }
}

// All rate constants of one cell, lanes over reactions.
__device__ __forceinline__ void cell_rate_constants(const DevProgram& P, int lane, double T, double Pa,
                                                 double* s_k) {
  for (int r = lane; r < P.n_rxn; r += kWave) rate_constant(P, r, T, Pa, s_k);
}

// ---------------------------------------------------------------------
// f(y) of one cell: per-type calc_deriv_contrib + time_derivative_output
// (camp_solver.c:901-954, time_derivative.c:46-97).  s_state holds the
// cell state with the solver variables already substituted, s_k the
// cell's rxn_env block.  Lane i handles species i, i+64, ...: it gathers
// its signed contributions into a double-double D (= production - loss)
// and their magnitudes into S (= production + loss).
// est != nullptr selects the Jacobian-extrapolated blend; est is then
// computed from the cell's J history (J_deriv + J_solver (y - J_state)).
// ---------------------------------------------------------------------
// Phase 1 of f(y): the rate of every term (reaction) once, into s_rate
// (n_terms double-doubles): k * prod(reactants) as the per-type
// calc_deriv_contrib computes it (rxn_arrhenius.c:143-147 and alike);
// first-order loss rounds k * y to double (rxn_first_order_loss.c:150).
// What f(y) reads of the program before any of it depends on y: the lane's
// first terms, the first records of its gather bin and the first batches of
// the estimate.  Loaded ahead of f's start, so that one trip to the caches
// covers what were five, one after another (each 300 to 600 cycles of the
// 13000 of a gas-phase f).
constexpr int kTermRegs = 4;
constexpr int kEstSets = 4, kEstAhead = 2;  // register sets; batches whose values are ahead
// One batch of the estimate's stream: the lane's columns, {position of its
// first value, stride between entries | (pass the batch ends + 1) << 16} and
// the values.  (The header comes by lane: a scalar load would be waited on at
// once.)
struct EstBatch {
  int4 c;
  int2 h;
  double v[kEstBatch];
};
struct FLoad {
  int4 tr[kTermRegs], a[4], fin;
  EstBatch B[kEstSets];
};
__device__ __forceinline__ void est_prog(const DevProgram& P, int lane, int n, EstBatch& S) {
  S.c = P.es_col[(size_t)n * kWave + lane];
  S.h = P.es_hdr[(size_t)n * kWave + lane];
}
__device__ __forceinline__ void f_load_terms(const DevProgram& P, int lane, FLoad& F) {
  lane = phase_lane(lane);
#pragma unroll
  for (int g = 0; g < kTermRegs; ++g) {
    int t = lane + g * kWave;
    F.tr[g] = t < P.n_terms ? P.t_rec[t] : make_int4(0, -1, -1, -1);
  }
}
__device__ __forceinline__ void f_load_gather(const DevProgram& P, int lane, FLoad& F) {
  lane = phase_lane(lane);
#pragma unroll
  for (int g = 0; g < 4; ++g) F.a[g] = P.fb_rec[g * kWave + lane];
#pragma unroll
  for (int u = 0; u < kEstSets; ++u) est_prog(P, lane, u, F.B[u]);
  F.fin = P.es_fin[lane];
}

// KT: the constants of a lane's first kTermRegs terms are in its registers
// (kt), the others' in global memory.
template <bool KT = false>
__device__ __forceinline__ void cell_rates(const DevProgram& P, int lane, const double* s_state,
                                           const double* s_k, double* s_rate, const FLoad& F,
                                           const double* kt = nullptr) {
  lane = phase_lane(lane);
  // a lane's terms in groups of four whose program loads are issued together
  constexpr int TG = kTermRegs;
  for (int t0 = lane; t0 < P.n_terms; t0 += TG * kWave) {
    int4 tr[TG];
#pragma unroll
    for (int g = 0; g < TG; ++g) {
      int t = t0 + g * kWave;
      tr[g] = F.tr[g];
      if (t0 != lane) tr[g] = t < P.n_terms ? P.t_rec[t] : make_int4(0, -1, -1, -1);
    }
#pragma unroll
    for (int g = 0; g < TG; ++g) {
      int t = t0 + g * kWave;
      if (t >= P.n_terms) break;
      int fl = tr[g].x >> 28;
      double k = KT && t0 == lane ? kt[g] : s_k[tr[g].x & 0x0FFFFFFF];
      double y0 = s_state[tr[g].y >= 0 ? tr[g].y : 0], y1 = s_state[tr[g].z >= 0 ? tr[g].z : 0],
             y2 = s_state[tr[g].w >= 0 ? tr[g].w : 0];
      dd rate = {k, 0.0};
      if (fl & 2) {
        rate = {k * y0, 0.0};
      } else {
        rate = tr[g].y >= 0 ? dd_mul_d(rate, y0) : rate;
        rate = tr[g].z >= 0 ? dd_mul_d(rate, y1) : rate;
        rate = tr[g].w >= 0 ? dd_mul_d(rate, y2) : rate;
      }
      reinterpret_cast<double2*>(s_rate)[t] = make_double2(rate.hi, rate.lo);
    }
  }
}

// The double whose high and low 32-bit words are hi and lo.
__host__ __device__ __forceinline__ double hilo_to_double(int hi, int lo) {
  unsigned long long b = ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo;
  return __builtin_bit_cast(double, b);
}

// LDS scratch of the f gather: per species value and magnitude sum, the
// partials of split species (hi, lo, magnitudes) and a spare partial that
// padding records write to.
__host__ __device__ inline size_t fb_lds_doubles(const DevProgram& P) {
  return 2 * (size_t)P.nv + 3 * ((size_t)P.fb_nparts + 1);
}
// The per-cell kernel places the f gather's scratch right after the LU
// values, where it also serves as the zero slot of the factorisation and the
// triangular solve (the 65th) and as the factorisation's tail buffers.
// the LU tail's buffers: a pivot's row and column, 8 groups of up to 5 doubles
constexpr int kLuTailStride = kLuTail / 8 + 1, kLuTailBuf = 2 * 8 * kLuTailStride;
__host__ __device__ inline size_t fb_scratch_doubles(const DevProgram& P) {
  size_t n = fb_lds_doubles(P);
  const size_t m = kLuTailBuf > kWave + 1 ? kLuTailBuf : kWave + 1;
  return n > m ? n : m;
}

// One record of the f gather, without branches: the term's rate (or a
// multi-phase slot value, whose coefficient is 1) times the yield (or -1),
// unless the record fails the negative-yield guard -rate * yield * h <=
// y[guard] (rxn_arrhenius.c:157 and alike), in which case its coefficient
// is zero.
// The product of the double-double rate and the coefficient is p + e
// (exact up to the rounding of lo * c); p joins the running sum Dh with an
// error-free TwoSum whose error, with e, goes to Dl, so Dh + Dl is the
// record sum to about 2^-100 of the magnitudes S (the reference's long
// double production/loss sums keep 2^-64).  A piece's last record (flag 16)
// stores the sums at the piece's target and restarts them from zero.
struct FOps {
  double hi, lo, sg;
};
__device__ __forceinline__ FOps f_operands(int4 rec, const double* s_state,
                                           const double* s_rate, const double* s_slot) {
  int flags = (int)((unsigned)rec.y >> 24);
  int g = (rec.y << 8) >> 8;  // sign-extended 24-bit guard (-1 = none)
  const double* src = (flags & 4) ? s_slot : s_rate;
  int idx = rec.x & 0xFFFF;
  FOps o;
  const double2 v = reinterpret_cast<const double2*>(src)[idx];  // (16-byte aligned)
  o.hi = v.x;
  o.lo = v.y;
  o.sg = s_state[g >= 0 ? g : 0];
  return o;
}
__host__ __device__ __forceinline__ void f_record(int4 rec, FOps o, double h, int nv, double* s_fb,
                                         double& Dh, double& Dl, double& S) {
  int flags = (int)((unsigned)rec.y >> 24);
  int g = (rec.y << 8) >> 8;
  double c = hilo_to_double(rec.w, rec.z);
  // (padding has coefficient 0 and no guard; a zero-rate term flagged 1
  // adds zero, as the reference's skip does)
  bool keep = g < 0 || -o.hi * c * h <= o.sg;
  c = keep ? c : 0.0;
  double p = o.hi * c;
  double e = fma(o.hi, c, -p);
  e = fma(o.lo, c, e);
  double s = Dh + p;
  double bb = s - Dh;
  double err = (Dh - (s - bb)) + (p - bb);
  Dh = s;
  Dl = Dl + (err + e);
  S += fabs(p);
  // whole species: value Dh + Dl at [t], S at [nv + t]; partial: (Dh, Dl,
  // S) at [t], [t + 1], [t + 2] (the lo store first, so that for a whole
  // species the value overwrites it)
  if (flags & 16) {
    int t = (int)((unsigned)rec.x >> 16);
    bool part = flags & 32;
    s_fb[part ? t + 1 : t] = Dl;
    s_fb[t] = part ? Dh : Dh + Dl;
    s_fb[part ? t + 2 : nv + t] = S;
    Dh = 0.0;
    Dl = 0.0;
    S = 0.0;
  }
}

// The f estimate's J history in the order its stream reads it (Program::es_hdr),
// then J_deriv by lane slot: est_doubles(P) doubles of the wavefront's scratch,
// refreshed with the history.  An entry per lane is then one run of
// consecutive doubles; read in place the elements were a cache line each (8
// lines an instruction against 64).
__host__ __device__ inline size_t est_doubles(const DevProgram& P) {
  return (size_t)P.es_n + (size_t)(P.nv + kWave - 1) / kWave * kWave;
}
__device__ __forceinline__ void est_stage(const DevProgram& P, int lane, const double* Js,
                                          const double* Jf, double* E) {
  lane = phase_lane(lane);
  // eight elements a lane at a time, the loads of each kind together (one after
  // another they are two trips to the caches per row of 64)
  constexpr int B = 8;
  for (int p0 = lane; p0 < P.es_n; p0 += B * kWave) {
    int e[B];
    double v[B];
#pragma unroll
    for (int u = 0; u < B; ++u) e[u] = P.es_src[min(p0 + u * kWave, P.es_n - 1)];
#pragma unroll
    for (int u = 0; u < B; ++u) v[u] = Js[e[u] >= 0 ? e[u] : 0];
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (p0 + u * kWave < P.es_n) E[p0 + u * kWave] = e[u] >= 0 ? v[u] : 0.0;
  }
  for (int s = lane; s < P.nv; s += kWave) E[P.es_n + s] = Jf[P.fs_species[s]];
  __threadfence_block();
  wsync();
}

// (STAGED: values in the stream's order, else the Jacobian's elements)
template <bool STAGED>
__device__ __forceinline__ void est_vals(const DevProgram& P, const double* Js, EstBatch& S) {
  int p = S.h.x;
  const int stride = S.h.y & 0xFFFF;
#pragma unroll
  for (int u = 0; u < kEstBatch; ++u, p += stride) {
    if (STAGED) {
      S.v[u] = Js[p];
    } else {
      const int e = P.es_src[p];
      S.v[u] = Js[e >= 0 ? e : 0];
    }
  }
}

// f(y) after cell_rates and a wave sync.  Phase 2: every lane walks its bin
// of fb_rows records (pieces of species' record lists, packed so that the
// lanes' bins are balanced) accumulating Dh + Dl (= production - loss,
// replacing CAMP's long double production/loss sums) and S (the
// magnitudes), with the next four records in flight while the current four
// are processed and each batch's LDS operands read before the batch is
// accumulated.  Phase 3: lane per species, the pieces of a split species
// are added in order, the Jacobian-based estimate J_hist (y - y_hist) +
// f_hist is formed (a stream of batches over the rows, y - y_hist once per
// species in dy), and the precision-loss blend of time_derivative.c:58-64
// gives f.  s_fb is LDS scratch of fb_lds_doubles, dy (use_est) of nv.
// STAGED: Js is est_stage's copy of the history (Jf unused).  DY: with dy; a
// program whose dy does not fit LDS forms y - y_hist for every entry.
template <bool STAGED, bool DY = true>
__device__ __forceinline__ void cell_deriv(const DevProgram& P, int lane, const double* s_state,
                                           const double* s_rate, const double* y,
                                           const double* Js, const double* Jy,
                                           const double* Jf, bool use_est, double h,
                                           double* out, double* s_fb, double* dy, FLoad& F,
                                           const double* s_slot = nullptr) {
  lane = phase_lane(lane);
  const int nv = P.nv, L = P.fb_rows;
  // (no solver variables: the estimate's stream is empty, and ends nowhere)
  use_est = use_est && nv > 0;
  const double* slot_or_rate = s_slot ? s_slot : s_rate;
  double jf = 0.0;
  if (use_est) {
#pragma unroll
    for (int u = 0; u < kEstAhead; ++u) est_vals<STAGED>(P, Js, F.B[u]);
    jf = STAGED ? Js[P.es_n + lane] : F.fin.x >= 0 ? Jf[F.fin.x] : 0.0;
    if (DY)
      for (int i = lane; i < nv; i += kWave) dy[i] = y[i] - Jy[i];
  }
  {
    const int4* fr = P.fb_rec + lane;
    // fb_rec has padding rows up to a multiple of 4 plus 4 beyond fb_rows
    int4 a0 = F.a[0], a1 = F.a[1], a2 = F.a[2], a3 = F.a[3];
    double Dh = 0.0, Dl = 0.0, S = 0.0;
    for (int j = 0; j < L; j += 4) {
      int4 c0 = a0, c1 = a1, c2 = a2, c3 = a3;
      a0 = fr[(j + 4) * kWave];
      a1 = fr[(j + 5) * kWave];
      a2 = fr[(j + 6) * kWave];
      a3 = fr[(j + 7) * kWave];
      FOps o0 = f_operands(c0, s_state, s_rate, slot_or_rate),
           o1 = f_operands(c1, s_state, s_rate, slot_or_rate),
           o2 = f_operands(c2, s_state, s_rate, slot_or_rate),
           o3 = f_operands(c3, s_state, s_rate, slot_or_rate);
      f_record(c0, o0, h, nv, s_fb, Dh, Dl, S);
      f_record(c1, o1, h, nv, s_fb, Dh, Dl, S);
      f_record(c2, o2, h, nv, s_fb, Dh, Dl, S);
      f_record(c3, o3, h, nv, s_fb, Dh, Dl, S);
    }
  }
  wsync();
  const double* part = s_fb + 2 * nv;
  // a species' value from its pieces, blended with its estimate
  auto finish = [&](int4 fin, double jf, double acc) {
    const int i = fin.x;
    if (i < 0) return;
    double Dhi = 0.0, S = 0.0;
    if (fin.z == 0) {
      Dhi = s_fb[i];
      S = s_fb[nv + i];
    } else if (fin.z > 0) {
      // the partials' (hi, lo) pairs are not normalised: TwoSum each first
      dd D = two_sum(part[3 * fin.y], part[3 * fin.y + 1]);
      S = part[3 * fin.y + 2];
      for (int k = 1; k < fin.z; ++k) {
        const double* q = part + 3 * (fin.y + k);
        D = dd_add(D, two_sum(q[0], q[1]));
        S += q[2];
      }
      Dhi = D.hi;
    }
    double v = 0.0;
    if (S != 0.0) {
      if (use_est) {
        double est = jf + acc;
        double inv = 1.0 / S;
        double sf = inv / (inv + 1.0e-14 / fabs(Dhi));
        v = sf * Dhi + (1.0 - sf) * est;
      } else {
        v = Dhi;
      }
    }
    out[i] = v;
  };
  if (!use_est) {
    for (int slot = lane; slot < (nv + kWave - 1) / kWave * kWave; slot += kWave)
      finish(P.es_fin[slot], 0.0, 0.0);
    return;
  }
  constexpr int NS = kEstSets, AH = kEstAhead;
  EstBatch(&B)[NS] = F.B;
  int4 fin = F.fin;
  double acc = 0.0;
  for (int n = 0;; n += NS) {
#pragma unroll
    for (int u = 0; u < NS; ++u) {
      EstBatch& S = B[u];
      est_vals<STAGED>(P, Js, B[(u + AH) % NS]);
      const int cw[4] = {S.c.x, S.c.y, S.c.z, S.c.w};
      double d[kEstBatch];
#pragma unroll
      for (int q = 0; q < kEstBatch; ++q) {
        const int col = q % 2 ? (unsigned)cw[q / 2] >> 16 : cw[q / 2] & 0xFFFF;
        const int at = col == 0xFFFF ? 0 : col;
        d[q] = DY ? dy[at] : y[at] - Jy[at];
      }
      __builtin_amdgcn_sched_barrier(0);  // (the loads ahead of their uses)
#pragma unroll
      for (int q = 0; q < kEstBatch; ++q) {
        const int col = q % 2 ? (unsigned)cw[q / 2] >> 16 : cw[q / 2] & 0xFFFF;
        const double t = acc + S.v[q] * d[q];
        acc = col == 0xFFFF ? acc : t;
      }
      const int pass = (__builtin_amdgcn_readfirstlane(S.h.y) >> 16) - 1;
      if (pass >= 0) {
        finish(fin, jf, acc);
        acc = 0.0;
        const int next = (pass + 1) * kWave;
        if (next >= nv) return;
        fin = P.es_fin[next + lane];
        jf = STAGED ? Js[P.es_n + next + lane] : fin.x >= 0 ? Jf[fin.x] : 0.0;
      }
      est_prog(P, lane, n + u + NS, S);
    }
  }
}

// camp_solver_update_model_state (camp_solver.c:805-833) for one cell:
// returns 1 (wave-uniform) if any y < -SMALL, else copies y into s_state.
__device__ __forceinline__ int cell_set_state(const DevProgram& P, int lane, const double* y,
                                              double* s_state) {
  lane = phase_lane(lane);
  constexpr int R = 2;  // rows a lane keeps between the check and the copy
  double v[R];
  int to[R], bad = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = lane + r * kWave;
    v[r] = i < P.nv ? y[i] : 0.0;
    to[r] = i < P.nv ? P.dep_state[i] : -1;
    bad |= v[r] < -1.0e-30;
  }
  for (int i = lane + R * kWave; i < P.nv; i += kWave) bad |= (y[i] < -1.0e-30);
  bad = wave_or(bad);
  if (bad) return 1;
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (to[r] >= 0) s_state[to[r]] = v[r] > -1.0e-30 ? v[r] : 1.0e-60;
  for (int i = lane + R * kWave; i < P.nv; i += kWave) {
    double w = y[i];
    s_state[P.dep_state[i]] = w > -1.0e-30 ? w : 1.0e-60;
  }
  wsync();
  return 0;
}

// ---------------------------------------------------------------------
// J(y) of one cell into the solver Jacobian (CSC element order): per-type
// calc_jac_contrib + jacobian_output + jac_map (camp_solver.c:1052-1106,
// Jacobian.c:223-241).
// ---------------------------------------------------------------------
// Operands of one J record.
struct GjOps {
  int e, last, g, h1, h2;
  double coef, k, y1, y2, yw, sg;
};
__device__ __forceinline__ GjOps gj_ops(int4 x, int4 w, const double* sy, const double* sk) {
  GjOps o;
  o.e = x.x & 0x3FFFFFFF;
  o.last = (x.x >> 30) & 1;
  o.g = x.y;
  o.coef = hilo_to_double(x.w, x.z);
  o.h1 = w.y >= 0;
  o.h2 = w.z >= 0;
  o.k = sk[w.x];
  o.y1 = sy[o.h1 ? w.y : 0];
  o.y2 = sy[o.h2 ? w.z : 0];
  o.yw = sy[w.w >= 0 ? w.w : 0];
  o.sg = sy[o.g >= 0 ? o.g : 0];
  return o;
}
// One J record: k * the other reactants; loss records (coefficient -1)
// unguarded, others guarded (rxn_arrhenius.c:186-207 and alike); the
// element's double-double sum stored after its last record.  A guarded
// record that fails adds an exact zero, which leaves the sum as skipping it
// would.
__device__ __forceinline__ void gj_acc(const GjOps& o, double h, int nnz, double* Jc, dd& D) {
  double v = o.k;
  if (o.h1) v *= o.y1;
  if (o.h2) v *= o.y2;
  double add;
  if (o.coef == -1.0) {
    add = -v;
  } else {
    bool keep = o.g < 0 || -v * o.yw * o.coef * h <= o.sg;
    add = keep ? o.coef * v : 0.0;
  }
  D = dd_add(D, dd{add, 0.0});
  if (o.last) {
    if (o.e < nnz) Jc[o.e] = D.hi;
    D = dd{0.0, 0.0};
  }
}

// J(y) of one gas-phase cell: lane j walks its run of whole elements in the
// per-cell J program (runs of near-equal record counts), four records in
// flight while the current four are accumulated, and writes each element
// after its last record.
__device__ __forceinline__ void cell_jac(const DevProgram& P, int lane, const double* s_state,
                                         const double* s_k, double h, double* J) {
  lane = phase_lane(lane);
  vm_drain();
  const int nnz = P.nnz;
  constexpr int RS = 2 * kWave;
  const int4* rec = P.cj_rec + 2 * lane;
  dd D = {0.0, 0.0};
  // the program has 4 rows of padding past cj_rows for the look-ahead
  int4 a0 = rec[0], b0 = rec[1], a1 = rec[RS], b1 = rec[RS + 1];
  int4 a2 = rec[2 * RS], b2 = rec[2 * RS + 1], a3 = rec[3 * RS], b3 = rec[3 * RS + 1];
  for (int r = 0; r < P.cj_rows; r += 4) {
    int4 x0 = a0, w0 = b0, x1 = a1, w1 = b1, x2 = a2, w2 = b2, x3 = a3, w3 = b3;
    const int4* nx = rec + (size_t)(r + 4) * RS;
    a0 = nx[0]; b0 = nx[1]; a1 = nx[RS]; b1 = nx[RS + 1];
    a2 = nx[2 * RS]; b2 = nx[2 * RS + 1]; a3 = nx[3 * RS]; b3 = nx[3 * RS + 1];
    GjOps o0 = gj_ops(x0, w0, s_state, s_k), o1 = gj_ops(x1, w1, s_state, s_k),
          o2 = gj_ops(x2, w2, s_state, s_k), o3 = gj_ops(x3, w3, s_state, s_k);
    gj_acc(o0, h, nnz, J, D);
    gj_acc(o1, h, nnz, J, D);
    gj_acc(o2, h, nnz, J, D);
    gj_acc(o3, h, nnz, J, D);
  }
}

// ---------------------------------------------------------------------
// Sparse LU of M = I - gamma*J (SUNMatScaleAddI) with the static pivot
// order of the program.  Returns 1 on a zero or non-finite pivot (a
// recoverable linear-setup failure).  lu holds lu_nnz values and, at lu_nnz +
// 64, the zero slot; buf is LDS scratch of kLuTailBuf doubles.
//
// One pivot after another, the factorisation is nv dependent steps whose lists
// of updates are read from L2 as they come up (1300 cycles a pivot for the
// CB05-scale mechanism, 2300 to 5000 for multi-phase cells, whose LU lives in
// global memory).  The elimination order has far fewer levels (46 of 72, 65 of
// 304 pivots), and most of them are the dense last pivots.  So every LU value is
// a task -- its products in pivot order, the same operations the pivot-wise
// elimination does on it, so the values are the same bit for bit -- and the
// host packs the tasks into groups of 64 lanes, longest chain first, each at
// least kLuDist groups after the values it reads are stored: a group's
// operands are loaded while the one before it runs.  The last lu_d pivots
// (up to kLuTail) are a dense block in registers (lane l holds rows 8 a + l / 8 and columns
// 8 b + l % 8), a pivot's row and column going through LDS.
// Cycles per factorisation: one CB05-scale cell 84k -> 49k (2000 cells 95k ->
// 55k), CB05cl_ae5 66k -> 21k, one multi-phase cell 743k -> 339k (1024 cells
// 1.60M -> 0.57M); half of the gas one is tasks, the rest the register block (a
// pivot: an LDS round trip, a division and up to 25 products, 350 to 850).
// ---------------------------------------------------------------------
struct LuGroup {
  int4 r, h;
  double src, a[4], b[4], dg;
};
__device__ __forceinline__ void lu_prog(const DevProgram& P, int lane, int n, LuGroup& S) {
  S.r = P.lg_rec[(size_t)(2 * n) * kWave + lane];
  S.h = P.lg_rec[(size_t)(2 * n + 1) * kWave + lane];
}
__device__ __forceinline__ void lu_src(const double* J, LuGroup& S) {
  S.src = J[S.h.x >= 0 ? S.h.x : 0];
}
__device__ __forceinline__ void lu_vals(const double* lu, LuGroup& S) {
  const int e[4] = {S.r.x, S.r.y, S.r.z, S.r.w};
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    S.a[u] = lu[e[u] & 0xFFFF];
    S.b[u] = lu[(unsigned)e[u] >> 16];
  }
  S.dg = lu[(unsigned)S.h.y >> 16];
}
// One group: the tasks' next four products; acc carries a task that goes on.
__device__ __forceinline__ void lu_run(const LuGroup& S, double gamma, double* lu, double& acc,
                                       bool& bad) {
  const int fl = S.h.z;
  double v = S.h.x >= 0 ? -gamma * S.src : 0.0;
  v = (fl & 8) ? v + 1.0 : v;
  acc = (fl & 1) ? v : acc;
#pragma unroll
  for (int u = 0; u < 4; ++u) acc = acc - S.a[u] * S.b[u];
  const double scaled = acc * (1.0 / S.dg);
  acc = (fl & 4) ? scaled : acc;
  if (fl & 2) {
    // (a pivot of the register block is checked there)
    bad |= (fl & 16) && !(acc != 0.0 && isfinite(acc));
    lu[S.h.y & 0xFFFF] = acc;
  }
  wsync();
}

// The block of the last lu_d pivots in memory, pivot by pivot, products of its
// entries only.  The dense elimination below also multiplies entries the pattern
// does not have; as zeros they change nothing unless a value is not finite.
__device__ __forceinline__ bool lu_tail_sparse(const DevProgram& P, int lane, double* lu) {
  const int d = P.lu_d, nb = (d + 7) / 8, r = lane >> 3, c = lane & 7;
  auto at = [&](int i, int j) {
    return i < d && j < d ? P.lt_pos[((i >> 3) * nb + (j >> 3)) * kWave + (i & 7) * 8 + (j & 7)]
                          : -1;
  };
  bool bad = false;
#pragma nounroll
  for (int k = 0; k < d; ++k) {
    const double piv = lu[at(k, k)];
    bad |= !(piv != 0.0 && isfinite(piv));
    const double rinv = 1.0 / piv;
    wsync();
#pragma nounroll
    for (int i = k + 1 + lane; i < d; i += kWave) {
      const int p = at(i, k);
      if (p >= 0) lu[p] = lu[p] * rinv;
    }
    wsync();
#pragma nounroll
    for (int b = (k >> 3) * (nb + 1); b < nb * nb; ++b) {
      const int i = 8 * (b / nb) + r, j = 8 * (b % nb) + c;
      if (i <= k || j <= k) continue;
      const int p = at(i, j), l = at(i, k), u = at(k, j);
      if (p >= 0 && l >= 0 && u >= 0) lu[p] = lu[p] - lu[l] * lu[u];
    }
    wsync();
  }
  return bad;
}

// The dense block of the last lu_d pivots, NB blocks of 8.  Returns whether a
// pivot is zero or not finite; EXACT: or any value, and then stores nothing.  A pivot's row and
// column go through LDS (buf) by lane: the NB values a lane needs of either are
// consecutive.
template <int NB, bool EXACT>
__device__ __forceinline__ bool lu_tail(const DevProgram& P, int lane, double* lu, double* buf) {
  constexpr int W = kLuTailStride;  // doubles per lane group of 8
  const int d = P.lu_d, r = lane >> 3, c = lane & 7;
  double a[NB][NB];
#pragma unroll
  for (int p = 0; p < NB; ++p)
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int at = P.lt_pos[(NB * p + q) * kWave + lane];
      a[p][q] = lu[at >= 0 ? at : P.lu_nnz + kWave];
    }
  double *ub = buf, *lb = buf + 8 * W;
  wsync();
  bool bad = false;
#pragma unroll
  for (int kp = 0; kp < NB; ++kp) {
    for (int kr = 0; kr < 8; ++kr) {
      if (8 * kp + kr >= d) break;
      if (r == kr) {
#pragma unroll
        for (int q = kp; q < NB; ++q) ub[W * c + q] = a[kp][q];
      }
      if (c == kr) {
#pragma unroll
        for (int p = kp; p < NB; ++p) lb[W * r + p] = a[p][kp];
      }
      wsync();
      const double piv = ub[W * kr + kp];
      double l[NB], u[NB];
#pragma unroll
      for (int p = kp; p < NB; ++p) {
        l[p] = lb[W * r + p];
        u[p] = ub[W * c + p];
      }
      bad |= !(piv != 0.0 && isfinite(piv));
      const double rinv = 1.0 / piv;
#pragma unroll
      for (int p = kp; p < NB; ++p) l[p] = l[p] * rinv;
#pragma unroll
      for (int p = kp; p < NB; ++p)
#pragma unroll
        for (int q = kp; q < NB; ++q) {
          const double v = a[p][q] - l[p] * u[q];
          a[p][q] = (p > kp || r > kr) && (q > kp || c > kr) ? v : a[p][q];
        }
      // the pivot's column keeps the scaled values
#pragma unroll
      for (int p = kp; p < NB; ++p) a[p][kp] = c == kr && (p > kp || r > kr) ? l[p] : a[p][kp];
      wsync();
    }
  }
  if (EXACT) {
#pragma unroll
    for (int p = 0; p < NB; ++p)
#pragma unroll
      for (int q = 0; q < NB; ++q) bad |= !isfinite(a[p][q]);
    if (__builtin_amdgcn_ballot_w64(bad) != 0) return true;
  }
#pragma unroll
  for (int p = 0; p < NB; ++p)
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int at = P.lt_pos[(NB * p + q) * kWave + lane];
      if (at >= 0) lu[at] = a[p][q];
    }
  wsync();
  return bad;
}

// EXACT: the block entry by entry where a value is not finite (lu_tail_sparse).
// The integrator does without: to it such factors are a failed set-up as a bad
// pivot is, and the code costs it registers (1 to 2 % of a step).
template <bool EXACT>
__device__ __forceinline__ int cell_lu_factor(const DevProgram& P, int lane, const double* J,
                                              double gamma, double* lu, double* buf) {
  lane = phase_lane(lane);
  if (lane == 0) lu[P.lu_nnz + kWave] = 0.0;
  wsync();
  vm_drain();
  constexpr int NS = 4;  // register sets (NS <= kLuPad)
  LuGroup S[NS];
  double acc = 0.0;
  bool bad = false;
#pragma unroll
  for (int u = 0; u < NS; ++u) lu_prog(P, lane, u, S[u]);
  lu_src(J, S[0]);
  lu_src(J, S[1]);
  lu_vals(lu, S[0]);
  bool done = P.lg_n == 0;
  for (int n = 0; !done; n += NS) {
#pragma unroll
    for (int u = 0; u < NS; ++u) {
      if (n + u >= P.lg_n) {
        done = true;
        break;
      }
      lu_vals(lu, S[(u + 1) % NS]);
      lu_src(J, S[(u + 2) % NS]);
      __builtin_amdgcn_sched_barrier(0);  // (the loads ahead of the chain)
      lu_run(S[u], gamma, lu, acc, bad);
      lu_prog(P, lane, n + u + NS, S[u]);
    }
  }
  bool odd = false;
  switch ((P.lu_d + 7) / 8) {
    case 0: break;  // no solver variables
    case 1: odd = lu_tail<1, EXACT>(P, lane, lu, buf); break;
    case 2: odd = lu_tail<2, EXACT>(P, lane, lu, buf); break;
    case 3: odd = lu_tail<3, EXACT>(P, lane, lu, buf); break;
    case 4: odd = lu_tail<4, EXACT>(P, lane, lu, buf); break;
    default: odd = lu_tail<5, EXACT>(P, lane, lu, buf); break;
  }
  if (EXACT && odd) odd = lu_tail_sparse(P, lane, lu);
  bad |= odd;
  return wave_or(bad ? 1 : 0);
}

__device__ __forceinline__ double readlane_d(double v, int l) {
  int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}

// ---------------------------------------------------------------------
// Triangular solves (LU) x = b.
//
// A sweep is a chain: unknown k needs every earlier unknown of its row.  Taken
// pivot by pivot (a column of L or U at a time) the CB05-scale mechanism with
// its aerosol is 608 dependent steps of about 1000 cycles, though its
// elimination order has only 63 (forward) and 58 (backward) levels.  So the
// pivots are split (Program::tri_e):
//  * the tail, the last min(64, nv) pivots, where the fill makes nearly every
//    pivot wait on the one before it: one unknown per lane in a register, the
//    pivot's value broadcast with v_readlane, one multiply-add per pivot;
//  * the head before it, in batches of rows whose unknowns are ready: a lane
//    takes up to 8 entries of one row, in the row's order, with the unknowns
//    in LDS, so that a batch costs one LDS round trip and independent rows
//    (the aerosol's size bins) run side by side.
// Every row adds its entries in elimination order, one product at a time, so
// the results are those of the pivot-by-pivot sweeps bit for bit, as long as they
// are finite and quot's operands in range (see cell_lu_solve).  All LU
// values and positions are known before the sweep and are loaded ahead of it
// (AH batches; the program NS ahead), so a batch waits on the unknowns only.
// Cycles per solve: 1024 multi-phase cells 557k -> 84k, one cell 381k -> 54k;
// 2000 CB05-scale gas cells 18.9k -> 10.9k, one cell 17.3k -> 10.0k.
//
// FMA (nv <= kTriInPlace): fused multiply-adds, the backward sweep on
// D^-1 U x = D^-1 y (weights and right-hand side times the reciprocal
// diagonal); otherwise separate products and a division by the diagonal.
// ---------------------------------------------------------------------
// AH: batches whose LU values are loaded ahead; NS: register sets of the
// pipelines, the look-ahead of the program (AH + 1 < NS <= kTriPad)

struct TriBatch {
  int4 a, b;
  int2 r;
  double w[8], dg;
};
__device__ __forceinline__ void tri_prog(const DevProgram& P, int lane, int n, TriBatch& S) {
  S.a = P.tri_e[(size_t)(2 * n) * kWave + lane];
  S.b = P.tri_e[(size_t)(2 * n + 1) * kWave + lane];
  S.r = P.tri_r[(size_t)n * kWave + lane];
}
template <bool FWD>
__device__ __forceinline__ void tri_vals(const double* lu, TriBatch& S) {
  const int e[8] = {S.a.x, S.a.y, S.a.z, S.a.w, S.b.x, S.b.y, S.b.z, S.b.w};
#pragma unroll
  for (int u = 0; u < 8; ++u) S.w[u] = lu[e[u] & 0xFFFF];
  S.dg = FWD ? 1.0 : lu[S.r.y];
}
template <bool FWD, bool FMA>
__device__ __forceinline__ void tri_run(const TriBatch& S, double* X) {
  const int e[8] = {S.a.x, S.a.y, S.a.z, S.a.w, S.b.x, S.b.y, S.b.z, S.b.w};
  const int row = S.r.x & 0xFFFF;
  const bool idle = row == 0xFFFF;
  double x[8];
  double acc = X[idle ? 0 : row];
#pragma unroll
  for (int u = 0; u < 8; ++u) x[u] = X[(unsigned)e[u] >> 16];
  __builtin_amdgcn_sched_barrier(0);  // (all nine reads in flight)
  double d = 1.0;
  if (!FWD && FMA) {
    d = 1.0 / S.dg;
    acc = (S.r.x & (1 << 16)) ? acc * d : acc;
  }
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    if (FMA) acc = fma(-(FWD ? S.w[u] : S.w[u] * d), x[u], acc);
    else acc = acc - S.w[u] * x[u];
  }
  if (!FWD && !FMA) acc = (S.r.x & (1 << 17)) ? acc / S.dg : acc;
  if (!idle) X[row] = acc;
  wsync();
}
// (both pipelines leave their loops in the middle: a step that was skipped
// instead would leave the compiler unsure how many loads are in flight, and
// it would wait for all of them)
template <bool FWD, bool FMA, int AH, int NS>
__device__ __forceinline__ void tri_head(const DevProgram& P, int lane, const double* lu,
                                         double* X) {
  const int n0 = FWD ? 0 : P.tri_nf + kTriPad, nb = FWD ? P.tri_nf : P.tri_nb;
  if (nb == 0) return;
  TriBatch S[NS];
#pragma unroll
  for (int u = 0; u < NS; ++u) tri_prog(P, lane, n0 + u, S[u]);
#pragma unroll
  for (int u = 0; u < AH; ++u) tri_vals<FWD>(lu, S[u]);
  for (int n = 0;; n += NS) {
#pragma unroll
    for (int u = 0; u < NS; ++u) {
      if (n + u >= nb) return;
      tri_vals<FWD>(lu, S[(u + AH) % NS]);
      __builtin_amdgcn_sched_barrier(0);  // keeps the loads ahead of the chain
      tri_run<FWD, FMA>(S[u], X);
      tri_prog(P, lane, n0 + n + u + NS, S[u]);
    }
  }
}

// The tail: x is the lane's unknown (row tri_s + lane); dg its diagonal and y
// the diagonal's reciprocal.
struct TailBlock {
  int4 t;
  double w[8];
};
__device__ __forceinline__ void tail_vals(const double* lu, TailBlock& S) {
  const int t[4] = {S.t.x, S.t.y, S.t.z, S.t.w};
#pragma unroll
  for (int u = 0; u < 8; ++u)
    S.w[u] = lu[u % 2 ? (unsigned)t[u / 2] >> 16 : t[u / 2] & 0xFFFF];
}
// x / dg for every lane: the quotient from the correctly rounded reciprocal y
// with two residual corrections, which is the correctly rounded quotient (P.
// Markstein, IBM J. Res. Dev. 34(1), 1990) in a third of the latency of the
// division, which sits on the chain of every pivot -- as long as nothing on the
// way over- or underflows.  quot_ok: the reciprocal and the first quotient are
// normal and the residual x - dg q, a multiple of 2^-104 of x, is exact.
__device__ __forceinline__ double quot(double x, double dg, double y) {
  double q = x * y;
  q = fma(fma(-dg, q, x), y, q);
  return fma(fma(-dg, q, x), y, q);
}
__device__ __forceinline__ bool quot_ok(double x, double dg, double q) {
  const double ax = fabs(x), ad = fabs(dg), aq = fabs(q);
  return ad >= 0x1p-1000 && ad <= 0x1p1000 &&
         (x == 0.0 || (ax >= 0x1p-900 && ax <= 0x1p1000 && aq >= 0x1p-900 && aq <= 0x1p1000));
}
// Eight pivots of the tail, k0 onwards (or downwards).
template <bool FWD, bool FMA>
__device__ __forceinline__ void tail_run(int k0, const TailBlock& S, double dg, double y,
                                         double& x) {
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const double v = !FWD && !FMA ? quot(x, dg, y) : x;
    const double xk = readlane_d(v, (FWD ? k0 + u : k0 - u) & (kWave - 1));
    if (FMA) x = fma(-(FWD ? S.w[u] : S.w[u] * y), xk, x);
    else x = x - S.w[u] * xk;
  }
}
// A full tail (64 pivots) is unrolled: a readlane of a fixed lane costs two
// thirds of one whose lane is a register (28 against 43 cycles with the
// multiply-add that waits on it).  Shorter tails loop over their blocks.
template <bool FWD, bool FMA, int AH>
__device__ __forceinline__ void tri_tail(const DevProgram& P, int lane, const double* lu,
                                         double dg, double y, double& x) {
  const int nb = FWD ? P.tt_nf : P.tt_nb;
  const int4* tb = P.tt + (size_t)(FWD ? 0 : P.tt_nf + kTriPad) * kWave + lane;
  if (P.tri_d == kWave) {
    TailBlock S[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) S[b].t = tb[b * kWave];
#pragma unroll
    for (int b = 0; b < AH; ++b) tail_vals(lu, S[b]);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      if (b + AH < 8) tail_vals(lu, S[b + AH]);
      __builtin_amdgcn_sched_barrier(0);
      tail_run<FWD, FMA>(FWD ? 8 * b : kWave - 1 - 8 * b, S[b], dg, y, x);
    }
    return;
  }
  for (int n = 0; n < nb; ++n) {
    TailBlock S;
    S.t = tb[n * kWave];
    tail_vals(lu, S);
    tail_run<FWD, FMA>(FWD ? 8 * n : P.tri_d - 1 - 8 * n, S, dg, y, x);
  }
}

// x in X (LDS): indexed by solver variable for FMA programs, else by pivot.
// Returns false where a quotient of the tail may not be the correctly rounded
// one (non-FMA programs).
template <bool FMA, int AH, int NS>
__device__ __forceinline__ bool tri_solve(const DevProgram& P, int lane, const double* lu,
                                          double* X) {
  vm_drain();
  const bool on = lane < P.tri_d;
  const int r = on ? P.tri_s + lane : 0;
  const int ix = FMA ? P.perm[r] : r;
  const double dg = on ? lu[P.diag_pos[r]] : 1.0;
  tri_head<true, FMA, AH, NS>(P, lane, lu, X);
  double x = on ? X[ix] : 0.0;
  tri_tail<true, FMA, AH>(P, lane, lu, 1.0, 1.0, x);
  const double y = 1.0 / dg;
  if (FMA) x *= y;
  tri_tail<false, FMA, AH>(P, lane, lu, dg, y, x);
  bool ok = true;
  if (!FMA) {
    const double q = quot(x, dg, y);
    ok = !on || quot_ok(x, dg, q);
    x = q;
  }
  if (on) X[ix] = x;
  wsync();
  tri_head<false, FMA, AH, NS>(P, lane, lu, X);
  return ok;
}

// The same solve of a program with separate products, entry by entry: no
// product with the padding's zeros, divisions by the diagonal.  With values
// that are not finite, or too small for quot, these are not the same.
__device__ __forceinline__ void tri_solve_sparse(const DevProgram& P, int lane, const double* lu,
                                                 double* X) {
  const int zero = P.lu_nnz + kWave;
  auto head = [&](bool fwd) {
    const int n0 = fwd ? 0 : P.tri_nf + kTriPad, nb = fwd ? P.tri_nf : P.tri_nb;
#pragma nounroll
    for (int n = 0; n < nb; ++n) {
      const int* e = (const int*)P.tri_e + (size_t)(n0 + n) * 2 * kWave * 4 + 4 * lane;
      const int2 r = P.tri_r[(size_t)(n0 + n) * kWave + lane];
      const int row = r.x & 0xFFFF;
      double acc = X[row == 0xFFFF ? 0 : row];
#pragma nounroll
      for (int u = 0; u < 8; ++u) {
        const int w = e[(u >> 2) * kWave * 4 + (u & 3)];
        if ((w & 0xFFFF) != zero) acc = acc - lu[w & 0xFFFF] * X[(unsigned)w >> 16];
      }
      if (!fwd && (r.x & (1 << 17))) acc = acc / lu[r.y];
      if (row != 0xFFFF) X[row] = acc;
      wsync();
    }
  };
  const int d = P.tri_d;
  auto tail = [&](bool fwd, double dg, double& x) {
    const int4* tb = P.tt + (size_t)(fwd ? 0 : P.tt_nf + kTriPad) * kWave + lane;
#pragma nounroll
    for (int k = 0; k < d; ++k) {
      const int* t = (const int*)(tb + (size_t)(k >> 3) * kWave);
      const int p = (int)(((unsigned)t[(k & 7) >> 1] >> (16 * (k & 1))) & 0xFFFF);
      const double xk = readlane_d(fwd ? x : x / dg, fwd ? k : d - 1 - k);
      if (p != zero && !(fwd && k == d - 1)) x = x - lu[p] * xk;
    }
  };
  const bool on = lane < d;
  const int r = on ? P.tri_s + lane : 0;
  const double dg = on ? lu[P.diag_pos[r]] : 1.0;
  head(true);
  double x = on ? X[r] : 0.0;
  tail(true, 1.0, x);
  tail(false, dg, x);
  if (on) X[r] = x / dg;
  wsync();
  head(false);
}

// Solve (LU) x = b in place; b in dep order, w a scratch vector (nv) in LDS,
// used past kTriInPlace.  FAR: the factors live in global memory (multi-phase
// programs) and are fetched two batches ahead instead of one.  EXACT: a solution
// with values that are not finite, or quotients outside quot's range, is that of
// the pivot-by-pivot sweeps too: entry by entry past kTriInPlace, NaN as a whole
// up to it.  The integrator does without: it rejects a correction that is not
// finite whatever values it has, and an ulp of one under 2^-900 decides nothing.
template <bool FAR, bool EXACT>
__device__ __forceinline__ void cell_lu_solve(const DevProgram& P, int lane, double* lu, double* b,
                                              double* w) {
  lane = phase_lane(lane);
  if (!FAR) {
    // the zero slot, 64 places after the LU values (the f gather's scratch
    // shares it)
    if (lane == 0) lu[P.lu_nnz + kWave] = 0.0;
    wsync();
  }
  if (P.nv <= kTriInPlace) {
    (void)tri_solve<true, FAR ? 2 : 1, 4>(P, lane, lu, b);
    if (!EXACT) return;
    bool odd = false;
    for (int i = lane; i < P.nv; i += kWave) odd |= !isfinite(b[i]);
    if (__builtin_amdgcn_ballot_w64(odd) != 0)
      for (int i = lane; i < P.nv; i += kWave) b[i] = __builtin_nan("");
    wsync();
    return;
  }
  for (int k = lane; k < P.nv; k += kWave) w[k] = b[P.perm[k]];
  wsync();
  bool ok = tri_solve<false, FAR ? 2 : 1, 4>(P, lane, lu, w);
  if (EXACT) {
    for (int k = lane; k < P.nv; k += kWave) ok = ok && isfinite(w[k]);
    if (__builtin_amdgcn_ballot_w64(!ok) != 0) {
      for (int k = lane; k < P.nv; k += kWave) w[k] = b[P.perm[k]];
      wsync();
      tri_solve_sparse(P, lane, lu, w);
    }
  }
  for (int k = lane; k < P.nv; k += kWave) b[P.perm[k]] = w[k];
  wsync();
}

}  // namespace camp
