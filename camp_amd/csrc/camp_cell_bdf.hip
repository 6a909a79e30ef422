// Persistent per-cell BDF kernel.
//
// Each wavefront pops cells from an atomic queue and integrates each cell
// from t0 to t1 on its own: variable-order (1-5) variable-step BDF in
// Nordsieck form with modified Newton and WRMS error control -- the CVODE
// algorithm that CAMP's solver_run drives (camp_solver.c:544-693; CVODE:
// Hindmarsh et al., ACM TOMS 31(3), 2005) -- but with order, step size,
// Newton iteration, Jacobian reuse and error test decided per cell instead
// of once for the whole block of cells.  What a step touches lives in LDS
// as far as it fits (Nordsieck history, work vectors, rates, LU factors; kPlaceLds
// and following say what lies where); the cell's saved Jacobian history (J_solver,
// J_state, J_deriv, camp_solver.c:1111-1114) has its place in HBM, because CAMP
// keeps it across calls.
#include <cstddef>
#include <cstdio>
#include <mutex>
#include <type_traits>

#include "camp_device.hpp"
#include "camp_kernels.hpp"
#include "camp_solver_impl.hpp"

namespace camp {

namespace {

constexpr int QMAX = 5;
constexpr double ETAMX1 = 10000.0, ETAMX2 = 10.0, ETAMX3 = 10.0, ETAMXF = 0.2;
constexpr double ETAMIN = 0.1, ETACF = 0.25, ADDON = 0.000001;
constexpr double BIAS1 = 6.0, BIAS2 = 6.0, BIAS3 = 10.0, THRESH = 1.5;
constexpr int SMALL_NST = 10, MXNEF1 = 3, SMALL_NEF = 2, LONG_WAIT = 10;
constexpr double CRDOWN = 0.3, DGMAX = 0.3, RDIV = 2.0, NLSCOEF = 0.1;
constexpr int MSBP = 20, MAXCOR = 3, MSBJ = 50;
constexpr double DGMAX_JBAD = 0.2;
constexpr int GUESS_MAX_ITER = 5;

enum { CV_SUCCESS = 0, CV_TOO_MUCH_WORK = -1, CV_TOO_MUCH_ACC = -2, CV_ERR_FAILURE = -3,
       CV_CONV_FAILURE = -4, CV_LSETUP_FAIL = -6, CV_LSOLVE_FAIL = -7, CV_RHSFUNC_FAIL = -8,
       CV_FIRST_RHSFUNC_ERR = -9, CV_REPTD_RHSFUNC_ERR = -10, CV_UNREC_RHSFUNC_ERR = -11,
       CV_ILL_INPUT = -22 };
enum { FIRST_CALL = 1, PREV_CONV_FAIL, PREV_ERR_FAIL };
enum { DO_ERROR_TEST = 2, PREDICT_AGAIN, CONV_FAIL, TRY_AGAIN, RHSFUNC_RECVR, NEWTON_F, ERR_TEST_F };
enum { CV_NO_FAILURES = 0, CV_FAIL_BAD_J = 1, CV_FAIL_OTHER = 2 };

__device__ __forceinline__ double rpowerr(double b, double e) { return b <= 0.0 ? 0.0 : pow(b, e); }
__device__ __forceinline__ double rpoweri(double b, int e) {
  double p = 1.0;
  for (int i = 1; i <= (e < 0 ? -e : e); ++i) p *= b;
  return e < 0 ? 1.0 / p : p;
}

// A condition on wave-uniform values as a scalar: every lane of the wavefront
// is active and agrees, but the compiler cannot see that of values that come
// through LDS or calls, and one branch it takes for divergent makes every
// control variable set under it per-lane (the whole integrator then ran under
// execution masks, with its control state copied between vector registers).
__device__ __forceinline__ bool uc(bool c) { return __builtin_amdgcn_ballot_w64(c) != 0; }

// A step-control value, the same in every lane, held in vector registers: in
// scalar ones each assignment was a v_readfirstlane pair and each use a copy
// back, 1k to 3k cycles of a step (10 species 46.7k -> 45.8k, with everything in
// LDS 56.1k -> 52.0k; CB05-scale, everything in LDS, 75.4k -> 72.5k).  A class of
// its own: as plain doubles the compiler, at the two-wavefront register bound,
// spills f's rate constants instead of the history passes' values (2000
// CB05-scale cells: f 13.8k instead of 13.3k cycles).
struct UDouble {
  double v;
  UDouble() = default;
  __device__ UDouble(double x) : v(x) {}
  __device__ UDouble& operator=(double x) {
    v = x;
    return *this;
  }
  __device__ UDouble& operator+=(double x) { return *this = v + x; }
  __device__ UDouble& operator-=(double x) { return *this = v - x; }
  __device__ UDouble& operator*=(double x) { return *this = v * x; }
  __device__ UDouble& operator/=(double x) { return *this = v / x; }
  __device__ operator double() const { return v; }
};

// MP selects the multi-phase instantiation: gas-phase programs run a kernel
// without the aerosol code (smaller code and register footprint).  PL: the
// variant.  KG: the rate constants are read in place in global memory (s_k)
// and, for the f terms, held by the lanes (kt).  GH: the J history lives in
// global memory, with a copy in f's order in the wavefront's scratch (E).
template <bool MP, int PL>
struct CellCv {
  static constexpr bool GH = MP || PL != kPlaceLds, KG = GH && !MP;

  // The kernel argument's program, read from kernarg memory anew where a phase
  // begins: the pointer is opaque to the compiler there, so the phase's fields
  // come with a few scalar loads.  Loaded once at the kernel's start, as the
  // compiler would otherwise, the ~90 pointers overflow the scalar registers
  // into lanes of vector registers, and each use costs a v_readlane pair (24
  // cycles each).
  static_assert(offsetof(CellBdfArgs, P) == 0, "the program is read at the kernel arguments' start");
  __device__ __forceinline__ static const DevProgram& program() {
    auto k = (const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(k));
    return *(const DevProgram*)(const __attribute__((address_space(4))) DevProgram*)k;
  }
  int lane, nv;
  double *s_state, *s_k, *s_rate, *z01, *z2, *ewt, *acor, *y, *tempv, *ftemp, *last, *acinit,
      *w, *lu, *s_fb, *E;
  double *Js, *Jy, *Jf;
  MpLds mpl;   // multi-phase extras (LDS); unused for gas-phase programs
  double* Jr;  // reaction Jacobian scratch (global) of multi-phase programs
  UDouble tn, h, hscale, hprime, next_h, eta, etamax, etaq, etaqm1, etaqp1, hu, init_h, rtol;
  double *l, *tq, *tau;  // small coefficient arrays, in LDS (uniform values)
  UDouble rl1, gamma, gammap, gamrat, crate, acnrm, saved_tq5;
  int q, qprime, L, qwait, jcur, use_acinit, guess_on, maxcf, max_steps, projected;
  int nst, nfe, nsetups, nni, ncfn, netf, nje, nstlp, nstlj;
  // the rate constants of the lane's first kTermRegs terms
  double kt[kTermRegs];
  __device__ __forceinline__ void load_term_constants() {
    const DevProgram& P = program();
#pragma unroll
    for (int g = 0; g < kTermRegs; ++g) {
      int t = lane + g * kWave;
      kt[g] = t < P.n_terms ? s_k[P.t_rec[t].x & 0x0FFFFFFF] : 0.0;
    }
  }
  // optional shader-clock counters (cycles in f, Jac, LU factor, LU solve)
  bool prof;
  long long c_f, c_j, c_lu, c_sol, c_fr, c_fg;
  __device__ __forceinline__ long long tick() const { return prof ? clock64() : 0; }

  // Nordsieck vectors 0 and 1 (read in every Newton iteration) and 2 to 5,
  // which may live apart
  __device__ __forceinline__ double* zn0() const { return z01; }
  __device__ __forceinline__ double* zn1() const { return z01 + nv; }
  __device__ __forceinline__ double* znh(int j) const { return z2 + (size_t)(j - 2) * nv; }
  __device__ __forceinline__ double zget(int j, int i) const {
    return j == 0 ? zn0()[i] : j == 1 ? zn1()[i] : znh(j)[i];
  }
  __device__ __forceinline__ void zset(int j, int i, double v) const {
    if (j == 0) zn0()[i] = v;
    else if (j == 1) zn1()[i] = v;
    else znh(j)[i] = v;
  }

  // body(i, on) over the lane's rows, two at a time where there are more than
  // 64: the second row's loads then overlap the first's (a second trip of the
  // loop costs its full latency, for 8 rows of a CB05-scale cell).  A lane
  // without a second row repeats its first one (on[1] false): same loads,
  // same stores.
  template <class B>
  __device__ __forceinline__ void rows(B body) const {
    for (int i0 = 0; i0 < nv; i0 += 2 * kWave) {
      const int i = i0 + lane;
      if (i0 + kWave < nv) {
        const bool two = i + kWave < nv;
        const int id[2] = {i, two ? i + kWave : i};
        body(id, two, std::integral_constant<int, 2>());
      } else if (i < nv) {
        const int id[2] = {i, i};
        body(id, false, std::integral_constant<int, 1>());
      }
    }
  }
  // f(order) with the method's order as a constant: the history loops then
  // have fixed bounds
  template <class F>
  __device__ __forceinline__ void by_order(F f) const {
    switch (q) {
      case 1: f(std::integral_constant<int, 1>()); break;
      case 2: f(std::integral_constant<int, 2>()); break;
      case 3: f(std::integral_constant<int, 3>()); break;
      case 4: f(std::integral_constant<int, 4>()); break;
      default: f(std::integral_constant<int, 5>()); break;
    }
  }

  __device__ __forceinline__ double wrms(const double* x) {
    double s = 0.0;
    for (int i = lane; i < nv; i += kWave) {
      double p = x[i] * ewt[i];
      s += p * p;
    }
    s = wave_sum(s);
    return sqrt(s / nv);
  }

  // the error weights of zn[0], and zn[0]'s WRMS norm under them
  __device__ __forceinline__ double ewt_set() {
    const DevProgram& P = program();
    double s = 0.0;
    rows([&](const int* id, bool two, auto R) {
      double wt[R], z[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        z[r] = zn0()[id[r]];
        wt[r] = P.abs_tol_dep[id[r]];
      }
#pragma unroll
      for (int r = 0; r < R; ++r) wt[r] = 1.0 / (rtol * fabs(z[r]) + wt[r]);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        ewt[id[r]] = wt[r];
        double p = z[r] * wt[r];
        s += r == 0 || two ? p * p : 0.0;
      }
    });
    wsync();
    return sqrt(wave_sum(s) / nv);
  }

  // CAMP f(): camp_solver.c:843-958 for one cell; est = false is the pure f
  // that Jac() runs first (camp_solver.c:1052-1063).  y -> ftemp always: fixed
  // arguments keep their address spaces known to the compiler.
  __device__ __forceinline__ int f(bool est) {
    const DevProgram& P = program();
    long long t0 = tick();
    double ts = next_h > 0.0 ? next_h : init_h;
    FLoad F;
    if (!MP) {
      f_load_terms(P, lane, F);
      f_load_gather(P, lane, F);
    }
    int bad = cell_set_state(P, lane, y, s_state);
    if (!bad) {
      if (MP) {
        mp_f_prologue(P, lane, s_state, s_k, mpl);
        f_load_terms(P, lane, F);
      }
      cell_rates<KG>(P, lane, s_state, s_k, s_rate, F, kt);
      if (MP) f_load_gather(P, lane, F);
      wsync();
      long long t1 = tick();
      if (prof && est) c_fr += t1 - t0;
      cell_deriv<GH>(P, lane, s_state, s_rate, y, GH ? E : Js, Jy, Jf, est, ts, ftemp, s_fb,
                     KG && PL != kPlaceWide ? tempv : w, F, MP ? mpl.slot : nullptr);
      wsync();
      if (prof && est) c_fg += clock64() - t1;
    }
    wsync();
    if (prof) (est ? c_f : c_j) += clock64() - t0;
    return bad;
  }

  // CAMP Jac() after its pure f: J into the cell's J_solver, save history
  __device__ __forceinline__ void jac() {
    const DevProgram& P = program();
    long long t0 = tick();
    double ts = next_h > 0.0 ? next_h : init_h;
    if (MP) {
      mp_refresh(P, lane, s_state, mpl);
      mp_j_prologue(P, lane, s_state, s_k, mpl);
      cell_jac_mp(P, lane, s_state, s_k, ts, mpl, Jr, Js);
    } else {
      const double* k = s_k;
      if (!MP && PL == kPlaceGlobal) {
        // J reads its constants at random: staged where the LU goes next
        for (int i = lane; i < P.n_env; i += kWave) lu[i] = s_k[i];
        wsync();
        k = lu;
      }
      cell_jac(P, lane, s_state, k, ts, Js);
    }
    for (int i = lane; i < nv; i += kWave) {
      Jy[i] = y[i];
      Jf[i] = ftemp[i];
    }
    __threadfence_block();
    wsync();
    stage_history(P);
    if (prof) c_j += clock64() - t0;
  }
  __device__ __forceinline__ void stage_history(const DevProgram& P) {
    if (GH) est_stage(P, lane, Js, Jf, E);
  }

  // The history updates below work on one row of the Nordsieck array at a
  // time, staged in registers: all of its loads are issued together and each
  // value is stored once, instead of a chain of dependent load-store steps
  // through the array (which may live in global memory).  Every element
  // sees the same operations in the same order as the column-wise loops of
  // CVODE (cvRescale, cvPredict, cvRestore, cvCompleteStep).
  __device__ __forceinline__ void hist_load(int i, double* z) const {
#pragma unroll
    for (int j = 0; j <= QMAX; ++j)
      if (j <= q) z[j] = zget(j, i);
  }

  __device__ __forceinline__ void rescale() {
    double fac[QMAX + 1];
    double factor = eta;
#pragma unroll
    for (int j = 1; j <= QMAX; ++j) {
      fac[j] = factor;
      factor *= eta;
    }
    by_order([&](auto Q) {
      rows([&](const int* id, bool, auto R) {
        double z[R][QMAX + 1];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int j = 1; j <= Q; ++j) z[r][j] = zget(j, id[r]);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int j = 1; j <= Q; ++j) zset(j, id[r], z[r][j] * fac[j]);
      });
    });
    h = hscale * eta;
    next_h = h;
    hscale = h;
    wsync();
  }

  // zn[j-1] += zn[j] (SIGN 1) or -= (SIGN -1), k = 1..q, j = q..k; a
  // prediction also goes to y, and its minimum is returned
  template <int SIGN>
  __device__ __forceinline__ double pascal() {
    double mn = 1.0e308;
    by_order([&](auto Q) {
      rows([&](const int* id, bool, auto R) {
        double z[R][QMAX + 1];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int j = 0; j <= Q; ++j) z[r][j] = zget(j, id[r]);
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
          for (int k = 1; k <= Q; ++k)
#pragma unroll
            for (int j = Q; j >= k; --j)
              z[r][j - 1] = SIGN > 0 ? z[r][j - 1] + z[r][j] : z[r][j - 1] - z[r][j];
#pragma unroll
          for (int j = 0; j < Q; ++j) zset(j, id[r], z[r][j]);
          if (SIGN > 0) {
            y[id[r]] = z[r][0];
            mn = fmin(mn, z[r][0]);
          }
        }
      });
    });
    wsync();
    return mn;
  }

  __device__ __forceinline__ double predict() {
    tn += h;
    return wave_min(pascal<1>());
  }

  __device__ __forceinline__ void restore(double saved_t) {
    tn = saved_t;
    pascal<-1>();
  }

  // cvSet and cvSetTqBDF.  All step-size quotients h / (h + tau_1 + ... +
  // tau_(j-1)) are formed at once (their divisions overlap; those past the
  // order are not used), and l is built in registers and stored once: loops
  // over the LDS arrays were a chain of LDS round trips and divisions.
  __device__ __forceinline__ void set() {
    double hs = h, x[QMAX + 2], L_[QMAX + 1];
#pragma unroll
    for (int j = 2; j <= QMAX + 1; ++j) {
      hs += tau[j - 1];
      x[j] = h / hs;
    }
    L_[0] = L_[1] = 1.0;
#pragma unroll
    for (int j = 2; j <= QMAX; ++j) L_[j] = 0.0;
    double alpha0 = -1.0, alpha0_hat = -1.0, xi_inv = 1.0, xistar_inv = 1.0, lq = 1.0, rq = 1.0;
    double xi_next = x[2];
    if (q > 1) {
#pragma unroll
      for (int j = 2; j < QMAX; ++j)
        if (j < q) {
          alpha0 -= 1.0 / j;
#pragma unroll
          for (int i = QMAX; i >= 1; --i)
            if (i <= j) L_[i] += L_[i - 1] * x[j];
        }
#pragma unroll
      for (int j = 2; j <= QMAX; ++j)
        if (j == q) {
          rq = 1.0 / j;
          xi_inv = x[j];
          xi_next = x[j + 1];
        }
      alpha0 -= rq;
      xistar_inv = -L_[1] - alpha0;
      alpha0_hat = -L_[1] - xi_inv;
#pragma unroll
      for (int i = QMAX; i >= 1; --i)
        if (i <= q) L_[i] += L_[i - 1] * xistar_inv;
#pragma unroll
      for (int j = 2; j <= QMAX; ++j)
        if (j == q) lq = L_[j];
    } else {
      lq = L_[1];
    }
    double A1 = 1.0 - alpha0_hat + alpha0;
    double A2 = 1.0 + q * A1;
    double tq2 = fabs(A1 / (alpha0 * A2));
    double tq5 = fabs(A2 * xistar_inv / (lq * xi_inv));
    tq[2] = tq2;
    tq[5] = tq5;
    if (qwait == 1) {
      if (q > 1) {
        double C = xistar_inv / lq;
        double A3 = alpha0 + rq;
        double A4 = alpha0_hat + xi_inv;
        double Cpinv = (1.0 - A4 + A3) / A3;
        tq[1] = fabs(C * Cpinv);
      } else {
        tq[1] = 1.0;
      }
      double A5 = alpha0 - (1.0 / (q + 1));
      double A6 = alpha0_hat - xi_next;
      double Cppinv = (1.0 - A6 + A5) / A2;
      tq[3] = fabs(Cppinv / (xi_next * (q + 2) * A5));
    }
    tq[4] = NLSCOEF / tq2;
#pragma unroll
    for (int j = 0; j <= QMAX; ++j)
      if (j <= q) l[j] = L_[j];
    rl1 = 1.0 / L_[1];
    gamma = h * rl1;
    if (nst == 0) gammap = gamma;
    gamrat = (nst > 0) ? gamma / gammap : 1.0;
  }

  __device__ __forceinline__ void increase_bdf() {
    double alpha0, alpha1, prod, xi, xiold, hsum, A1;
    for (int j = 0; j <= QMAX; ++j) l[j] = 0.0;
    l[2] = alpha1 = prod = xiold = 1.0;
    alpha0 = -1.0;
    hsum = hscale;
    if (q > 1) {
      for (int j = 1; j < q; ++j) {
        hsum += tau[j + 1];
        xi = hsum / hscale;
        prod *= xi;
        alpha0 -= 1.0 / (j + 1);
        alpha1 += 1.0 / xi;
        for (int i = j + 2; i >= 2; --i) l[i] = l[i] * xiold + l[i - 1];
        xiold = xi;
      }
    }
    A1 = (-alpha0 - alpha1) / prod;
    for (int i = lane; i < nv; i += kWave) {
      double v = A1 * znh(QMAX)[i];
      znh(L)[i] = v;
      for (int j = 2; j <= q; ++j) znh(j)[i] += l[j] * v;
    }
    wsync();
  }

  __device__ __forceinline__ void decrease_bdf() {
    double hsum, xi;
    for (int j = 0; j <= QMAX; ++j) l[j] = 0.0;
    l[2] = 1.0;
    hsum = 0.0;
    for (int j = 1; j <= q - 2; ++j) {
      hsum += tau[j];
      xi = hsum / hscale;
      for (int i = j + 2; i >= 2; --i) l[i] = l[i] * xi + l[i - 1];
    }
    for (int i = lane; i < nv; i += kWave)
      for (int j = 2; j < q; ++j) znh(j)[i] += (-l[j]) * znh(q)[i];
    wsync();
  }

  __device__ __forceinline__ void adjust_params() {
    if (qprime != q) {
      int dq = qprime - q;
      if (dq == 1) increase_bdf();
      else if (dq == -1) decrease_bdf();
      q = qprime;
      L = q + 1;
      qwait = L;
    }
    rescale();
  }

  // The jump of one guess_helper iteration (camp_solver.c:1321-1408, called
  // with h_n = h > 0): y moved along ftemp by the longest step that keeps it
  // non-negative; returns the step.
  __device__ __forceinline__ double guess_jump(int iter, double t_n, double t_0, double t_j) {
    double h_j = t_n - (t_0 + t_j);
    double best = h_j;
    int found = 0;
    for (int i = lane; i < nv; i += kWave) {
      double c = ftemp[i], t_star = -y[i] / c;
      if ((t_star > 0.0 || (t_star == 0.0 && c < 0.0)) && t_star < best) {
        best = t_star;
        found = 1;
      }
    }
    best = wave_min(best);
    found = wave_or(found);
    h_j = best;
    if (uc(found != 0)) h_j *= 0.95 + 0.1 * iter / (double)GUESS_MAX_ITER;
    h_j = t_n < t_0 + t_j + h_j ? t_n - (t_0 + t_j) : h_j;
    for (int i = lane; i < nv; i += kWave) y[i] += h_j * ftemp[i];
    wsync();
    return h_j;
  }

  // whether the linear setup needs a new Jacobian (cvLsSetup)
  __device__ __forceinline__ bool jac_bad(int convfail) {
    double dgamma = fabs(gamma / gammap - 1.0);
    return (nst == 0) || (nst > nstlj + MSBJ) ||
           ((convfail == CV_FAIL_BAD_J) && uc(dgamma < DGMAX_JBAD)) || (convfail == CV_FAIL_OTHER);
  }

  __device__ __forceinline__ int factor() {
    const DevProgram& P = program();
    long long t0 = tick();
    int rc = cell_lu_factor<false>(P, lane, Js, gamma, lu, s_fb);
    if (prof) c_lu += clock64() - t0;
    return rc;
  }

  __device__ __forceinline__ void lsolve(double* b) {
    const DevProgram& P = program();
    long long t0 = tick();
    cell_lu_solve<MP || PL == kPlaceGlobalLu || PL == kPlaceWide, false>(P, lane, lu, b, w);
    if (prof) c_sol += clock64() - t0;
    if (uc(gamrat != 1.0)) {
      double s = 2.0 / (1.0 + gamrat);
      for (int i = lane; i < nv; i += kWave) b[i] *= s;
      wsync();
    }
  }

  // Non-negativity safeguard (not in CVODE): CAMP's f() rejects y < -SMALL
  // (camp_solver.c:816-822), and cutting the step is CVODE's only answer,
  // so a species driven to ~0 by a fast loss stalls the integration.
  // Wherever f() would see the iterate y = zn0 + corr, components below
  // -SMALL by at most their tolerance (-y_i * ewt_i <= 1) are projected to
  // TINY (solver_run's floor, camp_solver.c:554-567) through corr.
  // Returns -1 (nothing below -SMALL), 0 (projected) or 1 (a larger
  // excursion: the recoverable f() failure it implies); wave-uniform.
  __device__ __forceinline__ int project(double* corr) {
    double worst = -1.0;
    for (int i = lane; i < nv; i += kWave)
      if (y[i] < -1.0e-30) worst = fmax(worst, -y[i] * ewt[i]);
    worst = -wave_min(-worst);
    if (uc(worst > 1.0)) return 1;
    if (uc(worst < 0.0)) return -1;
    for (int i = lane; i < nv; i += kWave)
      if (y[i] < -1.0e-30) {
        corr[i] = 1.0e-60 - zn0()[i];
        y[i] = 1.0e-60;
      }
    wsync();
    return 0;
  }

  // One Newton iteration up to the next f(y): NEWTON_F where it needs one
  // (y holds the iterate), else the nonlinear solve's outcome.  m, del and
  // delp carry the iteration count and the last two correction norms.
  // (the first iteration starts from the guess, or zero)
  __device__ __forceinline__ double correction(int m, int i) const {
    return m > 0 ? acor[i] : use_acinit ? acinit[i] : 0.0;
  }
  __device__ __forceinline__ int newton_pass(int& m, UDouble& delp) {
    rows([&](const int* id, bool, auto R) {
      double t[R], fv[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        t[r] = rl1 * zn1()[id[r]] + correction(m, id[r]);
        fv[r] = ftemp[id[r]];
      }
#pragma unroll
      for (int r = 0; r < R; ++r) tempv[id[r]] = gamma * fv[r] - t[r];
    });
    wsync();
    lsolve(tempv);
    nni++;
    // the correction's WRMS norm, the corrected state and the per-lane sum
    // of the new correction's norm in one pass over the rows (one round
    // trip for the error weights and zn[0] instead of two)
    double s_del = 0.0, s_acor = 0.0;
    rows([&](const int* id, bool two, auto R) {
      double t[R], wt[R], a[R], z[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        t[r] = tempv[id[r]];
        wt[r] = ewt[id[r]];
        a[r] = correction(m, id[r]);
        z[r] = zn0()[id[r]];
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        double p = t[r] * wt[r];
        a[r] += t[r];
        double pa = a[r] * wt[r];
        if (r == 0 || two) {
          s_del += p * p;
          s_acor += pa * pa;
        }
        acor[id[r]] = a[r];
        y[id[r]] = z[r] + a[r];
      }
    });
    double del = sqrt(wave_sum(s_del) / nv);
    wsync();
    if (m > 0) crate = fmax(CRDOWN * crate, del / delp);
    double dcon = del * fmin(1.0, crate) / tq[4];
    const bool ok = uc(dcon <= 1.0);
    if (!ok) {
      m++;
      if ((m == MAXCOR) || ((m >= 2) && uc(del > RDIV * delp))) return jcur ? CONV_FAIL : TRY_AGAIN;
    }
    int pr = project(acor);
    if (pr > 0) return jcur ? RHSFUNC_RECVR : TRY_AGAIN;
    if (!ok) {
      delp = del;
      return NEWTON_F;
    }
    projected = pr == 0;
    // (without a projection acor is the one summed above)
    acnrm = pr < 0 ? (m == 0 ? del : sqrt(wave_sum(s_acor) / nv)) : wrms(acor);
    jcur = 0;
    return CV_SUCCESS;
  }

  __device__ __forceinline__ int handle_nflag(int* nflagPtr, double saved_t, int* ncfPtr) {
    int nflag = *nflagPtr;
    if (nflag == CV_SUCCESS) return DO_ERROR_TEST;
    ncfn++;
    restore(saved_t);
    if (nflag == CV_LSETUP_FAIL || nflag == CV_LSOLVE_FAIL || nflag == CV_RHSFUNC_FAIL) return nflag;
    (*ncfPtr)++;
    etamax = 1.0;
    if (*ncfPtr == maxcf) {
      if (nflag == CONV_FAIL) return CV_CONV_FAILURE;
      if (nflag == RHSFUNC_RECVR) return CV_REPTD_RHSFUNC_ERR;
    }
    eta = ETACF;
    *nflagPtr = PREV_CONV_FAIL;
    rescale();
    return PREDICT_AGAIN;
  }

  __device__ __forceinline__ int do_error_test(int* nflagPtr, double saved_t, int* nefPtr, double* dsmPtr) {
    double dsm = acnrm * tq[2];
    *dsmPtr = dsm;
    if (uc(dsm <= 1.0)) return CV_SUCCESS;
    (*nefPtr)++;
    netf++;
    *nflagPtr = PREV_ERR_FAIL;
    restore(saved_t);
    if (*nefPtr == maxcf) return CV_ERR_FAILURE;
    etamax = 1.0;
    if (*nefPtr <= MXNEF1) {
      eta = 1.0 / (rpowerr(BIAS2 * dsm, 1.0 / L) + ADDON);
      eta = fmax(ETAMIN, fmax(eta, 0.0));
      if (*nefPtr >= SMALL_NEF) eta = fmin(eta, ETAMXF);
      rescale();
      return TRY_AGAIN;
    }
    if (q > 1) {
      eta = ETAMIN;
      decrease_bdf();
      L = q;
      q--;
      qwait = L;
      rescale();
      return TRY_AGAIN;
    }
    eta = ETAMIN;
    h *= eta;
    next_h = h;
    hscale = h;
    qwait = LONG_WAIT;
    return ERR_TEST_F;  // zn[1] restarts from f(zn[0])
  }

  __device__ __forceinline__ void complete_step() {
    nst++;
    hu = h;
    double ta[QMAX + 1];
#pragma unroll
    for (int i = 1; i <= QMAX; ++i) ta[i] = tau[i];
#pragma unroll
    for (int i = QMAX; i >= 2; --i)
      if (i <= q || (i == 2 && nst > 1)) tau[i] = ta[i - 1];
    tau[1] = h;
    qwait--;
    bool save = (qwait == 1) && (q != QMAX);
    by_order([&](auto Q) {
      double lj[Q + 1];
#pragma unroll
      for (int j = 0; j <= Q; ++j) lj[j] = l[j];
      rows([&](const int* id, bool, auto R) {
        double z[R][QMAX + 1], a[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          a[r] = acor[id[r]];
#pragma unroll
          for (int j = 0; j <= Q; ++j) z[r][j] = zget(j, id[r]);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int i = id[r];
#pragma unroll
          for (int j = 0; j <= Q; ++j) z[r][j] += lj[j] * a[r];
          // after a projection, components at TINY restart flat
          if (projected && y[i] == 1.0e-60) {
            z[r][0] = 1.0e-60;
#pragma unroll
            for (int j = 1; j <= Q; ++j) z[r][j] = 0.0;
          }
#pragma unroll
          for (int j = 0; j <= Q; ++j) zset(j, i, z[r][j]);
          if (save) znh(QMAX)[i] = a[r];
          last[i] = z[r][0];
        }
      });
    });
    if (save) saved_tq5 = tq[5];
    wsync();
  }

  __device__ __forceinline__ void set_eta() {
    if (uc(eta < THRESH)) {
      eta = 1.0;
      hprime = h;
    } else {
      eta = fmin(eta, etamax);
      hprime = h * eta;
    }
  }

  __device__ __forceinline__ void prepare_next_step(double dsm) {
    if (uc(etamax == 1.0)) {
      qwait = qwait > 2 ? qwait : 2;
      qprime = q;
      hprime = h;
      eta = 1.0;
      return;
    }
    double ddn = -1.0, dup = -1.0;
    if (qwait == 0) {
      if (q > 1) {
        ddn = wrms(znh(q)) * tq[1];
      }
      if (q != QMAX && uc(saved_tq5 != 0.0)) {
        double cquot = (tq[5] / saved_tq5) * rpoweri(h / tau[2], L);
        for (int i = lane; i < nv; i += kWave) tempv[i] = -cquot * znh(QMAX)[i] + acor[i];
        wsync();
        dup = wrms(tempv) * tq[3];
      }
    }
    // The candidate ratios eta = 1 / (b^(1/n) + ADDON): one per lane, so that
    // up to three powers (about 1000 cycles each) cost one, and none when all
    // lie under THRESH for certain -- b >= (2/3)^n, rounded up, puts eta
    // below 1.4999935 -- for then their values decide nothing.
    const int w = lane % 3;
    const int n = w == 0 ? L : w == 1 ? q : L + 1;
    const bool on = w == 0 || (w == 1 ? ddn >= 0.0 : dup >= 0.0);
    const double b = w == 0 ? BIAS2 * dsm : w == 1 ? BIAS1 * ddn : BIAS3 * dup;
    double lim = 1.0;
    for (int j = 0; j < n; ++j) lim *= 0.66667;
    const bool small = !on || b >= lim;
    if (__builtin_amdgcn_ballot_w64(!small) == 0) {
      if (qwait == 0) qwait = 2;
      eta = 1.0;
      qprime = q;
      hprime = h;
      return;
    }
    const double r = on ? 1.0 / (rpowerr(b, 1.0 / n) + ADDON) : 0.0;
    etaq = readlane_d(r, 0);
    if (qwait != 0) {
      eta = etaq;
      qprime = q;
      set_eta();
      return;
    }
    qwait = 2;
    etaqm1 = readlane_d(r, 1);
    etaqp1 = readlane_d(r, 2);
    double etam = fmax(etaqm1, fmax(etaq, etaqp1));
    if (uc(etam < THRESH)) {
      eta = 1.0;
      qprime = q;
    } else if (uc(etam == etaq)) {
      eta = etaq;
      qprime = q;
    } else if (uc(etam == etaqm1)) {
      eta = etaqm1;
      qprime = q - 1;
    } else {
      eta = etaqp1;
      qprime = q + 1;
      for (int i = lane; i < nv; i += kWave) znh(QMAX)[i] = acor[i];
      wsync();
    }
    set_eta();
  }

  // Measurement: the cycles of f(y), J(y), the LU factorisation (gamma =
  // 10) and one triangular solve at the cell's staged state, averaged over
  // reps repetitions, into pr[0..3].  Integrates nothing.
  __device__ int bench_phases(int reps, double* pr) {
    for (int i = lane; i < nv; i += kWave) y[i] = zn0()[i];
    wsync();
    next_h = init_h = 1.0;
    if (f(false)) return -101;
    jac();
    long long cf = 0, cj = 0, clu = 0, cs = 0;
    for (int r = 0; r < reps; ++r) {
      long long t0 = clock64();
      f(true);
      long long t1 = clock64();
      f(false);
      jac();
      long long t2 = clock64();
      gamma = 10.0;
      if (factor()) return -102;
      long long t3 = clock64();
      for (int i = lane; i < nv; i += kWave) tempv[i] = ftemp[i];
      wsync();
      long long t4 = clock64();
      lsolve(tempv);
      long long t5 = clock64();
      cf += t1 - t0;
      cj += t2 - t1;
      clu += t3 - t2;
      cs += t5 - t4;
    }
    if (lane == 0) {
      pr[0] = (double)cf / reps;
      pr[1] = (double)cj / reps;
      pr[2] = (double)clu / reps;
      pr[3] = (double)cs / reps;
    }
    return -100;
  }

  // CVodeReInit + CVodeSetInitStep + CVode(tout, CV_NORMAL); zn(0) holds y0
  // on entry, y holds y(tout) on successful exit.
  __device__ __forceinline__ int solve(double t0, double tout) {
    for (int i = lane; i < nv; i += kWave) last[i] = zn0()[i];
    tn = t0;
    q = 1;
    L = 2;
    qwait = L;
    qprime = 1;
    etamax = ETAMX1;
    hu = 0.0;
    nst = nfe = ncfn = netf = nni = nsetups = nstlp = nje = nstlj = 0;
    saved_tq5 = 0.0;
    crate = 1.0;
    gamrat = 1.0;
    gammap = 1.0;
    jcur = 0;
    projected = 0;
    eta = 1.0;
    for (int i = 0; i < 8; ++i) tau[i] = 0.0;
    for (int i = 0; i < 6; ++i) tq[i] = 0.0;
    init_h = tout - t0;
    next_h = 0.0;
    wsync();
    ewt_set();
    // The integrator as one loop over actions, so that f(y) -- which the
    // start, the guess helper, the predictor, Jac(), every Newton iteration
    // and the error test's restart call -- and the other phases each appear
    // once in the kernel: inlined at every call they made 130 KB of code (263
    // KB with aerosol), several times the instruction cache.  An action that
    // needs f puts its argument into y, sets where to go on (then) and hands
    // over to ACT_F; bad is f's outcome.
    enum { ACT_F, ACT_START, ACT_MAIN, ACT_PREDICT, ACT_GUESS, ACT_GUESS_F, ACT_NLS, ACT_NLS_F,
           ACT_JAC, ACT_FACTOR, ACT_NEWTON, ACT_NEWTON_F, ACT_NLS_END, ACT_RESTART };
    int act = ACT_F, then = ACT_START, bad = 0;
    bool f_est = true;
    auto call_f = [&](int next) {
      f_est = true;
      act = ACT_F;
      then = next;
    };
    for (int i = lane; i < nv; i += kWave) y[i] = zn0()[i];
    wsync();
    int nstloc = 0, ncf = 0, nef = 0, nflag = FIRST_CALL, convfail = 0, call_setup = 0, m = 0,
        iter = 0, rc = 0;
    double dsm = 0.0;
    UDouble saved_t = tn, delp = 0.0, t_j = 0.0;
    for (;;) {
      // (addresses derived from these are computed in the action that uses
      // them, not kept through all of them)
      nv = phase_uniform(nv);
      lane = phase_lane(lane);
      switch (act) {
        case ACT_F:
          if (f_est) nfe++;
          bad = f(f_est);
          act = then;
          break;
        case ACT_START:
          if (bad) return CV_FIRST_RHSFUNC_ERR;
          h = init_h;
          for (int i = lane; i < nv; i += kWave) zn1()[i] = ftemp[i] * h;
          wsync();
          hscale = h;
          hprime = h;
          act = ACT_MAIN;
          break;
        case ACT_MAIN: {  // CVode's loop, then the start of cvStep
          next_h = h;
          if (nstloc >= max_steps) return CV_TOO_MUCH_WORK;
          double nrm = ewt_set();  // (before the first step: as it is)
          if (uc(2.220446049250313e-16 * nrm > 1.0)) return CV_TOO_MUCH_ACC;
          saved_t = tn;
          dsm = 0.0;
          ncf = nef = 0;
          nflag = FIRST_CALL;
          if ((nst > 0) && uc(hprime != h)) adjust_params();
          act = ACT_PREDICT;
          break;
        }
        case ACT_PREDICT: {  // then the start of the nonlinear solve
          double mn = predict();
          set();
          convfail = ((nflag == FIRST_CALL) || (nflag == PREV_ERR_FAIL)) ? CV_NO_FAILURES
                                                                         : CV_FAIL_OTHER;
          call_setup = (nflag == PREV_CONV_FAIL) || (nflag == PREV_ERR_FAIL) || (nst == 0) ||
                       (nst >= nstlp + MSBP) || uc(fabs(gamrat - 1.0) > DGMAX);
          use_acinit = 0;
          if (uc(mn > -1.0e-30)) {
            call_f(ACT_NLS_F);  // y is the prediction
            break;
          }
          act = ACT_NLS;
          // the guess helper acts on a negative prediction only
          if (guess_on) {
            double c = 1.0 / h;
            for (int i = lane; i < nv; i += kWave) {
              double la = last[i];
              y[i] = la;
              ftemp[i] = c * (zn0()[i] - la);
            }
            wsync();
            t_j = 0.0;
            iter = 0;
            act = ACT_GUESS;
          }
          break;
        }
        case ACT_GUESS: {
          double t_n = tn, t_0 = t_n - h;
          if (iter < GUESS_MAX_ITER && uc(t_0 + t_j < t_n)) {
            t_j += guess_jump(iter, t_n, t_0, t_j);
            call_f(ACT_GUESS_F);
            break;
          }
          for (int i = lane; i < nv; i += kWave) acinit[i] = (y[i] - zn0()[i]) * 0.999;
          wsync();
          use_acinit = 1;
          act = ACT_NLS;
          break;
        }
        case ACT_GUESS_F:
          iter++;
          act = bad ? ACT_NLS : ACT_GUESS;
          break;
        case ACT_NLS: {
          double mn = 1.0e308;
          for (int i = lane; i < nv; i += kWave) {
            double v = use_acinit ? zn0()[i] + acinit[i] : zn0()[i];
            y[i] = v;
            mn = fmin(mn, v);
          }
          wsync();
          if (uc(wave_min(mn) < -1.0e-30)) {
            if (!use_acinit) {
              for (int i = lane; i < nv; i += kWave) acinit[i] = 0.0;
              wsync();
              use_acinit = 1;
            }
            project(acinit);
          }
          call_f(ACT_NLS_F);
          break;
        }
        case ACT_NLS_F:
          if (bad) {
            nflag = RHSFUNC_RECVR;
            act = ACT_NLS_END;
          } else if (!call_setup) {
            m = -1;
            act = ACT_NEWTON;
          } else if (jac_bad(convfail)) {
            nje++;
            nstlj = nst;
            jcur = 1;
            call_f(ACT_JAC);
            f_est = false;
          } else {
            jcur = 0;
            bad = 0;
            act = ACT_FACTOR;
          }
          break;
        case ACT_JAC:
          if (!bad) jac();
          act = ACT_FACTOR;
          break;
        case ACT_FACTOR:
          if (!bad) bad = uc(factor() != 0);
          nsetups++;
          call_setup = 0;
          gamrat = crate = 1.0;
          gammap = gamma;
          nstlp = nst;
          m = -1;
          act = ACT_NEWTON;
          if (bad) {
            nflag = CONV_FAIL;
            act = ACT_NLS_END;
          }
          break;
        case ACT_NEWTON:
          if (m < 0) {
            m = 0;
            delp = 0.0;
          }
          rc = newton_pass(m, delp);
          if (rc == NEWTON_F) {
            call_f(ACT_NEWTON_F);
          } else if (rc == TRY_AGAIN) {
            call_setup = 1;
            convfail = CV_FAIL_BAD_J;
            act = ACT_NLS;
          } else {
            nflag = rc;
            act = ACT_NLS_END;
          }
          break;
        case ACT_NEWTON_F:
          act = ACT_NEWTON;
          if (bad && jcur) {
            nflag = RHSFUNC_RECVR;
            act = ACT_NLS_END;
          } else if (bad) {
            call_setup = 1;
            convfail = CV_FAIL_BAD_J;
            act = ACT_NLS;
          }
          break;
        case ACT_NLS_END: {
          int kflag = handle_nflag(&nflag, saved_t, &ncf);
          act = ACT_PREDICT;
          if (kflag == PREDICT_AGAIN) break;
          if (kflag != DO_ERROR_TEST) return kflag;
          int eflag = do_error_test(&nflag, saved_t, &nef, &dsm);
          if (eflag == TRY_AGAIN) break;
          if (eflag == ERR_TEST_F) {
            for (int i = lane; i < nv; i += kWave) y[i] = zn0()[i];
            wsync();
            call_f(ACT_RESTART);
            break;
          }
          if (eflag != CV_SUCCESS) return eflag;
          complete_step();
          prepare_next_step(dsm);
          etamax = (nst <= SMALL_NST) ? ETAMX2 : ETAMX3;
          nstloc++;
          act = ACT_MAIN;
          if (uc((tn - tout) * h >= 0.0)) {
            double s = (tout - tn) / h;
            for (int i = lane; i < nv; i += kWave) {
              double z[QMAX + 1], v = 0.0;
              hist_load(i, z);
#pragma unroll
              for (int j = QMAX; j >= 0; --j)
                if (j <= q) v = j == q ? z[j] : z[j] + s * v;
              y[i] = v;
            }
            wsync();
            next_h = hprime;
            return CV_SUCCESS;
          }
          break;
        }
        case ACT_RESTART:
          if (bad) return CV_UNREC_RHSFUNC_ERR;
          for (int i = lane; i < nv; i += kWave) zn1()[i] = h * ftemp[i];
          wsync();
          act = ACT_PREDICT;
          break;
      }
    }
  }
};

}  // namespace

// MP: multi-phase program (PL then kPlaceGlobal); PL: the variant (see
// kPlaceLds and following).  Each is compiled for the wavefronts per SIMD its
// LDS footprint lets onto a CU (one or two), which bounds its registers.
// BENCH: the measurement variant (bench_phases instead of the solve).
template <bool MP, int PL, bool BENCH = false>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(MP || PL == kPlaceLds || PL == kPlaceWide ? 1 : 2)))
    k_cell_bdf(CellBdfArgs a) {
  extern __shared__ double smem[];
  const DevProgram& P = a.P;
  constexpr bool GH = MP || PL != kPlaceLds;
  constexpr bool GL = MP || PL == kPlaceGlobalLu || PL == kPlaceWide;
  constexpr int kPlace = MP ? kPlaceGlobal : PL;
  // the wavefront index is uniform: a scalar, so the cell's LDS and scratch
  // pointers derived from it live in scalar registers
  int lane = threadIdx.x % kWave, wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  int nv = P.nv;
  size_t per_cell = cell_bdf_lds_doubles(P, kPlace);
  double* base = smem + (size_t)wv * per_cell;
  double* scratch = GH ? a.wave_scratch + ((size_t)blockIdx.x * (blockDim.x / kWave) + wv) *
                                              cell_bdf_wave_scratch(P, kPlace)
                       : nullptr;
  CellCv<MP, PL> cv;
  cv.lane = lane;
  cv.nv = nv;
  cv.s_state = base;
  constexpr bool kConstLds = MP || !GH;  // (else see CellCv::kt)
  constexpr bool kNewtonLds = GH && !MP && PL != kPlaceWide;
  double* sk_end = cv.s_state + P.ns;
  if (kConstLds) {
    cv.s_k = sk_end;
    sk_end += P.n_env;
  }
  sk_end = cv.s_state + even_up(sk_end - cv.s_state);
  cv.mpl = mp_lds(P, sk_end,
                  MP ? scratch + (P.lu_nnz + kWave + 1) + P.rnnz : nullptr);
  cv.s_rate = sk_end + mp_lds_doubles(P);
  double* v = cv.s_rate + 2 * (size_t)P.n_terms;
  // With GH the Nordsieck history and the work vectors other than y, acor
  // and w live in the wavefront's global scratch (after the LU where it is
  // global, and for multi-phase programs the J_rxn and Jacobian scalars);
  // else all in LDS.
  double* g = MP   ? scratch + (P.lu_nnz + kWave + 1) + P.rnnz + mp_jsc_doubles(P)
              : GL ? scratch + P.lu_nnz + kWave + 1
                   : scratch;
  double*& vh = GH ? g : v;
  // gas-phase cells with the history in global memory keep what every Newton
  // iteration and step reads in LDS: zn[0], zn[1], the error weights and the
  // iteration's two work vectors (six cells still fit a CU, as the rate
  // constants stay in global memory and the lanes' registers)
  if (kNewtonLds) {
    cv.z01 = v; v += 2 * (size_t)nv;
    cv.ewt = v; v += nv;
    cv.tempv = v; v += nv;
    cv.ftemp = v; v += nv;
  } else {
    cv.z01 = vh; vh += 2 * (size_t)nv;
    cv.ewt = vh; vh += nv;
    cv.tempv = vh; vh += nv;
    cv.ftemp = vh; vh += nv;
  }
  // (kPlaceGlobalLu has room in LDS for all of the history)
  double*& v2 = !MP && PL == kPlaceGlobalLu ? v : vh;
  cv.z2 = v2; v2 += 4 * (size_t)nv;
  cv.last = v2; v2 += nv;
  cv.acinit = v2; v2 += nv;
  cv.E = nullptr;
  if (GH) {
    cv.E = vh; vh += est_doubles(P);
  }
  cv.acor = v; v += nv;
  cv.y = v; v += nv;
  // the solve's scratch w (used past kTriInPlace only) stays in LDS except where
  // it would take a place from another cell of a small program
  if (kNewtonLds) {
    cv.w = vh; vh += nv;
  } else {
    cv.w = v; v += nv;
  }
  // Without GH the J history (J_solver, J_state, J_deriv) is staged in LDS
  // for the whole solve; with GH it is used in place in HBM.
  double *h_js = nullptr, *h_jy = nullptr, *h_jf = nullptr;
  // the f gather's scratch follows the LU values (their zero slot lies in it)
  if (MP) {
    cv.lu = scratch;
    cv.Jr = scratch + P.lu_nnz + kWave + 1;
    cv.s_fb = v; v += fb_scratch_doubles(P);
  } else {
    cv.Jr = nullptr;
    if (GL) {
      cv.lu = scratch;
    } else {
      cv.lu = v;
      v += kNewtonLds ? cell_lu_lds(P) : P.lu_nnz;
    }
    cv.s_fb = v; v += fb_scratch_doubles(P);
    if (!GH) {
      h_js = v; v += P.nnz;
      h_jy = v; v += nv;
      h_jf = v; v += nv;
    }
  }
  cv.l = v;
  cv.tq = v + 6;
  cv.tau = v + 12;
  cv.rtol = a.rtol;
  cv.guess_on = a.guess_on;
  cv.maxcf = a.max_conv_fails;
  cv.max_steps = a.max_steps;
  cv.prof = !BENCH && a.prof != nullptr;

  for (;;) {
    const DevProgram& P = cv.program();
    int q = 0;
    if (lane == 0) q = atomicAdd(a.counter, 1);
    q = __builtin_amdgcn_readfirstlane(q);  // lane 0's ticket, as a scalar
    if (q >= a.nc) break;
    int cell = a.cell_list ? a.cell_list[q] : q;
    double t1 = a.cell_t1 ? a.cell_t1[cell] : a.t1;
    int nsteps = a.cell_nsteps ? a.cell_nsteps[cell] : 1;
    for (int step = 0; step < nsteps; ++step) {
      if (a.poison) {
        const double nan = __builtin_nan("");
        for (size_t i = lane; i < per_cell; i += kWave) base[i] = nan;
        if (GH)
          for (size_t i = lane; i < cell_bdf_wave_scratch(P, kPlace); i += kWave) scratch[i] = nan;
        __threadfence_block();
        wsync();
      }
      double* state_c = a.state + (size_t)cell * P.ns;
      double* renv_c = a.rxn_env + (size_t)cell * P.n_env;
      double* g_js = a.Js + (size_t)cell * P.nnz;
      double* g_jy = a.Jy + (size_t)cell * nv;
      double* g_jf = a.Jf + (size_t)cell * nv;
      if (GH) {
        cv.Js = g_js;
        cv.Jy = g_jy;
        cv.Jf = g_jf;
      } else {
        for (int e = lane; e < P.nnz; e += kWave) h_js[e] = g_js[e];
        for (int i = lane; i < nv; i += kWave) {
          h_jy[i] = g_jy[i];
          h_jf[i] = g_jf[i];
        }
        cv.Js = h_js;
        cv.Jy = h_jy;
        cv.Jf = h_jf;
      }
      // stage state (constants clamped in place) and rate data
      for (int i = lane; i < P.ns; i += kWave) {
        double s = state_c[i];
        cv.s_state[i] = s;
        if (a.var_type[i] != 1) {
          s = s > 1.0e-60 ? s : 1.0e-60;
          cv.s_state[i] = s;
          state_c[i] = s;
        }
      }
      if (!kConstLds)
        cv.s_k = renv_c;
      else
        for (int i = lane; i < P.n_env; i += kWave) cv.s_k[i] = renv_c[i];
      wsync();
      // rate constants for the cell's environment (rxn_update_env_state)
      double T = a.env[2 * cell], Pa = a.env[2 * cell + 1];
      cell_rate_constants(P, lane, T, Pa, cv.s_k);
      wsync();
      if (MP) mp_cell_env(P, lane, T, Pa, cv.mpl);
      if (!kConstLds) {
        __threadfence_block();
        cv.load_term_constants();
      } else {
        for (int i = lane; i < P.n_env; i += kWave) renv_c[i] = cv.s_k[i];
      }
      for (int i = lane; i < nv; i += kWave) {
        double s = cv.s_state[P.dep_state[i]];
        cv.zn0()[i] = s > 1.0e-60 ? s : 1.0e-60;
      }
      wsync();
      cv.stage_history(P);
      cv.c_f = cv.c_j = cv.c_lu = cv.c_sol = cv.c_fr = cv.c_fg = 0;
      long long c_start = cv.tick();
      int flag;
      if constexpr (BENCH)
        flag = cv.bench_phases(a.bench_reps, a.prof + (size_t)cell * kCellProf);
      else
        flag = cv.solve(a.t0, t1);
      if (flag >= 0) {
        for (int i = lane; i < nv; i += kWave) {
          double yv = cv.y[i];
          state_c[P.dep_state[i]] = yv > 0.0 ? yv : 0.0;
          if (MP) cv.s_state[P.dep_state[i]] = yv > 0.0 ? yv : 0.0;
        }
        if (MP) {
          // the post-solve sub_model_calculate (camp_solver.c:685-687) on the
          // final state; the sub models' outputs go back to the state array
          wsync();
          mp_zsr(P, lane, cv.mpl.sub_env, cv.s_state, cv.mpl.slot);
          for (int z = lane; z < P.n_zi; z += kWave)
            state_c[P.zi_water[z]] = cv.s_state[P.zi_water[z]];
        }
      }
      if (!GH) {
        wsync();
        for (int e = lane; e < P.nnz; e += kWave) g_js[e] = h_js[e];
        for (int i = lane; i < nv; i += kWave) {
          g_jy[i] = h_jy[i];
          g_jf[i] = h_jf[i];
        }
      }
      if (lane == 0) {
        double* st = a.stats + (size_t)cell * kCellStats;
        st[0] = cv.nst; st[1] = cv.nfe; st[2] = cv.nsetups; st[3] = cv.netf;
        st[4] = cv.nni; st[5] = cv.ncfn; st[6] = cv.nje; st[7] = flag;
        st[8] = cv.hu; st[9] = cv.next_h;
        if (a.fail_count && flag < 0) a.fail_count[cell] += 1;
        if (cv.prof) {
          double* pr = a.prof + (size_t)cell * kCellProf;
          pr[0] = (double)cv.c_f; pr[1] = (double)cv.c_j; pr[2] = (double)cv.c_lu;
          pr[3] = (double)cv.c_sol; pr[4] = (double)(clock64() - c_start);
          pr[5] = (double)cv.c_fr; pr[6] = (double)cv.c_fg;
        }
      }
      wsync();
    }
  }
}

// Per-cell LDS beyond 64 KiB per block (multi-phase programs, or several
// cells per workgroup) is opted into per kernel; gfx950 has 160 KiB per CU.
static const void* cell_bdf_fn(const DevProgram& P, int place) {
  if (P.mp) return (const void*)k_cell_bdf<true, kPlaceGlobal>;
  switch (place) {
    case kPlaceGlobal: return (const void*)k_cell_bdf<false, kPlaceGlobal>;
    case kPlaceGlobalLu: return (const void*)k_cell_bdf<false, kPlaceGlobalLu>;
    case kPlaceWide: return (const void*)k_cell_bdf<false, kPlaceWide>;
    default: return (const void*)k_cell_bdf<false, kPlaceLds>;
  }
}

void launch_cell_bdf(const CellBdfArgs& a, int grid, int block, size_t lds, hipStream_t s) {
  allow_lds(cell_bdf_fn(a.P, a.place), lds);
  if (a.P.mp)
    hipLaunchKernelGGL((k_cell_bdf<true, kPlaceGlobal>), dim3(grid), dim3(block), lds, s, a);
  else if (a.place == kPlaceGlobal)
    hipLaunchKernelGGL((k_cell_bdf<false, kPlaceGlobal>), dim3(grid), dim3(block), lds, s, a);
  else if (a.place == kPlaceGlobalLu)
    hipLaunchKernelGGL((k_cell_bdf<false, kPlaceGlobalLu>), dim3(grid), dim3(block), lds, s, a);
  else if (a.place == kPlaceWide)
    hipLaunchKernelGGL((k_cell_bdf<false, kPlaceWide>), dim3(grid), dim3(block), lds, s, a);
  else
    hipLaunchKernelGGL((k_cell_bdf<false, kPlaceLds>), dim3(grid), dim3(block), lds, s, a);
}

void launch_cell_bdf_bench(const CellBdfArgs& a, int grid, int block, size_t lds,
                           hipStream_t s) {
  allow_lds(cell_bdf_fn(a.P, a.place), lds);
  if (a.P.mp) {
    allow_lds((const void*)k_cell_bdf<true, kPlaceGlobal, true>, lds);
    hipLaunchKernelGGL((k_cell_bdf<true, kPlaceGlobal, true>), dim3(grid), dim3(block), lds, s,
                       a);
  } else if (a.place == kPlaceGlobal) {
    allow_lds((const void*)k_cell_bdf<false, kPlaceGlobal, true>, lds);
    hipLaunchKernelGGL((k_cell_bdf<false, kPlaceGlobal, true>), dim3(grid), dim3(block), lds, s,
                       a);
  } else if (a.place == kPlaceLds) {
    allow_lds((const void*)k_cell_bdf<false, kPlaceLds, true>, lds);
    hipLaunchKernelGGL((k_cell_bdf<false, kPlaceLds, true>), dim3(grid), dim3(block), lds, s, a);
  } else {
    die("phase measurement: placements 0 and 1 only");
  }
}

int cell_bdf_blocks_per_cu(const DevProgram& P, int place, int block, size_t lds) {
  if (block > 256 || lds > kMaxLds) return 0;
  const void* fn = cell_bdf_fn(P, place);
  allow_lds(fn, lds);
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, block, lds) != hipSuccess) return 0;
  return n;
}

// ---------------------------------------------------------------------
// The no-allocation entry point's scratch: the queue counter and the
// wavefronts' global scratch of camp_solver_run_device_noalloc.  Host code
// never uses the array's name as an address: each device's copy is looked
// up once, with that device current, with hipGetSymbolAddress.
// ---------------------------------------------------------------------
static __device__ __align__(256) double scratch[kNoAllocScratchDoubles];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {nullptr};
}  // namespace

// This device's copy of the scratch (nullptr, with a message, on failure).
double* noalloc_scratch() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    std::fprintf(stderr, "camp_solver_run_device_noalloc: no current HIP device\n");
    return nullptr;
  }
  std::lock_guard<std::mutex> g(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      std::fprintf(stderr, "camp_solver_run_device_noalloc: hipGetSymbolAddress failed: %s\n",
                   hipGetErrorString(e));
      return nullptr;
    }
    g_scratch_ptr[dev] = static_cast<double*>(ptr);
  }
  return g_scratch_ptr[dev];
}

}  // namespace camp

// camp_solver_run_device without any allocation (see include/camp_solver.h).
extern "C" int camp_solver_run_device_noalloc(void* solver_data, double* d_state, double* d_env,
                                              double t_initial, double t_final) {
  using namespace camp;
  Solver* s = static_cast<Solver*>(solver_data);
  if (!s || !s->m.initialized) return CAMP_NOALLOC_NOT_READY;
  // the solver's own device buffers are made by its first device call
  if (!s->stream) {
    std::fprintf(stderr, "camp_solver_run_device_noalloc: the solver's device buffers do not "
                         "exist yet (any earlier call that uses the device makes them)\n");
    return CAMP_NOALLOC_NOT_READY;
  }
  if (s->mode != CAMP_MODE_PER_CELL || s->profiling || s->eval_jac) {
    std::fprintf(stderr, "camp_solver_run_device_noalloc: per-cell mode only, without phase "
                         "timing or the Jacobian check\n");
    return CAMP_NOALLOC_UNSUPPORTED;
  }
  const size_t per_wave = cell_bdf_wave_scratch(s->P, s->variant());
  if (per_wave > kNoAllocScratchDoubles - kNoAllocHeaderDoubles) {
    std::fprintf(stderr, "camp_solver_run_device_noalloc: one wavefront needs %zu doubles of "
                         "scratch, more than the %zu available\n",
                 per_wave, kNoAllocScratchDoubles - kNoAllocHeaderDoubles);
    return CAMP_NOALLOC_TOO_LARGE;
  }
  double* sc = noalloc_scratch();
  if (!sc) return CAMP_NOALLOC_NOT_READY;
  s->upload_renv();
  if (s->m.n_rxn == 0) return CAMP_SOLVER_SUCCESS;
  int rc = s->run_cells(d_state, d_env, t_initial, t_final, sc, kNoAllocScratchDoubles);
  HIP_OK(hipStreamSynchronize(s->stream));
  return rc;
}
