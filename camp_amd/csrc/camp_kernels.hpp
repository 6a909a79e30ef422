// Launch interface between the host solver (camp_solver.cpp) and the HIP
// kernels (camp_kernels.hip, camp_cell_bdf.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "camp_device.hpp"
#include "camp_model.hpp"
#include "camp_mp_device.hpp"

namespace camp {

constexpr int kCellStats = 10;  // nst nfe nsetups netf nni ncfn nje flag hu next_h

// LDS of a CU.  A kernel opts into more than 64 KiB a block once and for all
// (the limit belongs to the function, which solvers and threads share: set to
// each launch's own size it would lower another's).
constexpr size_t kMaxLds = 160 * 1024;
inline void allow_lds(const void* fn, size_t lds) {
  if (lds > 65536 && lds <= kMaxLds)
    (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds);
}

// shader cycles per cell: f, Jac, LU factor, LU solve, whole solve, and the
// two parts of f (state update + rates, species gather + estimate blend)
constexpr int kCellProf = 7;

// Where a cell's working set lives in the persistent kernel.  Every variant
// keeps the state, the per-term rates, y, acor, the f gather's scratch and the
// BDF coefficient arrays l, tq and tau (24 slots) in LDS.
//  kPlaceLds     everything else too: rate constants, Nordsieck history (6
//                vectors), 8 work vectors, LU factors, J history (gas phase
//                only: 4 cells per CU for the CB05-scale mechanism);
//  kPlaceGlobal  gas phase: zn[0], zn[1], the error weights, tempv, ftemp and
//                the LU factors in LDS; Nordsieck vectors 2 to 5, last,
//                acinit, w and the J history in f's order in the wavefront's
//                global scratch; rate constants and J history in place in HBM
//                (6 cells per CU).  Multi-phase programs always run this
//                variant, with y, acor, w and the rate constants in LDS and
//                their other vectors, LU factors, reaction Jacobian and
//                per-instance Jacobian scalars in the scratch.
//  kPlaceGlobalLu  gas phase: the LU factors, w and the J history in f's order
//                in the scratch, all other vectors in LDS, rate constants and
//                J history in HBM (8 cells per CU).
//  kPlaceWide    gas phase: all vectors but y, acor and w, and the LU factors,
//                in the scratch.  Needs the least LDS; for programs of which no
//                cell fits with the placement asked for (the vectors in LDS
//                outgrow it with the number of solver variables).
// The gas-phase kernels of kPlaceGlobal and kPlaceGlobalLu are compiled for two
// wavefronts per SIMD, the others for one.
constexpr int kPlaceLds = 0, kPlaceGlobal = 1, kPlaceGlobalLu = 2, kNumPlacements = 3,
              kPlaceWide = 3;
// LU factors in the wavefront's global scratch
__host__ __device__ inline bool cell_lu_global(const DevProgram& P, int place) {
  return P.mp || place == kPlaceGlobalLu || place == kPlaceWide;
}
// vectors of a cell in LDS
__host__ __device__ inline int cell_lds_vectors(const DevProgram& P, int place) {
  return P.mp || place == kPlaceWide ? 3 : place == kPlaceLds ? 14 : place == kPlaceGlobal ? 7 : 13;
}
// rate constants in LDS (gas-phase cells with the J history in global memory
// read them there too)
__host__ __device__ inline size_t cell_lds_env(const DevProgram& P, int place) {
  return P.mp || place == kPlaceLds ? (size_t)P.n_env : 0;
}
// gas-phase kPlaceGlobal: the LU's LDS, where J(y) also stages the rate constants
__host__ __device__ inline size_t cell_lu_lds(const DevProgram& P) {
  return P.lu_nnz > P.n_env ? P.lu_nnz : P.n_env;
}
// LDS doubles of a cell; place: the variant launched (any for multi-phase)
__host__ __device__ inline size_t cell_bdf_lds_doubles(const DevProgram& P, int place) {
  const bool lds = !P.mp && place == kPlaceLds;
  return even_up(P.ns + cell_lds_env(P, place)) + mp_lds_doubles(P) +
         even_up(2 * (size_t)P.n_terms + (size_t)cell_lds_vectors(P, place) * P.nv + fb_scratch_doubles(P) +
         (cell_lu_global(P, place) ? 0 : place == kPlaceGlobal ? cell_lu_lds(P) : (size_t)P.lu_nnz) +
         (lds ? (size_t)P.nnz + 2 * (size_t)P.nv : 0) + 24);
}
// The variant that runs placement `place`, cpb cells a workgroup: itself where
// it fits a CU, else kPlaceWide.
inline int cell_placement(const DevProgram& P, int place, int cpb = 1) {
  if (P.mp) return kPlaceGlobal;
  return cpb * cell_bdf_lds_doubles(P, place) * sizeof(double) <= kMaxLds ? place : kPlaceWide;
}
// Global scratch doubles per wavefront: the LU factors where they are global
// (with the zero slot), for multi-phase programs then the reaction Jacobian and
// the per-instance Jacobian scalars, then the vectors not in LDS (of 14) and
// the J history in f's order.
__host__ __device__ inline size_t cell_bdf_wave_scratch(const DevProgram& P, int place) {
  if (!P.mp && place == kPlaceLds) return 0;
  return (cell_lu_global(P, place) ? (size_t)P.lu_nnz + kWave + 1 : 0) +
         (P.mp ? P.rnnz + mp_jsc_doubles(P) : 0) +
         (size_t)(14 - cell_lds_vectors(P, place)) * P.nv + est_doubles(P);
}

// The no-allocation entry point's scratch (a file-scope device array of
// kNoAllocScratchDoubles doubles, 96 MiB, 316 wavefronts of the CB05-scale
// mechanism with eight aerosol bins): the first kNoAllocHeaderDoubles
// (256 bytes) hold the queue counter, the rest the wavefronts' scratch.
constexpr size_t kNoAllocScratchDoubles = (size_t)12 << 20;
constexpr size_t kNoAllocHeaderDoubles = 32;

struct CellBdfArgs {
  DevProgram P;
  int nc;
  double* state;        // [nc][ns] in/out
  const double* env;    // [nc][2]
  double* rxn_env;      // [nc][n_env] in/out (rate constants written back)
  double *Js, *Jy, *Jf; // per-cell J history
  const int* var_type;  // [ns]
  double rtol, t0, t1;
  int max_steps, max_conv_fails, guess_on;
  int* counter;         // work queue head (zeroed before launch)
  double* stats;        // [nc][kCellStats]
  // Optional indirection used by the request server: queue position q
  // solves cell cell_list[q] (nullptr: cell q) over [t0, cell_t1[cell]]
  // (nullptr: [t0, t1]).  nc is then the length of cell_list.
  const int* cell_list = nullptr;
  const double* cell_t1 = nullptr;
  double* prof = nullptr;  // [cells][kCellProf] when phase timing is on
  int* fail_count = nullptr;  // per cell: incremented on each failed solve
  double* wave_scratch = nullptr;  // [grid waves][cell_bdf_wave_scratch]
  // Optional: cell solves cell_nsteps[cell] consecutive timesteps over
  // [t0, t1] in this launch, each exactly as a separate launch would
  // (state written back and restaged between them); nullptr: one.
  const int* cell_nsteps = nullptr;
  int place = kPlaceLds;  // the kernel variant (cell_placement)
  // Check of per-cell independence: when non-zero, every wavefront fills its
  // whole working memory (the cell's LDS region and, for multi-phase
  // programs, its global scratch) with quiet NaNs before it stages each
  // cell, so that any value a cell reads before writing shows in its result.
  int poison = 0;
  int bench_reps = 0;  // launch_cell_bdf_bench: repetitions per phase
};

void launch_cell_bdf(const CellBdfArgs& a, int grid, int block, size_t lds, hipStream_t s);
// the measurement variant: per cell, the cycles of f, J, LU and one solve
// into prof[cell][0..3] (gas-phase programs, placements 0 and 1)
void launch_cell_bdf_bench(const CellBdfArgs& a, int grid, int block, size_t lds, hipStream_t s);
// workgroups per CU of the variant (program kind and placement) at this
// block size and LDS, 0 if it does not fit
int cell_bdf_blocks_per_cu(const DevProgram& P, int place, int block, size_t lds);

__global__ void k_rates(DevProgram P, int nc, const double* env, double* rxn_env);
__global__ void k_deriv(DevProgram P, int nc, const double* y, const double* state,
                        const double* env, const double* rxn_env, const double* Js,
                        const double* Jy, const double* Jf, double* fout, double h, int use_est,
                        int* fail);
// Jr: reaction-Jacobian scratch [nc][rnnz] of multi-phase programs (else unused)
__global__ void k_jac(DevProgram P, int nc, const double* y, const double* state,
                      const double* env, const double* rxn_env, double* J, double h, double* Jr);
// LDS doubles per wavefront of k_deriv and k_jac (f's gather scratch and J's
// per-instance scalars share a place; the estimate's dy last, where it fits; without: k_check_jac, whose f takes no estimate), and wavefronts per
// block: one for multi-phase programs, whose per-cell extras are large, else up
// to four, as many as fit.
__host__ __device__ inline size_t fj_lds_doubles_no_dy(const DevProgram& P) {
  return even_up((size_t)P.ns + P.n_env) + mp_lds_doubles(P) +
         even_up(2 * (size_t)P.n_terms +
                 (mp_jsc_doubles(P) > fb_lds_doubles(P) ? mp_jsc_doubles(P) : fb_lds_doubles(P)));
}
__host__ __device__ inline bool fj_dy(const DevProgram& P) {
  return (fj_lds_doubles_no_dy(P) + even_up(P.nv)) * sizeof(double) <= kMaxLds;
}
__host__ __device__ inline size_t fj_lds_doubles(const DevProgram& P) {
  return fj_lds_doubles_no_dy(P) + (fj_dy(P) ? even_up(P.nv) : 0);
}
inline int fj_waves_per_block(const DevProgram& P) {
  int w = P.mp ? 1 : 4;
  while (w > 1 && w * fj_lds_doubles(P) * sizeof(double) > kMaxLds) w /= 2;
  return w;
}

// Lane-group f(y) and J(y) of gas-phase programs (lanes per cell = 8, 16
// or 32; camp_kernels.hip) and the compact rate-constant array they read.
__global__ void k_kval(DevProgram P, int nc, const double* rxn_env, double* kval);
// hp (may be null): the time step read from device memory instead of h
void launch_group_deriv(int lanes, const DevProgram& P, int nc, const double* y,
                        const double* state, const double* kval, const double* Js,
                        const double* Jy, const double* Jf, double* fout, double h,
                        const double* hp, int use_est, int* fail, hipStream_t st);
void launch_group_jac(int lanes, const DevProgram& P, int nc, const double* y,
                      const double* state, const double* kval, double* J, double h,
                      hipStream_t st);
// Per-cell LDS stride of the lane-group kernels: the state, (the blended f)
// the gather's running sums 2 nv + 2, the compact rate constants; odd, so
// that the cells of a wavefront start in different LDS banks.
__host__ __device__ inline int group_cell_stride(const DevProgram& P, bool fsum) {
  return (P.ns + (fsum ? 2 * P.nv + 2 : 0) + P.n_k) | 1;
}
inline size_t group_lds_bytes(const DevProgram& P, int lanes, bool fsum) {
  return (size_t)(kWave / lanes) * group_cell_stride(P, fsum) * sizeof(double);
}
// The J kernel also stages its cells' Jacobians (nnz each) and writes them
// out contiguously.
inline size_t group_jac_lds_bytes(const DevProgram& P, int lanes) {
  return group_lds_bytes(P, lanes, false) + (size_t)(kWave / lanes) * P.nnz * sizeof(double);
}
// LDS of k_lu_factor: the LU values, the zero slot and the tail's buffers
inline size_t lu_factor_lds_bytes(const DevProgram& P) {
  return ((size_t)P.lu_nnz + kWave + 1 + kLuTailBuf) * sizeof(double);
}
__global__ void k_lu_factor(DevProgram P, int nc, const double* J, double gamma, double* LU,
                            int* fail);
// sp (may be null): the scale read from device memory instead of s
__global__ void k_lu_solve(DevProgram P, int nc, const double* LU, double* b, double s,
                           const double* sp);
__global__ void k_vec_lin(long n, double a, const double* x, double b, const double* y,
                          double* z);
__global__ void k_vec_scale(long n, double a, double* x);
__global__ void k_vec_pascal(long n, int q, double* zn, int sign);
__global__ void k_vec_rescale(long n, int q, double eta, double* zn);
struct Coef6 {
  double v[6];
};
__global__ void k_vec_complete(long n, int q, Coef6 l6, const double* acor, double* zn, int save,
                               double* last, int projected, const double* y);
// ctl (may be null): rl1 = ctl[0], gamma = ctl[1] from device memory
__global__ void k_vec_resid(long n, double rl1, const double* zn1, const double* acor,
                            double gamma, const double* ftemp, double* tempv, const double* ctl);
__global__ void k_vec_newton_update(long n, const double* b, double* acor, const double* zn0,
                                    double* y);
__global__ void k_vec_ewt(long n, int nv, double rtol, const double* atol, const double* y,
                          double* ewt);
__global__ void k_vec_interp(long n, int q, double s, const double* zn, double* y);
__global__ void k_vec_wsq(long n, const double* x, const double* w, double* out);
__global__ void k_vec_min(long n, const double* x, double* out);
__global__ void k_gather_rows(long n, int len, long stride, const double* src, double* dst);
__global__ void k_vec_negmax(long n, const double* x, const double* w, double* out);
__global__ void k_vec_project(long n, const double* zn0, double* acor, double* y);
__global__ void k_vec_tstar(long n, const double* tmp1, const double* corr, double h_j,
                            double* out);
__global__ void k_fill(long n, double v, double* x);
__global__ void k_fill_int(long n, int v, int* x);
__global__ void k_check_jac(DevProgram P, int nc, const double* y, const double* state,
                            const double* env, const double* rxn_env, const double* J, double h_ts,
                            int* cell_fails);
inline size_t check_jac_lds_doubles(const DevProgram& P) {
  return fj_lds_doubles_no_dy(P) + 4 * (size_t)P.nv + 2 * (size_t)P.nnz;
}
// renv[c][upd_off[u]] = rates[c][u] for c < n_cells, u < n_upd
__global__ void k_scatter_rates(int n_cells, int n_upd, const int* upd_off, const double* rates,
                                int n_env, double* renv);
__global__ void k_clamp_constants(DevProgram P, int nc, const int* var_type, double* state);
__global__ void k_state_gather(DevProgram P, int nc, const double* state, double* y);
__global__ void k_state_take(DevProgram P, int nc, const double* state, double* y);
__global__ void k_state_scatter(DevProgram P, int nc, const double* y, double* state);

}  // namespace camp
