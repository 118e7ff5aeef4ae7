// Time integrators (internal): device-resident Krylov expv and Dormand-Prince 5(4).
#pragma once

#include <algorithm>
#include <cmath>
#include <memory>

#include "nc_sens.h"

struct nc_solver_s {
  nc_matrix_s* A = nullptr;  // borrowed; must outlive the solver (the base generator for SA)
  nc_sensmatrix_s* SA = nullptr;  // sensitivity operator (borrowed), or null
  int blocks = 1;                 // P+1 for the sensitivity system
  int64_t Nb = 0, Npb = 0;        // true and padded rows per block
  nc_solve_opts opts{};
  int method = NC_METHOD_KRYLOV;
  int64_t N = 0;   // true vector length (blocks * Nb)
  int64_t Np = 0;  // padded length (blocks * Npb, Npb a multiple of 1024); padding stays zero
  size_t vs = 8;
  double t = 0.0;
  bool have_state = false;
  hipStream_t s = nullptr;  // the matrix's stream
  nc::DevBuf<double> u;     // FP64 master state [p; sinks]
  nc::DevBuf<double> u0;    // state uploaded by the last set_state (for restart)
  double t0 = 0.0, beta0 = 0.0;
  nc::DevBuf<double> snaps; // n_out x Np (padded layout)
  int32_t n_snaps = 0;
  // reduction scratch
  nc::DevBuf<double> partials;
  unsigned red_blocks = 0;
  int64_t kn = 0, kblk = 0;  // Krylov columns: rows summed in blocks, and the blocks
  int kgroups = 0;           // their workgroups
  // Krylov
  int m = 30;
  nc::DevBuf<unsigned char> V;  // (m+1) x N, VT, unnormalised
  nc::DevBuf<double> q;         // FP64 mat-vec outputs of two columns
  nc::DevBuf<double> kbuf;      // H (m+2)^2 | sc (m+2) | misc (8) | sink rows
  double* hbuf = nullptr;       // pinned host copy of kbuf, written by the process's last launch
  double* hbuf_dev = nullptr;   // the same block as a device address
  double* hpart = nullptr;      // pinned host copy of per-block partial sums
  int64_t hpart_cap = 0;        // partial slots of hpart before its sink-value region
  double* hpart_dev = nullptr;  // the same pinned block as a device address: the RK error
                                // pass writes its partials there directly
  double beta = 0.0, t_new = 0.0, anorm = 0.0;
  bool started = false;
  hipGraph_t arnoldi_graph = nullptr;  // captured Arnoldi process (replayed every step)
  hipGraphExec_t arnoldi_exec = nullptr;
  uint64_t arnoldi_gen = 0;  // the matrix's launch_gen when the graph was captured
  // RK
  nc::DevBuf<unsigned char> rkv;   // VT copy of the stage input
  nc::DevBuf<unsigned char> rkv2;  // the other stage-input buffer (epilogue-formed stages)
  nc::DevBuf<double> k;            // 7 x N stage derivatives (FP64)
  nc::DevBuf<double> ytmp;         // N
  double h = 0.0;
  int ksw = 0;  // 1: RK stages 0 and 6 have traded slots in k
  bool fsal_valid = false;
  nc_solve_stats st{};
  // state list shared by the snapshot vectors handed out (nc_solver_get_fspvec)
  std::shared_ptr<nc::DevBuf<int32_t>> snap_states;
  uint64_t snap_space_uid = 0, snap_version = 0;
  ~nc_solver_s() {
    if (arnoldi_exec) (void)hipGraphExecDestroy(arnoldi_exec);
    if (arnoldi_graph) (void)hipGraphDestroy(arnoldi_graph);
    if (s) (void)hipStreamSynchronize(s);  // copies into the pinned blocks have landed
    if (hbuf) nc::pinned_free(hbuf);
    if (hpart) nc::pinned_free(hpart);
  }
};

namespace nc {
// FSP sink-mass budget of the adaptive solve: integration stops where
// g(t) = sum(sinks) - fsptol * t / tend crosses zero from below (fspsolve.jl:141-156).
struct EventSpec {
  double fsptol = 0.0, tend = 1.0;
  bool fired = false;
};
// The Krylov process of a small space in one launch (nc_krylov_small.hip): with nv >= 0 it
// first ends the step before, u <- cu u + sum_{i < nv} cs[i] V_{i+1}. H, the scales, norms
// and sink rows go to hbuf.
bool krylov_small_fits(const nc_solver_s* S);
void krylov_small_launch(nc_solver_s* S, int nv, double cu, const double* cs);
// Error per unit time that a step's estimate is held to. With full orthogonalisation the
// error lay two to three orders below the estimate, with two vectors it comes near it: held to
// the tolerance itself, FP64 errors grew by up to a thousand times (telegraph box of 120
// counts over 200 time units at 1e-9: full 49 steps, 6.5e-12; two vectors 63 steps, 2.5e-9).
// 10^(-m/10) of it makes every step a fifth shorter whatever m is, and the errors are the full
// form's or less (78 steps, 1.0e-13; sweep of 42 FP64 solves at 1e-9 and 1e-12: none above
// it). Not below 1e-14, where the estimate is rounding.
inline double krylov_step_tol(const nc_solver_s* S) {
  const double tol = S->opts.krylov_tol;
  return std::max(tol * std::pow(10.0, -0.1 * S->m), std::min(tol, 1e-14));
}
// Happy breakdown: the residual of the exhausted space is |beta| h per unit time, so h has to
// fall below the tolerance the caller asks for, per unit time too (Expokit's fixed 1e-7 let
// solves near a stationary state jump to the next output with 2e-5 of error), and in FP64
// storage below 1e-8 at any tolerance: that jump is most of the error there. In FP32 h does
// not fall much below 1e-7, and a smaller threshold costs four times the steps.
inline double krylov_breakdown_tol(const nc_solver_s* S) {
  const double most = S->vs == 8 ? 1e-8 : 1e-7;
  return std::max(std::min(S->opts.krylov_tol, most), 1e-14);
}
// Error that a step need not go below, relative to |V_0|: the first vector rounded to FP32 is
// off by about 2^-25 of its norm to begin with. Steps that followed the estimate further down
// resolved that rounding: near the stationary state of a telegraph box of 300 counts a
// tolerance of 1e-9 took 1,181 steps (93 ms) and 1e-12 1,659 (128 ms), now 765 (61 ms) and 784
// (62 ms) at the same error of 8e-9. Not below 12 vectors, where the steps are many and their
// truncation, unlike the rounding, does not average out (three vectors: 3e-9 of error would
// become 2e-7), and not for sensitivities, whose norm says nothing of the rounding of p.
inline double krylov_floor(const nc_solver_s* S) {
  return S->vs == 4 && S->m >= 12 && !S->SA ? 0x1p-26 : 0.0;
}
// Advance to t_target (or to the budget crossing when ev is given); with one_step the
// call returns after the first accepted step.
void krylov_advance(nc_solver_s* S, double t_target, EventSpec* ev = nullptr, bool one_step = false);
void rk_advance(nc_solver_s* S, double t_target, EventSpec* ev = nullptr, bool one_step = false);
// Internal entry points shared with the adaptive driver.
nc_solver_s* solver_create(nc_matrix_s* A, const nc_solve_opts* opts, nc_sensmatrix_s* SA = nullptr);
void solver_set_state_device(nc_solver_s* S, double t0, const double* u_dev);
// Step size the integrator would try next (RK: h, Krylov: tau), 0 before its first step.
double solver_step_hint(const nc_solver_s* S);
// Start the next step from h instead of the automatic first step (h <= 0: no change).
void solver_seed_step(nc_solver_s* S, double h);
void solver_reduce_setup(nc_solver_s* S);
}  // namespace nc
