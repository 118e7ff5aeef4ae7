// Device-resident time integration of the FSP ODE du/dt = A(t) u.
//
// Replaces the integrator loop of NumCME.jl's solve (src/transientcme/sparse/fspsolve.jl:
// 10-41, a DifferentialEquations.jl/CVODE call around matvec!) with:
//
//  * Krylov expv for time-invariant generators: incomplete orthogonalisation against the
//    last two basis vectors (nc_iop.h), FP64 dot products and coefficients, basis vectors
//    stored in the matrix precision, one launch per basis vector; the
//    (m+2)x(m+2) Hessenberg exponential, the local error estimate and the step-size
//    control run on the host, following R. B. Sidje, "Expokit: a software package for
//    computing matrix exponentials", ACM TOMS 24(1), 1998 (algorithm of its EXPV
//    routine). One host synchronisation per Krylov step.
//  * Dormand-Prince 5(4) (J. R. Dormand & P. J. Prince, J. Comput. Appl. Math. 6, 1980)
//    with FSAL, the Hairer-Norsett-Wanner RMS error norm computed on the device in FP64,
//    and output times hit exactly by step clamping.
//
// Vectors: the master state u is FP64; mat-vec inputs are stored in the matrix precision.
#include <algorithm>
#include <cmath>
#include <limits>
#include <type_traits>

#include "nc_fspvec.h"
#include "nc_solver.h"

namespace nc {

namespace {

constexpr int kBlock = 256;
constexpr int kMaxRedBlocks = 2048;

constexpr int kFinBlock = 1024;          // threads of the square-sum fold
constexpr unsigned kVecBlocks = 512;     // grid of the vector passes
constexpr int kLoadChunk = 8;  // basis vectors whose loads a vector pass issues together

__device__ inline double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

template <typename T, int R>
struct alignas(sizeof(T) * R) Pack {
  T v[R];
};

// The end of a Krylov step: u <- cu u + sum_i cs[i] V_{i+1} (the coefficients are kernel
// arguments: no upload), with the next step's V_0 in storage precision. HBM / Infinity
// Cache bound: every basis vector once.
template <typename BT>
struct CombineArgs {
  int64_t N;
  int nv;  // vectors V_1 .. V_nv
  const BT* V1;
  BT* v0;
  double* u;
  double cu;
  double cs[32];
};

// Each thread owns 4 consecutive rows and reads every stream with one 16-byte (FP32) or
// 32-byte (FP64) vector load per vector; N is a multiple of 4 and all vectors are zero
// beyond the true length, so no tail handling is needed. The basis is read in chunks of
// kLoadChunk vectors whose loads are issued together (unconditional, index clamped to
// nv - 1: a guarded load becomes a branch that waits for it) and kept ahead of their
// arithmetic by a scheduling barrier; left to itself the scheduler reuses one register set
// and waits after every load. Vectors beyond nv carry a zero coefficient.
template <typename BT, int MAXV>
__global__ __launch_bounds__(kBlock) void k_combine(CombineArgs<BT> a) {
  constexpr int R = 4;
  __shared__ double s_cs[32];
  if (threadIdx.x < 32) s_cs[threadIdx.x] = (int)threadIdx.x < a.nv ? a.cs[threadIdx.x] : 0.0;
  __syncthreads();
  const int64_t groups = a.N / R;
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  for (int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x; g < groups; g += stride) {
    const int64_t n0 = g * R;
    double x[R];
    const Pack<double, R> xi = *reinterpret_cast<const Pack<double, R>*>(a.u + n0);
    if constexpr (MAXV == 0) {
#pragma unroll
      for (int r = 0; r < R; ++r) x[r] = a.cu * xi.v[r];
    }
#pragma unroll
    for (int i0 = 0; i0 < MAXV; i0 += kLoadChunk) {
      Pack<BT, R> vv[kLoadChunk];
#pragma unroll
      for (int u = 0; u < kLoadChunk; ++u)
        if (i0 + u < MAXV)
          vv[u] = *reinterpret_cast<const Pack<BT, R>*>(a.V1 + (int64_t)min(i0 + u, a.nv - 1) * a.N + n0);
      __builtin_amdgcn_sched_barrier(0);
      if (i0 == 0) {
#pragma unroll
        for (int r = 0; r < R; ++r) x[r] = a.cu * xi.v[r];
      }
#pragma unroll
      for (int u = 0; u < kLoadChunk; ++u) {
        if (i0 + u >= MAXV) break;
#pragma unroll
        for (int r = 0; r < R; ++r) x[r] = __fma_rn(s_cs[i0 + u], (double)vv[u].v[r], x[r]);
      }
    }
    Pack<double, R> o;
    Pack<BT, R> ov;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      o.v[r] = x[r];
      ov.v[r] = (BT)x[r];
    }
    *reinterpret_cast<Pack<double, R>*>(a.u + n0) = o;
    *reinterpret_cast<Pack<BT, R>*>(a.v0 + n0) = ov;
  }
}

template <typename BT>
void launch_combine(const CombineArgs<BT>& a, unsigned grid, hipStream_t s) {
  switch ((a.nv + 7) / 8) {
    case 0: k_combine<BT, 0><<<grid, kBlock, 0, s>>>(a); break;
    case 1: k_combine<BT, 8><<<grid, kBlock, 0, s>>>(a); break;
    case 2: k_combine<BT, 16><<<grid, kBlock, 0, s>>>(a); break;
    case 3: k_combine<BT, 24><<<grid, kBlock, 0, s>>>(a); break;
    default: k_combine<BT, 32><<<grid, kBlock, 0, s>>>(a); break;
  }
  NC_CHECK_HIP(hipGetLastError());
}

// Column c's five sums from the stored vectors, where the mat-vec does not form them (nc_iop.h)
template <typename BT>
__global__ __launch_bounds__(kIopThreads) void k_krylov_sums(IopArgs p) {
  const int c = p.c, g = blockIdx.x;
  const BT* V = reinterpret_cast<const BT*>(p.V);
  const BT* __restrict__ v = V + (int64_t)c * p.ld;
  const BT* __restrict__ v1 = V + (int64_t)(c > 0 ? c - 1 : 0) * p.ld;
  const double* __restrict__ q = p.q[c & 1];
  const int64_t blk0 = (int64_t)g * p.nblk / p.groups, blk1 = (int64_t)(g + 1) * p.nblk / p.groups;
  double t[kIopSums] = {0.0, 0.0, 0.0, 0.0, 0.0};
  for (int64_t blk = blk0; blk < blk1; ++blk) {
    const int64_t i0 = blk * kIopRows + 2 * threadIdx.x;
    if (i0 >= p.n) continue;
    const Pack<double, 2> qv = *reinterpret_cast<const Pack<double, 2>*>(q + i0);
    const Pack<BT, 2> a = *reinterpret_cast<const Pack<BT, 2>*>(v + i0), b = *reinterpret_cast<const Pack<BT, 2>*>(v1 + i0);
#pragma unroll
    for (int r = 0; r < 2; ++r)
      if (i0 + r < p.n) iop_row_sums(a.v[r], c > 0 ? (double)b.v[r] : 0.0, qv.v[r], t);
  }
  iop_group_sums(t, p.part[c & 1], p.groups, g);
}

// The last column's norm and |A v_m| (avnorm of Expokit), the sink rows of the basis and of
// the state u, and the step's coefficients to the pinned host block the host reads next (one
// workgroup: no copy command, only the synchronisation).
template <typename BT>
__global__ __launch_bounds__(kIopThreads) void k_krylov_last(IopArgs p, int m, const double* u, int64_t ns, int R, double* host) {
  double tot[kIopSums];
  iop_fold<BT>(p, m, tot);
  const IopCoef o = iop_coef(tot, m, 0.0, p.btol);  // the coefficients of V_{m+1} are not used
  const KLayout L = p.L;
  if (threadIdx.x == 0) {
    p.kb[L.H(m, m - 1)] = o.nrm;
    p.kb[L.sc(m)] = o.sc;
    p.kb[L.misc(MISC_AVN)] = o.sc * sqrt(tot[4]);
  }
  const BT* V = reinterpret_cast<const BT*>(p.V);
  for (int t = threadIdx.x; t < (m + 2) * R; t += kIopThreads) {
    const int j = t / R, r = t % R;
    host[L.sinkv(0, 0, R) + t] = j <= m ? (double)V[(int64_t)j * p.ld + ns + r] : u[ns + r];
  }
  __syncthreads();
  for (int t = threadIdx.x; t < L.size(); t += kIopThreads) host[t] = p.kb[t];
}

// Sum of squares of x (N a multiple of 4) in two launches, deterministic.
__global__ __launch_bounds__(kBlock) void k_sumsq(int64_t N, const double* x, double* part) {
  double acc = 0.0;
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  for (int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x; g < N / 4; g += stride) {
    const Pack<double, 4> v = *reinterpret_cast<const Pack<double, 4>*>(x + 4 * g);
#pragma unroll
    for (int r = 0; r < 4; ++r) acc += v.v[r] * v.v[r];
  }
  __shared__ double red[kBlock / 64];
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < kBlock / 64; ++w) s += red[w];
    part[blockIdx.x] = s;
  }
}

// one workgroup; nblocks <= kFinBlock
__global__ __launch_bounds__(kFinBlock) void k_sumsq_fold(unsigned nblocks, const double* part, double* out) {
  __shared__ double wsum[kFinBlock / 64];
  const double v = wave_sum(threadIdx.x < nblocks ? part[threadIdx.x] : 0.0);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < kFinBlock / 64; ++w) s += wsum[w];
    *out = s;
  }
}

// |x|^2 of a padded solver vector into *out (device)
void launch_sumsq(const nc_solver_s* S, const double* x, double* out, hipStream_t s) {
  const unsigned grid = S->red_blocks;
  if (S->Np % 4 || grid > (unsigned)kFinBlock) throw Error(NC_ERR_INTERNAL, "square sum not set up");
  k_sumsq<<<grid, kBlock, 0, s>>>(S->Np, x, S->partials.p);
  k_sumsq_fold<<<1, kFinBlock, 0, s>>>(grid, S->partials.p, out);
  NC_CHECK_HIP(hipGetLastError());
}

// ---- Dormand-Prince 5(4) ------------------------------------------------------------
#define NC_DP_A                                                                  \
  {{0, 0, 0, 0, 0, 0},                                                           \
   {1.0 / 5, 0, 0, 0, 0, 0},                                                     \
   {3.0 / 40, 9.0 / 40, 0, 0, 0, 0},                                             \
   {44.0 / 45, -56.0 / 15, 32.0 / 9, 0, 0, 0},                                   \
   {19372.0 / 6561, -25360.0 / 2187, 64448.0 / 6561, -212.0 / 729, 0, 0},        \
   {9017.0 / 3168, -355.0 / 33, 46732.0 / 5247, 49.0 / 176, -5103.0 / 18656, 0}, \
   {35.0 / 384, 0, 500.0 / 1113, 125.0 / 192, -2187.0 / 6784, 11.0 / 84}}
__constant__ double c_dp_a[7][6] = NC_DP_A;
const double h_dp_a[7][6] = NC_DP_A;  // the same table for the host (mat-vec epilogues)
#undef NC_DP_A
const double h_dp_c[7] = {0, 1.0 / 5, 3.0 / 10, 4.0 / 5, 8.0 / 9, 1.0, 1.0};
// b - b* (5th minus embedded 4th order weights)
#define NC_DP_E {71.0 / 57600, 0, -71.0 / 16695, 71.0 / 1920, -17253.0 / 339200, 22.0 / 525, -1.0 / 40}
__constant__ double c_dp_e[7] = NC_DP_E;
const double h_dp_e[7] = NC_DP_E;  // the same weights for the host (the mat-vec's error epilogue)
#undef NC_DP_E

// Stage j lives in slot j of k, except that with sw = 1 stages 0 and 6 trade slots (an
// accepted step hands k6 = f(y_{n+1}) on as the next k0 by flipping sw, not by copying).
__device__ __host__ inline int rk_slot(int j, int sw) { return (sw && (j == 0 || j == 6)) ? 6 - j : j; }

// Stage input y_i = y + h * sum_{j<i} a_ij k_j ; writes the mat-vec copy, and at the last
// stage (i = 6, whose input is y_{n+1}) also the FP64 value (ytmp), the only stage input
// the error estimate and the accept read. The stage is a template argument so that its
// STAGE loads of k are issued together (a runtime trip count would wait for each before
// the next); two elements per thread.
template <typename VT, int STAGE>
__global__ __launch_bounds__(kBlock) void k_rk_stage(int64_t N, double h, const double* y, const double* k, int sw,
                                                     double* ytmp, VT* vin) {
  constexpr int R = 2;
  const int64_t stride = (int64_t)gridDim.x * kBlock * R;
  for (int64_t n = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * R; n < N; n += stride) {
    // a_61 = 0: the last stage does not read k1
    Pack<double, R> kv[STAGE];
#pragma unroll
    for (int j = 0; j < STAGE; ++j)
      if (!(STAGE == 6 && j == 1)) kv[j] = *reinterpret_cast<const Pack<double, R>*>(k + (int64_t)rk_slot(j, sw) * N + n);
    const Pack<double, R> yv = *reinterpret_cast<const Pack<double, R>*>(y + n);
    Pack<double, R> o;
    Pack<VT, R> ov;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      double acc = 0.0;
#pragma unroll
      for (int j = 0; j < STAGE; ++j)
        if (!(STAGE == 6 && j == 1)) acc += c_dp_a[STAGE][j] * kv[j].v[r];
      o.v[r] = yv.v[r] + h * acc;
      ov.v[r] = (VT)o.v[r];
    }
    if constexpr (STAGE == 6) *reinterpret_cast<Pack<double, R>*>(ytmp + n) = o;
    *reinterpret_cast<Pack<VT, R>*>(vin + n) = ov;
  }
}

template <typename VT>
void launch_rk_stage(int stage, unsigned grid, hipStream_t s, int64_t N, double h, const double* y, const double* k,
                     int sw, double* ytmp, VT* vin) {
  switch (stage) {
    case 1: k_rk_stage<VT, 1><<<grid, kBlock, 0, s>>>(N, h, y, k, sw, ytmp, vin); break;
    case 2: k_rk_stage<VT, 2><<<grid, kBlock, 0, s>>>(N, h, y, k, sw, ytmp, vin); break;
    case 3: k_rk_stage<VT, 3><<<grid, kBlock, 0, s>>>(N, h, y, k, sw, ytmp, vin); break;
    case 4: k_rk_stage<VT, 4><<<grid, kBlock, 0, s>>>(N, h, y, k, sw, ytmp, vin); break;
    case 5: k_rk_stage<VT, 5><<<grid, kBlock, 0, s>>>(N, h, y, k, sw, ytmp, vin); break;
    case 6: k_rk_stage<VT, 6><<<grid, kBlock, 0, s>>>(N, h, y, k, sw, ytmp, vin); break;
    default: throw Error(NC_ERR_INTERNAL, "bad RK stage");
  }
}

// Error norm sum_n (h*sum_j e_j k_j / (atol + rtol*max(|y|,|ynew|)))^2 with ynew = ytmp;
// one partial sum per block (folded on the host, which reads them back anyway). With
// R > 0, block 0 also gathers the sink rows ns..ns+R-1 of ynew, k0 and k6 behind the
// partials, so that one copy brings back everything the step controller needs.
__global__ __launch_bounds__(kBlock) void k_rk_err(int64_t N, double h, double atol, double rtol, const double* y,
                                                   const double* ynew, const double* k, int sw, int64_t ns, int R,
                                                   double* partials) {
  if (blockIdx.x == 0 && (int)threadIdx.x < R) {
    double* ex = partials + gridDim.x;
    const int r = threadIdx.x;
    ex[r] = ynew[ns + r];
    ex[R + r] = k[(int64_t)rk_slot(0, sw) * N + ns + r];
    ex[2 * R + r] = k[(int64_t)rk_slot(6, sw) * N + ns + r];
  }
  double acc = 0.0;
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  for (int64_t n = (int64_t)blockIdx.x * kBlock + threadIdx.x; n < N; n += stride) {
    double e = 0.0;
    // e_1 = 0 in Dormand-Prince 5(4): k1 is not read
#pragma unroll
    for (int j = 0; j < 7; ++j)
      if (j != 1) e += c_dp_e[j] * k[(int64_t)rk_slot(j, sw) * N + n];
    e *= h;
    const double sc = atol + rtol * fmax(fabs(y[n]), fabs(ynew[n]));
    const double r = e / sc;
    acc += r * r;
  }
  __shared__ double red[kBlock / 64];
  double v = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < kBlock / 64; ++w) s += red[w];
    partials[blockIdx.x] = s;
  }
}

// Cubic Hermite dense output on an accepted step, written over y:
// y(t + theta h) from y, y1 = y(t + h) and the derivatives k0 = f(y), k6 = f(y1).
__global__ __launch_bounds__(kBlock) void k_rk_hermite(int64_t N, double theta, double h, double* y, const double* y1,
                                                       const double* k0, const double* k6) {
  const double t2 = theta * theta, t3 = t2 * theta;
  const double a0 = 2 * t3 - 3 * t2 + 1, b0 = (t3 - 2 * t2 + theta) * h;
  const double a1 = -2 * t3 + 3 * t2, b1 = (t3 - t2) * h;
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  for (int64_t n = (int64_t)blockIdx.x * kBlock + threadIdx.x; n < N; n += stride)
    y[n] = a0 * y[n] + b0 * k0[n] + a1 * y1[n] + b1 * k6[n];
}

__global__ void k_copy_d(const double* in, double* out, int64_t N) {
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  for (int64_t n = (int64_t)blockIdx.x * kBlock + threadIdx.x; n < N; n += stride) out[n] = in[n];
}

template <typename VT>
__global__ void k_to_vt(const double* in, VT* out, int64_t N) {
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  for (int64_t n = (int64_t)blockIdx.x * kBlock + threadIdx.x; n < N; n += stride) out[n] = (VT)in[n];
}

double round_step(double x) {
  // Expokit rounds step sizes to 2 significant digits
  if (!(x > 0.0)) return x;
  const double s = std::pow(10.0, std::floor(std::log10(x)) - 1.0);
  return std::ceil(x / s) * s;
}

}  // namespace

void krylov_sums(const IopArgs& p, bool fp32, hipStream_t s) {
  if (fp32)
    k_krylov_sums<float><<<(unsigned)p.groups, kIopThreads, 0, s>>>(p);
  else
    k_krylov_sums<double><<<(unsigned)p.groups, kIopThreads, 0, s>>>(p);
  NC_CHECK_HIP(hipGetLastError());
}

void solver_reduce_setup(nc_solver_s* S) {
  // Grid of the vector passes: 1024 blocks of 256 threads for a Krylov basis stored in
  // FP32 and 512 otherwise (on the 1024^2 toggle-switch solve, 256 to 4096 blocks are
  // within 1% of each other since the passes issue their basis loads in batches)
  const unsigned vb = (S->method == NC_METHOD_KRYLOV && S->vs == 4) ? 1024u : kVecBlocks;
  S->red_blocks = std::min<unsigned>(vb, grid_for(S->Np / 4, kBlock));
  // Krylov columns: blocks of kIopRows state rows with the sink rows added by the fold; the
  // sensitivity system sums every padded row
  S->kn = S->SA ? S->Np : S->A->n;
  S->kblk = std::max<int64_t>((S->kn + kIopRows - 1) / kIopRows, 1);
  S->kgroups = iop_groups(S->kblk, !S->SA && krylov_small_shape(S->A));
  S->partials.reserve(std::max<size_t>(S->red_blocks, (size_t)2 * kIopSums * S->kgroups));
  if (!S->hpart) {
    // partials (up to kMaxRedBlocks, or one per row workgroup and sink row of the mat-vec's
    // error epilogue) and the RK step's 3 R gathered sink values, then the carried sinks of
    // u and the step's three sink sets (4 R) behind them
    S->hpart_cap = std::max<int64_t>(kMaxRedBlocks, matvec_err_parts(S->A));
    S->hpart = static_cast<double*>(pinned_alloc(sizeof(double) * (S->hpart_cap + 7 * kMaxReactions)));
    NC_CHECK_HIP(hipHostGetDevicePointer(reinterpret_cast<void**>(&S->hpart_dev), S->hpart, 0));
  }
}

// The right-hand-side operator: the FSP generator, or the block sensitivity operator.
static void op_apply(nc_solver_s* S, double t, const void* v, double* out) {
  if (S->SA)
    sens_matvec_launch(S->SA, t, v, S->Npb, out, S->Npb, S->s);
  else
    matvec_launch(S->A, t, v, out, false, S->s, true);
}

// Device (padded, block stride Npb) <-> host (contiguous, block stride Nb) copies.
static void copy_from_host(nc_solver_s* S, double* dev, const double* host) {
  if (S->blocks == 1)
    NC_CHECK_HIP(hipMemcpyAsync(dev, host, sizeof(double) * S->N, hipMemcpyHostToDevice, S->s));
  else
    NC_CHECK_HIP(hipMemcpy2DAsync(dev, sizeof(double) * S->Npb, host, sizeof(double) * S->Nb, sizeof(double) * S->Nb,
                                  S->blocks, hipMemcpyHostToDevice, S->s));
}
static void copy_to_host(nc_solver_s* S, double* host, const double* dev) {
  if (S->blocks == 1)
    NC_CHECK_HIP(hipMemcpyAsync(host, dev, sizeof(double) * S->N, hipMemcpyDeviceToHost, S->s));
  else
    NC_CHECK_HIP(hipMemcpy2DAsync(host, sizeof(double) * S->Nb, dev, sizeof(double) * S->Npb, sizeof(double) * S->Nb,
                                  S->blocks, hipMemcpyDeviceToHost, S->s));
  NC_CHECK_HIP(hipStreamSynchronize(S->s));
}

// ---- Krylov expv ---------------------------------------------------------------------
// The device work of one Krylov process: columns 0 .. m (nc_iop.h), each one launch where
// the generator's mat-vec has the column form, else V_c, q_c = A V_c and the sums by
// themselves; then the last column's norms and the read-back. Its launches and arguments
// are identical for every Krylov step, so it is captured once into a HIP graph and replayed.
template <typename BT>
static void krylov_process(nc_solver_s* S) {
  IopArgs p{};
  p.n = S->kn;
  p.tail1 = S->SA ? S->kn : S->A->n_rows;
  p.ld = S->Np;
  p.nblk = S->kblk;
  p.groups = S->kgroups;
  p.V = S->V.p;
  p.kb = S->kbuf.p;
  p.L = KLayout{S->m};
  p.btol = krylov_breakdown_tol(S);
  for (int h = 0; h < 2; ++h) {
    p.q[h] = S->q.p + (size_t)h * S->Np;
    p.part[h] = S->partials.p + (size_t)h * kIopSums * S->kgroups;
  }
  const bool fused = !S->SA && matvec_krylov_fusable(S->A);
  for (int c = 0; c <= S->m; ++c) {
    p.c = c;
    if (fused) {
      matvec_launch_krylov(S->A, S->s, p);
      continue;
    }
    if (c > 0) krylov_form(p, S->vs == 4, S->s);
    op_apply(S, 0.0, S->V.p + (size_t)c * S->Np * S->vs, p.q[c & 1]);
    krylov_sums(p, S->vs == 4, S->s);
  }
  k_krylov_last<BT><<<1, kIopThreads, 0, S->s>>>(p, S->m, S->u.p, S->A->n, S->A->nr, S->hbuf_dev);
  NC_CHECK_HIP(hipGetLastError());
}

static void arnoldi_launch(nc_solver_s* S) {
  if (S->A->precision == NC_FP32)
    krylov_process<float>(S);
  else
    krylov_process<double>(S);
}

static void arnoldi_run(nc_solver_s* S) {
  const bool use_graph = !S->A->timing && S->opts.no_graphs == 0;
  if (!use_graph) {
    arnoldi_launch(S);
    return;
  }
  if (S->arnoldi_exec && S->arnoldi_gen != S->A->launch_gen) {
    // the matrix's launch shape changed since the capture (autotune, set_rows_per_thread)
    NC_CHECK_HIP(hipStreamSynchronize(S->s));
    (void)hipGraphExecDestroy(S->arnoldi_exec);
    (void)hipGraphDestroy(S->arnoldi_graph);
    S->arnoldi_exec = nullptr;
    S->arnoldi_graph = nullptr;
  }
  if (!S->arnoldi_exec) {
    hipGraph_t g = nullptr;
    NC_CHECK_HIP(hipStreamBeginCapture(S->s, hipStreamCaptureModeThreadLocal));
    try {
      arnoldi_launch(S);
    } catch (...) {
      (void)hipStreamEndCapture(S->s, &g);
      if (g) (void)hipGraphDestroy(g);
      (void)hipGetLastError();
      throw;
    }
    NC_CHECK_HIP(hipStreamEndCapture(S->s, &g));
    NC_CHECK_HIP(hipGraphInstantiate(&S->arnoldi_exec, g, nullptr, nullptr, 0));
    S->arnoldi_graph = g;
    S->arnoldi_gen = S->A->launch_gen;
  }
  NC_CHECK_HIP(hipGraphLaunch(S->arnoldi_exec, S->s));
}

// Kernel timing of one solver's advance. The generator may be shared by several solvers
// (the flag and the event pool live on the matrix), so the solver's own time_kernels
// setting applies only while it advances, and the timings recorded meanwhile are
// credited to its own statistics.
struct TimingScope {
  nc_solver_s* S;
  bool was, was_plain;
  double ms0;
  int64_t n0;
  explicit TimingScope(nc_solver_s* s_) : S(s_), was(s_->A->timing), was_plain(s_->A->timing_plain) {
    S->A->timing = S->opts.time_kernels != 0;
    S->A->timing_plain = S->opts.time_kernels == 2;
    ms0 = S->A->timed_ms;
    n0 = S->A->timed_count;
  }
  ~TimingScope() {
    try {
      matvec_harvest_timing(S->A);
    } catch (...) {
    }
    S->st.matvec_ms += S->A->timed_ms - ms0;
    S->st.matvecs_timed += S->A->timed_count - n0;
    S->A->timing = was;
    S->A->timing_plain = was_plain;
  }
};

// Sink-mass budget of the adaptive solve (fspsolve.jl:145-148): g(t) = sum(sinks) - c t.
static double budget(const EventSpec* ev, double sink_sum, double t) {
  return sink_sum - ev->fsptol * t / ev->tend;
}

void krylov_advance(nc_solver_s* S, double t_target, EventSpec* ev, bool one_step) {
  TimingScope timing_scope(S);
  nc_matrix_s* A = S->A;
  const int m = S->m;
  const int64_t N = S->Np;
  const KLayout L{m};
  const int R = A->nr;
  hipStream_t s = S->s;
  const bool fp32 = A->precision == NC_FP32;
  const double tol = krylov_step_tol(S);
  const double btol = krylov_breakdown_tol(S), gamma = 0.9, delta = 1.2;
  const int mxrej = 10;
  if (!S->started) {
    // first step size from the norm estimate (Expokit)
    S->anorm = std::max(S->SA ? S->SA->norm1 : A->norm1, 1e-300);
    const double fact = std::pow((m + 1) / std::exp(1.0), m + 1) * std::sqrt(2.0 * M_PI * (m + 1));
    const double b = std::max(S->beta, 1e-300);
    S->t_new = round_step((1.0 / S->anorm) * std::pow((fact * tol) / (4.0 * b * S->anorm), 1.0 / m));
    S->started = true;
  }
  const double t_eps = 1e-13 * std::max(1.0, std::fabs(t_target));
  // the combination that ends a step: u <- pend_cu u + sum_i pend[i] V_{i+1}. A small space's
  // next process takes it with it; else, and after the last step here, it is a launch.
  const bool small = krylov_small_fits(S);
  bool pending = false;
  std::vector<double> pend;
  double pend_cu = 0.0;
  auto combine = [&](auto* v0) {
    CombineArgs<std::remove_pointer_t<decltype(v0)>> a{};
    a.N = N;
    a.nv = (int)pend.size();
    a.V1 = v0 + N;
    a.v0 = v0;
    a.u = S->u.p;
    a.cu = pend_cu;
    std::copy(pend.begin(), pend.end(), a.cs);
    launch_combine(a, S->red_blocks, s);
  };
  auto end_step = [&] {
    if (fp32)
      combine(reinterpret_cast<float*>(S->V.p));
    else
      combine(reinterpret_cast<double*>(S->V.p));
    pending = false;
  };
  while (S->t < t_target - t_eps) {
    if (S->opts.max_steps && S->st.steps >= S->opts.max_steps) {
      if (pending) end_step();
      throw Error(NC_ERR_NUMERIC, "Krylov integrator exceeded max_steps");
    }
    if (S->beta == 0.0) {  // zero vector stays zero
      S->t = t_target;
      break;
    }
    double t_step = std::min(t_target - S->t, S->t_new);
    if (small) {
      krylov_small_launch(S, pending ? (int)pend.size() : -1, pend_cu, pend.data());
      pending = false;
    } else {
      arnoldi_run(S);
    }
    S->st.matvecs += m + 1;
    NC_CHECK_HIP(hipStreamSynchronize(s));  // the process ends by writing hbuf
    S->st.host_syncs++;
    matvec_harvest_timing(A);
    const double* hb = S->hbuf;
    const double beta = hb[L.misc(MISC_BETA)];  // |V_0| as stored
    // happy breakdown detection
    int mb = m, k1 = 2;
    for (int j = 0; j < m; ++j) {
      if (hb[L.H(j + 1, j)] < btol) {
        mb = j + 1;
        k1 = 0;
        t_step = t_target - S->t;
        break;
      }
    }
    const double avnorm = hb[L.misc(MISC_AVN)];
    const double floor_err = krylov_floor(S) * beta;
    auto allowed = [&](double tau) { return std::max(tau * tol, floor_err); };  // error of a step tau
    const int mxf = mb + k1;  // size of the exponentiated matrix
    std::vector<double> F(mxf);  // first column of exp(tau H), H tridiagonal
    auto exp_tau = [&](double tau, std::vector<double>& out) {
      double lo[34], di[34], up[34];  // m <= 31
      auto h = [&](int i, int j) { return i < m + 1 && i < mb + 1 && j < mb ? tau * hb[L.H(i, j)] : 0.0; };
      for (int i = 0; i < mxf; ++i) {
        lo[i] = i > 0 ? (k1 != 0 && i == m + 1 ? tau : h(i, i - 1)) : 0.0;
        di[i] = h(i, i);
        up[i] = i + 1 < mxf ? h(i, i + 1) : 0.0;
      }
      expm_first_column(mxf, lo, di, up, out.data());
    };
    double err_loc = btol, xm = 1.0 / m;
    for (int ireject = 0;; ++ireject) {
      exp_tau(t_step, F);
      if (k1 == 0) {
        err_loc = btol;
        break;
      }
      const double phi1 = std::fabs(beta * F[m]);
      const double phi2 = std::fabs(beta * F[m + 1] * avnorm);
      if (phi1 > 10.0 * phi2) {
        err_loc = phi2;
        xm = 1.0 / m;
      } else if (phi1 > phi2) {
        err_loc = (phi1 * phi2) / (phi1 - phi2);
        xm = 1.0 / m;
      } else {
        err_loc = phi1;
        xm = 1.0 / (m - 1);
      }
      if (err_loc <= delta * allowed(t_step)) break;
      if (ireject == mxrej) throw Error(NC_ERR_NUMERIC, "Krylov step rejected too many times; tolerance too tight");
      // the step that the estimate's order asks for; from the second rejection on at most half:
      // near a stationary state of a stiff generator the estimate falls like tau, not
      // tau^m, and shrinking by a tenth each time used up the rejections (an exponential
      // costs 6 us, a step a hundred and more)
      const double fac = gamma * std::pow(allowed(t_step) / err_loc, xm);
      t_step = round_step(t_step * (ireject > 0 ? std::min(fac, 0.5) : fac));
      S->st.rejected++;
    }
    const int mx = mb + std::max(0, k1 - 1);
    // sink mass of w(tau) = beta V exp(tau H) e1, with the exact state for the first term
    auto sink_sum = [&](const std::vector<double>& Fm) {
      double tot = 0.0;
      for (int r = 0; r < R; ++r) {
        double v = Fm[0] * hb[L.sinkv(m + 1, r, R)];
        for (int i = 1; i < mx; ++i) v += beta * Fm[i] * hb[L.sc(i)] * hb[L.sinkv(i, r, R)];
        tot += v;
      }
      return tot;
    };
    bool fire = false;
    double sinks0 = 0.0;  // sink mass of the state at the start of the step
    for (int r = 0; r < R; ++r) sinks0 += hb[L.sinkv(m + 1, r, R)];
    if (ev && R > 0 && budget(ev, sinks0, S->t) <= 0.0 && budget(ev, sink_sum(F), S->t + t_step) > 0.0) {
      // the budget is crossed inside this step: locate the crossing on the exact Krylov
      // solution w(tau) by bisection (the reference's callback root-finds to eps)
      std::vector<double> Ft(mxf);
      double lo = 0.0, hi = t_step;
      for (int it = 0; it < 200 && hi - lo > 4.0 * std::numeric_limits<double>::epsilon() * std::max(1.0, S->t + hi); ++it) {
        const double mid = 0.5 * (lo + hi);
        exp_tau(mid, Ft);
        if (budget(ev, sink_sum(Ft), S->t + mid) > 0.0)
          hi = mid;
        else
          lo = mid;
      }
      t_step = hi;
      exp_tau(t_step, F);
      fire = true;
    }
    S->t += t_step;
    const bool hit = !fire && S->t >= t_target - t_eps;
    if (hit) S->t = t_target;
    // w_new = F_0 w + sum_{i>=1} beta F_i sc_i V_i
    pend_cu = F[0];
    pend.resize(mx - 1);
    for (int i = 1; i < mx; ++i) pend[i - 1] = (beta * F[i]) * hb[L.sc(i)];
    pending = true;
    if (!small || fire || hit || one_step) end_step();
    S->st.steps++;
    err_loc = std::max(err_loc, 1e-300);
    S->st.error_estimate += std::max(err_loc, S->anorm * 2.220446049250313e-16);
    if (k1 != 0 && !fire) S->t_new = round_step(gamma * t_step * std::pow(allowed(t_step) / err_loc, xm));
    if (fire) {
      ev->fired = true;
      break;
    }
    if (hit || one_step) break;
  }
}

// ---- Dormand-Prince 5(4) ---------------------------------------------------------------
void rk_advance(nc_solver_s* S, double t_target, EventSpec* ev, bool one_step) {
  TimingScope timing_scope(S);
  nc_matrix_s* A = S->A;
  const int64_t N = S->Np;  // padded: rows beyond the true length stay zero
  const int R = A->nr;
  const int64_t ns = A->n;
  hipStream_t s = S->s;
  const bool fp32 = A->precision == NC_FP32;
  const double rtol = S->opts.rtol, atol = S->opts.atol;
  const unsigned g = std::min<unsigned>(4096, grid_for(N, kBlock));  // elementwise stage kernels
  const unsigned g2 = std::min<unsigned>(4096, grid_for(N / 2, kBlock));  // two elements per thread
  double* k = S->k.p;
  auto kp = [&](int j) { return k + (int64_t)rk_slot(j, S->ksw) * N; };
  auto to_vin = [&](const double* src) {
    if (fp32)
      k_to_vt<float><<<g, kBlock, 0, s>>>(src, reinterpret_cast<float*>(S->rkv.p), N);
    else
      k_to_vt<double><<<g, kBlock, 0, s>>>(src, reinterpret_cast<double*>(S->rkv.p), N);
  };
  // The mat-vec that forms k_s also forms stage s + 1's input in its epilogue (the stored
  // generator at 2 rows per thread, and the sensitivity operator up to 16 blocks; the stage
  // pass runs on its own for stage 1 and for the computed modes);
  // the stage inputs alternate between two buffers, since a mat-vec gathers from its input
  // while its epilogue writes the next one.
  const bool fuse = S->rkv2.p && (S->SA ? sens_rk_fusable(S->SA) : matvec_rk_fusable(A));
  // the error pass in the epilogue of the step's last mat-vec (plain generator)
  const int64_t err_parts = matvec_err_parts(A);
  const bool efuse = fuse && !S->SA && err_parts <= S->hpart_cap;
  const int Rg = (ev && R > 0) ? R : 0;
  auto stages = [&](double h) {
    if (!S->SA) {
      double ts[5];
      for (int j = 0; j < 5; ++j) ts[j] = S->t + h_dp_c[j + 1] * h;  // the last two stages share theirs
      matrix_prepare_times(A, 5, ts);
    }
    unsigned char* cur = S->rkv.p;
    unsigned char* nxt = S->rkv2.p;
    for (int stage = 1; stage < 7; ++stage) {
      if (stage == 1 || !fuse) {
        if (fp32)
          launch_rk_stage<float>(stage, g2, s, N, h, S->u.p, k, S->ksw, S->ytmp.p, reinterpret_cast<float*>(cur));
        else
          launch_rk_stage<double>(stage, g2, s, N, h, S->u.p, k, S->ksw, S->ytmp.p, reinterpret_cast<double*>(cur));
        NC_CHECK_HIP(hipGetLastError());
      }
      const double ts = S->t + h_dp_c[stage] * h;
      if (fuse && stage < 6) {
        const int next = stage + 1;
        RkEpilogue e{};
        for (int j = 0; j < stage; ++j) {
          if (next == 6 && j == 1) continue;  // a_61 = 0: the last stage does not read k1
          e.mask |= 1 << j;
          e.k[j] = kp(j);
          e.a[j] = h_dp_a[next][j];
        }
        e.k[0] = kp(0);
        e.a_new = h_dp_a[next][stage];
        e.h = h;
        e.u = S->u.p;
        e.ytmp = next == 6 ? S->ytmp.p : nullptr;
        e.vin = nxt;
        if (S->SA)
          sens_matvec_launch(S->SA, ts, cur, S->Npb, kp(stage), S->Npb, s, &e);
        else
          matvec_launch_rk(A, ts, cur, kp(stage), s, e);
        std::swap(cur, nxt);
      } else if (efuse && stage == 6) {
        RkErrEpilogue e{};
        for (int j = 0; j < 6; ++j) e.k[j] = kp(j);
        for (int j = 0; j < 7; ++j) e.e[j] = h_dp_e[j];
        e.h = h;
        e.atol = atol;
        e.rtol = rtol;
        e.u = S->u.p;
        e.ynew = S->ytmp.p;
        e.part = S->hpart_dev;
        e.ex = S->hpart_dev + err_parts;
        e.n_ex = Rg;
        matvec_launch_err(A, ts, cur, kp(stage), s, e);
      } else {
        op_apply(S, ts, cur, kp(stage));
      }
      S->st.matvecs++;
    }
  };
  if (!S->fsal_valid) {
    to_vin(S->u.p);
    op_apply(S, S->t, S->rkv.p, kp(0));
    S->st.matvecs++;
    S->fsal_valid = true;
  }
  if (S->h <= 0.0) {
    // initial step (Hairer, Norsett & Wanner, Solving ODEs I, II.4): based on |f(t0,y0)|
    double* fn2 = static_cast<double*>(host_stage(5));
    launch_sumsq(S, kp(0), S->kbuf.p, s);
    NC_CHECK_HIP(hipMemcpyAsync(fn2, S->kbuf.p, sizeof(double), hipMemcpyDeviceToHost, s));
    NC_CHECK_HIP(hipStreamSynchronize(s));
    const double fnorm = std::sqrt(*fn2);
    S->h = S->opts.h0 > 0 ? S->opts.h0 : (fnorm > 0 ? 0.01 / fnorm : 1e-3);
    S->h = std::max(S->h, 1e-12);
  }
  // pinned: sinks of u, y_{n+1}, k0, k6 (R each), behind the readback region
  double* hs = S->hpart + S->hpart_cap + 3 * kMaxReactions;
  if (ev && R > 0) {
    NC_CHECK_HIP(hipMemcpyAsync(hs, S->u.p + ns, sizeof(double) * R, hipMemcpyDeviceToHost, s));
    NC_CHECK_HIP(hipStreamSynchronize(s));
  }
  const double t_eps = 1e-13 * std::max(1.0, std::fabs(t_target));
  double errsum = 0.0;
  while (S->t < t_target - t_eps) {
    if (S->opts.max_steps && S->st.steps + S->st.rejected >= S->opts.max_steps)
      throw Error(NC_ERR_NUMERIC, "RK integrator exceeded max_steps");
    double h = std::min(S->h, t_target - S->t);
    const bool clamped = h < S->h;
    stages(h);
    // after stage 6 the stage input is y + h*sum b_j k_j (row 7 of A): ytmp = y_{n+1}
    // the partials and the gathered sinks go straight to the pinned host block: the step's
    // read-back needs no copy launch, only the synchronisation
    if (!efuse) {
      k_rk_err<<<S->red_blocks, kBlock, 0, s>>>(N, h, atol, rtol, S->u.p, S->ytmp.p, k, S->ksw, ns, Rg, S->hpart_dev);
      NC_CHECK_HIP(hipGetLastError());
    }
    NC_CHECK_HIP(hipStreamSynchronize(s));
    const int64_t np = efuse ? err_parts : (int64_t)S->red_blocks;
    for (int r = 0; r < Rg; ++r) {  // sinks of y_{n+1}, k0 and k6 behind the partials
      hs[R + r] = S->hpart[np + r];
      hs[2 * R + r] = S->hpart[np + R + r];
      hs[3 * R + r] = S->hpart[np + 2 * R + r];
    }
    // four running sums (the epilogue's partials number one per row workgroup), then added
    double es[4] = {0.0, 0.0, 0.0, 0.0};
    int64_t b = 0;
    for (; b + 4 <= np; b += 4)
      for (int q = 0; q < 4; ++q) es[q] += S->hpart[b + q];
    for (; b < np; ++b) es[0] += S->hpart[b];
    errsum = (es[0] + es[1]) + (es[2] + es[3]);
    S->st.host_syncs++;
    matvec_harvest_timing(A);
    const double err = std::sqrt(errsum / (double)S->N);
    if (!std::isfinite(err)) throw Error(NC_ERR_NUMERIC, "non-finite RK error estimate");
    double fac = err > 0 ? 0.9 * std::pow(err, -0.2) : 5.0;
    if (err <= 1.0) {
      if (ev && R > 0) {
        double s0 = 0, s1 = 0, d0 = 0, d1 = 0;
        for (int r = 0; r < R; ++r) s0 += hs[r], s1 += hs[R + r], d0 += hs[2 * R + r], d1 += hs[3 * R + r];
        const double c = ev->fsptol / ev->tend;
        const double g0 = s0 - c * S->t, g1 = s1 - c * (S->t + h);
        if (g0 <= 0.0 && g1 > 0.0) {
          // cubic Hermite dense output of g on the step (derivatives from the FSAL stages),
          // crossing located by bisection; the event state is the same Hermite
          // interpolant of the whole state, so its sink mass is the root-found one
          const double dg0 = (d0 - c) * h, dg1 = (d1 - c) * h;
          auto herm = [&](double th) {
            const double t2 = th * th, t3 = t2 * th;
            return (2 * t3 - 3 * t2 + 1) * g0 + (t3 - 2 * t2 + th) * dg0 + (-2 * t3 + 3 * t2) * g1 + (t3 - t2) * dg1;
          };
          double lo = 0.0, hi = 1.0;
          for (int it = 0; it < 200 && (hi - lo) * h > 4.0 * std::numeric_limits<double>::epsilon() * std::max(1.0, S->t + h); ++it) {
            const double mid = 0.5 * (lo + hi);
            if (herm(mid) > 0.0)
              hi = mid;
            else
              lo = mid;
          }
          k_rk_hermite<<<g, kBlock, 0, s>>>(N, hi, h, S->u.p, S->ytmp.p, kp(0), kp(6));
          NC_CHECK_HIP(hipGetLastError());
          S->t += hi * h;
          S->st.steps++;
          S->fsal_valid = false;  // k0 no longer matches u
          ev->fired = true;
          break;
        }
      }
      // accept: u <- ytmp, k0 <- k6 (FSAL), by exchanging buffers
      std::swap(S->u, S->ytmp);
      S->ksw ^= 1;
      S->t += h;
      S->st.steps++;
      if (S->t > t_target - t_eps) S->t = t_target;
      for (int r = 0; ev && r < R; ++r) hs[r] = hs[R + r];
      fac = std::min(5.0, std::max(0.2, fac));
      if (!clamped || fac < 1.0) S->h = h * fac;
      if (one_step) break;
    } else {
      S->st.rejected++;
      S->h = h * std::max(0.2, fac);
    }
    if (S->h < 1e-14 * std::max(1.0, std::fabs(S->t))) throw Error(NC_ERR_NUMERIC, "RK step size underflow");
  }
}

}  // namespace nc

using namespace nc;

namespace {

static nc_solver_s* solver_create_impl(nc_matrix_s* A, const nc_solve_opts* opts, nc_sensmatrix_s* SA = nullptr) {
  {
    NC_REQUIRE(A, NC_ERR_ARG, "null matrix");
    auto S = new nc_solver_s();
    try {
      if (opts)
        S->opts = *opts;
      else
        nc_solve_opts_default(&S->opts);
      if (S->opts.krylov_m <= 0) S->opts.krylov_m = 30;
      if (S->opts.krylov_tol <= 0) S->opts.krylov_tol = 1e-12;
      if (S->opts.rtol <= 0) S->opts.rtol = 1e-8;
      if (S->opts.atol <= 0) S->opts.atol = 1e-14;
      NC_REQUIRE(S->opts.krylov_m >= 2 && S->opts.krylov_m <= 31, NC_ERR_ARG, "krylov_m must be in 2..31");
      S->A = A;
      S->s = A->stream.s;
      S->SA = SA;
      S->blocks = SA ? SA->P + 1 : 1;
      S->Nb = A->n_rows;
      S->Npb = (S->Nb + 1023) / 1024 * 1024;
      S->N = S->blocks * S->Nb;
      S->vs = A->vsize;
      const bool tv = !A->tv_r.empty();
      int method = S->opts.method;
      if (method == NC_METHOD_AUTO) method = tv ? NC_METHOD_RK45 : NC_METHOD_KRYLOV;
      NC_REQUIRE(!(method == NC_METHOD_KRYLOV && tv), NC_ERR_ARG,
                 "the Krylov integrator needs a time-invariant generator; use NC_METHOD_RK45");
      S->method = method;
      S->m = S->opts.krylov_m;
      S->Np = S->blocks * S->Npb;
      S->u.alloc(S->Np);
      NC_CHECK_HIP(hipMemsetAsync(S->u.p, 0, sizeof(double) * S->Np, S->s));
      const KLayout L{S->m};
      const int ksize = L.size_with_sinks(A->nr);
      S->kbuf.alloc(ksize);
      NC_CHECK_HIP(hipMemsetAsync(S->kbuf.p, 0, sizeof(double) * ksize, S->s));
      S->hbuf = static_cast<double*>(pinned_alloc(sizeof(double) * ksize));
      std::memset(S->hbuf, 0, sizeof(double) * ksize);
      NC_CHECK_HIP(hipHostGetDevicePointer(reinterpret_cast<void**>(&S->hbuf_dev), S->hbuf, 0));
      solver_reduce_setup(S);
      if (method == NC_METHOD_KRYLOV) {
        S->V.alloc((size_t)(S->m + 1) * S->Np * S->vs);
        S->q.alloc(2 * S->Np);  // columns alternate: a column gathers the last q while it writes its own
        NC_CHECK_HIP(hipMemsetAsync(S->V.p, 0, (size_t)(S->m + 1) * S->Np * S->vs, S->s));
        NC_CHECK_HIP(hipMemsetAsync(S->q.p, 0, sizeof(double) * 2 * S->Np, S->s));
      } else {
        S->rkv.alloc(S->Np * S->vs);
        S->k.alloc((size_t)7 * S->Np);
        S->ytmp.alloc(S->Np);
        NC_CHECK_HIP(hipMemsetAsync(S->rkv.p, 0, S->Np * S->vs, S->s));
        S->rkv2.alloc(S->Np * S->vs);
        NC_CHECK_HIP(hipMemsetAsync(S->rkv2.p, 0, S->Np * S->vs, S->s));
        NC_CHECK_HIP(hipMemsetAsync(S->k.p, 0, sizeof(double) * 7 * S->Np, S->s));
        NC_CHECK_HIP(hipMemsetAsync(S->ytmp.p, 0, sizeof(double) * S->Np, S->s));
      }
      NC_CHECK_HIP(hipStreamSynchronize(S->s));
    } catch (...) {
      delete S;
      throw;
    }
    return S;
  }
}

// Re-initialise integrator state from the device copy u0 (time t0, norm beta0).
static void solver_reinit(nc_solver_s* S) {
  {
    const unsigned gc = std::min<unsigned>(4096, grid_for(S->Np, kBlock));
    k_copy_d<<<gc, kBlock, 0, S->s>>>(S->u0.p, S->u.p, S->Np);
    S->t = S->t0;
    S->have_state = true;
    S->fsal_valid = false;
    S->started = false;
    S->h = 0.0;
    S->st = nc_solve_stats{};
    if (S->method == NC_METHOD_KRYLOV) {
      S->beta = S->beta0;
      const unsigned g = grid_for(S->Np, kBlock);
      if (S->A->precision == NC_FP32)
        k_to_vt<float><<<std::min(g, 4096u), kBlock, 0, S->s>>>(S->u.p, reinterpret_cast<float*>(S->V.p), S->Np);
      else
        k_to_vt<double><<<std::min(g, 4096u), kBlock, 0, S->s>>>(S->u.p, reinterpret_cast<double*>(S->V.p), S->Np);
    }
    NC_CHECK_HIP(hipGetLastError());
  }
}

static void solver_set_state_impl(nc_solver_s* S, double t0, const double* u) {
  NC_REQUIRE(S && u, NC_ERR_ARG, "null argument");
  if (!S->u0.p) {
    S->u0.alloc(S->Np);
    NC_CHECK_HIP(hipMemsetAsync(S->u0.p, 0, sizeof(double) * S->Np, S->s));
  }
  copy_from_host(S, S->u0.p, u);
  double b2 = 0.0;
  for (int64_t i = 0; i < S->N; ++i) b2 += u[i] * u[i];
  S->beta0 = std::sqrt(b2);
  S->t0 = t0;
  solver_reinit(S);
  NC_CHECK_HIP(hipStreamSynchronize(S->s));
}

static void solver_run_impl(nc_solver_s* S, int32_t n_out, const double* t_out) {
  {
    NC_REQUIRE(S && S->have_state, NC_ERR_ARG, "solver has no state; call nc_solver_set_state first");
    NC_REQUIRE(n_out >= 0 && (n_out == 0 || t_out), NC_ERR_ARG, "bad output times");
    for (int k = 0; k < n_out; ++k) {
      NC_REQUIRE(std::isfinite(t_out[k]) && t_out[k] >= S->t - 1e-12 * std::max(1.0, std::fabs(S->t)), NC_ERR_ARG,
                 "output times must be finite and not before the current time");
      NC_REQUIRE(k == 0 || t_out[k] >= t_out[k - 1], NC_ERR_ARG, "output times must be ascending");
    }
    if ((size_t)n_out * S->Np > S->snaps.n) S->snaps.alloc((size_t)std::max(n_out, 1) * S->Np);
    S->n_snaps = n_out;
    const unsigned g = std::min<unsigned>(4096, grid_for(S->Np, kBlock));
    for (int k = 0; k < n_out; ++k) {
      if (S->method == NC_METHOD_KRYLOV)
        krylov_advance(S, t_out[k]);
      else
        rk_advance(S, t_out[k]);
      k_copy_d<<<g, kBlock, 0, S->s>>>(S->u.p, S->snaps.p + (size_t)k * S->Np, S->Np);
      NC_CHECK_HIP(hipGetLastError());
    }
    NC_CHECK_HIP(hipStreamSynchronize(S->s));
    matvec_harvest_timing(S->A);
  }
}

}  // namespace

extern "C" {

int nc_solve_opts_default(nc_solve_opts* o) {
  if (!o) return NC_ERR_ARG;
  std::memset(o, 0, sizeof(*o));
  o->method = NC_METHOD_AUTO;
  o->krylov_m = 30;
  o->krylov_tol = 1e-12;
  o->rtol = 1e-8;
  o->atol = 1e-14;
  return NC_OK;
}

int nc_solver_create(nc_matrix A, const nc_solve_opts* opts, nc_solver* out) {
  return guard([&] {
    NC_REQUIRE(out, NC_ERR_ARG, "null argument");
    *out = solver_create_impl(A, opts);
  });
}

int nc_solver_destroy(nc_solver S) {
  return guard([&] { delete S; });
}

int nc_solver_set_state(nc_solver S, double t0, const double* u) {
  return guard([&] { solver_set_state_impl(S, t0, u); });
}

int nc_solver_restart(nc_solver S) {
  return guard([&] {
    NC_REQUIRE(S && S->u0.p, NC_ERR_ARG, "solver has no state; call nc_solver_set_state first");
    solver_reinit(S);
  });
}

int nc_solver_run(nc_solver S, int32_t n_out, const double* t_out) {
  return guard([&] { solver_run_impl(S, n_out, t_out); });
}

int nc_solver_get_snapshot(nc_solver S, int32_t k, double* u) {
  return guard([&] {
    NC_REQUIRE(S && u && k >= 0 && k < S->n_snaps, NC_ERR_ARG, "snapshot index out of range");
    copy_to_host(S, u, S->snaps.p + (size_t)k * S->Np);
  });
}

int nc_solver_get_fspvec(nc_solver S, int32_t k, int32_t block, nc_space space, nc_fspvec* p, double* sinks) {
  return guard([&] {
    NC_REQUIRE(S && space && p && k >= 0 && k < S->n_snaps, NC_ERR_ARG, "snapshot index out of range");
    NC_REQUIRE(block >= 0 && block < S->blocks, NC_ERR_ARG, "block index out of range");
    NC_REQUIRE(space->n == S->A->n && space->nr == S->A->nr, NC_ERR_ARG,
               "the state space does not match the solver's generator");
    if (!S->snap_states || S->snap_space_uid != space->uid || S->snap_version != space->version) {
      S->snap_states = share_states(space->states.p, space->n, space->ns, space->stream.s);
      NC_CHECK_HIP(hipStreamSynchronize(space->stream.s));
      S->snap_space_uid = space->uid;
      S->snap_version = space->version;
    }
    const double* base = S->snaps.p + (size_t)k * S->Np + (size_t)block * S->Npb;
    *p = fspvec_from_device(space->ns, space->n, S->snap_states, base, S->s);
    if (sinks)
      NC_CHECK_HIP(hipMemcpy(sinks, base + S->A->n, sizeof(double) * S->A->nr, hipMemcpyDeviceToHost));
  });
}

int nc_solver_get_state(nc_solver S, double* t, double* u) {
  return guard([&] {
    NC_REQUIRE(S, NC_ERR_ARG, "null solver");
    if (t) *t = S->t;
    if (u) copy_to_host(S, u, S->u.p);
  });
}

int nc_solver_stats(nc_solver S, nc_solve_stats* st) {
  return guard([&] {
    NC_REQUIRE(S && st, NC_ERR_ARG, "null argument");
    *st = S->st;
  });
}

static void solve_fixed_impl(nc_matrix_s* A, nc_sensmatrix_s* SA, const nc_solve_opts* opts, const double* u0,
                             int32_t n_out, const double* t_out, double* u_out, nc_solve_stats* st) {
  NC_REQUIRE(A && u0 && (n_out == 0 || (t_out && u_out)), NC_ERR_ARG, "null argument");
  nc_solver_s* S = solver_create_impl(A, opts, SA);
  struct Guard {
    nc_solver_s* S;
    ~Guard() { delete S; }
  } gd{S};
  const double t0 = n_out ? t_out[0] : 0.0;
  solver_set_state_impl(S, t0, u0);
  solver_run_impl(S, n_out, t_out);
  for (int k = 0; k < n_out; ++k) copy_to_host(S, u_out + (size_t)k * S->N, S->snaps.p + (size_t)k * S->Np);
  if (st) nc_solver_stats(S, st);
}

int nc_solve_fixed(nc_matrix A, const nc_solve_opts* opts, const double* u0, int32_t n_out, const double* t_out,
                   double* u_out, nc_solve_stats* st) {
  return guard([&] { solve_fixed_impl(A, nullptr, opts, u0, n_out, t_out, u_out, st); });
}

int nc_solver_create_sens(nc_sensmatrix SA, const nc_solve_opts* opts, nc_solver* out) {
  return guard([&] {
    NC_REQUIRE(SA && out, NC_ERR_ARG, "null argument");
    *out = solver_create_impl(SA->A, opts, SA);
  });
}

int nc_solve_sens_fixed(nc_sensmatrix SA, const nc_solve_opts* opts, const double* u0, int32_t n_out,
                        const double* t_out, double* u_out, nc_solve_stats* st) {
  return guard([&] {
    NC_REQUIRE(SA, NC_ERR_ARG, "null argument");
    solve_fixed_impl(SA->A, SA, opts, u0, n_out, t_out, u_out, st);
  });
}

}  // extern "C"

namespace nc {

nc_solver_s* solver_create(nc_matrix_s* A, const nc_solve_opts* opts, nc_sensmatrix_s* SA) {
  return solver_create_impl(A, opts, SA);
}

// Set the state from a device vector of the true length N, blocks contiguous (t0 is its
// time).
double solver_step_hint(const nc_solver_s* S) {
  if (S->method == NC_METHOD_KRYLOV) return S->started ? S->t_new : 0.0;
  return S->h;
}

void solver_seed_step(nc_solver_s* S, double h) {
  if (!(h > 0.0) || !std::isfinite(h)) return;
  if (S->method == NC_METHOD_KRYLOV) {
    S->anorm = std::max(S->SA ? S->SA->norm1 : S->A->norm1, 1e-300);
    S->t_new = h;
    S->started = true;
  } else {
    S->h = h;
  }
}

void solver_set_state_device(nc_solver_s* S, double t0, const double* u_dev) {
  if (!S->u0.p) {
    S->u0.alloc(S->Np);
    NC_CHECK_HIP(hipMemsetAsync(S->u0.p, 0, sizeof(double) * S->Np, S->s));
  }
  // u_dev holds the blocks contiguously (stride Nb); the solver pads each to Npb
  NC_CHECK_HIP(hipMemcpy2DAsync(S->u0.p, sizeof(double) * S->Npb, u_dev, sizeof(double) * S->Nb,
                                sizeof(double) * S->Nb, S->blocks, hipMemcpyDeviceToDevice, S->s));
  double* b2 = static_cast<double*>(host_stage(5));
  launch_sumsq(S, S->u0.p, S->kbuf.p, S->s);
  NC_CHECK_HIP(hipMemcpyAsync(b2, S->kbuf.p, sizeof(double), hipMemcpyDeviceToHost, S->s));
  NC_CHECK_HIP(hipStreamSynchronize(S->s));
  S->beta0 = std::sqrt(*b2);
  S->t0 = t0;
  solver_reinit(S);
  NC_CHECK_HIP(hipStreamSynchronize(S->s));
}

}  // namespace nc
