// The Krylov process of the device expv (internal, device code shared by its kernels).
//
// Incomplete orthogonalisation (Y. Saad, Math. Comp. 37, 1981; for the chemical master
// equation H. D. Vo and R. B. Sidje, "Approximating the large sparse matrix exponential
// using incomplete orthogonalization and Krylov subspaces of variable dimension", Numer.
// Linear Algebra Appl. 24, 2017): V_{c+1} = A v_c made orthogonal to V_c and V_{c-1} only.
// A V = V H holds, to the rounding of the stored vectors, whatever the angles between older
// ones, so exp(tau A) u is approximated by V exp(tau H) e1 as with full orthogonalisation, with
// the same error estimate, held lower (krylov_step_tol). A column then reads two basis vectors
// instead of all of them: the full form's two sweeps over 1..30 vectors took 60% of a solve on
// the 1024^2 toggle switch. The price is steps. Full form, this form with the estimate held to
// the tolerance, and as it is held:
//   telegraph 800 states   FP64 1e-9    73  102  118     39 ms,   8.8,  10.0
//   toggle    301 x 259    FP64 1e-12   60   82   94     32 ms,  19.2,  21.5
//   toggle    1024^2       FP32 1e-9    99  137  123    119 ms,  87.8,  78.5
//   toggle    1024^2       FP64 1e-9    88  154  194    158 ms, 119.6, 149.9
// (the breakdown threshold is no part of it: with Expokit's 1e-7 the second column reads 99,
// 82, 137, 154). Near the stationary state of a stiff box the full form's threshold saved it
// most steps, at 2e-5 of error: 8,000 telegraph states at 1e-9 FP64 219 and 868 steps, 119 and
// 163 ms, FP32 164 and 958, 87 and 185 ms.
//
// The basis is stored unnormalised with FP64 scales sc_c = 1 / |V_c|. Column c sums
//   T0 = V_c.q  T1 = V_{c-1}.q  T2 = V_c.V_c  T3 = V_{c-1}.V_c  T4 = q.q,   q = A V_c,
// from which (iop_coef) |V_c|, sc_c and the two coefficients follow: h solves the 2x2 Gram
// system of the stored (rounded) vectors. The next column's vector is
//   V_{c+1} = sc_c q - h1 sc_c V_c - h0 sc_{c-1} V_{c-1}          (iop_row)
// rounded to storage. Three ways to run a column give the same result bit for bit, since
// they share these functions and the order of the sums: one kernel that forms V_c while it
// gathers it (k_krylov_col), the separate form / mat-vec / sums kernels, and the
// one-workgroup process of small spaces.
//
// Order of the sums: rows in blocks of kIopRows, thread t takes rows 2t, 2t + 1 of its
// workgroup's blocks in ascending order; waves, then the wave sums one after the other; up
// to kIopGroups workgroups' partials; the tail rows (the sinks) one after the other, last.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace nc {

constexpr int kIopThreads = 256;
constexpr int kIopWaves = kIopThreads / 64;
constexpr int kIopRows = 2 * kIopThreads;  // rows per block
constexpr int kIopGroups = 512;  // workgroups of a column at most: every workgroup of the next
                                 // column folds their partials itself, 20 KB from L2 (1,024
                                 // groups: 2 us more a column)
constexpr int kIopSums = 5;
constexpr int kIopTail = 32;  // sink rows at most

// one: the one-workgroup process holds a space of this shape, and every form sums in its order
inline int iop_groups(int64_t nblk, bool one) {
  if (one) return 1;
  return nblk < kIopGroups ? (int)nblk : kIopGroups;
}

// kbuf layout (doubles)
struct KLayout {
  int m;
  __host__ __device__ int H(int i, int j) const { return i * (m + 2) + j; }
  __host__ __device__ int sc(int i) const { return (m + 2) * (m + 2) + i; }
  __host__ __device__ int misc(int i) const { return (m + 2) * (m + 2) + (m + 2) + i; }
  // sink rows of basis vector j (j <= m) and of the state (j = m+1), R sinks each
  __host__ __device__ int sinkv(int j, int r, int R) const { return misc(8) + j * R + r; }
  __host__ __device__ int size() const { return misc(8); }
  __host__ __device__ int size_with_sinks(int R) const { return size() + (m + 2) * R; }
};
enum { MISC_AVN = 0, MISC_BETA = 1 };

struct IopArgs {
  int64_t n;      // rows summed in blocks
  int64_t tail1;  // rows n .. tail1 - 1 (the sinks, at most kIopTail) are added by the fold
  int64_t ld;     // basis stride, a multiple of 1024; rows past the true length stay zero
  int64_t nblk;
  int32_t groups;
  int32_t c;        // column
  void* V;          // basis, matrix precision
  double* q[2];     // q of column c in q[c & 1]
  double* part[2];  // sums of column c in part[c & 1], value-major (kIopSums x groups)
  double* kb;
  KLayout L;
  double btol;
};

struct IopCoef {
  double nrm, sc, h1, h0;  // |V_c|, its scale, coefficients of v_c and v_{c-1}
  double xs, c1, c0;       // V_{c+1} = xs q + c1 V_c + c0 V_{c-1}
};

#if defined(__HIPCC__)

template <int CTRL>
__device__ inline double iop_dpp_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return v + __hiloint2double(hi, lo);
}

__device__ inline double iop_readlane(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Sum over the wave (all 64 lanes active), the same value in every lane: within rows of 16
// lanes by register permutes (no LDS traffic, unlike a shuffle), then the four row sums.
__device__ inline double iop_wave_sum(double v) {
  v = iop_dpp_add<0xB1>(v);   // lane ^ 1
  v = iop_dpp_add<0x4E>(v);   // lane ^ 2
  v = iop_dpp_add<0x141>(v);  // the other four of eight
  v = iop_dpp_add<0x140>(v);  // the other eight of sixteen
  return (iop_readlane(v, 0) + iop_readlane(v, 16)) + (iop_readlane(v, 32) + iop_readlane(v, 48));
}

// The five products of one row added to the running sums
__device__ inline void iop_row_sums(double x, double x1, double q, double (&t)[kIopSums]) {
  t[0] = __fma_rn(x, q, t[0]);
  t[1] = __fma_rn(x1, q, t[1]);
  t[2] = __fma_rn(x, x, t[2]);
  t[3] = __fma_rn(x1, x, t[3]);
  t[4] = __fma_rn(q, q, t[4]);
}

// Row of V_{c+1} in storage precision, as the FP64 value that storage holds
template <typename BT>
__device__ inline BT iop_row(double xs, double c1, double c0, double q, double v1, double v0) {
  return (BT)__fma_rn(c0, v0, __fma_rn(c1, v1, __dmul_rn(xs, q)));
}

// Column c's norm, scale and coefficients from its folded sums; scp = sc_{c-1} (c > 0).
__device__ inline IopCoef iop_coef(const double (&t)[kIopSums], int c, double scp, double btol) {
#pragma clang fp contract(off)
  IopCoef o;
  o.nrm = sqrt(t[2]);
  // the first vector is normalised however small; a vanished later one ends the space
  o.sc = o.nrm > (c == 0 ? 0.0 : btol) ? 1.0 / o.nrm : 0.0;
  const double a1 = (o.sc * o.sc) * t[0];
  o.h1 = a1;
  o.h0 = 0.0;
  if (c > 0) {
    const double s = scp * o.sc, a0 = s * t[1], g = s * t[3], det = 1.0 - g * g;
    o.h0 = a0;
    if (det > 1e-3) {  // nearly parallel stored vectors: any coefficients keep A V = V H
      // 1 / (1 - g^2); g is of the storage rounding almost always, no division then
      const double inv = fabs(g) < 1e-4 ? 1.0 + g * g : 1.0 / det;
      o.h1 = (a1 - g * a0) * inv;
      o.h0 = (a0 - g * a1) * inv;
    }
  }
  o.xs = o.sc;
  o.c1 = -(o.h1 * o.sc);
  o.c0 = -(o.h0 * scp);
  return o;
}

// Sums over the waves of a workgroup's wave sums
__device__ inline double iop_waves(const double (&s_w)[kIopWaves][kIopSums], int k) {
  double s = s_w[0][k];
#pragma unroll
  for (int w = 1; w < kIopWaves; ++w) s += s_w[w][k];
  return s;
}

// Sums of a workgroup's running sums into part (one value per group).
__device__ inline void iop_group_sums(double (&t)[kIopSums], double* part, int groups, int g) {
  __shared__ double s_w[kIopWaves][kIopSums];
#pragma unroll
  for (int k = 0; k < kIopSums; ++k) t[k] = iop_wave_sum(t[k]);
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int k = 0; k < kIopSums; ++k) s_w[threadIdx.x >> 6][k] = t[k];
  }
  __syncthreads();
  if (threadIdx.x < kIopSums) {
    const int k = threadIdx.x;
    part[(int64_t)k * groups + g] = iop_waves(s_w, k);
  }
}

// Tail rows added to the totals, one after the other (x, x1, q of tail row r in sx, sx1, sq,
// arrays of kIopTail). Four rows' values are loaded together (a row at a time was an LDS
// latency each); rows past the last weigh zero, which leaves a sum as it is.
__device__ inline void iop_add_tail(int rows, const double* sx, const double* sx1, const double* sq,
                                    double (&tot)[kIopSums]) {
  double tl[kIopSums] = {0.0, 0.0, 0.0, 0.0, 0.0};
  for (int r = 0; r < rows; r += 4) {
    double x[4], x1[4], q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = r + u < kIopTail ? r + u : 0;
      x[u] = sx[i], x1[u] = sx1[i], q[u] = sq[i];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool on = r + u < rows;  // the others may hold anything
      iop_row_sums(on ? x[u] : 0.0, on ? x1[u] : 0.0, on ? q[u] : 0.0, tl);
    }
  }
#pragma unroll
  for (int k = 0; k < kIopSums; ++k) tot[k] += tl[k];
}

// Fold of column c's partials by a workgroup: every thread gets the totals.
// Every workgroup of the following launch does this itself (a separate fold launch took
// 3.9 us a column).
template <typename BT>
__device__ inline void iop_fold(const IopArgs& a, int c, double (&tot)[kIopSums]) {
  __shared__ double s_w[kIopWaves][kIopSums];
  __shared__ double s_x[kIopTail], s_x1[kIopTail], s_q[kIopTail];
  const double* p = a.part[c & 1];
  const int t = threadIdx.x, groups = a.groups;
  const int rows = (int)(a.tail1 - a.n);
  constexpr int U = kIopGroups / kIopThreads;
  double v[kIopSums];
#pragma unroll
  for (int k = 0; k < kIopSums; ++k) {
    double x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = p[k * groups + min(t + u * kIopThreads, groups - 1)];
    v[k] = t < groups ? x[0] : 0.0;
#pragma unroll
    for (int u = 1; u < U; ++u) v[k] += t + u * kIopThreads < groups ? x[u] : 0.0;
  }
  if (t < rows) {
    const BT* V = reinterpret_cast<const BT*>(a.V) + a.n + t;
    s_x[t] = (double)V[(int64_t)c * a.ld];
    s_x1[t] = c > 0 ? (double)V[(int64_t)(c - 1) * a.ld] : 0.0;
    s_q[t] = a.q[c & 1][a.n + t];
  }
#pragma unroll
  for (int k = 0; k < kIopSums; ++k) v[k] = iop_wave_sum(v[k]);
  if ((t & 63) == 0) {
#pragma unroll
    for (int k = 0; k < kIopSums; ++k) s_w[t >> 6][k] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kIopSums; ++k) tot[k] = iop_waves(s_w, k);
  iop_add_tail(rows, s_x, s_x1, s_q, tot);
}

// The fold and coefficients of column c (read by column c + 1); workgroup 0 keeps them.
template <typename BT>
__device__ inline IopCoef iop_finish_column(const IopArgs& a, int c) {
  const double scp = c > 0 ? a.kb[a.L.sc(c - 1)] : 0.0;
  double tot[kIopSums];
  iop_fold<BT>(a, c, tot);
  const IopCoef o = iop_coef(tot, c, scp, a.btol);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.kb[a.L.H(c, c)] = o.h1;
    a.kb[a.L.sc(c)] = o.sc;
    if (c > 0) {
      a.kb[a.L.H(c - 1, c)] = o.h0;
      a.kb[a.L.H(c, c - 1)] = o.nrm;
    } else {
      a.kb[a.L.misc(MISC_BETA)] = o.nrm;
    }
  }
  return o;
}

#endif  // __HIPCC__

}  // namespace nc
