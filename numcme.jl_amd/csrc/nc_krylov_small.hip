// The Krylov process of a small space in one launch of one workgroup (see nc_iop.h for the
// method and the order of its sums, which the launches of larger spaces share).
#include "nc_solver.h"

namespace nc {
namespace {

constexpr int kT = kIopThreads;

template <typename VT>
struct SmallArgs {
  int64_t n, ld, Np;
  int32_t K, R, m;
  const double* diag;
  const int32_t* col;
  const VT* val;
  const int64_t* sink_off;
  const int32_t* sink_src;
  const VT* sink_val;
  VT* V;
  double* u;
  double* host;
  KLayout L;
  double btol;
  int32_t nv;  // >= 0: first u <- cu u + sum cs[i] V_{i+1} (the end of the step before)
  double cu;
  double cs[32];
};

template <typename T>
struct alignas(2 * sizeof(T)) Two {
  T v[2];
};

// The tree of the mat-vec's sink rows (lane l with l + 32, then 16, 8, 4, 2, 1; lane 0's sum)
// by register permutes: the halves and the odd rows of 16 swapped, then rotations within a
// row, whose lanes agree modulo the width already summed.
__device__ inline double tree_sum(double v) {
  auto swapped = [](auto pl, double x) {
    const auto lo = pl((uint32_t)__double2loint(x)), hi = pl((uint32_t)__double2hiint(x));
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
  };
  v = swapped([](uint32_t x) { return __builtin_amdgcn_permlane32_swap(x, x, false, false); }, v);
  v = swapped([](uint32_t x) { return __builtin_amdgcn_permlane16_swap(x, x, false, false); }, v);
  v = iop_dpp_add<0x128>(v);
  v = iop_dpp_add<0x124>(v);
  v = iop_dpp_add<0x122>(v);
  return iop_dpp_add<0x121>(v);
}

// Thread t owns rows 512 p + 2 t, + 1 for p < P: their matrix entries stay in registers for
// the whole process, the vector being multiplied lives in LDS, and a column is two barriers:
// one before its gathers, one at its sums. Latency bound (LDS gathers, the wave sums, one
// square root and one division): a column of 31 takes 1.9 us at 240 rows, 2.6 at 1,400 and
// 3.4 at 3,000, where the launches of the process cost 5 us a column. H and the sink values
// collect in LDS and go to the host's memory at the end, and nothing in the column loop is
// indexed by a loop counter (private memory): a wait for either also waits for the stores
// to host memory, 2.3, 3.0 and 4.4 us a column. KT: slots, entries past K weigh zero.
template <typename VT, int KT, int P>
__global__ __launch_bounds__(kT) void k_krylov_small(SmallArgs<VT> a) {
  __shared__ double s_x[kIopRows * P];
  __shared__ double s_w[kIopWaves][kIopSums];
  __shared__ double s_sv[3][kIopTail], s_sq[kIopTail];
  __shared__ double s_k[32][4], s_ks[32][kIopTail], s_avn;  // for the host, written at the end
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = (int)a.n, R = a.R;
  double dg[P][2];
  VT w[P][2][KT];
  uint16_t cl[P][2][KT];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int i0 = kIopRows * p + 2 * tid, ic = i0 < n ? i0 : 0;
    const Two<double> d = *reinterpret_cast<const Two<double>*>(a.diag + ic);
#pragma unroll
    for (int r = 0; r < 2; ++r) dg[p][r] = i0 + r < n ? d.v[r] : 0.0;
#pragma unroll
    for (int k = 0; k < KT; ++k) {
      const int64_t o = (int64_t)(k < a.K ? k : 0) * a.ld + ic;
      const Two<VT> wk = *reinterpret_cast<const Two<VT>*>(a.val + o);
      const Two<int32_t> ck = *reinterpret_cast<const Two<int32_t>*>(a.col + o);
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const bool on = k < a.K && i0 + r < n;
        w[p][r][k] = on ? wk.v[r] : (VT)0;
        cl[p][r][k] = (uint16_t)(on ? ck.v[r] : 0);
      }
    }
  }
  // the first 64 entries of this wave's first two sink rows
  int ss[2] = {0, 0};
  double sw[2] = {0.0, 0.0};
  int64_t e0[2] = {0, 0}, e1[2] = {0, 0};
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = wave + kIopWaves * j;
    if (r < R) {
      e0[j] = a.sink_off[r];
      e1[j] = a.sink_off[r + 1];
      if (e0[j] + lane < e1[j]) {
        ss[j] = a.sink_src[e0[j] + lane];
        sw[j] = (double)a.sink_val[e0[j] + lane];
      }
    }
  }
  double x[P][2], x1[P][2], q[P][2];  // V_c, V_{c-1} and q_c of the thread's rows
  double usink = 0.0;
  if (a.nv >= 0) {
    constexpr int C = P <= 2 ? 16 : 8;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int i0 = kIopRows * p + 2 * tid, ic = i0 < n ? i0 : 0;
      const Two<double> uv = *reinterpret_cast<const Two<double>*>(a.u + ic);
      double y[2] = {a.cu * uv.v[0], a.cu * uv.v[1]};
      for (int i = 0; i < a.nv; i += C) {
        Two<VT> vv[C];
#pragma unroll
        for (int u = 0; u < C; ++u)
          vv[u] = *reinterpret_cast<const Two<VT>*>(a.V + (int64_t)(min(i + u, a.nv - 1) + 1) * a.Np + ic);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < C; ++u)
#pragma unroll
          for (int r = 0; r < 2; ++r)
            if (i + u < a.nv) y[r] = __fma_rn(a.cs[i + u], (double)vv[u].v[r], y[r]);
      }
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        x[p][r] = 0.0;
        if (i0 + r < n) {
          x[p][r] = (double)(VT)y[r];
          a.u[i0 + r] = y[r];
          a.V[i0 + r] = (VT)y[r];
        }
      }
    }
    if (tid < R) {
      double y = a.cu * a.u[n + tid];
      for (int i = 0; i < a.nv; ++i) y = __fma_rn(a.cs[i], (double)a.V[(int64_t)(i + 1) * a.Np + n + tid], y);
      a.u[n + tid] = usink = y;
      a.V[n + tid] = (VT)y;
      s_sv[0][tid] = (double)(VT)y;
    }
  } else {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int i0 = kIopRows * p + 2 * tid, ic = i0 < n ? i0 : 0;
      const Two<VT> v = *reinterpret_cast<const Two<VT>*>(a.V + ic);
#pragma unroll
      for (int r = 0; r < 2; ++r) x[p][r] = i0 + r < n ? (double)v.v[r] : 0.0;
    }
    if (tid < R) {
      usink = a.u[n + tid];
      s_sv[0][tid] = (double)a.V[n + tid];
    }
  }
  const KLayout L = a.L;
  if (tid < R) {
    s_sv[2][tid] = 0.0;  // no vector before V_0
    a.host[L.sinkv(a.m + 1, tid, R)] = usink;
  }
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      s_x[kIopRows * p + 2 * tid + r] = x[p][r];
      x1[p][r] = 0.0;
    }
  double scp = 0.0;
  for (int c = 0; c <= a.m; ++c) {
    __syncthreads();
    double t[kIopSums] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        double acc = __dmul_rn(dg[p][r], x[p][r]);
#pragma unroll
        for (int k = 0; k < KT; ++k) acc = __fma_rn((double)w[p][r][k], s_x[cl[p][r][k]], acc);
        q[p][r] = acc;
      }
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int r = 0; r < 2; ++r) iop_row_sums(x[p][r], x1[p][r], q[p][r], t);  // rows past the states are zero
    // sink rows, one wave each, its entries in the order of the launches' 256 threads
    auto sink_row = [&](int r, int64_t b0, int64_t b1, bool kept, int src, double weight) {
      double s = 0.0;
      for (int v = 0; v < 4 && b0 + 64 * v < b1; ++v) {
        double acc = 0.0;
        int64_t e = b0 + 64 * v + lane;
        if (v == 0 && kept) {
          acc = __fma_rn(weight, s_x[src], acc);
          e += 256;
        }
        for (; e < b1; e += 256) acc = __fma_rn((double)a.sink_val[e], s_x[a.sink_src[e]], acc);
        s += tree_sum(acc);
      }
      if (lane == 0) s_sq[r] = s;
    };
    if (wave < R) sink_row(wave, e0[0], e1[0], true, ss[0], sw[0]);
    if (wave + kIopWaves < R) sink_row(wave + kIopWaves, e0[1], e1[1], true, ss[1], sw[1]);
    for (int r = wave + 2 * kIopWaves; r < R; r += kIopWaves)
      sink_row(r, a.sink_off[r], a.sink_off[r + 1], false, 0, 0.0);
#pragma unroll
    for (int k = 0; k < kIopSums; ++k) t[k] = iop_wave_sum(t[k]);
    if (lane == 0) {
#pragma unroll
      for (int k = 0; k < kIopSums; ++k) s_w[wave][k] = t[k];
    }
    __syncthreads();
    double tot[kIopSums];
#pragma unroll
    for (int k = 0; k < kIopSums; ++k) tot[k] = iop_waves(s_w, k);
    const double* sx = s_sv[c % 3];
    const double* sx1 = s_sv[(c + 2) % 3];
    iop_add_tail(R, sx, sx1, s_sq, tot);
    const IopCoef o = iop_coef(tot, c, scp, a.btol);
    if (tid == 0) {
      s_k[c][0] = o.nrm;
      s_k[c][1] = o.sc;
      s_k[c][2] = o.h1;
      s_k[c][3] = o.h0;
      if (c == a.m) s_avn = o.sc * sqrt(tot[4]);
    }
    if (tid < R) s_ks[c][tid] = sx[tid];
    if (c == a.m) break;
    VT* vn = a.V + (int64_t)(c + 1) * a.Np;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int i0 = kIopRows * p + 2 * tid;
      Two<VT> v;
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        v.v[r] = iop_row<VT>(o.xs, o.c1, o.c0, q[p][r], x[p][r], x1[p][r]);
        x1[p][r] = x[p][r];
        x[p][r] = (double)v.v[r];
        s_x[i0 + r] = x[p][r];
      }
      if (i0 + 1 < n)
        *reinterpret_cast<Two<VT>*>(vn + i0) = v;
      else if (i0 < n)
        vn[i0] = v.v[0];
    }
    if (tid < R) {
      const VT y = iop_row<VT>(o.xs, o.c1, o.c0, s_sq[tid], sx[tid], sx1[tid]);
      vn[n + tid] = y;
      s_sv[(c + 1) % 3][tid] = (double)y;
    }
    scp = o.sc;
  }
  __syncthreads();
  if (tid <= a.m) {
    const int c = tid;
    a.host[c > 0 ? L.H(c, c - 1) : L.misc(MISC_BETA)] = s_k[c][0];
    a.host[L.sc(c)] = s_k[c][1];
    if (c < a.m) {
      a.host[L.H(c, c)] = s_k[c][2];
      if (c > 0) a.host[L.H(c - 1, c)] = s_k[c][3];
    } else {
      a.host[L.misc(MISC_AVN)] = s_avn;
    }
  }
  for (int i = tid; i < (a.m + 1) * R; i += kT) a.host[L.sinkv(0, 0, R) + i] = s_ks[i / R][i % R];
}

template <typename VT>
void launch_t(nc_solver_s* S, int nv, double cu, const double* cs) {
  nc_matrix_s* A = S->A;
  SmallArgs<VT> a{};
  a.n = A->n;
  a.ld = A->ld;
  a.Np = S->Np;
  a.K = A->K;
  a.R = A->nr;
  a.m = S->m;
  a.diag = A->diag.p;
  a.col = A->col.p;
  a.val = reinterpret_cast<const VT*>(A->val.p);
  a.sink_off = A->sink_off.p;
  a.sink_src = A->sink_src.p;
  a.sink_val = reinterpret_cast<const VT*>(A->sink_val.p);
  a.V = reinterpret_cast<VT*>(S->V.p);
  a.u = S->u.p;
  a.host = S->hbuf_dev;
  a.L = KLayout{S->m};
  a.btol = krylov_breakdown_tol(S);
  a.nv = nv;
  a.cu = cu;
  for (int i = 0; i < nv; ++i) a.cs[i] = cs[i];
  hipStream_t s = S->s;
  const bool k4 = A->K <= 4;
  if (A->n <= kIopRows)
    k4 ? k_krylov_small<VT, 4, 1><<<1, kT, 0, s>>>(a) : k_krylov_small<VT, 8, 1><<<1, kT, 0, s>>>(a);
  else if (A->n <= 2 * kIopRows)
    k4 ? k_krylov_small<VT, 4, 2><<<1, kT, 0, s>>>(a) : k_krylov_small<VT, 8, 2><<<1, kT, 0, s>>>(a);
  else if (A->n <= 4 * kIopRows)
    k4 ? k_krylov_small<VT, 4, 4><<<1, kT, 0, s>>>(a) : k_krylov_small<VT, 8, 4><<<1, kT, 0, s>>>(a);
  else
    k_krylov_small<VT, 4, 8><<<1, kT, 0, s>>>(a);
  NC_CHECK_HIP(hipGetLastError());
}

}  // namespace

// One workgroup is faster than a launch per column while a column's work on one CU stays
// under a launch's latency.
bool krylov_small_fits(const nc_solver_s* S) {
  const nc_matrix_s* A = S->A;
  return !S->SA && !A->timing && A->mf_mode == 0 && A->tv_r.empty() && A->n_chunks == 0 && A->nr <= kIopTail &&
         krylov_small_shape(A);
}

void krylov_small_launch(nc_solver_s* S, int nv, double cu, const double* cs) {
  if (!krylov_small_fits(S) || nv > 32 || S->m > 31 || S->A->n_rows > S->Np)
    throw Error(NC_ERR_INTERNAL, "one-workgroup Krylov process misconfigured");
  if (S->A->precision == NC_FP32)
    launch_t<float>(S, nv, cu, cs);
  else
    launch_t<double>(S, nv, cu, cs);
}

}  // namespace nc
