// First column of exp(T) of a tridiagonal matrix (host), included twice by nc_util.hip:
// once compiled for AVX2 and FMA, once for the baseline instruction set.
// (No include guard: each inclusion defines the kernel in its own namespace.)
//
// Incomplete orthogonalisation over two vectors leaves a tridiagonal H, and a Krylov step
// needs exp(tau H) e1 alone. T = tau H stands for a generator's section with its spectrum
// about [-2c, 0], so T + c I with c the centre of the diagonal's range has half the norm,
// and exp(T) e1 = (e^{-c/s} exp((T + c I) / s))^s e1 with the inner exponential's column
// from its Taylor series, s a power of two (the scaling is exact). The terms grow to
// e^{|T + c I| / s}, e^{-c/s} takes that back; kTriExcess bounds what is left of it (a matrix
// that is far from normal) and so the digits lost. Against 80-bit arithmetic on 837 matrices
// of the process (toggle, telegraph and cascade; m 12 and 30; tolerances 1e-6 to 1e-12;
// norms 0.1 to 94) the absolute error is 7e-16 on average and 8.2e-15 at most, the dense
// Pade form's 1.0e-15 and 9.2e-15; m = 30 takes 5.9 us against 27.
typedef double v4t __attribute__((vector_size(32)));

constexpr double kTriPart = 8.0;    // norm of one part (4: 8.2 us, the same error)
constexpr double kTriExcess = 4.0;  // its norm less its shift

// lo[i] = T(i, i - 1), di[i] = T(i, i), up[i] = T(i, i + 1), n <= 64; false, and out not
// written: more than max_parts parts, or entries that are not finite
inline bool expm_tri(int n, const double* lo, const double* di, const double* up, int max_parts, double* out) {
  constexpr int kMax = 64;
  alignas(32) double l[kMax], d[kMax], u[kMax], sum[kMax];
  alignas(32) double xa[kMax + 8] = {}, xb[kMax + 8] = {};  // the vector at offset 4
  double dmin = di[0], dmax = di[0];
  for (int i = 1; i < n; ++i) {
    dmin = di[i] < dmin ? di[i] : dmin;
    dmax = di[i] > dmax ? di[i] : dmax;
  }
  const double c = -0.5 * (dmin + dmax);
  double norm = 0.0;
  for (int j = 0; j < n; ++j) {
    const double s = std::fabs(di[j] + c) + (j > 0 ? std::fabs(up[j - 1]) : 0.0) + (j + 1 < n ? std::fabs(lo[j + 1]) : 0.0);
    if (!(s <= kTriPart * max_parts)) return false;
    norm = s > norm ? s : norm;
  }
  int parts = 1;
  while (norm > kTriPart * parts || norm - c > kTriExcess * parts) {
    if (parts > max_parts / 2) return false;
    parts *= 2;
  }
  const double scale = 1.0 / parts, part = norm * scale, damp = std::exp(-c * scale);
  // up to the first term below 2^-57, and at least 8 terms into the last row, which term
  // n - 1 reaches first: the step's error estimate is the last rows, however small
  int deg = 1;
  for (double t = part; t > 6.9e-18; t *= part / deg) ++deg;
  deg = std::max(deg, n + 8);
  const int np = (n + 3) / 4 * 4;
  for (int i = 0; i < np; ++i) {
    l[i] = i > 0 && i < n ? lo[i] * scale : 0.0;
    d[i] = i < n ? (di[i] + c) * scale : 0.0;
    u[i] = i + 1 < n ? up[i] * scale : 0.0;
  }
  for (int i = 0; i < np; ++i) sum[i] = 0.0;
  sum[0] = 1.0;
  double *x = xa + 4, *y = xb + 4;
  for (int p = 0; p < parts; ++p) {
    for (int i = 0; i < np; ++i) x[i] = sum[i];
    for (int k = 1; k <= deg; ++k) {
      const double f = 1.0 / k;
      const v4t fv = {f, f, f, f};
      for (int i = 0; i < np; i += 4) {
        v4t xm, x0, xp, lv, dv, uv, sv;
        __builtin_memcpy(&xm, x + i - 1, sizeof(v4t));
        __builtin_memcpy(&x0, x + i, sizeof(v4t));
        __builtin_memcpy(&xp, x + i + 1, sizeof(v4t));
        __builtin_memcpy(&lv, l + i, sizeof(v4t));
        __builtin_memcpy(&dv, d + i, sizeof(v4t));
        __builtin_memcpy(&uv, u + i, sizeof(v4t));
        __builtin_memcpy(&sv, sum + i, sizeof(v4t));
        const v4t t = (lv * xm + dv * x0 + uv * xp) * fv;
        sv += t;
        __builtin_memcpy(y + i, &t, sizeof(v4t));
        __builtin_memcpy(sum + i, &sv, sizeof(v4t));
      }
      std::swap(x, y);
    }
    for (int i = 0; i < np; ++i) sum[i] *= damp;
  }
  for (int i = 0; i < n; ++i) out[i] = sum[i];
  return true;
}
