// Small dense FP64 linear algebra held in registers: the packed-Schur PSD test, the
// symmetric QR algorithm that projects element Hessians and the cyclic Jacobi eigensolver
// of the diagonal-block inverses (Golub & Van Loan, "Matrix Computations", sections 8.3
// and 8.5).
#pragma once
#include "common.hpp"

namespace ysp {

// Packed-Schur PSD test (hessianKernelHeader.pyx:79-141) on a packed lower triangle
// L[r*(r+1)/2 + c] (c <= r) that it overwrites.
template <int N>
__device__ __forceinline__ bool psd_test_packed(double* L) {
  double scale = 1.0;
#pragma unroll
  for (int r = 0; r < N; ++r) scale = fmax(scale, fabs(L[r * (r + 1) / 2 + r]));
  const double tol = scale * 1.0e-10;
  bool ok = true;
#pragma unroll
  for (int c = 0; c < N; ++c) {
    const double pivot = L[c * (c + 1) / 2 + c];
    if (pivot < -tol) ok = false;
    const bool small = fabs(pivot) <= tol;
    if (small) {
#pragma unroll
      for (int r = c + 1; r < N; ++r)
        if (fabs(L[r * (r + 1) / 2 + c]) > tol) ok = false;
    } else {
      const double inv = 1.0 / pivot;
#pragma unroll
      for (int r = c + 1; r < N; ++r) {
        const double factor = L[r * (r + 1) / 2 + c] * inv;
#pragma unroll
        for (int t = c + 1; t <= r; ++t)
          L[r * (r + 1) / 2 + t] = fma(-factor, L[t * (t + 1) / 2 + c], L[r * (r + 1) / 2 + t]);
      }
    }
  }
  return ok;
}

// Cyclic Jacobi eigen-decomposition of a symmetric N x N matrix held in registers.
// On return A is diagonal (eigenvalues) and V holds the eigenvectors as columns.
template <int N>
__device__ __forceinline__ void jacobi_eigen(double (&A)[N][N], double (&V)[N][N]) {
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) V[i][j] = (i == j) ? 1.0 : 0.0;
  double fro = 0.0;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) fro += A[i][j] * A[i][j];
  const double stop = fro * 1.0e-32;
  for (int sweep = 0; sweep < 24; ++sweep) {
    double off = 0.0;
#pragma unroll
    for (int p = 0; p < N; ++p)
#pragma unroll
      for (int q = p + 1; q < N; ++q) off += A[p][q] * A[p][q];
    if (off <= stop) break;
#pragma unroll
    for (int p = 0; p < N; ++p)
#pragma unroll
      for (int q = p + 1; q < N; ++q) {
        const double apq = A[p][q];
        if (apq == 0.0) continue;
        const double theta = (A[q][q] - A[p][p]) / (2.0 * apq);
        const double t = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(1.0 + theta * theta));
        const double c = 1.0 / sqrt(1.0 + t * t);
        const double s = t * c;
#pragma unroll
        for (int k = 0; k < N; ++k) {
          const double akp = A[k][p], akq = A[k][q];
          A[k][p] = c * akp - s * akq;
          A[k][q] = s * akp + c * akq;
        }
#pragma unroll
        for (int k = 0; k < N; ++k) {
          const double apk = A[p][k], aqk = A[q][k];
          A[p][k] = c * apk - s * aqk;
          A[q][k] = s * apk + c * aqk;
        }
#pragma unroll
        for (int k = 0; k < N; ++k) {
          const double vkp = V[k][p], vkq = V[k][q];
          V[k][p] = c * vkp - s * vkq;
          V[k][q] = s * vkp + c * vkq;
        }
      }
  }
}

// Index of (p, q), p <= q, in the packed upper triangle of an N x N symmetric matrix.
template <int N>
__host__ __device__ constexpr int upper_index(int p, int q) {
  return p * N - p * (p - 1) / 2 + (q - p);
}

// 1/x to full double precision for finite normal x: the hardware reciprocal estimate and
// two Newton steps (each at least doubles the correct bits).
__device__ __forceinline__ double recip_nr(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}

// 1/sqrt(x) for x well inside the normal range: the hardware estimate and two Newton steps.
__device__ __forceinline__ double rsqrt_pos(double x) {
  double y = __builtin_amdgcn_rsq(x);
  const double hx = 0.5 * x;
  y = y * fma(-hx * y, y, 1.5);
  return y * fma(-hx * y, y, 1.5);
}

// Eigen-decomposition A = V diag(d) V^T of a symmetric matrix from its packed upper
// triangle a (N(N+1)/2 entries, destroyed): Householder tridiagonalisation, the
// orthogonal factor formed in V, then implicit QR sweeps with Wilkinson's shift applied to
// V (Golub & Van Loan, "Matrix Computations", sections 8.3.1 to 8.3.3). Backward stable:
// eigenvalues and V diag(f(d)) V^T carry an error of a few ulp of the largest entry,
// whatever the spectrum (off-diagonals are dropped at 1e-16 of the Frobenius norm).
//
// One matrix per lane, every index a compile-time constant and no control flow inside a
// sweep (a branch around each rotation made the compiler copy V at every merge, as many
// moves as multiply-adds). Bound by FP64 VALU work and its dependent chains at two
// wavefronts per SIMD (254 VGPRs): SNH tets take 79 rotations each, about 117 with the
// wavefront's lanes waiting for the slowest at every eigenvalue, each 36 multiply-adds on V,
// about 35 on the tridiagonal and one reciprocal square root. The round-robin Jacobi it
// replaces took 5.6 sweeps of 36 rotations: the projection of the 37^3-cell cube's 173,000
// indefinite tets 256 -> 116 us, of a 48^3-cell cube's 378,000 tets 502 -> 206 us, of one
// wavefront 71 -> 38 us.
template <int N>
__device__ __forceinline__ void sym_eigen_packed(double (&a)[N * (N + 1) / 2], double (&d)[N],
                                                 double (&V)[N][N]) {
  constexpr int E = N > 1 ? N - 1 : 1;
  auto at = [](int i, int j) constexpr { return i <= j ? upper_index<N>(i, j) : upper_index<N>(j, i); };
  // entries scaled exactly to at most 1 (squares below must not leave the normal range)
  double big = 0.0;
#pragma unroll
  for (int i = 0; i < N * (N + 1) / 2; ++i) big = fmax(big, fabs(a[i]));
  const int ex = __builtin_amdgcn_frexp_exp(big);
#pragma unroll
  for (int i = 0; i < N * (N + 1) / 2; ++i) a[i] = __builtin_amdgcn_ldexp(a[i], -ex);
  constexpr double kTiny = 1.0e-290;
  double e[E], beta[E];
#pragma unroll
  for (int k = 0; k + 2 < N; ++k) {
    // reflector of column k below the diagonal: v in place of the column's entries
    double tail = 0.0;
#pragma unroll
    for (int i = k + 2; i < N; ++i) tail = fma(a[at(k, i)], a[at(k, i)], tail);
    const double x0 = a[at(k, k + 1)];
    d[k] = a[at(k, k)];
    e[k] = x0;
    beta[k] = 0.0;
    if (tail > kTiny) {
      const double n2 = fma(x0, x0, tail), norm = sqrt(n2);
      e[k] = x0 >= 0.0 ? -norm : norm;
      a[at(k, k + 1)] = x0 - e[k];
      const double b = recip_nr(fma(fabs(x0), norm, n2));
      beta[k] = b;
      double w[N], vw = 0.0;
#pragma unroll
      for (int i = k + 1; i < N; ++i) {
        double acc = 0.0;
#pragma unroll
        for (int j = k + 1; j < N; ++j) acc = fma(a[at(i, j)], a[at(k, j)], acc);
        w[i] = b * acc;
        vw = fma(w[i], a[at(k, i)], vw);
      }
      const double h = 0.5 * b * vw;
#pragma unroll
      for (int i = k + 1; i < N; ++i) w[i] = fma(-h, a[at(k, i)], w[i]);
#pragma unroll
      for (int i = k + 1; i < N; ++i)
#pragma unroll
        for (int j = i; j < N; ++j)
          a[at(i, j)] = fma(-w[i], a[at(k, j)], fma(-a[at(k, i)], w[j], a[at(i, j)]));
    }
  }
  if constexpr (N >= 2) {
    d[N - 2] = a[at(N - 2, N - 2)];
    e[N - 2] = a[at(N - 2, N - 1)];
  }
  d[N - 1] = a[at(N - 1, N - 1)];
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) V[i][j] = (i == j) ? 1.0 : 0.0;
#pragma unroll
  for (int k = N - 3; k >= 0; --k)
#pragma unroll
    for (int j = k + 1; j < N; ++j) {
      double acc = 0.0;
#pragma unroll
      for (int i = k + 1; i < N; ++i) acc = fma(a[at(k, i)], V[i][j], acc);
      acc *= beta[k];
#pragma unroll
      for (int i = k + 1; i < N; ++i) V[i][j] = fma(-acc, a[at(k, i)], V[i][j]);
    }
  if constexpr (N >= 2) {
    double fro = 0.0;
#pragma unroll
    for (int i = 0; i < N; ++i) fro = fma(d[i], d[i], fro);
#pragma unroll
    for (int i = 0; i + 1 < N; ++i) fro = fma(2.0 * e[i], e[i], fro);
    const double tol = 1.0e-16 * sqrt(fro);
    // stage H: sweeps of the leading (H + 1) x (H + 1) block until every lane's last
    // off-diagonal is negligible (lanes that are done take part with the identity)
#pragma unroll
    for (int H = N - 1; H >= 1; --H) {
      for (int it = 0; it < 40; ++it) {
        const bool open = fabs(e[H - 1]) > tol;
        if (!open) e[H - 1] = 0.0;
        if (!__any(open)) break;
        int lo = open ? 0 : H;                        // start of the unreduced block
#pragma unroll
        for (int i = 1; i < H; ++i) {
          const bool cut = !(fabs(e[i - 1]) > tol);
          e[i - 1] = cut ? 0.0 : e[i - 1];
          lo = (cut && open) ? i : lo;
        }
        const double half = 0.5 * (d[H - 1] - d[H]);
        const double root = sqrt(fma(half, half, e[H - 1] * e[H - 1]));
        const double den = half + (half >= 0.0 ? root : -root);
        const double mu = fma(-e[H - 1] * e[H - 1], recip_nr(open ? den : 1.0), d[H]);
        double x = 1.0, z = 0.0;                      // the identity up to lo
#pragma unroll
        for (int k = 0; k < H; ++k) {
          const bool first = k == lo;
          x = first ? d[k] - mu : x;
          z = first ? e[k] : z;
          // z = 0 is the identity exactly: a lane that waits keeps its matrix bit for bit,
          // so its result does not depend on which elements share the wavefront
          const double r2 = fma(x, x, z * z);
          const bool turn = z != 0.0 && r2 > kTiny;
          const double ir = rsqrt_pos(fmax(r2, kTiny));
          const double c = turn ? x * ir : 1.0, s = turn ? z * ir : 0.0;
          if (k > 0) e[k - 1] = first ? 0.0 : (turn ? r2 * ir : x);
          const double ek = e[k], u = fma(d[k] - d[k + 1], s, -2.0 * c * ek);
          d[k] = fma(-s, u, d[k]);
          d[k + 1] = fma(s, u, d[k + 1]);
          e[k] = fma(-c, u, -ek);
          x = e[k];
          if (k + 1 < H) {
            z = s * e[k + 1];
            e[k + 1] *= c;
          }
#pragma unroll
          for (int i = 0; i < N; ++i) {
            const double v0 = V[i][k], v1 = V[i][k + 1];
            V[i][k] = fma(c, v0, s * v1);
            V[i][k + 1] = fma(c, v1, -s * v0);
          }
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < N; ++i) d[i] = __builtin_amdgcn_ldexp(d[i], ex);
}

// a = V diag(f(d)) V^T for the eigen-decomposition a = V diag(d) V^T of a packed upper
// triangle.
template <int N, typename F>
__device__ __forceinline__ void map_spectrum_packed(double (&a)[N * (N + 1) / 2], F f) {
  double d[N], V[N][N];
  sym_eigen_packed<N>(a, d, V);
#pragma unroll
  for (int i = 0; i < N; ++i) d[i] = f(d[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    double t[N];
#pragma unroll
    for (int k = 0; k < N; ++k) t[k] = V[i][k] * d[k];
#pragma unroll
    for (int j = i; j < N; ++j) {
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < N; ++k) acc = fma(t[k], V[j][k], acc);
      a[upper_index<N>(i, j)] = acc;
    }
  }
}

// The projection of hessianKernelHeader.pyx:143-252: negative eigenvalues become 0 (method
// 2) or their absolute value (method 1); and what it adds to the matrix.
template <int N>
__device__ __forceinline__ void clamp_spectrum_packed(double (&a)[N * (N + 1) / 2], uint32_t method) {
  map_spectrum_packed<N>(a, [=](double d) { return d < 0.0 ? (method == 1 ? -d : 0.0) : d; });
}
template <int N>
__device__ __forceinline__ void clamp_change_packed(double (&a)[N * (N + 1) / 2], uint32_t method) {
  map_spectrum_packed<N>(a, [=](double d) { return d < 0.0 ? (method == 1 ? -2.0 * d : -d) : 0.0; });
}

}  // namespace ysp
