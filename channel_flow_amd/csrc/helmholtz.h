// Host set-up of the diagonalised wall-normal solves: the collocation systems
// of omega_y (get_coef_omegay, PF:3432-3455) and v (get_coef_v, PF:3348-3381),
// folded by parity, as two matrices that every mode shares and a diagonal.
//
// With c = dt/(2 re) and the parity half degrees l_i = 2i + par (i < n), interior
// points p = 1 .. m (m = n - 1) and Q = [-1^T ; I] (functions that vanish at the
// walls), M0 = T0_I Q, M2 = T2_I Q, M0^-1 M2 = V diag(lam) V^-1, L = V^-1 M0^-1:
//
// omega_y: x = Q V diag(1 / sigma) L b with sigma = 1 + c (k^2 - lam).
//
// v: the operator is (1 + c k^2 - c D^2)(D^2 - k^2), so with phi = (D^2 - k^2) v
// (an exact polynomial) the rows p = 2 .. m are the omega_y-type collocation of
// phi = b psi + Q z, psi = T_par, with two unknowns per half system: the right-hand
// side a at p = 1, where v has no row, and the wall value b of phi.  In the
// eigenbasis, with y = L f (f = 0 at p = 1), l1 = L e_1 and q = lam * (L psi_I),
//     v = Q V x,  x_j = s_j (y_j + a l1_j - B q_j),  s_j = 1 / (sigma_j (lam_j - k^2)),
// B = c b, and the conditions v' = 0 and D^2 v = b at the wall are
//     w1 . x = 0,  w2 . x = B / c
// with w1, w2 the first and second wall derivatives of Q V: two dot products
// and a 2 x 2 system per mode.  The discrete solution is the one of the dense
// half system.
//
// The decomposition is computed in extended precision (the double eigenpairs,
// then first-order corrections V (I + X), X_ij = E_ij / (lam_j - lam_i) with
// E = V^-1 (G V - V diag(lam))) and rounded once.  With eigenpairs of double accuracy the v
// solve loses three to six digits against the dense inverses; with these it is
// one to three digits closer to the solution in extended precision than the
// dense double inverses are (N = 32 .. 256: 1e-16 .. 1e-14 against 1e-14 .. 2e-11).
#pragma once
#include <cmath>
#include <initializer_list>
#include <thread>
#include <vector>

#include "eig.h"

namespace chf {
namespace la {

using LD = long double;
using LMat = std::vector<LD>;

struct HelmholtzHalf {
  bool ok = false;  // decomposed: set last, so false where that failed or threw on the way
  int m = 0;
  std::vector<double> L, V;               // m x m, row-major
  std::vector<double> lam, w1, w2, l1, q;  // m
  LMat t0, t2, t4;                         // m x n: T_l and its derivatives at the interior points
};

// T_l(y_p) and its second and fourth derivatives at the half system's interior
// points, rows p = 1 .. m, columns l_i (the fourth as the second derivative of
// the expansion T_l'' = sum_k c_k T_k, c_k = l (l^2 - k^2) / (k == 0 ? 2 : 1)).
inline void half_points(int N, int par, HelmholtzHalf& h) {
  const int m = h.m, n = m + 1;
  const LD pi = std::acos(-1.0L);
  std::vector<LD> cs(2 * (size_t)N), sn(2 * (size_t)N);
  for (int k = 0; k < 2 * N; ++k) {
    cs[k] = std::cos(pi * k / N);
    sn[k] = std::sin(pi * k / N);
  }
  for (LMat* t : {&h.t0, &h.t2, &h.t4}) t->assign((size_t)m * n, 0.0L);
  for (int r = 0; r < m; ++r) {
    const int p = r + 1;
    const LD c1 = cs[p], s1 = sn[p], is3 = 1.0L / (s1 * s1 * s1);
    LD sum = 0.0L, sumk = 0.0L;  // of T_k''/e_k and k^2 T_k''/e_k over the lower degrees (e_0 = 2, else 1)
    for (int i = 0; i < n; ++i) {
      const LD l = 2 * i + par;
      const size_t a = (size_t)((long)p * (2 * i + par) % (2L * N)), o = (size_t)r * n + i;
      h.t0[o] = cs[a];
      h.t2[o] = l * (sn[a] * c1 - l * cs[a] * s1) * is3;
      h.t4[o] = l * (l * l * sum - sumk);
      const LD e = l == 0.0L ? 2.0L : 1.0L;
      sum += h.t2[o] / e;
      sumk += l * l * h.t2[o] / e;
    }
  }
}

// a b (m x m) in extended precision: dot products, four columns at a time (the
// accumulators stay in registers; x87 stores are what the row form waits for), the
// rows of large ones by several threads (m = 96, the decomposition's products are
// 7 of its 13 ms in one; below 80 the threads cost what they save).
inline LMat lmul(const LMat& a, const LMat& b, int m) {
  LMat bt((size_t)m * m), c((size_t)m * m);
  for (int i = 0; i < m; ++i)
    for (int j = 0; j < m; ++j) bt[(size_t)j * m + i] = b[(size_t)i * m + j];
  auto rows = [&](int i0, int i1) {
    for (int i = i0; i < i1; ++i) {
      const LD* x = &a[(size_t)i * m];
      int j = 0;
      for (; j + 4 <= m; j += 4) {
        const LD *y0 = &bt[(size_t)j * m], *y1 = y0 + m, *y2 = y1 + m, *y3 = y2 + m;
        LD s0 = 0, s1 = 0, s2 = 0, s3 = 0;
        for (int k = 0; k < m; ++k) {
          const LD f = x[k];
          s0 += f * y0[k];
          s1 += f * y1[k];
          s2 += f * y2[k];
          s3 += f * y3[k];
        }
        LD* o = &c[(size_t)i * m + j];
        o[0] = s0; o[1] = s1; o[2] = s2; o[3] = s3;
      }
      for (; j < m; ++j) {
        LD s0 = 0;
        for (int k = 0; k < m; ++k) s0 += x[k] * bt[(size_t)j * m + k];
        c[(size_t)i * m + j] = s0;
      }
    }
  };
  constexpr int kThreads = 4;
  std::thread others[kThreads - 1];
  int done = 0;  // rows handed out
  if (m >= 80)
    for (std::thread& t : others) {
      try {
        t = std::thread(rows, done, done + m / kThreads);
      } catch (...) {
        break;  // the rest of the rows is done here
      }
      done += m / kThreads;
    }
  rows(done, m);
  for (std::thread& t : others)
    if (t.joinable()) t.join();
  return c;
}

// Inverse in extended precision: the double inverse Z and one Newton step,
// Z + Z (I - A Z) with the residual in extended precision (the correction is
// small, so its product may be in double).
inline bool linverse(const LMat& A, int m, LMat& out) {
  Mat Z;
  if (!inverse(Mat(A.begin(), A.end()), m, Z)) return false;
  out.assign(Z.begin(), Z.end());
  const LMat AZ = lmul(A, out, m);
  Mat R((size_t)m * m);
  for (int i = 0; i < m; ++i)
    for (int j = 0; j < m; ++j) R[(size_t)i * m + j] = (double)((i == j ? 1.0L : 0.0L) - AZ[(size_t)i * m + j]);
  const Mat C = matmul(Z, R, m, m, m);
  for (size_t i = 0; i < out.size(); ++i) {
    out[i] += C[i];
    if (!(std::fabs(R[i]) < 1e-7)) return false;  // its square is what is left
  }
  return true;
}

// The decomposition of one parity half system of degree N; false when the
// eigenvalues are not real, negative and distinct or the corrections do not
// converge.
inline bool helmholtz_half(int N, int par, HelmholtzHalf& out) {
  const int n = par ? (N + 1) / 2 : N / 2 + 1, m = n - 1;
  if (m < 1) return false;
  out.ok = false;
  out.m = m;
  half_points(N, par, out);
  LMat M0((size_t)m * m), M2((size_t)m * m), M0i;
  for (int r = 0; r < m; ++r)
    for (int k = 0; k < m; ++k) {
      M0[(size_t)r * m + k] = out.t0[(size_t)r * n + k + 1] - out.t0[(size_t)r * n];
      M2[(size_t)r * m + k] = out.t2[(size_t)r * n + k + 1] - out.t2[(size_t)r * n];
    }
  if (!linverse(M0, m, M0i)) return false;
  const LMat G = lmul(M0i, M2, m);
  std::vector<double> ev;
  Mat Vd, Vid;
  if (!eig_real(Mat(G.begin(), G.end()), m, ev, Vd)) return false;
  LMat V(Vd.begin(), Vd.end()), lam(ev.begin(), ev.end());
  bool converged = false;
  for (int it = 0; it < 6 && !converged; ++it) {
    // E = V^-1 (G V - V diag(lam)): the residual in extended precision is
    // small, so double serves for the rest of the correction
    const LMat GV = lmul(G, V, m);
    Mat W((size_t)m * m), X((size_t)m * m, 0.0);
    for (int i = 0; i < m; ++i)
      for (int j = 0; j < m; ++j) {
        const size_t o = (size_t)i * m + j;
        W[o] = (double)(GV[o] - V[o] * lam[j]);
        Vd[o] = (double)V[o];
      }
    if (!inverse(Vd, m, Vid)) return false;
    const Mat E = matmul(Vid, W, m, m, m);
    double big = 0.0;
    for (int i = 0; i < m; ++i)
      for (int j = 0; j < m; ++j) {
        if (i == j) continue;
        const double x = E[(size_t)i * m + j] / (double)(lam[j] - lam[i]);
        if (!std::isfinite(x)) return false;
        X[(size_t)i * m + j] = x;
        big = std::max(big, std::fabs(x));
      }
    for (int j = 0; j < m; ++j) {
      lam[j] += E[(size_t)j * m + j];
      for (int k = 0; k < m; ++k)  // second order, lest large lam_k disturb small lam_j
        if (k != j) lam[j] += E[(size_t)j * m + k] * X[(size_t)k * m + j];
    }
    const Mat C = matmul(Vd, X, m, m, m);
    for (size_t i = 0; i < V.size(); ++i) V[i] += C[i];
    converged = big < 1e-9;  // what is left is of the order of its square
  }
  LMat Vi;
  if (!converged || !linverse(V, m, Vi)) return false;
  const LMat L = lmul(Vi, M0i, m);
  out.L.assign(L.begin(), L.end());
  out.V.assign(V.begin(), V.end());
  out.lam.assign(lam.begin(), lam.end());
  out.w1.assign(m, 0.0);
  out.w2.assign(m, 0.0);
  out.l1.assign(m, 0.0);
  out.q.assign(m, 0.0);
  auto d1 = [](LD l) { return l * l; };
  auto d2 = [](LD l) { return l * l * (l * l - 1.0L) / 3.0L; };
  for (int j = 0; j < m; ++j) {
    if (!(lam[j] < 0.0L)) return false;  // the Dirichlet second derivative's spectrum
    LD w1 = 0.0L, w2 = 0.0L, ps = 0.0L;
    for (int r = 0; r < m; ++r) {
      const LD l = 2 * (r + 1) + par, v = V[(size_t)r * m + j];
      w1 += (d1(l) - d1((LD)par)) * v;
      w2 += (d2(l) - d2((LD)par)) * v;
      ps += L[(size_t)j * m + r] * out.t0[(size_t)r * n];
    }
    out.w1[j] = (double)w1;
    out.w2[j] = (double)w2;
    out.l1[j] = (double)L[(size_t)j * m];
    out.q[j] = (double)(lam[j] * ps);
  }
  out.ok = true;
  return true;
}

// The two wall conditions of the v solve for one k^2: the matrix that maps
// (d1, d2) = (w1 . s y, w2 . s y) to (a, B), row-major.
inline void wall_matrix(const HelmholtzHalf& h, double c, double k2, double out[4]) {
  double m11 = 0, m12 = 0, m21 = 0, m22 = -1.0 / c;
  for (int j = 0; j < h.m; ++j) {
    const double s = 1.0 / ((1.0 + c * (k2 - h.lam[j])) * (h.lam[j] - k2));
    m11 += h.w1[j] * s * h.l1[j];
    m12 -= h.w1[j] * s * h.q[j];
    m21 += h.w2[j] * s * h.l1[j];
    m22 -= h.w2[j] * s * h.q[j];
  }
  const double det = m11 * m22 - m12 * m21;
  out[0] = -m22 / det;
  out[1] = m12 / det;
  out[2] = m21 / det;
  out[3] = -m11 / det;
}

// One solve of a half system as the kernels do it: v (rows f of p = 2 .. m, f[0]
// unused) or omega_y (rows of p = 1 .. m) for one k^2, into x[n].
inline void helmholtz_solve(const HelmholtzHalf& h, bool is_v, double c, double k2, const double* f, double* x) {
  const int m = h.m;
  std::vector<double> y(m, 0.0);
  double d1 = 0, d2 = 0;
  for (int j = 0; j < m; ++j) {
    double t = 0;
    for (int r = is_v ? 1 : 0; r < m; ++r) t += h.L[(size_t)j * m + r] * f[r];
    const double sg = 1.0 + c * (k2 - h.lam[j]);
    y[j] = is_v ? t / (sg * (h.lam[j] - k2)) : t / sg;
    d1 += h.w1[j] * y[j];
    d2 += h.w2[j] * y[j];
  }
  if (is_v) {
    double w[4];
    wall_matrix(h, c, k2, w);
    const double a = w[0] * d1 + w[1] * d2, b = w[2] * d1 + w[3] * d2;
    for (int j = 0; j < m; ++j)
      y[j] += (a * h.l1[j] - b * h.q[j]) / ((1.0 + c * (k2 - h.lam[j])) * (h.lam[j] - k2));
  }
  x[0] = 0;
  for (int r = 0; r < m; ++r) {
    double t = 0;
    for (int j = 0; j < m; ++j) t += h.V[(size_t)r * m + j] * y[j];
    x[r + 1] = t;
    x[0] -= t;
  }
}

// Whether the decomposition reproduces direct solves of the half systems at
// one k^2 (v for k^2 > 0 only) to 1e-12 of the solution.  The direct solution is
// the double LU's, refined with residuals in extended precision.  The bar has a
// factor of ten: every degree from 4 to 256 comes within 1e-13, where the
// refinement stops, for c from 1e-15 to 1e5 and k^2 to 1e8.
inline bool helmholtz_verify(int par, const HelmholtzHalf& h, double c, double k2) {
  if (!h.ok) return false;
  const int m = h.m, n = m + 1;
  for (int is_v = 0; is_v < (k2 > 0.0 ? 2 : 1); ++is_v) {
    const int nbc = is_v ? 2 : 1;  // wall rows, then the points p >= nbc
    if (n <= nbc) continue;        // no interior row
    LMat A((size_t)n * n, 0.0L), ref(n, 0.0L);
    std::vector<double> f(m, 0.0), x(n, 0.0);
    for (int i = 0; i < n; ++i) {
      const LD l = 2 * i + par;
      A[i] = 1.0L;
      if (is_v) A[(size_t)n + i] = l * l;
      for (int r = nbc - 1; r < m; ++r) {
        const size_t o = (size_t)r * n + i;
        A[(size_t)(r + 1) * n + i] =
            is_v ? -c * h.t4[o] + (1.0L + 2.0L * c * k2) * h.t2[o] - k2 * (1.0L + (LD)c * k2) * h.t0[o]
                 : -c * h.t2[o] + (1.0L + (LD)c * k2) * h.t0[o];
      }
    }
    for (int r = nbc - 1; r < m; ++r) f[r] = std::sin(1.7 * r + 0.3) + 0.1 * r / m;
    Mat lu_(A.begin(), A.end());
    std::vector<int> piv;
    if (!lu(lu_, piv, n)) return false;
    LD step = 0.0L, size = 0.0L;
    for (int it = 0; it < 8; ++it) {
      Mat res(n);
      for (int i = 0; i < n; ++i) {
        LD t = i >= nbc ? (LD)f[i - 1] : 0.0L;
        for (int j = 0; j < n; ++j) t -= A[(size_t)i * n + j] * ref[j];
        res[i] = (double)t;
      }
      lu_solve(lu_, piv, n, res, 1);
      step = size = 0.0L;
      for (int i = 0; i < n; ++i) {
        ref[i] += res[i];
        step = std::max(step, std::fabs((LD)res[i]));
        size = std::max(size, std::fabs(ref[i]));
      }
      if (step <= 1e-13L * size) break;
    }
    helmholtz_solve(h, is_v != 0, c, k2, f.data(), x.data());
    LD err = step;  // not refined to the end: no better than the last correction
    for (int i = 0; i < n; ++i) err = std::max(err, std::fabs((LD)x[i] - ref[i]));
    if (!(err <= 1e-12L * size)) return false;
  }
  return true;
}

// Whether a half system is decomposed (here, unless `h` is already) and
// reproduces direct solves at each k^2; false, not an exception, without memory.
inline bool helmholtz_accept(int N, int par, HelmholtzHalf& h, double c, std::initializer_list<double> k2s) noexcept {
  try {
    if (!h.ok && !helmholtz_half(N, par, h)) return false;
    for (double k2 : k2s)
      if (!helmholtz_verify(par, h, c, k2)) return false;
    return true;
  } catch (...) {
    return false;
  }
}

}  // namespace la
}  // namespace chf
