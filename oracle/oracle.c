/* CPU restatement of the reference ADER-WENO solver.  TEST INFRASTRUCTURE ONLY:
 * see oracle.h.  Reference file:line citations are relative to the reference
 * tree (haranjackson/PyPDE).
 *
 * Operation-order conventions shared with the HIP kernels:
 *   - dot products:  acc = a[0]*b[0]; acc = fma(a[j], b[j], acc) for j = 1..;
 *   - every other expression is evaluated as written (-ffp-contract=off);
 *   - tables are computed in long double and rounded once to double.
 */
#include "oracle.h"

#include <float.h>
#include <math.h>
#include <stdlib.h>
#include <string.h>

#define MAXN 6
#define MAXV 17
#define MAXD 3
#define MAXND 216 /* MAXN^MAXD */
#define HOUSE_TINY 0x1p-900
#define NEWTON_A_TINY 1e-6 /* max |dt dS/dQ| below which the stiff step drops A */

/* Constants of the reference: types.h:18, weno.h:8-10, dg.h:8-9,
 * NumericalDiff.h:9. */
static const double WENO_LAMS = 1.0, WENO_LAMC = 1e5, WENO_EPS = 1e-14;
static const int DG_IT = 50;
static const double DG_TOL = 6e-6;
static const double FD_EPS = 1.4901161193847656e-08; /* sqrt(2^-52) */

/* ------------------------------------------------------------------ tables */

typedef long double ld;

/* Gauss-Legendre nodes/weights on [-1,1] by Newton iteration on P_N from
 * Chebyshev-like starting points; the reference gets the same quantities from
 * the companion-matrix eigenvalues plus one Newton step (legendre.cpp:136-197).
 * Returned ascending, mapped to [0,1] (basis.cpp:7-20). */
static void gl_nodes(int n, ld *x, ld *w) {
  for (int i = 0; i < n; i++) {
    ld z = cosl(3.14159265358979323846264338327950288L * ((ld)i + 0.75L) /
                ((ld)n + 0.5L));
    ld dp = 1.0L;
    for (int it = 0; it < 100; it++) {
      ld p0 = 1.0L, p1 = z;
      for (int k = 2; k <= n; k++) {
        ld p2 = ((ld)(2 * k - 1) * z * p1 - (ld)(k - 1) * p0) / (ld)k;
        p0 = p1;
        p1 = p2;
      }
      if (n == 1) p0 = 1.0L;
      dp = (ld)n * (z * p1 - p0) / (z * z - 1.0L);
      ld z1 = z;
      z = z1 - p1 / dp;
      if (fabsl(z - z1) <= 4.0L * LDBL_EPSILON) break;
    }
    {
      ld p0 = 1.0L, p1 = z;
      for (int k = 2; k <= n; k++) {
        ld p2 = ((ld)(2 * k - 1) * z * p1 - (ld)(k - 1) * p0) / (ld)k;
        p0 = p1;
        p1 = p2;
      }
      if (n == 1) p0 = 1.0L;
      dp = (ld)n * (z * p1 - p0) / (z * z - 1.0L);
    }
    x[n - 1 - i] = (1.0L + z) / 2.0L;
    w[n - 1 - i] = 1.0L / ((1.0L - z * z) * dp * dp);
  }
}

/* Power-basis coefficients of the Lagrange polynomials at the nodes
 * (basis.cpp:22-53): c[j][k] is the s^k coefficient of psi_j. */
static void lagrange_coeffs(int n, const ld *x, ld c[MAXN][MAXN]) {
  for (int j = 0; j < n; j++) {
    ld p[MAXN];
    for (int k = 0; k < n; k++) p[k] = 0.0L;
    p[0] = 1.0L;
    int deg = 0;
    for (int m = 0; m < n; m++) {
      if (m == j) continue;
      ld den = x[j] - x[m];
      for (int k = deg + 1; k >= 1; k--) p[k] = (p[k - 1] - x[m] * p[k]) / den;
      p[0] = (-x[m] * p[0]) / den;
      deg++;
    }
    for (int k = 0; k < n; k++) c[j][k] = p[k];
  }
}

static ld poly_eval(const ld *c, int len, ld s) {
  ld r = 0.0L;
  for (int k = len - 1; k >= 0; k--) r = r * s + c[k];
  return r;
}

/* Antiderivative integral of psi_j over [a, a+1]. */
static ld poly_int(const ld *c, int n, ld a) {
  ld P[MAXN + 1];
  P[0] = 0.0L;
  for (int k = 0; k < n; k++) P[k + 1] = c[k] / (ld)(k + 1);
  return poly_eval(P, n + 1, a + 1.0L) - poly_eval(P, n + 1, a);
}

/* Gauss-Jordan inverse with partial pivoting. */
static int ld_inverse(int n, ld A[MAXN][MAXN], ld R[MAXN][MAXN]) {
  ld M[MAXN][2 * MAXN];
  for (int i = 0; i < n; i++)
    for (int j = 0; j < 2 * n; j++)
      M[i][j] = j < n ? A[i][j] : (ld)(j - n == i);
  for (int k = 0; k < n; k++) {
    int p = k;
    for (int i = k + 1; i < n; i++)
      if (fabsl(M[i][k]) > fabsl(M[p][k])) p = i;
    if (M[p][k] == 0.0L) return -1;
    if (p != k)
      for (int j = 0; j < 2 * n; j++) {
        ld t = M[k][j];
        M[k][j] = M[p][j];
        M[p][j] = t;
      }
    ld piv = M[k][k];
    for (int j = 0; j < 2 * n; j++) M[k][j] /= piv;
    for (int i = 0; i < n; i++) {
      if (i == k) continue;
      ld f = M[i][k];
      for (int j = 0; j < 2 * n; j++) M[i][j] -= f * M[k][j];
    }
  }
  for (int i = 0; i < n; i++)
    for (int j = 0; j < n; j++) R[i][j] = M[i][n + j];
  return 0;
}

typedef struct {
  int N, D, V, Nd, Nd1, NT; /* N, ndim, nvar, N^D, N^(D-1), N^(D+1) */
  double x[MAXN], w[MAXN], end0[MAXN], end1[MAXN], der[MAXN][MAXN];
  double wmat[4][MAXN][MAXN], winv[4][MAXN][MAXN], sig[MAXN][MAXN];
  double dgmat[MAXN][MAXN], dginv[MAXN][MAXN];
  double flc[MAXN], flm[MAXN][MAXN][MAXN]; /* flm[k-1] = M_k */
  int nsten, soff[4];
  double slam[4];
  /* per-node tables (node idx = row-major multi-index k_0..k_{D-1}) */
  int kk[MAXND][MAXD];
  double WP[MAXND];  /* prod_d W[k_d]                      (stepper.cpp:31-40) */
  double IWP[MAXND]; /* 1 / WP */
} Tab;

int oracle_tables(int N, double *nodes, double *wghts, double *endvals,
                  double *dervals, double *weno_mat, double *weno_inv,
                  double *sig, double *dgmat, double *dginv, double *fl_c,
                  double *fl_m) {
  if (N < 1 || N > MAXN) return 1;
  int n = N;
  ld x[MAXN], w[MAXN], c[MAXN][MAXN];
  gl_nodes(n, x, w);
  lagrange_coeffs(n, x, c);
  if (nodes)
    for (int i = 0; i < n; i++) nodes[i] = (double)x[i];
  if (wghts)
    for (int i = 0; i < n; i++) wghts[i] = (double)w[i];
  /* ENDVALS[e][j] = psi_j(e) (basis.cpp:55-65) */
  ld e0[MAXN], e1[MAXN];
  for (int j = 0; j < n; j++) {
    e0[j] = poly_eval(c[j], n, 0.0L);
    e1[j] = poly_eval(c[j], n, 1.0L);
    if (endvals) {
      endvals[j] = (double)e0[j];
      endvals[n + j] = (double)e1[j];
    }
  }
  /* derivative coefficients */
  ld dc[MAXN][MAXN];
  for (int j = 0; j < n; j++) {
    for (int k = 0; k < n; k++) dc[j][k] = 0.0L;
    for (int k = 1; k < n; k++) dc[j][k - 1] = c[j][k] * (ld)k;
  }
  /* DERVALS[i][j] = psi_j'(x_i) (basis.cpp:67-76) */
  if (dervals)
    for (int i = 0; i < n; i++)
      for (int j = 0; j < n; j++)
        dervals[i * n + j] = (double)poly_eval(dc[j], n, x[i]);
  /* WENO stencil matrices (weno_matrices.cpp:8-33) and their inverses */
  int FN2 = (n - 1) / 2, CN2 = n / 2;
  int off[4] = {-(n - 1), 0, -CN2, -FN2};
  for (int s = 0; s < 4; s++) {
    ld A[MAXN][MAXN], R[MAXN][MAXN];
    for (int i = 0; i < n; i++)
      for (int j = 0; j < n; j++) A[i][j] = poly_int(c[j], n, (ld)(i + off[s]));
    if (ld_inverse(n, A, R)) return 2;
    for (int i = 0; i < n; i++)
      for (int j = 0; j < n; j++) {
        if (weno_mat) weno_mat[(s * n + i) * n + j] = (double)A[i][j];
        if (weno_inv) weno_inv[(s * n + i) * n + j] = (double)R[i][j];
      }
  }
  /* SIG[i][j] = sum_{a=1}^{n-1} int_0^1 psi_i^(a) psi_j^(a) (weno_matrices.cpp:36-51) */
  if (sig) {
    ld S[MAXN][MAXN];
    for (int i = 0; i < n; i++)
      for (int j = 0; j < n; j++) S[i][j] = 0.0L;
    ld di[MAXN][MAXN];
    for (int j = 0; j < n; j++)
      for (int k = 0; k < n; k++) di[j][k] = c[j][k];
    for (int a = 1; a < n; a++) {
      for (int j = 0; j < n; j++) {
        for (int k = 1; k < n; k++) di[j][k - 1] = di[j][k] * (ld)k;
        di[j][n - 1] = 0.0L;
      }
      for (int i = 0; i < n; i++)
        for (int j = 0; j < n; j++) {
          ld acc = 0.0L;
          for (int p = 0; p < n; p++)
            for (int q = 0; q < n; q++)
              acc += di[i][p] * di[j][q] / (ld)(p + q + 1);
          S[i][j] += acc;
        }
    }
    for (int i = 0; i < n; i++)
      for (int j = 0; j < n; j++) sig[i * n + j] = (double)S[i][j];
  }
  /* DG_MAT[i][j] = psi_i(1) psi_j(1) - int_0^1 psi_i' psi_j
   * (dg.cpp:38-40 with dg_matrices.cpp:28-55, the quadrature being exact) */
  ld G[MAXN][MAXN], GI[MAXN][MAXN];
  for (int i = 0; i < n; i++)
    for (int j = 0; j < n; j++) {
      ld acc = 0.0L;
      for (int p = 0; p < n; p++)
        for (int q = 0; q < n; q++) acc += dc[i][p] * c[j][q] / (ld)(p + q + 1);
      G[i][j] = e1[i] * e1[j] - acc;
    }
  if (ld_inverse(n, G, GI)) return 3;
  for (int i = 0; i < n; i++)
    for (int j = 0; j < n; j++) {
      if (dgmat) dgmat[i * n + j] = (double)G[i][j];
      if (dginv) dginv[i * n + j] = (double)GI[i][j];
    }
  /* Faddeev-LeVerrier on Tw = diag(1/W) DG_MAT: det(xI - Tw) = x^n + sum c_k x^k,
   * adj(xI - Tw) = sum_{k=1}^{n} M_k x^{n-k}.  Used by the stiff predictor's
   * Newton solve (a per-node Newton; the reference uses Newton-Krylov,
   * newton_krylov.cpp:144-183). */
  {
    ld T[MAXN][MAXN], Mk[MAXN][MAXN], TM[MAXN][MAXN], cc[MAXN + 1];
    for (int i = 0; i < n; i++)
      for (int j = 0; j < n; j++) T[i][j] = G[i][j] / w[i];
    for (int i = 0; i < n; i++)
      for (int j = 0; j < n; j++) Mk[i][j] = (ld)(i == j);
    cc[n] = 1.0L;
    for (int k = 1; k <= n; k++) {
      if (k > 1) {
        for (int i = 0; i < n; i++)
          for (int j = 0; j < n; j++) Mk[i][j] = TM[i][j] + (i == j ? cc[n - k + 1] : 0.0L);
      }
      for (int i = 0; i < n; i++)
        for (int j = 0; j < n; j++) {
          ld acc = 0.0L;
          for (int p = 0; p < n; p++) acc += T[i][p] * Mk[p][j];
          TM[i][j] = acc;
        }
      ld tr = 0.0L;
      for (int i = 0; i < n; i++) tr += TM[i][i];
      cc[n - k] = -tr / (ld)k;
      if (fl_m)
        for (int i = 0; i < n; i++)
          for (int j = 0; j < n; j++)
            fl_m[((k - 1) * n + i) * n + j] = (double)Mk[i][j];
    }
    if (fl_c)
      for (int k = 0; k < n; k++) fl_c[k] = (double)cc[k];
  }
  return 0;
}

static int tab_init(Tab *T, int N, int D, int V) {
  if (N < 1 || N > MAXN || D < 1 || D > MAXD || V < 1 || V > MAXV) return 1;
  memset(T, 0, sizeof(*T));
  T->N = N;
  T->D = D;
  T->V = V;
  T->Nd = 1;
  for (int d = 0; d < D; d++) T->Nd *= N;
  if (T->Nd > MAXND) return 1;
  T->Nd1 = T->Nd / N;
  T->NT = T->Nd * N;
  double endv[2 * MAXN], derv[MAXN * MAXN], wm[4 * MAXN * MAXN],
      wi[4 * MAXN * MAXN], sg[MAXN * MAXN], dg[MAXN * MAXN], dgi[MAXN * MAXN],
      flc[MAXN], flm[MAXN * MAXN * MAXN];
  if (oracle_tables(N, T->x, T->w, endv, derv, wm, wi, sg, dg, dgi, flc, flm))
    return 2;
  for (int i = 0; i < N; i++) {
    T->end0[i] = endv[i];
    T->end1[i] = endv[N + i];
    T->flc[i] = flc[i];
    for (int j = 0; j < N; j++) {
      T->der[i][j] = derv[i * N + j];
      T->sig[i][j] = sg[i * N + j];
      T->dgmat[i][j] = dg[i * N + j];
      T->dginv[i][j] = dgi[i * N + j];
      for (int s = 0; s < 4; s++) {
        T->wmat[s][i][j] = wm[(s * N + i) * N + j];
        T->winv[s][i][j] = wi[(s * N + i) * N + j];
      }
      for (int k = 0; k < N; k++) T->flm[k][i][j] = flm[(k * N + i) * N + j];
    }
  }
  /* stencils in the reference's order (weno.cpp:47-55) */
  int FN2 = (N - 1) / 2, CN2 = N / 2;
  T->nsten = 2;
  T->soff[0] = 0;
  T->slam[0] = WENO_LAMS;
  T->soff[1] = N - 1;
  T->slam[1] = WENO_LAMS;
  if (N > 2) {
    T->soff[2] = FN2;
    T->slam[2] = WENO_LAMC;
    T->nsten = 3;
    if (N % 2 == 0) {
      T->soff[3] = CN2;
      T->slam[3] = WENO_LAMC;
      T->nsten = 4;
    }
  }
  for (int idx = 0; idx < T->Nd; idx++) {
    int r = idx;
    for (int d = D - 1; d >= 0; d--) {
      T->kk[idx][d] = r % N;
      r /= N;
    }
    double p = T->w[T->kk[idx][0]];
    for (int d = 1; d < D; d++) p = p * T->w[T->kk[idx][d]];
    T->WP[idx] = p;
    T->IWP[idx] = 1.0 / p;
  }
  return 0;
}

/* ---------------------------------------------------------------- helpers */

static int ipow(int b, int e) {
  int r = 1;
  for (int i = 0; i < e; i++) r *= b;
  return r;
}

/* Derivative along axis d at node idx of a nodal tensor q (Nd x V rows):
 * DERVALS row k_d against the line through idx, then / dX[d]
 * (evaluations.cpp:23-47), as a product with rdx = 1 / dX[d]. */
static void node_deriv(const Tab *T, const double *q, int idx, int d,
                       double rdx, double *out) {
  int N = T->N, V = T->V;
  int stride = ipow(N, T->D - 1 - d);
  int kd = T->kk[idx][d];
  int base = idx - kd * stride;
  for (int v = 0; v < V; v++) {
    double acc = T->der[kd][0] * q[base * V + v];
    for (int j = 1; j < N; j++)
      acc = fma(T->der[kd][j], q[(base + j * stride) * V + v], acc);
    out[v] = acc * rdx;
  }
}

/* ---------------------------------------------------------- eigenvalues */

/* Householder reflector for x[0..m-1] (Golub & Van Loan, Alg. 5.1.1, with v
 * left unnormalised): P x = mu e_1, P = I - beta v v^T, v = (v0, x[1..m-1]),
 * beta = 2 / (v^T v).  Two divisions per reflector instead of m + 1.  Columns
 * whose tail is below 2^-900 in square norm are treated as already reduced
 * (the matrix is scaled to entries <= 1 first), which keeps beta finite. */
static double house(const double *x, int m, double *v) {
  double sigma = 0.0;
  for (int i = 1; i < m; i++) sigma = fma(x[i], x[i], sigma);
  if (sigma <= HOUSE_TINY) {
    v[0] = 1.0;
    for (int i = 1; i < m; i++) v[i] = 0.0;
    return 0.0;
  }
  double mu = sqrt(fma(x[0], x[0], sigma));
  double v0 = (x[0] <= 0.0) ? x[0] - mu : -sigma / (x[0] + mu);
  v[0] = v0;
  for (int i = 1; i < m; i++) v[i] = x[i];
  return 2.0 / fma(v0, v0, sigma);
}

/* The same reflector with one division, for the Hessenberg reduction of a
 * matrix scaled to entries <= 1: v^T v = 2 mu (mu - x0), so beta = 1 / (mu (mu
 * - x0)) when x0 <= 0 (v0 = x0 - mu); when x0 > 0 (v0 = -sigma / (x0 + mu))
 * beta = (x0 + mu) / (mu sigma), both quotients from r = 1 / ((x0 + mu) mu
 * sigma); *mu_out = mu (P x = mu e_1).  A tail below 2^-500 in square norm
 * counts as reduced, which keeps the product above 2^-1000. */
#define HOUSE1_TINY 0x1p-500
static double house1(const double *x, int m, double *v, double *mu_out) {
  double sigma = 0.0;
  for (int i = 1; i < m; i++) sigma = fma(x[i], x[i], sigma);
  if (sigma <= HOUSE1_TINY) {
    v[0] = 1.0;
    for (int i = 1; i < m; i++) v[i] = 0.0;
    return 0.0;
  }
  double mu = sqrt(fma(x[0], x[0], sigma));
  *mu_out = mu;
  int pos = x[0] > 0.0;
  double s = x[0] + mu;
  double r = 1.0 / (pos ? (s * mu) * sigma : mu * (mu - x[0]));
  v[0] = pos ? -sigma * ((r * mu) * sigma) : x[0] - mu;
  for (int i = 1; i < m; i++) v[i] = x[i];
  return pos ? s * (r * s) : r;
}

/* rows r0..r0+m-1, columns c0..c1: H = P H */
static void house_left(double *H, int n, const double *v, int m, double beta,
                       int r0, int c0, int c1) {
  for (int j = c0; j <= c1; j++) {
    double s = v[0] * H[r0 * n + j];
    for (int i = 1; i < m; i++) s = fma(v[i], H[(r0 + i) * n + j], s);
    s = beta * s;
    for (int i = 0; i < m; i++) H[(r0 + i) * n + j] = fma(-s, v[i], H[(r0 + i) * n + j]);
  }
}

/* rows r0..r1, columns c0..c0+m-1: H = H P */
static void house_right(double *H, int n, const double *v, int m, double beta,
                        int r0, int r1, int c0) {
  for (int i = r0; i <= r1; i++) {
    double s = v[0] * H[i * n + c0];
    for (int j = 1; j < m; j++) s = fma(v[j], H[i * n + c0 + j], s);
    s = beta * s;
    for (int j = 0; j < m; j++) H[i * n + c0 + j] = fma(-s, v[j], H[i * n + c0 + j]);
  }
}

/* Characteristic polynomial p(x) = det(xI - H) of an upper Hessenberg H
 * (n <= MAXV), monic, coefficients c[0..n]: leading principal minors expanded
 * along their last column,
 *   D_k = (x - h_kk) D_k-1 - sum_{m=1}^{k-1} h_{k-m,k} (prod_{j=k-m+1}^{k} h_{j,j-1}) D_{k-m-1}
 * (1-based; Wilkinson, The Algebraic Eigenvalue Problem, ch. 7). */
static void hess_charpoly(const double *H, int n, double *c) {
  double D[MAXV + 1][MAXV + 1];
  D[0][0] = 1.0;
  for (int k = 1; k <= n; k++) {
    double hkk = H[(k - 1) * n + (k - 1)];
    for (int i = 0; i <= k; i++) {
      double v = (i >= 1) ? D[k - 1][i - 1] : 0.0;
      if (i <= k - 1) v = fma(-hkk, D[k - 1][i], v);
      D[k][i] = v;
    }
    double prod = 1.0;
    for (int m = 1; m <= k - 1; m++) {
      /* prod = h_{k,k-1} h_{k-1,k-2} ... h_{k-m+1,k-m} (1-based) */
      prod = prod * H[(k - m) * n + (k - m - 1)];
      double t = H[(k - m - 1) * n + (k - 1)] * prod;
      for (int i = 0; i <= k - m - 1; i++) D[k][i] = fma(-t, D[k - m - 1][i], D[k][i]);
    }
  }
  for (int i = 0; i <= n; i++) c[i] = D[n][i];
}

/* One real root of the monic degree-n polynomial c (n >= 2) from x0, by
 * Halley's method for n <= 5 and by Laguerre's method above (both converge
 * cubically at simple roots and, from above the largest real root of a
 * real-rooted polynomial, decrease monotonically onto it; Halley's step needs
 * no square root, Laguerre's lands near the roots at once from a start far
 * outside them).  Halley: p p' / (p'^2 - p p''/2).  Laguerre: n / (G +-
 * sqrt((n-1)(n H - G^2))), G = p'/p, H = G^2 - p''/p, evaluated multiplied
 * through by p: n p / (p' +- sqrt((n-1)((n-1) p'^2 - n p p''))).  f = p''/2
 * comes from the fused Horner recurrence, whose first two steps are written
 * out (exact for c[n] = 1 and finite x).  Converged: |step| <= 4 eps |x|, or
 * |step| <= 1e-8 |x| with |step| |x| <= |previous step|^2 (superlinear
 * convergence seen: the remaining error is below |step|^2.5).  *dp receives
 * p' where p was last evaluated.  Returns 0 when it does not converge in
 * LAG_IT steps. */
#define LAG_IT 40
static int real_root(const double *c, int n, double x0, double *root, double *dp) {
  double x = x0, prev = 0.0;
  for (int it = 0; it < LAG_IT; it++) {
    double b1 = x + c[n - 1];
    double f = 1.0, d = x + b1, b = fma(x, b1, c[n - 2]);
    for (int j = n - 3; j >= 0; j--) {
      f = fma(x, f, d);
      d = fma(x, d, b);
      b = fma(x, b, c[j]);
    }
    *dp = d;
    if (b == 0.0) {
      *root = x;
      return 1;
    }
    double num, den;
    if (n <= 5) {
      num = b * d;
      den = fma(d, d, -(b * f));
    } else {
      double r = (double)(n - 1) * ((double)(n - 1) * (d * d) - (double)(2 * n) * (f * b));
      double sq = r > 0.0 ? sqrt(r) : 0.0;
      num = (double)n * b;
      den = (d >= 0.0) ? d + sq : d - sq;
    }
    if (!(den != 0.0)) return 0;
    double step = num / den;
    x = x - step;
    double as = fabs(step), ax = fabs(x);
    if (!(as > 4.0 * DBL_EPSILON * ax) || as <= DBL_MIN ||
        (as <= 1e-8 * ax && as * ax <= prev * prev)) {
      *root = x;
      return ax <= 1e300; /* finite */
    }
    prev = as;
  }
  return 0;
}

/* max |lambda| of an upper Hessenberg H (n >= 3, entries scaled to <= 1) from
 * its characteristic polynomial: the largest and smallest real roots by
 * real_root, checked for accuracy against the rounding error of evaluating
 * p, then a certificate that every other root is smaller in modulus -- the
 * remaining factor q = p / ((x - l1)(x - l2)) is centred on the mean of its roots, alpha, and its roots bounded by
 * |z - alpha| <= R, R = 2^(E+1) >= 2 max_k |t_k|^(1/(m-k)) (Fujiwara's bound
 * on the roots of t(y) = q(y + alpha), in powers of two: |t_k| < 2^e_k gives
 * |t_k|^(1/j) < 2^ceil(e_k/j)).  Returns 0 (caller falls back to QR) when a
 * root does not converge or the certificate fails: complex or repeated
 * extreme eigenvalues. */
static int charpoly_max_abs(const double *H, int n, double *out) {
  double c[MAXV + 1], q[MAXV + 1], t[MAXV + 1];
  hess_charpoly(H, n, c);
  /* starting points mu +- 1.001 sigma sqrt(n / 2), mu and sigma^2 the mean and
   * variance of the roots from c[n-1] and c[n-2] -- for a spectrum of pairs
   * u +- a_i around roots at u (the waves of a hyperbolic system) sigma^2 n / 2
   * = sum a_i^2, at or above the largest a_i^2 -- or +-||H||_inf when sigma^2
   * is not positive.  Any start is safe: the certificate decides. */
  double xhi, xlo;
  double inv_n = 1.0 / (double)n;
  double mu = -(c[n - 1] * inv_n);
  double s2 = fma(-mu, mu, fma(c[n - 1], c[n - 1], -2.0 * c[n - 2]) * inv_n);
  if (s2 > 0.0 && s2 <= 1e300) {
    double w = 1.001 * sqrt(s2 * (0.5 * (double)n));
    xhi = mu + w;
    xlo = mu - w;
  } else {
    double U = 0.0;
    for (int i = 0; i < n; i++) {
      double rs = 0.0;
      for (int j = 0; j < n; j++) rs = rs + fabs(H[i * n + j]);
      U = fmax(U, rs);
    }
    xhi = U;
    xlo = -U;
  }
  double l1, l2, d1, d2;
  if (!real_root(c, n, xhi, &l1, &d1) || !real_root(c, n, xlo, &l2, &d2)) return 0;
  double M = fmax(fabs(l1), fabs(l2));
  /* two distinct roots: from both ends the iterations can reach the one real
   * root, and deflating p by it twice would leave no certificate */
  if (!(l1 - l2 > 1e-9 * M)) return 0;
  /* accuracy: evaluating p rounds by up to 2 n eps sum_k |c_k| |x|^k, which
   * moves a root by that over |p'|; both must stay below 1e-11 M (a simple
   * root next to a cluster is ill-conditioned as a polynomial root) */
  {
    double a1 = fabs(l1), a2 = fabs(l2), E1 = 1.0, E2 = 1.0;
    for (int j = n - 1; j >= 0; j--) {
      E1 = fma(a1, E1, fabs(c[j]));
      E2 = fma(a2, E2, fabs(c[j]));
    }
    if (!((double)(2 * n) * DBL_EPSILON * E1 <= 1e-11 * M * fabs(d1))) return 0;
    if (!((double)(2 * n) * DBL_EPSILON * E2 <= 1e-11 * M * fabs(d2))) return 0;
  }
  /* q = p / (x - l1) / (x - l2), degree m = n - 2, monic */
  for (int i = 0; i <= n; i++) q[i] = c[i];
  int deg = n;
  double rr[2] = {l1, l2};
  for (int k = 0; k < 2; k++) {
    double nq[MAXV + 1];
    nq[deg - 1] = q[deg];
    for (int j = deg - 2; j >= 0; j--) nq[j] = fma(rr[k], nq[j + 1], q[j + 1]);
    deg -= 1;
    for (int j = 0; j <= deg; j++) q[j] = nq[j];
  }
  int m = deg;
  double alpha = -(q[m - 1] * (1.0 / (double)m));
  /* Taylor shift t(y) = q(y + alpha) */
  for (int i = 0; i <= m; i++) t[i] = q[i];
  for (int k = 0; k < m; k++)
    for (int j = m - 1; j >= k; j--) t[j] = fma(alpha, t[j + 1], t[j]);
  double tsum = 0.0;
  for (int k = 0; k < m; k++) tsum = tsum + fabs(t[k]);
  if (!(tsum <= DBL_MAX)) return 0;
  int emax = -2000;
  for (int k = 0; k < m; k++) {
    if (t[k] != 0.0) {
      int e;
      (void)frexp(t[k], &e);                 /* |t_k| = f 2^e, f in [0.5, 1) */
      int j = m - k;
      int ce = e >= 0 ? (e + j - 1) / j : -((-e) / j);
      emax = ce > emax ? ce : emax;
    }
  }
  double R = emax == -2000 ? 0.0 : ldexp(1.0, emax + 1);
  if (!(fabs(alpha) + R < M)) return 0;
  *out = M;
  return 1;
}

/* max |lambda| of a real n x n matrix, the quantity the reference takes from
 * Eigen's EigenSolver (system.cpp:28-43).  Method (EISPACK hqr structure,
 * eigenvalues only): scale by the power of two at or above the largest |entry|
 * (exact; Eigen's RealSchur divides by the largest |entry|, RealSchur.h:258-276),
 * Householder reduction to Hessenberg form, then Francis
 * double-shift QR steps (Golub & Van Loan Alg. 7.5.1-7.5.2) on the active
 * block, deflating on subdiagonals below eps (|h_kk| + |h_k-1,k-1|).  After 10
 * and 30 steps without deflation the origin is moved (exceptional shifts of
 * Wilkinson and of Moler, accumulated in `ex`), which is what lets clusters of
 * nearly equal small eigenvalues, as finite-difference Jacobians of
 * multi-wave systems produce, deflate at all.  After 40 n steps the remaining
 * diagonal entries stand in for the unresolved eigenvalues. */
double oracle_max_abs_eig(const double *A, int n) {
  double H[MAXV * MAXV];
  double scale = 0.0;
  for (int i = 0; i < n * n; i++) scale = fmax(scale, fabs(A[i]));
  if (!(scale >= DBL_MIN)) return (scale != scale) ? scale : 0.0;
  int e2;
  (void)frexp(scale, &e2);                 /* scale = m 2^e2, m in [0.5, 1) */
  /* up to n = 5, with the largest |entry| within 2^+-64, the matrix stays
   * unscaled: the reduction and the polynomial path then stay in the normal
   * range and commute exactly with scaling by a power of two; the QR
   * fallback, whose shifts are absolute, is scaled */
  int scaled = n > 5 || e2 < -64 || e2 > 64;
  double pw = ldexp(1.0, -e2);
  for (int i = 0; i < n * n; i++) H[i] = scaled ? A[i] * pw : A[i];
  double v[3], x[MAXV];
  for (int k = 0; k + 2 < n; k++) {
    int m = n - k - 1;
    double vv[MAXV];
    for (int i = 0; i < m; i++) x[i] = H[(k + 1 + i) * n + k];
    double mu = 0.0;
    double beta = house1(x, m, vv, &mu);
    if (beta != 0.0) {
      /* column k is x: P x = mu e_1, set rather than computed */
      house_left(H, n, vv, m, beta, k + 1, k + 1, n - 1);
      H[(k + 1) * n + k] = mu;
      for (int i = k + 2; i < n; i++) H[i * n + k] = 0.0;
      house_right(H, n, vv, m, beta, 0, n - 1, k + 1);
    }
  }
  {
    double r;
    if (n >= 3 && charpoly_max_abs(H, n, &r)) return scaled ? ldexp(r, e2) : r;
  }
  if (!scaled)
    for (int i = 0; i < n * n; i++) H[i] = H[i] * pw;
  double anorm = 0.0;
  for (int i = 0; i < n * n; i++) anorm = anorm + fabs(H[i]);
  double best = 0.0, ex = 0.0;
  int hi = n - 1, iter = 0, total = 0;
  while (hi >= 0) {
    int lo = hi;
    while (lo > 0) {
      double s = fabs(H[(lo - 1) * n + lo - 1]) + fabs(H[lo * n + lo]);
      if (s == 0.0) s = anorm;
      if (fabs(H[lo * n + lo - 1]) <= DBL_EPSILON * s) {
        H[lo * n + lo - 1] = 0.0;
        break;
      }
      lo--;
    }
    if (lo == hi) {
      best = fmax(best, fabs(H[hi * n + hi] + ex));
      hi -= 1;
      iter = 0;
      continue;
    }
    if (lo == hi - 1) {
      double a = H[(hi - 1) * n + hi - 1] + ex, b = H[(hi - 1) * n + hi];
      double c = H[hi * n + hi - 1], dd = H[hi * n + hi] + ex;
      double p = 0.5 * (a - dd);
      double bc = b * c;
      double disc = p * p + bc;
      if (disc >= 0.0) {
        double z = sqrt(disc);
        z = (p >= 0.0) ? p + z : p - z;
        double l1 = dd + z;
        double l2 = (z != 0.0) ? dd - bc / z : dd;
        best = fmax(best, fmax(fabs(l1), fabs(l2)));
      } else {
        double re = dd + p;
        best = fmax(best, sqrt(re * re - disc));
      }
      hi -= 2;
      iter = 0;
      continue;
    }
    if (total >= 40 * n) {
      for (int i = 0; i <= hi; i++) best = fmax(best, fabs(H[i * n + i] + ex));
      break;
    }
    /* shift data from the trailing 2x2 block */
    double sx = H[hi * n + hi], sy = H[(hi - 1) * n + hi - 1];
    double sw = H[hi * n + hi - 1] * H[(hi - 1) * n + hi];
    if (iter == 10) {
      ex = ex + sx;
      for (int i = 0; i <= hi; i++) H[i * n + i] = H[i * n + i] - sx;
      double s = fabs(H[hi * n + hi - 1]) + fabs(H[(hi - 1) * n + hi - 2]);
      sx = 0.75 * s;
      sy = sx;
      sw = -0.4375 * s * s;
    } else if (iter == 30) {
      double s = (sy - sx) / 2.0;
      s = s * s + sw;
      if (s > 0.0) {
        s = sqrt(s);
        if (sy < sx) s = -s;
        s = s + (sy - sx) / 2.0;
        s = sx - sw / s;
        ex = ex + s;
        for (int i = 0; i <= hi; i++) H[i * n + i] = H[i * n + i] - s;
        sx = 0.964;
        sy = 0.964;
        sw = 0.964;
      }
    }
    iter++;
    total++;
    /* first column of (H - s1)(H - s2), scaled by 1/h(lo+1,lo) */
    double h00 = H[lo * n + lo];
    double r = sx - h00, q = sy - h00;
    x[0] = (r * q - sw) / H[(lo + 1) * n + lo] + H[lo * n + lo + 1];
    x[1] = H[(lo + 1) * n + lo + 1] - h00 - r - q;
    x[2] = H[(lo + 2) * n + lo + 1];
    for (int k = lo; k <= hi - 2; k++) {
      if (k > lo) {
        x[0] = H[k * n + k - 1];
        x[1] = H[(k + 1) * n + k - 1];
        x[2] = H[(k + 2) * n + k - 1];
      }
      double beta = house(x, 3, v);
      if (beta != 0.0) {
        if (k > lo) {
          H[k * n + k - 1] = sqrt(x[0] * x[0] + (x[1] * x[1] + x[2] * x[2]));
          H[(k + 1) * n + k - 1] = 0.0;
          H[(k + 2) * n + k - 1] = 0.0;
        }
        house_left(H, n, v, 3, beta, k, k, hi);
        int rr = (k + 3 < hi) ? k + 3 : hi;
        house_right(H, n, v, 3, beta, lo, rr, k);
      }
    }
    x[0] = H[(hi - 1) * n + hi - 2];
    x[1] = H[hi * n + hi - 2];
    double beta = house(x, 2, v);
    if (beta != 0.0) {
      H[(hi - 1) * n + hi - 2] = sqrt(x[0] * x[0] + x[1] * x[1]);
      H[hi * n + hi - 2] = 0.0;
      house_left(H, n, v, 2, beta, hi - 1, hi - 1, hi);
      house_right(H, n, v, 2, beta, lo, hi, hi - 1);
    }
  }
  return ldexp(best, e2);
}

/* 1 / h_i for the forward-difference steps h_i = max(sqrt(eps)|q_i|,
 * sqrt(eps)) = 2^-26 m_i, m_i = max(|q_i|, 1) (exact: sqrt(eps) = 2^-26), with
 * one division for all of them: 1 / h_i = (2^26 / prod m) (prod_{j<i} m_j
 * prod_{j>i} m_j).  When prod m passes 2^1000 each is divided on its own. */
static void fd_recips(const double *q, int V, double *rh) {
  double m[MAXV], pre[MAXV + 1], suf[MAXV + 1];
  pre[0] = 1.0;
  for (int i = 0; i < V; i++) {
    m[i] = fmax(fabs(q[i]), 1.0);
    pre[i + 1] = pre[i] * m[i];
  }
  if (!(pre[V] <= 0x1p1000)) {
    for (int i = 0; i < V; i++) rh[i] = 1.0 / fmax(FD_EPS * fabs(q[i]), FD_EPS);
    return;
  }
  suf[V] = 1.0;
  for (int i = V - 1; i >= 0; i--) suf[i] = suf[i + 1] * m[i];
  double r = 0x1p26 / pre[V];
  for (int i = 0; i < V; i++) rh[i] = r * (pre[i] * suf[i + 1]);
}

/* A = dF/dQ by forward differences + B (system.cpp:6-26, NumericalDiff.h:6-44):
 * h_i = max(sqrt(eps)|q_i|, sqrt(eps)), column i = (F(q + h_i e_i) - F(q)) (1 / h_i)
 * with the reciprocals from fd_recips (the reference divides every entry by
 * h_i, which differs by a few roundings).
 * f0 (optional) receives F(q). */
static void system_matrix(oracle_F F, oracle_B B, const double *q,
                          const double *dq, int d, int V, double *A,
                          double *f0) {
  double qq[MAXV], dqq[MAXD * MAXV], v1[MAXV], v2[MAXV];
  memcpy(qq, q, V * sizeof(double));
  memcpy(dqq, dq, MAXD * V * sizeof(double));
  if (F) {
    double rh[MAXV];
    F(v1, qq, dqq, d);
    fd_recips(qq, V, rh);
    for (int i = 0; i < V; i++) {
      double qi0 = qq[i];
      double h = fmax(FD_EPS * fabs(qi0), FD_EPS);
      qq[i] = qi0 + h;
      F(v2, qq, dqq, d);
      qq[i] = qi0;
      for (int r = 0; r < V; r++) A[r * V + i] = (v2[r] - v1[r]) * rh[i];
    }
    if (f0) memcpy(f0, v1, V * sizeof(double));
  } else {
    for (int i = 0; i < V * V; i++) A[i] = 0.0;
  }
  if (B) {
    double b[MAXV * MAXV];
    B(b, qq, d);
    for (int i = 0; i < V * V; i++) A[i] = A[i] + b[i];
  }
}

void oracle_system_matrix(oracle_F F, oracle_B B, const double *q,
                          const double *dq, int d, int ndim, int V,
                          double *out) {
  double dqq[MAXD * MAXV] = {0};
  memcpy(dqq, dq, ndim * V * sizeof(double));
  system_matrix(F, B, q, dqq, d, V, out, NULL);
}

static double max_abs_eigs(oracle_F F, oracle_B B, const double *q,
                           const double *dq, int d, int V, double *f0) {
  double A[MAXV * MAXV];
  system_matrix(F, B, q, dq, d, V, A, f0);
  return oracle_max_abs_eig(A, V);
}

/* Viscous wave speed (system.cpp:53-61, NumericalDiff.h:6-44 with
 * secondOrder): 2 (N + 1) / dX_d max|lambda(dF_d / d(dQ_d))|, the Jacobian by
 * forward differences in the gradient components dQ[d V + i]. */
static double max_abs_eigs_second_order(oracle_F F, const double *q, const double *dq,
                                        int d, int V, int N, const double *dX) {
  double qq[MAXV], dqq[MAXD * MAXV], v1[MAXV], v2[MAXV], A[MAXV * MAXV];
  memcpy(qq, q, V * sizeof(double));
  memcpy(dqq, dq, MAXD * V * sizeof(double));
  F(v1, qq, dqq, d);
  for (int i = 0; i < V; i++) {
    double qi0 = dqq[d * V + i];
    double h = fmax(FD_EPS * fabs(qi0), FD_EPS);
    dqq[d * V + i] = qi0 + h;
    F(v2, qq, dqq, d);
    dqq[d * V + i] = qi0;
    double rh = 1.0 / h;
    for (int r = 0; r < V; r++) A[r * V + i] = (v2[r] - v1[r]) * rh;
  }
  return (double)(2 * (N + 1)) / dX[d] * oracle_max_abs_eig(A, V);
}

/* ------------------------------------------- |A| x for Roe and Osher fluxes */

/* Real Schur form T = Z^T H Z of an n x n matrix (H is overwritten by T, Z
 * receives the orthogonal factor): Householder Hessenberg reduction and
 * Francis double-shift QR as in oracle_max_abs_eig, here applied to the whole
 * matrix with the transformations accumulated in Z (the EISPACK hqr2
 * arrangement), exceptional shifts restored on the diagonal as each block
 * deflates, and every 2 x 2 block with real eigenvalues split by a rotation.
 * Returns 0, or 1 when the QR did not converge in 40 n steps (T is then
 * only partly reduced). */
static int real_schur(double *H, double *Z, int n) {
  double v[3], x[MAXV];
  for (int i = 0; i < n * n; i++) Z[i] = (i % (n + 1) == 0) ? 1.0 : 0.0;
  for (int k = 0; k + 2 < n; k++) {
    int m = n - k - 1;
    double vv[MAXV];
    for (int i = 0; i < m; i++) x[i] = H[(k + 1 + i) * n + k];
    double beta = house(x, m, vv);
    if (beta != 0.0) {
      house_left(H, n, vv, m, beta, k + 1, k, n - 1);
      house_right(H, n, vv, m, beta, 0, n - 1, k + 1);
      house_right(Z, n, vv, m, beta, 0, n - 1, k + 1);
    }
    for (int i = k + 2; i < n; i++) H[i * n + k] = 0.0;
  }
  double anorm = 0.0;
  for (int i = 0; i < n * n; i++) anorm = anorm + fabs(H[i]);
  double ex = 0.0;
  int hi = n - 1, iter = 0, total = 0;
  while (hi >= 0) {
    int lo = hi;
    while (lo > 0) {
      double s = fabs(H[(lo - 1) * n + lo - 1]) + fabs(H[lo * n + lo]);
      if (s == 0.0) s = anorm;
      if (fabs(H[lo * n + lo - 1]) <= DBL_EPSILON * s) {
        H[lo * n + lo - 1] = 0.0;
        break;
      }
      lo--;
    }
    if (lo == hi) {
      H[hi * n + hi] = H[hi * n + hi] + ex;
      hi -= 1;
      iter = 0;
      continue;
    }
    if (lo == hi - 1) {
      int na = hi - 1;
      H[na * n + na] = H[na * n + na] + ex;
      H[hi * n + hi] = H[hi * n + hi] + ex;
      double a = H[na * n + na], b = H[na * n + hi], c = H[hi * n + na], d = H[hi * n + hi];
      double p = 0.5 * (a - d);
      double disc = p * p + b * c;
      if (disc >= 0.0) {
        /* real pair: rotate so that the block becomes upper triangular */
        double z = sqrt(disc);
        z = (p >= 0.0) ? p + z : p - z;
        double xr = c, sr = fabs(xr) + fabs(z);
        double pr = xr / sr, qr = z / sr;
        double rr = sqrt(pr * pr + qr * qr);
        pr = pr / rr;
        qr = qr / rr;
        for (int j = na; j < n; j++) {
          double t = H[na * n + j];
          H[na * n + j] = qr * t + pr * H[hi * n + j];
          H[hi * n + j] = qr * H[hi * n + j] - pr * t;
        }
        for (int i = 0; i <= hi; i++) {
          double t = H[i * n + na];
          H[i * n + na] = qr * t + pr * H[i * n + hi];
          H[i * n + hi] = qr * H[i * n + hi] - pr * t;
        }
        for (int i = 0; i < n; i++) {
          double t = Z[i * n + na];
          Z[i * n + na] = qr * t + pr * Z[i * n + hi];
          Z[i * n + hi] = qr * Z[i * n + hi] - pr * t;
        }
        H[hi * n + na] = 0.0;
      }
      hi -= 2;
      iter = 0;
      continue;
    }
    if (total >= 40 * n) {
      for (int i = 0; i <= hi; i++) H[i * n + i] = H[i * n + i] + ex;
      return 1;
    }
    double sx = H[hi * n + hi], sy = H[(hi - 1) * n + hi - 1];
    double sw = H[hi * n + hi - 1] * H[(hi - 1) * n + hi];
    if (iter == 10) {
      ex = ex + sx;
      for (int i = 0; i <= hi; i++) H[i * n + i] = H[i * n + i] - sx;
      double s = fabs(H[hi * n + hi - 1]) + fabs(H[(hi - 1) * n + hi - 2]);
      sx = 0.75 * s;
      sy = sx;
      sw = -0.4375 * s * s;
    } else if (iter == 30) {
      double s = (sy - sx) / 2.0;
      s = s * s + sw;
      if (s > 0.0) {
        s = sqrt(s);
        if (sy < sx) s = -s;
        s = s + (sy - sx) / 2.0;
        s = sx - sw / s;
        ex = ex + s;
        for (int i = 0; i <= hi; i++) H[i * n + i] = H[i * n + i] - s;
        sx = 0.964;
        sy = 0.964;
        sw = 0.964;
      }
    }
    iter++;
    total++;
    double h00 = H[lo * n + lo];
    double r = sx - h00, q = sy - h00;
    x[0] = (r * q - sw) / H[(lo + 1) * n + lo] + H[lo * n + lo + 1];
    x[1] = H[(lo + 1) * n + lo + 1] - h00 - r - q;
    x[2] = H[(lo + 2) * n + lo + 1];
    for (int k = lo; k <= hi - 2; k++) {
      if (k > lo) {
        x[0] = H[k * n + k - 1];
        x[1] = H[(k + 1) * n + k - 1];
        x[2] = H[(k + 2) * n + k - 1];
      }
      double beta = house(x, 3, v);
      if (beta != 0.0) {
        if (k > lo) {
          H[k * n + k - 1] = sqrt(x[0] * x[0] + (x[1] * x[1] + x[2] * x[2]));
          H[(k + 1) * n + k - 1] = 0.0;
          H[(k + 2) * n + k - 1] = 0.0;
        }
        house_left(H, n, v, 3, beta, k, k, n - 1);
        int rr = (k + 3 < hi) ? k + 3 : hi;
        house_right(H, n, v, 3, beta, 0, rr, k);
        house_right(Z, n, v, 3, beta, 0, n - 1, k);
      }
    }
    x[0] = H[(hi - 1) * n + hi - 2];
    x[1] = H[hi * n + hi - 2];
    double beta = house(x, 2, v);
    if (beta != 0.0) {
      H[(hi - 1) * n + hi - 2] = sqrt(x[0] * x[0] + x[1] * x[1]);
      H[hi * n + hi - 2] = 0.0;
      house_left(H, n, v, 2, beta, hi - 1, hi - 1, n - 1);
      house_right(H, n, v, 2, beta, 0, hi, hi - 1);
      house_right(Z, n, v, 2, beta, 0, n - 1, hi - 1);
    }
  }
  return 0;
}

/* Divisor guard of the back substitution (as Eigen's EigenSolver): a zero
 * pivot of T - lambda becomes eps ||T||. */
static double guard_div(double w, double tn) {
  return (w == 0.0) ? DBL_EPSILON * tn : w;
}

/* y = |A| x = R |Lambda| R^-1 x for a real n x n matrix A, R its eigenvectors
 * (fluxes.cpp:20-70 forms exactly this from Eigen's EigenSolver).  Computed in
 * real arithmetic: from the real Schur form T = Z^T A Z, a basis Y of each
 * invariant subspace of T (the eigenvector of a real eigenvalue; real and
 * imaginary parts of the eigenvector of a complex pair, on which |A| acts as
 * |lambda| I), W = Z Y, then y = W D W^-1 x with D = |lambda| per column.
 * A is scaled by the power of two at or above its largest |entry| first. */
void oracle_abs_apply(const double *A, const double *xin, int n, double *y) {
  double T[MAXV * MAXV], Z[MAXV * MAXV], Y[MAXV * MAXV], W[MAXV * MAXV], D[MAXV];
  double scale = 0.0;
  for (int i = 0; i < n * n; i++) scale = fmax(scale, fabs(A[i]));
  if (!(scale >= DBL_MIN)) {
    for (int i = 0; i < n; i++) y[i] = (scale != scale) ? scale : 0.0;
    return;
  }
  int e2;
  (void)frexp(scale, &e2);
  double pw = ldexp(1.0, -e2);
  for (int i = 0; i < n * n; i++) T[i] = A[i] * pw;
  (void)real_schur(T, Z, n);
  double tn = 0.0;
  for (int i = 0; i < n * n; i++) tn = tn + fabs(T[i]);
  for (int i = 0; i < n * n; i++) Y[i] = 0.0;
  /* invariant-subspace bases, from the bottom block up */
  int en = n - 1;
  while (en >= 0) {
    if (en >= 1 && T[en * n + en - 1] != 0.0) {
      /* complex pair on rows en-1, en: eigenvector for lambda = a + i b */
      int na = en - 1;
      double a = 0.5 * (T[na * n + na] + T[en * n + en]);
      double pp = 0.5 * (T[na * n + na] - T[en * n + en]);
      double bb = sqrt(-(pp * pp + T[na * n + en] * T[en * n + na]));
      D[na] = ldexp(sqrt(a * a + bb * bb), e2);
      D[en] = D[na];
      /* vector (yr + i yi): rows na, en from (T_blk - lambda) y = 0 with y[en] = 1:
       * y[na] = (lambda - t_en,en) / t_en,na */
      double yr[MAXV], yi[MAXV];
      for (int i = 0; i < n; i++) {
        yr[i] = 0.0;
        yi[i] = 0.0;
      }
      yr[en] = 1.0;
      yr[na] = (a - T[en * n + en]) / T[en * n + na];
      yi[na] = bb / T[en * n + na];
      int i = na - 1;
      while (i >= 0) {
        if (i >= 1 && T[i * n + i - 1] != 0.0) {
          /* 2 x 2 block rows i-1, i: complex 2 x 2 solve (Cramer) */
          int im = i - 1;
          double s1r = 0.0, s1i = 0.0, s2r = 0.0, s2i = 0.0;
          for (int j = i + 1; j <= en; j++) {
            s1r = fma(T[im * n + j], yr[j], s1r);
            s1i = fma(T[im * n + j], yi[j], s1i);
            s2r = fma(T[i * n + j], yr[j], s2r);
            s2i = fma(T[i * n + j], yi[j], s2i);
          }
          /* [[t11 - lam, t12], [t21, t22 - lam]] [u1; u2] = -[s1; s2] */
          double m11r = T[im * n + im] - a, m11i = -bb, m12 = T[im * n + i];
          double m21 = T[i * n + im], m22r = T[i * n + i] - a, m22i = -bb;
          double detr = (m11r * m22r - m11i * m22i) - m12 * m21;
          double deti = m11r * m22i + m11i * m22r;
          if (detr == 0.0 && deti == 0.0) detr = DBL_EPSILON * tn;
          /* u1 = (-s1 m22 + s2 m12) / det, u2 = (-s2 m11 + s1 m21) / det */
          double n1r = -(s1r * m22r - s1i * m22i) + s2r * m12;
          double n1i = -(s1r * m22i + s1i * m22r) + s2i * m12;
          double n2r = -(s2r * m11r - s2i * m11i) + s1r * m21;
          double n2i = -(s2r * m11i + s2i * m11r) + s1i * m21;
          double dd = detr * detr + deti * deti;
          yr[im] = (n1r * detr + n1i * deti) / dd;
          yi[im] = (n1i * detr - n1r * deti) / dd;
          yr[i] = (n2r * detr + n2i * deti) / dd;
          yi[i] = (n2i * detr - n2r * deti) / dd;
          i -= 2;
        } else {
          double sr = 0.0, si = 0.0;
          for (int j = i + 1; j <= en; j++) {
            sr = fma(T[i * n + j], yr[j], sr);
            si = fma(T[i * n + j], yi[j], si);
          }
          /* (t_ii - a - i b) y_i = -s */
          double wr = guard_div(T[i * n + i] - a, tn), wi = -bb;
          double dd = wr * wr + wi * wi;
          yr[i] = -(sr * wr + si * wi) / dd;
          yi[i] = -(si * wr - sr * wi) / dd;
          i -= 1;
        }
      }
      for (int r = 0; r < n; r++) {
        Y[r * n + na] = yr[r];
        Y[r * n + en] = yi[r];
      }
      en -= 2;
    } else {
      double lam = T[en * n + en];
      D[en] = ldexp(fabs(lam), e2);
      double yv[MAXV];
      for (int i = 0; i < n; i++) yv[i] = 0.0;
      yv[en] = 1.0;
      int i = en - 1;
      while (i >= 0) {
        if (i >= 1 && T[i * n + i - 1] != 0.0) {
          int im = i - 1;
          double s1 = 0.0, s2 = 0.0;
          for (int j = i + 1; j <= en; j++) {
            s1 = fma(T[im * n + j], yv[j], s1);
            s2 = fma(T[i * n + j], yv[j], s2);
          }
          double m11 = T[im * n + im] - lam, m12 = T[im * n + i];
          double m21 = T[i * n + im], m22 = T[i * n + i] - lam;
          double det = guard_div(m11 * m22 - m12 * m21, tn);
          yv[im] = (-s1 * m22 + s2 * m12) / det;
          yv[i] = (-s2 * m11 + s1 * m21) / det;
          i -= 2;
        } else {
          double sacc = 0.0;
          for (int j = i + 1; j <= en; j++) sacc = fma(T[i * n + j], yv[j], sacc);
          yv[i] = -sacc / guard_div(T[i * n + i] - lam, tn);
          i -= 1;
        }
      }
      for (int r = 0; r < n; r++) Y[r * n + en] = yv[r];
      en -= 1;
    }
  }
  /* W = Z Y */
  for (int i = 0; i < n; i++)
    for (int j = 0; j < n; j++) {
      double acc = Z[i * n] * Y[j];
      for (int k = 1; k < n; k++) acc = fma(Z[i * n + k], Y[k * n + j], acc);
      W[i * n + j] = acc;
    }
  /* b = W^-1 x (LU, partial pivoting), b *= D, y = W b */
  double LU[MAXV * MAXV], b[MAXV];
  int piv[MAXV];
  memcpy(LU, W, sizeof(double) * n * n);
  for (int i = 0; i < n; i++) b[i] = xin[i];
  for (int k = 0; k < n; k++) {
    int p = k;
    for (int i = k + 1; i < n; i++)
      if (fabs(LU[i * n + k]) > fabs(LU[p * n + k])) p = i;
    piv[k] = p;
    if (p != k) {
      for (int j = 0; j < n; j++) {
        double t = LU[k * n + j];
        LU[k * n + j] = LU[p * n + j];
        LU[p * n + j] = t;
      }
      double t = b[k];
      b[k] = b[p];
      b[p] = t;
    }
    double piv_k = guard_div(LU[k * n + k], 1.0);
    for (int i = k + 1; i < n; i++) {
      double l = LU[i * n + k] / piv_k;
      LU[i * n + k] = l;
      for (int j = k + 1; j < n; j++) LU[i * n + j] = fma(-l, LU[k * n + j], LU[i * n + j]);
      b[i] = fma(-l, b[k], b[i]);
    }
  }
  for (int i = n - 1; i >= 0; i--) {
    double acc = b[i];
    for (int j = i + 1; j < n; j++) acc = fma(-LU[i * n + j], b[j], acc);
    b[i] = acc / guard_div(LU[i * n + i], 1.0);
  }
  (void)piv;
  for (int i = 0; i < n; i++) b[i] = b[i] * D[i];
  for (int i = 0; i < n; i++) {
    double acc = W[i * n] * b[0];
    for (int k = 1; k < n; k++) acc = fma(W[i * n + k], b[k], acc);
    y[i] = acc;
  }
}

double oracle_exp(double x) {
  /* Same method as pde_exp in pypde_amd/systems/pde_prelude.h (which system
   * sources call); duplicated here so the oracle is self-contained. */
  if (x > 709.782712893384) return 1.0 / 0.0;
  if (x < -745.1332191019412) return 0.0;
  double k = rint(x * 1.4426950408889634);
  double r = fma(-k, 0.6931471805599453, x);
  r = fma(-k, 2.3190468138462996e-17, r);
  static const double c[13] = {
      2.08767569878681e-09, 2.505210838544172e-08, 2.755731922398589e-07,
      2.7557319223985893e-06, 2.48015873015873e-05, 0.0001984126984126984,
      0.001388888888888889, 0.008333333333333333, 0.041666666666666664,
      0.16666666666666666, 0.5, 1.0, 1.0};
  double p = 1.6059043836821613e-10;
  for (int i = 0; i < 13; i++) p = fma(p, r, c[i]);
  return ldexp(p, (int)k);
}

/* ------------------------------------------------------------ boundaries */

/* Ghost index map (boundaries.cpp:7-23); reflective walls (code 2) are an
 * addition to the reference's codes: mirror image across the wall, signs from
 * `reflect`. */
static int ghost_src(int i, int N, int type, int n, int *flip) {
  int r = i - N;
  *flip = 0;
  if (r < 0) {
    if (type == 0) return 0;
    if (type == 1) return n + r;
    *flip = 1;
    return -r - 1;
  }
  if (r >= n) {
    if (type == 0) return n - 1;
    if (type == 1) return r - n;
    *flip = 1;
    return 2 * n - r - 1;
  }
  return r;
}

int oracle_boundaries(double *ub, const double *u, const int *nX, int ndim,
                      const int *bc, const double *reflect, int N, int V) {
  int nb[MAXD], ind[MAXD];
  long ncell = 1;
  for (int d = 0; d < ndim; d++) {
    nb[d] = nX[d] + 2 * N;
    ncell *= nb[d];
    ind[d] = 0;
  }
  for (long c = 0; c < ncell; c++) {
    long src = 0;
    double sgn[MAXV];
    for (int v = 0; v < V; v++) sgn[v] = 1.0;
    for (int d = 0; d < ndim; d++) {
      int flip;
      int s = ghost_src(ind[d], N, bc[d], nX[d], &flip);
      if (s < 0 || s >= nX[d]) return 1;
      src = src * nX[d] + s;
      if (flip && reflect)
        for (int v = 0; v < V; v++) sgn[v] = sgn[v] * reflect[d * V + v];
    }
    for (int v = 0; v < V; v++) ub[c * V + v] = u[src * V + v] * sgn[v];
    for (int d = ndim - 1; d >= 0; d--) {
      if (++ind[d] < nb[d]) break;
      ind[d] = 0;
    }
  }
  return 0;
}

/* ----------------------------------------------------------------- WENO */

/* One line window d[0..2N-2] (stride `st`) -> N nodal values (weno.cpp:26-59):
 * for each stencil c = M^-1 data, p = c^T SIG c + EPS, o = LAM / p^8,
 * num += o c, den += o; result num / den.  With at most three stencils the
 * weights are multiplied through by prod_r p_r^8 (o_s' = LAM_s prod_{r != s}
 * p_r^8, never below 1e-224) and the sums scaled by one reciprocal, which
 * saves a division per stencil; where that product form overflows the
 * division form is used.  Both give the reference's weights to a few ulps
 * (held to the reference's own weno_solver to 1e-12 at N = 3). */
static void weno_line(const Tab *T, const double *d, long st, double *out) {
  int N = T->N, NS = T->nsten;
  double num[MAXN], den = 0.0, c[4][MAXN], P[4];
  for (int s = 0; s < NS; s++) {
    const double *dd = d + (long)T->soff[s] * st;
    for (int k = 0; k < N; k++) {
      double acc = T->winv[s][k][0] * dd[0];
      for (int j = 1; j < N; j++) acc = fma(T->winv[s][k][j], dd[(long)j * st], acc);
      c[s][k] = acc;
    }
    double p = 0.0;
    for (int k = 0; k < N; k++) {
      double t = T->sig[k][0] * c[s][0];
      for (int j = 1; j < N; j++) t = fma(T->sig[k][j], c[s][j], t);
      p = (k == 0) ? c[s][0] * t : fma(c[s][k], t, p);
    }
    p = p + WENO_EPS;
    double p2 = p * p;
    double p4 = p2 * p2;
    P[s] = p4 * p4;
  }
  if (NS <= 3) {
    for (int k = 0; k < N; k++) num[k] = 0.0;
    for (int s = 0; s < NS; s++) {
      double o = T->slam[s];
      for (int r = 0; r < NS; r++)
        if (r != s) o = o * P[r];
      for (int k = 0; k < N; k++) num[k] = fma(o, c[s][k], num[k]);
      den = den + o;
    }
    if (den <= DBL_MAX) {
      double rden = 1.0 / den;
      for (int k = 0; k < N; k++) out[k] = num[k] * rden;
      return;
    }
    den = 0.0;
  }
  for (int k = 0; k < N; k++) num[k] = 0.0;
  for (int s = 0; s < NS; s++) {
    double o = T->slam[s] / P[s];
    for (int k = 0; k < N; k++) num[k] = fma(o, c[s][k], num[k]);
    den = den + o;
  }
  for (int k = 0; k < N; k++) out[k] = num[k] / den;
}

/* Dimension-by-dimension reconstruction (weno.cpp:61-121).  rec has shape
 * `shape` (cells) x V; result shape shrinks by 2(N-1) per axis and gains N^D
 * node indices. */
static double *weno_sweeps(const Tab *T, const double *ub, const int *shape_in) {
  int N = T->N, V = T->V, D = T->D;
  int shape[MAXD];
  long ncell = 1;
  for (int d = 0; d < D; d++) {
    shape[d] = shape_in[d];
    ncell *= shape[d];
  }
  double *rec = (double *)malloc(sizeof(double) * ncell * V);
  memcpy(rec, ub, sizeof(double) * ncell * V);
  for (int d = 0; d < D; d++) {
    long n1 = 1, n3 = 1;
    for (int i = 0; i < d; i++) n1 *= shape[i];
    long n2 = shape[d] - 2 * (N - 1);
    for (int i = d + 1; i < D; i++) n3 *= shape[i];
    long n4 = ipow(N, d);
    double *rec2 = (double *)malloc(sizeof(double) * n1 * n2 * n3 * n4 * N * V);
    long stride = n3 * n4 * V;
#pragma omp parallel for collapse(2) schedule(static)
    for (long i1 = 0; i1 < n1; i1++)
      for (long i3 = 0; i3 < n3; i3++)
        for (long i4 = 0; i4 < n4; i4++) {
          long indu = ((i1 * shape[d] * n3 + i3) * n4 + i4) * V;
          long indw = ((i1 * n2 * n3 + i3) * n4 + i4) * N * V;
          for (long i = 0; i < n2; i++)
            for (int v = 0; v < V; v++) {
              double out[MAXN];
              weno_line(T, rec + indu + i * stride + v, stride, out);
              for (int k = 0; k < N; k++)
                rec2[indw + i * N * stride + k * V + v] = out[k];
            }
        }
    free(rec);
    rec = rec2;
    shape[d] = (int)n2;
  }
  return rec;
}

int oracle_weno(double *wh, const double *u, const int *nX, int ndim, int N,
                int V) {
  Tab T;
  if (tab_init(&T, N, ndim, V)) return 1;
  long nout = 1;
  for (int d = 0; d < ndim; d++) {
    if (nX[d] - 2 * (N - 1) < 1) return 2;
    nout *= nX[d] - 2 * (N - 1);
  }
  double *r = weno_sweeps(&T, u, nX);
  memcpy(wh, r, sizeof(double) * nout * T.Nd * V);
  free(r);
  return 0;
}

/* ------------------------------------------------------------- timestep */

/* CFL step (stepper.cpp:35-76) over every reconstructed cell, the ghost layer
 * included (iterator.cpp:76): cell mean q and gradient dq by the tensor Gauss
 * weights, MAX = max_cells sum_d lambda_d / dX_d, dt = CFL / MAX, x0.2 while
 * count <= 5, clamped to tf - t. */
static double cell_speed(const Tab *T, oracle_F F, oracle_B B,
                         const double *wc, const double *dX, int second) {
  int V = T->V, D = T->D, Nd = T->Nd;
  double q[MAXV], dq[MAXD * MAXV] = {0}, tmp[MAXV];
  for (int v = 0; v < V; v++) {
    double acc = T->WP[0] * wc[v];
    for (int idx = 1; idx < Nd; idx++) acc = fma(T->WP[idx], wc[idx * V + v], acc);
    q[v] = acc;
  }
  for (int d = 0; d < D; d++) {
    double acc[MAXV];
    for (int idx = 0; idx < Nd; idx++) {
      node_deriv(T, wc, idx, d, 1.0 / dX[d], tmp);
      for (int v = 0; v < V; v++)
        acc[v] = (idx == 0) ? T->WP[0] * tmp[v] : fma(T->WP[idx], tmp[v], acc[v]);
    }
    for (int v = 0; v < V; v++) dq[d * V + v] = acc[v];
  }
  double sum = 0.0;
  for (int d = 0; d < D; d++) {
    double lam = max_abs_eigs(F, B, q, dq, d, V, NULL);
    if (second) lam = lam + max_abs_eigs_second_order(F, q, dq, d, V, T->N, dX);
    sum = sum + lam / dX[d];
  }
  return sum;
}

static double timestep_impl(oracle_F F, oracle_B B, const double *wh, long nw,
                            const double *dX, int ndim, int N, int V, double CFL,
                            double tf, double t, long count, int second) {
  Tab T;
  if (tab_init(&T, N, ndim, V)) return NAN;
  double MAX = 0.0;
#pragma omp parallel for reduction(max : MAX) schedule(static)
  for (long c = 0; c < nw; c++) {
    double s = cell_speed(&T, F, B, wh + c * T.Nd * V, dX, second);
    if (s > MAX) MAX = s;
  }
  double dt = CFL / MAX;
  if (count <= 5) dt = dt * 0.2;
  if (t + dt > tf) return tf - t;
  return dt;
}

double oracle_timestep(oracle_F F, oracle_B B, const double *wh, long nw,
                       const double *dX, int ndim, int N, int V, double CFL,
                       double tf, double t, long count) {
  return timestep_impl(F, B, wh, nw, dX, ndim, N, V, CFL, tf, t, count, 0);
}

/* ------------------------------------------------------------ predictor */

typedef struct {
  const Tab *T;
  oracle_F F;
  oracle_B B;
  oracle_S S;
  oracle_M M;
  const double *dX;
  double dt;
  double *dq; /* workspace: MAXND * MAXD * MAXV */
  double *f;  /* workspace: MAXD * MAXND * MAXV */
  int b_quirk;
} Ctx;

/* B(q) applied to a gradient dq.  Default: the matrix-vector product of the
 * documented PDE (solvers.py:108-121).  b_quirk = 1 reproduces what the
 * reference computes at dg.cpp:110 (row destination): `b * dq.row(i)` has
 * mismatched inner dimensions, which -DNDEBUG leaves unchecked, and Eigen
 * evaluates it as a depth-1 outer product, b(0,0) dq[v].  b_quirk = 2 is the
 * column-destination form of fv.cpp:234, b(v,0) dq[0]. */
static void b_times(const double *b, const double *dqd, int V, int quirk,
                    double *out) {
  for (int v = 0; v < V; v++) {
    if (quirk == 1) {
      out[v] = b[0] * dqd[v];
    } else if (quirk == 2) {
      out[v] = b[v * V] * dqd[0];
    } else {
      double acc = b[v * V] * dqd[0];
      for (int j = 1; j < V; j++) acc = fma(b[v * V + j], dqd[j], acc);
      out[v] = acc;
    }
  }
}

/* rhs(q) of the space-time system (dg.cpp:50-126):
 * r = W_t prod W_x (S(q) - sum_d (B_d(q) dq_d + d_d F_d(q, dq))), then
 * rhs = r dt + Ww with Ww[t][x] = psi_t(0) prod W_x w[x] (dg.cpp:156-171). */
static void dg_rhs(const Ctx *C, const double *w, const double *q, double *rhs) {
  const Tab *T = C->T;
  int N = T->N, D = T->D, V = T->V, Nd = T->Nd;
  double *dq = C->dq, *f = C->f;
  for (int t = 0; t < N; t++) {
    const double *qt = q + (long)t * Nd * V;
    for (int idx = 0; idx < Nd; idx++)
      for (int d = 0; d < D; d++)
        node_deriv(T, qt, idx, d, 1.0 / C->dX[d], dq + (idx * MAXD + d) * V);
    if (C->F)
      for (int idx = 0; idx < Nd; idx++) {
        double qq[MAXV], dqq[MAXD * MAXV] = {0};
        memcpy(qq, qt + idx * V, V * sizeof(double));
        memcpy(dqq, dq + idx * MAXD * V, D * V * sizeof(double));
        for (int d = 0; d < D; d++) C->F(f + (d * MAXND + idx) * V, qq, dqq, d);
      }
    for (int idx = 0; idx < Nd; idx++) {
      double r[MAXV], qq[MAXV];
      memcpy(qq, qt + idx * V, V * sizeof(double));
      if (C->S)
        C->S(r, qq);
      else
        for (int v = 0; v < V; v++) r[v] = 0.0;
      for (int d = 0; d < D; d++) {
        const double *dqd = dq + (idx * MAXD + d) * V;
        if (C->B) {
          double b[MAXV * MAXV], bd[MAXV];
          C->B(b, qq, d);
          b_times(b, dqd, V, C->b_quirk ? 1 : 0, bd);
          for (int v = 0; v < V; v++) r[v] = r[v] - bd[v];
        }
        if (C->F) {
          double df[MAXV];
          node_deriv(T, f + d * MAXND * V, idx, d, 1.0 / C->dX[d], df);
          for (int v = 0; v < V; v++) r[v] = r[v] - df[v];
        }
      }
      double c = T->w[t];
      for (int d = 0; d < D; d++) c = c * T->w[T->kk[idx][d]];
      double c0 = T->end0[t];
      for (int d = 0; d < D; d++) c0 = c0 * T->w[T->kk[idx][d]];
      for (int v = 0; v < V; v++) {
        double rr = r[v] * c;
        rhs[((long)t * Nd + idx) * V + v] = rr * C->dt + c0 * w[idx * V + v];
      }
    }
  }
}

/* Picard iteration q1 = DG_U^-1 rhs(q0) (dg.cpp:187-202), DG_U = DG_MAT (x) diag W
 * (x) ... (dg.cpp:42-47) applied as DG_MAT^-1 along time and 1/prod W per node.
 * Continues while any |q1 - q0| > DG_TOL (1 + |q0|), at most DG_IT times. */
static int picard_cell(const Ctx *C, const double *w, double *q, double *rhs,
                       double *q1) {
  const Tab *T = C->T;
  int N = T->N, V = T->V, Nd = T->Nd;
  long NTV = (long)T->NT * V;
  int it;
  for (it = 0; it < DG_IT; it++) {
    dg_rhs(C, w, q, rhs);
    int more = 0;
    for (int t = 0; t < N; t++)
      for (int idx = 0; idx < Nd; idx++)
        for (int v = 0; v < V; v++) {
          double acc = T->dginv[t][0] * rhs[(long)idx * V + v];
          for (int s = 1; s < N; s++)
            acc = fma(T->dginv[t][s], rhs[((long)s * Nd + idx) * V + v], acc);
          long e = ((long)t * Nd + idx) * V + v;
          q1[e] = acc * T->IWP[idx];
          if (fabs(q1[e] - q[e]) > DG_TOL * (1.0 + fabs(q[e]))) more = 1;
        }
    if (!more) {
      memcpy(q, q1, NTV * sizeof(double));
      return it + 1;
    }
    memcpy(q, q1, NTV * sizeof(double));
  }
  return it;
}

/* LU with partial pivoting of a V x V matrix, then solve for n right-hand sides
 * x_t = -P^-1 h_t.  Each pivot is inverted once (rd[k] = 1 / u_kk) and the
 * multipliers and the back substitution multiply by it. */
static void lu_solve_neg(int V, double *P, int n, double h[MAXN][MAXV]) {
  int piv[MAXV];
  double rd[MAXV];
  for (int k = 0; k < V; k++) {
    int p = k;
    for (int i = k + 1; i < V; i++)
      if (fabs(P[i * V + k]) > fabs(P[p * V + k])) p = i;
    piv[k] = p;
    if (p != k)
      for (int j = 0; j < V; j++) {
        double t = P[k * V + j];
        P[k * V + j] = P[p * V + j];
        P[p * V + j] = t;
      }
    rd[k] = 1.0 / P[k * V + k];
    for (int i = k + 1; i < V; i++) {
      double l = P[i * V + k] * rd[k];
      P[i * V + k] = l;
      for (int j = k + 1; j < V; j++) P[i * V + j] = fma(-l, P[k * V + j], P[i * V + j]);
    }
  }
  for (int t = 0; t < n; t++) {
    double *b = h[t];
    for (int k = 0; k < V; k++) {
      int p = piv[k];
      if (p != k) {
        double tmp = b[k];
        b[k] = b[p];
        b[p] = tmp;
      }
    }
    for (int i = 1; i < V; i++) {
      double acc = b[i];
      for (int j = 0; j < i; j++) acc = fma(-P[i * V + j], b[j], acc);
      b[i] = acc;
    }
    for (int i = V - 1; i >= 0; i--) {
      double acc = b[i];
      /* b[j] holds x_j = -y_j already */
      for (int j = i + 1; j < V; j++) acc = fma(P[i * V + j], b[j], acc);
      b[i] = -(acc * rd[i]);
    }
  }
}

/* Stiff predictor: Newton iteration on obj(q) = rhs(q) - (DG_MAT (x) W) q = 0
 * (dg.cpp:128-154, whose root the reference finds by Newton-Krylov,
 * dg.cpp:173-185, newton_krylov.cpp:144-183).
 *
 * The Jacobian here keeps the exact time coupling and the stiff source,
 * frozen per spatial node at the time-weighted mean state (flux and B terms
 * lagged):  J = W_x diag(W_t) (x) I (dt JS - Tw), Tw = diag(1/W) DG_MAT, solved
 * through (Tw - A)^-1 = -adj(xI - Tw)(A) p(A)^-1 with A = dt JS (the entries of
 * the polynomial matrix commute).  Where max |A| < NEWTON_A_TINY (the source
 * is not stiff there: unburnt gas with exp(-Ea rho/p) ~ 1e-9) the step uses
 * A = 0 exactly, which costs N^2 V multiply-adds instead of the V x V matrix
 * polynomial and LU.  The fixed point does not depend on J.
 *
 * Learned initial guess (guess != NULL): while the cell is still on its
 * guess, a cell residual max|obj| that is not finite or larger than at the
 * previous iterate abandons the guess; the iteration restarts from the plain
 * guess (w broadcast in time), counting the evaluations already spent.
 * Returns the number of residual evaluations; *fellback reports a restart. */
static void init_guess(const Tab *T, const double *w, double *q);

static int newton_cell(const Ctx *C, const double *w, double *q, double *rhs,
                       int learned, double tol, int maxit, int *fellback) {
  const Tab *T = C->T;
  int N = T->N, V = T->V, Nd = T->Nd;
  double r0 = 0.0;
  int it;
  *fellback = 0;
  for (it = 0; it < maxit; it++) {
    dg_rhs(C, w, q, rhs);
    /* residual G (kept in rhs) and its cell max-norm */
    double rmax = 0.0;
    for (int idx = 0; idx < Nd; idx++) {
      double wp = T->WP[idx];
      for (int t = 0; t < N; t++)
        for (int v = 0; v < V; v++) {
          double acc = (T->dgmat[t][0] * wp) * q[(long)idx * V + v];
          for (int s = 1; s < N; s++)
            acc = fma(T->dgmat[t][s] * wp, q[((long)s * Nd + idx) * V + v], acc);
          long e = ((long)t * Nd + idx) * V + v;
          rhs[e] = rhs[e] - acc;
          double a = fabs(rhs[e]);
          rmax = (a > rmax || a != a) ? a : rmax; /* keeps a NaN */
        }
    }
    if (learned) {
      /* still on the learned guess: a residual that is not finite, or larger
       * than at the previous iterate, abandons the guess */
      if (!(rmax <= (it > 0 ? r0 : DBL_MAX))) {
        init_guess(T, w, q);
        *fellback = 1;
        learned = 0;
        continue;
      }
      r0 = rmax;
    }
    int more = 0;
    for (int idx = 0; idx < Nd; idx++) {
      double g[MAXN][MAXV], h[MAXN][MAXV], qbar[MAXV], JS[MAXV * MAXV], A[MAXV * MAXV],
          P[MAXV * MAXV];
      double wp = T->WP[idx];
      for (int t = 0; t < N; t++)
        for (int v = 0; v < V; v++)
          g[t][v] = rhs[((long)t * Nd + idx) * V + v] * (1.0 / (T->w[t] * wp));
      for (int v = 0; v < V; v++) {
        double acc = T->w[0] * q[(long)idx * V + v];
        for (int t = 1; t < N; t++) acc = fma(T->w[t], q[((long)t * Nd + idx) * V + v], acc);
        qbar[v] = acc;
      }
      if (C->M) {
        C->M(JS, qbar);
      } else if (C->S) {
        double s0[MAXV], s1[MAXV], qq[MAXV];
        memcpy(qq, qbar, V * sizeof(double));
        C->S(s0, qq);
        for (int j = 0; j < V; j++) {
          double q0 = qq[j];
          double hh = fmax(FD_EPS * fabs(q0), FD_EPS);
          qq[j] = q0 + hh;
          C->S(s1, qq);
          qq[j] = q0;
          double rhh = 1.0 / hh;
          for (int i = 0; i < V; i++) JS[i * V + j] = (s1[i] - s0[i]) * rhh;
        }
      } else {
        for (int i = 0; i < V * V; i++) JS[i] = 0.0;
      }
      /* max |dt JS| as |dt| max |JS| (rounding is monotone: the same bits;
       * 0 for a NaN dt, as the NaN-skipping maximum of the products gives) */
      double amax = 0.0;
      for (int i = 0; i < V * V; i++) amax = fmax(amax, fabs(JS[i]));
      amax = fmax(0.0, fabs(C->dt) * amax);
      for (int i = 0; i < V * V; i++) A[i] = C->dt * JS[i];
      if (amax < NEWTON_A_TINY) {
        /* negligible source Jacobian: (Tw - A)^-1 = Tw^-1, i.e. dq_t =
         * -(sum_s M_N[t][s] g_s) (1 / c_0) (the A = 0 case of the general step) */
        for (int t = 0; t < N; t++)
          for (int v = 0; v < V; v++) {
            const double(*Mk)[MAXN] = T->flm[N - 1];
            double acc = Mk[t][0] * g[0][v];
            for (int s2 = 1; s2 < N; s2++) acc = fma(Mk[t][s2], g[s2][v], acc);
            h[t][v] = -(acc * (1.0 / T->flc[0]));
          }
      } else {
        /* h_t = sum_j A^j u_{t,j},  u_{t,j} = sum_s M_{N-j}[t][s] g_s  (Horner in A) */
        for (int t = 0; t < N; t++) {
          for (int j = N - 1; j >= 0; j--) {
            double u[MAXV];
            const double(*Mk)[MAXN] = T->flm[N - j - 1];
            for (int v = 0; v < V; v++) {
              double acc = Mk[t][0] * g[0][v];
              for (int s = 1; s < N; s++) acc = fma(Mk[t][s], g[s][v], acc);
              u[v] = acc;
            }
            if (j == N - 1) {
              for (int v = 0; v < V; v++) h[t][v] = u[v];
            } else {
              double Ah[MAXV];
              for (int i = 0; i < V; i++) {
                double acc = A[i * V] * h[t][0];
                for (int k = 1; k < V; k++) acc = fma(A[i * V + k], h[t][k], acc);
                Ah[i] = acc;
              }
              for (int v = 0; v < V; v++) h[t][v] = Ah[v] + u[v];
            }
          }
        }
        /* P = p(A) = A^N + c_{N-1} A^{N-1} + ... + c_0 I  (Horner) */
        for (int i = 0; i < V * V; i++) P[i] = A[i];
        for (int i = 0; i < V; i++) P[i * V + i] = P[i * V + i] + T->flc[N - 1];
        for (int j = N - 2; j >= 0; j--) {
          double PA[MAXV * MAXV];
          for (int i = 0; i < V; i++)
            for (int k = 0; k < V; k++) {
              double acc = P[i * V] * A[k];
              for (int m = 1; m < V; m++) acc = fma(P[i * V + m], A[m * V + k], acc);
              PA[i * V + k] = acc;
            }
          for (int i = 0; i < V * V; i++) P[i] = PA[i];
          for (int i = 0; i < V; i++) P[i * V + i] = P[i * V + i] + T->flc[j];
        }
        lu_solve_neg(V, P, N, h);
      }
      for (int t = 0; t < N; t++)
        for (int v = 0; v < V; v++) {
          long e = ((long)t * Nd + idx) * V + v;
          if (!(fabs(h[t][v]) <= tol * (1.0 + fabs(q[e])))) more = 1;
          q[e] = q[e] + h[t][v];
        }
    }
    if (!more) return it + 1;
  }
  return it;
}

static void init_guess(const Tab *T, const double *w, double *q) {
  for (int t = 0; t < T->N; t++)
    memcpy(q + (long)t * T->Nd * T->V, w, sizeof(double) * T->Nd * T->V);
}

typedef struct {
  long iters, cells, maxit, capped, fallbacks;
} PredStats;

static int predictor_impl(const Tab *T, oracle_F F, oracle_B B, oracle_S S,
                          oracle_M M, const double *wh, long nw,
                          const double *dX, double dt, int stiff,
                          const oracle_opts *opts, double *qh, int *iters,
                          PredStats *ps) {
  long NTV = (long)T->NT * T->V, NdV = (long)T->Nd * T->V;
  double tol = (opts && opts->newton_tol > 0) ? opts->newton_tol : 1e-12;
  int maxit = (opts && opts->newton_maxit > 0) ? opts->newton_maxit : 100;
  const double *guess = opts ? opts->guess : NULL;
  int gcheck = opts ? opts->guess_check : 0;
  long s_it = 0, s_max = 0, s_cap = 0, s_fb = 0;
#pragma omp parallel reduction(+ : s_it, s_cap, s_fb) reduction(max : s_max)
  {
    double *ws = (double *)malloc(sizeof(double) * (2 * MAXND * MAXD * MAXV + 2 * NTV));
    Ctx C = {T, F, B, S, M, dX, dt, ws, ws + MAXND * MAXD * MAXV, opts ? opts->b_quirk : 0};
    double *rhs = ws + 2 * MAXND * MAXD * MAXV, *q1 = rhs + NTV;
#pragma omp for schedule(dynamic, 16)
    for (long c = 0; c < nw; c++) {
      double *q = qh + c * NTV;
      const double *w = wh + c * NdV;
      int it;
      if (stiff) {
        int fb = 0;
        if (guess) {
          memcpy(q, guess + c * NTV, NTV * sizeof(double));
          it = newton_cell(&C, w, q, rhs, gcheck, tol, maxit, &fb);
        } else {
          init_guess(T, w, q);
          it = newton_cell(&C, w, q, rhs, 0, tol, maxit, &fb);
        }
        s_fb += fb;
        if (it >= maxit) s_cap++;
      } else {
        init_guess(T, w, q);
        it = picard_cell(&C, w, q, rhs, q1);
        if (it >= DG_IT) s_cap++;
      }
      if (iters) iters[c] = it;
      s_it += it;
      if (it > s_max) s_max = it;
    }
    free(ws);
  }
  if (ps) {
    ps->iters += s_it;
    ps->cells += nw;
    if (s_max > ps->maxit) ps->maxit = s_max;
    ps->capped += s_cap;
    ps->fallbacks += s_fb;
  }
  return 0;
}

int oracle_predictor(oracle_F F, oracle_B B, oracle_S S, oracle_M M,
                     const double *wh, long nw, const double *dX, int ndim,
                     int N, int V, double dt, int stiff, const oracle_opts *opts,
                     double *qh, int *iters) {
  Tab T;
  if (tab_init(&T, N, ndim, V)) return 1;
  return predictor_impl(&T, F, B, S, M, wh, nw, dX, dt, stiff, opts, qh, iters,
                        NULL);
}

int oracle_dg_obj(oracle_F F, oracle_B B, oracle_S S, const double *w,
                  const double *q, const double *dX, int ndim, int N, int V,
                  double dt, int b_quirk, double *res) {
  Tab T;
  if (tab_init(&T, N, ndim, V)) return 1;
  double *ws = (double *)malloc(sizeof(double) * 2 * MAXND * MAXD * MAXV);
  Ctx C = {&T, F, B, S, NULL, dX, dt, ws, ws + MAXND * MAXD * MAXV, b_quirk};
  dg_rhs(&C, w, q, res);
  free(ws);
  for (int t = 0; t < N; t++)
    for (int idx = 0; idx < T.Nd; idx++)
      for (int v = 0; v < V; v++) {
        double acc = 0.0;
        for (int s = 0; s < N; s++)
          acc += T.dgmat[t][s] * T.WP[idx] * q[((long)s * T.Nd + idx) * V + v];
        res[((long)t * T.Nd + idx) * V + v] -= acc;
      }
  return 0;
}

/* ------------------------------------------------------------------- FV */

/* Face trace of a cell's space-time tensor: line along axis d through the
 * transverse node j at end e (evaluations.cpp:49-70). */
static void face_trace(const Tab *T, const double *qc, int d, int e, int t,
                       int j, double *out) {
  int N = T->N, V = T->V, D = T->D;
  int stride = ipow(N, D - 1 - d);
  /* node index of (transverse j, k_d = 0): split j into the dims before/after d */
  int hi = j / stride, lo = j % stride;
  int base = hi * stride * N + lo;
  const double *ev = e ? T->end1 : T->end0;
  const double *qt = qc + (long)t * T->Nd * V;
  for (int v = 0; v < V; v++) {
    double acc = ev[0] * qt[base * V + v];
    for (int m = 1; m < N; m++) acc = fma(ev[m], qt[(base + m * stride) * V + v], acc);
    out[v] = acc;
  }
}

/* Gradient at the face point: the derivatives of qh(t) along every d_ at the
 * nodes of the line through transverse node j, extrapolated to side e
 * (fv.cpp:87-122: qh_derivatives, then endpts); out[d_ V + v]. */
static void face_grad_trace(const Tab *T, const double *qc, int d, int e, int t, int j,
                            const double *dX, double *out) {
  int N = T->N, V = T->V, D = T->D;
  int stride = ipow(N, D - 1 - d);
  int hi = j / stride, lo = j % stride;
  int base = hi * stride * N + lo;
  const double *ev = e ? T->end1 : T->end0;
  const double *qt = qc + (long)t * T->Nd * V;
  for (int d_ = 0; d_ < D; d_++) {
    double g[MAXN][MAXV];
    for (int m = 0; m < N; m++) node_deriv(T, qt, base + m * stride, d_, 1.0 / dX[d_], g[m]);
    for (int v = 0; v < V; v++) {
      double acc = ev[0] * g[0][v];
      for (int m = 1; m < N; m++) acc = fma(ev[m], g[m][v], acc);
      out[d_ * V + v] = acc;
    }
  }
}

/* f = D(qL, qR) + (F(qL) + F(qR)) (fluxes.cpp:79-101) with the dissipation
 *   Rusanov (0): max(lam(qL), lam(qR)) (qL - qR)           (fluxes.cpp:72-77)
 *   Roe (1):     |sum_i W_i A(q_i)| (qL - qR)               (fluxes.cpp:47-70)
 *   Osher (2):   sum_i W_i |A(q_i)| (qL - qR)               (fluxes.cpp:20-45)
 * on the path q_i = qR + x_i (qL - qR), dq_i = dqR + x_i (dqL - dqR),
 * A = dF/dQ + B, and with a viscous F (second) + max(lam2(qL), lam2(qR))
 * (qL - qR) (fluxes.cpp:96-100); Bint = (sum_i W_i B(qL + x_i (qR - qL)))
 * (qR - qL) (fluxes.cpp:103-116). */
static void face_flux(const Tab *T, oracle_F F, oracle_B B, int flux,
                      const double *qL, const double *qR, const double *dqL,
                      const double *dqR, int second, const double *dX, int d, double *f,
                      double *bint) {
  int V = T->V, N = T->N, D = T->D;
  if (F && flux == 0) {
    double fl[MAXV], fr[MAXV];
    double l1 = max_abs_eigs(F, B, qL, dqL, d, V, fl);
    double l2 = max_abs_eigs(F, B, qR, dqR, d, V, fr);
    double s = fmax(l1, l2);
    for (int v = 0; v < V; v++) f[v] = s * (qL[v] - qR[v]) + (fl[v] + fr[v]);
  } else if (F) {
    double fl[MAXV], fr[MAXV], Dq[MAXV], q[MAXV], A[MAXV * MAXV], Mx[MAXV * MAXV], y[MAXV],
        Dsum[MAXV], ftmp[MAXV], dq[MAXD * MAXV] = {0}, qq[MAXV], dqq[MAXD * MAXV] = {0};
    memcpy(qq, qL, V * sizeof(double));
    memcpy(dqq, dqL, D * V * sizeof(double));
    F(fl, qq, dqq, d);
    memcpy(qq, qR, V * sizeof(double));
    memcpy(dqq, dqR, D * V * sizeof(double));
    F(fr, qq, dqq, d);
    for (int v = 0; v < V; v++) Dq[v] = qL[v] - qR[v];
    for (int i = 0; i < N; i++) {
      for (int v = 0; v < V; v++) q[v] = fma(T->x[i], Dq[v], qR[v]);
      for (int k = 0; k < D * V; k++) dq[k] = fma(T->x[i], dqL[k] - dqR[k], dqR[k]);
      system_matrix(F, B, q, dq, d, V, A, ftmp);
      if (flux == 1) {
        for (int k = 0; k < V * V; k++) Mx[k] = (i == 0) ? T->w[0] * A[k] : fma(T->w[i], A[k], Mx[k]);
      } else {
        oracle_abs_apply(A, Dq, V, y);
        for (int v = 0; v < V; v++) Dsum[v] = (i == 0) ? T->w[0] * y[v] : fma(T->w[i], y[v], Dsum[v]);
      }
    }
    if (flux == 1) oracle_abs_apply(Mx, Dq, V, Dsum);
    for (int v = 0; v < V; v++) f[v] = Dsum[v] + (fl[v] + fr[v]);
  } else {
    for (int v = 0; v < V; v++) f[v] = 0.0;
  }
  if (F && second) {
    double m1 = max_abs_eigs_second_order(F, qL, dqL, d, V, N, dX);
    double m2 = max_abs_eigs_second_order(F, qR, dqR, d, V, N, dX);
    double s2 = fmax(m1, m2);
    for (int v = 0; v < V; v++) f[v] = f[v] + s2 * (qL[v] - qR[v]);
  }
  if (B) {
    double Dq[MAXV], Mx[MAXV * MAXV], b[MAXV * MAXV], q[MAXV];
    for (int v = 0; v < V; v++) Dq[v] = qR[v] - qL[v];
    for (int i = 0; i < N; i++) {
      for (int v = 0; v < V; v++) q[v] = fma(T->x[i], Dq[v], qL[v]);
      B(b, q, d);
      for (int k = 0; k < V * V; k++) Mx[k] = (i == 0) ? T->w[0] * b[k] : fma(T->w[i], b[k], Mx[k]);
    }
    for (int v = 0; v < V; v++) {
      double acc = Mx[v * V] * Dq[0];
      for (int k = 1; k < V; k++) acc = fma(Mx[v * V + k], Dq[k], acc);
      bint[v] = acc;
    }
  } else {
    for (int v = 0; v < V; v++) bint[v] = 0.0;
  }
}

/* Volume term (fv.cpp:33-85): sum over nodes of dt W_t prod W_x (S(qh) - sum_d
 * B_d(qh) d_d qh).  Summed per spatial node over t, then over nodes. */
static void cell_volume(const Tab *T, oracle_F F, oracle_B B, oracle_S S,
                        const double *qc, const double *dX, double dt, int quirk,
                        double *vol) {
  int N = T->N, V = T->V, D = T->D, Nd = T->Nd;
  (void)F;
  for (int v = 0; v < V; v++) vol[v] = 0.0;
  for (int idx = 0; idx < Nd; idx++) {
    double part[MAXV];
    for (int t = 0; t < N; t++) {
      const double *qt = qc + (long)t * Nd * V;
      double s[MAXV], qq[MAXV];
      memcpy(qq, qt + idx * V, V * sizeof(double));
      if (S)
        S(s, qq);
      else
        for (int v = 0; v < V; v++) s[v] = 0.0;
      if (B)
        for (int d = 0; d < D; d++) {
          double dqd[MAXV], b[MAXV * MAXV], bd[MAXV];
          node_deriv(T, qt, idx, d, 1.0 / dX[d], dqd);
          B(b, qq, d);
          b_times(b, dqd, V, quirk ? 2 : 0, bd);
          for (int v = 0; v < V; v++) s[v] = s[v] - bd[v];
        }
      double tmp = dt * T->w[t];
      for (int d = 0; d < D; d++) tmp = tmp * T->w[T->kk[idx][d]];
      for (int v = 0; v < V; v++) part[v] = (t == 0) ? tmp * s[v] : fma(tmp, s[v], part[v]);
    }
    for (int v = 0; v < V; v++) vol[v] = (idx == 0) ? part[v] : vol[v] + part[v];
  }
}

/* Corrector (fv.cpp:200-207 = centers then interfaces, fv.cpp:124-198).  For
 * an interior cell c the reference's face-cell loop visits, in order, the
 * faces c+1-e_d (c on the right, d = 0..D-1, each over t then transverse
 * node) and then the face-cell c+1 (c on the left, over t, then d, then
 * transverse node).  Face fluxes are evaluated once per face point and then
 * gathered per cell in exactly that order. */
static int fv_impl(oracle_F F, oracle_B B, oracle_S S, double *u, const double *qh,
                   const int *nX, int ndim, const double *dX, int flux, int N, int V,
                   double dt, int b_quirk, int second) {
  Tab T;
  if (tab_init(&T, N, ndim, V)) return 1;
  int D = ndim, Nd1 = T.Nd1;
  long NTV = (long)T.NT * V;
  int n2[MAXD];
  long ncell = 1;
  for (int d = 0; d < D; d++) {
    n2[d] = nX[d] + 2;
    ncell *= nX[d];
  }
  /* face arrays per d: shape (nX_d + 1) along d, nX_d' across; entries
   * [face][t][j][v] */
  double *ff[MAXD], *fb[MAXD];
  long nface[MAXD];
  for (int d = 0; d < D; d++) {
    long nf = 1;
    for (int e = 0; e < D; e++) nf *= (e == d) ? nX[e] + 1 : nX[e];
    nface[d] = nf;
    ff[d] = (double *)malloc(sizeof(double) * nf * N * Nd1 * V);
    fb[d] = (double *)malloc(sizeof(double) * nf * N * Nd1 * V);
#pragma omp parallel for schedule(dynamic, 64)
    for (long f = 0; f < nf; f++) {
      int fc[MAXD];
      long r = f;
      for (int e = D - 1; e >= 0; e--) {
        int ext = (e == d) ? nX[e] + 1 : nX[e];
        fc[e] = (int)(r % ext);
        r /= ext;
      }
      /* left w-cell (nX+2 coordinates) = face-cell F with F_e = fc_e + 1 across */
      long wl = 0, wr = 0;
      for (int e = 0; e < D; e++) {
        int Fe = (e == d) ? fc[e] : fc[e] + 1;
        wl = wl * n2[e] + Fe;
        wr = wr * n2[e] + Fe + (e == d);
      }
      for (int t = 0; t < N; t++)
        for (int j = 0; j < Nd1; j++) {
          double qL[MAXV], qR[MAXV], dqL[MAXD * MAXV] = {0}, dqR[MAXD * MAXV] = {0};
          face_trace(&T, qh + wl * NTV, d, 1, t, j, qL);
          face_trace(&T, qh + wr * NTV, d, 0, t, j, qR);
          if (second) {
            face_grad_trace(&T, qh + wl * NTV, d, 1, t, j, dX, dqL);
            face_grad_trace(&T, qh + wr * NTV, d, 0, t, j, dX, dqR);
          }
          long o = ((f * N + t) * Nd1 + j) * V;
          face_flux(&T, F, B, flux, qL, qR, dqL, dqR, second, dX, d, ff[d] + o, fb[d] + o);
        }
    }
  }
#pragma omp parallel for schedule(static)
  for (long c = 0; c < ncell; c++) {
    int cc[MAXD];
    long r = c;
    for (int e = D - 1; e >= 0; e--) {
      cc[e] = (int)(r % nX[e]);
      r /= nX[e];
    }
    double *uc = u + c * V;
    if (B || S) {
      long wc = 0;
      for (int e = 0; e < D; e++) wc = wc * n2[e] + cc[e] + 1;
      double vol[MAXV];
      cell_volume(&T, F, B, S, qh + wc * NTV, dX, dt, b_quirk, vol);
      for (int v = 0; v < V; v++) uc[v] = uc[v] + vol[v];
    }
    if (!(F || B)) continue;
    long fidx[2][MAXD];
    for (int d = 0; d < D; d++)
      for (int side = 0; side < 2; side++) {
        long f = 0;
        for (int e = 0; e < D; e++) {
          int ext = (e == d) ? nX[e] + 1 : nX[e];
          int fe = cc[e] + ((e == d) ? side : 0);
          f = f * ext + fe;
        }
        fidx[side][d] = f;
      }
    /* c is the right cell of faces c+1-e_d */
    for (int d = 0; d < D; d++)
      for (int t = 0; t < N; t++) {
        double c0 = (dt * T.w[t]) / (2.0 * dX[d]);
        for (int j = 0; j < Nd1; j++) {
          double tmp = c0;
          int rr = j;
          int jj[MAXD];
          for (int i = D - 2; i >= 0; i--) {
            jj[i] = rr % N;
            rr /= N;
          }
          for (int i = 0; i < D - 1; i++) tmp = tmp * T.w[jj[i]];
          long o = ((fidx[0][d] * N + t) * Nd1 + j) * V;
          for (int v = 0; v < V; v++) uc[v] = uc[v] - tmp * (fb[d][o + v] - ff[d][o + v]);
        }
      }
    /* c is the left cell of face-cell c+1 */
    for (int t = 0; t < N; t++)
      for (int d = 0; d < D; d++) {
        double c0 = (dt * T.w[t]) / (2.0 * dX[d]);
        for (int j = 0; j < Nd1; j++) {
          double tmp = c0;
          int rr = j;
          int jj[MAXD];
          for (int i = D - 2; i >= 0; i--) {
            jj[i] = rr % N;
            rr /= N;
          }
          for (int i = 0; i < D - 1; i++) tmp = tmp * T.w[jj[i]];
          long o = ((fidx[1][d] * N + t) * Nd1 + j) * V;
          for (int v = 0; v < V; v++) uc[v] = uc[v] - tmp * (fb[d][o + v] + ff[d][o + v]);
        }
      }
  }
  for (int d = 0; d < D; d++) {
    free(ff[d]);
    free(fb[d]);
  }
  return 0;
}

int oracle_fv(oracle_F F, oracle_B B, oracle_S S, double *u, const double *qh,
              const int *nX, int ndim, const double *dX, int flux, int N, int V,
              double dt, int b_quirk) {
  return fv_impl(F, B, S, u, qh, nX, ndim, dX, flux, N, V, dt, b_quirk, 0);
}

/* ---------------------------------------------------------------- driver */

/* Time loop of iterator.cpp:38-151 (serial over the whole grid; the reference's
 * slab split changes no arithmetic). */
int oracle_pde_solver(oracle_F F, oracle_B B, oracle_S S, oracle_M M, int useF,
                      int useB, int useS, double *u, double tf, const int *nX,
                      int ndim, const double *dX, double CFL, const int *bc,
                      int stiff, int flux, int N, int V, int ndt,
                      int secondOrder, double *ret, const oracle_opts *opts,
                      oracle_stats *stats) {
  if (!useF) F = NULL;
  if (!useB) B = NULL;
  if (!useS) S = NULL;
  if (!S) M = NULL;
  if (flux < 0 || flux > 2) return 11; /* Rusanov, Roe, Osher */
  if (ndt < 1) return 12;
  Tab T;
  if (tab_init(&T, N, ndim, V)) return 13;
  for (int d = 0; d < ndim; d++)
    if (bc[d] < 0 || bc[d] > 2) return 14;
  long ncell = 1, nub = 1, nw = 1;
  int nb[MAXD];
  for (int d = 0; d < ndim; d++) {
    ncell *= nX[d];
    nb[d] = nX[d] + 2 * N;
    nub *= nb[d];
    nw *= nX[d] + 2;
  }
  long NTV = (long)T.NT * V;
  double *ub = (double *)malloc(sizeof(double) * nub * V);
  double *qh = (double *)malloc(sizeof(double) * nw * NTV);
  const double *reflect = opts ? opts->reflect : NULL;
  long max_steps = opts ? opts->max_steps : 0;
  double t = 0.0;
  long count = 0;
  int push = 0, rc = 0;
  PredStats ps = {0, 0, 0, 0, 0};
  while (t < tf && (max_steps <= 0 || count < max_steps)) {
    oracle_boundaries(ub, u, nX, ndim, bc, reflect, N, V);
    double *wh = weno_sweeps(&T, ub, nb);
    double dt = timestep_impl(F, B, wh, nw, dX, ndim, N, V, CFL, tf, t, count, secondOrder);
    predictor_impl(&T, F, B, S, M, wh, nw, dX, dt, stiff, opts, qh, NULL, &ps);
    free(wh);
    fv_impl(F, B, S, u, qh, nX, ndim, dX, flux, N, V, dt, opts ? opts->b_quirk : 0, secondOrder);
    t += dt;
    count += 1;
    if (push < ndt && t >= (double)(push + 1) / (double)ndt * tf) {
      memcpy(ret + (long)push * ncell * V, u, sizeof(double) * ncell * V);
      push += 1;
    }
    int bad = 0;
    for (long i = 0; i < ncell * V; i++)
      if (u[i] != u[i]) bad = 1;
    if (bad) {
      rc = -(int)count;
      break;
    }
  }
  memcpy(ret + (long)(ndt - 1) * ncell * V, u, sizeof(double) * ncell * V);
  if (stats) {
    stats->steps = count;
    stats->t = t;
    stats->pred_iters = ps.iters;
    stats->pred_cells = ps.cells;
    stats->pred_maxit = ps.maxit;
    stats->pred_capped = ps.capped;
    stats->guess_fallbacks = ps.fallbacks;
  }
  free(ub);
  free(qh);
  return rc;
}
