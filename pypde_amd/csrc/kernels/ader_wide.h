// Wave speeds of systems with more than eight variables on small grids, one
// wavefront per matrix.  Compiled by hipRTC after ader_common.h where
// PDE_WIDE_EIG (or, for the helpers, PDE_WIDE_PRED) is 1.
//
// One lane per matrix, which larger grids take (wide_matrices in tune.h gives the
// line), leaves a small grid waiting: a 17 x 17 matrix and its reduction need
// some 600 registers, so they live in scratch (4-8 KB per lane), and a 200-cell
// line has only 402 face points, seven wavefronts on the whole GPU, each a serial
// chain of spilled accesses.  Here the matrix
// lies in LDS, lane j works on column j (left products, Jacobian columns) or
// row j (right products), and scalars are formed by every lane alike.  What
// bounds it is the latency of the dependent chains (Householder sums, Horner
// steps, QR sweeps), hidden only by other wavefronts.  On the 17-variable
// model, 200 cells, order 2, a launch: face flux 1340 -> 88.5 us and timestep
// 726 -> 72 us (a matrix takes about 19,000 cycles to reduce, 5,300 for its
// characteristic polynomial, 3,500 for the roots, 3,000 for the certificate
// and, for the half of them that need it, 88,000 for QR).
//
// Every sum keeps the order of the one-lane routines (fma chains from the
// first product), so the results are the same bits.
#pragma once

constexpr int VP = V | 1;  // LDS row stride in doubles: odd, so columns meet no bank conflicts
constexpr int WIDE_WAVES = 4;  // wavefronts (matrices) per workgroup of k_dt and k_eig_batch

struct WideMat {
  double H[V][VP];       // the matrix, destroyed
  double P[V + 1][VP + 1];  // leading principal minors' characteristic polynomials
};

// Orders this wavefront's LDS accesses (performed in issue order) for the compiler.
DEV void wide_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

DEV double wide_max(double x) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) x = dmax(x, __shfl_xor(x, o, 64));
  return x;
}

// Householder reduction of W.H to upper Hessenberg form (eig_prepare's loop),
// every index static: lane j takes column j of each left product and lane i
// row i of each right product.  The next reflector's column and the lane's own
// are read together, so a step meets two LDS round trips.  48,000
// -> 19,000 cycles against a loop over k with bounds on every row.
DEV void wide_hessenberg(WideMat& W, int lane) {
  static_for<0, V - 2>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
    constexpr int m = V - k - 1;
    const int own = lane < V ? lane : V - 1;
    double x[m], v[m], h[m];
#pragma unroll
    for (int i = 0; i < m; i++) x[i] = W.H[k + 1 + i][k];
#pragma unroll
    for (int i = 0; i < m; i++) h[i] = W.H[k + 1 + i][own];
    double mu, beta;
    if (house1<m>(x, v, &beta, &mu)) {
      auto reflect = [&]() {
        double s = v[0] * h[0];
#pragma unroll
        for (int i = 1; i < m; i++) s = dfma(v[i], h[i], s);
        s = beta * s;
#pragma unroll
        for (int i = 0; i < m; i++) h[i] = dfma(-s, v[i], h[i]);
      };
      reflect();
      if (lane > k && lane < V) {
#pragma unroll
        for (int i = 0; i < m; i++) W.H[k + 1 + i][lane] = h[i];
        W.H[lane][k] = lane == k + 1 ? mu : 0.0;
      }
      wide_sync();
#pragma unroll
      for (int j = 0; j < m; j++) h[j] = W.H[own][k + 1 + j];
      reflect();
      if (lane < V) {
#pragma unroll
        for (int j = 0; j < m; j++) W.H[lane][k + 1 + j] = h[j];
      }
      wide_sync();
    }
  });
}

// Value of the lane below (lane 0: its own), over the whole wavefront.
DEV double lane_below(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, 0x138, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), 0x138, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Coefficients c[0..V] of det(xI - H), H upper Hessenberg (hess_charpoly).
// Lane k forms the multipliers t_m of minor k (W.P[k][m]); then lane i carries
// coefficient i of every minor's polynomial in registers (33,000 -> 5,300
// cycles against polynomials in LDS).  A polynomial is 0 above its degree, so
// terms beyond it add nothing.
DEV void wide_charpoly(WideMat& W, int lane, double (&c)[V + 1]) {
  if (lane >= 1 && lane <= V) {
    double prod = 1.0;
#pragma unroll
    for (int m = 1; m < V; m++) {
      const int r = lane - m > 0 ? lane - m : 1;  // (unused past m = lane - 1)
      prod = prod * W.H[r][r - 1];
      W.P[lane][m] = W.H[r - 1][lane - 1] * prod;
    }
    W.P[lane][0] = W.H[lane - 1][lane - 1];
  }
  wide_sync();
  double p[V + 1];
  p[0] = lane == 0 ? 1.0 : 0.0;
#pragma unroll
  for (int k = 1; k <= V; k++) {
    const double below = lane_below(p[k - 1]);
    double v = lane >= 1 ? below : 0.0;
    v = dfma(-W.P[k][0], p[k - 1], v);
#pragma unroll
    for (int m = 1; m <= k - 1; m++) v = dfma(-W.P[k][m], p[k - m - 1], v);
    p[k] = v;
  }
  wide_sync();
  if (lane <= V) W.P[0][lane] = p[V];
  wide_sync();
#pragma unroll
  for (int j = 0; j <= V; j++) c[j] = W.P[0][j];
}

// Starting points of the root iterations (charpoly_setup).
DEV void wide_root_starts(const WideMat& W, const double (&c)[V + 1], int lane, double* xhi,
                          double* xlo) {
  constexpr double inv_v = 1.0 / (double)V;
  const double mu = -(c[V - 1] * inv_v);
  const double s2 = dfma(-mu, mu, dfma(c[V - 1], c[V - 1], -2.0 * c[V - 2]) * inv_v);
  if (s2 > 0.0 && s2 <= 1e300) {
    const double w = 1.001 * dsqrt(s2 * (0.5 * (double)V));
    *xhi = mu + w;
    *xlo = mu - w;
    return;
  }
  double rs = 0.0;
  if (lane < V) {
#pragma unroll
    for (int j = 0; j < V; j++) rs = rs + dabs(W.H[lane][j]);
  }
  const double u = wide_max(dmax(0.0, rs));
  *xhi = u;
  *xlo = -u;
}

// house<M>, every lane alike, with both forms of v0 computed and one selected.
// *head receives sqrt(x0^2 + (x1^2 (+ x2^2))), the entry the reflector leaves,
// whose square root overlaps the others'.  Its chain of a square root and two
// divisions is much of what a step of the QR waits for: without operand scaling
// (sqrt_mid, in house's range) face flux 92 -> 88.5 us, timestep 75 -> 72 us.
template <int M>
DEV double wide_house(const double (&x)[3], double (&v)[3], double* head) {
  double sigma = x[1] * x[1];
  double tail = sigma;
  if (M == 3) {
    sigma = dfma(x[2], x[2], sigma);
    tail = tail + x[2] * x[2];
  }
  const double mu2 = dfma(x[0], x[0], sigma), h2 = x[0] * x[0] + tail;
  v[1] = x[1];
  v[2] = x[2];
  if ((sigma > HOUSE_TINY) & (mu2 <= 0x1p60)) {
    const double mu = sqrt_mid(mu2);
    *head = sqrt_mid(h2);
    const double low = x[0] - mu, high = -div_mid(sigma, x[0] + mu);
    const double v0 = x[0] <= 0.0 ? low : high;
    v[0] = v0;
    return 2.0 * recip_mid(dfma(v0, v0, sigma));
  }
  const double mu = dsqrt(mu2);
  *head = dsqrt(h2);
  const double low = x[0] - mu, high = -sigma / (x[0] + mu);
  const double v0 = x[0] <= 0.0 ? low : high;
  v[0] = v0;
  const double beta = 2.0 / dfma(v0, v0, sigma);
  return sigma <= HOUSE_TINY ? 0.0 : beta;
}

// Francis double-shift QR on the scaled Hessenberg W.H (eig_qr): max |lambda|
// in the scaled units.
DEV double wide_qr(WideMat& W, int lane) {
  auto H = [&](int i, int j) -> double { return W.H[i][j]; };
  // entry of the column a right product just left in registers, from its row's lane
  auto pick = [](double x, int from) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane((int)b, from);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), from);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
  };
  double anorm = 0.0;
#pragma unroll 1
  for (int i = 0; i < V; i++)
#pragma unroll
    for (int j = 0; j < V; j++) anorm = anorm + dabs(W.H[i][j]);
  double best = 0.0, ex = 0.0;
  int hi = V - 1, iter = 0, total = 0;
  while (hi >= 0) {
    // the largest l <= hi whose subdiagonal entry is negligible
    bool small = false;
    if (lane >= 1 && lane <= hi) {
      double s = dabs(W.H[lane - 1][lane - 1]) + dabs(W.H[lane][lane]);
      if (s == 0.0) s = anorm;
      small = dabs(W.H[lane][lane - 1]) <= 2.220446049250313e-16 * s;
    }
    const unsigned long long mask = __ballot(small);
    const int lo = mask ? 63 - __builtin_clzll(mask) : 0;
    if (mask && lane == lo) W.H[lane][lane - 1] = 0.0;
    wide_sync();
    if (lo == hi) {
      best = dmax(best, dabs(H(hi, hi) + ex));
      hi -= 1;
      iter = 0;
      continue;
    }
    if (lo == hi - 1) {
      const double a = H(hi - 1, hi - 1) + ex, b = H(hi - 1, hi);
      const double c = H(hi, hi - 1), dd = H(hi, hi) + ex;
      const double p = 0.5 * (a - dd);
      const double bc = b * c;
      const double disc = p * p + bc;
      if (disc >= 0.0) {
        double z = dsqrt(disc);
        z = (p >= 0.0) ? p + z : p - z;
        const double l1 = dd + z;
        const double l2 = (z != 0.0) ? dd - bc / z : dd;
        best = dmax(best, dmax(dabs(l1), dabs(l2)));
      } else {
        const double re = dd + p;
        best = dmax(best, dsqrt(re * re - disc));
      }
      hi -= 2;
      iter = 0;
      continue;
    }
    if (total >= 40 * V) {
#pragma unroll 1
      for (int i = 0; i <= hi; i++) best = dmax(best, dabs(H(i, i) + ex));
      break;
    }
    double sx = H(hi, hi), sy = H(hi - 1, hi - 1);
    double sw = H(hi, hi - 1) * H(hi - 1, hi);
    auto shift_diagonal = [&](double s) {
      wide_sync();
      if (lane <= hi) W.H[lane][lane] = W.H[lane][lane] - s;
      wide_sync();
    };
    if (iter == 10) {
      ex = ex + sx;
      const double s = dabs(H(hi, hi - 1)) + dabs(H(hi - 1, hi - 2));
      shift_diagonal(sx);
      sx = 0.75 * s;
      sy = sx;
      sw = -0.4375 * s * s;
    } else if (iter == 30) {
      double s = (sy - sx) / 2.0;
      s = s * s + sw;
      if (s > 0.0) {
        s = dsqrt(s);
        if (sy < sx) s = -s;
        s = s + (sy - sx) / 2.0;
        s = sx - sw / s;
        ex = ex + s;
        shift_diagonal(s);
        sx = 0.964;
        sy = 0.964;
        sw = 0.964;
      }
    }
    iter++;
    total++;
    const double h00 = H(lo, lo);
    const double r = sx - h00, q = sy - h00;
    double x[3], v[3];
    x[0] = (r * q - sw) / H(lo + 1, lo) + H(lo, lo + 1);
    x[1] = H(lo + 1, lo + 1) - h00 - r - q;
    x[2] = H(lo + 2, lo + 1);
    // one reflector per row k: this lane's column of the left product is read
    // while the reflector is formed; the column that holds the next one's
    // entries is then in the lanes' registers
    auto chase = [&](int k, auto mc) {
      constexpr int m = decltype(mc)::value;
      const int own = lane < V ? lane : V - 1;
      double h[m];
#pragma unroll
      for (int i = 0; i < m; i++) h[i] = W.H[k + i][own];
      double head;
      const double beta = wide_house<m>(x, v, &head);
      double first = 0.0;  // H[lane][k] after this step
      if (beta != 0.0) {
        auto reflect = [&]() {
          double s = v[0] * h[0];
#pragma unroll
          for (int i = 1; i < m; i++) s = dfma(v[i], h[i], s);
          s = beta * s;
#pragma unroll
          for (int i = 0; i < m; i++) h[i] = dfma(-s, v[i], h[i]);
        };
        if (k > lo && lane < m) W.H[k + lane][k - 1] = lane == 0 ? head : 0.0;
        reflect();
        if (lane >= k && lane <= hi) {
#pragma unroll
          for (int i = 0; i < m; i++) W.H[k + i][lane] = h[i];
        }
        wide_sync();
        const int rr = (k + 3 < hi) ? k + 3 : hi;
#pragma unroll
        for (int j = 0; j < m; j++) h[j] = W.H[own][k + j];
        first = h[0];
        reflect();
        if (lane >= lo && lane <= rr) {
#pragma unroll
          for (int j = 0; j < m; j++) W.H[lane][k + j] = h[j];
          first = h[0];
        }
        wide_sync();
      } else {
        first = W.H[own][k];
      }
      if (m == 3) {
        x[0] = pick(first, k + 1);
        x[1] = pick(first, k + 2);
        x[2] = k + 3 < V ? pick(first, k + 3) : 0.0;
      }
    };
#pragma unroll 1
    for (int k = lo; k <= hi - 2; k++) chase(k, IC<3>{});
    chase(hi - 1, IC<2>{});
  }
  return best;
}

// max |lambda| of the matrix whose column `lane` is col (lanes >= V hold
// none): max_abs_eig over one wavefront, every lane returning the result.
DEV double wide_max_abs_eig(WideMat& W, const double (&col)[V], int lane) {
  double scale = 0.0;
  if (lane < V) {
#pragma unroll
    for (int r = 0; r < V; r++) scale = dmax(scale, dabs(col[r]));
  }
  scale = wide_max(scale);
  if (!(scale >= 2.2250738585072014e-308)) return (scale != scale) ? scale : 0.0;
  int e2;
  (void)__builtin_frexp(scale, &e2);
  const double pw = __builtin_ldexp(1.0, -e2);
  wide_sync();
  if (lane < V) {
#pragma unroll
    for (int r = 0; r < V; r++) W.H[r][lane] = col[r] * pw;
  }
  wide_sync();
  wide_hessenberg(W, lane);
  {
    // the two extreme roots iterate side by side: even lanes the largest, odd
    // lanes the smallest
    double c[1][V + 1], x0[1], root[1], dp[1], xhi, xlo, r;
    bool ok[1];
    wide_charpoly(W, lane, c[0]);
    wide_root_starts(W, c[0], lane, &xhi, &xlo);
    x0[0] = (lane & 1) ? xlo : xhi;
    real_roots<1>(c, x0, root, dp, ok);
    const double l1 = __shfl(root[0], 0, 64), l2 = __shfl(root[0], 1, 64);
    const double d1 = __shfl(dp[0], 0, 64), d2 = __shfl(dp[0], 1, 64);
    const bool both = (__ballot(ok[0]) & 3ull) == 3ull;
    if (both && charpoly_certify(c[0], l1, l2, d1, d2, &r)) return __builtin_ldexp(r, e2);
  }
  return __builtin_ldexp(wide_qr(W, lane), e2);
}

// Column `lane` of A = dF/dQ + B(q, d) by forward differences
// (system_matrix); f0 receives F(q).  q and dq are the same in every lane.  B
// is written once, to LDS (over W.P).
DEV void wide_system_column(WideMat& W, const double* q, const double* dq, int d, int lane,
                            double (&col)[V], double* f0) {
#if PDE_USE_F
  double v1[V], v2[V], m[V], rh[V], qq[V];
  F(v1, q, dq, d);
  fd_recips(q, m, rh);
  double r1 = 0.0;
#pragma unroll
  for (int i = 0; i < V; i++) {
    qq[i] = i == lane ? dfma(FD_EPS, m[i], q[i]) : q[i];
    r1 = i == lane ? rh[i] : r1;
  }
  F(v2, qq, dq, d);
#pragma unroll
  for (int r = 0; r < V; r++) {
    col[r] = (v2[r] - v1[r]) * r1;
    f0[r] = v1[r];
  }
#else
#pragma unroll
  for (int r = 0; r < V; r++) {
    col[r] = 0.0;
    f0[r] = 0.0;
  }
#endif
#if PDE_USE_B
  double* const b = &W.P[0][0];
  wide_sync();
  if (lane == 0) B(b, q, d);
  wide_sync();
#pragma unroll
  for (int r = 0; r < V; r++) col[r] = col[r] + b[r * V + (lane < V ? lane : 0)];
#endif
}

DEV double wide_max_abs_eigs(WideMat& W, const double* q, const double* dq, int d, int lane,
                             double* f0) {
  double col[V];
  wide_system_column(W, q, dq, d, lane, col, f0);
  return wide_max_abs_eig(W, col, lane);
}
