// Space-time predictor of systems with more than eight variables, one
// wavefront per cell.  Compiled by hipRTC after ader_step.h where PDE_WIDE_PRED
// is 1: on small grids, and for stiff systems of 14 variables and more on all.
//
// With one lane per spatial node the 17-variable stiff Newton step
// holds three 17 x 17 matrices per lane, 10,000 spilled registers, and 202
// cells of two nodes fill seven wavefronts.  Here a cell's iterate lies in
// LDS: F and S run with one lane per space-time node, everything elementwise
// with one lane per (node, variable), and the Newton step of a node with half
// a wavefront, lane j holding column j of the matrices (so that a pivot is
// found in one lane's registers).  What bounds it is the latency of those
// chains (the source Jacobian's S evaluation, the LU, the back substitution).
// 17-variable model, 200 cells, order 2, stiff: 1530 -> 114 us a launch.
//
// Every sum keeps the order of node_rhs and newton_node, so the results are
// the same bits.
#pragma once

// time nodes whose F is staged at once: all of them where they take 24 KB or less
constexpr int WIDE_T = D * NT * V <= 3072 ? N : 1;

struct WideGroup {
  double A[V][VP];  // source Jacobian, then U; also B or M as the system writes it
  double P[V][VP];  // p(A); row k then the multipliers of LU step k
  double row[V];    // 1 / pivot
  double h[N][V];   // Horner vectors, then the solution
  double qbar[V], s0[V];
};
struct WidePred {
  double q[N][ND][V], r[N][ND][V], w[ND][V];
  double f[D][WIDE_T][ND][V];
  WideGroup grp[2];
};

DEV double wide_weight(int node) {  // prod_d W[k_d]
  double p = 0.0;
#pragma unroll
  for (int d = 0; d < D; d++) {
    const double w = tw((node / ipow_c(N, D - 1 - d)) % N);
    p = d == 0 ? w : p * w;
  }
  return p;
}
// a prod_d W[k_d], the products in the order d = 0, 1
DEV double wide_scaled(double a, int node) {
#pragma unroll
  for (int d = 0; d < D; d++) a = a * tw((node / ipow_c(N, D - 1 - d)) % N);
  return a;
}
// derivative along d at a node of buf[node][v]
template <int d>
DEV double wide_deriv(const double (*buf)[V], int node, int v, double rdx) {
  constexpr int stride = ipow_c(N, D - 1 - d);
  const int kd = (node / stride) % N, base = node - kd * stride;
  double acc = tder(kd, 0) * buf[base][v];
#pragma unroll
  for (int j = 1; j < N; j++) acc = dfma(tder(kd, j), buf[base + j * stride][v], acc);
  return acc * rdx;
}

// sm.r = S(q) (r_out) and sm.f = F(q) for time nodes t0 .. t0 + nt - 1, one
// lane per space-time node.
DEV void wide_eval(WidePred& sm, int t0, int nt, bool with_f, const Geom& g, int lane) {
#pragma unroll 1
  for (int i = lane; i < nt * ND; i += 64) {
    const int tt = i / ND, node = i % ND, t = t0 + tt;
    double q[V], out[V];
#pragma unroll
    for (int v = 0; v < V; v++) q[v] = sm.q[t][node][v];
    callS(out, q);
#pragma unroll
    for (int v = 0; v < V; v++) sm.r[t][node][v] = out[v];
#if PDE_USE_F
    if (with_f) {
      double dq[D * V];
#pragma unroll
      for (int k = 0; k < D * V; k++) dq[k] = 0.0;
      if constexpr (PRED_DQ)
        static_for<0, D>([&](auto dc) {
          constexpr int d = decltype(dc)::value;
#pragma unroll
          for (int v = 0; v < V; v++)
            dq[d * V + v] = wide_deriv<d>(sm.q[t], node, v, 1.0 / g.dX[d]);
        });
      static_for<0, D>([&](auto dc) {
        constexpr int d = decltype(dc)::value;
        F(out, q, dq, d);
#pragma unroll
        for (int v = 0; v < V; v++) sm.f[d][tt][node][v] = out[v];
      });
    }
#endif
  }
  wide_sync();
}

#if PDE_USE_B
// sm.r -= B(q, d) dq_d at time nodes t0 .. t0 + nt - 1, four space-time nodes
// at a time: lanes 0..3 write their B (over the groups' matrices), then one
// lane per (node, variable); QUIRK as in b_times.
template <int d, int QUIRK>
DEV void wide_b_term(WidePred& sm, int t0, int nt, const Geom& g, int lane) {
  auto matrix = [&](int k) {
    WideGroup& G = sm.grp[k >> 1];
    return (k & 1) ? &G.P[0][0] : &G.A[0][0];
  };
#pragma unroll 1
  for (int i0 = 0; i0 < nt * ND; i0 += 4) {
    const int n = nt * ND - i0 < 4 ? nt * ND - i0 : 4;
    if (lane < n) B(matrix(lane), sm.q[t0 + (i0 + lane) / ND][(i0 + lane) % ND], d);
    wide_sync();
#pragma unroll 1
    for (int e = lane; e < n * V; e += 64) {
      const int k = e / V, v = e % V, t = t0 + (i0 + k) / ND, node = (i0 + k) % ND;
      const double* const bm = matrix(k);
      auto dq = [&](int j) { return wide_deriv<d>(sm.q[t], node, j, 1.0 / g.dX[d]); };
      double bd;
      if constexpr (QUIRK == 1) {
        bd = bm[0] * dq(v);
      } else if constexpr (QUIRK == 2) {
        bd = bm[v * V] * dq(0);
      } else {
        bd = bm[v * V] * dq(0);
#pragma unroll 1
        for (int j = 1; j < V; j++) bd = dfma(bm[v * V + j], dq(j), bd);
      }
      sm.r[t][node][v] = sm.r[t][node][v] - bd;
    }
    wide_sync();
  }
}
#endif

// sm.r = right-hand side of the space-time system (node_rhs).
DEV void wide_rhs(WidePred& sm, double dt, const Geom& g, int lane) {
#pragma unroll 1
  for (int t0 = 0; t0 < N; t0 += WIDE_T) {
    wide_eval(sm, t0, WIDE_T, true, g, lane);
    static_for<0, D>([&](auto dc) {
      constexpr int d = decltype(dc)::value;
#if PDE_USE_B
      wide_b_term<d, PDE_B_QUIRK ? 1 : 0>(sm, t0, WIDE_T, g, lane);
#endif
#if PDE_USE_F
#pragma unroll 1
      for (int e = lane; e < ND * V; e += 64) {
        const int node = e / V, v = e % V;
#pragma unroll
        for (int tt = 0; tt < WIDE_T; tt++)
          sm.r[t0 + tt][node][v] =
              sm.r[t0 + tt][node][v] - wide_deriv<d>(sm.f[d][tt], node, v, 1.0 / g.dX[d]);
      }
      wide_sync();
#endif
    });
  }
#pragma unroll 1
  for (int e = lane; e < ND * V; e += 64) {
    const int node = e / V, v = e % V;
#pragma unroll
    for (int t = 0; t < N; t++) {
      const double rr = sm.r[t][node][v] * wide_scaled(T_W[t], node);
      sm.r[t][node][v] = rr * dt + wide_scaled(T_END0[t], node) * sm.w[node][v];
    }
  }
  wide_sync();
}

DEV double group_max(double x) {
#pragma unroll
  for (int o = 16; o >= 1; o >>= 1) x = dmax(x, __shfl_xor(x, o, 64));
  return x;
}

#if PDE_STIFF
// Newton correction at one node (newton_node) by half a wavefront: lane l <
// V holds variable l, gt its scaled residuals, and receives its correction in
// delta.  True where the source Jacobian was solved.  Every lane calls it; a
// half without a node (on false) works on values it discards.
static_assert(V + N <= 32, "a half wavefront holds the columns and right-hand sides");
DEV bool wide_newton(WideGroup& G, const double (&qn)[N], const double (&gt)[N], double dt, int l,
                     double (&delta)[N]) {
  const unsigned long long half = 0xffffffffull << (threadIdx.x & 32u);
  const bool in = l < V;
  double qbar = T_W[0] * qn[0];
#pragma unroll
  for (int t = 1; t < N; t++) qbar = dfma(T_W[t], qn[t], qbar);
  if (in) G.qbar[l] = qbar;
  wide_sync();
  double col[V];
#if PDE_USE_M
  if (l == 0) M(&G.A[0][0], G.qbar);
  wide_sync();
#pragma unroll
  for (int i = 0; i < V; i++) col[i] = in ? (&G.A[0][0])[i * V + l] : 0.0;
#elif PDE_USE_S
  {
    // lanes l < V perturb variable l, the others evaluate S(qbar) itself
    double qq[V], s1[V], hl = FD_EPS;
#pragma unroll
    for (int v = 0; v < V; v++) {
      const double q0 = G.qbar[v];
      const double hh = dmax(FD_EPS * dabs(q0), FD_EPS);
      qq[v] = v == l ? q0 + hh : q0;
      hl = v == l ? hh : hl;
    }
    const double rhh = 1.0 / hl;
    S(s1, qq);
    if (l == V) {
#pragma unroll
      for (int v = 0; v < V; v++) G.s0[v] = s1[v];
    }
    wide_sync();
#pragma unroll
    for (int i = 0; i < V; i++) col[i] = in ? (s1[i] - G.s0[i]) * rhh : 0.0;
  }
#else
#pragma unroll
  for (int i = 0; i < V; i++) col[i] = 0.0;
#endif
  double amax = 0.0;
#pragma unroll
  for (int i = 0; i < V; i++) amax = dmax(amax, dabs(col[i]));
  amax = dmax(0.0, dabs(dt) * group_max(amax));
  const bool full = !(amax < NEWTON_A_TINY);
  if (!full) {
#pragma unroll
    for (int t = 0; t < N; t++) {
      double acc = T_FLM[N - 1][t][0] * gt[0];
#pragma unroll
      for (int s = 1; s < N; s++) acc = dfma(T_FLM[N - 1][t][s], gt[s], acc);
      delta[t] = -(acc * (1.0 / T_FLC[0]));
    }
  }
  if ((__ballot(full) & half) == 0ull) return false;
  wide_sync();
  if (in) {
#pragma unroll
    for (int i = 0; i < V; i++) G.A[i][l] = dt * col[i];
  }
  wide_sync();
  // h_t (Horner in A), lane i holding row i of A
  const int row = in ? l : 0;
  double b[N];
  {
    double Ar[V];
#pragma unroll
    for (int k = 0; k < V; k++) Ar[k] = G.A[row][k];
#pragma unroll
    for (int j = N - 1; j >= 0; j--) {
      double u[N];
#pragma unroll
      for (int t = 0; t < N; t++) {
        u[t] = T_FLM[N - j - 1][t][0] * gt[0];
#pragma unroll
        for (int s = 1; s < N; s++) u[t] = dfma(T_FLM[N - j - 1][t][s], gt[s], u[t]);
      }
      if (j == N - 1) {
#pragma unroll
        for (int t = 0; t < N; t++) b[t] = u[t];
      } else {
#pragma unroll
        for (int t = 0; t < N; t++) {
          double acc = Ar[0] * G.h[t][0];
#pragma unroll
          for (int k = 1; k < V; k++) acc = dfma(Ar[k], G.h[t][k], acc);
          b[t] = acc + u[t];
        }
      }
      wide_sync();
      if (in) {
#pragma unroll
        for (int t = 0; t < N; t++) G.h[t][l] = b[t];
      }
      wide_sync();
    }
  }
  // P = p(A), lane j holding column j; lane V + t holds right-hand side t
  double P[V];
#pragma unroll
  for (int i = 0; i < V; i++) {
    const double a = G.A[i][row];
    P[i] = i == l ? a + T_FLC[N - 1] : a;
  }
#pragma unroll
  for (int j = N - 2; j >= 0; j--) {
    // P <- P A + c_j I: the rows of P from LDS (A itself, shifted, the first time)
    double Ac[V], next[V];
#pragma unroll
    for (int m = 0; m < V; m++) Ac[m] = G.A[m][row];
    if (j < N - 2) {
      wide_sync();
      if (in) {
#pragma unroll
        for (int i = 0; i < V; i++) G.P[i][l] = P[i];
      }
      wide_sync();
    }
#pragma unroll
    for (int i = 0; i < V; i++) {
#pragma unroll
      for (int m = 0; m < V; m++) {
        const double e = j == N - 2 ? (m == i ? G.A[i][m] + T_FLC[N - 1] : G.A[i][m]) : G.P[i][m];
        next[i] = m == 0 ? e * Ac[0] : dfma(e, Ac[m], next[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < V; i++) P[i] = i == l ? next[i] + T_FLC[j] : next[i];
  }
#pragma unroll
  for (int t = 0; t < N; t++)
    if (l == V + t) {
#pragma unroll
      for (int i = 0; i < V; i++) P[i] = G.h[t][i];
    }
  // LU with partial pivoting (first largest pivot), the right-hand sides
  // carried along: lane k finds the pivot of step k in its own registers and
  // hands the multipliers to the others through LDS
#pragma unroll
  for (int k = 0; k < V; k++) {
    double most = 0.0;
#pragma unroll
    for (int i = k + 1; i < V; i++) most = dmax(most, dabs(P[i]));
    if ((__ballot(l == k && most > dabs(P[k])) & half) != 0ull) {
      int p = k;
      double best = dabs(P[k]);
#pragma unroll
      for (int i = k + 1; i < V; i++) {
        const double a = dabs(P[i]);
        if (a > best) {
          best = a;
          p = i;
        }
      }
      p = __shfl(p, (int)(threadIdx.x & 32u) + k, 64);
#pragma unroll
      for (int i = k + 1; i < V; i++) {
        if (p == i) {
          const double tmp = P[k];
          P[k] = P[i];
          P[i] = tmp;
        }
      }
    }
    if (l == k) {
      const double rk = 1.0 / P[k];
      G.row[k] = rk;
#pragma unroll
      for (int i = k + 1; i < V; i++) {
        P[i] = P[i] * rk;
        G.P[k][i] = P[i];
      }
    }
    wide_sync();
    if (l > k) {
#pragma unroll
      for (int i = k + 1; i < V; i++) P[i] = dfma(-G.P[k][i], P[k], P[i]);
    }
  }
  // back substitution in the right-hand sides' lanes, U's rows through LDS
  wide_sync();
  if (in) {
#pragma unroll
    for (int i = 0; i < V; i++) G.A[i][l] = P[i];
  }
  wide_sync();
  if (l >= V && l < V + N) {
    double x[V];
#pragma unroll
    for (int i = V - 1; i >= 0; i--) {  // x[j] is -y_j already
      double acc = P[i];
#pragma unroll
      for (int j = i + 1; j < V; j++) acc = dfma(G.A[i][j], x[j], acc);
      x[i] = -(acc * G.row[i]);
    }
#pragma unroll
    for (int i = 0; i < V; i++) G.h[l - V][i] = x[i];
  }
  wide_sync();
  if (full) {
#pragma unroll
    for (int t = 0; t < N; t++) delta[t] = G.h[t][row];
  }
  wide_sync();
  return full;
}
#endif

DEV void wide_predictor(WidePred& sm, const double* __restrict__ wh,
                        const double* __restrict__ guess, double* __restrict__ tr,
                        double* __restrict__ vol, double* __restrict__ qh, StepState* st,
                        const Geom& g, double newton_tol, int newton_maxit, const Blk& blk) {
  if (st->done) return;
  const double dt = st->dt;
  const int lane = threadIdx.x;
  const long cell = (long)xcd_order(blk.x, blk.n);
  if (cell >= g.nwc) return;
#pragma unroll 1
  for (int e = lane; e < ND * V; e += 64) {
    const int node = e / V, v = e % V;
    const double w = wh[(long)e * g.nwc + cell];
    sm.w[node][v] = w;
#pragma unroll
    for (int t = 0; t < N; t++)
      sm.q[t][node][v] =
          (PDE_GUESS && guess) ? guess[(long)((t * ND + node) * V + v) * g.nwc + cell] : w;
  }
  wide_sync();
#if PDE_STIFF
  const int maxit = newton_maxit;
#else
  const int maxit = DG_IT;
  (void)newton_tol;
  (void)newton_maxit;
#endif
  int it = 0, fellback = 0;
  unsigned int n_full = 0u, n_short = 0u;  // node corrections of this cell
#if PDE_STIFF && PDE_GUESS
  bool learned = guess != nullptr;
  double r0 = 0.0;
#endif
  bool active = true;
  while (active) {
    wide_rhs(sm, dt, g, lane);
    bool more = false;
#if PDE_STIFF
    // residual G = rhs - (DG_MAT (x) W) q   (dg.cpp:128-154)
    double rmax = 0.0;
    bool rnan = false;
#pragma unroll 1
    for (int e = lane; e < ND * V; e += 64) {
      const int node = e / V, v = e % V;
      const double WP = wide_weight(node);
#pragma unroll
      for (int t = 0; t < N; t++) {
        double acc = (T_DGMAT[t][0] * WP) * sm.q[0][node][v];
#pragma unroll
        for (int s = 1; s < N; s++) acc = dfma(T_DGMAT[t][s] * WP, sm.q[s][node][v], acc);
        const double G = sm.r[t][node][v] - acc;
        sm.r[t][node][v] = G;
        rmax = dmax(rmax, dabs(G));
        rnan = rnan || G != G;
      }
    }
    wide_sync();
    bool skip = false;
#if PDE_GUESS
    // a learned guess whose residual is not finite or grows sends the cell
    // back to the plain guess
    if (learned) {
      const double cm = wide_max(rmax);
      const bool keep =
          __ballot(rnan) == 0ull && cm <= (it > 0 ? r0 : 1.7976931348623157e308);
      if (!keep) {
#pragma unroll 1
        for (int e = lane; e < ND * V; e += 64)
#pragma unroll
          for (int t = 0; t < N; t++) sm.q[t][e / V][e % V] = sm.w[e / V][e % V];
        wide_sync();
        fellback = 1;
        learned = false;
        skip = true;
        more = true;
      } else {
        r0 = cm;
      }
    }
#else
    (void)rmax;
    (void)rnan;
#endif
    if (!skip) {
      const int l = lane & 31, v = l < V ? l : 0;
#pragma unroll 1
      for (int n0 = 0; n0 < ND; n0 += 2) {
        const int node = n0 + (lane >> 5);
        const bool on = node < ND;
        const int nn = on ? node : ND - 1;
        const double p = wide_weight(nn);
        double qn[N], gt[N], delta[N];
#pragma unroll
        for (int t = 0; t < N; t++) {
          qn[t] = sm.q[t][nn][v];
          gt[t] = sm.r[t][nn][v] * (1.0 / (T_W[t] * p));
        }
        const bool full = wide_newton(sm.grp[lane >> 5], qn, gt, dt, l, delta);
        if (on && l == 0) {
          if (full) n_full++;
          else n_short++;
        }
        if (on && l < V) {
#pragma unroll
          for (int t = 0; t < N; t++) {
            if (!(dabs(delta[t]) <= newton_tol * (1.0 + dabs(qn[t])))) more = true;
            sm.q[t][nn][v] = qn[t] + delta[t];
          }
        }
      }
      wide_sync();
    }
#else
    // Picard: q1 = DG_MAT^-1 rhs / prod W  (dg.cpp:187-202)
#pragma unroll 1
    for (int e = lane; e < ND * V; e += 64) {
      const int node = e / V, v = e % V;
      const double IWP = 1.0 / wide_weight(node);
      double rs[N];
#pragma unroll
      for (int t = 0; t < N; t++) rs[t] = sm.r[t][node][v];
#pragma unroll
      for (int t = 0; t < N; t++) {
        double acc = T_DGINV[t][0] * rs[0];
#pragma unroll
        for (int s = 1; s < N; s++) acc = dfma(T_DGINV[t][s], rs[s], acc);
        const double q1 = acc * IWP, q0 = sm.q[t][node][v];
        if (dabs(q1 - q0) > DG_TOL * (1.0 + dabs(q0))) more = true;
        sm.q[t][node][v] = q1;
      }
    }
    wide_sync();
#endif
    it++;
    active = __ballot(more) != 0ull && it < maxit;
  }
  // ---- traces, optional full qh, volume term (predictor_static_body)
  static_for<0, D>([&](auto dc) {
    constexpr int d = decltype(dc)::value;
    constexpr int stride = ipow_c(N, D - 1 - d);
#pragma unroll 1
    for (int i = lane; i < N * ND1 * V; i += 64) {
      const int v = i % V, j = (i / V) % ND1, t = i / (V * ND1);
      const int idx0 = (j / stride) * stride * N + j % stride;  // node with k_d = 0
#pragma unroll
      for (int e = 0; e < 2; e++) {
        double acc = (e ? T_END1[0] : T_END0[0]) * sm.q[t][idx0][v];
#pragma unroll
        for (int m = 1; m < N; m++)
          acc = dfma(e ? T_END1[m] : T_END0[m], sm.q[t][idx0 + m * stride][v], acc);
        tr[trace_at(g, ((d * 2 + e) * N + t) * ND1 + j, cell, 0) + v] = acc;
      }
    }
  });
  if (qh) {
#pragma unroll 1
    for (int i = lane; i < NT * V; i += 64)
      qh[(long)i * g.nwc + cell] = (&sm.q[0][0][0])[i];
  }
#if PDE_USE_S || PDE_USE_B
#pragma unroll 1
  for (int t0 = 0; t0 < N; t0 += WIDE_T) wide_eval(sm, t0, WIDE_T, false, g, lane);
#if PDE_USE_B
  static_for<0, D>([&](auto dc) {
    wide_b_term<decltype(dc)::value, PDE_B_QUIRK ? 2 : 0>(sm, 0, N, g, lane);
  });
#endif
  // per node the sum over t, then over nodes in order
#pragma unroll 1
  for (int e = lane; e < ND * V; e += 64) {
    const int node = e / V, v = e % V;
    double part = 0.0;
#pragma unroll
    for (int t = 0; t < N; t++) {
      const double tmp = wide_scaled(dt * T_W[t], node);
      part = t == 0 ? tmp * sm.r[0][node][v] : dfma(tmp, sm.r[t][node][v], part);
    }
    sm.r[0][node][v] = part;
  }
  wide_sync();
  if (lane < V) {
    double acc = sm.r[0][0][lane];
#pragma unroll
    for (int i = 1; i < ND; i++) acc = acc + sm.r[0][i][lane];
    vol[(long)lane * g.nwc + cell] = acc;
  }
#endif
  const unsigned long long w_full = wave_sum_u64(n_full), w_short = wave_sum_u64(n_short);
  if (lane == 0) {
    unsigned long long* ps = st->pstat[blk.x & 63];
    atomicAdd(&ps[0], (unsigned long long)it);
    atomicAdd(&ps[1], 1ull);
    if (it >= maxit) atomicAdd(&ps[2], 1ull);
    if (fellback) atomicAdd(&ps[3], 1ull);
    atomicMax(&ps[4], (unsigned long long)it);
    if (w_full) atomicAdd(&ps[5], w_full);
    if (w_short) atomicAdd(&ps[6], w_short);
  }
}

extern "C" __global__ void __launch_bounds__(64)
k_predictor_static(const double* __restrict__ wh, const double* __restrict__ guess,
                   double* __restrict__ tr, double* __restrict__ vol, double* __restrict__ qh,
                   StepState* st, Geom g, double newton_tol, int newton_maxit,
                   double* __restrict__ trd) {
  __shared__ WidePred sm;
  (void)trd;
  wide_predictor(sm, wh, guess, tr, vol, qh, st, g, newton_tol, newton_maxit, lin_blk());
}
#if PDE_BATCH
extern "C" __global__ void __launch_bounds__(64)
k_predictor_static_b(const Member* ms, const BlkMap* map, int nm, double newton_tol,
                     int newton_maxit) {
  __shared__ WidePred sm;
  PYPDE_BATCH_MEMBER
  wide_predictor(sm, M.wh, nullptr, M.tr, M.vol, nullptr, M.st, M.g, newton_tol, newton_maxit, b);
}
#endif
