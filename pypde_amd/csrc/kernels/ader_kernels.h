// ADER-WENO step kernels for MI355X (gfx950).  Compiled at run time by hipRTC
// after ader_common.h, with the problem's D, N, V, tables and system source.
//
// Device data layout (structure of arrays, cell index fastest):
//   u   [V][ncell]                          interior state
//   wh  [N^D * V][nwc]                      reconstruction, plane = node*V + v
//   tr  [2*D*N*N^(D-1)][ntb][V][TCW]        face traces of the predictor, plane
//                                           ((d*2+e)*N+t)*N^(D-1)+j; TCW cells per
//                                           block (trace_at)
//   vol [V][nwc]                            volume (source / B) integral
//   ff, fb [N*N^(D-1)*V][nf_d] per d        face flux / B path integral
// nwc = prod(nx_d + 2) reconstructed cells (one ghost layer, iterator.cpp:76).
#pragma once

struct Geom {
  int nx[2];     // interior cells per axis (nx[1] = 1 when D = 1)
  int nw[2];     // reconstructed cells per axis (nx + 2; nw[1] = 1 when D = 1)
  int nb[2];     // ghost-extended cells per axis (nx + 2N)
  int bc[2];     // 0 transmissive, 1 periodic, 2 reflective
  long ncell;    // prod nx
  long nwc;      // prod nw
  long nf[2];    // faces per direction: (nx_d + 1) * prod_{e != d} nx_e
  double dX[2];
  double refl[2][17];  // reflective-wall multipliers per axis (V <= 17)
  int ndt;
  // Flux-item index arithmetic without run-time division: n / nf[d] and n /
  // (faces per row along d: nx[1] for d = 0, nx[1] + 1 for d = 1) as
  // (n * mul) >> sh, exact for n < 2^31 (udiv); idx32 is 1 when every flux
  // item index and every w-cell index is below 2^31.
  unsigned fmul[2], fsh[2], rmul[2], rsh[2];
  int idx32;
  long ntb;  // trace blocks: ceil(nwc / TCW)
};

// Face traces in blocks of the TCW cells one predictor wavefront holds, their
// variables together: a wavefront writes whole cache lines (V TCW doubles a
// block: 128 bytes at order 4 with four variables, where rows of 4 cells in
// planes of one variable were 32-byte pieces that four wavefronts had to
// complete), and what a face point reads of a block, its V variables, lies in
// the same lines (2048 x 2048 at order 2, predictor 848 -> 729 us: it writes
// 2.1 GB of traces, which is what bounds it).
constexpr int TCW = PDE_WIDE_PRED ? 1 : 64 / ND;
DEV long trace_at(const Geom& g, int plane, long block, int slot) {
  return ((long)plane * g.ntb + block) * (V * TCW) + slot;  // + v * TCW
}

// n / d for n < 2^31 from d's multiplier m = ceil(2^sh / d), sh = 31 +
// ceil(log2 d): with n = q d + r, n m / 2^sh = q + (r + n e / 2^sh) / d, e =
// m d - 2^sh in [0, d), and n e < 2^31 d <= 2^sh keeps the bracket below d.
DEV unsigned udiv(unsigned n, unsigned m, unsigned sh) {
  return (unsigned)(((unsigned long long)n * m) >> sh);
}

struct StepState {
  double t, dt, tf, cfl;
  long long count, max_steps;
  int push, done, nan_step;
  int flip;  // 1D: the state lies in u2 (k_update_next)
  unsigned long long maxbits;   // unused (the wave-speed maximum lives in pstat[.][8])
  unsigned int nan_flag, pad2;
  unsigned long long pred_iters, pred_cells, pred_capped, pred_fallbacks;
  unsigned int pred_maxit, pad3;
  // stiff predictor: Newton corrections per spatial node with the full source
  // Jacobian solve and with the A = 0 shortcut, summed over nodes and steps
  unsigned long long pred_nfull, pred_nshort;
  unsigned long long pred_iters32;  // mixed precision: FP32-phase iterations over cells
  unsigned long long hot_count;     // split stiff predictor: cells handed to the hot pass
  // workgroups of k_dt and of the corrector that have finished this step: the
  // last one of each folds the step's partial results (dt; the step's
  // bookkeeping) and resets its ticket
  unsigned int dt_ticket, step_ticket;
  // predictor statistics spread over 64 slots, one 128-byte line each, so the
  // wavefronts' atomics do not queue on one address; the corrector's last
  // workgroup folds them into the totals above and clears them ([0]
  // iterations, [1] cells, [2] capped, [3] fallbacks, [4] max iterations, [5]
  // full and [6] shortcut node corrections, [7] FP32-phase iterations; [8]
  // k_dt's partial maximum, folded by k_dt's last workgroup; [9], [10] the
  // tickets of k_dt's and the corrector's workgroups, last_workgroup)
  unsigned long long pstat[64][16];
};

// A workgroup's coordinates within one grid's launch, and the number of
// workgroups of that launch: the hardware's own for a single grid, or one
// member's share of a batched ensemble launch.
struct Blk {
  unsigned int x, y, z, n;
};
DEV Blk hw_blk() {
  return {blockIdx.x, blockIdx.y, blockIdx.z, gridDim.x * gridDim.y * gridDim.z};
}
// Launches numbered in x alone: workgroups that do not fit in x continue in y
// (grid_of in grid.h), and the last row may hold some past the last one.
DEV unsigned int blk_x() { return blockIdx.y * gridDim.x + blockIdx.x; }
DEV Blk lin_blk() { return {blk_x(), 0u, 0u, gridDim.x * gridDim.y}; }

// Position of workgroup i of n in an order that gives each of the 8 XCDs
// runs of XCD_RUN consecutive positions: workgroups are dispatched to the
// XCDs round-robin (i to XCD i mod 8), so neighbouring positions, whose
// cells share cache lines, meet in one XCD's L2, while costly regions of a
// grid (a reaction zone) still spread over every XCD.  Runs of
// 8 x XCD_RUN positions go round the XCDs; the n mod (8 x XCD_RUN) last
// positions keep their order.  A bijection of [0, n).
constexpr unsigned int XCD_RUN = 16;
DEV unsigned int xcd_order(unsigned int i, unsigned int n) {
  constexpr unsigned int SPAN = 8u * XCD_RUN;
  if (i >= n - n % SPAN) return i;
  const unsigned int x = i & 7u, k = i >> 3;
  return (k / XCD_RUN) * SPAN + x * XCD_RUN + k % XCD_RUN;
}

// Every kernel of a step returns at once when the run has ended.  The flag was
// written by another kernel on another XCD, so reading it takes as long as
// any load from memory; where a kernel's own first loads do not depend on
// it, they are issued before the flag is tested (their addresses are valid
// either way), and this keeps the compiler from sinking them below the test
// (200 cells: predictor 7.3 -> 6.9 us, face flux 4.15 -> 3.9; viscous 64 x 64 0.3
// less each).
#define LOADS_FIRST() asm volatile("" ::: "memory")

DEV double wave_max(double x) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) x = dmax(x, __shfl_xor(x, o, 64));
  return x;
}
// True in every thread of the workgroup that is the last of the grid to
// reach this point; that workgroup also resets the ticket.  What the other
// workgroups hand over must be written with device-scope atomics (performed
// at the device's coherence point) and read back with atomics: each thread
// waits for its own atomics to be acknowledged before the workgroup draws its
// ticket, so the last ticket is drawn after every other workgroup's atomics
// have completed.  No device-scope fence is used: on gfx950 every such fence
// writes back or invalidates the XCD's L2, which costs more than a separate
// one-workgroup launch.  b.n is the number of workgroups drawing from the
// ticket, numbered by b.x; every thread of each of them must call it.
//
// Atomics on one address complete one after the other, about 12 ns apart, which
// bounds a launch of many short workgroups (k_dt on 2048 x 2048 cells, 32,800
// workgroups: 388 us, 232 with two levels).  Above 128 workgroups each
// therefore draws from one of 64 tickets, word `sub` of its pstat line, and
// the last of each of the 64 from the common one; below, the second round
// trip at the end would cost as much as it saves.
DEV bool last_workgroup(StepState* st, unsigned int* ticket, int sub, const Blk& b) {
  __shared__ unsigned int is_last;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned int n = b.n, last = 1u;
    if (n > 128u) {
      const unsigned int k = b.x & 63u, members = (n - k + 63u) >> 6;
      unsigned long long* own = &st->pstat[k][sub];
      last = atomicAdd(own, 1ull) == members - 1u ? 1u : 0u;
      if (last) atomicExch(own, 0ull);
      n = 64u;
    }
    if (last) {
      last = atomicAdd(ticket, 1u) == n - 1u ? 1u : 0u;
      if (last) atomicExch(ticket, 0u);
    }
    is_last = last;
  }
  __syncthreads();
  return is_last != 0u;
}
DEV void dt_finalize(StepState* st);

DEV unsigned long long wave_sum_u64(unsigned long long x) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}
DEV unsigned int wave_max_u32(unsigned int x) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    unsigned int y = __shfl_xor(x, o, 64);
    x = x > y ? x : y;
  }
  return x;
}

// --------------------------------------------------------------- WENO
// Boundary ghosts fused into the load, both sweeps staged in LDS
// (boundaries.cpp:25-53, weno.cpp:61-121).  ghost = false gives the
// reference's weno_solver semantics (no ghost extension).
// 2D: one variable per workgroup (coordinate z), a TX x TY tile of output cells
// per workgroup (256 threads); sweep 1 along axis 0 over the TX + 2N - 2 rows
// and TY + 2N - 2 columns the tile needs, then sweep 2 along axis 1 for every
// coefficient index k0.  The autotuner picks the tile per problem.  A thread
// of sweep 2 forms all the nodes of its cell and variable, so it also has
// their mean (k_dt's fma chain over the nodes): k_dt reads one value per
// variable instead of N^2 (512 x 512 at order 4 34 -> 21 us, the 1024 x 256
// channel at order 3 30 -> 24, for 0-1 us more here; at order 2 17 us less there
// for 17 more here).
template <int TX, int TY>
DEV void weno_2d(const double* __restrict__ u, double* __restrict__ wh, const Geom& g, int ghost,
                 int nin0, int nin1, long out_stride, double* __restrict__ wm, const Blk& b) {
  constexpr int H = 2 * N - 2;
  const int tid = threadIdx.x;
  constexpr int RX = TX + H, RY = TY + H, RYP = RY + 1;
  __shared__ double s0[RX][RYP];
  __shared__ double s1[N][TX][RYP];
  const int v = b.z;
  const int i0 = b.y * TX, j0 = b.x * TY;
  const int nb0 = ghost ? g.nb[0] : nin0, nb1 = ghost ? g.nb[1] : nin1;
  const int no0 = nb0 - H, no1 = nb1 - H;
  const long in_stride = ghost ? g.ncell : (long)nin0 * nin1;
  const int in_row = ghost ? g.nx[1] : nin1;
  for (int e = tid; e < RX * RY; e += 256) {
    int r = e / RY, c = e % RY;
    int I = i0 + r, J = j0 + c;
    double val = 0.0;
    if (I < nb0 && J < nb1) {
      bool f0 = false, f1 = false;
      int s0i = ghost ? ghost_src(I, g.bc[0], g.nx[0], &f0) : I;
      int s1i = ghost ? ghost_src(J, g.bc[1], g.nx[1], &f1) : J;
      double sg = 1.0;
      if (f0) sg = sg * g.refl[0][v];
      if (f1) sg = sg * g.refl[1][v];
      val = u[(long)v * in_stride + (long)s0i * in_row + s1i] * sg;
    }
    s0[r][c] = val;
  }
  __syncthreads();
  for (int e = tid; e < TX * RY; e += 256) {
    int r = e / RY, c = e % RY;
    if (i0 + r < no0) {
      double out[N];
      weno_line([&](int m) { return s0[r + m][c]; }, out);
#pragma unroll
      for (int k = 0; k < N; k++) s1[k][r][c] = out[k];
    }
  }
  __syncthreads();
  for (int e = tid; e < TX * TY; e += 256) {
    int c = e % TY, r = e / TY;
    int i = i0 + r, j = j0 + c;
    if (i < no0 && j < no1) {
      long cell = (long)i * no1 + j;
      double mean = 0.0;
#pragma unroll(N <= 3 ? N : 1)
      for (int k0 = 0; k0 < N; k0++) {
        double out[N];
        weno_line([&](int m) { return s1[k0][r][c + m]; }, out);
#pragma unroll
        for (int k1 = 0; k1 < N; k1++) {
          const int idx = k0 * N + k1;
          wh[(long)(idx * V + v) * out_stride + cell] = out[k1];
          mean = idx == 0 ? T_WP[0] * out[0] : dfma(T_WP[idx], out[k1], mean);
        }
      }
      if (wm) wm[(long)v * out_stride + cell] = mean;
    }
  }
}

// 1D: WENO1_W output cells per workgroup, all variables: 256, so that each
// thread takes V values; above V = 8 16, about one value per thread, as a
// grid of 200 cells and 17 variables was one workgroup's 17 turns otherwise
// (13.0 -> 4.7 us).  At V = 3 tiles of 64 and 256 measure the same.
constexpr int WENO1_W = V > 8 ? 16 : 256;
DEV void weno_1d(const double* __restrict__ u, double* __restrict__ wh, const Geom& g, int ghost,
                 int nin0, long out_stride, double* __restrict__ wm, const Blk& b) {
  constexpr int H = 2 * N - 2;
  const int tid = threadIdx.x;
  constexpr int TX = WENO1_W;
  constexpr int RX = TX + H;
  __shared__ double s0[V][RX];
  const int i0 = b.x * TX;
  const int nb0 = ghost ? g.nb[0] : nin0;
  const int no0 = nb0 - H;
  for (int e = tid; e < V * RX; e += 256) {
    int v = e / RX, r = e % RX;
    int I = i0 + r;
    double val = 0.0;
    if (I < nb0) {
      bool f0 = false;
      int s = ghost ? ghost_src(I, g.bc[0], g.nx[0], &f0) : I;
      double sg = 1.0;
      if (f0) sg = sg * g.refl[0][v];
      val = u[(long)v * (ghost ? g.ncell : nin0) + s] * sg;
    }
    s0[v][r] = val;
  }
  __syncthreads();
  for (int e = tid; e < V * TX; e += 256) {
    int v = e / TX, r = e % TX;
    int i = i0 + r;
    if (i < no0) {
      double out[N];
      weno_line([&](int m) { return s0[v][r + m]; }, out);
      double mean = 0.0;
#pragma unroll
      for (int k = 0; k < N; k++) {
        wh[(long)(k * V + v) * out_stride + i] = out[k];
        mean = k == 0 ? T_WP[0] * out[0] : dfma(T_WP[k], out[k], mean);
      }
      if (wm) wm[(long)v * out_stride + i] = mean;
    }
  }
}

#define PYPDE_WENO_KERNEL(NAME, TX, TY)                                                        \
  extern "C" __global__ void __launch_bounds__(256)                                            \
  NAME(const double* __restrict__ u, double* __restrict__ wh, const StepState* __restrict__ st, \
       Geom g, int ghost, int nin0, int nin1, long out_stride, double* __restrict__ wm) {      \
    if (st && st->done) return;                                                                \
    if constexpr (D == 1)                                                                      \
      weno_1d(u, wh, g, ghost, nin0, out_stride, wm, lin_blk());                               \
    else                                                                                       \
      weno_2d<TX, TY>(u, wh, g, ghost, nin0, nin1, out_stride, wm, hw_blk());                  \
  }
PYPDE_WENO_KERNEL(k_weno, 8, 32)
PYPDE_WENO_KERNEL(k_weno_4x64, 4, 64)
PYPDE_WENO_KERNEL(k_weno_16x16, 16, 16)
PYPDE_WENO_KERNEL(k_weno_16x32, 16, 32)

// ------------------------------------------------------------ timestep
// Largest sum_d lambda_d / dX_d over every reconstructed cell
// (stepper.cpp:42-65), reduced as IEEE bit patterns (all values >= 0).
template <int d>
DEV void cell_deriv(const double (&w)[ND][V], int idx, double rdx, double* out) {
  constexpr int stride = ipow_c(N, D - 1 - d);
  // idx is a compile-time constant at every call site after unrolling
  const int kd = (idx / stride) % N;
  const int base = idx - kd * stride;
#pragma unroll
  for (int v = 0; v < V; v++) {
    double acc = T_DER[kd][0] * w[base][v];
#pragma unroll
    for (int j = 1; j < N; j++) acc = dfma(T_DER[kd][j], w[base + j * stride][v], acc);
    out[v] = acc * rdx;
  }
}

// In 2D (V <= 5, no viscous term) two neighbouring lanes share a w-cell and
// take one direction each: twice the wavefronts (a 1024 x 256 grid's 8,272 in
// two rounds of the 4,096 slots at four per SIMD) with half the eigenvalue
// work per lane.  Both lanes form the cell's (l_0 / dX_0) + (l_1 /
// dX_1) from the pair's two terms.  The host launches DT_LANES * nwc threads.
constexpr bool DT_PAIR = (D == 2) && (V <= 5) && !PDE_SECOND;
// With a viscous F a w-cell has 2 D eigenvalue problems, each of which costs as
// much as a whole first-order cell: a wavefront takes one of them for 64
// cells and the sums go through LDS (64 x 64 cells, 69 wavefronts one after
// the other's problems otherwise: 22 -> 10.4 us).
constexpr int DT_LANES = PDE_WIDE_EIG ? 64 : PDE_SECOND ? 2 * D : DT_PAIR ? 2 : 1;

#if PDE_WIDE_EIG
// One wavefront per w-cell: the cell's mean (lane v takes variable v), then
// one eigenvalue problem per direction over the wavefront.
DEV void dt_body(const double* __restrict__ wh, const double* __restrict__ wm, StepState* st,
                 const Geom& g, const Blk& b) {
  __shared__ WideMat mats[WIDE_WAVES];
  if (st->done) return;
  const int lane = threadIdx.x & 63;
  WideMat& W = mats[threadIdx.x >> 6];
  const long c = (long)b.x * WIDE_WAVES + (threadIdx.x >> 6);
  double sum = 0.0;
  if (c < g.nwc) {
    if (lane < V) W.P[0][lane] = wm[(long)lane * g.nwc + c];
    wide_sync();
    double q[V], dq[D * V], f0[V];
#pragma unroll
    for (int v = 0; v < V; v++) q[v] = W.P[0][v];
#pragma unroll
    for (int i = 0; i < D * V; i++) dq[i] = 0.0;
    static_for<0, D>([&](auto dc) {
      constexpr int d = decltype(dc)::value;
      const double lam = wide_max_abs_eigs(W, q, dq, d, lane, f0);
      sum = sum + lam / g.dX[d];
    });
    if (!(sum > 0.0)) sum = 0.0;
  }
  if (lane == 0 && sum > 0.0)
    atomicMax(&st->pstat[b.x & 63][8], (unsigned long long)__double_as_longlong(sum));
  if (last_workgroup(st, &st->dt_ticket, 9, b)) dt_finalize(st);
}
#elif PDE_SECOND
DEV void dt_body(const double* __restrict__ wh, const double* __restrict__ wm, StepState* st,
                 const Geom& g, const Blk& b) {
  constexpr int CELLS = 256 / DT_LANES;  // a multiple of 64: `part` is the same in a wavefront
  if (st->done) return;
  __shared__ double lam[DT_LANES][CELLS];
  const int part = threadIdx.x / CELLS, k = threadIdx.x % CELLS;
  const long c = (long)b.x * CELLS + k;
  if (c < g.nwc) {
    double w[ND][V];
#pragma unroll
    for (int idx = 0; idx < ND; idx++)
#pragma unroll
      for (int v = 0; v < V; v++) w[idx][v] = wh[(long)(idx * V + v) * g.nwc + c];
    double q[V], dq[D * V];
#pragma unroll
    for (int v = 0; v < V; v++) q[v] = wm[(long)v * g.nwc + c];
    static_for<0, D>([&](auto dc) {
      constexpr int d = decltype(dc)::value;
      double acc[V], tmp[V];
#pragma unroll
      for (int idx = 0; idx < ND; idx++) {
        cell_deriv<d>(w, idx, 1.0 / g.dX[d], tmp);
#pragma unroll
        for (int v = 0; v < V; v++) acc[v] = (idx == 0) ? T_WP[0] * tmp[v] : dfma(T_WP[idx], tmp[v], acc[v]);
      }
#pragma unroll
      for (int v = 0; v < V; v++) dq[d * V + v] = acc[v];
    });
    static_for<0, D>([&](auto dc) {
      constexpr int d = decltype(dc)::value;
      double f0[V];
      if (part == 2 * d) lam[2 * d][k] = max_abs_eigs(q, dq, d, f0);
      if (part == 2 * d + 1) lam[2 * d + 1][k] = max_abs_eigs_second_order<d>(q, dq, g.dX[d]);
    });
  }
  __syncthreads();
  double sum = 0.0;
  if (part == 0 && c < g.nwc) {
#pragma unroll
    for (int d = 0; d < D; d++) sum = sum + (lam[2 * d][k] + lam[2 * d + 1][k]) / g.dX[d];
    if (!(sum > 0.0)) sum = 0.0;
  }
  const double m = wave_max(sum);
  if ((threadIdx.x & 63) == 0 && m > 0.0)
    atomicMax(&st->pstat[b.x & 63][8], (unsigned long long)__double_as_longlong(m));
  if (last_workgroup(st, &st->dt_ticket, 9, b)) dt_finalize(st);
}
#else
DEV void dt_body(const double* __restrict__ wh, const double* __restrict__ wm, StepState* st,
                 const Geom& g, const Blk& b) {
  const long item = (long)b.x * 256 + threadIdx.x;
  const long c = DT_PAIR ? (item >> 1) : item;
  const int stop = st->done;
  double q[V], dq[D * V];
  if (c < g.nwc) {
#pragma unroll
    for (int v = 0; v < V; v++) q[v] = wm[(long)v * g.nwc + c];
  }
  LOADS_FIRST();
  if (stop) return;
  // a first-order F takes no gradient (the reference gives it none)
#pragma unroll
  for (int i = 0; i < D * V; i++) dq[i] = 0.0;
  double sum = 0.0;
  if (c < g.nwc) {
    if constexpr (DT_PAIR) {
      const int dl = (int)(item & 1);
      double f0[V];
      const double part = max_abs_eigs(q, dq, dl, f0) / (dl ? g.dX[1] : g.dX[0]);
      const double other = __shfl_xor(part, 1, 64);
      sum = dl ? other + part : part + other;
    } else {
      static_for<0, D>([&](auto dc) {
        constexpr int d = decltype(dc)::value;
        double f0[V];
        sum = sum + max_abs_eigs(q, dq, d, f0) / g.dX[d];
      });
    }
    if (!(sum > 0.0)) sum = 0.0;
  }
  double m = wave_max(sum);
  if ((threadIdx.x & 63) == 0 && m > 0.0)
    atomicMax(&st->pstat[b.x & 63][8], (unsigned long long)__double_as_longlong(m));
  // the last workgroup to finish takes dt from the 64 slots
  if (last_workgroup(st, &st->dt_ticket, 9, b)) dt_finalize(st);
}
#endif

extern "C" __global__ void __launch_bounds__(256)
k_dt(const double* __restrict__ wh, const double* __restrict__ wm, StepState* st, Geom g) {
  dt_body(wh, wm, st, g, lin_blk());
}

// dt = CFL / MAX, x0.2 while count <= 5, clamped to tf - t (stepper.cpp:67-75),
// MAX the maximum over the 64 slots k_dt spreads its atomics over (IEEE bits
// of values >= 0 order as integers); each slot is read and cleared with one
// atomic exchange.  Run by the first wavefront of the last workgroup.
DEV void dt_finalize(StepState* st) {
  if (threadIdx.x >= 64) return;
  unsigned long long b = atomicExch(&st->pstat[threadIdx.x][8], 0ull);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    unsigned long long y = __shfl_xor(b, o, 64);
    b = b > y ? b : y;
  }
  if (threadIdx.x != 0) return;
  double MAX = __longlong_as_double((long long)b);
  double dt = st->cfl / MAX;
  if (st->count <= 5) dt = dt * 0.2;
  if (st->t + dt > st->tf) dt = st->tf - st->t;
  st->dt = dt;
  st->hot_count = 0ull;
}

// ------------------------------------------------------- eigen diagnostics
// The wave-speed and |A| routines on a batch of V x V matrices (row-major,
// one per thread), for checking them against the CPU restatement:
// which 0: max_abs_eig, out of n entries; 2: abs_apply(A_i, x_i) (Roe and
// Osher modules), out of n V.
extern "C" __global__ void __launch_bounds__(256)
k_eig_batch(const double* __restrict__ A, const double* __restrict__ x, double* __restrict__ out,
            long n, int which) {
#if PDE_WIDE_EIG
  // a workgroup's 256 matrices, 64 in turn per wavefront (which is 0: Roe and
  // Osher stop at V = 8)
  __shared__ WideMat mats[WIDE_WAVES];
  const int lane = threadIdx.x & 63;
  const long i0 = (long)blk_x() * 256 + (threadIdx.x & ~63u);
  for (long k = i0; k < i0 + 64 && k < n; k++) {
    double col[V];
#pragma unroll
    for (int r = 0; r < V; r++) col[r] = lane < V ? A[k * V * V + r * V + lane] : 0.0;
    const double lam = wide_max_abs_eig(mats[threadIdx.x >> 6], col, lane);
    if (lane == 0) out[k] = lam;
  }
  (void)x;
  (void)which;
#else
  const long i = (long)blk_x() * 256 + threadIdx.x;
  if (i >= n) return;
  double H[V * V];
#pragma unroll
  for (int k = 0; k < V * V; k++) H[k] = A[i * V * V + k];
  if (which == 0) {
    out[i] = max_abs_eig(H);
    return;
  }
#if PDE_FLUX != 0
  double xv[V], y[V];
#pragma unroll
  for (int v = 0; v < V; v++) xv[v] = x[i * V + v];
  abs_apply(H, xv, y);
#pragma unroll
  for (int v = 0; v < V; v++) out[i * V + v] = y[v];
#else
  (void)x;
#endif
#endif
}
