// sgeo_bvec.hip -- vector kernels and reductions of the multi-trial engine
// on the interleaved [equation][column] arrays.
//
// The equations are split into tiles of T (8 .. 256, a power of two chosen
// by the equation count only: enough tiles to fill the chip on small systems,
// at most 16,384 of them up to 4.19 million equations, where T has reached
// 256, and n / 256 above).  A tile's partial of
// a column is the sum of eight interleaved accumulators, accumulator i
// taking the equations 8 s + i of the tile in order of s, combined pairwise
// (0,1) (2,3) .., then the pairs, then the two halves; four or eight tiles
// make a group (tile_group), summed in order, and one partial leaves the
// block per group.  None
// of it depends on the column count B or on the launch, so a column's bits
// are the same in any engine, while the lanes are laid out for B: with 64
// columns a wave walks one equation at a time and keeps the eight
// accumulators of each column in registers; with 8, its lanes hold eight
// consecutive equations of the eight columns, one accumulator each (every
// load still covers whole lines); below, a wave holds several tiles.
//
// Measured against one thread per (column, chunk of consecutive equations),
// which used 32 of a line's 128 bytes per load at 8 columns, in us: update
// 97 -> 29 and x write 117 -> 44 on 25,344 elements, 8 columns; update 18.9
// -> 8.0 on 6,300, one column; update 111 -> 102, x write 233 -> 189 on
// 12,544, 64 columns, where both stream at 4.3 - 4.6 TB/s of the card's 4.8.
// The groups' partials are few enough for one final stage per reduction; it
// had been a grouping launch of 9 - 14 us and a final one of 4 - 6.
#pragma clang fp contract(off)

#include "sgeo_device.h"
#include "sgeo_internal.h"

namespace sgeo {

template <int B, int G>  // G tiles per group
struct Tile {
  static constexpr int NR = 64 / B < 8 ? 64 / B : 8;  // equations side by side per tile
  static constexpr int A = 8 / NR;                    // accumulators per lane
  static constexpr int TPW = 64 / (B * NR);           // tiles per wave
  static constexpr int W = TPW < G / 4 ? G / TPW : 4;  // waves per block
  static constexpr int NT = 64 * W;                    // threads per block
  static constexpr int GPB = W * TPW / G;              // groups per block
};

// One pass over this wave's tile(s).  f.load(g) reads what equation g of the
// lane's column needs, f.apply(data, g, v) does its work and gives the NK
// values to reduce; f.stage(g, n) (all lanes) prepares the n <= 64 equations
// from g.
// The loads of F::BATCH equations are issued together; g is clamped for them,
// never for apply.  Every thread of the block calls it.
template <int B, int G, int NK, class F>
__device__ __forceinline__ void tile_walk(F& f, int64_t n1, int T, bool act,
                                          const int (&kind)[NK], const bool (&is_max)[NK],
                                          const bool (&put)[NK], double* __restrict__ part,
                                          int64_t ng) {
  using S_ = Tile<B, G>;
  constexpr int NR = S_::NR, A = S_::A, TPW = S_::TPW, W = S_::W;
  constexpr int AB = A < F::BATCH ? A : F::BATCH;  // accumulators and steps of a batch
  constexpr int U = F::BATCH / AB;
  __shared__ double red[NK][W * TPW][B];
  const int t = threadIdx.x, l = t & 63, w = t >> 6;
  const int j = l % B, row = (l / B) % NR, sub = l / (B * NR);
  const int64_t tile = ((int64_t)blockIdx.x * W + w) * TPW + sub;
  const int64_t g0 = tile * T;
  const bool on = act && g0 < n1;
  double acc[NK][A];
#pragma unroll
  for (int k = 0; k < NK; k++)
#pragma unroll
    for (int a = 0; a < A; a++) acc[k][a] = 0.0;
  if (__any(on)) {
    const int S = T >> 3;
    for (int s0 = 0; s0 < S; s0 += 8) {
      const int s1 = s0 + 8 < S ? s0 + 8 : S;
      f.stage(g0 + 8 * s0, 8 * (s1 - s0));
      if (on)
        for (int s = s0; s < s1; s += U) {
#pragma unroll
          for (int a0 = 0; a0 < A; a0 += AB) {
            typename F::Data d[U][AB];
#pragma unroll
            for (int q = 0; q < U; q++)
#pragma unroll
              for (int a = 0; a < AB; a++) {
                const int64_t g = g0 + 8 * (s + q) + row + NR * (a0 + a);
                if (s + q < s1) d[q][a] = f.load(g < n1 ? g : n1 - 1);
              }
#pragma unroll
            for (int q = 0; q < U; q++)
#pragma unroll
              for (int a = 0; a < AB; a++) {
                const int64_t g = g0 + 8 * (s + q) + row + NR * (a0 + a);
                if (s + q < s1 && g < n1) {
                  double v[NK];
                  f.apply(d[q][a], g, v);
#pragma unroll
                  for (int k = 0; k < NK; k++) {
                    double& c = acc[k][a0 + a];
                    c = is_max[k] ? fmax(c, v[k]) : c + v[k];
                  }
                }
              }
          }
        }
    }
  }
#pragma unroll
  for (int k = 0; k < NK; k++) {
    int n = A;
#pragma unroll
    for (int b = 0; b < 3; b++) {  // accumulators i and i ^ (1 << b)
      if ((1 << b) < NR) {
#pragma unroll
        for (int a = 0; a < A; a++) {
          const double o = __shfl_xor(acc[k][a], B << b, 64);
          acc[k][a] = is_max[k] ? fmax(acc[k][a], o) : acc[k][a] + o;
        }
      } else {
#pragma unroll
        for (int a = 0; a < A / 2; a++)
          if (2 * a < n)
            acc[k][a] = is_max[k] ? fmax(acc[k][2 * a], acc[k][2 * a + 1])
                                  : acc[k][2 * a] + acc[k][2 * a + 1];
        n /= 2;
      }
    }
    if (row == 0) red[k][w * TPW + sub][j] = acc[k][0];
  }
  __syncthreads();
  if (t >= S_::GPB * B) return;
  const int q = t / B;  // group of the block; t % B is this lane's column
  const int64_t g = (int64_t)blockIdx.x * S_::GPB + q;
  if (g >= ng) return;
#pragma unroll
  for (int k = 0; k < NK; k++) {
    if (!put[k]) continue;
    double a = red[k][G * q][j];
#pragma unroll
    for (int i = 1; i < G; i++) {
      const double o = red[k][G * q + i][j];
      a = is_max[k] ? fmax(a, o) : a + o;
    }
    part[(kind[k] * ng + g) * B + j] = a;
  }
}

// --------------------------------------------------------------------------
// The final stage of a reduction combines the groups' partials and advances
// the columns' state machines.
//   RESID: r.z of the FP64 residual, max|x| (START).
//   ALPHA: the elements' p.Kp shares from the product (a "group" is one of
//          their tiles' groups, or an element below BFIN_DIRECT_ELEMENTS).
//   INNER: max|x|, r.z, max|p|.
// Row i of 256 takes the values i, i + 256, ..; the rows are combined by the
// bits of i from the highest down.  The order depends on the count of values
// only, wherever the stage runs: in a launch of its own (k_bfinalize), or,
// where the values are few (BFIN_FUSED), in every block of the kernel that
// needs its result: ALPHA in the update, INNER in the next step's direction.
// There each block reads all values, 2 - 3 us, and a step of a small system
// is three launches instead of five.  Plastic iterations against launches of
// their own everywhere: sweeps of 8 columns on 384 elements 72 -> 64 ms, one
// column on 6,300 elements 25.6 -> 24.0 and on 25,344 77.4 -> 73.5, two on
// 12,544 56.0 -> 53.9.  Above BFIN_FUSED the read costs more than the launch
// (8 columns on 25,344 elements, 6,300 values per kind: update 29 -> 37 us); a
// launch reads with a block per column, since few wide blocks cannot draw the
// values in fast enough (64 columns on 12,544 elements: 22 us by blocks of
// eight columns, 16 by one).
// --------------------------------------------------------------------------
#define BFIN_KINDS 4  // max|x|, r.z, max|p| of the steps on state 0 and state 1
#define BFIN_ROWS 256
#define BFIN_FUSED 4096  // values per kind, all columns

__device__ __forceinline__ int fin_states(int what) {
  return what == BFIN_RESID ? (BCOL_BIT(BCOL_START) | BCOL_BIT(BCOL_REPLACE))
                            : BCOL_BIT(BCOL_INNER);
}

// kind k of `what` combines by max (else by sum)
__device__ __forceinline__ constexpr bool fin_max(int what, int k) {
  return (what == BFIN_INNER && k != 1) || (what == BFIN_RESID && k == 1);
}

__device__ __forceinline__ constexpr int fin_kinds(int what) {
  return what == BFIN_INNER ? 3 : what == BFIN_RESID ? 2 : 1;
}

// Columns j0 .. j0 + CB - 1 by a block of NT threads: v[k] of column
// j0 + t % CB in every thread.  Kind k of value b at src[k][b * B + j]; kinds
// below k0 are left out (INNER of a step that did not write x has no max|x|:
// a third less to read).
template <int WHAT, int CB, int NT>
__device__ __forceinline__ void fin_combine(const double* const (&src)[3], int64_t ng, int B,
                                            int j0, int k0, double (&v)[3]) {
  constexpr int NK = fin_kinds(WHAT);
  constexpr int RPT = 256 * CB / NT > 0 ? 256 * CB / NT : 1;  // rows per thread
  constexpr int H = BFIN_ROWS / RPT;                          // rows after the thread's own
  static_assert(H % 8 == 0, "eight low rows");
  __shared__ double top[NK][H][CB], low[NK][8][CB];
  const int t = threadIdx.x, c = t % CB, row = t / CB;
  auto op = [](int k, double a, double b) { return fin_max(WHAT, k) ? fmax(a, b) : a + b; };
  if (row < H) {
    double a[NK][RPT];
#pragma unroll
    for (int k = 0; k < NK; k++)
#pragma unroll
      for (int m = 0; m < RPT; m++) a[k][m] = 0.0;
    constexpr int U = 8 / RPT;  // eight values of a kind in flight
    const int n = (int)ng;
    for (int b0 = row; b0 < n; b0 += U * BFIN_ROWS) {
      double y[NK][U][RPT];
#pragma unroll
      for (int k = 0; k < NK; k++)
        if (k >= k0)
#pragma unroll
          for (int u = 0; u < U; u++)
#pragma unroll
            for (int m = 0; m < RPT; m++) {  // past the end: the last value, not used
              const int b = min(b0 + u * BFIN_ROWS + m * H, n - 1);
              y[k][u][m] = src[k][b * B + j0 + c];
            }
#pragma unroll
      for (int k = 0; k < NK; k++)
        if (k >= k0)
#pragma unroll
          for (int u = 0; u < U; u++)
#pragma unroll
            for (int m = 0; m < RPT; m++)
              if (b0 + u * BFIN_ROWS + m * H < n) a[k][m] = op(k, a[k][m], y[k][u][m]);
    }
#pragma unroll
    for (int k = 0; k < NK; k++) {
#pragma unroll
      for (int h = RPT / 2; h > 0; h /= 2)
#pragma unroll
        for (int m = 0; m < h; m++) a[k][m] = op(k, a[k][m], a[k][m + h]);
      top[k][row][c] = a[k][0];
    }
  }
  __syncthreads();
  if (row < 8) {
    constexpr int N = H / 8;
#pragma unroll
    for (int k = 0; k < NK; k++) {
      double a[N];
#pragma unroll
      for (int m = 0; m < N; m++) a[m] = top[k][row + 8 * m][c];
#pragma unroll
      for (int h = N / 2; h > 0; h /= 2)
#pragma unroll
        for (int m = 0; m < h; m++) a[m] = op(k, a[m], a[m + h]);
      low[k][row][c] = a[0];
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NK; k++) {
    double a[8];
#pragma unroll
    for (int m = 0; m < 8; m++) a[m] = low[k][m][c];
#pragma unroll
    for (int h = 4; h > 0; h /= 2)
#pragma unroll
      for (int m = 0; m < h; m++) a[m] = op(k, a[m], a[m + h]);
    v[k] = a[0];
  }
}

// one column's step of its state machine; st: its state
__device__ __forceinline__ void fin_advance(int what, const double (&v)[3], BCol& c, int32_t& st,
                                            int xw) {
  switch (what) {
    case BFIN_RESID:  // v0 = r.z of the FP64 residual, v1 = max|x| (START)
      c.nrep += 1;
      if (st == BCOL_START) {
        c.rz = v[0];
        c.rz0 = v[0];
        c.it = 0;
        c.pending = 0;
        c.maxx = v[1];
        c.xsum = 0.0;
        c.npend = 0;
        st = (v[0] == 0.0) ? BCOL_DONE : BCOL_INNER;  // r = 0: x is exact
      } else {  // replaces r_{k+1}: beta = r.z (true) / r_k.z_k
        c.beta = v[0] / c.rz_prev;
        c.rz = v[0];
        c.rz0 = v[0];
        c.pending = 1;
        st = BCOL_INNER;
      }
      break;
    case BFIN_ALPHA:  // v0 = p.Kp
      c.alpha = c.rz / v[0];
      c.alpha_hist[(c.it + 1) & 7] = c.alpha;
      c.pending = 0;
      break;
    case BFIN_INNER: {  // v0 = max|x| (x written), v1 = r.z, v2 = max|p|
      c.it += 1;
      c.maxp = v[2];
      const double a = fabs(c.alpha) * v[2];
      const bool xit = (c.it & (c.xlen - 1)) == 0;
      if (xit != (xw != 0)) {
        // the step's update and the column disagree on whether x was
        // written (the engine's step phase and the column's iteration
        // count went apart): the column ends, and the host reports it
        c.xerr = 1;
        st = BCOL_FAIL;
        break;
      }
      bool stop;
      if (xit) {
        // relative update test of src/solver.f90:65 (after the x update)
        stop = a / v[0] <= c.tol;
        c.maxx = v[0];
        c.xsum = 0.0;
        c.npend = 0;
      } else {
        // x_it = x_w + sum of alpha_k p_k over the iterations after the last
        // write w is not written yet, but max|x_it| >= max|x_w| - xsum with
        // xsum the sum of |alpha_k| max|p_k|: a <= tol (max|x_w| - xsum)
        // passes the same test for certain.  Only inside the window of
        // relative width ~tol xsum / max|x| (~xlen tol^2 near convergence)
        // where the bound cannot decide does the solve iterate once more
        // than the test would.
        c.xsum += a;
        stop = a <= c.tol * (c.maxx - c.xsum);
        c.npend += 1;
      }
      if (stop) {
        st = BCOL_DONE;
      } else if (c.it >= c.maxiter) {
        st = BCOL_FAIL;
      } else {
        c.rz_prev = c.rz;
        // due for an FP64 residual: replaced at the next residual step, by
        // when the column may have iterated on
        if (v[1] <= c.inner_tol * c.rz0) c.want_rep = 1;
        c.beta = v[1] / c.rz;
        c.rz = v[1];
        c.pending = 1;
      }
      break;
    }
  }
}

// p_i = D r + beta p_{i-1} for INNER columns with a pending beta (i the
// iteration about to run; p_i in buffer i & pmask of the n1 x B buffers),
// and the partial of max|p_i| for the iteration's stop test (INNER kind 2)
template <int B>
struct PUpdate {
  static constexpr int BATCH = 4;
  struct Data {
    float r, p, d;
  };
  const float *r, *dinv, *pold;
  float* pnew;
  float beta;
  int j;
  __device__ __forceinline__ void stage(int64_t, int) {}
  __device__ __forceinline__ Data load(int64_t g) const {
    return {r[g * B + j], pold[g * B + j], dinv[g]};
  }
  __device__ __forceinline__ void apply(const Data& d, int64_t g, double (&v)[1]) {
    const float pg = d.d * d.r + beta * d.p;
    pnew[g * B + j] = pg;
    v[0] = fabs((double)pg);
  }
};

// FIN: every block first runs the INNER stage of the step before on the state
// (cst, bc); the first one writes the new state.  slot: where max|p| goes.
template <int B, int G, bool FIN>
__global__ __launch_bounds__((Tile<B, G>::NT)) void k_bpupdate(
    int64_t n1, int T, int64_t ng, const float* __restrict__ r, const float* __restrict__ dinv,
    float* __restrict__ p, double* part, int slot, const int32_t* __restrict__ cst,
    const BCol* __restrict__ bc, int32_t* __restrict__ cstn, BCol* __restrict__ bcn, int xw) {
  const int t = threadIdx.x, j = t % B;
  bool act = cst[j] == BCOL_INNER;
  int i, pm;
  float beta;
  if constexpr (FIN) {
    __shared__ float s_beta[B];
    __shared__ int32_t s_it[B], s_pm[B], s_act[B];
    double v[3];
    const double* const src[3] = {part, part + ng * B, part + (5 - slot) * ng * B};
    BCol c;
    int32_t st;
    if (t < B) {  // in flight beside the values
      c = bc[t];
      st = cst[t];
    }
    fin_combine<BFIN_INNER, B, Tile<B, G>::NT>(src, ng, B, 0, xw ? 0 : 1, v);
    if (t < B) {
      if (act) fin_advance(BFIN_INNER, v, c, st, xw);
      s_act[t] = st == BCOL_INNER && c.pending;
      s_beta[t] = (float)c.beta;
      s_it[t] = c.it;
      s_pm[t] = c.pmask;
      if (blockIdx.x == 0) {
        bcn[t] = c;
        cstn[t] = st;
      }
    }
    __syncthreads();
    act = s_act[j];
    i = s_it[j] + 1;
    pm = s_pm[j];
    beta = s_beta[j];
  } else {
    act = act && bc[j].pending;
    i = bc[j].it + 1;
    pm = bc[j].pmask;
    beta = (float)bc[j].beta;
  }
  const int64_t nv = n1 * B;
  PUpdate<B> f{r, dinv, p + ((i - 1) & pm) * nv, p + (i & pm) * nv, beta, j};
  tile_walk<B, G, 1>(f, n1, T, act, {slot}, {true}, {act}, part, ng);
}

// The update of an iteration, with kp assembled on the fly:
//   kp[g][j] = sum over the slots of Y (element order, FP32),
//   r -= alpha kp, z = D r,
// and the r.z partial (FP64, kind 1) for INNER columns.  x is written by
// k_bxfold on the steps that write it; max|p| comes from where p was formed
// (k_bpupdate, or k_bresid for p_1), so the update reads neither x nor p.
// The (at most 8 on hexahedral meshes) element contributions of an equation
// are loaded together, then summed in slot order.  Where a wave walks one
// tile (B >= 8) it first stages the row pointers and slots of 64 equations
// in its LDS rows, one coalesced load each, so the gathers wait on one memory
// level instead of three.
#define UPD_SL 512  // staged slots per wave (64 equations, 8 slots each)

// The contributions of a row.  Below eight columns a wave's lanes hold many
// rows and all eight are loaded, past a row's end its last one again:
// conditional loads compile to a branch each, and every slot's latency stood
// before the next one's (update of 6,300 elements, one column 9.0 -> 7.8 us;
// plastic iterations there 24.0 -> 22.9 ms, of 25,344 73.7 -> 65.0).
// From eight columns on the rows of a wave are few and the branches skip
// loads: unconditional ones cost 8 columns on 25,344 elements 6 %, 64 on
// 12,544 8 %.
template <int B, typename T>
__device__ __forceinline__ void gather8(const int32_t* __restrict__ slots,
                                        const T* __restrict__ Y, int32_t q0, int32_t q1, int j,
                                        T (&v)[8]) {
  if constexpr (B >= 8) {
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = q0 + k < q1 ? Y[(int64_t)slots[q0 + k] * B + j] : (T)0;
  } else {
    int32_t at[8];
#pragma unroll
    for (int k = 0; k < 8; k++) at[k] = slots[max(min(q0 + k, q1 - 1), 0)];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = Y[(int64_t)(q1 > q0 ? at[k] : 0) * B + j];
  }
}
template <int B>
struct Update {
  static constexpr int BATCH = 4;
  struct Data {
    float v[8], r, d;
    int32_t q0, q1;
  };
  const int32_t *rowptr, *slots;
  const float *Y, *dinv;
  float* r;
  int64_t n1;
  float alpha;
  int j;
  int32_t *rp, *sl;  // the wave's staged rows
  int64_t ga;        // first staged equation
  bool staged;
  __device__ __forceinline__ void stage(int64_t g0, int n) {
    staged = false;
    if constexpr (B >= 8) {
      const int ln = threadIdx.x & 63;
      ga = g0 > 0 ? g0 : 1;  // equation 0, the sink, has no update
      const int64_t ge = g0 + n < n1 ? g0 + n : n1;
      const int nr = (int)(ge - ga) + 1;  // <= 65; the walk stays below n1
      if (nr < 2) return;
      __builtin_amdgcn_wave_barrier();  // the rows staged before are read
      if (ln < nr) rp[ln] = rowptr[ga + ln];
      if (ln == 0 && nr > 64) rp[64] = rowptr[ga + 64];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const int32_t sb = rp[0], nsl = rp[nr - 1] - sb;
      if (nsl > UPD_SL) return;
      for (int k = ln; k < nsl; k += 64) sl[k] = slots[sb + k];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      staged = true;
    }
  }
  __device__ __forceinline__ Data load(int64_t g) const {
    Data d;
    if (B >= 8 && staged) {
      d.q0 = g > 0 ? rp[g - ga] : 0;
      d.q1 = g > 0 ? rp[g - ga + 1] : 0;
      const int32_t sb = rp[0];
#pragma unroll
      for (int k = 0; k < 8; k++)
        d.v[k] = d.q0 + k < d.q1 ? Y[(int64_t)sl[d.q0 + k - sb] * B + j] : 0.0f;
    } else {
      d.q0 = rowptr[g];  // row 0, the sink, is empty
      d.q1 = rowptr[g + 1];
      gather8<B>(slots, Y, d.q0, d.q1, j, d.v);
    }
    d.r = r[g * B + j];
    d.d = dinv[g];
    return d;
  }
  __device__ __forceinline__ void apply(const Data& d, int64_t g, double (&v)[1]) {
    float kp = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++)
      if (d.q0 + k < d.q1) kp = kp + d.v[k];
    for (int32_t q = d.q0 + 8; q < d.q1; q++) kp = kp + Y[(int64_t)slots[q] * B + j];
    const float rg = d.r - alpha * kp;
    r[g * B + j] = rg;
    const float zg = d.d * rg;
    v[0] = (double)rg * (double)zg;
  }
};

// FIN: every block first runs the ALPHA stage on the nfin values of fin; the
// first one writes alpha to the state, where no block of this launch reads it.
template <int B, int G, bool FIN>
__global__ __launch_bounds__((Tile<B, G>::NT)) void k_bupdate(
    int64_t n1, int T, int64_t ng, const int32_t* __restrict__ rowptr,
    const int32_t* __restrict__ slots, const float* __restrict__ Y,
    const float* __restrict__ dinv, float* __restrict__ r, double* __restrict__ part,
    const int32_t* __restrict__ cst, BCol* bc, const double* __restrict__ fin, int64_t nfin) {
  __shared__ int32_t idx[B >= 8 ? Tile<B, G>::W * (65 + UPD_SL) : 1];
  const int t = threadIdx.x, j = t % B;
  const bool act = cst[j] == BCOL_INNER;
  double alpha;
  if constexpr (FIN) {
    double v[3];
    const double* const src[3] = {fin, fin, fin};
    const double rz = bc[j].rz;
    const int i = bc[j].it + 1;
    fin_combine<BFIN_ALPHA, B, Tile<B, G>::NT>(src, nfin, B, 0, 0, v);
    alpha = rz / v[0];
    if (blockIdx.x == 0 && t < B && act) {
      bc[t].alpha = alpha;
      bc[t].alpha_hist[i & 7] = alpha;
      bc[t].pending = 0;
    }
  } else {
    alpha = bc[j].alpha;
  }
  int32_t* wr = idx + (B >= 8 ? (t >> 6) * (65 + UPD_SL) : 0);
  Update<B> f{rowptr, slots, Y, dinv, r, n1, (float)alpha, j, wr, wr + 65, 0, false};
  tile_walk<B, G, 1>(f, n1, T, act, {1}, {false}, {act}, part, ng);
}

// The x write of an iteration i with i % xlen == 0 (INNER columns), after
// the update of i: the npend deferred updates before i and i's own, in
// order, x += alpha_k p_k for k = i - np + 1 .. i (np = npend + 1 <= 8),
// and the max|x| partial (kind 0; x(0) = 0) for i's stop test.
template <int B>
struct XFold {
  static constexpr int BATCH = 2;
  struct Data {
    double x;
    float p[8];
  };
  double* x;
  const float* p;
  int j, np;
  double al[8];
  uint32_t pk[8];  // buffer offsets, (pmask + 1) n1 B < 2^32
  __device__ __forceinline__ void stage(int64_t, int) {}
  __device__ __forceinline__ Data load(int64_t g) const {
    Data d;
    const int64_t q = g * B + j;
    d.x = x[q];
#pragma unroll
    for (int k = 0; k < 8; k++) d.p[k] = p[pk[k] + q];  // k >= np: a repeated buffer
    return d;
  }
  __device__ __forceinline__ void apply(const Data& d, int64_t g, double (&v)[1]) {
    double xg = d.x;
#pragma unroll
    for (int k = 0; k < 8; k++)
      if (k < np) xg = xg + al[k] * (double)d.p[k];
    if (g == 0) xg = 0.0;
    x[g * B + j] = xg;
    v[0] = fabs(xg);
  }
};

template <int B, int G>
__global__ __launch_bounds__((Tile<B, G>::NT)) void k_bxfold(int64_t n1, int T, int64_t ng,
                                                double* __restrict__ x,
                                                const float* __restrict__ p,
                                                double* __restrict__ part,
                                                const int32_t* __restrict__ cst,
                                                const BCol* __restrict__ bc) {
  const int j = threadIdx.x % B;
  const BCol& bj = bc[j];
  const int i = bj.it + 1;
  // a column off the x-writing phase writes nothing here; the INNER finalize
  // reports it
  const bool act = cst[j] == BCOL_INNER && (i & (bj.xlen - 1)) == 0;
  XFold<B> f;
  f.x = x;
  f.p = p;
  f.j = j;
  f.np = act ? bj.npend + 1 : 0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int it = i - f.np + 1 + (k < f.np ? k : 0);
    f.al[k] = bj.alpha_hist[it & 7];
    f.pk[k] = (uint32_t)(it & bj.pmask) * (uint32_t)(n1 * B);
  }
  tile_walk<B, G, 1>(f, n1, T, act, {0}, {true}, {act}, part, ng);
}

// FP64 residual for START / REPLACE columns: r64 = load - sum Y64 (element
// order, FP64; Y64 holds the residual list's columns at their list places);
// r = (float) r64; START: p_1 = D r (buffer 1); partials r.(D r) and (START)
// max|x_0|, and for START the first iteration's max|p_1| (kind 2, the INNER
// reduction's third)
template <int B>
struct Resid {
  static constexpr int BATCH = 1;
  struct Data {
    double v[8], b, x;
    float d;
    int32_t q0, q1;
  };
  const int32_t *rowptr, *slots;
  const double *Y64, *rhs, *x;
  const float* dinv;
  float *r, *p1;
  int j, qs;
  bool start;
  __device__ __forceinline__ void stage(int64_t, int) {}
  __device__ __forceinline__ Data load(int64_t g) const {
    Data d;
    d.q0 = rowptr[g];
    d.q1 = rowptr[g + 1];
    gather8<B>(slots, Y64, d.q0, d.q1, qs, d.v);
    d.b = rhs[g * B + j];
    d.x = start ? x[g * B + j] : 0.0;
    d.d = dinv[g];
    return d;
  }
  __device__ __forceinline__ void apply(const Data& d, int64_t g, double (&v)[3]) {
    double kx = 0.0;
#pragma unroll
    for (int k = 0; k < 8; k++)
      if (d.q0 + k < d.q1) kx = kx + d.v[k];
    for (int32_t q = d.q0 + 8; q < d.q1; q++) kx = kx + Y64[(int64_t)slots[q] * B + qs];
    const double r64 = g == 0 ? 0.0 : d.b - kx;
    const float rg = (float)r64;
    const float zg = d.d * rg;
    r[g * B + j] = rg;
    if (start) p1[g * B + j] = zg;
    v[0] = (double)rg * (double)zg;
    v[1] = fabs(d.x);
    v[2] = start ? fabs((double)zg) : 0.0;
  }
};

template <int B, int G>
__global__ __launch_bounds__((Tile<B, G>::NT)) void k_bresid(
    int64_t n1, int T, int64_t ng, const int32_t* __restrict__ rowptr,
    const int32_t* __restrict__ slots, const double* __restrict__ Y64,
    const double* __restrict__ load, const float* __restrict__ dinv,
    const double* __restrict__ x, float* __restrict__ r, float* __restrict__ p,
    double* __restrict__ part, const int32_t* __restrict__ cst,
    const int32_t* __restrict__ rslot, const int32_t* __restrict__ rlist) {
  if (rlist[64] == 0) return;  // the common case: no column needs a residual
  const int j = threadIdx.x % B, st = cst[j];
  const bool act = st == BCOL_START || st == BCOL_REPLACE;
  Resid<B> f{rowptr, slots, Y64, load, x, dinv, r, p + n1 * B, j, act ? rslot[j] : 0,
             st == BCOL_START};
  tile_walk<B, G, 3>(f, n1, T, act, {0, 1, 2}, {false, true, true},
                  {act, act, st == BCOL_START}, part, ng);
}

// uerr per column: x(0)=0, partial max|x-oldx| and max|x|, oldx = x
template <int B>
struct UErr {
  static constexpr int BATCH = 4;
  struct Data {
    double x, o;
  };
  double *x, *oldx;
  int j;
  __device__ __forceinline__ void stage(int64_t, int) {}
  __device__ __forceinline__ Data load(int64_t g) const {
    return {x[g * B + j], oldx[g * B + j]};
  }
  __device__ __forceinline__ void apply(const Data& d, int64_t g, double (&v)[2]) {
    double xg = d.x;
    if (g == 0) {
      xg = 0.0;
      x[j] = 0.0;
    }
    oldx[g * B + j] = xg;
    v[0] = fabs(xg - d.o);
    v[1] = fabs(xg);
  }
};

template <int B, int G>
__global__ __launch_bounds__((Tile<B, G>::NT)) void k_buerr(int64_t n1, int T, int64_t ng,
                                               double* __restrict__ x,
                                               double* __restrict__ oldx,
                                               double* __restrict__ part,
                                               const int32_t* __restrict__ active) {
  const int j = threadIdx.x % B;
  const bool act = active[j] != 0;
  UErr<B> f{x, oldx, j};
  tile_walk<B, G, 2>(f, n1, T, act, {0, 1}, {true, true}, {act, act}, part, ng);
}

// the elements' p.Kp shares, as "equations" of the same tiles
template <int B>
struct Shares {
  static constexpr int BATCH = 4;
  typedef double Data;
  const double* e;
  int j;
  __device__ __forceinline__ void stage(int64_t, int) {}
  __device__ __forceinline__ double load(int64_t g) const { return e[g * B + j]; }
  __device__ __forceinline__ void apply(const double& d, int64_t, double (&v)[1]) { v[0] = d; }
};

template <int B, int G>
__global__ __launch_bounds__((Tile<B, G>::NT)) void k_bshares(int64_t n, int T, int64_t ng,
                                                 const double* __restrict__ edot,
                                                 double* __restrict__ part,
                                                 const int32_t* __restrict__ cst) {
  const int j = threadIdx.x % B;
  const bool act = cst[j] == BCOL_INNER;
  Shares<B> f{edot, j};
  tile_walk<B, G, 1>(f, n, T, act, {0}, {false}, {act}, part, ng);
}

// The deferred x updates of a column whose solve ended between two x
// writes (DONE or FAIL with npend > 0): x += alpha_k p_k for the npend
// iterations k after the last write, in order; k_bxlag_clear then clears
// npend.
__global__ __launch_bounds__(256) void k_bmaterialize(int64_t n1, int B,
                                                      double* __restrict__ x,
                                                      const float* __restrict__ p,
                                                      const int32_t* __restrict__ cst,
                                                      const BCol* __restrict__ bc) {
  const int64_t nv = n1 * B, stride = (int64_t)gridDim.x * blockDim.x;  // B divides it
  const int64_t q0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int j = (int)(q0 % B), st = cst[j];
  const BCol& bj = bc[j];
  const int np = bj.npend;  // at most 7
  if ((st != BCOL_DONE && st != BCOL_FAIL) || np == 0) return;
  double al[8];
  const float* pk[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int it = bj.it - np + 1 + (k < np ? k : 0);
    al[k] = bj.alpha_hist[it & 7];
    pk[k] = p + (it & bj.pmask) * nv;
  }
  for (int64_t q = q0; q < nv; q += stride) {
    double xg = 0.0;
    if (q >= B) {
      xg = x[q];
#pragma unroll
      for (int k = 0; k < 8; k++)
        if (k < np) xg = xg + al[k] * (double)pk[k][q];
    }
    x[q] = xg;
  }
}

__global__ void k_bxlag_clear(int B, const int32_t* __restrict__ cst,
                              BCol* __restrict__ bc) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= B) return;
  if (cst[j] == BCOL_DONE || cst[j] == BCOL_FAIL) bc[j].npend = 0;
}

// The stage in a launch of its own; state in (cst, bc), out (cstn, bcn), which
// may be the same.
template <int WHAT>
__global__ __launch_bounds__(256) void k_bfinalize(int64_t ng, int B, const double* s0,
                                                   const double* s1, const double* s2,
                                                   const int32_t* cst, const BCol* bc,
                                                   int32_t* cstn, BCol* bcn, int xw) {
  const int j = blockIdx.x;
  BCol c;
  int32_t st = cst[j];
  const bool act = (fin_states(WHAT) >> st) & 1;  // uniform per block
  if (threadIdx.x == 0) c = bc[j];
  double v[3];
  if (act) {
    const double* const src[3] = {s0, s1, s2};
    fin_combine<WHAT, 1, 256>(src, ng, B, j, WHAT == BFIN_INNER && !xw ? 1 : 0, v);
  } else if (cst == cstn) {
    return;
  }
  if (threadIdx.x != 0) return;
  if (act) fin_advance(WHAT, v, c, st, xw);
  bcn[j] = c;
  cstn[j] = st;
}

__global__ __launch_bounds__(256) void k_buerr_finalize(
    int64_t nch, int B, const double* __restrict__ part,
    PlasticScalars* __restrict__ ps, const int32_t* __restrict__ active,
    double nl_tol) {
  __shared__ double red[4];
  const int j = blockIdx.x;
  if (!active[j]) return;
  double vd = 0.0, vx = 0.0;
#pragma unroll 4
  for (int64_t b = threadIdx.x; b < nch; b += 256) {
    vd = fmax(vd, part[(0 * nch + b) * B + j]);
    vx = fmax(vx, part[(1 * nch + b) * B + j]);
  }
  vd = block_max<4>(vd, red);
  vx = block_max<4>(vx, red);
  if (threadIdx.x == 0) {
    const double uerr = vd / vx;
    ps[j].uerr = uerr;
    ps[j].xmax = vx;
    ps[j].nl_isconv = uerr <= nl_tol ? 1 : 0;
    ps[j].fmax_bits = 0ull;  // fmax = zero (src/slope.F90:286)
    ps[j].n_plastic = 0;
  }
}

// --------------------------------------------------------------------------
// launch wrappers
// --------------------------------------------------------------------------
// tile length, by the count of equations (or elements) only
static int tile_len(int64_t n) {
  int t = 8;
  while (t < 256 && n / t > 16384) t *= 2;
  return t;
}

// tiles per group, by the count only too: eight (blocks of eight waves where a
// wave walks one tile) halve what the final stages read, and cost the large
// systems' streaming kernels the waves that wait for the last tile.  Plastic
// iterations, four against eight: 11,800 equations (8 columns) 69.6 / 64.2 ms,
// 85,000 (8) 31.7 / 31.2, 160,000 (8) 44.9 / 46.2, 322,000 (64) 402 / 424.
static int tile_group(int64_t n) { return n <= (1 << 17) ? 8 : 4; }

static inline int64_t tile_groups(int64_t n) {
  const int64_t per = tile_group(n) * (int64_t)tile_len(n);
  return (n + per - 1) / per;
}

int64_t batch_partials(int64_t n1) { return BFIN_KINDS * tile_groups(n1); }

int64_t batch_element_partials(int32_t nelmt) { return (int64_t)nelmt + tile_groups(nelmt); }

#define SGEO_COLS(kern, n, ...)                                                             \
  do {                                                                                      \
    const int T_ = tile_len(n);                                                             \
    const int64_t ng_ = tile_groups(n);                                                     \
    switch (B) {                                                                            \
      SGEO_COL(kern, 64, n, __VA_ARGS__) SGEO_COL(kern, 32, n, __VA_ARGS__)                 \
      SGEO_COL(kern, 16, n, __VA_ARGS__) SGEO_COL(kern, 8, n, __VA_ARGS__)                  \
      SGEO_COL(kern, 4, n, __VA_ARGS__) SGEO_COL(kern, 2, n, __VA_ARGS__)                   \
      SGEO_COL(kern, 1, n, __VA_ARGS__)                                                     \
    }                                                                                       \
  } while (0)
#define SGEO_COLS8(kern, n, ...)                                                            \
  do {                                                                                      \
    const int T_ = tile_len(n);                                                             \
    const int64_t ng_ = tile_groups(n);                                                     \
    switch (B) {                                                                            \
      SGEO_COL(kern, 8, n, __VA_ARGS__) SGEO_COL(kern, 4, n, __VA_ARGS__)                   \
      SGEO_COL(kern, 2, n, __VA_ARGS__) SGEO_COL(kern, 1, n, __VA_ARGS__)                   \
    }                                                                                       \
  } while (0)
#define SGEO_COL(kern, BB, n, ...)                                                          \
  case BB:                                                                                  \
    if (tile_group(n) == 8) SGEO_COLG(kern, BB, 8, n, __VA_ARGS__);                         \
    else SGEO_COLG(kern, BB, 4, n, __VA_ARGS__);                                            \
    break;
#define SGEO_COLG(kern, BB, G, n, ...)                                                      \
  hipLaunchKernelGGL((kern<BB, G>),                                                         \
                     dim3((unsigned)((ng_ + Tile<BB, G>::GPB - 1) / Tile<BB, G>::GPB)),     \
                     dim3(Tile<BB, G>::NT), 0, s, n, T_, ng_, __VA_ARGS__)

template <int B, int G>
static constexpr auto k_bupdate_run = k_bupdate<B, G, false>;
template <int B, int G>
static constexpr auto k_bupdate_fin = k_bupdate<B, G, true>;
template <int B, int G>
static constexpr auto k_bpupdate_run = k_bpupdate<B, G, false>;
template <int B, int G>
static constexpr auto k_bpupdate_fin = k_bpupdate<B, G, true>;

void launch_bupdate(hipStream_t s, int64_t n1, int B, const int32_t* rowptr,
                    const int32_t* slots, const float* Y, const float* dinv, float* r,
                    double* part, const int32_t* cst, BCol* bc, const BFinSrc* fin) {
  if (fin)
    SGEO_COLS8(k_bupdate_fin, n1, rowptr, slots, Y, dinv, r, part, cst, bc, fin->v, fin->n);
  else
    SGEO_COLS(k_bupdate_run, n1, rowptr, slots, Y, dinv, r, part, cst, bc,
              (const double*)nullptr, (int64_t)0);
}

void launch_bxfold(hipStream_t s, int64_t n1, int B, double* x, const float* p,
                   double* part, const int32_t* cst, const BCol* bc) {
  SGEO_COLS(k_bxfold, n1, x, p, part, cst, bc);
}

// cur: the state (of two) that the step runs on, and where its max|p| goes;
// fin: the INNER stage of the step before, on the other state, comes first
void launch_bpupdate(hipStream_t s, int64_t n1, int B, const float* r,
                     const float* dinv, float* p, double* part, int32_t* cst, BCol* bc,
                     int cur, bool fin, int xw) {
  int32_t* cn = cst + cur * B;
  BCol* bn = bc + cur * B;
  if (fin)
    SGEO_COLS8(k_bpupdate_fin, n1, r, dinv, p, part, 2 + cur,
               (const int32_t*)(cst + (cur ^ 1) * B), (const BCol*)(bc + (cur ^ 1) * B), cn, bn,
               xw);
  else
    SGEO_COLS(k_bpupdate_run, n1, r, dinv, p, part, 2 + cur, (const int32_t*)cn,
              (const BCol*)bn, (int32_t*)nullptr, (BCol*)nullptr, 0);
}

void launch_bresid(hipStream_t s, int64_t n1, int B, const int32_t* rowptr,
                   const int32_t* slots, const double* Y64, const double* load,
                   const float* dinv, const double* x, float* r, float* p,
                   double* part, const int32_t* cst, const int32_t* rslot,
                   const int32_t* rlist) {
  SGEO_COLS(k_bresid, n1, rowptr, slots, Y64, load, dinv, x, r, p, part, cst, rslot, rlist);
}

void launch_bmaterialize(hipStream_t s, int64_t n1, int B, double* x, const float* p,
                         const int32_t* cst, BCol* bc) {
  const int64_t nb = (n1 * B + 255) / 256;
  hipLaunchKernelGGL(k_bmaterialize, dim3((unsigned)(nb < 4096 ? nb : 4096)), dim3(256), 0, s,
                     n1, B, x, p, cst, bc);
  hipLaunchKernelGGL(k_bxlag_clear, dim3((B + 63) / 64), dim3(64), 0, s, B, cst, bc);
}

void launch_buerr(hipStream_t s, int64_t n1, int B, double* x, double* oldx,
                  double* part, PlasticScalars* ps, const int32_t* active,
                  double nl_tol) {
  SGEO_COLS(k_buerr, n1, x, oldx, part, active);
  hipLaunchKernelGGL(k_buerr_finalize, dim3(B), dim3(256), 0, s, tile_groups(n1), B, part, ps,
                     active, nl_tol);
}

// up to here the final stage reads the elements' shares themselves: 16 per
// row, less than the launch that would group them.  By the element count
// only: the grouping is part of the order of the sum.
#define BFIN_DIRECT_ELEMENTS 4096

BFinSrc launch_bshares(hipStream_t s, int32_t nelmt, int B, double* edot, const int32_t* cst) {
  if (nelmt <= BFIN_DIRECT_ELEMENTS) return {edot, nelmt};
  double* groups = edot + (int64_t)nelmt * B;
  SGEO_COLS(k_bshares, (int64_t)nelmt, (const double*)edot, groups, cst);
  return {groups, tile_groups(nelmt)};
}

bool batch_fuse_inner(int64_t n1, int B) { return B <= 8 && tile_groups(n1) * B <= BFIN_FUSED; }
bool batch_fuse_alpha(const BFinSrc& q, int B) { return B <= 8 && q.n * B <= BFIN_FUSED; }

template <int WHAT>
static void finalize(hipStream_t s, int64_t ng, int B, const double* s0, const double* s1,
                     const double* s2, const int32_t* cst, const BCol* bc, int32_t* cstn,
                     BCol* bcn, int xw) {
  hipLaunchKernelGGL(k_bfinalize<WHAT>, dim3(B), dim3(256), 0, s, ng, B, s0, s1, s2, cst, bc,
                     cstn, bcn, xw);
}

void launch_bfin_resid(hipStream_t s, int64_t n1, int B, const double* part, int32_t* cst,
                       BCol* bc) {
  const int64_t ng = tile_groups(n1);
  finalize<BFIN_RESID>(s, ng, B, part, part + ng * B, part, cst, bc, cst, bc, 0);
}

void launch_bfin_alpha(hipStream_t s, const BFinSrc& q, int B, int32_t* cst, BCol* bc) {
  finalize<BFIN_ALPHA>(s, q.n, B, q.v, q.v, q.v, cst, bc, cst, bc, 0);
}

// from state cur (of two) to state 0; xw: the step's update wrote x (checked
// against each column)
void launch_bfin_inner(hipStream_t s, int64_t n1, int B, const double* part, int32_t* cst,
                       BCol* bc, int cur, int xw) {
  const int64_t ng = tile_groups(n1), nk = ng * B;
  finalize<BFIN_INNER>(s, ng, B, part, part + nk, part + (2 + cur) * nk,
                       cst + cur * B, bc + cur * B, cst, bc, xw);
}

}  // namespace sgeo
