// sgeo_pcg.hip -- EBE matrix-vector product, assembly and the Jacobi-PCG
// vector kernels (src/solver.f90:14-79) for gfx950.
//
// Reductions are two-phase: every block of a vector kernel writes its
// partial sums/maxima to a scratch array, and they are combined in a fixed
// order after a kernel boundary: in the tree-ordered iteration by every block
// of the kernel that needs the result (above PCG_DIRECT partials by
// k_pcg_collapse before it), at a solve's start and in the reference-order mode
// by a one-block finalize kernel.  The kernel boundary provides the
// visibility; no device-scope fences or atomics are issued per block (on a
// multi-XCD MI355X a device-scope release writes back the L2, which made a
// last-block-done pattern cost an order of magnitude more than the streaming
// itself).  The order is fixed, so results are deterministic run to run.
//
// Contraction is off: element products and vector updates round each
// operation as the reference does.
#pragma clang fp contract(off)

#include <algorithm>

#include "sgeo_device.h"
#include "sgeo_internal.h"

namespace sgeo {

static inline unsigned nblk(int64_t n, int per) {
  return (unsigned)((n + per - 1) / per);
}

static inline unsigned grid_stride_blocks(int64_t n) {
  const int64_t b = (n + SGEO_VEC_THREADS - 1) / SGEO_VEC_THREADS;
  return (unsigned)(b < 65536 ? (b > 0 ? b : 1) : 65536);
}

// the block's sum of v (NW waves) into its partial
template <int NW>
__device__ __forceinline__ void put_share(double v, double* __restrict__ part, int blk) {
  __shared__ double red[NW];
  v = block_sum<NW>(v, red);
  if (threadIdx.x == 0) part[blk] = v;
}

// --------------------------------------------------------------------------
// EBE product, element part: Y[e] = K_e p_e
// --------------------------------------------------------------------------
// Three elements per 256-thread block: thread t owns row r = t % 81 of
// element 3*blockIdx + t / 81 (threads 243..255 idle).  Column c of the
// three column-major K_e is read by the block as three contiguous 648-byte
// runs, so every wave-wide load is (nearly) full width.  p_e is gathered
// into LDS once; row r sums c = 0..80 in order, as matmul(km, p(egdof))
// (src/solver.f90:57).
// skip_mode: 0 none, 1 return when sc->done, 2 return when !sc->u_nonzero.
// back: the elements from the last to the first.  A solve alternates, so that
// an iteration starts with the matrices that the last one left in the 256 MB
// MALL (30,030 elements, 1.6 GB: solves of 200 iterations 65.8 -> 64.2 ms).
// part (may be NULL): the block's share of p.Kp = sum_e p_e . Y_e.
template <typename KT>
__global__ __launch_bounds__(256) void k_ebe_elem(
    int32_t nelmt, const KT* __restrict__ K, const int32_t* __restrict__ gdof,
    const double* __restrict__ p, double* __restrict__ Y, double* __restrict__ part,
    const PcgScalars* __restrict__ sc, int skip_mode, int back) {
  if (skip_mode == 1 && sc->done) return;
  if (skip_mode == 2 && !sc->u_nonzero) return;
  __shared__ double pe[3][81];
  const int t = threadIdx.x;
  const int el = t / 81, r = t - 81 * el;
  const int blk = back ? gridDim.x - 1 - blockIdx.x : blockIdx.x;
  const int64_t e = (int64_t)blk * 3 + el;
  const bool valid = (t < 243) && (e < nelmt);
  if (valid) pe[el][r] = p[gdof[e * 81 + r]];
  __syncthreads();
  double d = 0.0;
  if (valid) {
    const KT* ke = K + e * 6561 + r;
    const double* pl = pe[el];
    double a = 0.0;
#pragma unroll 27
    for (int c = 0; c < 81; c++) a = a + (double)ke[c * 81] * pl[c];
    Y[e * 81 + r] = a;
    d = a * pl[r];
  }
  if (part) put_share<4>(d, part, blk);
}

// --------------------------------------------------------------------------
// EBE product on symmetric-packed storage (the fast path)
// --------------------------------------------------------------------------
// K_e keeps its upper triangle U(r,c), r <= c, column by column:
// U(r,c) at c(c+1)/2 + r, 3321 entries padded to SGEO_KPACK = 3328 so each
// element starts 16-byte aligned.  A 128-thread block stages an element's
// packed matrix in LDS with 16-byte loads (each stored entry crosses HBM
// once), then thread r < 81 forms y_r = sum_c K(r,c) p_c, c ascending, with
// K(r,c) = U(min(r,c), max(r,c)).  FP32 matrices: k_ebe_packed, a block per
// element; FP64: k_ebe_packed_pipe.
// The reference's K_e is symmetric only to the last bit, so this path
// agrees with the full-storage product to rounding, not bit for bit.

// Row r of the packed matrix u times pe, c ascending.  The place of K(r,c) is
// a choice of two bases plus a constant of c; written with the index formula
// in a loop, its 21 integer operations per entry, not the loads, set the time
// of the product.  Nine entries are read ahead of the nine being added.
// Measured: 9,315 elements 57.8 -> 43.9 us per product, 5.7 TB/s, which is
// what the full-storage product reads at; plastic iterations 145 -> 121 ms.
template <typename KT>
__device__ __forceinline__ double packed_row(const KT* u, const double* pe, int r) {
  int rbase = r * (r + 1) / 2;
  double a = 0.0;
  // ties the places read next to the sum so far: formed ahead, and the entries
  // read ahead, they would take every register
  auto pin = [&]() { asm volatile("" : "+v"(rbase), "+v"(r), "+v"(a)); };
  KT k[2][9];
  double q[2][9];
  auto fetch = [&](int b) {
#pragma unroll
    for (int i = 0; i < 9; i++) {
      const int c = 9 * b + i, col = c * (c + 1) / 2;
      const KT* at = u + (c < r ? rbase + (c - col) : r);
      k[b & 1][i] = at[col];
      q[b & 1][i] = pe[c];
    }
  };
  fetch(0);
#pragma unroll
  for (int b = 0; b < 9; b++) {
    pin();
    if (b < 8) fetch(b + 1);
#pragma unroll
    for (int i = 0; i < 9; i++) a = a + (double)k[b & 1][i] * q[b & 1][i];
  }
  return a;
}

__global__ __launch_bounds__(128) void k_ebe_packed(
    int32_t nelmt, const float* __restrict__ KP, const int32_t* __restrict__ gdof,
    const double* __restrict__ p, double* __restrict__ Y, double* __restrict__ part,
    const PcgScalars* __restrict__ sc, int skip_mode) {
  if (skip_mode == 1 && sc->done) return;
  if (skip_mode == 2 && !sc->u_nonzero) return;
  typedef float v4f __attribute__((ext_vector_type(4)));
  constexpr int NV = SGEO_KPACK / 4;
  __shared__ __align__(16) float u[SGEO_KPACK];
  __shared__ double pe[81];
  const int64_t e = blockIdx.x;
  const int t = threadIdx.x;
  const v4f* src = reinterpret_cast<const v4f*>(KP + e * SGEO_KPACK);
  v4f* dst = reinterpret_cast<v4f*>(u);
#pragma unroll 4
  for (int q = t; q < NV; q += 128) dst[q] = __builtin_nontemporal_load(src + q);
  if (t < 81) pe[t] = p[gdof[e * 81 + t]];
  __syncthreads();
  double d = 0.0;
  if (t < 81) {
    const int r = t;
    const double a = packed_row(u, pe, r);
    Y[e * 81 + r] = a;
    d = a * pe[r];
  }
  if (part) put_share<2>(d, part, blockIdx.x);
}

// FP64, persistent and pipelined: a few 128-thread
// blocks per CU walk the elements.  While element e is multiplied from LDS,
// the next element's packed K is in flight into registers (16-byte loads) and
// its gathered p into a register, with gdof read
// one element further ahead; both reach LDS after the product, behind the
// block's barrier.  Row r sums c ascending.
__global__ __launch_bounds__(128) void k_ebe_packed_pipe(
    int32_t nelmt, const double* __restrict__ KP, const int32_t* __restrict__ gdof,
    const double* __restrict__ p, double* __restrict__ Y, double* __restrict__ part,
    const PcgScalars* __restrict__ sc, int skip_mode, int back) {
  if (skip_mode == 1 && sc->done) return;
  if (skip_mode == 2 && !sc->u_nonzero) return;
  typedef double v2d __attribute__((ext_vector_type(2)));
  constexpr int NV = SGEO_KPACK / 2;        // 16-byte pieces per element
  constexpr int PT = (NV + 127) / 128;      // per thread
  __shared__ __align__(16) double u[SGEO_KPACK];
  __shared__ double pe[2][81];
  const int t = threadIdx.x;
  // this block's elements, blockIdx.x and every gridDim.x-th after it, from
  // the last to the first when `back`
  int64_t stride = gridDim.x, e = blockIdx.x;
  if (back) {
    e = e < nelmt ? e + (nelmt - 1 - e) / stride * stride : -1;
    stride = -stride;
  }
  auto in = [&](int64_t q) { return q >= 0 && q < nelmt; };
  v2d kr[PT];
  int32_t gn = 0;  // gdof of the next element
  if (in(e)) {
    const v2d* src = reinterpret_cast<const v2d*>(KP + e * SGEO_KPACK);
#pragma unroll
    for (int i = 0; i < PT; i++) {
      const int q = t + 128 * i;
      if (q < NV) kr[i] = src[q];
    }
    if (t < 81) pe[0][t] = p[gdof[e * 81 + t]];
    if (t < 81 && in(e + stride)) gn = gdof[(e + stride) * 81 + t];
  }
  const int r = t;
  int cur = 0;
  double share = 0.0;
  for (; in(e); e += stride) {
    v2d* dst = reinterpret_cast<v2d*>(u);
#pragma unroll
    for (int i = 0; i < PT; i++) {
      const int q = t + 128 * i;
      if (q < NV) dst[q] = kr[i];
    }
    __syncthreads();  // K of e and pe[cur] visible
    const int64_t en = e + stride;
    double pn = 0.0;
    if (in(en)) {  // in flight during the product
      const v2d* src = reinterpret_cast<const v2d*>(KP + en * SGEO_KPACK);
#pragma unroll
      for (int i = 0; i < PT; i++) {
        const int q = t + 128 * i;
        if (q < NV) kr[i] = src[q];
      }
      if (t < 81) pn = p[gn];
    }
    int32_t gnn = 0;
    if (t < 81 && in(en + stride)) gnn = gdof[(en + stride) * 81 + t];
    if (t < 81) {
      const double* pl = pe[cur];
      const double a = packed_row(u, pl, r);
      Y[e * 81 + r] = a;
      share = share + a * pl[r];
      pe[cur ^ 1][t] = pn;
    }
    gn = gnn;
    __syncthreads();  // u and pe[cur] free, pe[cur ^ 1] visible
    cur ^= 1;
  }
  if (part) put_share<2>(share, part, blockIdx.x);
}

// blocks per CU of the persistent FP64 product (LDS 28 KB per block)
#define EBE_PIPE_BLOCKS_PER_CU 5

// full (reference layout) -> packed upper triangle, zero padding
template <typename KT>
__global__ void k_pack_upper(int32_t nelmt, const double* __restrict__ K,
                             KT* __restrict__ KP) {
  const int64_t n = (int64_t)nelmt * SGEO_KPACK;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t e = q / SGEO_KPACK;
    const int i = (int)(q - e * SGEO_KPACK);
    KT v = (KT)0;
    if (i < 3321) {
      // column c with c(c+1)/2 <= i < (c+1)(c+2)/2, row r = i - c(c+1)/2
      int c = (int)((sqrt(8.0 * i + 1.0) - 1.0) * 0.5);
      while (c * (c + 1) / 2 > i) c--;
      while ((c + 1) * (c + 2) / 2 <= i) c++;
      const int r = i - c * (c + 1) / 2;
      v = (KT)K[e * 6561 + r + 81 * c];
    }
    KP[q] = v;
  }
}

// plain copy of n doubles (bandwidth calibration)
__global__ __launch_bounds__(256) void k_copy(int64_t n, const double2* __restrict__ a,
                                              double2* __restrict__ b) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n;
       q += (int64_t)gridDim.x * blockDim.x)
    b[q] = a[q];
}

// --------------------------------------------------------------------------
// assembly: out_g = sum over the element slots of g, ascending element order
// (the order of kp(egdof)=kp(egdof)+... in src/solver.f90:54-58)
// --------------------------------------------------------------------------
__device__ __forceinline__ double gather_row(const int32_t* __restrict__ rowptr,
                                             const int32_t* __restrict__ slots,
                                             const double* __restrict__ Y,
                                             int64_t g) {
  double acc = 0.0;
  const int32_t b = rowptr[g], en = rowptr[g + 1];
  for (int32_t s = b; s < en; s++) acc = acc + Y[slots[s]];
  return acc;
}

__global__ __launch_bounds__(SGEO_VEC_THREADS) void k_assemble(
    int64_t n1, const int32_t* __restrict__ rowptr,
    const int32_t* __restrict__ slots, const double* __restrict__ Y,
    double* __restrict__ out, const PcgScalars* __restrict__ sc,
    int skip_mode) {
  if (skip_mode == 2 && !sc->u_nonzero) return;
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n1;
       g += (int64_t)gridDim.x * blockDim.x)
    out[g] = (g == 0) ? 0.0 : gather_row(rowptr, slots, Y, g);
}

// out_g = out_g (+|-) its Y terms in element order; out[0] = 0
// (bodyload(egdof)=bodyload(egdof)+bload, src/slope.F90:382;
//  extload(egdof)=extload(egdof)-eld*gam, src/preprocess.f90:136)
__global__ __launch_bounds__(SGEO_VEC_THREADS) void k_assemble_acc(
    int64_t n1, const int32_t* __restrict__ rowptr,
    const int32_t* __restrict__ slots, const double* __restrict__ Y,
    double* __restrict__ out, int subtract,
    const PlasticScalars* __restrict__ ps) {
  if (ps && ps->nl_isconv) return;  // no body load once converged
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n1;
       g += (int64_t)gridDim.x * blockDim.x) {
    if (g == 0) { out[0] = 0.0; continue; }
    double acc = out[g];
    const int32_t b = rowptr[g], en = rowptr[g + 1];
    if (subtract) {
      for (int32_t s = b; s < en; s++) acc = acc - Y[slots[s]];
    } else {
      for (int32_t s = b; s < en; s++) acc = acc + Y[slots[s]];
    }
    out[g] = acc;
  }
}

// --------------------------------------------------------------------------
// PCG vector kernels: partial sums per block
// --------------------------------------------------------------------------
#define VEC_LOOP(g)                                                         \
  const int64_t base = (int64_t)blockIdx.x * SGEO_VEC_THREADS * SGEO_VEC_ITEMS; \
  _Pragma("unroll") for (int k_ = 0; k_ < SGEO_VEC_ITEMS; k_++)            \
    for (int64_t g = base + threadIdx.x + (int64_t)k_ * SGEO_VEC_THREADS;  \
         g < n1; g = n1)

// max|u| at entry (src/solver.f90:39)
__global__ __launch_bounds__(SGEO_VEC_THREADS) void k_pcg_begin(
    int64_t n1, const double* __restrict__ u, double* __restrict__ part) {
  __shared__ double red[SGEO_VEC_THREADS / 64];
  double m = 0.0;
  VEC_LOOP(g) { m = fmax(m, fabs(u[g])); }
  m = block_max<SGEO_VEC_THREADS / 64>(m, red);
  if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// The kernels of the reference-order mode, whose dot products k_pcg_seqdot
// forms.
// r = f - kp (kp = K u if u != 0, else 0); z = dinv*r; p = z
__global__ __launch_bounds__(SGEO_VEC_THREADS) void k_pcg_init(
    int64_t n1, const double* __restrict__ f, const double* __restrict__ kp,
    const double* __restrict__ dinv, double* __restrict__ r,
    double* __restrict__ z, double* __restrict__ p, const PcgScalars* __restrict__ sc) {
  const bool unz = sc->u_nonzero != 0;
  VEC_LOOP(g) {
    const double rg = f[g] - (unz ? kp[g] : 0.0);
    const double zg = dinv[g] * rg;
    r[g] = rg;
    z[g] = zg;
    p[g] = zg;
  }
}

// kp = assemble(Y); partial max|p|
__global__ __launch_bounds__(SGEO_VEC_THREADS) void k_pcg_assemble_max(
    int64_t n1, const int32_t* __restrict__ rowptr,
    const int32_t* __restrict__ slots, const double* __restrict__ Y,
    const double* __restrict__ p, double* __restrict__ kp,
    double* __restrict__ part, const PcgScalars* __restrict__ sc) {
  if (sc->done) return;
  __shared__ double red[SGEO_VEC_THREADS / 64];
  double m = 0.0;
  VEC_LOOP(g) {
    kp[g] = (g == 0) ? 0.0 : gather_row(rowptr, slots, Y, g);
    m = fmax(m, fabs(p[g]));
  }
  const double bm = block_max<SGEO_VEC_THREADS / 64>(m, red);
  if (threadIdx.x == 0) part[blockIdx.x] = bm;
}

// u += alpha p; partial max|u|; r -= alpha kp; z = dinv r
__global__ __launch_bounds__(SGEO_VEC_THREADS) void k_pcg_update(
    int64_t n1, const double* __restrict__ p, const double* __restrict__ kp,
    const double* __restrict__ dinv, double* __restrict__ u,
    double* __restrict__ r, double* __restrict__ z, double* __restrict__ part,
    const PcgScalars* __restrict__ sc) {
  if (sc->done) return;
  __shared__ double red[SGEO_VEC_THREADS / 64];
  const double alpha = sc->alpha;
  double m = 0.0;
  VEC_LOOP(g) {
    const double ug = u[g] + alpha * p[g];
    u[g] = ug;
    m = fmax(m, fabs(ug));
    const double rg = r[g] - alpha * kp[g];
    r[g] = rg;
    z[g] = dinv[g] * rg;
  }
  const double bm = block_max<SGEO_VEC_THREADS / 64>(m, red);
  if (threadIdx.x == 0) part[blockIdx.x] = bm;
}

// p = z + beta p
__global__ __launch_bounds__(SGEO_VEC_THREADS) void k_pcg_pupdate(
    int64_t n1, const double* __restrict__ z, double* __restrict__ p,
    const PcgScalars* __restrict__ sc) {
  if (sc->done) return;
  const double beta = sc->beta;
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n1;
       g += (int64_t)gridDim.x * blockDim.x)
    p[g] = z[g] + beta * p[g];
}

// --------------------------------------------------------------------------
// finalize: one block combines the nb partials in index order
// --------------------------------------------------------------------------
enum FinWhat {
  FIN_BEGIN = 0,   // max|u|  -> u_nonzero, reset
  FIN_RZ = 1,      // r.z     -> rz
  FIN_MAXP = 2,    // max|p|  (reference-order mode)
  FIN_UPDATE = 3,  // max|u|  -> stop test (reference-order mode)
};

__global__ __launch_bounds__(256) void k_pcg_finalize(
    int nb, const double* __restrict__ part, PcgScalars* __restrict__ sc,
    int what, double tol, int32_t maxiter) {
  __shared__ double red[4];
  if (what >= FIN_MAXP && sc->done) return;
  double v = 0.0;
#pragma unroll 4
  for (int b = threadIdx.x; b < nb; b += 256)
    v = what == FIN_RZ ? v + part[b] : fmax(v, part[b]);
  v = what == FIN_RZ ? block_sum<4>(v, red) : block_max<4>(v, red);
  if (threadIdx.x != 0) return;
  switch (what) {
    case FIN_BEGIN:
      sc->u_nonzero = v > 0.0 ? 1 : 0;
      sc->iter = 0;
      sc->done = 0;
      sc->conv_iter = 0;
      sc->tol = tol;
      sc->maxiter = maxiter;
      break;
    case FIN_RZ:
      sc->rz = v;
      break;
    case FIN_MAXP:
      sc->maxp = v;
      break;
    case FIN_UPDATE: {
      const int it = sc->iter + 1;
      sc->iter = it;
      sc->maxu = v;
      // src/solver.f90:65: stop after the u update, before the r update
      if (fabs(sc->alpha) * sc->maxp / v <= sc->tol) {
        sc->done = 1;
        sc->conv_iter = it;
      } else if (it >= sc->maxiter) {
        sc->done = 2;
        sc->conv_iter = sc->maxiter + 1;  // DO-loop variable after exhaustion
      }
      break;
    }
  }
}

// --------------------------------------------------------------------------
// The iteration with tree-ordered reductions.  Linear solves run three
// kernels:
//   the element product, with its blocks' shares of p.Kp (p.Kp = sum_e
//     p_e . Y_e, so alpha needs no assembled vector),
//   k_pcg_step<true>: kp summed on the fly, u += alpha p, r -= alpha kp,
//     partials of max|u| and r.z (z = dinv r is formed, not stored),
//   k_pcg_dir: the stop test, p = z + beta p, partials of max|p|.
// A trial's solves multiply the stored matrices and form p.Kp from the
// assembled vector (k_pcg_asm, then k_pcg_step<false>): their x enters the
// yield function, which at the corners of the Mohr-Coulomb pyramid turns the
// last bits of x into relative changes of 1e-7 (asin near 1), so they keep the
// summation order they have always had.  That keeps a trial's bits; whether
// the other order is any less accurate has not been measured.
// Every block combines the partials that the kernel before it left, all in
// the same order, so that no one-block kernel stands between them; above
// PCG_DIRECT partials k_pcg_collapse does it once, in that order, since each
// block reading thousands would cost more than the extra launch.  The
// scalars are double-buffered: the kernels of iteration `it` read
// sc[it & 1] while k_pcg_dir's first block writes sc[(it + 1) & 1].
// A block holds one equation per thread: the three dependent loads of a
// gathered row set the time of small systems.  Blocks of 1,024 keep a
// trial's partials (four values per lane, 256 equations apart, then the
// lanes) and their number low; linear solves of up to 2^18 equations take
// blocks of 256, four times as many compute units at work.
// Measured, us per iteration without the product: 28,969 equations 29
// before (five kernels, four rows per thread one after another), 12.7 with
// blocks of 1,024, 10.6 with 256, 9.5 with the partials of all kinds in
// flight together; 3,489,480 equations 141 before, 112 now.
// --------------------------------------------------------------------------
#define PCG_DIRECT 1024
#define PCG_BLOCK 1024
static_assert(PCG_BLOCK == SGEO_VEC_THREADS * SGEO_VEC_ITEMS, "partials of 1,024 equations");

// v[k] = sum (bit k of MAXES: max) of in[k][0..n) over the block in
// k_pcg_finalize's order, in every thread.  The kinds' values are in flight
// together: one after another each cost the latency of values that other XCDs
// wrote, and two barriers.
template <int NK, int MAXES>
__device__ __forceinline__ void combine(const double* const (&in)[NK], int n, double (&v)[NK]) {
  if (n == 1) {
#pragma unroll
    for (int k = 0; k < NK; k++) v[k] = in[k][0];
    return;
  }
  __shared__ double red[NK][4];
  const int t = threadIdx.x;
  auto op = [](int k, double a, double b) { return (MAXES >> k) & 1 ? fmax(a, b) : a + b; };
  if (t < 256) {
    double a[NK];
#pragma unroll
    for (int k = 0; k < NK; k++) a[k] = 0.0;
    for (int b0 = t; b0 < n; b0 += 4 * 256) {
      double y[NK][4];
#pragma unroll
      for (int k = 0; k < NK; k++)
#pragma unroll
        for (int i = 0; i < 4; i++)  // past the end: the last value, not used
          y[k][i] = in[k][min(b0 + 256 * i, n - 1)];
#pragma unroll
      for (int k = 0; k < NK; k++)
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (b0 + 256 * i < n) a[k] = op(k, a[k], y[k][i]);
    }
#pragma unroll
    for (int k = 0; k < NK; k++) {
      a[k] = (MAXES >> k) & 1 ? wave_max(a[k]) : wave_sum(a[k]);
      if ((t & 63) == 0) red[k][t >> 6] = a[k];
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NK; k++) {
    v[k] = 0.0;
#pragma unroll
    for (int i = 0; i < 4; i++) v[k] = op(k, v[k], red[k][i]);
  }
}

// partials in[k][0..n) -> out[k]: max|u|, r.z and max|p|, or p.Kp alone (the
// others NULL).  One block.
struct Kinds {
  const double* in[3];
};
__global__ __launch_bounds__(256) void k_pcg_collapse(int n, Kinds kinds,
                                                      double* __restrict__ out,
                                                      const PcgScalars* __restrict__ sc) {
  if (sc->done) return;
  if (!kinds.in[1]) {  // p.Kp alone
    double v[1];
    combine<1, 0>({kinds.in[0]}, n, v);
    if (threadIdx.x == 0) out[0] = v[0];
    return;
  }
  double v[3];
  combine<3, 5>({kinds.in[0], kinds.in[1], kinds.in[2]}, n, v);
  if (threadIdx.x < 3) out[threadIdx.x] = v[threadIdx.x];
}

// the block's partials of NK kinds (bit k of MAXES: a max) from its threads'
// values
template <int BS, int NK, int MAXES>
__device__ __forceinline__ void block_partials(const double (&v)[NK],
                                               double* const (&part)[NK]) {
  __shared__ double lds[NK][BS > 256 ? BS : 1], red[NK][4];
  const int t = threadIdx.x;
  auto op = [](int k, double a, double b) { return (MAXES >> k) & 1 ? fmax(a, b) : a + b; };
  if (BS > 256) {
#pragma unroll
    for (int k = 0; k < NK; k++) lds[k][t] = v[k];
    __syncthreads();
  }
  if (t < 256) {
#pragma unroll
    for (int k = 0; k < NK; k++) {
      double a = BS > 256 ? 0.0 : v[k];
#pragma unroll
      for (int i = 0; i < BS / 256 && BS > 256; i++) a = op(k, a, lds[k][t + 256 * i]);
      a = (MAXES >> k) & 1 ? wave_max(a) : wave_sum(a);
      if ((t & 63) == 0) red[k][t >> 6] = a;
    }
  }
  __syncthreads();
  if (t < NK) {
#pragma unroll
    for (int k = 0; k < NK; k++) {
      if (t != k) continue;
      double s = 0.0;
#pragma unroll
      for (int i = 0; i < 4; i++) s = op(k, s, red[k][i]);
      part[k][blockIdx.x] = s;
    }
  }
}

// r = f - kp (kp = K u if u != 0, else 0); p = z = dinv r; r.z and max|p|
template <int BS>
__global__ __launch_bounds__(BS) void k_pcg_start(
    int64_t n1, const double* __restrict__ f, const double* __restrict__ kp,
    const double* __restrict__ dinv, double* __restrict__ r, double* __restrict__ p,
    double* __restrict__ part_rz, double* __restrict__ part_p,
    const PcgScalars* __restrict__ sc) {
  const int64_t g = (int64_t)blockIdx.x * BS + threadIdx.x;
  double s = 0.0, m = 0.0;
  if (g < n1) {
    const double rg = f[g] - (sc->u_nonzero ? kp[g] : 0.0);
    const double zg = dinv[g] * rg;
    r[g] = rg;
    p[g] = zg;
    s = rg * zg;
    m = fabs(zg);
  }
  block_partials<BS, 2, 2>({s, m}, {part_rz, part_p});
}

// The row's element contributions (at most 8 on hexahedral meshes), then
// summed in slot order.  All eight are loaded, past the row's end its last one
// again: conditional loads compile to a branch each, and every slot's latency
// stood before the next one's (solves of 1,152 elements 10.5 -> 9.7 ms, 4,921
// packed 15.0 -> 14.0, 144,000 packed 30.3 -> 29.0).
__device__ __forceinline__ double gather_row8(const int32_t* __restrict__ rowptr,
                                              const int32_t* __restrict__ slots,
                                              const double* __restrict__ Y, int64_t g) {
  const int32_t q0 = rowptr[g], q1 = rowptr[g + 1];
  int32_t at[8];
  double v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) at[i] = slots[max(min(q0 + i, q1 - 1), 0)];
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = Y[q1 > q0 ? at[i] : 0];
  double kp = 0.0;
#pragma unroll
  for (int i = 0; i < 8; i++) kp = q0 + i < q1 ? kp + v[i] : kp;
  for (int32_t q = q0 + 8; q < q1; q++) kp = kp + Y[slots[q]];
  return kp;
}

// kp and the partial of p.kp
template <int BS>
__global__ __launch_bounds__(BS) void k_pcg_asm(
    int64_t n1, const int32_t* __restrict__ rowptr, const int32_t* __restrict__ slots,
    const double* __restrict__ Y, const double* __restrict__ p, double* __restrict__ kp,
    double* __restrict__ part, const PcgScalars* __restrict__ sc) {
  if (sc->done) return;
  const int64_t g = (int64_t)blockIdx.x * BS + threadIdx.x;
  double s = 0.0;
  if (g < n1) {
    const double v = g == 0 ? 0.0 : gather_row8(rowptr, slots, Y, g);
    kp[g] = v;
    s = p[g] * v;
  }
  block_partials<BS, 1, 0>({s}, {part});
}

// n_dot partials of p.Kp in `dot`; FUSED: kp is summed from Y here
template <int BS, bool FUSED>
__global__ __launch_bounds__(BS) void k_pcg_step(
    int64_t n1, const int32_t* __restrict__ rowptr, const int32_t* __restrict__ slots,
    const double* __restrict__ Y, const double* __restrict__ kp,
    const double* __restrict__ p, const double* __restrict__ dinv, double* __restrict__ u,
    double* __restrict__ r, const double* __restrict__ dot, int n_dot,
    double* __restrict__ part_u, double* __restrict__ part_rz, PcgScalars* __restrict__ sc) {
  if (sc->done) return;
  const int64_t g = (int64_t)blockIdx.x * BS + threadIdx.x;
  const bool in = g < n1;
  const double rz = sc->rz;
  double v = 0.0, ug = 0.0, pg = 0.0, rg = 0.0, dg = 0.0;
  if (in) {  // in flight while the partials are combined
    ug = u[g];
    pg = p[g];
    rg = r[g];
    dg = dinv[g];
    if (!FUSED) v = kp[g];
    else if (g > 0) v = gather_row8(rowptr, slots, Y, g);
  }
  double c[1];
  combine<1, 0>({dot}, n_dot, c);
  const double pkp = c[0];
  const double alpha = rz / pkp;
  double m = 0.0, s = 0.0;
  if (in) {
    ug = ug + alpha * pg;
    u[g] = ug;
    m = fabs(ug);
    rg = rg - alpha * v;
    r[g] = rg;
    s = rg * (dg * rg);
  }
  block_partials<BS, 2, 1>({m, s}, {part_u, part_rz});
  if (blockIdx.x == 0 && threadIdx.x == 0) {  // read by later kernels only
    sc->pkp = pkp;
    sc->alpha = alpha;
  }
}

// n_part partials of max|u|, r.z and this iteration's max|p|
template <int BS>
__global__ __launch_bounds__(BS) void k_pcg_dir(
    int64_t n1, const double* __restrict__ r, const double* __restrict__ dinv,
    double* __restrict__ p, const double* __restrict__ part_u,
    const double* __restrict__ part_rz, const double* __restrict__ part_p, int n_part,
    double* __restrict__ part_pn, const PcgScalars* __restrict__ sc,
    PcgScalars* __restrict__ scn) {
  const bool writer = blockIdx.x == 0 && threadIdx.x == 0;
  if (sc->done) {
    if (writer) *scn = *sc;
    return;
  }
  const int64_t g = (int64_t)blockIdx.x * BS + threadIdx.x;
  const bool in = g < n1;
  double rg = 0.0, dg = 0.0, pg = 0.0;
  if (in) {
    rg = r[g];
    dg = dinv[g];
    pg = p[g];
  }
  PcgScalars n = *sc;
  double c[3];
  combine<3, 5>({part_u, part_rz, part_p}, n_part, c);
  const double maxu = c[0], rz = c[1], maxp = c[2];
  const int it = n.iter + 1;
  // src/solver.f90:65: the relative update of u
  const bool conv = fabs(n.alpha) * maxp / maxu <= n.tol;
  const bool fail = !conv && it >= n.maxiter;
  const double beta = rz / n.rz;
  if (writer) {
    n.iter = it;
    n.maxu = maxu;
    n.maxp = maxp;
    if (conv) {
      n.done = 1;
      n.conv_iter = it;
    } else if (fail) {
      n.done = 2;
      n.conv_iter = n.maxiter + 1;  // DO-loop variable after exhaustion
    } else {
      n.beta = beta;
      n.rz = rz;
    }
    *scn = n;
  }
  if (conv || fail) return;
  double m = 0.0;
  if (in) {
    pg = dg * rg + beta * pg;
    p[g] = pg;
    m = fabs(pg);
  }
  block_partials<BS, 1, 1>({m}, {part_pn});
}

// --------------------------------------------------------------------------
// reference-order dot products: s = ((0 + a0 b0) + a1 b1) + ..., exactly the
// sequential dot_product of src/solver.f90:61-62,72.  One block: waves 1-3
// stage rounded products of the next chunk in LDS while lane 0 of wave 0
// adds the current chunk in index order.  O(n) latency-bound; meant for
// bit-for-bit parity runs, the tree reductions above are the fast path.
// --------------------------------------------------------------------------
#define SEQ_CHUNK 1536
__device__ double seq_dot(int64_t n1, const double* __restrict__ a,
                          const double* __restrict__ b, double* buf) {
  const int t = threadIdx.x;
  const int64_t nch = (n1 + SEQ_CHUNK - 1) / SEQ_CHUNK;
  double s = 0.0;
  for (int j = t; j < SEQ_CHUNK; j += blockDim.x)
    buf[j] = (j < n1) ? a[j] * b[j] : 0.0;
  __syncthreads();
  for (int64_t c = 0; c < nch; c++) {
    const double* cur = buf + (c & 1) * SEQ_CHUNK;
    if (t < 64) {
      if (t == 0) {
        const int64_t cnt = (c == nch - 1) ? n1 - c * SEQ_CHUNK : SEQ_CHUNK;
        for (int64_t j = 0; j < cnt; j++) s = s + cur[j];
      }
    } else if (c + 1 < nch) {
      double* nxt = buf + ((c + 1) & 1) * SEQ_CHUNK;
      const int64_t base = (c + 1) * SEQ_CHUNK;
      for (int j = t - 64; j < SEQ_CHUNK; j += blockDim.x - 64) {
        const int64_t g = base + j;
        nxt[j] = (g < n1) ? a[g] * b[g] : 0.0;
      }
    }
    __syncthreads();
  }
  return s;  // valid in thread 0
}

// which: 0 initial rz; 1 alpha = rz / p.kp; 2 beta from r.z
__global__ __launch_bounds__(256) void k_pcg_seqdot(
    int64_t n1, const double* __restrict__ a, const double* __restrict__ b,
    PcgScalars* __restrict__ sc, int which) {
  __shared__ double buf[2 * SEQ_CHUNK];
  if (which != 0 && sc->done) return;
  const double s = seq_dot(n1, a, b, buf);
  if (threadIdx.x == 0) {
    if (which == 0) {
      sc->rz = s;
    } else if (which == 1) {
      sc->pkp = s;
      sc->alpha = sc->rz / s;
    } else {
      sc->beta = s / sc->rz;
      sc->rz = s;
    }
  }
}

// --------------------------------------------------------------------------
// plastic-iteration vector kernels (src/slope.F90:288-309)
// --------------------------------------------------------------------------
// load = extload + bodyload; load(0) = 0
__global__ void k_load(int64_t n1, const double* __restrict__ ext,
                       const double* __restrict__ body, double* __restrict__ load) {
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n1;
       g += (int64_t)gridDim.x * blockDim.x)
    load[g] = (g == 0) ? 0.0 : ext[g] + body[g];
}

// x(0)=0; partial max|x-oldx| and max|x|; oldx = x
__global__ __launch_bounds__(SGEO_VEC_THREADS) void k_uerr(
    int64_t n1, double* __restrict__ x, double* __restrict__ oldx,
    double* __restrict__ part) {
  __shared__ double red[SGEO_VEC_THREADS / 64];
  double md = 0.0, mx = 0.0;
  VEC_LOOP(g) {
    double xg = x[g];
    if (g == 0) { xg = 0.0; x[0] = 0.0; }
    md = fmax(md, fabs(xg - oldx[g]));
    mx = fmax(mx, fabs(xg));
    oldx[g] = xg;
  }
  const double bd = block_max<SGEO_VEC_THREADS / 64>(md, red);
  const double bx = block_max<SGEO_VEC_THREADS / 64>(mx, red);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = bd;
    part[gridDim.x + blockIdx.x] = bx;
  }
}

// uerr = max|x-oldx| / max|x|; nl_isconv = uerr <= nl_tol; fmax = 0
__global__ __launch_bounds__(256) void k_uerr_finalize(
    int nb, const double* __restrict__ part, PlasticScalars* __restrict__ ps,
    double nl_tol) {
  __shared__ double red[4];
  double vd = 0.0, vx = 0.0;
  for (int b = threadIdx.x; b < nb; b += 256) {
    vd = fmax(vd, part[b]);
    vx = fmax(vx, part[nb + b]);
  }
  vd = block_max<4>(vd, red);
  vx = block_max<4>(vx, red);
  if (threadIdx.x == 0) {
    const double uerr = vd / vx;
    ps->uerr = uerr;
    ps->xmax = vx;
    ps->nl_isconv = uerr <= nl_tol ? 1 : 0;
    ps->fmax_bits = 0ull;  // fmax = zero (src/slope.F90:286)
    ps->n_plastic = 0;
  }
}

// --------------------------------------------------------------------------
// inverse map (equation -> element slots) built on the device: the same
// CSR a stable counting sort on the host builds (slots of every equation
// g >= 1 in ascending e*81+i order; the index-0 sink stays empty, no assembly
// reads it).  Every kernel checks the equation range itself.
// --------------------------------------------------------------------------
__global__ void k_fill_i32(int64_t n, int32_t* __restrict__ a, int32_t v) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n;
       q += (int64_t)gridDim.x * blockDim.x)
    a[q] = v;
}

// cnt[g + 1] = slots of equation g (1 <= g <= neq); *bad = 1 if an entry
// lies outside 0..neq (such entries are skipped)
__global__ void k_csr_count(int64_t ns, int32_t neq, const int32_t* __restrict__ gdof,
                            int32_t* __restrict__ cnt, int32_t* __restrict__ bad) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < ns;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int32_t g = gdof[q];
    if (g < 0 || g > neq) {
      *bad = 1;
      continue;
    }
    if (g > 0) atomicAdd(&cnt[g + 1], 1);
  }
}

// *longest (zero before) = the largest count of cnt[g + 1], 1 <= g < n1
__global__ __launch_bounds__(SGEO_VEC_THREADS) void k_csr_longest(
    int64_t n1, const int32_t* __restrict__ cnt, int32_t* __restrict__ longest) {
  int32_t m = 0;
  for (int64_t g = 1 + blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n1;
       g += (int64_t)gridDim.x * blockDim.x)
    m = max(m, cnt[g + 1]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off, 64));
  if ((threadIdx.x & 63) == 0) atomicMax(longest, m);
}

// In-place inclusive scan: each block of 1024 threads scans its SCAN_SEG
// entries (four per thread) and leaves their total; the totals are scanned by
// one block (total NULL: rounds of SCAN_SEG, the running sum carried) and
// k_scan_add adds them to the segments after them.  One block over 1.6 M
// entries had taken 0.92 ms, a latency-bound round after another; the three
// launches take 19 us.
#define SCAN_SEG 4096
__global__ __launch_bounds__(1024) void k_scan_i32(int64_t n, int32_t* __restrict__ a,
                                                   int32_t* __restrict__ total) {
  __shared__ int32_t wsum[16];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  int32_t carry = 0;
  const int64_t first = (int64_t)blockIdx.x * SCAN_SEG;
  const int64_t last = total ? min(n, first + SCAN_SEG) : n;
  for (int64_t base = first; base < last; base += SCAN_SEG) {
    const int64_t i0 = base + (int64_t)t * 4;
    int32_t v[4], s = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      s += (i0 + k < n) ? a[i0 + k] : 0;
      v[k] = s;
    }
    int32_t x = s;  // inclusive scan of the thread totals across the wave
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int32_t y = __shfl_up(x, off, 64);
      if (lane >= off) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    if (w == 0) {
      int32_t ws = lane < 16 ? wsum[lane] : 0;
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) {
        const int32_t y = __shfl_up(ws, off, 64);
        if (lane >= off) ws += y;
      }
      if (lane < 16) wsum[lane] = ws;
    }
    __syncthreads();
    const int32_t excl = carry + (x - s) + (w > 0 ? wsum[w - 1] : 0);
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (i0 + k < n) a[i0 + k] = v[k] + excl;
    carry += wsum[15];
    __syncthreads();  // wsum is rewritten by the next round
  }
  if (total && t == 0) total[blockIdx.x] = carry;
}

__global__ __launch_bounds__(SGEO_VEC_THREADS) void k_scan_add(
    int64_t n, int32_t* __restrict__ a, const int32_t* __restrict__ total) {
  const int64_t i = SCAN_SEG + blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) a[i] += total[i / SCAN_SEG - 1];
}

// cursor[g] = rowptr[g]; slots[cursor[g]++] = q for every entry of g >= 1
__global__ void k_csr_fill(int64_t ns, int32_t neq, const int32_t* __restrict__ gdof,
                           int32_t* __restrict__ cursor, int32_t* __restrict__ slots) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < ns;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int32_t g = gdof[q];
    if (g < 1 || g > neq) continue;
    slots[atomicAdd(&cursor[g], 1)] = (int32_t)q;
  }
}

// each equation's slots in ascending order (the fill's atomics leave them
// in arrival order); rows hold at most a node's element count
__global__ void k_csr_sort(int64_t n1, const int32_t* __restrict__ rowptr,
                           int32_t* __restrict__ slots) {
  for (int64_t g = 1 + blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n1;
       g += (int64_t)gridDim.x * blockDim.x) {
    const int32_t b = rowptr[g], e = rowptr[g + 1];
    for (int32_t i = b + 1; i < e; i++) {
      const int32_t v = slots[i];
      int32_t j = i - 1;
      while (j >= b && slots[j] > v) {
        slots[j + 1] = slots[j];
        j--;
      }
      slots[j + 1] = v;
    }
  }
}

__global__ void k_copy_i32(int64_t n, const int32_t* __restrict__ a, int32_t* __restrict__ b) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n;
       q += (int64_t)gridDim.x * blockDim.x)
    b[q] = a[q];
}

// *a = v, queued on the stream (a kernel, not a memset node)
void launch_set_i32(hipStream_t s, int32_t* a, int32_t v) {
  hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, s, (int64_t)1, a, v);
}

// The two halves of the map in caller memory.  count: rowptr (n1 + 1 entries)
// of gdof (ns entries); flags[0] (zeroed here) reports entries outside 0..neq,
// flags[1] the longest row.  fill: slots.  tmp and cursor (n1 entries each) are
// temporaries.
// A row is sorted by one thread inserting its entries one after another: for
// rows as short as a mesh's.
void launch_csr_count(hipStream_t s, int64_t ns, int32_t neq, const int32_t* gdof,
                      int32_t* rowptr, int32_t* tmp, int32_t* flags) {
  const int64_t n1 = (int64_t)neq + 1;
  hipLaunchKernelGGL(k_fill_i32, dim3(grid_stride_blocks(n1 + 1)), dim3(SGEO_VEC_THREADS),
                     0, s, n1 + 1, rowptr, 0);
  hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, s, (int64_t)2, flags, 0);
  hipLaunchKernelGGL(k_csr_count, dim3(grid_stride_blocks(ns)), dim3(SGEO_VEC_THREADS), 0,
                     s, ns, neq, gdof, rowptr, flags);
  hipLaunchKernelGGL(k_csr_longest, dim3(std::min(256u, grid_stride_blocks(n1))),
                     dim3(SGEO_VEC_THREADS), 0, s, n1, rowptr, flags + 1);
  const int64_t ne = n1 + 1, nseg = (ne + SCAN_SEG - 1) / SCAN_SEG;  // nseg <= n1
  hipLaunchKernelGGL(k_scan_i32, dim3((unsigned)nseg), dim3(1024), 0, s, ne, rowptr, tmp);
  if (nseg > 1) {
    hipLaunchKernelGGL(k_scan_i32, dim3(1), dim3(1024), 0, s, nseg, tmp, (int32_t*)nullptr);
    hipLaunchKernelGGL(k_scan_add, dim3(nblk(ne - SCAN_SEG, SGEO_VEC_THREADS)),
                       dim3(SGEO_VEC_THREADS), 0, s, ne, rowptr, tmp);
  }
}

void launch_csr_fill(hipStream_t s, int64_t ns, int32_t neq, const int32_t* gdof,
                     const int32_t* rowptr, int32_t* slots, int32_t* cursor) {
  const int64_t n1 = (int64_t)neq + 1;
  hipLaunchKernelGGL(k_copy_i32, dim3(grid_stride_blocks(n1)), dim3(SGEO_VEC_THREADS), 0,
                     s, n1, rowptr, cursor);
  hipLaunchKernelGGL(k_csr_fill, dim3(grid_stride_blocks(ns)), dim3(SGEO_VEC_THREADS), 0,
                     s, ns, neq, gdof, cursor, slots);
  hipLaunchKernelGGL(k_csr_sort, dim3(grid_stride_blocks(n1)), dim3(SGEO_VEC_THREADS), 0,
                     s, n1, rowptr, slots);
}

// --------------------------------------------------------------------------
// launch wrappers
// --------------------------------------------------------------------------
void launch_ebe_elem_f64(hipStream_t s, int32_t nelmt, const double* K,
                         const int32_t* gdof, const double* p, double* Y, double* part,
                         const PcgScalars* sc, int skip_mode, int back) {
  if (nelmt <= 0) return;
  hipLaunchKernelGGL(k_ebe_elem<double>, dim3(nblk(nelmt, 3)), dim3(256), 0, s,
                     nelmt, K, gdof, p, Y, part, sc, skip_mode, back);
}

void launch_ebe_elem_f32k(hipStream_t s, int32_t nelmt, const float* K,
                          const int32_t* gdof, const double* p, double* Y, double* part,
                          const PcgScalars* sc, int skip_mode, int back) {
  if (nelmt <= 0) return;
  hipLaunchKernelGGL(k_ebe_elem<float>, dim3(nblk(nelmt, 3)), dim3(256), 0, s,
                     nelmt, K, gdof, p, Y, part, sc, skip_mode, back);
}

void launch_ebe_packed_f64(hipStream_t s, int32_t nelmt, int n_cu, const double* KP,
                           const int32_t* gdof, const double* p, double* Y, double* part,
                           const PcgScalars* sc, int skip_mode, int back) {
  if (nelmt <= 0) return;
  hipLaunchKernelGGL(k_ebe_packed_pipe, dim3((unsigned)ebe_packed_blocks(nelmt, n_cu)),
                     dim3(128), 0, s, nelmt, KP, gdof, p, Y, part, sc, skip_mode, back);
}

void launch_ebe_packed_f32(hipStream_t s, int32_t nelmt, const float* KP,
                           const int32_t* gdof, const double* p, double* Y, double* part,
                           const PcgScalars* sc, int skip_mode) {
  if (nelmt <= 0) return;
  hipLaunchKernelGGL(k_ebe_packed, dim3(nelmt), dim3(128), 0, s, nelmt,
                     KP, gdof, p, Y, part, sc, skip_mode);
}

int ebe_elem_blocks(int32_t nelmt) { return (int)nblk(nelmt, 3); }
int ebe_packed_blocks(int32_t nelmt, int n_cu) {
  return std::min<int64_t>((int64_t)n_cu * EBE_PIPE_BLOCKS_PER_CU, nelmt);
}

void launch_pack_upper_f64(hipStream_t s, int32_t nelmt, const double* K,
                           double* KP) {
  hipLaunchKernelGGL(k_pack_upper<double>,
                     dim3(grid_stride_blocks((int64_t)nelmt * SGEO_KPACK)),
                     dim3(SGEO_VEC_THREADS), 0, s, nelmt, K, KP);
}

void launch_pack_upper_f32(hipStream_t s, int32_t nelmt, const double* K,
                           float* KP) {
  hipLaunchKernelGGL(k_pack_upper<float>,
                     dim3(grid_stride_blocks((int64_t)nelmt * SGEO_KPACK)),
                     dim3(SGEO_VEC_THREADS), 0, s, nelmt, K, KP);
}

void launch_copy(hipStream_t s, int64_t n_double2, const double* a, double* b) {
  hipLaunchKernelGGL(k_copy, dim3(grid_stride_blocks(n_double2)),
                     dim3(256), 0, s, n_double2, (const double2*)a, (double2*)b);
}

void launch_assemble(hipStream_t s, int64_t n1, const int32_t* rowptr,
                     const int32_t* slots, const double* Y, double* out,
                     const PcgScalars* sc, int skip_mode) {
  hipLaunchKernelGGL(k_assemble, dim3(grid_stride_blocks(n1)),
                     dim3(SGEO_VEC_THREADS), 0, s, n1, rowptr, slots, Y, out,
                     sc, skip_mode);
}

void launch_assemble_acc(hipStream_t s, int64_t n1, const int32_t* rowptr,
                         const int32_t* slots, const double* Y, double* out,
                         int subtract, const PlasticScalars* ps) {
  hipLaunchKernelGGL(k_assemble_acc, dim3(grid_stride_blocks(n1)),
                     dim3(SGEO_VEC_THREADS), 0, s, n1, rowptr, slots, Y, out,
                     subtract, ps);
}

void launch_pcg_begin(hipStream_t s, int64_t n1, const double* u, double* part,
                      PcgScalars* sc, double tol, int32_t maxiter) {
  const unsigned nb = vec_reduce_blocks(n1);
  hipLaunchKernelGGL(k_pcg_begin, dim3(nb), dim3(SGEO_VEC_THREADS), 0, s, n1, u,
                     part);
  hipLaunchKernelGGL(k_pcg_finalize, dim3(1), dim3(256), 0, s, (int)nb, part, sc,
                     (int)FIN_BEGIN, tol, maxiter);
}

// reference-order dot products (k_pcg_seqdot)
void launch_pcg_init(hipStream_t s, int64_t n1, const double* f,
                     const double* kp, const double* dinv, double* r, double* z,
                     double* p, PcgScalars* sc) {
  const unsigned nb = vec_reduce_blocks(n1);
  hipLaunchKernelGGL(k_pcg_init, dim3(nb), dim3(SGEO_VEC_THREADS), 0, s, n1, f,
                     kp, dinv, r, z, p, sc);
  hipLaunchKernelGGL(k_pcg_seqdot, dim3(1), dim3(256), 0, s, n1, r, z, sc, 0);
}

void launch_pcg_assemble(hipStream_t s, int64_t n1, const int32_t* rowptr,
                             const int32_t* slots, const double* Y,
                             const double* p, double* kp, double* part,
                             PcgScalars* sc) {
  const unsigned nb = vec_reduce_blocks(n1);
  hipLaunchKernelGGL(k_pcg_assemble_max, dim3(nb), dim3(SGEO_VEC_THREADS), 0, s,
                     n1, rowptr, slots, Y, p, kp, part, sc);
  hipLaunchKernelGGL(k_pcg_finalize, dim3(1), dim3(256), 0, s, (int)nb, part, sc,
                     (int)FIN_MAXP, 0.0, 0);
  hipLaunchKernelGGL(k_pcg_seqdot, dim3(1), dim3(256), 0, s, n1, p, kp, sc, 1);
}

void launch_pcg_update(hipStream_t s, int64_t n1, const double* p,
                       const double* kp, const double* dinv, double* u,
                       double* r, double* z, double* part, PcgScalars* sc) {
  const unsigned nb = vec_reduce_blocks(n1);
  hipLaunchKernelGGL(k_pcg_update, dim3(nb), dim3(SGEO_VEC_THREADS), 0, s, n1, p,
                     kp, dinv, u, r, z, part, sc);
  hipLaunchKernelGGL(k_pcg_finalize, dim3(1), dim3(256), 0, s, (int)nb, part, sc,
                     (int)FIN_UPDATE, 0.0, 0);
  hipLaunchKernelGGL(k_pcg_seqdot, dim3(1), dim3(256), 0, s, n1, r, z, sc, 2);
}

void launch_pcg_pupdate(hipStream_t s, int64_t n1, const double* z, double* p,
                        const PcgScalars* sc) {
  hipLaunchKernelGGL(k_pcg_pupdate, dim3(grid_stride_blocks(n1)),
                     dim3(SGEO_VEC_THREADS), 0, s, n1, z, p, sc);
}

// equations per block (n_dot 0: a trial's solve, or one without shares)
static inline int pcg_block(int n_dot, int64_t n1) {
  return n_dot > 0 && n1 <= (1 << 18) ? 256 : PCG_BLOCK;
}

// doubles of a solve's partials: p.Kp (n_dot shares, or one per block of
// equations), max|u| and r.z, two generations of max|p|, collapsed forms
size_t pcg_tree_part(int n_dot, int64_t n1) {
  const int nv = (int)nblk(n1, pcg_block(n_dot, n1));
  return (size_t)std::max(n_dot, nv) + 4 * (size_t)nv + 4;
}

PcgPart pcg_part(double* part, int n_dot, int64_t n1) {
  PcgPart q;
  q.block = pcg_block(n_dot, n1);
  q.n_vec = (int)nblk(n1, q.block);
  q.n_dot = n_dot > 0 ? n_dot : q.n_vec;  // 0: from the assembled vector
  q.dot = part;
  q.u = q.dot + std::max(q.n_dot, q.n_vec);
  q.rz = q.u + q.n_vec;
  q.p[0] = q.rz + q.n_vec;
  q.p[1] = q.p[0] + q.n_vec;
  q.c_dot = q.p[1] + q.n_vec;
  q.c_vec = q.c_dot + 1;
  return q;
}

void launch_pcg_start(hipStream_t s, int64_t n1, const double* f, const double* kp,
                      const double* dinv, double* r, double* p, const PcgPart& q,
                      PcgScalars* sc) {
  const auto k = q.block == 256 ? k_pcg_start<256> : k_pcg_start<PCG_BLOCK>;
  hipLaunchKernelGGL(k, dim3(q.n_vec), dim3(q.block), 0, s, n1, f, kp, dinv, r, p, q.rz,
                     q.p[0], (const PcgScalars*)sc);
  hipLaunchKernelGGL(k_pcg_finalize, dim3(1), dim3(256), 0, s, q.n_vec, (const double*)q.rz,
                     sc, (int)FIN_RZ, 0.0, 0);
}

// what follows the product in iteration `it` (0-based; sc: two buffers);
// kp: NULL when the product left its shares of p.Kp
void launch_pcg_iteration(hipStream_t s, int64_t n1, int it, const int32_t* rowptr,
                          const int32_t* slots, const double* Y, double* kp,
                          const double* dinv, double* u, double* r, double* p,
                          const PcgPart& q, PcgScalars* sc) {
  PcgScalars *cur = sc + (it & 1), *nxt = sc + (~it & 1);
  const PcgScalars* cc = cur;
  const double *dot = q.dot, *pu = q.u, *prz = q.rz, *pp = q.p[it & 1];
  const dim3 grid(q.n_vec), block(q.block);
  int nd = q.n_dot, np = q.n_vec;
  if (kp)
    hipLaunchKernelGGL(k_pcg_asm<PCG_BLOCK>, grid, block, 0, s, n1, rowptr, slots, Y,
                       (const double*)p, kp, q.dot, cc);
  if (nd > PCG_DIRECT) {
    hipLaunchKernelGGL(k_pcg_collapse, dim3(1), dim3(256), 0, s, nd,
                       Kinds{{dot, nullptr, nullptr}}, q.c_dot, cc);
    dot = q.c_dot;
    nd = 1;
  }
  const auto step = kp               ? k_pcg_step<PCG_BLOCK, false>
                    : q.block == 256 ? k_pcg_step<256, true>
                                     : k_pcg_step<PCG_BLOCK, true>;
  hipLaunchKernelGGL(step, grid, block, 0, s, n1, rowptr, slots, Y, (const double*)kp,
                     (const double*)p, dinv, u, r, dot, nd, q.u, q.rz, cur);
  if (np > PCG_DIRECT) {
    hipLaunchKernelGGL(k_pcg_collapse, dim3(1), dim3(256), 0, s, np, Kinds{{pu, prz, pp}},
                       q.c_vec, cc);
    pu = q.c_vec;
    prz = pu + 1;
    pp = pu + 2;
    np = 1;
  }
  const auto dir = q.block == 256 ? k_pcg_dir<256> : k_pcg_dir<PCG_BLOCK>;
  hipLaunchKernelGGL(dir, grid, block, 0, s, n1, (const double*)r, dinv, p, pu, prz, pp, np,
                     q.p[~it & 1], cc, nxt);
}

void launch_load(hipStream_t s, int64_t n1, const double* ext,
                 const double* body, double* load) {
  hipLaunchKernelGGL(k_load, dim3(grid_stride_blocks(n1)),
                     dim3(SGEO_VEC_THREADS), 0, s, n1, ext, body, load);
}

void launch_uerr(hipStream_t s, int64_t n1, double* x, double* oldx,
                 double* part, PlasticScalars* ps, double nl_tol) {
  const unsigned nb = vec_reduce_blocks(n1);
  hipLaunchKernelGGL(k_uerr, dim3(nb), dim3(SGEO_VEC_THREADS), 0, s, n1, x, oldx,
                     part);
  hipLaunchKernelGGL(k_uerr_finalize, dim3(1), dim3(256), 0, s, (int)nb, part, ps,
                     nl_tol);
}

}  // namespace sgeo
