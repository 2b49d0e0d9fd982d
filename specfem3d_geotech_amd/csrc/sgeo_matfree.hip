// sgeo_matfree.hip -- EBE products of built meshes without the stored element
// matrices: Y_e = K_e p_e = sum_i B_i^T C B_i p_e detJ_i w_i, evaluated at
// the 27 GLL points from the element's corners.  With collocated 3-point
// GLL bases every reference derivative at a point is a combination of the
// three nodes of a grid line, so a product takes about 3,300 operations
// instead of 6,561 multiply-adds and reads 1 KB of geometry and numbering
// instead of 27 KB (packed FP64) of matrix.  The rounding differs from the
// stored matrices' (each term is formed once instead of through the rounded
// entries of K_e); the operator is the same.
#pragma clang fp contract(off)

#include <algorithm>
#include <utility>

#include "sgeo_device.h"
#include "sgeo_internal.h"

namespace sgeo {

// l_m'(xi_q): row q of the reference derivative matrix, column m
template <typename T>
struct DRow {
  T a, b, c;
};
template <typename T>
__device__ __forceinline__ DRow<T> d_row(int q) {  // (d(q,0), d(q,1), d(q,2))
  return q == 0 ? DRow<T>{(T)-1.5, (T)2, (T)-0.5}
                : q == 1 ? DRow<T>{(T)-0.5, (T)0, (T)0.5} : DRow<T>{(T)0.5, (T)-2, (T)1.5};
}
template <typename T>
__device__ __forceinline__ DRow<T> d_col(int m) {  // (d(0,m), d(1,m), d(2,m))
  return m == 0 ? DRow<T>{(T)-1.5, (T)-0.5, (T)0.5}
                : m == 1 ? DRow<T>{(T)2, (T)0, (T)-2} : DRow<T>{(T)-0.5, (T)0.5, (T)1.5};
}

// Adjugate of the Jacobian J(a,b) = dx_b/dxi_a at GLL point (ix, iy, iz) of
// a hex8 element, and det J: J^-1 = adj / det.  At the GLL points the
// trilinear map's derivative along an axis is a mean of the four edges
// along it, weighted by the (0, 1/4, 1/2, 1) position between them.
// xc[g*3 + b]: corner g (EXODUS order), axis b.
__device__ __forceinline__ double adjugate_point(int ix, int iy, int iz, const double* xc,
                                                 double adj[3][3]) {
  const double xm = 0.5 * (2 - ix), xp = 0.5 * ix, ym = 0.5 * (2 - iy), yp = 0.5 * iy;
  const double zm = 0.5 * (2 - iz), zp = 0.5 * iz;
  double J[3][3];
#pragma unroll
  for (int b = 0; b < 3; b++) {
    double c[8];
#pragma unroll
    for (int g = 0; g < 8; g++) c[g] = xc[g * 3 + b];
    double s = (0.5 * ym * zm) * (c[1] - c[0]);
    s = __builtin_fma(0.5 * yp * zm, c[2] - c[3], s);
    s = __builtin_fma(0.5 * ym * zp, c[5] - c[4], s);
    J[0][b] = __builtin_fma(0.5 * yp * zp, c[6] - c[7], s);
    s = (0.5 * xm * zm) * (c[3] - c[0]);
    s = __builtin_fma(0.5 * xp * zm, c[2] - c[1], s);
    s = __builtin_fma(0.5 * xm * zp, c[7] - c[4], s);
    J[1][b] = __builtin_fma(0.5 * xp * zp, c[6] - c[5], s);
    s = (0.5 * xm * ym) * (c[4] - c[0]);
    s = __builtin_fma(0.5 * xp * ym, c[5] - c[1], s);
    s = __builtin_fma(0.5 * xm * yp, c[7] - c[3], s);
    J[2][b] = __builtin_fma(0.5 * xp * yp, c[6] - c[2], s);
  }
  adj[0][0] = J[1][1] * J[2][2] - J[2][1] * J[1][2];
  adj[0][1] = J[2][1] * J[0][2] - J[0][1] * J[2][2];
  adj[0][2] = J[0][1] * J[1][2] - J[1][1] * J[0][2];
  adj[1][0] = J[2][0] * J[1][2] - J[1][0] * J[2][2];
  adj[1][1] = J[0][0] * J[2][2] - J[2][0] * J[0][2];
  adj[1][2] = J[1][0] * J[0][2] - J[0][0] * J[1][2];
  adj[2][0] = J[1][0] * J[2][1] - J[2][0] * J[1][1];
  adj[2][1] = J[2][0] * J[0][1] - J[0][0] * J[2][1];
  adj[2][2] = J[0][0] * J[1][1] - J[1][0] * J[0][1];
  return J[0][0] * adj[0][0] + J[0][1] * adj[1][0] + J[0][2] * adj[2][0];
}

// R(b, c) of one point from the reference derivatives H(b, c) = d u_c / d xi_b:
//   g = adj H (the gradient times det), sigma = C(g) w / det,
//   R(b, c) = sum_a sigma(c, a) adj(a, b),
// so that B^T C B u detJ w at the point is sum_b d_b(node) R(b, c).
// lam, mu: the Lame parameters times w / det.
template <typename T, typename FMA>
__device__ __forceinline__ void point_flux(const T adj[3][3], T lam, T mu, const T H[3][3],
                                           T R[3][3], FMA fma) {
  T g[3][3];  // g[c][a] = sum_b adj[a][b] H[b][c]
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int a = 0; a < 3; a++)
      g[c][a] = fma(adj[a][2], H[2][c], fma(adj[a][1], H[1][c], adj[a][0] * H[0][c]));
  const T tr = lam * ((g[0][0] + g[1][1]) + g[2][2]), mu2 = mu + mu;
  const T s00 = fma(mu2, g[0][0], tr), s11 = fma(mu2, g[1][1], tr), s22 = fma(mu2, g[2][2], tr);
  const T s01 = mu * (g[0][1] + g[1][0]), s12 = mu * (g[1][2] + g[2][1]),
          s20 = mu * (g[2][0] + g[0][2]);
  const T s[3][3] = {{s00, s01, s20}, {s01, s11, s12}, {s20, s12, s22}};
#pragma unroll
  for (int b = 0; b < 3; b++)
#pragma unroll
    for (int c = 0; c < 3; c++)
      R[b][c] = fma(s[c][2], adj[2][b], fma(s[c][1], adj[1][b], s[c][0] * adj[0][b]));
}

// --------------------------------------------------------------------------
// FP64 product of one vector: nine elements per 256-thread block, a thread
// per GLL point, then per node.
//
// The element vectors are gathered into LDS; each thread evaluates its
// point's Jacobian from the corners in LDS (recomputing it takes about 150
// operations and saves 2 KB of geometry per element), the point's flux R
// (point_flux) and leaves the nine values in LDS; then each thread sums its
// node's three components over the points of the node's three grid lines.
// Blocks are mapped so that each XCD walks a contiguous eighth of the
// elements: neighbours' gathers meet in that XCD's L2.
//
// Measured on 144,000 elements: 109 us (124 with the gathers awaited before
// the Jacobians were formed) against 801 us for the packed matrices
// (k_ebe_packed_pipe, 4.8 TB/s, at the copy rate); on 4,921, 8 against 33 us.
// The 262 MB it must move take 55 us at that rate (200 MB of them cross HBM).
// Counters: vector issue active 46 % of the time, LDS 44 % (63 values per
// point; 8 % are bank conflicts), the waves waiting 61 % of their cycles at
// four per SIMD (124 registers).  Five waves per SIMD gain 2.6 % on 144,000 elements
// and lose 2 % on 4,921; six spill into the time of both (129 us).
// --------------------------------------------------------------------------
#define MF_EPB 9
#define MF_XCD 8

__global__ __launch_bounds__(256) void k_mf64(
    int32_t nelmt, int32_t nblk, const double* __restrict__ corners,
    const int32_t* __restrict__ gdof, const int32_t* __restrict__ mat_id,
    const double2* __restrict__ lame, const double* __restrict__ p, double* __restrict__ Y,
    double* __restrict__ part, const PcgScalars* __restrict__ sc, int skip_mode) {
  if (skip_mode == 1 && sc->done) return;
  if (skip_mode == 2 && !sc->u_nonzero) return;
  const int32_t per = gridDim.x / MF_XCD;  // the grid is a multiple of MF_XCD
  const int32_t blk = (blockIdx.x % MF_XCD) * per + blockIdx.x / MF_XCD;
  if (blk >= nblk) return;  // uniform per block
  __shared__ double s_u[MF_EPB * 81];
  __shared__ __align__(16) double s_xc[MF_EPB * 24];
  __shared__ double s_R[MF_EPB][9][27];
  const int t = threadIdx.x;
  const int64_t e0 = (int64_t)blk * MF_EPB;
  const int ne = nelmt - e0 < MF_EPB ? (int)(nelmt - e0) : MF_EPB;
  const int32_t* gd = gdof + e0 * 81;
  int32_t g[3];
  double ug[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {  // 9 * 81 = 729 <= 3 * 256
    const int q = t + 256 * k;
    g[k] = q < ne * 81 ? gd[q] : 0;
  }
  if (t < ne * 24) s_xc[t] = corners[e0 * 24 + t];
  const int el = t / 27, i = t - 27 * el;
  const bool on = el < ne;
  const int iz = i / 9, iy = (i - 9 * iz) / 3, ix = i - 9 * iz - 3 * iy;
  double2 lm = {0.0, 0.0};
  if (on) lm = lame[mat_id[e0 + el] - 1];
  __syncthreads();
  // the gathers are in flight while the Jacobians are formed
#pragma unroll
  for (int k = 0; k < 3; k++) ug[k] = p[g[k]];
  auto fma = [](double a, double b, double c) { return __builtin_fma(a, b, c); };
  double adj[3][3], w = 0.0;
  if (on) w = gll_weight(i) / adjugate_point(ix, iy, iz, s_xc + el * 24, adj);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const int q = t + 256 * k;
    if (q < ne * 81) s_u[q] = ug[k];
  }
  __syncthreads();
  if (on) {
    const double* u = s_u + el * 81;
    double H[3][3], R[3][3];
    const DRow<double> dx = d_row<double>(ix), dy = d_row<double>(iy), dz = d_row<double>(iz);
    const int nx = i - ix, ny = i - 3 * iy, nz = i - 9 * iz;  // first nodes of the lines
#pragma unroll
    for (int c = 0; c < 3; c++) {
      H[0][c] = fma(dx.c, u[3 * (nx + 2) + c], fma(dx.b, u[3 * (nx + 1) + c], dx.a * u[3 * nx + c]));
      H[1][c] = fma(dy.c, u[3 * (ny + 6) + c], fma(dy.b, u[3 * (ny + 3) + c], dy.a * u[3 * ny + c]));
      H[2][c] = fma(dz.c, u[3 * (nz + 18) + c], fma(dz.b, u[3 * (nz + 9) + c], dz.a * u[3 * nz + c]));
    }
    point_flux<double>(adj, lm.x * w, lm.y * w, H, R, fma);
#pragma unroll
    for (int b = 0; b < 3; b++)
#pragma unroll
      for (int c = 0; c < 3; c++) s_R[el][3 * b + c][i] = R[b][c];
  }
  __syncthreads();
  double d = 0.0;  // the node's share of p.Kp
  if (on) {
    const DRow<double> dx = d_col<double>(ix), dy = d_col<double>(iy), dz = d_col<double>(iz);
    const int nx = i - ix, ny = i - 3 * iy, nz = i - 9 * iz;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const double *rx = s_R[el][c] + nx, *ry = s_R[el][3 + c] + ny, *rz = s_R[el][6 + c] + nz;
      double y = fma(dx.c, rx[2], fma(dx.b, rx[1], dx.a * rx[0]));
      y = fma(dy.c, ry[6], fma(dy.b, ry[3], fma(dy.a, ry[0], y)));
      y = fma(dz.c, rz[18], fma(dz.b, rz[9], fma(dz.a, rz[0], y)));
      d = fma(s_u[el * 81 + 3 * i + c], y, d);
      s_u[el * 81 + 3 * i + c] = y;  // read back only after the barrier
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const int q = t + 256 * k;
    if (q < ne * 81) Y[e0 * 81 + q] = s_u[q];
  }
  if (part) {  // the block's, by block index within the element order
    d = block_sum<4>(d, s_xc);
    if (t == 0) part[blk] = d;
  }
}

// Lame parameters (lambda, mu) of each material from E and nu
__global__ void k_lame(int nmat, const double* __restrict__ ym, const double* __restrict__ nu,
                       double2* __restrict__ lame) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= nmat) return;
  const Cmat c = cmat_of(ym[m], nu[m]);
  lame[m] = double2{c.c12, c.c44};
}

void launch_lame(hipStream_t s, int nmat, const double* ym, const double* nu, double2* lame) {
  hipLaunchKernelGGL(k_lame, dim3((nmat + 63) / 64), dim3(64), 0, s, nmat, ym, nu, lame);
}

int mf64_blocks(int32_t nelmt) { return (nelmt + MF_EPB - 1) / MF_EPB; }

void launch_mf64(hipStream_t s, int32_t nelmt, const double* corners, const int32_t* gdof,
                 const int32_t* mat_id, const double2* lame, const double* p, double* Y,
                 double* part, const PcgScalars* sc, int skip_mode) {
  if (nelmt <= 0) return;
  const int32_t nblk = mf64_blocks(nelmt);
  const unsigned grid = (unsigned)((nblk + MF_XCD - 1) / MF_XCD * MF_XCD);
  hipLaunchKernelGGL(k_mf64, dim3(grid), dim3(256), 0, s, nelmt, nblk, corners, gdof, mat_id,
                     lame, p, Y, part, sc, skip_mode);
}

// --------------------------------------------------------------------------
// FP32 product of the batched engine's columns from the geometry
// --------------------------------------------------------------------------
// Per GLL point 12 floats (three float4): adj(a, b) / 2 row by row, lambda
// w / det, mu w / det, 2 mu w / det, rounded once from FP64.  The halves let
// a line's derivatives be formed without its factors 1/2: with the line's
// node values a, b, c, m = c - a and q = (a + c) - 2 b, twice the
// derivatives at the three points are m - 2 q, m and m + 2 q, and the
// transposed sums take the coefficients of 2 D.  A power of two per point
// moves from the Lame terms to adj, whose largest entry becomes 1 .. 2: with
// elements of length h they are E / h^3 and h^2, and FP32 would end for h below about
// 1e-11 or above 1e14 where their product, E h as in the matrices, does not.
// It enters a flux twice and leaves it exactly, so it changes no bit elsewhere.
//
// Both kernels below form every value by the same operations in the same
// order, so a column's bits do not depend on which one ran, on B or on the
// launch geometry: a point's flux from point_flux; a node's sum over the
// points of its three grid lines in ascending point order (at the point on
// the node itself x, y, z); the element's share of p.Kp in FP64 (exact
// products) over the node's three components, then over the nodes 0..8,
// 9..17 and 18..26 one after another, then the three.
//
// Against the packed FP32 matrices (rounded entries, 81-term FP32 sums) the
// product's error is smaller: relative to 64 bits 6.7e-8 against 1.1e-7 on
// random vectors, 6.6e-8 against 1.8e-7 on CG directions and 6.0e-6 against
// 3.9e-5 on the solution itself (1,152 elements).
__global__ __launch_bounds__(256) void k_point_geometry(
    int32_t nelmt, const double* __restrict__ corners, const int32_t* __restrict__ mat_id,
    const double2* __restrict__ lame, float4* __restrict__ geo) {
  const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (q >= (int64_t)nelmt * 27) return;
  const int64_t e = q / 27;
  const int i = (int)(q - e * 27);
  double xc[24], adj[3][3];
  for (int k = 0; k < 24; k++) xc[k] = corners[e * 24 + k];
  const double det = adjugate_point(i % 3, (i / 3) % 3, i / 9, xc, adj);
  const double w = gll_weight(i) / det;
  const double2 lm = lame[mat_id[e] - 1];
  double f[12] = {0.5 * adj[0][0], 0.5 * adj[0][1], 0.5 * adj[0][2], 0.5 * adj[1][0],
                  0.5 * adj[1][1], 0.5 * adj[1][2], 0.5 * adj[2][0], 0.5 * adj[2][1],
                  0.5 * adj[2][2], lm.x * w,        lm.y * w,        2.0 * lm.y * w};
  double big = 0.0;
  for (int k = 0; k < 9; k++) big = fmax(big, fabs(f[k]));
  const int sh = big > 0.0 && big < INFINITY ? ilogb(big) : 0;
  for (int k = 0; k < 12; k++) f[k] = ldexp(f[k], k < 9 ? -sh : 2 * sh);
  float4* o = geo + q * 3;
  for (int k = 0; k < 3; k++)
    o[k] = float4{(float)f[4 * k], (float)f[4 * k + 1], (float)f[4 * k + 2], (float)f[4 * k + 3]};
}

__device__ __forceinline__ float fmaf1(float a, float b, float c) {
  return __builtin_fmaf(a, b, c);
}

// the nine fluxes of a point from its geometry and twice the reference
// derivatives
template <typename Next>
__device__ __forceinline__ void point_flux32(const float4& g0, const float4& g1,
                                             const float4& g2, const float H[3][3],
                                             float R[3][3], Next next) {
  const float A[3][3] = {{g0.x, g0.y, g0.z}, {g0.w, g1.x, g1.y}, {g1.z, g1.w, g2.x}};
  const float lam = g2.y, mu = g2.z, mu2 = g2.w;
  float g[3][3];  // g[c][a]
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int a = 0; a < 3; a++)
      g[c][a] = fmaf1(A[a][2], H[2][c], fmaf1(A[a][1], H[1][c], A[a][0] * H[0][c]));
  next();
  const float tr = lam * ((g[0][0] + g[1][1]) + g[2][2]);
  const float s00 = fmaf1(mu2, g[0][0], tr), s11 = fmaf1(mu2, g[1][1], tr),
              s22 = fmaf1(mu2, g[2][2], tr);
  const float s01 = mu * (g[0][1] + g[1][0]), s12 = mu * (g[1][2] + g[2][1]),
              s20 = mu * (g[2][0] + g[0][2]);
  const float s[3][3] = {{s00, s01, s20}, {s01, s11, s12}, {s20, s12, s22}};
#pragma unroll
  for (int b = 0; b < 3; b++)
#pragma unroll
    for (int c = 0; c < 3; c++)
      R[b][c] = fmaf1(s[c][2], A[2][b], fmaf1(s[c][1], A[1][b], s[c][0] * A[0][b]));
}

// twice the derivative at point `q` of a line with node values a, b, c
__device__ __forceinline__ float line_deriv(int q, float a, float b, float c) {
  const float m = c - a;
  if (q == 1) return m;
  return fmaf1(q == 0 ? -2.0f : 2.0f, fmaf1(-2.0f, b, a + c), m);
}

// twice l_m'(xi_q): what node m of a line receives from its point q
__device__ __forceinline__ constexpr float d2(int q, int m) {
  constexpr float d[3][3] = {{-3.0f, 4.0f, -1.0f}, {-1.0f, 0.0f, 1.0f}, {1.0f, -4.0f, 3.0f}};
  return d[q][m];
}

// keeps the compiler from carrying what it knows of v past this place, in
// either direction
__device__ __forceinline__ void pin(float& v) { asm volatile("" : "+v"(v)); }

// Point I of an element in registers: u its 81 values, y its 81 sums, g the
// point's geometry (replaced by the next point's, read from LDS while the flux
// is formed).  The compiler keeps no differences of z grid lines from one plane
// of points to the next, and finishes a point before the next: otherwise
// neither would fit the registers.
template <int I>
__device__ __forceinline__ void lane_point(float (&u)[81], float (&y)[81], const float4* ge,
                                           float4 (&g)[3]) {
  constexpr int ix = I % 3, iy = (I / 3) % 3, iz = I / 9;
  constexpr int nx = I - ix, ny = I - 3 * iy, nz = I - 9 * iz;
  if constexpr (I % 9 == 0) {
#pragma unroll
    for (int r = 0; r < 81; r++) pin(u[r]);
  }
  float H[3][3], R[3][3];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    H[0][c] = line_deriv(ix, u[3 * nx + c], u[3 * (nx + 1) + c], u[3 * (nx + 2) + c]);
    H[1][c] = line_deriv(iy, u[3 * ny + c], u[3 * (ny + 3) + c], u[3 * (ny + 6) + c]);
    H[2][c] = line_deriv(iz, u[3 * nz + c], u[3 * (nz + 9) + c], u[3 * (nz + 18) + c]);
  }
  float4 h[3] = {g[0], g[1], g[2]};
  point_flux32(g[0], g[1], g[2], H, R, [&]() {
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (I < 26) {
#pragma unroll
      for (int k = 0; k < 3; k++) h[k] = ge[3 * I + 3 + k];
    }
    __builtin_amdgcn_sched_barrier(0);
  });
#pragma unroll
  for (int k = 0; k < 3; k++) g[k] = h[k];
  // a node's first term starts its sum
#pragma unroll
  for (int m = 0; m < 3; m++)
#pragma unroll
    for (int c = 0; c < 3; c++) {
      float& a = y[3 * (nx + m) + c];
      if (d2(ix, m) != 0.0f) a = I == 0 ? d2(ix, m) * R[0][c] : fmaf1(d2(ix, m), R[0][c], a);
    }
#pragma unroll
  for (int m = 0; m < 3; m++)
#pragma unroll
    for (int c = 0; c < 3; c++) {
      float& a = y[3 * (ny + 3 * m) + c];
      if (d2(iy, m) != 0.0f)
        a = I < 3 && m > 0 ? d2(iy, m) * R[1][c] : fmaf1(d2(iy, m), R[1][c], a);
    }
#pragma unroll
  for (int m = 0; m < 3; m++)
#pragma unroll
    for (int c = 0; c < 3; c++) {
      float& a = y[3 * (nz + 9 * m) + c];
      if (d2(iz, m) != 0.0f)
        a = I < 9 && m > 0 ? d2(iz, m) * R[2][c] : fmaf1(d2(iz, m), R[2][c], a);
    }
#pragma unroll
  for (int m = 0; m < 3; m++)
#pragma unroll
    for (int c = 0; c < 3; c++) {
      pin(y[3 * (nx + m) + c]);
      if (m != iy) pin(y[3 * (ny + 3 * m) + c]);
      if (m != iz) pin(y[3 * (nz + 9 * m) + c]);
    }
}

template <int... I>
__device__ __forceinline__ void lane_points(float (&u)[81], float (&y)[81], const float4* ge,
                                            std::integer_sequence<int, I...>) {
  float4 g[3] = {ge[0], ge[1], ge[2]};
  (lane_point<I>(u, y, ge, g), ...);
}

// A lane per (element, column): 64 / B elements per wave, the element's 81
// values and 81 sums in registers, the 27 points unrolled; one wave per
// block, two per SIMD.  The elements' geometry is loaded into LDS beside the
// gathers: read point by point from memory (through the scalar cache at
// B = 64) every line's latency stood in the wave's way, 1.72 ms on 144,000
// elements.  Of the 1.15 ms that remain 0.78 are the 3,340 vector instructions
// of a wave at one per 4 cycles and SIMD (counted); the rest is the start of
// each wave (a chain of four dependent loads).  It moves 4.5 GB meanwhile.
// Measured against k_bmv_mfma: 144,000 elements, 64 columns 1.15 against
// 1.80 ms, 8 columns 0.185 against 0.80; 12,544 elements, 64 columns 109
// against 165 us; 25,344, 8 columns 35 against 146.
template <int B>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_bmf_lane(
    int32_t nelmt, int lx, const float4* __restrict__ geo, const int32_t* __restrict__ gdof,
    const int32_t* __restrict__ eorder, const float* __restrict__ P, int64_t nv,
    float* __restrict__ Y, double* __restrict__ edot, const int32_t* __restrict__ cst,
    const BCol* __restrict__ bc, int want_mask) {
  constexpr int EPW = 64 / B;
  const int l = threadIdx.x, j = l % B;
  // this XCD's share of the walk (one of 1 << lx), and the wave's place in it
  const int xcd = blockIdx.x & ((1 << lx) - 1);
  const int32_t xe0 = (int32_t)((int64_t)nelmt * xcd >> lx);
  const int32_t xe1 = (int32_t)((int64_t)nelmt * (xcd + 1) >> lx);
  const int32_t wi = xe0 + (int32_t)(blockIdx.x >> lx) * EPW;
  if (wi >= xe1) return;
  const bool in = wi + l / B < xe1;
  const int32_t e = B == 64 ? eorder[wi] : eorder[in ? wi + l / B : wi];
  // the loads of a wave's start stand in one chain (element, numbering,
  // gathers): everything that does not depend on it is issued beside it
  constexpr int NG = (EPW * 81 + 63) / 64;
  __shared__ float4 s_geo[NG * 64];
  float4 gr[NG];
#pragma unroll
  for (int k = 0; k < NG; k++) {
    const int q = l + 64 * k, es = q / 81;
    const int32_t eg = B == 64 ? e : __shfl(e, es < EPW ? es * B : 0);
    gr[k] = geo[(int64_t)eg * 81 + (es < EPW ? q - 81 * es : 0)];
  }
  const bool jv = (want_mask >> cst[j]) & 1, on = jv && in;
  const unsigned long long any = __ballot(jv);
  if (any == 0) return;
  // the column's search direction of the iteration being computed; lanes of
  // columns outside the mask compute on the first wanted column's (their own
  // direction can sit in another buffer, whose lines nobody else reads)
  const int jr = jv ? j : __builtin_ctzll(any) % B;
  const float* pj = P + (int64_t)((bc[jr].it + 1) & bc[jr].pmask) * nv + jr;
  const int32_t* gd = gdof + (int64_t)e * 81;
  float u[81], y[81];
#pragma unroll
  for (int r = 0; r < 81; r++) u[r] = pj[(int64_t)gd[r] * B];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int k = 0; k < NG; k++) s_geo[l + 64 * k] = gr[k];
  __syncthreads();
  lane_points(u, y, s_geo + (l / B) * 81, std::make_integer_sequence<int, 27>());
  double s[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
#pragma unroll
    for (int n = 9 * k; n < 9 * k + 9; n++) {
      double d = (double)u[3 * n] * (double)y[3 * n];
      d = __builtin_fma((double)u[3 * n + 1], (double)y[3 * n + 1], d);
      d = __builtin_fma((double)u[3 * n + 2], (double)y[3 * n + 2], d);
      s[k] = n == 9 * k ? d : s[k] + d;
    }
  }
  if (on) {
    float* ye = Y + (int64_t)e * 81 * B + j;
#pragma unroll
    for (int r = 0; r < 81; r++) ye[r * B] = y[r];
    edot[(int64_t)e * B + j] = (s[0] + s[1]) + s[2];
  }
}

// A thread per (point, element, column), eight (element, column) slots per
// block, the exchange between points and nodes through LDS: 27 times the
// threads of the lane kernel for the same columns.  Below BMF_POINT_SLOTS
// slots the lane kernel leaves most of the chip idle while each of its waves
// runs 3,400 operations one after another.  Measured against k_bmv_mfma:
// 384 elements, 8 columns 4.7 against 8.7 us; 6,300, one column 6.0 against
// 38; 144,000, one column 75 against 760.
__global__ __launch_bounds__(256) void k_bmf_point(
    int32_t nslot, int lb, const float4* __restrict__ geo, const int32_t* __restrict__ gdof,
    const float* __restrict__ P, int64_t nv, float* __restrict__ Y, double* __restrict__ edot,
    const int32_t* __restrict__ cst, const BCol* __restrict__ bc, int want_mask) {
  __shared__ float s_u[81 * 8];
  __shared__ float s_R[9 * 27 * 8];
  __shared__ double s_t[27 * 8], s_s[3 * 8];
  const int t = threadIdx.x, k = t & 7, i = t >> 3;  // slot of the block, point
  const int32_t slot = blockIdx.x * 8 + k;
  const int B = 1 << lb, j = slot & (B - 1);
  const int64_t e = slot >> lb;
  const bool on = slot < nslot && ((want_mask >> cst[j]) & 1);
  if (!__syncthreads_or(on)) return;
  const float* pj = P + (int64_t)((bc[j].it + 1) & bc[j].pmask) * nv + j;
#pragma unroll
  for (int q = 0; q < 3; q++) {
    const int r = i + 32 * q;
    if (r < 81) s_u[r * 8 + k] = on ? pj[(int64_t)gdof[e * 81 + r] << lb] : 0.0f;
  }
  const bool point = i < 27;
  float4 g0, g1, g2;
  if (point && on) {
    const float4* ge = geo + (e * 27 + i) * 3;
    g0 = ge[0];
    g1 = ge[1];
    g2 = ge[2];
  }
  const int iz = i / 9, iy = (i - 9 * iz) / 3, ix = i - 9 * iz - 3 * iy;
  __syncthreads();
  if (point && on) {
    float H[3][3], R[3][3];
    auto deriv = [&](int q, int n0, int st, int c) {  // line_deriv, q at run time
      const float a = s_u[(3 * n0 + c) * 8 + k], b = s_u[(3 * (n0 + st) + c) * 8 + k];
      const float d = s_u[(3 * (n0 + 2 * st) + c) * 8 + k];
      return fmaf1(2.0f * (float)(q - 1), fmaf1(-2.0f, b, a + d), d - a);
    };
#pragma unroll
    for (int c = 0; c < 3; c++) {
      H[0][c] = deriv(ix, i - ix, 1, c);
      H[1][c] = deriv(iy, i - 3 * iy, 3, c);
      H[2][c] = deriv(iz, i - 9 * iz, 9, c);
    }
    point_flux32(g0, g1, g2, H, R, []() {});
#pragma unroll
    for (int b = 0; b < 3; b++)
#pragma unroll
      for (int c = 0; c < 3; c++) s_R[((3 * b + c) * 27 + i) * 8 + k] = R[b][c];
  }
  __syncthreads();
  if (point && on) {
    double d = 0.0;
    // 2 l_m'(xi_q) of the lines' points q = 0, 1, 2 at this node's place m
    auto coef = [](int m, float (&o)[3]) {
      o[0] = m == 0 ? -3.0f : m == 1 ? 4.0f : -1.0f;
      o[1] = m == 0 ? -1.0f : m == 1 ? 0.0f : 1.0f;
      o[2] = m == 0 ? 1.0f : m == 1 ? -4.0f : 3.0f;
    };
    float cx[3], cy[3], cz[3];
    coef(ix, cx);
    coef(iy, cy);
    coef(iz, cz);
    const int nx = i - ix, ny = i - 3 * iy, nz = i - 9 * iz;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const float* rx = s_R + (c * 27 + nx) * 8 + k;
      const float* ry = s_R + ((3 + c) * 27 + ny) * 8 + k;
      const float* rz = s_R + ((6 + c) * 27 + nz) * 8 + k;
      const float x[3] = {rx[0], rx[8], rx[16]}, v[3] = {ry[0], ry[24], ry[48]},
                  z[3] = {rz[0], rz[72], rz[144]};
      // ascending point order: the lower points of z, y and x, the node's
      // own point, then the upper ones of x, y and z
      float y = 0.0f;
#pragma unroll
      for (int q = 0; q < 2; q++) y = fmaf1(q < iz ? cz[q] : 0.0f, z[q], y);
#pragma unroll
      for (int q = 0; q < 2; q++) y = fmaf1(q < iy ? cy[q] : 0.0f, v[q], y);
#pragma unroll
      for (int q = 0; q < 2; q++) y = fmaf1(q < ix ? cx[q] : 0.0f, x[q], y);
      y = fmaf1(ix == 0 ? cx[0] : ix == 1 ? cx[1] : cx[2], ix == 0 ? x[0] : ix == 1 ? x[1] : x[2], y);
      y = fmaf1(iy == 0 ? cy[0] : iy == 1 ? cy[1] : cy[2], iy == 0 ? v[0] : iy == 1 ? v[1] : v[2], y);
      y = fmaf1(iz == 0 ? cz[0] : iz == 1 ? cz[1] : cz[2], iz == 0 ? z[0] : iz == 1 ? z[1] : z[2], y);
#pragma unroll
      for (int q = 1; q < 3; q++) y = fmaf1(q > ix ? cx[q] : 0.0f, x[q], y);
#pragma unroll
      for (int q = 1; q < 3; q++) y = fmaf1(q > iy ? cy[q] : 0.0f, v[q], y);
#pragma unroll
      for (int q = 1; q < 3; q++) y = fmaf1(q > iz ? cz[q] : 0.0f, z[q], y);
      float& u = s_u[(3 * i + c) * 8 + k];
      d = __builtin_fma((double)u, (double)y, d);
      u = y;  // read back only after the barrier
    }
    s_t[i * 8 + k] = d;
  }
  __syncthreads();
  if (on) {
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const int r = i + 32 * q;
      if (r < 81) Y[((e * 81 + r) << lb) + j] = s_u[r * 8 + k];
    }
    if (i < 3) {
      double s = s_t[9 * i * 8 + k];
#pragma unroll
      for (int n = 1; n < 9; n++) s = s + s_t[(9 * i + n) * 8 + k];
      s_s[i * 8 + k] = s;
    }
  }
  __syncthreads();
  if (on && i == 0) edot[(e << lb) + j] = (s_s[k] + s_s[8 + k]) + s_s[16 + k];
}

// Up to here a wave of the lane kernel, alone on its SIMD, takes longer than
// the whole point kernel: 9,216 slots 9.8 against 6.3 us, 18,432 10.1 against
// 11.2, 36,864 11.3 against 18.9.  One and two columns always go by points:
// the lane kernel would gather 64 or 32 elements' scattered values per load
// (144,000 elements, one column: 75 us by points, 115 by lanes).
#define BMF_POINT_SLOTS 16384

void launch_point_geometry(hipStream_t s, int32_t nelmt, const double* corners,
                           const int32_t* mat_id, const double2* lame, float4* geo) {
  if (nelmt <= 0) return;
  hipLaunchKernelGGL(k_point_geometry, dim3((unsigned)(((int64_t)nelmt * 27 + 255) / 256)),
                     dim3(256), 0, s, nelmt, corners, mat_id, lame, geo);
}

bool bmf_by_points(int32_t nelmt, int B) {
  return B < 4 || (int64_t)nelmt * B <= BMF_POINT_SLOTS;
}

// Product of the engine's columns from the geometry.  Of the launch geometry
// the lane kernel takes the XCD split of its walk; it is not persistent (a
// fixed number of blocks per CU left the last of them running alone).
void launch_bmf(hipStream_t s, int32_t nelmt, int B, BmvGeom geom, const float4* geo,
                const int32_t* gdof, const int32_t* eorder, const float* P, int64_t nv,
                float* Y, double* edot, const int32_t* cst, const BCol* bc, int want_mask) {
  if (nelmt <= 0) return;
  if (bmf_by_points(nelmt, B)) {
    const int64_t nslot = (int64_t)nelmt * B;
    int lb = 0;
    while ((1 << lb) < B) lb++;
    hipLaunchKernelGGL(k_bmf_point, dim3((unsigned)((nslot + 7) / 8)), dim3(256), 0, s,
                       (int32_t)nslot, lb, geo, gdof, P, nv, Y, edot, cst, bc, want_mask);
    return;
  }
  const int lx = geom.xcd_split ? 3 : 0, nx = 1 << lx;  // MF_XCD XCDs
  // one wave per block; every XCD's share may round up
  const int64_t per = 64 / B, share = (nelmt + nx - 1) / nx;
  const unsigned g = (unsigned)((share + per - 1) / per * nx);
#define SGEO_LANE(BB)                                                                        \
  case BB:                                                                                   \
    hipLaunchKernelGGL(k_bmf_lane<BB>, dim3(g), dim3(64), 0, s, nelmt, lx, geo,              \
                       gdof, eorder, P, nv, Y, edot, cst, bc, want_mask);                    \
    break;
  switch (B) {
    SGEO_LANE(64)
    SGEO_LANE(32)
    SGEO_LANE(16)
    SGEO_LANE(8)
    SGEO_LANE(4)
  }
#undef SGEO_LANE
}

}  // namespace sgeo
