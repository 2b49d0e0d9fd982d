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
// Measured: 111 us on 144,000 elements against 801 us for the packed
// matrices (k_ebe_packed_pipe, 4.8 TB/s, at the copy rate), 7.9 against
// 33 us on 4,921.  The 262 MB it must move take 55 us at that rate; the rest
// is the LDS traffic (63 values per point) and the latency of the gathers.
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
  __shared__ double s_xc[MF_EPB * 24];
  __shared__ double s_R[MF_EPB][9][27];
  const int t = threadIdx.x;
  const int64_t e0 = (int64_t)blk * MF_EPB;
  const int ne = nelmt - e0 < MF_EPB ? (int)(nelmt - e0) : MF_EPB;
  const int32_t* gd = gdof + e0 * 81;
#pragma unroll
  for (int k = 0; k < 3; k++) {  // 9 * 81 = 729 <= 3 * 256
    const int q = t + 256 * k;
    if (q < ne * 81) s_u[q] = p[gd[q]];
  }
  if (t < ne * 24) s_xc[t] = corners[e0 * 24 + t];
  const int el = t / 27, i = t - 27 * el;
  const bool on = el < ne;
  const int iz = i / 9, iy = (i - 9 * iz) / 3, ix = i - 9 * iz - 3 * iy;
  double2 lm = {0.0, 0.0};
  if (on) lm = lame[mat_id[e0 + el] - 1];
  __syncthreads();
  auto fma = [](double a, double b, double c) { return __builtin_fma(a, b, c); };
  if (on) {
    double adj[3][3];
    const double det = adjugate_point(ix, iy, iz, s_xc + el * 24, adj);
    const double w = gll_weight(i) / det;
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

}  // namespace sgeo
