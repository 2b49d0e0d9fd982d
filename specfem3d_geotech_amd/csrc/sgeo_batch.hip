// sgeo_batch.hip -- multi-trial (multi-RHS) kernels of the mixed-precision
// EBE-PCG: B strength-reduction trials share one mesh and one elastic
// stiffness (the viscoplastic method never changes K, src/slope.F90:288), so
// every CG iteration applies K once to all B columns.  Here: the FP32 product
// of uploaded matrices, the FP64 residual product, and the columns' body
// passes and state.  Built meshes' FP32 products come from the geometry
// (sgeo_matfree.hip); the vector kernels and reductions are in sgeo_bvec.hip.
//
// Vectors are interleaved [n1][B] (column fastest): an element gathers 81
// contiguous B-vectors and every update is unit-stride.  The inner CG
// vectors (r, p) and the element product are FP32 (K p is summed from the
// element products inside the update, never stored); dot products, the
// solution x, the FP64 true residual f - K x and all plastic state are FP64.
// Every reduction combines the partials of groups of tiles in a fixed order,
// so a column's arithmetic does not depend on B or on the other columns: a
// trial gives the same bits alone and in any batch.
#pragma clang fp contract(off)

#include "sgeo_device.h"
#include "sgeo_internal.h"

namespace sgeo {

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bool wanted(const int32_t* cst, int j, int mask) {
  return (mask >> cst[j]) & 1;
}

// --------------------------------------------------------------------------
// FP32 batched element product of uploaded matrices, on MFMA:
//   Y[e][r][j] = sum_c K_e(r,c) P[g(e,c)][j]
// with v_mfma_f32_16x16x4f32 (A 16x4, B 4x16, D 16x16): rows 0..79 in 5
// tiles of 16, columns in tiles of 16 (B < 16: one partial tile), k in 21
// steps of 4 (81 -> 84).  Row 80 is a dot product on the vector ALUs: lane
// (j, kq) sums K(80, 4s+kq) P(4s+kq, j) over the k-steps s -- the B operand
// it already holds -- and the four kq partials are added across lanes in a
// fixed order.  A sixth MFMA row tile would spend 15 of its 16 rows on
// zero padding.  One element per block of 4 waves; wave w takes column
// tile n = w % NT and row tiles m = w / NT (+ 4 / NT ...); the wave of each
// column tile with the fewest row tiles also takes row 80.
// The packed upper triangle of K_e is unpacked (with its mirror) into LDS
// row by row, Kf[r * BMV_RLD + slot(c)] with slot(c) = (c % 4) * 24 + c / 4:
// lane (i, kq) of k-steps 4m .. 4m+3 needs K(r, 4s + kq) for s = 4m .. 4m+3,
// which sit at four consecutive slots, so one 16-byte read serves four
// MFMAs; zero padded for k = 81..83.  BMV_RLD = 100 floats puts the 16 rows
// of a read on disjoint groups of four banks and keeps every read 16-byte
// aligned.
// A column's result depends only on its own P column, so trials are
// independent of the batch; columns not in `want_mask` are not written.
//
// The epilogue also forms the element's share of p.Kp,
//   edot[e][j] = sum_r P(g(e,r), j) Y[e][r][j]   (FP64 sums of exact products),
// since p.Kp = sum_g p_g sum_{e,r: g(e,r)=g} Y[e][r] = sum_e p_e . Y_e.  The
// accumulator of row tile mt holds Y(16 mt + 4 kq + v, j) in lane (kq, j),
// register v, while the B operand of k-step 4 mt + i holds P(16 mt + 4 i +
// kq, j) in lane (kq, j).  A 4x4 transpose of (lane group, register) -- two
// v_permlane32_swap and two v_permlane16_swap -- puts Y(16 mt + 4 i + kq, j)
// in register i of lane (kq, j), beside its P.  The share is summed in one
// order for every column tiling: per lane, row tiles 0..4 (each the four
// products i = 0..3 in order), then row 80 in lane group 0, then the four
// lane groups (xor 16, xor 32; IEEE addition commutes, so all four lanes
// hold the same sum).  When a column tile's row tiles are spread over
// several waves (B <= 32), the per-tile sums meet in LDS and one wave adds
// them in that order.  Per-element shares keep the reduction independent of
// which block computed an element.
// --------------------------------------------------------------------------
#define BMV_RLD 100
#define BMV_KC 84
__device__ __forceinline__ constexpr int bmv_slot(int c) { return (c & 3) * 24 + (c >> 2); }

// (lane group, register) transpose of a 4x4 block of 16-lane groups:
// on return a[i] in lane group g holds what a[g] held in lane group i
__device__ __forceinline__ void lanegroup_transpose4(float (&a)[4]) {
  uint32_t u0 = __float_as_uint(a[0]), u1 = __float_as_uint(a[1]);
  uint32_t u2 = __float_as_uint(a[2]), u3 = __float_as_uint(a[3]);
  // lanes 32..63 of the first operand <-> lanes 0..31 of the second
  auto s02 = __builtin_amdgcn_permlane32_swap(u0, u2, false, false);
  auto s13 = __builtin_amdgcn_permlane32_swap(u1, u3, false, false);
  // odd 16-lane rows of the first operand <-> even rows of the second
  auto t01 = __builtin_amdgcn_permlane16_swap(s02[0], s13[0], false, false);
  auto t23 = __builtin_amdgcn_permlane16_swap(s02[1], s13[1], false, false);
  a[0] = __uint_as_float(t01[0]);
  a[1] = __uint_as_float(t01[1]);
  a[2] = __uint_as_float(t23[0]);
  a[3] = __uint_as_float(t23[1]);
}

__device__ __forceinline__ int tri_col(int q) {  // c with c(c+1)/2 <= q < (c+1)(c+2)/2
  int c = (int)((sqrtf(8.0f * (float)q + 1.0f) - 1.0f) * 0.5f);
  if ((c + 1) * (c + 2) / 2 <= q) c++;
  if (c * (c + 1) / 2 > q) c--;
  return c;
}

// Persistent and software-pipelined: the grid holds a few blocks per CU.
// The elements are taken in the order eorder[] (spatially compact runs,
// built with the engine).  With nxcd = 8, each XCD (blocks are dispatched
// to the 8 XCDs round-robin) walks its own contiguous eighth of that order,
// so elements in flight together share nodes and their gathered P rows hit
// in that XCD's L2; nxcd = 1 is a plain grid-stride walk.  While element e is multiplied, K
// and gdof of the block's next element are already in registers, and the
// next element's P rows are gathered before its K is unpacked.  The grid
// size and nxcd change which block computes an element, never how: the
// launch geometry does not change any result bit.
#define BMV_XCD 8

template <int NT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
void k_bmv_mfma(int32_t nelmt, int B, int nxcd,
                                                  const float* __restrict__ KP,
                                                  const int32_t* __restrict__ gdof,
                                                  const int32_t* __restrict__ eorder,
                                                  const float* __restrict__ P,
                                                  int64_t nv,
                                                  float* __restrict__ Y,
                                                  double* __restrict__ edot,
                                                  const int32_t* __restrict__ cst,
                                                  const BCol* __restrict__ bc,
                                                  int want_mask) {
  constexpr int NS = 4 / NT;             // waves per column tile
  constexpr int NMT = 5;                 // MFMA row tiles: rows 0..79
  constexpr int NM = (NMT + NS - 1) / NS;  // row tiles per wave
  constexpr int KPT = (3321 + 255) / 256;  // packed entries per thread
  __shared__ __align__(16) float Kf[81 * BMV_RLD];
  __shared__ int32_t sg[2][BMV_KC];
  // p.Kp shares of the row tiles (and row 80) of each column tile, when they
  // come from several waves
  __shared__ double xs[NS > 1 ? NT : 1][NS > 1 ? NMT + 1 : 1][64];
  const int t = threadIdx.x;
  // range of the element walk eorder[] of this block's XCD, and the block's
  // stride within it; wi is the walk position, e = eorder[wi] the element
  const int xcd = blockIdx.x % nxcd;
  const int nbx = gridDim.x / nxcd;  // grid is a multiple of nxcd
  const int64_t xe0 = (int64_t)nelmt * xcd / nxcd;
  const int64_t xe1 = (int64_t)nelmt * (xcd + 1) / nxcd;
  int64_t wi = xe0 + blockIdx.x / nxcd;
  int64_t e = wi < xe1 ? eorder[wi] : 0;
  // column tile of this wave; columns outside the mask are neither
  // gathered nor multiplied nor stored, but the wave keeps to the block's
  // barriers
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int l = t & 63;
  const int n = w % NT, mpart = NS == 1 ? 0 : w / NT;
  const int j = n * 16 + (l & 15);
  const bool jv = j < B && wanted(cst, j, want_mask);
  const bool wave_on = __any(jv);
  const int jl = j < B ? j : B - 1;
  // lanes of columns not in the mask (and past B) gather nothing: their B
  // operand is 0 and their results are not stored.  Their own search
  // direction can sit in any of the ring's buffers, so a gather there would
  // fetch lines no wanted column uses.
  // the column's search direction of the iteration being computed
  // (pmask + 1) n1 B < 2^32, checked when the engine is made
  const uint32_t poff = (uint32_t)((bc[jl].it + 1) & bc[jl].pmask) * (uint32_t)nv;
  const int kq = l >> 4;
  const bool row80 = mpart == NS - 1;  // wave-uniform
  // zero padding, once: k columns 81..83 (rows 0..80)
  for (int q = t; q < 3 * 81; q += 256) Kf[(q % 81) * BMV_RLD + bmv_slot(81 + q / 81)] = 0.0f;
  if (t >= 81 && t < BMV_KC) { sg[0][t] = 0; sg[1][t] = 0; }
  // LDS addresses of this thread's packed entries q = t + 256 i (fixed for
  // the kernel): K(r, c) at r*RLD + slot(c) and its mirror at c*RLD +
  // slot(r), both below 2^16, packed in one word
  uint32_t kaddr[KPT];
#pragma unroll
  for (int i = 0; i < KPT; i++) {
    const int q = t + 256 * i;
    const int c = q < 3321 ? tri_col(q) : 0;
    const int r = q < 3321 ? q - c * (c + 1) / 2 : 0;
    kaddr[i] = (uint32_t)(r * BMV_RLD + bmv_slot(c)) |
               ((uint32_t)(c * BMV_RLD + bmv_slot(r)) << 16);
  }
  // prologue: K and gdof of the first element
  float kreg[KPT];
  int32_t greg = 0;
  if (wi < xe1) {
    const float* src = KP + e * SGEO_KPACK;
#pragma unroll
    for (int i = 0; i < KPT; i++) {
      const int q = t + 256 * i;
      kreg[i] = q < 3321 ? src[q] : 0.0f;
    }
    if (t < 81) greg = gdof[e * 81 + t];
  }
  if (t < 81) sg[0][t] = greg;
  __syncthreads();
  float bv[21];
  if (wave_on && wi < xe1) {
#pragma unroll
    for (int s = 0; s < 21; s++)
      bv[s] = jv ? P[(uint32_t)(sg[0][4 * s + kq] * B + jl) + poff] : 0.0f;
  }
  int cur = 0;
  for (; wi < xe1; wi += nbx) {
    // unpack the packed upper triangle (and its mirror) of element e
#pragma unroll
    for (int i = 0; i < KPT; i++) {
      if (t + 256 * i < 3321) {
        Kf[kaddr[i] & 0xffffu] = kreg[i];
        Kf[kaddr[i] >> 16] = kreg[i];
      }
    }
    __syncthreads();
    const int64_t wn = wi + nbx;
    const int64_t en = wn < xe1 ? eorder[wn] : 0;
    if (wn < xe1) {  // next element's K and gdof, in flight during the MFMAs
      const float* src = KP + en * SGEO_KPACK;
#pragma unroll
      for (int i = 0; i < KPT; i++) {
        const int q = t + 256 * i;
        kreg[i] = q < 3321 ? src[q] : 0.0f;
      }
      if (t < 81) greg = gdof[en * 81 + t];
    }
    if (wave_on) {
      f32x4 acc[NM];
#pragma unroll
      for (int i = 0; i < NM; i++) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      float r80 = 0.0f;
      // k-steps s = 0..19 four at a time (one 16-byte read per row tile),
      // then s = 20; every accumulator sums its k-steps in order 0..20
      const float* kr = Kf + (l & 15) * BMV_RLD + kq * 24;  // row (l & 15), group kq
#pragma unroll
      for (int m = 0; m < 5; m++) {
        f32x4 a[NM];
        f32x4 a80;
#pragma unroll
        for (int i = 0; i < NM; i++) {
          const int mt = mpart + i * NS;  // wave-uniform
          if (NM * NS > NMT && mt >= NMT) break;
          a[i] = *reinterpret_cast<const f32x4*>(kr + mt * 16 * BMV_RLD + 4 * m);
        }
        if (row80)
          a80 = *reinterpret_cast<const f32x4*>(Kf + 80 * BMV_RLD + kq * 24 + 4 * m);
#pragma unroll
        for (int ss = 0; ss < 4; ss++) {
          const int s = 4 * m + ss;
#pragma unroll
          for (int i = 0; i < NM; i++) {
            const int mt = mpart + i * NS;
            if (NM * NS > NMT && mt >= NMT) break;
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][ss], bv[s], acc[i], 0, 0, 0);
          }
          if (row80) r80 = __builtin_fmaf(a80[ss], bv[s], r80);
        }
      }
#pragma unroll
      for (int i = 0; i < NM; i++) {
        const int mt = mpart + i * NS;
        if (NM * NS > NMT && mt >= NMT) break;
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[mt * 16 * BMV_RLD + 20], bv[20],
                                                      acc[i], 0, 0, 0);
      }
      if (row80) r80 = __builtin_fmaf(Kf[80 * BMV_RLD + kq * 24 + 20], bv[20], r80);
      if (row80) {  // the four k-groups of column j: lanes j, j+16, j+32, j+48
        r80 = r80 + __shfl_xor(r80, 16);
        r80 = r80 + __shfl_xor(r80, 32);
      }
      if (jv) {
#pragma unroll
        for (int i = 0; i < NM; i++) {
          const int mt = mpart + i * NS;
          if (NM * NS > NMT && mt >= NMT) break;
#pragma unroll
          for (int v = 0; v < 4; v++)
            Y[(e * 81 + mt * 16 + 4 * kq + v) * B + j] = acc[i][v];
        }
        if (row80 && kq == 0) Y[(e * 81 + 80) * B + j] = r80;
      }
      // the element's share of p.Kp, per lane: row tiles in order, then row 80
      double dsum = 0.0;
#pragma unroll
      for (int i = 0; i < NM; i++) {
#pragma unroll
        for (int mc = 0; mc < NMT; mc++) {
          if (mc != mpart + i * NS) continue;  // wave-uniform; keeps bv indices static
          float a[4] = {acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
          lanegroup_transpose4(a);
          double u = (double)a[0] * (double)bv[4 * mc];
          u = u + (double)a[1] * (double)bv[4 * mc + 1];
          u = u + (double)a[2] * (double)bv[4 * mc + 2];
          u = u + (double)a[3] * (double)bv[4 * mc + 3];
          if (NS == 1) dsum = dsum + u;
          else xs[n][mc][l] = u;
        }
      }
      const double d80 = (row80 && kq == 0) ? (double)r80 * (double)bv[20] : 0.0;
      if (NS == 1) {
        dsum = dsum + d80;
        dsum = dsum + __shfl_xor(dsum, 16);
        dsum = dsum + __shfl_xor(dsum, 32);
        if (jv && kq == 0) edot[e * B + j] = dsum;
      } else if (row80) {
        xs[n][NMT][l] = d80;
      }
    }
    if (t < 81) sg[cur ^ 1][t] = greg;
    __syncthreads();  // Kf free for the next element, its gdof visible
    cur ^= 1;
    if (NS > 1 && wave_on && mpart == 0) {  // the shares of the column tile's waves
      double dsum = 0.0;
#pragma unroll
      for (int mc = 0; mc <= NMT; mc++) dsum = dsum + xs[n][mc][l];
      dsum = dsum + __shfl_xor(dsum, 16);
      dsum = dsum + __shfl_xor(dsum, 32);
      if (jv && kq == 0) edot[e * B + j] = dsum;
    }
    if (wave_on && wn < xe1) {
#pragma unroll
      for (int s = 0; s < 21; s++)
        bv[s] = jv ? P[(uint32_t)(sg[cur][4 * s + kq] * B + jl) + poff] : 0.0f;
    }
    e = en;
  }
}

// --------------------------------------------------------------------------
// FP64 batched element product for the true residual f - K x, on the FP64
// MFMA (v_mfma_f64_16x16x4f64), for the columns of the residual list only:
//   Y64[e][r][q] = sum_c K_e(r,c) X[g(e,c)][rlist[q]],  q < nres = rlist[64],
// with the list's columns packed into tiles of 16 (q = 16 n + lane % 16), so
// the work scales with the columns that need a residual, not with B.  The
// packed upper triangle of K_e (FP64) is unpacked into LDS as
// Kf64[c * B64_LDK + r]; rows 0..79 are 5 row tiles of 16, k runs in 21
// steps of 4 (81 -> 84, zero padded), row 80 is a dot product on the vector
// ALUs as in the FP32 product.  The list length is read on the device, so
// one captured launch serves any list.  Operand layouts: A (16x4) lane l
// holds A(l % 16, l / 16); B (4x16) lane l holds B(l / 16, l % 16); D (16x16)
// lane l, register v holds D(4 v + l / 16, l % 16) -- rows interleaved,
// unlike the FP32 instruction's 4 (l / 16) + v.  A column's sums do not
// depend on its place in the list.
// Persistent and pipelined like the FP32 product: K and gdof of the block's
// next element are loaded during the MFMAs.
// --------------------------------------------------------------------------
#define B64_LDK 88
typedef double f64x4 __attribute__((ext_vector_type(4)));

// Wave w multiplies list tile w (list places 16 w .. 16 w + 15) over all
// row tiles; waves past the list idle.
__device__ __forceinline__ void bmv64_element(
    int64_t e, int nres, int B, const double* __restrict__ X, double* __restrict__ Y,
    const int32_t* __restrict__ rlist, const double* Kf, const int32_t* sgc, int w, int l) {
  constexpr int NMT = 5;
  if (w * 16 >= nres) return;  // wave-uniform: no column in this tile
  const int q = w * 16 + (l & 15);  // list place of this lane's column
  const bool qv = q < nres;
  const int jc = rlist[qv ? q : 0];
  const int kq = l >> 4;
  double bv[21];
#pragma unroll
  for (int s = 0; s < 21; s++) bv[s] = X[(uint32_t)(sgc[4 * s + kq] * B + jc)];
  f64x4 acc[NMT];
#pragma unroll
  for (int i = 0; i < NMT; i++) acc[i] = f64x4{0.0, 0.0, 0.0, 0.0};
  double r80 = 0.0;
#pragma unroll
  for (int s = 0; s < 21; s++) {
    const double* kc = Kf + (4 * s + kq) * B64_LDK + (l & 15);
#pragma unroll
    for (int i = 0; i < NMT; i++)
      acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(kc[i * 16], bv[s], acc[i], 0, 0, 0);
    r80 = r80 + Kf[(4 * s + kq) * B64_LDK + 80] * bv[s];
  }
  // the four k-groups of the column: lanes p, p+16, p+32, p+48
  r80 = r80 + __shfl_xor(r80, 16);
  r80 = r80 + __shfl_xor(r80, 32);
  if (!qv) return;
#pragma unroll
  for (int i = 0; i < NMT; i++)
#pragma unroll
    for (int v = 0; v < 4; v++) Y[(e * 81 + i * 16 + 4 * v + kq) * B + q] = acc[i][v];
  if (kq == 0) Y[(e * 81 + 80) * B + q] = r80;
}

__global__ __launch_bounds__(256) void k_bmv64(int32_t nelmt, int B,
                                               const double* __restrict__ KP,
                                               const int32_t* __restrict__ gdof,
                                               const double* __restrict__ X,
                                               double* __restrict__ Y,
                                               const int32_t* __restrict__ rlist) {
  constexpr int KPT = (3321 + 255) / 256;
  __shared__ double Kf[BMV_KC * B64_LDK];
  __shared__ int32_t sg[2][BMV_KC];
  const int nres = __builtin_amdgcn_readfirstlane(rlist[64]);
  if (nres == 0) return;  // the common case: no column needs a residual
  const int t = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int l = t & 63;
  for (int q = t; q < 3 * 81; q += 256) Kf[(81 + q / 81) * B64_LDK + q % 81] = 0.0;
  if (t >= 81 && t < BMV_KC) { sg[0][t] = 0; sg[1][t] = 0; }
  uint32_t kaddr[KPT];
#pragma unroll
  for (int i = 0; i < KPT; i++) {
    const int q = t + 256 * i;
    const int c = q < 3321 ? tri_col(q) : 0;
    const int r = q < 3321 ? q - c * (c + 1) / 2 : 0;
    kaddr[i] = (uint32_t)(c * B64_LDK + r) | ((uint32_t)(r * B64_LDK + c) << 16);
  }
  int64_t e = blockIdx.x;
  double kreg[KPT];
  int32_t greg = 0;
  if (e < nelmt) {
    const double* src = KP + e * SGEO_KPACK;
#pragma unroll
    for (int i = 0; i < KPT; i++) {
      const int q = t + 256 * i;
      kreg[i] = q < 3321 ? src[q] : 0.0;
    }
    if (t < 81) greg = gdof[e * 81 + t];
  }
  if (t < 81) sg[0][t] = greg;
  int cur = 0;
  for (; e < nelmt; e += gridDim.x) {
#pragma unroll
    for (int i = 0; i < KPT; i++) {
      if (t + 256 * i < 3321) {
        Kf[kaddr[i] & 0xffffu] = kreg[i];
        Kf[kaddr[i] >> 16] = kreg[i];
      }
    }
    __syncthreads();  // K_e and its gdof visible
    const int64_t en = e + gridDim.x;
    if (en < nelmt) {  // next element's K and gdof, in flight during the MFMAs
      const double* src = KP + en * SGEO_KPACK;
#pragma unroll
      for (int i = 0; i < KPT; i++) {
        const int q = t + 256 * i;
        kreg[i] = q < 3321 ? src[q] : 0.0;
      }
      if (t < 81) greg = gdof[en * 81 + t];
    }
    bmv64_element(e, nres, B, X, Y, rlist, Kf, sg[cur], w, l);
    if (t < 81) sg[cur ^ 1][t] = greg;
    __syncthreads();  // Kf free for the next element, its gdof visible
    cur ^= 1;
  }
}

// At a residual step: INNER columns due for a replacement become REPLACE
// (their last iteration left r_{k+1}, rz_prev = r_k.z_k and a pending beta,
// which the FP64 residual's finalize recomputes), and the columns that need
// an FP64 residual now (START, REPLACE) form the residual list, in column
// order: rlist[0..nres-1], rlist[64] = nres, rslot[j] = column j's place.
// One wave (B <= 64).
__global__ __launch_bounds__(64) void k_bpromote(int B, int32_t* __restrict__ cst,
                                                 BCol* __restrict__ bc,
                                                 int32_t* __restrict__ rlist,
                                                 int32_t* __restrict__ rslot) {
  const int j = threadIdx.x;
  bool want = false;
  if (j < B) {
    int st = cst[j];
    if (st == BCOL_INNER && bc[j].want_rep) {
      st = BCOL_REPLACE;
      cst[j] = st;
      bc[j].want_rep = 0;
    }
    want = st == BCOL_START || st == BCOL_REPLACE;
  }
  const unsigned long long m = __ballot(want);
  const int slot = __popcll(m & ((1ull << j) - 1ull));
  if (want) {
    rlist[slot] = j;
    rslot[j] = slot;
  }
  if (j == 0) rlist[64] = __popcll(m);
}

// load[g][j] = ext[g] + body[g][j] (load(0)=0) for active columns
__global__ void k_bload(int64_t n1, int B, const double* __restrict__ ext,
                        const double* __restrict__ body, double* __restrict__ load,
                        const int32_t* __restrict__ active) {
  const int64_t n = n1 * B;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t g = q / B;
    const int j = (int)(q - g * B);
    if (!active[j]) continue;
    load[q] = (g == 0) ? 0.0 : ext[g] + body[q];
  }
}

// body[g][j] += its element body loads (element order) unless the column's
// trial converged or is on its last iteration (src/slope.F90:380-384)
__global__ void k_bbody_assemble(int64_t n1, int B, int32_t nel,
                                 const int32_t* __restrict__ rowptr,
                                 const int32_t* __restrict__ slots,
                                 const double* __restrict__ BL,
                                 double* __restrict__ body,
                                 const int32_t* __restrict__ active,
                                 const int32_t* __restrict__ is_last,
                                 const PlasticScalars* __restrict__ ps) {
  const int64_t n = n1 * B;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t g = q / B;
    const int j = (int)(q - g * B);
    if (!active[j] || is_last[j] || ps[j].nl_isconv) continue;
    if (g == 0) { body[q] = 0.0; continue; }
    double acc = body[q];
    const double* blj = BL + (int64_t)j * nel * 81;
    for (int32_t w = rowptr[g]; w < rowptr[g + 1]; w++) acc = acc + blj[slots[w]];
    body[q] = acc;
  }
}

// column j of an interleaved [n1][B] array: set from src (contiguous n1,
// NULL = zero) or copy out to dst (contiguous)
__global__ void k_col_io(int64_t n1, int B, int j, double* __restrict__ a,
                         const double* __restrict__ src, double* __restrict__ dst) {
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n1;
       g += (int64_t)gridDim.x * blockDim.x) {
    if (dst) dst[g] = a[g * B + j];
    else a[g * B + j] = src ? src[g] : 0.0;
  }
}

// FP32 copy of an FP64 vector
__global__ void k_to_f32(int64_t n, const double* __restrict__ a,
                         float* __restrict__ b) {
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n;
       g += (int64_t)gridDim.x * blockDim.x)
    b[g] = (float)a[g];
}

// --------------------------------------------------------------------------
// launch wrappers
// --------------------------------------------------------------------------
static inline unsigned grid_stride(int64_t n) {
  const int64_t b = (n + 255) / 256;
  return (unsigned)(b < 65536 ? (b > 0 ? b : 1) : 65536);
}

static inline int bmv_threads(int B) {
  int t = 81 * B;
  if (t > 256) t = 256;
  t = (t + 63) / 64 * 64;
  return t < 64 ? 64 : t;
}

// Launch geometry of the persistent MFMA product: blocks per CU (at most 3:
// the kernel is built for 3 waves per SIMD, at most 168 VGPRs) and the
// XCD-aware element split (nxcd 8) or a plain grid-stride walk (nxcd 1).
void launch_bmv_mfma_f32(hipStream_t s, int32_t nelmt, int B, int n_cu, BmvGeom geom,
                         const float* KP, const int32_t* gdof, const int32_t* eorder,
                         const float* P, int64_t nv, float* Y, double* edot,
                         const int32_t* cst, const BCol* bc, int want_mask) {
  const int nx = geom.xcd_split ? BMV_XCD : 1;
  const int bpc = geom.blocks_per_cu < 1 ? 1 : geom.blocks_per_cu > 4 ? 4 : geom.blocks_per_cu;
  int64_t g = (int64_t)n_cu * bpc;
  const int64_t need = ((int64_t)nelmt + nx - 1) / nx * nx;
  if (g > need) g = need;
  g = (g + nx - 1) / nx * nx;  // a multiple of the XCD count
  const dim3 grid((unsigned)g);
  if (B >= 64)
    hipLaunchKernelGGL(k_bmv_mfma<4>, grid, dim3(256), 0, s, nelmt, B, nx, KP, gdof,
                       eorder, P, nv, Y, edot, cst, bc, want_mask);
  else if (B == 32)
    hipLaunchKernelGGL(k_bmv_mfma<2>, grid, dim3(256), 0, s, nelmt, B, nx, KP, gdof,
                       eorder, P, nv, Y, edot, cst, bc, want_mask);
  else
    hipLaunchKernelGGL(k_bmv_mfma<1>, grid, dim3(256), 0, s, nelmt, B, nx, KP, gdof,
                       eorder, P, nv, Y, edot, cst, bc, want_mask);
}

// FP64 residual product: persistent, 2 blocks per CU (60 KB of LDS each);
// every block returns at once when the residual list is empty
void launch_bmv_f64(hipStream_t s, int32_t nelmt, int B, int n_cu, const double* KP,
                    const int32_t* gdof, const double* X, double* Y,
                    const int32_t* rlist) {
  int64_t g = (int64_t)n_cu * 2;
  if (g > nelmt) g = nelmt;
  if (g < 1) g = 1;
  hipLaunchKernelGGL(k_bmv64, dim3((unsigned)g), dim3(256), 0, s, nelmt, B, KP, gdof, X,
                     Y, rlist);
}

void launch_bpromote(hipStream_t s, int B, int32_t* cst, BCol* bc, int32_t* rlist,
                     int32_t* rslot) {
  hipLaunchKernelGGL(k_bpromote, dim3(1), dim3(64), 0, s, B, cst, bc, rlist, rslot);
}

void launch_bload(hipStream_t s, int64_t n1, int B, const double* ext,
                  const double* body, double* load, const int32_t* active) {
  hipLaunchKernelGGL(k_bload, dim3(grid_stride(n1 * B)), dim3(256), 0, s, n1, B,
                     ext, body, load, active);
}

void launch_col_io(hipStream_t s, int64_t n1, int B, int j, double* a,
                   const double* src, double* dst) {
  hipLaunchKernelGGL(k_col_io, dim3(grid_stride(n1)), dim3(256), 0, s, n1, B, j,
                     a, src, dst);
}

void launch_to_f32(hipStream_t s, int64_t n, const double* a, float* b) {
  hipLaunchKernelGGL(k_to_f32, dim3(grid_stride(n)), dim3(256), 0, s, n, a, b);
}

void launch_bbody_assemble(hipStream_t s, int64_t n1, int B, int32_t nel,
                           const int32_t* rowptr, const int32_t* slots,
                           const double* BL, double* body, const int32_t* active,
                           const int32_t* is_last, const PlasticScalars* ps) {
  hipLaunchKernelGGL(k_bbody_assemble, dim3(grid_stride(n1 * B)), dim3(256), 0, s,
                     n1, B, nel, rowptr, slots, BL, body, active, is_last, ps);
}

}  // namespace sgeo
