// A panel's diagonal block and the rows below it on the matrix cores (gfx950).
//
// diag_potrf_inv factors and inverts a diagonal block of up to 128 columns in LDS by one
// workgroup, for k_small_fronts; block_substitute solves sixteen rows a wave against a factored block without leaving the wave's registers.
#pragma once

#include "gemm_kernels.hpp"

namespace fc {

constexpr int DB = 16;  // columns of a diagonal-block step: one MFMA tile

// d = sqrt(p) and rd = 1 / sqrt(p), both to within a rounding or so: the hardware's estimate, one
// coupled Newton step on (sqrt p, 1 / (2 sqrt p)), then each corrected by its own residual.
__device__ __forceinline__ void root_pair(double p, double& d, double& rd) {
  const double y = __builtin_amdgcn_rsq(p);
  double s = p * y, h = 0.5 * y;
  const double e = fma(-h, s, 0.5);
  s = fma(s, e, s);
  h = fma(h, e, h);
  d = fma(fma(-s, s, p), h, s);
  const double r = h + h;
  rd = fma(fma(-d, r, 1.0), r, r);
}

// The h x h block (h <= NMAX, whole steps of DB columns) at S[0.., 0..], factored with the
// reference's pivot test (cholesky.rs:1161) and inverted, in FP64 (EXACT: the quotients by the
// pivot's root rounded as divisions, for FP64 storage). On entry S holds A in its lower
// triangle over the 16 nb x 16 nb square (nb = ceil(h / 16)), zeros above it, and an identity in
// the rows and columns past h; on return S[i][j] = L(i, j) for i >= j, S[k][i] = Linv(i, k) for
// i > k and xd[i] = Linv(i, i). IB is 16 x 17 of LDS. NW waves call it; it ends on a barrier.
//
// A block of 128 columns is a chain of 128 dependent pivots, so what sets its time is the
// latency of a step. Each step of 16 columns is taken by every wave on its own copy of the 16 x 16
// pivot block (lanes 0..15, a row a lane) with 48 other rows in the wave's other lanes: the
// rows below, and, since the rows of an identity appended below the block become the columns of
// the inverse, the identity's rows too. One instruction stream then gives L, the rows below it by
// true substitution and the inverse, with the pivot column broadcast by scalar reads (no
// LDS round trip and no barrier inside a step). Row c of the identity is nonzero from column c
// on, so its entries live in the upper triangle of S and each step has 16 nb rows to take. The
// trailing update S(r, j) -= P(r) L(j)^T (rows below, and identity rows already started) goes
// through the 16x16x4 MFMA, a tile a wave, NT tiles of a wave in flight at once.
template <int NMAX, int NW, bool EXACT>
__device__ inline void diag_potrf_inv(double (*S)[NMAX + 1], double* xd, double (*IB)[DB + 1], int h, int tid,
                                      const double* __restrict__ dg, int64_t col,
                                      unsigned long long* __restrict__ fail) {
  constexpr int ROWS = 64 - DB;  // rows a wave takes beside the pivot block
  static_assert(NW * ROWS >= NMAX, "a step's rows fit the workgroup's waves");
  constexpr int NT = 3;
  const int lane = tid & 63, wave = tid >> 6;
  const int nb = (h + DB - 1) / DB;
  for (int kb = 0; kb < nb; ++kb) {
    const int c0 = DB * kb;
    // slot 0..15: the identity's rows c0 ..; then the block's other rows in order
    const int slot = wave * ROWS + lane - DB;
    const bool piv = lane < DB, ident = !piv && slot < DB, act = !piv && slot < DB * nb;
    const int row = piv ? c0 + lane : (slot - DB < c0 ? slot - DB : slot);  // (unused for the identity)
    const bool work = wave * ROWS < DB * nb;  // uniform
    double a[DB];
    if (work) {
      const double* src = S[(piv || (act && !ident)) ? row : c0];
#pragma unroll
      for (int t = 0; t < DB; ++t) a[t] = src[c0 + t];
      if (ident)
#pragma unroll
        for (int t = 0; t < DB; ++t) a[t] = t == slot ? 1.0 : 0.0;
    }
    const double dl = (lane < DB && c0 + lane < h) ? fabs(dg[c0 + lane]) : 0.0;
    __syncthreads();  // every copy of the pivot block read before it is overwritten
    if (work) {
double pv = 0.0;  // lane j: pivot j
      double p = readlane_d(a[0], 0), d, rd;
      root_pair(p, d, rd);
#pragma unroll
      for (int j = 0; j < DB; ++j) {
        pv = lane == j ? p : pv;
        double l = a[j] * rd;
        if constexpr (EXACT) l = fma(fma(-l, d, a[j]), rd, l);  // a[j] / d to a rounding
        a[j] = l;
        // the next pivot first: its reciprocal root is the step's dependent chain, the other
        // columns' updates fill it (one scheduling region a step: the broadcasts of several steps
        // together do not fit the scalar registers)
        if (j + 1 < DB) {
          a[j + 1] = fma(-l, readlane_d(l, j + 1), a[j + 1]);
          p = readlane_d(a[j + 1], j + 1);
          root_pair(p, d, rd);
        }
#pragma unroll
        for (int k = j + 2; k < DB; ++k) a[k] = fma(-l, readlane_d(l, k), a[k]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (wave == 0 && lane < DB && c0 + lane < h && (!(pv > PIVOT_TOL * dl) || !isfinite(pv)))
        atomicMin(fail, (unsigned long long)(col + c0 + lane));
      if (ident) {
#pragma unroll
        for (int t = 0; t < DB; ++t) {
          IB[slot][t] = a[t];
          if (t > slot) S[c0 + slot][c0 + t] = a[t];
          if (t == slot) xd[c0 + slot] = a[t];
        }
      } else if (act || (piv && wave == 0)) {
#pragma unroll
        for (int t = 0; t < DB; ++t)
          if (!piv || t <= lane) S[row][c0 + t] = a[t];
      }
    }
    __syncthreads();
    // tiles (r, j), j > kb: rows r >= j (below) and r <= kb (the identity's)
    const int nj = nb - 1 - kb;
    const int tiles = nj * (nj + 1) / 2 + nj * (kb + 1);
    for (int t0 = wave; t0 < tiles; t0 += NW * NT) {
      int rb[NT], jb[NT];
      v4d acc[NT];
#pragma unroll
      for (int q = 0; q < NT; ++q) {
        int t = min(t0 + NW * q, tiles - 1), j = 0;
        while (t >= (kb + 1) + (nj - j)) t -= (kb + 1) + (nj - j), ++j;  // column kb + 1 + j
        jb[q] = kb + 1 + j;
        rb[q] = t <= kb ? t : jb[q] + t - (kb + 1);
        acc[q] = v4d{0, 0, 0, 0};
      }
      const int r = lane & 15, g = lane >> 4;
      double fj[NT][4], fi[NT][4];
#pragma unroll
      for (int q = 0; q < NT; ++q)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          fj[q][s] = S[DB * jb[q] + r][c0 + 4 * s + g];
          fi[q][s] = rb[q] == kb ? IB[r][4 * s + g] : S[DB * rb[q] + r][c0 + 4 * s + g];
        }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int q = 0; q < NT; ++q) acc[q] = Mma<double>::step(fj[q][s], fi[q][s], acc[q]);
#pragma unroll
      for (int q = 0; q < NT; ++q)
        if (t0 + NW * q < tiles)
#pragma unroll
          for (int v = 0; v < 4; ++v) S[DB * rb[q] + r][DB * jb[q] + g + 4 * v] -= acc[q][v];
    }
    __syncthreads();
  }
}

// X L11^T = B for sixteen rows a wave, by blocks of 16 columns in the wave's registers:
//   X_k = (B_k - sum_{j < k} X_j L_kj^T) L_kk^-T
// x[k] holds B_k on entry and X_k on return, in the MFMA's output layout (entry v of a lane: row
// lane % 16, column 16 k + row(lane, v)). That layout is also the layout of the next product's
// row operand when the products sum their 16 columns in the order row(lane, s), so no value moves
// between lanes. Lop(k, j, s), Xop(k, s) and Dop(k, s) return the lane's column operand: entry
// (lane % 16, row(lane, s)) of L_kj, L_kk^-1 and L_kk. REFINE corrects each X_k once against L_kk
// (a product with an explicit inverse alone is not backward stable).
template <typename M, int NBK, bool REFINE, class FL, class FX, class FD>
__device__ __forceinline__ void block_substitute(typename Mma<M>::acc_t (&x)[NBK], int nb, FL Lop, FX Xop, FD Dop) {
  typedef typename Mma<M>::acc_t acc_t;
#pragma unroll
  for (int k = 0; k < NBK; ++k) {
    if (k >= nb) break;
    acc_t b = x[k];
#pragma unroll
    for (int j = 0; j < k; ++j)
#pragma unroll
      for (int s = 0; s < 4; ++s) b = Mma<M>::step(-Lop(k, j, s), x[j][s], b);
    acc_t y = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; ++s) y = Mma<M>::step(Xop(k, s), b[s], y);
    if constexpr (REFINE) {
#pragma unroll
      for (int s = 0; s < 4; ++s) b = Mma<M>::step(-Dop(k, s), y[s], b);
#pragma unroll
      for (int s = 0; s < 4; ++s) y = Mma<M>::step(Xop(k, s), b[s], y);
    }
    x[k] = y;
  }
}

}  // namespace fc
