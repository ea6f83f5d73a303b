// Kernels of the multifrontal numeric phase (gfx950). All are work-list kernels: workgroup b
// runs item items[item0 + b] of its launch; one launch covers one level of the front tree.
//
// Per level: the children's update matrices are added into the fronts' L parts (extend-add);
// each front is factored by panels of 128 columns, left-looking inside the front like the
// reference's panel loop (cholesky.rs:1138-1186, panels of 64 there): the panel minus its
// products with the front's earlier columns (MFMA GEMM), its diagonal block factored with the
// pivot test of cholesky.rs:1161, the rows below solved against it; then the front's update
// matrix U = -L21 L21^T (MFMA SYRK) and the children's update matrices added into it. The
// dense kernels are in gemm_kernels.hpp; these are the entry, scaling and extend-add steps.
#pragma once

#include "device.hpp"

namespace fc {

// ------------------------------------------------------------------------------------------
// Matrix entries into the factor storage

template <typename T>
__global__ void k_scatter_a(const double* __restrict__ aval, const int64_t* __restrict__ a_pos, int64_t nnz,
                            T* __restrict__ L) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < nnz; e += (int64_t)gridDim.x * blockDim.x)
    L[a_pos[e]] = (T)aval[e];
}

__global__ void k_gather_diag(const double* __restrict__ aval, const int64_t* __restrict__ diag_src, int64_t n,
                              double* __restrict__ diag) {
  for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < n; c += (int64_t)gridDim.x * blockDim.x)
    diag[c] = diag_src[c] >= 0 ? aval[diag_src[c]] : 0.0;
}

// Per front: the exponent e of the smallest power of two with sqrt(A_ii) <= 2^e over the
// front's rows. For an SPD matrix every factor entry satisfies |L_ij| <= sqrt(A_ii) (row i of L
// has squared norm A_ii), so 2^-e scales the front's columns into [-1, 1]. 0 when no row has a
// positive finite diagonal.
__global__ __launch_bounds__(256) void k_front_scale(const FrontDev* __restrict__ fronts, const int32_t* __restrict__ rows,
                                                     const double* __restrict__ diag, int64_t nf,
                                                     int32_t* __restrict__ fexp) {
  __shared__ double red[4];
  for (int64_t f = blockIdx.x; f < nf; f += gridDim.x) {
    const FrontDev F = fronts[f];
    const int32_t* fr = rows + F.rows_off;
    double mx = 0.0;
    for (int i = threadIdx.x; i < F.m; i += blockDim.x) {
      const double d = diag[fr[i]];
      if (isfinite(d) && d > mx) mx = d;
    }
    for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
      mx = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
      int e = 0;
      if (mx > 0.0) (void)frexp(sqrt(mx), &e);
      fexp[f] = e;
    }
    __syncthreads();
  }
}

template <typename T>
__global__ void k_fill(T* __restrict__ p, int64_t len, T v) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < len; e += (int64_t)gridDim.x * blockDim.x) p[e] = v;
}

// ------------------------------------------------------------------------------------------
// Extend-add: the workgroup owns the parent's columns [a, b) and adds every child's update
// matrix entries that land there, child after child (in increasing order), so each entry
// receives its contributions in a fixed order and no two workgroups write the same entry.
// Item: f, a, b, and at ranges[c .. c + d) the children's column runs that land in [a, b),
// window of at most EA_COLS parent columns after window, children in increasing order within a
// window (children with none are not listed; the runs are found when the launches are planned).
//
// Wave v takes the window's columns win + v and win + v + 4, through every child: a column's entries
// stay with one wave, whose memory operations are in order, so the children need no barrier. Lanes
// run along the child's rows, both columns together (one read of the row map for the two), EA_BATCH
// rows of each in flight. Bound: HBM, 12 bytes a child's FP32 entry (20 FP64) and the row maps; in
// levels of few columns, the chain of a workgroup's ranges (three memory round trips each). Taken
// as one flat range of 8 columns by the whole workgroup, with a barrier after each child and
// selects to find an entry's column, a launch of the cantilever's FP64 factor took 64 us (now 7), of
// the 28^3 cube's 91 us (48), of the 40^3 cube's mixed one 136 us (97).
template <typename T>
__global__ __launch_bounds__(256) void k_extend_add(const Item* __restrict__ items, const EaRange* __restrict__ ranges,
                                                    const FrontDev* __restrict__ fronts,
                                                    const int32_t* __restrict__ rel, T* L, const T* __restrict__ U,
                                                    T* Uw) {
  // U (children, read) and Uw (this front, written) are disjoint blocks of one arena
  const Item it = items[blockIdx.x];
  const FrontDev P = fronts[it.f];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t pmu = P.m - P.w;
  for (int q = it.c; q < it.c + it.d; ++q) {
    const EaRange rg = ranges[q];
    const int32_t* r = rel + rg.rel;
    // the child's columns that land on the wave's two: lane l looks at column jc0 + l
    const int mine = lane < rg.jc1 - rg.jc0 ? r[rg.jc0 + lane] - rg.win - wave : -1;
    const uint64_t m0 = __ballot(mine == 0), m1 = __ballot(mine == 4);
    if (!(m0 | m1)) continue;
    int jc[2];
    T* d[2];
    const T* s[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint64_t m = h ? m1 : m0;
      const int p = rg.win + wave + 4 * h;
      jc[h] = m ? rg.jc0 + __ffsll((unsigned long long)m) - 1 : rg.cmu;  // none: no row
      d[h] = p < P.w ? L + P.lpos + (int64_t)p * P.ld : Uw + P.upos + (int64_t)(p - P.w) * pmu - P.w;
      s[h] = U + rg.u + (int64_t)min(jc[h], rg.cmu - 1) * rg.cmu;
    }
    // rows from the first column's on; a lane's rows past the range read its last one (in bounds)
    // and store nothing
    for (int i0 = min(jc[0], jc[1]) + lane; i0 < rg.cmu; i0 += 64 * EA_BATCH) {
      int ri[EA_BATCH];
      T sv[2][EA_BATCH], dv[2][EA_BATCH];
#pragma unroll
      for (int k = 0; k < EA_BATCH; ++k) {
        const int i = min(i0 + 64 * k, rg.cmu - 1);
        ri[k] = r[i];
#pragma unroll
        for (int h = 0; h < 2; ++h) sv[h][k] = i >= jc[h] ? s[h][i] : T(0);
      }
#pragma unroll
      for (int k = 0; k < EA_BATCH; ++k)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int i = i0 + 64 * k;
          dv[h][k] = (i < rg.cmu && i >= jc[h]) ? d[h][ri[k]] : T(0);
        }
#pragma unroll
      for (int k = 0; k < EA_BATCH; ++k)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int i = i0 + 64 * k;
          if (i < rg.cmu && i >= jc[h]) d[h][ri[k]] = dv[h][k] + sv[h][k];
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the next child's loads stay behind these stores
  }
}

}  // namespace fc
