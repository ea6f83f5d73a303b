// Dense kernels of a front's partial factorization on the matrix cores (gfx950).
//
// The Schur products of the numeric phase are items of one kernel, k_gemm (k_gemm_b16 in the mixed form):
//   panel update   L[r.., c0..c1) -= L[r.., 0..c0) L[c0..c1, 0..c0)^T      (G_SUB)
//   update matrix  U[i.., j..)     = -L[W+i.., 0..W) L[W+j.., 0..W)^T        (G_NEG)
// (a panel's diagonal block and the rows below it are panel_kernels.hpp's). A launch with few
// output tiles is split along k: each piece writes its partial tile (G_PART) and k_reduce_parts adds
// the pieces in a fixed order, so results do not depend on scheduling.
//
// Tile: TB x TB per workgroup of 4 waves (128, or 64 in launches of few tiles: GB_FEW), each wave a
// quarter as blocks of the 16x16x4 MFMA; k staged in LDS (16 at a time, 32 for the smaller tile),
// the next stage prefetched into registers while the current one is multiplied (one barrier a
// stage). The MFMA's first operand is taken from the j side so that a lane's output column index
// runs along C's rows: 16 lanes store 16 consecutive rows of a column (coalesced, C is column-major).
#pragma once

#include "device.hpp"

namespace fc {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int GB = 128;  // tile edge
constexpr int GB2 = 64;  // tile edge of launches with few tiles
constexpr int GK = 16;   // k per LDS stage
constexpr int NB = 128;  // panel width of the factorization (columns of a diagonal block)

enum GemmMode : int32_t { G_SUB = 0, G_NEG = 1, G_PART = 2 };
enum GemmSrc : int8_t { S_L = 0, S_U = 1, S_PART = 2 };

struct GemmItem {
  int64_t a, b, c;        // element offsets: A(i, k) = A[a + k lda + i], B(j, k), C(i, j) = C[c + j ldc + i]
  int32_t lda, ldb, ldc;
  int32_t m, n, k;        // rows of C (and A), columns of C (rows of B), depth
  int32_t mode;           // GemmMode
  int32_t diag;           // store C(i, j) only when i - j + diag >= 0
  int8_t csrc, pad0, pad1, pad2;
  int32_t front;          // the front both operands come from (its scale in the mixed form)
};
static_assert(sizeof(GemmItem) == 64, "GemmItem layout");

struct ReduceItem {
  int64_t c;              // output offset in csrc
  int64_t part0;          // first partial tile (tile x tile, column-major) in the split-K workspace
  int32_t ldc, m, n, mode, diag, parts;
  int8_t csrc, pad0, pad1, pad2;
  int32_t tile;           // edge of the partial tiles (TB)
};
static_assert(sizeof(ReduceItem) == 48, "ReduceItem layout");

template <typename T>
struct Mma;
template <>
struct Mma<double> {
  typedef v4d acc_t;
  static __device__ __forceinline__ acc_t step(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // output v of lane l is D(row(l, v), l % 16) (measured on gfx950)
  static __device__ __forceinline__ int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};
template <>
struct Mma<float> {
  typedef v4f acc_t;
  static __device__ __forceinline__ acc_t step(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

template <typename T, int TB>
__global__ __launch_bounds__(256, 2) void k_gemm(const GemmItem* __restrict__ items, T* L, T* U, T* Part) {
  constexpr int PAD = 4;
  constexpr int KS = TB == GB ? GK : 2 * GK;  // k per LDS stage (the same loads a thread either way)
  constexpr int NQ = TB / 32;                 // 16 x 16 blocks of a wave's quarter, each way
  constexpr int LK = 256 / TB, LR = KS / LK;  // the loader: a thread one row, every LK-th k
  __shared__ T As[2][KS][TB + PAD];
  __shared__ T Bs[2][KS][TB + PAD];
  const GemmItem it = items[blockIdx.x];
  const T* __restrict__ A = L + it.a;
  const T* __restrict__ B = L + it.b;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wi = (wave >> 1) * (TB / 2), wj = (wave & 1) * (TB / 2);
  const int lrow = tid & (TB - 1), lk = tid / TB;
  const bool arow = lrow < it.m, brow = lrow < it.n;
  T ra[LR], rb[LR];
  auto load = [&](int ks) {
#pragma unroll
    for (int r = 0; r < LR; ++r) {
      const int k = ks + lk + LK * r;
      const bool kin = k < it.k;
      ra[r] = (arow && kin) ? A[(int64_t)k * it.lda + lrow] : T(0);
      rb[r] = (brow && kin) ? B[(int64_t)k * it.ldb + lrow] : T(0);
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int r = 0; r < LR; ++r) {
      As[buf][lk + LK * r][lrow] = ra[r];
      Bs[buf][lk + LK * r][lrow] = rb[r];
    }
  };
  typename Mma<T>::acc_t acc[NQ][NQ];
#pragma unroll
  for (int bi = 0; bi < NQ; ++bi)
#pragma unroll
    for (int bj = 0; bj < NQ; ++bj) acc[bi][bj] = typename Mma<T>::acc_t{0, 0, 0, 0};
  const int stages = (it.k + KS - 1) / KS;
  load(0);
  store(0);
  __syncthreads();
  for (int s = 0; s < stages; ++s) {
    const int cur = s & 1;
    if (s + 1 < stages) load((s + 1) * KS);
#pragma unroll
    for (int kk = 0; kk < KS; kk += 4) {
      T fj[NQ], fi[NQ];
#pragma unroll
      for (int b = 0; b < NQ; ++b) {
        fj[b] = Bs[cur][kk + (lane >> 4)][wj + 16 * b + (lane & 15)];
        fi[b] = As[cur][kk + (lane >> 4)][wi + 16 * b + (lane & 15)];
      }
#pragma unroll
      for (int bi = 0; bi < NQ; ++bi)
#pragma unroll
        for (int bj = 0; bj < NQ; ++bj) acc[bi][bj] = Mma<T>::step(fj[bj], fi[bi], acc[bi][bj]);
    }
    if (s + 1 < stages) store(cur ^ 1);
    __syncthreads();
  }
  // acc[bi][bj][v] = C(wi + 16 bi + lane % 16, wj + 16 bj + row(lane, v))
  const int il = lane & 15;
  if (it.mode == G_PART) {
    T* P = Part + it.c;
#pragma unroll
    for (int bi = 0; bi < NQ; ++bi)
#pragma unroll
      for (int bj = 0; bj < NQ; ++bj)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int i = wi + 16 * bi + il, j = wj + 16 * bj + Mma<T>::row(lane, v);
          P[(int64_t)j * TB + i] = acc[bi][bj][v];
        }
    return;
  }
  T* C = (it.csrc == S_L ? L : U) + it.c;
  // By row blocks: G_SUB reads the block's 16 old values first, every load in flight at
  // once, through a buffer resource (a tile spans far below 2 GiB of its array; an entry outside
  // the tile reads 0 from the range check and is not stored). An update and its load in one
  // branch made the compiler wait for each load in turn: 64 round trips a tile.
  const auto rc = raw_rsrc(C);
  const uint32_t ldcb = (uint32_t)it.ldc * sizeof(T);
#pragma unroll
  for (int bi = 0; bi < NQ; ++bi) {
    T old[NQ][4] = {};
    if (it.mode == G_SUB) {
#pragma unroll
      for (int bj = 0; bj < NQ; ++bj)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int i = wi + 16 * bi + il, j = wj + 16 * bj + Mma<T>::row(lane, v);
          const bool in = i < it.m && j < it.n && i - j + it.diag >= 0;
          old[bj][v] = buf_load<T>(rc, in ? (uint32_t)(i * sizeof(T)) : 0x80000000u, (uint32_t)j * ldcb);
        }
    }
#pragma unroll
    for (int bj = 0; bj < NQ; ++bj)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = wi + 16 * bi + il, j = wj + 16 * bj + Mma<T>::row(lane, v);
        if (i < it.m && j < it.n && i - j + it.diag >= 0) {
          const T x = acc[bi][bj][v];
          C[(int64_t)j * it.ldc + i] = it.mode == G_SUB ? old[bj][v] - x : -x;
        }
      }
  }
}

// ------------------------------------------------------------------------------------------
// The Schur products of the mixed form on the 16x16x32 BF16 matrix cores with FP32
// accumulation. Both operands of a product come from one front, whose columns are scaled by
// that front's power of two 2^-fexp[front] (which bounds them by 1: |L_ij| <= sqrt(A_ii) for an
// SPD matrix); the result is scaled back exactly. With TERMS = 3 each scaled value x is carried
// as hi = bf16(x) and lo = bf16(x - hi) and a product is hi*hi + hi*lo + lo*hi, about 16
// significant bits; TERMS = 1 keeps hi*hi.
//
// The BF16 copies are written once per panel, by the kernels that finish it (the diagonal
// block's by k_potrf_blk, the rows below by k_trsm<float, true>), in a k-chunked
// layout: entry (i, j) at bpos + ((j / 32) ld + i) 32 + j % 32, zero past the front's width up to
// a multiple of 32, so a 128-row x 32-column stage of an operand is one contiguous 8 KB block
// per copy and a product's last stage needs no bounds. The product kernel moves it into LDS with the
// direct global-to-LDS loads (no registers on the way), 1 KB (16 rows) per wave instruction,
// while the previous stage is multiplied. Tiles, modes and split-k pieces are those of k_gemm
// (128 x 128, 4 waves of 64 x 64).
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
constexpr int BK = 32;  // k per stage: one MFMA depth, one chunk of the copies

// LDS address of a shared-memory pointer, and a 16-byte LDS read issued as an instruction the
// compiler does not track: it would otherwise wait for every direct global-to-LDS load in
// flight before any LDS read. The caller waits (lgkm_wait) before using the values.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
template <int OFF>
__device__ __forceinline__ v8bf lds_read16(uint32_t a) {
  v8bf r;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(a), "i"(OFF));
  return r;
}

// Fragments of NQ 16-row blocks (1 KB apart) from LDS address a.
template <int NQ>
__device__ __forceinline__ void read_rows(v8bf (&f)[NQ], uint32_t a) {
  f[0] = lds_read16<0>(a);
  f[1] = lds_read16<1024>(a);
  if constexpr (NQ == 4) {
    f[2] = lds_read16<2048>(a);
    f[3] = lds_read16<3072>(a);
  }
}

// Wait until the fragments read above are in their registers (the same statement that names them
// as changed, so that nothing uses one before).
__device__ __forceinline__ void frags_wait(v8bf (&a)[2], v8bf (&b)[2]) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a[0]), "+v"(a[1]), "+v"(b[0]), "+v"(b[1]));
}
__device__ __forceinline__ void frags_wait(v8bf (&a)[4], v8bf (&b)[4]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]));
}
__device__ __forceinline__ void frags_wait(v8bf (&a)[2], v8bf (&b)[2], v8bf (&c)[2], v8bf (&d)[2]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(a[0]), "+v"(a[1]), "+v"(b[0]), "+v"(b[1]), "+v"(c[0]), "+v"(c[1]), "+v"(d[0]), "+v"(d[1]));
}
__device__ __forceinline__ void frags_wait(v8bf (&a)[4], v8bf (&b)[4], v8bf (&c)[4], v8bf (&d)[4]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]),
                 "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3]), "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3]));
}

// A product's tile (TB x TB) with both operands staged through LDS by direct loads, 64 KB of
// stages for three terms (two workgroups share a CU): two of a 128 x 128 tile, four of a 64 x 64
// one, whose launches have few tiles and so wait on each stage's load rather than on the matrix
// cores.
//
// Stage buffer: copy t of A (TB rows x 32 k), then copy t of B. A row's four 16-byte chunks sit
// in the order chunk ^ (row / 2 % 4), the arrangement under which the fragment reads measure
// free of bank conflicts on gfx950; a wave's direct load fills 1 KB = 16 rows, lane l taking
// the chunk of LDS slot l.
// Rows past the tile's m (n) load the last row of the tile (in bounds); their products land in
// entries that are not stored. The copies are zero past the front's width, so the last stage
// needs no k bound.
template <int TERMS, int TB>
__global__ __launch_bounds__(256, 2) void k_gemm_b16(const GemmItem* __restrict__ items, const FrontDev* __restrict__ fronts,
                                                     const __bf16* __restrict__ Lh, const __bf16* __restrict__ Ll,
                                                     float* L, float* U, float* Part, const int32_t* __restrict__ fexp) {
  static_assert(TERMS == 1 || TERMS == 3, "one or three BF16 products");
  constexpr int NS = TERMS == 3 ? 2 : 1;       // hi (and lo) copies of each operand
  constexpr int NQ = TB / 32;                  // 16 x 16 blocks of a wave's quarter, each way
  constexpr int NBUF = TB == GB ? 2 : 4;       // stage buffers: 64 KB of LDS for three terms
  constexpr int CE = TB * BK;                  // elements of one copy of one operand per stage
  constexpr int SE = 2 * NS * CE;              // elements of a stage buffer
  constexpr int PW = 2 * NS * (TB / 16) / 4;   // 1 KB direct loads per wave per stage
  __shared__ __attribute__((aligned(16))) __bf16 S[NBUF * SE];
  const GemmItem it = items[blockIdx.x];
  const FrontDev F = fronts[it.front];
  const int e = fexp[it.front];
  // the operands' first rows and columns in the front, and their origins in the copies
  const int64_t oa = it.a - F.lpos, ob = it.b - F.lpos;
  const int64_t chunk = (int64_t)F.ld * BK;  // elements from one k-chunk of a row to the next
  const int64_t a0 = F.bpos + (oa / F.ld) / BK * chunk + (oa % F.ld) * BK;
  const int64_t b0 = F.bpos + (ob / F.ld) / BK * chunk + (ob % F.ld) * BK;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wi = (wave >> 1) * (TB / 2), wj = (wave & 1) * (TB / 2);
  const int lrow = lane >> 2, lch = (lane & 3) ^ ((lrow >> 1) & 3);  // the row and chunk slot l holds
  auto issue = [&](int s, int buf) {
#pragma unroll
    for (int q = 0; q < PW; ++q) {
      const int g = wave + 4 * q;            // which 1 KB block of the stage: operand, copy, rows
      const int op = g / (NS * TB / 16), t = g / (TB / 16) % NS, rb = g % (TB / 16);
      const int row = rb * 16 + lrow;
      const int64_t src = (op == 0 ? a0 + (int64_t)min(row, it.m - 1) * BK
                                   : b0 + (int64_t)min(row, it.n - 1) * BK) + s * chunk + lch * 8;
      const __bf16* gp = (t == 0 ? Lh : Ll) + src;
      __bf16* lp = S + buf * SE + (op * NS + t) * CE + rb * 16 * BK;
      __builtin_amdgcn_global_load_lds((const void*)gp, (__attribute__((address_space(3))) void*)lp, 16, 0, 0);
    }
  };
  v4f acc[NQ][NQ];
#pragma unroll
  for (int bi = 0; bi < NQ; ++bi)
#pragma unroll
    for (int bj = 0; bj < NQ; ++bj) acc[bi][bj] = v4f{0, 0, 0, 0};
  const int stages = (it.k + BK - 1) / BK;
  // a lane's fragment: row lane % 16 of a 16-row block, k chunk lane / 16 (byte offset in a copy)
  const int fr = lane & 15;
  const uint32_t foff = (uint32_t)(fr * 4 + ((lane >> 4) ^ ((fr >> 1) & 3))) * 16;
  const uint32_t sbase = lds_addr(S);
  auto mul = [&](int buf) {
    const uint32_t ah = sbase + (uint32_t)(buf * SE + wi * BK) * 2 + foff;
    const uint32_t bh = sbase + (uint32_t)(buf * SE + NS * CE + wj * BK) * 2 + foff;
    v8bf fi[NQ], fj[NQ], gi[NQ], gj[NQ];
    read_rows<NQ>(fi, ah);
    read_rows<NQ>(fj, bh);
    if constexpr (TERMS == 3) {
      read_rows<NQ>(gi, ah + CE * 2);
      read_rows<NQ>(gj, bh + CE * 2);
    }
    if constexpr (TERMS == 3) frags_wait(fi, fj, gi, gj);
    else frags_wait(fi, fj);
    if constexpr (TERMS == 3) {
#pragma unroll
      for (int bi = 0; bi < NQ; ++bi)
#pragma unroll
        for (int bj = 0; bj < NQ; ++bj)
          acc[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gj[bj], fi[bi], acc[bi][bj], 0, 0, 0);
#pragma unroll
      for (int bi = 0; bi < NQ; ++bi)
#pragma unroll
        for (int bj = 0; bj < NQ; ++bj)
          acc[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fj[bj], gi[bi], acc[bi][bj], 0, 0, 0);
    }
#pragma unroll
    for (int bi = 0; bi < NQ; ++bi)
#pragma unroll
      for (int bj = 0; bj < NQ; ++bj)
        acc[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fj[bj], fi[bi], acc[bi][bj], 0, 0, 0);
  };
  // NBUF - 1 stages in flight: stage s waits for the wave's own loads up to it (those of the NBUF - 2
  // later stages may be out, PW each; near the end, for all), then meets the others at the
  // barrier, which also frees buffer (s - 1) % NBUF for stage s + NBUF - 1.
#pragma unroll
  for (int s = 0; s < NBUF - 1; ++s)
    if (s < stages) issue(s, s);
  for (int s = 0; s < stages; ++s) {
    if (s + NBUF - 2 < stages) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NBUF - 2) * PW) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (s + NBUF - 1 < stages) issue(s + NBUF - 1, (s + NBUF - 1) % NBUF);
    mul(s % NBUF);
  }
  // acc[bi][bj][v] = C(wi + 16 bi + lane % 16, wj + 16 bj + 4 (lane / 16) + v) / sc^2
  const float unscale = ldexpf(1.0f, 2 * e);
  const int il = lane & 15;
  if (it.mode == G_PART) {
    float* P = Part + it.c;
#pragma unroll
    for (int bi = 0; bi < NQ; ++bi)
#pragma unroll
      for (int bj = 0; bj < NQ; ++bj)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int i = wi + 16 * bi + il, j = wj + 16 * bj + Mma<float>::row(lane, v);
          P[(int64_t)j * TB + i] = acc[bi][bj][v] * unscale;
        }
    return;
  }
  float* C = (it.csrc == S_L ? L : U) + it.c;
  // by row blocks, G_SUB's 16 old values of a block loaded first (as in k_gemm)
  const auto rc = raw_rsrc(C);
  const uint32_t ldcb = (uint32_t)it.ldc * sizeof(float);
#pragma unroll
  for (int bi = 0; bi < NQ; ++bi) {
    float old[NQ][4] = {};
    if (it.mode == G_SUB) {
#pragma unroll
      for (int bj = 0; bj < NQ; ++bj)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int i = wi + 16 * bi + il, j = wj + 16 * bj + Mma<float>::row(lane, v);
          const bool in = i < it.m && j < it.n && i - j + it.diag >= 0;
          old[bj][v] = buf_load<float>(rc, in ? (uint32_t)(i * sizeof(float)) : 0x80000000u, (uint32_t)j * ldcb);
        }
    }
#pragma unroll
    for (int bj = 0; bj < NQ; ++bj)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = wi + 16 * bi + il, j = wj + 16 * bj + Mma<float>::row(lane, v);
        if (i < it.m && j < it.n && i - j + it.diag >= 0) {
          const float x = acc[bi][bj][v] * unscale;
          C[(int64_t)j * it.ldc + i] = it.mode == G_SUB ? old[bj][v] - x : -x;
        }
      }
  }
}

// Sum of the partial tiles of a split product, in order, applied to C as its mode says. Each
// tile is shared by RSPLIT workgroups.
constexpr int RSPLIT = 16;

template <typename T>
__global__ __launch_bounds__(256) void k_reduce_parts(const ReduceItem* __restrict__ items, T* L, T* U,
                                                      const T* __restrict__ Part) {
  const ReduceItem it = items[blockIdx.x / RSPLIT];
  T* C = (it.csrc == S_L ? L : U) + it.c;
  const int tb = it.tile, tt = tb * tb, chunk = tt / RSPLIT;
  const int e0 = (blockIdx.x % RSPLIT) * chunk;
  for (int e = e0 + threadIdx.x; e < e0 + chunk; e += blockDim.x) {
    const int i = e % tb, j = e / tb;
    if (i >= it.m || j >= it.n || i - j + it.diag < 0) continue;
    T* p = C + (int64_t)j * it.ldc + i;
    const T old = it.mode == G_SUB ? *p : T(0);
    // the pieces in order, eight loads in flight at a time (one round trip per piece otherwise)
    T s = 0;
    int q = 0;
    for (; q + 8 <= it.parts; q += 8) {
      T v[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) v[t] = Part[it.part0 + (int64_t)(q + t) * tt + e];
#pragma unroll
      for (int t = 0; t < 8; ++t) s += v[t];
    }
    for (; q < it.parts; ++q) s += Part[it.part0 + (int64_t)q * tt + e];
    *p = it.mode == G_SUB ? old - s : -s;
  }
}

}  // namespace fc
