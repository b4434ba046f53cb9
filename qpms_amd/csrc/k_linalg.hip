// Dense complex linear algebra for the mode problem on gfx950: blocked
// right-looking LU with partial pivoting (zgetrf / cgetrf semantics,
// row-major, 1-based ipiv), triangular solves, and the FP32-LU + FP64
// iterative-refinement solver.
//
// Reference call sites: scatsystem.c:2214 (LAPACKE_zgetrf), 2270 (zgetrs),
// beyn.c:556-561 (zgetrf + zgetrs with l right-hand sides).
//
// LU structure (getrf_batched): outer blocks of LU_NB = 256 columns.
//   k_strip       factors a tall strip of PW = 32 columns with partial pivoting
//                 in one launch, the rows in registers; its workgroups agree on
//                 each pivot through memory. They wait for one another, so they
//                 announce themselves first, and where they do not all get onto
//                 the device in time one of them does the strip alone;
//   k_ts_*        the same with tournament pivoting, no workgroup waiting for
//                 another: for strips of more workgroups than may wait for one
//                 another (strip_most);
//   k_swap_u      the strip's interchanges and U = L11^{-1} A12 in the rest of
//                 its outer block, by substitution; k_u12 the block's U12 in the
//                 columns beyond;
//   k_gemm_sub    C -= A B (k_gemm_cu beside the trailing update): the rank-PW
//                 updates inside an outer block and the rank-256 trailing update
//                 A22 -= L21 U12 (the O(n^3) part, rocBLAS or k_cgemm3m by size
//                 class). FP64 uses v_mfma_f64_16x16x4f64, FP32
//                 v_mfma_f32_16x16x4f32; the complex product is four real MFMA
//                 chains on de-interleaved LDS tiles.
// Solves (getrs_batched): k_tri, both sweeps in one launch.
// Every kernel takes a batch index in blockIdx.z with per-matrix strides, so
// the Beyn quadrature nodes factor in one launch sequence.
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <algorithm>
#include <type_traits>
#include <mutex>
#include <rocblas/rocblas.h>
#include "qpms_internal.h"
#include "dev_launch.hpp"

typedef double v2d __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

#define HIPCHK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) \
  qpms_hip_die(__FILE__, __LINE__, __func__, "HIP error %d (%s) in %s", (int)e_, hipGetErrorString(e_), #x); } while (0)

namespace {

template <class T> struct C2;
template <> struct C2<double> { typedef v2d t; };
template <> struct C2<float> { typedef v2f t; };

template <class T> __device__ __forceinline__ typename C2<T>::t cmul(typename C2<T>::t a, typename C2<T>::t b) {
  return typename C2<T>::t{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
// y - a b with one rounding of y's size (as two chained FMAs a part it is two)
template <class T> __device__ __forceinline__ typename C2<T>::t cless(typename C2<T>::t y, typename C2<T>::t a, typename C2<T>::t b) {
  return typename C2<T>::t{y.x - fma(a.x, b.x, -a.y * b.y), y.y - fma(a.x, b.y, a.y * b.x)};
}
template <class T> __device__ __forceinline__ typename C2<T>::t cdiv(typename C2<T>::t a, typename C2<T>::t b) {
  // Smith's algorithm
  if (fabs(b.x) >= fabs(b.y)) {
    T r = b.y / b.x, d = b.x + b.y * r;
    return typename C2<T>::t{(a.x + a.y * r) / d, (a.y - a.x * r) / d};
  } else {
    T r = b.x / b.y, d = b.x * r + b.y;
    return typename C2<T>::t{(a.x * r + a.y) / d, (a.y * r - a.x) / d};
  }
}


// ---------------------------------------------------------------------------
// C[M x N] -= A[M x K] * B[K x N] (complex, row-major), MFMA.
// Block: 256 threads = 4 waves, C tile 64 x 64, each wave a 32 x 32 quadrant
// made of 2 x 2 MFMA 16x16 tiles, K step 16 (= 4 MFMA k-steps of 4).
// LDS tiles are de-interleaved: Ar, Ai [64][16+1], Br, Bi [16][64+1].
// Complex: Cr -= Ar Br - Ai Bi ; Ci -= Ar Bi + Ai Br  → accumulate
//   Pr = Ar Br + (-Ai) Bi and Pi = Ar Bi + Ai Br, then C -= P.
// MFMA 16x16x4 lane layout: a = A[l%16][l/16], b = B[l/16][l%16],
// acc[i] = D[MF<T>::row(l/16, i)][l%16].
// ---------------------------------------------------------------------------
template <class T> struct MF;
// Output row of accumulator element i held by lane group lk (= lane / 16):
// the f64 16x16x4 instruction interleaves the four lane groups row by row,
// the f32 one gives each lane group four consecutive rows.
template <> struct MF<double> {
  typedef v4d acc;
  static __device__ __forceinline__ acc mma(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int i) { return lk + 4 * i; }
};
template <> struct MF<float> {
  typedef v4f acc;
  static __device__ __forceinline__ acc mma(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int i) { return 4 * lk + i; }
};

constexpr int GT = 64, GK = 16;

template <class T>
__global__ __launch_bounds__(256) void k_gemm_sub(int M, int N, int K, const typename C2<T>::t *A, long lda, long sA,
                                                  const typename C2<T>::t *B, long ldb, long sB,
                                                  typename C2<T>::t *C, long ldc, long sC) {
  typedef typename C2<T>::t cT;
  typedef typename MF<T>::acc acc_t;
  A += (long)blockIdx.z * sA;
  B += (long)blockIdx.z * sB;
  C += (long)blockIdx.z * sC;
  __shared__ T Ar[GT][GK + 1], Ai[GT][GK + 1], Br[GK][GT + 1], Bi[GK][GT + 1];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int wm = (wv >> 1) * 32, wn = (wv & 1) * 32;  // wave quadrant
  // grid-stride over C tiles (a grid smaller than the tile count keeps its
  // workgroups on few CUs)
  for (int m0 = blockIdx.y * GT; m0 < M; m0 += gridDim.y * GT)
  for (int n0 = blockIdx.x * GT; n0 < N; n0 += gridDim.x * GT) {
  acc_t pr[2][2], pi[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) { pr[a][b] = acc_t{0, 0, 0, 0}; pi[a][b] = acc_t{0, 0, 0, 0}; }
  const int lr = lane & 15, lk = lane >> 4;
  for (int k0 = 0; k0 < K; k0 += GK) {
    // load A tile 64 x 16 (1024 complex, 4 per thread) and B tile 16 x 64
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int idx = tid + 256 * e;
      const int ar = idx >> 4, ak = idx & 15;
      cT va = cT{0, 0};
      if (m0 + ar < M && k0 + ak < K) va = A[(long)(m0 + ar) * lda + k0 + ak];
      Ar[ar][ak] = va.x;
      Ai[ar][ak] = va.y;
      const int bk = idx >> 6, bn = idx & 63;
      cT vb = cT{0, 0};
      if (k0 + bk < K && n0 + bn < N) vb = B[(long)(k0 + bk) * ldb + n0 + bn];
      Br[bk][bn] = vb.x;
      Bi[bk][bn] = vb.y;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GK; kk += 4) {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const T ar = Ar[wm + a * 16 + lr][kk + lk], ai = Ai[wm + a * 16 + lr][kk + lk];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const T br = Br[kk + lk][wn + b * 16 + lr], bi = Bi[kk + lk][wn + b * 16 + lr];
          pr[a][b] = MF<T>::mma(ar, br, pr[a][b]);
          pr[a][b] = MF<T>::mma(-ai, bi, pr[a][b]);
          pi[a][b] = MF<T>::mma(ar, bi, pi[a][b]);
          pi[a][b] = MF<T>::mma(ai, br, pi[a][b]);
        }
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = m0 + wm + a * 16 + MF<T>::row(lk, i), col = n0 + wn + b * 16 + lr;
        if (row < M && col < N) {
          cT c = C[(long)row * ldc + col];
          c.x -= pr[a][b][i];
          c.y -= pi[a][b][i];
          C[(long)row * ldc + col] = c;
        }
      }
  }
}

// ---------------------------------------------------------------------------
// Small helpers
// ---------------------------------------------------------------------------
__global__ void k_iota(int n, int *p, long sP) {
  p += (long)blockIdx.z * sP;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = i;
}

// perm from LAPACK-style pivots (where a caller hands in pivots without the
// permutation): each lane follows one row through the interchanges, the same for
// all, 64 of them loaded at a time while the ones before are gone through; a wave
// ends when its rows' places lie behind it. One thread making the interchanges
// one by one took 0.11 us each (1.0 ms at order 9216).
__global__ __launch_bounds__(64) void k_perm_from_ipiv(int n, const int *__restrict__ ipiv, int *__restrict__ perm) {
  const int lane = threadIdx.x, t = blockIdx.x * 64 + lane;
  int pos = t, next = ipiv[min(lane, n - 1)] - 1;
  for (int i0 = 0; i0 < n && __ballot(pos >= i0 && t < n); i0 += 64) {
    const int own = i0 + lane < n ? next : i0 + lane;   // behind the end: stays where it is
    next = ipiv[min(i0 + 64 + lane, n - 1)] - 1;
#pragma unroll 16
    for (int q = 0; q < 64; ++q) {
      const int i = i0 + q, p = __builtin_amdgcn_readlane(own, q);
      pos = pos == i ? p : pos == p ? i : pos;
    }
  }
  if (t < n) perm[pos] = t;
}

// C[:, 0:NR] -= A B for few right-hand sides (NR <= 4), FP64 complex: one
// wave per row of A with its lanes 16 bytes apart along the row (each wave
// load is 1 KiB contiguous), the NR sums reduced across the wave. A is read
// once, so the residuals of the iterative refinement run at HBM speed; the
// tiled GEMM would give each 64-row tile one workgroup and leave most CUs idle.
template <int NR>
__global__ __launch_bounds__(256) void k_gemv_sub_f64(int M, int K, const v2d *__restrict__ A, long lda, long sA,
                                                      const v2d *__restrict__ B, long ldb, long sB,
                                                      v2d *__restrict__ C, long ldc, long sC) {
  const int lane = threadIdx.x & 63;
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int z = blockIdx.y;
  if (i >= M) return;
  const v2d *a = A + (long)z * sA + (long)i * lda;
  const v2d *b = B + (long)z * sB;
  double sr[NR], si[NR];
#pragma unroll
  for (int n = 0; n < NR; ++n) sr[n] = si[n] = 0.0;
#pragma unroll 4
  for (int k = lane; k < K; k += 64) {
    const v2d x = __builtin_nontemporal_load(a + k);
#pragma unroll
    for (int n = 0; n < NR; ++n) {
      const v2d y = b[(long)k * ldb + n];
      sr[n] += x.x * y.x - x.y * y.y;
      si[n] += x.x * y.y + x.y * y.x;
    }
  }
#pragma unroll
  for (int n = 0; n < NR; ++n)
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      sr[n] += __shfl_xor(sr[n], o);
      si[n] += __shfl_xor(si[n], o);
    }
  if (lane == 0) {
    v2d *c = C + (long)z * sC + (long)i * ldc;
#pragma unroll
    for (int n = 0; n < NR; ++n) c[n] = v2d{c[n].x - sr[n], c[n].y - si[n]};
  }
}

// Element-wise conversions and copies: grid-stride loops, so that a launch
// covers any n (a batch of Beyn nodes at order 49152 is 4.8e9 elements, more
// work-items than one dispatch can name).
__global__ void k_d2f(long n, const v2d *x, v2f *y) {
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256)
    y[i] = v2f{(float)x[i].x, (float)x[i].y};
}
__global__ void k_f2d_add(long n, const v2f *d, v2d *x) {
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256)
    x[i] = v2d{x[i].x + (double)d[i].x, x[i].y + (double)d[i].y};
}
__global__ void k_copy2d(long n, const v2d *x, v2d *y) {
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) y[i] = x[i];
}
// Sum of |z|^2 into out[blockIdx.x] (partial sums, finished on the host).
__global__ void k_sumsq(long n, const v2d *x, double *out) {
  __shared__ double s[256];
  double a = 0;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256)
    a += x[i].x * x[i].x + x[i].y * x[i].y;
  s[threadIdx.x] = a;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) s[threadIdx.x] += s[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = s[0];
}

// M = I - T W for one particle's block row: T (nr x nr), W rows (nr x L), the
// identity lands at columns col0..col0+nr-1.
__global__ void k_block_tw(int nr, int L, const v2d *T, const v2d *W, v2d *M, int col0) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  const int i = blockIdx.y;
  if (j >= L) return;
  double re = (j - col0 == i) ? 1.0 : 0.0, im = 0.0;
  for (int k = 0; k < nr; ++k) {
    const v2d t = T[(long)i * nr + k], w = W[(long)k * L + j];
    re -= t.x * w.x - t.y * w.y;
    im -= t.x * w.y + t.y * w.x;
  }
  M[(long)i * L + j] = v2d{re, im};
}

}  // namespace

// ===========================================================================
// Host drivers
// ===========================================================================
// ---------------------------------------------------------------------------
// Tall-strip panel: LU with tournament pivoting (CALU / TSLU, Grigori,
// Demmel & Xiang 2011). The strip (rows c0..n-1, columns c0..c0+w-1,
// w <= PW) is split into chunks of R = 256 rows staged in LDS, one row per
// thread:
//   k_ts_local   each workgroup runs partial-pivoting elimination on its
//                chunk only to choose w candidate rows, and writes their
//                indices and original values;
//   k_ts_merge   up to R / PW candidate sets per workgroup are merged the
//                same way, level by level, until one set remains;
//   the last level (local when one chunk covers the strip, else the last
//                merge) also writes the w x w block L11\U11 as its
//                elimination left the pivot rows, the zgetrf-style
//                interchanges (ipiv, perm), info on a zero pivot, the
//                list of rows the interchanges move, and L11^{-1} and
//                U11^{-1};
//   k_ts_apply   moves those rows in every column of the matrix (one gather
//                per column block) and stores L11\U11;
//   then every other strip row gets L21 = A21 U11^{-1} and the next PW rows
//   of the outer block U = L11^{-1} A12, as MFMA products (k_gemm_sub).
// No workgroup ever waits for another one; each step is its own launch.
// ---------------------------------------------------------------------------
constexpr int PW_ = 32;           // strip width (FP32 and FP64)
constexpr int TS_THREADS = 256;   // threads per tournament workgroup (one row each)
constexpr int TS_WAVES = TS_THREADS / 64;
// LDS row stride (complex): conflict-free row-per-lane access with 16-byte
// lane accesses (two FP32 complex values, or one FP64)
template <class T> struct TsStride;
template <> struct TsStride<float> { static constexpr int XS = PW_ + 2; };
template <> struct TsStride<double> { static constexpr int XS = PW_ + 1; };

template <class T> struct PanelW { static constexpr int W = PW_; };
// rows per tournament workgroup, one per thread: the chunk is staged in LDS
// (70 KB FP32, 135 KB FP64)
template <class T> struct TsRows { static constexpr int R = TS_THREADS; };
template <class T> constexpr int ts_fan() { return TsRows<T>::R / PW_; }   // candidate sets merged per workgroup
template <class T> constexpr size_t ts_lds() { return (size_t)TsRows<T>::R * TsStride<T>::XS * sizeof(typename C2<T>::t); }

// Per matrix: two candidate buffers of Gmax sets (index + PW values each),
// then one output slot per strip of an outer block (the last tournament
// level's L11\U11, moved-row list and its length), kept until the block's
// interchanges have been applied to the columns outside it.
constexpr int TS_SLOTS = 8;   // strips per outer block (LU_NB / PW)
template <class T>
struct PanelWS {
  static size_t set_bytes() { return ((size_t)PW_ * 4 + (size_t)PW_ * PW_ * sizeof(typename C2<T>::t) + 255) / 256 * 256; }
  // slot of a strip: its interchanges (src[i], the strip row that ends as row i of
  // the top PW; to[i], where row i of the top went), then (tournament) L11\U11 and
  // U11^{-1}, PW x PW each
  static constexpr size_t LU_OFF = 2 * PW_ * 4, UINV_OFF = LU_OFF + (size_t)PW_ * PW_ * sizeof(typename C2<T>::t);
  static size_t fin_bytes() { return UINV_OFF + (size_t)PW_ * PW_ * sizeof(typename C2<T>::t); }
  static int sets(int n) { return (n + TsRows<T>::R - 1) / TsRows<T>::R; }
};

// Workgroup state of the elimination: each wave's packed winner and winning
// row per column (two slot sets, alternating), the pivot rows as they were
// when chosen (urow[j][j + p] = column j + p of pivot j: its U part), and
// the pivots.
template <class T>
struct TsShared {
  typedef typename C2<T>::t cT;
  unsigned long long wp[2][TS_WAVES];
  __align__(16) cT cand[2][TS_WAVES][PW_];
  __align__(16) cT urow[PW_ + 1][PW_];   // one row more: pivot j's shifted row runs j positions past its own
  int sel[PW_];    // block row of pivot j
  int skey[PW_];   // key (strip row) of pivot j
  T sval[PW_];     // 1 if the pivot j is not zero, else 0
};

// Arg-max over a wave, by DPP moves only (xor 1, xor 2, rotate 4, rotate 8
// inside each 16-lane row, then the row broadcasts; lane 63 ends with the
// wave's winner) of one packed 64-bit key per lane:
//   bits 63..32  the order bits of |x_j|_1 plus one (0: no live row) -- all 32
//                bits of an FP32 value, the upper 32 of an FP64 one (order
//                kept up to 2^-20 relative; nearer ties go to the key, as do
//                exact ties in izamax's first-maximum rule);
//   bits 31..10  0x3FFFFF - key (the smaller strip row wins a tie);
//   bits  9..0   the row within the workgroup (< 512).
// NaN magnitudes rank as zero. Non-negative floats order as their bits.
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false); }
__device__ __forceinline__ unsigned int ts_order_bits(float a) { return __float_as_uint(a); }
__device__ __forceinline__ unsigned int ts_order_bits(double a) {
  return (unsigned int)((unsigned long long)__double_as_longlong(a) >> 32);
}
template <class T>
__device__ __forceinline__ unsigned long long ts_pack(bool live, T a, int key, int row) {
  if (!(a == a)) a = 0;
  const unsigned int hi = live ? ts_order_bits(a) + 1u : 0u;
  return ((unsigned long long)hi << 32) | ((unsigned long long)(0x3FFFFFu - (unsigned)key) << 10) | (unsigned)row;
}
template <int CTRL>
__device__ __forceinline__ unsigned long long dpp_u64(unsigned long long v) {
  const unsigned lo = (unsigned)dpp_i<CTRL>((int)(unsigned)v), hi = (unsigned)dpp_i<CTRL>((int)(unsigned)(v >> 32));
  return ((unsigned long long)hi << 32) | lo;
}
// row broadcasts for the rows the mask enables; the others receive 0
template <int CTRL, int RM>
__device__ __forceinline__ unsigned long long dppm_u64(unsigned long long v) {
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)v, CTRL, RM, 0xF, false);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(v >> 32), CTRL, RM, 0xF, false);
  return ((unsigned long long)hi << 32) | lo;
}
__device__ __forceinline__ unsigned long long umax64(unsigned long long a, unsigned long long b) { return b > a ? b : a; }
__device__ __forceinline__ unsigned long long wave_amax(unsigned long long v) {
  v = umax64(v, dpp_u64<0xB1>(v));          // quad_perm [1,0,3,2]
  v = umax64(v, dpp_u64<0x4E>(v));          // quad_perm [2,3,0,1]
  v = umax64(v, dpp_u64<0x124>(v));         // row_ror 4
  v = umax64(v, dpp_u64<0x128>(v));         // row_ror 8: every lane of a row holds the row's winner
  v = umax64(v, dppm_u64<0x142, 0xA>(v));   // row_bcast 15: rows 1, 3 take rows 0, 2
  v = umax64(v, dppm_u64<0x143, 0xC>(v));   // row_bcast 31: rows 2, 3 take row 1
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, 63);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), 63);
  return ((unsigned long long)hi << 32) | lo;
}

// 1 / p for the pivot as conj(p) / |p|^2 while |p|^2 is comfortably normal
// (FP32: the hardware reciprocal, one rounding more than a division; FP64: one
// IEEE division), instead of Smith's three dependent divisions, which remain
// for tiny or huge pivots.
template <class T> __device__ __forceinline__ typename C2<T>::t ts_crcp(typename C2<T>::t p);
template <> __device__ __forceinline__ v2f ts_crcp<float>(v2f p) {
  const float d = p.x * p.x + p.y * p.y;
  if (d > 1e-30f && d < 1e30f) {
    const float r = __builtin_amdgcn_rcpf(d);
    return v2f{p.x * r, -p.y * r};
  }
  return cdiv<float>(v2f{1, 0}, p);
}
template <> __device__ __forceinline__ v2d ts_crcp<double>(v2d p) {
  const double d = p.x * p.x + p.y * p.y;
  if (d > 1e-280 && d < 1e280) {
    const double r = 1.0 / d;
    return v2d{p.x * r, -p.y * r};
  }
  return cdiv<double>(v2d{1, 0}, p);
}

// Partial-pivoting elimination over the R rows of a workgroup staged in LDS
// (X[row][XS]), used only to choose pivot rows. Row i belongs to thread i
// (keys distinct, < 0 for an empty row), which holds it in registers. Per
// column j, a rolled loop (its body is a few KB of code, so the workgroup's
// single pass does not wait on instruction fetch):
//   the wave arg-max of |x_j|_1 on packed keys; each wave's winning lane
//   writes its row and lane 0 the packed key into LDS slots that alternate
//   between columns; one barrier; every thread combines the waves' keys and
//   reads the pivot row from its wave's slot (one broadcast address per
//   access); the chosen row stores itself as it is (its U part) and drops
//   out; every live row stores its multiplier l in X[row][j] and subtracts l
//   times the pivot row (four FMAs per complex entry).
// The row is kept rotated, x[p] = column j + p, shifting by one per column
// (zeros enter on the right, and stay zero: no column mask is needed).
// A wave reaches column j + 2's slots only after every wave has passed
// column j + 1's barrier, so two slot sets suffice. On return X[row][c] holds
// the multipliers of each row for the columns before its selection (all
// columns for rows not chosen), sh.urow the chosen rows' U parts and
// sh.sel/skey/sval the pivots; returns their number.
template <class T>
__device__ __forceinline__ int ts_gepp(typename C2<T>::t *X, int key, int w, TsShared<T> &sh) {
  typedef typename C2<T>::t cT;
  constexpr int XS = TsStride<T>::XS;
  static_assert(TsRows<T>::R == TS_THREADS, "one row per thread");
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  bool live = key >= 0;
  cT x[PW_];
#pragma unroll
  for (int c = 0; c < PW_; ++c) x[c] = X[t * XS + c];
  int ns = 0;
  for (int j = 0; j < w; ++j) {
    const int par = j & 1;
    const cT xj = x[0];
    const unsigned long long v = wave_amax(ts_pack<T>(live, fabs(xj.x) + fabs(xj.y), live ? key : 0, t));
    if (t == (int)(v & 0x3FFu)) {
#pragma unroll
      for (int p = 0; p < PW_; ++p) sh.cand[par][wave][p] = x[p];
    }
    if (lane == 0) sh.wp[par][wave] = v;
    __syncthreads();
    unsigned long long m = sh.wp[par][0];
#pragma unroll
    for (int q = 1; q < TS_WAVES; ++q) m = umax64(m, sh.wp[par][q]);
    const unsigned int mhi = (unsigned int)(m >> 32);
    if (mhi == 0) break;   // no row left (uniform)
    const int pr = (int)(m & 0x3FFu), pk = (int)(0x3FFFFFu - (unsigned)((m >> 10) & 0x3FFFFFu));
    const bool nonzero = mhi > 1u;   // the pivot's |x_j|_1 is not zero (uniform)
    if (t == 0) { sh.sel[j] = pr; sh.skey[j] = pk; sh.sval[j] = nonzero ? T(1) : T(0); }
    ns = j + 1;
    if (t == pr) {
      live = false;
      cT *dst = &sh.urow[j][j];
#pragma unroll
      for (int p = 0; p < PW_; ++p) dst[p] = x[p];
    }
    // Every thread shifts (straight-line code, so the shift stays in place in
    // the registers); rows that are not live, and every row at a zero pivot,
    // shift with l = 0. A live row keeps its entry at a zero pivot.
    const cT *P = sh.cand[par][pr >> 6];
    cT l = cT{0, 0};
    if (live && nonzero) l = cmul<T>(xj, ts_crcp<T>(P[0]));
    if (live) X[t * XS + j] = nonzero ? l : xj;
#pragma unroll
    for (int p = 0; p + 1 < PW_; ++p) {
      const cT u = P[p + 1], y = x[p + 1];
      x[p] = cT{fma(-l.x, u.x, fma(l.y, u.y, y.x)), fma(-l.x, u.y, fma(-l.y, u.x, y.y))};
    }
    x[PW_ - 1] = cT{0, 0};
  }
  __syncthreads();
  return ns;
}

// U11^{-1} of a strip's PW x PW L\U into out (row-major), for the strip's L21 as
// a product. v: entries e = t + TS_THREADS q of L\U. PW backward right-looking
// steps, each entry owned by one thread, one barrier per step, in the LDS of X
// (whose rows are no longer needed). A zero diagonal entry of U is taken as one:
// the row's L21 entry is then kept, as a zero pivot leaves it.
template <class T>
__device__ __forceinline__ void ts_u_inverse(typename C2<T>::t *X, const typename C2<T>::t *v, char *out) {
  typedef typename C2<T>::t cT;
  constexpr int PP = PW_ * PW_, NE = PP / TS_THREADS;
  const int t = threadIdx.x;
  cT *LU = X, *Z = X + PP, *dinv = X + 2 * PP;   // Z: U^{-1} with unscaled rows
  __syncthreads();   // every read of X's rows is done
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    const int e = t + TS_THREADS * q;
    LU[e] = v[q];
    Z[e] = (e / PW_ == e % PW_) ? cT{1, 0} : cT{0, 0};
  }
  __syncthreads();
  if (t < PW_) {
    const cT d = LU[t * PW_ + t];
    dinv[t] = (d.x == 0 && d.y == 0) ? cT{1, 0} : cdiv<T>(cT{1, 0}, d);
  }
  __syncthreads();
  for (int s = PW_ - 1; s >= 0; --s) {   // rows above s take row s divided by its diagonal
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      const int e = t + TS_THREADS * q, i = e / PW_, c = e % PW_;
      if (i < s) {
        const cT u = cmul<T>(LU[i * PW_ + s], dinv[s]), z = Z[s * PW_ + c];
        Z[e] = cT{Z[e].x - (u.x * z.x - u.y * z.y), Z[e].y - (u.x * z.y + u.y * z.x)};
      }
    }
    __syncthreads();
  }
  cT *o = reinterpret_cast<cT *>(out);
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    const int e = t + TS_THREADS * q;
    o[e] = cmul<T>(Z[e], dinv[e / PW_]);
  }
}

// Output of the last tournament level: L11\U11 rows, ipiv (1-based, matrix
// rows), perm, info, U11^{-1}, and where the interchanges take rows from and
// to, from a list of the rows they touch. The list starts as the w top rows; each interchange
// i <-> p is applied to it with wave ballots (a row not yet listed sits at
// its own index).
template <class T>
__device__ __forceinline__ void ts_finish(typename C2<T>::t *X, int ns, int w, int c0, TsShared<T> &sh,
                                          char *fin, int *ipiv, int *perm, int *info) {
  typedef typename C2<T>::t cT;
  constexpr int XS = TsStride<T>::XS, NE = PW_ * PW_ / TS_THREADS;
  const int t = threadIdx.x;
  cT *lu = reinterpret_cast<cT *>(fin + PanelWS<T>::LU_OFF);
  int *src = reinterpret_cast<int *>(fin), *to = src + PW_;
  cT v[NE];   // entries t + TS_THREADS q of L11\U11
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    const int e = t + TS_THREADS * q, i = e / PW_, c = e % PW_;
    v[q] = (i < ns && c < w) ? (c >= i ? sh.urow[i][c] : X[sh.sel[i] * XS + c]) : cT{0, 0};
    lu[e] = v[q];
  }
  if (t < 64) {
    int id = (t < w) ? t : -1, pos = id, nlist = w;
    for (int i = 0; i < ns; ++i) {
      const int tg = sh.skey[i];
      const unsigned long long mt = __ballot(id == tg);
      const int lt = mt ? __ffsll((long long)mt) - 1 : -1;
      const int p = (lt >= 0) ? __shfl(pos, lt) : tg;
      const unsigned long long mi = __ballot(id >= 0 && pos == i);
      const int li = __ffsll((long long)mi) - 1;
      if (p != i) {
        if (t == li) pos = p;
        if (lt >= 0) {
          if (t == lt) pos = i;
        } else {
          if (t == nlist) { id = tg; pos = i; }
          ++nlist;
        }
      }
      if (t == 0) ipiv[c0 + i] = c0 + p + 1;
    }
    if (t == 0) {
      int z0 = 0;
      for (int i = ns - 1; i >= 0; --i)
        if (sh.sval[i] == 0) z0 = c0 + i + 1;
      if (z0 && *info == 0) *info = z0;
    }
    if (t < nlist && pos < w) src[pos] = id;
    if (t < nlist && id < w) to[id] = pos;
    const bool mv = (t < nlist) && id != pos;
    if (perm) {   // the moved rows as one gather: every lane loads before any stores
      const int pv = mv ? perm[c0 + id] : 0;
      if (mv) perm[c0 + pos] = pv;
    }
  }
  ts_u_inverse<T>(X, v, fin + PanelWS<T>::UINV_OFF);
}

template <class T>
__global__ __launch_bounds__(TS_THREADS) void k_ts_local(int n, int c0, int w, const typename C2<T>::t *A, long lda,
                                                         long sA, char *ws, long sW, long setb, long finoff,
                                                         int final_, int *ipiv, long sP, int *perm, int *info) {
  typedef typename C2<T>::t cT;
  constexpr int R = TsRows<T>::R, XS = TsStride<T>::XS;
  extern __shared__ __align__(16) char smem_raw[];
  cT *X = reinterpret_cast<cT *>(smem_raw);
  __shared__ TsShared<T> sh;
  const int z = blockIdx.z, g = blockIdx.x, t = threadIdx.x;
  A += (long)z * sA;
  ws += (long)z * sW;
  const int m = n - c0, r0 = g * R, nr = min(R, m - r0);
  {   // coalesced along each row; every load in flight before the first LDS store
    constexpr int PER = R * PW_ / TS_THREADS;
    cT v[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = t + TS_THREADS * q, r = e / PW_, c = e % PW_;
      v[q] = (r < nr && c < w) ? A[(long)(c0 + r0 + r) * lda + c0 + c] : cT{0, 0};
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = t + TS_THREADS * q;
      X[(e / PW_) * XS + e % PW_] = v[q];
    }
  }
  __syncthreads();
  const int ns = ts_gepp<T>(X, t < nr ? r0 + t : -1, w, sh);
  if (final_) {
    ts_finish<T>(X, ns, w, c0, sh, ws + finoff, ipiv + (long)z * sP, perm ? perm + (long)z * sP : nullptr, info + z);
    return;
  }
  char *set = ws + (long)g * setb;
  int *oidx = reinterpret_cast<int *>(set);
  cT *oval = reinterpret_cast<cT *>(set + PW_ * 4);
  if (t < PW_) oidx[t] = (t < ns) ? sh.skey[t] : -1;
  constexpr int PO = PW_ * PW_ / TS_THREADS;
  cT v[PO];
#pragma unroll
  for (int q = 0; q < PO; ++q) {   // the chosen rows' original values
    const int e = t + TS_THREADS * q, i = e / PW_, c = e % PW_;
    v[q] = (i < ns && c < w) ? A[(long)(c0 + sh.skey[i]) * lda + c0 + c] : cT{0, 0};
  }
#pragma unroll
  for (int q = 0; q < PO; ++q) {
    const int e = t + TS_THREADS * q;
    if (e < ns * PW_) oval[e] = v[q];
  }
}

template <class T>
__global__ __launch_bounds__(TS_THREADS) void k_ts_merge(int c0, int w, int nin, const char *wsin, char *wsout,
                                                         long sW, long setb, char *wsfin, int final_, int *ipiv,
                                                         long sP, int *perm, int *info) {
  typedef typename C2<T>::t cT;
  constexpr int R = TsRows<T>::R, F = ts_fan<T>(), XS = TsStride<T>::XS;
  extern __shared__ __align__(16) char smem_raw[];
  cT *X = reinterpret_cast<cT *>(smem_raw);
  __shared__ TsShared<T> sh;
  const int z = blockIdx.z, b = blockIdx.x, t = threadIdx.x;
  const char *in = wsin + (long)z * sW;
  const int s0 = b * F, nset = min(F, nin - s0);
  {   // every load in flight before the first LDS store
    constexpr int PER = R * PW_ / TS_THREADS;
    cT v[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = t + TS_THREADS * q, r = e / PW_, c = e % PW_, si = r / PW_, i = r % PW_;
      v[q] = (si < nset) ? reinterpret_cast<const cT *>(in + (long)(s0 + si) * setb + PW_ * 4)[i * PW_ + c]
                         : cT{0, 0};
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = t + TS_THREADS * q;
      X[(e / PW_) * XS + e % PW_] = v[q];
    }
  }
  int key = -1;
  if (t < R && t / PW_ < nset) key = reinterpret_cast<const int *>(in + (long)(s0 + t / PW_) * setb)[t % PW_];
  __syncthreads();
  const int ns = ts_gepp<T>(X, key, w, sh);
  if (final_) {
    ts_finish<T>(X, ns, w, c0, sh, wsfin + (long)z * sW, ipiv + (long)z * sP, perm ? perm + (long)z * sP : nullptr,
                 info + z);
    return;
  }
  char *out = wsout + (long)z * sW + (long)b * setb;
  int *oidx = reinterpret_cast<int *>(out);
  cT *oval = reinterpret_cast<cT *>(out + PW_ * 4);
  if (t < PW_) oidx[t] = (t < ns) ? sh.skey[t] : -1;
  constexpr int PO = PW_ * PW_ / TS_THREADS;
  cT v[PO];
#pragma unroll
  for (int q = 0; q < PO; ++q) {   // the chosen rows' original values, from their input set
    const int e = t + TS_THREADS * q, i = e / PW_, c = e % PW_, r = sh.sel[i];
    v[q] = (i < ns) ? reinterpret_cast<const cT *>(in + (long)(s0 + r / PW_) * setb + PW_ * 4)[(r % PW_) * PW_ + c]
                    : cT{0, 0};
  }
#pragma unroll
  for (int q = 0; q < PO; ++q) {
    const int e = t + TS_THREADS * q;
    if (e < ns * PW_) oval[e] = v[q];
  }
}

// ---------------------------------------------------------------------------
// Partial-pivoting strips (k_strip), for the entry points that return the
// factors (qpms_hip_zgetrf_dev and the ABI factorisation built on it): the
// pivots of zgetrf (zgetf2's column loop, scatsystem.c:2214): pivot j is the
// first row of largest |re| + |im| in column j at or below the diagonal, taken
// in full double (or float) precision. One launch factors a whole strip: the
// workgroups hold its rows in registers for all of its columns and agree on
// each pivot through memory. L21 is left in place by the elimination.
//
// Layout. A wave holds RT tiles of 16 rows; lane (rq, cq) = (lane % 16,
// lane / 16) holds row rq of each tile and columns 4 i + cq, i = 0..7: the
// accumulator layout of the 16 x 16 x 4 matrix instructions for the transposed
// tile. Four columns (a chunk, register i) are factored with a row per lane: a
// 4 x 4 transposition by lane swaps gives lane (rq, cq) row rq of tile cq and
// its four entries y. Transposed back, register i is, as it stands, the right
// operand of the rank-4 update of the columns beyond, whose left operand is the
// chunk's U rows: four products per tile of 16 x 16. So a column step touches
// four columns only. With a row per lane throughout and rank-1 updates of the
// whole row, a column took 2.2 us beside its exchange (each wave took the whole
// pivot row from LDS, and the row's owner wrote it there one lane wide).
//
// Exchange. Every word carries the column's tag beside its payload (a
// candidate is two words: magnitude and position; a row is its entries' 32-bit
// halves), so a reader needs no flag and no fence: it reads a word until the
// tag is the column's. Words are relaxed agent-scope atomics, which pass the
// XCDs' own L2s: about 1.3 us per column for 2 to 32 workgroups. One wave of a
// workgroup reads them (every wave reading them took three times as long: the
// words of a column lie in a few lines that all workgroups ask for). Sets of
// words alternate between columns (candidates) and chunks (rows): a workgroup
// writes a set again only after it has seen every workgroup's candidate of a
// later column, hence after all of them have read the set. k_strip_init clears
// the words before a factorisation; within one, neighbouring columns' tags
// differ. One launch per column instead, with the strip read and written by
// each, took 11.9 us per column at order 2190 and 18.9 us at 9216.
//
// Waiting. A workgroup may wait for another one only when all of them are on
// the device. They announce themselves first: whoever has seen everybody moves
// the strip's state word from 0 to GO, whoever has waited longer than the limit
// moves it from 0 to ALONE, and the word's value after the attempt decides for
// everybody. After GO every workgroup has started and none ends before the
// last column, so every later wait ends. After
// ALONE the workgroup that set it factors the strip by itself in memory and
// the others leave without having written to the matrix.
// ---------------------------------------------------------------------------
constexpr int ST_GO = 1, ST_ALONE = 2;
constexpr int ST_RT = 4;   // row tiles per wave
// waves per workgroup: FP64 one per SIMD, FP32 two
template <class T> constexpr int st_w() { return sizeof(T) == 8 ? 4 : 8; }
template <class T> constexpr int st_rows() { return st_w<T>() * 16 * ST_RT; }   // 256 (FP64), 512 rows per workgroup
typedef unsigned long long st_u64;
constexpr st_u64 ST_LIMIT = 10000000ull;   // ticks of the 100 MHz clock (0.1 s) to wait for everybody
// words of one row: the reciprocal of its pivot, then its entries
template <class T> constexpr int st_ew() { return (int)sizeof(typename C2<T>::t) / 4; }
template <class T> constexpr int st_words() { return (1 + PW_) * st_ew<T>(); }
// Per-matrix workspace of the strips: a state word per strip, two sets of
// candidates, the announcements, two sets of four rows per workgroup.
constexpr long ST_STATE = 0;
constexpr long st_cand_off(int n) { return ST_STATE + ((long)((n + PW_ - 1) / PW_) * 4 + 255) / 256 * 256; }
template <class T> constexpr int st_groups(int rows) { return (rows + st_rows<T>() - 1) / st_rows<T>(); }
template <class T> constexpr long st_meet_off(int n) { return st_cand_off(n) + 2L * st_groups<T>(n) * 2 * 8; }
template <class T> constexpr long st_row_off(int n) { return st_meet_off<T>(n) + (long)st_groups<T>(n) * 8; }
template <class T> constexpr long st_ws_bytes(int n) { return st_row_off<T>(n) + 8L * st_groups<T>(n) * st_words<T>() * 8; }

__global__ __launch_bounds__(256) void k_strip_init(char *ws, long sW, long bytes) {
  st_u64 *p = reinterpret_cast<st_u64 *>(ws + (long)blockIdx.z * sW);
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < bytes / 8; i += (long)gridDim.x * 256) p[i] = 0;
}

__device__ __forceinline__ st_u64 st_load(const st_u64 *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_store(st_u64 *p, st_u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A candidate's two words: 21 bits of tag above 43 bits of the rank, and above
// its other 21 bits and 22 bits of the position.
__device__ __forceinline__ void st_pack(unsigned tag, st_u64 rank, int pos, st_u64 &a, st_u64 &b) {
  a = ((st_u64)tag << 43) | (rank >> 21);
  b = ((st_u64)tag << 43) | ((rank & 0x1fffffull) << 22) | (unsigned)pos;
}
__device__ __forceinline__ bool st_unpack(unsigned tag, st_u64 a, st_u64 b, st_u64 &rank, int &pos) {
  rank = (a << 21) | ((b >> 22) & 0x1fffffull);
  pos = (int)(b & 0x3fffffull);
  return (a >> 43) == tag && (b >> 43) == tag;
}
// A row's rank in the pivot search: the bits of |x|_1 (non-negative floating
// values order as their bits) plus two, 1 where that is no number, 0 for no row.
__device__ __forceinline__ st_u64 st_bits(double a) { return (st_u64)__double_as_longlong(a); }
__device__ __forceinline__ st_u64 st_bits(float a) { return (st_u64)__float_as_uint(a); }
template <class T> __device__ __forceinline__ st_u64 st_rank(bool live, typename C2<T>::t x) {
  const T a = fabs(x.x) + fabs(x.y);
  return live ? ((a == a) ? st_bits(a) + 2 : 1) : 0;
}
__device__ __forceinline__ bool st_before(st_u64 r, int p, st_u64 r2, int p2) { return r > r2 || (r == r2 && p < p2); }
template <int CTRL, int RM>
__device__ __forceinline__ unsigned st_dmax(unsigned v) {   // lanes without a source keep their own value
  const unsigned o = (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, RM, 0xF, false);
  return o > v ? o : v;
}
__device__ __forceinline__ unsigned st_wave_max(unsigned v) {
  v = st_dmax<0xB1, 0xF>(v);    // quad_perm [1,0,3,2]
  v = st_dmax<0x4E, 0xF>(v);    // quad_perm [2,3,0,1]
  v = st_dmax<0x124, 0xF>(v);   // row_ror 4
  v = st_dmax<0x128, 0xF>(v);   // row_ror 8
  v = st_dmax<0x142, 0xA>(v);   // row_bcast 15
  v = st_dmax<0x143, 0xC>(v);   // row_bcast 31
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}
// The lane of a wave with the largest rank, the smallest position among equal
// ones; rank and pos become that lane's. One DPP chain on the ranks' leading 32
// bits (FP32: all of them); only where lanes tie, one more for the other bits
// and one for the positions (a flat cluster's matrix has many entries that are
// exactly zero: taken one by one, their ties made a column three times as long).
template <bool WIDE>
__device__ __forceinline__ int st_wave_best(st_u64 &rank, int &pos) {
  const unsigned lo = (unsigned)rank, hi = (unsigned)(rank >> 32), own = WIDE ? hi : lo;
  const unsigned m = st_wave_max(own);
  st_u64 eq = __ballot(own == m && rank != 0);
  if (eq == 0) {   // no row in the wave
    rank = 0;
    return 0;
  }
  bool in = own == m && rank != 0;
  if (WIDE && (eq & (eq - 1))) {   // uniform
    const unsigned m2 = st_wave_max(in ? lo : 0u);
    in = in && lo == m2;
    eq = __ballot(in);
  }
  if (eq & (eq - 1)) {
    const unsigned m3 = st_wave_max(in ? 0x7fffffffu - (unsigned)pos : 0u);
    eq = __ballot(in && 0x7fffffffu - (unsigned)pos == m3);
  }
  const int l = __ffsll((long long)eq) - 1;
  rank = ((st_u64)(unsigned)__builtin_amdgcn_readlane((int)hi, l) << 32) | (unsigned)__builtin_amdgcn_readlane((int)lo, l);
  pos = __builtin_amdgcn_readlane(pos, l);
  return l;
}

template <class T>
struct StShared {
  typedef typename C2<T>::t cT;
  // rows in rotated order (entry 4 q + c is register q's column c: the chunk's
  // four entries first): the workgroup's candidate on its way to memory, the
  // chunk's pivot rows as they were when chosen, and their pivots' reciprocals
  __align__(16) cT own[PW_], urow[4][PW_], rcp[4], orcp;
  st_u64 rank[2][st_w<T>()];
  int pos[2][st_w<T>()];
  st_u64 prank;
  int ppos;
  int from[4];                     // the workgroups that had the chunk's pivots
  int piv[PW_], nz[PW_];
  int state;
};

// The strip's pivots (strip rows piv, nz[i] = 0 for a zero one) to ipiv and info.
__device__ __forceinline__ void st_pivots(int c0, int w, const int *piv, const int *nz, int *ipiv, int *info) {
  for (int i = 0; i < w; ++i) {
    ipiv[c0 + i] = c0 + piv[i] + 1;
    if (!nz[i] && *info == 0) *info = c0 + i + 1;
  }
}

// The strip's rows (S = row c0, column c0; m of them) factored in memory by one
// workgroup, after ALONE: a plain column loop.
template <class T>
__device__ __noinline__ void st_alone(int m, int w, typename C2<T>::t *S, long lda, StShared<T> &sh) {
  typedef typename C2<T>::t cT;
  constexpr bool WIDE = sizeof(T) == 8;
  const int t = threadIdx.x, nt = st_w<T>() * 64, lane = t & 63, wave = t >> 6;
  for (int j = 0; j < w; ++j) {
    st_u64 rank = 0;
    int pos = 0x3fffff;
    for (int i = j + t; i < m; i += nt) {
      const st_u64 r = st_rank<T>(true, S[(long)i * lda + j]);
      if (r > rank) { rank = r; pos = i; }   // a thread's rows come in rising order
    }
    (void)st_wave_best<WIDE>(rank, pos);
    if (lane == 0) { sh.rank[0][wave] = rank; sh.pos[0][wave] = pos; }
    __syncthreads();
    for (int q = 0; q < st_w<T>(); ++q)
      if (q == 0 || st_before(sh.rank[0][q], sh.pos[0][q], rank, pos)) { rank = sh.rank[0][q]; pos = sh.pos[0][q]; }
    if (t == 0) { sh.piv[j] = pos; sh.nz[j] = rank > 2; }
    if (t < w) {   // the interchange
      const cT a = S[(long)j * lda + t], b = S[(long)pos * lda + t];
      S[(long)j * lda + t] = b;
      if (pos != j) S[(long)pos * lda + t] = a;
    }
    __syncthreads();
    if (rank > 2) {
      const cT rcp = ts_crcp<T>(S[(long)j * lda + j]);
      for (int i = j + 1 + t; i < m; i += nt) {
        const cT l = cmul<T>(S[(long)i * lda + j], rcp);
        S[(long)i * lda + j] = l;
        for (int c = j + 1; c < w; ++c) {
          const cT u = S[(long)j * lda + c], y = S[(long)i * lda + c];
          S[(long)i * lda + c] = cless<T>(y, l, u);
        }
      }
    }
    __syncthreads();
  }
}

// Strips and slabs left to one workgroup so far (tests and probes read it).
__device__ unsigned g_alone;

// Everybody here? (one wave) Announces workgroup g with `tag` in the words `at`
// and waits for the others; returns 1 (go on), 0 (leave) or -1 (do the strip
// alone).
__device__ __forceinline__ int st_rendezvous(int g, int G, unsigned tag, st_u64 *at, int *state, st_u64 limit) {
  const int lane = threadIdx.x & 63;
  if (lane == 0) st_store(at + g, tag);
  const st_u64 t0 = wall_clock64();
  bool late = false;
  for (int c = lane; c < G; c += 64)
    while (!late && st_load(at + c) != tag) late = wall_clock64() - t0 > limit;
  const bool stop = __ballot(late) != 0;
  int seen = 0;
  if (lane == 0 && __hip_atomic_compare_exchange_strong(state, &seen, stop ? ST_ALONE : ST_GO, __ATOMIC_RELAXED,
                                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    seen = stop ? -1 : ST_GO;
  if (lane == 0 && seen == -1) atomicAdd(&g_alone, 1u);
  seen = __builtin_amdgcn_readfirstlane(seen);
  return seen == ST_ALONE ? 0 : seen;
}

// One column's exchange (one wave, all lanes; its candidate's words are on
// their way): the reciprocal and row `own` to memory, everybody's candidates, and
// the reciprocal and the chunk's entries of the winner's row to rcp and prow;
// rank, p and the result become the winner's rank, position and workgroup.
template <class T>
__device__ __forceinline__ int st_exchange(int g, int G, unsigned tag, const st_u64 *cw, st_u64 *rw,
                                           const typename C2<T>::t &orcp, const typename C2<T>::t *own,
                                           typename C2<T>::t &rcp, typename C2<T>::t *prow, st_u64 &rank, int &p) {
  constexpr int NW = st_words<T>(), EW = st_ew<T>();
  const int lane = threadIdx.x & 63;
  const st_u64 hi = (st_u64)tag << 32;
  // reciprocal and chunk first
  if (lane < EW) st_store(rw + g * NW + lane, hi | reinterpret_cast<const unsigned *>(&orcp)[lane]);
#pragma unroll
  for (int e = 0; e < PW_ * EW / 64; ++e)
    st_store(rw + g * NW + EW + 64 * e + lane, hi | reinterpret_cast<const unsigned *>(own)[64 * e + lane]);
  st_u64 best = 0;
  int bp = 0x3fffff, bg = 0;
  for (int c = lane; c < G; c += 64) {
    st_u64 r2;
    int p2;
    while (!st_unpack(tag, st_load(cw + 2 * c), st_load(cw + 2 * c + 1), r2, p2)) {}
    if (st_before(r2, p2, best, bp)) { best = r2; bp = p2; bg = c; }
  }
  const int bl = st_wave_best<sizeof(T) == 8>(best, bp);
  bg = __builtin_amdgcn_readlane(bg, bl);
  if (lane < 5 * EW) {
    st_u64 v;
    do v = st_load(rw + bg * NW + lane); while ((unsigned)(v >> 32) != tag);
    unsigned *to = lane < EW ? reinterpret_cast<unsigned *>(&rcp) + lane : reinterpret_cast<unsigned *>(prow) + lane - EW;
    *to = (unsigned)v;
  }
  rank = best;
  p = bp;
  return bg;
}

// Transposes four registers against the four rows of 16 lanes: v[a] of lane
// (rq, b) becomes v[b] of lane (rq, a).
__device__ __forceinline__ void st_transpose(unsigned (&v)[4]) {
  const auto a = __builtin_amdgcn_permlane16_swap(v[0], v[1], false, false);   // odd rows of the first <-> even of the second
  const auto b = __builtin_amdgcn_permlane16_swap(v[2], v[3], false, false);
  const auto c = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);   // upper half of the first <-> lower of the second
  const auto d = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
  v[0] = c[0];
  v[1] = d[0];
  v[2] = c[1];
  v[3] = d[1];
}
__device__ __forceinline__ void st_transpose(float (&v)[4]) {
  unsigned u[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) u[c] = __float_as_uint(v[c]);
  st_transpose(u);
#pragma unroll
  for (int c = 0; c < 4; ++c) v[c] = __uint_as_float(u[c]);
}
__device__ __forceinline__ void st_transpose(double (&v)[4]) {
  unsigned lo[4], hi[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const st_u64 b = (st_u64)__double_as_longlong(v[c]);
    lo[c] = (unsigned)b;
    hi[c] = (unsigned)(b >> 32);
  }
  st_transpose(lo);
  st_transpose(hi);
#pragma unroll
  for (int c = 0; c < 4; ++c) v[c] = __longlong_as_double((long long)(((st_u64)hi[c] << 32) | lo[c]));
}
// of four values, the lane's own
template <class T> __device__ __forceinline__ T st_own4(int cq, T a, T b, T c, T d) {
  const T e = (cq & 1) ? b : a, f = (cq & 1) ? d : c;
  return (cq & 2) ? f : e;
}

// Rows never move: each thread follows its row's position (the interchanges of
// zgetrf as integers) and the rows are stored there at the end.
template <class T>
__global__ __launch_bounds__(st_w<T>() * 64, 2) void k_strip(int n, int c0, int w, typename C2<T>::t *A, long lda,
                                                             long sA, char *ws, long sW, long finoff, st_u64 limit,
                                                             int *ipiv, long sP, int *info) {
  typedef typename C2<T>::t cT;
  typedef typename MF<T>::acc acc_t;
  constexpr bool WIDE = sizeof(T) == 8;
  constexpr int RT = ST_RT, NW = st_words<T>(), W = st_w<T>();
  static_assert(RT == 4, "a tile per row of lanes in a chunk");
  __shared__ StShared<T> sh;
  const int z = blockIdx.z, g = blockIdx.x, G = gridDim.x, t = threadIdx.x, lane = t & 63, rq = lane & 15, cq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  A += (long)z * sA;
  char *wz = ws + (long)z * sW;
  int *src = reinterpret_cast<int *>(wz + finoff), *moved_to = src + PW_;   // PanelWS's slot
  st_u64 *gcand = reinterpret_cast<st_u64 *>(wz + st_cand_off(n)), *grow = reinterpret_cast<st_u64 *>(wz + st_row_off<T>(n));
  const int m = n - c0, row0 = g * st_rows<T>() + wave * 16 * RT;
  int pos = row0 + lane;             // of row rq of tile cq
  const bool live_row = pos < m;
  bool live = live_row;
  unsigned el = 0;                   // the chunk's steps that eliminated the row
  // register q at chunk i is column 4 ((i + q) % 8) + cq: rotated by one per chunk,
  // so that all indices are compile-time and one body serves every chunk
  acc_t xr[RT][2], xi[RT][2];
#pragma unroll
  for (int T_ = 0; T_ < RT; ++T_) {
    // rows past the last and columns past the strip repeat the last one (never chosen, never stored)
    const cT *row = A + (long)(c0 + min(row0 + 16 * T_ + rq, m - 1)) * lda + c0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const cT v = row[min(4 * i + cq, w - 1)];
      xr[T_][i / 4][i % 4] = v.x;
      xi[T_][i / 4][i % 4] = v.y;
    }
  }
  if (G > 1) {
    if (wave == 0)
      sh.state = st_rendezvous(g, G, (unsigned)c0 + 1u, reinterpret_cast<st_u64 *>(wz + st_meet_off<T>(n)),
                               reinterpret_cast<int *>(wz + ST_STATE) + c0 / PW_, limit);
    __syncthreads();
    const int st = sh.state;
    if (st != ST_GO) {
      if (st == -1) {
        st_alone<T>(m, w, A + (long)c0 * lda + c0, lda, sh);
        if (t < w) {   // the interchanges followed forth from row t and back from place t
          int f = t, b = sh.piv[t];
          for (int i = 0; i < w; ++i) f = f == i ? sh.piv[i] : f == sh.piv[i] ? i : f;
          for (int i = t - 1; i >= 0; --i) b = b == i ? sh.piv[i] : b == sh.piv[i] ? i : b;
          moved_to[t] = f;
          src[t] = b;
        }
        if (t == 0) st_pivots(c0, w, sh.piv, sh.nz, ipiv + (long)z * sP, info + z);
      }
      return;
    }
  }
  T ya[4], yb[4];   // the row's entries in the chunk: column 4 i + (k + c) % 4 in [c] at step k
#pragma unroll 1
  for (int j = 0; j < PW_; ++j) {
    const int k = j & 3, i = j >> 2;
    if (k == 0) {   // a new chunk
      el = 0;
#pragma unroll
      for (int T_ = 0; T_ < RT; ++T_) { ya[T_] = xr[T_][0][0]; yb[T_] = xi[T_][0][0]; }
      st_transpose(ya);
      st_transpose(yb);
    }
    const int open = 4 - k;   // [0..open-1] are columns j.. of the chunk
    bool nz = false;
    cT P[4], rcp = cT{0, 0};
#pragma unroll
    for (int c = 0; c < 4; ++c) P[c] = cT{0, 0};
    if (j < w) {   // uniform
      const int par = j & 1;
      st_u64 rank = st_rank<T>(live, cT{ya[0], yb[0]});
      int p = pos;
      const int wl = st_wave_best<WIDE>(rank, p);
      if (lane == 0) { sh.rank[par][wave] = rank; sh.pos[par][wave] = p; }
      // each row's reciprocal, in case it is chosen: made while the waves meet
      const bool some = ya[0] != 0 || yb[0] != 0;
      const cT own_rcp = some ? ts_crcp<T>(cT{ya[0], yb[0]}) : cT{0, 0};
      __syncthreads();
      int bw = 0;   // the waves' best
      rank = sh.rank[par][0];
      p = sh.pos[par][0];
#pragma unroll
      for (int v = 1; v < W; ++v)
        if (st_before(sh.rank[par][v], sh.pos[par][v], rank, p)) { rank = sh.rank[par][v]; p = sh.pos[par][v]; bw = v; }
      const bool mine = wave == __builtin_amdgcn_readfirstlane(bw);
      // the row beyond the chunk (needed at the chunk's end only)
      auto hand_rest = [&](cT *own) {
        if (rq == (wl & 15)) {
#pragma unroll
          for (int T_ = 0; T_ < RT; ++T_)
            if (T_ == (wl >> 4)) {   // uniform
#pragma unroll
              for (int q = 1; q < 8; ++q) own[4 * q + cq] = cT{xr[T_][q / 4][q % 4], xi[T_][q / 4][q % 4]};
            }
        }
      };
      if (mine) {   // its wave hands it on
        const unsigned tag = (unsigned)((c0 + j) % 0x1fffff) + 1u;
        st_u64 *cw = gcand + par * G * 2;
        if (G > 1) {
          st_u64 wa, wb;
          st_pack(tag, rank, p, wa, wb);
          if (lane < 2) st_store(cw + 2 * g + lane, lane ? wb : wa);
        }
        cT *own = G > 1 ? sh.own : sh.urow[k];
        if (lane == wl) {
#pragma unroll
          for (int c = 0; c < 4; ++c) own[(k + c) & 3] = cT{ya[c], yb[c]};
          if (G > 1) sh.orcp = own_rcp;
          else sh.rcp[k] = own_rcp;
        }
        if (G > 1) {
          hand_rest(own);
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the row, across the wave's lanes
          __builtin_amdgcn_wave_barrier();
          const int from = st_exchange<T>(g, G, tag, cw, grow + ((i & 1) * 4 + k) * G * NW, sh.orcp, sh.own, sh.rcp[k],
                                          sh.urow[k], rank, p);
          if (lane == 0) { sh.prank = rank; sh.ppos = p; sh.from[k] = from; }
        }
      }
      __syncthreads();
      if (G == 1 && mine) hand_rest(sh.urow[k]);
      if (G > 1) {
        rank = sh.prank;
        p = sh.ppos;
      }
      nz = rank > 2;   // uniform
      if (t == 0) { sh.piv[j] = p; sh.nz[j] = nz; }
#pragma unroll
      for (int c = 0; c < 4; ++c) P[c] = sh.urow[k][(k + c) & 3];
      rcp = sh.rcp[k];
      const bool chosen = live && pos == p;
      if (live && pos == j) pos = p;   // the top row takes the pivot's place
      if (chosen) { live = false; pos = j; }
    }
    {   // the step in the chunk, as a rotation by one
      const bool e = live && nz;
      const T a0 = ya[0], b0 = yb[0];
      const cT l = cmul<T>(cT{a0, b0}, rcp);
#pragma unroll
      for (int c = 1; c < 4; ++c) {
        const cT f = cless<T>(cT{ya[c], yb[c]}, l, P[c]);
        ya[c - 1] = (e && c < open) ? f.x : ya[c];
        yb[c - 1] = (e && c < open) ? f.y : yb[c];
      }
      ya[3] = e ? l.x : a0;
      yb[3] = e ? l.y : b0;
      if (e) el |= 1u << k;
    }
    if (k == 3) {
      T ma[4], mb[4];   // the row's multipliers, zero where it was not eliminated; then the lane's operands
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        ma[c] = ((el >> c) & 1) ? ya[c] : T(0);
        mb[c] = ((el >> c) & 1) ? yb[c] : T(0);
      }
      st_transpose(ya);
      st_transpose(yb);
      if (j + 1 < w) {   // the columns beyond: x -= (multipliers) (U rows)
        if (__ballot(el != 15u) == 0) {
#pragma unroll
          for (int c = 0; c < 4; ++c) { ma[c] = ya[c]; mb[c] = yb[c]; }
        } else {
          st_transpose(ma);
          st_transpose(mb);
        }
        if (G > 1 && wave < 4) {
          const unsigned tag = (unsigned)((c0 + 4 * i + wave) % 0x1fffff) + 1u;
          const st_u64 *src = grow + (((i & 1) * 4 + wave) * G + sh.from[wave]) * NW + st_ew<T>();
#pragma unroll
          for (int e = 0; e < PW_ * st_ew<T>() / 64; ++e) {
            st_u64 v;
            do v = st_load(src + 64 * e + lane); while ((unsigned)(v >> 32) != tag);
            reinterpret_cast<unsigned *>(sh.urow[wave])[64 * e + lane] = (unsigned)v;
          }
        }
        __syncthreads();
        // U rows by substitution with the pivot rows' multipliers, each lane for
        // one column of each half and one row (cq)
        cT L[6];
#pragma unroll
        for (int s = 0, e = 0; s < 3; ++s)
#pragma unroll
          for (int r = s + 1; r < 4; ++r, ++e) {
            const cT v = sh.urow[r][s];
            L[e] = sh.nz[4 * i + s] ? v : cT{0, 0};   // (1,0) (2,0) (3,0) (2,1) (3,1) (3,2)
          }
        // the lane's operand row rq of a product: register rq / 4 of lanes with cq =
        // rq % 4 (FP64), register rq % 4 of lanes with cq = rq / 4 (FP32)
        const int oq = WIDE ? rq >> 2 : rq & 3, oc = WIDE ? rq & 3 : rq >> 2;
        T ur[2], ui[2];
        bool odd = false;   // a value that is no finite number takes part
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
          cT u[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) u[r] = sh.urow[r][4 * (4 * ct + oq) + oc];
          u[1] = cless<T>(u[1], L[0], u[0]);
          u[2] = cless<T>(cless<T>(u[2], L[1], u[0]), L[3], u[1]);
          u[3] = cless<T>(cless<T>(cless<T>(u[3], L[2], u[0]), L[4], u[1]), L[5], u[2]);
          const bool use = 4 * ct + oq > 0 && i + 4 * ct + oq < 8 && sh.nz[4 * i + cq];   // an open column
          ur[ct] = use ? st_own4(cq, u[0].x, u[1].x, u[2].x, u[3].x) : T(0);
          ui[ct] = use ? st_own4(cq, u[0].y, u[1].y, u[2].y, u[3].y) : T(0);
          odd |= !(fabs(ur[ct]) + fabs(ui[ct]) < T(INFINITY));
        }
#pragma unroll
        for (int T_ = 0; T_ < RT; ++T_) odd |= !(fabs(ma[T_]) + fabs(mb[T_]) < T(INFINITY));
        if (__ballot(odd)) {
          // With an infinity or NaN about, a product with zero is not nothing: such
          // factors become zero, and NaN goes to the entries they reach, which a
          // product of zeros and ones finds (a step that eliminates the row, times a
          // bad U entry; a bad multiplier, times an open column).
          unsigned es[4] = {el & 1u, (el >> 1) & 1u, (el >> 2) & 1u, (el >> 3) & 1u};
          st_transpose(es);
#pragma unroll
          for (int ct = 0; ct < 2; ++ct) {
            const bool bad = !(fabs(ur[ct]) + fabs(ui[ct]) < T(INFINITY));
            const T one = (4 * ct + oq > 0 && i + 4 * ct + oq < 8) ? T(1) : T(0);
#pragma unroll
            for (int T_ = 0; T_ < RT; ++T_) {
              const bool badl = !(fabs(ma[T_]) + fabs(mb[T_]) < T(INFINITY));
              acc_t hit = acc_t{0, 0, 0, 0};
              hit = MF<T>::mma(bad ? T(1) : T(0), es[T_] ? T(1) : T(0), hit);
              hit = MF<T>::mma(one, badl ? T(1) : T(0), hit);
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (hit[e] > 0) xr[T_][ct][e] = xi[T_][ct][e] = T(NAN);
            }
            if (bad) ur[ct] = ui[ct] = 0;
          }
#pragma unroll
          for (int T_ = 0; T_ < RT; ++T_)
            if (!(fabs(ma[T_]) + fabs(mb[T_]) < T(INFINITY))) ma[T_] = mb[T_] = 0;
        }
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
          if (ct == 1 && i >= 4) continue;   // finished columns (uniform)
#pragma unroll
          for (int T_ = 0; T_ < RT; ++T_) {   // the four products' sum, then one rounding of x's size
            acc_t pr = acc_t{0, 0, 0, 0}, pi = pr;
            pr = MF<T>::mma(ur[ct], ma[T_], pr);
            pi = MF<T>::mma(ui[ct], ma[T_], pi);
            pr = MF<T>::mma(-ui[ct], mb[T_], pr);
            pi = MF<T>::mma(ur[ct], mb[T_], pi);
            xr[T_][ct] -= pr;
            xi[T_][ct] -= pi;
            if (WIDE) __builtin_amdgcn_sched_barrier(0);   // else more sums at a time than registers
          }
        }
      }
      // the finished chunk goes behind the others; the pins keep the rotation in
      // place (as a parallel move it took a second set of registers)
#pragma unroll
      for (int T_ = 0; T_ < RT; ++T_) {
#pragma unroll
        for (int q = 0; q < 7; ++q) {
          xr[T_][q / 4][q % 4] = xr[T_][(q + 1) / 4][(q + 1) % 4];
          xi[T_][q / 4][q % 4] = xi[T_][(q + 1) / 4][(q + 1) % 4];
        }
        xr[T_][1][3] = ya[T_];
        xi[T_][1][3] = yb[T_];
        asm("" : "+v"(xr[T_][0]), "+v"(xr[T_][1]), "+v"(xi[T_][0]), "+v"(xi[T_][1]));
      }
    }
  }
  unsigned at[4] = {(unsigned)pos, (unsigned)pos, (unsigned)pos, (unsigned)pos};
  st_transpose(at);   // [T] = the position of row rq of tile T
#pragma unroll
  for (int T_ = 0; T_ < RT; ++T_)
    if (row0 + 16 * T_ + rq < m) {
      cT *row = A + (long)(c0 + (int)at[T_]) * lda + c0;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (4 * i + cq < w) row[4 * i + cq] = cT{xr[T_][i / 4][i % 4], xi[T_][i / 4][i % 4]};
    }
  if (live_row && pos < w) src[pos] = row0 + lane;
  if (live_row && row0 + lane < w) moved_to[row0 + lane] = pos;
  if (g == 0 && t == 0) st_pivots(c0, w, sh.piv, sh.nz, ipiv + (long)z * sP, info + z);
}

// Row interchanges of strips as gathers A[c0 + to] = A[c0 + from] over their
// moved rows, per block of AP_COLS columns: every moved entry is loaded into
// registers, then (after a barrier) stored.
//   k_ts_apply:  a tournament strip on its own columns, then its L11\U11;
//   k_ts_apply_defer: the strips of an outer block (slots 0..nslots-1, strip
//                c0 = K0 + PW slot, in order) on every column outside
//                [skip_lo, skip_hi).
constexpr int AP_COLS = 32;
template <class T>
__device__ __forceinline__ void ts_gather(int n, int c0, const char *fin, typename C2<T>::t *A, long lda, int j0,
                                          int *from, int *to, int *count, bool colok) {
  typedef typename C2<T>::t cT;
  const int t = threadIdx.x;
  if (t < 64) {   // lanes 0..31: what comes to the top; 32..63: what leaves it
    const int *src = reinterpret_cast<const int *>(fin), *dst = src + PW_, w = min(PW_, n - c0), i = t & (PW_ - 1);
    const int f = t < PW_ ? (i < w ? src[i] : i) : i, d = t < PW_ ? i : (i < w ? dst[i] : i);
    const bool mv = t < PW_ ? f != d : d >= w && i < w;
    const unsigned long long mm = __ballot(mv);
    const int slot = __popcll(mm & ((1ull << t) - 1ull));
    if (mv) { from[slot] = f; to[slot] = d; }
    if (t == 0) *count = __popcll(mm);
  }
  __syncthreads();
  const int k = *count;
  const int c = t % AP_COLS, r4 = t / AP_COLS;
  constexpr int RP = 256 / AP_COLS, NQ = 2 * PW_ / RP;   // rows per pass; passes over the longest list
  cT v[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {   // every load in flight, then (after the barrier) every store
    const int e = r4 + RP * q;
    v[q] = (colok && e < k) ? A[(long)(c0 + from[e]) * lda + j0 + c] : cT{0, 0};
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int e = r4 + RP * q;
    if (colok && e < k) A[(long)(c0 + to[e]) * lda + j0 + c] = v[q];
  }
  __syncthreads();
}

template <class T>
__global__ __launch_bounds__(256) void k_ts_apply(int n, int c0, int w, typename C2<T>::t *A, long lda, const char *fin) {
  typedef typename C2<T>::t cT;
  __shared__ int from[2 * PW_], to[2 * PW_], count;
  const int t = threadIdx.x, c = t % AP_COLS, r4 = t / AP_COLS;
  const bool colok = c < w;
  ts_gather<T>(n, c0, fin, A, lda, c0, from, to, &count, colok);
  const cT *lu = reinterpret_cast<const cT *>(fin + PanelWS<T>::LU_OFF);
  if (colok)
    for (int i = r4; i < w; i += 256 / AP_COLS) A[(long)(c0 + i) * lda + c0 + c] = lu[i * PW_ + c];
}

template <class T>
__global__ __launch_bounds__(256) void k_ts_apply_defer(int n, int K0, int nslots, typename C2<T>::t *A, long lda,
                                                        long sA, const char *fin0, long finb, long sW, int skip_lo,
                                                        int skip_hi) {
  __shared__ int from[2 * PW_], to[2 * PW_], count;
  const int z = blockIdx.z, j0 = blockIdx.x * AP_COLS;
  if (j0 >= skip_lo && j0 + AP_COLS <= skip_hi) return;   // whole block inside the skipped columns (uniform)
  A += (long)z * sA;
  fin0 += (long)z * sW;
  const int c = threadIdx.x % AP_COLS;
  const bool colok = j0 + c < n && (j0 + c < skip_lo || j0 + c >= skip_hi);
  for (int q = 0; q < nslots; ++q) ts_gather<T>(n, K0 + PW_ * q, fin0 + q * finb, A, lda, j0, from, to, &count, colok);
}

// Forward substitution with a unit lower 32 x 32 block for the 16 columns of a
// wave, four lanes per column (lane = 4 column + class): x[q] is row 4 q + class.
// Each step's solved entry goes round its four lanes by DPP. The rolled loop
// over groups of four rows keeps the group at hand in x[0] and hands it to
// out(kb, value) when it is done. A thread per column instead has 496 dependent
// updates in a row; a product with the inverse needs the inverse (26 us for the
// launch that made it).
// lane class K's value
template <int K> __device__ __forceinline__ unsigned su_dpp(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, K * 0x55, 0xF, 0xF, true);
}
template <int K> __device__ __forceinline__ float su_bc(float v) { return __uint_as_float(su_dpp<K>(__float_as_uint(v))); }
template <int K> __device__ __forceinline__ double su_bc(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = su_dpp<K>((unsigned)b), hi = su_dpp<K>((unsigned)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
constexpr int SU_LS = PW_ + 1;   // LDS row stride of the lower block
template <class T, class Out>
__device__ __forceinline__ void su_solve(const typename C2<T>::t *L, int cls, typename C2<T>::t (&x)[8], Out out) {
  typedef typename C2<T>::t cT;
  cT less[8];   // the rows' products so far, subtracted as a sum: one rounding of x's size
#pragma unroll
  for (int q = 0; q < 8; ++q) less[q] = cT{0, 0};
#pragma unroll 1
  for (int kb = 0; kb < 8; ++kb) {
    auto step = [&](auto kc) {
      constexpr int K = decltype(kc)::value;
      const cT w = x[0] - less[0], v = cT{su_bc<K>(w.x), su_bc<K>(w.y)};
      const int k = 4 * kb + K;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (q >= 8 - kb) continue;   // rows beyond the block (uniform)
        const cT l = L[(4 * (kb + q) + cls) * SU_LS + k];
        const cT y = cT{fma(l.x, v.x, fma(-l.y, v.y, less[q].x)), fma(l.x, v.y, fma(l.y, v.x, less[q].y))};
        if (q > 0 || cls > K) less[q] = y;
      }
    };
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 3>{});
    out(kb, x[0] - less[0]);
#pragma unroll
    for (int q = 0; q < 7; ++q) {
      x[q] = x[q + 1];
      less[q] = less[q + 1];
    }
  }
}

// A strip's interchanges on the block's other columns [lo, hi), and U = L11^{-1}
// A12 on those behind the strip: 64 columns per workgroup, 16 per wave. The
// first nl workgroups take the columns before the strip, the others those
// behind; workgroup 0 also brings perm up to date.
template <class T>
__global__ __launch_bounds__(256) void k_swap_u(int n, int c0, int w, typename C2<T>::t *A, long lda, long sA,
                                                const char *fin, long sW, int lo, int hi, int nl, int *perm, long sP) {
  typedef typename C2<T>::t cT;
  __shared__ __align__(16) cT L[PW_ * SU_LS];
  const int z = blockIdx.z, b = blockIdx.x, t = threadIdx.x, lane = t & 63, cls = lane & 3;
  A += (long)z * sA;
  fin += (long)z * sW;
  const int *src = reinterpret_cast<const int *>(fin), *to = src + PW_;
  if (b == 0 && perm && t < 2 * PW_) {
    int *pz = perm + (long)z * sP + c0;
    const int i = t & (PW_ - 1);
    const bool mv = i < w && (t < PW_ || to[i] >= w);
    const int f = mv ? (t < PW_ ? src[i] : i) : 0, d = mv ? (t < PW_ ? i : to[i]) : 0;
    const int v = mv ? pz[f] : 0;   // one wave: every lane loads before any stores
    __builtin_amdgcn_s_waitcnt(0);
    if (mv) pz[d] = v;
  }
  const bool behind = b >= nl;
  const int col = (behind ? c0 + w + (b - nl) * 64 : lo + b * 64) + (t >> 6) * 16 + (lane >> 2);
  const bool ok = col < (behind ? hi : c0);
  if (behind)
    for (int e = t; e < PW_ * PW_; e += 256) {
      const int i = e / PW_, k = e % PW_;
      L[i * SU_LS + k] = (i < w && k < i) ? A[(long)(c0 + i) * lda + c0 + k] : cT{0, 0};
    }
  cT x[8], y[8];   // rows 4 q + cls of the new top, and of the old top where they leave it
  int d[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int i = 4 * q + cls;
    const bool in = ok && i < w;
    const int s = in ? src[i] : 0;
    d[q] = in ? to[i] : 0;
    x[q] = in ? A[(long)(c0 + s) * lda + col] : cT{0, 0};
    y[q] = in && d[q] >= w ? A[(long)(c0 + i) * lda + col] : cT{0, 0};
  }
  __builtin_amdgcn_s_waitcnt(0);   // the four lanes of a column read each other's rows: all loads are done
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (ok && d[q] >= w) A[(long)(c0 + d[q]) * lda + col] = y[q];
  auto put = [&](int q, cT v) {
    const int i = 4 * q + cls;
    if (ok && i < w) A[(long)(c0 + i) * lda + col] = v;
  };
  if (behind) {
    su_solve<T>(L, cls, x, put);
  } else {
#pragma unroll
    for (int q = 0; q < 8; ++q) put(q, x[q]);
  }
}

// U12 = L11^{-1} A12 of an outer block (nb <= 256 rows at A, unit lower L in the
// columns before them) for 16 columns per workgroup, held in LDS for the whole
// solve: per 32 rows one wave substitutes (su_solve), then the four waves
// subtract L21 times the solved rows from the rows below with matrix
// instructions, L read as operands straight from the matrix (all workgroups
// read the same 512 KB). As eight products with inverses and seven updates it
// was 15 dependent launches, about 200 us per block.
constexpr int U12_C = 16, U12_XS = U12_C + 1;
template <class T> constexpr size_t u12_lds() { return (size_t)(256 * U12_XS + PW_ * SU_LS) * sizeof(typename C2<T>::t); }
template <class T>
__global__ __launch_bounds__(256) void k_u12(int nb, int ncols, const typename C2<T>::t *Lm, long lda, long sA,
                                             typename C2<T>::t *B) {
  typedef typename C2<T>::t cT;
  typedef typename MF<T>::acc acc_t;
  extern __shared__ __align__(16) char smem_raw[];
  cT *X = reinterpret_cast<cT *>(smem_raw), *L = X + 256 * U12_XS;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, j0 = blockIdx.x * U12_C, nc = min(U12_C, ncols - j0);
  Lm += (long)blockIdx.z * sA;
  B += (long)blockIdx.z * sA + j0;
  {
    const int c = t % U12_C, r = t / U12_C;
    cT v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = (c < nc && r + 16 * q < nb) ? B[(long)(r + 16 * q) * lda + c] : cT{0, 0};
#pragma unroll
    for (int q = 0; q < 16; ++q) X[(r + 16 * q) * U12_XS + c] = v[q];
  }
  const int lr = lane & 15, lk = lane >> 4;
  for (int s = 0; s < nb; s += PW_) {
    const int w = min(PW_, nb - s);
#pragma unroll
    for (int e = t; e < PW_ * PW_; e += 256) {
      const int i = e / PW_, k = e % PW_;
      L[i * SU_LS + k] = (i < w && k < i) ? Lm[(long)(s + i) * lda + s + k] : cT{0, 0};
    }
    __syncthreads();
    if (wave == 0) {
      const int cls = lane & 3, c = lane >> 2;
      cT x[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) x[q] = X[(s + 4 * q + cls) * U12_XS + c];
      su_solve<T>(L, cls, x, [&](int q, cT v) { X[(s + 4 * q + cls) * U12_XS + c] = v; });
    }
    __syncthreads();
    for (int r0 = s + PW_ + 16 * wave; r0 < nb; r0 += 64) {   // 16 rows at a time
      cT a[8];
#pragma unroll
      for (int q = 0; q < 8; ++q)
        a[q] = (r0 + lr < nb) ? Lm[(long)(r0 + lr) * lda + s + 4 * q + lk] : cT{0, 0};
      acc_t pr = acc_t{0, 0, 0, 0}, pi = acc_t{0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const cT b = X[(s + 4 * q + lk) * U12_XS + lr];
        pr = MF<T>::mma(a[q].x, b.x, pr);
        pi = MF<T>::mma(a[q].x, b.y, pi);
        pr = MF<T>::mma(-a[q].y, b.y, pr);
        pi = MF<T>::mma(a[q].y, b.x, pi);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        cT &x = X[(r0 + MF<T>::row(lk, e)) * U12_XS + lr];
        x = cT{x.x - pr[e], x.y - pi[e]};
      }
    }
    __syncthreads();
  }
  const int c = t % U12_C;
  for (int r = t / U12_C; r < nb; r += 16)
    if (c < nc) B[(long)r * lda + c] = X[r * U12_XS + c];
}

// ---------------------------------------------------------------------------
// Trailing update C -= A B of the LU (M x N x K = n-k x n-k x 256): a plain
// complex GEMM, handed to rocBLAS (cgemm / zgemm on MFMA, FP32 or FP64
// accumulation) when it is large; k_gemm_sub otherwise, or everywhere with
// QPMS_HIP_GEMM=own. Row-major C = A B is column-major C^T = B^T A^T.
// ---------------------------------------------------------------------------
static bool use_rocblas() {
  static int v = -1;
  if (v < 0) {
    const char *e = getenv("QPMS_HIP_GEMM");
    v = !(e && !strcmp(e, "own"));
  }
  return v == 1;
}

// Per-stream state of the LU driver: a rocBLAS handle bound to the stream, the
// lookahead's two events, and the workspace of callers that bring none. Created
// on a stream's first use; qh_stream_release() destroys it, and callers that
// destroy a stream (the serving loop's lanes) must call it first, so that a later
// stream created at the same address never inherits a dead stream's state.
struct LaCtx {
  hipEvent_t go, done;   // ordering of the caller's stream against the device's side stream
};

constexpr int STREAM_TAB = 64;
struct StreamState {
  hipStream_t key;
  rocblas_handle blas;   // nullptr until the first library GEMM on the stream
  bool la;               // lookahead context created
  LaCtx lc;
  char *ws;              // see ws_for
  size_t ws_bytes;
};
static std::mutex g_tab_mu;
static StreamState g_tab[STREAM_TAB];
static int g_ntab = 0;

static StreamState *state_for(hipStream_t s) {   // caller holds g_tab_mu
  for (int i = 0; i < g_ntab; ++i) if (g_tab[i].key == s) return &g_tab[i];
  if (g_ntab == STREAM_TAB)
    qpms_hip_die(__FILE__, __LINE__, __func__, "more than %d live streams use the LU (release them)", STREAM_TAB);
  StreamState &e = g_tab[g_ntab++];
  e = StreamState{};
  e.key = s;
  return &e;
}

static rocblas_handle blas_for(hipStream_t s) {
  std::lock_guard<std::mutex> g(g_tab_mu);
  StreamState *e = state_for(s);
  if (!e->blas) {
    rocblas_handle h;
    if (rocblas_create_handle(&h) != rocblas_status_success)
      qpms_hip_die(__FILE__, __LINE__, __func__, "rocblas_create_handle failed");
    if (rocblas_set_stream(h, s) != rocblas_status_success)
      qpms_hip_die(__FILE__, __LINE__, __func__, "rocblas_set_stream failed");
    e->blas = h;
  }
  return e->blas;
}

// Workspace of the factorisations on a stream whose callers bring none. It holds
// words that a strip's workgroups wait on, so no two streams may share one.
static char *ws_for(hipStream_t s, size_t bytes) {
  std::lock_guard<std::mutex> g(g_tab_mu);
  StreamState *e = state_for(s);
  if (bytes > e->ws_bytes) {
    HIPCHK(hipStreamSynchronize(s));   // earlier factorisations may use it
    qh_dfree(e->ws);
    e->ws = (char *)qh_dmalloc(bytes);
    e->ws_bytes = bytes;
  }
  return e->ws;
}

// CUs kept free of the side stream's trailing update, so that the next
// block's strips (latency-bound launches of tens of workgroups, launched as
// whole-CU workgroups) find CUs while it runs: QPMS_HIP_LU_RESERVE (default
// 32; 0: no CU mask, the strips then wait for CUs to drain).
static int lu_reserve_cus() {
  static int v = -1;
  if (v < 0) {
    const char *e = getenv("QPMS_HIP_LU_RESERVE");
    v = e ? std::max(0, atoi(e)) : 32;
  }
  return v;
}

// The side stream of the lookahead: one per device for the whole process,
// masked to all CUs but the reserved ones, shared by every caller stream (the
// bulk updates of concurrent factorisations queue on it, each ordered against
// its own caller by that caller's events). Every further hardware queue
// costs: with several masked side streams alive, factorisations measured up
// to 1.6 x slower, depending on the order the queues were created in.
constexpr int LA_MAX_DEV = 64;
static hipStream_t g_la_side[LA_MAX_DEV];
static bool g_la_masked[LA_MAX_DEV];
static hipStream_t la_side(bool *masked) {   // caller holds g_tab_mu
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= LA_MAX_DEV) qpms_hip_die(__FILE__, __LINE__, __func__, "device %d outside the table", dev);
  if (!g_la_side[dev]) {
    const int reserve = lu_reserve_cus();
    int ncu = 0;
    HIPCHK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    if (reserve > 0 && ncu > 2 * reserve && ncu <= 32 * 32) {
      uint32_t mask[32] = {0};
      for (int i = 0; i < ncu - reserve; ++i) mask[i / 32] |= 1u << (i % 32);
      HIPCHK(hipExtStreamCreateWithCUMask(&g_la_side[dev], (uint32_t)((ncu + 31) / 32), mask));
      g_la_masked[dev] = true;
    } else {
      HIPCHK(hipStreamCreateWithFlags(&g_la_side[dev], hipStreamNonBlocking));
      g_la_masked[dev] = false;
    }
  }
  *masked = g_la_masked[dev];
  return g_la_side[dev];
}

// Lookahead context of a caller stream: its two events (created on first use).
static LaCtx *la_for(hipStream_t s, hipStream_t *side, bool *masked) {
  std::lock_guard<std::mutex> g(g_tab_mu);
  StreamState *e = state_for(s);
  if (!e->la) {
    HIPCHK(hipEventCreateWithFlags(&e->lc.go, hipEventDisableTiming));
    HIPCHK(hipEventCreateWithFlags(&e->lc.done, hipEventDisableTiming));
    e->la = true;
  }
  *side = la_side(masked);
  return &e->lc;
}

// Destroys the per-stream state of `stream` (rocBLAS handle, lookahead events,
// workspace), after waiting for its work on the shared side stream.
extern "C" void qh_stream_release(void *stream) {
  hipStream_t s = (hipStream_t)stream;
  std::lock_guard<std::mutex> g(g_tab_mu);
  for (int i = 0; i < g_ntab; ++i) {
    if (g_tab[i].key != s) continue;
    StreamState &e = g_tab[i];
    if (e.la) {   // the caller's own work on the shared side stream ends before its events go
      HIPCHK(hipEventSynchronize(e.lc.done));
      HIPCHK(hipEventDestroy(e.lc.go));
      HIPCHK(hipEventDestroy(e.lc.done));
    }
    if (e.blas) rocblas_destroy_handle(e.blas);
    qh_dfree(e.ws);   // waits for what uses it
    g_tab[i] = g_tab[--g_ntab];
    return;
  }
}

// Number of streams with live per-stream state (tests check that servers
// release theirs).
extern "C" int qh_stream_state_count(void) {
  std::lock_guard<std::mutex> g(g_tab_mu);
  return g_ntab;
}

static bool stream_capturing(hipStream_t s) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(s, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone;
}

template <class T>
static void trailing_gemm(int M, int N, int K, int batch, const typename C2<T>::t *A, long lda, long sA,
                          const typename C2<T>::t *B, long ldb, long sB, typename C2<T>::t *C, long ldc, long sC,
                          hipStream_t s, bool own_only = false) {
  if (M <= 0 || N <= 0 || K <= 0) return;
  // inside a captured graph only hand-written kernels (a library call may
  // record allocations or memsets into the graph)
  const bool capturing = stream_capturing(s);
  if (capturing) own_only = true;
  if (sizeof(T) == 4 && (!own_only || capturing)) {
    // FP32: the variant the autotuner picked for this size class
    int v = qh_lu_gemm_variant(M, N, batch > 1);
    if (v == 0 && capturing) v = qh_lu_gemm_best_own(M, N, batch > 1);
    qh_lu_gemm_run(v, M, N, K, batch, (const float *)A, lda, sA, (const float *)B, ldb, sB, (float *)C, ldc, sC,
                   v == 0 ? (void *)blas_for(s) : nullptr, s);
    return;
  }
  if (own_only || !use_rocblas() || (long)M * N < 512L * 512) {
    QH_LAUNCH(k_gemm_sub<T>, dim3((N + GT - 1) / GT, (M + GT - 1) / GT, batch), dim3(256), 0, s, M, N, K, A,
                       lda, sA, B, ldb, sB, C, ldc, sC);
    return;
  }
  rocblas_handle h = blas_for(s);
  rocblas_status st;
  if (sizeof(T) == 4) {
    const rocblas_float_complex al = {-1.f, 0.f}, be = {1.f, 0.f};
    st = rocblas_cgemm_strided_batched(h, rocblas_operation_none, rocblas_operation_none, N, M, K, &al,
                                       (const rocblas_float_complex *)B, (rocblas_int)ldb, sB,
                                       (const rocblas_float_complex *)A, (rocblas_int)lda, sA, &be,
                                       (rocblas_float_complex *)C, (rocblas_int)ldc, sC, batch);
  } else {
    const rocblas_double_complex al = {-1.0, 0.0}, be = {1.0, 0.0};
    st = rocblas_zgemm_strided_batched(h, rocblas_operation_none, rocblas_operation_none, N, M, K, &al,
                                       (const rocblas_double_complex *)B, (rocblas_int)ldb, sB,
                                       (const rocblas_double_complex *)A, (rocblas_int)lda, sA, &be,
                                       (rocblas_double_complex *)C, (rocblas_int)ldc, sC, batch);
  }
  if (st != rocblas_status_success)
    qpms_hip_die(__FILE__, __LINE__, __func__, "rocBLAS GEMM failed (status %d)", (int)st);
}

constexpr int LU_NB = 256;   // outer block: K of the trailing GEMM
static_assert(LU_NB / PW_ == TS_SLOTS, "one output slot per strip of an outer block");

static bool use_lookahead() {
  static int v = -1;
  if (v < 0) {
    const char *e = getenv("QPMS_HIP_LU_LOOKAHEAD");
    v = !(e && !strcmp(e, "0"));
  }
  return v == 1;
}

// C -= A B (or C = A B, ASSIGN) for K <= PW: the products of strips (the
// in-block rank-PW update, L21 = A21 U11^{-1} after a tournament) that run as
// whole-CU workgroups, beside the trailing update (one workgroup per CU).
// The workgroup is gcu_q quarters of 256 threads, each quarter on its own
// 64 x 64 tile of C, so that a CU has that many tiles in flight; a tile's A
// (64 x K) and B (K x 64) are staged whole (one load round trip for the
// products instead of one per GK slice), and the waves of the quarters hide
// each other's latency. The quarters step through groups of tiles together
// (every barrier is reached by all of them; a quarter past the last tile
// loads and stores nothing).
template <class T> constexpr int gcu_q() { return sizeof(T) == 4 ? 4 : 2; }
template <class T> constexpr size_t gcu_quarter_lds() {
  return (size_t)(2 * GT * (PW_ + 1) + 2 * PW_ * (GT + 1)) * sizeof(T);
}
template <class T> constexpr size_t gcu_lds() { return gcu_q<T>() * gcu_quarter_lds<T>(); }

template <class T, bool ASSIGN>
__global__ __launch_bounds__(gcu_q<T>() * 256) void k_gemm_cu(int M, int N, int K, const typename C2<T>::t *A,
                                                               long lda, const typename C2<T>::t *B, long ldb,
                                                               typename C2<T>::t *C, long ldc) {
  typedef typename C2<T>::t cT;
  typedef typename MF<T>::acc acc_t;
  constexpr int Q = gcu_q<T>(), AS = PW_ + 1, BS = GT + 1;
  extern __shared__ __align__(16) char smem_raw[];
  const int sub = threadIdx.x >> 8, tid = threadIdx.x & 255, lane = tid & 63, wv = tid >> 6;
  T *Ar = reinterpret_cast<T *>(smem_raw + sub * gcu_quarter_lds<T>());
  T *Ai = Ar + GT * AS, *Br = Ai + GT * AS, *Bi = Br + PW_ * BS;
  const int wm = (wv >> 1) * 32, wn = (wv & 1) * 32;   // wave quadrant of the tile
  const int lr = lane & 15, lk = lane >> 4;
  const int tn = (N + GT - 1) / GT, nt = ((M + GT - 1) / GT) * tn, ngrp = (nt + Q - 1) / Q;
  for (int g = blockIdx.x; g < ngrp; g += gridDim.x) {
    const int tile = g * Q + sub;
    const bool valid = tile < nt;
    const int m0 = valid ? (tile / tn) * GT : M, n0 = valid ? (tile % tn) * GT : N;
    cT va[GT * PW_ / 256], vb[PW_ * GT / 256];
#pragma unroll
    for (int e = 0; e < GT * PW_ / 256; ++e) {
      const int idx = tid + 256 * e;
      const int ar = idx / PW_, ak = idx % PW_, bk = idx / GT, bn = idx % GT;
      va[e] = (m0 + ar < M && ak < K) ? A[(long)(m0 + ar) * lda + ak] : cT{0, 0};
      vb[e] = (bk < K && n0 + bn < N) ? B[(long)bk * ldb + n0 + bn] : cT{0, 0};
    }
    __syncthreads();   // the previous group's reads of the tiles are done
#pragma unroll
    for (int e = 0; e < GT * PW_ / 256; ++e) {
      const int idx = tid + 256 * e;
      const int ar = idx / PW_, ak = idx % PW_, bk = idx / GT, bn = idx % GT;
      Ar[ar * AS + ak] = va[e].x;
      Ai[ar * AS + ak] = va[e].y;
      Br[bk * BS + bn] = vb[e].x;
      Bi[bk * BS + bn] = vb[e].y;
    }
    __syncthreads();
    acc_t pr[2][2], pi[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) { pr[a][b] = acc_t{0, 0, 0, 0}; pi[a][b] = acc_t{0, 0, 0, 0}; }
#pragma unroll
    for (int kk = 0; kk < PW_; kk += 4) {
      if (kk >= K) break;   // uniform; entries past K are zero
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const T ar = Ar[(wm + a * 16 + lr) * AS + kk + lk], ai = Ai[(wm + a * 16 + lr) * AS + kk + lk];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const T br = Br[(kk + lk) * BS + wn + b * 16 + lr], bi = Bi[(kk + lk) * BS + wn + b * 16 + lr];
          pr[a][b] = MF<T>::mma(ar, br, pr[a][b]);
          pr[a][b] = MF<T>::mma(-ai, bi, pr[a][b]);
          pi[a][b] = MF<T>::mma(ar, bi, pi[a][b]);
          pi[a][b] = MF<T>::mma(ai, br, pi[a][b]);
        }
      }
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = m0 + wm + a * 16 + MF<T>::row(lk, i), col = n0 + wn + b * 16 + lr;
          if (row < M && col < N) {
            if (ASSIGN) {
              C[(long)row * ldc + col] = cT{pr[a][b][i], pi[a][b][i]};
            } else {
              const cT c = C[(long)row * ldc + col];
              C[(long)row * ldc + col] = cT{c.x - pr[a][b][i], c.y - pi[a][b][i]};
            }
          }
        }
  }
}

// Strips that run beside the side stream's trailing update launch every
// kernel with a dynamic-LDS request that fills the rest of a CU's 160 KB, so
// that none of their workgroups shares a CU with a GEMM workgroup (they would
// get a small share of its issue slots); they then run on the CUs the side
// stream's mask leaves free. The request per kernel is set once with its
// dynamic-LDS limit, from the kernel's static LDS.
constexpr size_t CU_LDS = (size_t)160 << 10;
static size_t whole_cu_lds(const void *fn) {
  hipFuncAttributes at;
  HIPCHK(hipFuncGetAttributes(&at, fn));
  const size_t stat = at.sharedSizeBytes;
  const size_t pad = (CU_LDS > stat + 512 ? CU_LDS - stat - 512 : 0) / 256 * 256;
  if (pad > 0) HIPCHK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)pad));
  return pad;
}
template <class T>
struct WholeCu {   // dynamic-LDS requests of the strip kernels for whole-CU launches
  size_t local, merge, apply, gemm_assign, gemm_sub, strip, swap_u;
};
template <class T>
static const WholeCu<T> &whole_cu() {
  static WholeCu<T> w;
  static std::once_flag once;
  std::call_once(once, [] {
    w.local = std::max(whole_cu_lds((const void *)k_ts_local<T>), ts_lds<T>());
    w.merge = std::max(whole_cu_lds((const void *)k_ts_merge<T>), ts_lds<T>());
    w.apply = whole_cu_lds((const void *)k_ts_apply<T>);
    w.gemm_assign = std::max(whole_cu_lds((const void *)k_gemm_cu<T, true>), gcu_lds<T>());
    w.gemm_sub = std::max(whole_cu_lds((const void *)k_gemm_cu<T, false>), gcu_lds<T>());
    w.strip = whole_cu_lds((const void *)k_strip<T>);
    w.swap_u = whole_cu_lds((const void *)k_swap_u<T>);
  });
  return w;
}

// The tournament kernels stage a chunk of more than 64 KB of LDS: raise
// their dynamic-LDS limit once (before any launch sequence is captured).
template <class T>
static void ts_prepare() {
  static std::once_flag once;
  std::call_once(once, [] {
    HIPCHK(hipFuncSetAttribute((const void *)k_ts_local<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)ts_lds<T>()));
    HIPCHK(hipFuncSetAttribute((const void *)k_ts_merge<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)ts_lds<T>()));
  });
  (void)whole_cu<T>();   // raises the limits further for whole-CU launches
  static std::once_flag u12;
  std::call_once(u12, [] {
    HIPCHK(hipFuncSetAttribute((const void *)k_u12<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)u12_lds<T>()));
  });
}

extern "C" void qh_cgemm3m_prepare(void);
// Every kernel attribute the LU paths set, set now (the serving loop calls
// this at creation, before it captures any launch sequence into a graph).
template <class T> static void tr_prepare();
extern "C" void qh_lu_prepare(void) {
  ts_prepare<float>();
  ts_prepare<double>();
  tr_prepare<float>();
  tr_prepare<double>();
  qh_cgemm3m_prepare();
}

// Most workgroups of a strip that wait for one another: those of a quarter of the
// device (64 CUs, two FP64 workgroups or one FP32 one each), as for the slabs of the
// solves, so that of four hardware queues' launches one is always complete. Beside a
// trailing update, as many as CUs are kept free of it. (Two strips that share those
// end with the update: the side stream's next one waits for one of them.)
template <class T>
static int strip_most(bool beside) {
  return beside ? lu_reserve_cus() : sizeof(T) == 8 ? 128 : 64;
}
// Whether a factorisation may use the tournament for some of its blocks (see
// getrf_batched): single matrices with strips of more workgroups than that.
template <class T>
static bool may_tournament(int n, int batch, bool pp, int most) {
  return !pp && batch == 1 && (st_groups<T>(n) > most || (use_lookahead() && st_groups<T>(n) > strip_most<T>(true)));
}
// Workspace of one matrix: the strips' words, the tournament's two candidate
// buffers (the second holds the first merge level's output, a set per workgroup
// of fan-in sets) where it may be used, the output slots.
template <class T>
struct LuWS {
  size_t strip, buf_a, buf_b, fin, bytes;   // offsets, total
  LuWS(int n, int batch, bool pp, int most = strip_most<T>(false)) {
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    const size_t sets = may_tournament<T>(n, batch, pp, most) ? (size_t)PanelWS<T>::sets(n) : 0;
    strip = 0;
    buf_a = up((size_t)st_ws_bytes<T>(n));
    buf_b = buf_a + sets * PanelWS<T>::set_bytes();
    fin = buf_b + (sets + ts_fan<T>() - 1) / ts_fan<T>() * PanelWS<T>::set_bytes();
    bytes = fin + up(TS_SLOTS * PanelWS<T>::fin_bytes());
  }
};
// Workspace bytes for getrf_batched<T>(n, batch).
template <class T>
static size_t getrf_ws_bytes(int n, int batch) {
  return (size_t)batch * LuWS<T>(n, batch, false).bytes;
}

// Blocked right-looking LU of `batch` n x n matrices (stride sA), in place. Outer
// blocks of LU_NB columns; inside a block the columns are factorised PW at a time
// (k_strip), the block's remaining columns updated by substitution (k_swap_u) and a
// GEMM (K = PW); then U12 = L11^{-1} A12 in one launch (k_u12), and the trailing A22
// -= L21 U12 (K = LU_NB).
// ipiv (1-based, stride sP) lists the row interchanges as zgetrf's does;
// perm (optional) tracks P; info[z] gets the first zero pivot. ws: the call's own
// until its work is done, LuWS<T>(n, batch, pp, most).bytes per matrix.
template <class T>
static void getrf_batched(int n, int batch, typename C2<T>::t *A, long lda, long sA, int *ipiv, long sP,
                          int *perm, int *dinfo, hipStream_t s, char *ws, bool lookahead = true,
                          bool own_gemm = false, bool pp = false, st_u64 wait = ST_LIMIT,
                          int most = strip_most<T>(false)) {
  typedef typename C2<T>::t cT;
  constexpr int PW = PanelW<T>::W;
  const dim3 b256(256);
  if (n <= 0 || batch <= 0) return;
  if (n >= (1 << 22)) qpms_hip_die(__FILE__, __LINE__, __func__, "order %d above the pivot search's 2^22 rows", n);
  const LuWS<T> lay(n, batch, pp, most);
  const long sW = (long)lay.bytes;
  const long setb = (long)PanelWS<T>::set_bytes();
  const dim3 bts(TS_THREADS);
  ts_prepare<T>();
  char *bufA = ws + lay.buf_a, *bufB = ws + lay.buf_b, *fin0 = ws + lay.fin;
  const long finb = (long)PanelWS<T>::fin_bytes();
  QH_LAUNCH(k_strip_init, dim3((unsigned)std::min((st_ws_bytes<T>(n) / 8 + 255) / 256, 1024L), 1, batch), b256, 0, s, ws,
            sW, st_ws_bytes<T>(n));
  // The strips of the outer block [k0, k0 + nb): pivots, interchanges on the
  // block's own columns, L21, then the block's remaining columns by TRSM and the
  // rank-w update. Touches only the block's columns (rows >= k0). wcu: beside a
  // trailing update, as whole-CU workgroups. Strips of more workgroups than
  // strip_most go by tournament, whose workgroups do not wait for each other
  // (single matrices, where the caller leaves the pivots to the library).
  auto block_strips = [&](int k0, int nb, hipStream_t st, bool wcu) {
    constexpr int F = ts_fan<T>();
    const bool tour = !pp && batch == 1 && st_groups<T>(n - k0) > (wcu ? strip_most<T>(true) : most);
    const WholeCu<T> &W = whole_cu<T>();
    const dim3 bcu(gcu_q<T>() * 256);
    auto gcu_grid = [](int M, int N) {
      const int nt = ((M + GT - 1) / GT) * ((N + GT - 1) / GT);
      return dim3(std::min((nt + gcu_q<T>() - 1) / gcu_q<T>(), 4096));
    };
    for (int j0 = 0; j0 < nb; j0 += PW) {
      const int w = min(PW, nb - j0), c0 = k0 + j0;
      char *fin = fin0 + (long)(j0 / PW) * finb;
      const int rest = k0 + nb - (c0 + w), mr = n - c0 - w;
      if (!tour) {   // the strip factored in place (L21 included), its interchanges and U on the block's other columns
        QH_LAUNCH(k_strip<T>, dim3(st_groups<T>(n - c0), 1, batch), dim3(st_w<T>() * 64), wcu ? W.strip : 0, st, n, c0, w,
                  A, lda, sA, ws, sW, (long)(fin - ws), wait, ipiv, sP, dinfo);
        const int nl = (c0 - k0 + 63) / 64, nu = (rest + 63) / 64;
        if (nl + nu > 0 || perm)
          QH_LAUNCH(k_swap_u<T>, dim3(std::max(nl + nu, 1), 1, batch), b256, wcu ? W.swap_u : 0, st, n, c0, w, A, lda, sA,
                    fin, sW, k0, k0 + nb, nl, perm, sP);
      } else {
        const int G = (n - c0 + TsRows<T>::R - 1) / TsRows<T>::R;
        QH_LAUNCH(k_ts_local<T>, dim3(G), bts, W.local, st, n, c0, w, A, lda, sA, bufA, sW, setb, (long)(fin - bufA),
                  G == 1 ? 1 : 0, ipiv, sP, perm, dinfo);
        char *cur = bufA, *nxt = bufB;
        for (int nsets = G; nsets > 1; nsets = (nsets + F - 1) / F) {
          const int nout = (nsets + F - 1) / F;
          QH_LAUNCH(k_ts_merge<T>, dim3(nout), bts, W.merge, st, c0, w, nsets, cur, nxt, sW, setb, fin,
                    nout == 1 ? 1 : 0, ipiv, sP, perm, dinfo);
          std::swap(cur, nxt);
        }
        const int nl = (c0 - k0 + 63) / 64, nu = (rest + 63) / 64;
        QH_LAUNCH(k_ts_apply<T>, dim3(1), b256, W.apply, st, n, c0, w, A, lda, fin);
        if (nl + nu > 0)
          QH_LAUNCH(k_swap_u<T>, dim3(nl + nu), b256, W.swap_u, st, n, c0, w, A, lda, sA, fin, sW, k0, k0 + nb, nl,
                    (int *)nullptr, sP);
        if (mr > 0)   // L21 = A21 U11^{-1}
          QH_LAUNCH((k_gemm_cu<T, true>), gcu_grid(mr, w), bcu, W.gemm_assign, st, mr, w, w,
                    A + (long)(c0 + w) * lda + c0, lda, reinterpret_cast<const cT *>(fin + PanelWS<T>::UINV_OFF), (long)PW,
                    A + (long)(c0 + w) * lda + c0, lda);
      }
      if (wcu) {   // single matrix, whole-CU launches (k_gemm_cu: several tiles per CU, K <= PW)
        if (rest > 0 && mr > 0)   // the block's next columns: A22 -= L21 U
          QH_LAUNCH((k_gemm_cu<T, false>), gcu_grid(mr, rest), bcu, W.gemm_sub, st, mr, rest, w,
                    A + (long)(c0 + w) * lda + c0, lda, A + (long)c0 * lda + c0 + w, lda,
                    A + (long)(c0 + w) * lda + c0 + w, lda);
        continue;
      }
      if (rest > 0 && mr > 0)   // the block's next columns: A22 -= L21 U
        QH_LAUNCH(k_gemm_sub<T>, dim3((rest + GT - 1) / GT, (mr + GT - 1) / GT, batch), b256, 0, st, mr, rest, w,
                  A + (long)(c0 + w) * lda + c0, lda, sA, A + (long)c0 * lda + c0 + w, lda, sA,
                  A + (long)(c0 + w) * lda + c0 + w, lda, sA);
    }
  };
  // Lookahead: once the trailing update has reached block k+1's columns, the
  // rest of it runs on the side stream (masked off a few CUs) while block
  // k+1's strips run here; the side stream's update is enqueued first, so it
  // starts at once, and the strips find the reserved CUs free. Block k+1's
  // interchanges are applied to the columns outside it afterwards (the strips
  // touch only their own block), after the side stream's update. Single
  // matrices only: a batch's strips already fill the device (batch x tens of
  // workgroups), and as whole-CU workgroups on the reserved CUs they would
  // queue (a batch of 8 at order 9216: 274 us per tournament launch).
  const bool la = lookahead && use_lookahead() && batch == 1 && n > 2 * LU_NB && !stream_capturing(s);
  hipStream_t side = nullptr;
  bool masked = false;
  LaCtx *cx = la ? la_for(s, &side, &masked) : nullptr;
  if (perm) QH_LAUNCH(k_iota, dim3((n + 255) / 256, 1, batch), b256, 0, s, n, perm, sP);
  block_strips(0, min(LU_NB, n), s, false);
  for (int k0 = 0; k0 < n; k0 += LU_NB) {
    const int nb = min(LU_NB, n - k0);
    if (n > nb)
      QH_LAUNCH(k_ts_apply_defer<T>, dim3((n + AP_COLS - 1) / AP_COLS, 1, batch), b256, 0, s, n, k0,
                         (nb + PW - 1) / PW, A, lda, sA, fin0, finb, sW, k0, k0 + nb);
    const int nr = n - k0 - nb;
    if (nr > 0) {
      QH_LAUNCH(k_u12<T>, dim3((nr + U12_C - 1) / U12_C, 1, batch), b256, u12_lds<T>(), s, nb, nr,
                (const cT *)(A + (long)k0 * lda + k0), lda, sA, A + (long)k0 * lda + k0 + nb);
      // A22 -= L21 U12: the next block's columns first, then the rest and the next block's strips
      const int nb1 = min(LU_NB, nr);
      trailing_gemm<T>(nr, nb1, nb, batch, A + (long)(k0 + nb) * lda + k0, lda, sA, A + (long)k0 * lda + k0 + nb, lda,
                       sA, A + (long)(k0 + nb) * lda + k0 + nb, lda, sA, s, own_gemm);
      // A strip's workgroups wait for each other, so each needs one of the CUs kept
      // free for it: beside the update on a shared CU the slowest held all of them up
      // (order 9216: 1.8 ms for the first strip of a block, 0.1 ms alone).
      const bool split = la && nr > nb1 && !(pp && st_groups<T>(nr) > strip_most<T>(true));
      if (nr > nb1) {
        hipStream_t sg = split ? side : s;
        if (split) {
          HIPCHK(hipEventRecord(cx->go, s));
          HIPCHK(hipStreamWaitEvent(sg, cx->go, 0));
        }
        trailing_gemm<T>(nr, nr - nb1, nb, batch, A + (long)(k0 + nb) * lda + k0, lda, sA,
                         A + (long)k0 * lda + k0 + nb + nb1, lda, sA, A + (long)(k0 + nb) * lda + k0 + nb + nb1, lda,
                         sA, sg, own_gemm);
        if (split) HIPCHK(hipEventRecord(cx->done, sg));
      }
      block_strips(k0 + nb, nb1, s, split && masked);
      if (split) HIPCHK(hipStreamWaitEvent(s, cx->done, 0));
    }
  }
  HIPCHK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Both triangular solves with a factorisation, one launch (k_tri): workgroup g
// of G owns the 64-row blocks g, g + G, ... of 16 right-hand-side columns. For a
// block it subtracts the products with the blocks solved before (each wave a
// quarter of their columns, by matrix instructions, the sums added in a fixed
// order), substitutes with its diagonal block, and publishes the result; backward the
// same from below.
//
// What bounds it: the chain of blocks, 7 to 8 us each in FP64 and 5 in FP32 for up to
// four columns, 11 to 14 and 7 to 10 for 16 (the words' way to the next workgroup, 64
// matrix instructions in a row for the last block's columns, 2 of the 7 us, and the
// substitution, 2 to 3 us). As launches per 64-row block (a wave substituting, 18-22
// us, then an update, 17 us) an FP64 solve of order 9216 took 10.5 ms, now 2.4; per
// 256-row block (130 us + 70 us) an FP32 one of order 9990 with 32 right-hand sides 16
// ms, now 3.1. With the diagonal block's inverse, made while others were solving, in
// the substitution's place the blocks took 6.3 and 4.1 us, but the error (FP64 factors
// of random matrices and of clusters', orders 64 to 512, against 80 bits) was 1.3 to 2
// times that of the launches' substitution; now it is 0.2 to 1.0 times. Loading the
// next product's operands or words ahead gained nothing.
//
// Published values carry a tag (1 forward, 2 backward) beside each 32 bits, as
// the strips' words do, so a reader needs no flag. Forward values are all read
// before the last block is solved forward, hence before any backward one
// replaces them. The workgroups of a slab announce themselves first
// (st_rendezvous); where they do not all get onto the device in time, one of
// them takes all blocks and the others leave.
// ---------------------------------------------------------------------------
constexpr int TR_B = 64, TR_C = 16, TR_VS = TR_B + 1, TR_XS = TR_C + 1;
constexpr int TR_MEET = 128;   // most workgroups of a slab
template <class T> constexpr size_t tr_lds() {   // the diagonal block without its diagonal, the waves' sums, the diagonal
  return (size_t)(TR_B * TR_VS + 4 * TR_B * TR_XS + TR_B) * sizeof(typename C2<T>::t);
}
template <class T> constexpr size_t tr_slab_bytes(int n, int nrhs) {
  return 256 + TR_MEET * 8 + (size_t)((n + TR_B - 1) / TR_B) * TR_B * (nrhs < TR_C ? nrhs : TR_C) * st_ew<T>() * 8;
}
constexpr int TR_MOST = 64 * TR_C;   // most right-hand sides of a launch (a grid's rows, and the words' memory)
template <class T> constexpr size_t tr_ws_bytes(int n, int nrhs) {
  if (nrhs > TR_MOST) nrhs = TR_MOST;
  return (size_t)((nrhs + TR_C - 1) / TR_C) * ((tr_slab_bytes<T>(n, nrhs) + 255) / 256 * 256);
}

template <class F, int... K>
__device__ __forceinline__ void tr_each(F f, std::integer_sequence<int, K...>) {
  (f(std::integral_constant<int, K>{}), ...);
}

// 1 / d 2^e in two parts (the second the first one's error) for a diagonal entry d of
// U, e = 0 unless its square or reciprocal might leave the range. A product with both
// parts is as good as a division by d, and no division waits in the chain of rows.
template <class T> struct TrRecip {
  typename C2<T>::t hi, lo;
  int e;
};
template <class T>
__device__ __forceinline__ TrRecip<T> tr_recip(typename C2<T>::t d) {
#pragma clang fp contract(off)
  typedef typename C2<T>::t cT;
  constexpr T BIG = sizeof(T) == 8 ? T(0x1p500) : T(0x1p60f);
  TrRecip<T> r;
  const T m = fmax(fabs(d.x), fabs(d.y));
  r.e = 0;
  if (m > 0 && m < T(INFINITY) && !(m > 1 / BIG && m < BIG)) {
    r.e = ilogb(m);
    d = cT{ldexp(d.x, -r.e), ldexp(d.y, -r.e)};
  }
  r.hi = cdiv<T>(cT{1, 0}, d);
  // 1 - d hi, exactly but for the products' own errors: the two products of the real
  // part add up to one, those of the imaginary part to nothing
  const T a = d.x * r.hi.x, b = -d.y * r.hi.y, ea = fma(d.x, r.hi.x, -a), eb = fma(-d.y, r.hi.y, -b);
  const T c = d.x * r.hi.y, f = d.y * r.hi.x, ec = fma(d.x, r.hi.y, -c), ef = fma(d.y, r.hi.x, -f);
  const cT err = cT{((1 - fmax(a, b)) - fmin(a, b)) - (ea + eb), -(c + f) - (ec + ef)};
  r.lo = cmul<T>(err, r.hi);
  return r;
}

// The value of lane K: of the lane's row of 16 (LN = 16), of the wave.
template <int LN, int K> __device__ __forceinline__ unsigned tr_lane(unsigned v) {
  if constexpr (LN == 16) return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x150 + K, 0xF, 0xF, true);   // row_newbcast
  else return (unsigned)__builtin_amdgcn_readlane((int)v, K);
}
template <int LN, int K> __device__ __forceinline__ float tr_bc(float v) { return __uint_as_float(tr_lane<LN, K>(__float_as_uint(v))); }
template <int LN, int K> __device__ __forceinline__ double tr_bc(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = tr_lane<LN, K>((unsigned)b), hi = tr_lane<LN, K>((unsigned)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// v / d
template <class T>
__device__ __forceinline__ typename C2<T>::t tr_div(typename C2<T>::t v, const TrRecip<T> &d, bool scaled) {
  typedef typename C2<T>::t cT;
  const cT h = d.hi, l = d.lo;
  const cT y = cT{fma(v.x, h.x, fma(-v.y, h.y, fma(v.x, l.x, -v.y * l.y))), fma(v.x, h.y, fma(v.y, h.x, fma(v.x, l.y, v.y * l.x)))};
  return scaled ? cT{ldexp(y.x, -d.e), ldexp(y.y, -d.e)} : y;
}

// Substitution with a triangular block of LN R rows at V (LDS, row stride TR_VS;
// strictly lower or upper, zeros elsewhere; UPPER: dinv the lane's diagonal entries'
// reciprocals), LN lanes per column: x[q] is row LN q + cls of the lane's column,
// less[q] what the rows solved before the block take from it. The row's other products
// are added to less, and the sum subtracted once: subtracted one by one they cost a
// rounding of x's size each. Every step's solved entry goes round the column's lanes.
// All lanes add: the zeros keep the solved rows, but for an entry that is no finite
// number; with any of those, or diagonal entries near the limits of the range, the rows
// are solved again, under conditions. V's entries come four steps ahead.
// What bounds it: a step's instructions, with one wave on a SIMD; with a wave on all
// four, V's way from LDS as much.
template <class T, bool UPPER, int LN, int R>
__device__ __forceinline__ void tr_substitute(const typename C2<T>::t *V, const TrRecip<T> (&dinv)[R], int cls,
                                              typename C2<T>::t (&x)[R], typename C2<T>::t (&less)[R]) {
  typedef typename C2<T>::t cT;
  constexpr int N = LN * R;
  bool odd = false;
  if (UPPER)
#pragma unroll
    for (int q = 0; q < R; ++q) odd |= dinv[q].e != 0;
  const bool scaled = __any(odd);
  cT l[2][4][R], pre[R], pim[R], rest[R];   // 8 steps' products with l's real and imaginary part; x - less
#pragma unroll
  for (int q = 0; q < R; ++q) {
    pre[q] = pim[q] = cT{0, 0};
    rest[q] = x[q] - less[q];
  }
  auto load = [&](auto cc) {   // the entries of steps 4 C .. 4 C + 3
    constexpr int C = decltype(cc)::value, Q = UPPER ? R - 1 - 4 * C / LN : 4 * C / LN;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int col = UPPER ? N - 1 - 4 * C - i : 4 * C + i;
#pragma unroll
      for (int q = UPPER ? 0 : Q; q <= (UPPER ? Q : R - 1); ++q) l[C & 1][i][q] = V[(LN * q + cls) * TR_VS + col];
    }
    asm volatile("" ::: "memory");   // not earlier than here, nor later
  };
  load(std::integral_constant<int, 0>{});
  auto chunk = [&](auto cc) {
    constexpr int C = decltype(cc)::value, Q = UPPER ? R - 1 - 4 * C / LN : 4 * C / LN;
    if constexpr (C + 1 < N / 4) load(std::integral_constant<int, C + 1>{});
    auto step = [&](auto ic) {
      constexpr int I = decltype(ic)::value, K = UPPER ? LN - 1 - (4 * C + I) % LN : (4 * C + I) % LN;
      cT v = rest[Q] - cT{pre[Q].x - pim[Q].y, pre[Q].y + pim[Q].x};
      if (UPPER) v = tr_div<T>(v, dinv[Q], false);
      v = cT{tr_bc<LN, K>(v.x), tr_bc<LN, K>(v.y)};
#pragma unroll
      for (int q = UPPER ? 0 : Q; q <= (UPPER ? Q : R - 1); ++q) {
        const cT e = l[C & 1][I][q];
        pre[q] = cT{fma(e.x, v.x, pre[q].x), fma(e.x, v.y, pre[q].y)};
        pim[q] = cT{fma(e.y, v.x, pim[q].x), fma(e.y, v.y, pim[q].y)};
      }
      __builtin_amdgcn_sched_barrier(0);   // put off, the other rows' products would hold their factors in registers
    };
    tr_each(step, std::make_integer_sequence<int, 4>{});
    if constexpr (C % 2 == 1 && C + 1 < N / 4) {
#pragma unroll
      for (int q = UPPER ? 0 : Q; q <= (UPPER ? Q : R - 1); ++q) {
        less[q] += cT{pre[q].x - pim[q].y, pre[q].y + pim[q].x};
        pre[q] = pim[q] = cT{0, 0};
        rest[q] = x[q] - less[q];
      }
    }
  };
  cT start[R];
#pragma unroll
  for (int q = 0; q < R; ++q) start[q] = less[q];
  tr_each(chunk, std::make_integer_sequence<int, N / 4>{});
#pragma unroll
  for (int q = 0; q < R; ++q) {
    less[q] += cT{pre[q].x - pim[q].y, pre[q].y + pim[q].x};
    odd |= !(fabs(less[q].x) + fabs(less[q].y) < T(INFINITY));
  }
  if (__any(odd)) {
#pragma unroll
    for (int q = 0; q < R; ++q) less[q] = start[q];
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int Q = UPPER ? R - 1 - u : u;
#pragma unroll 1
      for (int j = 0; j < LN; j += 8) {   // the same roundings as above
#pragma unroll
        for (int q = 0; q < R; ++q) {
          pre[q] = pim[q] = cT{0, 0};
          rest[q] = x[q] - less[q];
        }
#pragma unroll 1
        for (int i = j; i < j + 8; ++i) {
          const int k = UPPER ? LN - 1 - i : i, from = (threadIdx.x & 63 & -LN) | k;
          cT v = rest[Q] - cT{pre[Q].x - pim[Q].y, pre[Q].y + pim[Q].x};
          if (UPPER) v = tr_div<T>(v, dinv[Q], scaled);
          v = cT{__shfl(v.x, from), __shfl(v.y, from)};
#pragma unroll
          for (int q = UPPER ? 0 : Q; q <= (UPPER ? Q : R - 1); ++q) {
            const cT e = V[(LN * q + cls) * TR_VS + LN * Q + k];
            if (q != Q || (UPPER ? cls < k : cls > k)) {
              pre[q] = cT{fma(e.x, v.x, pre[q].x), fma(e.x, v.y, pre[q].y)};
              pim[q] = cT{fma(e.y, v.x, pim[q].x), fma(e.y, v.y, pim[q].y)};
            }
          }
        }
#pragma unroll
        for (int q = 0; q < R; ++q) less[q] += cT{pre[q].x - pim[q].y, pre[q].y + pim[q].x};
      }
    }
  }
#pragma unroll
  for (int q = 0; q < R; ++q) {
    x[q] -= less[q];
    if (UPPER) x[q] = tr_div<T>(x[q], dinv[q], scaled);
  }
}

template <class T>
__device__ __forceinline__ typename C2<T>::t tr_value(const st_u64 (&w)[sizeof(T) == 8 ? 4 : 2]) {
  if constexpr (sizeof(T) == 8)
    return v2d{__longlong_as_double((long long)((w[1] << 32) | (unsigned)w[0])),
               __longlong_as_double((long long)((w[3] << 32) | (unsigned)w[2]))};
  else
    return v2f{__uint_as_float((unsigned)w[0]), __uint_as_float((unsigned)w[1])};
}
template <class T>
__device__ __forceinline__ void tr_publish(st_u64 *at, unsigned tag, typename C2<T>::t v) {
  const st_u64 hi = (st_u64)tag << 32;
  if constexpr (sizeof(T) == 8) {
    const st_u64 a = (st_u64)__double_as_longlong(v.x), b = (st_u64)__double_as_longlong(v.y);
    st_store(at, hi | (unsigned)a);
    st_store(at + 1, hi | (unsigned)(a >> 32));
    st_store(at + 2, hi | (unsigned)b);
    st_store(at + 3, hi | (unsigned)(b >> 32));
  } else {
    st_store(at, hi | __float_as_uint(v.x));
    st_store(at + 1, hi | __float_as_uint(v.y));
  }
}

template <class T>
__global__ __launch_bounds__(256, (sizeof(T) == 4 ? 2 : 1)) void k_tri(int n, int nrhs, const typename C2<T>::t *LU, long lda, long sA,
                                                const int *perm, long sP, typename C2<T>::t *B, long ldb, long sB,
                                                char *ws, long sW, long slabb, st_u64 limit) {
  typedef typename C2<T>::t cT;
  typedef typename MF<T>::acc acc_t;
  constexpr int EW = st_ew<T>();
  extern __shared__ __align__(16) char smem_raw[];
  cT *V = reinterpret_cast<cT *>(smem_raw);
  cT *S = V + TR_B * TR_VS, *D = S + 4 * TR_B * TR_XS;
  __shared__ int go;
  const int z = blockIdx.z, t = threadIdx.x, lane = t & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int g = blockIdx.x, G = gridDim.x;
  const int j0 = blockIdx.y * TR_C, nc = min(TR_C, nrhs - j0), cs = min(TR_C, nrhs);   // columns, words' column stride
  LU += (long)z * sA;
  perm += (long)z * sP;
  B += (long)z * sB + j0;
  char *wz = ws + (long)z * sW + (long)blockIdx.y * slabb;
  st_u64 *X = reinterpret_cast<st_u64 *>(wz + 256 + TR_MEET * 8);
  if (G > 1) {
    if (wave == 0) go = st_rendezvous(g, G, 1u, reinterpret_cast<st_u64 *>(wz + 256), reinterpret_cast<int *>(wz), limit);
    __syncthreads();
    if (go == 0) return;
    if (go < 0) { g = 0; G = 1; }
  }
  const int nblk = (n + TR_B - 1) / TR_B;
  auto sweep = [&](auto up) {
    constexpr bool UPPER = decltype(up)::value;
    constexpr unsigned tag = UPPER ? 2u : 1u;
    const int mine = (nblk - 1 - g) / G + 1;   // blocks of this workgroup
    for (int b = 0; b < mine; ++b) {
      const int i = g + G * (UPPER ? mine - 1 - b : b), r0 = i * TR_B;
      // the diagonal block
      {
        cT v[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const int e = t + 256 * q, r = e >> 6, c = e & 63;
          const bool in = r0 + r < n && r0 + c < n && (UPPER ? c >= r : c < r);
          v[q] = in ? LU[(long)(r0 + r) * lda + r0 + c] : cT{UPPER && r == c ? T(1) : T(0), 0};
        }
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const int e = t + 256 * q, r = e >> 6, c = e & 63;
          if (UPPER && r == c) D[r] = v[q];
          V[r * TR_VS + c] = r == c ? cT{0, 0} : v[q];
        }
        __syncthreads();
      }
      TrRecip<T> dinv[2][2], dinv1[1];   // its diagonal's reciprocals, as the substitutions take them
      if (UPPER) {
        if (cs > 4) {
#pragma unroll
          for (int q = 0; q < 4; ++q) dinv[q >> 1][q & 1] = tr_recip<T>(D[16 * q + lr]);
        } else {
          dinv1[0] = tr_recip<T>(D[lane]);
        }
      }
      // this wave's 16 rows of the right-hand side, as results of matrix
      // instructions: rows of P B, or what the forward sweep left
      const int rw = r0 + 16 * wave;
      acc_t rr, ri;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = rw + MF<T>::row(lk, e);
        cT v = cT{0, 0};
        if (UPPER) {
          if (lr < cs) {
            st_u64 w[EW];
            bool ok;
            do {
              ok = true;
#pragma unroll
              for (int k = 0; k < EW; ++k) { w[k] = st_load(X + ((long)r * cs + lr) * EW + k); ok &= (w[k] >> 32) == 1u; }
            } while (!ok);
            v = tr_value<T>(w);
          }
        } else if (r < n && lr < nc) {
          v = B[(long)perm[r] * ldb + lr];
        }
        rr[e] = v.x;
        ri[e] = v.y;
      }
      // less the products with the blocks solved before, a quarter of their columns per wave
      // (block by block, added in LDS: as one chain over all blocks their rounding
      // errors were twice as large at order 1024)
      acc_t pr[4], pi[4];
      auto sums = [&](bool first) {
#pragma unroll
        for (int T_ = 0; T_ < 4; ++T_) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            cT &at = S[(wave * TR_B + 16 * T_ + MF<T>::row(lk, e)) * TR_XS + lr];
            const cT v = cT{pr[T_][e], pi[T_][e]};
            at = first ? v : at + v;
          }
          pr[T_] = pi[T_] = acc_t{0, 0, 0, 0};
        }
      };
#pragma unroll
      for (int T_ = 0; T_ < 4; ++T_) pr[T_] = pi[T_] = acc_t{0, 0, 0, 0};
      const int nb = UPPER ? nblk - 1 - i : i;
      for (int q = 0; q < nb; ++q) {
        const int k0 = (UPPER ? nblk - 1 - q : q) * TR_B + 16 * wave + lk;
        cT a[4][4], x[4];
#pragma unroll
        for (int T_ = 0; T_ < 4; ++T_)
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) {
            const int r = r0 + 16 * T_ + lr, c = k0 + 4 * ks;
            a[T_][ks] = (r < n && c < n) ? LU[(long)r * lda + c] : cT{0, 0};
          }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) x[ks] = cT{0, 0};
        if (lr < cs) {
          st_u64 w[4][EW];
          bool ok;
          do {
            ok = true;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
#pragma unroll
              for (int k = 0; k < EW; ++k) {
                w[ks][k] = st_load(X + ((long)(k0 + 4 * ks) * cs + lr) * EW + k);
                ok &= (w[ks][k] >> 32) == tag;
              }
          } while (!ok);
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) x[ks] = tr_value<T>(w[ks]);
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
          for (int T_ = 0; T_ < 4; ++T_) {
            pr[T_] = MF<T>::mma(a[T_][ks].x, x[ks].x, pr[T_]);
            pi[T_] = MF<T>::mma(a[T_][ks].x, x[ks].y, pi[T_]);
            pr[T_] = MF<T>::mma(-a[T_][ks].y, x[ks].y, pr[T_]);
            pi[T_] = MF<T>::mma(a[T_][ks].y, x[ks].x, pi[T_]);
          }
        if (q + 1 < nb) sums(q == 0);
      }
      sums(nb <= 1);
      __syncthreads();
      cT sum[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const cT *at = S + (16 * wave + MF<T>::row(lk, e)) * TR_XS + lr;
        sum[e] = (at[0] + at[TR_B * TR_XS]) + (at[2 * TR_B * TR_XS] + at[3 * TR_B * TR_XS]);
      }
      // a wave's rows and their sums to the lanes that solve their columns, in parts that
      // no other wave reads
      auto part = [&](int r, int c, int p) { return S + (long)(((r >> 4) ^ p) * TR_B + r) * TR_XS + c; };
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 16 * wave + MF<T>::row(lk, e);
        *part(r, lr, 0) = cT{rr[e], ri[e]};
        *part(r, lr, 1) = sum[e];
      }
      __syncthreads();
      auto done = [&](int row, int c, cT x) {
        const int r = r0 + row;
        if (c < cs) tr_publish<T>(X + ((long)r * cs + c) * EW, tag, x);
        if (UPPER && r < n && c < nc) B[(long)r * ldb + c] = x;
      };
      // up to four columns a wave each (order 1040, one column: 223 us in FP64, 151 in
      // FP32, against 259 and 191 with 16 lanes), more 16 lanes each
      if (cs <= 4) {
        if (wave < cs) {
          cT xs[1] = {*part(lane, wave, 0)}, ls[1] = {*part(lane, wave, 1)};
          tr_substitute<T, UPPER, 64, 1>(V, dinv1, lane, xs, ls);
          done(lane, wave, xs[0]);
        }
      } else {   // the block's halves one after the other (as one 11.4, 7.8 us a block, so 10.7, 6.9)
        const int c = 4 * wave + lk;
        auto half = [&](auto hc) {
          constexpr int H = decltype(hc)::value, o = 32 * H;
          constexpr bool SECOND = UPPER ? H == 0 : H == 1;
          if (4 * wave < cs) {   // uniform
            cT xs[2], ls[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              const int r = o + 16 * q + lr;
              xs[q] = *part(r, c, 0);
              ls[q] = *part(r, c, 1);
              if (SECOND) ls[q] += *part(r, c, 2) + *part(r, c, 3);
            }
            tr_substitute<T, UPPER, 16, 2>(V + o * TR_VS + o, dinv[H], lr, xs, ls);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              const int r = o + 16 * q + lr;
              done(r, c, xs[q]);
              if (!SECOND) *part(r, c, 0) = xs[q];
            }
          }
        };
        half(std::integral_constant<int, UPPER ? 1 : 0>{});
        __syncthreads();
        {   // what the first half takes from the second: 16 rows and 16 columns of V per wave
          constexpr int o0 = UPPER ? 32 : 0, o1 = 32 - o0;
          const int rt = o1 + 16 * (wave & 1), kt = o0 + 16 * (wave >> 1);
          acc_t rx = acc_t{0, 0, 0, 0}, iy = rx, ix = rx, ry = rx;   // short chains, for their rounding errors too
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) {
            const cT a = V[(rt + lr) * TR_VS + kt + 4 * ks + lk], x = *part(kt + 4 * ks + lk, lr, 0);
            rx = MF<T>::mma(a.x, x.x, rx);
            ry = MF<T>::mma(a.x, x.y, ry);
            iy = MF<T>::mma(a.y, x.y, iy);
            ix = MF<T>::mma(a.y, x.x, ix);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) *part(rt + MF<T>::row(lk, e), lr, 2 + (wave >> 1)) = cT{rx[e] - iy[e], ry[e] + ix[e]};
        }
        __syncthreads();
        half(std::integral_constant<int, UPPER ? 0 : 1>{});
      }
      __syncthreads();
    }
  };
  sweep(std::false_type{});
  sweep(std::true_type{});
}
template <class T>
static void tr_prepare() {
  static std::once_flag once;
  std::call_once(once, [] {
    HIPCHK(hipFuncSetAttribute((const void *)k_tri<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)tr_lds<T>()));
  });
}
template <class T> static size_t getrs_ws_bytes(int n, int nrhs, int batch) {
  return (size_t)batch * tr_ws_bytes<T>(n, nrhs);
}

// B (n x nrhs, ldb) <- A^{-1} B given LU and the row permutation. ws:
// getrs_ws_bytes<T>(n, nrhs, batch) bytes.
template <class T>
static void getrs_batched(int n, int nrhs, int batch, const typename C2<T>::t *LU, long lda, long sA,
                          const int *perm, long sP, typename C2<T>::t *B, long ldb, long sB, void *ws, hipStream_t s,
                          st_u64 wait = ST_LIMIT) {
  if (n <= 0 || nrhs <= 0 || batch <= 0) return;
  if (nrhs > TR_MOST) {   // in turns
    for (int j = 0; j < nrhs; j += std::min(TR_MOST, nrhs - j))
      getrs_batched<T>(n, std::min(TR_MOST, nrhs - j), batch, LU, lda, sA, perm, sP, B + j, ldb, sB, ws, s, wait);
    return;
  }
  tr_prepare<T>();
  const int nblk = (n + TR_B - 1) / TR_B, nslab = (nrhs + TR_C - 1) / TR_C;
  const long slabb = (long)((tr_slab_bytes<T>(n, nrhs) + 255) / 256 * 256), sW = slabb * nslab;
  qh_zero(ws, (size_t)batch * sW, s);
  // A workgroup's next block, up to nblk products of 64 x 64 blocks (2 us each), has to
  // be ready when the chain (5 to 14 us a block) gets there: nblk / 4 of them keep up
  // with one slab. A slab gets no more than a quarter of the device (which holds 256
  // workgroups in FP64, 512 in FP32), so that of the slabs of four hardware queues one
  // is always complete and the others wait for its end only. Several slabs or matrices
  // share the device, more of them take turns: a 16-matrix batch of order 9216 with 64
  // right-hand sides (FP32) takes 23 ms with two workgroups per slab, 12 with eight.
  const long quarter = sizeof(T) == 8 ? 64 : 128, slabs = (long)nslab * batch;
  const int G = (int)std::max(1L, std::min({(long)nblk, (long)TR_MEET, quarter, 4 * quarter / slabs}));
  QH_LAUNCH(k_tri<T>, dim3(G, nslab, batch), dim3(256), tr_lds<T>(), s, n, nrhs, LU, lda, sA, perm, sP, B, ldb, sB,
            (char *)ws, sW, slabb, wait);
  HIPCHK(hipGetLastError());
}

extern "C" int qpms_hip_zgetrf_dev(size_t n, _Complex double *A_dev, int *ipiv_dev, void *stream) {
  hipStream_t s = (hipStream_t)qh_stream(stream);
  // the info word and the workspace, this call's own
  int *dinfo = (int *)qh_dmalloc(256 + (n < (1u << 22) ? LuWS<double>((int)n, 1, true).bytes : 0));
  HIPCHK(hipMemsetAsync(dinfo, 0, sizeof(int), s));
  getrf_batched<double>((int)n, 1, (v2d *)A_dev, (long)n, 0, ipiv_dev, 0, nullptr, dinfo, s, (char *)dinfo + 256,
                        true, false, /*pp=*/true);
  int info = 0;
  HIPCHK(hipMemcpyAsync(&info, dinfo, sizeof(int), hipMemcpyDeviceToHost, s));
  HIPCHK(hipStreamSynchronize(s));
  qh_dfree(dinfo);
  return info;
}

// The partial-pivoting LU of one FP64 or FP32 (prec 64, 32) matrix with the
// strips' wait for their workgroups as an argument (clock ticks; 0: a strip of
// several workgroups is left to the first one that does not see the others at
// once). info: a device word. Tests reach both ways through a strip with it.
extern "C" int qh_getrf_pp(int prec, int n, double *A, int *ipiv, int *info, unsigned long long wait, void *stream) {
  hipStream_t s = (hipStream_t)qh_stream(stream);
  qh_zero(info, sizeof(int), s);
  char *ws = ws_for(s, prec == 32 ? LuWS<float>(n, 1, true).bytes : LuWS<double>(n, 1, true).bytes);
  if (prec == 32)
    getrf_batched<float>(n, 1, (v2f *)A, n, 0, ipiv, 0, nullptr, info, s, ws, true, false, true, wait);
  else
    getrf_batched<double>(n, 1, (v2d *)A, n, 0, ipiv, 0, nullptr, info, s, ws, true, false, true, wait);
  return 0;
}

// The LU of one matrix with the tournament for strips of more than `most`
// workgroups, no lookahead; waits. Tests reach it at small orders.
extern "C" int qh_getrf_most(int prec, int n, double *A, int *ipiv, int *perm, int *info, int most, void *stream) {
  hipStream_t s = (hipStream_t)qh_stream(stream);
  qh_zero(info, sizeof(int), s);
  char *ws = (char *)qh_dmalloc(prec == 32 ? LuWS<float>(n, 1, false, most).bytes : LuWS<double>(n, 1, false, most).bytes);
  if (prec == 32)
    getrf_batched<float>(n, 1, (v2f *)A, n, 0, ipiv, n, perm, info, s, ws, false, false, false, ST_LIMIT, most);
  else
    getrf_batched<double>(n, 1, (v2d *)A, n, 0, ipiv, n, perm, info, s, ws, false, false, false, ST_LIMIT, most);
  HIPCHK(hipStreamSynchronize(s));
  qh_dfree(ws);
  return 0;
}

// ---------------------------------------------------------------------------
// Whole-factorisation timing for the GEMM autotuner: FP32 LUs of a
// well-conditioned pseudo-random matrix (entries in [-1/2, 1/2]^2 from a hash
// of the indices, 3 sqrt(n) added on the diagonal), with lookahead, as the
// serving loop and the LU entry points run them, on a stream of their own.
// ---------------------------------------------------------------------------
__global__ void k_tune_fill(long n, v2f *A) {
  const long tot = n * n;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < tot; e += (long)gridDim.x * blockDim.x) {
    unsigned long long h = (unsigned long long)e * 0x9E3779B97F4A7C15ull;
    h ^= h >> 29;
    h *= 0xBF58476D1CE4E5B9ull;
    h ^= h >> 32;
    const float re = (float)(h & 0xFFFFFF) * (1.f / 16777216.f) - 0.5f;
    const float im = (float)((h >> 24) & 0xFFFFFF) * (1.f / 16777216.f) - 0.5f;
    A[e] = v2f{re + ((e / n == e % n) ? 3.f * sqrtf((float)n) : 0.f), im};
  }
}

namespace {
struct TuneCtx {
  v2f *A;
  char *ws;
  int *ipiv, *info;
  hipStream_t s;
  hipEvent_t e0, e1;
  int nmax;
};
float tune_lu(int n, void *p) {
  TuneCtx &c = *static_cast<TuneCtx *>(p);
  if (n > c.nmax) return -1.f;
  float best = -1.f;
  for (int rep = 0; rep < 2; ++rep) {   // the first run warms the shapes' kernels up
    QH_LAUNCH(k_tune_fill, dim3(qh_stride_blocks((long)n * n)), dim3(256), 0, c.s, (long)n, c.A);
    HIPCHK(hipEventRecord(c.e0, c.s));
    getrf_batched<float>(n, 1, c.A, n, 0, c.ipiv, n, nullptr, c.info, c.s, c.ws, true);
    HIPCHK(hipEventRecord(c.e1, c.s));
    HIPCHK(hipEventSynchronize(c.e1));
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, c.e0, c.e1));
    if (rep) best = ms;
  }
  return best;
}
}  // namespace

// Tunes the single-matrix classes by whole factorisations (largest order
// that fits the free memory, at most 16384; the class above keeps its GEMM
// timing). Returns the classes tuned.
extern "C" int qh_autotune_lu(float *report) {
  TuneCtx c{};
  HIPCHK(hipStreamCreateWithFlags(&c.s, hipStreamNonBlocking));   // released with its LU state at the end
  for (int n = 16384; n >= 2048 && !c.A; n /= 2) {
    void *a = nullptr, *w = nullptr;
    if (hipMalloc(&a, (size_t)n * n * 8) != hipSuccess ||
        hipMalloc(&w, getrf_ws_bytes<float>(n, 1) + 8 * (size_t)n + 256) != hipSuccess) {
      (void)hipGetLastError();
      if (a) HIPCHK(hipFree(a));
      if (w) HIPCHK(hipFree(w));
      continue;
    }
    c.A = (v2f *)a;
    c.ws = (char *)w;
    c.nmax = n;
  }
  if (!c.A) {
    HIPCHK(hipStreamDestroy(c.s));
    return 0;
  }
  c.ipiv = (int *)(c.ws + getrf_ws_bytes<float>(c.nmax, 1));
  c.info = c.ipiv + c.nmax;
  HIPCHK(hipEventCreate(&c.e0));
  HIPCHK(hipEventCreate(&c.e1));
  const int tuned = qh_autotune_lu_classes(tune_lu, &c, report);
  HIPCHK(hipStreamSynchronize(c.s));
  HIPCHK(hipEventDestroy(c.e0));
  HIPCHK(hipEventDestroy(c.e1));
  HIPCHK(hipFree(c.A));
  HIPCHK(hipFree(c.ws));
  qh_stream_release(c.s);
  HIPCHK(hipStreamDestroy(c.s));
  return tuned;
}

// ---------------------------------------------------------------------------
// Allocation-free variant of qpms_hip_zgetrf_dev for callers that cannot
// allocate device memory (code under graph capture, serving loops that
// forbid hipMalloc). Its scratch -- the info word and the strip workspace
// -- is the file-scope array below; the GEMMs are the
// hand-written kernel (the library GEMM may allocate) and there is no
// lookahead side stream. The host never names the array in a kernel
// argument or copy: it uses the device address hipGetSymbolAddress returned
// for the current device at initialisation.
// ---------------------------------------------------------------------------
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)16 << 20;
static __device__ __align__(256) char scratch[NOALLOC_SCRATCH_BYTES];
constexpr int NOALLOC_MAX_DEV = 64;
static char *g_scratch_ptr[NOALLOC_MAX_DEV];   // device address of `scratch`, per device
static std::mutex g_scratch_mu[NOALLOC_MAX_DEV];   // held by the call that uses the array, until its work is done

// Called by the library's initialisation with the device current (once per
// device); records the device address of the scratch array.
extern "C" void qh_noalloc_scratch_init(void) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= NOALLOC_MAX_DEV)
    qpms_hip_die(__FILE__, __LINE__, __func__, "device %d outside the scratch table", dev);
  void *p = nullptr;
  HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  g_scratch_ptr[dev] = (char *)p;
}

// Largest order the entry point takes (its strips' words and slots, after a
// 256-byte info word, fit the scratch array).
constexpr int NOALLOC_MAX_N = 125952;
extern "C" size_t qpms_hip_zgetrf_noalloc_max_n(void) { return NOALLOC_MAX_N; }

extern "C" int qpms_hip_zgetrf_dev_noalloc(size_t n, _Complex double *A_dev, int *ipiv_dev, void *stream) {
  hipStream_t s = (hipStream_t)qh_stream(stream);
  if (n == 0) return 0;
  if (n > (size_t)NOALLOC_MAX_N) {
    fprintf(stderr, "qpms_hip_zgetrf_dev_noalloc: order %zu is above the largest order %d of the %zu-byte scratch "
            "array\n", n, NOALLOC_MAX_N, NOALLOC_SCRATCH_BYTES);
    return -1;
  }
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  char *base = (dev >= 0 && dev < NOALLOC_MAX_DEV) ? g_scratch_ptr[dev] : nullptr;
  if (!base) qpms_hip_die(__FILE__, __LINE__, __func__, "scratch of device %d not initialised", dev);
  if (256 + LuWS<double>((int)n, 1, true).bytes > NOALLOC_SCRATCH_BYTES)
    qpms_hip_die(__FILE__, __LINE__, __func__, "scratch too small for order %zu", n);
  std::lock_guard<std::mutex> turn(g_scratch_mu[dev]);
  int *dinfo = (int *)base;
  qh_zero(dinfo, 256, s);   // a kernel: the info word must start at zero on every call
  getrf_batched<double>((int)n, 1, (v2d *)A_dev, (long)n, 0, ipiv_dev, 0, nullptr, dinfo, s, base + 256,
                        /*lookahead=*/false, /*own_gemm=*/true, /*pp=*/true);
  int info = 0;
  HIPCHK(hipMemcpyAsync(&info, dinfo, sizeof(int), hipMemcpyDeviceToHost, s));
  HIPCHK(hipStreamSynchronize(s));
  return info;
}

extern "C" int qpms_hip_zgetrs_dev(size_t n, size_t nrhs, const _Complex double *LU_dev, const int *ipiv_dev,
                                   _Complex double *B_dev, void *stream) {
  hipStream_t s = (hipStream_t)qh_stream(stream);
  if (n == 0 || nrhs == 0) return 0;
  const size_t wb = getrs_ws_bytes<double>((int)n, (int)nrhs, 1);
  char *ws = (char *)qh_dmalloc(wb + n * sizeof(int));
  int *perm = (int *)(ws + wb);
  QH_LAUNCH(k_perm_from_ipiv, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, s, (int)n, ipiv_dev, perm);
  getrs_batched<double>((int)n, (int)nrhs, 1, (const v2d *)LU_dev, (long)n, 0, perm, 0, (v2d *)B_dev, (long)nrhs, 0, ws, s);
  HIPCHK(hipStreamSynchronize(s));
  qh_dfree(ws);
  return 0;
}

extern "C" int qh_launch_block_tw(size_t nr, size_t L, const double *T, const double *W, double *M, size_t col0,
                                  void *stream) {
  QH_LAUNCH(k_block_tw, dim3((unsigned)((L + 255) / 256), (unsigned)nr), dim3(256), 0,
                     (hipStream_t)qh_stream(stream), (int)nr, (int)L, (const v2d *)T, (const v2d *)W, (v2d *)M,
                     (int)col0);
  HIPCHK(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------
// Batched LU / solve entry points used by Beyn and the serving loop. Without a
// workspace of the caller's: that of the stream, one thread at a time.
// ---------------------------------------------------------------------------
extern "C" int qh_getrf_batched_f64(int n, int batch, double *A, long sA, int *ipiv, int *perm, int *info,
                                    void *stream) {
  hipStream_t s = (hipStream_t)qh_stream(stream);
  if (n <= 0 || batch <= 0) return 0;
  getrf_batched<double>(n, batch, (v2d *)A, n, sA, ipiv, n, perm, info, s, ws_for(s, getrf_ws_bytes<double>(n, batch)));
  return 0;
}
extern "C" size_t qh_getrf_ws_bytes(int prec, int n, int batch) {
  return prec == 32 ? getrf_ws_bytes<float>(n, batch) : getrf_ws_bytes<double>(n, batch);
}
// Caller-workspace entry points: their callers (the serving loop's lanes)
// already overlap work across several streams, so no lookahead side stream.
extern "C" int qh_getrf_batched_ws_f64(int n, int batch, double *A, long sA, int *ipiv, int *perm, int *info, void *ws,
                                       void *stream) {
  getrf_batched<double>(n, batch, (v2d *)A, n, sA, ipiv, n, perm, info, (hipStream_t)qh_stream(stream), (char *)ws,
                        false);
  return 0;
}
extern "C" int qh_getrf_batched_ws_f32(int n, int batch, float *A, long sA, int *ipiv, int *perm, int *info, void *ws,
                                       void *stream) {
  getrf_batched<float>(n, batch, (v2f *)A, n, sA, ipiv, n, perm, info, (hipStream_t)qh_stream(stream), (char *)ws,
                       false);
  return 0;
}
// The same with lookahead when `lookahead` (large orders): the bulk of each
// trailing GEMM runs on a side stream of `stream` while the next block's
// strips run on `stream` (the side stream belongs to `stream` until
// released).
extern "C" int qh_getrf_batched_wsla_f32(int n, int batch, float *A, long sA, int *ipiv, int *perm, int *info,
                                         void *ws, int lookahead, void *stream) {
  getrf_batched<float>(n, batch, (v2f *)A, n, sA, ipiv, n, perm, info, (hipStream_t)qh_stream(stream), (char *)ws,
                       lookahead != 0);
  return 0;
}
extern "C" int qh_getrf_batched_wsla_f64(int n, int batch, double *A, long sA, int *ipiv, int *perm, int *info,
                                         void *ws, int lookahead, void *stream) {
  getrf_batched<double>(n, batch, (v2d *)A, n, sA, ipiv, n, perm, info, (hipStream_t)qh_stream(stream), (char *)ws,
                        lookahead != 0);
  return 0;
}
// Strips of factorisations and slabs of solves that one workgroup had to do alone,
// since the library was loaded (waits for the device).
extern "C" unsigned qh_alone_count(void) {
  unsigned n = 0;
  HIPCHK(hipMemcpyFromSymbol(&n, HIP_SYMBOL(g_alone), sizeof n));
  return n;
}
// Solves with batched factorisations. The workspace form neither allocates nor
// waits.
extern "C" size_t qh_getrs_ws_bytes(int prec, int n, int nrhs, int batch) {
  return prec == 32 ? getrs_ws_bytes<float>(n, nrhs, batch) : getrs_ws_bytes<double>(n, nrhs, batch);
}
extern "C" int qh_getrs_ws_f64(int n, int nrhs, int batch, const double *LU, long sA, const int *perm, double *B,
                               long sB, void *ws, void *stream) {
  getrs_batched<double>(n, nrhs, batch, (const v2d *)LU, n, sA, perm, n, (v2d *)B, nrhs, sB, ws,
                        (hipStream_t)qh_stream(stream));
  return 0;
}
extern "C" int qh_getrs_ws_f32(int n, int nrhs, int batch, const float *LU, long sA, const int *perm, float *B, long sB,
                               void *ws, void *stream) {
  getrs_batched<float>(n, nrhs, batch, (const v2f *)LU, n, sA, perm, n, (v2f *)B, nrhs, sB, ws,
                       (hipStream_t)qh_stream(stream));
  return 0;
}
// The same for matrices one behind the other, with the limit of the slabs'
// rendezvous (0: one workgroup takes the slab unless it sees the others at once).
// Tests reach both ways through a solve with it.
extern "C" int qh_getrs_wait(int prec, int n, int nrhs, int batch, const double *LU, const int *perm, double *B,
                             unsigned long long wait, void *stream) {
  hipStream_t s = (hipStream_t)qh_stream(stream);
  void *ws = qh_dmalloc(qh_getrs_ws_bytes(prec, n, nrhs, batch));
  const long sA = (long)n * n, sB = (long)n * nrhs;
  if (prec == 32)
    getrs_batched<float>(n, nrhs, batch, (const v2f *)LU, n, sA, perm, n, (v2f *)B, nrhs, sB, ws, s, wait);
  else
    getrs_batched<double>(n, nrhs, batch, (const v2d *)LU, n, sA, perm, n, (v2d *)B, nrhs, sB, ws, s, wait);
  HIPCHK(hipStreamSynchronize(s));
  qh_dfree(ws);
  return 0;
}
// (work: n x nrhs x batch entries of scratch, as an earlier form of the solve
// needed; its own words are allocated here)
extern "C" int qh_getrs_batched_f64(int n, int nrhs, int batch, const double *LU, long sA, const int *perm, double *B, long sB,
                                    double *work, void *stream) {
  (void)work;
  void *ws = qh_dmalloc(getrs_ws_bytes<double>(n, nrhs, batch));
  qh_getrs_ws_f64(n, nrhs, batch, LU, sA, perm, B, sB, ws, stream);
  HIPCHK(hipStreamSynchronize((hipStream_t)qh_stream(stream)));
  qh_dfree(ws);
  return 0;
}
extern "C" int qh_getrf_batched_f32(int n, int batch, float *A, long sA, int *ipiv, int *perm, int *info,
                                    void *stream) {
  hipStream_t s = (hipStream_t)qh_stream(stream);
  if (n <= 0 || batch <= 0) return 0;
  getrf_batched<float>(n, batch, (v2f *)A, n, sA, ipiv, n, perm, info, s, ws_for(s, getrf_ws_bytes<float>(n, batch)));
  return 0;
}
// (work: n x nrhs x batch entries of scratch, as an earlier form of the solve
// needed; its own words are allocated here)
extern "C" int qh_getrs_batched_f32(int n, int nrhs, int batch, const float *LU, long sA, const int *perm, float *B, long sB,
                                    float *work, void *stream) {
  (void)work;
  void *ws = qh_dmalloc(getrs_ws_bytes<float>(n, nrhs, batch));
  qh_getrs_ws_f32(n, nrhs, batch, LU, sA, perm, B, sB, ws, stream);
  HIPCHK(hipStreamSynchronize((hipStream_t)qh_stream(stream)));
  qh_dfree(ws);
  return 0;
}
// C -= A B (FP64 complex, batched, row-major, packed leading dimensions)
extern "C" int qh_gemm_sub_f64(int M, int N, int K, int batch, const double *A, long lda, long sA, const double *B,
                               long ldb, long sB, double *C, long ldc, long sC, void *stream) {
  if (M <= 0 || N <= 0 || batch <= 0) return 0;
  if (N <= 4) {   // few right-hand sides: stream A once, a wave per row
    const dim3 g((unsigned)((M + 3) / 4), (unsigned)batch);
    hipStream_t s = (hipStream_t)qh_stream(stream);
#define QH_GV(NR) QH_LAUNCH(k_gemv_sub_f64<NR>, g, dim3(256), 0, s, M, K, (const v2d *)A, lda, sA, \
                                     (const v2d *)B, ldb, sB, (v2d *)C, ldc, sC)
    switch (N) { case 1: QH_GV(1); break; case 2: QH_GV(2); break; case 3: QH_GV(3); break; default: QH_GV(4); }
#undef QH_GV
    HIPCHK(hipGetLastError());
    return 0;
  }
  // more right-hand sides (the refinement residuals of Beyn nodes, N = l):
  // the library GEMM outside graph capture (it streams A near the HBM rate;
  // the tiled kernel reached a fifth of it at N = 32), the tiled kernel inside
  trailing_gemm<double>(M, N, K, batch, (const v2d *)A, lda, sA, (const v2d *)B, ldb, sB, (v2d *)C, ldc, sC,
                        (hipStream_t)qh_stream(stream));
  HIPCHK(hipGetLastError());
  return 0;
}
extern "C" int qh_gemm_sub_f32(int M, int N, int K, int batch, const float *A, long lda, long sA, const float *B,
                               long ldb, long sB, float *C, long ldc, long sC, void *stream) {
  QH_LAUNCH(k_gemm_sub<float>, dim3((N + GT - 1) / GT, (M + GT - 1) / GT, batch), dim3(256), 0,
                     (hipStream_t)qh_stream(stream), M, N, K, (const v2f *)A, lda, sA, (const v2f *)B, ldb, sB,
                     (v2f *)C, ldc, sC);
  HIPCHK(hipGetLastError());
  return 0;
}
extern "C" int qh_d2f(long n, const double *x, float *y, void *stream) {
  QH_LAUNCH(k_d2f, dim3(qh_stride_blocks(n)), dim3(256), 0, (hipStream_t)qh_stream(stream), n,
                     (const v2d *)x, (v2f *)y);
  return 0;
}
extern "C" int qh_f2d_add(long n, const float *d, double *x, void *stream) {
  QH_LAUNCH(k_f2d_add, dim3(qh_stride_blocks(n)), dim3(256), 0, (hipStream_t)qh_stream(stream), n,
                     (const v2f *)d, (v2d *)x);
  return 0;
}
extern "C" int qh_copy_c64(long n, const double *x, double *y, void *stream) {
  QH_LAUNCH(k_copy2d, dim3(qh_stride_blocks(n)), dim3(256), 0, (hipStream_t)qh_stream(stream), n,
                     (const v2d *)x, (v2d *)y);
  return 0;
}
// Frobenius norm of n complex values (synchronises).
extern "C" double qh_norm2_c64(long n, const double *x, void *stream) {
  hipStream_t s = (hipStream_t)qh_stream(stream);
  const int nb = 512;
  double *part = (double *)qh_dmalloc(nb * sizeof(double));
  QH_LAUNCH(k_sumsq, dim3(nb), dim3(256), 0, s, n, (const v2d *)x, part);
  double h[nb];
  HIPCHK(hipMemcpyAsync(h, part, sizeof h, hipMemcpyDeviceToHost, s));
  HIPCHK(hipStreamSynchronize(s));
  qh_dfree(part);
  double t = 0;
  for (int i = 0; i < nb; ++i) t += h[i];
  return sqrt(t);
}

// ---------------------------------------------------------------------------
// Mixed precision: FP32 LU on MFMA + FP64 iterative refinement.
// ---------------------------------------------------------------------------
extern "C" int qpms_hip_solve_mixed_dev(size_t n_, size_t nrhs_, const _Complex double *A_dev,
                                        _Complex double *B_dev, _Complex double *X_dev, double tol, int maxit,
                                        void *stream) {
  hipStream_t s = (hipStream_t)qh_stream(stream);
  const int n = (int)n_, nrhs = (int)nrhs_;
  const long nn = (long)n * n, nb = (long)n * nrhs;
  float *A32 = (float *)qh_dmalloc(nn * sizeof(v2f));
  int *ipiv = (int *)qh_dmalloc(n * sizeof(int));
  int *perm = (int *)qh_dmalloc(n * sizeof(int));
  int *dinfo = (int *)qh_dmalloc(sizeof(int));
  double *R = (double *)qh_dmalloc(nb * sizeof(v2d));
  float *R32 = (float *)qh_dmalloc(nb * sizeof(v2f));
  // words of the solves, and before them of the factorisation
  void *W32 = qh_dmalloc(std::max(getrs_ws_bytes<float>(n, nrhs, 1), getrf_ws_bytes<float>(n, 1)));
  HIPCHK(hipMemsetAsync(dinfo, 0, sizeof(int), s));
  qh_d2f(nn, (const double *)A_dev, A32, s);
  getrf_batched<float>(n, 1, (v2f *)A32, n, 0, ipiv, 0, perm, dinfo, s, (char *)W32);
  HIPCHK(hipMemsetAsync(X_dev, 0, nb * sizeof(v2d), s));
  const double normA = qh_norm2_c64(nn, (const double *)A_dev, s);
  const double normB = qh_norm2_c64(nb, (const double *)B_dev, s);
  int it = 0, ok = 0;
  double prev = INFINITY;
  qh_copy_c64(nb, (const double *)B_dev, R, s);
  for (it = 0; it < maxit; ++it) {
    qh_d2f(nb, R, R32, s);
    getrs_batched<float>(n, nrhs, 1, (const v2f *)A32, n, 0, perm, 0, (v2f *)R32, nrhs, 0, W32, s);
    qh_f2d_add(nb, R32, (double *)X_dev, s);
    // R = B - A X
    qh_copy_c64(nb, (const double *)B_dev, R, s);
    qh_gemm_sub_f64(n, nrhs, n, 1, (const double *)A_dev, n, 0, (const double *)X_dev, nrhs, 0, R, nrhs, 0, s);
    const double nr = qh_norm2_c64(nb, R, s);
    const double nx = qh_norm2_c64(nb, (const double *)X_dev, s);
    const double rel = nr / (normA * nx + normB * 1e-300);
    if (rel <= tol) { ok = 1; ++it; break; }
    if (!(rel < 0.5 * prev)) {   // stalled: accept at the FP64 rounding floor
      ok = (rel <= 1e-14);
      ++it;
      break;
    }
    prev = rel;
  }
  qh_dfree(A32); qh_dfree(ipiv); qh_dfree(perm); qh_dfree(dinfo); qh_dfree(R); qh_dfree(R32); qh_dfree(W32);
  if (ok) return it;
  // Refinement stalled: FP64 LU fallback on the GPU.
  double *A64 = (double *)qh_dmalloc(nn * sizeof(v2d));
  int *ip = (int *)qh_dmalloc(n * sizeof(int));
  int *pm = (int *)qh_dmalloc(n * sizeof(int));
  int *inf = (int *)qh_dmalloc(sizeof(int));
  void *work = qh_dmalloc(std::max(getrs_ws_bytes<double>(n, nrhs, 1), getrf_ws_bytes<double>(n, 1)));
  HIPCHK(hipMemsetAsync(inf, 0, sizeof(int), s));
  qh_copy_c64(nn, (const double *)A_dev, A64, s);
  qh_copy_c64(nb, (const double *)B_dev, (double *)X_dev, s);
  getrf_batched<double>(n, 1, (v2d *)A64, n, 0, ip, 0, pm, inf, s, (char *)work);
  getrs_batched<double>(n, nrhs, 1, (const v2d *)A64, n, 0, pm, 0, (v2d *)X_dev, nrhs, 0, work, s);
  HIPCHK(hipStreamSynchronize(s));
  qh_dfree(A64); qh_dfree(ip); qh_dfree(pm); qh_dfree(inf); qh_dfree(work);
  return -1;
}
