// dense.hip -- batched dense linear algebra on gfx950 for the fermion-bag
// determinants (full_determinant.c:144-186, fluctuation_determinant.c:
// 126-301, fermion_matrix.c:355-427): partial-pivot LU, log|det| and sign,
// inverse from the LU factors, GEMM updates on the matrix cores.
//
// A batch is a set of row-major square matrices in one device buffer:
// matrix b has order n[b], starts at element off[b], its pivots at poff[b].
// Every kernel takes the whole batch; matrices of different orders share a
// launch (blocks of a matrix that is already finished return at once).
//
// LU: right-looking with partial pivoting (the factors equal those of
// LAPACK's whole-row interchanges).  Up to order PR*PT, blocks of LOB = 128
// columns, each factored as register panels of 16 (FP64) or 32 columns, which also
// interchange the block's other columns and solve for U to their right
// (k_lu_panel_reg), and updates inside the block (k_lu_update); then, outside
// it, one launch for all interchanges of the block and U12 = L11^{-1} A12
// (k_lu_right), and one for A22 -= L21 U12, on MFMA 16x16x4 tiles.  Larger
// orders use panels of NB = 32 columns reduced through LDS, with a trailing
// update per panel.
#include "th2d_internal.h"

#include <mutex>

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "../../include/th2d_bag.h"

namespace {

constexpr int NB = 32;    // LU panel width
constexpr int BM = 64;    // GEMM tile rows
constexpr int BN = 64;    // GEMM tile cols
constexpr int BK = 16;    // GEMM k chunk

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

template <typename T> struct Mfma;
// Operand layout of both 16x16x4 instructions (lane l): A[l%16][l/16],
// B[l/16][l%16].  Result register r of lane l holds row row(l, r) and
// column l%16 -- rows are blocked by lane group in FP32 (4*(l/16) + r)
// but interleaved in FP64 (4*r + l/16), as measured on gfx950.
template <> struct Mfma<double> {
  using acc = v4d;
  static __device__ __forceinline__ acc op(double a, double b, acc c)
  {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * r + (lane >> 4); }
  // the row of operand lane i that puts row 4 g + r in register r of lane group g
  static __device__ __forceinline__ int solve_row(int i) { return 4 * (i & 3) + (i >> 2); }
};
template <> struct Mfma<float> {
  using acc = v4f;
  static __device__ __forceinline__ acc op(float a, float b, acc c)
  {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
  static __device__ __forceinline__ int solve_row(int i) { return i; }
};

// C[i][j] += alpha * sum_k A[i][k] B[k][j] for one BM x BN tile at
// (i0, j0); rows >= M, cols >= N, k >= K are skipped.  256 threads: wave w
// owns the 32x32 quadrant (w/2, w%2) as 2x2 MFMA blocks of 16x16; a
// thread's results sit at rows Mfma<T>::row(lane, r) of each block.
template <typename T, bool USE_MFMA>
__device__ void gemm_tile(const T *A, long lda, const T *B, long ldb, T *C, long ldc, int M, int N,
                          int K, T alpha, int i0, int j0, T *sA, T *sB)
{
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int wr = (wv >> 1) * 32, wc = (wv & 1) * 32;
  using Acc = typename Mfma<T>::acc;
  Acc acc[2][2];
  T vacc[4][4];
  if (USE_MFMA) {
    for (int a = 0; a < 2; a++)
      for (int b = 0; b < 2; b++) acc[a][b] = Acc{0, 0, 0, 0};
  } else {
    for (int a = 0; a < 4; a++)
      for (int b = 0; b < 4; b++) vacc[a][b] = 0;
  }
  // software pipeline: the next chunk's A and B entries are loaded into
  // registers while the current chunk is multiplied out of LDS
  constexpr int EA = BM * BK / 256, EB = BK * BN / 256;
  T ra[EA], rb[EB];
  // an FP64 tile inside the matrix loads its chunks without bounds checks
  // (a uniform branch per chunk), so the loads issue back to back; in FP32
  // the second path costs registers, and so occupancy
  const bool inner = sizeof(T) == 8 && i0 + BM <= M && j0 + BN <= N;
  auto fetch = [&](int k0) {
    if (inner && k0 + BK <= K) {
#pragma unroll
      for (int q = 0; q < EA; q++) {
        const int e = tid + q * 256, r = e / BK, c = e - r * BK;
        ra[q] = A[(i0 + r) * lda + k0 + c];
      }
#pragma unroll
      for (int q = 0; q < EB; q++) {
        const int e = tid + q * 256, r = e / BN, c = e - r * BN;
        rb[q] = B[(k0 + r) * ldb + j0 + c];
      }
      return;
    }
#pragma unroll
    for (int q = 0; q < EA; q++) {
      const int e = tid + q * 256, r = e / BK, c = e - r * BK;
      const int gi = i0 + r, gk = k0 + c;
      ra[q] = (gi < M && gk < K) ? A[gi * lda + gk] : (T)0;
    }
#pragma unroll
    for (int q = 0; q < EB; q++) {
      const int e = tid + q * 256, r = e / BN, c = e - r * BN;
      const int gk = k0 + r, gj = j0 + c;
      rb[q] = (gk < K && gj < N) ? B[gk * ldb + gj] : (T)0;
    }
  };
  fetch(0);
  for (int k0 = 0; k0 < K; k0 += BK) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < EA; q++) {
      const int e = tid + q * 256, r = e / BK, c = e - r * BK;
      sA[r * (BK + 1) + c] = ra[q];
    }
#pragma unroll
    for (int q = 0; q < EB; q++) {
      const int e = tid + q * 256, r = e / BN, c = e - r * BN;
      sB[r * (BN + 1) + c] = rb[q];
    }
    __syncthreads();
    if (k0 + BK < K) fetch(k0 + BK);
    if (USE_MFMA) {
#pragma unroll
      for (int kk = 0; kk < BK; kk += 4) {
        T av[2], bv[2];
        for (int a = 0; a < 2; a++) av[a] = sA[(wr + a * 16 + (lane & 15)) * (BK + 1) + kk + (lane >> 4)];
        for (int b = 0; b < 2; b++) bv[b] = sB[(kk + (lane >> 4)) * (BN + 1) + wc + b * 16 + (lane & 15)];
        for (int a = 0; a < 2; a++)
          for (int b = 0; b < 2; b++) acc[a][b] = Mfma<T>::op(av[a], bv[b], acc[a][b]);
      }
    } else {
      // thread owns the entries of the MFMA result layout:
      // rows wr + a*16 + row(lane, r), cols wc + b*16 + lane%16
      for (int kk = 0; kk < BK; kk++)
        for (int a = 0; a < 2; a++)
          for (int r = 0; r < 4; r++) {
            T av = sA[(wr + a * 16 + Mfma<T>::row(lane, r)) * (BK + 1) + kk];
            for (int b = 0; b < 2; b++)
              vacc[a * 2 + b][r] += av * sB[kk * (BN + 1) + wc + b * 16 + (lane & 15)];
          }
    }
  }
  for (int a = 0; a < 2; a++)
    for (int b = 0; b < 2; b++)
      for (int r = 0; r < 4; r++) {
        int gi = i0 + wr + a * 16 + Mfma<T>::row(lane, r);
        int gj = j0 + wc + b * 16 + (lane & 15);
        if (inner || (gi < M && gj < N)) {
          T v = USE_MFMA ? acc[a][b][r] : vacc[a * 2 + b][r];
          C[gi * ldc + gj] += alpha * v;
        }
      }
}

struct BatchView {
  const long *off;
  const int *n;
  const long *poff;
  int count;
};

// ----------------------------------------------------------------- LU ---
template <typename T>
__global__ void __launch_bounds__(256) k_lu_panel(T *base, BatchView bv, int *pivb, int *info,
                                                  int k)
{
  __shared__ double sval[256];
  __shared__ int sidx[256];
  const int b = blockIdx.x;
  const int n = bv.n[b];
  if (k >= n) return;
  T *A = base + bv.off[b];
  int *piv = pivb + bv.poff[b];
  const int jb = min(NB, n - k), tid = threadIdx.x;
  for (int j = k; j < k + jb; j++) {
    // pivot: largest |a_ij|, i >= j; ties to the smaller row
    double best = -1.0;
    int bi = n;
    for (int i = j + tid; i < n; i += 256) {
      double v = fabs((double)A[(long)i * n + j]);
      if (v > best) {
        best = v;
        bi = i;
      }
    }
    sval[tid] = best;
    sidx[tid] = bi;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
      if (tid < s) {
        double v2 = sval[tid + s];
        int i2 = sidx[tid + s];
        if (v2 > sval[tid] || (v2 == sval[tid] && i2 < sidx[tid])) {
          sval[tid] = v2;
          sidx[tid] = i2;
        }
      }
      __syncthreads();
    }
    const int p = sidx[0];
    const double pabs = sval[0];
    __syncthreads();
    if (tid == 0) {
      piv[j] = p;
      if (pabs == 0.0 && info[b] == 0) info[b] = j + 1;
    }
    if (p != j)
      for (int c = tid; c < n; c += 256) {
        T t0 = A[(long)j * n + c];
        A[(long)j * n + c] = A[(long)p * n + c];
        A[(long)p * n + c] = t0;
      }
    __syncthreads();
    const T pv = A[(long)j * n + j];
    if (pv != (T)0)
      for (int i = j + 1 + tid; i < n; i += 256) A[(long)i * n + j] /= pv;
    __syncthreads();
    const int w = k + jb - 1 - j;  // remaining panel columns
    if (w > 0)
      for (long e = tid; e < (long)(n - j - 1) * w; e += 256) {
        int i = j + 1 + (int)(e / w), c = j + 1 + (int)(e % w);
        A[(long)i * n + c] -= A[(long)i * n + j] * A[(long)j * n + c];
      }
    __syncthreads();
  }
}

constexpr int PT = 1024;  // most threads of the register panel
constexpr int PR = 3;     // panel rows per thread
constexpr int LOB = 128;  // outer block of the register-panel LU
template <typename T> constexpr int PW = sizeof(T) == 8 ? 16 : 32;  // panel columns

// DPP move of a lane's unsigned value; lanes the move does not write get 0.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ unsigned dpp_or0(unsigned v)
{
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xf, false);
}

// Maximum over lanes 0..15, read from lane 0: quads, half-rows, the row.
__device__ __forceinline__ unsigned row16_max(unsigned v)
{
  v = max(v, dpp_or0<0xB1, 0xf>(v));   // quad_perm [1,0,3,2]
  v = max(v, dpp_or0<0x4E, 0xf>(v));   // quad_perm [2,3,0,1]
  v = max(v, dpp_or0<0x141, 0xf>(v));  // row_half_mirror
  v = max(v, dpp_or0<0x140, 0xf>(v));  // row_mirror
  return (unsigned)__builtin_amdgcn_readlane((int)v, 0);
}

// Wave64 maximum: within rows, then rows 0..3 into lane 63.
__device__ __forceinline__ unsigned wave_max(unsigned v)
{
  v = max(v, dpp_or0<0xB1, 0xf>(v));
  v = max(v, dpp_or0<0x4E, 0xf>(v));
  v = max(v, dpp_or0<0x141, 0xf>(v));
  v = max(v, dpp_or0<0x140, 0xf>(v));
  v = max(v, dpp_or0<0x142, 0xa>(v));  // row_bcast:15 into rows 1, 3
  v = max(v, dpp_or0<0x143, 0xc>(v));  // row_bcast:31 into rows 2, 3
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// A pivot candidate's magnitude as integers that order alike: the upper (or,
// in FP32, the only) half plus one, so that 0 is "no candidate", and the
// lower half.
struct PivKey {
  unsigned hi, lo;
};
__device__ __forceinline__ PivKey piv_key(double v)  // v >= 0, or -1: none
{
  const long long b = __double_as_longlong(v);
  return {v < 0.0 ? 0u : (unsigned)(b >> 32) + 1u, (unsigned)b};
}
__device__ __forceinline__ PivKey piv_key(float v)
{
  return {v < 0.0f ? 0u : __float_as_uint(v) + 1u, 0u};
}

// Lane l's value, in scalar registers (one cost per wave, not per row).
__device__ __forceinline__ float lane_get(float v, int l)
{
  return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), l));
}
__device__ __forceinline__ double lane_get(double v, int l)
{
  const long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)b, l);
  const unsigned hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | lo);
}

// Division of a panel column by its pivot (0: left as it is), with the
// reciprocal taken once: the panel is bound by VALU issue, and the scaled
// division is ten operations.  FP64: the quotient corrected by its residual;
// a pivot far from 1 and its column are scaled by a power of two first (the
// column is no larger, so nothing overflows; below an infinite pivot, 0).
// FP32: the product in FP64.
template <typename T> struct PanelDiv;
template <> struct PanelDiv<double> {
  double p, r, s;
  __device__ __forceinline__ explicit PanelDiv(double pv)
  {
    const double m = fabs(pv);
    s = lane_get(m > 1.7976931348623157e308 ? 0.0
                : m > 0x1p500 ? 0x1p-500 : (m < 0x1p-500 && m > 0.0 ? 0x1p500 : 1.0), 0);
    p = lane_get(s == 0.0 || m == 0.0 ? 1.0 : pv * s, 0);
    double q = __builtin_amdgcn_rcp(p);
    q = __builtin_fma(q, __builtin_fma(-p, q, 1.0), q);
    q = __builtin_fma(q, __builtin_fma(-p, q, 1.0), q);
    r = lane_get(q, 0);
  }
  __device__ __forceinline__ double operator()(double a) const
  {
    a *= s;
    const double q = a * r;
    return __builtin_fma(r, __builtin_fma(-p, q, a), q);
  }
};
template <> struct PanelDiv<float> {
  double r;
  __device__ __forceinline__ explicit PanelDiv(float pv)
  {
    const double p = pv == 0.0f ? 1.0 : (double)pv;
    double q = __builtin_amdgcn_rcp(p);
    q = __builtin_fma(q, __builtin_fma(-p, q, 1.0), q);
    q = __builtin_fma(q, __builtin_fma(-p, q, 1.0), q);
    r = lane_get(fabs(p) > 3.4028234663852886e38 ? 0.0 : q, 0);
  }
  __device__ __forceinline__ float operator()(float a) const { return (float)((double)a * r); }
};

// One element of a matrix by a buffer access at a byte offset from its
// first element.  An offset at or beyond the resource's size (the matrix's
// n*n elements) reads 0 and drops the store.
constexpr unsigned BUF_OOR = 0x80000000u;
template <typename T>
__device__ __forceinline__ T buf_ld(__amdgpu_buffer_rsrc_t rs, unsigned voff)
{
  if constexpr (sizeof(T) == 8)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rs, voff, 0, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(rs, voff, 0, 0));
}
template <typename T>
__device__ __forceinline__ void buf_st(__amdgpu_buffer_rsrc_t rs, unsigned voff, T v)
{
  typedef unsigned u2v __attribute__((ext_vector_type(2)));
  if constexpr (sizeof(T) == 8)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2v, v), rs, voff, 0, 0);
  else
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rs, voff, 0, 0);
}

// Rows that an ordered run of interchanges moves: for the final row `dst`,
// the row its content comes from (pv[j]: the partner of row k + j).
__device__ __forceinline__ int swap_source(int dst, int k, int jb, const int *pv)
{
  int pos = dst;
  for (int j = jb - 1; j >= 0; j--) {
    const int p = pv[j], r = k + j;
    pos = pos == r ? p : (pos == p ? r : pos);
  }
  return pos;
}

// Panel of W = PW columns held in registers: one block of NT threads per matrix
// (256, 512 or 1024, the fewest that hold the rows left), row k + t + q*NT of
// the panel in thread t, slot q < PR (orders up to PR*PT).  Rows stay where
// they are; an interchange exchanges their positions (pos, from k).  Per
// column, with one barrier: each wave finds its largest |a_ij| and the
// smallest position attaining it (so ties go as in k_lu_panel) and posts it
// with that row's columns from j to LDS; after the barrier every wave reduces
// the NT/64 posts to the pivot and every thread scales its entries of the
// column and updates the panel's later columns, in registers.  Then the rows
// go out to their positions, and the panel's interchanges and U of its rows
// to the block's other columns (k0 <= c < k1).  k_lu_right applies the block's
// interchanges to the rest, so the factors equal those of whole-row swaps.
//
// Bound by a column's chain (posts, barrier, reduction, reciprocal: some 2500
// cycles) and, with 16 waves, by VALU issue.  Keys as integers, one reciprocal
// per column, the pivot's row in scalar registers and no exchange of rows: for
// 64 matrices of order 256..2304 an FP64 panel of 16 columns with 1024 threads
// 55 -> 47 us, and with the block's interchanges and U, which were a launch of
// 8-12 us.  (FP64 panels of 32 columns with up to 512 threads saved a tenth of
// their time, but a row takes 32 one-column updates in turn instead of 16 and a
// product: |A - L U| grew by 6 % on bag matrices.)  116..128 registers and 38 KB
// of LDS with 256 threads let four matrices share a CU: 1000 FP64 matrices of
// order 64 take 179 us (402 with one per CU).
template <typename T, int NT>
__global__ void __launch_bounds__(NT)
k_lu_panel_reg(T *base, BatchView bv, int *pivb, int *info, int k, int k0, int k1)
{
  constexpr int NW = NT / 64, W = PW<T>;
  static_assert(NW <= 16 && NT >= 2 * LOB && 2 * W <= NT, "posts in a row of lanes; the gather");
  // double-buffered by column parity: a buffer is rewritten two columns
  // later, after every thread has passed the barrier between
  __shared__ uint4 post[2][NW];  // key, row
  __shared__ __align__(16) T wrow[2][NW][W];  // each wave's candidate row
  __shared__ __align__(16) T sLt[W * W];      // L of the panel's rows, by columns
  __shared__ int pv[W], dst[2 * W], src[2 * W];
  __shared__ T stage[NT * (W + 1)];  // one slab of NT rows (at most 136 KiB)
  const int b = blockIdx.x;
  const int n = bv.n[b];
  if (k >= n) return;
  T *A = base + bv.off[b];
  int *piv = pivb + bv.poff[b];
  const int left = n - k, jb = min(W, left);
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  T a[PR][W];
  int pos[PR];  // -1: no such row
#pragma unroll
  for (int q = 0; q < PR; q++) {
    pos[q] = tid + q * NT < left ? tid + q * NT : -1;
#pragma unroll
    for (int c = 0; c < W; c++) a[q][c] = (T)0;
  }
  // rows arrive through LDS in slabs of NT rows, one per q, read
  // row-contiguously (W consecutive lanes per row) rather than one row per
  // lane; a thread's loads of a slab are all issued before the first wait.
  // Thread t moves column t % W of rows t / W + m * NT / W; elements
  // outside the matrix get an out-of-range offset.
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc(A, 0, (int)((long)n * n * sizeof(T)), 0x00020000);
  const int sc = tid % W, sr = tid / W;
  constexpr int SRS = NT / W;  // rows between a thread's elements
  auto soff = [&](int sr, int sc, int r0, int m) {
    const int i = k + r0 + sr + m * SRS;
    return (sc < jb && i < n) ? (unsigned)(((long)i * n + k + sc) * sizeof(T)) : BUF_OOR;
  };
#pragma unroll
  for (int q = 0; q < PR; q++) {
    const int r0 = q * NT;  // first panel row of the slab, from k
    if (r0 >= left) break;
    if (q) __syncthreads();  // the previous slab has been read
    T v[W];
#pragma unroll
    for (int m = 0; m < W; m++) v[m] = buf_ld<T>(rs, soff(sr, sc, r0, m));
#pragma unroll
    for (int m = 0; m < W; m++) stage[(sr + m * SRS) * (W + 1) + sc] = v[m];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < W; c++) a[q][c] = stage[tid * (W + 1) + c];
  }
#pragma clang loop unroll(full)
  for (int j = 0; j < W; j++) {
    if (j >= jb) continue;  // (a full unroll keeps a[][] in registers)
    const int par = j & 1;
    __builtin_amdgcn_sched_barrier(0);
    // the thread's largest |a_ij| of the rows left, first position on ties
    T best = -1;
    int bp = 0, bq = 0;
#pragma unroll
    for (int q = 0; q < PR; q++) {
      const T v = sizeof(T) == 8 ? (T)fabs(a[q][j]) : (T)fabsf(a[q][j]);
      if (pos[q] >= j && (v > best || (v == best && pos[q] < bp))) {
        best = v;
        bp = pos[q];
        bq = q;
      }
    }
    // the wave's
    const PivKey key = piv_key(best);
    const unsigned mh = wave_max(key.hi);
    unsigned long long at = __ballot(key.hi == mh);
    if (at & (at - 1)) {  // several with the same upper half
      const unsigned ml = wave_max(key.hi == mh ? key.lo : 0u);
      const bool on = key.hi == mh && key.lo == ml;
      const unsigned mp = wave_max(on ? ~(unsigned)bp : 0u);
      at = __ballot(on && (unsigned)bp == ~mp);
    }
    const int ls = __builtin_ctzll(at), qs = __builtin_amdgcn_readlane(bq, ls);
    if (lane == ls) {
      post[par][wv] = make_uint4(key.hi, key.lo, (unsigned)bp, 0u);
#pragma unroll
      for (int q = 0; q < PR; q++)
        if (q == qs) {
#pragma unroll
          for (int c = 0; c < W; c++)
            if (c >= j) wrow[par][wv][c] = a[q][c];
          __asm__ volatile("; slot %0" ::"i"(q));  // (else the slots' stores are merged
        }                                          // behind moves of the whole row)
    }
    __syncthreads();
    // every wave reduces the posts itself, one per lane: the largest, and the
    // smallest position at it
    int at16 = lane;  // (its address is formed here, not kept through the loop)
    __asm__ volatile("" : "+v"(at16));
    uint4 pk = post[par][at16 & (NW - 1)];
    if (at16 >= NW) pk.x = 0u;
    const unsigned gh = row16_max(pk.x);
    at = __ballot(pk.x == gh) & ((1ull << NW) - 1);
    if (at & (at - 1)) {
      const unsigned gl = row16_max(pk.x == gh ? pk.y : 0u);
      const unsigned gp = row16_max(pk.x == gh && pk.y == gl ? ~pk.z : 0u);
      at &= __ballot(pk.y == gl && pk.z == ~gp);
    }
    const int bw = __builtin_ctzll(at);
    // (no number among the candidates: position j stays, with NaN below)
    const int p = gh ? __builtin_amdgcn_readlane((int)pk.z, bw) : j;
    if (tid == 0) {
      pv[j] = k + p;
      if (gh == 1u && __builtin_amdgcn_readlane((int)pk.y, bw) == 0 && info[b] == 0)
        info[b] = k + j + 1;
    }
    T pl = wrow[par][bw][lane % W];  // column c of the pivot's row in lane c
    if (!gh) pl = (T)NAN;
#pragma unroll
    for (int q = 0; q < PR; q++) pos[q] = pos[q] == p ? j : (pos[q] == j ? p : pos[q]);
    const PanelDiv<T> div(lane_get(pl, j));
#pragma unroll
    for (int q = 0; q < PR; q++) {
      __builtin_amdgcn_sched_barrier(0);
      if (pos[q] > j) a[q][j] = div(a[q][j]);
    }
    // eight columns of the pivot's row at a time in scalar registers, for all
    // slots (from LDS for each slot: bound by LDS reads with 16 waves)
    constexpr int UC = 8;
#pragma unroll
    for (int h = 0; h < W / UC; h++) {
      const int c0 = j + 1 + h * UC;
      if (c0 >= W) continue;
      __builtin_amdgcn_sched_barrier(0);
      T u[UC];
#pragma unroll
      for (int i = 0; i < UC; i++) u[i] = c0 + i < W ? lane_get(pl, (c0 + i) % W) : (T)0;
#pragma unroll
      for (int q = 0; q < PR; q++)
        if (pos[q] > j) {
#pragma unroll
          for (int c = 0; c < W; c++)  // constant trip count: indices fold after unrolling
            if (c >= c0 && c < c0 + UC) a[q][c] -= a[q][j] * u[c - c0];
        }
    }
  }
  // the thread's row and column in a slab, recomputed here rather than
  // kept in registers through the column loop
  int t2 = tid;
  __asm__ volatile("" : "+v"(t2));
  const int sc2 = t2 % W, sr2 = t2 / W;
  if (tid < 2 * W) src[tid] = dst[tid] = -1;
#pragma unroll
  for (int q = 0; q < PR; q++) {
    const int r0 = q * NT;
    if (r0 >= left) break;
    __syncthreads();  // the slab before has been stored, the lists are cleared
#pragma unroll
    for (int t = 0; t < PR; t++)
      if (pos[t] >= r0 && pos[t] < r0 + NT) {
#pragma unroll
        for (int c = 0; c < W; c++) stage[(pos[t] - r0) * (W + 1) + c] = a[t][c];
        if (q == 0 && pos[t] < W) {
          dst[pos[t]] = k + pos[t];
          src[pos[t]] = k + tid + t * NT;
#pragma unroll
          for (int c = 0; c < W; c++) sLt[c * W + pos[t]] = a[t][c];
        }
        // (only rows that were among the panel's can have moved below them)
        if (t == 0 && tid < W && pos[0] >= W) {
          dst[W + tid] = k + pos[0];
          src[W + tid] = k + tid;
        }
      }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < W; m++)
      buf_st<T>(rs, soff(sr2, sc2, r0, m), stage[(sr2 + m * SRS) * (W + 1) + sc2]);
  }
  if (tid < jb) piv[k + tid] = pv[tid];
  if (k1 - k0 <= W) return;
  // the block's other columns: thread c of the first 128 takes the panel's
  // rows of column k0 + c, thread 128 + c the rows below that they exchange
  // with
  const int c = k0 + (tid & (LOB - 1)), half = tid / LOB;
  const bool mine = half < 2 && c < min(k1, n) && !(c >= k && c < k + W);
  T x[W];
#pragma unroll
  for (int r = 0; r < W; r++) {
    const int s = src[(half & 1) * W + r];  // (rows and columns that are not there: any in range)
    x[r] = A[(long)(s >= 0 ? s : k) * n + min(c, n - 1)];
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's rows are here
  __syncthreads();                     // and every wave's
  if (!mine) return;
  if (half == 0 && c > k) {  // (the panel is whole)
#pragma unroll
    for (int q = 0; q + 1 < W; q++) {
      if (q % 4 == 0) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = q + 1; r < W; r++) x[r] -= sLt[q * W + r] * x[q];
    }
  }
#pragma unroll
  for (int r = 0; r < W; r++) {
    const int d = dst[half * W + r];
    if (d >= 0) A[(long)d * n + c] = x[r];
  }
}

// U12 = L11^{-1} A12 on rows k..k+jb-1 of the columns from k + jb on, unit
// lower L11 of order jb <= JB (the LDS panels' block rows).  One thread per
// column; its column of U12 lives in registers (the loops over the JB
// rows unroll fully, so every index is a constant), L11 in LDS.
template <typename T, int JB>
__global__ void __launch_bounds__(256) k_lu_trsm(T *base, BatchView bv, int k)
{
  __shared__ T sL[JB * JB];
  const int b = blockIdx.y;
  const int n = bv.n[b];
  if (k >= n) return;
  const int jb = min(JB, n - k);
  const int cb = k + jb;
  if (cb >= n) return;
  T *A = base + bv.off[b];
  for (int e = threadIdx.x; e < jb * jb; e += 256) {
    const int r = e / jb, q = e - r * jb;
    sL[r * JB + q] = A[(long)(k + r) * n + k + q];
  }
  __syncthreads();
  const int c = cb + blockIdx.x * 256 + threadIdx.x;
  if (c >= n) return;
  T x[JB];
#pragma unroll
  for (int r = 0; r < JB; r++) x[r] = r < jb ? A[(long)(k + r) * n + c] : (T)0;
#pragma unroll
  for (int r = 1; r < JB; r++) {
    if (r < jb) {
      T s = x[r];
#pragma unroll
      for (int q = 0; q < r; q++) s -= sL[r * JB + q] * x[q];
      x[r] = s;
      A[(long)(k + r) * n + c] = s;
    }
  }
}

// A[r0:r1, c0:c1] -= A[r0:r1, kk:kk+K] A[kk:kk+K, c0:c1], every range
// clipped to the matrix's order: the trailing and in-block updates of the
// LU (L21 U12).
// (FP64 on the matrix cores: at most 128 VGPRs, four waves per SIMD)
template <typename T, bool MF>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 && MF ? 4 : 1)))
    k_lu_update(T *base, BatchView bv, int kk, int K, int r0, int r1, int c0, int c1)
{
  __shared__ T sA[BM * (BK + 1)];
  __shared__ T sB[BK * (BN + 1)];
  const int b = blockIdx.z;
  const int n = bv.n[b];
  const int kn = min(K, n - kk), m = min(r1, n) - r0, mc = min(c1, n) - c0;
  if (kn <= 0 || m <= 0 || mc <= 0) return;
  const int ti = blockIdx.y * BM, tj = blockIdx.x * BN;
  if (ti >= m || tj >= mc) return;
  T *A = base + bv.off[b];
  gemm_tile<T, MF>(A + (long)r0 * n + kk, n, A + (long)kk * n + c0, n, A + (long)r0 * n + c0, n,
                   m, mc, kn, (T)-1, ti, tj, sA, sB);
}

// log|det| and sign from the factors: sign = prod sign(u_ii) * (-1)^{#swaps}
template <typename T>
__global__ void __launch_bounds__(256) k_lu_logdet(const T *base, BatchView bv, const int *pivb,
                                                   const int *info, double *logabs, int *sign)
{
  __shared__ double sh[4];
  __shared__ int shn[256];
  const int b = blockIdx.x;
  const int n = bv.n[b];
  const T *A = base + bv.off[b];
  const int *piv = pivb + bv.poff[b];
  double acc = 0.0;
  int neg = 0;
  for (int i = threadIdx.x; i < n; i += 256) {
    double u = (double)A[(long)i * n + i];
    acc += log(fabs(u));
    neg += (u < 0) + (piv[i] != i);
  }
  double s = block_sum(acc, sh);
  shn[threadIdx.x] = neg;
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    for (int q = 0; q < 256; q++) t += shn[q];
    if (info[b]) {
      logabs[b] = -INFINITY;
      sign[b] = 0;
    } else {
      logabs[b] = n ? s : 0.0;
      sign[b] = (t & 1) ? -1 : 1;
    }
  }
}

// ------------------------------------------------- 128 x 64 GEMM tile ---
// Tile of CM x CN results held in registers by 256 threads: wave w owns
// rows 32 w .. 32 w + 31 as 2 x 4 MFMA blocks of 16 x 16.  Chunks of CK are
// double-buffered in LDS (one barrier per chunk; the next chunk's entries
// are in flight while this one is multiplied).  128 x 64 halves the LDS and
// global reads per flop of the 64 x 64 tile of gemm_tile; the B rows are CNP
// elements apart, so that the four k rows of an FP32 operand read fall on
// different banks.
constexpr int CM = 128, CN = 64, CK = 16, CNP = CN + 16;

// Workgroups go to the 8 XCDs in turn, and each XCD has its own L2: groups
// of gs tiles that read the same rows of a factor are given to one XCD
// (consecutive workgroups of it), so that the rows are fetched once per group
// instead of once per tile.  Workgroup id -> tile `w` of group `g` of matrix
// b, for `ng` groups per matrix; xcd_grid gives the number of workgroups.
struct XcdTile {
  int b, g, w;
};
__device__ __forceinline__ XcdTile xcd_tile(unsigned id, int gs, int ng)
{
  const unsigned r = id >> 3;
  const int gid = (int)(r / (unsigned)gs) * 8 + (int)(id & 7), b = gid / ng;
  // (rotated by the matrix: else, with ng even, a partly empty last group of
  // every matrix would fall on the same XCDs)
  return XcdTile{b, (gid + b) % ng, (int)(r % (unsigned)gs)};
}
inline unsigned xcd_grid(int gs, int ng, int count)
{
  return (unsigned)((((long)ng * count + 7) / 8) * 8 * gs);
}

// tx x ty tiles in gx x gy groups of sx x sy, at most 8 x 8 tiles to a group
// (and no more than there are: a group's unused tiles are workgroups too).
struct TileGroups {
  int gx, gy, sx, sy;
  TileGroups(int tx, int ty)
      : gx((tx + 7) / 8), gy((ty + 7) / 8), sx(std::min(tx, 8)), sy(std::min(ty, 8))
  {
  }
  unsigned grid(int count) const { return xcd_grid(sx * sy, gx * gy, count); }
  __device__ __forceinline__ XcdTile tile(unsigned id, int &row, int &col) const
  {
    const XcdTile xt = xcd_tile(id, sx * sy, gx * gy);
    row = xt.g / gx * sy + xt.w / sx;
    col = xt.g % gx * sx + xt.w % sx;
    return xt;
  }
};

template <typename T> struct TileMem {
  T a[2][CM * (CK + 1)];
  T b[2][CK * CNP];
};
template <typename T> using TileAcc = typename Mfma<T>::acc[2][4];

// Elements of a row-major matrix from (row, column 0) on, by buffer loads at
// 32-bit offsets: an element outside the range is given the offset OOR,
// beyond the resource, and reads as 0 without a branch.
template <typename R> struct TileSrc {
  const R *p;
  long ld;
  int rows, cols;  // what is left of the matrix from p
  // column offset c, row r0 (uniform) + r
  __device__ __forceinline__ R get(long r0, int r, int c0, int c) const
  {
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void *)(p + r0 * ld + c0), 0, 0x7fffffff, 0x00020000);
    const bool in = r0 + r < rows && c0 + c < cols;
    return buf_ld<R>(rs, in ? (unsigned)((r * ld + c) * sizeof(R)) : BUF_OOR);
  }
};

// tot -= A B (SLICED) or tot += A B of depth K, A and B given by their sources and, as they go to
// LDS, by ca(v, r, k) and cb(v, k, c) (a conversion, a triangle's mask).
// MF: on the matrix cores, else on the vector ALUs in the same result
// layout.  A chunk's entries are loaded two chunks ahead (one ahead, a
// workgroup alone on its CU waited for them: 1.8 us per chunk whose products
// take 0.45) and first touched when they go to LDS.  SLICED: the product is summed in slices of
// depth CS, each subtracted from `tot` by itself: one chain of 2304 terms was
// off by 1.4 times as much as the slices.
constexpr int CS = 32;
template <typename T, bool MF, bool SLICED, typename R, typename CA, typename CB>
__device__ __forceinline__ void tile_mac(TileAcc<T> &tot, int K, TileMem<T> &sm,
                                         const TileSrc<R> &A, const TileSrc<R> &B, CA ca, CB cb)
{
  if (K <= 0) return;
  TileAcc<T> own;
  TileAcc<T> &acc = SLICED ? own : tot;
  if (SLICED)
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int c = 0; c < 4; c++) acc[a][c] = typename Mfma<T>::acc{0, 0, 0, 0};
  const int tid = threadIdx.x, lane = tid & 63, wr = (tid >> 6) * 32;
  constexpr int EA = CM * CK / 256, EB = CK * CN / 256;
  const int ar = tid / CK, ac = tid % CK, br = tid / CN, bc = tid % CN;
  R ra[2][EA], rb[2][EB];  // chunk i in set i & 1
  auto fetch = [&](auto set, int k0) {
#pragma unroll
    for (int q = 0; q < EA; q++) ra[set][q] = A.get(0, ar + q * (256 / CK), k0, ac);
#pragma unroll
    for (int q = 0; q < EB; q++) rb[set][q] = B.get(k0, br + q * (256 / CN), 0, bc);
  };
  auto put = [&](auto set, int k0) {
#pragma unroll
    for (int q = 0; q < EA; q++) {
      const int r = ar + q * (256 / CK);
      sm.a[set][r * (CK + 1) + ac] = ca(ra[set][q], r, k0 + ac);
    }
#pragma unroll
    for (int q = 0; q < EB; q++) {
      const int k = br + q * (256 / CN);
      sm.b[set][k * CNP + bc] = cb(rb[set][q], k0 + k, bc);
    }
  };
  // chunk at k0, in LDS buffer (and register set) `set`; entries past K read
  // as 0 without a memory access, so the last chunks fetch and put no less
  auto step = [&](auto set, int k0) {
    constexpr int P = decltype(set)::value;
    __syncthreads();  // the chunk is in LDS; every wave has left the other buffer
    fetch(set, k0 + 2 * CK);
    const T *pa = sm.a[P], *pb = sm.b[P];
    if constexpr (MF) {
#pragma unroll
      for (int kk = 0; kk < CK; kk += 4) {
        T av[2], bv[4];
#pragma unroll
        for (int a = 0; a < 2; a++) av[a] = pa[(wr + a * 16 + (lane & 15)) * (CK + 1) + kk + (lane >> 4)];
#pragma unroll
        for (int b = 0; b < 4; b++) bv[b] = pb[(kk + (lane >> 4)) * CNP + b * 16 + (lane & 15)];
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
          for (int b = 0; b < 4; b++) acc[a][b] = Mfma<T>::op(av[a], bv[b], acc[a][b]);
      }
    } else {
      for (int kk = 0; kk < CK; kk++)
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const T av = pa[(wr + a * 16 + Mfma<T>::row(lane, r)) * (CK + 1) + kk];
#pragma unroll
            for (int b = 0; b < 4; b++) acc[a][b][r] += av * pb[kk * CNP + b * 16 + (lane & 15)];
          }
    }
    put(std::integral_constant<int, P ^ 1>{}, k0 + CK);
  };
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  static_assert(CS == 2 * CK, "a slice of the sum is two chunks");
  fetch(even, 0);
  fetch(odd, CK);
  put(even, 0);
  for (int k0 = 0; k0 < K; k0 += CS) {
    step(even, k0);
    step(odd, k0 + CK);
    if (SLICED)
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
          tot[a][c] -= acc[a][c];
          acc[a][c] = typename Mfma<T>::acc{0, 0, 0, 0};
        }
  }
}

// ------------------------------------------------------------ inverse ---
// A = P^T L U (rows exchanged in order by the pivots), A^-1 = U^-1 L^-1 P:
//   1. Z = L^-1, block rows of IB = 128 from the top; only columns up to the
//      block's last row are not zero, the others are never touched;
//   2. Z = U^-1 Z, block rows from the bottom;
//   3. X = Z P, a permutation of the columns.
// Each block row is one left-looking launch over the batch: a workgroup
// accumulates F[block, done rows] Z[done rows, 64 columns] in registers,
// subtracts it from the right-hand side and solves with the 128 x 128
// diagonal block by substitution (block_solve), so X is read and written once
// per phase.  4/3 n^3 flop; bound by the matrix cores where the batch fills the
// chip.  (Rank-32 updates of all of X after each 32-row solve took
// 2 n^3 flop and read and wrote X 72 times at order 2304: for 64 FP32
// matrices of order 256..2304, 21.3 ms.)
// Row permutation of the pivots: element v of the identity ends at position
// `pos` after the exchanges (perm[pos] = v).  One thread per element follows
// it through the pivots, which are the same address in every lane: 16 at a
// time in scalar registers, since one load per step is one latency per step.
constexpr int PC = 16;
__global__ void __launch_bounds__(256) k_perm(BatchView bv, const int *__restrict__ pivb,
                                              int *permb, long pstride)
{
  const int b = blockIdx.y;
  const int n = bv.n[b];
  if ((int)(blockIdx.x * 256) >= n) return;
  const int *__restrict__ piv = pivb + bv.poff[b];
  int *perm = permb + (pstride > 0 ? pstride * b : bv.poff[b]);
  const int v = blockIdx.x * 256 + threadIdx.x;
  int pos = v;
  int j = 0;
  for (; j + PC <= n; j += PC) {
    int p[PC];
#pragma unroll
    for (int t = 0; t < PC; t++) p[t] = piv[j + t];
#pragma unroll
    for (int t = 0; t < PC; t++) pos = pos == j + t ? p[t] : (pos == p[t] ? j + t : pos);
  }
  for (; j < n; j++) {
    const int p = piv[j];
    pos = pos == j ? p : (pos == p ? j : pos);
  }
  if (v < n) perm[pos] = v;
}

constexpr int IB = CM;     // block rows of the inverse

// x / u with r = 1 / u taken once for a column: the quotient corrected by its
// residual (FP64) or formed in FP64 (FP32); where that is not finite, the
// division itself.
__device__ __forceinline__ double near_rcp(double u)
{
  double r = __builtin_amdgcn_rcp(u);
  r = __builtin_fma(r, __builtin_fma(-u, r, 1.0), r);
  return __builtin_fma(r, __builtin_fma(-u, r, 1.0), r);
}
__device__ __forceinline__ double quot(double x, double u, double r)
{
  double q = x * r;
  q = __builtin_fma(r, __builtin_fma(-u, q, x), q);
  if (!(fabs(q) <= 1.7976931348623157e308)) q = x / u;
  return q;
}
__device__ __forceinline__ float quot(float x, float u, double r)
{
  float q = (float)((double)x * r);
  if (!(fabsf(q) <= 3.4028234663852886e38f)) q = x / u;
  return q;
}

// out <- T^-1 acc for the 128 x 64 tile of right-hand sides in acc and the
// triangle T (unit lower, or upper) of order jb <= 128 at D, by substitution:
// 32-row slices in turn, each followed by the update of the slices to come.
// In a slice, wave w solves 16 of the columns.  Lane (l15, g = l / 16) holds
// rows 4 g .. 4 g + 3 of column l15 of each 16-row tile: group b's turn comes
// with every earlier row subtracted, it substitutes in its 4 x 4 triangle, and
// its four rows go out to the later groups one product each (the other groups'
// rows enter as 0, so nothing but these rows is multiplied).  Bound by the
// chain of these products, 24 per slice.  Products with inverted triangles of 32
// rows took as long for the lower triangles and 7 % less per launch for the
// upper ones (64 FP32 matrices of order 256..2304: 203 us, 218 here), with
// residuals larger by 7-20 % on bag matrices and without bound where a triangle
// is ill-conditioned.
// `sol` is SOL<T, MF> elements of LDS: the slice before (sX) and after (sY) its
// solve, the four triangles, and (vector ALUs) the waves' blocks of T.
constexpr int SST = 34;
template <typename T, bool MF> constexpr int SOL = (MF ? 4 : 8) * 32 * SST + 2 * 32 * (CN + 1);
template <typename T, bool MF, bool UPPER>
__device__ __forceinline__ void block_solve(TileAcc<T> &acc, const T *D, long ld, int jb, T *sol,
                                            T *out, long ldo, int cols)
{
  constexpr int SXW = CN + 1, SX = 32 * SXW, ST = 32 * SST;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, l4 = lane >> 4;
  T *const sT = sol, *const sX = sol + 4 * ST, *const sY = sX + SX;
  {
    // the wave's diagonal block, identity past the matrix
    T *const st = sT + wv * ST;
    const TileSrc<T> Dw{D + (long)(wv * 32) * ld + wv * 32, ld, jb - wv * 32, jb - wv * 32};
    T v[16];
#pragma unroll
    for (int q = 0; q < 16; q++) v[q] = Dw.get(0, 2 * q + (lane >> 5), 0, lane & 31);
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int r = 2 * q + (lane >> 5), c = lane & 31;
      st[r * SST + c] = r == c && wv * 32 + r >= jb ? (T)1 : v[q];
    }
  }
#pragma unroll 1
  for (int q = 0; q < 4; q++) {
    const int s = UPPER ? 3 - q : q;  // the slice solved now, held by wave s
    if (s * 32 >= jb) continue;
    if (wv == s) {
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
          for (int r = 0; r < 4; r++)
            sX[(a * 16 + Mfma<T>::row(lane, r)) * SXW + c * 16 + l15] =
                s * 32 + a * 16 + Mfma<T>::row(lane, r) < jb ? acc[a][c][r] : (T)0;
    }
    const bool later = UPPER ? wv < s : wv > s;  // (uniform) the wave's slice is still to come
    T av[8][2];
    const TileSrc<T> E{D + (long)(wv * 32) * ld + s * 32, ld, jb - wv * 32, jb - s * 32};
    if (later)
#pragma unroll
      for (int kk = 0; kk < 8; kk++)
#pragma unroll
        for (int a = 0; a < 2; a++) av[kk][a] = E.get(0, a * 16 + l15, 0, kk * 4 + l4);
    __syncthreads();
    const T *const ti = sT + s * ST;
    if constexpr (MF) {
      const int col = wv * 16 + l15;
      const int ar = Mfma<T>::solve_row(l15);  // the row that operand lane l15 stands for
      typename Mfma<T>::acc x[2];
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int r = 0; r < 4; r++) x[a][r] = sX[(a * 16 + 4 * l4 + r) * SXW + col];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int a = UPPER ? 1 - h : h;
        const T *const ta = ti + a * 16 * SST + a * 16;  // the tile's triangle
        T d[4][4], v[4];
        double rc[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
#pragma unroll
          for (int j = 0; j < 4; j++)
            if (UPPER ? j >= i : j < i) d[i][j] = ta[(4 * l4 + i) * SST + 4 * l4 + j];
          v[i] = ta[ar * SST + 4 * l4 + i];
          v[i] = (UPPER ? (ar >> 2) < l4 : (ar >> 2) > l4) ? -v[i] : (T)0;
          if (UPPER) rc[i] = near_rcp((double)d[i][i]);
        }
        if (h == 1) {  // the other tile's rows, in the wave's columns of sY
          const int o = UPPER ? 16 : 0;
#pragma unroll
          for (int kk = 0; kk < 4; kk++)
            x[a] = Mfma<T>::op(-ti[(a * 16 + ar) * SST + o + kk * 4 + l4],
                               sY[(o + kk * 4 + l4) * SXW + col], x[a]);
        }
        T res[4] = {0, 0, 0, 0};
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const int b = UPPER ? 3 - g : g;
          T y[4];
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const int r = UPPER ? 3 - i : i;
            y[r] = x[a][r];
#pragma unroll
            for (int j = 0; j < i; j++) {
              const int c = UPPER ? 3 - j : j;
              y[r] -= d[r][c] * y[c];
            }
            if (UPPER) y[r] = quot(y[r], d[r][r], rc[r]);
          }
#pragma unroll
          for (int r = 0; r < 4; r++) res[r] = l4 == b ? y[r] : res[r];
          if (g < 3)
#pragma unroll
            for (int r = 0; r < 4; r++) x[a] = Mfma<T>::op(v[r], l4 == b ? y[r] : (T)0, x[a]);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int row = a * 16 + 4 * l4 + r;
          sY[row * SXW + col] = res[r];
          if (s * 32 + row < jb && col < cols) out[(long)(s * 32 + row) * ldo + col] = res[r];
        }
        __builtin_amdgcn_wave_barrier();
      }
    } else {
      // wave w holds rows 8 w .. 8 w + 7 of every column
      T x[8];
#pragma unroll
      for (int r = 0; r < 8; r++) x[r] = sX[(wv * 8 + r) * SXW + lane];
#pragma unroll 1
      for (int g = 0; g < 4; g++) {
        const int b = UPPER ? 3 - g : g;
        const T *const tb = ti + wv * 8 * SST + b * 8;  // the wave's rows, wave b's columns
        if (wv == b) {
#pragma unroll
          for (int i = 0; i < 8; i++) {
            const int r = UPPER ? 7 - i : i;
#pragma unroll
            for (int j = 0; j < i; j++) {
              const int c = UPPER ? 7 - j : j;
              x[r] -= tb[r * SST + c] * x[c];
            }
            if (UPPER) x[r] /= tb[r * SST + r];
            const int row = b * 8 + r;
            sY[row * SXW + lane] = x[r];
            if (s * 32 + row < jb && lane < cols) out[(long)(s * 32 + row) * ldo + lane] = x[r];
          }
        }
        __syncthreads();
        if (UPPER ? wv < b : wv > b)
#pragma unroll
          for (int c = 0; c < 8; c++) {
            const T yc = sY[(b * 8 + (UPPER ? 7 - c : c)) * SXW + lane];
#pragma unroll
            for (int r = 0; r < 8; r++) x[r] -= tb[r * SST + (UPPER ? 7 - c : c)] * yc;
          }
      }
    }
    __syncthreads();
    if (later) {  // acc -= F[own slice, solved slice] y
      TileAcc<T> part;
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 4; c++) part[a][c] = typename Mfma<T>::acc{0, 0, 0, 0};
      if constexpr (MF) {
#pragma unroll
        for (int kk = 0; kk < 8; kk++) {
          T yv[4];
#pragma unroll
          for (int c = 0; c < 4; c++) yv[c] = sY[(kk * 4 + l4) * SXW + c * 16 + l15];
#pragma unroll
          for (int a = 0; a < 2; a++)
#pragma unroll
            for (int c = 0; c < 4; c++) part[a][c] = Mfma<T>::op(av[kk][a], yv[c], part[a][c]);
        }
      } else {
        T *const se = sY + SX + wv * ST;  // the wave's own
#pragma unroll
        for (int kk = 0; kk < 8; kk++)
#pragma unroll
          for (int a = 0; a < 2; a++) se[(a * 16 + l15) * SST + kk * 4 + l4] = av[kk][a];
        __builtin_amdgcn_wave_barrier();
#pragma unroll 2
        for (int k = 0; k < 32; k++)
#pragma unroll
          for (int a = 0; a < 2; a++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const T v = se[(a * 16 + Mfma<T>::row(lane, r)) * SST + k];
#pragma unroll
              for (int c = 0; c < 4; c++) part[a][c][r] += v * sY[k * SXW + c * 16 + l15];
            }
      }
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[a][c] -= part[a][c];
    }
  }
}

// Block row t (from the top, or from the bottom when UPPER) of Z for every
// matrix that has one.
template <typename T, bool MF, bool UPPER>
__global__ void __launch_bounds__(256, MF ? 2 : 1) k_inv_rows(const T *LU, T *X, BatchView bv, int t,
                                                     TileGroups tg)
{
  // the solve's LDS follows the product's in the same memory
  __shared__ __align__(16) union {
    TileMem<T> mem;
    T sol[SOL<T, MF>];
  } sh;
  int tr, tc;
  const int b = tg.tile(blockIdx.x, tr, tc).b;
  if (b >= bv.count) return;
  const int n = bv.n[b];
  const int nb = (n + IB - 1) / IB;
  if (t >= nb) return;
  const int k0 = (UPPER ? nb - 1 - t : t) * IB, j0 = tc * CN;
  if (j0 >= n || (!UPPER && j0 >= k0 + IB)) return;  // (L^-1 is 0 there)
  const int jb = min(IB, n - k0);
  const T *F = LU + bv.off[b];
  T *Z = X + bv.off[b];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15;
  // the right-hand side (the identity, or L^-1) minus the product with the
  // rows already done (for L^-1: from the columns' own block row, above
  // which they are 0)
  TileAcc<T> acc;
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = k0 + wv * 32 + a * 16 + Mfma<T>::row(lane, r), col = j0 + c * 16 + l15;
        T rhs = row == col ? (T)1 : (T)0;
        if (UPPER) {
          rhs = 0;
          if (j0 < k0 + IB && row < n && col < n) rhs = Z[(long)row * n + col];
        }
        acc[a][c][r] = rhs;
      }
  const int kb = UPPER ? k0 + IB : j0 / IB * IB, K = UPPER ? n - kb : k0 - kb;
  tile_mac<T, MF, true>(
      acc, K, sh.mem, TileSrc<T>{F + (long)k0 * n + kb, n, jb, K},
      TileSrc<T>{Z + (long)kb * n + j0, n, K, n - j0}, [](T v, int, int) { return v; },
      [](T v, int, int) { return v; });
  __syncthreads();  // the product's LDS is free
  block_solve<T, MF, UPPER>(acc, F + (long)k0 * n + k0, n, jb, sh.sol, Z + (long)k0 * n + j0, n,
                            n - j0);
}

// The inverse of matrices of order n <= 64, one wave each: lane l solves for
// column l of Z = U^-1 L^-1, four rows at a time from the rows before (LU and Z
// in LDS, the coefficients the same in every lane), and with `permute` writes
// it as the column of A^-1 it is.  Bound by LDS reads and their latency.  A
// workgroup of k_inv_rows per matrix and phase is mostly idle at such orders:
// 1000 FP64 matrices of order 16 take 30 us here (431 in k_inv_rows with groups
// of eight tiles), of order 64 172 (468).  A few matrices of order above 32 are
// better off there: one of order 64 takes 49 us, 77 here.
constexpr int IS = 64;
inline bool small_inverse(const th2d_ctx *c, const th2d_batch *bt)
{
  return bt->max_n <= 32 || (bt->max_n <= IS && bt->count > c->num_cu);
}
template <typename T>
__global__ void __launch_bounds__(64) k_inv_small(const T *LU, T *X, BatchView bv, const int *pivb,
                                                  int nmax, int permute)
{
  extern __shared__ double is_raw[];
  const int b = blockIdx.x, lane = threadIdx.x;
  const int n = bv.n[b];
  if (n < 1 || n > nmax) return;  // (nmax <= IS)
  const int m = (n + 3) & ~3;  // identity beyond n
  T *S = (T *)is_raw, *Z = S + m * m;
  const T *F = LU + bv.off[b];
  for (int e = lane; e < m * m; e += 64) {
    const int r = e / m, c = e - r * m;
    S[e] = r < n && c < n ? F[r * n + c] : (r == c ? (T)1 : (T)0);
  }
  __syncthreads();
  if (lane < m) {
    T *z = Z + lane;
    for (int i = 0; i < m; i += 4) {  // L z = e_lane
      const T *si = S + i * m;
      T x[4];
#pragma unroll
      for (int t = 0; t < 4; t++) x[t] = i + t == lane ? (T)1 : (T)0;
      for (int q = 0; q < i; q += 4)
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const T y = z[(q + u) * m];
#pragma unroll
          for (int t = 0; t < 4; t++) x[t] -= si[t * m + q + u] * y;
        }
#pragma unroll
      for (int t = 0; t < 4; t++) {
#pragma unroll
        for (int u = 0; u < t; u++) x[t] -= si[t * m + i + u] * x[u];
        z[(i + t) * m] = x[t];
      }
    }
    for (int i = m - 4; i >= 0; i -= 4) {  // U z = z
      const T *si = S + i * m;
      T x[4];
#pragma unroll
      for (int t = 0; t < 4; t++) x[t] = z[(i + t) * m];
      for (int q = i + 4; q < m; q += 4)
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const T y = z[(q + u) * m];
#pragma unroll
          for (int t = 0; t < 4; t++) x[t] -= si[t * m + q + u] * y;
        }
#pragma unroll
      for (int t = 3; t >= 0; t--) {
#pragma unroll
        for (int u = 3; u > t; u--) x[t] -= si[t * m + i + u] * x[u];
        x[t] /= si[t * m + i + t];
        z[(i + t) * m] = x[t];
      }
    }
  }
  int col = lane;
  if (permute) {
    // element `lane` of the identity ends at position pos
    const int *piv = pivb + bv.poff[b];
    int pos = lane;
    for (int j = 0; j < n; j++) {
      const int p = piv[j];
      pos = pos == j ? p : (pos == p ? j : pos);
    }
    __syncthreads();  // the factors have been read: their LDS holds the columns
    int *pm = (int *)is_raw;
    if (lane < n) pm[pos] = lane;
    __syncthreads();
    if (lane < n) col = pm[lane];
  }
  if (lane < n) {
    T *Xb = X + bv.off[b] + col;
    for (int r = 0; r < n; r++) Xb[r * n] = Z[r * m + lane];
  }
}

// After the block of columns k .. k + 127: its interchanges on 64 of the
// other columns per workgroup, as a gather of the rows they touch, and to the
// right of the block U12 = L11^-1 A12 of its rows (block_solve).  `left`
// workgroups of a matrix take the columns before k.  (Interchanges one after
// the other, and U12 by four 32-row solves and updates in between, took 175 us
// for the first block of 64 FP64 matrices of order 256..2304; this takes 131.)
template <typename T, bool MF>
__global__ void __launch_bounds__(256, MF ? 2 : 1) k_lu_right(T *base, BatchView bv, const int *pivb, int k)
{
  __shared__ int pv[LOB], dst[2 * LOB], src[2 * LOB];
  __shared__ __align__(16) T sol[SOL<T, MF>];
  static_assert(LOB == CM && LOB == 128, "a block is a tile's rows");
  const int b = blockIdx.y;
  const int n = bv.n[b];
  if (k >= n) return;
  const int jb = min(LOB, n - k);
  const bool right = (int)blockIdx.x >= k / CN;
  const int c0 = right ? k + LOB + ((int)blockIdx.x - k / CN) * CN : (int)blockIdx.x * CN;
  if (c0 >= n) return;
  const int cols = min(CN, n - c0);
  T *A = base + bv.off[b];
  const int tid = threadIdx.x, lane = tid & 63, l15 = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid < jb) pv[tid] = pivb[bv.poff[b] + k + tid];
  __syncthreads();
  {
    const int j = tid % LOB;
    int d = -1;
    if (j < jb) d = tid < LOB ? k + j : (pv[j] >= k + jb ? pv[j] : -1);
    dst[tid] = d;
    src[tid] = d >= 0 ? swap_source(d, k, jb, pv) : -1;
  }
  __syncthreads();
  // the block's rows in the tile's layout, the rows below one per load
  const TileSrc<T> S{A + c0, n, n, cols};
  TileAcc<T> acc;
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int q = src[wv * 32 + a * 16 + Mfma<T>::row(lane, r)];
#pragma unroll
      for (int c = 0; c < 4; c++) acc[a][c][r] = S.get(0, q >= 0 ? q : n, 0, c * 16 + l15);
    }
  T below[32];
#pragma unroll
  for (int i = 0; i < 32; i++) {
    const int q = src[LOB + wv * 32 + i];
    below[i] = S.get(0, q >= 0 ? q : n, 0, lane);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's rows are here
  __syncthreads();                     // and every wave's
#pragma unroll
  for (int i = 0; i < 32; i++) {
    const int q = dst[LOB + wv * 32 + i];
    if (q >= 0 && lane < cols) A[(long)q * n + c0 + lane] = below[i];
  }
  if (right) {  // (a block with columns to its right is whole)
    block_solve<T, MF, false>(acc, A + (long)k * n + k, n, jb, sol, A + (long)k * n + c0, n, cols);
    return;
  }
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int t = wv * 32 + a * 16 + Mfma<T>::row(lane, r);
#pragma unroll
      for (int c = 0; c < 4; c++)
        if (t < jb && c * 16 + l15 < cols) A[(long)(k + t) * n + c0 + c * 16 + l15] = acc[a][c][r];
    }
}

// A22 -= L21 U12 beyond the block of columns k .. k + 127, one 128 x 64 tile
// per workgroup; 8 x 8 tiles of a matrix share an XCD, and with it the rows of
// L21 and the columns of U12.
template <typename T, bool MF>
__global__ void __launch_bounds__(256, 2) k_lu_trail(T *base, BatchView bv, int k, TileGroups tg)
{
  __shared__ TileMem<T> mem;
  int tr, tc;
  const XcdTile xt = tg.tile(blockIdx.x, tr, tc);
  if (xt.b >= bv.count) return;
  const int n = bv.n[xt.b], ce = k + LOB;
  const int i0 = ce + tr * CM, j0 = ce + tc * CN;
  if (i0 >= n || j0 >= n) return;
  T *A = base + bv.off[xt.b];
  const int lane = threadIdx.x & 63, wr = (threadIdx.x >> 6) * 32, l15 = lane & 15;
  TileAcc<T> acc;
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int c = 0; c < 4; c++) acc[a][c] = typename Mfma<T>::acc{0, 0, 0, 0};
  tile_mac<T, MF, false>(
      acc, LOB, mem, TileSrc<T>{A + (long)i0 * n + k, n, n - i0, LOB},
      TileSrc<T>{A + (long)k * n + j0, n, LOB, n - j0}, [](T v, int, int) { return v; },
      [](T v, int, int) { return v; });
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int row = i0 + wr + a * 16 + Mfma<T>::row(lane, r);
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int col = j0 + c * 16 + l15;
        if (row < n && col < n) A[(long)row * n + col] -= acc[a][c][r];
      }
    }
}

// X = Z P in place: row by row through LDS (up to PERM_LDS bytes a row), or,
// for longer rows, the column exchanges in reverse order, one thread per row.
constexpr size_t PERM_LDS = 64 << 10;
template <typename T>
__global__ void __launch_bounds__(256) k_permute_cols(T *X, BatchView bv, const int *permb,
                                                      long pstride)
{
  extern __shared__ double perm_raw[];
  T *row = (T *)perm_raw;
  const int b = blockIdx.y;
  const int n = bv.n[b];
  const int *perm = permb + (pstride > 0 ? pstride * b : bv.poff[b]);
  T *Z = X + bv.off[b];
  for (int r = blockIdx.x; r < n; r += gridDim.x) {
    T *p = Z + (long)r * n;
    for (int c = threadIdx.x; c < n; c += 256) row[perm[c]] = p[c];
    __syncthreads();
    for (int c = threadIdx.x; c < n; c += 256) p[c] = row[c];
    __syncthreads();
  }
}

template <typename T>
__global__ void __launch_bounds__(256) k_exchange_cols(T *X, BatchView bv, const int *pivb)
{
  const int b = blockIdx.y;
  const int n = bv.n[b];
  const int *piv = pivb + bv.poff[b];
  for (int r = blockIdx.x * 256 + threadIdx.x; r < n; r += gridDim.x * 256) {
    T *p = X + bv.off[b] + (long)r * n;
    for (int j = n - 1; j >= 0; j--) {
      const int q = piv[j];
      if (q != j) {
        const T v = p[j];
        p[j] = p[q];
        p[q] = v;
      }
    }
  }
}

// generic batched GEMM: C += alpha A B (jobs in device memory)
template <typename T, bool MF>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 && MF ? 4 : 1)))
    k_gemm_jobs(T *base, const th2d_gemm_job *jobs, double alpha)
{
  __shared__ T sA[BM * (BK + 1)];
  __shared__ T sB[BK * (BN + 1)];
  const th2d_gemm_job J = jobs[blockIdx.z];
  const int ti = blockIdx.y * BM, tj = blockIdx.x * BN;
  if (ti >= J.M || tj >= J.N) return;
  gemm_tile<T, MF>(base + J.a, J.lda, base + J.b, J.ldb, base + J.c, J.ldc, J.M, J.N, J.K,
                   (T)alpha, ti, tj, sA, sB);
}

__global__ void k_f64_to_f32_n(float *d, const double *s, long n)
{
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256)
    d[i] = (float)s[i];
}

// ---- FP64 correction of an FP32 LU's log-determinant ---------------------
// Partial sums of tr(B^-1 E) with B = P^T L U, E = A - B the FP64 residual of
// the FP32 factorisation and Z = U^-1 L^-1 (FP32, k_inv_rows): with the rows
// of E in the factorisation's order,
//   tr(B^-1 E) = sum_{r,i} Z[i][r] (A[perm[r]][i] - (L U)[r][i]).
// A workgroup forms one 128 x 64 tile of L U in FP64 on the matrix cores,
// from the FP32 factors promoted as they are loaded (the triangles masked:
// depth min(r, i) + 1 only), and takes its part of the trace from the
// registers, so L U never goes to memory.  (Promoting L and U to dense FP64
// matrices first and reading the product back for the trace took 5.4 ms for
// 64 matrices of order 256..2304, 2.8 of them the product.)
// Tiles of a group share an XCD: L rows and U columns.
template <bool MF>
__global__ void __launch_bounds__(256, 2) k_refine_trace(const double *A, const float *LU32,
                                                         const float *Z, const int *permb,
                                                         BatchView bv, double *part, int nparts,
                                                         TileGroups tg)
{
  __shared__ union {
    TileMem<double> mem;
    float z[CN * (CM + 1)];
  } sh;
  __shared__ double red[4];
  int tr, tc;
  const XcdTile xt = tg.tile(blockIdx.x, tr, tc);
  const int b = xt.b;
  if (b >= bv.count) return;
  const int n = bv.n[b];
  const int tx = (n + CN - 1) / CN, ty = (n + CM - 1) / CM;
  // the deepest tiles first
  const int ti = ty - 1 - tr, tj = tx - 1 - tc;
  if (ti < 0 || tj < 0) return;
  const int tile = ti * tx + tj, i0 = ti * CM, j0 = tj * CN;
  const long off = bv.off[b];
  const float *F = LU32 + off;
  const int *perm = permb + bv.poff[b];
  const int tid = threadIdx.x, lane = tid & 63, wr = (tid >> 6) * 32;
  TileAcc<double> acc;
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int c = 0; c < 4; c++) acc[a][c] = v4d{0, 0, 0, 0};
  const int K = min(n, min(i0 + CM, j0 + CN));
  // depth up to the first diagonal element of the tile's rows or columns,
  // then the rest with the triangles masked
  const int K1 = min(i0, j0);
  tile_mac<double, MF, false>(
      acc, K1, sh.mem, TileSrc<float>{F + (long)i0 * n, n, n - i0, K1},
      TileSrc<float>{F + j0, n, K1, n - j0}, [](float v, int, int) { return (double)v; },
      [](float v, int, int) { return (double)v; });
  __syncthreads();
  tile_mac<double, MF, false>(
      acc, K - K1, sh.mem, TileSrc<float>{F + (long)i0 * n + K1, n, n - i0, K - K1},
      TileSrc<float>{F + (long)K1 * n + j0, n, K - K1, n - j0},
      [&](float v, int r, int k) {  // L
        const int row = i0 + r - K1;
        return k < row ? (double)v : (k == row ? 1.0 : 0.0);
      },
      [&](float v, int k, int c) { return k + K1 <= j0 + c ? (double)v : 0.0; });  // U
  __syncthreads();
  // Z[j0 ..][i0 ..] (64 rows of 128) through LDS, read by columns
#pragma unroll 8
  for (int e = tid; e < CN * CM; e += 256) {
    const int c = e / CM, r = e % CM;
    sh.z[c * (CM + 1) + r] = Z[off + (long)min(j0 + c, n - 1) * n + min(i0 + r, n - 1)];
  }
  __syncthreads();
  double sum = 0.0;
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int lr = wr + a * 16 + Mfma<double>::row(lane, r), row = i0 + lr;
      const double *pa = A + off + (long)perm[min(row, n - 1)] * n;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int lc = c * 16 + (lane & 15), col = j0 + lc;
        const double e = pa[min(col, n - 1)] - acc[a][c][r];
        if (row < n && col < n) sum += (double)sh.z[lc * (CM + 1) + lr] * e;
      }
    }
  const double s = block_sum(sum, red);
  if (tid == 0) part[(long)b * nparts + tile] = s;
}

// logabs[b] += the matrix's partial sums, in a fixed order.
__global__ void __launch_bounds__(256) k_add_correction(const double *part, int nparts,
                                                        BatchView bv, const int *info,
                                                        double *logabs)
{
  __shared__ double red[4];
  const int b = blockIdx.x;
  const int n = bv.n[b];
  if (info[b]) return;
  const int nt = ((n + CN - 1) / CN) * ((n + CM - 1) / CM);
  double acc = 0.0;
  for (int q = threadIdx.x; q < nt; q += 256) acc += part[(long)b * nparts + q];
  const double s = block_sum(acc, red);
  if (threadIdx.x == 0) logabs[b] += s;
}

static int g_use_mfma = -1;
static int g_lu_reg_panel = 1;  // register panel when it fits (th2d_set_lu_panel)
bool use_mfma()
{
  if (g_use_mfma < 0) {
    const char *e = getenv("TH2D_DENSE_MFMA");
    g_use_mfma = e ? atoi(e) != 0 : 1;
  }
  return g_use_mfma != 0;
}

BatchView view(const th2d_batch *b) { return BatchView{b->off, b->n, b->poff, b->count}; }

template <typename T>
void launch_update(th2d_ctx *c, bool mf, T *A, BatchView bv, int count, int kk, int K, int r0,
                   int r1, int c0, int c1, int N)
{
  const int rows = std::min(r1, N) - r0, cols = std::min(c1, N) - c0;
  if (rows <= 0 || cols <= 0) return;
  dim3 g((cols + BN - 1) / BN, (rows + BM - 1) / BM, count);
  if (mf)
    hipLaunchKernelGGL((k_lu_update<T, true>), g, dim3(256), 0, c->stream, A, bv, kk, K, r0, r1, c0,
                       c1);
  else
    hipLaunchKernelGGL((k_lu_update<T, false>), g, dim3(256), 0, c->stream, A, bv, kk, K, r0, r1, c0,
                       c1);
}

template <typename T, int NT>
void launch_panel(th2d_ctx *c, T *A, BatchView bv, int count, int *piv, int *info, int kk, int k,
                  int ce)
{
  hipLaunchKernelGGL((k_lu_panel_reg<T, NT>), dim3(count), dim3(NT), 0, c->stream, A, bv, piv,
                     info, kk, k, ce);
}

template <typename T, bool MF>
void lu_blocks(th2d_ctx *c, const th2d_batch *bt, T *A, int *piv, int *info)
{
  const BatchView bv = view(bt);
  const int N = bt->max_n, cnt = bt->count;
  constexpr int END = 1 << 30;  // a range bound past every order
  constexpr int W = PW<T>;
  for (int k = 0; k < N; k += LOB) {
    const int ce = std::min(k + LOB, N), rows = N - k;  // the most rows a matrix has left
    for (int kk = k; kk < ce; kk += W) {
      if (rows <= PR * 256) launch_panel<T, 256>(c, A, bv, cnt, piv, info, kk, k, ce);
      else if (rows <= PR * 512) launch_panel<T, 512>(c, A, bv, cnt, piv, info, kk, k, ce);
      else launch_panel<T, PT>(c, A, bv, cnt, piv, info, kk, k, ce);
      const int cb = kk + W;
      if (cb < ce) launch_update<T>(c, MF, A, bv, cnt, kk, W, cb, END, cb, ce, N);
    }
    const int tiles = k / CN + (N - ce + CN - 1) / CN;
    if (tiles > 0)
      hipLaunchKernelGGL((k_lu_right<T, MF>), dim3(tiles, cnt), dim3(256), 0, c->stream, A, bv, piv,
                         k);
    if (ce >= N) break;
    // FP64: 64 x 64 tiles, four waves per SIMD (first of 17 launches 713 us; 128
    // x 64 tiles at two: 851).  FP32: 128 x 64 (all 17: 2.2 ms; 64 x 64: 3.5).
    if constexpr (sizeof(T) == 8) {
      launch_update<T>(c, MF, A, bv, cnt, k, LOB, ce, END, ce, END, N);
    } else {
      const TileGroups tg((N - ce + CN - 1) / CN, (N - ce + CM - 1) / CM);
      hipLaunchKernelGGL((k_lu_trail<T, MF>), dim3(tg.grid(cnt)), dim3(256), 0, c->stream, A, bv, k,
                         tg);
    }
  }
}

template <typename T>
int lu_run(th2d_ctx *c, const th2d_batch *bt, T *A, int *piv, int *info)
{
  BatchView bv = view(bt);
  TH2D_TRY(th2d_memset(c, info, 0, sizeof(int) * bt->count));
  const bool mf = use_mfma();
  const int N = bt->max_n, cnt = bt->count;
  constexpr int END = 1 << 30;  // a range bound past every order
  if (bt->max_n <= PR * PT && g_lu_reg_panel) {
    if (mf) lu_blocks<T, true>(c, bt, A, piv, info);
    else lu_blocks<T, false>(c, bt, A, piv, info);
  } else {
    // the LDS-reduction panel of width NB, which swaps whole rows itself
    for (int k = 0; k < N; k += NB) {
      hipLaunchKernelGGL(k_lu_panel<T>, dim3(cnt), dim3(256), 0, c->stream, A, bv, piv, info, k);
      const int rest = N - k - NB;
      if (rest > 0) {
        hipLaunchKernelGGL((k_lu_trsm<T, NB>), dim3((rest + 255) / 256, cnt), dim3(256), 0,
                           c->stream, A, bv, k);
        launch_update<T>(c, mf, A, bv, cnt, k, NB, k + NB, END, k + NB, END, N);
      }
    }
  }
  TH2D_HIP(hipGetLastError());
  return TH2D_OK;
}

// Z = U^-1 L^-1 of every matrix (k_inv_rows), in X.
template <typename T, bool MF>
void inverse_rows(th2d_ctx *c, const th2d_batch *bt, const T *LU, T *X)
{
  const BatchView bv = view(bt);
  const int N = bt->max_n, nb = (N + IB - 1) / IB;
  const int ct = (N + CN - 1) / CN;
  for (int t = 0; t < nb; t++) {
    const TileGroups tg(std::min(ct, (t + 1) * (IB / CN)), 1);
    hipLaunchKernelGGL((k_inv_rows<T, MF, false>), dim3(tg.grid(bt->count)), dim3(256), 0, c->stream,
                       LU, X, bv, t, tg);
  }
  const TileGroups tg(ct, 1);
  for (int t = 0; t < nb; t++)
    hipLaunchKernelGGL((k_inv_rows<T, MF, true>), dim3(tg.grid(bt->count)), dim3(256), 0, c->stream,
                       LU, X, bv, t, tg);
}

template <typename T>
void inverse_small(th2d_ctx *c, const th2d_batch *bt, const T *LU, const int *piv, T *X,
                   int permute)
{
  const int m = (bt->max_n + 3) & ~3;
  hipLaunchKernelGGL(k_inv_small<T>, dim3(bt->count), dim3(64), 2 * sizeof(T) * m * m, c->stream, LU,
                     X, view(bt), piv, bt->max_n, permute);
}

template <typename T>
void inverse_unpermuted(th2d_ctx *c, const th2d_batch *bt, const T *LU, T *X)
{
  if (small_inverse(c, bt)) {
    inverse_small<T>(c, bt, LU, nullptr, X, 0);
    return;
  }
  if (use_mfma()) inverse_rows<T, true>(c, bt, LU, X);
  else inverse_rows<T, false>(c, bt, LU, X);
}

void perm_launch(th2d_ctx *c, const th2d_batch *bt, const int *piv, int *perm, long pstride)
{
  hipLaunchKernelGGL(k_perm, dim3((bt->max_n + 255) / 256, bt->count), dim3(256), 0, c->stream,
                     view(bt), piv, perm, pstride);
}

// The inverse in launches alone (no allocation, no host wait): perm is the
// scratch of each matrix's permutation, at its pivot offset poff[b] (pstride
// 0) or at b * pstride.
template <typename T>
int inverse_launch(th2d_ctx *c, const th2d_batch *bt, const T *LU, const int *piv, T *X,
                   int *perm, long pstride)
{
  const BatchView bv = view(bt);
  const int N = bt->max_n;
  if (N < 1) return TH2D_OK;
  if (small_inverse(c, bt)) {
    inverse_small<T>(c, bt, LU, piv, X, 1);
    TH2D_HIP(hipGetLastError());
    return TH2D_OK;
  }
  inverse_unpermuted<T>(c, bt, LU, X);
  if (sizeof(T) * (size_t)N <= PERM_LDS) {
    perm_launch(c, bt, piv, perm, pstride);
    hipLaunchKernelGGL(k_permute_cols<T>, dim3(std::min(N, 1024), bt->count), dim3(256),
                       sizeof(T) * (size_t)N, c->stream, X, bv, (const int *)perm, pstride);
  } else {
    hipLaunchKernelGGL(k_exchange_cols<T>, dim3((N + 255) / 256, bt->count), dim3(256), 0,
                       c->stream, X, bv, piv);
  }
  TH2D_HIP(hipGetLastError());
  return TH2D_OK;
}

template <typename T>
int inverse_run(th2d_ctx *c, const th2d_batch *bt, const T *LU, const int *piv, T *X)
{
  // scratch: permutation per matrix (same offsets as the pivots)
  long total = 0;
  std::vector<long> h(bt->count);
  TH2D_HIP(hipMemcpyAsync(h.data(), bt->poff, sizeof(long) * bt->count, hipMemcpyDeviceToHost,
                          c->stream));
  TH2D_HIP(hipStreamSynchronize(c->stream));
  for (int i = 0; i < bt->count; i++) total = std::max(total, h[i]);
  TH2D_TRY(th2d_buf_reserve(c->bag, sizeof(int) * (size_t)(total + bt->max_n + 64)));
  return inverse_launch<T>(c, bt, LU, piv, X, (int *)c->bag.ptr, 0);
}

}  // namespace

// ---- the allocation-free inverse ------------------------------------------
// Its permutation scratch is a file-scope device array: each GPU holds its
// own copy until the process ends.  Host code uses the per-device address
// from hipGetSymbolAddress (looked up when a context is created on that
// device), never the array's name.  Calls that overlap on one GPU share
// the array and race.
constexpr long kNoAllocPermInts = 1L << 22;  // 16 MiB: count * max_n <= 4,194,304
static __device__ __align__(256) int scratch[kNoAllocPermInts];
static std::mutex g_scratch_mu;
static int *g_scratch_ptr[64];

namespace th2d {
int noalloc_scratch_init(int device)
{
  if (device < 0 || device >= 64) return TH2D_EARG;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[device]) return TH2D_OK;
  void *p = nullptr;
  TH2D_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  g_scratch_ptr[device] = (int *)p;
  return TH2D_OK;
}
}  // namespace th2d

static int *noalloc_scratch(int device)
{
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  return (device >= 0 && device < 64) ? g_scratch_ptr[device] : nullptr;
}


// ================================================================ ABI ===
extern "C" int th2d_lu_batched(th2d_ctx *c, const th2d_batch *b, void *A, int precision, int *piv,
                               int *info)
{
  if (!c || !b || !A || !piv || !info || b->count < 1 || b->max_n < 0) return TH2D_EARG;
  if (precision == TH2D_PREC_F64) return lu_run<double>(c, b, (double *)A, piv, info);
  if (precision == TH2D_PREC_F32) return lu_run<float>(c, b, (float *)A, piv, info);
  return TH2D_EARG;
}

extern "C" int th2d_lu_logdet(th2d_ctx *c, const th2d_batch *b, const void *LU, int precision,
                              const int *piv, const int *info, double *logabs, int *sign)
{
  if (!c || !b || !LU || !piv || !info || !logabs || !sign || b->count < 1) return TH2D_EARG;
  BatchView bv = view(b);
  if (precision == TH2D_PREC_F64)
    hipLaunchKernelGGL(k_lu_logdet<double>, dim3(b->count), dim3(256), 0, c->stream,
                       (const double *)LU, bv, piv, info, logabs, sign);
  else if (precision == TH2D_PREC_F32)
    hipLaunchKernelGGL(k_lu_logdet<float>, dim3(b->count), dim3(256), 0, c->stream,
                       (const float *)LU, bv, piv, info, logabs, sign);
  else return TH2D_EARG;
  TH2D_HIP(hipGetLastError());
  return TH2D_OK;
}

// log|det A| of FP32 factors, corrected in FP64: log det A = log det B +
// tr(B^-1 E) + O(|B^-1 E|^2) with B = P^T L U (the FP32 factors), E = A - B
// formed in FP64 from the promoted factors and B^-1 the FP32 inverse from the
// same factors (k_inv_rows, its columns not permuted back: k_refine_trace).
extern "C" int th2d_lu_logdet_refined(th2d_ctx *c, const th2d_batch *b, const double *A,
                                      const float *LU32, const int *piv, const int *info,
                                      double *logabs, int *sign)
{
  if (!c || !b || !A || !LU32 || !piv || !info || !logabs || !sign || b->count < 1)
    return TH2D_EARG;
  TH2D_TRY(th2d_lu_logdet(c, b, LU32, TH2D_PREC_F32, piv, info, logabs, sign));
  const int count = b->count;
  std::vector<long> off(count), poff(count);
  std::vector<int> n(count);
  TH2D_HIP(hipMemcpyAsync(off.data(), b->off, sizeof(long) * count, hipMemcpyDeviceToHost, c->stream));
  TH2D_HIP(hipMemcpyAsync(poff.data(), b->poff, sizeof(long) * count, hipMemcpyDeviceToHost,
                          c->stream));
  TH2D_HIP(hipMemcpyAsync(n.data(), b->n, sizeof(int) * count, hipMemcpyDeviceToHost, c->stream));
  TH2D_HIP(hipStreamSynchronize(c->stream));
  long total = 0, ptotal = 0;
  int nmax = 0;
  for (int q = 0; q < count; q++) {
    total = std::max(total, off[q] + (long)n[q] * n[q]);
    ptotal = std::max(ptotal, poff[q] + (long)n[q]);
    nmax = std::max(nmax, n[q]);
  }
  if (nmax < 1) return TH2D_OK;
  const int nparts = ((nmax + CN - 1) / CN) * ((nmax + CM - 1) / CM);  // tiles of a matrix
  // scratch: Z (FP32, the batch's layout), perm, partials
  const size_t zb = (sizeof(float) * (size_t)total + 255) & ~(size_t)255;
  const size_t pb = (sizeof(int) * (size_t)ptotal + 255) & ~(size_t)255;
  TH2D_TRY(th2d_buf_reserve(c->misc, zb + pb + sizeof(double) * (size_t)count * nparts));
  float *Z = (float *)c->misc.ptr;
  int *perm = (int *)((char *)c->misc.ptr + zb);
  double *part = (double *)((char *)c->misc.ptr + zb + pb);
  const BatchView bv = view(b);
  inverse_unpermuted<float>(c, b, LU32, Z);
  perm_launch(c, b, piv, perm, 0);
  const TileGroups tg((nmax + CN - 1) / CN, (nmax + CM - 1) / CM);
  const dim3 grid(tg.grid(count));
  if (use_mfma())
    hipLaunchKernelGGL(k_refine_trace<true>, grid, dim3(256), 0, c->stream, A, LU32,
                       (const float *)Z, (const int *)perm, bv, part, nparts, tg);
  else
    hipLaunchKernelGGL(k_refine_trace<false>, grid, dim3(256), 0, c->stream, A, LU32,
                       (const float *)Z, (const int *)perm, bv, part, nparts, tg);
  hipLaunchKernelGGL(k_add_correction, dim3(count), dim3(256), 0, c->stream, part, nparts, bv,
                     info, logabs);
  TH2D_HIP(hipGetLastError());
  return TH2D_OK;
}

extern "C" int th2d_lu_inverse(th2d_ctx *c, const th2d_batch *b, const void *LU, int precision,
                               const int *piv, void *X)
{
  if (!c || !b || !LU || !piv || !X || LU == X || b->count < 1) return TH2D_EARG;
  if (precision == TH2D_PREC_F64) return inverse_run<double>(c, b, (const double *)LU, piv, (double *)X);
  if (precision == TH2D_PREC_F32) return inverse_run<float>(c, b, (const float *)LU, piv, (float *)X);
  return TH2D_EARG;
}

extern "C" int th2d_lu_inverse_noalloc(th2d_ctx *c, const th2d_batch *b, const void *LU,
                                       int precision, const int *piv, void *X)
{
  if (!c || !b || !LU || !piv || !X || LU == X || b->count < 1 || b->max_n < 1) return TH2D_EARG;
  if ((long)b->count * b->max_n > kNoAllocPermInts) return TH2D_EARG;  // beyond the scratch
  int *perm = noalloc_scratch(c->device);
  if (!perm) return TH2D_EARG;  // no context was created on this device
  if (precision == TH2D_PREC_F64)
    return inverse_launch<double>(c, b, (const double *)LU, piv, (double *)X, perm, b->max_n);
  if (precision == TH2D_PREC_F32)
    return inverse_launch<float>(c, b, (const float *)LU, piv, (float *)X, perm, b->max_n);
  return TH2D_EARG;
}

extern "C" int th2d_gemm_batched(th2d_ctx *c, void *base, int precision,
                                 const th2d_gemm_job *jobs_dev, int count, int max_m, int max_n,
                                 double alpha)
{
  if (!c || !base || !jobs_dev || count < 1 || max_m < 0 || max_n < 0) return TH2D_EARG;
  if (!max_m || !max_n) return TH2D_OK;
  dim3 g((max_n + BN - 1) / BN, (max_m + BM - 1) / BM, count);
  const bool mf = use_mfma();
  if (precision == TH2D_PREC_F64) {
    if (mf) hipLaunchKernelGGL((k_gemm_jobs<double, true>), g, dim3(256), 0, c->stream, (double *)base, jobs_dev, alpha);
    else hipLaunchKernelGGL((k_gemm_jobs<double, false>), g, dim3(256), 0, c->stream, (double *)base, jobs_dev, alpha);
  } else if (precision == TH2D_PREC_F32) {
    if (mf) hipLaunchKernelGGL((k_gemm_jobs<float, true>), g, dim3(256), 0, c->stream, (float *)base, jobs_dev, alpha);
    else hipLaunchKernelGGL((k_gemm_jobs<float, false>), g, dim3(256), 0, c->stream, (float *)base, jobs_dev, alpha);
  } else return TH2D_EARG;
  TH2D_HIP(hipGetLastError());
  return TH2D_OK;
}

extern "C" int th2d_set_dense_mfma(int on)
{
  g_use_mfma = on ? 1 : 0;
  return TH2D_OK;
}

extern "C" int th2d_set_lu_lookahead(int on)
{
  (void)on;  // the blocks run in order
  return TH2D_OK;
}

extern "C" int th2d_set_lu_panel(int reg)
{
  g_lu_reg_panel = reg ? 1 : 0;
  return TH2D_OK;
}

extern "C" int th2d_copy_f64_to_f32(th2d_ctx *c, float *d, const double *s, long n)
{
  if (!c || (!d && n) || (!s && n) || n < 0) return TH2D_EARG;
  if (!n) return TH2D_OK;
  long blocks = std::min(4096L, (n + 255) / 256);
  hipLaunchKernelGGL(k_f64_to_f32_n, dim3((unsigned)blocks), dim3(256), 0, c->stream, d, s, n);
  TH2D_HIP(hipGetLastError());
  return TH2D_OK;
}
