// lu.hip -- blocked complex LU with partial pivoting, triangular solves
// and the refinement helpers, complex128 and complex64.
//
// Right-looking blocked algorithm (outer block nb, inner block 32):
//  * a 32-column sub-panel is factored in one launch: row-by-row partial
//    pivoting (lu_panel.inc), or tournament pivoting (k_panel_ts below) for
//    the mixed solver's complex64 factors;
//  * row interchanges are applied to the other columns,
//  * U12 = L11^{-1} A12 (unit-lower triangular solve),
//  * A22 -= A21 U12 on the matrix cores: v_mfma_f64_16x16x4f64 for
//    complex128 and v_mfma_f32_16x16x4f32 for complex64, four real
//    products per complex product.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <type_traits>
#include <vector>

#include "gate.h"
#include "lu.h"
#include "lu_dev.h"
#include "prof.h"
#include "ws.h"

namespace scuffx {


typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

template <typename T> struct CT;
// Both 16x16x4 instructions take A[i][k] from lane i + 16k and B[k][j]
// from lane j + 16k; result element r of a lane sits in column lane % 16
// and row 4*(lane/16) + r for f32 but row lane/16 + 4r for f64 (measured
// on gfx950 with a one-wave probe).
template <> struct CT<double2> {
  typedef double R;
  typedef d4 V4;
  __device__ static inline V4 mfma(R a, R b, V4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  __device__ static inline V4 zero() { return V4{0, 0, 0, 0}; }
  __device__ static inline int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <> struct CT<double> {
  typedef double R;
  typedef d4 V4;
  __device__ static inline V4 mfma(R a, R b, V4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  __device__ static inline V4 zero() { return V4{0, 0, 0, 0}; }
  __device__ static inline int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <> struct CT<float2> {
  typedef float R;
  typedef f4 V4;
  __device__ static inline V4 mfma(R a, R b, V4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  __device__ static inline V4 zero() { return V4{0, 0, 0, 0}; }
  __device__ static inline int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

// ---------------------------------------------------------------------
// C[m x n] -= A[m x k] B[k x n]  (ACC)  or  C = A B  (!ACC);
// 64x64 block tile, 4 waves of 32x32, K staged 16 at a time through LDS
// as separate real/imag planes, four real MFMAs per complex product.
// ---------------------------------------------------------------------
#define GBM 64
#define GBN 64
#define GBK 16

// G3M (complex64 only): three real products per complex product instead of
// four (Gauss / "3M": T1 = Ar Br, T2 = Ai Bi, T3 = (Ar + Ai)(Br + Bi),
// Re = T1 - T2, Im = T3 - T1 - T2; normwise stable, Higham, SIAM J. Matrix
// Anal. Appl. 13 (1992) 681-687), a quarter fewer MFMAs
template <typename T, bool ACC, bool G3M = false>
__global__ void __launch_bounds__(256)
k_gemm(long m, long n, long k, const T *A, long lda, const T *B, long ldb, T *C, long ldc, long bsa)
{
  {
    const long z = blockIdx.z;   // instance of a batch (bsa elements apart)
    A += z * bsa; B += z * bsa; C += z * bsa;
  }
  typedef typename CT<T>::R R;
  typedef typename CT<T>::V4 V4;
  __shared__ R sAr[GBK][GBM + 4], sAi[GBK][GBM + 4], sBr[GBK][GBN + 4], sBi[GBK][GBN + 4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave >> 1, wc = wave & 1;
  const long row0 = (long)blockIdx.x * GBM, col0 = (long)blockIdx.y * GBN;
  V4 accr[2][2], acci[2][2], acc3[2][2];
  for (int a = 0; a < 2; a++)
    for (int b = 0; b < 2; b++) { accr[a][b] = CT<T>::zero(); acci[a][b] = CT<T>::zero(); acc3[a][b] = CT<T>::zero(); }
  // tiles of chunk k0 into registers: all eight global loads in flight
  // before any LDS store
  auto load = [&](long k0, T (&v)[4], T (&u)[4]) {
    if (row0 + GBM <= m && col0 + GBN <= n && k0 + GBK <= k) {
#pragma unroll
      for (int s = 0; s < 4; s++) {
        v[s] = A[(row0 + (tid & 63)) + (k0 + (tid >> 6) + 4 * s) * lda];
        u[s] = B[(k0 + (tid & 15)) + (col0 + (tid >> 4) + 16 * s) * ldb];
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4; s++) {
        int i = tid & 63, kk = (tid >> 6) + 4 * s;
        long gi = row0 + i, gk = k0 + kk;
        if (gi < m && gk < k) v[s] = A[gi + gk * lda]; else { v[s] = zero_v<T>(); }
        int kb = tid & 15, j = (tid >> 4) + 16 * s;
        long gkb = k0 + kb, gj = col0 + j;
        if (gkb < k && gj < n) u[s] = B[gkb + gj * ldb]; else { u[s] = zero_v<T>(); }
      }
    }
  };
  // the next chunk's loads are issued before this chunk's products
  // (complex64: 98 registers, four waves per SIMD; complex128: two)
  constexpr bool PF = true;
  T v[4], u[4];
  if (PF && k > 0) load(0, v, u);
  for (long k0 = 0; k0 < k; k0 += GBK) {
    if (!PF) load(k0, v, u);
#pragma unroll
    for (int s = 0; s < 4; s++) {
      int i = tid & 63, kk = (tid >> 6) + 4 * s;
      sAr[kk][i] = v[s].x; sAi[kk][i] = v[s].y;
      int kb = tid & 15, j = (tid >> 4) + 16 * s;
      sBr[kb][j] = u[s].x; sBi[kb][j] = u[s].y;
    }
    __syncthreads();
    if (PF && k0 + GBK < k) load(k0 + GBK, v, u);
    for (int kk0 = 0; kk0 < GBK; kk0 += 4) {
      int kk = kk0 + (lane >> 4);
      R ar[2], ai[2], br[2], bi[2];
      for (int t = 0; t < 2; t++) {
        ar[t] = sAr[kk][wr * 32 + t * 16 + (lane & 15)];
        ai[t] = sAi[kk][wr * 32 + t * 16 + (lane & 15)];
        br[t] = sBr[kk][wc * 32 + t * 16 + (lane & 15)];
        bi[t] = sBi[kk][wc * 32 + t * 16 + (lane & 15)];
      }
      if constexpr (G3M) {
        // accr: T1, acci: T2, acc3: T3
        R as[2], bs[2];
        for (int t = 0; t < 2; t++) { as[t] = ar[t] + ai[t]; bs[t] = br[t] + bi[t]; }
        for (int ti = 0; ti < 2; ti++)
          for (int tj = 0; tj < 2; tj++) {
            accr[ti][tj] = CT<T>::mfma(ar[ti], br[tj], accr[ti][tj]);
            acci[ti][tj] = CT<T>::mfma(ai[ti], bi[tj], acci[ti][tj]);
            acc3[ti][tj] = CT<T>::mfma(as[ti], bs[tj], acc3[ti][tj]);
          }
      } else {
        for (int ti = 0; ti < 2; ti++)
          for (int tj = 0; tj < 2; tj++) {
            // acc = Re/Im of -(A B) when accumulating into C, +(A B) otherwise
            const R sg = ACC ? (R)-1 : (R)1;
            accr[ti][tj] = CT<T>::mfma(sg * ar[ti], br[tj], accr[ti][tj]);
            accr[ti][tj] = CT<T>::mfma(-sg * ai[ti], bi[tj], accr[ti][tj]);
            acci[ti][tj] = CT<T>::mfma(sg * ar[ti], bi[tj], acci[ti][tj]);
            acci[ti][tj] = CT<T>::mfma(sg * ai[ti], br[tj], acci[ti][tj]);
          }
      }
    }
    __syncthreads();
  }
  for (int ti = 0; ti < 2; ti++)
    for (int tj = 0; tj < 2; tj++)
      for (int r = 0; r < 4; r++) {
        long gi = row0 + wr * 32 + ti * 16 + CT<T>::row(lane, r);
        long gj = col0 + wc * 32 + tj * 16 + (lane & 15);
        if (gi < m && gj < n) {
          R re = accr[ti][tj][r], im = acci[ti][tj][r];
          if constexpr (G3M) {
            const R t1 = accr[ti][tj][r], t2 = acci[ti][tj][r];
            re = ACC ? t2 - t1 : t1 - t2;
            im = ACC ? (t1 + t2) - acc3[ti][tj][r] : acc3[ti][tj][r] - (t1 + t2);
          }
          T c;
          if (ACC) { c = C[gi + gj * ldc]; c.x += re; c.y += im; }
          else { c.x = re; c.y = im; }
          C[gi + gj * ldc] = c;
        }
      }
}

// Real (double) C -= A B or C = A B: the same 64x64 tile and k-chunk
// staging, one v_mfma_f64_16x16x4f64 per product; each wave owns a 32x64
// strip (2 x 4 tiles of 16x16), so one LDS read of A feeds four products.
template <bool ACC>
__global__ void __launch_bounds__(256)
k_gemm_r(long m, long n, long k, const double *A, long lda, const double *B, long ldb, double *C, long ldc, long bsa)
{
  {
    const long z = blockIdx.z;
    A += z * bsa; B += z * bsa; C += z * bsa;
  }
  __shared__ double sA[GBK][2 * GBM + 4], sB[GBK][GBN + 4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long row0 = (long)blockIdx.x * 2 * GBM, col0 = (long)blockIdx.y * GBN;
  d4 acc[2][4];
  for (int a = 0; a < 2; a++) for (int b = 0; b < 4; b++) acc[a][b] = d4{0, 0, 0, 0};
  // A chunk: 128 rows x 16, B chunk: 16 x 64 per k-chunk
  auto load = [&](long k0, double (&v)[8], double (&u)[4]) {
    if (row0 + 2 * GBM <= m && col0 + GBN <= n && k0 + GBK <= k) {
#pragma unroll
      for (int q = 0; q < 8; q++) v[q] = A[(row0 + (tid & 127)) + (k0 + (tid >> 7) + 2 * q) * lda];
#pragma unroll
      for (int q = 0; q < 4; q++) u[q] = B[(k0 + (tid & 15)) + (col0 + (tid >> 4) + 16 * q) * ldb];
    } else {
#pragma unroll
      for (int q = 0; q < 8; q++) {
        long gi = row0 + (tid & 127), gk = k0 + (tid >> 7) + 2 * q;
        v[q] = (gi < m && gk < k) ? A[gi + gk * lda] : 0.0;
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        long gk = k0 + (tid & 15), gj = col0 + (tid >> 4) + 16 * q;
        u[q] = (gk < k && gj < n) ? B[gk + gj * ldb] : 0.0;
      }
    }
  };
  double v[8], u[4];
  if (k > 0) load(0, v, u);
  for (long k0 = 0; k0 < k; k0 += GBK) {
#pragma unroll
    for (int q = 0; q < 8; q++) sA[(tid >> 7) + 2 * q][tid & 127] = v[q];
#pragma unroll
    for (int q = 0; q < 4; q++) sB[tid & 15][(tid >> 4) + 16 * q] = u[q];
    __syncthreads();
    if (k0 + GBK < k) load(k0 + GBK, v, u);
    for (int kk0 = 0; kk0 < GBK; kk0 += 4) {
      const int kk = kk0 + (lane >> 4);
      double ar[2], br[4];
      for (int t = 0; t < 2; t++) ar[t] = sA[kk][wave * 32 + t * 16 + (lane & 15)];
      for (int t = 0; t < 4; t++) br[t] = sB[kk][t * 16 + (lane & 15)];
      const double sg = ACC ? -1.0 : 1.0;
      for (int ti = 0; ti < 2; ti++)
        for (int tj = 0; tj < 4; tj++)
          acc[ti][tj] = __builtin_amdgcn_mfma_f64_16x16x4f64(sg * ar[ti], br[tj], acc[ti][tj], 0, 0, 0);
    }
    __syncthreads();
  }
  for (int ti = 0; ti < 2; ti++)
    for (int tj = 0; tj < 4; tj++)
      for (int r = 0; r < 4; r++) {
        long gi = row0 + wave * 32 + ti * 16 + (lane >> 4) + 4 * r;
        long gj = col0 + tj * 16 + (lane & 15);
        if (gi < m && gj < n) {
          if (ACC) C[gi + gj * ldc] += acc[ti][tj][r];
          else C[gi + gj * ldc] = acc[ti][tj][r];
        }
      }
}

static int gemm_kind(const double2 *) { return PK_GEMM_C128; }
static int gemm_kind(const float2 *) { return PK_GEMM_C64; }
static int gemm_kind(const double *) { return PK_GEMM_F64; }

// lds_pad: extra (unused) LDS per workgroup, which caps how many of its
// workgroups share a CU
template <typename T, bool ACC>
static void gemm(long m, long n, long k, const T *A, long lda, const T *B, long ldb, T *C, long ldc,
                 hipStream_t s, unsigned lds_pad = 0, int nbat = 1, long bsa = 0, bool g3m = false)
{
  if (m <= 0 || n <= 0 || k <= 0 || nbat <= 0) return;
  int tok = prof_begin(s, gemm_kind(A));
  if constexpr (IsReal<T>::v) {
    dim3 grid((unsigned)((m + 2 * GBM - 1) / (2 * GBM)), (unsigned)((n + GBN - 1) / GBN), (unsigned)nbat);
    hipLaunchKernelGGL((k_gemm_r<ACC>), grid, dim3(256), lds_pad, s, m, n, k, A, lda, B, ldb, C, ldc, bsa);
    prof_end(s, tok, 2.0 * (double)m * (double)n * (double)k * nbat);
  } else {
    dim3 grid((unsigned)((m + GBM - 1) / GBM), (unsigned)((n + GBN - 1) / GBN), (unsigned)nbat);
    if (std::is_same<T, float2>::value && ACC && g3m)
      hipLaunchKernelGGL((k_gemm<T, ACC, true>), grid, dim3(256), lds_pad, s, m, n, k, A, lda, B, ldb, C, ldc, bsa);
    else
      hipLaunchKernelGGL((k_gemm<T, ACC>), grid, dim3(256), lds_pad, s, m, n, k, A, lda, B, ldb, C, ldc, bsa);
    prof_end(s, tok, 8.0 * (double)m * (double)n * (double)k * nbat);
  }
}

template <typename T>
static void gemm_sub(long m, long n, long k, const T *A, long lda, const T *B, long ldb, T *C, long ldc,
                     hipStream_t s, unsigned lds_pad = 0, int nbat = 1, long bsa = 0, bool g3m = false)
{
  gemm<T, true>(m, n, k, A, lda, B, ldb, C, ldc, s, lds_pad, nbat, bsa, g3m);
}

// The mixed solver's complex64 factorization (a preconditioner for the
// complex128 refinement) updates with three real products per complex
// product; SCUFFX_GEMM_3M=0, read at every factorization, keeps four (its
// normwise error is 2-4x smaller, which matters only past condition
// numbers of ~1e7, where complex64 factors barely precondition anyway)
static bool mixed_gemm_3m()
{
  const char *e = getenv("SCUFFX_GEMM_3M");
  return !(e && !strcmp(e, "0"));
}

__global__ void k_fill_u64(unsigned long long *w, unsigned long long v, long n)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) w[i] = v;
}

// inverse of a panel's unit-lower w x w block (identity outside it), column
// t of it by substitution: for the block rows of the mixed solver's
// factorization with row-by-row pivoting
template <typename T>
__global__ void __launch_bounds__(64) k_unit_inv(const T *A, long lda, long r0, int w, T *linv)
{
  __shared__ T L[PW][PW + 1];
  const int t = threadIdx.x;
  for (int e = t; e < PW * PW; e += 64) {
    const int rr = e % PW, q = e / PW;
    L[rr][q] = (rr < w && q < w) ? A[(r0 + rr) + (r0 + q) * lda] : zero_v<T>();
  }
  __syncthreads();
  if (t >= PW) return;
  T x[PW];
#pragma unroll
  for (int r = 0; r < PW; r++) {
    T v = (r == t) ? unit_v<T>() : zero_v<T>();
    if (r < w && t < w) {
#pragma unroll
      for (int k = 0; k < r; k++) v = csub(v, cmul(L[r][k], x[k]));
    }
    x[r] = v;
  }
#pragma unroll
  for (int r = 0; r < PW; r++) linv[(long)t * PW + r] = x[r];
}

// ---------------------------------------------------------------------
// Tournament-pivoting panel for the complex64 factorization of the mixed
// solver (communication-avoiding LU, "TSLU": Grigori, Demmel and Xiang,
// SIAM J. Matrix Anal. Appl. 32 (2011) 1317-1350).  Each workgroup factors
// its 256 rows x w columns in LDS with partial pivoting and nominates the w
// rows it pivoted on; groups of TS_FAN nominee sets are stacked and factored
// again, up a tree, until one workgroup factors the last stack: its w pivot
// rows, in order, are the panel's pivots and its factors the w x w diagonal
// block L11\U11.  Every workgroup then writes its rows of the permuted panel:
// the diagonal block, or L21 rows = (original row) U11^-1 by substitution.
// Pivot choices differ from row-by-row partial pivoting (the complex128
// path keeps that); the mixed solver's refinement in complex128 takes the
// factors as a preconditioner.  Cross-workgroup data moves only through
// agent-scope relaxed atomics, data drained before a flag: three
// waits per panel (two at most 64 workgroups) instead of one per column.
// ---------------------------------------------------------------------
#define TS_FAN 8
#define TS_SET 128                  // u64 words of one nominee set: row indices [PW], flag,
#define TS_IDX 0                    // references [PW] (row of each nominee's original values in
#define TS_FLAG (PW + 8)            // the copy area: workgroup * 256 + row)
#define TS_REF (PW + 16)
#define TS_TOP (PW * PW)            // root area: final block [PW][PW], (spare) [PW][PW], plan, flag
#define TS_PLAN (2 * PW * PW)
#define TS_NPLAN (2 * PW * PW + 2 * PW)
#define TS_FIN (2 * PW * PW + 2 * PW + 8)
#define TS_UREP 2176                // first replica (workgroup g reads replica g % 8)
#define TS_REP 1056                 // u64 words between replicas of the final block
#define TS_ROOT (2176 + 8 * TS_REP) // root area + 8 replicas of the final block

// the tournament's scratch: sets of all levels [levels + 1][Gmax], the
// copy area [Gmax][256][PW] (each workgroup's rows as loaded), the root area
__host__ __device__ inline long ts_copy_off(int levels, long Gmax) { return (long)(levels + 1) * Gmax * TS_SET; }
__host__ __device__ inline long ts_root_off(int levels, long Gmax) { return ts_copy_off(levels, Gmax) + Gmax * 256 * PW; }

__host__ __device__ inline int ts_levels(long G)
{
  int l = 0;
  for (long c = G; c > 1; c = (c + TS_FAN - 1) / TS_FAN) l++;
  return l;
}

// 1/a for complex64 with hardware reciprocals (about 1 ulp each; the
// tournament panel's pivots), scaled by max(|re|, |im|) against overflow
// and underflow of |a|^2
__device__ inline float2 crecip_fast(float2 a)
{
  const float s = fmaxf(fabsf(a.x), fabsf(a.y)), is = __builtin_amdgcn_rcpf(s);
  const float xs = a.x * is, ys = a.y * is;
  const float d = __builtin_amdgcn_rcpf(fmaf(xs, xs, ys * ys)) * is;
  float2 r;
  r.x = xs * d;
  r.y = -ys * d;
  return r;
}

// r - l c with fused multiply-adds (complex64)
__device__ inline float2 cfms(float2 r, float2 l, float2 c)
{
  float2 o;
  o.x = fmaf(-l.x, c.x, fmaf(l.y, c.y, r.x));
  o.y = fmaf(-l.x, c.y, fmaf(-l.y, c.x, r.y));
  return o;
}

// partial-pivoting LU (largest |re|+|im|, lowest row on ties) of the rows
// [0, nr) the threads of the workgroup hold in registers (thread t: row t,
// r[0..w-1]), rows left in place: spiv[j] = row of pivot j, srank[t] = j
// on pivot rows (else -1); each row ends as its row of the packed factors
// (multipliers left of its pivot step, or its U row).  Returns min(w, nr);
// *zero = first step with a zero pivot or -1.  The pivot search compares
// keys bits(|re|+|im|) + 1 (0: row already a pivot or absent), which order
// as the non-negative magnitudes do.  One barrier per column: the winning
// row of each wave goes through LDS (two buffers: a wave writes buffer
// j & 1 again only after every wave has passed step j + 1's barrier, i.e.
// has read it).
__device__ __attribute__((always_inline)) inline int ts_lu(float2 (&r)[PW], int nr, int w, int *spiv, int *srank,
                                                           unsigned long long (*wkv)[4], float2 (*cand)[4][PW],
                                                           int *zero)
{
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  bool used = t >= nr;
  srank[t] = -1;
  const int np = min(w, nr);
  int z = -1;
#pragma unroll
  for (int j = 0; j < PW; j++) {
    if (j < np) {
      const unsigned key = used ? 0u : __float_as_uint(fabsf(r[j].x) + fabsf(r[j].y)) + 1u;
      const unsigned wm = wave_max_key(key);
      const unsigned long long hit = __ballot(wm != 0 && key == wm);
      const int wl = hit ? __ffsll(hit) - 1 : -1;
      if (lane == wl) {
#pragma unroll
        for (int q = j; q < PW; q++) cand[j & 1][wave][q] = r[q];
        // the wave's key and row in one word: the largest word has the
        // largest key and, among equal keys, the lowest row
        wkv[j & 1][wave] = ((unsigned long long)wm << 32) | (unsigned)(255 - t);
      }
      if (lane == 0 && wl < 0) wkv[j & 1][wave] = 0ull;
      __syncthreads();
      unsigned long long best = wkv[j & 1][0];
#pragma unroll
      for (int q = 1; q < 4; q++) best = max(best, wkv[j & 1][q]);
      const unsigned b0 = (unsigned)(best >> 32);
      const int p = 255 - (int)(unsigned)best;
      const int pw = p >> 6;
      if (t == p) { used = true; srank[t] = j; }
      if (t == 0) spiv[j] = p;
      if (b0 == 1u && z < 0) z = j;
      if (!used) {
        float2 l = r[j];
        if (b0 != 1u) { l = cmul(l, crecip_fast(cand[j & 1][pw][j])); r[j] = l; }
#pragma unroll
        for (int q = j + 1; q < PW; q++) r[q] = cfms(r[q], l, cand[j & 1][pw][q]);
      }
    }
  }
  __syncthreads();
  *zero = z;
  return np;
}

// nominees in the level-l set of workgroup g: min(w, rows of workgroups g
// .. g + TS_FAN^l - 1), by induction over the merges
__device__ inline int ts_count(long g, long span, long m, int w)
{
  const long rows = min(span * 256, m - g * 256);
  return (int)min((long)w, rows);
}

// wave 0 waits until the n <= 64 words f[k * stride] hold seq (bounded),
// then the workgroup synchronizes
__device__ void ts_wait(const unsigned long long *f, long stride, int n, unsigned long long seq, unsigned *err)
{
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    unsigned spins = 0;
    for (;;) {
      bool ok = true;
      if (lane < n) ok = ld_coh(f + lane * stride) == seq;
      if (__ballot(!ok) == 0) break;
      if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) break;
      if (++spins > GBAR_SPIN) { __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); break; }
      __builtin_amdgcn_s_sleep(1);
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  }
  __syncthreads();
}

// panel rows [r0, r0 + m) x columns [r0, r0 + w), w <= PW; grid: one
// workgroup per 256 rows, all co-resident; outputs as k_panel_x (factors in
// place, ipiv, info, the net row permutation in S.plan, the inverse of the
// unit-lower diagonal block in S.linv)
// (at most 168 VGPRs, so that a workgroup fits on SIMDs that run three
// waves of the trailing GEMM instead of waiting for them to retire)
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
k_panel_ts(float2 *A, long lda, long r0, long m, int w, int *ipiv, int *info, PanelScratch S, int Gmax, unsigned seq0,
           BStride bs)
{
  constexpr int NR = 256;
  __shared__ float2 sF[PW][PW + 1];     // final block, row-major
  __shared__ float2 cand[2][NR / 64][PW];
  __shared__ float2 sRd[PW];
  __shared__ unsigned long long wkv[2][NR / 64];
  __shared__ int spiv[PW], srank[NR], ssrc[NR], sfrom[NR];
  __shared__ long sidx[NR];
  // the panel is the critical path and the trailing GEMM shares its CUs:
  // its waves win instruction issue on their SIMDs
  {
    // instance blockIdx.y of a batch
    const long bi = blockIdx.y;
    A += bi * bs.a;
    ipiv += bi * bs.p;
    info = bshift(info, bi * bs.s);
    S = S.shift(bi * bs.s);
  }
  __builtin_amdgcn_s_setprio(3);
  // workgroups 0 .. G - 1 hold the panel's rows; workgroup G only inverts
  // the final block's unit-lower triangle, beside the others' last phase
  const int t = threadIdx.x, G = gridDim.x - 1, g = blockIdx.x;
  const long lo = r0 + (long)g * NR;
  const int nrow = (int)max(0L, min((long)NR, r0 + m - lo));
  const long i = lo + t;
  const unsigned long long seq = seq0;
  unsigned *err = S.bar + 64;
  unsigned long long *ts = S.ts;
  unsigned long long *copy = ts + ts_copy_off(ts_levels(Gmax), Gmax);
  unsigned long long *root = ts + ts_root_off(ts_levels(Gmax), Gmax);
  const int nl = ts_levels(G);
  if (g == G) {
    ts_wait(root + TS_FIN, 0, 1, seq, err);
    // (all of this thread's loads in flight before the first LDS store)
    float2 fv[PW * PW / NR];
#pragma unroll
    for (int u = 0; u < PW * PW / NR; u++) fv[u] = ld_coh((const float2 *)(root + t + u * NR));
#pragma unroll
    for (int u = 0; u < PW * PW / NR; u++) {
      const int e = t + u * NR, rr = e / PW, q = e % PW;
      if (rr < w && q < w) sF[rr][q] = fv[u];
    }
    __syncthreads();
    // the inverse of the unit-lower w x w block, column t by substitution
    if (S.linv && t < PW) {
      float2 x[PW];
#pragma unroll
      for (int rr = 0; rr < PW; rr++) {
        float2 val;
        val.x = (rr == t) ? 1 : 0; val.y = 0;
        if (rr < w && t < w) {
#pragma unroll
          for (int k = 0; k < rr; k++) val = cfms(val, sF[rr][k], x[k]);
        }
        x[rr] = val;
      }
      float2 *li = (float2 *)S.linv + (r0 / PW) * PW * PW + (long)t * PW;
#pragma unroll
      for (int rr = 0; rr < PW; rr++) li[rr] = x[rr];
    }
    return;
  }

  // own rows into registers (A keeps the original values until the last
  // phase, which re-reads them); workgroup 0 also publishes rows r0 .. r0 +
  // w - 1 (those the interchanges displace)
  // (columns from w on hold zeros; their loads repeat column w - 1, so
  // that the loads are not split by per-column branches)
  float2 r[PW];
#pragma unroll
  for (int q = 0; q < PW; q++) r[q] = zero_v<float2>();
  if (t < nrow) {
#pragma unroll
    for (int q = 0; q < PW; q++) {
      const float2 v = A[i + (r0 + min(q, w - 1)) * lda];
      r[q] = q < w ? v : zero_v<float2>();
    }
  }
  // every row's original values to the copy area (read by the merges and,
  // for the rows the interchanges displace from the diagonal block, by the
  // last phase); drained before this workgroup's first flag
  if (t < nrow) {
#pragma unroll
    for (int q = 0; q < PW; q++) st_coh((float2 *)(copy + ((long)g * NR + t) * PW + q), r[q]);
  }
  sidx[t] = lo + t;
  // stage 0: this workgroup's rows; stage l >= 1: workgroups g % TS_FAN^l
  // == 0 stack the nominee sets of g, g + sp, .., g + (TS_FAN - 1) sp (sp =
  // TS_FAN^(l-1)) from stage l - 1.  The last stage runs on workgroup 0.
  int zero = -1;
  long sp = 1;
  for (int l = 0; l <= nl; l++) {
    int nr = nrow;
    const unsigned long long *prev = ts + (long)(l > 0 ? l - 1 : 0) * Gmax * TS_SET;
    if (l > 0) {
      if (g % (sp * TS_FAN)) break;
      const int nch = (int)min((long)TS_FAN, (G - g + sp - 1) / sp);
      ts_wait(prev + (long)g * TS_SET + TS_FLAG, sp * TS_SET, nch, seq, err);
      // the stack: child k's nominees at rows sbase[k] ..
      int sbase[TS_FAN + 1];
      sbase[0] = 0;
#pragma unroll
      for (int k = 0; k < TS_FAN; k++)
        sbase[k + 1] = sbase[k] + (k < nch ? ts_count(g + k * sp, sp, m, w) : 0);
      nr = sbase[TS_FAN];
#pragma unroll
      for (int q = 0; q < PW; q++) { r[q] = zero_v<float2>(); }
      if (t < nr) {
        int k = 0;
#pragma unroll
        for (int q = 1; q < TS_FAN; q++)
          if (t >= sbase[q]) k = q;
        const int rr = t - sbase[k];
        const unsigned long long *cs = prev + (g + k * sp) * TS_SET;
        const int ref = (int)ld_coh(cs + TS_REF + rr);
        const unsigned long long *os = copy + (long)ref * PW;   // the row's original values
#pragma unroll
        for (int q = 0; q < PW; q++) r[q] = ld_coh((const float2 *)(os + q));
        sidx[t] = (long)ld_coh(cs + TS_IDX + rr);
        ssrc[t] = ref;
      }
    }
    const int np = ts_lu(r, nr, w, spiv, srank, wkv, cand, &zero);
    if (l == nl) {
      // workgroup 0: the final block in pivot order
      const int k = t < nr ? srank[t] : -1;
      if (k >= 0) {
#pragma unroll
        for (int q = 0; q < PW; q++) sF[k][q] = r[q];
      }
      break;
    }
    // nominees: original values of the pivot rows
    unsigned long long *set = ts + ((long)l * Gmax + g) * TS_SET;
    const int k = t < nr ? srank[t] : -1;
    if (k >= 0) {
      // references to the original values in the copy area
      st_coh(set + TS_REF + k, (unsigned long long)(l == 0 ? g * NR + t : ssrc[t]));
      st_coh(set + TS_IDX + k, (unsigned long long)sidx[t]);
    }
    (void)np;
    drain();
    __syncthreads();
    if (t == 0) st_coh(set + TS_FLAG, seq);
    if (l > 0) sp *= TS_FAN;
  }

  if (g == 0) {
    // publish the final block, and its upper triangle U11 in eight
    // replicas (read by all workgroups at once); ipiv, the net
    // permutation and info
    __syncthreads();
    for (int e = t; e < PW * PW; e += NR) {
      const int rr = e / PW, q = e % PW;
      if (rr < w && q < w) {
        st_coh((float2 *)(root + rr * PW + q), sF[rr][q]);
        if (q >= rr)
          for (int c = 0; c < 8; c++) st_coh((float2 *)(root + TS_UREP + c * TS_REP + rr * PW + q), sF[rr][q]);
      }
    }
    if (t < 64) {
      // lanes hold (position, original row now there) for every touched
      // position: lanes 0..w-1 the diagonal block's, pivot rows from
      // below appended (lane indices are wave-uniform: lane reads)
      int row = (t < w) ? (int)(r0 + t) : -1, content = row;
      const int Rl = (t < w) ? (int)sidx[spiv[t]] : -1;    // original row of pivot t
      int cnt = w;
      for (int j = 0; j < w; j++) {
        const int R = __builtin_amdgcn_readlane(Rl, j);
        const unsigned long long hit = __ballot(content == R);
        int ip;
        if (hit) ip = __ffsll(hit) - 1;
        else { ip = cnt; if (t == cnt) { row = R; content = R; } cnt++; }
        const int pos = __builtin_amdgcn_readlane(row, ip);
        if (t == 0) ipiv[r0 + j] = pos + 1;
        const int cj = __builtin_amdgcn_readlane(content, j), cp = __builtin_amdgcn_readlane(content, ip);
        if (t == j) content = cp;
        if (t == ip) content = cj;
      }
      if (t < cnt) {
        S.plan[t] = (int)row;
        S.plan[PW * 2 + t] = (int)content;
        st_coh(root + TS_PLAN + t, ((unsigned long long)row << 32) | (unsigned long long)content);
      }
      if (t == 0) {
        S.plan[PW * 4] = cnt;
        st_coh(root + TS_NPLAN, (unsigned long long)cnt);
        if (zero >= 0 && *info == 0) *info = (int)(r0 + zero + 1);
      }
    }
    drain();
    __syncthreads();
    if (t == 0) st_coh(root + TS_FIN, seq);
  }

  // every workgroup: its rows of the permuted panel.  The row's original
  // values (the panel never writes them before this phase, and only this
  // thread writes its row after it) are loaded before the root's flag is
  // awaited; a row displaced from the diagonal block reloads below.
  float2 v[PW];
#pragma unroll
  for (int q = 0; q < PW; q++) { v[q] = zero_v<float2>(); }
  if (t < nrow && i >= r0 + w) {
    // plain loads (opaque address, as above); columns from w on repeat
    // column w - 1 and are never used
    float2 *Ai = A + i + r0 * lda;
    asm volatile("" : "+v"(Ai));
#pragma unroll
    for (int q = 0; q < PW; q++) v[q] = Ai[min(q, w - 1) * lda];
  }
  ts_wait(root + TS_FIN, 0, 1, seq, err);
  // workgroup 0 (the diagonal block's rows) reads the whole final
  // block, the others U11 from replica g % 8; with the plan words, all
  // loads in flight at once
  float2 fv[PW * PW / NR];
  {
    const unsigned long long *fb = g == 0 ? root : root + TS_UREP + (g & 7) * TS_REP;
#pragma unroll
    for (int u = 0; u < PW * PW / NR; u++) fv[u] = ld_coh((const float2 *)(fb + t + u * NR));
  }
  int npl = 0;
  unsigned long long pe = 0;
  if (t < 2 * PW) {
    npl = (int)ld_coh(root + TS_NPLAN);
    pe = ld_coh(root + TS_PLAN + t);
  }
#pragma unroll
  for (int u = 0; u < PW * PW / NR; u++) {
    const int e = t + u * NR, rr = e / PW, q = e % PW;
    if (rr < w && q < w && (g == 0 || q >= rr)) sF[rr][q] = fv[u];
  }
  // displaced rows of this workgroup: sfrom[row - lo] = original row
  sfrom[t] = -1;
  __syncthreads();
  if (t < 2 * PW) {
    const long dst = (long)(pe >> 32);
    if (t < npl && dst >= lo && dst < lo + nrow) sfrom[dst - lo] = (int)(pe & 0xFFFFFFFFull);
  }
  __syncthreads();
  if (t < w) {
    const float2 d = sF[t][t];
    sRd[t] = (d.x != 0 || d.y != 0) ? crecip(d) : d;
  }
  __syncthreads();
  if (t < nrow) {
    if (i < r0 + w) {
#pragma unroll
      for (int q = 0; q < PW; q++)
        if (q < w) A[i + (r0 + q) * lda] = sF[i - r0][q];
    } else {
      const long c = sfrom[t] >= 0 ? sfrom[t] : i;
      if (c == i) {
        // the values loaded above
      } else if (c >= r0 && c < r0 + w) {
        // a row displaced from the diagonal block (no other source exists;
        // anything else is reported as a failed panel)
#pragma unroll
        for (int q = 0; q < PW; q++) v[q] = ld_coh((const float2 *)(copy + (c - r0) * PW + q));
      } else {
        __hip_atomic_store(err, 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      // x U11 = (original row); a zero pivot leaves its column unscaled
#pragma unroll
      for (int q = 0; q < PW; q++) {
        if (q < w) {
          float2 x = v[q];
#pragma unroll
          for (int k = 0; k < q; k++) x = cfms(x, v[k], sF[k][q]);
          const float2 rd = sRd[q];
          if (rd.x != 0 || rd.y != 0) x = cmul(x, rd);
          v[q] = x;
        }
      }
#pragma unroll
      for (int q = 0; q < PW; q++)
        if (q < w) A[i + (r0 + q) * lda] = v[q];
    }
  }
}

// applies nplans consecutive panel row permutations (each: dst <- src on
// at most 2 PW rows, stride 4 PW + 1 ints) to the columns [c0, c1) except
// [s0, s1); one wave per column, four columns in flight per wave, plans in
// order within a column
#define PLAN_LEN (4 * PW + 1)
template <typename T>
__global__ void __launch_bounds__(256)
k_laswp_plans(T *A, long lda, long c0, long c1, long s0, long s1, const int *plans, int nplans, BStride bs)
{
  {
    const long bi = blockIdx.y;   // instance of a batch
    A += bi * bs.a;
    plans = bshift(plans, bi * bs.s);
  }
  const int lane = threadIdx.x & 63;
  const long skip = s1 - s0;
  const long ncol = (c1 - c0) - skip;
  const long nw = (long)gridDim.x * (blockDim.x >> 6);
  for (long c4 = ((long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 4; c4 < ncol; c4 += nw * 4) {
    long cc[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      long c = c0 + c4 + u;
      cc[u] = c < s0 ? c : c + skip;
    }
    for (int pl = 0; pl < nplans; pl++) {
      const int *plan = plans + (long)pl * PLAN_LEN;
      const int cnt = plan[PW * 4];
      const long dst = lane < cnt ? plan[lane] : 0, src = lane < cnt ? plan[PW * 2 + lane] : 0;
      T v[4];
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (c4 + u < ncol && lane < cnt) v[u] = A[src + cc[u] * lda];
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (c4 + u < ncol && lane < cnt) A[dst + cc[u] * lda] = v[u];
      // the next plan's loads see these stores
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    }
  }
}

template <typename T>
static void laswp_plans(T *A, long lda, long c0, long c1, long s0, long s1, const int *plans, int nplans,
                        hipStream_t st, int nbat = 1, BStride bs = BStride())
{
  long ncol = (c1 - c0) - (s1 - s0);
  if (ncol <= 0 || nplans <= 0) return;
  long nwaves = (ncol + 3) / 4;
  unsigned blocks = (unsigned)std::min<long>(4096, (nwaves + 3) / 4);
  hipLaunchKernelGGL(k_laswp_plans<T>, dim3(blocks, (unsigned)nbat), dim3(256), 0, st, A, lda, c0, c1, s0, s1, plans,
                     nplans, bs);
}

// row interchanges rows [k1,k2) (absolute, ipiv 1-based) on columns [c0,c1)
template <typename T>
__global__ void k_laswp(T *A, long lda, long c0, long c1, long k1, long k2, const int *ipiv)
{
  long c = c0 + (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= c1) return;
  for (long s = k1; s < k2; s++) {
    long p = ipiv[s] - 1;
    if (p != s) { T t = A[s + c * lda]; A[s + c * lda] = A[p + c * lda]; A[p + c * lda] = t; }
  }
}

template <typename T>
static void laswp(T *A, long lda, long c0, long c1, long k1, long k2, const int *ipiv, hipStream_t s)
{
  if (c1 <= c0 || k2 <= k1) return;
  hipLaunchKernelGGL(k_laswp<T>, dim3((unsigned)((c1 - c0 + 255) / 256)), dim3(256), 0, s, A, lda, c0, c1, k1, k2, ipiv);
}

// lane k's value in every lane (k wave-uniform)
__device__ inline float readlane_f(float v, int k) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k)); }
__device__ inline double readlane_f(double v, int k)
{
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xFFFFFFFF), k), hi = __builtin_amdgcn_readlane((int)(b >> 32), k);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ inline double readlane_t(double v, int k) { return readlane_f(v, k); }
template <typename T> __device__ inline T readlane_t(T v, int k)
{
  T r;
  r.x = readlane_f(v.x, k);
  r.y = readlane_f(v.y, k);
  return r;
}

__device__ inline double fma_r(double a, double b, double c) { return fma(a, b, c); }
__device__ inline float fma_r(float a, float b, float c) { return fmaf(a, b, c); }
// l x, and r - l x, with fused multiply-adds
__device__ inline double fmul_t(double l, double x) { return l * x; }
__device__ inline double2 fmul_t(double2 l, double2 x)
{
  return make_double2(fma(l.x, x.x, -(l.y * x.y)), fma(l.x, x.y, l.y * x.x));
}
__device__ inline float2 fmul_t(float2 l, float2 x)
{
  return make_float2(fmaf(l.x, x.x, -(l.y * x.y)), fmaf(l.x, x.y, l.y * x.x));
}
__device__ inline double fnma_t(double r, double l, double x) { return fma(-l, x, r); }
__device__ inline double2 fnma_t(double2 r, double2 l, double2 x)
{
  return make_double2(fma(-l.x, x.x, fma(l.y, x.y, r.x)), fma(-l.x, x.y, fma(-l.y, x.x, r.y)));
}
__device__ inline float2 fnma_t(float2 r, float2 l, float2 x)
{
  return make_float2(fmaf(-l.x, x.x, fmaf(l.y, x.y, r.x)), fmaf(-l.x, x.y, fmaf(-l.y, x.x, r.y)));
}

// One panel's interchanges on the columns [c0, c1) outside the panel
// [s0, s1) and, on the columns right of the panel, the substitution with the
// panel block's unit-lower triangle on its w rows from r0, in one launch:
// one wave per column.  Lane e holds plan entry e (dst <- src, all sources
// read before any write); entries 0..w-1 are the rows r0 .. r0 + w - 1, so
// after the interchange lanes 0..w-1 hold the panel rows of the column and
// step q passes x_q by lane reads.  Bound: the chain of w - 1 steps (about
// 1 us); a wave per column leaves the other columns' chains to hide it.  A
// launch of the interchanges and one of a substitution with a column per
// thread (L and B through LDS, one wave per 64 columns) took 8 + 54 us per
// complex128 panel at order 3840; this one takes 7 us.
template <typename T>
__global__ void __launch_bounds__(256)
k_swap_trsm(T *A, long lda, long c0, long c1, long s0, long s1, const int *plan, int w, long r0)
{
  const int lane = threadIdx.x & 63;
  const long ci = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const long nleft = s0 - c0;
  if (ci >= (c1 - c0) - (s1 - s0)) return;
  const long c = ci < nleft ? c0 + ci : s1 + (ci - nleft);
  const int cnt = plan[PW * 4];
  T v = zero_v<T>();
  long dst = -1;
  if (lane < cnt) {
    dst = plan[lane];
    v = A[plan[PW * 2 + lane] + c * lda];
  }
  if (c >= s1) {
    // this lane's row of L11 (a clamped row and column elsewhere), all
    // loads in flight before the substitution
    T lr[PW];
    const T *Lr = A + (r0 + (lane < w ? lane : 0)) + r0 * lda;
#pragma unroll
    for (int k = 0; k < PW; k++) lr[k] = Lr[(k < w ? k : 0) * lda];
#pragma unroll
    for (int k = 0; k < PW; k++) {
      if (k < w) {
        const T x = readlane_t(v, k);
        if (lane > k && lane < w) v = csub(v, cmul(lr[k], x));
      }
    }
  }
  if (lane < cnt) A[dst + c * lda] = v;
}

template <typename T>
static void swap_trsm(T *A, long lda, long c0, long c1, long s0, long s1, const int *plan, int w, long r0, hipStream_t s)
{
  const long ncol = (c1 - c0) - (s1 - s0);
  if (ncol <= 0) return;
  int tok = prof_begin(s, std::is_same<T, float2>::value ? PK_TRSM_C64 : PK_TRSM_C128);
  hipLaunchKernelGGL(k_swap_trsm<T>, dim3((unsigned)((ncol + 3) / 4)), dim3(256), 0, s, A, lda, c0, c1, s0, s1, plan, w,
                     r0);
  prof_end(s, tok, 4.0 * (double)w * (double)w * (double)(c1 - s1));
}

// B[jb x ncol] <- L^-1 B for the unit-lower jb x jb diagonal block at
// A(r0, r0), jb <= 256, in one launch: NC columns per workgroup, thread t
// holds row t of each.  Per 32-row panel the wave that holds its rows
// substitutes by lane reads and passes the 32 values of every column
// through LDS; the rows below subtract L(row, panel) x, each thread's 32
// values of L loaded before the barrier (they do not depend on x) and used
// for all NC columns.  NC = 1 where columns are few (the next block's 256:
// latency counts), 4 where they fill the GPU (a quarter of the reads of L:
// 0.5 MB per workgroup in complex128).  At order 3840: 40 us for the next
// block, 150 us beside it for the rest, where 32-row substitutions and
// updates in 15 launches took 540 us for each.
template <typename T, int NC>
__global__ void __launch_bounds__(256)
k_trsm_sub(const T *A, long lda, long r0, int jb, T *B, long ldb, long ncol)
{
  __shared__ T xs[2][NC][PW];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, row = threadIdx.x;
  const long c0 = (long)blockIdx.x * NC;
  T b[NC];
#pragma unroll
  for (int u = 0; u < NC; u++) {
    b[u] = zero_v<T>();
    if (row < jb && c0 + u < ncol) b[u] = B[row + (c0 + u) * ldb];
  }
  for (int i = 0; i * PW < jb; i++) {
    const int i0 = PW * i, w = min(PW, jb - i0), si = i / 2, l0 = PW * (i & 1);
    const bool below = row >= i0 + w && row < jb;
    const T *Lr = A + (r0 + (row < jb ? row : 0)) + (r0 + i0) * lda;
    T lv[PW];
    if (wv >= si) {
      // (the panel's own rows: their row of the triangle; rows below:
      // their row of L; clamped columns past w are not used)
#pragma unroll
      for (int k = 0; k < PW; k++) lv[k] = Lr[(k < w ? k : 0) * lda];
    }
    if (wv == si) {
      const bool mine = lane >= l0 && lane < l0 + w;
#pragma unroll
      for (int k = 0; k < PW; k++) {
        if (k < w) {
#pragma unroll
          for (int u = 0; u < NC; u++) {
            const T x = readlane_t(b[u], l0 + k);
            if (mine && lane - l0 > k) b[u] = csub(b[u], cmul(lv[k], x));
          }
        }
      }
      if (mine) {
#pragma unroll
        for (int u = 0; u < NC; u++) xs[i & 1][u][lane - l0] = b[u];
      }
    }
    __syncthreads();
    if (below) {
      // (the product summed from zero and subtracted once, as the GEMM
      // update does: subtracting term by term rounds against b 32 times)
      T d[NC];
#pragma unroll
      for (int u = 0; u < NC; u++) d[u] = zero_v<T>();
#pragma unroll
      for (int k = 0; k < PW; k++)
        if (k < w) {
#pragma unroll
          for (int u = 0; u < NC; u++) d[u] = fnma_t(d[u], lv[k], xs[i & 1][u][k]);
        }
#pragma unroll
      for (int u = 0; u < NC; u++) b[u] = cadd(b[u], d[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < NC; u++)
    if (row < jb && c0 + u < ncol) B[row + (c0 + u) * ldb] = b[u];
}

template <typename T>
static void trsm_block(const T *A, long lda, long r0, int nb, T *B, long ldb, long ncol, hipStream_t s)
{
  if (ncol <= 0 || nb <= 0) return;
  int tok = prof_begin(s, std::is_same<T, float2>::value ? PK_TRSM_C64 : PK_TRSM_C128);
  if (ncol <= 512)
    hipLaunchKernelGGL((k_trsm_sub<T, 1>), dim3((unsigned)ncol), dim3(256), 0, s, A, lda, r0, nb, B, ldb, ncol);
  else
    hipLaunchKernelGGL((k_trsm_sub<T, 4>), dim3((unsigned)((ncol + 3) / 4)), dim3(256), 0, s, A, lda, r0, nb, B, ldb, ncol);
  prof_end(s, tok, 4.0 * (double)nb * (double)nb * (double)ncol);
}

// B[w x ncol] <- Linv B for a w x w (w <= PW) inverse of a unit-lower
// panel block, in place: each workgroup stages Linv and a 64-column tile
// of B in LDS; thread (row, column group) forms one row of 8 columns
template <typename T>
__global__ void __launch_bounds__(256)
k_trmm_strip(const T *Linv, int w, T *B, long ldb, long ncol)
{
  __shared__ T Ls[PW][PW + 1];
  __shared__ T Bt[PW][64 + 1];
  const int t = threadIdx.x;
  const long c0 = (long)blockIdx.x * 64;
  const bool full = (w == PW && c0 + 64 <= ncol);
  {
    T lv[4], bv[8];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      int e = t + 256 * u, r = e & (PW - 1), k = e / PW;
      lv[u] = Linv[r + k * PW];
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      int e = t + 256 * u, r = e & (PW - 1), c = e / PW;
      if (full || (r < w && c0 + c < ncol)) bv[u] = B[r + (c0 + c) * ldb];
      else { bv[u] = zero_v<T>(); }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      int e = t + 256 * u, r = e & (PW - 1), k = e / PW;
      Ls[r][k] = lv[u];
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      int e = t + 256 * u, r = e & (PW - 1), c = e / PW;
      Bt[r][c] = bv[u];
    }
  }
  __syncthreads();
  const int r = t & (PW - 1), cg = t >> 5;
  T acc[8];
#pragma unroll
  for (int u = 0; u < 8; u++) { acc[u] = zero_v<T>(); }
#pragma unroll 8
  for (int k = 0; k < PW; k++) {
    const T a = Ls[r][k];
#pragma unroll
    for (int u = 0; u < 8; u++) acc[u] = cadd(acc[u], cmul(a, Bt[k][cg * 8 + u]));
  }
  if (r < w) {
#pragma unroll
    for (int u = 0; u < 8; u++) {
      long c = c0 + cg * 8 + u;
      if (c < ncol) B[r + c * ldb] = acc[u];
    }
  }
}

template <typename T>
static void trmm_strip(const T *Linv, int w, T *B, long ldb, long ncol, hipStream_t s)
{
  if (ncol <= 0 || w <= 0) return;
  int tok = prof_begin(s, std::is_same<T, double2>::value ? PK_TRSM_C128 : PK_TRSM_C64);
  hipLaunchKernelGGL(k_trmm_strip<T>, dim3((unsigned)((ncol + 63) / 64)), dim3(256), 0, s, Linv, w, B, ldb, ncol);
  prof_end(s, tok, 4.0 * (double)w * (double)w * (double)ncol);
}

// One panel's interchanges on the columns [c0, c1) outside the panel
// [s0, s1) and, on the columns right of the panel, the product of the
// panel block's unit-lower inverse with its w rows from r0 (what
// laswp_plans and trmm_strip do, in one launch): one wave per column.
// Lane e holds plan entry e (dst <- src, all sources read before any
// write); entries 0..w-1 are the rows r0 .. r0 + w - 1, so after the
// interchange lanes 0..w-1 hold the panel rows of the column.
template <typename T>
__global__ void __launch_bounds__(256)
k_swap_trmm(T *A, long lda, long c0, long c1, long s0, long s1, const int *plan, const T *Linv, int w, long r0,
            BStride bs)
{
  {
    const long bi = blockIdx.y;   // instance of a batch
    A += bi * bs.a;
    plan = bshift(plan, bi * bs.s);
    Linv = bshift(Linv, bi * bs.s);
  }
  const int lane = threadIdx.x & 63;
  const long ci = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const long nleft = s0 - c0;
  if (ci >= (c1 - c0) - (s1 - s0)) return;
  const long c = ci < nleft ? c0 + ci : s1 + (ci - nleft);
  const int cnt = plan[PW * 4];
  T v = zero_v<T>();
  long dst = -1;
  if (lane < cnt) {
    dst = plan[lane];
    v = A[plan[PW * 2 + lane] + c * lda];
  }
  if (c >= s1) {
    // this lane's row of Linv, all loads in flight before the products
    T lr[PW];
    const int q = lane < w ? lane : 0;
#pragma unroll
    for (int k = 0; k < PW; k++) lr[k] = Linv[q + k * PW];
    T acc = zero_v<T>();
#pragma unroll
    for (int k = 0; k < PW; k++) {
      if (k < w) {
        T vk;
        vk.x = readlane_f(v.x, k);
        vk.y = readlane_f(v.y, k);
        acc = cadd(acc, cmul(lr[k], vk));
      }
    }
    if (lane < w) v = acc;
  }
  if (lane < cnt) A[dst + c * lda] = v;
}

template <typename T>
static void swap_trmm(T *A, long lda, long c0, long c1, long s0, long s1, const int *plan, const T *Linv, int w,
                      long r0, hipStream_t s, int nbat = 1, BStride bs = BStride())
{
  const long ncol = (c1 - c0) - (s1 - s0);
  if (ncol <= 0) return;
  int tok = prof_begin(s, std::is_same<T, double2>::value ? PK_TRSM_C128 : PK_TRSM_C64);
  hipLaunchKernelGGL(k_swap_trmm<T>, dim3((unsigned)((ncol + 3) / 4), (unsigned)nbat), dim3(256), 0, s, A, lda, c0, c1,
                     s0, s1, plan, Linv, w, r0, bs);
  prof_end(s, tok, 4.0 * (double)w * (double)w * (double)(c1 - s1));
}

// trsm_block with the panels' block inverses: per 32-row step a product
// with the step's inverse instead of substitution, then the GEMM update
template <typename T>
static void trsm_block_inv(const T *A, long lda, long r0, int nb, const T *linv, T *B, long ldb, long ncol,
                           hipStream_t s)
{
  for (int i0 = 0; i0 < nb; i0 += PW) {
    int w = std::min(PW, nb - i0);
    trmm_strip(linv + (long)(i0 / PW) * PW * PW, w, B + i0, ldb, ncol, s);
    if (i0 + w < nb)
      gemm_sub((long)(nb - i0 - w), ncol, (long)w, A + (r0 + i0 + w) + (r0 + i0) * lda, lda, B + i0, ldb,
               B + i0 + w, ldb, s);
  }
}

// B[jb x ncol] <- L^-1 B for the unit-lower jb x jb diagonal block of a
// 256-column block (jb <= 256) in one launch, with the panels' inverses:
// per 32-row panel i, B_i <- Linv_i B_i, then the rows below minus
// L(below, panel i) B_i (what trsm_block_inv does in 15 launches for the
// next block's columns).  One workgroup per column: wave v holds rows
// 64 v + lane (jb / 64 waves); the wave that holds panel i's rows forms x_i = Linv_i B_i
// by lane reads and passes it to the others through LDS, so the rows
// below are updated by four waves at once.
template <typename T>
__global__ void __launch_bounds__(256)
k_trsm_blk(const T *A, long lda, long r0, int jb, const T *linv, T *B, long ldb, long ncol, BStride bs)
{
  {
    const long bi = blockIdx.y;   // instance of a batch
    A += bi * bs.a;
    B += bi * bs.a;
    linv = bshift(linv, bi * bs.s);
  }
  __shared__ T xs[2][PW];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const long c = blockIdx.x;
  if (c >= ncol) return;
  const int row = lane + 64 * wv;
  T b = zero_v<T>();
  if (row < jb) b = B[row + c * ldb];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int i0 = PW * i;
    if (i0 < jb) {
      const int w = min(PW, jb - i0), si = i / 2, l0 = PW * (i & 1);
      if (wv == si) {
        // x = Linv_i b_i on the lanes holding the panel's rows
        const T *Li = linv + (long)i * PW * PW;
        const bool mine = lane >= l0 && lane < l0 + w;
        // this lane's row of Linv_i, all loads in flight before the products
        T lr[PW];
        const int q = mine ? lane - l0 : 0;
#pragma unroll
        for (int k = 0; k < PW; k++) lr[k] = Li[q + k * PW];
        T acc = zero_v<T>();
#pragma unroll
        for (int k = 0; k < PW; k++) {
          if (k < w) {
            T bk;
            bk.x = readlane_f(b.x, l0 + k);
            bk.y = readlane_f(b.y, l0 + k);
            acc = cadd(acc, cmul(lr[k], bk));
          }
        }
        if (mine) { b = acc; xs[i & 1][lane - l0] = acc; }
      }
      __syncthreads();
      // rows below the panel: minus L(rows, panel) x
      if (i0 + w < jb && row >= i0 + w && row < jb) {
        const T *Lr = A + (r0 + row) + (r0 + i0) * lda;
        T lv[PW];
#pragma unroll
        for (int k = 0; k < PW; k++) lv[k] = Lr[(k < w ? k : 0) * lda];
        T a = b;
#pragma unroll
        for (int k = 0; k < PW; k++)
          if (k < w) a = csub(a, cmul(lv[k], xs[i & 1][k]));
        b = a;
      }
    }
  }
  if (row < jb) B[row + c * ldb] = b;
}

// The same solve where columns are many (complex64, jb = 16 NT): a wave
// holds 16 columns of all jb rows in the matrix unit's result layout, lane (j,
// q) rows 4 q + r of column j in word r, which is also the layout of a right
// operand whose k-step r takes rows 4 q + r: products feed products without
// leaving the registers, and no wave waits for another.  Bound: the matrix
// units, 32 cycles an instruction (576 for 128 rows).  A wave per 64 rows of
// one column by lane reads (k_trsm_blk, still better for a single
// factorization's next 256 columns, where only 16 waves would run) took 358 us
// a launch in the batch of 32 at N=3840, this one 73.
template <int NT>
__global__ void __launch_bounds__(256)
k_trsm_mm(const float2 *A, long lda, long r0, const float2 *linv, float2 *B, long ldb, long ncol, BStride bs)
{
  typedef CT<float2> M;
  {
    const long bi = blockIdx.y;   // instance of a batch
    A += bi * bs.a;
    B += bi * bs.a;
    linv = bshift(linv, bi * bs.s);
  }
  const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4;
  const long c0 = ((long)blockIdx.x * 4 + (threadIdx.x >> 6)) * 16;
  if (c0 >= ncol) return;
  float2 *Bc = B + 4 * q + min(c0 + j, ncol - 1) * ldb;
  f4 br[NT], bi[NT];
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const float2 v = Bc[16 * t + r];
      br[t][r] = v.x;
      bi[t][r] = v.y;
    }
  // acc += s a x
  auto mac = [&](float2 a, float xr, float xi, f4 &re, f4 &im) __attribute__((always_inline)) {
    re = M::mfma(a.x, xr, re);
    im = M::mfma(a.x, xi, im);
    re = M::mfma(-a.y, xi, re);
    im = M::mfma(a.y, xr, im);
  };
  const float2 *Ap = A + (r0 + j) + (r0 + 4 * q) * lda;
#pragma unroll
  for (int i = 0; i < NT / 2; i++) {
    // X = Linv_i B_i (its upper right 16 x 16 part is zero)
    const float2 *Li = linv + (long)i * PW * PW + j + 4 * q * PW;
    f4 xr[2], xi[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
      xr[u] = M::zero();
      xi[u] = M::zero();
#pragma unroll
      for (int t = 0; t <= u; t++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          mac(Li[16 * u + (16 * t + r) * PW], br[2 * i + t][r], bi[2 * i + t][r], xr[u], xi[u]);
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
      br[2 * i + u] = xr[u];
      bi[2 * i + u] = xi[u];
    }
    // the rows below: B_k -= L_ki X
#pragma unroll
    for (int k = 2 * i + 2; k < NT; k++)
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          float2 a = Ap[16 * k + (PW * i + 16 * t + r) * lda];
          a.x = -a.x;
          a.y = -a.y;
          mac(a, xr[t][r], xi[t][r], br[k], bi[k]);
        }
  }
  if (c0 + j < ncol) {
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) Bc[16 * t + r] = make_float2(br[t][r], bi[t][r]);
  }
}

// whether it takes a solve: its block widths, and 4096 columns, i.e. a wave for
// a quarter of the SIMDs.  The N=15360 mixed solve takes 136.9 ms with this
// line, 138.9 with 16384, 138.5 without the kernel and 143.8 with it for every
// solve; the batch 149.2, 150.0 and 161.0
static bool trsm_mm(const float2 *A, long lda, long r0, int jb, const float2 *linv, float2 *B, long ldb, long ncol,
                    hipStream_t s, int nbat = 1, BStride bs = BStride())
{
  if ((jb != 128 && jb != 256) || ncol * nbat < 4096) return false;
  int tok = prof_begin(s, PK_TRSM_C64);
  const dim3 grid((unsigned)((ncol + 63) / 64), (unsigned)nbat);
  if (jb == 128) hipLaunchKernelGGL(k_trsm_mm<8>, grid, dim3(256), 0, s, A, lda, r0, linv, B, ldb, ncol, bs);
  else hipLaunchKernelGGL(k_trsm_mm<16>, grid, dim3(256), 0, s, A, lda, r0, linv, B, ldb, ncol, bs);
  prof_end(s, tok, 4.0 * (double)jb * (double)jb * (double)ncol * nbat);
  return true;
}

template <typename T>
static void trsm_blk(const T *A, long lda, long r0, int jb, const T *linv, T *B, long ldb, long ncol, hipStream_t s,
                     int nbat = 1, BStride bs = BStride())
{
  if (ncol <= 0 || jb <= 0) return;
  if constexpr (std::is_same<T, float2>::value)
    if (trsm_mm(A, lda, r0, jb, linv, B, ldb, ncol, s, nbat, bs)) return;
  int tok = prof_begin(s, std::is_same<T, double2>::value ? PK_TRSM_C128 : PK_TRSM_C64);
  // one wave per 64 rows of the block: two for a 128-column block
  const unsigned nthr = jb <= 128 ? 128u : 256u;
  hipLaunchKernelGGL(k_trsm_blk<T>, dim3((unsigned)ncol, (unsigned)nbat), dim3(nthr), 0, s, A, lda, r0, jb, linv, B,
                     ldb, ncol, bs);
  prof_end(s, tok, 4.0 * (double)jb * (double)jb * (double)ncol);
}

static Gate g_gates[64];

PanelPass::PanelPass(long workgroups, long slots)
{
  hipGetDevice(&dev_);
  dev_ &= 63;
  share_ = (double)workgroups / (double)std::max(1L, slots);
  if (share_ > 0) g_gates[dev_].enter(share_);
}

PanelPass::~PanelPass()
{
  if (share_ > 0) g_gates[dev_].leave(share_);
}

// second stream of the lookahead (default priority, non-blocking), one per
// device, created on first use.  (Keeping its kernels off a share of the
// CUs with a CU-masked stream was measured 1.7x slower on gfx950.)
static hipStream_t side_stream()
{
  static hipStream_t st[64] = {nullptr};
  int d = 0;
  hipGetDevice(&d);
  if (!st[d & 63]) hipStreamCreateWithFlags(&st[d & 63], hipStreamNonBlocking);
  return st[d & 63];
}

// Right-looking blocked LU with one block of lookahead.  Block b (nb
// columns from K) is factored in 32-column panels on the caller's stream
// (panel, its row interchanges inside the block, small TRSM and GEMM for
// the block's remaining columns); the next block's columns are then
// updated on the same stream, while the rest of the trailing matrix is
// updated on the side stream.  The next block's panels therefore run
// while the big GEMM of this block does.  Row interchanges on columns
// left of a block are applied at the end (nothing reads those rows in
// between), so the side stream's GEMM never sees its L21 rows move.
template <typename T>
int lu_factor(T *A, long n, long lda, int *d_ipiv, int *info, hipStream_t stream, int nb, int fast)
{
  if (n < 0 || lda < std::max(1L, n)) return -1;
  if (n == 0) return 0;
  if (nb > 256) nb = 256;
  if (nb % PW) nb = 256;
  const int ib = PW;
  constexpr int NR = 256;
  const long Gmax = (n + NR - 1) / NR;
  // the mixed solver's complex64 factorization pivots by tournament
  // (SCUFFX_MIXED_PIVOTING=partial, read at every factorization: row by
  // row, as the complex128 path)
  const char *piv_env = getenv("SCUFFX_MIXED_PIVOTING");
  const bool partial_env = piv_env && !strcmp(piv_env, "partial");
  if (IsReal<T>::v) fast = 0;     // the explicit-inverse block rows are a complex64 option
  const bool tourn = fast && std::is_same<T, float2>::value && !partial_env;
  const bool g3m = tourn && mixed_gemm_3m();
  int lrows = 0;
  const void *panel_one = panel_x_kernel<T>(true), *panel_two = panel_x_kernel<T>(false);
  const void *panel_loc = panel_l_kernel<T>(&lrows);
  const void *panel_fn = tourn ? (const void *)k_panel_ts : Gmax <= PX_ONE ? panel_one : panel_two;
  int dev = 0, ncu = 0, perCU = 0;
  hipGetDevice(&dev);
  hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, panel_fn, NR, 0);
  if (!tourn && Gmax > PX_ONE) {           // (its last panels are of the other kernel)
    int one = 0;
    hipOccupancyMaxActiveBlocksPerMultiprocessor(&one, panel_one, NR, 0);
    perCU = std::min(perCU, one);
  }
  // the tournament launches one more workgroup (it inverts the diagonal block)
  const long slots = (long)std::max(1, ncu) * std::max(1, perCU), grid = Gmax + (tourn ? 1 : 0);
  if (slots < grid) return -5;                                        // not co-resident
  if (Gmax > 64 * KEYS_PER_LANE) return -5;                           // more workgroups than polled keys
  const long npanels = (n + PW - 1) / PW;
  // panel scratch, carved from one workspace: time-out word (its own cache
  // lines), info, all panel plans, the panels' inverses, the tournament's or
  // the exact panel's exchange area
  PanelScratch S;
  size_t off_info = 96 * sizeof(unsigned), off_plan = off_info + 64;
  size_t off_li = off_plan + 256 * ((sizeof(int) * PLAN_LEN * npanels + 255) / 256);
  size_t off_ts = off_li + 256 * (((fast ? sizeof(T) * PW * PW * npanels : 0) + 255) / 256);
  const size_t ts_words = tourn ? (size_t)ts_root_off(ts_levels(Gmax), Gmax) + TS_ROOT : 0;
  const size_t x_words = tourn ? 0 : 2 * (size_t)PW * Gmax * PXW<T>::n;
  size_t total = off_ts + sizeof(unsigned long long) * (ts_words + x_words);
  char *wsb = (char *)ws_get(WS_PANEL, total);
  if (!wsb) return -2;
  S.linv = fast ? (void *)(wsb + off_li) : nullptr;
  S.ts = tourn ? (unsigned long long *)(wsb + off_ts) : nullptr;
  S.xch = tourn ? nullptr : (unsigned long long *)(wsb + off_ts);
  S.bar = (unsigned *)wsb;
  int *dinfo = (int *)(wsb + off_info);
  int *plans = (int *)(wsb + off_plan);
  // panels of one workgroup wait for nobody
  PanelPass pass(!tourn && n <= lrows ? 0 : perCU < 2 ? slots : grid, slots);
  // The trailing update runs beside the next panels on a second stream,
  // unless the panel needs more than half of the resident workgroup slots
  // of its kernel: then the GEMM's workgroups, dispatched without pause
  // on the other stream, could keep part of the panel's grid waiting until
  // its bounded waits expire (seen with 480 panel workgroups in 512 slots; 240
  // in 512, complex128 of order 61440, run beside it).  Everything then runs
  // on the caller's stream.
  const bool overlap = 2 * grid <= slots;
  hipStream_t side = overlap ? side_stream() : stream;
  hipEvent_t evP = nullptr, evR = nullptr;
  hipEventCreateWithFlags(&evP, hipEventDisableTiming);
  hipEventCreateWithFlags(&evR, hipEventDisableTiming);
  hipMemsetAsync(dinfo, 0, sizeof(int), stream);
  hipMemsetAsync(S.bar, 0, sizeof(unsigned) * 96, stream);
  // tournament sets and flags start at sequence 0, which no panel uses; the
  // exact panel's slots with the sentinel
  if (tourn) hipMemsetAsync(S.ts, 0, sizeof(unsigned long long) * ts_words, stream);
  else
    hipLaunchKernelGGL(k_fill_u64, dim3((unsigned)((x_words + 255) / 256)), dim3(256), 0, stream, S.xch,
                       (unsigned long long)PX_SENT, (long)x_words);
  // the side stream starts after the caller's stream has the matrix ready
  hipEventRecord(evR, stream);
  hipStreamWaitEvent(side, evR, 0);
  int rc = 0;
  int gmaxi = (int)Gmax;
  for (long K = 0; K < n && rc == 0; K += nb) {
    const long jb = std::min<long>(nb, n - K);
    const long p0 = K / PW;                 // first panel of the block
    for (long j0 = K; j0 < K + jb; j0 += ib) {
      int w = (int)std::min<long>(ib, K + jb - j0);
      long m = n - j0;
      long G = (m + NR - 1) / NR;
      long r0 = j0;
      S.plan = plans + (j0 / PW) * PLAN_LEN;
      // column sequence numbers: fresh for every panel of this factorization
      unsigned seq0 = (unsigned)(j0 + 1);
      BStride one;
      void *args[] = {(void *)&A, (void *)&lda, (void *)&r0, (void *)&m, (void *)&w, (void *)&d_ipiv,
                      (void *)&dinfo, (void *)&S, (void *)&gmaxi, (void *)&seq0, (void *)&one};
      int tok = prof_begin(stream, IsReal<T>::v ? PK_PANEL_F64
                                   : std::is_same<T, double2>::value ? PK_PANEL_C128 : PK_PANEL_C64);
      // neither panel has a grid barrier, only bounded waits for workgroups
      // that become resident as the trailing update's retire: an ordinary
      // launch keeps it on the stream's own hardware queue (a cooperative
      // launch goes through a queue of its own, with a cross-queue handoff
      // before and after every panel)
      hipError_t e = tourn        ? hipLaunchKernel(panel_fn, dim3((unsigned)G + 1), dim3(NR), args, 0, stream)
                     : m <= lrows ? hipLaunchKernel(panel_loc, dim3(1), dim3((unsigned)lrows), args, 0, stream)
                                  : hipLaunchKernel(G <= PX_ONE ? panel_one : panel_two, dim3((unsigned)G), dim3(NR), args, 0,
                                                    stream);
      // algorithmic flops of the m x w panel: per column, one complex
      // reciprocal-multiply per row below it and a complex rank-1 update
      double pflops = 0;
      for (int j = 0; j < w; j++) pflops += (double)(m - j - 1) * (6.0 + 8.0 * (double)(w - j - 1));
      prof_end(stream, tok, pflops);
      if (e != hipSuccess) { rc = -3; break; }
      if (S.linv && !tourn)
        hipLaunchKernelGGL(k_unit_inv<T>, dim3(1), dim3(64), 0, stream, A, lda, r0, w, (T *)S.linv + (j0 / PW) * PW * PW);
      // this panel's interchanges on the block's other columns, with the
      // substitution (fast: the product by the panel block's inverse) on the
      // columns right of it
      long nr = K + jb - (j0 + w);
      if (fast) {
        if constexpr (!IsReal<T>::v)
          swap_trmm(A, lda, K, K + jb, j0, j0 + w, S.plan, (const T *)S.linv + (j0 / PW) * PW * PW, w, j0, stream);
      } else
        swap_trsm(A, lda, K, K + jb, j0, j0 + w, S.plan, w, j0, stream);
      if (nr > 0) {
        gemm_sub(n - j0 - w, nr, (long)w, A + (j0 + w) + j0 * lda, lda, A + j0 + (j0 + w) * lda, lda,
                 A + (j0 + w) + (j0 + w) * lda, lda, stream, 0, 1, 0, g3m);
      }
    }
    if (rc) break;
    const int bplans = (int)((jb + PW - 1) / PW);
    const long c1 = K + jb;                               // first column right of the block
    const long nnext = std::min<long>(nb, n - c1), c2 = c1 + nnext;
    hipEventRecord(evP, stream);
    // the next block's columns (caller's stream), after the side stream
    // has finished the previous block's update of them
    if (nnext > 0) {
      hipStreamWaitEvent(stream, evR, 0);
      laswp_plans(A, lda, c1, c2, 0, 0, plans + p0 * PLAN_LEN, bplans, stream);
      if (fast) {
        if constexpr (!IsReal<T>::v)
          trsm_blk(A, lda, K, (int)jb, (const T *)S.linv + p0 * PW * PW, A + K + c1 * lda, lda, nnext, stream);
      } else
        trsm_block(A, lda, K, (int)jb, A + K + c1 * lda, lda, nnext, stream);
      gemm_sub(n - c1, nnext, jb, A + c1 + K * lda, lda, A + K + c1 * lda, lda, A + c1 + c1 * lda, lda, stream, 0, 1, 0,
               g3m);
    }
    // the rest of the trailing matrix (side stream)
    if (c2 < n) {
      hipStreamWaitEvent(side, evP, 0);
      laswp_plans(A, lda, c2, n, 0, 0, plans + p0 * PLAN_LEN, bplans, side);
      if (fast) {
        if constexpr (!IsReal<T>::v)
          {
            const T *li = (const T *)S.linv + p0 * PW * PW;
            bool done = false;
            if constexpr (std::is_same<T, float2>::value)
              done = trsm_mm(A, lda, K, (int)jb, li, A + K + c2 * lda, lda, n - c2, side);
            if (!done) trsm_block_inv(A, lda, K, (int)jb, li, A + K + c2 * lda, lda, n - c2, side);
          }
      } else
        trsm_block(A, lda, K, (int)jb, A + K + c2 * lda, lda, n - c2, side);
      // beside tournament panels: at most three trailing-GEMM workgroups
      // per CU (44 KB of LDS each), so that a panel workgroup (168 VGPRs
      // per wave, 12 KB) finds room on every CU instead of waiting for
      // GEMM workgroups to retire
      const unsigned pad = tourn ? 44u * 1024u - (unsigned)(4 * GBK * (GBM + 4) * sizeof(float)) : 0u;
      gemm_sub(n - c1, n - c2, jb, A + c1 + K * lda, lda, A + K + c2 * lda, lda, A + c1 + c2 * lda, lda, side, pad, 1,
               0, g3m);
      hipEventRecord(evR, side);
    }
    // this block's interchanges on the columns left of it.  Nothing reads
    // those rows again during the factorization (the trailing updates read
    // only the current block's L21), so with two streams they run on the
    // side stream behind this block's update, in block order, instead of
    // all at the end of the caller's stream
    if (side != stream && K > 0) {
      if (c2 >= n) hipStreamWaitEvent(side, evP, 0);   // no trailing update queued for this block
      laswp_plans(A, lda, 0, K, 0, 0, plans + p0 * PLAN_LEN, bplans, side);
    }
  }
  // join the side stream (one stream: the deferred interchanges on the
  // columns left of each block, now)
  hipEventRecord(evR, side);
  hipStreamWaitEvent(stream, evR, 0);
  if (rc == 0 && side == stream)
    for (long K = nb; K < n; K += nb) {
      const long jb = std::min<long>(nb, n - K);
      laswp_plans(A, lda, 0, K, 0, 0, plans + (K / PW) * PLAN_LEN, (int)((jb + PW - 1) / PW), stream);
    }
  unsigned tmo = 0;
  hipMemcpyAsync(info, dinfo, sizeof(int), hipMemcpyDeviceToHost, stream);
  hipMemcpyAsync(&tmo, S.bar + 64, sizeof(unsigned), hipMemcpyDeviceToHost, stream);
  hipStreamSynchronize(stream);
  hipStreamSynchronize(side);
  hipEventDestroy(evP);
  hipEventDestroy(evR);
  if (prof_enabled()) prof_collect();
  if (tmo && rc == 0) rc = tmo == 1 ? -6 : -3;
  if (rc == 0 && hipGetLastError() != hipSuccess) rc = -3;
  return rc;
}

// ---------------------------------------------------------------------
// triangular solves, in one launch per triangle: one right-hand side down
// the 64-row blocks (k_trsv_chain),
// several right-hand sides and transposed systems as a chain of block
// products on the matrix cores with substitution (k_trsm_chain).
// ---------------------------------------------------------------------
template <typename T>
__global__ void k_laswp_rev(T *B, long ldb, long n, long nrhs, const int *ipiv)
{
  long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nrhs) return;
  for (long s = n - 1; s >= 0; s--) {
    long p = ipiv[s] - 1;
    if (p != s) { T t = B[s + c * ldb]; B[s + c * ldb] = B[p + c * ldb]; B[p + c * ldb] = t; }
  }
}

// The row interchanges of ipiv (LAPACK order, each row s swapped with a
// row p >= s) composed into one permutation: perm[s] is the row whose
// content ends up in row s.  One wave walks the interchanges in order on
// an LDS copy of the permutation; a ballot over 64 pivots at a time skips
// the rows that stay (most of them for a BEM matrix).  The right-hand
// sides are then gathered (forward) or scattered (reverse) in parallel,
// instead of one thread per column walking all n interchanges in memory.
#define PERM_LDS_MAX 20480
__global__ void __launch_bounds__(64) k_perm_build(const int *ipiv, long n, int *perm, long sp, long sperm)
{
  ipiv += (long)blockIdx.x * sp;   // instance blockIdx.x of a batch
  perm += (long)blockIdx.x * sperm;
  __shared__ int P[PERM_LDS_MAX], V[PERM_LDS_MAX];
  const int lane = threadIdx.x;
  for (long i = lane; i < n; i += 64) { P[i] = (int)i; V[i] = ipiv[i] - 1; }
  __syncthreads();
  for (long s0 = 0; s0 < n; s0 += 64) {
    const long s = s0 + lane;
    const int p = s < n ? V[s] : (int)s;
    unsigned long long m = __ballot(s < n && p != s && p > s && p < n);   // interchanges stay below row n
    while (m) {
      const int b = __ffsll(m) - 1;
      m &= m - 1;
      const int pp = __shfl(p, b);
      // one lane swaps; the wave's LDS operations complete in order
      if (lane == 0) { const int a = P[s0 + b]; P[s0 + b] = P[pp]; P[pp] = a; }
    }
  }
  __syncthreads();
  for (long i = lane; i < n; i += 64) perm[i] = P[i];
}

// out[s] = in[perm[s]]
template <typename T>
__global__ void __launch_bounds__(256) k_perm_apply(const T *in, T *out, const int *perm, long n, long sin, long sout,
                                                    long sperm)
{
  {
    const long z = blockIdx.z;   // instance of a batch
    in += z * sin; out += z * sout; perm += z * sperm;
  }
  const long s = (long)blockIdx.x * 256 + threadIdx.x;
  if (s < n) out[s] = in[perm[s]];
}

// applies the interchanges of ipiv to b (as laswp with increment 1); tmp
// holds n elements; perm_ready: perm_buf already holds the composed
// permutation of ipiv
template <typename T>
static void apply_row_perm(T *b, long n, const int *ipiv, T *tmp, hipStream_t s, int *perm_buf, bool perm_ready)
{
  int *perm = n > PERM_LDS_MAX ? nullptr : perm_buf ? perm_buf : (int *)ws_get(WS_PERM, sizeof(int) * n);
  if (!perm) {
    // beyond the LDS copy: the interchanges one after another
    laswp(b, n, 0, 1, 0, n, ipiv, s);
    return;
  }
  if (!(perm_ready && perm == perm_buf)) hipLaunchKernelGGL(k_perm_build, dim3(1), dim3(64), 0, s, ipiv, n, perm, 0L, 0L);
  hipLaunchKernelGGL(k_perm_apply<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, b, tmp, perm, n, 0L, 0L, 0L);
  hipMemcpyAsync(b, tmp, sizeof(T) * n, hipMemcpyDeviceToDevice, s);
}

// Inverses of the diagonal 64x64 blocks of L (unit lower, blockIdx.y = 0)
// and U (blockIdx.y = 1), identity past row n: every block step of a
// refined complex64 solve is then a product.  Columns of the inverse by
// substitution, so that L X and U X, not X L and X U, are the identity to
// rounding (the transpose of U^T's inverse converged ten times slower in the
// refinement).  One workgroup a block, a wave for 16 columns of the inverse, a
// lane for a row; a step passes one row's values of every column by lane
// reads.  Bound: issue of the lane reads and updates.  A column per thread of
// one wave, its sums from LDS, took 100 us for each triangle, this 59 us for
// both (order 2501, in complex128, which substitutes by now; the first 16 (q + 1)
// columns only in steps 16 q ..: 78 us with every column in every step).
#define TB 64
template <typename T>
__global__ void __launch_bounds__(256)
k_tri_inv(const T *LU, long lda, long n, T *invL, T *invU, long sa, long sinv)
{
  __shared__ T D[TB][TB + 1];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const bool up = blockIdx.y != 0;
  const long z = blockIdx.z, kb = (long)blockIdx.x * TB;   // instance z of a batch
  const int bs = (int)std::min<long>(TB, n - kb);
  LU += z * sa + kb + kb * lda;
  // the rows and columns of U in reverse: a lower triangle as well
  {
    T v[16];
#pragma unroll
    for (int u = 0; u < 16; u++)      // (past the edge a valid element, replaced by the identity)
      v[u] = LU[min(lane, bs - 1) + min(wave + 4 * u, bs - 1) * lda];
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int c = wave + 4 * u;
      if (lane >= bs || c >= bs) v[u] = lane == c ? unit_v<T>() : zero_v<T>();
      if (up) D[TB - 1 - lane][TB - 1 - c] = v[u]; else D[lane][c] = v[u];
    }
  }
  __syncthreads();
  const T rd = up ? crecip(D[lane][lane]) : unit_v<T>();
  T y[16];
#pragma unroll
  for (int u = 0; u < 16; u++) y[u] = lane == wave + 4 * u ? unit_v<T>() : zero_v<T>();
  // steps 16 q .. 16 q + 15 concern the first 16 (q + 1) columns
  auto steps = [&](auto qc) __attribute__((always_inline)) {
    constexpr int q = decltype(qc)::value;
#pragma unroll 2
    for (int k = 16 * q; k < 16 * q + 16; k++) {
      const T d = D[lane][k], rk = readlane_t(rd, k);
#pragma unroll
      for (int u = 0; u < 4 * q + 4; u++) {
        T x = readlane_t(y[u], k);
        if (up) {
          x = cmul(x, rk);
          if (lane == k) y[u] = x;
        }
        if (lane > k) y[u] = fnma_t(y[u], d, x);
      }
    }
  };
  steps(std::integral_constant<int, 0>{});
  steps(std::integral_constant<int, 1>{});
  steps(std::integral_constant<int, 2>{});
  steps(std::integral_constant<int, 3>{});
  T *o = (up ? invU : invL) + z * sinv + (long)blockIdx.x * TB * TB;
  const int r = up ? TB - 1 - lane : lane;
#pragma unroll
  for (int u = 0; u < 16; u++) o[r + (up ? TB - 1 - wave - 4 * u : wave + 4 * u) * TB] = y[u];
}

template <typename T>
static void tri_inv(const T *LU, long lda, long n, T *invL, T *invU, hipStream_t s, int nbat = 1, long sa = 0,
                    long sinv = 0)
{
  const long nblk = (n + TB - 1) / TB;
  hipLaunchKernelGGL(k_tri_inv<T>, dim3((unsigned)nblk, 2, (unsigned)nbat), dim3(256), 0, s, LU, lda, n, invL, invU, sa,
                     sinv);
}

// one block step: x_b = inv(D_b) r_b (every workgroup, from L2), the
// solution written to Xout by workgroup 0, and the rows outside the block
// updated with x_b (LOWER: rows below, else rows above)
template <typename T, bool LOWER>
__global__ void __launch_bounds__(256)
k_trsv_inv(const T *LU, long lda, long n, long kb, int bs, const T *invb, T *Bin, T *Xout, long sa, long sinv, long sb,
           long sx)
{
  {
    const long z = blockIdx.z;   // instance of a batch
    LU += z * sa; invb += z * sinv; Bin += z * sb; Xout += z * sx;
  }
  __shared__ T rs[TB], xs[TB];
  const int t = threadIdx.x;
  T *b = Bin, *xo = Xout;
  if (t < TB) {
    if (t < bs) rs[t] = b[kb + t]; else { rs[t] = zero_v<T>(); }
  }
  __syncthreads();
  if (t < TB) {
    T acc = zero_v<T>();
#pragma unroll
    for (int k0 = 0; k0 < TB; k0 += 16) {
      T a[16];
#pragma unroll
      for (int u = 0; u < 16; u++) a[u] = invb[t + (k0 + u) * TB];
#pragma unroll
      for (int u = 0; u < 16; u++) {
        T v = rs[k0 + u];
        mac(acc, a[u], v);
      }
    }
    xs[t] = acc;
  }
  __syncthreads();
  if (blockIdx.x == 0 && t < bs) xo[kb + t] = xs[t];
  const long row = LOWER ? kb + bs + (long)blockIdx.x * 256 + t : (long)blockIdx.x * 256 + t;
  const long rend = LOWER ? n : kb;
  if (row < rend) {
    T acc = zero_v<T>();
    const T *Lr = LU + row + kb * lda;
    T bo = b[row];
    if (bs == TB) {
      // full block: 16 independent loads in flight per batch
#pragma unroll
      for (int i0 = 0; i0 < TB; i0 += 16) {
        T a[16];
#pragma unroll
        for (int u = 0; u < 16; u++) a[u] = Lr[(long)(i0 + u) * lda];
#pragma unroll
        for (int u = 0; u < 16; u++) {
          T v = xs[i0 + u];
          mac(acc, a[u], v);
        }
      }
    } else {
      for (int i = 0; i < bs; i++) {
        T a = Lr[(long)i * lda], v = xs[i];
        mac(acc, a, v);
      }
    }
    b[row] = csub(bo, acc);
  }
}

// One right-hand side, all block steps in one launch.  A workgroup owns the
// 64 rows of a block, which it takes in solve order from a ticket, so that it
// only ever waits for workgroups that have started (no residency is needed, and
// an ordinary launch stays on the stream's own queue): it subtracts the off-diagonal
// blocks' products with every earlier solution block as that block is
// published (forward: blocks k < g of L; backward: k > g of U), then
// solves with the diagonal block and publishes its own 64 values.  The
// output starts filled with a sentinel (a NaN bit pattern in every 64-bit
// word that no solve produces), and every entry is written once, by an
// agent-scope relaxed atomic store: a reader that sees a word other than
// the sentinel sees its final value, so no flag or store drain is needed
// (one memory round trip per block step).  Every wait is bounded (error
// word, as in the panel).  Thread t handles row t % 64 and the 16 columns
// 16 (t / 64) .. of a block; the four partial sums meet in LDS.  The next
// block's 16 values per thread are loaded before the wait.  The forward
// solve, which reads its right-hand side b once per row, leaves the
// sentinel in b (mark), where the backward solve writes its output.
// SUB: the diagonal block by substitution, one wave, x_k by lane reads.  Not
// SUB: by its explicit inverse, for callers that refine the solution in higher
// precision.  Products with the inverse of a badly scaled block (dielectric
// surfaces near the low-frequency limit, whose electric and magnetic rows differ by
// 1e6) lose digits that no residual of their own brings back further down:
// eps = 10 sphere of 960 functions at frequency 0.001i in complex128: forward
// error 2e-4 with the inverses, 9e-9 by substitution.
#define SCUFFX_CHAIN_SENT 0x7FF4DEADBEEF0003ULL

// a loaded value is final once none of its 64-bit words is the sentinel
template <typename T>
__device__ inline bool chain_val_set(const T &v)
{
  unsigned long long w[sizeof(T) / 8];
  __builtin_memcpy(w, &v, sizeof(T));
  bool set = true;
#pragma unroll
  for (int j = 0; j < (int)(sizeof(T) / 8); j++) set = set && (w[j] != SCUFFX_CHAIN_SENT);
  return set;
}

template <typename T>
__device__ inline void chain_mark(T *p)
{
  unsigned long long *w = (unsigned long long *)p;
#pragma unroll
  for (int j = 0; j < (int)(sizeof(T) / 8); j++) st_coh(w + j, SCUFFX_CHAIN_SENT);
}

template <typename T>
__global__ void k_chain_fill(T *x, long n)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    unsigned long long *w = (unsigned long long *)(x + i);
#pragma unroll
    for (int j = 0; j < (int)(sizeof(T) / 8); j++) w[j] = SCUFFX_CHAIN_SENT;
  }
}

template <typename T, bool LOWER, bool SUB>
__global__ void __launch_bounds__(256)
k_trsv_chain(const T *LU, long lda, long n, const T *inv, T *bin, T *xout, int mark, unsigned *err, unsigned *ticket)
{
  __shared__ unsigned s_tk;
  __shared__ T part[4][TB];
  __shared__ T bx[TB];
  __shared__ T sD[SUB ? TB : 1][TB];       // [column][row] of the diagonal block
  const int t = threadIdx.x, r = t & (TB - 1), q = t >> 6;
  const long nblk = (n + TB - 1) / TB;
  if (t == 0) s_tk = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const long nk = s_tk;                      // blocks before this one in solve order
  if (nk >= nblk) return;
  const long g = LOWER ? nk : nblk - 1 - nk;
  const long row = g * TB + r;
  const int bs = (int)std::min<long>(TB, n - g * TB);
  T b = zero_v<T>();
  if (q == 0 && r < bs) {
    b = bin[row];
    if (mark) chain_mark(bin + row);
  }
  auto blk = [&](long i) { return LOWER ? i : nblk - 1 - i; };
  auto load = [&](long k, T (&a)[16]) {
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const long col = k * TB + q * 16 + u;
      if (r < bs && col < n) a[u] = LU[row + col * lda];
      else { a[u] = zero_v<T>(); }
    }
  };
  // the inverse diagonal block, in the same registers once no block is left
  const T *ib = inv + g * TB * TB;
  auto load_inv = [&](T (&m)[16]) {
#pragma unroll
    for (int u = 0; u < 16; u++) m[u] = ib[r + (long)(q * 16 + u) * TB];
  };
  // SUB: the diagonal block into LDS and its diagonal's reciprocals, ahead of
  // the waits (zero past row n, where nothing uses the results)
  T rd = unit_v<T>();
  if constexpr (SUB) {
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int c = q * 16 + u;
      const T v = LU[g * TB + min(r, bs - 1) + (g * TB + min(c, bs - 1)) * lda];
      sD[c][r] = r < bs && c < bs ? v : zero_v<T>();
    }
    if (!LOWER && q == 0 && r < bs) rd = crecip(LU[row + row * lda]);
    __syncthreads();
  }
  T a[16];
  if (nk > 0) load(blk(0), a);
  else if (!SUB) load_inv(a);
  for (long i = 0; i < nk; i++) {
    const long k = blk(i);
    // this thread's 16 values of block k, once published (bounded)
    // (all 16 loads in flight at once; the whole set again while any
    // still holds the sentinel)
    T x[16];
    unsigned spins = 0;
    for (;;) {
      bool ready = true;
#pragma unroll
      for (int u = 0; u < 16; u++) {
        const long col = k * TB + q * 16 + u;
        x[u] = col < n ? ld_coh(xout + col) : zero_v<T>();
      }
#pragma unroll
      for (int u = 0; u < 16; u++) ready = ready && chain_val_set(x[u]);
      if (ready) break;
      if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) break;
      if (++spins > GBAR_SPIN) { __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); break; }
      __builtin_amdgcn_s_sleep(1);
    }
    T acc = zero_v<T>();
#pragma unroll
    for (int u = 0; u < 16; u++) {
      mac(acc, a[u], x[u]);
    }
    if (i + 1 < nk) load(blk(i + 1), a);
    else if (!SUB) load_inv(a);
    part[q][r] = acc;
    __syncthreads();
    if (q == 0) {
      T s4 = part[0][r];
      s4 = cadd(s4, part[1][r]); s4 = cadd(s4, part[2][r]); s4 = cadd(s4, part[3][r]);
      b = csub(b, s4);
    }
    __syncthreads();
  }
  if constexpr (SUB) {
    // own block: a lane a row, its products summed by themselves
    if (q != 0) return;
    T z = zero_v<T>();
#pragma unroll
    for (int j = 0; j < TB; j++) {
      const int k = LOWER ? j : TB - 1 - j;
      T v = cadd(b, z);
      if (!LOWER) v = cmul(v, rd);
      v = readlane_t(v, k);
      if (LOWER ? r > k : r < k) z = fnma_t(z, sD[k][r], v);
    }
    T xg = cadd(b, z);
    if (!LOWER) xg = cmul(xg, rd);
    if (r < bs) st_coh(xout + row, xg);
    return;
  }
  // own block: x_g = inv(D_g) b_g
  if (q == 0) bx[r] = b;
  __syncthreads();
  T acc = zero_v<T>();
#pragma unroll
  for (int u = 0; u < 16; u++) {
    const T m = a[u], v = bx[q * 16 + u];
    mac(acc, m, v);
  }
  part[q][r] = acc;
  __syncthreads();
  if (q == 0 && r < bs) {
    T xg = part[0][r];
    xg = cadd(xg, part[1][r]); xg = cadd(xg, part[2][r]); xg = cadd(xg, part[3][r]);
    st_coh(xout + row, xg);
  }
}

// Several right-hand sides, or transposed systems, in one launch per
// triangle: workgroup (block g of 64 rows, tile of 16 columns) subtracts the
// products with every earlier solution block on the matrix cores as that
// block is published, then substitutes through its diagonal block and
// publishes its own 64 x 16 values.  FWD: blocks in ascending order.  The
// matrix is L (FWD) or U, TRANS: U^T (FWD) or L^T, whose blocks are read as
// they lie (a lane then owns a row segment of 16 words).  Published values
// lie packed, [tile][row][16], filled with the sentinel first, as in
// k_trsv_chain: one memory round trip per block step, no barrier until the
// last (each wave holds 16 rows and polls the words it multiplies).
// Workgroups take their place in solve order from a ticket, so a wait is
// only ever for a workgroup that has started: any grid makes progress.
// Every wait is bounded all the same.
// The diagonal block is substituted in four sub-blocks of 16 rows: a lane
// holds one row of one column (each wave four columns) and a step passes x_k
// to the 16 lanes of its column by a row broadcast; the waves whose rows lie
// further then subtract the sub-block's products on the matrix cores.  (A
// lane for each of the 64 rows, x_k by lane reads, took 10 us a block in
// complex128; products with the explicit inverse 2 us, but where the block is
// badly scaled, eps = 10 spheres at imaginary frequency 0.001, they lose every
// digit.)  The entries of the first sub-block wait in LDS.
// Rounding: a block's 64 products are summed two k-steps at a time, a
// sub-block's own by themselves, and subtracted once, not term by term from the
// right-hand side.  Transposed systems (EXACT) also keep what the
// subtractions lose (two-sums, added back before each use) and multiply by
// reciprocals in two words.  Their error then is that of a dot product of 256
// partial sums and one division a row: 0.81 to 0.97 of it over orders 100 to 1500
// and the three types, where one sum over four blocks, products subtracted term by term
// and rounded reciprocals had 1.7 to 3.8 times as much.  Untransposed it is 0.4 to
// 0.9 of what products with the blocks' inverses had (2 to 16 columns; up to
// 1.7 before), inverses of order 64 and up at most that of substitution in
// 256-row blocks (1.02; up to 1.28 before).  One transposed system, order 3840,
// complex128: 1.69 -> 1.96 ms; two untransposed columns 1.43 -> 1.46 ms.
// bin: column-major right-hand sides, row r taken from pin[r] if given, or
// null: packed in win.  bout: column-major results or null, row r to pout[r]
// if given.  cj: 1 conjugates the right-hand sides, 2 the results in bout.
// Bound: the chain of block steps up to a few hundred columns (a round trip,
// 16 complex 16x16x4 products and 64 substitution steps per wave), the
// matrix units past that.  N=3840 complex128: 12 us a step (16 transposed);
// 181 columns 2.1 ms, where substitution in 256-row blocks by one workgroup a
// column and GEMM updates took 6.0; one transposed system 2.0 ms, where a single
// workgroup with a reduction per row took 24.
template <typename T> struct ChainArgs {
  const T *A; long lda; long n;
  const T *bin; long ldb; const int *pin; const T *win;
  T *w; T *bout; long ldo; const int *pout;
  long nrhs; int cj; unsigned *err, *ticket;
};

// acc += a x for one k-step of the matrix instruction
template <typename T>
__device__ inline void chain_mac(T a, T x, typename CT<T>::V4 &re, typename CT<T>::V4 &im)
{
  if constexpr (IsReal<T>::v) re = CT<T>::mfma(a, x, re);
  else {
    re = CT<T>::mfma(a.x, x.x, re);
    im = CT<T>::mfma(a.x, x.y, im);
    re = CT<T>::mfma(-a.y, x.y, re);
    im = CT<T>::mfma(a.y, x.x, im);
  }
}
// h - v, what its rounding lost added to l (Knuth's two-sum)
template <typename R> __device__ inline void two_diff(R &h, R &l, R v)
{
  const R z = h - v, w = z - h;
  l += (h - (z - w)) - (v + w);
  h = z;
}
__device__ inline void sub2(double &h, double &l, double v) { two_diff(h, l, v); }
template <typename T> __device__ inline void sub2(T &h, T &l, T v)
{
  two_diff(h.x, l.x, v.x);
  two_diff(h.y, l.y, v.y);
}
// a reciprocal rh of d and what it lacks: 1 / d = rh + rl to twice the
// precision (0 where the reciprocal is not finite)
__device__ inline double recip_lo(double d, double rh)
{
  const double rl = fma(-d, rh, 1.0) * rh;
  return isfinite(rl) ? rl : 0.0;
}
template <typename T> __device__ inline T recip_lo(T d, T rh)
{
  const T rl = cmul(fnma_t(unit_v<T>(), d, rh), rh);
  return isfinite(rl.x) && isfinite(rl.y) ? rl : zero_v<T>();
}
// v (rh + rl)
__device__ inline double mul2(double v, double rh, double rl) { return fma(v, rh, v * rl); }
template <typename T> __device__ inline T mul2(T v, T rh, T rl)
{
  const T t = fmul_t(v, rl);
  T q;
  q.x = fma_r(v.x, rh.x, fma_r(-v.y, rh.y, t.x));
  q.y = fma_r(v.x, rh.y, fma_r(v.y, rh.x, t.y));
  return q;
}
// v of lane k of this lane's row of 16
template <int K> __device__ inline float row_bcast(float v)
{
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + K, 0xF, 0xF, false));
}
template <int K> __device__ inline double row_bcast(double v)
{
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xFFFFFFFF), 0x150 + K, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x150 + K, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <int K, typename T> __device__ inline T row_bcast(T v)
{
  T r;
  r.x = row_bcast<K>(v.x);
  r.y = row_bcast<K>(v.y);
  return r;
}
template <typename T> __device__ inline T chain_elem(typename CT<T>::V4 re, typename CT<T>::V4 im, int r)
{
  if constexpr (IsReal<T>::v) return re[r];
  else { T v; v.x = re[r]; v.y = im[r]; return v; }
}

template <typename T, bool FWD, bool TRANS>
__global__ void __launch_bounds__(256, 2) k_trsm_chain(ChainArgs<T> p)
{
  typedef typename CT<T>::V4 V4;
  constexpr int NC = 16;
  constexpr bool UNIT = FWD != TRANS, EXACT = TRANS;
  __shared__ T sb[TB][NC + 1];                     // right-hand sides, then solutions
  __shared__ T sl[EXACT ? TB : 1][NC + 1];         // what their roundings lost
  __shared__ T sm[16][17], sr[TB];                 // first diagonal sub-block; the diagonal's reciprocals
  __shared__ T srl[EXACT ? TB : 1];                // what the reciprocals lack
  __shared__ unsigned s_tk;
  const int t = threadIdx.x, lane = t & 63, i = lane & 15, kq = lane >> 4, w0 = (t >> 6) * 16;
  if (t == 0) s_tk = __hip_atomic_fetch_add(p.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const long n = p.n, lda = p.lda, nblk = (n + TB - 1) / TB, ntile = (p.nrhs + NC - 1) / NC;
  const long nk = s_tk / ntile, tile = s_tk % ntile;      // blocks before this one in solve order
  if (nk >= nblk) return;
  auto blk = [&](long q) { return FWD ? q : nblk - 1 - q; };
  const long g = blk(nk);
  const int bs = (int)std::min<long>(TB, n - g * TB);
  T *wt = p.w + tile * nblk * TB * NC;
  // this lane's 16 values of block (g, k): matrix row 16 kq + s of the
  // k-step, row w0 + i of the block
  auto load = [&](long k, T (&a)[16]) {
    const long row = g * TB + w0 + i, col = k * TB + 16 * kq;
    if (std::max(g, k) * TB + TB <= n) {
      const T *q = TRANS ? p.A + col + row * lda : p.A + row + col * lda;
#pragma unroll
      for (int s = 0; s < 16; s++) a[s] = TRANS ? q[s] : q[s * lda];
    } else {
      const long rc = min(row, n - 1);
#pragma unroll
      for (int s = 0; s < 16; s++) {
        const long cc = min(col + s, n - 1);
        a[s] = TRANS ? p.A[cc + rc * lda] : p.A[rc + cc * lda];
        if (row >= n || col + s >= n) a[s] = zero_v<T>();
      }
    }
  };
  // sub-block u in solve order covers the rows from sub(u); its diagonal part:
  // this lane's row i (clamped past the edge, where nothing uses the values),
  // columns in solve order; the part left of wave row w0 for its k-steps
  const T *Ad = p.A + g * TB * (lda + 1);
  auto sub = [&](int u) { return 16 * (FWD ? u : 3 - u); };
  auto at = [&](int r, int k) { return TRANS ? Ad[min(k, bs - 1) + min(r, bs - 1) * lda] : Ad[min(r, bs - 1) + min(k, bs - 1) * lda]; };
  auto dload = [&](int u, T (&d)[16]) {
#pragma unroll
    for (int s = 0; s < 16; s++) d[s] = at(sub(u) + i, sub(u) + (FWD ? s : 15 - s));
  };
  auto fload = [&](int u, T (&f)[12]) {       // f[4 u ..]
#pragma unroll
    for (int s = 0; s < 4; s++) f[4 * u + s] = at(w0 + i, sub(u) + 4 * s + kq);
  };
  // the first sub-block, the diagonal's reciprocals and the right-hand side,
  // loaded ahead
  {
    const int s = t >> 4;
    sm[s][i] = at(sub(0) + i, sub(0) + (FWD ? s : 15 - s));
    if (!UNIT && t < TB) {
      const T d = at(t, t), rd = t < bs ? crecip(d) : unit_v<T>();
      sr[t] = rd;
      if (EXACT) srl[EXACT ? t : 0] = t < bs ? recip_lo(d, rd) : zero_v<T>();
    }
  }
  // b: the right-hand side less the products so far; bl (EXACT): the sum of
  // what its roundings lost
  T b[4], bl[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int br = w0 + CT<T>::row(lane, r);
    const long row = g * TB + br, c = tile * NC + i;
    b[r] = bl[r] = zero_v<T>();
    if (p.bin) {
      if (br < bs && c < p.nrhs) b[r] = conj_if(p.bin[(p.pin ? p.pin[row] : row) + c * p.ldb], p.cj & 1);
    } else if (br < bs) b[r] = p.win[(tile * nblk * TB + row) * NC + i];
  }
  __syncthreads();
  // ns k-steps' products, summed by two each and added up, taken from b
  auto take = [&](const T *a, const T *x, int ns) __attribute__((always_inline)) {
    V4 re = CT<T>::zero(), im = CT<T>::zero();
#pragma unroll
    for (int s = 0; s < ns; s += 2) {
      V4 tr = CT<T>::zero(), ti = CT<T>::zero();
      chain_mac<T>(a[s], x[s], tr, ti);
      chain_mac<T>(a[s + 1], x[s + 1], tr, ti);
      re += tr;
      im += ti;
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const T v = chain_elem<T>(re, im, r);
      if (EXACT) sub2(b[r], bl[r], v);
      else b[r] = csub(b[r], v);
    }
  };
  T a[16], x[16];
  if (nk > 0) load(blk(0), a);
  for (long q = 0; q < nk; q++) {
    const T *xs = wt + (blk(q) * TB + 16 * kq) * NC + i;
    unsigned spins = 0;
    for (;;) {
      bool ready = true;
#pragma unroll
      for (int s = 0; s < 16; s++) x[s] = ld_coh(xs + s * NC);
#pragma unroll
      for (int s = 0; s < 16; s++) ready = ready && chain_val_set(x[s]);
      if (ready) break;
      if (__hip_atomic_load(p.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) break;
      if (++spins > GBAR_SPIN) { __hip_atomic_store(p.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); break; }
      __builtin_amdgcn_s_sleep(1);
    }
    take(a, x, 16);
    if (q + 1 < nk) load(blk(q + 1), a);
  }
  // this wave's place in the block's solve order, its columns
  const int me = FWD ? w0 / 16 : 3 - w0 / 16, c4 = w0 / 4;
  T f[12];
#pragma unroll
  for (int s = 0; s < 16; s++) x[s] = sm[s][i];
  dload(1, a);
#pragma unroll
  for (int u = 0; u < 3; u++)
    if (u < me) fload(u, f);
  auto solve = [&](auto uc, T (&d)[16]) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value;
    if (me == u) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int br = w0 + CT<T>::row(lane, r);
        sb[br][i] = br < bs ? b[r] : zero_v<T>();
        if (EXACT) sl[br][i] = br < bs ? bl[r] : zero_v<T>();
      }
    }
    __syncthreads();
    const int row = sub(u) + i;
    // y + yl: what is left (EXACT: yl as bl, else the products' own sum)
    T y = sb[row][c4 + kq], yl = EXACT ? sl[EXACT ? row : 0][c4 + kq] : zero_v<T>();
    const T rd = UNIT ? unit_v<T>() : sr[row], rl = UNIT || !EXACT ? zero_v<T>() : srl[EXACT ? row : 0];
    auto value = [&]() __attribute__((always_inline)) {
      const T z = cadd(y, yl);
      return UNIT ? z : EXACT ? mul2(z, rd, rl) : cmul(z, rd);
    };
    static_for<0, 15>([&](auto sc) __attribute__((always_inline)) {
      constexpr int s = decltype(sc)::value, k = FWD ? s : 15 - s;
      const T v = row_bcast<k>(value());
      if (FWD ? i > k : i < k) {
        if (EXACT) sub2(y, yl, fmul_t(d[s], v));
        else yl = fnma_t(yl, d[s], v);
      }
    });
    sb[row][c4 + kq] = value();
    __syncthreads();
    if constexpr (u < 3)
      if (u < me) {
        T z[4];
#pragma unroll
        for (int s = 0; s < 4; s++) z[s] = sb[sub(u) + 4 * s + kq][i];
        take(f + 4 * u, z, 4);
      }
  };
  solve(std::integral_constant<int, 0>{}, x);
  dload(2, x);
  solve(std::integral_constant<int, 1>{}, a);
  dload(3, a);
  solve(std::integral_constant<int, 2>{}, x);
  solve(std::integral_constant<int, 3>{}, a);
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int br = w0 + kq + 4 * r;
    const long row = g * TB + br, c = tile * NC + i;
    const T v = sb[br][i];
    st_coh(wt + row * NC + i, v);
    if (p.bout && br < bs && c < p.nrhs) p.bout[(p.pout ? p.pout[row] : row) + c * p.ldo] = conj_if(v, (p.cj & 2) != 0);
  }
}

__global__ void k_zero_u64(unsigned long long *w, long n)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) w[i] = 0ull;
}

// lower (forward) then upper (backward) solve of one right-hand side in
// two launches, by substitution if the block inverses are null; returns -2
// without a workspace, -6 on a time-out
template <typename T>
static int trsv_chain(const T *LU, long lda, long n, const T *invL, const T *invU, T *B, T *W, hipStream_t s,
                      unsigned long long *words)
{
  const long nblk = (n + TB - 1) / TB;
  char *w = words ? (char *)words : (char *)ws_get(WS_CHAIN, sizeof(unsigned long long) * (2 * nblk + 8));
  if (!w) return -2;
  unsigned *err = (unsigned *)w, *ticket = (unsigned *)(w + sizeof(unsigned long long));
  // cleared and filled by kernels (not memset nodes, so that a captured
  // sequence does the same on every replay)
  hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, s, (unsigned long long *)w, 8L);
  hipLaunchKernelGGL(k_chain_fill<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, W, n);
  auto both = [&](auto sub) {
    hipLaunchKernelGGL((k_trsv_chain<T, true, decltype(sub)::value>), dim3((unsigned)nblk), dim3(256), 0, s, LU, lda, n,
                       invL, B, W, 1, err, ticket);
    hipLaunchKernelGGL((k_trsv_chain<T, false, decltype(sub)::value>), dim3((unsigned)nblk), dim3(256), 0, s, LU, lda, n,
                       invU, W, B, 0, err, ticket + 2);
  };
  if constexpr (std::is_same<T, float2>::value) {
    if (invL) both(std::false_type{});
    else both(std::true_type{});
  } else
    both(std::true_type{});
  if (hipGetLastError() != hipSuccess) return -3;
  unsigned tmo = 0;
  hipMemcpyAsync(&tmo, err, sizeof(unsigned), hipMemcpyDeviceToHost, s);
  hipStreamSynchronize(s);
  return tmo ? -6 : 0;
}

// one triangle of k_trsm_chain
template <typename T>
static void trsm_launch(bool fwd, bool trans, const ChainArgs<T> &p, hipStream_t s)
{
  const long nblk = (p.n + TB - 1) / TB, ntile = (p.nrhs + 15) / 16;
  const dim3 grid((unsigned)(nblk * ntile));
  if (fwd && !trans) hipLaunchKernelGGL((k_trsm_chain<T, true, false>), grid, dim3(256), 0, s, p);
  else if (!trans) hipLaunchKernelGGL((k_trsm_chain<T, false, false>), grid, dim3(256), 0, s, p);
  else if (fwd) hipLaunchKernelGGL((k_trsm_chain<T, true, true>), grid, dim3(256), 0, s, p);
  else hipLaunchKernelGGL((k_trsm_chain<T, false, true>), grid, dim3(256), 0, s, p);
}

// op(A) X = B for any number of right-hand sides, at most CHAIN_COLS at a
// time: that bounds the workspace, and 64 tiles a block step fill the GPU.
#define CHAIN_COLS 1024
template <typename T>
static int trsm_chain(const T *LU, long lda, long n, const int *ipiv, bool tr, bool cj, long nrhs, T *B, long ldb,
                      hipStream_t s)
{
  const long nblk = (n + TB - 1) / TB, cols = std::min<long>(nrhs, CHAIN_COLS);
  const size_t wlen = (size_t)nblk * TB * 16 * ((cols + 15) / 16);      // elements of one packed set
  T *W1 = (T *)ws_get(WS_SOLVE_W, sizeof(T) * wlen), *W2 = (T *)ws_get(WS_PERM_TMP, sizeof(T) * wlen);
  unsigned long long *word = (unsigned long long *)ws_get(WS_CHAIN, sizeof(unsigned long long) * (2 * nblk + 8));
  int *perm = n > PERM_LDS_MAX ? nullptr : (int *)ws_get(WS_PERM, sizeof(int) * n);
  if (!W1 || !W2 || !word || (n <= PERM_LDS_MAX && !perm)) return -2;
  if (perm) hipLaunchKernelGGL(k_perm_build, dim3(1), dim3(64), 0, s, ipiv, n, perm, 0L, 0L);
  ChainArgs<T> p;
  p.lda = lda;
  p.err = (unsigned *)word;
  auto fill = [&](T *w, long ncol) {
    const long ne = nblk * TB * 16 * ((ncol + 15) / 16);
    hipLaunchKernelGGL(k_chain_fill<T>, dim3((unsigned)((ne + 255) / 256)), dim3(256), 0, s, w, ne);
  };
  // the time-out word once, the two tickets before every set of columns
  hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, s, word, 1L);
  for (long c0 = 0; c0 < nrhs; c0 += CHAIN_COLS) {
    const long nc = std::min<long>(CHAIN_COLS, nrhs - c0);
    T *Bc = B + c0 * ldb;
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, s, word + 1, 2L);
    p.nrhs = nc;
    if (!perm && !tr) laswp(Bc, ldb, 0, nc, 0, n, ipiv, s);
    fill(W1, nc);
    fill(W2, nc);
    p.A = LU; p.n = n; p.ldb = p.ldo = ldb;
    p.bin = Bc; p.pin = tr ? nullptr : perm; p.win = nullptr;
    p.w = W1; p.bout = nullptr; p.pout = nullptr; p.cj = cj ? 1 : 0; p.ticket = (unsigned *)(word + 1);
    trsm_launch(true, tr, p, s);
    p.bin = nullptr; p.pin = nullptr; p.win = W1;
    p.w = W2; p.bout = Bc; p.pout = tr ? perm : nullptr; p.cj = cj ? 2 : 0; p.ticket = (unsigned *)(word + 2);
    trsm_launch(false, tr, p, s);
    if (!perm && tr)
      hipLaunchKernelGGL(k_laswp_rev<T>, dim3((unsigned)((nc + 63) / 64)), dim3(64), 0, s, Bc, ldb, n, nc, ipiv);
  }
  unsigned tmo = 0;
  hipMemcpyAsync(&tmo, p.err, sizeof(unsigned), hipMemcpyDeviceToHost, s);
  hipStreamSynchronize(s);
  if (hipGetLastError() != hipSuccess) return -3;
  return tmo ? -6 : 0;
}

template <typename T>
size_t solve_ws_bytes(long n, bool refined)
{
  auto r256 = [](size_t b) { return 256 * ((b + 255) / 256); };
  const long nblk = (n + TB - 1) / TB;
  return r256(sizeof(T) * n) + (refined ? 2 * r256(sizeof(T) * nblk * TB * TB) : 0) + r256(sizeof(int) * n) +
         r256(sizeof(unsigned long long) * (2 * nblk + 8));
}

template <typename T>
SolveWs<T> solve_ws_carve(char *base, long n, bool refined)
{
  auto r256 = [](size_t b) { return 256 * ((b + 255) / 256); };
  const long nblk = (n + TB - 1) / TB;
  SolveWs<T> w;
  w.W = (T *)base; base += r256(sizeof(T) * n);
  w.refined = refined;
  if (refined) {
    w.invL = (T *)base; base += r256(sizeof(T) * nblk * TB * TB);
    w.invU = (T *)base; base += r256(sizeof(T) * nblk * TB * TB);
  }
  w.perm = (int *)base; base += r256(sizeof(int) * n);
  w.chain = (unsigned long long *)base;
  return w;
}

template <typename T>
int lu_solve(const T *LU, long n, long lda, const int *d_ipiv, char trans, long nrhs, T *B, long ldb,
             hipStream_t stream, SolveWs<T> *ws)
{
  if (n < 0 || nrhs < 0 || lda < std::max(1L, n) || ldb < std::max(1L, n)) return -1;
  if (n == 0 || nrhs == 0) return 0;
  if (ws && !((trans == 'N' || trans == 'n') && nrhs == 1)) return -1;
  const bool tr = trans == 'T' || trans == 't' || trans == 'C' || trans == 'c', cj = trans == 'C' || trans == 'c';
  if (!tr && trans != 'N' && trans != 'n') return -1;
  if (!tr && nrhs == 1) {
    T *W = ws ? ws->W : (T *)ws_get(WS_SOLVE_W, sizeof(T) * n);
    if (!W) return -2;
    // a solve after the first with the same factors reuses the block
    // inverses and the composed permutation
    const bool cached = ws && ws->inv_ready;
    T *invL = nullptr, *invU = nullptr;
    if constexpr (std::is_same<T, float2>::value)
      if (ws && ws->refined) {
        invL = ws->invL;
        invU = ws->invU;
        if (!cached) tri_inv(LU, lda, n, invL, invU, stream);
      }
    if (ws) ws->inv_ready = true;
    apply_row_perm(B, n, d_ipiv, W, stream, ws ? ws->perm : nullptr, cached);
    return trsv_chain(LU, lda, n, invL, invU, B, W, stream, ws ? ws->chain : nullptr);
  }
  return trsm_chain(LU, lda, n, d_ipiv, tr, cj, nrhs, B, ldb, stream);
}

// log det of an LU-factored matrix: sum of log |U_ii| and of arg U_ii, plus
// pi for every row interchange (deterministic two-pass reduction)
template <typename T>
__global__ void __launch_bounds__(256) k_logdet(const T *LU, long n, long lda, const int *ipiv, double *out)
{
  __shared__ double s0[256], s1[256];
  double a = 0, b = 0;
  for (long i = threadIdx.x; i < n; i += 256) {
    T d = LU[i + i * lda];
    double re = re_of(d), im = im_of(d);
    a += 0.5 * log(re * re + im * im);
    b += atan2(im, re);
    if (ipiv[i] != i + 1) b += 3.14159265358979323846;
  }
  s0[threadIdx.x] = a; s1[threadIdx.x] = b;
  __syncthreads();
  for (int q = 128; q > 0; q >>= 1) {
    if (threadIdx.x < q) { s0[threadIdx.x] += s0[threadIdx.x + q]; s1[threadIdx.x] += s1[threadIdx.x + q]; }
    __syncthreads();
  }
  if (threadIdx.x == 0) { out[0] = s0[0]; out[1] = s1[0]; }
}

// trace of a square matrix (complex sum of the diagonal)
template <typename T>
__global__ void __launch_bounds__(256) k_trace(const T *A, long n, long lda, double *out)
{
  __shared__ double s0[256], s1[256];
  double a = 0, b = 0;
  for (long i = threadIdx.x; i < n; i += 256) { T d = A[i + i * lda]; a += re_of(d); b += im_of(d); }
  s0[threadIdx.x] = a; s1[threadIdx.x] = b;
  __syncthreads();
  for (int q = 128; q > 0; q >>= 1) {
    if (threadIdx.x < q) { s0[threadIdx.x] += s0[threadIdx.x + q]; s1[threadIdx.x] += s1[threadIdx.x + q]; }
    __syncthreads();
  }
  if (threadIdx.x == 0) { out[0] = s0[0]; out[1] = s1[0]; }
}

template <typename T>
int lu_logdet(const T *LU, long n, long lda, const int *ipiv, double out[2], hipStream_t s)
{
  double *d = (double *)ws_get(WS_SMALL, 256);
  if (!d) return -2;
  hipLaunchKernelGGL(k_logdet<T>, dim3(1), dim3(256), 0, s, LU, n, lda, ipiv, d);
  hipMemcpyAsync(out, d, 2 * sizeof(double), hipMemcpyDeviceToHost, s);
  return hipStreamSynchronize(s) == hipSuccess ? 0 : -3;
}

template <typename T>
int mat_trace(const T *A, long n, long lda, double out[2], hipStream_t s)
{
  double *d = (double *)ws_get(WS_SMALL, 256);
  if (!d) return -2;
  hipLaunchKernelGGL(k_trace<T>, dim3(1), dim3(256), 0, s, A, n, lda, d);
  hipMemcpyAsync(out, d, 2 * sizeof(double), hipMemcpyDeviceToHost, s);
  return hipStreamSynchronize(s) == hipSuccess ? 0 : -3;
}

template int lu_logdet<double2>(const double2 *, long, long, const int *, double *, hipStream_t);
template int lu_logdet<double>(const double *, long, long, const int *, double *, hipStream_t);
template int mat_trace<double>(const double *, long, long, double *, hipStream_t);
template int lu_factor<double>(double *, long, long, int *, int *, hipStream_t, int, int);
template int lu_solve<double>(const double *, long, long, const int *, char, long, double *, long, hipStream_t,
                              SolveWs<double> *);
template int lu_logdet<float2>(const float2 *, long, long, const int *, double *, hipStream_t);
template int mat_trace<double2>(const double2 *, long, long, double *, hipStream_t);
template int mat_trace<float2>(const float2 *, long, long, double *, hipStream_t);
template int lu_factor<double2>(double2 *, long, long, int *, int *, hipStream_t, int, int);
template int lu_factor<float2>(float2 *, long, long, int *, int *, hipStream_t, int, int);
template int lu_solve<double2>(const double2 *, long, long, const int *, char, long, double2 *, long, hipStream_t,
                               SolveWs<double2> *);
template int lu_solve<float2>(const float2 *, long, long, const int *, char, long, float2 *, long, hipStream_t,
                              SolveWs<float2> *);
template size_t solve_ws_bytes<double2>(long, bool);
template size_t solve_ws_bytes<float2>(long, bool);
template SolveWs<double2> solve_ws_carve<double2>(char *, long, bool);
template SolveWs<float2> solve_ws_carve<float2>(char *, long, bool);

// ---------------------------------------------------------------------
// one-right-hand-side solve that allocates nothing: the buffers of a
// SolveWs (W, composed permutation, one-launch words) are carved from a
// fixed device array, one copy per GPU, held until the process ends.  Every call on a GPU
// shares that GPU's array, so calls that overlap on one GPU race.
// ---------------------------------------------------------------------
constexpr long r256_const(long b) { return 256 * ((b + 255) / 256); }
constexpr long NOALLOC_NBLK = (NOALLOC_MAX_N + TB - 1) / TB;
constexpr long NOALLOC_BYTES = r256_const((long)sizeof(double2) * NOALLOC_MAX_N) +
                               r256_const((long)sizeof(int) * NOALLOC_MAX_N) +
                               r256_const((long)sizeof(unsigned long long) * (2 * NOALLOC_NBLK + 8));
static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

long noalloc_scratch_bytes() { return NOALLOC_BYTES; }

// device address of this GPU's copy of `scratch`, looked up once per device
// with that device current (the array's name in host code is only a
// host-side stand-in, never a device address)
static void *noalloc_scratch_ptr()
{
  static std::mutex mu;
  static void *ptr[64] = {nullptr};
  int d = 0;
  if (hipGetDevice(&d) != hipSuccess || d < 0 || d >= 64) return nullptr;
  std::lock_guard<std::mutex> lk(mu);
  if (!ptr[d]) {
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return nullptr;
    ptr[d] = p;
  }
  return ptr[d];
}

template <typename T>
int lu_solve_noalloc(const T *LU, long n, long lda, const int *d_ipiv, T *B, hipStream_t stream)
{
  if (n < 0 || lda < std::max(1L, n)) return -1;
  if (n > NOALLOC_MAX_N || (long)solve_ws_bytes<T>(n, false) > NOALLOC_BYTES) return -7;
  if (n == 0) return 0;
  char *base = (char *)noalloc_scratch_ptr();
  if (!base) return -3;
  SolveWs<T> w = solve_ws_carve<T>(base, n, false);
  w.inv_ready = false;   // the array holds whatever the last call left
  return lu_solve<T>(LU, n, lda, d_ipiv, 'N', 1, B, std::max(1L, n), stream, &w);
}
template int lu_solve_noalloc<double2>(const double2 *, long, long, const int *, double2 *, hipStream_t);
template int lu_solve_noalloc<float2>(const float2 *, long, long, const int *, float2 *, hipStream_t);

// ---------------------------------------------------------------------
// refinement helpers
// ---------------------------------------------------------------------
#define RES_COLCHUNK 512
__global__ void __launch_bounds__(256)
k_resid_partial(const double2 *A, long n, long lda, const double2 *x, double2 *work, long sa, long sx, long sw)
{
  {
    const long z = blockIdx.z;   // instance of a batch
    A += z * sa; x += z * sx; work += z * sw;
  }
  long i = (long)blockIdx.x * 256 + threadIdx.x;
  long c0 = (long)blockIdx.y * RES_COLCHUNK, c1 = std::min(n, c0 + RES_COLCHUNK);
  if (i >= n) return;
  double sr = 0, si = 0;
  for (long c = c0; c < c1; c++) {
    double2 a = A[i + c * lda], v = x[c];
    sr += a.x * v.x - a.y * v.y;
    si += a.x * v.y + a.y * v.x;
  }
  work[blockIdx.y * n + i] = make_double2(sr, si);
}

__global__ void k_resid_final(long n, int nch, const double2 *b, const double2 *work, double2 *r, long sb, long sw,
                              long srr)
{
  {
    const long z = blockIdx.y;   // instance of a batch
    if (b) b += z * sb;
    work += z * sw; r += z * srr;
  }
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double sr = 0, si = 0;
  for (int q = 0; q < nch; q++) { sr += work[q * n + i].x; si += work[q * n + i].y; }
  r[i] = b ? make_double2(b[i].x - sr, b[i].y - si) : make_double2(sr, si);
}

long residual_chunks(long n) { return (n + RES_COLCHUNK - 1) / RES_COLCHUNK; }

int residual_c128(const double2 *A, long n, long lda, const double2 *x, const double2 *b, double2 *r,
                  double2 *work, hipStream_t stream)
{
  int nch = (int)((n + RES_COLCHUNK - 1) / RES_COLCHUNK);
  hipLaunchKernelGGL(k_resid_partial, dim3((unsigned)((n + 255) / 256), nch), dim3(256), 0, stream, A, n, lda, x, work,
                     0L, 0L, 0L);
  hipLaunchKernelGGL(k_resid_final, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, n, nch, b, work, r, 0L, 0L,
                     0L);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

__global__ void k_c128_to_c64(const double2 *x, float2 *y, long rows, long cols, long ldx, long ldy)
{
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x, c = blockIdx.y;
  if (i >= rows) return;
  for (; c < cols; c += gridDim.y) {
    double2 v = x[i + c * ldx];
    y[i + c * ldy] = make_float2((float)v.x, (float)v.y);
  }
}

int convert_c128_to_c64(const double2 *x, float2 *y, long rows, long cols, long ldx, long ldy, hipStream_t stream)
{
  unsigned gy = (unsigned)std::min<long>(cols, 65535);
  hipLaunchKernelGGL(k_c128_to_c64, dim3((unsigned)((rows + 255) / 256), gy), dim3(256), 0, stream, x, y, rows, cols, ldx, ldy);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// real parts of a complex128 block into a real matrix (column-major, or
// packed upper storage of a square block: dst[r + c (c+1)/2], r <= c)
__global__ void k_re_part(const double2 *x, long ldx, double *y, long ldy, long rows, long cols, int packed)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  for (long c = blockIdx.y; c < cols; c += gridDim.y) {
    if (i >= rows) return;
    const double v = x[i + c * ldx].x;
    if (!packed) y[i + c * ldy] = v;
    else if (i <= c) y[i + c * (c + 1) / 2] = v;
  }
}

int real_part_c128(const double2 *x, long ldx, double *y, long ldy, long rows, long cols, int packed,
                   hipStream_t stream)
{
  if (rows <= 0 || cols <= 0) return 0;
  unsigned gy = (unsigned)std::min<long>(cols, 65535);
  hipLaunchKernelGGL(k_re_part, dim3((unsigned)((rows + 255) / 256), gy), dim3(256), 0, stream, x, ldx, y, ldy, rows,
                     cols, packed);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// full n x n matrix from packed upper storage (symmetric: A(r,c) = A(c,r))
template <typename T>
__global__ void k_unpack_sym(const T *P, T *A, long lda, long n)
{
  const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
  for (long c = blockIdx.y; c < n; c += gridDim.y) {
    if (r >= n) return;
    const long lo = r < c ? r : c, hi = r < c ? c : r;
    A[r + c * lda] = P[lo + hi * (hi + 1) / 2];
  }
}

template <typename T>
int unpack_symmetric(const T *P, T *A, long lda, long n, hipStream_t stream)
{
  if (n <= 0) return 0;
  unsigned gy = (unsigned)std::min<long>(n, 65535);
  hipLaunchKernelGGL(k_unpack_sym<T>, dim3((unsigned)((n + 255) / 256), gy), dim3(256), 0, stream, P, A, lda, n);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
template int unpack_symmetric<double>(const double *, double *, long, long, hipStream_t);
template int unpack_symmetric<double2>(const double2 *, double2 *, long, long, hipStream_t);
template int unpack_symmetric<float2>(const float2 *, float2 *, long, long, hipStream_t);

// identity matrix (n x n, column-major)
template <typename T>
__global__ void k_identity(T *A, long lda, long n)
{
  const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
  for (long c = blockIdx.y; c < n; c += gridDim.y) {
    if (r >= n) return;
    A[r + c * lda] = r == c ? unit_v<T>() : zero_v<T>();
  }
}

// first zero diagonal entry (1-based) of U, or 0
template <typename T>
__global__ void k_first_zero_diag(const T *LU, long lda, long n, int *out)
{
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    if (!nonzero(LU[i + i * lda])) atomicMin(out, (int)(i + 1));
}

// LUInvert (zgetri / dgetri semantics): A <- A^{-1} from its LU factors
// (unit-lower L, U, ipiv), as the solution of A X = I with nrhs = n; W holds
// n x n elements plus one int.  info = first zero diagonal of U (A unchanged)
template <typename T>
int lu_invert(T *A, long n, long lda, const int *ipiv, T *W, int *info, hipStream_t s)
{
  *info = 0;
  if (n <= 0) return 0;
  int *dz = (int *)(W + n * n);
  const int big = 0x7F7F7F7F;          // every byte 0x7F: larger than any index
  hipMemsetAsync(dz, 0x7F, sizeof(int), s);
  hipLaunchKernelGGL(k_first_zero_diag<T>, dim3((unsigned)std::min<long>(1024, (n + 255) / 256)), dim3(256), 0, s, A,
                     lda, n, dz);
  int z = 0;
  hipMemcpyAsync(&z, dz, sizeof(int), hipMemcpyDeviceToHost, s);
  if (hipStreamSynchronize(s) != hipSuccess) return -3;
  if (z != big) { *info = z; return 0; }
  unsigned gy = (unsigned)std::min<long>(n, 65535);
  hipLaunchKernelGGL(k_identity<T>, dim3((unsigned)((n + 255) / 256), gy), dim3(256), 0, s, W, n, n);
  int rc = lu_solve<T>(A, n, lda, ipiv, 'N', n, W, n, s);
  if (rc) return rc;
  hipMemcpy2DAsync(A, sizeof(T) * lda, W, sizeof(T) * n, sizeof(T) * n, n, hipMemcpyDeviceToDevice, s);
  return hipStreamSynchronize(s) == hipSuccess ? 0 : -3;
}
template int lu_invert<double2>(double2 *, long, long, const int *, double2 *, int *, hipStream_t);
template int lu_invert<float2>(float2 *, long, long, const int *, float2 *, int *, hipStream_t);
template int lu_invert<double>(double *, long, long, const int *, double *, int *, hipStream_t);

__global__ void k_c64_to_c128(const float2 *x, double2 *y, long n)
{
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = make_double2(x[i].x, x[i].y);
}
int convert_c64_to_c128(const float2 *x, double2 *y, long n, hipStream_t stream)
{
  hipLaunchKernelGGL(k_c64_to_c128, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, x, y, n);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

__global__ void k_axpy64(const float2 *d, double2 *x, long n)
{
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) { x[i].x += (double)d[i].x; x[i].y += (double)d[i].y; }
}
int axpy_c64_into_c128(const float2 *d, double2 *x, long n, hipStream_t stream)
{
  hipLaunchKernelGGL(k_axpy64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, d, x, n);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

__global__ void k_absmax(const double2 *x, long n, double *out)
{
  __shared__ double s[256];
  double m = 0;
  for (long i = threadIdx.x; i < n; i += 256) m = fmax(m, fabs(x[i].x) + fabs(x[i].y));
  s[threadIdx.x] = m;
  __syncthreads();
  for (int q = 128; q > 0; q >>= 1) { if (threadIdx.x < q) s[threadIdx.x] = fmax(s[threadIdx.x], s[threadIdx.x + q]); __syncthreads(); }
  if (threadIdx.x == 0) *out = s[0];
}
double absmax_c128(const double2 *x, long n, double *work, hipStream_t stream)
{
  hipLaunchKernelGGL(k_absmax, dim3(1), dim3(256), 0, stream, x, n, work);
  double h = 0;
  hipMemcpyAsync(&h, work, sizeof(double), hipMemcpyDeviceToHost, stream);
  hipStreamSynchronize(stream);
  return h;
}

// ---------------------------------------------------------------------
// Batched complex64 LU with tournament pivoting: nbat matrices of equal
// order n at A + b sa, factored in lockstep, every step one launch over
// the whole batch (panels: (G + 1) x nbat workgroups; updates: grid.y or
// grid.z = instance).  No lookahead (the batch fills the GPU), no host
// synchronization, no allocation and no memset, so that a stream capture
// records it.  The per-instance panel scratch (layout of lu_factor's
// complex64 tournament path) is cleared by a kernel at the start.
// ---------------------------------------------------------------------
struct BatchLayout {
  size_t off_info, off_plan, off_li, off_ts, total;
  long Gmax, npanels;
};

static BatchLayout batch_layout(long n)
{
  auto r256 = [](size_t b) { return 256 * ((b + 255) / 256); };
  BatchLayout L;
  L.Gmax = (n + 255) / 256;
  L.npanels = (n + PW - 1) / PW;
  L.off_info = 96 * sizeof(unsigned);
  L.off_plan = L.off_info + 64;
  L.off_li = L.off_plan + r256(sizeof(int) * PLAN_LEN * L.npanels);
  L.off_ts = L.off_li + r256(sizeof(float2) * PW * PW * L.npanels);
  const size_t ts_words = (size_t)ts_root_off(ts_levels(L.Gmax), L.Gmax) + TS_ROOT;
  L.total = r256(L.off_ts + sizeof(unsigned long long) * ts_words);
  return L;
}

size_t lu_batch_scratch_bytes(long n) { return batch_layout(n).total; }

__global__ void k_batch_status(const char *scratch, long sS, long off_info, int nbat, int *status)
{
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nbat) return;
  const char *base = scratch + (long)b * sS;
  status[2 * b] = *(const int *)(base + off_info);
  status[2 * b + 1] = (int)((const unsigned *)base)[64];
}

long lu_batch_slots()
{
  int dev = 0, ncu = 0, perCU = 0;
  hipGetDevice(&dev);
  hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, (const void *)k_panel_ts, 256, 0);
  return (long)std::max(1, ncu) * std::max(1, perCU);
}

long lu_batch_workgroups(long n, int nbat) { return nbat * ((n + 255) / 256 + 1); }

int lu_batch_max(long n) { return (int)(lu_batch_slots() / lu_batch_workgroups(n, 1)); }

int lu_factor_batch(float2 *A, long n, long lda, int nbat, long sa, int *ipiv, long sp, void *scratch, int *status,
                    hipStream_t s, int nb)
{
  if (n <= 0 || nbat <= 0 || lda < n || !scratch || !status) return -1;
  if (nb <= 0 || nb > 256 || nb % PW) return -1;
  const BatchLayout L = batch_layout(n);
  if (L.Gmax > 64 * KEYS_PER_LANE) return -5;
  if (nbat > lu_batch_max(n)) return -5;      // every panel workgroup of the batch must be co-resident
  const long sS = (long)L.total;
  char *base = (char *)scratch;
  const long nwords = (long)nbat * sS / 8;
  hipLaunchKernelGGL(k_zero_u64, dim3((unsigned)((nwords + 255) / 256)), dim3(256), 0, s,
                     (unsigned long long *)base, nwords);
  PanelScratch S;
  S.bar = (unsigned *)base;
  int *dinfo = (int *)(base + L.off_info);
  int *plans = (int *)(base + L.off_plan);
  S.xch = nullptr;
  S.linv = (void *)(base + L.off_li);
  S.ts = (unsigned long long *)(base + L.off_ts);
  const float2 *linv = (const float2 *)S.linv;
  const bool g3m = mixed_gemm_3m();
  BStride bs;
  bs.a = sa; bs.p = sp; bs.s = sS;
  int gmaxi = (int)L.Gmax;
  for (long K = 0; K < n; K += nb) {
    const long jb = std::min<long>(nb, n - K);
    const long p0 = K / PW;
    for (long j0 = K; j0 < K + jb; j0 += PW) {
      int w = (int)std::min<long>(PW, K + jb - j0);
      long m = n - j0, G = (m + 255) / 256, r0 = j0;
      S.plan = plans + (j0 / PW) * PLAN_LEN;
      unsigned seq0 = (unsigned)(j0 + 1);
      void *args[] = {(void *)&A, (void *)&lda, (void *)&r0, (void *)&m, (void *)&w, (void *)&ipiv,
                      (void *)&dinfo, (void *)&S, (void *)&gmaxi, (void *)&seq0, (void *)&bs};
      int tok = prof_begin(s, PK_PANEL_C64);
      hipError_t e = hipLaunchKernel((const void *)k_panel_ts, dim3((unsigned)G + 1, (unsigned)nbat), dim3(256), args,
                                     0, s);
      prof_end(s, tok, 0.0);
      if (e != hipSuccess) return -3;
      swap_trmm(A, lda, K, K + jb, j0, j0 + w, S.plan, linv + (j0 / PW) * PW * PW, w, j0, s, nbat, bs);
      const long nr = K + jb - (j0 + w);
      if (nr > 0)
        gemm_sub(n - j0 - w, nr, (long)w, A + (j0 + w) + j0 * lda, lda, A + j0 + (j0 + w) * lda, lda,
                 A + (j0 + w) + (j0 + w) * lda, lda, s, 0, nbat, sa, g3m);
    }
    const long c1 = K + jb;
    if (c1 < n) {
      const int bplans = (int)((jb + PW - 1) / PW);
      laswp_plans(A, lda, c1, n, 0, 0, plans + p0 * PLAN_LEN, bplans, s, nbat, bs);
      trsm_blk(A, lda, K, (int)jb, linv + p0 * PW * PW, A + K + c1 * lda, lda, n - c1, s, nbat, bs);
      gemm_sub(n - c1, n - c1, jb, A + c1 + K * lda, lda, A + K + c1 * lda, lda, A + c1 + c1 * lda, lda, s, 0, nbat,
               sa, g3m);
    }
  }
  // interchanges of each block on the columns left of it
  for (long K = nb; K < n; K += nb) {
    const long jb = std::min<long>(nb, n - K);
    laswp_plans(A, lda, 0, K, 0, 0, plans + (K / PW) * PLAN_LEN, (int)((jb + PW - 1) / PW), s, nbat, bs);
  }
  hipLaunchKernelGGL(k_batch_status, dim3((unsigned)((nbat + 63) / 64)), dim3(64), 0, s, (const char *)base, sS,
                     (long)L.off_info, nbat, status);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// Batched one-right-hand-side solves with batched complex64 factors:
// prepare (composed row permutations and inverses of the 64 x 64 diagonal
// blocks of L and U, once per factorization), then any number of solves
// of B (n per instance, sb apart) in place.  No host synchronization.
struct BatchSolveLayout {
  size_t off_invL, off_invU, off_W, total;
};
static BatchSolveLayout batch_solve_layout(long n)
{
  auto r256 = [](size_t b) { return 256 * ((b + 255) / 256); };
  const long nblk = (n + TB - 1) / TB;
  BatchSolveLayout L;
  L.off_invL = r256(sizeof(int) * n);
  L.off_invU = L.off_invL + r256(sizeof(float2) * nblk * TB * TB);
  L.off_W = L.off_invU + r256(sizeof(float2) * nblk * TB * TB);
  L.total = L.off_W + r256(sizeof(float2) * n);
  return L;
}
size_t lu_solve_batch_bytes(long n) { return batch_solve_layout(n).total; }

int lu_solve_batch_prepare(const float2 *LU, long n, long lda, int nbat, long sa, const int *ipiv, long sp, void *ws,
                           hipStream_t s)
{
  if (n <= 0 || nbat <= 0 || n > PERM_LDS_MAX || !ws) return -1;
  const BatchSolveLayout L = batch_solve_layout(n);
  const long sw = (long)L.total, nblk = (n + TB - 1) / TB;
  char *base = (char *)ws;
  hipLaunchKernelGGL(k_perm_build, dim3((unsigned)nbat), dim3(64), 0, s, ipiv, n, (int *)base, sp, sw / 4);
  tri_inv(LU, lda, n, (float2 *)(base + L.off_invL), (float2 *)(base + L.off_invU), s, nbat, sa, sw / 8);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

__global__ void k_copy_batch(const float2 *in, long sin, float2 *out, long sout, long n)
{
  const long i = (long)blockIdx.x * 256 + threadIdx.x, z = blockIdx.z;
  if (i < n) out[z * sout + i] = in[z * sin + i];
}

int lu_solve_batch(const float2 *LU, long n, long lda, int nbat, long sa, float2 *B, long sb, void *ws, hipStream_t s)
{
  if (n <= 0 || nbat <= 0 || !ws) return -1;
  const BatchSolveLayout L = batch_solve_layout(n);
  const long sw = (long)L.total;
  char *base = (char *)ws;
  const int *perm = (const int *)base;
  const float2 *invL = (const float2 *)(base + L.off_invL), *invU = (const float2 *)(base + L.off_invU);
  float2 *W = (float2 *)(base + L.off_W);
  const long swp = sw / 4, swe = sw / 8;   // the stride in ints and in complex64 elements
  // W = P B
  hipLaunchKernelGGL(k_perm_apply<float2>, dim3((unsigned)((n + 255) / 256), 1, (unsigned)nbat), dim3(256), 0, s,
                     (const float2 *)B, W, perm, n, sb, swe, swp);
  // L y = W: W is the running right-hand side, y lands in B
  for (long kb = 0; kb < n; kb += TB) {
    const int bs = (int)std::min<long>(TB, n - kb);
    const long rows = n - kb - bs;
    dim3 grid((unsigned)std::max<long>(1, (rows + 255) / 256), 1, (unsigned)nbat);
    hipLaunchKernelGGL((k_trsv_inv<float2, true>), grid, dim3(256), 0, s, LU, lda, n, kb, bs,
                       invL + (kb / TB) * TB * TB, W, B, sa, swe, swe, sb);
  }
  // U x = y: B is the running right-hand side, x lands in W
  const long last = ((n - 1) / TB) * TB;
  for (long kb = last; kb >= 0; kb -= TB) {
    const int bs = (int)std::min<long>(TB, n - kb);
    dim3 grid((unsigned)std::max<long>(1, (kb + 255) / 256), 1, (unsigned)nbat);
    hipLaunchKernelGGL((k_trsv_inv<float2, false>), grid, dim3(256), 0, s, LU, lda, n, kb, bs,
                       invU + (kb / TB) * TB * TB, B, W, sa, swe, sb, swe);
  }
  // B = x
  hipLaunchKernelGGL(k_copy_batch, dim3((unsigned)((n + 255) / 256), 1, (unsigned)nbat), dim3(256), 0, s,
                     (const float2 *)W, swe, B, sb, n);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// per instance of a batch: max|r_i| / max|b_i| (|re| + |im|), vectors n apart
__global__ void k_batch_relres(const double2 *r, const double2 *b, long n, double *out)
{
  __shared__ double sr[256], sb[256];
  const long z = blockIdx.x;
  r += z * n; b += z * n;
  double mr = 0, mb = 0;
  for (long i = threadIdx.x; i < n; i += 256) {
    mr = fmax(mr, fabs(r[i].x) + fabs(r[i].y));
    mb = fmax(mb, fabs(b[i].x) + fabs(b[i].y));
  }
  sr[threadIdx.x] = mr; sb[threadIdx.x] = mb;
  __syncthreads();
  for (int q = 128; q > 0; q >>= 1) {
    if (threadIdx.x < q) { sr[threadIdx.x] = fmax(sr[threadIdx.x], sr[threadIdx.x + q]); sb[threadIdx.x] = fmax(sb[threadIdx.x], sb[threadIdx.x + q]); }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[z] = sb[0] > 0 ? sr[0] / sb[0] : sr[0];
}
int batch_relres(const double2 *r, const double2 *b, long n, int nbat, double *out, hipStream_t s)
{
  hipLaunchKernelGGL(k_batch_relres, dim3((unsigned)nbat), dim3(256), 0, s, r, b, n, out);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

__global__ void k_zero_c128(double2 *x, long n)
{
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) x[i] = make_double2(0.0, 0.0);
}
int zero_c128(double2 *x, long n, hipStream_t s)
{
  if (n <= 0) return 0;
  hipLaunchKernelGGL(k_zero_c128, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, n);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// r = b - A x for a batch (A + z sa, x / b / r n apart, work n * chunks apart)
int residual_c128_batch(const double2 *A, long n, long lda, long sa, int nbat, const double2 *x, const double2 *b,
                        double2 *r, double2 *work, hipStream_t stream)
{
  const int nch = (int)((n + RES_COLCHUNK - 1) / RES_COLCHUNK);
  hipLaunchKernelGGL(k_resid_partial, dim3((unsigned)((n + 255) / 256), nch, (unsigned)nbat), dim3(256), 0, stream, A,
                     n, lda, x, work, sa, n, n * (long)nch);
  hipLaunchKernelGGL(k_resid_final, dim3((unsigned)((n + 255) / 256), (unsigned)nbat), dim3(256), 0, stream, n, nch, b,
                     work, r, n, n * (long)nch, n);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace scuffx
