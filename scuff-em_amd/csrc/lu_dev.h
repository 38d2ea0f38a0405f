// lu_dev.h -- device helpers shared by the LU's translation units: complex
// and real arithmetic, the coherent exchange words of the panels, the panel
// scratch.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

namespace scuffx {

template <typename T> __device__ inline T cmul(T a, T b) { T r; r.x = a.x * b.x - a.y * b.y; r.y = a.x * b.y + a.y * b.x; return r; }
template <typename T> __device__ inline T csub(T a, T b) { T r; r.x = a.x - b.x; r.y = a.y - b.y; return r; }
template <typename T> __device__ inline T cadd(T a, T b) { T r; r.x = a.x + b.x; r.y = a.y + b.y; return r; }
template <typename T> __device__ inline T crecip(T a)
{
  // Smith's algorithm for 1/a
  T r;
  typedef decltype(a.x) R;
  if (fabs(a.x) >= fabs(a.y)) { R t = a.y / a.x, d = a.x + a.y * t; r.x = 1 / d; r.y = -t / d; }
  else { R t = a.x / a.y, d = a.x * t + a.y; r.x = t / d; r.y = -1 / d; }
  return r;
}
// real (double) counterparts, so that the panel and the solves also
// instantiate for real matrices (LHM_REAL, dgetrf/dgetrs semantics)
__device__ inline double cmul(double a, double b) { return a * b; }
__device__ inline double csub(double a, double b) { return a - b; }
__device__ inline double cadd(double a, double b) { return a + b; }
__device__ inline double crecip(double a) { return 1.0 / a; }
// pivot magnitude |re| + |im| (izamax / idamax)
__device__ inline double mag1(double a) { return fabs(a); }
template <typename T> __device__ inline auto mag1(T a) -> decltype(a.x) { return fabs(a.x) + fabs(a.y); }
__device__ inline bool nonzero(double a) { return a != 0; }
template <typename T> __device__ inline bool nonzero(T a) { return a.x != 0 || a.y != 0; }
template <typename T> __device__ inline T zero_v() { T r; r.x = 0; r.y = 0; return r; }
template <> __device__ inline double zero_v<double>() { return 0; }
template <typename T> __device__ inline T unit_v() { T r; r.x = 1; r.y = 0; return r; }
template <> __device__ inline double unit_v<double>() { return 1; }
// acc += a b, real and imaginary parts each as one expression
template <typename T> __device__ inline void mac(T &acc, T a, T b)
{
  acc.x += a.x * b.x - a.y * b.y;
  acc.y += a.x * b.y + a.y * b.x;
}
__device__ inline void mac(double &acc, double a, double b) { acc += a * b; }
// conj(a) if cj (identity for real)
template <typename T> __device__ inline T conj_if(T a, bool cj) { if (cj) a.y = -a.y; return a; }
__device__ inline double conj_if(double a, bool) { return a; }
template <typename T> __device__ inline double re_of(T a) { return a.x; }
template <typename T> __device__ inline double im_of(T a) { return a.y; }
__device__ inline double re_of(double a) { return a; }
__device__ inline double im_of(double) { return 0; }
template <typename T> struct IsReal { static const bool v = false; };
template <> struct IsReal<double> { static const bool v = true; };

// Strides between the instances of a batch of equal-size factorizations:
// matrix elements (a), pivot entries (p) and bytes of each instance's
// panel scratch (s).  A single factorization is a batch of one, strides 0;
// batched kernels take the instance from blockIdx.y or blockIdx.z.
struct BStride {
  long a = 0, p = 0, s = 0;
};
template <typename P> __device__ inline P *bshift(P *p, long bytes)
{
  return p ? (P *)((char *)p + bytes) : p;
}

#define PW 32

struct PanelScratch {
  unsigned *bar;   // [64]: time-out word of the bounded waits
  int *plan;       // [4*PW+1]: dst rows [2*PW], src rows [2*PW], count of the panel's net row permutation
  void *linv;      // [npanels][PW][PW] T or null: inverse of each panel's unit-lower block (column-major)
  unsigned long long *ts;   // tournament-pivoting sets and root area (k_panel_ts), or null
  unsigned long long *xch;  // exchange area of k_panel_x: 2 sets of [PW][Gmax] slots, or null
  // the same scratch of the instance `bytes` further on (a batch's scratch
  // areas are equal and contiguous)
  __device__ inline PanelScratch shift(long bytes) const
  {
    PanelScratch o = *this;
    o.bar = bshift(bar, bytes);
    o.plan = bshift(plan, bytes); o.linv = bshift((char *)linv, bytes); o.ts = bshift(ts, bytes); o.xch = bshift(xch, bytes);
    return o;
  }
};


// Cross-workgroup exchange inside the panel without grid barriers: the
// shared words are read and written only by agent-scope relaxed atomics
// (coherent across the XCDs' L2s).  A writer waits for its data stores to
// complete (s_waitcnt) before it stores the flag that readers poll
// (tournament), or every word starts as a sentinel and is final once it
// differs (exact panel, solve chain).  No release/acquire fences, hence no L2 write-back or
// invalidation while the trailing GEMM runs beside the panel.
__device__ inline void st_coh(unsigned long long *p, unsigned long long v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline unsigned long long ld_coh(const unsigned long long *p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_coh(float2 *p, float2 v)
{
  unsigned long long u = ((unsigned long long)__float_as_uint(v.y) << 32) | __float_as_uint(v.x);
  st_coh((unsigned long long *)p, u);
}
__device__ inline float2 ld_coh(const float2 *p)
{
  unsigned long long u = ld_coh((const unsigned long long *)p);
  float2 v;
  v.x = __uint_as_float((unsigned)u);
  v.y = __uint_as_float((unsigned)(u >> 32));
  return v;
}
__device__ inline void st_coh(double2 *p, double2 v)
{
  st_coh((unsigned long long *)p, (unsigned long long)__double_as_longlong(v.x));
  st_coh((unsigned long long *)p + 1, (unsigned long long)__double_as_longlong(v.y));
}
__device__ inline void st_coh(double *p, double v)
{
  st_coh((unsigned long long *)p, (unsigned long long)__double_as_longlong(v));
}
__device__ inline double ld_coh(const double *p)
{
  return __longlong_as_double((long long)ld_coh((const unsigned long long *)p));
}
__device__ inline double2 ld_coh(const double2 *p)
{
  double2 v;
  v.x = __longlong_as_double((long long)ld_coh((const unsigned long long *)p));
  v.y = __longlong_as_double((long long)ld_coh((const unsigned long long *)p + 1));
  return v;
}
// polls before a wait gives up (about a second); the kernel then
// finishes and the host reports the time-out
#define GBAR_SPIN (1u << 20)
// keys one lane of the polling wave holds: up to 64 * 8 workgroups
#define KEYS_PER_LANE 8

// every memory operation this thread issued has completed; the signal
// fences keep the compiler from moving memory operations across it
__device__ inline void drain()
{
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// maximum of a 32-bit key over the wave, in every lane: within each row
// of 16 lanes by DPP (quad swaps, half-row and row mirrors), then over the
// four rows by lane reads (the result is wave-uniform).  All lanes active.
__device__ inline unsigned wave_max_key(unsigned k)
{
  k = max(k, (unsigned)__builtin_amdgcn_update_dpp(0, (int)k, 0xB1, 0xF, 0xF, false));    // quad_perm 1,0,3,2
  k = max(k, (unsigned)__builtin_amdgcn_update_dpp(0, (int)k, 0x4E, 0xF, 0xF, false));    // quad_perm 2,3,0,1
  k = max(k, (unsigned)__builtin_amdgcn_update_dpp(0, (int)k, 0x141, 0xF, 0xF, false));   // row_half_mirror
  k = max(k, (unsigned)__builtin_amdgcn_update_dpp(0, (int)k, 0x140, 0xF, 0xF, false));   // row_mirror
  const unsigned a = __builtin_amdgcn_readlane(k, 0), b = __builtin_amdgcn_readlane(k, 16);
  const unsigned c = __builtin_amdgcn_readlane(k, 32), d = __builtin_amdgcn_readlane(k, 48);
  return max(max(a, b), max(c, d));
}

// f(0), f(1), .. f(N - 1) with compile-time indices (a loop of this size is
// past the compiler's limit for unrolling, and a rolled one would index the
// row's registers, i.e. keep it in scratch memory)
template <int J, int N, typename F> __device__ __attribute__((always_inline)) inline void static_for(F &&f)
{
  if constexpr (J < N) {
    f(std::integral_constant<int, J>{});
    static_for<J + 1, N>(f);
  }
}

// slots of the exact panel's exchange area (lu_panel.inc): one per column
// and workgroup, 64-bit words {key, position, the candidate row}
template <typename T> struct XW;          // 64-bit words of one entry
template <> struct XW<double2> { static const int n = 2; };
template <> struct XW<double> { static const int n = 1; };
template <> struct XW<float2> { static const int n = 1; };
template <typename T> struct PXW { static const int n = 2 + PW * XW<T>::n; };   // words of one slot
#define PX_ONE 15
#define PX_SENT 0x7FF4DEADBEEF0005ULL

// the exact panel's kernel for up to PX_ONE workgroups (one) or any number:
// arguments (T *A, long lda, long r0, long m, int w, int *ipiv, int *info,
// PanelScratch S, int Gmax), one workgroup of 256 threads per 256 rows
template <typename T> const void *panel_x_kernel(bool one);
// the same for up to *rows rows, one workgroup of *rows threads: arguments
// (T *A, long lda, long r0, long m, int w, int *ipiv, int *info, PanelScratch S)
template <typename T> const void *panel_l_kernel(int *rows);

}  // namespace scuffx
