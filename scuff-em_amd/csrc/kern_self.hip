// kern_self.hip -- self (common-triangle) panel integrals by the
// generalized Taylor-Duffy method, every frequency.
//
// For a panel paired with itself the reference calls TaylorDuffy with
// P = {1, (x-Q).(x'-Q')}, the Helmholtz kernel e^{ikr}/4 pi r, and
// H0 = I_1 - 4 I_0/k^2, H1 = 0 (PanelPanelInteractions.cc:449-491).  The
// remaining 1-D integral is done by p-adaptive Clenshaw-Curtis
// quadrature, relative tolerance 1e-10, at most 1000 new points
// (TaylorDuffy.cc:152-367, libs/libSGJC/pcubature.c:323-385).
// One wave per (panel, region) job: the kernel values at a node serve all
// nine (Qa, Qb).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bem.h"
#include "exprel.h"

namespace scuffx {

#define TD_NWP 5
#define TD_MAXM 9            // 2^(9+1)+1 = 1025 nodes reached by MaxEval=1000
#define TD_NPRE 64           // cache entries computed up front, one per lane

__constant__ double c_ccx[512];            // nodes x_i, layout as the oracle
__constant__ double c_ccw[TD_MAXM + 1 + (1 << (TD_MAXM + 1))];

// common-triangle Upsilon coefficients (TaylorDuffy.cc:966-1057):
// U[d][n][0..2] = coefficients of 1, y, y^2; only M13,M14,M23,M24,V,S
// are non-zero for P in {1, PMCHWG1}.  Powers n outside the range that the
// sums take (below) are left zero.
struct CTPoly { double U[3][TD_NWP][3]; };

__device__ void ct_upsilon(double M13, double M14, double M23, double M24, double V1, double V2,
                           double V3, double V4, double S, CTPoly &P)
{
  const double M11 = 0, M12 = 0, M22 = 0, M33 = 0, M34 = 0, M44 = 0;
  for (int d = 0; d < 3; d++) for (int n = 0; n < TD_NWP; n++) for (int j = 0; j < 3; j++) P.U[d][n][j] = 0.0;
  double (*U)[TD_NWP][3] = P.U;
  U[0][0][0] = M11/4 + M12/4 + M13/2 + M14/4 + M22/12 + M23/4 + M24/6 + M33/4
               + M34/4 + M44/12 + (2*V1)/3 + V2/3 + (2*V3)/3 + V4/3 + S;
  U[0][1][1] = M12/3 + M14/3 + M22/6 + M23/3 + M24/3 + M34/3 + M44/6 + V2/2 + V4/2;
  U[0][1][0] = -(2*M11)/3 - (5*M12)/6 - (4*M13)/3 - (5*M14)/6 - M22/3 - (5*M23)/6
               - (2*M24)/3 - (2*M33)/3 - (5*M34)/6 - M44/3 - (3*V1)/2 - V2 - (3*V3)/2 - V4 - 2*S;
  U[0][2][2] = M22/4 + M44/4;
  U[0][2][1] = -M12/2 - M14 - M22/2 - M23 - M24 - M34/2 - M44/2 - V2 - V4;
  U[0][2][0] = (3*M11)/4 + M12 + M13 + M14 + M22/2 + M23 + M24 + (3*M33)/4 + M34 + M44/2
               + V1 + V2 + V3 + V4 + S;
  U[0][3][2] = -M22/2 - M44/2;
  U[0][3][1] = M14 + M22/2 + M23 + M24 + M44/2 + V2/2 + V4/2;
  U[0][3][0] = -M11/2 - M12/2 - M14/2 - M22/3 - M23/2 - (2*M24)/3 - M33/2 - M34/2 - M44/3
               - V1/6 - V2/3 - V3/6 - V4/3;
  U[0][4][2] = M22/4 + M44/4;
  U[0][4][1] = M12/6 - M14/3 - M22/6 - M23/3 - M24/3 + M34/6 - M44/6;
  U[0][4][0] = M11/6 + M12/12 - M13/6 + M14/12 + M22/12 + M23/12 + M24/6 + M33/6 + M34/12 + M44/12;

  U[1][0][0] = U[0][0][0];
  U[1][1][1] = -M11/3 - M12/2 - (2*M13)/3 - M14/2 - M22/6 - M23/2 - M24/3 - M33/3
               - M34/2 - M44/6 - V1/2 - V2/2 - V3/2 - V4/2;
  U[1][1][0] = -M11/3 - M12/3 - (2*M13)/3 - M14/3 - M22/6 - M23/3 - M24/3 - M33/3
               - M34/3 - M44/6 - 2*S - V1 - V2/2 - V3 - V4/2;
  U[1][2][2] = M11/4 + M12/2 + M22/4 + M33/4 + M34/2 + M44/4;
  U[1][2][1] = M11/2 + M12/2 + M13 + M14 + M23 + M24 + M33/2 + M34/2 + V1 + V2 + V3 + V4;
  U[1][2][0] = M22/4 + M44/4 + S;
  U[1][3][2] = -M11/2 - M12 - M22/2 - M33/2 - M34 - M44/2;
  U[1][3][1] = M12/2 - M14/2 + M22/2 - M23/2 - M24 + M34/2 + M44/2 - V1/2 - V2/2 - V3/2 - V4/2;
  U[1][3][0] = -M22/3 + M24/3 - M44/3 + V1/3 + V2/6 + V3/3 + V4/6;
  U[1][4][2] = M11/4 + M12/2 + M22/4 + M33/4 + M34/2 + M44/4;
  U[1][4][1] = -M11/6 - M12/2 - M13/3 - M22/3 + M24/3 - M33/6 - M34/2 - M44/3;
  U[1][4][0] = M11/12 + M12/12 + M13/6 + M14/12 + M22/6 + M23/12 - M24/6 + M33/12 + M34/12 + M44/6;

  U[2][0][0] = M11/4 + M12/4 + M13/2 + M14/4 + M22/12 + M23/4 + M24/6 + M33/4
               + M34/4 + M44/12 + S + (2*V1)/3 + V2/3 + (2*V3)/3 + V4/3;
  U[2][1][1] = -M11/3 - M12/6 - (2*M13)/3 - M14/6 - M23/6 - M33/3 - M34/6 - V1/2 - V3/2;
  U[2][1][0] = -M11/3 - M12/3 - (2*M13)/3 - M14/3 - M22/6 - M23/3 - M24/3 - M33/3 - M34/3
               - M44/6 - 2*S - V1 - V2/2 - V3 - V4/2;
  U[2][2][2] = M11/4 + M33/4;
  U[2][2][1] = M11/2 + M12/2 + M13 + M33/2 + M34/2 + V1 + V3;
  U[2][2][0] = M22/4 + M44/4 + S;
  U[2][3][2] = -M11/2 - M33/2;
  U[2][3][1] = -M12/2 + M14/2 + M23/2 - M34/2 - V1/2 - V3/2;
  U[2][3][0] = -M22/3 + M24/3 - M44/3 + V1/3 + V2/6 + V3/3 + V4/6;
  U[2][4][2] = M11/4 + M33/4;
  U[2][4][1] = -M11/6 + M12/6 - M13/3 - M14/3 - M23/3 - M33/6 + M34/6;
  U[2][4][0] = M11/12 + M12/12 + M13/6 + M14/12 + M22/6 + M23/12 - M24/6 + M33/12 + M34/12 + M44/6;

  // range of w-powers with a coefficient above 1e-8 (TaylorDuffy.cc:1507-1520)
  int nMin = TD_NWP - 1, nMax = -1;
  for (int n = 0; n < TD_NWP; n++)
    for (int d = 0; d < 3; d++)
      for (int j = 0; j < 3; j++)
        if (fabs(U[d][n][j]) > 1.0e-8) { if (n < nMin) nMin = n; if (n > nMax) nMax = n; }
  for (int n = 0; n < TD_NWP; n++)
    if (n < nMin || n > nMax)
      for (int d = 0; d < 3; d++)
        for (int j = 0; j < 3; j++) U[d][n][j] = 0.0;
}

// polynomial 0: P = 1, 1 + 3 qa + qb: PMCHWG1 of (Qa, Qb)
#define CT_NP 10
#define CT_NV (2 * CT_NP)                // real values of a node
struct CTJob { double A2, AdB, B2; CTPoly P[CT_NP]; cplx k; };

// integrand at y for all ten polynomials.  The job (J, in LDS) is shared by
// the wave; the kernel values K_n(X_d) = e^{ikX} ExpRel_n(-ikX) / (n X) of
// every power are formed once, from one sine, cosine and pair of
// exponentials a distance
__device__ inline void ct_integrand(const CTJob &J, double y, double *f)
{
#pragma clang fp contract(fast)
#pragma unroll
  for (int v = 0; v < CT_NV; v++) f[v] = 0.0;
  const cplx IK = IMUL(J.k);
#pragma unroll 1
  for (int d = 0; d < 3; d++) {
    const double u1 = d == 0 ? 1.0 : y, u2 = d == 0 ? y : d == 1 ? y - 1 : 1.0;
    const double X = sqrt(J.A2 * u1 * u1 + 2.0 * J.AdB * u1 * u2 + J.B2 * u2 * u2), iX = 1.0 / X;
    const cplx IKX = IK * X;
    double sn, cs;
    sincos(IKX.i, &sn, &cs);
    const double ep = exp(IKX.r), em = exp(-IKX.r);
    cplx ER[TD_NER];
    exprels(TD_NWP, -IKX, mk(em * cs, -(em * sn)), ER);
    const cplx e = mk(ep * cs * iX, ep * sn * iX);
    cplx K[TD_NWP];
#pragma unroll
    for (int n = 0; n < TD_NWP; n++) K[n] = (1.0 / (n + 1)) * cmulf(e, ER[n + 1]);
#pragma unroll
    for (int p = 0; p < CT_NP; p++)
#pragma unroll
      for (int n = 0; n < TD_NWP; n++) {
        const double c = J.P[p].U[d][n][0] + y * J.P[p].U[d][n][1];
        f[2 * p] += c * K[n].r;
        f[2 * p + 1] += c * K[n].i;
      }
  }
#pragma unroll
  for (int v = 0; v < CT_NV; v++) f[v] *= 1.0 / (4.0 * M_PI);
}

// weight of cache entry e in the Clenshaw-Curtis rule of the given order
// (entries: center, the pair at x0, then level l >= 1 pairs from 2^l + 1),
// 0 for entries of levels above the order; order < 0: one-point rule
__device__ inline double cc_weight(int e, int order)
{
  if (order < 0) return e == 0 ? 2.0 : 0.0;
  const double *w = c_ccw + order + (1 << order) - 1;
  if (e == 0) return w[0];
  if (e < 3) return w[1];
  const int l = 31 - __clz(e - 1);          // level of the entry
  if (l > order) return 0.0;
  const int nl = 1 << (l - 1);
  return w[1 + nl + ((e - (1 << l) - 1) >> 1)];
}

// node of cache entry e (entries as in cc_weight)
__device__ inline double cc_node(int e)
{
  if (e == 0) return 0.5;
  const int l = e < 3 ? 0 : 31 - __clz(e - 1), k = e < 3 ? e - 1 : e - (1 << l) - 1;
  const double x = c_ccx[(e < 3 ? 0 : 1 << (l - 1)) + (k >> 1)];
  return (k & 1) ? 0.5 - 0.5 * x : 0.5 + 0.5 * x;
}

// One wave per (panel, region) job.  The p-adaptive cubature of each (Qa,
// Qb) stops by itself (P = 1 and its PMCHWG1 within 1e-10 of the next lower
// order's, at most 1000 new points, as the reference does), but all nine
// read the same nodes, whose ten integrands share the kernel values.  The
// first TD_NPRE nodes, one per lane (orders 0 .. 4), come before the first
// test, order 5's last one if it is asked for; their sums are taken from LDS,
// a lane per order and value.  Later orders, if any, keep their nodes in a
// scratch slab.  Bound: latency of a job's kernel values and sums (0.3 to 1.1
// waves a SIMD; 7 to 30 % of the cycles issue vector instructions).  Bodies of
// N=7155: 0.61 ms an assembly, where a wave for each (Qa, Qb), with the
// exponentials of every power and polynomial its own, took 2.9
__global__ void __launch_bounds__(64)
k_self(const double *V, const int *PVI, int nP, int nreg, const RegionK *regs,
       double *HS, double *scratch, int njobs)
{
  const int lane = threadIdx.x;
  // the job's constants in LDS (read by every lane at the same address), the
  // node values, the sums of orders -1 .. 5
  __shared__ CTJob J;
  __shared__ double vals[TD_NPRE + 1][CT_NV + 1];
  __shared__ double S[7][CT_NV];
  for (int job = blockIdx.x; job < njobs; job += gridDim.x) {
    const int r = job % nreg, p = job / nreg;
    const double *V1 = V + 3 * PVI[3 * p], *V2 = V + 3 * PVI[3 * p + 1], *V3 = V + 3 * PVI[3 * p + 2];
    if (lane < CT_NP) {
      double A[3], B[3], D[3], DP[3];
      sub3(V2, V1, A); sub3(V3, V2, B);
      if (lane == 0) {
        J.A2 = dot3(A, A); J.AdB = dot3(A, B); J.B2 = dot3(B, B);
        J.k = regs[r].k;
        ct_upsilon(0, 0, 0, 0, 0, 0, 0, 0, 1.0, J.P[0]);
      } else {
        const int qa = (lane - 1) / 3, qb = (lane - 1) % 3;
        sub3(V1, V + 3 * PVI[3 * p + qa], D); sub3(V1, V + 3 * PVI[3 * p + qb], DP);
        ct_upsilon(dot3(A, A), dot3(A, B), dot3(B, A), dot3(B, B), dot3(A, DP), dot3(B, DP),
                   dot3(D, A), dot3(D, B), dot3(D, DP), J.P[lane]);
      }
    }
    __syncthreads();
    const double Vol = 0.5;
    double f[CT_NV];
    ct_integrand(J, cc_node(lane), f);
#pragma unroll
    for (int v = 0; v < CT_NV; v++) vals[lane][v] = f[v];
    __syncthreads();
    // sums of the orders lane / 20 and lane / 20 + 3 (up to 4 here)
    const int cv = lane % CT_NV, og = lane / CT_NV;
    auto rule = [&](int o) {
      double a = 0.0;
      const int ne = (1 << (o + 1)) + 1;
      for (int e = 0; e < ne; e++) a += vals[e][cv] * (cc_weight(e, o) * Vol);
      S[o + 1][cv] = a;
    };
    if (og < 3) {
      if (og == 0) S[0][cv] = vals[0][cv] * (2.0 * Vol);
      rule(og);
      if (og < 2) rule(og + 3);
    }
    __syncthreads();
    // lanes 0 .. 8: combination q; open: not converged yet
    const bool mine = lane < 9;
    const int q = mine ? lane : 0;
    bool open = mine;
    double R[4] = {0, 0, 0, 0};
    auto test = [&](int m) {
      if (!open) return;
      bool conv = true;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int v = c < 2 ? c : 2 * q + c;
        R[c] = S[m + 1][v];
        const double e = fabs(R[c] - S[m][v]);
        if (e > 0.0 && e > fabs(R[c]) * 1.0e-10) conv = false;
      }
      if (conv) open = false;
    };
    for (int m = 0; m <= 4; m++) test(m);
    if (__ballot(open)) {
      if (lane == 0) {
        ct_integrand(J, cc_node(TD_NPRE), f);
#pragma unroll
        for (int v = 0; v < CT_NV; v++) vals[TD_NPRE][v] = f[v];
      }
      __syncthreads();
      if (og == 0) rule(5);
      __syncthreads();
      test(5);
      double *slab = scratch + (long long)blockIdx.x * SCUFFX_SELF_SLAB;
      long numEval = 62;
      for (int m = 6; m <= TD_MAXM && numEval <= 1000 && __ballot(open); m++) {
        const int ne = (1 << (m + 1)) + 1;
        for (int e = (1 << m) + 1 + lane; e < ne; e += 64) {
          ct_integrand(J, cc_node(e), f);
#pragma unroll
          for (int v = 0; v < CT_NV; v++) slab[(long)(e - TD_NPRE - 1) * CT_NV + v] = f[v];
        }
        numEval += 1 << m;
        __syncthreads();
#pragma unroll
        for (int v = 0; v < CT_NV; v++) f[v] = 0.0;
        for (int e = lane; e < ne; e += 64) {
          const double w = cc_weight(e, m) * Vol;
          const double *x = e <= TD_NPRE ? &vals[e][0] : slab + (long)(e - TD_NPRE - 1) * CT_NV;
#pragma unroll
          for (int v = 0; v < CT_NV; v++) f[v] += x[v] * w;
        }
#pragma unroll
        for (int v = 0; v < CT_NV; v++) {
          for (int off = 32; off > 0; off >>= 1) f[v] += __shfl_xor(f[v], off);
          // (row 5: the order before, row 6: this one)
          if (lane == 0) { S[5][v] = S[6][v]; S[6][v] = f[v]; }
        }
        __syncthreads();
        test(5);
      }
    }
    if (mine) {
      const cplx I0 = mk(R[0], R[1]), I1 = mk(R[2], R[3]), k = J.k;
      const cplx H0 = I1 - 4.0 * I0 / (k * k);
      double *o = HS + ((long long)p * nreg + r) * 18 + 2 * q;
      o[0] = H0.r; o[1] = H0.i;
    }
    __syncthreads();   // the next job's constants overwrite this one's
  }
}

static_assert(SCUFFX_SELF_SLAB == ((2 << TD_MAXM) - TD_NPRE) * CT_NV, "scratch slab size");

static bool g_cc_ready[64] = {false};

hipError_t launch_self(hipStream_t stream, const double *V, const int *PVI, int nP, int nreg,
                       const RegionK *regs, double *HS, double *scratch)
{
  int dev = 0;
  hipGetDevice(&dev);
  if (!g_cc_ready[dev & 63]) {
    // Clenshaw-Curtis nodes and weights in the nested layout of
    // pcubature.c: x[0]=1; level m>=1 at offset 2^(m-1); weights of
    // rule order m (2^(m+1) intervals) at offset m+2^m-1:
    // [center, level-0 node, level-1 nodes, ...]
    static double hx[512], hw[TD_MAXM + 1 + (1 << (TD_MAXM + 1))];
    const long double pi = 3.141592653589793238462643383279502884L;
    hx[0] = 1.0;
    for (int m = 1; m <= TD_MAXM; m++)
      for (int i = 0; i < (1 << (m - 1)); i++)
        hx[(1 << (m - 1)) + i] = (double)cosl((2 * i + 1) * pi / (long double)(1L << (m + 1)));
    auto wt = [&](long n, long j) {
      long double s = 0;
      for (long k = 1; k <= n / 2; k++) {
        long double b = (k == n / 2) ? 1.0L : 2.0L;
        s += b / (4.0L * k * k - 1.0L) * cosl(2.0L * pi * (long double)((j * k) % n) / (long double)n);
      }
      long double cj = (j == 0 || j == n) ? 1.0L : 2.0L;
      return (double)(cj / (long double)n * (1.0L - s));
    };
    for (int m = 0; m <= TD_MAXM; m++) {
      long n = 1L << (m + 1);
      double *w = hw + m + (1 << m) - 1;
      w[0] = wt(n, n / 2);
      w[1] = wt(n, 0);
      int q = 2;
      for (int l = 1; l <= m; l++)
        for (int i = 0; i < (1 << (l - 1)); i++) w[q++] = wt(n, (2 * i + 1) * (n >> (l + 1)));
    }
    hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_ccx), hx, sizeof(hx));
    if (e != hipSuccess) return e;
    e = hipMemcpyToSymbol(HIP_SYMBOL(c_ccw), hw, sizeof(hw));
    if (e != hipSuccess) return e;
    g_cc_ready[dev & 63] = true;
  }
  const int njobs = nP * nreg;
  if (njobs <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_self, dim3(std::min(njobs, SCUFFX_SELF_SLABS)), dim3(64), 0, stream, V, PVI, nP, nreg, regs, HS,
                     scratch, njobs);
  return hipGetLastError();
}

}  // namespace scuffx
