// kern_grad.hip -- displacement derivatives of a BEM block between two
// distinct surfaces (GradM of AssembleBEMMatrixBlock).
//
// For every RWG pair the four panel-pair integrals are differentiated with
// respect to a rigid displacement of the row surface
// (PanelPanelInteractions.cc:132-199, :176-180):
//   dH0/dx_m = sum w w' R_m (F.F' + 4/(ik)^2) Psi
//   dH1/dx_m = sum w w' [R_m ((F x F').R) Zeta + (F x F')_m Psi]
// with Phi = e^{ikr}/4 pi r, Psi = Phi (ik - 1/r)/r,
// Zeta = Phi ((ik)^2 - 3ik/r + 3/r^2)/r^2, R = x - x'.  Panel pairs with
// relative distance > 4 use the 6-point rule, nearer ones the 78-point
// rule without desingularization, as the reference does when gradients
// are requested (:504-510).  The edge-pair combination and the region
// prefactors follow EdgeEdgeInteractions.cc:183-198 and
// SurfaceSurfaceInteractions.cc:212-327.
#include <hip/hip_runtime.h>

#include "bem.h"
#include "tcr20.inc"

namespace scuffx {

__constant__ double c_gtcr4[18] = SCUFFX_TCR4_INIT;
__constant__ double c_gtcr20[234];

#define SCUFFX_INV4PI_G 0.079577471545947667884

// gradient of one panel-pair integral: G[2m] (H0 part), G[2m+1] (H1 part);
// angular derivatives about the GS.n axes: T[2t], T[2t+1]
// (PanelPanelInteractions.cc:182-199: dX = Gamma X, dF = Gamma F,
//  dH0 += hPlus (R.dX) Psi + (dF.F') Phi,
//  dH1 += hTimes (R.dX) Zeta + ((dF x F').R + (F x F').dX) Psi)
__device__ void ppi_grad(const double *Va0, const double *Va1, const double *Va2, const double *Qa,
                         const double *Vb0, const double *Vb1, const double *Vb2, const double *Qb,
                         cplx k, int high, const GammaSet &GS, cplx G[6], cplx T[6])
{
  double A[3], B[3], AP[3], BP[3];
  sub3(Va1, Va0, A); sub3(Va2, Va0, B);
  sub3(Vb1, Vb0, AP); sub3(Vb2, Vb0, BP);
  const double *rule = high ? c_gtcr20 : c_gtcr4;
  const int np = high ? 78 : 6;
  cplx ik = IMUL(k), ik2 = ik * ik, c4 = 4.0 / ik2;
  for (int m = 0; m < 6; m++) { G[m] = mk(0, 0); T[m] = mk(0, 0); }
  const int ntq = GS.n;
  for (int i = 0; i < np; i++) {
    const double u = rule[3 * i], v = rule[3 * i + 1], w = rule[3 * i + 2];
    double X[3], F[3];
    for (int c = 0; c < 3; c++) { X[c] = Va0[c] + u * A[c] + v * B[c]; F[c] = X[c] - Qa[c]; }
    // rotated position and source vector of the outer point, per axis
    double dX[3][3], dF[3][3];
    for (int t = 0; t < ntq; t++)
      for (int m = 0; m < 3; m++) {
        dX[t][m] = 0; dF[t][m] = 0;
        for (int q = 0; q < 3; q++) {
          dX[t][m] += GS.g[9 * t + m + 3 * q] * X[q];
          dF[t][m] += GS.g[9 * t + m + 3 * q] * F[q];
        }
      }
    cplx GI[6], TI[6];
    for (int m = 0; m < 6; m++) { GI[m] = mk(0, 0); TI[m] = mk(0, 0); }
    for (int j = 0; j < np; j++) {
      const double up = rule[3 * j], vp = rule[3 * j + 1], wp = rule[3 * j + 2];
      double FP[3], R[3];
      for (int c = 0; c < 3; c++) {
        double XP = Vb0[c] + up * AP[c] + vp * BP[c];
        FP[c] = XP - Qb[c];
        R[c] = X[c] - XP;
      }
      double r2 = R[0] * R[0] + R[1] * R[1] + R[2] * R[2], r = sqrt(r2), ir = 1.0 / r;
      // (real and imaginary wavenumbers skip the exponential or the sine and
      // cosine: exact there)
      double e = 1.0, sn = 0.0, cs = 1.0;
      if (k.i != 0) e = exp(-k.i * r);
      if (k.r != 0) sincos(k.r * r, &sn, &cs);
      cplx Phi = mk(e * cs, e * sn) * (SCUFFX_INV4PI_G * ir * wp);
      cplx Psi = Phi * (ik - mk(ir, 0)) * ir;
      cplx Zeta = Phi * (ik2 - 3.0 * ir * ik + mk(3.0 * ir * ir, 0)) * (ir * ir);
      double FxFP[3];
      cross3(F, FP, FxFP);
      cplx hPlus = mk(F[0] * FP[0] + F[1] * FP[1] + F[2] * FP[2], 0) + c4;
      double hTimes = FxFP[0] * R[0] + FxFP[1] * R[1] + FxFP[2] * R[2];
      cplx hPsi = hPlus * Psi, tZeta = hTimes * Zeta;
      for (int m = 0; m < 3; m++) {
        GI[2 * m] += R[m] * hPsi;
        GI[2 * m + 1] += R[m] * tZeta + FxFP[m] * Psi;
      }
      for (int t = 0; t < ntq; t++) {
        double Puv = R[0] * dX[t][0] + R[1] * dX[t][1] + R[2] * dX[t][2];
        double dFFP = dF[t][0] * FP[0] + dF[t][1] * FP[1] + dF[t][2] * FP[2];
        double dFxFP[3];
        cross3(dF[t], FP, dFxFP);
        double c1 = dFxFP[0] * R[0] + dFxFP[1] * R[1] + dFxFP[2] * R[2]
                    + FxFP[0] * dX[t][0] + FxFP[1] * dX[t][1] + FxFP[2] * dX[t][2];
        TI[2 * t] += Puv * hPsi + dFFP * Phi;
        TI[2 * t + 1] += Puv * tZeta + c1 * Psi;
      }
    }
    for (int m = 0; m < 6; m++) { G[m] += w * GI[m]; T[m] += w * TI[m]; }
  }
}

// one thread per (ea, eb) of the block; GB holds three column-major
// NBF_a x NBF_b matrices (leading dimension ldg, gstride elements apart),
// overwritten
__global__ void __launch_bounds__(128)
k_grad_stamp(int nEa, const int *EIa, const double *ELa, const double *Va, const int *PVIa, const double *PCa,
             int nEb, const int *EIb, const double *ELb, const double *Vb, const int *PVIb, const double *PCb,
             int pecA, int pecB, int nreg, const RegionK *regs, double2 *GB, long ldg, long gstride,
             GammaSet GS, double2 *TB)
{
  int ea = blockIdx.x * blockDim.x + threadIdx.x;
  int eb = blockIdx.y;
  if (ea >= nEa || eb >= nEb) return;
  int pA[2] = {EIa[4 * ea], EIa[4 * ea + 1]}, qA[2] = {EIa[4 * ea + 2], EIa[4 * ea + 3]};
  int pB[2] = {EIb[4 * eb], EIb[4 * eb + 1]}, qB[2] = {EIb[4 * eb + 2], EIb[4 * eb + 3]};
  double LL = ELa[ea] * ELb[eb];
  const int nd = 3 + GS.n;           // displacement components, then axes
  cplx m00[6], m01[6], m11[6];
  for (int m = 0; m < 6; m++) { m00[m] = mk(0, 0); m01[m] = mk(0, 0); m11[m] = mk(0, 0); }
  for (int r = 0; r < nreg; r++) {
    cplx k = regs[r].k;
    cplx S0[6], S1[6];
    for (int m = 0; m < 6; m++) { S0[m] = mk(0, 0); S1[m] = mk(0, 0); }
    for (int s = 0; s < 2; s++)
      for (int t = 0; t < 2; t++) {
        if (pA[s] < 0 || pB[t] < 0) continue;
        const int pa = pA[s], pb = pB[t];
        const double *a0 = Va + 3 * PVIa[3 * pa], *a1 = Va + 3 * PVIa[3 * pa + 1], *a2 = Va + 3 * PVIa[3 * pa + 2];
        const double *b0 = Vb + 3 * PVIb[3 * pb], *b1 = Vb + 3 * PVIb[3 * pb + 1], *b2 = Vb + 3 * PVIb[3 * pb + 2];
        const double *Qa = Va + 3 * PVIa[3 * pa + qA[s]], *Qb = Vb + 3 * PVIb[3 * pb + qB[t]];
        // relative centroid distance (AssessPanelPair.cc:161-166)
        double dc[3] = {PCa[4 * pa] - PCb[4 * pb], PCa[4 * pa + 1] - PCb[4 * pb + 1], PCa[4 * pa + 2] - PCb[4 * pb + 2]};
        double rRel = sqrt(dc[0] * dc[0] + dc[1] * dc[1] + dc[2] * dc[2]) / fmax(PCa[4 * pa + 3], PCb[4 * pb + 3]);
        cplx G[6], TT[6];
        ppi_grad(a0, a1, a2, Qa, b0, b1, b2, Qb, k, rRel > 4.0 ? 0 : 1, GS, G, TT);
        double sg = ((s + t) & 1) ? -1.0 : 1.0;
        for (int m = 0; m < 3; m++) { S0[m] += sg * G[2 * m]; S1[m] += sg * G[2 * m + 1]; }
        for (int q = 0; q < GS.n; q++) { S0[3 + q] += sg * TT[2 * q]; S1[3 + q] += sg * TT[2 * q + 1]; }
      }
    cplx cpre = mk(LL, 0) / IMUL(k);
    for (int m = 0; m < nd; m++) {
      cplx g0 = LL * S0[m], g1 = cpre * S1[m];
      m00[m] += regs[r].pf1 * g0;
      m01[m] += regs[r].pf2 * g1;
      m11[m] += regs[r].pf3 * g0;
    }
  }
  for (int m = 0; m < nd; m++) {
    double2 *T = (m < 3) ? GB + (long)m * gstride : TB + (long)(m - 3) * gstride;
    if (pecA && pecB) {
      T[ea + (long)eb * ldg] = make_double2(m00[m].r, m00[m].i);
    } else if (pecA) {
      T[ea + (long)(2 * eb) * ldg] = make_double2(m00[m].r, m00[m].i);
      T[ea + (long)(2 * eb + 1) * ldg] = make_double2(m01[m].r, m01[m].i);
    } else if (pecB) {
      T[2 * ea + (long)eb * ldg] = make_double2(m00[m].r, m00[m].i);
      T[2 * ea + 1 + (long)eb * ldg] = make_double2(m01[m].r, m01[m].i);
    } else {
      long x = 2 * ea, y = 2 * eb;
      T[x + y * ldg] = make_double2(m00[m].r, m00[m].i);
      T[(x + 1) + y * ldg] = make_double2(m01[m].r, m01[m].i);
      T[x + (y + 1) * ldg] = make_double2(m01[m].r, m01[m].i);
      T[(x + 1) + (y + 1) * ldg] = make_double2(m11[m].r, m11[m].i);
    }
  }
}

// Between perfectly conducting surfaces only dH0 is wanted, and a panel pair's
// integrals serve the nine edge pairs that meet it.  With x, y from the
// panels' centroids, R = D + x - y,
//   dH0/dx_m (Qa, Qb) = A_m - Qb.B_m - Qa.C_m + (Qa.Qb + 4/(ik)^2) E_m,
//   A_m = sum R_m (x.y) Psi, B_m = sum R_m x Psi, C_m = sum R_m y Psi,
//   E_m = sum R_m Psi,
// and the sums over y for one x need sum {1, y, y y} Psi only (ten words).
// One thread per (row panel, slot) writes the 9 x 3 values of each region; the
// band's column edges are then combined from them, as the matrix is.  Bound:
// FP64 vector issue at one wave a SIMD (50 % of the cycles, 16 TFLOP/s).  Two N=1920 spheres: under 0.9 ms, where each edge pair
// integrated its four panel pairs by itself in 8.7.
__global__ void __launch_bounds__(128)
k_grad_pair(const double *Va, const int *PVIa, const double *PCa, int nPa, const double *Vb, const int *PVIb,
            const double *PCb, const int *slotPanels, int nreg, const RegionK *regs, double *HB, long rowsCap)
{
#pragma clang fp contract(fast)
  const int pa = blockIdx.x * blockDim.x + threadIdx.x, slot = blockIdx.y;
  if (pa >= nPa) return;
  const int pb = slotPanels[slot];
  double Pa[9], Pb[9], D[3];            // vertices from the centroids
  for (int c = 0; c < 3; c++) {
    for (int v = 0; v < 3; v++) {
      Pa[3 * v + c] = Va[3 * PVIa[3 * pa + v] + c] - PCa[4 * pa + c];
      Pb[3 * v + c] = Vb[3 * PVIb[3 * pb + v] + c] - PCb[4 * pb + c];
    }
    D[c] = PCa[4 * pa + c] - PCb[4 * pb + c];
  }
  // relative centroid distance (AssessPanelPair.cc:161-166)
  const double rRel = sqrt(D[0] * D[0] + D[1] * D[1] + D[2] * D[2]) / fmax(PCa[4 * pa + 3], PCb[4 * pb + 3]);
  const double *rule = rRel > 4.0 ? c_gtcr4 : c_gtcr20;
  const int np = rRel > 4.0 ? 6 : 78;
  for (int r = 0; r < nreg; r++) {
    const cplx k = regs[r].k;
    cplx A[3], B[3][3], C[3][3], E[3];
    for (int m = 0; m < 3; m++) {
      A[m] = mk(0, 0); E[m] = mk(0, 0);
      for (int c = 0; c < 3; c++) { B[m][c] = mk(0, 0); C[m][c] = mk(0, 0); }
    }
#pragma unroll 1
    for (int i = 0; i < np; i++) {
      const double u = rule[3 * i], v = rule[3 * i + 1], w = rule[3 * i + 2] * SCUFFX_INV4PI_G;
      double x[3], Dx[3];
      for (int c = 0; c < 3; c++) {
        x[c] = Pa[c] + u * (Pa[3 + c] - Pa[c]) + v * (Pa[6 + c] - Pa[c]);
        Dx[c] = D[c] + x[c];
      }
      cplx q0 = mk(0, 0), q[3], Q[6];     // Q: xx, yy, zz, xy, xz, yz
      for (int c = 0; c < 3; c++) q[c] = mk(0, 0);
      for (int c = 0; c < 6; c++) Q[c] = mk(0, 0);
#pragma unroll 1
      for (int j = 0; j < np; j++) {
        const double up = rule[3 * j], vp = rule[3 * j + 1];
        double y[3], R[3];
        for (int c = 0; c < 3; c++) {
          y[c] = Pb[c] + up * (Pb[3 + c] - Pb[c]) + vp * (Pb[6 + c] - Pb[c]);
          R[c] = Dx[c] - y[c];
        }
        const double rr = sqrt(R[0] * R[0] + R[1] * R[1] + R[2] * R[2]), ir = 1.0 / rr;
        double e = rule[3 * j + 2] * ir, sn = 0.0, cs = 1.0;
        if (k.i != 0) e *= exp(-k.i * rr);
        if (k.r != 0) sincos(k.r * rr, &sn, &cs);
        // Psi = Phi (ik - 1/r) / r
        const double a = -(k.i + ir) * ir, b = k.r * ir, fr = e * cs, fi = e * sn;
        const cplx g = mk(fr * a - fi * b, fr * b + fi * a);
        q0 += g;
        for (int c = 0; c < 3; c++) q[c] += y[c] * g;
        Q[0] += (y[0] * y[0]) * g; Q[1] += (y[1] * y[1]) * g; Q[2] += (y[2] * y[2]) * g;
        Q[3] += (y[0] * y[1]) * g; Q[4] += (y[0] * y[2]) * g; Q[5] += (y[1] * y[2]) * g;
      }
      for (int m = 0; m < 3; m++) {
        const cplx N = w * (Dx[m] * q0 - q[m]);
        E[m] += N;
        for (int c = 0; c < 3; c++) {
          const cplx M = w * (Dx[m] * q[c] - Q[c == m ? c : c + m + 2]);
          A[m] += x[c] * M;
          B[m][c] += x[c] * N;
          C[m][c] += M;
        }
      }
    }
    const cplx ik = IMUL(k), c4 = 4.0 / (ik * ik);
    double *out = HB + (((long)slot * rowsCap + pa) * nreg + r) * 54;
    for (int a = 0; a < 3; a++)
      for (int b = 0; b < 3; b++) {
        const double *qa = Pa + 3 * a, *qb = Pb + 3 * b;
        const cplx qq = mk(dot3(qa, qb), 0) + c4;
        for (int m = 0; m < 3; m++) {
          cplx h = A[m] + qq * E[m];
          for (int c = 0; c < 3; c++) h = h - qb[c] * B[m][c] - qa[c] * C[m][c];
          double *o = out + (3 * (3 * a + b) + m) * 2;
          o[0] = h.r; o[1] = h.i;
        }
      }
  }
}

// the band's column edges from its records: grid.y = column edge
__global__ void __launch_bounds__(256)
k_grad_comb(int nEa, const int *EIa, const double *ELa, const int *bandCols, const int *colSlots, const int *EIb,
            const double *ELb, int nreg, const RegionK *regs, const double *HB, long rowsCap, double2 *GB, long ldg,
            long gstride)
{
  const int ea = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  if (ea >= nEa) return;
  const int eb = bandCols[j];
  const double LL = ELa[ea] * ELb[eb];
  cplx m00[3] = {mk(0, 0), mk(0, 0), mk(0, 0)};
  for (int r = 0; r < nreg; r++) {
    cplx S[3] = {mk(0, 0), mk(0, 0), mk(0, 0)};
#pragma unroll
    for (int st = 0; st < 4; st++) {
      const int s = st >> 1, t = st & 1;
      const int pa = EIa[4 * ea + s], pb = EIb[4 * eb + t];
      if (pa < 0 || pb < 0) continue;
      const int q = 3 * EIa[4 * ea + 2 + s] + EIb[4 * eb + 2 + t];
      const double *h = HB + (((long)colSlots[2 * j + t] * rowsCap + pa) * nreg + r) * 54 + 6 * q;
      const double sg = s == t ? 1.0 : -1.0;
      for (int m = 0; m < 3; m++) S[m] += sg * mk(h[2 * m], h[2 * m + 1]);
    }
    for (int m = 0; m < 3; m++) m00[m] += regs[r].pf1 * (LL * S[m]);
  }
  for (int m = 0; m < 3; m++) GB[(long)m * gstride + ea + (long)eb * ldg] = make_double2(m00[m].r, m00[m].i);
}

static bool g_gtcr20_ready[64] = {false};

static hipError_t grad_tables()
{
  int dev = 0;
  hipGetDevice(&dev);
  if (!g_gtcr20_ready[dev & 63]) {
    hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_gtcr20), scuffx_tcr20, sizeof(scuffx_tcr20));
    if (e != hipSuccess) return e;
    g_gtcr20_ready[dev & 63] = true;
  }
  return hipSuccess;
}

hipError_t launch_grad_band(hipStream_t stream, int nEa, const int *EIa, const double *ELa, const double *Va,
                            const int *PVIa, const double *PCa, int nPa, const int *EIb, const double *ELb,
                            const double *Vb, const int *PVIb, const double *PCb, const int *slotPanels, int nslots,
                            const int *bandCols, const int *colSlots, int ncols, int nreg, const RegionK *regs,
                            double *HB, long rowsCap, double2 *GB, long ldg, long gstride)
{
  if (nPa <= 0 || nslots <= 0 || ncols <= 0 || nEa <= 0) return hipSuccess;
  hipError_t e = grad_tables();
  if (e != hipSuccess) return e;
  if (nreg > 0)
    hipLaunchKernelGGL(k_grad_pair, dim3((nPa + 127) / 128, nslots), dim3(128), 0, stream, Va, PVIa, PCa, nPa, Vb, PVIb,
                       PCb, slotPanels, nreg, regs, HB, rowsCap);
  hipLaunchKernelGGL(k_grad_comb, dim3((nEa + 255) / 256, ncols), dim3(256), 0, stream, nEa, EIa, ELa, bandCols,
                     colSlots, EIb, ELb, nreg, regs, HB, rowsCap, GB, ldg, gstride);
  return hipGetLastError();
}

hipError_t launch_grad(hipStream_t stream, int nEa, const int *EIa, const double *ELa, const double *Va,
                       const int *PVIa, const double *PCa, int nEb, const int *EIb, const double *ELb,
                       const double *Vb, const int *PVIb, const double *PCb, int pecA, int pecB, int nreg,
                       const RegionK *regs, double2 *GB, long ldg, long gstride, const GammaSet &GS,
                       double2 *TB)
{
  hipError_t e = grad_tables();
  if (e != hipSuccess) return e;
  if (nEa <= 0 || nEb <= 0) return hipSuccess;
  dim3 grid((nEa + 127) / 128, nEb);
  hipLaunchKernelGGL(k_grad_stamp, grid, dim3(128), 0, stream, nEa, EIa, ELa, Va, PVIa, PCa, nEb, EIb, ELb, Vb,
                     PVIb, PCb, pecA, pecB, nreg, regs, GB, ldg, gstride, GS, TB);
  return hipGetLastError();
}

}  // namespace scuffx
