// dg_line.hpp -- whole runs of small 1-D Euler meshes (with or without artificial viscosity) in one launch.
//
// A step of a few hundred line elements is a chain of ten launches whose kernels each wait for a few
// loads: 57 us a step, of which the arithmetic is a few per cent. Here one workgroup owns the mesh, one
// thread an element. The state stays in registers for all steps of the call, traces and normal
// artificial fluxes cross to the neighbours through LDS, and a stage costs two workgroup barriers.
// Bound by the latency of a thread's own chain of FP64 operations: 200 elements P2 with artificial
// viscosity take 27 us a step.
#ifndef SDG_DG_LINE_HPP_
#define SDG_DG_LINE_HPP_

#include <hip/hip_runtime.h>

#include "dg_kernels.hpp"

namespace sdg {

// elements of the largest mesh: eight wavefronts of 256 registers, one workgroup on one CU
constexpr int kLineMaxElements = 512;
// steps of one launch: longer calls take several, so that no kernel holds a CU for long
constexpr int kLineMaxSteps = 4096;

struct LineRun {
  double* U;        // state at the start and, replaced, at the end
  double* Uf;       // traces of the final state
  double* nodeav;   // artificial viscosity of the last step's start (null without)
  double* rel;      // monitor of the last step
  int* status;      // [0] NaN stop flag, [1] steps taken (both zeroed by the caller)
  double c0[3], c1[3], c2dt[3];
  int stages, nsteps;
};

template <int N, bool AV>
__global__ __launch_bounds__(kLineMaxElements) void lineRunKernel(Geo g, Phys ph, LineRun a) {
  constexpr int NV = 3, M = kLineMaxElements;
  __shared__ double sT[AV ? 1 : 2][2][NV][M];  // [buffer][side][variable][element] traces
  __shared__ double sV[AV ? 2 : 1][NV][AV ? M : 1];  // normal artificial fluxes
  __shared__ unsigned long long sE[AV ? M : 1];      // element viscosities (bits)
  __shared__ double red[NV][M / 64];
  __shared__ int sNan;
  const TensorOps& t = g.tens;
  const int e = threadIdx.x;
  const bool ok = e < g.E;
  const int ec = ok ? e : 0;
  if (a.status[0]) return;  // stopped by an earlier launch of the same call
  if (e == 0) sNan = 0;
  // geometry, neighbours (slot s: side lofs[s] of the element)
  const double dj = g.detj[ec], gi = g.ginv[ec], idj = 1.0 / dj;
  int nb[2], side[2];
  double nrm[2], jw[2];
#pragma unroll
  for (int s = 0; s < 2; s++) {
    nb[s] = g.snb[ec * 2 + s];
    side[s] = g.sfp[ec * 2 + s] & 1;
    nrm[s] = g.egeo[(ec * 2 + s) * 2];
    jw[s] = g.egeo[(ec * 2 + s) * 2 + 1];
  }
  // end points: lf row of slot s
  const int end0 = t.side[0], end1 = t.side[1];
  int share[2] = {-1, -1}, tag[2] = {0, 0};  // the element that shares vertex j
  double top = 0.0;
  if constexpr (AV) {
    top = ph.av_factor * (g.inrad[ec] / static_cast<double>(g.order));
    for (int j = 0; j < 2; j++) {
      tag[j] = g.ntag[ec * 2 + j];
      for (int s = 0; s < 2; s++)
        if (nb[s] >= 0) {
          const int m = nb[s] / 2;
          if (g.ntag[m * 2] == tag[j] || g.ntag[m * 2 + 1] == tag[j]) share[j] = m;
        }
    }
  }
  double um[NV][N], u0[NV][N], iw[N];
#pragma unroll
  for (int i = 0; i < N; i++) iw[i] = 1.0 / t.w[i];
#pragma unroll
  for (int v = 0; v < NV; v++)
#pragma unroll
    for (int k = 0; k < N; k++) um[v][k] = a.U[(ec * NV + v) * N + k];
  double R[NV][N];
  int taken = 0;
#pragma unroll 1
  for (int step = 0; step < a.nsteps; step++) {
    double av[2] = {0.0, 0.0};  // node viscosities of the two vertices
    if constexpr (AV) {  // the sensor of avSensorKernel
      double num = 0.0, den = 0.0;
#pragma unroll
      for (int i = 0; i < N; i++) {
        double all = 0.0, high = 0.0;
#pragma unroll
        for (int k = 0; k < N; k++) {
          const double x = t.B[i * N + k] * um[0][k];
          all += x;
          if (k >= ph.av_low) high += x;
        }
        const double w = dj * t.w[i];
        num += high * (high * w);
        den += all * (all * w);
      }
      const double s = log10(num / den);
      double eps;
      if (s < ph.av_s0 - ph.av_tol)
        eps = 0.0;
      else if (s > ph.av_s0 + ph.av_tol)
        eps = top;
      else
        eps = top * (1.0 + sin(3.14159265358979323846 * (s - ph.av_s0) / (2.0 * ph.av_tol))) / 2.0;
      const unsigned long long bits = static_cast<unsigned long long>(__double_as_longlong(eps));
      if (ok) sE[e] = bits;
      __syncthreads();
#pragma unroll
      for (int j = 0; j < 2; j++) {
        unsigned long long b = bits;
        if (share[j] >= 0) b = sE[share[j]] > b ? sE[share[j]] : b;
        av[j] = __longlong_as_double(static_cast<long long>(b));
      }
    } else {
      __syncthreads();  // sNan of the step before
    }
    if (sNan == (1 << NV) - 1) break;
#pragma unroll
    for (int v = 0; v < NV; v++)
#pragma unroll
      for (int k = 0; k < N; k++) u0[v][k] = um[v][k];
#pragma unroll 1
    for (int st = 0; st < a.stages; st++) {
      const int buf = AV ? 0 : (step * a.stages + st) & 1;
      double u[NV][N], to[2][NV], tn[2][NV];
#pragma unroll
      for (int v = 0; v < NV; v++) {
#pragma unroll
        for (int i = 0; i < N; i++) {
          double s = 0.0;
#pragma unroll
          for (int k = 0; k < N; k++) s += t.B[i * N + k] * um[v][k];
          u[v][i] = s;
        }
#pragma unroll
        for (int s = 0; s < 2; s++) {
          const int row = (s == 0 ? end0 : end1) * N;
          double x = 0.0;
#pragma unroll
          for (int i = 0; i < N; i++) x += t.lf[row + i] * u[v][i];
          to[s][v] = x;
          if (ok) sT[buf][s][v][e] = x;
        }
      }
      __syncthreads();
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int v = 0; v < NV; v++) tn[s][v] = nb[s] >= 0 ? sT[buf][nb[s] & 1][v][nb[s] >> 1] : to[s][v];
      double gr[AV ? NV : 1][AV ? N : 1], vo[2][NV];
      if constexpr (AV) {  // volume gradient at the nodes, eps grad u . n at the faces
        double al[2][NV];
#pragma unroll
        for (int s = 0; s < 2; s++) {
          if (nb[s] >= 0) {
#pragma unroll
            for (int v = 0; v < NV; v++) al[s][v] = ((tn[s][v] - to[s][v]) / 2.0) * jw[s];
          } else {
            const int bp = -1 - nb[s];
            double wd[4], uvg[NV], uig[NV];
            for (int i = 0; i < 4; i++) wd[i] = g.bdata[bp * 4 + i];
            boundaryGradientStates<1>(ph, g.btype[bp], &nrm[s], to[s], wd, uvg, uig);
            for (int v = 0; v < NV; v++) al[s][v] = (uvg[v] - to[s][v]) * jw[s];
          }
        }
#pragma unroll
        for (int i = 0; i < N; i++) {
          const double inw = idj * iw[i];
#pragma unroll
          for (int v = 0; v < NV; v++) {
            double s = 0.0;
#pragma unroll
            for (int m = 0; m < N; m++) s += t.Dn[i * N + m] * u[v][m];
            gr[v][i] = gi * s + (t.lf[end0 * N + i] * al[0][v] * nrm[0] + t.lf[end1 * N + i] * al[1][v] * nrm[1]) * inw;
          }
        }
#pragma unroll
        for (int s = 0; s < 2; s++) {
          const int row = (s == 0 ? end0 : end1) * N;
          const double eps = g.nodf[s * 2] * av[0] + g.nodf[s * 2 + 1] * av[1];
#pragma unroll
          for (int v = 0; v < NV; v++) {
            double x = 0.0;
#pragma unroll
            for (int i = 0; i < N; i++) x += t.lf[row + i] * gr[v][i];
            vo[s][v] = eps * (x * nrm[s]);
            if (ok) sV[s][v][e] = vo[s][v];
          }
        }
        __syncthreads();
      }
      // volume flux, weak divergence against the modal basis (R: the reference residual)
#pragma unroll
      for (int v = 0; v < NV; v++)
#pragma unroll
        for (int i = 0; i < N; i++) R[v][i] = 0.0;
#pragma unroll
      for (int m = 0; m < N; m++) {
        double x[NV], w[4], f[NV];
        for (int v = 0; v < NV; v++) x[v] = u[v][m];
        computational<1>(ph, x, w);
        const double et = w[2] + w[1] * w[1] / 2.0;
        f[0] = w[0] * w[1];
        f[1] = w[0] * w[1] * w[1] + w[3];
        f[2] = (w[0] * et + w[3]) * w[1];
        const double G = gi * (dj * t.w[m]);
        if constexpr (AV) {
          const double eps = t.nodt[m * 2] * av[0] + t.nodt[m * 2 + 1] * av[1];
#pragma unroll
          for (int v = 0; v < NV; v++) f[v] -= eps * gr[v][m];
        }
#pragma unroll
        for (int v = 0; v < NV; v++)
#pragma unroll
          for (int b = 0; b < N; b++) R[v][b] += g.dV[m * N + b] * (f[v] * G);
      }
      // numerical fluxes of the two end points with the face's left / right roles
#pragma unroll 1
      for (int s = 0; s < 2; s++) {
        double h[NV], uo[NV], un[NV], vs[NV];
        for (int v = 0; v < NV; v++) {
          uo[v] = s == 0 ? to[0][v] : to[1][v];
          un[v] = s == 0 ? tn[0][v] : tn[1][v];
          vs[v] = AV ? (s == 0 ? vo[0][v] : vo[1][v]) : 0.0;
        }
        const double n = s == 0 ? nrm[0] : nrm[1], w = s == 0 ? jw[0] : jw[1];
        const int nbs = s == 0 ? nb[0] : nb[1], sd = s == 0 ? side[0] : side[1];
        if (nbs < 0) {
          boundaryFlux<1, false>(ph, g, -1 - nbs, uo, nullptr, false, 0.0, 0.0, h);
          for (int v = 0; v < NV; v++) h[v] = vs[v] * w - h[v];
        } else {
          double ul[NV], ur[NV], wl[4], wr[4];
          for (int v = 0; v < NV; v++) {
            ul[v] = sd == 0 ? uo[v] : un[v];
            ur[v] = sd == 0 ? un[v] : uo[v];
          }
          const double nl = sd == 0 ? n : -n;
          computational<1>(ph, ul, wl);
          computational<1>(ph, ur, wr);
          convectiveFlux<1>(ph, &nl, ul, wl, ur, wr, h);
          for (int v = 0; v < NV; v++) {
            double x = h[v];
            if constexpr (AV) {
              const double vn = sV[nbs & 1][v][nbs >> 1];
              x -= sd == 0 ? (vs[v] - vn) / 2.0 : (vn - vs[v]) / 2.0;
            }
            x *= w;
            h[v] = sd == 0 ? -x : x;
          }
        }
#pragma unroll
        for (int v = 0; v < NV; v++)
#pragma unroll
          for (int b = 0; b < N; b++) R[v][b] += g.Vf[s * N + b] * h[v];
      }
      // The monitor's NaN test on the modes: an infinite flux at an end point meets the exact zero of the
      // other end's mode, one inside makes the two end modes of opposite infinities, so that their sum is
      // NaN where a node's value is.
      if (st == a.stages - 1) {
        int bad = 0;
        for (int v = 0; v < NV; v++) {
          double s = 0.0;
          for (int i = 0; i < N; i++) s += R[v][i];
          bad |= isnan(s) ? 1 << v : 0;
        }
        if (ok && bad) atomicOr(&sNan, bad);
      }
      // RK update
#pragma unroll
      for (int v = 0; v < NV; v++) {
#pragma unroll
        for (int k = 0; k < N; k++) {
          double s = 0.0;
#pragma unroll
          for (int b = 0; b < N; b++) s += R[v][b] * g.Minv[b * N + k];
          double x = um[v][k] * a.c1[st];
          x += a.c0[st] * u0[v][k];
          um[v][k] = x + a.c2dt[st] * (s * idj);
        }
      }
    }
    taken++;
    if constexpr (AV)
      if (ok)
        for (int j = 0; j < 2; j++) a.nodeav[tag[j]] = av[j];
  }
  // final state, its traces, the monitor of the last step (mean over the nodes of |R V^T|)
  if (ok) {
#pragma unroll
    for (int v = 0; v < NV; v++) {
#pragma unroll
      for (int k = 0; k < N; k++) a.U[(e * NV + v) * N + k] = um[v][k];
#pragma unroll
      for (int s = 0; s < 2; s++) {
        const int row = (s == 0 ? end0 : end1) * N;
        double x = 0.0;
#pragma unroll
        for (int i = 0; i < N; i++) {
          double n = 0.0;
#pragma unroll
          for (int k = 0; k < N; k++) n += t.B[i * N + k] * um[v][k];
          x += t.lf[row + i] * n;
        }
        a.Uf[(e * NV + v) * 2 + s] = x;
      }
    }
  }
  if (taken == 0) return;
  double mon[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) {
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < N; i++) {
      double x = 0.0;
#pragma unroll
      for (int k = 0; k < N; k++) x += t.B[i * N + k] * R[v][k];
      s += fabs(x);
    }
    s = ok ? s / N : 0.0;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) s += __shfl_down(s, d);
    mon[v] = s;
  }
  if ((e & 63) == 0)
    for (int v = 0; v < NV; v++) red[v][e >> 6] = mon[v];
  __syncthreads();
  if (e == 0) {
    const int waves = blockDim.x >> 6;
    bool all_nan = true;
    for (int v = 0; v < NV; v++) {
      double s = 0.0;
      for (int w = 0; w < waves; w++) s += red[v][w];
      s /= static_cast<double>(g.E);
      a.rel[v] = s;
      all_nan = all_nan && isnan(s);
    }
    if (all_nan) a.status[0] = 1;
    a.status[1] += taken;
  }
}

}  // namespace sdg

#endif  // SDG_DG_LINE_HPP_
