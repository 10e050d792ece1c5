// dg_quad.hpp -- sum-factorised FP64 stage kernels for (affine) quadrangles P1..P5.
//
// The operators are the 1-D operators of dg_tensor.hpp along the two axes (basis B, collocation
// derivative Dn at the Gauss nodes, end-point values lf, diagonal mass w |J|), so a contraction costs
// N instead of N^2 products per node. A lane is at once a node (N^2) and a face point (4 N) of its
// element, and a workgroup is one wavefront of 64 / max(N^2, 4N) elements: phases that need each
// other's values synchronise within the wavefront, no barrier waits for another one, and small
// meshes still spread over the card (48^2 cells P3: 576 workgroups).
//   quadGrad      Navier-Stokes (BR1 / BR2) or Euler with artificial viscosity: the weak divergence of
//                 the volume flux -> Rvol (nodes), the own normal viscous flux -> Vn (face points)
//   quadResidual  numerical flux of the element's own face points from both sides' traces and Vn,
//                 residual, RK update, next traces, monitor; Euler: the volume flux too (one kernel)
// A face point's numerical flux is evaluated by both parents with the face's left/right roles, which
// gives bit-identical values; one pass per face point instead (a kernel in between) would save those
// instructions but write and read the flux through HBM and cost a launch per stage.
#ifndef SDG_DG_QUAD_HPP_
#define SDG_DG_QUAD_HPP_

#include <hip/hip_runtime.h>

#include "dg_tensor.hpp"

namespace sdg {

template <int N>
struct QuadShape {
  static constexpr int D = 2, NV = 4, NG = 8, NPT = N * N, NAQ = 4 * N;
  static constexpr int LPE = NPT > NAQ ? NPT : NAQ;  // lanes per element
  static constexpr int EPB = 64 / LPE;               // elements per wavefront
  // LDS doubles per element, congruent to 2 mod 32 so that the elements of a half wavefront use
  // different banks
  static constexpr int pad(int n) { return (n + 29) / 32 * 32 + 2; }
};

// the order's tables, staged per workgroup with one round of loads
template <int N>
struct QuadLds {
  static constexpr int NPT = N * N, NAQ = 4 * N;
  double B[NPT], Binv[NPT], Dn[NPT], lf[2 * N], wn[NPT], fw[NAQ];
  short perm[NPT], iperm[NPT], slot_of[4 * NPT], base[NAQ], stride[NAQ], lofs[NAQ];  // per face point: axis stride, row of lf
};

template <int N>
__device__ __forceinline__ void stageQuadTables(const TensorOps& t, QuadLds<N>& L) {
  constexpr int NPT = N * N, NAQ = 4 * N, NS = (4 * NPT + 63) / 64;
  static_assert(NPT <= 64 && NAQ <= 64, "one table entry per lane");
  const int tid = threadIdx.x;
  const int i2 = tid < NPT ? tid : 0, ia = tid < NAQ ? tid : 0;
  const double b = t.B[i2], bi = t.Binv[i2], dn = t.Dn[i2], lf = t.lf[tid < 2 * N ? tid : 0];
  const short pm = t.perm[i2], ip = t.iperm[i2], bs = t.base[ia];
  const double w0 = t.w[i2 % N], w1 = t.w[i2 / N], fw = t.fwt[ia];
  const int ax = t.axis[ia / N], sd = t.side[ia / N];
  short so[NS];
#pragma unroll
  for (int k = 0; k < NS; k++) so[k] = t.slot_of[tid + 64 * k < 4 * NPT ? tid + 64 * k : 0];
  if (tid < NPT) {
    L.B[tid] = b;
    L.Binv[tid] = bi;
    L.Dn[tid] = dn;
    L.perm[tid] = pm;
    L.iperm[tid] = ip;
    L.wn[tid] = w0 * w1;
  }
  if (tid < 2 * N) L.lf[tid] = lf;
  if (tid < NAQ) {
    L.base[tid] = bs;
    L.fw[tid] = fw;
    L.stride[tid] = static_cast<short>(ax == 0 ? 1 : N);
    L.lofs[tid] = static_cast<short>(sd * N);
  }
#pragma unroll
  for (int k = 0; k < NS; k++)
    if (tid + 64 * k < 4 * NPT) L.slot_of[tid + 64 * k] = so[k];
}

// the lanes of the workgroup's single wavefront see each other's LDS writes
__device__ __forceinline__ void waveSync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// out[c] = sum_m M[i][m] in[c][line of the node along the axis][m] (T: M transposed), C components
template <int N, int C, bool T>
__device__ __forceinline__ void quadLine(const double* M, int i, int q0, int st, const double* in, double* out) {
  double m[N];
#pragma unroll
  for (int k = 0; k < N; k++) m[k] = T ? M[k * N + i] : M[i * N + k];
#pragma unroll
  for (int c = 0; c < C; c++) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < N; k++) s += m[k] * in[c * N * N + q0 + k * st];
    out[c] = s;
  }
}

// the four variables of a node through a 2-D operator M x M: X (LDS, input and scratch) -> out
// (registers); every lane of the wavefront calls it
template <int N, bool T>
__device__ __forceinline__ void quadApply(const double* M, int ix, int iy, bool node, double* X, double* Y, double* out) {
  constexpr int NPT = N * N;
  const int q = ix + N * iy;
  if (node) quadLine<N, 4, T>(M, ix, N * iy, 1, X, out);
  if (node)
    for (int v = 0; v < 4; v++) Y[v * NPT + q] = out[v];
  waveSync();
  if (node) quadLine<N, 4, T>(M, iy, ix, N, Y, out);
}

// nodal state of the modal one staged in X (tensor order)
template <int N>
__device__ __forceinline__ void quadNodal(const QuadLds<N>& L, int ix, int iy, bool node, double* X, double* Y, double* u) {
  quadApply<N, false>(L.B, ix, iy, node, X, Y, u);
}

// traces of the nodal field X at the element's own face point sl
template <int N>
__device__ __forceinline__ void quadTrace(const QuadLds<N>& L, const double* X, int sl, double* out) {
  const int b = L.base[sl], st = L.stride[sl];
  const double* l = L.lf + L.lofs[sl];
#pragma unroll
  for (int v = 0; v < 4; v++) {
    double acc = 0.0;
#pragma unroll
    for (int i = 0; i < N; i++) acc += l[i] * X[v * N * N + b + i * st];
    out[v] = acc;
  }
}

// ---- kernel 1: gradient, volume flux, own normal viscous flux -----------------------------------
// Bound by memory on large meshes, by the latency of its chain of phases on small ones; all loads of
// the wavefront are issued before the first wait.
// VISC 0: Euler with artificial viscosity (volume gradient); 1, 2: Navier-Stokes BR1 / BR2.
template <int N, int VISC>
__global__ __launch_bounds__(64) void quadGrad(Geo g, Phys ph, StageArgs a) {
  using S = QuadShape<N>;
  constexpr int D = 2, NV = 4, NG = 8, NPT = S::NPT, NAQ = S::NAQ, EPB = S::EPB;
  constexpr int REG = S::pad(2 * NV * NPT + 2 * NV * NAQ + 8);
  __shared__ double sm[EPB * REG];
  __shared__ QuadLds<N> sT;
  if (a.status && a.status[0]) return;
  const TensorOps& t = g.tens;
  stageQuadTables<N>(t, sT);
  const int lane = threadIdx.x, le = lane / S::LPE, ln = lane % S::LPE;
  const int64_t e = static_cast<int64_t>(blockIdx.x) * EPB + le;
  const bool ok = le < EPB && e < g.E, node = ok && ln < NPT, slot = ok && ln < NAQ;
  double* X = sm + (le < EPB ? le : 0) * REG;  // modal state, then nodal; W: gradient field, flux field
  double* Y = X + NV * NPT;
  double* W = X;
  double* Al = X + 2 * NV * NPT;  // alpha [v][slot]
  double* Be = Al + NV * NAQ;     // beta [v][slot]
  double* Nr = Be + NV * NAQ;     // outward normal per face (straight faces: one per face)
  const int q = ln < NPT ? ln : 0, sl = ln < NAQ ? ln : 0, ix = q % N, iy = q / N;
  const int64_t ec = ok ? e : 0, es = ec * NAQ + sl;
  double um[NV], uo[NV], un[NV], n[D];
  const int nbs = g.snb[es];
#pragma unroll
  for (int v = 0; v < NV; v++) um[v] = a.U[(ec * NV + v) * NPT + q];
#pragma unroll
  for (int v = 0; v < NV; v++) uo[v] = a.Uf_in[(ec * NV + v) * NAQ + sl];
  const double* eg = g.egeo + (ec * 4 + sl / N) * 3;
  for (int d = 0; d < D; d++) n[d] = eg[d];
  const double jw = eg[2] * t.fwt[sl], dj = g.detj[ec];
  double gi[D * D];
  for (int i = 0; i < D * D; i++) gi[i] = g.ginv[ec * D * D + i];
  {
    const int64_t nb0 = nbs >= 0 ? static_cast<int64_t>(nbs / NAQ) * NV * NAQ + nbs % NAQ : ec * NV * NAQ + sl;
#pragma unroll
    for (int v = 0; v < NV; v++) un[v] = a.Uf_in[nb0 + v * NAQ];
  }
  double eps_q = 0.0, eps_s = 0.0;
  if constexpr (VISC == 0) {
    for (int j = 0; j < 4; j++) {
      const double av = g.nodeav[g.ntag[ec * 4 + j]];
      eps_q += t.nodt[q * 4 + j] * av;
      eps_s += g.nodf[sl * 4 + j] * av;
    }
  }
  waveSync();  // the tables
  if (node) {
    const int tq = sT.perm[q];
    for (int v = 0; v < NV; v++) X[v * NPT + tq] = um[v];
  }
  double be[NV];
  if (slot) {
    double al[NV];
    if (nbs >= 0) {
#pragma unroll
      for (int v = 0; v < NV; v++) {
        al[v] = ((uo[v] + un[v]) / 2.0 - uo[v]) * jw;
        be[v] = ((un[v] - uo[v]) / 2.0) * jw;
      }
    } else {  // boundary face point: the boundary condition's gradient states
      const int bp = -1 - nbs;
      double wd[D + 3], uvg[NV], uig[NV];
      for (int i = 0; i < D + 3; i++) wd[i] = g.bdata[static_cast<int64_t>(bp) * (D + 3) + i];
      boundaryGradientStates<D>(ph, g.btype[bp], n, uo, wd, uvg, uig);
      for (int v = 0; v < NV; v++) {
        al[v] = (uvg[v] - uo[v]) * jw;
        be[v] = uig[v] * jw;
      }
    }
#pragma unroll
    for (int v = 0; v < NV; v++) {
      Al[v * NAQ + sl] = al[v];
      if constexpr (VISC != 0) Be[v * NAQ + sl] = be[v];
    }
    if (sl % N == 0)
      for (int d = 0; d < D; d++) Nr[(sl / N) * D + d] = n[d];
  }
  waveSync();
  double u[NV] = {1.0, 0.0, 0.0, 1.0};
  quadNodal<N>(sT, ix, iy, node, X, Y, u);
  if (node)
    for (int v = 0; v < NV; v++) X[v * NPT + q] = u[v];  // the modal values were last read before quadNodal's sync
  waveSync();
  // gradient at the node: J^-T (Dn u) + the face corrections
  double wt[NG], wf[NG];  // total gradient; the gradient with the faces' average traces
  const double jq = dj * sT.wn[q], ijw = 1.0 / jq;
  if (node) {
    double d0[NV], d1[NV];
    quadLine<N, NV, false>(sT.Dn, ix, N * iy, 1, X, d0);
    quadLine<N, NV, false>(sT.Dn, iy, ix, N, X, d1);
#pragma unroll
    for (int v = 0; v < NV; v++)
#pragma unroll
      for (int d = 0; d < D; d++) wt[v * D + d] = wf[v * D + d] = gi[d] * d0[v] + gi[d + D] * d1[v];
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int i = t.axis[s] == 0 ? ix : iy, so = s * N + sT.slot_of[s * NPT + q];
      const double c = sT.lf[t.side[s] * N + i] * ijw, n0 = Nr[s * D], n1 = Nr[s * D + 1];
#pragma unroll
      for (int v = 0; v < NV; v++) {
        const double al = Al[v * NAQ + so] * c;
        wf[v * D] += al * n0;
        wf[v * D + 1] += al * n1;
        if constexpr (VISC != 0) {
          const double b = Be[v * NAQ + so] * c;
          wt[v * D] += (al + b) * n0;
          wt[v * D + 1] += (al + b) * n1;
        }
      }
    }
  }
  waveSync();  // X is read; W takes the gradient fields
  if (a.Wout) {  // modal coefficients of the total gradient (sdg_get_gradient)
    if (node)
      for (int r = 0; r < NG; r++) W[r * NPT + q] = wt[r];
    waveSync();
    if (node) {
      const int b = sT.iperm[q];
#pragma unroll 1
      for (int r = 0; r < NG; r++) {
        double s = 0.0;
        for (int j = 0; j < N; j++)
          for (int i = 0; i < N; i++) s += sT.Binv[ix * N + i] * sT.Binv[iy * N + j] * W[r * NPT + i + N * j];
        a.Wout[(e * NPT + b) * NG + r] = s;
      }
    }
    waveSync();
  }
  if (node)
#pragma unroll
    for (int r = 0; r < NG; r++) W[r * NPT + q] = VISC == 1 ? wt[r] : wf[r];
  waveSync();
  if (slot) {  // the gradient at the own face point and the normal viscous flux there
    const int b = sT.base[sl], st = sT.stride[sl];
    const double* l = sT.lf + sT.lofs[sl];
    double gs[NG], vn[NV];
#pragma unroll
    for (int r = 0; r < NG; r++) {
      double acc = 0.0;
#pragma unroll
      for (int i = 0; i < N; i++) acc += l[i] * W[r * NPT + b + i * st];
      gs[r] = acc;
    }
    if constexpr (VISC == 0) {
#pragma unroll
      for (int v = 0; v < NV; v++) vn[v] = eps_s * (gs[v * D] * n[0] + gs[v * D + 1] * n[1]);
    } else {
      if constexpr (VISC == 2) {  // BR2: the own face's lift
        const double kf = (sT.lofs[sl] == 0 ? t.kappa[0] : t.kappa[1]) / (dj * sT.fw[sl]);
#pragma unroll
        for (int r = 0; r < NG; r++) gs[r] += kf * be[r / D] * n[r % D];
      }
      if (nbs < 0)
        for (int r = 0; r < NG; r++) a.Gf[(e * NG + r) * NAQ + sl] = gs[r];
      double ws[D + 3], pg[NG], fv[D * NV];
      computational<D>(ph, uo, ws);
      primitiveGradient<D>(ph, ws, uo, gs, pg);
      viscousRawFlux<D>(ph, ws, pg, fv);
#pragma unroll
      for (int v = 0; v < NV; v++) vn[v] = fv[D * v] * n[0] + fv[1 + D * v] * n[1];
    }
#pragma unroll
    for (int v = 0; v < NV; v++) a.Vn[(e * NV + v) * NAQ + sl] = vn[v];
  }
  waveSync();  // W takes the volume flux [b NV + v][node]
  double src = 0.0;
  if (node) {
    double w[D + 3], fv[D * NV], G[D * D], out[D * NV];
    computational<D>(ph, u, w);
    if (ph.source == kSourceBoussinesq) src = boussinesqSource<D>(ph, w) * jq;
    if constexpr (VISC == 0) {
#pragma unroll
      for (int r = 0; r < NG; r++) fv[(r % D) + D * (r / D)] = eps_q * wf[r];
    } else {
      double pg[NG];
      primitiveGradient<D>(ph, w, u, wt, pg);
      viscousRawFlux<D>(ph, w, pg, fv);
    }
    for (int i = 0; i < D * D; i++) G[i] = gi[i] * jq;
    volumeFlux<double, D, true>(a, w, fv, G, out);
#pragma unroll
    for (int i = 0; i < D * NV; i++) W[i * NPT + q] = out[i];
  }
  waveSync();
  if (node) {
    double r0[NV], r1[NV];
    quadLine<N, NV, true>(sT.Dn, ix, N * iy, 1, W, r0);
    quadLine<N, NV, true>(sT.Dn, iy, ix, N, W + NV * NPT, r1);
    r0[D] += src;
#pragma unroll
    for (int v = 0; v < NV; v++) a.Rvol[(e * NV + v) * NPT + q] = r0[v] + r1[v];
  }
}

// ---- kernel 2: face fluxes, residual, update, next traces, monitor ------------------------------
// KIND 0: Navier-Stokes, 1: Euler with artificial viscosity (both after quadGrad), 2: Euler
template <int N, int KIND>
__global__ __launch_bounds__(64) void quadResidual(Geo g, Phys ph, StageArgs a) {
  using S = QuadShape<N>;
  constexpr int D = 2, NV = 4, NG = 8, NPT = S::NPT, NAQ = S::NAQ, EPB = S::EPB;
  constexpr int REG = S::pad(2 * NV * NPT + NV * NAQ);
  __shared__ double sm[EPB * REG];
  __shared__ QuadLds<N> sT;
  if (a.status && a.status[0]) return;
  const TensorOps& t = g.tens;
  stageQuadTables<N>(t, sT);
  const int lane = threadIdx.x, le = lane / S::LPE, ln = lane % S::LPE;
  const int64_t e = static_cast<int64_t>(blockIdx.x) * EPB + le;
  const bool ok = le < EPB && e < g.E, node = ok && ln < NPT, slot = ok && ln < NAQ;
  double* X = sm + (le < EPB ? le : 0) * REG;
  double* Y = X + NV * NPT;
  double* H = Y + NV * NPT;  // signed face flux [v][slot]
  const int q = ln < NPT ? ln : 0, sl = ln < NAQ ? ln : 0, ix = q % N, iy = q / N;
  const int64_t ec = ok ? e : 0, es = ec * NAQ + sl;
  const int nbs = g.snb[es], side = g.sfp[es] & 1, tq = t.perm[q];
  double um[NV], us[NV], uo[NV], un[NV], vo[NV], vb[NV], rv[NV], n[D];
#pragma unroll
  for (int v = 0; v < NV; v++) {
    uo[v] = a.Uf_in[(ec * NV + v) * NAQ + sl];
    um[v] = a.U[(ec * NV + v) * NPT + q];
    us[v] = a.c0 != 0.0 ? a.Un[(ec * NV + v) * NPT + q] : 0.0;
    if constexpr (KIND != 2) {
      vo[v] = a.Vn[(ec * NV + v) * NAQ + sl];
      rv[v] = a.Rvol[(ec * NV + v) * NPT + q];
    }
  }
  const double* eg = g.egeo + (ec * 4 + sl / N) * 3;
  for (int d = 0; d < D; d++) n[d] = eg[d];
  const double jw = eg[2] * t.fwt[sl], dj = g.detj[ec];
  {
    const int64_t nb0 = nbs >= 0 ? static_cast<int64_t>(nbs / NAQ) * NV * NAQ + nbs % NAQ : ec * NV * NAQ + sl;
#pragma unroll
    for (int v = 0; v < NV; v++) {
      un[v] = a.Uf_in[nb0 + v * NAQ];
      if constexpr (KIND != 2) vb[v] = a.Vn[nb0 + v * NAQ];
    }
  }
  waveSync();  // the tables
  const double jq = dj * sT.wn[q];
  double R[NV] = {0.0, 0.0, 0.0, 0.0};
  if constexpr (KIND == 2) {  // the volume flux and its weak divergence
    if (node)
      for (int v = 0; v < NV; v++) X[v * NPT + tq] = um[v];
    waveSync();
    double u[NV] = {1.0, 0.0, 0.0, 1.0};
    quadNodal<N>(sT, ix, iy, node, X, Y, u);
    waveSync();
    double src = 0.0;
    if (node) {
      double w[D + 3], G[D * D], out[D * NV];
      computational<D>(ph, u, w);
      if (ph.source == kSourceBoussinesq) src = boussinesqSource<D>(ph, w) * jq;
      for (int i = 0; i < D * D; i++) G[i] = g.ginv[e * D * D + i] * jq;
      volumeFlux<double, D, false>(a, w, nullptr, G, out);
#pragma unroll
      for (int i = 0; i < D * NV; i++) X[i * NPT + q] = out[i];  // X and Y: [b NV + v][node]
    }
    waveSync();
    if (node) {
      double r1[NV];
      quadLine<N, NV, true>(sT.Dn, ix, N * iy, 1, X, R);
      quadLine<N, NV, true>(sT.Dn, iy, ix, N, Y, r1);
      R[D] += src;
#pragma unroll
      for (int v = 0; v < NV; v++) R[v] += r1[v];
    }
  }
  if (slot) {
    double h[NV];
    if (nbs < 0) {
      double gb[NG];
      if constexpr (KIND == 0)
        for (int r = 0; r < NG; r++) gb[r] = a.Gf[(e * NG + r) * NAQ + sl];
      boundaryFlux<D, KIND == 0>(ph, g, -1 - nbs, uo, gb, false, 0.0, 0.0, h);
      for (int v = 0; v < NV; v++) h[v] = KIND == 1 ? vo[v] * jw - h[v] : -h[v];
    } else {
      double ul[NV], ur[NV], wl[D + 3], wr[D + 3], nl[D];
#pragma unroll
      for (int v = 0; v < NV; v++) {
        ul[v] = side == 0 ? uo[v] : un[v];
        ur[v] = side == 0 ? un[v] : uo[v];
      }
      for (int d = 0; d < D; d++) nl[d] = side == 0 ? n[d] : -n[d];
      computational<D>(ph, ul, wl);
      computational<D>(ph, ur, wr);
      convectiveFlux<D>(ph, nl, ul, wl, ur, wr, h);
#pragma unroll
      for (int v = 0; v < NV; v++) {
        double x = h[v];
        if constexpr (KIND != 2) {  // both sides' Vn are along their own outward normal
          const double vl = side == 0 ? vo[v] : vb[v], vr = side == 0 ? vb[v] : vo[v];
          x -= (vl - vr) / 2.0;
        }
        x *= jw;
        h[v] = side == 0 ? -x : x;
      }
    }
#pragma unroll
    for (int v = 0; v < NV; v++) H[v * NAQ + sl] = h[v];
  }
  waveSync();
  if (node) {
    if constexpr (KIND != 2)
#pragma unroll
      for (int v = 0; v < NV; v++) R[v] = rv[v];
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int i = t.axis[s] == 0 ? ix : iy, so = s * N + sT.slot_of[s * NPT + q];
      const double l = sT.lf[t.side[s] * N + i];
#pragma unroll
      for (int v = 0; v < NV; v++) R[v] += l * H[v * NAQ + so];
    }
  }
  if (a.mode == 1 || a.last_stage) {  // (B^T x B^T) R: the reference residual; its values at the nodes
    double r[NV];
    if (node)
      for (int v = 0; v < NV; v++) X[v * NPT + q] = R[v];
    waveSync();
    quadApply<N, true>(sT.B, ix, iy, node, X, Y, r);
    if (a.mode == 1) {
      if (node)
        for (int v = 0; v < NV; v++) a.Rout[(e * NV + v) * NPT + sT.iperm[q]] = r[v];
      return;
    }
    if (node)
      for (int v = 0; v < NV; v++) X[v * NPT + q] = r[v];
    waveSync();
    quadApply<N, false>(sT.B, ix, iy, node, X, Y, r);
    waveSync();
    // monitor: mean over the nodes of |R V^T| (TimeIntegration.cpp:279-298), one lane per variable
    if (node)
      for (int v = 0; v < NV; v++) X[v * NPT + q] = fabs(r[v]);
    waveSync();
    if (ok && ln < NV) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < NPT; k++) s += X[ln * NPT + k];
      a.mon[e * NV + ln] = s / NPT;
    }
    waveSync();
  }
  // increment R / (w |J|) -> modal, RK update in the modal order, traces of the new state
  double inc[NV] = {0.0, 0.0, 0.0, 0.0};
  if (node) {
    const double ijw = 1.0 / jq;
    for (int v = 0; v < NV; v++) X[v * NPT + q] = R[v] * ijw;
  }
  waveSync();
  quadApply<N, false>(sT.Binv, ix, iy, node, X, Y, inc);
  // the lane's coefficients um, us are the modes q, its increment that of tensor index q
  if (node)
    for (int v = 0; v < NV; v++) X[v * NPT + q] = inc[v];
  waveSync();
  double nu[NV];
  if (node) {
    const int step = a.rec ? a.status[1] + (a.last_stage ? 1 : 0) : 0, stage = a.last_stage ? 0 : a.rec_stage + 1;
#pragma unroll
    for (int v = 0; v < NV; v++) {
      const int64_t gi = (e * NV + v) * NPT + q;
      double x = um[v] * a.c1;
      x += a.c0 * us[v];
      x += a.c2dt * X[v * NPT + tq];
      a.Uo[gi] = x;
      if (a.rec && step < a.rec_nsteps) a.rec[(static_cast<int64_t>(step) * a.rec_S + stage) * a.rec_n + gi] = x;
      nu[v] = x;
    }
  }
  waveSync();
  if (node)
    for (int v = 0; v < NV; v++) X[v * NPT + tq] = nu[v];
  waveSync();
  quadNodal<N>(sT, ix, iy, node, X, Y, nu);
  if (node)
    for (int v = 0; v < NV; v++) X[v * NPT + q] = nu[v];
  waveSync();
  if (slot) {
    double tr[NV];
    quadTrace<N>(sT, X, sl, tr);
    const int step = a.rec_t ? a.status[1] + (a.last_stage ? 1 : 0) : 0, stage = a.last_stage ? 0 : a.rec_stage + 1;
#pragma unroll
    for (int v = 0; v < NV; v++) {
      const int64_t ti = (e * NV + v) * NAQ + sl;
      a.Uf_out[ti] = tr[v];
      if (a.rec_t && step < a.rec_nsteps) a.rec_t[(static_cast<int64_t>(step) * a.rec_S + stage) * a.rec_nt + ti] = tr[v];
    }
  }
}

// traces from the state in HBM with the stage kernel's own arithmetic (restarts, checkpoints)
template <int N>
__global__ __launch_bounds__(64) void quadTraceKernel(Geo g, const double* U, double* Uf_out) {
  using S = QuadShape<N>;
  constexpr int NV = 4, NPT = S::NPT, NAQ = S::NAQ, EPB = S::EPB, REG = S::pad(2 * NV * NPT);
  __shared__ double sm[EPB * REG];
  __shared__ QuadLds<N> sT;
  const TensorOps& t = g.tens;
  stageQuadTables<N>(t, sT);
  const int lane = threadIdx.x, le = lane / S::LPE, ln = lane % S::LPE;
  const int64_t e = static_cast<int64_t>(blockIdx.x) * EPB + le;
  const bool ok = le < EPB && e < g.E, node = ok && ln < NPT, slot = ok && ln < NAQ;
  double* X = sm + (le < EPB ? le : 0) * REG;
  double* Y = X + NV * NPT;
  const int q = ln < NPT ? ln : 0, ix = q % N, iy = q / N;
  waveSync();
  if (node)
    for (int v = 0; v < NV; v++) X[v * NPT + sT.perm[q]] = U[(e * NV + v) * NPT + q];
  waveSync();
  double nu[NV];
  quadNodal<N>(sT, ix, iy, node, X, Y, nu);
  if (node)
    for (int v = 0; v < NV; v++) X[v * NPT + q] = nu[v];
  waveSync();
  if (slot) {
    double tr[NV];
    quadTrace<N>(sT, X, ln, tr);
    for (int v = 0; v < NV; v++) Uf_out[(e * NV + v) * NAQ + ln] = tr[v];
  }
}

}  // namespace sdg

#endif  // SDG_DG_QUAD_HPP_
