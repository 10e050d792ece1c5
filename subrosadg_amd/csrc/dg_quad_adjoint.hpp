// dg_quad_adjoint.hpp -- transpose of the sum-factorised quadrangle stage kernels (Navier-Stokes, FP64,
// periodic meshes): the steps of dg_tensor_adjoint.hpp on two axes, in the layout of dg_quad.hpp (a lane a
// node and a face point, one wavefront per workgroup).
//   quadAdjVolume  nodal state and gradients again, mu (the adjoint of the nodal residual), its face
//                  traces, the pointwise volume-flux VJP, the face points' gradients
//   (nsAdjFaceRevKernel / nsAdjFaceKernel: the face points' VJP)
//   quadAdjLift    gradient adjoints back through the lifting
//   quadAdjGather  trace adjoints and the nodal adjoint back to the modes, transpose of the RK stage
// 64^2 P3, us per launch on the dense matrix-core kernels and here: volume 19.9 and 10.5, lift 11.5 and
// 6.7, gather 7.4 and 5.2. All three are bound by the latency of their phases at that size (1024
// wavefronts on 1024 SIMDs).
#ifndef SDG_DG_QUAD_ADJOINT_HPP_
#define SDG_DG_QUAD_ADJOINT_HPP_

#include <hip/hip_runtime.h>

#include "dg_adjoint.hpp"
#include "dg_quad.hpp"

namespace sdg {

template <int N, int VISC>
__global__ __launch_bounds__(64) void quadAdjVolume(Geo g, Phys ph, StageArgs a, AdjArgs j) {
  using S = QuadShape<N>;
  constexpr int D = 2, NV = 4, NG = 8, NPT = S::NPT, NAQ = S::NAQ, EPB = S::EPB;
  constexpr int REG = S::pad(3 * NV * NPT + NV * NAQ + 8);
  __shared__ double sm[EPB * REG];
  __shared__ QuadLds<N> sT;
  const TensorOps& t = g.tens;
  stageQuadTables<N>(t, sT);
  const int lane = threadIdx.x, le = lane / S::LPE, ln = lane % S::LPE;
  const int64_t e = static_cast<int64_t>(blockIdx.x) * EPB + le;
  const bool ok = le < EPB && e < g.E, node = ok && ln < NPT, slot = ok && ln < NAQ;
  double* X = sm + (le < EPB ? le : 0) * REG;  // state; with Y the gradient field W
  double* Y = X + NV * NPT;
  double* W = X;
  double* Mu = Y + NV * NPT;
  double* Be = Mu + NV * NPT;  // beta, which is alpha on an interior face
  double* Nr = Be + NV * NAQ;
  const int q = ln < NPT ? ln : 0, sl = ln < NAQ ? ln : 0, ix = q % N, iy = q / N;
  const int64_t ec = ok ? e : 0, es = ec * NAQ + sl;
  double um[NV], lm[NV], uo[NV], un[NV], n[D], gi[D * D];
  const int nbs = g.snb[es];
#pragma unroll
  for (int v = 0; v < NV; v++) {
    um[v] = a.U[(ec * NV + v) * NPT + q];
    lm[v] = j.lam[(ec * NV + v) * NPT + q];
    uo[v] = a.Uf_in[(ec * NV + v) * NAQ + sl];
  }
  const double* eg = g.egeo + (ec * 4 + sl / N) * 3;
  for (int d = 0; d < D; d++) n[d] = eg[d];
  const double jw = eg[2] * t.fwt[sl], dj = g.detj[ec];
  for (int i = 0; i < D * D; i++) gi[i] = g.ginv[ec * D * D + i];
  {
    const int64_t nb0 = nbs >= 0 ? static_cast<int64_t>(nbs / NAQ) * NV * NAQ + nbs % NAQ : ec * NV * NAQ + sl;
#pragma unroll
    for (int v = 0; v < NV; v++) un[v] = a.Uf_in[nb0 + v * NAQ];
  }
  waveSync();  // the tables
  const double jq = dj * sT.wn[q], ijw = 1.0 / jq;
  if (node) {
    const int tq = sT.perm[q];
    for (int v = 0; v < NV; v++) {
      X[v * NPT + tq] = um[v];
      Mu[v * NPT + tq] = lm[v];
    }
  }
  double be[NV];
  if (slot) {
#pragma unroll
    for (int v = 0; v < NV; v++) {
      be[v] = ((un[v] - uo[v]) / 2.0) * jw;
      Be[v * NAQ + sl] = be[v];
    }
    if (sl % N == 0)
      for (int d = 0; d < D; d++) Nr[(sl / N) * D + d] = n[d];
  }
  waveSync();
  double u[NV] = {1.0, 0.0, 0.0, 1.0}, mu[NV];
  quadNodal<N>(sT, ix, iy, node, X, Y, u);
  waveSync();
  if (j.apply_minv) {  // the increment is (B^-1 x B^-1)(R / (w |J|))
    quadApply<N, true>(sT.Binv, ix, iy, node, Mu, Y, mu);
#pragma unroll
    for (int v = 0; v < NV; v++) mu[v] *= ijw;
  } else {  // the reference residual (B^T x B^T) R
    quadApply<N, false>(sT.B, ix, iy, node, Mu, Y, mu);
  }
  waveSync();
  if (node)
    for (int v = 0; v < NV; v++) {
      X[v * NPT + q] = u[v];
      Mu[v * NPT + q] = mu[v];
    }
  waveSync();
  double wt[NG], wf[NG];  // total and face gradient at the node
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
      const double c = sT.lf[t.side[s] * N + i] * ijw;
#pragma unroll
      for (int v = 0; v < NV; v++) {
        const double b = Be[v * NAQ + so] * c;
#pragma unroll
        for (int d = 0; d < D; d++) {
          wf[v * D + d] += (VISC == 2 ? b : 2.0 * b) * Nr[s * D + d];
          wt[v * D + d] += 2.0 * b * Nr[s * D + d];
        }
      }
    }
  }
  waveSync();  // X is read
  if (node) {
#pragma unroll
    for (int r = 0; r < NG; r++) W[r * NPT + q] = wf[r];
    // W-bar_a = Dn_a mu, then the pointwise VJP of the volume flux
    double fbar[D * NV], G[D * D], Fb[D * NV], gb[NG], ub[NV];
    quadLine<N, NV, false>(sT.Dn, ix, N * iy, 1, Mu, fbar);
    quadLine<N, NV, false>(sT.Dn, iy, ix, N, Mu, fbar + NV);
    for (int i = 0; i < D * D; i++) G[i] = gi[i] * jq;
    volumeFluxBar<D>(fbar, G, Fb);
    volumeFluxStateVjp<D>(ph, u, wt, Fb, ub);
#pragma unroll
    for (int v = 0; v < NV; v++) j.Ua[(e * NV + v) * NPT + q] = ub[v];
    volumeFluxVjpDir<D>(ph, u, wt, Fb, NV, gb);
#pragma unroll
    for (int r = 0; r < NG; r++) j.RtV[(e * NG + r) * NPT + q] = gb[r];
  }
  waveSync();
  if (slot) {  // H-bar and the gradient the face flux differentiates the viscous flux at
    const int b = sT.base[sl], st = sT.stride[sl];
    const double* l = sT.lf + sT.lofs[sl];
    double hb[NV];
    quadTrace<N>(sT, Mu, sl, hb);
#pragma unroll
    for (int v = 0; v < NV; v++) j.Hb[(e * NV + v) * NAQ + sl] = hb[v];
    const double kf = (sT.lofs[sl] == 0 ? t.kappa[0] : t.kappa[1]) / (dj * sT.fw[sl]);
#pragma unroll
    for (int r = 0; r < NG; r++) {
      double acc = 0.0;
#pragma unroll
      for (int i = 0; i < N; i++) acc += l[i] * W[r * NPT + b + i * st];
      if constexpr (VISC == 2) acc += kf * be[r / D] * n[r % D];
      a.Gf[(e * NG + r) * NAQ + sl] = acc;
    }
  }
}

template <int N, int VISC>
__global__ __launch_bounds__(64) void quadAdjLift(Geo g, Phys ph, StageArgs a, AdjArgs j) {
  using S = QuadShape<N>;
  constexpr int D = 2, NV = 4, NG = 8, NPT = S::NPT, NAQ = S::NAQ, EPB = S::EPB;
  constexpr int REG = S::pad(NG * NPT + NG * NAQ);
  __shared__ double sm[EPB * REG];
  __shared__ QuadLds<N> sT;
  const TensorOps& t = g.tens;
  stageQuadTables<N>(t, sT);
  const int lane = threadIdx.x, le = lane / S::LPE, ln = lane % S::LPE;
  const int64_t e = static_cast<int64_t>(blockIdx.x) * EPB + le;
  const bool ok = le < EPB && e < g.E, node = ok && ln < NPT, slot = ok && ln < NAQ;
  double* Z = sm + (le < EPB ? le : 0) * REG;
  double* Gb = Z + NG * NPT;  // face-gradient adjoints [r][slot]
  const int q = ln < NPT ? ln : 0, sl = ln < NAQ ? ln : 0, ix = q % N, iy = q / N;
  const int64_t ec = ok ? e : 0;
  double gt[NG], gf[NG], gs[NG], yb[NV], gi[D * D], n[D];
#pragma unroll
  for (int r = 0; r < NG; r++) {
    gt[r] = j.RtV[(ec * NG + r) * NPT + q];
    gs[r] = j.GFb[(ec * NG + r) * NAQ + sl];
  }
#pragma unroll
  for (int v = 0; v < NV; v++) yb[v] = j.Ua[(ec * NV + v) * NPT + q];
  const double* eg = g.egeo + (ec * 4 + sl / N) * 3;
  for (int d = 0; d < D; d++) n[d] = eg[d];
  const double jw = g.snb[ec * NAQ + sl] >= 0 ? eg[2] * t.fwt[sl] : 0.0, dj = g.detj[ec];
  for (int i = 0; i < D * D; i++) gi[i] = g.ginv[ec * D * D + i];
  if (slot)
#pragma unroll
    for (int r = 0; r < NG; r++) Gb[r * NAQ + sl] = gs[r];
  waveSync();
  if (node) {  // the face-gradient field's adjoint, then Dr-bar[v][ax] = sum_d J^-T[d][ax] (.)[v][d]
#pragma unroll
    for (int r = 0; r < NG; r++) gf[r] = 0.0;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int i = t.axis[s] == 0 ? ix : iy, so = s * N + sT.slot_of[s * NPT + q];
      const double l = sT.lf[t.side[s] * N + i];
#pragma unroll
      for (int r = 0; r < NG; r++) gf[r] += l * Gb[r * NAQ + so];
    }
    if constexpr (VISC == 1)
#pragma unroll
      for (int r = 0; r < NG; r++) {
        gt[r] += gf[r];
        gf[r] = 0.0;
      }
#pragma unroll
    for (int v = 0; v < NV; v++)
#pragma unroll
      for (int ax = 0; ax < D; ax++) {
        double s = 0.0;
#pragma unroll
        for (int d = 0; d < D; d++) s += gi[d + D * ax] * (gt[v * D + d] + gf[v * D + d]);
        Z[(ax * NV + v) * NPT + q] = s;
      }
  }
  waveSync();
  if (node) {  // Y-bar += sum_a Dn_a^T Dr-bar_a
    double r0[NV], r1[NV];
    quadLine<N, NV, true>(sT.Dn, ix, N * iy, 1, Z, r0);
    quadLine<N, NV, true>(sT.Dn, iy, ix, N, Z + NV * NPT, r1);
#pragma unroll
    for (int v = 0; v < NV; v++) j.Ua[(e * NV + v) * NPT + q] = yb[v] + (r0[v] + r1[v]);
  }
  waveSync();
  if (node) {  // alpha enters the total and the face gradient, beta the total one, both as lf_s(i) n / (w |J|)
    const double inw = 1.0 / (sT.wn[q] * dj);
#pragma unroll
    for (int r = 0; r < NG; r++) Z[r * NPT + q] = inw * (2.0 * gt[r] + gf[r]);
  }
  waveSync();
  if (slot) {
    const int b = sT.base[sl], st = sT.stride[sl];
    const double* l = sT.lf + sT.lofs[sl];
    const double kf = (sT.lofs[sl] == 0 ? t.kappa[0] : t.kappa[1]) / (dj * sT.fw[sl]);
#pragma unroll
    for (int v = 0; v < NV; v++) {
      double ab = 0.0;
#pragma unroll
      for (int d = 0; d < D; d++) {
        double acc = 0.0;
#pragma unroll
        for (int i = 0; i < N; i++) acc += l[i] * Z[(v * D + d) * NPT + b + i * st];
        if constexpr (VISC == 2) acc += kf * gs[v * D + d];  // the own face's lift
        ab += acc * n[d];
      }
      const double sb = ab * jw / 2.0;  // alpha = beta = (u_n - u_o)/2 |J_f| w
      j.Pown[(e * NV + v) * NAQ + sl] = -sb;
      j.Qnb[(e * NV + v) * NAQ + sl] = sb;
    }
  }
  (void)ph;
  (void)a;
}

template <int N>
__global__ __launch_bounds__(64) void quadAdjGather(Geo g, Phys ph, StageArgs a, AdjArgs j) {
  using S = QuadShape<N>;
  constexpr int NV = 4, NPT = S::NPT, NAQ = S::NAQ, EPB = S::EPB;
  constexpr int REG = S::pad(2 * NV * NPT + NV * NAQ);
  __shared__ double sm[EPB * REG];
  __shared__ QuadLds<N> sT;
  const TensorOps& t = g.tens;
  stageQuadTables<N>(t, sT);
  const int lane = threadIdx.x, le = lane / S::LPE, ln = lane % S::LPE;
  const int64_t e = static_cast<int64_t>(blockIdx.x) * EPB + le;
  const bool ok = le < EPB && e < g.E, node = ok && ln < NPT, slot = ok && ln < NAQ;
  double* X = sm + (le < EPB ? le : 0) * REG;
  double* Y = X + NV * NPT;
  double* T = Y + NV * NPT;  // trace adjoints [v][slot]
  const int q = ln < NPT ? ln : 0, sl = ln < NAQ ? ln : 0, ix = q % N, iy = q / N;
  const int64_t ec = ok ? e : 0;
  const int nbs = g.snb[ec * NAQ + sl];
  double x[NV], yb[NV], l[NV], ac[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) {
    const int64_t o = (ec * NV + v) * NAQ + sl;
    x[v] = j.UFf[o] + j.Pown[o];
    yb[v] = j.Ua[(ec * NV + v) * NPT + q];
    l[v] = j.rk ? j.lam[(ec * NV + v) * NPT + q] : 0.0;
    ac[v] = j.rk && !j.rk_first ? j.acc[(ec * NV + v) * NPT + q] : 0.0;
  }
  if (nbs >= 0)
#pragma unroll
    for (int v = 0; v < NV; v++) x[v] += j.Qnb[(static_cast<int64_t>(nbs / NAQ) * NV + v) * NAQ + nbs % NAQ];
  if (slot)
#pragma unroll
    for (int v = 0; v < NV; v++) T[v * NAQ + sl] = x[v];
  waveSync();
  if (node) {  // u_s = sum_i lf_s(i) Y(line)
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int i = t.axis[s] == 0 ? ix : iy, so = s * N + sT.slot_of[s * NPT + q];
      const double c = sT.lf[t.side[s] * N + i];
#pragma unroll
      for (int v = 0; v < NV; v++) yb[v] += c * T[v * NAQ + so];
    }
#pragma unroll
    for (int v = 0; v < NV; v++) X[v * NPT + q] = yb[v];
  }
  waveSync();
  double r[NV];
  quadApply<N, true>(sT.B, ix, iy, node, X, Y, r);  // Y = (B x B) c
  if (node)  // tensor order -> the lane's mode q
    for (int v = 0; v < NV; v++) X[v * NPT + q] = r[v];
  waveSync();
  if (node) {
    const int tq = sT.perm[q];
#pragma unroll
    for (int v = 0; v < NV; v++) {
      const int64_t o = (e * NV + v) * NPT + q;
      const double vjp = X[v * NPT + tq];
      if (!j.rk) {
        j.out[o] = vjp;
      } else {
        const double al = j.rk_first ? j.c0 * l[v] : j.c0 * l[v] + ac[v];
        const double ln2 = j.c2dt * vjp + j.c1 * l[v];
        if (j.rk_last) {
          j.lam[o] = al + ln2;
        } else {
          j.acc[o] = al;
          j.lam[o] = ln2;
        }
      }
    }
  }
  (void)ph;
  (void)a;
}

}  // namespace sdg

#endif  // SDG_DG_QUAD_ADJOINT_HPP_
