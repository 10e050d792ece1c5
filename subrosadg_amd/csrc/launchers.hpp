// launchers.hpp -- kernel sets: the stage, trace, sensor and adjoint kernels of an element size as
// launch functions, and the selection by element type and order. The sets of each element type are
// compiled in a translation unit of their own (sdg_launch_*.hip), so that they build in parallel.
#ifndef SDG_LAUNCHERS_HPP_
#define SDG_LAUNCHERS_HPP_

#include <hip/hip_runtime.h>

#include "../../include/sdg.h"
#include "dg_adjoint.hpp"
#include "dg_kernels.hpp"
#include "dg_line.hpp"
#include "dg_mfma.hpp"
#include "dg_quad.hpp"
#include "dg_quad_adjoint.hpp"
#include "dg_tensor.hpp"
#include "dg_tensor_adjoint.hpp"

namespace sdg {

using StageFn = void (*)(hipStream_t, const Geo&, const Phys&, const StageArgs&);
using TraceFn = void (*)(hipStream_t, const Geo&, const double*, void*, const MixRef&);
using DtFn = void (*)(hipStream_t, const Geo&, const Phys&, const double*, const double*, double, int, double*);
using MonFn = void (*)(hipStream_t, const double*, int, double*, int*);
using SrcFn = void (*)(hipStream_t, const Geo&, const Phys&, const double*, double*, const double*);
using AdjFn = void (*)(hipStream_t, const Geo&, const Phys&, const StageArgs&, const AdjArgs&);
using AvFn = void (*)(hipStream_t, const Geo&, const Phys&, const double*, double*);
using LineFn = void (*)(hipStream_t, const Geo&, const Phys&, const LineRun&);
using BlockFn = void (*)(hipStream_t, const Geo&, const Phys&, const double*, double*);

struct Launchers {
  bool mfma = false;
  bool tensor = false;  // hexahedra, Navier-Stokes: sum-factorised stage kernels
  bool quad = false;    // quadrangles: sum-factorised stage kernels
  StageFn euler = nullptr;
  StageFn ns_grad_br1 = nullptr;
  StageFn ns_grad_br2 = nullptr;
  StageFn ns_flux = nullptr;
  StageFn ns_face = nullptr;  // matrix-core path: face fluxes before ns_flux
  TraceFn trace = nullptr;
  TraceFn trace64 = nullptr;  // FP64 traces of the FP64 state (the adjoint of mixed-precision contexts)
  SrcFn source = nullptr;  // modal Boussinesq source (all kernel sets but the sum-factorised one)
  DtFn dt = nullptr;
  MonFn monitor = nullptr;
  // Euler with artificial viscosity (vector kernels): gradient pass + volume flux, face fluxes +
  // residual + update, and the per-step sensor
  StageFn av_grad = nullptr;
  StageFn av_flux = nullptr;
  StageFn av_ns_grad[2] = {nullptr, nullptr};  // Navier-Stokes with artificial viscosity: BR1, BR2
  StageFn av_ns_flux = nullptr;
  AvFn av_sensor = nullptr;
  // Navier-Stokes BR2 raw files: per boundary face the parent's volume gradient plus that face's lift
  BlockFn br2_blocks = nullptr;
  LineFn line_run[2] = {nullptr, nullptr};  // lines, Euler: whole runs of small meshes (without / with AV)
  // discrete adjoint (Navier-Stokes, FP64: the dense matrix-core set, or the sum-factorised set on hexahedra)
  AdjFn adj_volume[2] = {nullptr, nullptr};  // BR1, BR2
  AdjFn adj_face = nullptr;
  AdjFn adj_lift[2] = {nullptr, nullptr};
  AdjFn adj_gather = nullptr;
};

inline int blocksFor(int E, int epb) { return (E + epb - 1) / epb; }

// Grids of at most this many workgroups take kWideWaves wavefronts each in the gradient and residual
// kernels. Microseconds a launch at 507 to 1024, 2025 to 2048 and 12800 workgroups, with the tile count's
// wavefronts and with four: quadrangles P3 FP64 gradient 12.8 and 12.0, 17.7 and 20.2, 52.5 and 69.5.
constexpr int kWideGrid = 1024;
// In FP64 the residual kernel takes four for any grid where the flux panel it stages has 24 rows or more:
// quadrangles P3 10.3 and 7.9 us at 256 workgroups, 32.0 and 30.4 at 6400; tetrahedra P2 22.7 and 20.0 at
// 3456. Below (triangles P1, P2, tetrahedra P1) and in mixed precision it loses on large grids: triangles
// P2 12.8 and 15.5 us at 5000 workgroups, quadrangles P4 mixed 35.3 and 40.8 at 6400.
constexpr int kWideRows = 24;

template <typename TC, int D, int NB, int NQ, int NF, int NFQ, int VISC>
void launchGradMfma(hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
  constexpr int W = MfmaShape<NB, NQ, NF * NFQ>::WAVES;
  const int grid = blocksFor(g.E, 16 / ((D + 2) * D));
  if (W < kWideWaves && grid <= kWideGrid)
    hipLaunchKernelGGL((nsGradMfma<TC, D, NB, NQ, NF, NFQ, VISC, kWideWaves>), dim3(grid), dim3(64 * kWideWaves), 0, st, g, ph, a);
  else
    hipLaunchKernelGGL((nsGradMfma<TC, D, NB, NQ, NF, NFQ, VISC, W>), dim3(grid), dim3(64 * W), 0, st, g, ph, a);
}
template <typename TC, int D, int NB, int NQ, int NF, int NFQ>
void launchResidualMfma(hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
  constexpr int W = sizeof(TC) == 8 && NQ * D >= kWideRows ? kWideWaves : MfmaShape<NB, NQ, NF * NFQ>::WAVES;
  const int grid = blocksFor(g.E, 16 / (D + 2));
  if (W < kWideWaves && grid <= kWideGrid)
    hipLaunchKernelGGL((nsResidualMfma<TC, D, NB, NQ, NF, NFQ, kWideWaves>), dim3(grid), dim3(64 * kWideWaves), 0, st, g, ph, a);
  else
    hipLaunchKernelGGL((nsResidualMfma<TC, D, NB, NQ, NF, NFQ, W>), dim3(grid), dim3(64 * W), 0, st, g, ph, a);
}

// VALU kernels: any size; MFMA kernels: bases that fill 16x16 tiles. TC is the contraction type of
// the matrix-core kernels: double (FP64 mode) or float (mixed-precision mode).
template <int D, int NB, int NQ, int NF, int NFQ, bool MFMA, typename TC = double, bool ADJOINT = true>
Launchers makeLaunchers() {
  using S = Sizes<D, NB, NQ, NF, NFQ>;
  constexpr int EPB = S::EPB;
  constexpr int NV = D + 2;
  Launchers l;
  l.mfma = MFMA;
  if constexpr (MFMA) {
    constexpr int EPB_S = 16 / NV, EPB_G = 16 / (NV * D);
    l.euler = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      hipLaunchKernelGGL((eulerStageMfma<TC, D, NB, NQ, NF, NFQ>), dim3(blocksFor(g.E, EPB_S)),
                         dim3(MfmaShape<NB, NQ, NF * NFQ>::NT), 0, st, g, ph, a);
    };
    l.ns_grad_br1 = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      launchGradMfma<TC, D, NB, NQ, NF, NFQ, 1>(st, g, ph, a);
    };
    l.ns_grad_br2 = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      launchGradMfma<TC, D, NB, NQ, NF, NFQ, 2>(st, g, ph, a);
    };
    l.ns_face = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      hipLaunchKernelGGL((nsFaceFluxKernel<TC, D, NF, NFQ>), dim3(blocksFor((g.F + g.Fb) * NFQ, kThreads)),
                         dim3(kThreads), 0, st, g, ph, a);
    };
    l.ns_flux = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      launchResidualMfma<TC, D, NB, NQ, NF, NFQ>(st, g, ph, a);
    };
    {  // Euler with artificial viscosity: volume gradient, AV fluxes (both precision modes)
      l.av_grad = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
        launchGradMfma<TC, D, NB, NQ, NF, NFQ, 0>(st, g, ph, a);
      };
      l.av_flux = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
        hipLaunchKernelGGL((nsFaceFluxKernel<TC, D, NF, NFQ, false, true>),
                           dim3(blocksFor((g.F + g.Fb) * NFQ, kThreads)), dim3(kThreads), 0, st, g, ph, a);
        launchResidualMfma<TC, D, NB, NQ, NF, NFQ>(st, g, ph, a);
      };
      l.av_sensor = [](hipStream_t st, const Geo& g, const Phys& ph, const double* U, double* node) {
        hipLaunchKernelGGL((avSensorKernel<D, NB, NQ>), dim3(blocksFor(g.E, kThreads)), dim3(kThreads),
                           0, st, g, ph, U, node);
      };
    }
    if constexpr (ADJOINT && sizeof(TC) == 8) {
      l.adj_volume[0] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
        hipLaunchKernelGGL((nsAdjVolumeMfma<D, NB, NQ, NF, NFQ, 1>), dim3(blocksFor(g.E, EPB_G)),
                           dim3(AdjShape<D, NB, NQ, NF * NFQ>::NT), 0, st, g, ph, a, j);
      };
      l.adj_volume[1] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
        hipLaunchKernelGGL((nsAdjVolumeMfma<D, NB, NQ, NF, NFQ, 2>), dim3(blocksFor(g.E, EPB_G)),
                           dim3(AdjShape<D, NB, NQ, NF * NFQ>::NT), 0, st, g, ph, a, j);
      };
      l.adj_face = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
        if (ph.flux <= SDG_FLUX_ROE)  // reverse mode, one thread per face point
          hipLaunchKernelGGL((nsAdjFaceRevKernel<D, NF, NFQ>), dim3(blocksFor(g.F * NFQ, kThreads)),
                             dim3(kThreads), 0, st, g, ph, a, j);
        else  // dual numbers, one thread per (state component or gradient, side, face point)
          hipLaunchKernelGGL((nsAdjFaceKernel<D, NF, NFQ>),
                             dim3(blocksFor(g.F * NFQ * 2 * (D + 3), kThreads)),
                             dim3(kThreads), 0, st, g, ph, a, j);
      };
      l.adj_lift[0] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
        hipLaunchKernelGGL((nsAdjLiftMfma<D, NB, NQ, NF, NFQ, 1>), dim3(blocksFor(g.E, EPB_G)),
                           dim3(AdjShape<D, NB, NQ, NF * NFQ>::NT), 0, st, g, ph, a, j);
      };
      l.adj_lift[1] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
        hipLaunchKernelGGL((nsAdjLiftMfma<D, NB, NQ, NF, NFQ, 2>), dim3(blocksFor(g.E, EPB_G)),
                           dim3(AdjShape<D, NB, NQ, NF * NFQ>::NT), 0, st, g, ph, a, j);
      };
      l.adj_gather = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
        hipLaunchKernelGGL((nsAdjGatherMfma<D, NB, NQ, NF, NFQ>), dim3(blocksFor(g.E, EPB_S)),
                           dim3(AdjShape<D, NB, NQ, NF * NFQ>::NT), 0, st, g, ph, a, j);
      };
    }
  } else {
    l.euler = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      hipLaunchKernelGGL((eulerStageKernel<D, NB, NQ, NF, NFQ, EPB>), dim3(blocksFor(g.E, EPB)),
                         dim3(kThreads), 0, st, g, ph, a);
    };
    l.ns_grad_br1 = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      hipLaunchKernelGGL((nsGradKernel<D, NB, NQ, NF, NFQ, EPB, 1>), dim3(blocksFor(g.E, EPB)),
                         dim3(kThreads), 0, st, g, ph, a);
    };
    l.ns_grad_br2 = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      hipLaunchKernelGGL((nsGradKernel<D, NB, NQ, NF, NFQ, EPB, 2>), dim3(blocksFor(g.E, EPB)),
                         dim3(kThreads), 0, st, g, ph, a);
    };
    l.ns_flux = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      hipLaunchKernelGGL((nsFluxKernel<D, NB, NQ, NF, NFQ, EPB>), dim3(blocksFor(g.E, EPB)), dim3(kThreads),
                         0, st, g, ph, a);
    };
    l.av_grad = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      hipLaunchKernelGGL((nsGradKernel<D, NB, NQ, NF, NFQ, EPB, 0>), dim3(blocksFor(g.E, EPB)),
                         dim3(kThreads), 0, st, g, ph, a);
    };
    l.av_flux = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      hipLaunchKernelGGL((nsFluxKernel<D, NB, NQ, NF, NFQ, EPB, 1>), dim3(blocksFor(g.E, EPB)),
                         dim3(kThreads), 0, st, g, ph, a);
    };
    l.av_ns_grad[0] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      hipLaunchKernelGGL((nsGradKernel<D, NB, NQ, NF, NFQ, EPB, 1, true>), dim3(blocksFor(g.E, EPB)),
                         dim3(kThreads), 0, st, g, ph, a);
    };
    l.av_ns_grad[1] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      hipLaunchKernelGGL((nsGradKernel<D, NB, NQ, NF, NFQ, EPB, 2, true>), dim3(blocksFor(g.E, EPB)),
                         dim3(kThreads), 0, st, g, ph, a);
    };
    l.av_ns_flux = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
      hipLaunchKernelGGL((nsFluxKernel<D, NB, NQ, NF, NFQ, EPB, 2>), dim3(blocksFor(g.E, EPB)),
                         dim3(kThreads), 0, st, g, ph, a);
    };
    l.av_sensor = [](hipStream_t st, const Geo& g, const Phys& ph, const double* U, double* node) {
      hipLaunchKernelGGL((avSensorKernel<D, NB, NQ>), dim3(blocksFor(g.E, kThreads)), dim3(kThreads), 0,
                         st, g, ph, U, node);
    };
  }
  if constexpr (MFMA) {
    // the stage tail's own contraction (bit-identical traces after a host-side state change)
    l.trace = [](hipStream_t st, const Geo& g, const double* U, void* Uf, const MixRef& mix) {
      hipLaunchKernelGGL((mfmaTraceKernel<TC, D, NB, NF, NFQ>), dim3(blocksFor(g.E, 16 / (D + 2))),
                         dim3(MfmaShape<NB, NB, NF * NFQ>::NT), 0, st, g, U, Uf, mix);
    };
  } else {
    l.trace = [](hipStream_t st, const Geo& g, const double* U, void* Uf, const MixRef& mix) {
      const int64_t n = static_cast<int64_t>(g.E) * (D + 2) * NF * NFQ;
      hipLaunchKernelGGL((traceKernel<D, NB, NQ, NF, NFQ>), dim3((n + kThreads - 1) / kThreads),
                         dim3(kThreads), 0, st, g, U, Uf, mix);
    };
  }
  l.source = [](hipStream_t st, const Geo& g, const Phys& ph, const double* U, double* out, const double* Li) {
    constexpr int NM = NQ > NB ? NQ : NB, EPBS = kThreads / NM > 0 ? kThreads / NM : 1;
    hipLaunchKernelGGL((sourceKernel<D, NB, NQ>), dim3(blocksFor(g.E, EPBS)), dim3(kThreads), 0, st, g, ph,
                       U, out, Li);
  };
  l.br2_blocks = [](hipStream_t st, const Geo& g, const Phys& ph, const double* U, double* out) {
    hipLaunchKernelGGL((br2BoundaryBlockKernel<D, NB, NQ, NF, NFQ>), dim3(g.Fb), dim3(kThreads), 0, st, g, ph,
                       U, out);
  };
  l.dt = [](hipStream_t st, const Geo& g, const Phys& ph, const double* U, const double* me, double cfl, int order,
            double* out) {
    hipLaunchKernelGGL((dtKernel<D, NB, NQ, NF, NFQ>), dim3(blocksFor(g.E, DtShape<D, NB, NQ>::EPB)),
                       dim3(kThreads), 0, st, g, ph, U, me, cfl, order, out);
  };
  l.monitor = [](hipStream_t st, const double* mon, int E, double* rel, int* status) {
    // mon holds E x NV per-element values followed by kMonitorBlocks x NV partial sums
    double* part = const_cast<double*>(mon) + static_cast<int64_t>(E) * (D + 2);
    hipLaunchKernelGGL((monitorKernel<D + 2>), dim3(monitorBlocks(E, D + 2)), dim3(kThreads), 0, st, mon, E, part, rel,
                       status);
  };
  return l;
}

// Kernel set for (element type, order). Mixed precision runs on the matrix-core kernels only.
template <int D, int NB, int NQ, int NF, int NFQ>
bool pickMfma(bool force_valu, bool mixed, Launchers& l) {
  if (mixed)
    l = makeLaunchers<D, NB, NQ, NF, NFQ, true, float>();
  else
    l = force_valu ? makeLaunchers<D, NB, NQ, NF, NFQ, false>() : makeLaunchers<D, NB, NQ, NF, NFQ, true>();
  return true;
}
// Simplices: the FP64 matrix-core kernels, without the mixed mode and the adjoint of pickMfma
template <int D, int NB, int NQ, int NF, int NFQ>
bool pickSimplex(bool force_valu, bool mixed, Launchers& l) {
  if (mixed) return false;
  l = force_valu ? makeLaunchers<D, NB, NQ, NF, NFQ, false>() : makeLaunchers<D, NB, NQ, NF, NFQ, true, double, false>();
  return true;
}
template <int D, int NB, int NQ, int NF, int NFQ>
bool pickValu(bool mixed, Launchers& l) {
  if (mixed) return false;
  l = makeLaunchers<D, NB, NQ, NF, NFQ, false>();
  return true;
}

// Navier-Stokes on hexahedra P2..P4: the sum-factorised stage kernels replace the matrix-core
// gradient and residual kernels (the face-flux kernel, the adjoint kernels and Euler stay).
template <typename TC, int N>
void useTensorKernels(Launchers& l) {
  constexpr int EPB = TensorShape<N>::EPB, TPB = TensorShape<N>::TPB;
  l.ns_grad_br1 = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
    hipLaunchKernelGGL((nsGradTensor<TC, N, 1>), dim3(blocksFor(g.E, EPB)), dim3(TPB), 0, st, g, ph, a);
  };
  l.ns_grad_br2 = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
    hipLaunchKernelGGL((nsGradTensor<TC, N, 2>), dim3(blocksFor(g.E, EPB)), dim3(TPB), 0, st, g, ph, a);
  };
  // face fluxes from the elements' own normal viscous fluxes (written by the gradient kernel)
  l.ns_face = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
    constexpr int NFQ = N * N;
    hipLaunchKernelGGL((nsFaceFluxKernel<TC, 3, 6, NFQ, true>), dim3(blocksFor((g.F + g.Fb) * NFQ, kThreads)),
                       dim3(kThreads), 0, st, g, ph, a);
  };
  l.ns_flux = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
    hipLaunchKernelGGL((nsResidualTensor<TC, N>), dim3(blocksFor(g.E, EPB)), dim3(TPB), 0, st, g, ph,
                       a);
  };
  l.trace = [](hipStream_t st, const Geo& g, const double* U, void* Uf, const MixRef& mix) {
    hipLaunchKernelGGL((tensorTraceKernel<TC, N>), dim3(blocksFor(g.E, EPB)), dim3(TPB), 0, st, g, U,
                       Uf, mix);
  };
  // the transpose of these stage kernels, FP64 in both precision modes: a mixed-precision context's
  // adjoint differentiates the FP64 residual at the states of its run, on FP64 traces (trace64)
  l.trace64 = [](hipStream_t st, const Geo& g, const double* U, void* Uf, const MixRef& mix) {
    hipLaunchKernelGGL((tensorTraceKernel<double, N>), dim3(blocksFor(g.E, EPB)), dim3(TPB), 0, st, g, U, Uf, mix);
  };
  l.adj_volume[0] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
    hipLaunchKernelGGL((nsAdjVolumeTensor<N, 1>), dim3(blocksFor(g.E, EPB)), dim3(TPB), 0, st, g, ph, a, j);
  };
  l.adj_volume[1] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
    hipLaunchKernelGGL((nsAdjVolumeTensor<N, 2>), dim3(blocksFor(g.E, EPB)), dim3(TPB), 0, st, g, ph, a, j);
  };
  l.adj_face = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
    constexpr int NFQ = N * N;
    if (ph.flux <= SDG_FLUX_ROE)
      hipLaunchKernelGGL((nsAdjFaceRevKernel<3, 6, NFQ>), dim3(blocksFor(g.F * NFQ, kThreads)),
                         dim3(kThreads), 0, st, g, ph, a, j);
    else
      hipLaunchKernelGGL((nsAdjFaceKernel<3, 6, NFQ>), dim3(blocksFor(g.F * NFQ * 2 * 6, kThreads)),
                         dim3(kThreads), 0, st, g, ph, a, j);
  };
  l.adj_lift[0] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
    hipLaunchKernelGGL((nsAdjLiftTensor<N, 1>), dim3(blocksFor(g.E, EPB)), dim3(TPB), 0, st, g, ph, a, j);
  };
  l.adj_lift[1] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
    hipLaunchKernelGGL((nsAdjLiftTensor<N, 2>), dim3(blocksFor(g.E, EPB)), dim3(TPB), 0, st, g, ph, a, j);
  };
  l.adj_gather = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
    hipLaunchKernelGGL((nsAdjGatherTensor<N>), dim3(blocksFor(g.E, EPB)), dim3(TPB), 0, st, g, ph, a, j);
  };
  l.tensor = true;
}
// Navier-Stokes (BR1 or BR2, FP64 or mixed) with artificial viscosity on the sum-factorised kernels: the
// gradient kernel adds eps grad U (the volume gradient) to the volume flux and to each side's normal
// viscous flux, boundary points keep the volume-gradient trace (GfV) for the boundary flux
template <typename TC, int N>
void useTensorAvKernels(Launchers& l) {
  constexpr int EPB = TensorShape<N>::EPB, TPB = TensorShape<N>::TPB;
  l.av_ns_grad[0] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
    hipLaunchKernelGGL((nsGradTensor<TC, N, 1, true>), dim3(blocksFor(g.E, EPB)), dim3(TPB), 0, st, g, ph, a);
  };
  l.av_ns_grad[1] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
    hipLaunchKernelGGL((nsGradTensor<TC, N, 2, true>), dim3(blocksFor(g.E, EPB)), dim3(TPB), 0, st, g, ph, a);
  };
  l.ns_face = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
    constexpr int NFQ = N * N;
    hipLaunchKernelGGL((nsFaceFluxKernel<TC, 3, 6, NFQ, true, true>),
                       dim3(blocksFor((g.F + g.Fb) * NFQ, kThreads)), dim3(kThreads), 0, st, g, ph, a);
  };
  l.av_ns_flux = l.ns_flux;
}
template <typename TC>
bool selectTensorAvT(int order, Launchers& l) {
  switch (order) {
    case 2: useTensorAvKernels<TC, 3>(l); return true;
    case 3: useTensorAvKernels<TC, 4>(l); return true;
    case 4: useTensorAvKernels<TC, 5>(l); return true;
    default: return false;
  }
}
// Quadrangles, FP64: the sum-factorised stage kernels replace those of every stage, and their
// transpose the adjoint kernels where the size has an adjoint. 256^2 P3 Euler with artificial viscosity: 95 us of kernels a stage, 260 us on the matrix-core
// kernels; 48^2 P3 Navier-Stokes: 14.3 us and 28 us; 32^2 P2 Euler: 7.1 us and 8.5 us on the vector kernel.
template <int N>
bool pickQuad(Launchers& l) {
  constexpr int EPB = QuadShape<N>::EPB;
  l.ns_grad_br1 = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
    hipLaunchKernelGGL((quadGrad<N, 1>), dim3(blocksFor(g.E, EPB)), dim3(64), 0, st, g, ph, a);
  };
  l.ns_grad_br2 = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
    hipLaunchKernelGGL((quadGrad<N, 2>), dim3(blocksFor(g.E, EPB)), dim3(64), 0, st, g, ph, a);
  };
  l.av_grad = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
    hipLaunchKernelGGL((quadGrad<N, 0>), dim3(blocksFor(g.E, EPB)), dim3(64), 0, st, g, ph, a);
  };
  l.ns_face = nullptr;
  l.ns_flux = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
    hipLaunchKernelGGL((quadResidual<N, 0>), dim3(blocksFor(g.E, EPB)), dim3(64), 0, st, g, ph, a);
  };
  l.av_flux = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
    hipLaunchKernelGGL((quadResidual<N, 1>), dim3(blocksFor(g.E, EPB)), dim3(64), 0, st, g, ph, a);
  };
  l.euler = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a) {
    hipLaunchKernelGGL((quadResidual<N, 2>), dim3(blocksFor(g.E, EPB)), dim3(64), 0, st, g, ph, a);
  };
  l.trace = [](hipStream_t st, const Geo& g, const double* U, void* Uf, const MixRef&) {
    hipLaunchKernelGGL((quadTraceKernel<N>), dim3(blocksFor(g.E, EPB)), dim3(64), 0, st, g, U, static_cast<double*>(Uf));
  };
  if (l.adj_face) {  // P3..P5: the transpose of these kernels (the face kernel is the generic one)
    l.adj_volume[0] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
      hipLaunchKernelGGL((quadAdjVolume<N, 1>), dim3(blocksFor(g.E, EPB)), dim3(64), 0, st, g, ph, a, j);
    };
    l.adj_volume[1] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
      hipLaunchKernelGGL((quadAdjVolume<N, 2>), dim3(blocksFor(g.E, EPB)), dim3(64), 0, st, g, ph, a, j);
    };
    l.adj_lift[0] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
      hipLaunchKernelGGL((quadAdjLift<N, 1>), dim3(blocksFor(g.E, EPB)), dim3(64), 0, st, g, ph, a, j);
    };
    l.adj_lift[1] = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
      hipLaunchKernelGGL((quadAdjLift<N, 2>), dim3(blocksFor(g.E, EPB)), dim3(64), 0, st, g, ph, a, j);
    };
    l.adj_gather = [](hipStream_t st, const Geo& g, const Phys& ph, const StageArgs& a, const AdjArgs& j) {
      hipLaunchKernelGGL((quadAdjGather<N>), dim3(blocksFor(g.E, EPB)), dim3(64), 0, st, g, ph, a, j);
    };
  }
  l.quad = true;
  return true;
}

// Lines: the vector kernels, and the whole-run kernels of small Euler meshes
template <int N>
bool pickLine(bool mixed, Launchers& l) {
  if (!pickValu<1, N, N, 2, 1>(mixed, l)) return false;
  l.line_run[0] = [](hipStream_t st, const Geo& g, const Phys& ph, const LineRun& a) {
    hipLaunchKernelGGL((lineRunKernel<N, false>), dim3(1), dim3((g.E + 63) / 64 * 64), 0, st, g, ph, a);
  };
  l.line_run[1] = [](hipStream_t st, const Geo& g, const Phys& ph, const LineRun& a) {
    hipLaunchKernelGGL((lineRunKernel<N, true>), dim3(1), dim3((g.E + 63) / 64 * 64), 0, st, g, ph, a);
  };
  return true;
}

template <int N>
bool pickTensor(bool mixed, Launchers& l) {
  if (mixed)
    useTensorKernels<float, N>(l);
  else
    useTensorKernels<double, N>(l);
  return true;
}

// Kernel set of an element type and order; false where there is none. force_valu: the vector kernels.
bool selectLine(int order, bool mixed, Launchers& l);
bool selectTriangle(int order, bool force_valu, bool mixed, Launchers& l);
bool selectQuadrangle(int order, bool force_valu, bool mixed, Launchers& l);
bool selectTetrahedron(int order, bool force_valu, bool mixed, Launchers& l);
bool selectPyramid(int order, bool mixed, Launchers& l);
bool selectHexahedron(int order, bool force_valu, bool mixed, Launchers& l);
// hexahedra P2..P4, Navier-Stokes: replaces the stage kernels by the sum-factorised ones
bool selectTensor(int order, bool mixed, Launchers& l);
// quadrangles P1..P5, FP64: replaces the stage kernels by the sum-factorised ones
bool selectQuadTensor(int order, Launchers& l);
// the hexahedra's kernels with artificial viscosity, after selectTensor
bool selectTensorAv(int order, bool mixed, Launchers& l);

}  // namespace sdg

#endif  // SDG_LAUNCHERS_HPP_
