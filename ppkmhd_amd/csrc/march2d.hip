// Single-pass 2D MHD step: one kernel reads the state once and writes the interior of the new
// state once (wave program and data flow: march2d_body.hpp).  The ghost cells of the new state
// come from the step's ghost fill, which writes each ghost value to both states.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "march2d_body.hpp"

namespace ppk {
namespace PPK_NS {
namespace march2k {

// One wave per strip (or pair of 32-column strips), four waves per block that do not interact.
// Bound by instruction issue (about 1,460 FP64 and 400 other instructions per row and wave, 4
// cycles each, reciprocals and square roots 16): two waves per SIMD at 256 registers (2
// spilled) take 1.9 times the time of one.  Measured per launch: 2048^2 0.287 ms (14.6 G
// cell-updates/s), where the three-kernel form's kernels take 0.875 ms, 1024^2 87 us, 256^2 23 us,
// 64^2 16 us.  HBM traffic 168 bytes per cell (the state once each way is 128).
// RS, ST, ISO: as k_march3d (Riemann solver; minmod factor fixed; isothermal branches).
template <int RS, int ST, int ISO>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_march2d(const double *__restrict__ Uin, double *__restrict__ Uout, double *__restrict__ parts,
          DevParams pk, double *ctrl, double *host, int fold) {
  if (ctrl[CTRL_ACTIVE] == 0.0) return;
  __shared__ double ring[kWaves * kRing];
  DevParams p = pk;
  if (!ISO) p.cIso = 0.0;
  if (ST) p.slope_type = double(ST);
  const int wave = threadIdx.x >> 6;
  const int w = xcd_remap(blockIdx.x, gridDim.x) * kWaves + wave;
  const Geom g = geom_of(p);
  if (w >= g.waves()) return;  // whole waves only
  if (w == 0 && threadIdx.x == 0) step_end(ctrl, host);
  const double m = march2d<RS>(Uin, Uout, p, g, w, ctrl[CTRL_DT], fold != 0, ring + wave * kRing);
  if (fold && (threadIdx.x & 63) == 0) parts[w] = m;
}

}  // namespace march2k

hipError_t march2d_godunov(const DevParams &p, const double *Uin, double *Uout, double *parts,
                           double *ctrl, double *host, int fold_cfl, hipStream_t s, StageTimer *tm) {
  using namespace march2k;
  const Geom g = geom_of(p);
  const dim3 grid((unsigned)((g.waves() + kWaves - 1) / kWaves)), block(64 * kWaves);
  if (tm) tm->mark(ST_FUSED_MARCH, true);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, s, Uin, Uout, parts, p, ctrl, host, fold_cfl);
  };
  const int minmod = p.slope_type == 1.0 ? 1 : 0, iso = p.cIso > 0 ? 1 : 0;
  auto pick = [&](auto rs) {
    constexpr int RS = decltype(rs)::value;
    if (minmod)
      iso ? launch(k_march2d<RS, 1, 1>) : launch(k_march2d<RS, 1, 0>);
    else
      iso ? launch(k_march2d<RS, 0, 1>) : launch(k_march2d<RS, 0, 0>);
  };
  switch (p.riemann) {
    case PPK_RIEMANN_HLLD: pick(std::integral_constant<int, PPK_RIEMANN_HLLD>{}); break;
    case PPK_RIEMANN_HLL: pick(std::integral_constant<int, PPK_RIEMANN_HLL>{}); break;
    default: pick(std::integral_constant<int, PPK_RIEMANN_LLF>{}); break;
  }
  if (tm) tm->mark(ST_FUSED_MARCH, false);
  return hipGetLastError();
}

}  // namespace PPK_NS
}  // namespace ppk
