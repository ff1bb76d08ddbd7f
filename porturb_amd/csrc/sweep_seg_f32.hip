// sweep_seg_f32.hip -- the FP32 segment sweeps (k_sweep<ORD, float, DIR, MODE>, sweep_f32_core.h) in a
// translation unit of their own, for parallel compilation; like all sweeps built with -mllvm
// -disable-machine-licm (porturb_amd/build.py): the x sweep then takes 70 VGPRs at WENO-9 without spills.
#include "sweep_f32_core.h"

namespace pu {

template <int ORD>
static void launch_ord(int dir, bool combine, hipStream_t s, const float *prim, const uint16_t *codes, float *tend,
                       const SweepParams &P, const FuseArgs<float> &FA) {
  using X = f32::SegShape<0>;
  using L = f32::SegShape<1>;
  constexpr int NL = L::BS - 2;
  const dim3 bx(X::BX, X::BY), bl(L::BX, L::BY);
  const unsigned wx = (unsigned)((P.nx + L::BX - 1) / L::BX);
  if (dir == 0) {
    static_assert(X::BX == SX_BX && X::BY == SX_BY, "x_position");
    const dim3 grd(x_blocks(P.nx, P.ny), 1, (unsigned)P.nz);
    if (combine) hipLaunchKernelGGL((f32::k_sweep<ORD, float, 0, 2>), grd, bx, 0, s, prim, codes, tend, P, FA);
    else hipLaunchKernelGGL((f32::k_sweep<ORD, float, 0, 1>), grd, bx, 0, s, prim, codes, tend, P, FA);
  } else if (dir == 1) {
    const dim3 grd(wx, (unsigned)((P.ny + NL - 1) / NL), (unsigned)P.nz);
    hipLaunchKernelGGL((f32::k_sweep<ORD, float, 1, 1>), grd, bl, 0, s, prim, codes, tend, P, FA);
  } else {
    const dim3 grd(wx, (unsigned)P.ny, (unsigned)((P.nz + NL - 1) / NL));
    hipLaunchKernelGGL((f32::k_sweep<ORD, float, 2, 0>), grd, bl, 0, s, prim, codes, tend, P, FA);
  }
}

int launch_seg_f32(int ord, int dir, bool combine, hipStream_t s, const float *prim, const uint16_t *codes, float *tend,
                   const SweepParams &P, const FuseArgs<float> &FA) {
  switch (ord) {
    case 3: launch_ord<3>(dir, combine, s, prim, codes, tend, P, FA); break;
    case 5: launch_ord<5>(dir, combine, s, prim, codes, tend, P, FA); break;
    case 7: launch_ord<7>(dir, combine, s, prim, codes, tend, P, FA); break;
    case 9: launch_ord<9>(dir, combine, s, prim, codes, tend, P, FA); break;
    case 11: launch_ord<11>(dir, combine, s, prim, codes, tend, P, FA); break;
    default: return fail(PU_ERR_UNSUPPORTED, "unsupported ord");
  }
  PU_HIP_CHECK(hipGetLastError());
  return PU_OK;
}

}  // namespace pu
