// sweep_x_f32.hip -- the FP32 x sweep (k_sweep_x<ORD, float, MODE>, sweep_core.h) in a translation
// unit of its own, built with -mllvm -disable-machine-licm (porturb_amd/build.py).
#include "sweep_core.h"

namespace pu {

template <int ORD>
static void launch_ord(int mode, dim3 grid, dim3 block, hipStream_t s, const float *prim, const uint16_t *codes,
                       float *tend, const SweepParams &P, const FuseArgs<float> &FA) {
  if (mode == 2)
    hipLaunchKernelGGL((k_sweep_x<ORD, float, 2>), grid, block, 0, s, prim, codes, tend, P, FA);
  else
    hipLaunchKernelGGL((k_sweep_x<ORD, float, 1>), grid, block, 0, s, prim, codes, tend, P, FA);
}

int launch_x_f32(int ord, int mode, dim3 grid, dim3 block, hipStream_t s, const float *prim, const uint16_t *codes,
                 float *tend, const SweepParams &P, const FuseArgs<float> &FA) {
  switch (ord) {
    case 3: launch_ord<3>(mode, grid, block, s, prim, codes, tend, P, FA); break;
    case 5: launch_ord<5>(mode, grid, block, s, prim, codes, tend, P, FA); break;
    case 7: launch_ord<7>(mode, grid, block, s, prim, codes, tend, P, FA); break;
    case 9: launch_ord<9>(mode, grid, block, s, prim, codes, tend, P, FA); break;
    case 11: launch_ord<11>(mode, grid, block, s, prim, codes, tend, P, FA); break;
    default: return fail(PU_ERR_UNSUPPORTED, "unsupported ord");
  }
  PU_HIP_CHECK(hipGetLastError());
  return PU_OK;
}

}  // namespace pu
