// sweep_zwall_f32.hip -- the FP32 whole-column z sweep (f32::k_sweep_zwall<ORD, float>, sweep_f32_core.h) in
// a translation unit of its own, for parallel compilation; like all sweeps built with -mllvm
// -disable-machine-licm (porturb_amd/build.py):
// without it the compiler hoists the limiter's constants out of the chunk loop into registers and
// the kernel loses a wave per SIMD.
#include "sweep_f32_core.h"

namespace pu {

int launch_zwall_f32(int ord, dim3 grid, dim3 block, hipStream_t s, const float *prim, const uint16_t *codes,
                     float *tend, const SweepParams &P) {
  switch (ord) {
    case 3: hipLaunchKernelGGL((f32::k_sweep_zwall<3, float>), grid, block, 0, s, prim, codes, tend, P); break;
    case 5: hipLaunchKernelGGL((f32::k_sweep_zwall<5, float>), grid, block, 0, s, prim, codes, tend, P); break;
    case 7: hipLaunchKernelGGL((f32::k_sweep_zwall<7, float>), grid, block, 0, s, prim, codes, tend, P); break;
    case 9: hipLaunchKernelGGL((f32::k_sweep_zwall<9, float>), grid, block, 0, s, prim, codes, tend, P); break;
    case 11: hipLaunchKernelGGL((f32::k_sweep_zwall<11, float>), grid, block, 0, s, prim, codes, tend, P); break;
    default: return fail(PU_ERR_UNSUPPORTED, "unsupported ord");
  }
  PU_HIP_CHECK(hipGetLastError());
  return PU_OK;
}

}  // namespace pu
