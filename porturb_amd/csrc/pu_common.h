// pu_common.h -- internal definitions shared by the HIP kernels and the C ABI of libporturb.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstddef>
#include <type_traits>
#include <string>
#include <map>
#include <vector>
#include "porturb.h"

namespace pu {

// Conserved-state indices (dynamics_rk.h:33-38) and the pressure slot of the reconstructed
// fields (dynamics_rk.h:496).
constexpr int idR = 0, idU = 1, idV = 2, idW = 3, idT = 4, idP = 5, NUM_STATE = 5;

// Reconstruction halo of the primitive-field array: hs cells for the stencils of interior cells
// plus one more for the neighbour-cell reconstruction each line segment needs at its ends.
__host__ __device__ constexpr int prim_halo(int hs) { return hs + 1; }

// x position of interior cell 0 in the primitive-field and flag arrays, and the alignment of their
// rows (elements): rows start on 128-byte boundaries for float and double and the interior of
// every row starts on one, so the row segments the kernels read and write map onto whole cache
// lines.  PRIM_OX >= prim_halo(hs) for every order.
constexpr int PRIM_OX = 32, PRIM_ROW_ALIGN = 32;

struct Grid {
  int nx, ny, nz, hs, hp;          // hp = prim_halo(hs)
  int ox;                          // x offset of the interior (PRIM_OX); y/z offsets are hp
  long long nxh, nyh, nzh;         // extents of the primitive-field array (nxh: padded row pitch)
  long long n3() const { return (long long)nx * ny * nz; }
  long long nh() const { return nxh * nyh * nzh; }
};

// Timing of one kernel family with HIP events around each launch.
struct KernelTimer {
  double total_ms = 0;
  long long count = 0;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> pending;
};

}  // namespace pu

struct pu_ctx {
  pu_config cfg;
  hipStream_t stream = nullptr;
  int device = 0;                  // the HIP device current when the context was created
  pu::Grid g{};
  int nv = 0;                      // 5 + num_tracers  (conserved variables)
  int nf = 0;                      // nv + 1           (reconstructed fields incl. pressure)
  bool dycore_ready = false;
  bool les_ready = false;
  // kernels of the y and z sweeps ([1], [2]): by the rule of rule_takes_segments or, where the environment variable
  // PORTURB_SEGMENT_SWEEPS is set when the context is created, segments in the directions of
  // PORTURB_SEGMENT_DIRS (both if that is not set) and whole lines where they apply in the others
  enum SweepRoute { ROUTE_RULE, ROUTE_LINES, ROUTE_SEGMENTS } sweep_route[3] = {ROUTE_RULE, ROUTE_RULE, ROUTE_RULE};
  // hydrostatic background, FP64 (host + device copies)
  std::vector<double> hy_cells[3];     // dens, theta, pressure: [nz+2hs]
  std::vector<double> hy_edges[3];     // [nz+1]
  double *d_hy = nullptr;              // device: [3*(nz+2hs)] cells then [3*(nz+1)] edges
  // immersed data
  uint16_t *d_codes = nullptr;         // stencil codes along x, y, z [3][n3] (sweep_core.h SC_*)
  uint8_t *d_any10 = nullptr;          // dycore_any_immersed10 [n3]
  int     *d_tau = nullptr;            // dycore_immersed_tau [n3]
  double  *d_relax = nullptr;          // pow(prop, immersed_power)/tau [n3]
  uint8_t *d_imm_les = nullptr;        // immersed_proportion_halos (hs=1) as 0 / partial / 1 codes
  double  *d_imm_les_val = nullptr;    // immersed_proportion_halos values [nz+2][ny+2][nx+2]
  // dycore work arrays (element type follows cfg.precision)
  void *d_U = nullptr, *d_Us = nullptr;        // [nv][n3]
  void *d_Ulo = nullptr, *d_Uslo = nullptr;    // FP32 only: compensation of rho, rho*theta [2][n3]
  void *d_tend = nullptr;                      // [nv][n3]
  void *d_prim = nullptr;                      // [nf][nzh][nyh][nxh]
  // LES work arrays
  double *d_les = nullptr;                     // primitive closure state, halo 1
  // learned subgrid closure (attached network, its per-cell outputs and the static mask of cells
  // whose level and 3x3x3 neighbourhood allow it)
  const pu_mlp *sgs_model = nullptr;
  float   *d_sgs_tau = nullptr;                // [3][n3][4]: per face direction d, (tau_0d, tau_1d, tau_2d, q_d)
  uint8_t *d_sgs_flags = nullptr;              // [n3]
  uint8_t *d_sgs_valid = nullptr;              // [n3]
  float   *d_sgs_fmul = nullptr;               // [108]
  bool     sgs_valid_ready = false;
  // surface fluxes: halo'd immersed roughness and temperature boxes
  double  *d_sfc_rough = nullptr, *d_sfc_temp = nullptr;
  bool     sfc_ready = false;
  // horizontal means per level (forcing modules): [3][nz] means + [3][nz][16] partial sums
  double  *d_col = nullptr;
  // reductions
  double *d_red = nullptr;                     // scratch for reductions
  // timing
  hipEvent_t t0 = nullptr, t1 = nullptr;
  bool kernel_timing = false;
  std::map<std::string, pu::KernelTimer> timers;
};

namespace pu {

void set_error(const std::string &msg);
int  fail(int code, const std::string &msg);

#define PU_HIP_CHECK(expr)                                                                  \
  do {                                                                                      \
    hipError_t _e = (expr);                                                                 \
    if (_e != hipSuccess)                                                                   \
      return ::pu::fail(PU_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(_e));     \
  } while (0)

// XCD-aware block order.  The dispatcher hands workgroups to the 8 XCDs of an MI355X round-robin
// by linear workgroup id, and each XCD has its own L2; blocks that share cache lines (x-neighbours)
// should therefore run on the same XCD.  This maps the hardware id so that consecutive logical
// ids land on one XCD: hardware id h (XCD h % 8, slot h / 8) -> logical id
// start(XCD) + slot, a bijection on [0, nblocks).
__device__ __forceinline__ unsigned xcd_swizzle(unsigned h, unsigned nblocks) {
  const unsigned nx = 8, q = nblocks / nx, r = nblocks % nx;
  const unsigned xcd = h % nx, slot = h / nx;
  return xcd < r ? xcd * (q + 1) + slot : r * (q + 1) + (xcd - r) * q + slot;
}

// Logical 3-D block index of the current workgroup after the swizzle (x fastest).
__device__ __forceinline__ void swizzled_block(unsigned &bx, unsigned &by, unsigned &bz) {
  const unsigned nb = gridDim.x * gridDim.y * gridDim.z;
  const unsigned h = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  const unsigned l = xcd_swizzle(h, nb);
  bx = l % gridDim.x;
  by = (l / gridDim.x) % gridDim.y;
  bz = l / (gridDim.x * gridDim.y);
}

// Reciprocal of a positive, normal argument: v_rcp_f32 in FP32; in FP64 v_rcp_f64 (2^-24) refined by
// one third-order step, r (1 + e + e^2) with e = 1 - x r: its error e^3 is below 2^-70, so the result
// is as accurate as after two Newton steps with one multiply-add less.
template <class T> __device__ __forceinline__ T recip(T x) {
  if constexpr (std::is_same<T, float>::value) {
    return __builtin_amdgcn_rcpf(x);
  } else {
    const double r = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, r, 1.0);
    return fma(r, fma(e, e, e), r);
  }
}

// x^a in FP64 for 0 < x < inf and |a ln x| < 700 (anything else goes to the library's pow): exp(a ln x)
// with the logarithm and the product held as sums of two doubles, so that the result is off by little
// more than its last rounding.  ln m, m in [sqrt(1/2), sqrt(2)), is 2 atanh s, s = (m - 1) / (m + 1); the
// series in s^2 <= 0.0295 and the Taylor terms of exp on |r| <= ln(2) / 2 end below 2^-57 of the result.
// About 80 instructions on the way through, the library's pow 226.
// Against 80-bit powl over [1e-5, 1e6] with exponents 1.4, 1/1.4, 0.4 and -2.5: at most 0.69 ulp, rms 0.290
// (the library's: 1.36 and 0.42).
__device__ __forceinline__ double pow_pos(double x, double a) {
  constexpr double LN2_HI = 0x1.62e42fee00000p-1, LN2_LO = 0x1.a39ef35793c76p-33;     // LN2_HI: 33 bits, its multiples are exact
  double m = __builtin_amdgcn_frexp_mant(x);
  const bool low = m < 0.70710678118654752;
  m = low ? m + m : m;
  const double k = (double)(__builtin_amdgcn_frexp_exp(x) - (low ? 1 : 0));
  const double n = m - 1., d = m + 1., dl = m - (d - 1.);                             // m + 1 = d + dl
  const double rd = recip(d), s = n * rd, sl = fma(-s, dl, fma(-s, d, n)) * rd, z = s * s;
  double p = 2. / 21.;
  p = fma(p, z, 2. / 19.);
  p = fma(p, z, 2. / 17.);
  p = fma(p, z, 2. / 15.);
  p = fma(p, z, 2. / 13.);
  p = fma(p, z, 2. / 11.);
  p = fma(p, z, 2. / 9.);
  p = fma(p, z, 2. / 7.);
  p = fma(p, z, 2. / 5.);
  p = fma(p, z, 2. / 3.);
  const double k0 = k * LN2_HI, s2 = s + s, lh = k0 + s2;                             // ln x = lh + ll
  const double ll = (s2 - (lh - k0)) + fma(k, LN2_LO, fma(s * z, p, sl + sl));
  const double yh = a * lh, yl = fma(a, ll, fma(a, lh, -yh));
  if (!(x > 0. && x < HUGE_VAL && fabs(yh) < 700.)) return pow(x, a);
  const double q = rint(yh * 1.4426950408889634);
  const double r0 = fma(-q, LN2_HI, yh), c = fma(-q, LN2_LO, yl), r = r0 + c, rl = c - (r - r0);
  double e = 1. / 6227020800.;
  e = fma(e, r, 1. / 479001600.);
  e = fma(e, r, 1. / 39916800.);
  e = fma(e, r, 1. / 3628800.);
  e = fma(e, r, 1. / 362880.);
  e = fma(e, r, 1. / 40320.);
  e = fma(e, r, 1. / 5040.);
  e = fma(e, r, 1. / 720.);
  e = fma(e, r, 1. / 120.);
  e = fma(e, r, 1. / 24.);
  e = fma(e, r, 1. / 6.);
  e = fma(e, r, 0.5);
  const double h = 1. + r;
  return ldexp(h + (fma(r * r, e, rl) + (r - (h - 1.))), (int)q);
}

// Square root.  FP64: v_rsq_f64 refined by Goldschmidt's iteration and one residual step, without the library's
// scaling of every argument.  It is the library's result for every normal argument tried (12 million in
// [1e-290, 1e290]); below 1e-290 the residual underflows and the last bits differ.  Zero and +inf, where the
// iteration meets 0 * inf, are their own roots; negative arguments and NaN give NaN.
__device__ __forceinline__ float root(float x) { return sqrtf(x); }
__device__ __forceinline__ double root(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, q = 0.5 * y;
  const double e = fma(-q, g, 0.5);
  g = fma(g, e, g);
  q = fma(q, e, q);
  g = fma(fma(-g, g, x), q, g);
  return __builtin_amdgcn_class(x, 0x260) ? x : g;      // -0, +0, +inf
}

// Tracer pointer bundles passed by value to kernels.
struct TracerPtrs { double *p[PU_MAX_TRACERS]; };
struct TracerPtrsC { const double *p[PU_MAX_TRACERS]; };

// Kernel-timing helpers: record events around a launch when timing is enabled.
struct LaunchTimer {
  pu_ctx *ctx; const char *name; hipEvent_t a = nullptr, b = nullptr;
  LaunchTimer(pu_ctx *c, const char *n) : ctx(c), name(n) {
    if (ctx->kernel_timing) {
      hipEventCreate(&a); hipEventCreate(&b);
      hipEventRecord(a, ctx->stream);
    }
  }
  ~LaunchTimer() {
    if (ctx->kernel_timing) {
      hipEventRecord(b, ctx->stream);
      ctx->timers[name].pending.emplace_back(a, b);
    }
  }
};

void collect_timers(pu_ctx *ctx);

// Launchers implemented in the kernel translation units.
int launch_prep(pu_ctx *ctx, const void *U, const void *Ulo, hipStream_t s);
int launch_c2d_prep(pu_ctx *ctx, const pu_coupler_state *cs, hipStream_t s);
// Sweeps z, y, x.  stage < 0: tendencies into d_tend; stage 0..2: the x sweep also applies the
// stage combination (sources, SSPRK3 stage, clip, nrelax immersed relaxations) for every cell it
// finishes
int launch_sweeps(pu_ctx *ctx, hipStream_t s, int stage = -1, double dt = 0., int nrelax = 0);
// whether the y (dir 1) or z (dir 2) sweep of a grid takes the segment kernel when no route is forced
bool rule_takes_segments(const pu_config &c, const Grid &g, int dir);
int launch_convert_c2d(pu_ctx *ctx, const pu_coupler_state *cs, int relax, hipStream_t s);
int launch_convert_d2c(pu_ctx *ctx, pu_coupler_state *cs, hipStream_t s);
int launch_tend_export(pu_ctx *ctx, double *tend, hipStream_t s);
int launch_census(pu_ctx *ctx, hipStream_t s, unsigned long long *counts);
int dycore_init_device(pu_ctx *ctx, const pu_coupler_state *cs);
int les_apply_device(pu_ctx *ctx, pu_coupler_state *cs, double dt);
int les_prim_device(pu_ctx *ctx, const pu_coupler_state *cs);   // closure box d_les only
// learned closure: prediction and flags into ctx->d_sgs_tau / d_sgs_flags from ctx->d_les
int sgs_infer_device(pu_ctx *ctx, double dt);
int les_init_device(pu_ctx *ctx, const pu_coupler_state *cs);
int fill_device(double *ptr, double value, size_t count);
int copy_device(void *dst, const void *src, size_t bytes);
// k_copy of bytes (a multiple of 16, 16-byte aligned pointers) on stream s, not waited for
int launch_copy(void *dst, const void *src, size_t bytes, hipStream_t s);
int les_set_immersed_halos_device(pu_ctx *ctx, const double *halos);
int diagnostics_device(pu_ctx *ctx, const pu_coupler_state *cs, double *mass, double *maxw, double *maxabsw);
int case_init_device(const pu_config *cfg, int case_id, unsigned long long seed, pu_coupler_state *cs,
                     double *imm, hipStream_t s);

}  // namespace pu
