// les_kernels.hip -- LES_Closure::apply (les_closure.h:30-323) on gfx950.
//
// Two launches per call:
//   k_les_prim   : coupler state -> primitive closure fields (rho_d, u, v, w, theta, K, q_l) on a
//                  halo-1 box, with the periodic/precursor x/y halos (coupler.h:785-851) and the
//                  z wall/periodic halos (les_closure.h:418-536) computed in place;
//   k_les_update : the face fluxes (:92-229), the TKE source (:233-278) and the forward-Euler update
//                  (:280-320) written straight back to the coupler entries (:375-414).  A block
//                  computes each face of its tile once and exchanges the fluxes between lanes and
//                  through LDS, so no flux arrays go to HBM.
// In the FP64 dycore mode the closure runs in double; in the FP32 mode its box, fluxes and
// tendencies are float and the tendencies are applied as increments to the double entries.
#include "pu_common.h"
#include <cmath>
#include <type_traits>

namespace pu {

struct LesParams {
  int nx, ny, nz, ntr_all, nq, idTKE, bc_x, bc_y, bc_z, enable_gravity, dns;
  long long nxh, nyh, nzh, nh, n3;
  int qidx[PU_MAX_TRACERS];        // tracer index of each diffused tracer
  double dx, dy, dz, delta, grav, nu, total_mult, diss_mult, shear_mult, dt;
  double visc_max_x, visc_max_y, visc_max_z;
  double rdelta, nu_pr, rR_d;      // 1 / delta, nu / Pr (Pr = 0.7), 1 / R_d
  double rdx, rdy, rdz;            // 1 / dx, 1 / dy, 1 / dz
  double R_d, C0, gamma;
  // learned closure: per-cell stresses/heat fluxes per face direction d, [3][n3] of
  // (tau_0d, tau_1d, tau_2d, q_d), and flags [n3] (null: eddy viscosity only)
  const float4 *tau;
  const unsigned char *sflags;
};

// The update's constants in its type (converted once on the host, not by every lane).
template <class T> struct LesNum {
  T rdx, rdy, rdz, r2dx, r2dy, r2dz, delta, rdelta, grav, nu, nu_pr, mix, diss, shear, dt, gamma;
  T half_vmax[3];
  LesNum(const LesParams &P)
      : rdx((T)P.rdx), rdy((T)P.rdy), rdz((T)P.rdz), r2dx(T(0.5) * rdx), r2dy(T(0.5) * rdy), r2dz(T(0.5) * rdz),
        delta((T)P.delta), rdelta((T)P.rdelta), grav((T)P.grav), nu((T)P.nu), nu_pr((T)P.nu_pr),
        mix((T)P.total_mult * T(0.1)), diss((T)P.diss_mult), shear((T)P.shear_mult), dt((T)P.dt), gamma((T)P.gamma),
        half_vmax{T(0.5) * (T)P.visc_max_x, T(0.5) * (T)P.visc_max_y, T(0.5) * (T)P.visc_max_z} {}
};

// periodic image of an index at most one period outside [0, n) (every use here is one cell away)
__device__ __forceinline__ int wrapl(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// fields of the closure box: 0 rho_d, 1 u, 2 v, 3 w, 4 theta, 5 K, 6+q diffused tracer mixing ratios
// (values computed in FP64, stored as T: double, or float for the FP32 dycore mode)
template <class T>
__global__ __launch_bounds__(256) void k_les_prim(const double *__restrict__ rd_, const double *__restrict__ uu,
                                                  const double *__restrict__ vv, const double *__restrict__ ww,
                                                  const double *__restrict__ tt, TracerPtrsC trc,
                                                  T *__restrict__ F, LesParams P) {
  // grid: (blocks over one halo'd level's nxh*nyh points, nzh levels)
  const int nxyh = (int)(P.nxh * P.nyh);
  const int p = blockIdx.x * blockDim.x + threadIdx.x, kh = blockIdx.y;
  if (p >= nxyh) return;
  const int jh = p / (int)P.nxh, ih = p - jh * (int)P.nxh;
  const long long id = (long long)kh * nxyh + p;
  int i = ih - 1, j = jh - 1, k = kh - 1;
  bool ox = i < 0 || i >= P.nx, oy = j < 0 || j >= P.ny;
  // x/y source (periodic exchange; precursor replaces only the face halos, corners stay periodic)
  int is = i, js = j;
  if (ox && oy) { is = wrapl(i, P.nx); js = wrapl(j, P.ny); }
  else if (ox) is = P.bc_x == PU_BC_PRECURSOR ? (i < 0 ? 0 : P.nx - 1) : wrapl(i, P.nx);
  else if (oy) js = P.bc_y == PU_BC_PRECURSOR ? (j < 0 ? 0 : P.ny - 1) : wrapl(j, P.ny);
  bool zhalo = k < 0 || k >= P.nz;
  int ks = k;
  if (zhalo) ks = P.bc_z == PU_BC_PERIODIC ? wrapl(k, P.nz) : (k < 0 ? 0 : P.nz - 1);
  long long sid = ((long long)ks * P.ny + js) * P.nx + is;
  double rho_d = rd_[sid];
  double vals[6];
  vals[0] = rho_d;
  vals[1] = uu[sid];
  vals[2] = vv[sid];
  vals[3] = ww[sid];
  vals[4] = pow_pos(rho_d * P.R_d * tt[sid] / P.C0, 1. / P.gamma) / rho_d;
  vals[5] = fmax(0., trc.p[P.idTKE][sid] / rho_d);
  if (zhalo && P.bc_z != PU_BC_PERIODIC) {
    vals[3] = 0.;
    // hydrostatic extrapolation of rho from the first interior level (les_closure.h:503-510)
    double g = P.enable_gravity ? P.grav : 0.;
    double rho0_gm1 = pow_pos(rho_d, P.gamma - 1), theta0_g = pow_pos(vals[4], P.gamma);
    double sgn = k < 0 ? 1. : -1.;
    vals[0] = pow_pos(rho0_gm1 + sgn * g * (P.gamma - 1) * P.dz * 1 / (P.gamma * P.C0 * theta0_g), 1. / (P.gamma - 1));
  }
  for (int f = 0; f < 6; f++) F[(long long)f * P.nh + id] = (T)vals[f];
  for (int q = 0; q < P.nq; q++) F[(long long)(6 + q) * P.nh + id] = (T)(trc.p[P.qidx[q]][sid] / rho_d);
}

// Fluxes of one face, as the two cells beside it use them; all zero on a face of a fully immersed cell.
template <class T> struct Face {
  T f[6];      // ru rv rw rt tke, and -rho * viscosity for the diffused tracers
};

// The closure box as the face fluxes read it: field f at box index idx, the immersed proportion,
// and the box strides.  Tile: the block's cells plus a one-cell halo staged in LDS.
// Cells of one block tile: a row of 16 lanes is a row of cells in x, a wave a level of 16 x 4 cells, so
// that the high x face comes from the next lane, the high y face from the lane 16 above and the high z
// face from the next wave.
constexpr int LTX = 16, LTY = 4, LTZ = 4;
static_assert(LTX == 16 && LTX * LTY == 64, "one cell per thread: 16 lanes along x, a wave per level");
constexpr int LES_THREADS = LTX * LTY * LTZ;
constexpr int LBX = LTX + 2, LBY = LTY + 2, LBZ = LTZ + 2;   // tile + one-cell halo

// Coordinates of box point q < 1024: q / LBX and row / LBY as multiplications (exact in that range).
struct BoxPoint {
  int i, j, k;
  __device__ __forceinline__ BoxPoint(unsigned q) {
    const unsigned row = (q * (65536u / LBX + 1)) >> 16;
    k = (int)((row * (256u / LBY + 1)) >> 8);
    i = (int)(q - row * LBX);
    j = (int)(row - (unsigned)k * LBY);
  }
};

template <class T> struct TileBox {
  const T *sm;                               // closure fields of the tile + halo, [field][n]
  const uint8_t *icode;                      // immersed codes of the box points: 0 none, 1 partial, 2 full
  const float4 *tau;                         // learned closure: global [3][n3] per-direction stresses, or null
  long long n3;
  const unsigned char *flag;                 // learned closure: [n] flags of the box points
  static constexpr int sx = 1, sy = LBX, sz = LBX * LBY, n = LBX * LBY * LBZ;
  __device__ T S(int f, int idx) const { return sm[f * n + idx]; }
  __device__ bool imm_full(int idx) const { return icode[idx] == 2; }   // immersed proportion == 1
  __device__ bool imm_any(int idx) const { return icode[idx] != 0; }    // immersed proportion > 0
};

// Face flux on the low face of box cell c in direction DIR (les_closure.h:92-229).  T = double
// reproduces the reference's formulas in FP64; T = float evaluates them in FP32 (the FP32 dycore mode).
// gm, gc: the global cell ids of the face's low and high cells (periodic boundaries wrapped), used
// by the learned closure only.
template <int DIR, class T>
__device__ __forceinline__ Face<T> face_flux(const TileBox<T> &B, const LesParams &P, const LesNum<T> &C, int c, long long gm, long long gc) {
  constexpr int sx = TileBox<T>::sx, sy = TileBox<T>::sy, sz = TileBox<T>::sz;
  const int sn = DIR == 0 ? sx : (DIR == 1 ? sy : sz);            // normal stride
  const int m = c - sn;                                            // the low neighbour
  auto S = [&](int f, int idx) { return B.S(f, idx); };
  Face<T> fc = {};
  if (B.imm_full(m) || B.imm_full(c)) return fc;
  int both = 0;
  float4 ta = {}, tb = {};
  auto load_tau = [&]() {
    both = B.flag[m] & B.flag[c];
    if (both) {
      ta = B.tau[DIR * B.n3 + gm];
      tb = B.tau[DIR * B.n3 + gc];
    }
  };
  // read ahead in FP32; in FP64 that takes 133 VGPRs instead of 122, a wave less where LDS has room for four blocks,
  // and where it has not (three diffused tracers, 500x310x60) ran 1037 us instead of 1032
  if (sizeof(T) == 4 && B.tau) load_tau();
  const T h = T(0.5);
  const T rdx = C.rdx, rdy = C.rdy, rdz = C.rdz, r2dx = C.r2dx, r2dy = C.r2dy, r2dz = C.r2dz;
  T du_dx, du_dy, du_dz, dv_dx, dv_dy, dv_dz, dw_dx, dw_dy, dw_dz, dt_dz, dtn, dKn;
  if (DIR == 0) {
    du_dz = h * ((S(1, m + sz) - S(1, m - sz)) * r2dz + (S(1, c + sz) - S(1, c - sz)) * r2dz);
    dw_dz = h * ((S(3, m + sz) - S(3, m - sz)) * r2dz + (S(3, c + sz) - S(3, c - sz)) * r2dz);
    dt_dz = h * ((S(4, m + sz) - S(4, m - sz)) * r2dz + (S(4, c + sz) - S(4, c - sz)) * r2dz);
    du_dy = h * ((S(1, m + sy) - S(1, m - sy)) * r2dy + (S(1, c + sy) - S(1, c - sy)) * r2dy);
    dv_dy = h * ((S(2, m + sy) - S(2, m - sy)) * r2dy + (S(2, c + sy) - S(2, c - sy)) * r2dy);
    du_dx = (S(1, c) - S(1, m)) * rdx;
    dv_dx = (S(2, c) - S(2, m)) * rdx;
    dw_dx = (S(3, c) - S(3, m)) * rdx;
    dtn = (S(4, c) - S(4, m)) * rdx;
    dKn = (S(5, c) - S(5, m)) * rdx;
    dv_dz = dw_dy = T(0);
  } else if (DIR == 1) {
    dv_dz = h * ((S(2, m + sz) - S(2, m - sz)) * r2dz + (S(2, c + sz) - S(2, c - sz)) * r2dz);
    dw_dz = h * ((S(3, m + sz) - S(3, m - sz)) * r2dz + (S(3, c + sz) - S(3, c - sz)) * r2dz);
    dt_dz = h * ((S(4, m + sz) - S(4, m - sz)) * r2dz + (S(4, c + sz) - S(4, c - sz)) * r2dz);
    du_dx = h * ((S(1, m + sx) - S(1, m - sx)) * r2dx + (S(1, c + sx) - S(1, c - sx)) * r2dx);
    dv_dx = h * ((S(2, m + sx) - S(2, m - sx)) * r2dx + (S(2, c + sx) - S(2, c - sx)) * r2dx);
    du_dy = (S(1, c) - S(1, m)) * rdy;
    dv_dy = (S(2, c) - S(2, m)) * rdy;
    dw_dy = (S(3, c) - S(3, m)) * rdy;
    dtn = (S(4, c) - S(4, m)) * rdy;
    dKn = (S(5, c) - S(5, m)) * rdy;
    du_dz = dw_dx = T(0);
  } else {
    du_dx = h * ((S(1, m + sx) - S(1, m - sx)) * r2dx + (S(1, c + sx) - S(1, c - sx)) * r2dx);
    dw_dx = h * ((S(3, m + sx) - S(3, m - sx)) * r2dx + (S(3, c + sx) - S(3, c - sx)) * r2dx);
    dv_dy = h * ((S(2, m + sy) - S(2, m - sy)) * r2dy + (S(2, c + sy) - S(2, c - sy)) * r2dy);
    dw_dy = h * ((S(3, m + sy) - S(3, m - sy)) * r2dy + (S(3, c + sy) - S(3, c - sy)) * r2dy);
    du_dz = (S(1, c) - S(1, m)) * rdz;
    dv_dz = (S(2, c) - S(2, m)) * rdz;
    dw_dz = (S(3, c) - S(3, m)) * rdz;
    dt_dz = (S(4, c) - S(4, m)) * rdz;
    dtn = dt_dz;
    dKn = (S(5, c) - S(5, m)) * rdz;
    du_dy = dv_dx = T(0);
  }
  const T rho = h * (S(0, m) + S(0, c));
  const T K = h * (S(5, m) + S(5, c));
  const T t = h * (S(4, m) + S(4, c));
  // les_closure.h:116-127 with the divisions as reciprocal multiplies (t, N + 1e-20 > 0) and
  // km / Pr_t = km (1 + 2 ell) / delta
  const T sK = root(K);
  const T N = dt_dz >= T(0) && P.enable_gravity ? root(C.grav * recip(t) * dt_dz) : T(0);
  const T ell = fmin(T(0.76) * sK * recip(N + T(1.e-20)), C.delta);
  const T km = C.mix * ell * sK;
  const T visc_tot = P.dns ? C.nu : fmin(km + C.nu, C.half_vmax[DIR]);
  const T visc_tot_th = P.dns ? C.nu : fmin(km * (T(1) + T(2) * ell) * C.rdelta + C.nu_pr, C.half_vmax[DIR]);
  const T t23 = T(2. / 3.);
  fc.f[5] = -rho * visc_tot;
  if (DIR == 0) {
    fc.f[0] = -rho * visc_tot * (du_dx + du_dx - t23 * (du_dx + dv_dy + dw_dz));
    fc.f[1] = -rho * visc_tot * (dv_dx + du_dy);
    fc.f[2] = -rho * visc_tot * (dw_dx + du_dz);
  } else if (DIR == 1) {
    fc.f[0] = -rho * visc_tot * (du_dy + dv_dx);
    fc.f[1] = -rho * visc_tot * (dv_dy + dv_dy - t23 * (du_dx + dv_dy + dw_dz));
    fc.f[2] = -rho * visc_tot * (dw_dy + dv_dz);
  } else {
    fc.f[0] = -rho * visc_tot * (du_dz + dw_dx);
    fc.f[1] = -rho * visc_tot * (dv_dz + dw_dy);
    fc.f[2] = -rho * visc_tot * (dw_dz + dw_dz - t23 * (du_dx + dv_dy + dw_dz));
  }
  fc.f[3] = -rho * visc_tot_th * (dtn);
  fc.f[4] = -rho * visc_tot * T(2) * (dKn);
  if (B.tau) {
    // Learned closure (no reference counterpart): on a face whose two cells both hold the
    // network's flag, the momentum fluxes become rho * avg(tau_{i,DIR}) (bit 0) and the theta
    // flux rho * avg(q_DIR) (bit 1).  Box points outside the domain carry flag 0 unless the
    // boundary is periodic (then they hold the wrapped cell's values).  The network's outputs are
    // stored per face direction, so a face reads one 16-byte vector of each of its two cells.
    if (sizeof(T) == 8) load_tau();
    if (both & 1) {
      fc.f[0] = rho * (h * ((T)ta.x + (T)tb.x));
      fc.f[1] = rho * (h * ((T)ta.y + (T)tb.y));
      fc.f[2] = rho * (h * ((T)ta.z + (T)tb.z));
    }
    if (both & 2) fc.f[3] = rho * (h * ((T)ta.w + (T)tb.w));
  }
  return fc;
}

// value of the next lane of the 16-lane row (row_shl:1)
template <class T> __device__ __forceinline__ T from_next_in_row(T v) {
  if constexpr (sizeof(T) == 8) {
    const unsigned long long x = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0x101, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(x >> 32), 0x101, 0xf, 0xf, true);
    return __builtin_bit_cast(T, ((unsigned long long)hi << 32) | lo);
  } else {
    return __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x101, 0xf, 0xf, true));
  }
}

// Where faces wait in LDS for the cells below them, by the thread that reads them: high z and high y
// faces of every cell and the tile's high x faces; values of a field together.
struct FaceSlots {
  static constexpr int Z = 0, Y = Z + LES_THREADS, X = Y + LES_THREADS, N = X + LTY * LTZ;
};

// One block: an LTX x LTY x LTZ tile of cells.  The closure box values of the tile plus a one-cell halo
// (fields rho_d, u, v, w, theta, K and the diffused tracers, and the box points' immersed codes as
// bytes) are staged in LDS once.  Each thread evaluates the three low faces of its cell; the tile's 144
// high faces are a fourth face of waves 0 (y), 1 (z) and 2 (x).  The fluxes wait in the LDS of the box's
// first fields, which nothing reads any more after the TKE source, so that they take no LDS of their own:
// what bounds the kernel is the latency of its dependent chains (two square roots and two reciprocals a
// face, about 40 LDS reads) at the waves that fit.  In FP64 a block takes 31.8 KB and 5.2 KB for each
// diffused tracer: four blocks a CU (as many as 122 VGPRs allow) with none or one, three with two or three
// (the usual four tracers of which three diffuse); in FP32 half of that, six blocks (77 VGPRs) up to three.
// With the prim kernel, us when each cell computed its six faces and now, three diffused tracers: 384x250x100
// in FP64 960, 871; 512x256x128 in FP32 1182, 1140, with learned stresses 1419, 1296.
// T = double: the reference's update in FP64 (les_closure.h:280-320, :404-413).  T = float: the
// tendencies in FP32, applied as increments to the FP64 coupler entries (u += dt tend_u / rho,
// T *= (1 + dt tend_theta / (rho theta))^gamma, TKE and tracer masses += dt tend), so the entries
// keep their FP64 resolution.
template <class T>
__global__ __launch_bounds__(LES_THREADS) void k_les_update(const T *__restrict__ F, const uint8_t *__restrict__ icode,
                                                    double *uu, double *vv, double *ww, double *tt, TracerPtrs trc,
                                                    LesParams P, LesNum<T> C) {
  extern __shared__ __align__(16) unsigned char smraw[];
  T *sm = reinterpret_cast<T *>(smraw);
  const int nfl = 6 + P.nq;
  unsigned bx, by, bz;
  swizzled_block(bx, by, bz);
  const int i0 = bx * LTX, j0 = by * LTY, k0 = bz * LTZ;
  constexpr int NB = TileBox<T>::n;
  constexpr int PER = (NB + LES_THREADS - 1) / LES_THREADS;         // box points per thread
  // Everything the block needs is loaded before the first LDS write, so it waits on memory once (for
  // more than FB fields, once per FB).  Points past the halo (ragged last tiles) belong to no face of a
  // cell inside; they read its last point and carry no flag.
  long long goff[PER];
#pragma unroll
  for (int e = 0; e < PER; e++) {
    const BoxPoint b(min((int)threadIdx.x + LES_THREADS * e, NB - 1));
    const int ih = min(i0 + b.i, (int)P.nxh - 1), jh = min(j0 + b.j, (int)P.nyh - 1), kh = min(k0 + b.k, (int)P.nzh - 1);
    goff[e] = ((long long)kh * (int)P.nyh + jh) * (int)P.nxh + ih;
  }
  uint8_t ib[PER];
#pragma unroll
  for (int e = 0; e < PER; e++) ib[e] = icode[goff[e]];
  unsigned char fb[PER] = {};
  if (P.sflags) {
    // the network's flags of the box points (interior cells; periodic boundaries wrap)
#pragma unroll
    for (int e = 0; e < PER; e++) {
      const int q = threadIdx.x + LES_THREADS * e;
      const BoxPoint b(q);
      int i = i0 + b.i - 1, j = j0 + b.j - 1, k = k0 + b.k - 1;
      bool ok = q < NB;
      // points more than one cell past the domain belong to no cell's faces (ragged last tiles)
      if (i < 0 || i >= P.nx) { if (P.bc_x == PU_BC_PERIODIC && i <= P.nx) i = wrapl(i, P.nx); else ok = false; }
      if (j < 0 || j >= P.ny) { if (P.bc_y == PU_BC_PERIODIC && j <= P.ny) j = wrapl(j, P.ny); else ok = false; }
      if (k < 0 || k >= P.nz) { if (P.bc_z == PU_BC_PERIODIC && k <= P.nz) k = wrapl(k, P.nz); else ok = false; }
      if (ok) fb[e] = P.sflags[((long long)k * P.ny + j) * P.nx + i];
    }
  }
  constexpr int FB = 4;
  for (int f0 = 0; f0 < nfl; f0 += FB) {
    T buf[FB][PER];
#pragma unroll
    for (int df = 0; df < FB; df++)
#pragma unroll
      for (int e = 0; e < PER; e++)
        buf[df][e] = F[(long long)min(f0 + df, nfl - 1) * P.nh + goff[e]];      // no branch between the loads
#pragma unroll
    for (int df = 0; df < FB; df++)
#pragma unroll
      for (int e = 0; e < PER; e++) {
        const int q = threadIdx.x + LES_THREADS * e;
        if (f0 + df < nfl && q < NB) sm[(f0 + df) * NB + q] = buf[df][e];
      }
  }
  T *xch = sm;                                  // the faces take the place of box fields 0 .. 5 (see below)
  static_assert(6 * FaceSlots::N <= 6 * NB, "the faces fit the fields that they overwrite");
  uint8_t *sic = reinterpret_cast<uint8_t *>(sm + NB * nfl);
  unsigned char *sflag = P.sflags ? sic + NB : nullptr;
#pragma unroll
  for (int e = 0; e < PER; e++) {
    const int q = threadIdx.x + LES_THREADS * e;
    if (q < NB) {
      sic[q] = ib[e];
      if (P.sflags) sflag[q] = fb[e];
    }
  }
  __syncthreads();
  const int li = threadIdx.x % LTX, lj = (threadIdx.x / LTX) % LTY, lk = threadIdx.x / (LTX * LTY);
  const int i = i0 + li, j = j0 + lj, k = k0 + lk;
  const TileBox<T> B{sm, sic, P.sflags ? P.tau : nullptr, P.n3, sflag};
  constexpr int sx = TileBox<T>::sx, sy = TileBox<T>::sy, sz = TileBox<T>::sz;
  const int c = ((lk + 1) * LBY + (lj + 1)) * LBX + (li + 1);
  auto S = [&](int f, int idx) { return B.S(f, idx); };
  // Global ids of a face's two cells, read only by the learned closure where both carry a flag
  // (out-of-domain cells carry one only where their boundary wraps).
  auto low_face = [&](auto dir, int ii, int jj, int kk) {           // of the tile's cell (ii, jj, kk), one past its end included
    constexpr int DIR = decltype(dir)::value;
    long long gm = 0, gc = 0;
    if (P.sflags) {
      const int iw = wrapl(i0 + ii, P.nx), jw = wrapl(j0 + jj, P.ny), kw = wrapl(k0 + kk, P.nz);
      gc = ((long long)kw * P.ny + jw) * P.nx + iw;
      if (DIR == 0) gm = gc + (iw == 0 ? P.nx - 1 : -1);
      if (DIR == 1) gm = gc + (long long)(jw == 0 ? P.ny - 1 : -1) * P.nx;
      if (DIR == 2) gm = gc + (long long)(kw == 0 ? P.nz - 1 : -1) * P.nx * P.ny;
    }
    return face_flux<DIR>(B, P, C, ((kk + 1) * LBY + (jj + 1)) * LBX + (ii + 1), gm, gc);
  };
  auto put = [&](const Face<T> &fc, int slot) {
#pragma unroll
    for (int f = 0; f < 6; f++) xch[f * FaceSlots::N + slot] = fc.f[f];
  };
  using std::integral_constant;
  // All threads take part, those of cells past the domain too: the low face of the first of them is a
  // high face of the last cell inside, and the box is defined everywhere.
  const int lane = threadIdx.x & 63;
  Face<T> fe = {};
  int es = -1;
  if (lk == 0) {
    const int ke = lane / LTX;
    fe = low_face(integral_constant<int, 1>{}, li, LTY, ke);
    es = FaceSlots::Y + (ke * LTY + LTY - 1) * LTX + li;
  } else if (lk == 1) {
    fe = low_face(integral_constant<int, 2>{}, li, lj, LTZ);
    es = FaceSlots::Z + LTX * LTY * (LTZ - 1) + lane;
  } else if (lk == 2 && lane < LTY * LTZ) {
    fe = low_face(integral_constant<int, 0>{}, LTX, lane % LTY, lane / LTY);
    es = FaceSlots::X + lane;
  }
  const Face<T> fz = low_face(integral_constant<int, 2>{}, li, lj, lk);
  const Face<T> fx = low_face(integral_constant<int, 0>{}, li, lj, lk);
  const Face<T> fy = low_face(integral_constant<int, 1>{}, li, lj, lk);
  const T h = T(0.5);
  const T rdx = C.rdx, rdy = C.rdy, rdz = C.rdz, r2dx = C.r2dx, r2dy = C.r2dy, r2dz = C.r2dz;
  const T rdelta = C.rdelta;
  // TKE source (les_closure.h:233-278)
  const T rho = S(0, c), K = S(5, c), t = S(4, c);
  const T dt_dz = (S(4, c + sz) - S(4, c - sz)) * r2dz;
  const T sK = root(K), rt_ = recip(t);
  const T N = dt_dz >= T(0) && P.enable_gravity ? root(C.grav * rt_ * dt_dz) : T(0);
  const T ell = fmin(T(0.76) * sK * recip(N + T(1.e-20)), C.delta);
  const T km = T(0.1) * ell * sK;
  T src = T(0);
  if (!B.imm_full(c)) {
    // -(g rho km) / (t Pr_t) dt_dz with 1 / Pr_t = (1 + 2 ell) / delta
    if (P.enable_gravity) src += -(C.grav * rho * km) * (rt_ * (T(1) + T(2) * ell) * rdelta) * dt_dz;
    src -= C.diss * rho * (T(0.19) + T(0.51) * ell * rdelta) * rdelta * (K * sK);
    int im1 = B.imm_any(c - sx) ? c : c - sx, ip1 = B.imm_any(c + sx) ? c : c + sx;
    int jm1 = B.imm_any(c - sy) ? c : c - sy, jp1 = B.imm_any(c + sy) ? c : c + sy;
    int km1 = B.imm_any(c - sz) ? c : c - sz, kp1 = B.imm_any(c + sz) ? c : c + sz;
    const T du_dx = (S(1, c + sx) - S(1, c - sx)) * r2dx;
    const T dv_dx = (S(2, ip1) - S(2, im1)) * r2dx;
    const T dw_dx = (S(3, ip1) - S(3, im1)) * r2dx;
    const T du_dy = (S(1, jp1) - S(1, jm1)) * r2dy;
    const T dv_dy = (S(2, c + sy) - S(2, c - sy)) * r2dy;
    const T dw_dy = (S(3, jp1) - S(3, jm1)) * r2dy;
    const T du_dz = (S(1, kp1) - S(1, km1)) * r2dz;
    const T dv_dz = (S(2, kp1) - S(2, km1)) * r2dz;
    const T dw_dz = (S(3, c + sz) - S(3, c - sz)) * r2dz;
    const T j1_i1 = (du_dx + du_dx) * du_dx, j1_i2 = (dv_dx + du_dy) * dv_dx, j1_i3 = (dw_dx + du_dz) * dw_dx;
    const T j2_i1 = (du_dy + dv_dx) * du_dy, j2_i2 = (dv_dy + dv_dy) * dv_dy, j2_i3 = (dw_dy + dv_dz) * dw_dy;
    const T j3_i1 = (du_dz + dw_dx) * du_dz, j3_i2 = (dv_dz + dw_dy) * dv_dz, j3_i3 = (dw_dz + dw_dz) * dw_dz;
    src += C.shear * rho * km * (j1_i1 + j1_i2 + j1_i3 + j2_i1 + j2_i2 + j2_i3 + j3_i1 + j3_i2 + j3_i3);
  }
  const T uc = S(1, c), vc = S(2, c), wc = S(3, c);
  __syncthreads();
  if (es >= 0) put(fe, es);
  if (lk > 0) put(fz, FaceSlots::Z + (int)threadIdx.x - LTX * LTY);
  if (lj > 0) put(fy, FaceSlots::Y + (int)threadIdx.x - LTX);
  __syncthreads();
  // the high faces: x from the next lane (the last of a row from LDS), y and z from LDS
  auto high = [&](int f, T &x1, T &y1, T &z1) {
    const T *e = xch + f * FaceSlots::N;
    const T xe = e[FaceSlots::X + lk * LTY + lj], xn = from_next_in_row(fx.f[f]);
    x1 = li == LTX - 1 ? xe : xn;
    y1 = e[FaceSlots::Y + threadIdx.x];
    z1 = e[FaceSlots::Z + threadIdx.x];
  };
  T tend[5];
#pragma unroll
  for (int f = 0; f < 5; f++) {
    T x1, y1, z1;
    high(f, x1, y1, z1);
    tend[f] = -(x1 - fx.f[f]) * rdx - (y1 - fy.f[f]) * rdy - (z1 - fz.f[f]) * rdz;
  }
  T vx1 = T(0), vy1 = T(0), vz1 = T(0);
  if (P.nq > 0) high(5, vx1, vy1, vz1);
  if (i >= P.nx || j >= P.ny || k >= P.nz) return;
  const long long id = ((long long)k * P.ny + j) * P.nx + i;
  tend[4] += src;
  const T dt = C.dt;
  const T rrho = recip(rho);
  if constexpr (std::is_same<T, double>::value) {
    const double ru = uc * rho + dt * tend[0];
    const double rv = vc * rho + dt * tend[1];
    const double rw = wc * rho + dt * tend[2];
    const double rt = t * rho + dt * tend[3];
    const double rk = fmax(0., K * rho + dt * tend[4]);
    uu[id] = ru * rrho;
    vv[id] = rv * rrho;
    ww[id] = rw * rrho;
    tt[id] = P.C0 * pow_pos(rt, P.gamma) * (rrho * P.rR_d);
    trc.p[P.idTKE][id] = rk;
  } else {
    uu[id] += (double)(dt * tend[0] * rrho);
    vv[id] += (double)(dt * tend[1] * rrho);
    ww[id] += (double)(dt * tend[2] * rrho);
    const T x = dt * tend[3] * rrho * recip(t);                  // relative change of rho*theta
    const double T0 = tt[id];
    tt[id] = T0 + T0 * (double)expm1f(C.gamma * log1pf(x));
    double *tke = trc.p[P.idTKE];
    tke[id] = fmax(0., fmax(0., tke[id]) + (double)(dt * tend[4]));
  }
  // diffused tracers: flux -rho*visc*dq/dn on each open face
  if (P.nq == 0) return;
  const bool cf = B.imm_full(c);
  const bool ox0 = !(cf || B.imm_full(c - sx)), ox1 = !(cf || B.imm_full(c + sx));
  const bool oy0 = !(cf || B.imm_full(c - sy)), oy1 = !(cf || B.imm_full(c + sy));
  const bool oz0 = !(cf || B.imm_full(c - sz)), oz1 = !(cf || B.imm_full(c + sz));
  for (int q = 0; q < P.nq; q++) {
    auto Q = [&](int idx) { return B.S(6 + q, idx); };
    const T qx0 = ox0 ? fx.f[5] * ((Q(c) - Q(c - sx)) * rdx) : T(0);
    const T qx1 = ox1 ? vx1 * ((Q(c + sx) - Q(c)) * rdx) : T(0);
    const T qy0 = oy0 ? fy.f[5] * ((Q(c) - Q(c - sy)) * rdy) : T(0);
    const T qy1 = oy1 ? vy1 * ((Q(c + sy) - Q(c)) * rdy) : T(0);
    const T qz0 = oz0 ? fz.f[5] * ((Q(c) - Q(c - sz)) * rdz) : T(0);
    const T qz1 = oz1 ? vz1 * ((Q(c + sz) - Q(c)) * rdz) : T(0);
    const T tq = -(qx1 - qx0) * rdx - (qy1 - qy0) * rdy - (qz1 - qz0) * rdz;
    if constexpr (std::is_same<T, double>::value) trc.p[P.qidx[q]][id] = Q(c) * rho + dt * tq;
    else trc.p[P.qidx[q]][id] += (double)(dt * tq);
  }
}

static int les_params(pu_ctx *ctx, const pu_coupler_state *cs, double dt, LesParams &P, TracerPtrs &tp,
                      TracerPtrsC &tpc) {
  const pu_config &c = ctx->cfg;
  if (c.idTKE < 0 || c.idTKE >= c.num_tracers) return fail(PU_ERR_ARG, "LES closure needs a TKE tracer (idTKE)");
  P = LesParams{};
  P.nx = c.nx; P.ny = c.ny; P.nz = c.nz; P.ntr_all = c.num_tracers; P.idTKE = c.idTKE;
  P.bc_x = c.bc_x; P.bc_y = c.bc_y; P.bc_z = c.bc_z;
  P.enable_gravity = c.enable_gravity; P.dns = c.dns;
  P.nxh = c.nx + 2; P.nyh = c.ny + 2; P.nzh = c.nz + 2; P.nh = P.nxh * P.nyh * P.nzh;
  P.n3 = (long long)c.nx * c.ny * c.nz;
  P.nq = 0;
  for (int tr = 0; tr < c.num_tracers; tr++) if (c.tracer_diffuse[tr]) P.qidx[P.nq++] = tr;
  P.dx = c.xlen / c.nx; P.dy = c.ylen / c.ny; P.dz = c.zlen / c.nz;
  P.delta = std::pow(P.dx * P.dy * P.dz, 1. / 3.);
  P.rdelta = 1. / P.delta;
  P.nu_pr = c.kinematic_viscosity / 0.7;
  P.rR_d = 1. / c.R_d;
  P.rdx = 1. / P.dx; P.rdy = 1. / P.dy; P.rdz = 1. / P.dz;
  P.grav = c.grav; P.nu = c.kinematic_viscosity;
  P.total_mult = c.les_total_mult; P.diss_mult = c.les_dissipation_mult; P.shear_mult = c.les_shear_prod_mult;
  P.dt = dt;
  P.visc_max_x = 0.25 * P.dx * P.dx / dt; P.visc_max_y = 0.25 * P.dy * P.dy / dt; P.visc_max_z = 0.25 * P.dz * P.dz / dt;
  P.R_d = c.R_d; P.C0 = c.C0; P.gamma = c.gamma_d;
  P.tau = nullptr;
  P.sflags = nullptr;
  for (int tr = 0; tr < PU_MAX_TRACERS; tr++) {
    tp.p[tr] = tr < c.num_tracers ? cs->tracers[tr] : nullptr;
    tpc.p[tr] = tp.p[tr];
  }
  return PU_OK;
}

template <class T>
static int launch_les_prim(pu_ctx *ctx, const pu_coupler_state *cs, const LesParams &P, const TracerPtrsC &tpc) {
  hipLaunchKernelGGL(k_les_prim<T>, dim3((unsigned)((P.nxh * P.nyh + 255) / 256), (unsigned)P.nzh), dim3(256), 0,
                     ctx->stream, cs->density_dry,
                     cs->uvel, cs->vvel, cs->wvel, cs->temp, tpc, (T *)ctx->d_les, P);
  PU_HIP_CHECK(hipGetLastError());
  return PU_OK;
}

template <class T>
static int launch_les_update(pu_ctx *ctx, pu_coupler_state *cs, const LesParams &P, const TracerPtrs &tp) {
  const dim3 grd((unsigned)((P.nx + LTX - 1) / LTX), (unsigned)((P.ny + LTY - 1) / LTY), (unsigned)((P.nz + LTZ - 1) / LTZ));
  // box fields (<= 114 KB for 16 tracers in FP64), the immersed codes and the network's flags
  const size_t lds = sizeof(T) * TileBox<T>::n * (6 + P.nq) + TileBox<T>::n * (P.sflags ? 2 : 1);
  if (lds > 65536)
    PU_HIP_CHECK(hipFuncSetAttribute((const void *)k_les_update<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(k_les_update<T>, grd, dim3(LES_THREADS), lds, ctx->stream, (const T *)ctx->d_les,
                     (const uint8_t *)ctx->d_imm_les, cs->uvel, cs->vvel, cs->wvel, cs->temp, tp, P, LesNum<T>(P));
  PU_HIP_CHECK(hipGetLastError());
  return PU_OK;
}

int les_prim_device(pu_ctx *ctx, const pu_coupler_state *cs) {
  LesParams P;
  TracerPtrs tp;
  TracerPtrsC tpc;
  int rc = les_params(ctx, cs, 1., P, tp, tpc);
  if (rc) return rc;
  return ctx->cfg.precision == PU_FP32 ? launch_les_prim<float>(ctx, cs, P, tpc) : launch_les_prim<double>(ctx, cs, P, tpc);
}

int les_apply_device(pu_ctx *ctx, pu_coupler_state *cs, double dt) {
  LesParams P;
  TracerPtrs tp;
  TracerPtrsC tpc;
  int rc = les_params(ctx, cs, dt, P, tp, tpc);
  if (rc) return rc;
  const bool f32 = ctx->cfg.precision == PU_FP32;
  {
    LaunchTimer lt(ctx, "les");
    rc = f32 ? launch_les_prim<float>(ctx, cs, P, tpc) : launch_les_prim<double>(ctx, cs, P, tpc);
    if (rc) return rc;
  }
  if (ctx->sgs_model) {
    LaunchTimer lt(ctx, "sgs");
    rc = sgs_infer_device(ctx, dt);
    if (rc) return rc;
    P.tau = reinterpret_cast<const float4 *>(ctx->d_sgs_tau);
    P.sflags = ctx->d_sgs_flags;
  }
  {
    LaunchTimer lt(ctx, "les");
    rc = f32 ? launch_les_update<float>(ctx, cs, P, tp) : launch_les_update<double>(ctx, cs, P, tp);
    if (rc) return rc;
  }
  return PU_OK;
}

}  // namespace pu
