// sweep_core.h -- the FP64 sweep kernels (WENO limiter, Riemann flux, flux divergence and the fused
// stage combination): the x sweep k_sweep_x, the whole-column z sweep k_sweep_zwall, the whole-line
// y sweep k_sweep_yline and the general y/z segment sweep k_sweep_seg, launched by dycore_kernels.hip,
// with what they share with the FP32 kernels (T = double throughout the kernels here).
//
// Every sweep works in two phases.  Phase A reconstructs density, normal velocity and pressure on
// both faces of a cell and solves the acoustic Riemann problem at its low face, which fixes the face's
// upwind side.  Phase B reconstructs each transported quantity (transverse velocities, theta, tracers)
// only there: one value per face instead of two per cell, of which the flux would use one.  A face
// whose upwind cell is the upper one reads that cell's stencil in reverse order and takes the same
// right-face expressions, so a wave with both directions runs one code path.  With the full limiter
// that is 7 of 10 fields (4 tracers) at 0.6 of the operations.
//   The kernels are bound by VALU issue (67-70 % of the SIMD cycles where every stencil takes the limiter, with 2900
// instructions per cell and sweep of ten fields, 4350 before; 52-59 % where two fifths are flat).  At
// 1024x1024x128 WENO-9, ms per launch: z 18.1 -> 14.1, y 19.4 -> 14.8, x 22.7 -> 16.3; of it the upwind side
// 0.84, the register cap with constants left in the loops 0.95, offsets and bases without 64-bit address
// arithmetic 0.96.
// FP32 has kernels of its own (sweep_f32_core.h).
#pragma once
#include "pu_common.h"
#include "weno_ops.h"
#include <type_traits>

namespace pu {

struct SweepParams {
  int nx, ny, nz, hs, hp, ox, ntr, bc_along, wall_z, weno_all;
  long long n3, nxh, nyh, nzh, nh;
  double rd;                       // 1/dx, 1/dy or 1/dz
  const double *hy_rc, *hy_tc;     // cells [nz+2hs]
  const double *hy_re, *hy_te;     // edges [nz+1]
};

__device__ __forceinline__ int wrapi(int i, int n) { i %= n; return i < 0 ? i + n : i; }
__device__ __forceinline__ int clampi(int i, int lo, int hi) { return i < lo ? lo : (i > hi ? hi : i); }

// ------------------------------------------------------------------------------------------------
// WENO limiter (WenoLimiter.h compute_limited_edges / gll_1 / gll_2 / convexify / map_rs)
// ------------------------------------------------------------------------------------------------

// Build switch for the flat-stencil branch of the limiters (1: on).
#ifndef PU_FLAT_SHORTCUT
#define PU_FLAT_SHORTCUT 1
#endif
template <class T> __device__ __forceinline__ bool flat_stencil(T tot) { return PU_FLAT_SHORTCUT && tot <= T(1.e-20); }

// P[m] = prod_{j != m} D[j]
template <class T, int S> __device__ __forceinline__ void excl_products(const T *D, T *P) {
  T pre[S];
  pre[0] = T(1);
#pragma unroll
  for (int m = 1; m < S; m++) pre[m] = pre[m - 1] * D[m - 1];
  T suf = T(1);
#pragma unroll
  for (int m = S - 1; m >= 0; m--) { P[m] = pre[m] * suf; suf *= D[m]; }
}

// Stencil code of a cell along one direction (k_any_z_codes, init_kernels.hip): 0 for a cell whose
// stencil and 10-cell box hold no immersed cell.  In the order the stencil is read, `lo` points at
// its start and `gap` points at its end are immersed ones to be replaced by the nearest valid point
// (dynamics_rk.h:478-493), `first` / `last` tell whether the neighbour before / after the cell is
// immersed (the limiter's imm_L, imm_R), `any` whether any cell of the 10-cell box is.
constexpr unsigned SC_LO = 0xf, SC_GAP = 0xf0, SC_CLAMP = 0xff, SC_FIRST = 0x100, SC_LAST = 0x200, SC_ANY = 0x400;
__device__ __forceinline__ unsigned reverse_code(unsigned c) {
  return ((c & SC_LO) << 4) | ((c & SC_GAP) >> 4) | ((c & SC_FIRST) << 1) | ((c & SC_LAST) >> 1) | (c & SC_ANY);
}

// What the limiter needs of a stencil besides the candidates' face values: the (unnormalised)
// nonlinear weights without their ideal factors, b[m] = 1 / (TV_m^2 + eps) up to a common factor.
// Candidate values are carried as differences e[m] from the cell's own average sc: a convex
// combination of them is sc + sum w_m e_m.  All multiply-adds of the limiter are explicit: a stencil
// gives the same value to the last bit in every kernel.
//
// The mathematics of the reference (WenoLimiter.h gll_1/gll_2) with a few roundings reordered:
//  * TV normalisation: with tot = sum(TV) > 1e-20 the reference uses TV_m/tot, so
//    d_m/((TV_m/tot)^2 + 1e-20) = tot^2 * d_m/(TV_m^2 + 1e-20*tot^2); the common factor tot^2
//    cancels in the weight normalisation, leaving D_m = TV_m^2 + 1e-20*tot^2.  imm_L/imm_R take a
//    maximum, which commutes with the positive scaling.
//  * w_m = d_m/D_m normalised equals d_m*P_m / sum_k d_k*P_k with P_m = prod_{j!=m} D_j
//    (D >= 1e-20*tot^2 keeps products of S-1 factors far from underflow in double).
template <int ORD, class T>
__device__ __forceinline__ void base_weights(T *TV, T tot, unsigned code, T *b) {
#pragma clang fp contract(off)
  constexpr int S = pu_weno::Ops<ORD>::S;
  if (code & (SC_FIRST | SC_LAST)) {
    T mx = TV[0];
#pragma unroll
    for (int m = 1; m < S; m++) mx = fmax(mx, TV[m]);
    if (code & SC_FIRST) TV[S - 1] = mx;
    if (code & SC_LAST) TV[0] = mx;
  }
  T D[S];
  const T eps = PU_FLAT_SHORTCUT || tot > T(1.e-20) ? T(1.e-20) * (tot * tot) : T(1.e-20);
#pragma unroll
  for (int m = 0; m < S; m++) D[m] = fma(TV[m], TV[m], eps);
  excl_products<T, S>(D, b);
}

// The valid stencil point that stands for point q when the points outside [lo, hi] are replaced
// (lo <= hs <= hi).
template <int ORD> __device__ __forceinline__ int valid_point(int q, int lo, int hi) {
  return q <= (ORD - 1) / 2 ? max(q, lo) : min(q, hi);
}

// Limited face value from the base weights b and the candidates' values e of one side (RIGHT: the
// face after the cell in stencil order).
//  * map_rs (k=6, m=3, s=2000) returns A_m/B_m; the renormalised mapped weights are
//    A_m*Q_m / sum A_k*Q_k with Q_m = prod_{j!=m} B_j, and the one division goes to the face value.
template <int ORD, class T, bool RIGHT>
__device__ __forceinline__ T limited_value(const T *b, const T *e, T sc, bool do_map) {
#pragma clang fp contract(off)
  using O = pu_weno::Ops<ORD>;
  constexpr int S = O::S;
  T w[S], ideal[S];
#pragma unroll
  for (int m = 0; m < S; m++) {
    ideal[m] = T(RIGHT ? O::idealR(m) : O::idealL(m));
    w[m] = ideal[m] * b[m];
  }
  T sum = w[0];
#pragma unroll
  for (int m = 1; m < S; m++) sum = fma(ideal[m], b[m], sum);
  const T r = recip(sum);
  auto dot = [&]() {
    T v = w[0] * e[0];
#pragma unroll
    for (int m = 1; m < S; m++) v = fma(w[m], e[m], v);
    return v;
  };
  if (!do_map) return fma(dot(), r, sc);
  T A[S], B[S];
#pragma unroll
  for (int m = 0; m < S; m++) {
    const T d = ideal[m], x = w[m] * r;
    if constexpr (O::use_map_rs) {
      const T dl = fma(w[m], r, -d), d2 = dl * dl, t1 = d2 * d2 * d2, ww = fma(-x, x, x), t2 = ww * ww * ww;
      B[m] = fma(T(2000), t2, t1);
      A[m] = fma(d, B[m], t1 * dl);
    } else {                                             // map_w (ord 3)
      B[m] = fma(T(1) - T(2) * d, x, d * d);
      A[m] = x * fma(x, x, fma(T(-3) * d, x, fma(d, d, d)));
    }
  }
  T Q[S];
  excl_products<T, S>(B, Q);
#pragma unroll
  for (int m = 0; m < S; m++) w[m] = A[m] * Q[m];
  sum = w[0];
#pragma unroll
  for (int m = 1; m < S; m++) sum = fma(A[m], Q[m], sum);
  return fma(dot(), recip(sum), sc);
}

// The linear (ideal-weight) reconstruction.
template <int ORD, class T, bool RIGHT>
__device__ __forceinline__ T linear_value(const T *e, T sc) {
#pragma clang fp contract(off)
  using O = pu_weno::Ops<ORD>;
  T dot = T(RIGHT ? O::idealR(0) : O::idealL(0)) * e[0];
#pragma unroll
  for (int m = 1; m < O::S; m++) dot = fma(T(RIGHT ? O::idealR(m) : O::idealL(m)), e[m], dot);
  return sc + dot;
}

// First differences and the candidates' total variations; returns their sum.
template <int ORD, class T>
__device__ __forceinline__ T variations(const T *s, T *d, T *TV) {
  using O = pu_weno::Ops<ORD>;
#pragma unroll
  for (int i = 0; i < ORD - 1; i++) d[i] = s[i + 1] - s[i];
  O::template tv<T>(d, TV);
  T tot = TV[0];
#pragma unroll
  for (int m = 1; m < O::S; m++) tot += TV[m];
  return tot;
}

// Flat stencils: with tot <= 1e-20 (the reference's convexify guard) every weight denominator
// rounds to 1e-20, the weights are the ideal ones and the map leaves them unchanged, so the limited
// values are the linear reconstruction to rounding.  Decided per stencil from its own values (the
// result does not depend on which cells share a wave); a wave of flat stencils skips the limiter.
// Both interface values of a cell from its stencil.
template <int ORD, class T>
__device__ __forceinline__ void cell_values(const T *s, unsigned code, bool use_weno, T &qL, T &qR) {
  using O = pu_weno::Ops<ORD>;
  T d[ORD - 1], TV[O::S], eL[O::S], eR[O::S];
  const T tot = variations<ORD, T>(s, d, TV);
  O::template edgeL<T>(d, eL);
  O::template edgeR<T>(d, eR);
  const T sc = s[O::hs];
  if (!use_weno || flat_stencil(tot)) {
    qL = linear_value<ORD, T, false>(eL, sc);
    qR = linear_value<ORD, T, true>(eR, sc);
    return;
  }
  T b[O::S];
  base_weights<ORD, T>(TV, tot, code, b);
  const bool do_map = !(code & SC_ANY);
  qL = limited_value<ORD, T, false>(b, eL, sc, do_map);
  qR = limited_value<ORD, T, true>(b, eR, sc, do_map);
}

// FP64: the value at the face after the cell, in the order the stencil is read.
template <int ORD, class T>
__device__ __forceinline__ T face_value(const T *s, unsigned code, bool use_weno) {
  using O = pu_weno::Ops<ORD>;
  T d[ORD - 1], TV[O::S], e[O::S];
  const T tot = variations<ORD, T>(s, d, TV);
  O::template edgeR<T>(d, e);
  const T sc = s[O::hs];
  if (!use_weno || flat_stencil(tot)) return linear_value<ORD, T, true>(e, sc);
  T b[O::S];
  base_weights<ORD, T>(TV, tot, code, b);
  return limited_value<ORD, T, true>(b, e, sc, !(code & SC_ANY));
}

// Stencil loads.  `base` is uniform over the wave (a scalar register pair) and the lane's part an
// offset in bytes: 32 bits wherever the host knows it fits (OFF = unsigned: the load takes it as it
// is, without 64-bit address arithmetic per point), 64 otherwise.
template <class T, class OFF> __device__ __forceinline__ T load_at(const T *base, OFF off) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + off);
}
template <class T> __device__ __forceinline__ void store_at(T *base, unsigned off, T v) {
  *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + off) = v;
}

// A cell's stencil in memory order; `base`: its first point for lane offset 0, sstride its step
// (uniform).  clamp: replace immersed points (transverse velocities and pressure).
template <int ORD, class T, class OFF>
__device__ __forceinline__ void load_stencil(const T *base, long long sstride, OFF off, unsigned code, bool clamp, T *s) {
  if (clamp && (code & SC_CLAMP)) {
    const int lo = code & SC_LO, hi = ORD - 1 - (int)((code & SC_GAP) >> 4);
#pragma unroll
    for (int q = 0; q < ORD; q++)
      s[q] = load_at<T, OFF>(base, off + (OFF)valid_point<ORD>(q, lo, hi) * (OFF)(sstride * (long long)sizeof(T)));
  } else {
#pragma unroll
    for (int q = 0; q < ORD; q++) s[q] = load_at<T, OFF>(base + q * sstride, off);
  }
}

// The stencil of a face's upwind cell, read from the upwind end.  The points' offsets are the same
// for every transported quantity, so they are worked out once per face and a load costs no address
// arithmetic; the transverse velocities (the first two quantities) take them with immersed points
// replaced, plain() gives the others theirs.
template <int ORD, class OFF> struct UpwindStencil {
  OFF off[ORD], off0, step;
  unsigned code;                   // in reading order
  // lane: the lane's offset of the lower neighbour's first point; left: the lower neighbour is
  // upwind; lower_code / own_code: stencil codes of the two cells
  __device__ __forceinline__ void setup(OFF lane, OFF stride, bool left, unsigned lower_code, unsigned own_code) {
    off0 = left ? lane : lane + (OFF)ORD * stride;
    step = left ? stride : (OFF)0 - stride;
    code = left ? lower_code : (own_code ? reverse_code(own_code) : 0u);
    plain();
    if (code & SC_CLAMP) {
      const int lo = code & SC_LO, hi = ORD - 1 - (int)((code & SC_GAP) >> 4);
#pragma unroll
      for (int q = 0; q < ORD; q++) off[q] = off0 + (OFF)valid_point<ORD>(q, lo, hi) * step;
    }
  }
  __device__ __forceinline__ void plain() {
    off[0] = off0;
#pragma unroll
    for (int q = 1; q < ORD; q++) off[q] = off[q - 1] + step;
  }
  template <class T> __device__ __forceinline__ void load(const T *base, T *s) const {
#pragma unroll
    for (int q = 0; q < ORD; q++) s[q] = load_at<T, OFF>(base, off[q]);
  }
};

// acoustic upwind state of one face (dynamics_rk.h:640-651): mass flux, pressure, upwind side.  The
// multiply-adds are written out, here and in carried(): every FP64 kernel then rounds a face's fluxes
// the same way, whatever code surrounds them.
template <class T> struct Upw {
  T ru, p;
  bool left;
  __device__ __forceinline__ T momentum(T uL, T uR) const { return fma(ru, left ? uL : uR, p); }
};

template <class T>
__device__ __forceinline__ Upw<T> riemann(T rL, T uL, T pL, T rR, T uR, T pR, T hr) {
#pragma clang fp contract(off)
  const T ruL = uL * (rL + hr), ruR = uR * (rR + hr);
  Upw<T> u;
  u.p = T(0.5) * fma(T(-350.), ruR - ruL, pL + pR);
  u.ru = T(0.5) * fma(T(-1. / 350.), pR - pL, ruL + ruR);
  u.left = u.ru > 0;
  return u;
}

// Flux of a transported value: rounded by itself, never fused into the divergence that follows, so
// that a face's two cells see the same flux.  The z kernels, which store the divergence, then give the same
// tendencies to the last bit; the y kernels add it to what z left, a sum that the compiler fuses differently in
// lines and segments (1e-13 of a tendency).
template <class T> __device__ __forceinline__ T carried(T ru, T v) {
#pragma clang fp contract(off)
  return ru * v;
}

// The transported quantities of a sweep in their order: the transverse velocities (stencils with
// immersed points replaced), theta (its hydrostatic part is added at the face), the tracers.  Calls
// f(is theta, primitive field, conserved field, quantity) for each.  PEEL: each of the first three
// from its own call site, so that the code for each holds only its own cases; the x sweep, whose
// stage combination differs by field, gains by it, the chunk-walking sweeps lose registers.
template <int DIR, bool PEEL, class US, class F> __device__ __forceinline__ void transport_all(US &us, int ntr, F &&f) {
  constexpr int first = DIR == 0 ? idV : idU, second = DIR == 2 ? idV : idW;
  if constexpr (PEEL) {
    f(false, first, first, 0);
    f(false, second, second, 1);
    us.plain();
    f(true, (int)idT, (int)idT, 2);
    for (int tr = 0; tr < ntr; tr++) f(false, NUM_STATE + 1 + tr, NUM_STATE + tr, 3 + tr);
  } else {
    for (int b = 0; b < 3 + ntr; b++) {
      if (b == 2) us.plain();
      const int l = b == 0 ? first : (b == 1 ? second : (b == 2 ? idT : NUM_STATE + b - 2));
      f(b == 2, l, b < 3 ? l : NUM_STATE + b - 3, b);
    }
  }
}

// Block of a chunk-walking sweep: CH_BX cells across, CH_BS along (at 512x512x128 WENO-9 in FP64 per
// launch 8x32 ran 3.42 (z) and 3.57 ms (y), 16x16 3.45 and 3.76, 4x64 3.7 and 3.6, 16x32 3.9 and 4.1;
// FP32 likewise).
constexpr int CH_BX = 8, CH_BS = 32;

// FP64 sweeps: at most 96 VGPRs (5 waves per SIMD), 128 at WENO-11 (4 waves; 96 cost it up to 30 spills).
// Spilled VGPRs as built: y lines 14 at WENO-5 and 27 at WENO-7 (the one-sided reconstructions at the periodic
// end), x with the stage combination 6 and z lines 2 at WENO-9, elsewhere none.  At WENO-9 and 1024x1024x128 x
// writes 11.8 GB a launch for 9.7 GB of results (without spills 9.7); z 10.2 and y, which spills nothing, 10.1.
__host__ __device__ constexpr int f64_waves(int ord) { return ord <= 9 ? 5 : 4; }
constexpr int SW_NQ = 5 + PU_MAX_TRACERS;     // fluxes of a face: mass, normal momentum, transported

// Whether the lane offsets of a line kernel (a chunk of 32 cells and its halo along the sweep) fit
// 32 bits: sstride = elements of es bytes between cells along the sweep.
static inline bool offsets_fit(long long sstride, int hp, size_t es) {
  return (CH_BS + 2 * hp + 2) * sstride * (long long)es + 4096 < (1LL << 32);
}

// ------------------------------------------------------------------------------------------------
// z sweep between solid walls (the first sweep of a stage, writing the tendencies): one block per
// BX columns walks the whole column in chunks of BS cells, every thread owning one cell per chunk.
// Walls need no neighbour cells (the wall faces take the adjacent cell's own values,
// dynamics_rk.h:864-888), and the face between two chunks takes the lower chunk's top values from
// a small LDS carry, so no cell is reconstructed twice (the segment kernel reconstructs 160 cells
// for each 128-level column).  Thread (x, t) of chunk q owns cell r = BS q + t: it computes the
// face below r (r = 0: the bottom wall) and finishes the tendency of cell r-1; the thread of the
// top cell also finishes its own tendency with the top wall face, whose Riemann state with w = 0
// on both sides and equal left/right values is exactly mass flux 0 and pressure p (every other
// flux through it is 0).  Otherwise the arithmetic of k_sweep_seg<ORD, T, 2>, operand for operand.
// A face's fluxes alternate between two LDS buffers, so a transported quantity costs one barrier.
// ------------------------------------------------------------------------------------------------

template <int ORD, class T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(f64_waves(ORD))))
void k_sweep_zwall(const T *__restrict__ prim,
                                                             const uint16_t *__restrict__ codes, T *__restrict__ tend,
                                                             SweepParams P) {
  constexpr int BX = CH_BX, BS = CH_BS, NT = BX * BS, hs = (ORD - 1) / 2;
  __shared__ T sQ[3][NT], sA[2][NT], sB[2][NT];
  __shared__ T carQ[2][3][BX], carF[2][SW_NQ][BX];          // by chunk parity

  const int tx = threadIdx.x, ty = threadIdx.y, lin = ty * BX + tx;
  unsigned bx, by, bz;
  swizzled_block(bx, by, bz);
  const int i = bx * BX + tx, j = by, nz = P.nz;
  const bool col_ok = i < P.nx;
  const long long plane = P.nxh * P.nyh, cplane = (long long)P.nx * P.ny;
  const unsigned stride = (unsigned)(plane * (long long)sizeof(T));
  const unsigned lane = (unsigned)((ty * plane + tx) * (long long)sizeof(T));
  const unsigned clane = (unsigned)((ty * cplane + tx) * (long long)sizeof(T));    // tendencies, one cell below
  const unsigned ctop = clane + (unsigned)(cplane * (long long)sizeof(T));
  const T rd = (T)P.rd;
  const int nchunk = (nz + BS - 1) / BS;

  for (int q = 0; q < nchunk; q++) {
    const int r = q * BS + ty;
    const bool valid = col_ok && r < nz;
    const bool bot = r == 0, top = valid && r == nz - 1;
    const bool carry_in = ty == 0 && q > 0;          // face below r: values of the previous chunk
    const bool carry_out = ty == BS - 1;
    const int pin = (q + 1) & 1, pout = q & 1;
    // first stencil point of the cell below the chunk's first one, at the block's first column
    const T *row = prim + ((long long)(q * BS) * P.nyh + (j + P.hp)) * P.nxh + (P.ox + (int)bx * BX);
    // cell of lane (0, 0) one level below the chunk, in the cell arrays
    const long long below = ((long long)(q * BS - 1) * P.ny + j) * P.nx + (int)bx * BX;
    unsigned own = 0, lower = 0;
    T hr = 0, ht = 0;
    if (valid) {
      const long long cid = ((long long)r * P.ny + j) * P.nx + i;
      own = codes[cid];
      if (r > 0) lower = codes[cid - cplane];
      hr = (T)P.hy_re[r];
      ht = (T)P.hy_te[r];
    }
    const bool weno = P.weno_all || (own & SC_ANY);

    // ---- phase A: density, w, pressure -> acoustic upwinding ----
    T qLr = 0, qRr = 0, qLu = 0, qRu = 0, qLp = 0, qRp = 0;
    if (valid) {
      T s[ORD];
      load_stencil<ORD, T, unsigned>(row + (long long)idR * P.nh + plane, plane, lane, own, false, s);
      cell_values<ORD, T>(s, own, weno, qLr, qRr);
      load_stencil<ORD, T, unsigned>(row + (long long)idW * P.nh + plane, plane, lane, own, false, s);
      cell_values<ORD, T>(s, own, weno, qLu, qRu);
      load_stencil<ORD, T, unsigned>(row + (long long)idP * P.nh + plane, plane, lane, own, true, s);
      cell_values<ORD, T>(s, own, weno, qLp, qRp);
    }
    sQ[0][lin] = qRr; sQ[1][lin] = qRu; sQ[2][lin] = qRp;
    __syncthreads();
    Upw<T> up{T(0), T(0), true};
    T Fr = 0, Fu = 0;
    if (valid) {
      T rL, uL, pL;
      if (carry_in) { rL = carQ[pin][0][tx]; uL = carQ[pin][1][tx]; pL = carQ[pin][2][tx]; }
      else if (ty > 0) { rL = sQ[0][lin - BX]; uL = sQ[1][lin - BX]; pL = sQ[2][lin - BX]; }
      else { rL = 0; uL = 0; pL = 0; }
      T rR = qLr, uR = qLu, pR = qLp;
      if (bot) { rL = rR; uL = 0; uR = 0; pL = pR; }
      up = riemann(rL, uL, pL, rR, uR, pR, hr);
      Fr = up.ru;
      Fu = up.momentum(uL, uR);
    }
    sA[0][lin] = Fr; sA[1][lin] = Fu;
    __syncthreads();
    if (valid) {
      if (r > 0) {
        const T Fr0 = ty > 0 ? sA[0][lin - BX] : carF[pin][0][tx];
        const T Fu0 = ty > 0 ? sA[1][lin - BX] : carF[pin][1][tx];
        store_at(tend + ((long long)idR * P.n3 + below), clane, -(Fr - Fr0) * rd);
        store_at(tend + ((long long)idW * P.n3 + below), clane, -(Fu - Fu0) * rd);
      }
      if (top) {
        store_at(tend + ((long long)idR * P.n3 + below), ctop, -(T(0) - Fr) * rd);
        store_at(tend + ((long long)idW * P.n3 + below), ctop, -(qRp - Fu) * rd);
      }
    }
    if (carry_out) {
      carQ[pout][0][tx] = qRr; carQ[pout][1][tx] = qRu; carQ[pout][2][tx] = qRp;
      carF[pout][0][tx] = Fr; carF[pout][1][tx] = Fu;
    }

    // ---- phase B: the transported quantities, one at a time ----
    // tendency of the cell below the face (and of the top cell) from the fluxes in sF
    auto finish = [&](const T *sF, int fidx, int b, T F) {
      if (valid) {
        T *tp = tend + ((long long)fidx * P.n3 + below);
        if (r > 0) store_at(tp, clane, -(F - (ty > 0 ? sF[lin - BX] : carF[pin][2 + b][tx])) * rd);
        if (top) store_at(tp, ctop, -(T(0) - F) * rd);
      }
      if (carry_out) carF[pout][2 + b][tx] = F;
    };
    UpwindStencil<ORD, unsigned> us;
    us.setup(lane, stride, up.left && !bot, lower, own);
    const bool weno_up = P.weno_all || (us.code & SC_ANY);
    transport_all<2, false>(us, P.ntr, [&](bool theta, int l, int fidx, int b) {
      T F = 0;
      if (valid) {
        T s[ORD];
        us.load(row + (long long)l * P.nh, s);
        T v = face_value<ORD, T>(s, us.code, weno_up);
        if (theta) v = (bot ? T(0) : v) + ht;
        F = carried(up.ru, v);
      }
      T *sF = sB[b & 1];
      sF[lin] = F;
      __syncthreads();
      finish(sF, fidx, b, F);
    });
  }
}


struct CombineParams {
  int nx, ny, nz, hs, ntr, stage, nrelax, enable_gravity, coriolis;
  int sim2d;                        // ny == 1: the V tendency is zero (dynamics_rk.h:716)
  long long n3;
  double cu, cs, ct;                // the stage's combination: cu*U + cs*Us + ct*tendency
  double grav, fcor;
  const double *hy_r, *hy_t;        // cells
  const double *relax;              // [n3]
  unsigned int positive_mask;       // bit tr set if tracer tr is positive-definite
};

// Conserved value as double: FP32 storage adds the compensation term of rho (l=0), rho*theta (l=4).
template <class ST>
__device__ __forceinline__ double load_cons(const ST *U, const ST *Ulo, int l, long long id, long long n3) {
  double v = (double)U[(long long)l * n3 + id];
  if constexpr (std::is_same<ST, float>::value) {
    if (l == idR) v += (double)Ulo[id];
    else if (l == idT) v += (double)Ulo[n3 + id];
  }
  return v;
}

template <class ST>
__device__ __forceinline__ void store_cons(ST *U, ST *Ulo, int l, long long id, long long n3, double v) {
  if constexpr (std::is_same<ST, float>::value) {
    float hi = (float)v;
    U[(long long)l * n3 + id] = hi;
    if (l == idR) Ulo[id] = (float)(v - (double)hi);
    else if (l == idT) Ulo[n3 + id] = (float)(v - (double)hi);
  } else {
    U[(long long)l * n3 + id] = v;
  }
}

template <class ST> struct FuseArgs {
  ST *U, *Ulo, *Us, *Uslo;
  CombineParams C;
};

// The same in double for cells addressed as a uniform cell number plus the lane's byte offset.
__device__ __forceinline__ double load_cons_at(const double *U, int l, long long cell, unsigned lane, long long n3) {
  return load_at<double, unsigned>(U + ((long long)l * n3 + cell), lane);
}

// The stage-input state of a cell the combination needs, read before any field of the cell is
// overwritten (stage 1 writes Us in place), and its relaxation multiplier and targets.
struct StageIn { double rho, u, v, mult, trr, trt; };

template <class ST>
__device__ __forceinline__ StageIn stage_inputs(const FuseArgs<ST> &F, long long id, int k) {
  const CombineParams &P = F.C;
  const ST *Sin = P.stage == 0 ? F.U : F.Us;
  const ST *Sinlo = P.stage == 0 ? F.Ulo : F.Uslo;
  StageIn S;
  S.rho = load_cons(Sin, Sinlo, idR, id, P.n3);
  S.u = P.coriolis ? load_cons(Sin, Sinlo, idU, id, P.n3) : 0.;
  S.v = P.coriolis ? load_cons(Sin, Sinlo, idV, id, P.n3) : 0.;
  S.mult = P.relax[id];
  S.trr = P.hy_r[P.hs + k];
  S.trt = P.hy_r[P.hs + k] * P.hy_t[P.hs + k];
  return S;
}

// ------------------------------------------------------------------------------------------------
// SSPRK3 stage combination of one conserved field of one cell (time_step_rk_3_3,
// dynamics_rk.h:279-367): gravity and Coriolis sources, the stage's convex combination, the
// positivity clip of the last stage and nrelax immersed relaxations (enforce_immersed_boundaries,
// :370-473).  tn: the field's tendency; un, us: its values in U and (stages 1, 2) Us.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ double combine_value(const CombineParams &P, int l, double tn, double un, double us,
                                                const StageIn &S) {
  if (l == idV && P.sim2d) tn = 0.;
  if (l == idW && P.enable_gravity) tn += -P.grav * (S.rho - S.trr);
  if (P.coriolis && l == idU) tn += P.fcor * S.v;
  if (P.coriolis && l == idV) tn -= P.fcor * S.u;
  double v = fma(P.ct, tn, fma(P.cu, un, P.cs * us));
  // a cell outside immersed regions has multiplier 0: its relaxations change nothing but the clip,
  // which is idempotent (the last stage clips before the first relaxation as well)
  const bool positive = l >= NUM_STATE && ((P.positive_mask >> (l - NUM_STATE)) & 1u);
  if (S.mult != 0.) {
    const double target = l == idR ? S.trr : (l == idT ? S.trt : 0.);
    if (P.stage == 2 && positive) v = fmax(0., v);
    for (int r = 0; r < P.nrelax; r++) {
      v = v + (target - v) * S.mult;
      if (positive) v = fmax(0., v);
    }
  } else if (positive) {
    v = fmax(0., v);
  }
  return v;
}

// ------------------------------------------------------------------------------------------------
// y sweep along periodic lines (adds to the tendencies): one block walks BX whole lines in chunks of
// BS cells, every thread owning one cell per chunk, so no cell is reconstructed twice (the segment
// kernel reconstructs 1120 cells for each 1024-cell line).  Thread t of chunk q owns cell
// r = BS q + t: it computes the face below it and finishes the tendency of cell r-1; the face between
// two chunks takes the lower chunk's top values from an LDS carry.  The thread of cell 0
// reconstructs the upper values of cell -1 (cell N-1 seen through the periodic halo: three one-sided
// reconstructions once per line) and so has the periodic face from the start; its fluxes are kept
// in LDS for cell N-1, whose upper face it is.  Otherwise the arithmetic of k_sweep_seg<ORD, T, 1>.
// ------------------------------------------------------------------------------------------------

template <int ORD, class T>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(f64_waves(ORD))))
void k_sweep_yline(const T *__restrict__ prim, const uint16_t *__restrict__ codes, T *__restrict__ tend, SweepParams P) {
  constexpr int BX = CH_BX, BS = CH_BS, NT = BX * BS, hs = (ORD - 1) / 2;
  __shared__ T sQ[3][NT], sA[2][NT], sB[2][NT];
  __shared__ T carQ[2][3][BX], carF[2][SW_NQ][BX];          // by chunk parity
  __shared__ T firstF[SW_NQ][BX];                            // the periodic face

  const int tx = threadIdx.x, ty = threadIdx.y, lin = ty * BX + tx;
  unsigned bx, by, bz;
  swizzled_block(bx, by, bz);
  const int i = bx * BX + tx, k = by, N = P.ny;
  const bool col_ok = i < P.nx;
  const unsigned stride = (unsigned)(P.nxh * (long long)sizeof(T));
  const unsigned lane = (unsigned)((ty * P.nxh + tx) * (long long)sizeof(T));
  const unsigned clane = (unsigned)((ty * (long long)P.nx + tx) * (long long)sizeof(T));   // tendencies, one cell below
  const unsigned clast = clane + (unsigned)(P.nx * (long long)sizeof(T));
  const T rd = (T)P.rd;
  const T hr = (T)P.hy_rc[P.hs + k], ht = (T)P.hy_tc[P.hs + k];
  const int nchunk = (N + BS - 1) / BS;
  const long long cline = (long long)k * P.ny * P.nx + i;      // cell 0 of the thread's line

  for (int q = 0; q < nchunk; q++) {
    const int r = q * BS + ty;
    const bool valid = col_ok && r < N;
    const bool carry_in = ty == 0 && q > 0, carry_out = ty == BS - 1;
    const bool first = r == 0, last = valid && r == N - 1;
    const int pin = (q + 1) & 1, pout = q & 1;
    const T *row = prim + ((long long)(k + P.hp) * P.nyh + q * BS) * P.nxh + (P.ox + (int)bx * BX);
    // cell of lane (0, 0) one row below the chunk, in the cell arrays
    const long long below = ((long long)k * P.ny + (q * BS - 1)) * P.nx + (int)bx * BX;
    unsigned own = 0, lower = 0;
    if (valid) {
      const long long cid = cline + (long long)r * P.nx;
      own = codes[cid];
      lower = codes[first ? cline + (long long)(N - 1) * P.nx : cid - P.nx];
    }
    const bool weno = P.weno_all || (own & SC_ANY);
    // the incoming tendencies are loaded ahead of the reconstructions that complete them
    auto incoming = [&](int fidx) {
      return valid && r > 0 ? load_at<T, unsigned>(tend + ((long long)fidx * P.n3 + below), clane) : T(0);
    };
    auto finish = [&](int fidx, T v) { store_at(tend + ((long long)fidx * P.n3 + below), clane, v); };
    auto finish_last = [&](int fidx, T v) {
      T *tp = tend + ((long long)fidx * P.n3 + below);
      store_at(tp, clast, load_at<T, unsigned>(tp, clast) + v);
    };

    // ---- phase A: density, v, pressure -> acoustic upwinding ----
    T qLr = 0, qRr = 0, qLu = 0, qRu = 0, qLp = 0, qRp = 0;
    const T tr0 = incoming(idR), tu0 = incoming(idV);
    T rL = 0, uL = 0, pL = 0;
    if (valid) {
      T s[ORD];
      load_stencil<ORD, T, unsigned>(row + (long long)idR * P.nh + P.nxh, P.nxh, lane, own, false, s);
      cell_values<ORD, T>(s, own, weno, qLr, qRr);
      load_stencil<ORD, T, unsigned>(row + (long long)idV * P.nh + P.nxh, P.nxh, lane, own, false, s);
      cell_values<ORD, T>(s, own, weno, qLu, qRu);
      load_stencil<ORD, T, unsigned>(row + (long long)idP * P.nh + P.nxh, P.nxh, lane, own, true, s);
      cell_values<ORD, T>(s, own, weno, qLp, qRp);
      if (first) {
        const bool weno_lo = P.weno_all || (lower & SC_ANY);
        load_stencil<ORD, T, unsigned>(row + (long long)idR * P.nh, P.nxh, lane, lower, false, s);
        rL = face_value<ORD, T>(s, lower, weno_lo);
        load_stencil<ORD, T, unsigned>(row + (long long)idV * P.nh, P.nxh, lane, lower, false, s);
        uL = face_value<ORD, T>(s, lower, weno_lo);
        load_stencil<ORD, T, unsigned>(row + (long long)idP * P.nh, P.nxh, lane, lower, true, s);
        pL = face_value<ORD, T>(s, lower, weno_lo);
      }
    }
    sQ[0][lin] = qRr; sQ[1][lin] = qRu; sQ[2][lin] = qRp;
    __syncthreads();
    Upw<T> up{T(0), T(0), true};
    T Fr = 0, Fu = 0;
    if (valid) {
      if (carry_in) { rL = carQ[pin][0][tx]; uL = carQ[pin][1][tx]; pL = carQ[pin][2][tx]; }
      else if (ty > 0) { rL = sQ[0][lin - BX]; uL = sQ[1][lin - BX]; pL = sQ[2][lin - BX]; }
      up = riemann(rL, uL, pL, qLr, qLu, qLp, hr);
      Fr = up.ru;
      Fu = up.momentum(uL, qLu);
    }
    sA[0][lin] = Fr; sA[1][lin] = Fu;
    if (first) { firstF[0][tx] = Fr; firstF[1][tx] = Fu; }
    __syncthreads();
    if (valid && r > 0) {
      const T Fr0 = ty > 0 ? sA[0][lin - BX] : carF[pin][0][tx];
      const T Fu0 = ty > 0 ? sA[1][lin - BX] : carF[pin][1][tx];
      finish(idR, tr0 + -(Fr - Fr0) * rd);
      finish(idV, tu0 + -(Fu - Fu0) * rd);
    }
    if (last) {
      finish_last(idR, -(firstF[0][tx] - Fr) * rd);
      finish_last(idV, -(firstF[1][tx] - Fu) * rd);
    }
    if (carry_out) {
      carQ[pout][0][tx] = qRr; carQ[pout][1][tx] = qRu; carQ[pout][2][tx] = qRp;
      carF[pout][0][tx] = Fr; carF[pout][1][tx] = Fu;
    }

    // ---- phase B: the transported quantities, one at a time ----
    auto complete = [&](const T *sF, int fidx, int b, T F, T t0) {
      if (valid && !first) finish(fidx, t0 + -(F - (ty > 0 ? sF[lin - BX] : carF[pin][2 + b][tx])) * rd);
      if (last) finish_last(fidx, -(firstF[2 + b][tx] - F) * rd);
      if (carry_out) carF[pout][2 + b][tx] = F;
    };
    UpwindStencil<ORD, unsigned> us;
    us.setup(lane, stride, up.left, lower, own);
    const bool weno_up = P.weno_all || (us.code & SC_ANY);
    transport_all<1, false>(us, P.ntr, [&](bool theta, int l, int fidx, int b) {
      const T t0 = incoming(fidx);
      T F = 0;
      if (valid) {
        T s[ORD];
        us.load(row + (long long)l * P.nh, s);
        T v = face_value<ORD, T>(s, us.code, weno_up);
        if (theta) v += ht;
        F = carried(up.ru, v);
      }
      T *sF = sB[b & 1];
      sF[lin] = F;
      if (first) firstF[2 + b][tx] = F;
      __syncthreads();
      complete(sF, fidx, b, F, t0);
    });
  }
}

// ------------------------------------------------------------------------------------------------
// x sweep (the last of a stage): a wave owns 64 consecutive positions of a level's rows, 62 of them for
// itself and one at each end whose reconstruction the end faces need.  A row is its cells and the
// position before and after them, and the next row follows on in the same wave (x_position), so that rows
// whose length is no multiple of 62 leave no lanes idle but the last wave's (us per launch, against waves
// that end with their row: 64^3 order 5 31 -> 23.5, 150x70x51 order 7 62 -> 54, 512x512x128 order 9 4.22 ->
// 4.06 ms; FP32 500x310x90 order 9 1358 -> 1240).  Lane t computes the low
// face of its cell; upper values and fluxes pass between neighbouring lanes by wave shifts, so the
// kernel has no LDS and no barrier and its waves run independently.
// MODE 1 adds to the tendencies, MODE 2 takes each cell's finished tendency straight into the stage
// combination (combine_value).  The stage runs z, y, x: this sweep's waves take 64 cells of a row, so
// the stage-state reads and writes of the combination are coalesced.
// ------------------------------------------------------------------------------------------------
constexpr int SX_BX = 64, SX_BY = 4, SX_NC = SX_BX - 2;
// Waves that a row gets to itself where they take no more than its positions end to end would (its length a
// multiple of 62 or up to two short of one), else 0 (us per launch, end to end and in waves of their own:
// 62x300x100 FP32 order 5 125, 117, order 9 167, 161, FP64 order 9 220, 214; 124x90x40 FP32 order 5 36.9, 34.4).
__host__ __device__ __forceinline__ int x_row_waves(int n) { const int w = (n + SX_NC - 1) / SX_NC; return w * SX_NC <= n + 2 ? w : 0; }
// blocks of a level: its positions, ny (nx + 2) without the first and the last, or its rows' own waves
inline unsigned x_blocks(int nx, int ny) {
  const int own = x_row_waves(nx);
  const long long waves = own ? (long long)ny * own : (ny * (nx + 2LL) - 2 + SX_NC - 1) / SX_NC;
  return (unsigned)((waves + SX_BY - 1) / SX_BY);
}
// Row j and cell c (-1 .. n; past n no cell) of lane t of wave w of a level; j0: lane 0's row.
__device__ __forceinline__ void x_position(int w, int t, int n, int &j0, int &j, int &c) {
  const int own = x_row_waves(n);
  if (own) {
    j = j0 = w / own;
    c = (w - j0 * own) * SX_NC + t - 1;
    return;
  }
  const int f0 = w * SX_NC;
  j = j0 = f0 / (n + 2);
  c = f0 - j0 * (n + 2) + t;
  while (c >= n + 2) { c -= n + 2; j++; }
  c--;
}

// the value of the neighbouring lane below / above (wave shifts by one lane)
template <int CTRL> __device__ __forceinline__ int wave_shift(int v) {
  return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);
}
template <int CTRL, class T> __device__ __forceinline__ T wave_shift_value(T v) {
  if constexpr (sizeof(T) == 8) {
    const long long x = __builtin_bit_cast(long long, v);
    const unsigned lo = (unsigned)wave_shift<CTRL>((int)x), hi = (unsigned)wave_shift<CTRL>((int)(x >> 32));
    return __builtin_bit_cast(T, (long long)(((unsigned long long)hi << 32) | lo));
  } else {
    return __builtin_bit_cast(T, wave_shift<CTRL>(__builtin_bit_cast(int, v)));
  }
}
template <class T> __device__ __forceinline__ T from_lane_below(T v) { return wave_shift_value<0x138>(v); }   // wave_shr:1
template <class T> __device__ __forceinline__ T from_lane_above(T v) { return wave_shift_value<0x130>(v); }   // wave_shl:1

template <int ORD, class T, int MODE>
__global__ __launch_bounds__(SX_BX * SX_BY)
__attribute__((amdgpu_waves_per_eu(f64_waves(ORD))))
void k_sweep_x(const T *__restrict__ prim, const uint16_t *__restrict__ codes, T *__restrict__ tend, SweepParams P,
               FuseArgs<T> FA) {
  constexpr int hs = (ORD - 1) / 2, hp = hs + 1;
  const int t = threadIdx.x, ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
  unsigned bx, by, bz;
  swizzled_block(bx, by, bz);
  const int k = bz, n = P.nx;
  int j0, j, c;
  x_position((int)bx * SX_BY + ty, t, n, j0, j, c);
  if (j0 >= P.ny) return;
  const bool periodic = P.bc_along == PU_BC_PERIODIC;
  const bool in_range = j < P.ny && c <= n, inner = c >= 0 && c < n;
  const bool do_recon = in_range && (periodic || inner);
  const bool has_face = in_range && t >= 1 && c >= 0;
  const bool has_tend = in_range && t >= 1 && t <= SX_NC && inner;
  const bool bface_lo = !periodic && c == 0, bface_hi = !periodic && c == n;

  // first stencil point of the cell below row j0's cell -1, and the lane's offset from there; the same of
  // the cell arrays
  const T *row = prim + ((long long)(k + hp) * P.nyh + (j0 + hp)) * P.nxh + (P.ox - 1 - hp);
  const unsigned lane = (unsigned)(((j - j0) * (int)P.nxh + c + 1) * (int)sizeof(T));
  const long long cell0 = ((long long)k * P.ny + j0) * P.nx - 1;
  const unsigned clane = (unsigned)(((j - j0) * n + c + 1) * (int)sizeof(T));
  const long long crow = ((long long)k * P.ny + j) * P.nx;
  // a periodic neighbour cell past either end is the wrapped interior cell
  unsigned own = 0;
  if (do_recon) own = codes[crow + (c < 0 ? c + n : (c >= n ? c - n : c))];
  const unsigned lower = from_lane_below(own);
  const bool weno = P.weno_all || (own & SC_ANY);

  const T rd = (T)P.rd;
  const T hr = (T)P.hy_rc[hs + k], ht = (T)P.hy_tc[hs + k];
  StageIn S{0., 0., 0., 0., 0., 0.};
  if constexpr (MODE == 2) {
    if (has_tend) S = stage_inputs(FA, crow + c, k);
  }
  // the values a cell's finished tendency is combined with are loaded before the field's
  // reconstruction, so their latency hides behind it
  struct Pre { T t; double u, us; };
  auto prefetch = [&](int fidx) {
    Pre p{T(0), 0., 0.};
    if (has_tend) {
      p.t = load_at<T, unsigned>(tend + ((long long)fidx * P.n3 + cell0), clane);
      if constexpr (MODE == 2) {
        p.u = load_cons_at(FA.U, fidx, cell0, clane, P.n3);
        if (FA.C.stage > 0) p.us = load_cons_at(FA.Us, fidx, cell0, clane, P.n3);
      }
    }
    return p;
  };
  // F: the flux through the cell's low face; completes the cell's tendency of one field
  auto finish = [&](int fidx, T F, const Pre &pf) {
    const T v = -(from_lane_above(F) - F) * rd;
    if (!has_tend) return;
    if constexpr (MODE == 2)
      store_at((FA.C.stage == 2 ? FA.U : FA.Us) + ((long long)fidx * P.n3 + cell0), clane,
               combine_value(FA.C, fidx, pf.t + v, pf.u, pf.us, S));
    else
      store_at(tend + ((long long)fidx * P.n3 + cell0), clane, pf.t + v);
  };

  // ---- phase A: density, u, pressure -> acoustic upwinding ----
  T qLr = 0, qRr = 0, qLu = 0, qRu = 0, qLp = 0, qRp = 0;
  const Pre preR = prefetch(idR), preU = prefetch(idU);
  if (do_recon) {
    T s[ORD];
    load_stencil<ORD, T, unsigned>(row + (long long)idR * P.nh + 1, 1, lane, own, false, s);
    cell_values<ORD, T>(s, own, weno, qLr, qRr);
    load_stencil<ORD, T, unsigned>(row + (long long)idU * P.nh + 1, 1, lane, own, false, s);
    cell_values<ORD, T>(s, own, weno, qLu, qRu);
    load_stencil<ORD, T, unsigned>(row + (long long)idP * P.nh + 1, 1, lane, own, true, s);
    cell_values<ORD, T>(s, own, weno, qLp, qRp);
  }
  T rL = from_lane_below(qRr), uL = from_lane_below(qRu), pL = from_lane_below(qRp);
  Upw<T> up{T(0), T(0), true};
  T Fr = 0, Fu = 0;
  if (has_face) {
    T rR = qLr, uR = qLu, pR = qLp;
    if (bface_lo) { rL = rR; uL = uR; pL = pR; }
    if (bface_hi) { rR = rL; uR = uL; pR = pL; }
    up = riemann(rL, uL, pL, rR, uR, pR, hr);
    Fr = up.ru;
    Fu = up.momentum(uL, uR);
  }
  finish(idR, Fr, preR);
  finish(idU, Fu, preU);

  // ---- phase B: the transported quantities, one at a time ----
  // (the faces of an open boundary take the inner cell's value from either side)
  UpwindStencil<ORD, unsigned> us;
  us.setup(lane, (unsigned)sizeof(T), (up.left || bface_hi) && !bface_lo, lower, own);
  const bool weno_up = P.weno_all || (us.code & SC_ANY);
  transport_all<0, true>(us, P.ntr, [&](bool theta, int l, int fidx, int) {
    const Pre pf = prefetch(fidx);
    T F = 0;
    if (has_face) {
      T s[ORD];
      us.load(row + (long long)l * P.nh, s);
      T v = face_value<ORD, T>(s, us.code, weno_up);
      if (theta) v += ht;
      F = carried(up.ru, v);
    }
    finish(fidx, F, pf);
  });
}

// ------------------------------------------------------------------------------------------------
// General y or z sweep (open y boundaries, periodic z, lines whose offsets need 64 bits): a 256-thread
// block covers line segments of 30 cells along the sweep plus one neighbour cell at each end (the
// cell whose reconstruction the segment's end faces need), 8 cells wide.  z writes the tendencies
// (the first sweep of a stage), y adds to them.
// ------------------------------------------------------------------------------------------------
constexpr int SG_BX = 8, SG_BS = 32, SG_NC = SG_BS - 2;

template <int ORD, class T, int DIR>
__global__ __launch_bounds__(SG_BX * SG_BS) void k_sweep_seg(const T *__restrict__ prim,
                                                             const uint16_t *__restrict__ codes, T *__restrict__ tend,
                                                             SweepParams P) {
  static_assert(DIR == 1 || DIR == 2, "y or z");
  constexpr int BX = SG_BX, NC = SG_NC, NT = SG_BX * SG_BS, hs = (ORD - 1) / 2;
  __shared__ T sQ[3][NT], sA[2][NT], sB[2][NT];
  const int tx = threadIdx.x, t = threadIdx.y, lin = t * BX + tx;
  unsigned bx, by, bz;
  swizzled_block(bx, by, bz);
  const int i = bx * BX + tx, n = DIR == 1 ? P.ny : P.nz;
  const int c0 = (int)(DIR == 1 ? by : bz) * NC - 1, c = c0 + t;
  const int jk = DIR == 1 ? (int)bz : (int)by;                 // level (y) or row (z) of the lines
  const bool across_ok = i < P.nx;
  const bool in_range = across_ok && c <= n;
  const bool periodic = P.bc_along == PU_BC_PERIODIC;
  const bool do_recon = in_range && (periodic || (c >= 0 && c < n));
  const bool has_face = in_range && t >= 1;
  const bool has_tend = across_ok && t >= 1 && t <= NC && c < n;
  const bool bface_lo = !periodic && c == 0, bface_hi = !periodic && c == n;
  const bool wallz = DIR == 2 && P.wall_z;

  const long long sstride = DIR == 1 ? P.nxh : P.nxh * P.nyh, cstride = DIR == 1 ? P.nx : (long long)P.nx * P.ny;
  // first stencil point of the cell below the segment's first one (c0 - 1 - hs = c0 - hp)
  const T *row = prim + (P.ox + (int)bx * BX) +
                 (DIR == 1 ? ((long long)(jk + P.hp) * P.nyh + c0) * P.nxh : ((long long)c0 * P.nyh + (jk + P.hp)) * P.nxh);
  const long long stride = sstride * (long long)sizeof(T), lane = t * stride + tx * (long long)sizeof(T);
  const long long cline = (DIR == 1 ? (long long)jk * P.ny * P.nx : (long long)jk * P.nx) + i;
  const long long cid = cline + c * cstride;
  // a periodic neighbour cell past either end is the wrapped interior cell
  auto code_of = [&](int cell) { return (unsigned)codes[cline + (cell < 0 ? cell + n : (cell >= n ? cell - n : cell)) * cstride]; };
  unsigned own = 0, lower = 0;
  if (do_recon) own = code_of(c);
  if (has_face && !bface_lo) lower = code_of(c - 1);
  const bool weno = P.weno_all || (own & SC_ANY);
  const T rd = (T)P.rd;
  // hydrostatic add-back: cell values for y faces, edge values for z faces (:642-645, :686-689)
  T hr = 0, ht = 0;
  if (has_face) {
    if (DIR == 2) { hr = (T)P.hy_re[c]; ht = (T)P.hy_te[c]; }
    else { hr = (T)P.hy_rc[hs + jk]; ht = (T)P.hy_tc[hs + jk]; }
  }
  auto put = [&](int fidx, T v) {
    T *tp = tend + (long long)fidx * P.n3 + cid;
    if (DIR == 1) *tp = *tp + v;
    else *tp = v;
  };

  // ---- phase A: density, normal velocity, pressure -> acoustic upwinding ----
  constexpr int ln = 1 + DIR;
  T qLr = 0, qRr = 0, qLu = 0, qRu = 0, qLp = 0, qRp = 0;
  if (do_recon) {
    T s[ORD];
    load_stencil<ORD, T, long long>(row + (long long)idR * P.nh + sstride, sstride, lane, own, false, s);
    cell_values<ORD, T>(s, own, weno, qLr, qRr);
    load_stencil<ORD, T, long long>(row + (long long)ln * P.nh + sstride, sstride, lane, own, false, s);
    cell_values<ORD, T>(s, own, weno, qLu, qRu);
    load_stencil<ORD, T, long long>(row + (long long)idP * P.nh + sstride, sstride, lane, own, true, s);
    cell_values<ORD, T>(s, own, weno, qLp, qRp);
  }
  sQ[0][lin] = qRr; sQ[1][lin] = qRu; sQ[2][lin] = qRp;
  __syncthreads();
  Upw<T> up{T(0), T(0), true};
  T Fr = 0, Fu = 0;
  if (has_face) {
    T rL = sQ[0][lin - BX], uL = sQ[1][lin - BX], pL = sQ[2][lin - BX];
    T rR = qLr, uR = qLu, pR = qLp;
    if (bface_lo) { rL = rR; uL = uR; pL = pR; }
    if (bface_hi) { rR = rL; uR = uL; pR = pL; }
    if (wallz && (bface_lo || bface_hi)) { uL = 0; uR = 0; }     // W = 0 on both sides at walls
    up = riemann(rL, uL, pL, rR, uR, pR, hr);
    Fr = up.ru;
    Fu = up.momentum(uL, uR);
  }
  sA[0][lin] = Fr; sA[1][lin] = Fu;
  __syncthreads();
  if (has_tend) {
    put(idR, -(sA[0][lin + BX] - Fr) * rd);
    put(ln, -(sA[1][lin + BX] - Fu) * rd);
  }

  // ---- phase B: the transported quantities, one at a time ----
  const bool left = (up.left || bface_hi) && !bface_lo;
  const bool wall = wallz && (bface_lo || bface_hi);
  auto through = [&](bool theta, T v) {
    if (theta) v = (wall ? T(0) : v) + ht;
    return carried(up.ru, v);
  };
  auto finish = [&](int fidx, int b, T F) {
    T *sF = sB[b & 1];
    sF[lin] = F;
    __syncthreads();
    if (has_tend) put(fidx, -(sF[lin + BX] - F) * rd);
  };
  UpwindStencil<ORD, long long> us;
  us.setup(lane, stride, left, lower, own);
  const bool weno_up = P.weno_all || (us.code & SC_ANY);
  transport_all<DIR, false>(us, P.ntr, [&](bool theta, int l, int fidx, int b) {
    T F = 0;
    if (has_face) {
      T s[ORD];
      us.load(row + (long long)l * P.nh, s);
      F = through(theta, face_value<ORD, T>(s, us.code, weno_up));
    }
    finish(fidx, b, F);
  });
}

// FP32 (sweep_f32_core.h): whole-column z sweep (sweep_zwall_f32.hip), whole-line y sweep
// (sweep_yline_f32.hip), segment sweeps (sweep_seg_f32.hip; dir 0: adds to the tendencies or, with
// combine, finishes them through the stage combination; 1: adds; 2: writes)
int launch_zwall_f32(int ord, dim3 grid, dim3 block, hipStream_t s, const float *prim, const uint16_t *codes,
                     float *tend, const SweepParams &P);
int launch_yline_f32(int ord, dim3 grid, dim3 block, hipStream_t s, const float *prim, const uint16_t *codes,
                     float *tend, const SweepParams &P);
int launch_seg_f32(int ord, int dir, bool combine, hipStream_t s, const float *prim, const uint16_t *codes, float *tend,
                   const SweepParams &P, const FuseArgs<float> &FA);

}  // namespace pu
