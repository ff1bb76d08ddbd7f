// sweep_f32_core.h -- the FP32 sweep kernels: the x and segment sweep k_sweep, the whole-column z sweep
// k_sweep_zwall and the whole-line y sweep k_sweep_yline.  Every field is reconstructed on both sides of
// a cell from its stencil in memory order.  The upwind-side evaluation of the FP64 sweeps
// (sweep_core.h), which reads half of the stencils in reverse, is not used in FP32: the limiter's map
// turns one rounding of a velocity (5e-7 at 8 m/s) into up to 4e-5 where a weight sits on its steep part,
// so that an FP32 run stays comparable with earlier ones only if every stencil keeps its order of
// evaluation (upwind-side FP32 sweeps moved single cells of w by up to 1e-3 of its rms in one step of the
// 512x512x128 urban boundary layer, at 0.92 of these kernels' time).
#pragma once
#include "sweep_core.h"

namespace pu {
namespace f32 {

constexpr int NQ = 6 + PU_MAX_TRACERS;     // carried face values: rho, normal velocity, p, then the transported fields

template <class T, int S> __device__ __forceinline__ void convexify(T *w) {
  T tot = w[0];
#pragma unroll
  for (int m = 1; m < S; m++) tot += w[m];
  if (tot > T(1.e-20)) {
    T r = recip(tot);
#pragma unroll
    for (int m = 0; m < S; m++) w[m] *= r;
  }
}

template <class T> __device__ __forceinline__ T map_rs(T w, T d) {     // k=6, m=3, s=2000
  T dl = w - d;
  T d2 = dl * dl;
  T t1 = d2 * d2 * d2;
  T ww = fma(-w, w, w);
  T t2 = ww * ww * ww;
  return d + (t1 * dl) * recip(t1 + T(2000) * t2);
}

// Both interface values of a cell; flat stencils take the linear reconstruction.
template <int ORD, class T>
__device__ __forceinline__ void weno_edges(const T *s, bool do_map, bool imm_L, bool imm_R, T &qL, T &qR) {
  using O = pu_weno::Ops<ORD>;
  constexpr int S = O::S;
  T d[ORD - 1], TV[S];
#pragma unroll
  for (int i = 0; i < ORD - 1; i++) d[i] = s[i + 1] - s[i];
  O::template tv<T>(d, TV);
  if constexpr (PU_FLAT_SHORTCUT) {                              // flat stencils: see cell_values
    T tot = TV[0];
#pragma unroll
    for (int m = 1; m < S; m++) tot += TV[m];
    if (tot <= T(1.e-20)) {
      qL = O::template linL<T>(s);
      qR = O::template linR<T>(s);
      return;
    }
  }
  convexify<T, S>(TV);
  if (imm_L || imm_R) {
    T mx = TV[0];
#pragma unroll
    for (int m = 1; m < S; m++) mx = fmax(mx, TV[m]);
    if (imm_L) TV[S - 1] = mx;
    if (imm_R) TV[0] = mx;
  }
  T rinv[S];
#pragma unroll
  for (int m = 0; m < S; m++) rinv[m] = recip(TV[m] * TV[m] + T(1.e-20));
  T wl[S], wr[S];
#pragma unroll
  for (int m = 0; m < S; m++) { wl[m] = T(O::idealL(m)) * rinv[m]; wr[m] = T(O::idealR(m)) * rinv[m]; }
  convexify<T, S>(wl);
  convexify<T, S>(wr);
  if (do_map && ORD <= 9) {
    // map_rs(w, d) = A/B; the renormalised mapped weights are A_m Q_m / sum_k A_k Q_k with
    // Q_m = prod_{j != m} B_j, and the one division goes to the face value.  Safe in FP32 up to
    // ord 9: the weights are normalised, so B_m = (w-d)^6 + 2000 (w(1-w))^3 lies in
    // [0.99 d_m^6, 32], and with the ideal weights of ord <= 9 (>= 1/126) a product of S-1 factors
    // stays above 1e-29 and below 1e6 (ord 11 could reach 1e-42: it keeps the divisions below).
#pragma unroll
    for (int side = 0; side < 2; side++) {
      T *w = side == 0 ? wl : wr;
      T A[S], B[S], Q[S];
#pragma unroll
      for (int m = 0; m < S; m++) {
        const T d = T(side == 0 ? O::idealL(m) : O::idealR(m));
        const T x = w[m];
        if constexpr (O::use_map_rs) {
          const T dl = x - d, d2 = dl * dl, t1 = d2 * d2 * d2, ww = fma(-x, x, x), t2 = ww * ww * ww;
          B[m] = fma(T(2000), t2, t1);
          A[m] = fma(d, B[m], t1 * dl);
        } else {
          B[m] = d * d + (T(1) - T(2) * d) * x;
          A[m] = x * (d + d * d - T(3) * d * x + x * x);
        }
      }
      excl_products<T, S>(B, Q);
      T sum = T(0);
#pragma unroll
      for (int m = 0; m < S; m++) { w[m] = A[m] * Q[m]; sum += w[m]; }
      if (side == 0) qL = O::template combL<T>(s, w) * recip(sum);
      else qR = O::template combR<T>(s, w) * recip(sum);
    }
  } else if (do_map) {
#pragma unroll
    for (int m = 0; m < S; m++) {
      wl[m] = map_rs(wl[m], T(O::idealL(m)));
      wr[m] = map_rs(wr[m], T(O::idealR(m)));
    }
    // renormalisation folded into the face value (the mapped weights sum to about one)
    T sl = wl[0], sr = wr[0];
#pragma unroll
    for (int m = 1; m < S; m++) { sl += wl[m]; sr += wr[m]; }
    qL = O::template combL<T>(s, wl) * recip(sl);
    qR = O::template combR<T>(s, wr) * recip(sr);
  } else {
    qL = O::template combL<T>(s, wl);
    qR = O::template combR<T>(s, wr);
  }
}

// What a cell's stencil code says about its reconstruction (dynamics_rk.h:572-607 with
// modify_stencil_immersed_der0, :478-493): the zero-derivative clamp window [lo, hi] used for the
// transverse velocities and p, imm_L / imm_R, do_map = no immersed cell within the 10-cell box, and
// WENO or the linear reconstruction.
template <int ORD> struct StencilFlags {
  static constexpr int hs = (ORD - 1) / 2;
  int lo = 0, hi = ORD - 1;
  bool imm_L = false, imm_R = false, do_map = true, use_weno = true;

  // c: the cell's stencil code
  __device__ __forceinline__ void setup(unsigned c, int weno_all) {
    lo = c & SC_LO;
    hi = ORD - 1 - (int)((c & SC_GAP) >> 4);
    imm_L = (c & SC_FIRST) != 0;
    imm_R = (c & SC_LAST) != 0;
    do_map = !(c & SC_ANY);
    use_weno = (c & SC_ANY) || weno_all;
  }

  // both interface values of the cell whose field value sits at p (stride sstride along the sweep)
  template <class T>
  __device__ __forceinline__ void recon(const T *p, long long sstride, bool modify, T &qL, T &qR) const {
    p -= (long long)hs * sstride;
    T s[ORD];
    if (modify) {
#pragma unroll
      for (int q = 0; q < ORD; q++) s[q] = p[(long long)valid_point<ORD>(q, lo, hi) * sstride];
    } else {
#pragma unroll
      for (int q = 0; q < ORD; q++) s[q] = p[(long long)q * sstride];
    }
    if (use_weno) {
      weno_edges<ORD, T>(s, do_map, imm_L, imm_R, qL, qR);
    } else {
      qL = pu_weno::Ops<ORD>::template linL<T>(s);
      qR = pu_weno::Ops<ORD>::template linR<T>(s);
    }
  }
};

// acoustic upwind state of one face (dynamics_rk.h:640-651): mass flux, pressure, upwind side
template <class T> struct Upw { T ru, p; bool left; };

template <class T>
__device__ __forceinline__ Upw<T> riemann(T rL, T uL, T pL, T rR, T uR, T pR, T hr) {
  rL += hr; rR += hr;
  const T cs = T(350.);
  T ruL = uL * rL, ruR = uR * rR;
  Upw<T> u;
  u.p = T(0.5) * (pL + pR - cs * (ruR - ruL));
  u.ru = T(0.5) * (ruL + ruR - (pR - pL) * T(1. / 350.));
  u.left = u.ru > 0;
  return u;
}

// z sweep between solid walls (writes the tendencies): the chunk walk of the FP64 kernel with both values
// of every cell exchanged through LDS.
template <int ORD, class T>
__global__ __launch_bounds__(256) void k_sweep_zwall(const T *__restrict__ prim,
                                                             const uint16_t *__restrict__ codes,
                                                             T *__restrict__ tend,
                                                             SweepParams P) {
  constexpr int BX = CH_BX, BS = CH_BS, NT = BX * BS;
  __shared__ T bufA0[NT], bufA1[NT], bufA2[NT], bufB0[NT], bufB1[NT];
  __shared__ T carQ[2][NQ][BX], carF[2][NQ][BX];     // by chunk parity

  const int tx = threadIdx.x, ty = threadIdx.y, lin = ty * BX + tx;
  unsigned bx, by, bz;
  swizzled_block(bx, by, bz);
  const int i = bx * BX + tx, j = by, nz = P.nz;
  const bool col_ok = i < P.nx;
  const long long sstride = P.nxh * P.nyh;
  const T rd = (T)P.rd;
  const int nchunk = (nz + BS - 1) / BS;
  const int nB = 3 + P.ntr;

  for (int q = 0; q < nchunk; q++) {
    const int r = q * BS + ty;
    const bool valid = col_ok && r < nz;
    const bool bot = r == 0, top = valid && r == nz - 1;
    const bool carry_in = ty == 0 && q > 0;          // face below r: values of the previous chunk
    const bool carry_out = ty == BS - 1;
    const int pin = (q + 1) & 1, pout = q & 1;
    const long long base = ((long long)(r + P.hp) * P.nyh + (j + P.hp)) * P.nxh + (i + P.ox);
    const long long cid = ((long long)r * P.ny + j) * P.nx + i;

    StencilFlags<ORD> sf;
    if (valid) sf.setup(codes[cid], P.weno_all);
    auto recon = [&](int l, bool modify, T &qL, T &qR) {
      sf.template recon<T>(prim + (long long)l * P.nh + base, sstride, modify, qL, qR);
    };
    T hr = 0, ht = 0;
    if (valid) { hr = (T)P.hy_re[r]; ht = (T)P.hy_te[r]; }

    // ---- phase A: density, w, pressure -> acoustic upwinding ----
    T qLr = 0, qRr = 0, qLu = 0, qRu = 0, qLp = 0, qRp = 0;
    if (valid) {
      recon(idR, false, qLr, qRr);
      recon(idW, false, qLu, qRu);
      recon(idP, true, qLp, qRp);
    }
    bufA0[lin] = qRr; bufA1[lin] = qRu; bufA2[lin] = qRp;
    __syncthreads();
    Upw<T> up{T(0), T(0), true};
    T Fr = 0, Fu = 0;
    if (valid) {
      T rL, uL, pL;
      if (carry_in) { rL = carQ[pin][0][tx]; uL = carQ[pin][1][tx]; pL = carQ[pin][2][tx]; }
      else if (ty > 0) { rL = bufA0[lin - BX]; uL = bufA1[lin - BX]; pL = bufA2[lin - BX]; }
      else { rL = 0; uL = 0; pL = 0; }
      T rR = qLr, uR = qLu, pR = qLp;
      if (bot) { rL = rR; uL = 0; uR = 0; pL = pR; }
      up = riemann(rL, uL, pL, rR, uR, pR, hr);
      Fr = up.ru;
      Fu = up.ru * (up.left ? uL : uR) + up.p;
    }
    bufB0[lin] = Fr; bufB1[lin] = Fu;
    __syncthreads();
    if (valid) {
      if (r > 0) {
        const T Fr0 = ty > 0 ? bufB0[lin - BX] : carF[pin][0][tx];
        const T Fu0 = ty > 0 ? bufB1[lin - BX] : carF[pin][1][tx];
        tend[(long long)idR * P.n3 + cid - (long long)P.nx * P.ny] = -(Fr - Fr0) * rd;
        tend[(long long)idW * P.n3 + cid - (long long)P.nx * P.ny] = -(Fu - Fu0) * rd;
      }
      if (top) {
        tend[(long long)idR * P.n3 + cid] = -(T(0) - Fr) * rd;
        tend[(long long)idW * P.n3 + cid] = -(qRp - Fu) * rd;
      }
    }
    if (carry_out) {
      carQ[pout][0][tx] = qRr; carQ[pout][1][tx] = qRu; carQ[pout][2][tx] = qRp;
      carF[pout][0][tx] = Fr; carF[pout][1][tx] = Fu;
    }

    // ---- phase B: the advected fields, one at a time ----
    for (int b = 0; b < nB; b++) {
      int l, fidx;
      bool modify = false;
      if (b == 0) { l = idU; fidx = idU; modify = true; }
      else if (b == 1) { l = idV; fidx = idV; modify = true; }
      else if (b == 2) { l = idT; fidx = idT; }
      else { l = NUM_STATE + 1 + (b - 3); fidx = NUM_STATE + (b - 3); }
      T qL = 0, qR = 0;
      if (valid) recon(l, modify, qL, qR);
      bufA0[lin] = qR;
      __syncthreads();
      T F = 0;
      if (valid) {
        T vL = carry_in ? carQ[pin][3 + b][tx] : (ty > 0 ? bufA0[lin - BX] : T(0)), vR = qL;
        if (bot) vL = vR;
        if (bot && l == idT) { vL = 0; vR = 0; }
        if (l == idT) { vL += ht; vR += ht; }
        F = up.ru * (up.left ? vL : vR);
      }
      bufB0[lin] = F;
      __syncthreads();
      if (valid) {
        T *tp = tend + (long long)fidx * P.n3 + cid;
        if (r > 0) tp[-(long long)P.nx * P.ny] = -(F - (ty > 0 ? bufB0[lin - BX] : carF[pin][2 + b][tx])) * rd;
        if (top) *tp = -(T(0) - F) * rd;
      }
      if (carry_out) { carQ[pout][3 + b][tx] = qR; carF[pout][2 + b][tx] = F; }
    }
  }
}


// y sweep along periodic lines (adds to the tendencies), chunks of BS cells with an LDS carry.  The
// periodic face between cells N-1 and 0 is computed last, by the thread of cell N-1, from cell 0's
// lower values kept in LDS; the tendencies of cells 0 and N-1, which need it, are finished after the
// last chunk.
//   Waves per SIMD by order: the low orders fit 72 VGPRs, and the schedule made for seven waves runs faster there
// than the one for six; the high ones lose more to the spills that 72 cost them (us per launch at 7 and 6:
// 700x24x144 order 3 122, 135, order 5 148, 163, order 7 168, 183, order 9 219, 210; 512x256x128 order 3
// 664, 714, order 5 817, 879, order 7 944, 995).  With six order 9 still spills 1 VGPR and order 11 7.
constexpr int yline_f32_waves(int ord) { return ord <= 7 ? 7 : 6; }
template <int ORD, class T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(yline_f32_waves(ORD))))
void k_sweep_yline(const T *__restrict__ prim, const uint16_t *__restrict__ codes,
                                                             T *__restrict__ tend,
                                                     SweepParams P) {
  constexpr int BX = CH_BX, BS = CH_BS, NA = BX, NT = BX * BS, nbs = BX;
  __shared__ T bufA0[NT], bufA1[NT], bufA2[NT], bufB0[NT], bufB1[NT];
  __shared__ T carQ[2][NQ][NA], carF[2][NQ][NA];          // by chunk parity
  __shared__ T firstQ[NQ][NA], firstF[NQ][NA];             // cell 0's lower values, face 1's fluxes
  __shared__ T lastF[NQ][NA], wrapF[NQ][NA], wrapU[2][NA]; // faces N-1 and N (= 0)

  const int tx = threadIdx.x, ty = threadIdx.y, lin = ty * BX + tx;
  const int t = ty, a = tx;
  unsigned bx, by, bz;
  swizzled_block(bx, by, bz);
  const int k = by;
  const int i = bx * BX + tx, N = P.ny;
  const bool across_ok = i < P.nx;
  const long long sstride = P.nxh, cstride = P.nx;
  const T rd = (T)P.rd;
  const T hr = (T)P.hy_rc[P.hs + k], ht = (T)P.hy_tc[P.hs + k];
  const int nchunk = (N + BS - 1) / BS;
  const int nB = 3 + P.ntr;
  constexpr int ln = idV, lt1 = idU;
  auto field_of = [&](int b, int &l, int &fidx, bool &modify) {
    modify = b < 2;
    if (b == 0) { l = lt1; fidx = lt1; }
    else if (b == 1) { l = idW; fidx = idW; }
    else if (b == 2) { l = idT; fidx = idT; }
    else { l = NUM_STATE + 1 + (b - 3); fidx = NUM_STATE + (b - 3); }
  };
  auto cell_id = [&](int r) { return ((long long)k * P.ny + r) * P.nx + i; };

  // the incoming tendency a cell's finished one adds to is loaded before the field's reconstruction
  // (27.1 -> 26.3 ms per step at 1024x1024x128)
  auto load_pre = [&](int fidx, long long cell, bool on) { return on ? tend[(long long)fidx * P.n3 + cell] : T(0); };
  auto finish = [&](int fidx, long long cell, T v, T pf) { tend[(long long)fidx * P.n3 + cell] = pf + v; };

  for (int q = 0; q < nchunk; q++) {
    const int r = q * BS + t;
    const bool valid = across_ok && r < N;
    const bool carry_in = t == 0 && q > 0, carry_out = t == BS - 1;
    const bool first = valid && r == 0, second = valid && r == 1, wrapper = valid && r == N - 1;
    const bool has_face = valid && r >= 1, has_tend = valid && r >= 2;
    const int pin = (q + 1) & 1, pout = q & 1;
    const long long cid = cell_id(r), eid = cid - cstride;   // own cell, tendency cell r-1
    const long long base = ((long long)(k + P.hp) * P.nyh + (r + P.hp)) * P.nxh + (i + P.ox);

    StencilFlags<ORD> sf;
    if (valid) sf.setup(codes[cid], P.weno_all);
    auto recon = [&](int l, bool modify, T &qL, T &qR) {
      sf.template recon<T>(prim + (long long)l * P.nh + base, sstride, modify, qL, qR);
    };
    auto prefetch = [&](int fidx) { return load_pre(fidx, eid, has_tend); };

    // ---- phase A: density, normal velocity, pressure -> acoustic upwinding ----
    T qLr = 0, qRr = 0, qLu = 0, qRu = 0, qLp = 0, qRp = 0;
    const T preR = prefetch(idR), preU = prefetch(ln);
    if (valid) {
      recon(idR, false, qLr, qRr);
      recon(ln, false, qLu, qRu);
      recon(idP, true, qLp, qRp);
    }
    bufA0[lin] = qRr; bufA1[lin] = qRu; bufA2[lin] = qRp;
    if (first) { firstQ[0][a] = qLr; firstQ[1][a] = qLu; firstQ[2][a] = qLp; }
    __syncthreads();
    Upw<T> up{T(0), T(0), true};
    T Fr = 0, Fu = 0;
    if (has_face) {
      T rL, uL, pL;
      if (carry_in) { rL = carQ[pin][0][a]; uL = carQ[pin][1][a]; pL = carQ[pin][2][a]; }
      else { rL = bufA0[lin - nbs]; uL = bufA1[lin - nbs]; pL = bufA2[lin - nbs]; }
      up = riemann(rL, uL, pL, qLr, qLu, qLp, hr);
      Fr = up.ru;
      Fu = up.ru * (up.left ? uL : qLu) + up.p;
    }
    if (wrapper) {
      const T uR = firstQ[1][a];
      const Upw<T> w = riemann(qRr, qRu, qRp, firstQ[0][a], uR, firstQ[2][a], hr);
      wrapU[0][a] = w.ru; wrapU[1][a] = w.left ? T(1) : T(0);
      wrapF[0][a] = w.ru; wrapF[1][a] = w.ru * (w.left ? qRu : uR) + w.p;
      lastF[0][a] = Fr; lastF[1][a] = Fu;
    }
    bufB0[lin] = Fr; bufB1[lin] = Fu;
    if (second) { firstF[0][a] = Fr; firstF[1][a] = Fu; }
    __syncthreads();
    if (has_tend) {
      const T Fr0 = carry_in ? carF[pin][0][a] : bufB0[lin - nbs];
      const T Fu0 = carry_in ? carF[pin][1][a] : bufB1[lin - nbs];
      finish(idR, eid, -(Fr - Fr0) * rd, preR);
      finish(ln, eid, -(Fu - Fu0) * rd, preU);
    }
    if (carry_out) {
      carQ[pout][0][a] = qRr; carQ[pout][1][a] = qRu; carQ[pout][2][a] = qRp;
      carF[pout][0][a] = Fr; carF[pout][1][a] = Fu;
    }

    // ---- phase B: the advected fields, one at a time ----
    for (int b = 0; b < nB; b++) {
      int l, fidx;
      bool modify;
      field_of(b, l, fidx, modify);
      T qL = 0, qR = 0;
      const T pf = prefetch(fidx);
      if (valid) recon(l, modify, qL, qR);
      bufA0[lin] = qR;
      if (first) firstQ[3 + b][a] = qL;
      __syncthreads();
      T F = 0;
      if (has_face) {
        T vL = carry_in ? carQ[pin][3 + b][a] : bufA0[lin - nbs], vR = qL;
        if (l == idT) { vL += ht; vR += ht; }
        F = up.ru * (up.left ? vL : vR);
      }
      if (wrapper) {
        T vL = qR, vR = firstQ[3 + b][a];
        if (l == idT) { vL += ht; vR += ht; }
        wrapF[2 + b][a] = wrapU[0][a] * (wrapU[1][a] != T(0) ? vL : vR);
        lastF[2 + b][a] = F;
      }
      bufB0[lin] = F;
      if (second) firstF[2 + b][a] = F;
      __syncthreads();
      if (has_tend) finish(fidx, eid, -(F - (carry_in ? carF[pin][2 + b][a] : bufB0[lin - nbs])) * rd, pf);
      if (carry_out) { carQ[pout][3 + b][a] = qR; carF[pout][2 + b][a] = F; }
    }
  }
  __syncthreads();

  // ---- cells 0 (thread t = 0) and N-1 (t = 1): the periodic face closes their tendencies ----
  if (across_ok && t < 2) {
    const int slot_lo = t == 0 ? 0 : 1;                 // which face arrays bound the cell
    const long long cell = cell_id(t == 0 ? 0 : N - 1);
    auto close = [&](int slot, int fidx) {
      const T Fhi = slot_lo == 0 ? firstF[slot][a] : wrapF[slot][a];
      const T Flo = slot_lo == 0 ? wrapF[slot][a] : lastF[slot][a];
      finish(fidx, cell, -(Fhi - Flo) * rd, load_pre(fidx, cell, true));
    };
    close(0, idR);
    close(1, ln);
    for (int b = 0; b < nB; b++) {
      int l, fidx;
      bool modify;
      field_of(b, l, fidx, modify);
      close(2 + b, fidx);
    }
  }
}

// Segment sweep: a 256-thread block covers line segments of BS-2 cells along the sweep plus one neighbour
// cell at each end (the cell whose reconstruction the segment's end faces need).  x always (its rows laid
// end to end, x_position; neighbours by wave shifts: 2 % less than through LDS with two barriers a field),
// y and z where the line kernels do not apply.  MODE: 0 writes the tendencies (z), 1 adds to them,
// 2 (x) takes each cell's finished tendency straight into the stage combination.
template <int DIR> struct SegShape { static constexpr int BX = 8, BY = 32, BS = 32; };
template <> struct SegShape<0> { static constexpr int BX = 64, BY = 4, BS = 64; };

// x, waves per SIMD by order: up to WENO-5 the kernel fits 64 VGPRs; above that 80 leave room for loads in
// flight (us per launch at 8 and 6 waves: 512x256x128 order 3 875, 939, order 5 1011, 1036, order 7 1200,
// 1176, order 9 1521, 1418).
constexpr int x_f32_waves(int ord) { return ord <= 5 ? 8 : 6; }
// Whether a wave's row is worked out in scalar registers.  Orders 7 and 9 run 0.5 to 1 % slower so, order 3
// 8 % and order 11 1 % faster (124x90x40 order 3 35.0 and 29.2 us with the wave cap; 512x256x128 order 11
// 1949, 1928).
constexpr bool x_f32_scalar_row(int ord) { return ord <= 5 || ord >= 11; }
// a - b, never fused with the product that made one of them
template <class T> __device__ __forceinline__ T plain_difference(T a, T b) {
#pragma clang fp contract(off)
  return a - b;
}

template <int ORD, class T, int DIR, int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DIR == 0 ? x_f32_waves(ORD) : 1)))
void k_sweep(const T *__restrict__ prim, const uint16_t *__restrict__ codes,
                                                             T *__restrict__ tend,
                                               SweepParams P, FuseArgs<T> FA) {
  constexpr int hs = (ORD - 1) / 2;
  constexpr int BX = SegShape<DIR>::BX, BY = SegShape<DIR>::BY, BS = SegShape<DIR>::BS;
  constexpr int NC = BS - 2;
  constexpr int NT = BX * BY;
  // x: a wave is a row and neighbours pass values by wave shifts; y and z: through LDS
  constexpr int NS = DIR == 0 ? 1 : NT;
  __shared__ T bufA0[NS], bufA1[NS], bufA2[NS], bufB0[NS], bufB1[NS];

  const int tx = threadIdx.x;
  const int ty = DIR == 0 && x_f32_scalar_row(ORD) ? __builtin_amdgcn_readfirstlane(threadIdx.y) : (int)threadIdx.y;
  const int lin = ty * BX + tx;
  const int t = DIR == 0 ? tx : ty;
  constexpr int nbs = DIR == 0 ? 1 : BX;
  unsigned bx, by, bz;
  swizzled_block(bx, by, bz);
  int i, j, k, c, nal;
  if (DIR == 0) { int j0; x_position((int)bx * BY + ty, tx, P.nx, j0, j, c); i = c; k = bz; nal = P.nx; }
  else if (DIR == 1) { i = bx * BX + tx; c = by * NC - 1 + ty; j = c; k = bz; nal = P.ny; }
  else { i = bx * BX + tx; j = by; c = bz * NC - 1 + ty; k = c; nal = P.nz; }
  const bool across_ok = DIR == 0 ? (j < P.ny) : (i < P.nx);
  const bool in_range = across_ok && c >= -1 && c <= nal;
  const bool periodic = P.bc_along == PU_BC_PERIODIC;
  const bool ghost = c < 0 || c >= nal;
  const bool do_recon = in_range && (!ghost || periodic);
  const bool has_face = in_range && t >= 1 && c >= 0;
  const bool has_tend = has_face && t <= NC && c < nal;
  const bool bface_lo = !periodic && c == 0;
  const bool bface_hi = !periodic && c == nal;
  const bool wallz = DIR == 2 && P.wall_z;

  const long long sstride = DIR == 0 ? 1 : (DIR == 1 ? P.nxh : P.nxh * P.nyh);
  const long long base = ((long long)(k + P.hp) * P.nyh + (j + P.hp)) * P.nxh + (i + P.ox);

  StencilFlags<ORD> sf;
  if (do_recon) {
    // A periodic neighbour cell past either end is the wrapped interior cell: its flags come from
    // that cell's own position (the z halos of the flag array hold "immersed", not a periodic copy,
    // dynamics_rk.h:1031-1034; the reference takes that face state from the wrapped cell's
    // reconstruction through edge_exchange, :890-908).
    const int cw = wrapi(c, nal);
    int ci = i, cj = j, ck = k;
    if (DIR == 0) ci = cw; else if (DIR == 1) cj = cw; else ck = cw;
    sf.setup(codes[((long long)ck * P.ny + cj) * P.nx + ci], P.weno_all);
  }
  auto recon = [&](int l, bool modify, T &qL, T &qR) {
    sf.template recon<T>(prim + (long long)l * P.nh + base, sstride, modify, qL, qR);
  };

  const long long cid = ((long long)k * P.ny + j) * P.nx + i;
  const T rd = (T)P.rd;
  StageIn S{0., 0., 0., 0., 0., 0.};
  if constexpr (MODE == 2) {
    if (has_tend) S = stage_inputs(FA, cid, k);
  }
  auto accumulate = [&](int fidx, T v) {
    T *tp = tend + (long long)fidx * P.n3 + cid;
    if constexpr (MODE == 2) {
      const T tsum = *tp + v;
      const double un = load_cons(FA.U, FA.Ulo, fidx, cid, P.n3);
      const double us = FA.C.stage > 0 ? load_cons(FA.Us, FA.Uslo, fidx, cid, P.n3) : 0.;
      const double w = combine_value(FA.C, fidx, (double)tsum, un, us, S);
      if (FA.C.stage == 2) store_cons(FA.U, FA.Ulo, fidx, cid, P.n3, w);
      else store_cons(FA.Us, FA.Uslo, fidx, cid, P.n3, w);
    } else if constexpr (MODE == 1) {
      *tp = *tp + v;
    } else {
      *tp = v;
    }
  };

  // hydrostatic add-back: cell values for x/y faces, edge values for z faces (:642-645, :686-689)
  T hr = 0, ht = 0;
  if (has_face) {
    if (DIR == 2) { hr = (T)P.hy_re[c]; ht = (T)P.hy_te[c]; }
    else { hr = (T)P.hy_rc[hs + k]; ht = (T)P.hy_tc[hs + k]; }
  }

  // ---- phase A: density, normal velocity, pressure -> acoustic upwinding ----
  constexpr int ln = 1 + DIR;
  T qLr = 0, qRr = 0, qLu = 0, qRu = 0, qLp = 0, qRp = 0;
  if (do_recon) {
    recon(idR, false, qLr, qRr);
    recon(ln, false, qLu, qRu);
    recon(idP, true, qLp, qRp);
  }
  T rL = 0, uL = 0, pL = 0;
  if constexpr (DIR == 0) {
    rL = from_lane_below(qRr); uL = from_lane_below(qRu); pL = from_lane_below(qRp);
  } else {
    bufA0[lin] = qRr; bufA1[lin] = qRu; bufA2[lin] = qRp;
    __syncthreads();
    if (has_face) { rL = bufA0[lin - nbs]; uL = bufA1[lin - nbs]; pL = bufA2[lin - nbs]; }
  }
  Upw<T> up{T(0), T(0), true};
  T Fr = 0, Fu = 0;
  if (has_face) {
    T rR = qLr, uR = qLu, pR = qLp;
    if (bface_lo) { rL = rR; uL = uR; pL = pR; }
    if (bface_hi) { rR = rL; uR = uL; pR = pL; }
    if (wallz && (bface_lo || bface_hi)) { uL = 0; uR = 0; }     // W = 0 on both sides at walls
    up = riemann(rL, uL, pL, rR, uR, pR, hr);
    Fr = up.ru;
    Fu = up.ru * (up.left ? uL : uR) + up.p;
  }
  // x: the flux through the cell's high face less the one through its low face
  auto difference = [&](T F) { return plain_difference(from_lane_above(F), F); };
  if constexpr (DIR != 0) {
    bufB0[lin] = Fr; bufB1[lin] = Fu;
    __syncthreads();
  }
  const T dr = DIR == 0 ? difference(Fr) : T(0), du = DIR == 0 ? difference(Fu) : T(0);
  if (has_tend) {
    accumulate(idR, -(DIR == 0 ? dr : bufB0[lin + nbs] - bufB0[lin]) * rd);
    accumulate(ln, -(DIR == 0 ? du : bufB1[lin + nbs] - bufB1[lin]) * rd);
  }

  // ---- phase B: the advected fields, one at a time ----
  constexpr int lt1 = DIR == 0 ? idV : idU;
  constexpr int lt2 = DIR == 2 ? idV : idW;
  const int nB = 3 + P.ntr;
  for (int b = 0; b < nB; b++) {
    int l, fidx;
    bool modify = false;
    if (b == 0) { l = lt1; fidx = lt1; modify = true; }
    else if (b == 1) { l = lt2; fidx = lt2; modify = true; }
    else if (b == 2) { l = idT; fidx = idT; }
    else { l = NUM_STATE + 1 + (b - 3); fidx = NUM_STATE + (b - 3); }
    T qL = 0, qR = 0;
    if (do_recon) recon(l, modify, qL, qR);
    T vL = 0;
    if constexpr (DIR == 0) {
      vL = from_lane_below(qR);
    } else {
      bufA0[lin] = qR;
      __syncthreads();
      if (has_face) vL = bufA0[lin - nbs];
    }
    T F = 0;
    if (has_face) {
      T vR = qL;
      if (bface_lo) vL = vR;
      if (bface_hi) vR = vL;
      if (wallz && (bface_lo || bface_hi) && l == idT) { vL = 0; vR = 0; }
      if (l == idT) { vL += ht; vR += ht; }
      F = up.ru * (up.left ? vL : vR);
    }
    if constexpr (DIR == 0) {
      const T dF = difference(F);
      if (has_tend) accumulate(fidx, -dF * rd);
    } else {
      bufB0[lin] = F;
      __syncthreads();
      if (has_tend) accumulate(fidx, -(bufB0[lin + nbs] - bufB0[lin]) * rd);
    }
  }
}

}  // namespace f32
}  // namespace pu
