// adjoint3d.hip -- reverse mode of one TVD-RK stage of normal motion,
//   out = a*u_c + b*(u_s + dt*L(u_s)),  L_i = -V_i sqrt(G_i),
// where G_i is the Godunov |grad phi|^2 of the six HJ-WENO5 one-sided
// derivatives of u_s at cell i (the forward of lsmhip_weno5_stage_normal and
// of the chain HJ_WENO5 -> ADD_[CONST_]NORMAL_VEL_TERM -> TVD_RK3_STAGEn,
// src/toolbox/lsm_spatial_derivatives3d.f.in:1161-1611,
// src/toolbox/lsm_level_set_evolution3d.f.in:131-349,
// src/toolbox/lsm_tvd_runge_kutta3d.f:269-500).  No counterpart in the
// reference, which has no derivatives of its time stepping.
//
// Given lam_out = dJ/d out on the fill box, the stage adds
//   lam_s += b*lam_out + (b dt dL/du_s)^T lam_out   (over the ghost box),
//   lam_c += a*lam_out,
//   lam_V += -b dt sqrt(G) lam_out                  (when V is a field).
// The Godunov selection takes one of an axis's two one-sided derivatives, so
// cell i's part of dL/du_s is, per axis, one coefficient c = b dt lam_out(i)
// dL/dp times the gradient of one WENO5 value, which depends on u_s(i-3 .. i+3)
// through six undivided differences.
//   1. adj_coef_kernel, over the fill box where lam_out is not zero: the six
//      WENO5 values, the selection, lam_c, lam_V and b*lam_out, and per axis c
//      with the side taken (three fields and a byte of flags in the caller's
//      scratch).
//   2. adj_march_kernel, along j with the x axis and along k: the gradients at
//      each cell, formed once, added into the six differences they belong to
//      (registers along the march, lane shuffles along x), and each difference
//      into the two values it is made of.
// No atomics, and the sums are deterministic.  The flags carry the support of
// lam_out: a gradient of a level-set loss lives near the interface, and waves
// without a flagged cell read one byte per cell and nothing else.
//
// adj_weights_kernel and adj_gather_kernel do the same through 21 weights per
// cell in scratch.  They serve calls whose outputs overlap an input (the second
// pass of the marches reads u_s again, after the first has written: pass 1
// reads all inputs but lam_out, which pass 2 reads at its own cell) or one
// another (adj_coef_kernel reads all three before it writes any: each array is
// added to by itself here, so one array takes the sum), and small grids (marched).
//
// Derivatives follow the implemented functions: the WENO5 weights
// a_k = d_k/(S_k + eps)^2 with eps = 1e-6 max v^2 (the max contributes through
// its argmax), the Godunov max/min selections (the branch the forward's
// maxr takes, the plus branch on ties), and sqrt(G) (zero derivative where
// G = 0).
#include "lsmhip_core.hpp"
#include "reduce.hpp"
#include "stencil.hpp"

#include <initializer_list>

using namespace lsmhip;

namespace {

constexpr int kQ = 21;  // 3 axes x 7 stencil offsets

// 1/x for x between 1e-12 and 1e13 (the normalised smoothness terms and their
// weights).  FP32: the hardware reciprocal and one Newton step, 0.5 ulp but for
// rare last bits, in 3 instructions instead of the division's ten.
__device__ __forceinline__ float recip(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.f), r, r);
}
__device__ __forceinline__ double recip(double x) { return 1.0 / x; }

// Value of one WENO5 reconstruction and its gradient with respect to v1..v5.
// W is homogeneous of degree 1 in v (eps = 1e-6 max v^2 scales with v^2), so
// its gradient is homogeneous of degree 0 and is evaluated on v / max|v|: the
// weights then stay in range in FP32 whatever the scale of v (the FP32 forward
// normalises the same way).  The 1e-36 floor of eps is below FP64 rounding of
// the normalised eps and is left out; v = 0 gives the linear-weight limit.
template <class T>
__device__ __forceinline__ T weno5_grad(const T vin[5], T g[5]) {
  int am = 0;
  T ma = fabs(vin[0]), vmax = vin[0];
#pragma unroll
  for (int k = 1; k < 5; k++)
    if (fabs(vin[k]) > ma) {
      ma = fabs(vin[k]);
      vmax = vin[k];
      am = k;
    }
  if (ma == T(0)) {  // d/dv of the linear-weight combination 0.1 p1 + 0.6 p2 + 0.3 p3
    g[0] = T(0.1 / 3.0);
    g[1] = T(-0.7 / 6.0 - 0.1);
    g[2] = T(1.1 / 6.0 + 0.5 + 0.1);
    g[3] = T(0.2 + 0.25);
    g[4] = T(-0.05);
    return T(0);
  }
  const T sc = T(1) / ma;
  T v[5];
#pragma unroll
  for (int k = 0; k < 5; k++) v[k] = vin[k] * sc;
  vmax *= sc;
  const T eps = T(1e-6) * (vmax * vmax);
  const T a1 = v[0] - T(2) * v[1] + v[2], b1 = v[0] - T(4) * v[1] + T(3) * v[2];
  const T a2 = v[1] - T(2) * v[2] + v[3], b2 = v[1] - v[3];
  const T a3 = v[2] - T(2) * v[3] + v[4], b3 = T(3) * v[2] - T(4) * v[3] + v[4];
  const T c13 = T(13.0 / 12.0);
  const T S1 = c13 * a1 * a1 + T(0.25) * b1 * b1;
  const T S2 = c13 * a2 * a2 + T(0.25) * b2 * b2;
  const T S3 = c13 * a3 * a3 + T(0.25) * b3 * b3;
  const T p1 = T(1.0 / 3.0) * v[0] - T(7.0 / 6.0) * v[1] + T(11.0 / 6.0) * v[2];
  const T p2 = -T(1.0 / 6.0) * v[1] + T(5.0 / 6.0) * v[2] + T(1.0 / 3.0) * v[3];
  const T p3 = T(1.0 / 3.0) * v[2] + T(5.0 / 6.0) * v[3] - T(1.0 / 6.0) * v[4];
  const T e1 = S1 + eps, e2 = S2 + eps, e3 = S3 + eps;
  const T r1 = recip(e1), r2 = recip(e2), r3 = recip(e3);
  const T al1 = T(0.1) * (r1 * r1), al2 = T(0.6) * (r2 * r2), al3 = T(0.3) * (r3 * r3);
  const T inv = recip(al1 + al2 + al3);
  const T w1 = al1 * inv, w2 = al2 * inv, w3 = al3 * inv;
  const T W = w1 * p1 + w2 * p2 + w3 * p3;
  // dW/dS_k = -2 w_k (p_k - W) / (S_k + eps); eps enters every S_k
  const T t1 = T(-2) * w1 * (p1 - W) * r1, t2 = T(-2) * w2 * (p2 - W) * r2, t3 = T(-2) * w3 * (p3 - W) * r3;
  const T s6 = T(13.0 / 6.0), s3 = T(13.0 / 3.0);
  g[0] = w1 * T(1.0 / 3.0) + t1 * (s6 * a1 + T(0.5) * b1);
  g[1] = w1 * T(-7.0 / 6.0) + w2 * T(-1.0 / 6.0) + t1 * (-s3 * a1 - T(2) * b1) + t2 * (s6 * a2 + T(0.5) * b2);
  g[2] = w1 * T(11.0 / 6.0) + w2 * T(5.0 / 6.0) + w3 * T(1.0 / 3.0) + t1 * (s6 * a1 + T(1.5) * b1) +
         t2 * (-s3 * a2) + t3 * (s6 * a3 + T(1.5) * b3);
  g[3] = w2 * T(1.0 / 3.0) + w3 * T(5.0 / 6.0) + t2 * (s6 * a2 - T(0.5) * b2) + t3 * (-s3 * a3 - T(2) * b3);
  g[4] = w3 * T(-1.0 / 6.0) + t3 * (s6 * a3 + T(0.5) * b3);
  const T ge = (t1 + t2 + t3) * T(2e-6) * vmax;
#pragma unroll
  for (int k = 0; k < 5; k++) g[k] += k == am ? ge : T(0);  // (g[am] would put g in memory)
  return W * ma;
}

struct AdjArgs {
  const real_t* us;
  const real_t* lam_out;
  real_t* lam_us;
  real_t* lam_uc;
  real_t* lam_v;
  const real_t* vnf;
  real_t vn;
  real_t a, b, dt;
  real_t inv[3];
  real_t* q;  // kQ fields over the ghost box
  real_t* c[3];          // the axes' coefficients (marches)
  unsigned char* flags;  // bits 0-2: the axis has a coefficient; 3-5: of its plus derivative
  Box gb, fb;
  long long vol;
  int sy, sz;
};

__device__ __forceinline__ long long goff(const AdjArgs& A, int i, int j, int k) {
  return (long long)(i - A.gb.ilo) + (long long)A.sy * (j - A.gb.jlo) + (long long)A.sz * (k - A.gb.klo);
}

__global__ void __launch_bounds__(256) adj_weights_kernel(AdjArgs A) {
  LSMHIP_CELL(A.fb);
  const long long o = goff(A, i, j, k);
  const real_t lam = A.lam_out[o];
  const real_t v = A.vnf ? A.vnf[o] : A.vn;
  const real_t coef = A.b * A.dt * lam;
  if (A.lam_uc && A.a != real_t(0)) A.lam_uc[o] += A.a * lam;
  const bool moving = fabs(v) >= kZeroTol;
  if (coef == real_t(0) || !moving) {
#pragma unroll
    for (int q = 0; q < kQ; q++) A.q[q * A.vol + o] = real_t(0);
    return;
  }
  const long long step[3] = {1, A.sy, A.sz};
  real_t gp[3][5], gm[3][5], pp[3], pm[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    real_t f[7];
#pragma unroll
    for (int s = -3; s <= 3; s++) f[s + 3] = A.us[o + s * step[d]];
    real_t D[6];  // D[t+2] = f(t) - f(t-1), t = -2..3
#pragma unroll
    for (int t = -2; t <= 3; t++) D[t + 2] = f[t + 3] - f[t + 2];
    const real_t h = A.inv[d];
    real_t vp[5] = {D[5] * h, D[4] * h, D[3] * h, D[2] * h, D[1] * h};
    real_t vm[5] = {D[0] * h, D[1] * h, D[2] * h, D[3] * h, D[4] * h};
    pp[d] = weno5_grad(vp, gp[d]);
    pm[d] = weno5_grad(vm, gm[d]);
  }
  // Godunov selection per axis: the selected one-sided value enters G squared
  const bool vpos = v > real_t(0);
  real_t G = real_t(0), selp[3], selm[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const real_t xm = vpos ? maxr(pm[d], real_t(0)) : minr(pm[d], real_t(0));
    const real_t xp = vpos ? minr(pp[d], real_t(0)) : maxr(pp[d], real_t(0));
    if (xm * xm > xp * xp) {  // maxr of the forward: the plus branch on ties
      G += xm * xm;
      selm[d] = xm;
      selp[d] = real_t(0);
    } else {
      G += xp * xp;
      selm[d] = real_t(0);
      selp[d] = xp;
    }
  }
  const real_t sg = sqrt(G);
  if (A.lam_v && A.vnf) A.lam_v[o] += -A.b * A.dt * sg * lam;
  // dL/dp = -V sel / sqrt(G), bounded by |V| since |sel| <= sqrt(G); zero where G vanishes
  const real_t rs = sg > real_t(0) ? real_t(1) / sg : real_t(0);
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const real_t cp = coef * (-v) * (selp[d] * rs) * A.inv[d], cm = coef * (-v) * (selm[d] * rs) * A.inv[d];
    real_t w[7] = {0, 0, 0, 0, 0, 0, 0};  // w[s+3], s = -3..3
#pragma unroll
    for (int kk = 0; kk < 5; kk++) {
      const int tp = 3 - kk;  // plus: v_k = D(4-k), k = kk+1
      w[tp + 3] += cp * gp[d][kk];
      w[tp + 2] -= cp * gp[d][kk];
      const int tm = kk - 2;  // minus: v_k = D(k-3)
      w[tm + 3] += cm * gm[d][kk];
      w[tm + 2] -= cm * gm[d][kk];
    }
#pragma unroll
    for (int s = 0; s < 7; s++) A.q[(d * 7 + s) * A.vol + o] = w[s];
  }
}

__global__ void __launch_bounds__(256) adj_gather_kernel(AdjArgs A) {
  LSMHIP_CELL(A.gb);
  const long long o = goff(A, i, j, k);
  const Box& f = A.fb;
  real_t acc = f.has(i, j, k) ? A.b * A.lam_out[o] : real_t(0);
  const int c[3] = {i, j, k};
  const long long step[3] = {1, A.sy, A.sz};
  const int lo[3] = {f.ilo, f.jlo, f.klo}, hi[3] = {f.ihi, f.jhi, f.khi};
  bool in_t[3] = {i >= f.ilo && i <= f.ihi, j >= f.jlo && j <= f.jhi, k >= f.klo && k <= f.khi};
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const bool tr = in_t[(d + 1) % 3] && in_t[(d + 2) % 3];
    if (!tr) continue;
#pragma unroll
    for (int s = -3; s <= 3; s++) {
      const int src = c[d] - s;  // cell i = j - s e_d whose stencil offset s names j
      if (src >= lo[d] && src <= hi[d]) acc += A.q[(d * 7 + s + 3) * A.vol + o - s * step[d]];
    }
  }
  A.lam_us[o] += acc;
}

// WENO5 derivatives and square root of the forward stage (fused3d.hip).
__device__ __forceinline__ void weno_pm(const double f[7], double inv, double& p, double& m) {
  stencil::plus_minus<5>(f, inv, p, m);
}
__device__ __forceinline__ void weno_pm(const float f[7], float inv, float& p, float& m) {
  stencil::fastf::plus_minus(f, inv, p, m);
}

// One thread per (i, j) column of kp planes, lam_out one plane ahead.  Where
// lam_out is sparse this is bound by reading it and writing the flag byte;
// where it is dense by the stencil loads and about 400 VALU instructions per
// cell.  Lanes past the fill box stay in the wave with lam = 0, and everything
// past the ballot is computed by whole waves: an FP64 wave of eight lanes or
// fewer issues about 3.5 times slower.
__global__ void __launch_bounds__(256) adj_coef_kernel(AdjArgs A, int kp) {
  const Box& fb = A.fb;
  const int i = fb.ilo + (int)(blockIdx.x / kXcds) * kBX + (int)threadIdx.x;
  const int j = fb.jlo + (int)((blockIdx.x % kXcds) * gridDim.y + blockIdx.y) * kBY + (int)threadIdx.y;
  const int k0 = fb.klo + kp * (int)blockIdx.z, k1 = min(k0 + kp - 1, fb.khi);
  if (j > fb.jhi) return;  // the whole wave
  const bool in = i <= fb.ihi;
  long long o = goff(A, in ? i : fb.ihi, j, k0);
  const long long step[3] = {1, A.sy, A.sz};
  real_t lam = in ? A.lam_out[o] : real_t(0);
  for (int k = k0; k <= k1; k++, o += A.sz) {
    const real_t ahead = in && k < k1 ? A.lam_out[o + A.sz] : real_t(0);
    int flag = 0;
    const bool live = lam != real_t(0);
    if (__ballot(live)) {
      // all loads before any arithmetic: one memory round trip
      const bool has_c = A.lam_uc && A.a != real_t(0), has_v = A.lam_v && A.vnf;
      real_t f[3][7];
#pragma unroll
      for (int d = 0; d < 3; d++)
#pragma unroll
        for (int s = -3; s <= 3; s++) f[d][s + 3] = A.us[o + s * step[d]];
      real_t v = A.vn, was_c = real_t(0), was_v = real_t(0);
      if (live) {
        const real_t was = A.lam_us[o];
        if (A.vnf) v = A.vnf[o];
        if (has_c) was_c = A.lam_uc[o];
        if (has_v) was_v = A.lam_v[o];
        A.lam_us[o] = was + A.b * lam;
        if (has_c) A.lam_uc[o] = was_c + A.a * lam;
      }
      const real_t coef = A.b * A.dt * lam;
      const bool active = coef != real_t(0) && fabs(v) >= kZeroTol;
      if (__ballot(active)) {
        real_t pp[3], pm[3];
#pragma unroll
        for (int d = 0; d < 3; d++) weno_pm(f[d], A.inv[d], pp[d], pm[d]);
        // Godunov selection per axis: the selected one-sided value enters G squared
        const bool vpos = v > real_t(0);
        real_t G = real_t(0), sel[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
          const real_t xm = vpos ? maxr(pm[d], real_t(0)) : minr(pm[d], real_t(0));
          const real_t xp = vpos ? minr(pp[d], real_t(0)) : maxr(pp[d], real_t(0));
          const bool plus = !(xm * xm > xp * xp);  // maxr of the forward: the plus branch on ties
          sel[d] = plus ? xp : xm;
          G += sel[d] * sel[d];
          flag |= plus ? 8 << d : 0;
        }
        const real_t sg = sqrt(G);
        // dL/dp = -V sel / sqrt(G), bounded by |V| since |sel| <= sqrt(G); zero where G vanishes
        const real_t rs = sg > real_t(0) ? real_t(1) / sg : real_t(0);
        real_t c[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
          c[d] = coef * (-v) * (sel[d] * rs) * A.inv[d];
          flag |= c[d] != real_t(0) ? 1 << d : 0;
        }
        if (active) {
          if (has_v) A.lam_v[o] = was_v - A.b * A.dt * sg * lam;
#pragma unroll
          for (int d = 0; d < 3; d++)
            if (flag & (1 << d)) A.c[d][o] = c[d];
        } else {
          flag = 0;
        }
      }
    }
    if (in) A.flags[o] = (unsigned char)flag;
    lam = ahead;
  }
}

// c times the gradient of the selected WENO5 value with respect to the six
// differences D(-2 .. 3), D(t) = u(t) - u(t-1), from u(-3 .. 3): zero where
// on is false, whatever u holds.
__device__ __forceinline__ void diff_grad(const real_t w[7], bool on, bool plus, real_t c, real_t add[6]) {
  real_t D[6], v[5], g[5];
#pragma unroll
  for (int t = 0; t < 6; t++) D[t] = w[t + 1] - w[t];
#pragma unroll
  for (int q = 0; q < 5; q++) v[q] = plus ? D[5 - q] : D[q];
  weno5_grad(v, g);
#pragma unroll
  for (int t = 0; t < 6; t++) {
    const real_t gp = t >= 1 ? g[t >= 1 ? 5 - t : 0] : real_t(0), gm = t <= 4 ? g[t <= 4 ? t : 0] : real_t(0);
    add[t] = on ? c * (plus ? gp : gm) : real_t(0);
  }
}

// The march along AX (1: j, 2: k) over the targets lo-3 .. hi+3, cut into
// chunks of len.  A thread owns a column; e[t] is the running sum of the
// difference at m - 2 + t over the cells up to m.  After cell m the difference
// at m - 2 is whole, and with the one before it the target m - 3.  X adds the x
// axis at the target's plane: a wave holds 64 cells of a row and the 58 targets
// all of whose cells it holds, and each lane takes the seven weights that name
// its cell from the lanes around it.  Waves are independent: no LDS, no barrier.
// Along j rather than k for the x axis only because one march has to take it.
// Bound by latency and the flag bytes where lam_out is sparse, by VALU issue
// (about 130 instructions a gradient) where it is dense; times at the launch.
constexpr int kColX = 58;
template <int AX, bool X>
__global__ void __launch_bounds__(256) adj_march_kernel(AdjArgs A, int len) {
  const Box& f = A.fb;
  const int lane = (int)threadIdx.x;
  const int i = X ? f.ilo - 6 + (int)blockIdx.x * kColX + lane : f.ilo + (int)blockIdx.x * kBX + lane;
  const int other = (AX == 1 ? f.klo : f.jlo) + (int)blockIdx.y * kBY + (int)threadIdx.y;
  if (other > (AX == 1 ? f.khi : f.jhi)) return;  // the whole wave
  const int lo = AX == 1 ? f.jlo : f.klo, hi = AX == 1 ? f.jhi : f.khi;
  const int t0 = lo - 3 + (int)blockIdx.z * len, t1 = min(t0 + len - 1, hi + 3);
  const bool col = i >= f.ilo && i <= f.ihi;              // the column's cells are in the fill box
  const int ic = min(max(i, f.ilo - 3), f.ihi + 3);       // an address inside the ghost box for any lane
  const bool owns = X ? lane >= 3 && lane < 3 + kColX && i <= f.ihi + 3 : col;
  const long long st = AX == 1 ? A.sy : A.sz;
  const long long base = AX == 1 ? goff(A, ic, lo, other) : goff(A, ic, other, lo);  // cell m: base + (m - lo) st
  auto flag_at = [&](int m) {
    return col && m >= lo && m <= hi ? (int)A.flags[base + (m - lo) * st] : 0;
  };
  real_t e[6] = {0, 0, 0, 0, 0, 0}, prev = real_t(0);
  int f1 = 0, f2 = 0, f3 = 0;  // flags of cells m - 1, m - 2, m - 3
  int quiet = 6;               // cells since the last contribution along the march (6: none is left in e, prev)
  constexpr int kAhead = 8;    // flags are loaded this many cells at a time
  for (int m0 = t0 - 3; m0 <= t1 + 3; m0 += kAhead) {
    unsigned long long batch = 0;
#pragma unroll
    for (int q = 0; q < kAhead; q++) batch |= (unsigned long long)flag_at(m0 + q) << (8 * q);
    if (!__ballot((batch | (unsigned long long)(f1 | f2 | f3)) != 0) && quiet >= 6) {
      f1 = f2 = f3 = 0;
      continue;  // nothing in these cells, and nothing left of earlier ones
    }
    for (int q = 0; q < kAhead && m0 + q <= t1 + 3; q++) {
      const int m = m0 + q;
      const int fl = (int)(batch & 0xff);
      batch >>= 8;
      const bool on = (fl >> AX) & 1, onx = X && (f3 & 1);
      const bool any = __ballot(on) != 0, anyx = X && __ballot(onx) != 0;
      quiet = any ? 0 : quiet + 1;
      const long long o = base + (m - lo) * st, ot = o - 3 * st;
      const bool writes = owns && m - 3 >= t0 && m - 3 <= t1;
      // every load of the iteration before any of its arithmetic: one memory round trip
      real_t w[7], wx[7], c = real_t(0), cx = real_t(0), was = real_t(0);
      if (any) {  // m is a cell of the fill box: m -+ 3 lie in the ghost box
#pragma unroll
        for (int s = -3; s <= 3; s++) w[s + 3] = A.us[o + s * st];
        if (on) c = A.c[AX][o];
      }
      const long long oc = ot + (onx ? 0 : min(max(i, f.ilo), f.ihi) - ic);  // i -+ 3 lie in the ghost box
      if (anyx) {  // plane m - 3 holds cells of the fill box
#pragma unroll
        for (int s = -3; s <= 3; s++) wx[s + 3] = A.us[oc + s];
        if (onx) cx = A.c[0][oc];
      }
      if ((quiet <= 6 || anyx) && writes) was = A.lam_us[ot];
      if (any) {
        real_t add[6];
        diff_grad(w, on, (fl >> (3 + AX)) & 1, c, add);
#pragma unroll
        for (int t = 0; t < 6; t++) e[t] += add[t];
      }
      real_t val = prev - e[0];
      prev = e[0];
#pragma unroll
      for (int t = 0; t < 5; t++) e[t] = e[t + 1];
      e[5] = real_t(0);
      if (anyx) {
        real_t add[6];
        diff_grad(wx, onx, (f3 >> 3) & 1, cx, add);
#pragma unroll
        for (int s = -3; s <= 3; s++) {  // the weight of u(i + s), taken by lane + s
          const real_t ws = (s >= -2 ? add[s >= -2 ? s + 2 : 0] : real_t(0)) - (s <= 2 ? add[s <= 2 ? s + 3 : 0] : real_t(0));
          val += __shfl(ws, lane - s, 64);
        }
      }
      f3 = f2;
      f2 = f1;
      f1 = fl;
      if (writes && val != real_t(0)) A.lam_us[ot] = was + val;
    }
  }
}

// Adjoint of the periodic fill: every ghost value is a copy of the interior
// cell one period away, so its adjoint is added there and the ghost zeroed.
// Only the interior cells that have a copy are visited: nlo cells at the low
// end of an axis (copied past its high end), nhi at the high end; first the
// slabs normal to z, then those normal to y between them, then x.  A ghost has
// one source (ghost layers are no wider than the period), so the thread that
// adds it zeroes it.  256^3 with three ghost layers, FP32: 96 + 24 us -> 13 us
// (every interior cell testing 26 copies, and a pass over the ghost box).
struct FoldBox {
  Box gb, fb;
  int nlo[3], nhi[3];
  long long cz, cy, cx;  // cells of the three groups of slabs
};
__global__ void __launch_bounds__(256) fold_kernel(real_t* lam, FoldBox F, int sy, int sz) {
  long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  const Box &gb = F.gb, &fb = F.fb;
  const int n[3] = {fb.nx(), fb.ny(), fb.nz()};
  const int s0 = F.nlo[0] + F.nhi[0], s1 = F.nlo[1] + F.nhi[1];
  int c[3];
  if (t < F.cz) {
    c[0] = (int)(t % n[0]);
    c[1] = (int)(t / n[0] % n[1]);
    const int q = (int)(t / ((long long)n[0] * n[1]));
    c[2] = q < F.nlo[2] ? q : n[2] - F.nhi[2] + q - F.nlo[2];
  } else if ((t -= F.cz) < F.cy) {
    c[0] = (int)(t % n[0]);
    const int q = (int)(t / n[0] % s1);
    c[1] = q < F.nlo[1] ? q : n[1] - F.nhi[1] + q - F.nlo[1];
    c[2] = F.nlo[2] + (int)(t / ((long long)n[0] * s1));
  } else if ((t -= F.cy) < F.cx) {
    const int my = n[1] - s1, q = (int)(t % s0);
    c[0] = q < F.nlo[0] ? q : n[0] - F.nhi[0] + q - F.nlo[0];
    c[1] = F.nlo[1] + (int)(t / s0 % my);
    c[2] = F.nlo[2] + (int)(t / ((long long)s0 * my));
  } else {
    return;
  }
  c[0] += fb.ilo;
  c[1] += fb.jlo;
  c[2] += fb.klo;
  const int glo[3] = {gb.ilo, gb.jlo, gb.klo}, ghi[3] = {gb.ihi, gb.jhi, gb.khi};
  real_t acc = real_t(0);
  for (int a = -1; a <= 1; a++)
    for (int bb = -1; bb <= 1; bb++)
      for (int cc = -1; cc <= 1; cc++) {
        if (a == 0 && bb == 0 && cc == 0) continue;
        const int q[3] = {c[0] + a * n[0], c[1] + bb * n[1], c[2] + cc * n[2]};
        bool ok = true;
        for (int d = 0; d < 3; d++) ok = ok && q[d] >= glo[d] && q[d] <= ghi[d];
        if (ok) {
          real_t* g = lam + ((q[0] - gb.ilo) + (long long)sy * (q[1] - gb.jlo) + (long long)sz * (q[2] - gb.klo));
          acc += *g;
          *g = real_t(0);
        }
      }
  lam[(c[0] - gb.ilo) + (long long)sy * (c[1] - gb.jlo) + (long long)sz * (c[2] - gb.klo)] += acc;
}

constexpr double kPi = 3.14159265358979323846;
constexpr double kOneOverPi = 0.31830988618379;

// Smoothed Heaviside of src/toolbox/lsm_calculus_toolbox.f:25-58 and its derivative.
__device__ __forceinline__ double heaviside(double v, double e) {
  if (v < -e) return 0.0;
  if (v > e) return 1.0;
  return 0.5 * (1.0 + v / e + kOneOverPi * sin(kPi * v / e));
}
__device__ __forceinline__ double heaviside_d(double v, double e) {
  if (v < -e || v > e) return 0.0;
  return 0.5 / e * (1.0 + kOneOverPi * kPi * cos(kPi * v / e));
}

struct MismatchOp {
  const real_t *phi, *tgt;
  Box gb;
  int sy, sz;
  double e, dV;
  __device__ double operator()(int i, int j, int k) const {
    const long long o = (i - gb.ilo) + (long long)sy * (j - gb.jlo) + (long long)sz * (k - gb.klo);
    const double r = heaviside((double)phi[o], e) - heaviside((double)tgt[o], e);
    return r * r * dV;
  }
};

__global__ void __launch_bounds__(256) mismatch_grad_kernel(real_t* grad, const real_t* phi, const real_t* tgt,
                                                            Box gb, Box fb, int sy, int sz, double e, double dV) {
  LSMHIP_CELL(gb);
  const long long o = (i - gb.ilo) + (long long)sy * (j - gb.jlo) + (long long)sz * (k - gb.klo);
  double g = 0.0;
  if (fb.has(i, j, k)) {
    const double p = (double)phi[o];
    g = 2.0 * (heaviside(p, e) - heaviside((double)tgt[o], e)) * heaviside_d(p, e) * dV;
  }
  grad[o] = (real_t)g;
}

// The marches are chains of a memory round trip per cell, seven at the least, which
// a small grid has too few columns to hide, while its 21 weights a cell lie in the
// caches.  By the fill box's waves (rows cut into 64 cells), and by those that the
// weights' kernels launch for them (rows in groups of 32: many more where there are
// few rows along j); a stage, us, weights / marches, lam_out not zero within 4 cells
// of an interface and everywhere:
//   FP32 64^3 (4096 waves) 32 / 51, 37 / 56; 96^3 (18432) 59 / 63, 70 / 84; 104^3
//   (21632) 73 / 71, 87 / 90; 112^3 (25088) 77 / 72, 94 / 111; 128^3 (32768) 120 / 82,
//   133 / 126; 512 x 4 x 512 (16384, 131072 launched) 335 / 130 both
//   FP64 64^3 40 / 68, 47 / 79; 96^3 89 / 111, 110 / 157; 60 x 90 x 200 (18000)
//   113 / 124, 149 / 195; 104^3 124 / 126, 157 / 174; 60 x 120 x 200 (24000) 203 / 144,
//   232 / 228; 112^3 169 / 147, 201 / 224; 120^3 (28800) 201 / 152, 236 / 246; 128^3
//   266 / 163, 290 / 252
// The line is drawn for gradients near an interface, which is what a loss of a level
// set has.
bool marched(const Box& f) {
  const dim3 g = grid_for(f);
  const long long waves = (long long)((f.nx() + 63) / 64) * f.ny() * f.nz();
  return waves >= 24000 || (long long)g.x * g.y * g.z * kBY >= 32768;
}

}  // namespace

// ---------------------------------------------------------------------------
// Entry points (no counterpart in the reference).  Arrays are device arrays on
// the ghost box gb; the stage is the one lsmhip_weno5_stage_normal computes.
// ---------------------------------------------------------------------------

// Reverse of one normal-motion stage (stage 1, 2, 3 of TVD-RK3 or 22 = TVD-RK2
// stage 2).  Accumulates into lam_us (ghost box), lam_uc (fill box; ignored for
// stage 1, may be null) and lam_vn (fill box, only when vn_field is given; may
// be null).  lam_out is read on fb.  scratch: 21 * |gb| reals.  Returns 0 or -1.
LSMHIP_EXPORT int lsmhip_weno5_stage_normal_adjoint(real_t* lam_us, real_t* lam_uc, real_t* lam_vn,
                                                    const real_t* lam_out, const real_t* phi_stage,
                                                    LSMHIP_BOXP(gb), LSMHIP_BOXP(fb), int stage, real_t vn,
                                                    const real_t* vn_field, real_t dt, real_t dx, real_t dy,
                                                    real_t dz, real_t* scratch) {
  LSMHIP_REQUIRE_ARRAYS_OR(-1, lam_us, lam_out, phi_stage, scratch);
  const char* who = "lsmhip_weno5_stage_normal_adjoint";
  AdjArgs A{};
  A.gb = LSMHIP_BOX(gb);
  A.fb = LSMHIP_BOX(fb);
  if (A.fb.empty()) return 0;
  if (!check_box(A.gb, A.fb.widen(3, 3, 3), who, "phi_stage") || !check_size(A.gb, who)) return -1;
  if (!lam_us || !lam_out || !phi_stage || !scratch) {
    set_error(kErrArg, "%s: lam_us, lam_out, phi_stage and scratch are required", who);
    return -1;
  }
  switch (stage) {
    case 1: A.a = 0; A.b = 1; break;
    case 2: A.a = real_t(0.75); A.b = real_t(0.25); break;
    case 3: A.a = real_t(1.0 / 3.0); A.b = real_t(2.0 / 3.0); break;
    case 22: A.a = real_t(0.5); A.b = real_t(0.5); break;
    default:
      set_error(kErrArg, "%s: stage must be 1, 2, 3 or 22, got %d", who, stage);
      return -1;
  }
  A.us = phi_stage;
  A.lam_out = lam_out;
  A.lam_us = lam_us;
  A.lam_uc = stage == 1 ? nullptr : lam_uc;
  A.lam_v = lam_vn;
  A.vnf = vn_field;
  A.vn = vn;
  A.dt = dt;
  A.inv[0] = real_t(1) / dx;
  A.inv[1] = real_t(1) / dy;
  A.inv[2] = real_t(1) / dz;
  A.q = scratch;
  A.vol = A.gb.volume();
  A.sy = A.gb.nx();
  A.sz = A.gb.nx() * A.gb.ny();
  auto overlap = [&](const real_t* a, const real_t* b) { return a && b && a < b + A.vol && b < a + A.vol; };
  bool shared = false;
  for (const real_t* out : {A.lam_us, A.lam_uc, A.lam_v})
    for (const real_t* in : {A.us, A.lam_out, A.vnf}) shared = shared || overlap(out, in);
  shared = shared || overlap(A.lam_us, A.lam_uc) || overlap(A.lam_us, A.lam_v) || overlap(A.lam_uc, A.lam_v);
  if (shared || !marched(A.fb)) {
    hipLaunchKernelGGL(adj_weights_kernel, grid_for(A.fb), block2d(), 0, stream(), A);
    hipLaunchKernelGGL(adj_gather_kernel, grid_for(A.gb), block2d(), 0, stream(), A);
    return finish(who) ? 0 : -1;
  }
  // The marches.  256^3 FP32, a stage of a loss near one interface (lam_out not
  // zero within some 30 cells of it): 1153 us through the 21 weights, 275 us here
  // (102 the coefficients, 108 and 64 the two marches).
  for (int d = 0; d < 3; d++) A.c[d] = scratch + d * A.vol;
  A.flags = reinterpret_cast<unsigned char*>(scratch + 3 * A.vol);
  const Box& f = A.fb;
  // enough waves for the chip before longer columns (256^3: 1 plane 116 us, 2 107, 4 103, 8 102, 16 107)
  const dim3 one = grid_for(f);
  const long long waves = (long long)one.x * one.y * one.z * kBY;
  const int kp = waves >= 8 * 8192 ? 8 : waves >= 2 * 8192 ? 2 : 1;
  hipLaunchKernelGGL(adj_coef_kernel, grid_for_cells(f, kp), block2d(), 0, stream(), A, kp);
  // Length of the march's chunks (columns: blocks side by side, n: targets along
  // the march).  A chunk forms six gradients more than it has targets, and it is
  // one serial chain of memory round trips where it meets flagged cells, so the
  // chip needs many: 4096 blocks or more (256^3, the march along j with x / along
  // k: 1024 blocks 160 / 103 us, 2048 131 / 75, 4096 108 / 64, 8192 100 / 60, which
  // repeats the gradients of half the cells where lam_out is dense).
  auto march_len = [&](long long columns, int n) {
    const long long want = (4096 + columns - 1) / columns;
    const int len = (int)((n + want - 1) / want);
    return len < 8 ? 8 : len > 64 ? 64 : len;
  };
  const unsigned by = (unsigned)((f.nz() + kBY - 1) / kBY), bz = (unsigned)((f.ny() + kBY - 1) / kBY);
  const unsigned tx = (unsigned)((f.nx() + 6 + kColX - 1) / kColX), ti = (unsigned)((f.nx() + kBX - 1) / kBX);
  const int ly = march_len((long long)tx * by, f.ny() + 6), lz = march_len((long long)ti * bz, f.nz() + 6);
  hipLaunchKernelGGL((adj_march_kernel<1, true>), dim3(tx, by, (unsigned)((f.ny() + 6 + ly - 1) / ly)), block2d(), 0,
                     stream(), A, ly);
  hipLaunchKernelGGL((adj_march_kernel<2, false>), dim3(ti, bz, (unsigned)((f.nz() + 6 + lz - 1) / lz)), block2d(), 0,
                     stream(), A, lz);
  return finish(who) ? 0 : -1;
}

// Adjoint of lsmhip_fill_ghosts(kind = periodic, all faces): adds every ghost
// entry of lam to the interior cell it copies and zeroes the ghosts.
LSMHIP_EXPORT int lsmhip_periodic_fill_adjoint(real_t* lam, LSMHIP_BOXP(gb), LSMHIP_BOXP(fb)) {
  LSMHIP_REQUIRE_ARRAYS_OR(-1, lam);
  const char* who = "lsmhip_periodic_fill_adjoint";
  Box g = LSMHIP_BOX(gb), f = LSMHIP_BOX(fb);
  if (f.empty()) return 0;
  if (!check_box(g, f, who, "lam") || !check_size(g, who)) return -1;
  if (g.ilo < f.ilo - f.nx() || g.ihi > f.ihi + f.nx() || g.jlo < f.jlo - f.ny() || g.jhi > f.jhi + f.ny() ||
      g.klo < f.klo - f.nz() || g.khi > f.khi + f.nz()) {
    set_error(kErrArg, "%s: ghost layers wider than the period", who);
    return -1;
  }
  FoldBox F{g, f, {}, {}, 0, 0, 0};
  const int n[3] = {f.nx(), f.ny(), f.nz()};
  const int below[3] = {f.ilo - g.ilo, f.jlo - g.jlo, f.klo - g.klo};
  const int above[3] = {g.ihi - f.ihi, g.jhi - f.jhi, g.khi - f.khi};
  for (int d = 0; d < 3; d++) {  // the ghosts above an axis copy its low cells, those below its high ones
    F.nlo[d] = above[d];
    F.nhi[d] = below[d] < n[d] - above[d] ? below[d] : n[d] - above[d];
  }
  F.cz = (long long)(F.nlo[2] + F.nhi[2]) * n[0] * n[1];
  const long long mz = n[2] - F.nlo[2] - F.nhi[2], my = n[1] - F.nlo[1] - F.nhi[1];
  F.cy = mz * (F.nlo[1] + F.nhi[1]) * n[0];
  F.cx = mz * my * (F.nlo[0] + F.nhi[0]);
  const long long cells = F.cz + F.cy + F.cx;
  if (cells == 0) return 0;  // no ghost layers
  hipLaunchKernelGGL(fold_kernel, dim3((unsigned)((cells + 255) / 256)), dim3(256), 0, stream(), lam, F, g.nx(),
                     g.nx() * g.ny());
  return finish(who) ? 0 : -1;
}

// J = sum over fb of (H_eps(phi) - H_eps(target))^2 dx dy dz, accumulated in
// FP64 (H_eps of src/toolbox/lsm_calculus_toolbox.f:25-58), and, when grad is
// not null, dJ/dphi on gb (zero off fb).  Returns 0 or -1.
LSMHIP_EXPORT int lsmhip_heaviside_mismatch(double* loss, real_t* grad, const real_t* phi, const real_t* target,
                                            LSMHIP_BOXP(gb), LSMHIP_BOXP(fb), double dx, double dy, double dz,
                                            double epsilon) {
  LSMHIP_REQUIRE_ARRAYS_OR(-1, loss, phi, target);
  const char* who = "lsmhip_heaviside_mismatch";
  Box g = LSMHIP_BOX(gb), f = LSMHIP_BOX(fb);
  if (!check_box(g, f, who, "phi") || !check_size(g, who)) return -1;
  MismatchOp op{phi, target, g, g.nx(), g.nx() * g.ny(), epsilon, dx * dy * dz};
  double s = 0.0;
  if (!f.empty() && !reduce::box_sum(who, f, op, &s)) return -1;
  if (loss) *loss = s;
  if (grad) {
    hipLaunchKernelGGL(mismatch_grad_kernel, grid_for(g), block2d(), 0, stream(), grad, phi, target, g, f, g.nx(),
                       g.nx() * g.ny(), epsilon, dx * dy * dz);
    if (!finish(who)) return -1;
  }
  return 0;
}
