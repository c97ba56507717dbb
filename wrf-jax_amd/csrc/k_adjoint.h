// Tangent-linear and adjoint of the scalar transport of one RK stage:
// advect_scalar (flux form, 5th-order horizontal / 3rd-order vertical,
// specified boundaries; module_advect_em.py:90-369, _fast.py:1437-1769)
// followed by rk_update_scalar (module_em.py:1437-1598) with the stage's
// recorded mass fluxes (ru_m, rv_m, ww_m) and column masses (mu_1, mu_2):
//   tend  = A q_in                   (A: the advect_scalar operator)
//   q_out = (m_old q_old + dt msfty [inner] tend) / m_new
// with m = c1h (mu + mub) + c2h.  For fixed fluxes the stage is linear in
// (q_old, q_in), so the tangent-linear stage is the stage itself: the
// dycore's advect_scalar kernel, which ends with the update (k_advect.h,
// kAdvTransport).  The adjoint is its transpose, k_ad_update then k_ad_advect
// (q_in_bar += A^T tend_bar).  In a window of stages run backwards, a
// stage's q_in_bar is the next one's q_out_bar at the same point, so
// k_ad_advect forms that stage's update in place of writing it (AdNext).
#pragma once

#include "wrfdc_common.h"

struct StageMass {
  const float *mu_1, *mu_2;  // recorded column masses of the stage (perturbation; + mub)
};

// column masses and map factor of the update at one point
struct StageCoef {
  float oldm, newm, msfty;
  bool inner;
};
__device__ __forceinline__ StageCoef stage_coef(CtxPtr x, const StageMass &sm, int i, int k, int j) {
  StageCoef c;
  const int sz = x->spec_zone;
  c.inner = i >= 1 + sz && i <= x->ide - sz - 1 && j >= 1 + sz && j <= x->jde - sz - 1;
  const float mub = A2(FL(mub), i, j), c1 = A1(FL(c1h), k), c2 = A1(FL(c2h), k);
  c.oldm = c1 * (A2(sm.mu_1, i, j) + mub) + c2;
  c.newm = c1 * (A2(sm.mu_2, i, j) + mub) + c2;
  c.msfty = A2(FL(msfty), i, j);
  return c;
}

// transpose of the update: q_old_bar += (m_old / m_new) q_out_bar,
// tend_bar = dt msfty [inner] / m_new q_out_bar; first: qbar_old starts from 0
__global__ void k_ad_update(const DevCtx *xv, R3 r, StageMass sm, const float *__restrict__ qbar_out, float *__restrict__ qbar_old,
                            float *__restrict__ tbar, float dt, int first) {
  const CtxPtr x = ctx_ptr(xv);
  GET_IKJ_P(r);
  const StageCoef c = stage_coef(x, sm, i, k, j);
  const float qb = A3(qbar_out, i, k, j);
  const float q0 = first ? 0.f : A3(qbar_old, i, k, j);
  A3(qbar_old, i, k, j) = q0 + c.oldm / c.newm * qb;
  A3(tbar, i, k, j) = c.inner ? dt * c.msfty / c.newm * qb : 0.f;
}

// Coefficient of q(f + m) in the flux through a face, for the velocity's
// sign s (flux5 / flux3 of module_advect_em.py:29-57); the second order's is
// 1/2 for m = -1 and 0.
template <int M>
__device__ __forceinline__ float coef5(bool up) {
  constexpr float p[6] = {2.f / 60.f, -13.f / 60.f, 47.f / 60.f, 27.f / 60.f, -3.f / 60.f, 0.f};
  constexpr float n[6] = {0.f, -3.f / 60.f, 27.f / 60.f, 47.f / 60.f, -13.f / 60.f, 2.f / 60.f};
  return up ? p[M + 3] : n[M + 3];
}
template <int M>
__device__ __forceinline__ float coef3(bool up) {
  constexpr float p[6] = {0.f, -2.f / 12.f, 10.f / 12.f, 4.f / 12.f, 0.f, 0.f};
  constexpr float n[6] = {0.f, 0.f, 4.f / 12.f, 10.f / 12.f, -2.f / 12.f, 0.f};
  return up ? p[M + 3] : n[M + 3];
}

// Horizontal part of A^T at one point c of a row of cells: the faces f = c -
// M, M in [-3, 2], whose fluxes read it.  Face f's dual is F_bar(f) = msf(f)
// rd tbar(f) [f has a tendency: 2 .. e-2] - msf(f-1) rd tbar(f-1) [f-1 has].
// t, ms: tbar and msf at cells c-3 .. c+3; v: the velocities of faces c-2 ..
// c+3.  Faces exist in [2, e-1]: second order at 2 and e-1, 5th in [4, e-3],
// else 3rd.  fast (uniform over the wave): all six faces are of 5th order and
// their cells have tendencies.
template <int M>
__device__ __forceinline__ void ad_face(const float t[7], const float ms[7], const float v[6], float rd, int c, int e, bool fast, float &acc) {
  constexpr int q = 3 - M;  // t[q]: cell f, t[q - 1]: cell f - 1, v[q - 1]: face f
  const int f = c - M;
  const float vel = v[q - 1];
  const bool up = vel >= 0.f;
  const float hi = ms[q] * rd * t[q], lo = ms[q - 1] * rd * t[q - 1];
  float coef = coef5<M>(up), fb = (0.f + hi) - lo;
  if (!fast) {
    fb = 0.f;
    if (f <= e - 2) fb += hi;
    if (f - 1 >= 2) fb -= lo;
    const bool five = f >= 4 && f <= e - 3, two = f == 2 || f == e - 1;
    constexpr bool in2 = M == -1 || M == 0, in3 = M >= -2 && M <= 1;  // cells a 2nd- / 3rd-order flux reads
    coef = five ? coef : two ? 0.5f : coef3<M>(up);
    // a face whose flux does not read c adds nothing: 0 times its values would
    // not be 0 where they are infinite or NaN
    if (f < 2 || f > e - 1 || !(five || (two ? in2 : in3))) return;
  }
  acc += vel * coef * fb;
}
__device__ __forceinline__ void ad_row(const float t[7], const float ms[7], const float v[6], float rd, int c, int e, bool fast, float &acc) {
  ad_face<-3>(t, ms, v, rd, c, e, fast, acc);
  ad_face<-2>(t, ms, v, rd, c, e, fast, acc);
  ad_face<-1>(t, ms, v, rd, c, e, fast, acc);
  ad_face<0>(t, ms, v, rd, c, e, fast, acc);
  ad_face<1>(t, ms, v, rd, c, e, fast, acc);
  ad_face<2>(t, ms, v, rd, c, e, fast, acc);
}

// what a stage's q_in_bar becomes in a window run backwards
enum { kAdAdd = 0,   // q_in_bar += A^T tbar (a stage on its own; the last stage of a window)
       kAdNext = 1,  // stages 3 and 2: the q_out_bar of the stage before, whose update follows here
       kAdStep = 2   // stage 1: complete once acc is added, the q_out_bar of the previous step's stage 3
};
struct AdNext {
  StageMass sm;  // the next stage's masses
  float *tbar;   // and its tend_bar
  float dt;
};

// A^T tend_bar at the mass points [1, ide-1] x [1, kde-1] x [1, jde-1]
// (gather: each point collects the faces whose fluxes read it).  Vertical
// faces f in [3, ktf-1] are 3rd order with the velocity's sign reversed (eta
// falls upward), f = 2 and ktf second order through fzm / fzp, 1 and kde
// zero.  qbar: q_in_bar (kAdAdd) or the window's accumulated q_old_bar.
//
// Bound by loads: 47 per point.  All of them go out first, unclamped through
// buffer descriptors (what lies outside the field is not used), and only then
// the orders are chosen; with a branch and a switch around each face's loads
// and a division per coefficient the stage took 76 us at 200x200x45 and its
// update 12 us in a pass of its own, 28 us together this way.
template <int MODE>
__global__ void __launch_bounds__(256) k_ad_advect(const DevCtx *xv, R3 r, const float *__restrict__ tbar, const float *__restrict__ ru,
                                                   const float *__restrict__ rv, const float *__restrict__ rom, float *__restrict__ qbar,
                                                   AdNext nx) {
  const CtxPtr x = ctx_ptr(xv);
  GET_IKJ(r);
  const int ide = x->ide, jde = x->jde, ktf = x->kde - 1;
  const float rdx = x->rdx, rdy = x->rdy;
  const float *rdzw = FL(rdnw), *fzm = FL(fnm), *fzp = FL(fnp);
  const unsigned n3 = (unsigned)x->n3, n2 = (unsigned)x->n2, sk = (unsigned)x->ip, sj = (unsigned)(x->kde * x->ip);
  const BufF bt = bufv(tbar, n3), bu = bufv(ru, n3), bv = bufv(rv, n3), bw = bufv(rom, n3), bm = bufv(FL(msftx), n2);
  const unsigned o = XI3(i, k, j), o2 = XI2(i, j);
  float tx[7], ty[7], tz[5], mx[7], my[7], u[6], v[6], w[4];
#pragma unroll
  for (int q = 0; q < 7; q++) {
    tx[q] = bld(bt, o + (unsigned)(q - 3));
    ty[q] = bld(bt, o + (unsigned)(q - 3) * sj);
    mx[q] = bld(bm, o2 + (unsigned)(q - 3));
    my[q] = bld(bm, o2 + (unsigned)(q - 3) * sk);
  }
#pragma unroll
  for (int q = 0; q < 6; q++) {
    u[q] = bld(bu, o + (unsigned)(q - 2));
    v[q] = bld(bv, o + (unsigned)(q - 2) * sj);
  }
#pragma unroll
  for (int q = 0; q < 5; q++) tz[q] = bld(bt, o + (unsigned)(q - 2) * sk);
#pragma unroll
  for (int q = 0; q < 4; q++) w[q] = bld(bw, o + (unsigned)(q - 1) * sk);
  const float q0 = elem(qbar, o);
  float acc = 0.f;
  // 5th-order faces and tendencies on both sides: f in [4, e-3] for f = c-2 .. c+3
  const bool fx = i >= 6 && i <= ide - 6, fy = j >= 6 && j <= jde - 6;
  ad_row(tx, mx, u, rdx, i, ide, __all(fx), acc);
  ad_row(ty, my, v, rdy, j, jde, fy, acc);
  // vertical faces f = k - m, m in [-2, 1]: tz[3 - m - 1] is cell f, w[1 - m] face f
#pragma unroll
  for (int m = -2; m <= 1; m++) {
    const int f = k - m;
    if (f < 2 || f > ktf) continue;
    const float vel = w[1 - m];
    float coef;
    if (f == 2 || f == ktf) coef = m == 0 ? A1(fzm, f) : (m == -1 ? A1(fzp, f) : 0.f);
    else coef = m == -2 ? coef3<-2>(-vel >= 0.f) : m == -1 ? coef3<-1>(-vel >= 0.f) : m == 0 ? coef3<0>(-vel >= 0.f) : coef3<1>(-vel >= 0.f);
    // V_bar(f) = rdzw(f) tbar(f) - rdzw(f-1) tbar(f-1), tendencies at [1, ktf]
    float vb = 0.f;
    vb += A1(rdzw, f) * tz[2 - m];
    vb -= A1(rdzw, f - 1) * tz[1 - m];
    if (coef != 0.f) acc += vel * coef * vb;
  }
  if (MODE == kAdAdd) {
    elem(qbar, o) = q0 + acc;
  } else {
    const StageCoef c = stage_coef(x, nx.sm, i, k, j);
    const float qb = MODE == kAdNext ? 0.f + acc : q0 + acc;
    elem(qbar, o) = (MODE == kAdNext ? q0 : 0.f) + c.oldm / c.newm * qb;
    elem(nx.tbar, o) = c.inner ? nx.dt * c.msfty / c.newm * qb : 0.f;
  }
}
