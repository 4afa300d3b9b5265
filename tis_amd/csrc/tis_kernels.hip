// tis_kernels.hip -- CDNA4 (gfx950) kernels of the DT15 TIS force-and-
// integrate path.  One wave (64 lanes) per work tile; a tile is 64 beads (or
// 64 charges) of one system.  Each lane owns one bead and gathers every force
// on it in a fixed order (bonded terms via the incidence list, excluded
// volume via its own neighbour list, Debye-Hueckel via the per-charge sums of
// the pre-pass), accumulating in FP64.  Pair arithmetic (mWCA, DH) is FP32 on
// FP64 coordinate differences; cutoff and list tests are FP64 with the
// reference's rounding.  Reference routines restated (src/ of the reference):
//   force_bond.F90:40-58, force_bangle.F90:40-84, force_dtrna_stack.F90:53-165,
//   force_dtrna_stack_nlocal.F90:48-263, force_dtrna_hbond15.F90:91-535,
//   force_exv_dt15.F90:53-115, force_ele_DH.F90:68-118,
//   neighbor_list.F90:56-87 + neighbor_assign.F90:481-559, neighbor_list_ele.F90:123-210,
//   neighbor_list_hb.F90:59-78, util_periodic.F90:26-36, time_integral.F90:149-183,
//   time_integral_pre.F90:176-179, energy_*.F90.
#include <type_traits>

#include "tis_dev.h"

// Multiply-adds are fused where one expression writes them, and nowhere else:
// a term evaluated by two kernels (the per-step passes and k_window) then has
// the same bits in both, whatever code surrounds it.
#pragma clang fp contract(on)

namespace tis {

// Coordinates as the terms read them: component d of bead g, from an SoA
// array in global memory or (k_window) from the workgroup's copy of its
// system's beads in LDS.
struct GlobalX {
  const double *p;
  int n;
  __device__ double operator()(int d, int g) const { return p[(size_t)d * n + g]; }
};
struct LocalX {
  const double *p;   // [3][n], bead off first
  int n, off;
  __device__ double operator()(int d, int g) const { return p[d * n + g - off]; }
};

__device__ inline void ld3(const double *X, int n, int g, double r[3]) {
  r[0] = X[g]; r[1] = X[n + g]; r[2] = X[2 * n + g];
}
__device__ inline double dot3(const double a[3], const double b[3]) {
  return (a[0] * b[0] + a[1] * b[1]) + a[2] * b[2];
}
__device__ inline void cross3(const double a[3], const double b[3], double c[3]) {
  c[0] = a[1] * b[2] - a[2] * b[1];
  c[1] = a[2] * b[0] - a[0] * b[2];
  c[2] = a[0] * b[1] - a[1] * b[0];
}
__device__ inline double wrap_pi(double d) {
  if (d > kPi) return d - 2.0 * kPi;
  if (d < -kPi) return d + 2.0 * kPi;
  return d;
}
__device__ inline void vsub(const double *X, int n, int a, int b, double v[3]) {
  v[0] = X[a] - X[b]; v[1] = X[n + a] - X[n + b]; v[2] = X[2 * n + a] - X[2 * n + b];
}
template <class XA>
__device__ inline void vsub(const XA &X, int a, int b, double v[3]) {
  v[0] = X(0, a) - X(0, b); v[1] = X(1, a) - X(1, b); v[2] = X(2, a) - X(2, b);
}

// The FP32 record of a bead (see kNearMargin): position and excluded-volume
// species.
__device__ inline float4 near_pos(double x, double y, double z, int species) {
  const bool ok = fabs(x) <= kNearMax && fabs(y) <= kNearMax && fabs(z) <= kNearMax;
  return make_float4(ok ? (float)x : __builtin_nanf(""), (float)y, (float)z, __int_as_float(species));
}

// The value of v at lane r (the same for every lane) of the wave.
__device__ inline double at_lane(double v, int r) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, r);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), r);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// ------------------------------------------------------------------ bonded
// Each bonded term is evaluated once (one lane per term) and its per-bead
// forces are written to the slots of the beads' incidence lists.

// force_bond.F90:40-58: fo[0..2] on bead 1, fo[3..5] on bead 2
template <class XA>
__device__ inline void bond_eval(const XA &X, int i, int j, double nat, double coef, double fo[6]) {
  double v[3];
  vsub(X, j, i, v);
  double dist = sqrt(dot3(v, v));
  double dd = dist - nat;
  double fr = coef * (-2.0 * dd / dist);
  for (int d = 0; d < 3; ++d) { fo[d] = -(fr * v[d]); fo[3 + d] = fr * v[d]; }
}

// force_bangle.F90:40-84
template <class XA>
__device__ inline void angle_eval(const XA &X, int i1, int i2, int i3, double nat, double coef, double fo[9]) {
  for (int k = 0; k < 9; ++k) fo[k] = 0.0;
  if (coef < 1.0e-6) return;
  double v21[3], v32[3];
  vsub(X, i2, i1, v21);
  vsub(X, i3, i2, v32);
  double c11 = dot3(v21, v21), c22 = dot3(v32, v32), c21 = dot3(v32, v21);
  double ct = -c21 / sqrt(c11 * c22);
  ct = ct > 1.0 ? 1.0 : (ct < -1.0 ? -1.0 : ct);
  double dba = acos(ct) - nat;
  double t3 = c11 * c22 - c21 * c21;
  if (t3 <= 1.0) t3 = 1.0;
  double fr = 2.0 * coef * dba / sqrt(t3);
  for (int d = 0; d < 3; ++d) {
    double f21 = fr * (v21[d] * (c21 / c11) - v32[d]);
    double f32 = fr * (v32[d] * (c21 / c22) - v21[d]);
    fo[d] = -f21; fo[3 + d] = f21 - f32; fo[6 + d] = f32;
  }
}

// force_dtrna_stack.F90:53-165: fo[3*k + d] on bead k of B1 B2 P1 S1 P2 S2 P3
template <class XA>
__device__ inline void stack_eval(const XA &X, const int m7[7], const double nat[3], const double cf[4],
                                  double fo[21]) {
  double v21[3], v34[3], v54[3], v56[3], v76[3], m[3], nn[3], fi[3], fl[3];
  vsub(X, m7[1], m7[0], v21);
  vsub(X, m7[2], m7[3], v34);
  vsub(X, m7[4], m7[3], v54);
  vsub(X, m7[4], m7[5], v56);
  vsub(X, m7[6], m7[5], v76);
  double ediv = 1.0;
  double dist = sqrt(dot3(v21, v21));
  double dd = dist - nat[0];
  ediv += cf[1] * dd * dd;
  for (int d = 0; d < 3; ++d) {
    fi[d] = 2.0 * cf[1] * dd / dist * v21[d];
    fo[d] = -fi[d]; fo[3 + d] = fi[d];
  }
  cross3(v34, v54, m);
  cross3(v54, v56, nn);
  double dmm = dot3(m, m), dnn = dot3(nn, nn), d5454 = dot3(v54, v54);
  double abs54 = sqrt(d5454), d5654 = dot3(v56, v54);
  double d3454o = dot3(v34, v54) / d5454, d5654o = d5654 / d5454;
  double dph = wrap_pi(atan2(dot3(v34, nn) * sqrt(d5454), dot3(m, nn)) - nat[1]);
  ediv += cf[2] * dph * dph;
  for (int d = 0; d < 3; ++d) {
    fi[d] = 2.0 * cf[2] * dph * abs54 / dmm * m[d];
    fl[d] = -2.0 * cf[2] * dph * abs54 / dnn * nn[d];
    fo[6 + d] = fi[d];
    fo[9 + d] = (-1.0 + d3454o) * fi[d] - d5654o * fl[d];
    fo[12 + d] = (-1.0 + d5654o) * fl[d] - d3454o * fi[d];
    fo[15 + d] = fl[d];
  }
  cross3(v76, v56, m);
  for (int d = 0; d < 3; ++d) nn[d] = -nn[d];
  dmm = dot3(m, m);
  double d5656 = dot3(v56, v56), abs56 = sqrt(d5656);
  double d7656o = dot3(v76, v56) / d5656, d5456o = d5654 / d5656;
  dph = wrap_pi(atan2(dot3(v76, nn) * sqrt(d5656), dot3(m, nn)) - nat[2]);
  ediv += cf[3] * dph * dph;
  for (int d = 0; d < 3; ++d) {
    fi[d] = 2.0 * cf[3] * dph * abs56 / dmm * m[d];
    fl[d] = -2.0 * cf[3] * dph * abs56 / dnn * nn[d];
    fo[18 + d] = fi[d];
    fo[15 + d] += (-1.0 + d7656o) * fi[d] - d5456o * fl[d];
    fo[12 + d] += -d7656o * fi[d] + (-1.0 + d5456o) * fl[d];
    fo[9 + d] += fl[d];
  }
  double sc = cf[0] / (ediv * ediv);
  for (int k = 0; k < 21; ++k) fo[k] *= sc;
}

__device__ inline void put_slots(const DevPtrs &P, int64_t base, int term, int nslot, const double *fo) {
  float *o = P.fslot + 3 * (base + (int64_t)nslot * term);   // the term's nslot 12-byte slots, contiguous
  for (int k = 0; k < 3 * nslot; ++k) o[k] = (float)fo[k];
}

// st_status of force_dtrna_stack_nlocal.F90:83-92 evaluated where it is
// read: consecutive stack st is off when one of the exclusive tertiary
// stacks that name it has d - d0 < 10 (the same FP64 operations as
// tstack_eval).
__device__ inline bool stack_on(const DevPtrs &P, const double *X, const double *PX, int st) {
  const int n = P.ntot;
  for (int e = P.st_exoff[st]; e < P.st_exoff[st + 1]; ++e) {
    const int t = P.st_ex[e];
    const DSys *sp = P.sys + P.tst_sys[t];
    const int32_t *m6 = P.tst_mp + 6 * t;
    double v12[3];
    if (sp->periodic) { vsub(PX, n, m6[0], m6[1], v12); pbneighbor(*sp, v12); }
    else vsub(X, n, m6[0], m6[1], v12);
    const double d1212 = dot3(v12, v12), a12 = sqrt(d1212);
    if (a12 - P.tst_nat[6 * t] < 10.0) return false;
  }
  return true;
}

// Bonded terms of the launch range: one lane per consecutive stack, angle or
// bond, in that order (the heaviest terms start first; the force pass runs
// these blocks last).

__device__ inline void bonded_lane(const DevPtrs &P, const double *X, const double *PX, const BondedRange &R,
                                   int t) {
  const int nb = R.nb, na = R.na, ns = R.ns, b0 = R.b0, a0 = R.a0, s0 = R.s0;
  if (t >= nb + na + ns) return;
  t = t < ns ? t + nb + na : (t < ns + na ? t - ns + nb : t - ns - na);   // stacks, angles, bonds
  if (t < nb) {
    double fo[6];
    const int b = b0 + t;
    bond_eval(GlobalX{X, P.ntot}, P.bd_mp[2 * b], P.bd_mp[2 * b + 1], P.bd_nat[b], P.bd_coef[b], fo);
    put_slots(P, P.sb_bd, b0 + t, 2, fo);
    return;
  }
  t -= nb;
  if (t < na) {
    double fo[9];
    const int a = a0 + t;
    angle_eval(GlobalX{X, P.ntot}, P.ba_mp[3 * a], P.ba_mp[3 * a + 1], P.ba_mp[3 * a + 2], P.ba_nat[a], P.ba_coef[a],
               fo);
    put_slots(P, P.sb_ba, a0 + t, 3, fo);
    return;
  }
  t -= na;
  if (t < ns) {
    const int st = s0 + t;
    double fo[21];
    if (stack_on(P, X, PX, st))
      stack_eval(GlobalX{X, P.ntot}, P.st_mp + 7 * st, P.st_nat + 3 * st, P.st_coef + 4 * st, fo);
    else for (int k = 0; k < 21; ++k) fo[k] = 0.0;
    put_slots(P, P.sb_st, st, 7, fo);
  }
}

// ------------------------------------------------------------------ tertiary stack
// force_dtrna_stack_nlocal.F90:48-263 for one tertiary stack: all six slots
// into fo[18] (the exclusion of secondary stacks when d < 10 is stack_on).
__device__ void tstack_eval(const DevPtrs &P, const DSys &s, const double *X, const double *PX,
                            int t, double fo[18]) {
  const int n = P.ntot;
  const int32_t *m6 = P.tst_mp + 6 * t;
  const double *nat = P.tst_nat + 6 * t, *cf = P.tst_coef + 7 * t;
  const double *Y = s.periodic ? PX : X;
  double v12[3], v13[3], v53[3], v42[3], v46[3], fi[3], fk[3], fl[3];
  vsub(Y, n, m6[0], m6[1], v12);
  if (s.periodic) pbneighbor(s, v12);
  double d1212 = dot3(v12, v12), a12 = sqrt(d1212);
  double dd = a12 - nat[0];
  vsub(Y, n, m6[0], m6[2], v13);
  vsub(Y, n, m6[4], m6[2], v53);
  vsub(Y, n, m6[3], m6[1], v42);
  vsub(Y, n, m6[3], m6[5], v46);
  if (s.periodic) { pbneighbor(s, v13); pbneighbor(s, v53); pbneighbor(s, v42); pbneighbor(s, v46); }
  for (int k = 0; k < 18; ++k) fo[k] = 0.0;
  double d1313 = dot3(v13, v13), d4242 = dot3(v42, v42);
  double a13 = sqrt(d1313), a42 = sqrt(d4242);
  double d1213 = dot3(v13, v12), d1242 = dot3(v12, v42), d4246 = dot3(v42, v46), d1353 = dot3(v13, v53);
  double o1213_1212 = d1213 / d1212, o1213_1313 = d1213 / d1313, o1242_1212 = d1242 / d1212;
  double o4246_4242 = d4246 / d4242, o1242_4242 = d1242 / d4242, o1353_1313 = d1353 / d1313;
  double ediv = 1.0 + cf[1] * dd * dd;
  for (int d = 0; d < 3; ++d) {
    fi[d] = 2.0 * cf[1] * dd * v12[d] / a12;
    fo[d] = fi[d]; fo[3 + d] = -fi[d];
  }
  double da = acos(d1213 / (a13 * a12)) - nat[1];
  double pre = 2.0 * cf[2] * da / sqrt(d1313 * d1212 - d1213 * d1213);
  for (int d = 0; d < 3; ++d) {
    fi[d] = pre * (v12[d] - o1213_1313 * v13[d]);
    fk[d] = pre * (v13[d] - o1213_1212 * v12[d]);
    fo[6 + d] += fi[d]; fo[3 + d] += fk[d]; fo[d] = fo[d] - fi[d] - fk[d];
  }
  ediv += cf[2] * da * da;
  da = acos(d1242 / (a12 * a42)) - nat[2];
  pre = 2.0 * cf[3] * da / sqrt(d1212 * d4242 - d1242 * d1242);
  for (int d = 0; d < 3; ++d) {
    fi[d] = -pre * (v42[d] - o1242_1212 * v12[d]);
    fk[d] = -pre * (v12[d] - o1242_4242 * v42[d]);
    fo[d] += fi[d]; fo[9 + d] += fk[d]; fo[3 + d] = fo[3 + d] - fi[d] - fk[d];
  }
  ediv += cf[3] * da * da;
  double c4212[3], c1213[3], m[3], nn[3];
  cross3(v42, v12, c4212);
  cross3(v12, v13, c1213);
  double c4212a = dot3(c4212, c4212), c1213a = dot3(c1213, c1213);
  double dph = wrap_pi(atan2(dot3(v42, c1213) * sqrt(d1212), dot3(c4212, c1213)) - nat[3]);
  ediv += cf[4] * dph * dph;
  pre = 2.0 * cf[4] * dph * a12;
  for (int d = 0; d < 3; ++d) {
    fi[d] = pre / c4212a * c4212[d];
    fl[d] = -pre / c1213a * c1213[d];
    fo[9 + d] += fi[d];
    fo[3 + d] += (-1.0 + o1242_1212) * fi[d] - o1213_1212 * fl[d];
    fo[d] += (-1.0 + o1213_1212) * fl[d] - o1242_1212 * fi[d];
    fo[6 + d] += fl[d];
  }
  cross3(v53, v13, m);
  for (int d = 0; d < 3; ++d) nn[d] = -c1213[d];
  double dmm = dot3(m, m), dnn = c1213a;
  dph = wrap_pi(atan2(dot3(v53, nn) * a13, dot3(m, nn)) - nat[4]);
  ediv += cf[5] * dph * dph;
  pre = 2.0 * cf[5] * dph * a13;
  for (int d = 0; d < 3; ++d) {
    fi[d] = pre / dmm * m[d];
    fl[d] = -pre / dnn * nn[d];
    fo[12 + d] += fi[d];
    fo[6 + d] += (-1.0 + o1353_1313) * fi[d] - o1213_1313 * fl[d];
    fo[d] += (-1.0 + o1213_1313) * fl[d] - o1353_1313 * fi[d];
    fo[3 + d] += fl[d];
  }
  for (int d = 0; d < 3; ++d) m[d] = -c4212[d];
  cross3(v42, v46, nn);
  dmm = c4212a; dnn = dot3(nn, nn);
  dph = wrap_pi(atan2(dot3(v12, nn) * a42, dot3(m, nn)) - nat[5]);
  ediv += cf[6] * dph * dph;
  pre = 2.0 * cf[6] * dph * a42;
  for (int d = 0; d < 3; ++d) {
    fi[d] = pre / dmm * m[d];
    fl[d] = -pre / dnn * nn[d];
    fo[d] += fi[d];
    fo[3 + d] += (-1.0 + o1242_4242) * fi[d] - o4246_4242 * fl[d];
    fo[9 + d] += (-1.0 + o4246_4242) * fl[d] - o1242_4242 * fi[d];
    fo[15 + d] += fl[d];
  }
  double sc = cf[0] / (ediv * ediv);
  for (int k = 0; k < 18; ++k) fo[k] *= sc;
}

// ------------------------------------------------------------------ hbond15
// force_dtrna_hbond15.F90:91-353 (default branch).  Returns 1 and fills
// fo[18], *ene when |r12 - r0| <= hb_cutoff_dist.
template <class XA>
__device__ inline int hbond_eval(const DSys &s, const XA &X, const XA &PX, const int m6[6], const double nat[6],
                                 const double cf[7], double fo[18], double *ene) {
  const double MAXC = cos((double)(0.57f / 180.0f) * kPi);  // const_physical.F90:37-38
  double v12[3], v13[3], v53[3], v42[3], v46[3], fi[3], fk[3], fl[3];
  if (s.periodic) { vsub(PX, m6[0], m6[1], v12); pbneighbor(s, v12); }
  else vsub(X, m6[0], m6[1], v12);
  double d1212 = dot3(v12, v12), a12 = sqrt(d1212);
  double dd = a12 - nat[0];
  if (fabs(dd) > s.hb_cut) return 0;
  double ex = -cf[1] * dd * dd;
  for (int d = 0; d < 3; ++d) {
    fi[d] = (2.0 * cf[1] * dd / a12) * v12[d];
    fo[d] = fi[d]; fo[3 + d] = -fi[d];
  }
  for (int k = 6; k < 18; ++k) fo[k] = 0.0;
  vsub(X, m6[0], m6[2], v13);
  vsub(X, m6[4], m6[2], v53);
  vsub(X, m6[3], m6[1], v42);
  vsub(X, m6[3], m6[5], v46);
  if (s.periodic) { pbneighbor(s, v13); pbneighbor(s, v53); pbneighbor(s, v42); pbneighbor(s, v46); }
  double d1313 = dot3(v13, v13), d4242 = dot3(v42, v42);
  double a13 = sqrt(d1313), a42 = sqrt(d4242);
  double d1213 = dot3(v13, v12), d1242 = dot3(v12, v42), d4246 = dot3(v42, v46), d1353 = dot3(v13, v53);
  double o1213_1212 = d1213 / d1212, o1213_1313 = d1213 / d1313, o1242_1212 = d1242 / d1212;
  double o4246_4242 = d4246 / d4242, o1242_4242 = d1242 / d4242, o1353_1313 = d1353 / d1313;
  double c312 = d1213 / (a13 * a12);
  if (fabs(c312) > MAXC) d1213 = copysign(a12 * a13 * MAXC, c312);
  double da = acos(c312) - nat[1];
  double pre = 2.0 * cf[2] * da / sqrt(d1313 * d1212 - d1213 * d1213);
  for (int d = 0; d < 3; ++d) {
    fi[d] = pre * (v12[d] - o1213_1313 * v13[d]);
    fk[d] = pre * (v13[d] - o1213_1212 * v12[d]);
    fo[6 + d] += fi[d]; fo[3 + d] += fk[d]; fo[d] = fo[d] - fi[d] - fk[d];
  }
  ex = ex - cf[2] * da * da;
  double c124 = d1242 / (a12 * a42);
  if (fabs(c124) > MAXC) d1242 = copysign(a12 * a42 * MAXC, c124);
  da = acos(c124) - nat[2];
  pre = 2.0 * cf[3] * da / sqrt(d1212 * d4242 - d1242 * d1242);
  for (int d = 0; d < 3; ++d) {
    fi[d] = -pre * (v42[d] - o1242_1212 * v12[d]);
    fk[d] = -pre * (v12[d] - o1242_4242 * v42[d]);
    fo[d] += fi[d]; fo[9 + d] += fk[d]; fo[3 + d] = fo[3 + d] - fi[d] - fk[d];
  }
  ex = ex - cf[3] * da * da;
  double c4212[3], c1213[3], c5313[3], c4246[3], nn[3];
  cross3(v42, v12, c4212);
  cross3(v12, v13, c1213);
  double c4212a = dot3(c4212, c4212), c1213a = dot3(c1213, c1213);
  if (fabs(c124) > MAXC) c4212a = d4242 * d1212 * (1.0 - MAXC * MAXC);
  if (fabs(c312) > MAXC) c1213a = d1212 * d1313 * (1.0 - MAXC * MAXC);
  double dph = wrap_pi(atan2(dot3(v42, c1213) * a12, dot3(c4212, c1213)) - nat[3]);
  ex = ex - cf[4] * dph * dph;
  pre = 2.0 * cf[4] * dph * a12;
  for (int d = 0; d < 3; ++d) {
    fi[d] = pre / c4212a * c4212[d];
    fl[d] = -pre / c1213a * c1213[d];
    fo[9 + d] += fi[d];
    fo[3 + d] += (-1.0 + o1242_1212) * fi[d] - o1213_1212 * fl[d];
    fo[d] += (-1.0 + o1213_1212) * fl[d] - o1242_1212 * fi[d];
    fo[6 + d] += fl[d];
  }
  cross3(v53, v13, c5313);
  for (int d = 0; d < 3; ++d) nn[d] = -c1213[d];
  double c5313a = dot3(c5313, c5313);
  double c531 = d1353 / (a13 * sqrt(dot3(v53, v53)));
  if (fabs(c531) > MAXC) c5313a = dot3(v53, v53) * d1313 * (1.0 - MAXC * MAXC);
  dph = wrap_pi(atan2(dot3(v53, nn) * a13, dot3(c5313, nn)) - nat[4]);
  ex = ex - cf[5] * dph * dph;
  pre = 2.0 * cf[5] * dph * a13;
  for (int d = 0; d < 3; ++d) {
    fi[d] = pre / c5313a * c5313[d];
    fl[d] = -pre / c1213a * nn[d];
    fo[12 + d] += fi[d];
    fo[6 + d] += (-1.0 + o1353_1313) * fi[d] - o1213_1313 * fl[d];
    fo[d] += (-1.0 + o1213_1313) * fl[d] - o1353_1313 * fi[d];
    fo[3 + d] += fl[d];
  }
  for (int d = 0; d < 3; ++d) nn[d] = -c4212[d];
  cross3(v42, v46, c4246);
  double c4246a = dot3(c4246, c4246);
  double c246 = d4246 / (a42 * sqrt(dot3(v46, v46)));
  if (fabs(c246) > MAXC) c4246a = dot3(v46, v46) * d4242 * (1.0 - MAXC * MAXC);
  dph = wrap_pi(atan2(dot3(v12, c4246) * a42, dot3(nn, c4246)) - nat[5]);
  ex = ex - cf[6] * dph * dph;
  pre = 2.0 * cf[6] * dph * a42;
  for (int d = 0; d < 3; ++d) {
    fi[d] = pre / c4212a * nn[d];
    fl[d] = -pre / c4246a * c4246[d];
    fo[d] += fi[d];
    fo[3 + d] += (-1.0 + o1242_4242) * fi[d] - o4246_4242 * fl[d];
    fo[9 + d] += (-1.0 + o4246_4242) * fl[d] - o1242_4242 * fi[d];
    fo[15 + d] += fl[d];
  }
  double e = cf[0] * exp(ex);
  *ene = e;
  for (int k = 0; k < 18; ++k) fo[k] = e * fo[k];
  return 1;
}

__device__ inline int hbond_at(const DevPtrs &P, const DSys &s, const double *X, const double *PX, int h,
                               double fo[18], double *ene) {
  return hbond_eval(s, GlobalX{X, P.ntot}, GlobalX{PX, P.ntot}, P.hb_mp + 6 * h, P.hb_nat + 6 * h, P.hb_coef + 7 * h,
                    fo, ene);
}

__device__ inline int site_count(const DevPtrs &P, int site) {
  return __hip_atomic_load(&P.site_cnt[site], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Orders the memory operations of a wave's lanes around it.
// A list build that overflowed the per-bead capacity (TIS_CNT_NB_OVERFLOW,
// set by the list passes) stops the run: every later kernel of the step
// sequence returns at once, so the state stays as it was when that
// rebuild's step began, and the host grows the capacity and resumes from
// that step.
__device__ inline bool run_stopped(const DevPtrs &P) {
  return __builtin_nontemporal_load(&P.counters[5]) != 0ull;
}

// The same, decided once for the whole block: in a kernel whose own blocks
// raise the flag (a list that overflows), the waves of a block that starts
// meanwhile could read it differently, and those that go on would work without
// the others' share.  Contains a barrier: every thread of the block calls it.
__device__ inline bool block_stopped(const DevPtrs &P) {
  __shared__ int stop;
  if (threadIdx.x == 0) stop = run_stopped(P) ? 1 : 0;
  __syncthreads();
  return stop != 0;
}

__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

__device__ inline bool site_in_excess(const DevPtrs &P, int site) {
  return site_count(P, site) - P.site_val[site] > 0;
}

// The hbond state the valence pass works on, in global memory: candidates q
// and sites k are numbered within the system.
struct GlobalHb {
  const DevPtrs &P;
  const DSys &s;
  __device__ bool excess(int k) const { return site_in_excess(P, s.sitoff + k); }
  __device__ bool formed(int q) const { return P.hb_inlist[s.hoff + q] && P.hb_status[s.hoff + q]; }
  __device__ int site(int q, int k) const {
    const int st = P.hb_site[6 * (s.hoff + q) + k];
    return st < 0 ? -1 : st - s.sitoff;
  }
  __device__ double ene(int q) const { return P.hb_ene[s.hoff + q]; }
  __device__ int seq(int i) const { return P.hb_seq[s.hoff + i]; }
  __device__ void set_seq(int i, int q) const { P.hb_seq[s.hoff + i] = q; }
  // lane 0: hbond q deleted
  __device__ void drop(int q) const {
    P.hb_status[s.hoff + q] = 0;
    P.hb_ene[s.hoff + q] = 0.0;
  }
  __device__ void drop_site(int k) const { atomicSub(&P.site_cnt[s.sitoff + k], 1); }
};

// Valence-limit deletion of force_dtrna_hbond15.F90:373-510 for one system,
// run by the whole wave (every lane calls it).  The scans are wave-wide:
// sites in excess are counted and the pick-th one found by ballots over
// chunks of 64 sites, and the listed, formed hbonds of the picked site are
// gathered in list order by ballots over chunks of 64 candidates into the
// system's scratch sequence (one entry per candidate, so any length fits).
// A sequence of at most 64 is moved into registers (lane i holds element i);
// a longer one is shuffled and chosen from by lane 0 in the scratch copy.
// The generator is counter-based, so a deletion's draws (the site, one per
// element for the shuffle, one per element but the first for the Metropolis
// choice) are taken by the lanes at once, lane i draw i, and the choice tests
// every remaining element against the current one together, taking the first
// that is accepted: the draws and decisions of a serial pass, so that the
// result equals the oracle's bit for bit, without a Philox evaluation and an
// exponential per element in series.  Lane 0 applies each deletion; the fence
// after it orders the next scan's reads.
template <class Hb>
__device__ inline int hbond_valence_wave(const DevPtrs &P, const DSys &s, uint64_t step, int lane, const Hb &hb) {
  const uint64_t below = (1ull << lane) - 1ull;
  int ndel = 0;
  uint32_t draw = 0;
  for (int iter = 0; iter < (1 << 20); ++iter) {
    int nex = 0;
    for (int k0 = 0; k0 < s.nsite; k0 += kTile) {
      const int k = k0 + lane;
      nex += __popcll(__ballot(k < s.nsite && hb.excess(k)));
    }
    if (nex == 0) break;
    const double u0 = uniform01(P.seed, s.key, step, 0, draw + (uint32_t)lane);
    const int pick = (int)ceil(at_lane(u0, 0) * nex) - 1;  // uniform in (0,1): 0 <= pick < nex
    int site = -1;
    for (int k0 = 0, c = 0; k0 < s.nsite; k0 += kTile) {
      const int k = k0 + lane;
      const bool ex = k < s.nsite && hb.excess(k);
      const uint64_t b = __ballot(ex);
      const int n = __popcll(b);
      if (pick < c + n) {
        const uint64_t w = __ballot(ex && c + __popcll(b & below) == pick);
        site = k0 + __builtin_ctzll(w);
        break;
      }
      c += n;
    }
    // hbonds of the site in list order into the scratch sequence
    int nseq = 0;
    for (int q0 = 0; q0 < s.nhb; q0 += kTile) {
      const int q = q0 + lane;
      bool m = false;
      if (q < s.nhb && hb.formed(q))
        for (int k = 0; k < 6; ++k) m = m || hb.site(q, k) == site;
      const uint64_t b = __ballot(m);
      if (m) hb.set_seq(nseq + __popcll(b & below), q);
      nseq += __popcll(b);
    }
    if (nseq == 0) break;
    wave_sync();
    int del;
    if (nseq <= kTile) {
      // draws 1 .. nseq shuffle, nseq + 1 .. 2 nseq - 1 choose
      const double u1 = 2 * nseq > kTile ? uniform01(P.seed, s.key, step, 0, draw + (uint32_t)(kTile + lane)) : 0.0;
      int myh = lane < nseq ? hb.seq(lane) : -1;
      for (int i = 0; i < nseq; ++i) {
        const double rnd = i + 1 < kTile ? at_lane(u0, i + 1) : at_lane(u1, i + 1 - kTile);
        const int isw = (int)ceil(rnd * nseq) - 1;  // 0 <= isw < nseq
        const int a = __builtin_amdgcn_readlane(myh, i), c = __builtin_amdgcn_readlane(myh, isw);
        if (lane == i) myh = c;
        if (lane == isw) myh = a;
      }
      const double myene = lane < nseq ? hb.ene(myh) : 0.0;
      const int ir = nseq + lane;
      const double r0 = __shfl(u0, ir & (kTile - 1)), r1 = __shfl(u1, ir & (kTile - 1));
      const double myrnd = ir < kTile ? r0 : r1;
      int at = 0;
      for (;;) {
        const double ratio = exp((myene - at_lane(myene, at)) * s.beta_hb);
        const uint64_t b = __ballot(lane > at && lane < nseq && myrnd < ratio);
        if (b == 0) break;
        at = __builtin_ctzll(b);
      }
      del = __builtin_amdgcn_readlane(myh, at);
    } else {
      del = -1;
      if (lane == 0) {
        uint32_t d = draw + 1u;
        for (int i = 0; i < nseq; ++i) {
          const double r = uniform01(P.seed, s.key, step, 0, d++);
          const int isw = (int)ceil(r * nseq) - 1;
          const int a = hb.seq(i);
          hb.set_seq(i, hb.seq(isw));
          hb.set_seq(isw, a);
        }
        del = hb.seq(0);
        double edel = hb.ene(del);
        for (int i = 1; i < nseq; ++i) {
          const int j = hb.seq(i);
          const double ej = hb.ene(j);
          const double ratio = exp((ej - edel) * s.beta_hb);
          if (uniform01(P.seed, s.key, step, 0, d++) < ratio) { del = j; edel = ej; }
        }
      }
      del = __shfl(del, 0);
    }
    draw += 2u * (uint32_t)nseq;
    if (lane == 0) {
      hb.drop(del);
      // excess -= 1 where positive; count kept as valence + excess
      for (int k = 0; k < 6; ++k) {
        const int st = hb.site(del, k);
        if (st >= 0 && hb.excess(st)) hb.drop_site(st);
      }
    }
    ++ndel;
    wave_sync();
  }
  return ndel;
}

// One hbond of a system none of whose sites can exceed its valence: every
// listed hbond within the cutoff stays (force_dtrna_hbond15.F90:91-353 without
// the valence pass), so the hbonds of all such systems are independent lanes.
__device__ inline void hbond_lane(const DevPtrs &P, const double *X, const double *PX, int h) {
  const DSys &s = P.sys[P.hb_sys[h]];
  int st = 0;
  double e = 0.0, fo[18];
  if (P.hb_inlist[h]) st = hbond_at(P, s, X, PX, h, fo, &e);
  if (!st) for (int q = 0; q < 18; ++q) fo[q] = 0.0;
  P.hb_status[h] = (uint8_t)st;
  P.hb_ene[h] = e;
  put_slots(P, P.sb_hb, h, 6, fo);
}

// ------------------------------------------------------------------ terms pass
// One wave per system that has tertiary stacks or hbond candidates some of
// whose sites can exceed their valence: tertiary stack forces, and for the
// latter the hbond geometry of listed candidates and the valence pass.  Forces go to per-term slots gathered by k_main.  The phases of a
// system are ordered by wave-level fences: the four waves of a block serve
// four systems.

__device__ void terms_wave(const DevPtrs &P, const double *X, const double *PX, int isys, int32_t t_local) {
  const int lane = threadIdx.x & (kTile - 1), nt = kTile;
  const DSys s = P.sys[isys];
  const uint64_t step = *P.stepbase + (uint64_t)t_local + 1u - s.step_origin;
  for (int k = lane; k < s.ntst; k += nt) {
    double fo[18];
    tstack_eval(P, s, X, PX, s.toff + k, fo);
    put_slots(P, P.sb_tst, s.toff + k, 6, fo);
  }
  // no site can exceed its valence: the hbonds run as lanes of their own
  // (hbond_lane)
  if (!s.hb_excess_possible) return;
  for (int k = lane; k < s.nsite; k += nt) P.site_cnt[s.sitoff + k] = 0;
  wave_sync();
  for (int k = lane; k < s.nhb; k += nt) {
    int h = s.hoff + k;
    int st = 0;
    double e = 0.0, fo[18];
    if (P.hb_inlist[h]) st = hbond_at(P, s, X, PX, h, fo, &e);
    P.hb_status[h] = (uint8_t)st;
    P.hb_ene[h] = e;
    if (st) {
      for (int q = 0; q < 18; ++q) P.for_hb[(size_t)q * P.nhb + h] = fo[q];
      for (int q = 0; q < 6; ++q) {
        int site = P.hb_site[6 * h + q];
        if (site >= 0) atomicAdd(&P.site_cnt[site], 1);
      }
    }
  }
  wave_sync();
  int any = 0;
  for (int k = lane; k < s.nsite; k += nt)
    if (site_count(P, s.sitoff + k) - P.site_val[s.sitoff + k] > 0) any = 1;
  if (__any(any)) {
    const int nd = hbond_valence_wave(P, s, step, lane, GlobalHb{P, s});
    if (nd && lane == 0) atomicAdd(&P.counters[2], (unsigned long long)nd);
  }
  wave_sync();
  // forces of the hbonds that survive into their beads' slots
  for (int k = lane; k < s.nhb; k += nt) {
    const int h = s.hoff + k;
    double fo[18];
    const bool on = P.hb_status[h] != 0;
    for (int q = 0; q < 18; ++q) fo[q] = on ? P.for_hb[(size_t)q * P.nhb + h] : 0.0;
    put_slots(P, P.sb_hb, h, 6, fo);
  }
}

// ------------------------------------------------------------------ electrostatics
// Pair magnitude dv (force on i = -dv * (x_j - x_i)) in FP32 for the three
// forms: Debye-Hueckel (force_ele_DH.F90:100-112, clamped at DE_MAX), plain
// Coulomb (force_ele_coulomb.F90:75-79) and the Ewald real-space term
// (force_ele_coulomb_ewld.F90:128-132).
// Hardware reciprocal square root and base-2 exponential (about 1 ulp);
// d2 is a normal positive number here and exp underflows to 0 gracefully.
__device__ inline float hw_rsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ inline float hw_exp(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896341f); }

template <int FORM>
__device__ inline float ele_dv(const DSys &s, float qq, float d2, unsigned &nclamp, bool count) {
  const float rinv = hw_rsq(d2);
  if (FORM == 0) {
    const float rcd = (float)s.rcdist;
    const float d1 = d2 * rinv;
    const float dv = qq * rinv * rinv * (rinv + rcd) * hw_exp(-d1 * rcd);
    const bool cl = dv > (float)kDeMax;
    nclamp += (cl && count) ? 1u : 0u;
    return cl ? (float)kDeMax : dv;
  } else if (FORM == 1) {
    return qq * rinv * rinv * rinv;
  } else {
    const float d1 = d2 * rinv;
    return qq * (erfcf((float)s.ew_alpha * d1) * rinv + (float)s.ew_beta * hw_exp(-(float)s.ew_a2 * d2)) * rinv * rinv;
  }
}

// Staging of the J chunk of each wave's chunk pair.
struct EleLds {
  EleWave w[kWaves];
};

// Whole-wave rotation by one lane (DPP wave_rol:1): each lane receives the
// value of a neighbouring lane.  The direction is read off at run time from
// the lane ids (wave_dir), so the pair schedule below does not depend on it.
__device__ inline uint32_t wave_rot(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x134, 0xF, 0xF, false);
}
__device__ inline double wave_rot(double v) {
  const uint64_t b = __double_as_longlong(v);
  const uint64_t lo = wave_rot((uint32_t)b), hi = wave_rot((uint32_t)(b >> 32));
  return __longlong_as_double((long long)(lo | (hi << 32)));
}
// The lane's number within its wave, counted where it is needed: k_force's pair
// blocks would otherwise keep threadIdx in scratch from the kernel's start (29.3
// us on the batch of 576 systems, 28.1 without).
__device__ inline int wave_lane() { return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }
// +1 or 63 (= -1 mod 64): which neighbour's value wave_rot brings
__device__ inline int wave_dir() {
  const int lane = wave_lane();
  return __builtin_amdgcn_readfirstlane(((int)wave_rot((uint32_t)lane) - lane) & (kTile - 1));
}

// force_ele_DH.F90:68-118, force_ele_coulomb.F90:63-84 and the real-space
// loop of force_ele_coulomb_ewld.F90:118-137, by chunk pairs (I, J), I <= J, of
// a system's charges (chunks of 64).  At step k lane l pairs its charge i of
// chunk I with j = (l + dir k) mod 64 of chunk J (staged in LDS); the force on
// i accumulates in the lane, the opposite force on j in a register that
// rotates with the schedule, so after 64 steps lane l holds the sum for j = l.
// The diagonal chunk (J = I) runs k = 1..32 (k = 32 for lanes < 32 only),
// which meets every unordered pair of the chunk once.  List membership from
// the bit matrix, cutoff test in FP64, pair arithmetic in FP32, accumulation
// in FP64; periodic pairs (ele_pair_periodic) take the mirror code the list
// stored for them (v = x_j - x_i + shift, util_pbneighbor.F90:22-35).  The
// forces on chunk I go to slot 0 of the task's partial buffer, those on
// chunk J (I < J) to slot 1, and k_main sums a charge's slots in task order:
// a fixed order, so results are bitwise reproducible.
__host__ __device__ inline int64_t ele_task_index(int I, int J, int nch) {
  return (int64_t)I * (2 * nch - I + 1) / 2 + (J - I);
}

// ele_pair_unrolled, a chunk pair of a non-periodic system per wave: the J
// chunk is staged twice over in an order where lane l meets, at step k, entry
// c + k (c = l for dir = 1, 63 - l for dir = 63), so the reads of eight
// consecutive steps take immediate offsets from one address; the list bits
// are turned into the same order once (bit k of mr is the pair of step k); a
// pair that is not on gets charge product 0, so its force is exactly zero
// and adds nothing, with no branch; the DE_MAX clamps are counted per wave; the
// DH exponent takes its scale as one constant, -rcd log2(e).
// Absent charges sit far apart (kFar, charge 0; -kFar on the I side): their
// pairs stay finite and off.
constexpr double kFar = 1e15;

// Where lane l's charge of a chunk is staged (and again 64 entries on).
__device__ inline int stage_at(int lane, int dir) { return dir == 1 ? lane : kTile - 1 - lane; }

// The pairs of one chunk pair from registers (chunk I: position, charge
// product factor, list bits m64 of its row against chunk J, nj charges) and
// the staged chunk J: sums on chunk I in F, on chunk J in G (the diagonal
// chunk's are added to F).  Returns the clamps (the same on every lane).
template <int FORM>
__device__ inline uint32_t ele_pair_sums(const DSys &s, bool diag, int nj, bool valid, uint64_t m64, double xi0,
                                         double xi1, double xi2, float qiC, int dir, const EleWave *JE, double F[3],
                                         double G[3]) {
  const int lane = wave_lane();
  const int c = stage_at(lane, dir);
  const double cut2 = FORM == 0 ? s.dh_cut2 : s.cl_cut2;
  // bit k of mr: the pair of step k, j = (lane + dir k) mod 64
  uint64_t mr = __builtin_rotateright64(dir == 1 ? m64 : __builtin_bitreverse64(m64), (uint64_t)c);
  if (diag && lane >= 32) mr &= ~(1ull << 32);   // step 32 of the diagonal chunk: lanes < 32 only
  double F0 = 0.0, F1 = 0.0, F2 = 0.0, G0 = 0.0, G1 = 0.0, G2 = 0.0;
  uint32_t nclamp = 0;
  const float rcd = (float)s.rcdist, nrl = -rcd * 1.44269504088896341f;   // exp(-r rcd) = 2^(r nrl)
  // eight steps from k0; BITS false: every pair of the chunk pair is listed,
  // so only the cutoff decides (a charge beyond nq has charge 0 and adds 0)
  auto steps8 = [&](const int k0, const uint32_t b8, auto bits_t) {
    constexpr bool BITS = decltype(bits_t)::value;
    const double *px = JE->x + c + k0, *py = JE->y + c + k0, *pz = JE->z + c + k0;
    const float *pq = JE->q + c + k0;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      const double v0 = px[kk] - xi0, v1 = py[kk] - xi1, v2 = pz[kk] - xi2;
      const double d2 = v0 * v0 + v1 * v1 + v2 * v2;
      const bool on = (!BITS || ((b8 >> kk) & 1u)) && d2 <= cut2;
      float sq = pq[kk];
      asm volatile("" : "+v"(sq));   // read for every lane: a select below, not a branch
      const float qq = on ? qiC * sq : 0.0f;
      // every pair listed: an off pair is beyond the cutoff (d2 > 0)
      const float d2f = BITS && !on ? 1.0f : (float)d2;
      const float rinv = hw_rsq(d2f);
      float dv;
      if (FORM == 0) {
        const float d1 = d2f * rinv;
        dv = qq * rinv * rinv * (rinv + rcd) * __builtin_amdgcn_exp2f(d1 * nrl);
        const bool cl = dv > (float)kDeMax;
        nclamp += (uint32_t)__popcll(__ballot(cl));
        dv = cl ? (float)kDeMax : dv;
      } else {
        dv = qq * rinv * rinv * rinv;
      }
      const double dd = (double)dv;
      F0 -= dd * v0; F1 -= dd * v1; F2 -= dd * v2;
      G0 += dd * v0; G1 += dd * v1; G2 += dd * v2;
      G0 = wave_rot(G0); G1 = wave_rot(G1); G2 = wave_rot(G2);
    }
  };
  if (__any(m64 != 0)) {
    // every valid j listed for every valid lane (off-diagonal chunk pairs)
    const uint64_t vjm = nj >= kTile ? ~0ull : (1ull << nj) - 1ull;
    const bool all_listed = !diag && __all(!valid || (m64 & vjm) == vjm);
    if (all_listed) {
#pragma unroll 1
      for (int k0 = 0; k0 < kTile; k0 += 8) steps8(k0, 0u, std::false_type{});
    } else {
      const int k_begin = diag ? 1 : 0, k_end = diag ? 33 : kTile;
#pragma unroll 1
      for (int k0 = k_begin; k0 < k_end; k0 += 8) steps8(k0, (uint32_t)(mr >> k0), std::true_type{});
    }
  }
  if (diag) {
    const int src = (lane - dir * 33) & (kTile - 1);
    F0 += __shfl(G0, src); F1 += __shfl(G1, src); F2 += __shfl(G2, src);
  }
  F[0] = F0; F[1] = F1; F[2] = F2;
  G[0] = G0; G[1] = G1; G[2] = G2;
  return nclamp;
}

template <int FORM>
__device__ inline void ele_pair_unrolled(const DevPtrs &P, const DSys &s, const double *Y, int I, int J, int dir,
                                         EleWave *JE) {
  // the chunk pair is the wave's: uniform, so the step loops are scalar
  I = __builtin_amdgcn_readfirstlane(I);
  J = __builtin_amdgcn_readfirstlane(J);
  const int lane = wave_lane();
  const int c = stage_at(lane, dir);
  const int n = P.ntot;
  const int qi = I * kTile + lane;
  const bool valid = qi < s.nq;
  double xi0 = -kFar, xi1 = -kFar, xi2 = -kFar, chi = 0.0;
  if (valid) {
    const int gi = P.qbead[s.qoff + qi];
    xi0 = Y[gi]; xi1 = Y[n + gi]; xi2 = Y[2 * n + gi];
    chi = P.charge[gi];
  }
  const int jt = J * kTile;
  {
    const bool vj = jt + lane < s.nq;
    const int gj = vj ? P.qbead[s.qoff + jt + lane] : 0;
    const double x = vj ? Y[gj] : kFar, y = vj ? Y[n + gj] : kFar, z = vj ? Y[2 * n + gj] : kFar;
    const float q = vj ? (float)P.charge[gj] : 0.0f;
    JE->x[c] = x; JE->y[c] = y; JE->z[c] = z; JE->q[c] = q;
    JE->x[c + kTile] = x; JE->y[c + kTile] = y; JE->z[c + kTile] = z; JE->q[c + kTile] = q;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const float qiC = (float)(chi * s.ele_coef);
  const uint32_t *row = P.qmask + s.moff + (int64_t)(valid ? qi : 0) * s.mwords;
  uint64_t m64 = 0;
  if (valid) {
    const int wb = jt >> 5;
    m64 = row[wb];
    if (wb + 1 < s.mwords) m64 |= (uint64_t)row[wb + 1] << 32;
  }
  const bool diag = I == J;
  const int nj = s.nq - jt < kTile ? s.nq - jt : kTile;
  double F[3], G[3];
  const uint32_t nclamp = ele_pair_sums<FORM>(s, diag, nj, valid, m64, xi0, xi1, xi2, qiC, dir, JE, F, G);
  double *pp = P.pp + s.pp_off + ele_task_index(I, J, s.nqt) * (6 * kTile);
  if (!diag) {
    pp[3 * kTile + lane] = G[0]; pp[4 * kTile + lane] = G[1]; pp[5 * kTile + lane] = G[2];
  }
  pp[lane] = F[0]; pp[kTile + lane] = F[1]; pp[2 * kTile + lane] = F[2];
  if (lane == 0 && nclamp) atomicAdd(&P.counters[1], (unsigned long long)nclamp);
}

// A chunk pair of a periodic system, by a block: the four waves take a
// quarter of the steps each, and the quarters' sums, brought to one order of
// charges in LDS, are added as (q0 + q1) + (q2 + q3).  A periodic system is
// one box whose chunk pairs leave most of the chip idle, so the time is one
// wave's chain; its mirror codes, a byte load per step on that chain before,
// are loaded ahead for all of a wave's steps (packed four to a word, bit 7: the
// pair is listed).  640 charges (55 chunk pairs): the force pass took 32.8 us
// with a wave per chunk pair, 10.8 now.
template <int FORM>
__device__ inline void ele_pair_periodic(const DevPtrs &P, const DSys &s, const double *Y, int I, int J, int dir,
                                         EleLds &lds) {
  const int tid = (int)threadIdx.x, lane = tid & (kTile - 1);
  const int part = __builtin_amdgcn_readfirstlane(tid / kTile);
  const int n = P.ntot;
  EleWave &JE = lds.w[0];
  double(*red)[6][kTile] = reinterpret_cast<double(*)[6][kTile]>(&lds.w[1]);   // quarters 1-3
  static_assert(sizeof(EleWave) >= 6 * kTile * sizeof(double), "the quarters' sums do not fit");
  const int qi = I * kTile + lane, jt = J * kTile;
  const bool valid = qi < s.nq, diag = I == J;
  const int ns = diag ? 8 : 16, kb = diag ? 1 + 8 * part : 16 * part;   // this wave's steps
  uint64_t m64 = 0;
  if (valid) {
    const uint32_t *row = P.qmask + s.moff + (int64_t)qi * s.mwords;
    const int wb = jt >> 5;
    m64 = row[wb];
    if (wb + 1 < s.mwords) m64 |= (uint64_t)row[wb + 1] << 32;
  }
  uint32_t pk[4] = {0u, 0u, 0u, 0u};
  {
    const uint8_t *mrow = P.qmirror + s.mioff + (int64_t)(valid ? qi : 0) * s.nq + jt;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int k = kb + u, jl = (lane + dir * k) & (kTile - 1);
      const bool bit = ((m64 >> jl) & 1u) && u < ns && !(diag && k == 32 && lane >= 32);
      const uint32_t code = mrow[bit ? jl : 0];   // unlisted: the row's first, unused
      pk[u >> 2] |= (bit ? code | 0x80u : 0u) << (8 * (u & 3));
    }
  }
  double xi0 = 0.0, xi1 = 0.0, xi2 = 0.0, chi = 0.0;
  if (valid) {
    const int gi = P.qbead[s.qoff + qi];
    xi0 = Y[gi]; xi1 = Y[n + gi]; xi2 = Y[2 * n + gi];
    chi = P.charge[gi];
  }
  if (part == 0) {
    const bool vj = jt + lane < s.nq;
    const int gj = vj ? P.qbead[s.qoff + jt + lane] : 0;
    JE.x[lane] = vj ? Y[gj] : 0.0; JE.y[lane] = vj ? Y[n + gj] : 0.0; JE.z[lane] = vj ? Y[2 * n + gj] : 0.0;
    JE.q[lane] = vj ? (float)P.charge[gj] : 0.0f;
  }
  __syncthreads();
  const float qiC = (float)(chi * s.ele_coef);
  const double cut2 = FORM == 0 ? s.dh_cut2 : s.cl_cut2;
  double F[3] = {0.0, 0.0, 0.0}, G[3] = {0.0, 0.0, 0.0};
  unsigned nclamp = 0;
  const bool any = __any(m64 != 0);
#pragma unroll 1
  for (int k0 = 0; any && k0 < ns; k0 += 4) {
    const uint32_t w = pk[0];
    pk[0] = pk[1]; pk[1] = pk[2]; pk[2] = pk[3];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int jl = (lane + dir * (kb + k0 + u)) & (kTile - 1);
      const int code = (int)((w >> (8 * u)) & 0x7fu);
      const bool bit = (w >> (8 * u)) & 0x80u;
      const double v0 = (JE.x[jl] - xi0) + mirror_shift(s, code, 0);
      const double v1 = (JE.y[jl] - xi1) + mirror_shift(s, code, 1);
      const double v2 = (JE.z[jl] - xi2) + mirror_shift(s, code, 2);
      const double d2 = v0 * v0 + v1 * v1 + v2 * v2;
      const bool on = bit && d2 <= cut2;
      float dv = ele_dv<FORM>(s, qiC * JE.q[jl], on ? (float)d2 : 1.0f, nclamp, on);
      const double dd = on ? (double)dv : 0.0;
      F[0] -= dd * v0; F[1] -= dd * v1; F[2] -= dd * v2;
      G[0] += dd * v0; G[1] += dd * v1; G[2] += dd * v2;
      for (int d = 0; d < 3; ++d) G[d] = wave_rot(G[d]);
    }
  }
  if (nclamp) atomicAdd(&P.counters[1], (unsigned long long)nclamp);
  // lane l's G is now the sum on charge l + dir (kb + ns)
  const int turn = dir * (kb + ns);
  if (part > 0) {
    for (int d = 0; d < 3; ++d) {
      red[part - 1][d][lane] = F[d];
      red[part - 1][3 + d][(lane + turn) & (kTile - 1)] = G[d];
    }
  }
  __syncthreads();
  if (part > 0) return;
  double *pp = P.pp + s.pp_off + ele_task_index(I, J, s.nqt) * (6 * kTile);
  for (int d = 0; d < 3; ++d) {
    const double g0 = __shfl(G[d], (lane - turn) & (kTile - 1));
    const double f = (F[d] + red[0][d][lane]) + (red[1][d][lane] + red[2][d][lane]);
    const double g = (g0 + red[0][3 + d][lane]) + (red[1][3 + d][lane] + red[2][3 + d][lane]);
    if (!diag) pp[(3 + d) * kTile + lane] = g;
    pp[d * kTile + lane] = diag ? f + g : f;
  }
}

// ------------------------------------------------------------------ Ewald reciprocal space
// force_ele_coulomb_ewld.F90:62-84.  The phase k.r = 2 pi (h . r/L) is
// formed in FP64 from fractional coordinates and reduced to (-1/2, 1/2]
// turns before the FP32 sincospi, so its rounding does not grow with |h| or
// the box; structure factors and forces accumulate in FP64.
//
// The vectors are one of each pair h, -h, with twice the coefficient: the
// phase of -h is the negative, exactly, so the other half would repeat the
// same cosines and opposite sines.
//
// Pass 1: partial structure factors.  One lane per reciprocal vector of a
// 64-vector tile, over one 64-charge chunk staged in LDS (broadcast reads),
// a quarter of the chunk per wave, the quarters added as (q0 + q1) + (q2 +
// q3): bound by the sines' arithmetic, which a wave per tile and chunk left
// to a few waves and their latency.  |h| <= 10, 640 charges: 10.5 us for all
// vectors with a wave per tile and chunk, 5.4 now.
// EXACT (energy evaluation) takes sin/cos in FP64.
struct EwLds {
  double fx[kTile], fy[kTile], fz[kTile], fq[kTile];
  double red[kWaves - 1][2][kTile];
};
template <bool EXACT>
__device__ inline void ewald_sk_block(const DevPtrs &P, const double *PX, const EwTask &tk, EwLds &L) {
  auto &fx = L.fx; auto &fy = L.fy; auto &fz = L.fz; auto &fq = L.fq; auto &red = L.red;
  const DSys s = P.sys[tk.sys];
  const int lane = threadIdx.x & (kTile - 1), w = threadIdx.x / kTile, n = P.ntot;
  const int k = tk.a * kTile + lane;
  const int kg = s.ewk0 + min(k, s.nk - 1);
  const double hx = P.ewh[kg], hy = P.ewh[P.nktot + kg], hz = P.ewh[2 * P.nktot + kg];
  if (w == 0) {
    const int qi = tk.b * kTile + lane;
    if (qi < s.nq) {
      const int g = P.qbead[s.qoff + qi];
      fx[lane] = PX[g] * s.ew_invL; fy[lane] = PX[n + g] * s.ew_invL; fz[lane] = PX[2 * n + g] * s.ew_invL;
      fq[lane] = P.charge[g];
    } else {
      fx[lane] = fy[lane] = fz[lane] = 0.0; fq[lane] = 0.0;
    }
  }
  __syncthreads();
  constexpr int kPart = kTile / kWaves;
  const int j0 = w * kPart, j1 = min(j0 + kPart, s.nq - tk.b * kTile);
  double sc = 0.0, ss = 0.0;
  if (EXACT) {
    for (int j = j0; j < j1; ++j) {
      double t = hx * fx[j] + hy * fy[j] + hz * fz[j];
      t -= rint(t);
      double sn, cs;
      sincospi(2.0 * t, &sn, &cs);
      sc += fq[j] * cs;
      ss += fq[j] * sn;
    }
  } else {
#pragma unroll 4
    for (int j = j0; j < j1; ++j) {
      double t = hx * fx[j] + hy * fy[j] + hz * fz[j];
      t -= rint(t);
      float sn, cs;
      sincospif((float)(2.0 * t), &sn, &cs);
      sc += fq[j] * (double)cs;
      ss += fq[j] * (double)sn;
    }
  }
  if (w > 0) {
    red[w - 1][0][lane] = sc;
    red[w - 1][1][lane] = ss;
  }
  __syncthreads();
  if (w > 0 || k >= s.nk) return;
  double *o = P.psk + s.psk_off + 2 * ((int64_t)tk.b * s.nk + k);
  o[0] = (sc + red[0][0][lane]) + (red[1][0][lane] + red[2][0][lane]);
  o[1] = (ss + red[0][1][lane]) + (red[1][1][lane] + red[2][1][lane]);
}

// for the energies: sines in FP64 (the force pass runs its own in k_force)
__global__ __launch_bounds__(kTile * kWaves) void k_ewald_sk(DevPtrs P, const double *PX, const EwTask *tasks) {
  __shared__ EwLds lds;
  if (run_stopped(P)) return;
  ewald_sk_block<true>(P, PX, tasks[blockIdx.x], lds);
}

// The force pass, one launch with six kinds of blocks: a tile of reciprocal
// vectors over a charge chunk per block (ewald_sk_block, which only the second
// reciprocal pass reads: a launch of its own took 5.4 us), 256 hbond lanes per
// block (hbond_lane: the hbonds of systems without valence-limited sites, one
// lane each, first because each lane is a long FP64 chain), four systems'
// tertiary stacks and valence-limited hbonds per block (terms_wave, one wave
// each), an electrostatic chunk pair of a periodic system per block
// (ele_pair_periodic), four of others per block (ele_pair_unrolled, one wave
// each), then the bonded terms, 256 lanes per block (bonded_lane).  k_main
// gathers all of their outputs.
template <int PPW, int TPL, int WPE>
__global__ __launch_bounds__(kTile * kWaves) __attribute__((amdgpu_waves_per_eu(WPE)))
void k_force(DevPtrs P, const double *X, const double *PX, const int32_t *systask, int ntask,
             const EwTask *ptasks, int npt, const EwTask *xtasks, int nxt, const EwTask *ktasks, int nkt,
             BondedRange br, int32_t t_local) {
  constexpr int ppw = PPW, tpl = TPL;
  __shared__ EleLds lds;
  if (run_stopped(P)) return;
  int b = (int)blockIdx.x;
  if (b < nkt) {
    static_assert(sizeof(EwLds) <= sizeof(EleLds), "the reciprocal pass works in the pair pass's LDS");
    ewald_sk_block<false>(P, PX, ktasks[b], reinterpret_cast<EwLds &>(lds));
    return;
  }
  b -= nkt;
  const int nhdb = (br.nhd + kTile * kWaves - 1) / (kTile * kWaves);   // blocks of 256 hbond lanes
  const int npb = (npt + kWaves * ppw - 1) / (kWaves * ppw);   // blocks of 4 ppw chunk pairs
  const int ntb = (ntask + kWaves - 1) / kWaves;   // blocks of four system terms passes
  if (b < nhdb) {
    const int t = b * (kTile * kWaves) + (int)threadIdx.x;
    if (t < br.nhd) hbond_lane(P, X, PX, P.hb_dense[br.hd0 + t]);
    return;
  }
  b -= nhdb;
  if (b < ntb) {
    const int task = b * kWaves + (int)threadIdx.x / kTile;
    if (task < ntask) terms_wave(P, X, PX, systask[task], t_local);
    return;
  }
  b -= ntb;
  if (b < nxt) {
    const EwTask tk = xtasks[b];
    const DSys s = P.sys[tk.sys];
    const int dir = wave_dir();
    if (s.ele_form == 0) ele_pair_periodic<0>(P, s, PX, tk.a, tk.b, dir, lds);
    else if (s.ele_form == 1) ele_pair_periodic<1>(P, s, PX, tk.a, tk.b, dir, lds);
    else ele_pair_periodic<2>(P, s, PX, tk.a, tk.b, dir, lds);
    return;
  }
  b -= nxt;
  if (b >= npb) {
    // tpl bonded terms per lane, a grid-wide stride apart
    const int nbb = (int)gridDim.x - nkt - nhdb - ntb - nxt - npb;
    for (int i = 0; i < tpl; ++i)
      bonded_lane(P, X, PX, br, (b - npb + i * nbb) * (kTile * kWaves) + (int)threadIdx.x);
    return;
  }
  const int dir = wave_dir();
  const int w = (int)threadIdx.x / kTile;
  EleWave *JE = &lds.w[w];
  // ppw consecutive chunk pairs per wave, one after the other through the
  // wave's LDS slice
#pragma unroll 1
  for (int i = 0; i < ppw; ++i) {
    const int task = (b * kWaves + w) * ppw + i;
    if (task >= npt) return;
    if (i) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    const EwTask tk = ptasks[task];
    const DSys s = P.sys[tk.sys];
    // (an Ewald system is periodic: not among these)
    if (s.ele_form == 0) ele_pair_unrolled<0>(P, s, X, tk.a, tk.b, dir, JE);
    else ele_pair_unrolled<1>(P, s, X, tk.a, tk.b, dir, JE);
  }
}

template __global__ void k_force<1, 1, 4>(DevPtrs, const double *, const double *, const int32_t *, int, const EwTask *,
                                          int, const EwTask *, int, const EwTask *, int, BondedRange, int32_t);
template __global__ void k_force<2, 1, 4>(DevPtrs, const double *, const double *, const int32_t *, int, const EwTask *,
                                          int, const EwTask *, int, const EwTask *, int, BondedRange, int32_t);
template __global__ void k_force<1, 2, 4>(DevPtrs, const double *, const double *, const int32_t *, int, const EwTask *,
                                          int, const EwTask *, int, const EwTask *, int, BondedRange, int32_t);
template __global__ void k_force<2, 2, 4>(DevPtrs, const double *, const double *, const int32_t *, int, const EwTask *,
                                          int, const EwTask *, int, const EwTask *, int, BondedRange, int32_t);
template __global__ void k_force<1, 1, 2>(DevPtrs, const double *, const double *, const int32_t *, int, const EwTask *,
                                          int, const EwTask *, int, const EwTask *, int, BondedRange, int32_t);

// ------------------------------------------------------------------ Ewald reciprocal space, pass 2
// Forces.  A block takes a 64-charge tile and a chunk of kEwKChunk
// reciprocal vectors: it first sums the partial structure factors of its
// vectors into LDS (even charge chunks, odd ones, then both), then each wave
// sweeps an eighth of them for its lane's charge; partial forces per chunk go
// to pf (summed by k_main).  Bound as pass 1: 14.9 us for all vectors in
// chunks of 256 by four waves, 7.8 now, and k_main 11.1 -> 8.1 us with half as
// many partial forces to add.
__global__ __launch_bounds__(kEwThreads) void k_ewald_f(DevPtrs P, const double *PX, const EwTask *tasks) {
  constexpr int kW = kEwThreads / kTile, kPart = kEwKChunk / kW;
  static_assert(kEwThreads == 4 * kEwKChunk, "a thread per vector, component and half of the charge chunks");
  __shared__ double shx[kEwKChunk], shy[kEwKChunk], shz[kEwKChunk], sfc[kEwKChunk];
  __shared__ double sum[2][2][kEwKChunk];   // [half][cosine, sine][vector]
  __shared__ double red[3][kW][kTile];
  if (run_stopped(P)) return;
  const EwTask tk = tasks[blockIdx.x];
  const DSys s = P.sys[tk.sys];
  const int tid = threadIdx.x, n = P.ntot;
  const int lane = tid & (kTile - 1), w = tid / kTile;
  const int qi = tk.a * kTile + lane;
  const bool valid = qi < s.nq;
  const int g = P.qbead[s.qoff + min(qi, s.nq - 1)];
  const double x0 = PX[g] * s.ew_invL, x1 = PX[n + g] * s.ew_invL, x2 = PX[2 * n + g] * s.ew_invL;
  {
    const int v = tid & (kEwKChunk - 1), part = tid / kEwKChunk, comp = part & 1, half = part >> 1;
    const int k = tk.b * kEwKChunk + v;
    double a = 0.0, fc = 0.0, hx = 0.0, hy = 0.0, hz = 0.0;
    if (k < s.nk) {
      const double *ps = P.psk + s.psk_off + 2 * (int64_t)k + comp;
#pragma unroll 8
      for (int c = half; c < s.nqc; c += 2) a += ps[2 * (int64_t)c * s.nk];
      const int kg = s.ewk0 + k;
      if (part == 0) {
        fc = P.ewc[kg]; hx = P.ewh[kg]; hy = P.ewh[P.nktot + kg]; hz = P.ewh[2 * P.nktot + kg];
      }
    }
    sum[half][comp][v] = a;
    if (part == 0) { shx[v] = hx; shy[v] = hy; shz[v] = hz; sfc[v] = fc; }
  }
  __syncthreads();
  double f0 = 0.0, f1 = 0.0, f2 = 0.0;
  const int kb = w * kPart, ke = min(kb + kPart, s.nk - tk.b * kEwKChunk);
#pragma unroll 4
  for (int k = kb; k < ke; ++k) {
    double t = shx[k] * x0 + shy[k] * x1 + shz[k] * x2;
    t -= rint(t);
    float sn, cs;
    sincospif((float)(2.0 * t), &sn, &cs);
    const double sck = sum[0][0][k] + sum[1][0][k], ssk = sum[0][1][k] + sum[1][1][k];
    const double term = sfc[k] * ((double)sn * sck - (double)cs * ssk);
    f0 += term * shx[k]; f1 += term * shy[k]; f2 += term * shz[k];
  }
  red[0][w][lane] = f0; red[1][w][lane] = f1; red[2][w][lane] = f2;
  __syncthreads();
  if (w < 3 && valid) {
    const double scale = s.ew_fscale * P.charge[g];
    double f = red[w][0][lane];
    for (int q = 1; q < kW; ++q) f += red[w][q][lane];
    P.pf[s.pf_off + ((int64_t)tk.b * 3 + w) * s.nq + qi] = scale * f;
  }
}

// ------------------------------------------------------------------ main pass
// mode 0: store F; mode 1: Langevin step; mode 2: initial acceleration;
// mode 3: store F and predict positions from the stored v, a; mode 4: mode
// 2 or 3 per system (DSys::init_accel).
// Langevin (time_integral.F90:169-183, then the next step's position update
// :152-160): a' = F/m + c1 xi; v = c2 v + c3 (a + a'); a = a';
// x_next = x + c4 v + (dt^2/2) a.
// A bead's integrator inputs (Langevin constants, 1/m, v, a, x, wrapped x,
// displacement since the last rebuild), loaded before the barrier of k_main
// so that their latency overlaps the other wave's work.
struct BeadState { double r[4], rcm, v[3], a[3], x[3], px[3], o[3]; };

__device__ inline void load_state(const DevPtrs &P, const DSys &s, int g, const double *X, const double *PX,
                                  BeadState &b) {
  const int n = P.ntot;
  const LangClass &lc = P.lcls[s.lc0 + P.lcl[g]];
  for (int k = 0; k < 4; ++k) b.r[k] = lc.r[k];
  b.rcm = lc.rcm;
  for (int d = 0; d < 3; ++d) {
    b.v[d] = P.v[d * n + g];
    b.a[d] = P.a[d * n + g];
    b.x[d] = X[d * n + g];
    b.px[d] = s.periodic ? PX[d * n + g] : 0.0;
    b.o[d] = P.dyn ? P.dxyz[d * n + g] : 0.0;
  }
}

// One component: force, noise, velocity and acceleration (both updated);
// returns the displacement of the next position update.
__device__ inline double langevin_update(const double r[4], double rcm, double tstep2, int mode, double F, double gs,
                                         double &v, double &a) {
#pragma clang fp contract(off)
  double af = F * rcm + r[0] * gs;
  double vv = v;
  const double a0 = a;
  if (mode == 3) af = a0;
  if (mode == 1) vv = r[1] * vv + r[2] * (a0 + af);
  v = vv;
  a = af;
  return r[3] * vv + tstep2 * af;
}

__device__ inline void integrate(const DevPtrs &P, const DSys &s, int g, const BeadState &b, const double gs[3],
                                 const double F[3], double *XN, double *PXN, float4 *XFN, int mode, double dxo[3]) {
#pragma clang fp contract(off)
  const int n = P.ntot;
  double y[3];
  for (int d = 0; d < 3; ++d) {
    double v = b.v[d], a = b.a[d];
    const double dx = langevin_update(b.r, b.rcm, P.tstep2, mode, F[d], gs[d], v, a);
    P.v[d * n + g] = v;
    P.a[d * n + g] = a;
    dxo[d] = dx;
    y[d] = b.x[d] + dx;
    XN[d * n + g] = y[d];
    if (s.periodic) { y[d] = b.px[d] + dx; PXN[d * n + g] = y[d]; }
  }
  XFN[g] = near_pos(y[0], y[1], y[2], P.species[g]);
}

// The boxes of a tile of 64 positions (one per lane of the wave): the tile's
// box to *tile and, for bead tiles (groups != nullptr), the boxes of its four
// 16-bead groups.
__device__ inline void tile_boxes(double p0, double p1, double p2, BBox *tile, BBox *groups) {
  const int lane = threadIdx.x & (kTile - 1);
  double lo[3] = {p0, p1, p2}, hi[3] = {p0, p1, p2};
#pragma unroll
  for (int off = 1; off < kTile; off <<= 1) {
    for (int d = 0; d < 3; ++d) {
      lo[d] = fmin(lo[d], __shfl_xor(lo[d], off));
      hi[d] = fmax(hi[d], __shfl_xor(hi[d], off));
    }
    // after the offsets 1..8 each group of 16 lanes holds its group's box
    if (off == 8 && groups && (lane & 15) == 0) {
      BBox b;
      for (int d = 0; d < 3; ++d) { b.lo[d] = lo[d]; b.hi[d] = hi[d]; }
      groups[lane / 16] = b;
    }
  }
  if (lane == 0) {
    BBox b;
    for (int d = 0; d < 3; ++d) { b.lo[d] = lo[d]; b.hi[d] = hi[d]; }
    *tile = b;
  }
}

// The force on a bead is (S + Q) + ((E0 + E2) + (E1 + E3)): its bonded slots
// S in incidence order, its electrostatic sums Q (ele_sums) and its
// excluded-volume neighbours in groups of four, group k of the list in E of
// k mod 4 -- a fixed order that every pass keeps (k_main, k_window), however
// it shares the parts out, so results are bitwise reproducible.
// One neighbour within its contact distance (force_exv_dt15.F90:53-115): the
// mWCA factor (a/dr)^14 amplifies rounding 14-fold, so this formula runs in
// FP64 (only pairs within D_ij reach it).  Returns whether it was clamped.
__device__ inline bool exv_contact(double a, double dij, double coef, const double v[3], double d2, double (&F)[3]) {
  const double dist = sqrt(d2);
  const double dr = dist + a - dij;
  const double id = 1.0 / dr, ar = a * id, r2 = ar * ar, r6 = r2 * r2 * r2, r12 = r6 * r6;
  double dv = fabs(12.0 * coef * (r12 - r6) * id / dist);
  const bool cl = dv > kDeMax;
  if (cl) dv = kDeMax;
  F[0] -= dv * v[0]; F[1] -= dv * v[1]; F[2] -= dv * v[2];
  return cl;
}

// Excluded volume of one bead: the neighbour groups k mod 4 = k0 in E[0] and,
// with NE = 2, k mod 4 = k0 + 2 in E[1].
// Bound: the gathers.  Two or three of a hundred listed pairs are in contact
// (the list radius is 11.2 A for a contact distance of 3.2 A), so the list is
// sifted in FP32 first: one 16-byte load per neighbour (position and species),
// eight in flight with the next eight list entries behind them, and the pairs
// that may touch go to a queue of the lane in LDS.  The queue's pairs are
// evaluated in FP64, two at a time: as many rounds as the fullest queue of the
// wave needs, where evaluating in list order took a round for almost every
// entry, some lane of 64 being in contact in it.  Each lane keeps its list
// order, so the sums keep their bits.
constexpr int kNearQueue = 16;
// a wave's queue: list entries and species (LDS: k_main runs four waves per
// SIMD up to 20 KB a block)
struct NearQueue { uint32_t e[kNearQueue * kTile]; uint8_t sp[kNearQueue * kTile]; };

template <int NE>
__device__ inline unsigned exv_bead(const DevPtrs &P, const DSys &s, const double *Y, const float4 *XF, int g, int k0,
                                    int cnt, const SpPair *tab, NearQueue &queue,
                                    double (&E)[NE][3]) {
  constexpr int kStep = NE == 2 ? 8 : 16;   // list entries from one group of the wave to the next
  const int n = P.ntot, lane = threadIdx.x & (kTile - 1);
  const float4 fi = XF[g];
  unsigned nclamp = 0;
  int nq = 0;
  uint32_t his = 0;   // bit q: queue entry q belongs to E[1]
  auto entries = [&](int m0, uint32_t (&e)[8]) {
    // entries past cnt re-read entry cnt - 1 and are skipped
#pragma unroll
    for (int u = 0; u < 8; ++u) e[u] = P.nb[(size_t)min(m0 + (u & 3) + kStep * (u >> 2), cnt - 1) * n + g];
  };
  // kFl queue entries a round: two where the chip is idle (NE = 1), one where
  // registers decide how many waves run
  constexpr int kFl = NE == 1 ? 2 : 1;
  auto flush = [&]() {
    if (__any(nq > 0)) {
      const double xi[3] = {Y[g], Y[n + g], Y[2 * n + g]};
      for (int q = 0; __any(q < nq); q += kFl) {
        if (q >= nq) continue;
        uint32_t qe[kFl];
        double y[kFl][3];
        SpPair t[kFl];
#pragma unroll
        for (int u = 0; u < kFl; ++u) {
          const int at = min(q + u, nq - 1) * kTile + lane;
          qe[u] = queue.e[at];
          const int j = (int)(qe[u] & kIdxMask);
          y[u][0] = Y[j]; y[u][1] = Y[n + j]; y[u][2] = Y[2 * n + j];
          t[u] = tab[queue.sp[at]];
        }
#pragma unroll
        for (int u = 0; u < kFl; ++u) {
          if (q + u >= nq) continue;
          double v[3] = {y[u][0] - xi[0], y[u][1] - xi[1], y[u][2] - xi[2]};
          if (s.periodic) {
            const int code = (int)(qe[u] >> kMirrorShift);
            for (int d = 0; d < 3; ++d) v[d] += mirror_shift(s, code, d);
          }
          const double d2 = dot3(v, v);
          if (d2 > t[u].dij2) continue;
          const bool cl = NE == 2 && ((his >> (q + u)) & 1u) ? exv_contact(s.exv_a, t[u].dij, t[u].coef, v, d2, E[NE - 1])
                                                     : exv_contact(s.exv_a, t[u].dij, t[u].coef, v, d2, E[0]);
          if (cl && g < (int)(qe[u] & kIdxMask)) ++nclamp;
        }
      }
    }
    nq = 0;
    his = 0;
  };
  // (the entries in flight do not live across a flush: registers)
  int m0 = 4 * k0;
  while (__any(m0 < cnt)) {
    uint32_t e[8] = {}, en[8] = {};
    if (m0 < cnt) entries(m0, e);
    do {
      if (m0 < cnt) {
        float4 f[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) f[u] = XF[e[u] & kIdxMask];
        if (m0 + 2 * kStep < cnt) entries(m0 + 2 * kStep, en);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          float v0 = f[u].x - fi.x, v1 = f[u].y - fi.y, v2 = f[u].z - fi.z;
          if (s.periodic) {
            const int code = (int)(e[u] >> kMirrorShift);
            v0 += (float)mirror_shift(s, code, 0); v1 += (float)mirror_shift(s, code, 1);
            v2 += (float)mirror_shift(s, code, 2);
          }
          const bool far = v0 * v0 + v1 * v1 + v2 * v2 > s.exv_near2;
          if (!far && m0 + (u & 3) + kStep * (u >> 2) < cnt) {
            queue.e[nq * kTile + lane] = e[u];
            queue.sp[nq * kTile + lane] = (uint8_t)__float_as_int(f[u].w);
            if (NE == 2) his |= (uint32_t)(u >> 2) << nq;
            ++nq;
          }
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) e[u] = en[u];
      }
      m0 += 2 * kStep;
    } while (__any(m0 < cnt) && !__any(nq > kNearQueue - 8));
    flush();
  }
  return nclamp;
}

// The two largest values over the wave (merge of top-2 pairs).
__device__ inline void top2_wave(double d2, double &a, double &b) {
  a = d2; b = -1.0;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double a2 = __shfl_xor(a, off), b2 = __shfl_xor(b, off);
    const double hi = fmax(a, a2), lo = fmax(fmin(a, a2), fmax(b, b2));
    a = hi; b = lo;
  }
}

// The two largest squared displacements of a bead tile since the last
// rebuild (-1 marks lanes without a bead), for the rebuild decision of the
// next step (system_trigger).
__device__ inline void tile_top2(const DevPtrs &P, int tile, double d2) {
  double a, b;
  top2_wave(d2, a, b);
  if ((threadIdx.x & (kTile - 1)) == 0) { P.ttop[2 * tile] = a; P.ttop[2 * tile + 1] = b; }
}

// dxyz_mp of time_integral.F90:160: |dxyz|^2 before the update (as
// :64 computes it), then dxyz += dx; the update is kept for a rebuild.
__device__ inline double accumulate_displacement(const DevPtrs &P, int g, const double o[3], const double dx[3]) {
#pragma clang fp contract(off)
  const int n = P.ntot;
  const double o0 = o[0], o1 = o[1], o2 = o[2];
  const double d2 = o0 * o0 + o1 * o1 + o2 * o2;
  P.dxyz[g] = o0 + dx[0]; P.dxyz[n + g] = o1 + dx[1]; P.dxyz[2 * n + g] = o2 + dx[2];
  P.dlast[g] = dx[0]; P.dlast[n + g] = dx[1]; P.dlast[2 * n + g] = dx[2];
  return d2;
}

// Electrostatic pair sums of the force pass (the chunk-pair task slots that
// hold the charge, in task order, four tasks' loads in flight at a time),
// then the Ewald reciprocal partial forces in chunk order, added to F.
__device__ inline void ele_sums(const DevPtrs &P, const DSys &s, int g, double F[3]) {
  const int q = P.qidx[g];
  if (q < 0) return;
  const int lq = q - s.qoff, C = lq / kTile, lc = lq % kTile;
  for (int I0 = 0; I0 < s.nqt; I0 += 4) {
    double f[4][3];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int I = min(I0 + u, s.nqt - 1);
      const int a = I <= C ? I : C, bb = I <= C ? C : I;
      const int slot = I < C ? 1 : 0;
      const double *pp = P.pp + s.pp_off + ele_task_index(a, bb, s.nqt) * (6 * kTile) + slot * 3 * kTile + lc;
      f[u][0] = pp[0]; f[u][1] = pp[kTile]; f[u][2] = pp[2 * kTile];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (I0 + u < s.nqt) { F[0] += f[u][0]; F[1] += f[u][1]; F[2] += f[u][2]; }
  }
  if (s.ele_form == 2) {
    const double *pf = P.pf + s.pf_off + lq;
#pragma unroll 4
    for (int c = 0; c < s.nkc; ++c)
      for (int d = 0; d < 3; ++d) F[d] += pf[((int64_t)c * 3 + d) * s.nq];
  }
}

// The step index of a bead's noise and valence draws in mode (after mode 4
// resolves to 2 or 3 per system).
__device__ inline int resolve_mode(const DSys &s, int mode) { return mode == 4 ? (s.init_accel ? 2 : 3) : mode; }
__device__ inline uint64_t noise_step(const DevPtrs &P, const DSys &s, int32_t t_local, int mode) {
  return *P.stepbase + (uint64_t)t_local + (mode == 2 ? 0u : 1u) - s.step_origin;
}

// A bead's force stored, then the integrator with the noise gs; returns the squared displacement since the last
// rebuild before this step's update (and accumulates the update) when
// rebuilds are displacement-triggered.
__device__ inline double main_tail(const DevPtrs &P, const DSys &s, int g, const double F[3], const BeadState &b,
                                   const double gs[3], double *XN, double *PXN, float4 *XFN, int mode) {
  const int n = P.ntot;
  P.f[g] = F[0]; P.f[n + g] = F[1]; P.f[2 * n + g] = F[2];
  if (mode == 0) return -1.0;
  double dx[3];
  integrate(P, s, g, b, gs, F, XN, PXN, XFN, resolve_mode(s, mode), dx);
  if (!P.dyn) return -1.0;
  return accumulate_displacement(P, g, b.o, dx);
}


// XW = 0: two waves share a tile of 64 beads: wave 0 sums each bead's bonded
// slots, wave 1 draws its Langevin noise and adds its electrostatic sums, and
// each takes half of the excluded-volume groups; XW = 4: those two and four
// more waves, each a quarter of the groups, for launches that leave the chip
// idle, where a tile's chain of loads sets the time.  Wave 0 integrates after
// the barrier, from state loaded before it.
// Bound: latency (incidence -> slot; list entry -> position; contact pairs),
// four waves per SIMD; then the state, records and slots it moves (107 MB).  576
// systems, 237,111 beads: 33.2 us with every listed pair evaluated in FP64,
// 26.8 sifted (19.6 without excluded volume, 21.3 without the slots).  A
// 2,000-nt chain (94 tiles): 12.0 us, 11.5 sifted by two waves, 9.5 by six;
// 10 tiles: 8.4 by two, 5.7 by six.
template <int XW>
__global__ __launch_bounds__(kTile *(2 + XW)) __attribute__((amdgpu_waves_per_eu(4))) void k_main(
    DevPtrs P, const double *X, const double *PX, const float4 *XF, double *XN, double *PXN, float4 *XFN,
    const Tile *tiles, int ntile, int32_t t_local, int mode, int do_dh, int count_step) {
  constexpr int kEw = XW ? XW : 2;   // waves with excluded-volume groups
  __shared__ double red[2][3][kTile], rex[kEw][3][kTile], gsh[3][kTile];
  __shared__ NearQueue queue[kEw];
  if (run_stopped(P)) return;
  // steps completed in the current run (the host resumes a stopped run
  // after the last of them)
  if (count_step && blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&P.counters[6], 1ull);
  const int lane = threadIdx.x & (kTile - 1), w = threadIdx.x / kTile;
  const Tile tl = tiles[blockIdx.x];
  const DSys s = P.sys[tl.sys];
  // a displacement-triggered rebuild of this step is counted here, in the
  // step's last kernel, so that a step the run resumes from counts once
  if (mode == 1 && P.dyn && tl.start == 0 && threadIdx.x == 0 && P.sys_flag[tl.sys])
    atomicAdd(&P.counters[3], 1ull);
  const int li = tl.start + lane;
  const bool valid = li < s.nmp;
  const int g = s.off + (valid ? li : 0);
  const int n = P.ntot;
  // wave 0: the bonded slots S, wave 1: the electrostatic sums Q, in F
  double F[3] = {0.0, 0.0, 0.0};
  if (valid) {
    if (w == 1) {
      // the Langevin noise of the bead (wave 0 integrates after the
      // barrier) and its electrostatic sums
      if (mode != 0) {
        const int m = resolve_mode(s, mode);
        double gs[3];
        gauss3(P.seed, s.key, noise_step(P, s, t_local, m), (uint32_t)li, gs);
        gsh[0][lane] = gs[0]; gsh[1][lane] = gs[1]; gsh[2][lane] = gs[2];
      }
      if (do_dh && s.ele_form >= 0) ele_sums(P, s, g, F);
    } else if (w == 0) {
      // bonded slots in incidence order, eight loads in flight at a time
      // (slots past ie re-read slot ie - 1 and are not added)
      // (the next eight slot indices load while these slots are read)
      const int ib = P.inc_off[g], ie = P.inc_off[g + 1];
      int32_t at[8] = {}, atn[8] = {};
      if (ib < ie) {
#pragma unroll
        for (int u = 0; u < 8; ++u) at[u] = P.inc_slot[min(ib + u, ie - 1)];
      }
      for (int k0 = ib; k0 < ie; k0 += 8) {
        float sl[8][3];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const float *q = P.fslot + 3 * (int64_t)at[u];
          sl[u][0] = q[0]; sl[u][1] = q[1]; sl[u][2] = q[2];
        }
        if (k0 + 8 < ie) {
#pragma unroll
          for (int u = 0; u < 8; ++u) atn[u] = P.inc_slot[min(k0 + 8 + u, ie - 1)];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (k0 + u < ie) { F[0] += (double)sl[u][0]; F[1] += (double)sl[u][1]; F[2] += (double)sl[u][2]; }
#pragma unroll
        for (int u = 0; u < 8; ++u) at[u] = atn[u];
      }
    }
    if (w < 2)
      for (int d = 0; d < 3; ++d) red[w][d][lane] = F[d];
    // excluded volume (force_exv_dt15.F90:53-115), owner view of each pair
    if (XW == 0 || w >= 2) {
      const int k0 = XW ? w - 2 : w;
      const double *Y = s.periodic ? PX : X;
      const SpPair *tab = P.sptab + s.sptab + (int)P.species[g] * s.nspecies;
      double E[XW ? 1 : 2][3] = {};
      const unsigned nclamp = exv_bead(P, s, Y, XF, g, k0, min(P.nb_cnt[g], P.nb_cap), tab, queue[k0], E);
      if (nclamp) atomicAdd(&P.counters[0], (unsigned long long)nclamp);
      for (int d = 0; d < 3; ++d) rex[k0][d][lane] = XW ? E[0][d] : E[0][d] + E[XW ? 0 : 1][d];
    }
  }
  BeadState bs;
  if (w == 0 && valid && mode != 0) load_state(P, s, g, X, PX, bs);
  __syncthreads();
  if (w != 0) return;
  double d2 = -1.0;   // squared displacement since the last rebuild, before this update
  if (valid) {
    const double gs[3] = {gsh[0][lane], gsh[1][lane], gsh[2][lane]};
    for (int d = 0; d < 3; ++d) {
      const double E02 = XW ? rex[0][d][lane] + rex[kEw - 2][d][lane] : rex[0][d][lane];
      const double E13 = XW ? rex[1][d][lane] + rex[kEw - 1][d][lane] : rex[1][d][lane];
      F[d] = (red[0][d][lane] + red[1][d][lane]) + (E02 + E13);
    }
    d2 = main_tail(P, s, g, F, bs, gs, XN, PXN, XFN, mode);
  }
  if (P.dyn && mode != 0) {
    const int it = s.bt0 + tl.start / kTile;
    tile_top2(P, it, d2);
    // the tile's boxes at this step's positions, which a displacement-triggered
    // rebuild before the next step builds its lists from and culls by (k_lists
    // then runs without k_prep; lanes past the last bead take the tile's first
    // bead, as bbox_tile)
    if (!s.periodic) {
      double p[3] = {0.0, 0.0, 0.0};
      if (valid) {
#pragma unroll
        for (int d = 0; d < 3; ++d) p[d] = bs.x[d];
      }
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double p0 = __shfl(p[d], 0);
        p[d] = valid ? p[d] : p0;
      }
      tile_boxes(p[0], p[1], p[2], &P.bbox[it], &P.sbox[4 * it]);
    }
  }
}

template __global__ void k_main<0>(DevPtrs, const double *, const double *, const float4 *, double *, double *,
                                   float4 *, const Tile *, int, int32_t, int, int, int);
template __global__ void k_main<4>(DevPtrs, const double *, const double *, const float4 *, double *, double *,
                                   float4 *, const Tile *, int, int32_t, int, int, int);

// ------------------------------------------------------------------ lists
// util_periodic.F90:26-36 on the current coordinates; with with_pred the
// predicted wrapped positions px + (c4 v + dt^2/2 a) are refreshed too.
__device__ inline void wrap_bead(const DevPtrs &P, const DSys &s, const double *X, double *PXc, double *PXp,
                                 float4 *XFc, float4 *XFp, int g, int with_pred) {
#pragma clang fp contract(off)
  const int n = P.ntot;
  double yc[3], yp[3] = {0.0, 0.0, 0.0};
  for (int d = 0; d < 3; ++d) {
    double pw = s.box[d], pmax = 0.5 * pw, pmin = -0.5 * pw;
    double tx = X[d * n + g];
    if (tx > pmax) tx = tx - pw * (double)((int)((tx - pmax) / pw) + 1);
    else if (tx < pmin) tx = tx + pw * (double)((int)((pmin - tx) / pw) + 1);
    yc[d] = tx;
    PXc[d * n + g] = tx;
    if (with_pred) {
      double dx = P.lcls[s.lc0 + P.lcl[g]].r[3] * P.v[d * n + g] + P.tstep2 * P.a[d * n + g];
      yp[d] = tx + dx;
      PXp[d * n + g] = yp[d];
    }
  }
  XFc[g] = near_pos(yc[0], yc[1], yc[2], P.species[g]);
  if (with_pred) XFp[g] = near_pos(yp[0], yp[1], yp[2], P.species[g]);
}

// DT15 keep rule for lo < hi (neighbor_assign.F90:481-559)
__device__ inline bool exv_keep(const DSys &s, int ulo, int uhi, int clo, int tlo, int lo, int hi) {
  if (ulo != uhi) return true;
  if (clo != 2) return true;  // ion / ligand unit
  int sep = tlo == 2 ? s.nsep[0] : (tlo == 4 ? s.nsep[1] : (tlo == 3 ? s.nsep[2] : -1));
  if (sep < 0) return false;
  return hi >= lo + sep;
}

// Bounding box of bead tile or charge tile `it` (tile tl) from the
// coordinates the lists are built from (non-periodic systems only cull by
// boxes).
__device__ inline void bbox_tile(const DevPtrs &P, const DSys &s, const double *X, const Tile tl, int it,
                                 bool charge) {
  const int lane = threadIdx.x;
  const double *Y = X;
  const int n = P.ntot;
  const int li = tl.start + lane;
  const int lim = charge ? s.nq : s.nmp;
  const int first = charge ? P.qbead[s.qoff + tl.start] : s.off + tl.start;
  int g = first;
  if (li < lim) g = charge ? P.qbead[s.qoff + li] : s.off + li;
  tile_boxes(Y[g], Y[n + g], Y[2 * n + g], charge ? &P.qbbox[it] : &P.bbox[it], charge ? nullptr : &P.sbox[4 * it]);
}

// squared distance bounds between two boxes (FP64); conservative culling
// margins of 1e-9 relative cover the rounding of the per-pair test.
__device__ inline double box_dmin2(const BBox &a, const BBox &b) {
  double s2 = 0.0;
  for (int d = 0; d < 3; ++d) {
    double g = fmax(0.0, fmax(b.lo[d] - a.hi[d], a.lo[d] - b.hi[d]));
    s2 += g * g;
  }
  return s2;
}
__device__ inline double box_dmax2(const BBox &a, const BBox &b) {
  double s2 = 0.0;
  for (int d = 0; d < 3; ++d) {
    double g = fmax(fabs(b.hi[d] - a.lo[d]), fabs(a.hi[d] - b.lo[d]));
    s2 += g * g;
  }
  return s2;
}

// exv lists (neighbor_list.F90:56-87 + neighbor_assign.F90): every bead of
// the tile scans the system's bead tiles that its tile's box can reach,
// staged through LDS, with the FP64 test d^2 < (cutoff + margin)^2 rounded as
// the reference rounds it.
constexpr int kRl2Lds = 16;       // unit-pair radius tables up to 16 x 16 units are staged in LDS

__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A list block's waves share the tiles that its own tile may meet out in units
// of 32 beads (or charges).
constexpr int kUnit = 32, kUnitsRound = kTile;   // beads of a unit, units per round (one lane's box test each)

template <int W>
struct ListLds {
  double sx[W][kUnit], sy[W][kUnit], sz[W][kUnit];
  int su[W][kUnit], stc[W][kUnit];
  double rl2[kRl2Lds * kRl2Lds];
  uint32_t bits[kUnitsRound][kTile];   // [unit met][bead]: listed beads of the unit
};

// The pair vector x_hi - x_lo of the reference's lower-index-first loops
// from x_j - x_i (i: this lane's bead or charge): IEEE subtraction is
// antisymmetric, so a negation gives the bits of the reversed difference;
// non-periodic pairs need only |v|^2, which the sign does not change.
__device__ inline void pair_vec(const DSys &s, double xj0, double xj1, double xj2, const double xi[3], bool own_lo,
                                double v[3]) {
  v[0] = __dadd_rn(xj0, -xi[0]); v[1] = __dadd_rn(xj1, -xi[1]); v[2] = __dadd_rn(xj2, -xi[2]);
  if (s.periodic && !own_lo) { v[0] = -v[0]; v[1] = -v[1]; v[2] = -v[2]; }
}

// squared distance from a point to a box (FP64)
__device__ inline double point_box_d2(const double p[3], const BBox &b) {
  double s2 = 0.0;
  for (int d = 0; d < 3; ++d) {
    double g = fmax(0.0, fmax(b.lo[d] - p[d], p[d] - b.hi[d]));
    s2 += g * g;
  }
  return s2;
}

// The candidate pair (li, lj2) of a non-periodic system at squared distance
// d2, every test evaluated and combined (no branch per test): the unit-pair
// radius of neighbor_list.F90 and the exclusions of neighbor_assign.F90
// (exv_keep, by selects).  tcj: type | class << 8 of bead lj2.
template <bool ONE_UNIT>
__device__ inline bool exv_listed(const DSys &s, double d2, int li, int ui, int ti, int ci, int lj2, int uj, int tcj,
                                  const double *rl2) {
  const bool own_lo = li < lj2;
  const int ulo = own_lo ? ui : uj, uhi = own_lo ? uj : ui;
  const double r2 = ONE_UNIT ? s.rl2max : rl2[ulo * s.nunit + uhi];
  const int tlo = own_lo ? ti : (tcj & 0xFF), clo = own_lo ? ci : (tcj >> 8);
  const int lo = own_lo ? li : lj2, hi = own_lo ? lj2 : li;
  int sep = -1;
  sep = tlo == 2 ? s.nsep[0] : sep;
  sep = tlo == 4 ? s.nsep[1] : sep;
  sep = tlo == 3 ? s.nsep[2] : sep;
  const bool keep = (ulo != uhi) | (clo != 2) | ((sep >= 0) & (hi >= lo + sep));
  return (lj2 != li) & (d2 < s.rl2max) & (d2 < r2) & keep;
}

// A block per bead tile: units of 32 beads whose boxes (two of 16 beads) the
// tile can reach within the largest list radius, tested 64 at a time (one lane
// each), are dealt out to the waves; a wave stages its unit and forms, for
// each bead of the tile, a bit per listed bead of the unit.  The bits give
// each unit's first slot, so that the waves then write their entries, which
// stay in ascending order.  Bound by the latency of the staging and of the 32
// tests of a unit: with a wave per tile, which met the tiles one after the
// other, a build took 122 us for 960 compact beads, 35 us for
// the 6,000 of a long hairpin; by eight waves 23.6 and 11.8 us.
template <bool RL2_LDS, bool ONE_UNIT, int W>
__device__ inline void list_exv_tile_t(const DevPtrs &P, const DSys &s, const double *X, const Tile tl, int it,
                                       ListLds<W> &L) {
  const int lane = threadIdx.x & (kTile - 1), w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kTile);
  const int li = tl.start + lane;
  const bool valid = li < s.nmp;
  const int n = P.ntot;
  const int g = s.off + (valid ? li : 0);
  auto &sx = L.sx[w]; auto &sy = L.sy[w]; auto &sz = L.sz[w];
  auto &su = L.su[w]; auto &stc = L.stc[w];
  if (RL2_LDS && !ONE_UNIT) {
    for (int k = (int)threadIdx.x; k < s.nunit * s.nunit; k += kTile * W) L.rl2[k] = P.rl2[s.uoff + k];
    __syncthreads();
  }
  double xi[3] = {0, 0, 0};
  int ui = 0, ti = 0, ci = 0;
  if (valid) { ld3(X, n, g, xi); ui = P.unit[g]; ti = P.mptype[g]; ci = P.iclass[g]; }
  const BBox bi = P.bbox[it];
  const double cut2 = s.rl2max * (1.0 + 1e-9);
  const int nu = (s.nmp + kUnit - 1) / kUnit;
  int cnt = 0;
  for (int u0 = 0; u0 < nu; u0 += kUnitsRound) {
    const int ul = u0 + lane;
    bool reach = false;
    if (ul < nu) {
      const BBox *sb = P.sbox + 4 * s.bt0 + 2 * ul;   // (its second group may be past the last bead)
      reach = !(box_dmin2(bi, sb[0]) > cut2) || (ul * kUnit + 16 < s.nmp && !(box_dmin2(bi, sb[1]) > cut2));
    }
    const uint64_t units = __ballot(reach);   // the same in every wave
    int q = 0;
    for (uint64_t todo = units; todo; todo &= todo - 1, ++q) {
      if ((q & (W - 1)) != w) continue;
      const int unit = u0 + __builtin_ctzll(todo), jt = unit * kUnit;
      const int kend = min(kUnit, s.nmp - jt);
      if (lane < kUnit) {   // past the last bead: its copy, whose bits are dropped
        const int gj = s.off + min(jt + lane, s.nmp - 1);
        sx[lane] = X[gj]; sy[lane] = X[n + gj]; sz[lane] = X[2 * n + gj];
        su[lane] = P.unit[gj];
        stc[lane] = (int)P.mptype[gj] | ((int)P.iclass[gj] << 8);
      }
      wave_lds_sync();
      uint32_t bits = 0u;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (16 * h >= kend) continue;
        const bool need = valid && point_box_d2(xi, P.sbox[4 * s.bt0 + 2 * unit + h]) <= cut2;
        if (!__any(need)) continue;
        // every test evaluated and combined (no branch per test)
#pragma unroll
        for (int dk = 0; dk < 16; ++dk) {
          const int k = 16 * h + dk;
          const double d2 = sq3_separate(sx[k] - xi[0], sy[k] - xi[1], sz[k] - xi[2]);
          // one unit: its radius is rl2max and both beads are in it
          const bool in = exv_listed<ONE_UNIT>(s, d2, li, ui, ti, ci, jt + k, ONE_UNIT ? ui : su[k], stc[k],
                                               RL2_LDS ? L.rl2 : P.rl2 + s.uoff);
          bits |= in && k < kend ? 1u << k : 0u;
        }
      }
      wave_lds_sync();
      L.bits[q][lane] = valid ? bits : 0u;
    }
    __syncthreads();
    q = 0;
    for (uint64_t todo = units; todo; todo &= todo - 1, ++q) {
      uint32_t bits = L.bits[q][lane];
      const int c = __popc(bits);
      if ((q & (W - 1)) == w) {
        const uint32_t j0 = (uint32_t)(s.off + (u0 + __builtin_ctzll(todo)) * kUnit);
        for (int slot = cnt; bits; bits &= bits - 1u, ++slot)
          if (slot < P.nb_cap) P.nb[(size_t)slot * n + g] = j0 + (uint32_t)__builtin_ctz(bits);
      }
      cnt += c;
    }
    __syncthreads();   // the bits are read before the next round's
  }
  if (w == 0 && valid) {
    P.nb_cnt[g] = cnt;
    if (cnt > P.nb_cap) atomicMax(&P.counters[5], (unsigned long long)cnt);
  }
}

// the unit-pair radii from LDS when the table fits there (a compile-time
// choice: a run-time one makes every radius read a generic-pointer load).
// Non-periodic systems only (k_lpair builds the periodic ones).
template <int W>
__device__ inline void list_exv_tile(const DevPtrs &P, const DSys &s, const double *X, const Tile tl, int it,
                                     ListLds<W> &L) {
  if (s.nunit == 1) list_exv_tile_t<true, true, W>(P, s, X, tl, it, L);
  else if (s.nunit <= kRl2Lds) list_exv_tile_t<true, false, W>(P, s, X, tl, it, L);
  else list_exv_tile_t<false, false, W>(P, s, X, tl, it, L);
}

// ele bit matrix (neighbor_list_ele.F90:123-210): bit (qi, qj) set when the
// pair is in the list; radius (margin + cutoff)^2 per i_DH_cutoff_type.  Tile
// pairs whose boxes lie entirely inside (outside) the radius are filled with
// ones (zeros) without per-pair tests; the rest are tested pair by pair.
// A box of charge tile t (charges [64 t, 64 t + 64) of system s): the union
// of the boxes of the bead tiles that hold them (charges follow bead order).
__device__ inline BBox charge_tile_union_box(const DevPtrs &P, const DSys &s, int t) {
  const int q0 = t * kTile, q1 = min(q0 + kTile, s.nq) - 1;
  const int t0 = (P.qbead[s.qoff + q0] - s.off) / kTile, t1 = (P.qbead[s.qoff + q1] - s.off) / kTile;
  BBox b = P.bbox[s.bt0 + t0];
  for (int k = t0 + 1; k <= t1; ++k) {
    const BBox c = P.bbox[s.bt0 + k];
    for (int d = 0; d < 3; ++d) { b.lo[d] = fmin(b.lo[d], c.lo[d]); b.hi[d] = fmax(b.hi[d], c.hi[d]); }
  }
  return b;
}

// A block per charge tile, its rows' words (32 charges each) dealt out to the
// waves.
// (union_boxes: the charge tiles' boxes from the bead tiles' boxes instead of
// qbbox, which only k_prep computes; conservative, so the decisions below
// stay exact)
template <int W>
__device__ inline void list_ele_tile(const DevPtrs &P, const DSys &s, const double *X, const Tile tl, int it,
                                     ListLds<W> &L, bool union_boxes) {
  const int lane = threadIdx.x & (kTile - 1), w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kTile);
  auto &sx = L.sx[w]; auto &sy = L.sy[w]; auto &sz = L.sz[w];
  const int qi = tl.start + lane;
  const bool valid = qi < s.nq;
  const int n = P.ntot;
  double xi[3] = {0, 0, 0};
  if (valid) ld3(X, n, P.qbead[s.qoff + qi], xi);
  uint32_t *row = P.qmask + s.moff + (int64_t)(valid ? qi : 0) * s.mwords;
  const BBox bi = union_boxes ? charge_tile_union_box(P, s, tl.start / kTile) : P.qbbox[it];
  for (int j0 = 0; j0 < s.nqt; j0 += kTile) {
    // mode of the tile pairs (it, j0 + lane), decided at once: 0 none, 1 all,
    // 2 test
    int lmode = 2;
    if (j0 + lane < s.nqt) {
      const BBox bj = union_boxes ? charge_tile_union_box(P, s, j0 + lane) : P.qbbox[s.qt0 + j0 + lane];
      if (box_dmin2(bi, bj) > s.ele_rl2 * (1.0 + 1e-9)) lmode = 0;
      else if (box_dmax2(bi, bj) < s.ele_rl2 * (1.0 - 1e-9)) lmode = 1;
    }
    for (int u = 2 * j0 + w; u < min(s.mwords, 2 * (j0 + kTile)); u += W) {
      const int jt = u * kUnit, kend = min(kUnit, s.nq - jt);
      const int mode = __shfl(lmode, u / 2 - j0);
      uint32_t bits = 0u;
      if (mode == 1) {
        bits = kend >= kUnit ? 0xFFFFFFFFu : (1u << kend) - 1u;
        if (qi >= jt && qi < jt + kend) bits &= ~(1u << (qi - jt));
      } else if (mode == 2) {
        if (lane < kUnit) {   // past the last charge: its copy, whose bits are dropped
          const int gj = P.qbead[s.qoff + min(jt + lane, s.nq - 1)];
          sx[lane] = X[gj]; sy[lane] = X[n + gj]; sz[lane] = X[2 * n + gj];
        }
        wave_lds_sync();
#pragma unroll 16
        for (int k = 0; k < kUnit; ++k) {
          double v[3];
          pair_vec(s, sx[k], sy[k], sz[k], xi, qi < jt + k, v);
          const double d2 = sq3_exact(v[0], v[1], v[2]);
          bits |= d2 < s.ele_rl2 && qi != jt + k && k < kend ? 1u << k : 0u;
        }
        wave_lds_sync();
      }
      if (valid) row[u] = bits;
    }
  }
}

// hb candidate list (neighbor_list_hb.F90:59-78; radius mloop_dtrna.F90:149):
// whether the bases at (wrapped) difference v are listed
__device__ inline bool hb_listed(const DSys &s, const double v[3], double nat0) {
#pragma clang fp contract(off)
  const double d2 = sq3_exact(v[0], v[1], v[2]);
  const double r = __dadd_rn(__dadd_rn(nat0, s.hb_cut), s.margin);
  return d2 < __dmul_rn(r, r);
}
__device__ inline void list_hb_entry(const DevPtrs &P, const DSys &s, const double *X, const double *PX, int h) {
  const int n = P.ntot;
  const int a = P.hb_mp[6 * h], b = P.hb_mp[6 * h + 1];
  const double *Y = s.periodic ? PX : X;
  double v[3] = {__dadd_rn(Y[a], -Y[b]), __dadd_rn(Y[n + a], -Y[n + b]), __dadd_rn(Y[2 * n + a], -Y[2 * n + b])};
  if (s.periodic) pbneighbor(s, v);
  P.hb_inlist[h] = (uint8_t)hb_listed(s, v, P.hb_nat[6 * h]);
}

// ------------------------------------------------------------------ lists by tile pairs

// The exv and electrostatic lists of periodic systems by pairs of tiles, which
// one wave per tile (k_lists) would walk one after the other.  Pass 1, a block
// per pair: each wave tests a quarter of tile b's beads (or charges) against
// tile a's, a bit per listed one; the bits of a bead pair go to lmask, those
// of a charge pair are the list rows themselves, with the mirror codes beside
// them.  Pass 2 (k_lpair_put), a wave per bead pair: the entries of the set
// bits from the slot that the bits of the tiles before give, so the order is
// ascending whatever the split.  Bound by the latency of the tests: 793 beads
// and 640 charges took 98 us with one wave per pair, 64 tests in a row, twice
// (the entries counted first), 23.8 us now.
struct PairLds {
  double sx[kTile], sy[kTile], sz[kTile];
  int su[kTile], stc[kTile];
  double rl2[kRl2Lds * kRl2Lds];
  uint32_t bits[kWaves][kTile];
};

// beads j0 .. j1 - 1 of the staged tile at jt listed for this lane's bead, bit
// 0: j0
template <bool RL2_LDS>
__device__ inline uint32_t exv_pair_bits(const DevPtrs &P, const DSys &s, int li, const double xi[3], int ui, int ti,
                                         int ci, int jt, int j0, int j1, const PairLds &L) {
  uint32_t bits = 0u;
  for (int k = j0; k < j1; ++k) {
    const int lj2 = jt + k;
    const bool own_lo = li < lj2;
    double v[3];
    pair_vec(s, L.sx[k], L.sy[k], L.sz[k], xi, own_lo, v);
    pbneighbor(s, v);
    const double d2 = sq3_exact(v[0], v[1], v[2]);
    if (lj2 == li || !(d2 < s.rl2max)) continue;
    const int uj = L.su[k];
    const int ulo = own_lo ? ui : uj, uhi = own_lo ? uj : ui;
    const double r2 = RL2_LDS ? L.rl2[ulo * s.nunit + uhi] : P.rl2[s.uoff + ulo * s.nunit + uhi];
    if (!(d2 < r2)) continue;
    const int tj = L.stc[k] & 0xFF, cj = L.stc[k] >> 8;
    const bool keep = own_lo ? exv_keep(s, ui, uj, ci, ti, li, lj2) : exv_keep(s, uj, ui, cj, tj, lj2, li);
    if (keep) bits |= 1u << (k - j0);
  }
  return bits;
}

// gate: only the systems whose displacement trigger fires (sys_flag)
__global__ __launch_bounds__(kTile * kWaves) void k_lpair(DevPtrs P, const double *PX, const EwTask *bpairs, int nbp,
                                                          const EwTask *qpairs, int gate) {
  __shared__ PairLds L;
  if (run_stopped(P)) return;
  constexpr int kPart = kTile / kWaves;
  const int tid = (int)threadIdx.x, w = tid / kTile, lane = tid & (kTile - 1), n = P.ntot;
  const int b = (int)blockIdx.x;
  const EwTask tp = b < nbp ? bpairs[b] : qpairs[b - nbp];
  if (gate && P.sys_flag[tp.sys] == 0) return;
  const DSys s = P.sys[tp.sys];
  const int jt = tp.b * kTile;
  double xi[3] = {0, 0, 0};
  if (b < nbp) {
    const int li = tp.a * kTile + lane, g = s.off + li, kend = min(kTile, s.nmp - jt);
    const bool valid = li < s.nmp;
    const bool rl2_lds = s.nunit <= kRl2Lds;
    if (rl2_lds)
      for (int k = tid; k < s.nunit * s.nunit; k += kTile * kWaves) L.rl2[k] = P.rl2[s.uoff + k];
    if (w == 0 && lane < kend) {
      const int gj = s.off + jt + lane;
      L.sx[lane] = PX[gj]; L.sy[lane] = PX[n + gj]; L.sz[lane] = PX[2 * n + gj];
      L.su[lane] = P.unit[gj];
      L.stc[lane] = (int)P.mptype[gj] | ((int)P.iclass[gj] << 8);
    }
    int ui = 0, ti = 0, ci = 0;
    if (valid) { ld3(PX, n, g, xi); ui = P.unit[g]; ti = P.mptype[g]; ci = P.iclass[g]; }
    __syncthreads();
    const int j0 = w * kPart, j1 = min(j0 + kPart, kend);
    uint32_t bits = 0u;
    if (valid)
      bits = rl2_lds ? exv_pair_bits<true>(P, s, li, xi, ui, ti, ci, jt, j0, j1, L)
                     : exv_pair_bits<false>(P, s, li, xi, ui, ti, ci, jt, j0, j1, L);
    L.bits[w][lane] = bits;
    __syncthreads();
    if (w == 0) {
      static_assert(kWaves == 4, "four quarters of 16 bits");
      const uint32_t lo = L.bits[0][lane] | (L.bits[1][lane] << 16), hi = L.bits[2][lane] | (L.bits[3][lane] << 16);
      P.lmask[(size_t)(s.lp_off + (int64_t)tp.a * s.nbt + tp.b) * kTile + lane] = (uint64_t)lo | ((uint64_t)hi << 32);
    }
    return;
  }
  // charge pair: the bit words of tile a's rows for tile b
  const int qi = tp.a * kTile + lane, kend = min(kTile, s.nq - jt);
  const bool valid = qi < s.nq;
  if (valid) ld3(PX, n, P.qbead[s.qoff + qi], xi);
  if (w == 0 && lane < kend) {
    const int gj = P.qbead[s.qoff + jt + lane];
    L.sx[lane] = PX[gj]; L.sy[lane] = PX[n + gj]; L.sz[lane] = PX[2 * n + gj];
  }
  __syncthreads();
  uint32_t bits = 0u;
  if (valid) {
    uint8_t *mrow = P.qmirror + s.mioff + (int64_t)qi * s.nq + jt;
    const int j0 = w * kPart, j1 = min(j0 + kPart, kend);
    for (int k = j0; k < j1; ++k) {
      const bool own_lo = qi < jt + k;
      double v[3];
      pair_vec(s, L.sx[k], L.sy[k], L.sz[k], xi, own_lo, v);
      const int code = pbneighbor(s, v);
      const double d2 = sq3_exact(v[0], v[1], v[2]);
      if (qi == jt + k || !(d2 < s.ele_rl2)) continue;
      bits |= 1u << (k - j0);
      mrow[k] = (uint8_t)(own_lo ? code : mirror_flip(code));
    }
  }
  L.bits[w][lane] = bits;
  __syncthreads();
  if (w == 0 && valid) {
    uint32_t *row = P.qmask + s.moff + (int64_t)qi * s.mwords + (jt >> 5);
    row[0] = L.bits[0][lane] | (L.bits[1][lane] << 16);
    if ((jt >> 5) + 1 < s.mwords) row[1] = L.bits[2][lane] | (L.bits[3][lane] << 16);
  }
}

__global__ __launch_bounds__(kTile * kWaves) void k_lpair_put(DevPtrs P, const double *PX, const EwTask *bpairs,
                                                              int nbp, int gate) {
  __shared__ double sx[kWaves][kTile], sy[kWaves][kTile], sz[kWaves][kTile];
  if (run_stopped(P)) return;
  const int w = (int)threadIdx.x / kTile, lane = (int)threadIdx.x & (kTile - 1), n = P.ntot;
  const int p = (int)blockIdx.x * kWaves + w;
  if (p >= nbp) return;
  const EwTask bp = bpairs[p];
  if (gate && P.sys_flag[bp.sys] == 0) return;
  const DSys s = P.sys[bp.sys];
  const int li = bp.a * kTile + lane, g = s.off + li, jt = bp.b * kTile;
  const uint64_t *row = P.lmask + (size_t)(s.lp_off + (int64_t)bp.a * s.nbt) * kTile + lane;
  uint64_t mask = row[(size_t)bp.b * kTile];   // 0 in lanes past the system's beads
  int off = 0;
#pragma unroll 8
  for (int j = 0; j < bp.b; ++j) off += __popcll(row[(size_t)j * kTile]);
  if (bp.b == s.nbt - 1 && li < s.nmp) {
    const int tot = off + __popcll(mask);
    P.nb_cnt[g] = tot;
    if (tot > P.nb_cap) atomicMax(&P.counters[5], (unsigned long long)tot);
  }
  if (!__any(mask != 0)) return;
  if (jt + lane < s.nmp) {
    const int gj = s.off + jt + lane;
    sx[w][lane] = PX[gj]; sy[w][lane] = PX[n + gj]; sz[w][lane] = PX[2 * n + gj];
  }
  double xi[3] = {0, 0, 0};
  if (mask) ld3(PX, n, g, xi);
  wave_lds_sync();
  for (; mask; mask &= mask - 1, ++off) {
    const int k = __builtin_ctzll(mask);
    const bool own_lo = li < jt + k;
    double v[3];
    pair_vec(s, sx[w][k], sy[w][k], sz[w][k], xi, own_lo, v);
    const int code = pbneighbor(s, v);
    if (off < P.nb_cap)
      P.nb[(size_t)off * n + g] =
          ((uint32_t)(own_lo ? code : mirror_flip(code)) << kMirrorShift) | (uint32_t)(s.off + jt + k);
  }
}

// The list passes of one rebuild in two launches.  gate = 0 builds for every
// system of the launch range; gate = 1 only for the systems whose
// displacement trigger fires (decided in k_prep from the tile pairs the
// previous k_main wrote, recorded in sys_flag for k_lists); all other blocks
// return at once.
//
// k_prep: blocks [0, nbt) bead tiles (periodic: wrap into the box and refresh
// the predicted wrapped positions; else the tile's bounding box; with gate,
// dxyz restarts from the last step's displacement), blocks [nbt, nbt + nqt)
// charge-tile boxes.
// time_integral.F90:57-75: the two largest squared displacements of the
// system (merged over its tiles' pairs; the merge is exact in any order) and
// sqrt(m1) + sqrt(m2) > margin.
__device__ inline bool system_trigger(const DevPtrs &P, const DSys &s) {
  double a = 0.0, b = 0.0;
  for (int t = (int)threadIdx.x & (kTile - 1); t < s.nbt; t += kTile) {
    const double t1 = P.ttop[2 * (s.bt0 + t)], t2 = P.ttop[2 * (s.bt0 + t) + 1];
    const double hi = fmax(a, t1), lo = fmax(fmin(a, t1), fmax(b, t2));
    a = hi; b = lo;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double a2 = __shfl_xor(a, off), b2 = __shfl_xor(b, off);
    const double hi = fmax(a, a2), lo = fmax(fmin(a, a2), fmax(b, b2));
    a = hi; b = lo;
  }
  return sqrt(a) + sqrt(b) > s.margin;
}

// ------------------------------------------------------------------ state transfers
// A system's state between the caller's (3, n) order, in pinned host memory
// that the kernels read and write themselves, and the arena's [3][ntot]: one
// launch each way.  (Three pageable copies with a wait each took 67 us for a
// system of any size; about 12 now.)

// buf[3 i + d] = base[d][off + i]; report (may be null) gets the overflow
// flag, and n may be 0 for that alone
__global__ __launch_bounds__(256) void k_state_out(const double *base, int ntot, int off, int n, double *buf,
                                                   const unsigned long long *counters, unsigned long long *report) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k < 3 * n) buf[k] = base[(size_t)(k % 3) * ntot + off + k / 3];
  if (k == 0 && report) report[0] = counters[5];
}

// base[d][off + i] = buf[3 i + d], with the FP32 records when xf is given (the
// coordinates of a system that is not periodic)
__global__ __launch_bounds__(256) void k_state_in(DevPtrs P, double *base, int off, int n, const double *buf,
                                                  float4 *xf) {
  const int i = blockIdx.x * 256 + threadIdx.x, N = P.ntot, g = off + i;
  if (i >= n) return;
  const double x = buf[3 * i], y = buf[3 * i + 1], z = buf[3 * i + 2];
  base[g] = x; base[N + g] = y; base[2 * (size_t)N + g] = z;
  if (xf) xf[g] = near_pos(x, y, z, P.species[g]);
}

// the FP32 records of [g0, g0 + n) from x (a new layout)
__global__ __launch_bounds__(256) void k_near(DevPtrs P, const double *X, float4 *XF, int g0, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x, g = g0 + i, N = P.ntot;
  if (i < n) XF[g] = near_pos(X[g], X[N + g], X[2 * (size_t)N + g], P.species[g]);
}

// The end of a run: its stop flag and completed steps to the host; both are
// zero between calls (the host clears them itself when the run has to resume).
__global__ void k_run_report(unsigned long long *counters, unsigned long long *report) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    report[0] = counters[5];
    report[1] = counters[6];
    if (counters[5] == 0ull) counters[6] = 0ull;
  }
}

__global__ __launch_bounds__(kTile) void k_prep(DevPtrs P, const double *X, double *PXc, double *PXp, float4 *XFc,
                                                float4 *XFp, const Tile *btiles, int bt0, int nbt, const Tile *qtiles, int qt0,
                                                int nqt, int with_pred, int gate) {
  if (run_stopped(P)) return;
  const int b = (int)blockIdx.x;
  const bool charge = b >= nbt;
  const int it = charge ? qt0 + b - nbt : bt0 + b;
  const Tile tl = charge ? qtiles[it] : btiles[it];
  const DSys s = P.sys[tl.sys];
  if (gate) {
    // every block of the system reaches the same decision; the first bead
    // tile records it for k_lists and k_main (which counts the rebuild)
    const bool fire = system_trigger(P, s);
    if (!charge && tl.start == 0 && threadIdx.x == 0) P.sys_flag[tl.sys] = fire ? 1 : 0;
    if (!fire) return;
  }
  if (!charge) {
    const int li = tl.start + (int)threadIdx.x;
    if (li < s.nmp) {
      const int g = s.off + li, n = P.ntot;
      if (s.periodic) wrap_bead(P, s, X, PXc, PXp, XFc, XFp, g, with_pred);
      if (gate)
        for (int d = 0; d < 3; ++d) P.dxyz[d * n + g] = P.dlast[d * n + g];
    }
  }
  if (!s.periodic) bbox_tile(P, s, X, tl, it, charge);
}

// k_lists, W waves per block: [0, nbt) exv lists of bead tiles,
// [nbt, nbt + nqt) ele bit rows of charge tiles, then 64 W hbond candidates per
// block.
template <int W>
__global__ __launch_bounds__(kTile * W) void k_lists(DevPtrs P, const double *X, const double *PX, const Tile *btiles,
                                                 int bt0, int nbt, const Tile *qtiles, int qt0, int nqt, int h0,
                                                 int nh, int gate) {
  __shared__ ListLds<W> lds;
  if (block_stopped(P)) return;
  const int b = (int)blockIdx.x;
  if (b < nbt + nqt) {
    const bool charge = b >= nbt;
    const int it = charge ? qt0 + b - nbt : bt0 + b;
    const Tile tl = charge ? qtiles[it] : btiles[it];
    if (gate == 1 && !P.sys_flag[tl.sys]) return;
    const DSys s = P.sys[tl.sys];
    if (gate == 2) {
      // without k_prep (non-periodic batch): k_prep's decision, taken by
      // every block of the system, and its displacement reset; the bead
      // tiles' boxes are k_main's of this step's coordinates
      const bool fire = system_trigger(P, s);
      if (!charge && tl.start == 0 && threadIdx.x == 0) P.sys_flag[tl.sys] = fire ? 1 : 0;
      if (!fire) return;
      if (!charge) {
        const int li = tl.start + (int)threadIdx.x, n = P.ntot;
        if ((int)threadIdx.x < kTile && li < s.nmp)
          for (int d = 0; d < 3; ++d) P.dxyz[d * n + s.off + li] = P.dlast[d * n + s.off + li];
        // the system's hbond candidates, shared out over its bead tiles
        for (int k = tl.start * W + (int)threadIdx.x; k < s.nhb; k += s.nbt * kTile * W)
          list_hb_entry(P, s, X, PX, s.hoff + k);
      }
    }
    if (s.periodic) return;   // built by tile pairs (k_lpair)
    if (charge) list_ele_tile(P, s, X, tl, it, lds, gate == 2);
    else list_exv_tile(P, s, X, tl, it, lds);
    return;
  }
  const int k = (b - nbt - nqt) * (kTile * W) + (int)threadIdx.x;
  if (k >= nh) return;
  const int h = h0 + k;
  if (gate && !P.sys_flag[P.hb_sys[h]]) return;
  list_hb_entry(P, P.sys[P.hb_sys[h]], X, PX, h);
}

template __global__ void k_lists<kListWide>(DevPtrs, const double *, const double *, const Tile *, int, int, const Tile *, int,
                                    int, int, int, int);
template __global__ void k_lists<kListFew>(DevPtrs, const double *, const double *, const Tile *, int, int, const Tile *, int,
                                    int, int, int, int);

// ------------------------------------------------------------------ windows of steps
// Steps of small systems without leaving the workgroup: one workgroup takes
// one system through n Langevin steps with its list rebuilds, its
// coordinates, slot forces, pair sums, term parameters, incidence and
// neighbour lists in LDS (win_layout), velocities and accelerations in the
// registers of one thread per bead.
// Bound: a step of a 64-nt hairpin is some 8,000 wave instructions, most of
// them FP64, on the four SIMDs of one CU; its longest chain is the 32
// dependent pair steps of a charge chunk.  As two launches per step (k_force,
// k_main) and three per rebuild every hand-over went through L2: 17.6 us a
// step for that hairpin against 10.1 here, 64 of them 18.1 against 10.3.
// Per step: (1) the terms as tasks of one wave each, longest first, taken
// from a counter in LDS (chunk pairs of charges, 64 hbonds, 64 stacks, the
// noise of 64 beads, half the neighbour groups of 64 beads, 64 angles, 64
// bonds); (2) after a barrier, each bead's thread sums them, integrates, and
// stages the next position where the next step's tasks read it.  Systems with
// valence-limited hbonds take the hbonds first and run the valence pass (one
// wave) beside the remaining tasks.
// Every term, list and sum is that of the per-step passes, in their order, so
// results do not depend on which of them ran.
//
// back: [9][ntot], takes x, v and a of the launch's start (k_window_back).
// cu: the buffer of the current positions at *stepbase; phase: steps since
// the last fixed rebuild was due; rebuild: the interval, 0 for the
// displacement trigger.  A rebuild that overflows the list capacity raises
// TIS_CNT_NB_OVERFLOW and the system stops before that step; the others
// complete the launch, and win_at keeps how far each system came, so the
// launch can be repeated when the capacity has grown.

// The hbond state of the valence pass in LDS.
struct LocalHb {
  double *e;
  int32_t *cnt;
  const int32_t *val;
  const uint16_t *hbsite;   // 0xFFFF: none
  uint16_t *sq;
  uint8_t *stat;
  float *slot;              // the hbonds' slot forces
  __device__ bool excess(int k) const { return *(volatile int32_t *)&cnt[k] - val[k] > 0; }
  __device__ bool formed(int q) const { return *(volatile uint8_t *)&stat[q] != 0; }
  __device__ int site(int q, int k) const {
    const int st = hbsite[6 * q + k];
    return st == 0xFFFF ? -1 : st;
  }
  __device__ double ene(int q) const { return e[q]; }
  __device__ int seq(int i) const { return sq[i]; }
  __device__ void set_seq(int i, int q) const { sq[i] = (uint16_t)q; }
  __device__ void drop(int q) const {
    stat[q] = 0;
    e[q] = 0.0;
    for (int k = 0; k < 18; ++k) slot[18 * q + k] = 0.0f;
  }
  __device__ void drop_site(int k) const { *(volatile int32_t *)&cnt[k] = cnt[k] - 1; }
};

// the next task of the workgroup's counter, the same for the whole wave
__device__ inline int take_task(int *next) {
  int k = 0;
  if ((threadIdx.x & (kTile - 1)) == 0) k = atomicAdd(next, 1);
  return __builtin_amdgcn_readfirstlane(k);
}

// (I, J), I <= J, of chunk pair k of nqt chunks
__device__ inline void chunk_pair(int k, int nqt, int &I, int &J) {
  int i = 0, first = 0;
  while (k >= first + (nqt - i)) { first += nqt - i; ++i; }
  I = i;
  J = i + k - first;
}

__global__ __launch_bounds__(kWinThreads) __attribute__((amdgpu_waves_per_eu(2))) void k_window(
    DevPtrs P, const int32_t *wsys, double *back, int rows, int cu, int n, int phase, int rebuild) {
  extern __shared__ __align__(16) char lds[];
  constexpr int T = kWinThreads, W = T / kTile;
  __shared__ int next[3];
  __shared__ unsigned over;
  __shared__ double top[W][2];
  if (block_stopped(P)) return;
  const int isys = wsys[blockIdx.x];
  const DSys s = P.sys[isys];
  const uint64_t base = *P.stepbase;
  const int ce = cu ^ (n & 1);
  int from = 0, cb = cu;
  {
    const uint64_t at = P.win_at[isys];
    if ((at >> 1) > base) { from = (int)min((at >> 1) - base, (uint64_t)n); cb = (int)(at & 1); }
  }
  if (from == n && cb == ce) return;
  const WinLds L = win_layout(s, rows);
  const int tid = (int)threadIdx.x, lane = tid & (kTile - 1), w = tid / kTile, N = P.ntot, nb = s.nmp;
  float4 *xf = (float4 *)(lds + L.xf);
  double *x = (double *)(lds + L.x), *e = (double *)(lds + L.e), *gn = (double *)(lds + L.g),
         *pp = (double *)(lds + L.pp), *hene = (double *)(lds + L.ene), *rl2 = (double *)(lds + L.rl2),
         *bdp = (double *)(lds + L.bd), *bap = (double *)(lds + L.ba), *stp = (double *)(lds + L.st),
         *hbp = (double *)(lds + L.hb);
  EleWave *je = (EleWave *)(lds + L.je);
  SpPair *sptab = (SpPair *)(lds + L.sptab);
  uint64_t *mask = (uint64_t *)(lds + L.mask);
  uint32_t *seg = (uint32_t *)(lds + L.slot);
  float *qic = (float *)(lds + L.qic), *slot = (float *)(lds + L.slot);
  uint32_t *meta = (uint32_t *)(lds + L.meta);   // type | class << 8 | unit << 16
  int32_t *scnt = (int32_t *)(lds + L.cnt), *sval = (int32_t *)(lds + L.val);
  uint16_t *list = (uint16_t *)(lds + L.list), *inc = (uint16_t *)(lds + L.inc), *incoff = (uint16_t *)(lds + L.incoff),
           *nbc = (uint16_t *)(lds + L.nb), *bdm = (uint16_t *)(lds + L.bdm), *bam = (uint16_t *)(lds + L.bam),
           *stm = (uint16_t *)(lds + L.stm), *hbm = (uint16_t *)(lds + L.hbm), *hbsite = (uint16_t *)(lds + L.hbsite),
           *sq = (uint16_t *)(lds + L.seq), *qb = (uint16_t *)(lds + L.qb);
  int16_t *qidx = (int16_t *)(lds + L.qidx);
  uint8_t *spec = (uint8_t *)(lds + L.spec), *stat = (uint8_t *)(lds + L.stat), *inl = (uint8_t *)(lds + L.inl);
  const int nq = s.ele_form >= 0 ? s.nq : 0, nqt = s.ele_form >= 0 ? s.nqt : 0, np = nqt * (nqt + 1) / 2;
  const int nbt = s.nbt, nbd = s.nbd, nba = s.nba, nst = s.nst, nhb = s.nhb;
  const bool vlim = s.hb_excess_possible != 0, dyn = rebuild == 0;
  const int dir = wave_dir();
  // slot bases within the system
  const int lb_ba = 2 * nbd, lb_st = lb_ba + 3 * nba, lb_hb = lb_st + 7 * nst;
  float *hslot = slot + 3 * lb_hb;

  // ---- the system into LDS and registers
  const double *XC = P.x[cb], *XP = P.x[cb ^ 1];
  const bool own = tid < nb;
  const int g = s.off + (own ? tid : 0);
  double xc[3], v[3], a[3], ds[3] = {0.0, 0.0, 0.0}, dl[3] = {0.0, 0.0, 0.0}, lr[4], rcm;
  {
    const LangClass &lc = P.lcls[s.lc0 + P.lcl[g]];
    for (int k = 0; k < 4; ++k) lr[k] = lc.r[k];
    rcm = lc.rcm;
    for (int d = 0; d < 3; ++d) {
      xc[d] = XC[(size_t)d * N + g]; v[d] = P.v[(size_t)d * N + g]; a[d] = P.a[(size_t)d * N + g];
      if (dyn) { ds[d] = P.dxyz[(size_t)d * N + g]; dl[d] = P.dlast[(size_t)d * N + g]; }
    }
    // for k_window_back
    if (own && from == 0)
      for (int d = 0; d < 3; ++d) {
        back[(size_t)d * N + g] = xc[d];
        back[(size_t)(3 + d) * N + g] = v[d];
        back[(size_t)(6 + d) * N + g] = a[d];
      }
  }
  const int ib0 = P.inc_off[s.off];
  if (own) {
    for (int d = 0; d < 3; ++d) x[d * nb + tid] = XP[(size_t)d * N + g];
    xf[tid] = near_pos(x[tid], x[nb + tid], x[2 * nb + tid], P.species[g]);
    meta[tid] = (uint32_t)(uint8_t)P.mptype[g] | (uint32_t)(uint8_t)P.iclass[g] << 8 | (uint32_t)P.unit[g] << 16;
    incoff[tid] = (uint16_t)(P.inc_off[g] - ib0);
    qidx[tid] = (int16_t)(nq > 0 && P.qidx[g] >= 0 ? P.qidx[g] - s.qoff : -1);
    spec[tid] = P.species[g];
  }
  const int ninc = P.inc_off[s.off + nb] - ib0;
  if (tid == 0) {
    incoff[nb] = (uint16_t)ninc;
    next[0] = next[1] = next[2] = 0;
    over = 0;
  }
  for (int k = tid; k < ninc; k += T) {
    const int64_t at = P.inc_slot[ib0 + k];
    int64_t l;
    if (at >= P.sb_hb) l = at - P.sb_hb - 6 * (int64_t)s.hoff + lb_hb;
    else if (at >= P.sb_st) l = at - P.sb_st - 7 * (int64_t)s.soff + lb_st;
    else if (at >= P.sb_ba) l = at - P.sb_ba - 3 * (int64_t)s.aoff + lb_ba;
    else l = at - 2 * (int64_t)s.boff;
    inc[k] = (uint16_t)l;
  }
  for (int k = tid; k < nbd; k += T) {
    const int t = s.boff + k;
    for (int q = 0; q < 2; ++q) bdm[q * nbd + k] = (uint16_t)(P.bd_mp[2 * t + q] - s.off);
    bdp[k] = P.bd_nat[t]; bdp[nbd + k] = P.bd_coef[t];
  }
  for (int k = tid; k < nba; k += T) {
    const int t = s.aoff + k;
    for (int q = 0; q < 3; ++q) bam[q * nba + k] = (uint16_t)(P.ba_mp[3 * t + q] - s.off);
    bap[k] = P.ba_nat[t]; bap[nba + k] = P.ba_coef[t];
  }
  for (int k = tid; k < nst; k += T) {
    const int t = s.soff + k;
    for (int q = 0; q < 7; ++q) stm[q * nst + k] = (uint16_t)(P.st_mp[7 * t + q] - s.off);
    for (int q = 0; q < 3; ++q) stp[q * nst + k] = P.st_nat[3 * t + q];
    for (int q = 0; q < 4; ++q) stp[(3 + q) * nst + k] = P.st_coef[4 * t + q];
  }
  for (int k = tid; k < nhb; k += T) {
    const int t = s.hoff + k;
    for (int q = 0; q < 6; ++q) hbm[q * nhb + k] = (uint16_t)(P.hb_mp[6 * t + q] - s.off);
    for (int q = 0; q < 6; ++q) hbp[q * nhb + k] = P.hb_nat[6 * t + q];
    for (int q = 0; q < 7; ++q) hbp[(6 + q) * nhb + k] = P.hb_coef[7 * t + q];
    inl[k] = P.hb_inlist[t];
  }
  for (int k = tid; k < s.nspecies * s.nspecies; k += T) sptab[k] = P.sptab[s.sptab + k];
  for (int k = tid; k < s.nunit * s.nunit; k += T) rl2[k] = P.rl2[s.uoff + k];
  for (int k = tid; k < nqt * kTile; k += T) {
    const int c = stage_at(k % kTile, dir);
    const bool val = k < nq;
    const int gq = val ? P.qbead[s.qoff + k] : 0;
    EleWave &E = je[k / kTile];
    const double px = val ? XP[gq] : kFar, py = val ? XP[N + gq] : kFar, pz = val ? XP[2 * (size_t)N + gq] : kFar;
    const float q = val ? (float)P.charge[gq] : 0.0f;
    E.x[c] = px; E.y[c] = py; E.z[c] = pz; E.q[c] = q;
    E.x[c + kTile] = px; E.y[c + kTile] = py; E.z[c + kTile] = pz; E.q[c + kTile] = q;
    qic[k] = val ? (float)(P.charge[gq] * s.ele_coef) : 0.0f;
    if (val) qb[k] = (uint16_t)(gq - s.off);
  }
  if (vlim) {
    for (int k = tid; k < s.nsite; k += T) { scnt[k] = 0; sval[k] = P.site_val[s.sitoff + k]; }
    for (int k = tid; k < 6 * nhb; k += T) {
      const int st = P.hb_site[6 * (size_t)s.hoff + k];
      hbsite[k] = (uint16_t)(st < 0 ? 0xFFFF : st - s.sitoff);
    }
  }
  if (dyn && lane == 0) {
    top[w][0] = w < nbt ? P.ttop[2 * (s.bt0 + w)] : 0.0;
    top[w][1] = w < nbt ? P.ttop[2 * (s.bt0 + w) + 1] : 0.0;
  }
  const uint64_t step0 = base + 1u - s.step_origin;
  const LocalX lx{x, nb, 0};
  const LocalHb hb{hene, scnt, sval, hbsite, sq, stat, hslot};
  // tasks of a step, in the order they are taken; valence-limited systems
  // take the first nfirst (hbonds, stacks) before the others
  const int t_hb = (nhb + kTile - 1) / kTile, t_st = (nst + kTile - 1) / kTile;
  const int t_ba = (nba + kTile - 1) / kTile, t_bd = (nbd + kTile - 1) / kTile;
  const int nfirst = vlim ? t_hb + t_st : 0;
  const int nrest = np + (vlim ? 0 : t_hb + t_st) + 3 * nbt + t_ba + t_bd;
  unsigned clamp_exv = 0, clamp_ele = 0, ndel = 0, nfire = 0;
  __syncthreads();

  // whether the lists are rebuilt before step t: at the fixed interval, or by
  // the displacement trigger (system_trigger on the tiles' two largest)
  auto due = [&](int t) {
    if (!dyn) return (phase + t) % rebuild == 0;
    double m1 = 0.0, m2 = 0.0;
    for (int q = 0; q < nbt; ++q) {
      const double hi = fmax(m1, top[q][0]), lo = fmax(fmin(m1, top[q][0]), fmax(m2, top[q][1]));
      m1 = hi; m2 = lo;
    }
    return sqrt(m1) + sqrt(m2) > s.margin;
  };
  if (from < n && !due(from)) {
    // the lists as they stand
    if (own) {
      const int cnt = min(P.nb_cnt[g], P.nb_cap);
      nbc[tid] = (uint16_t)cnt;
    }
    __syncthreads();
    for (int k = tid; k < rows * nb; k += T) {
      const int m = k / nb, i = k % nb;
      if (m >= nbc[i]) continue;
      const int j = (int)(P.nb[(size_t)m * N + s.off + i] & kIdxMask) - s.off;
      list[k] = (uint16_t)(j | (int)spec[j] << 10);
    }
    for (int k = tid; k < np * kTile; k += T) {
      int I, J;
      chunk_pair(k / kTile, nqt, I, J);
      const int qi = I * kTile + k % kTile;
      uint64_t m = 0;
      if (qi < nq) {
        const uint32_t *row = P.qmask + s.moff + (int64_t)qi * s.mwords;
        m = row[2 * J];
        if (2 * J + 1 < s.mwords) m |= (uint64_t)row[2 * J + 1] << 32;
      }
      mask[k] = m;
    }
    __syncthreads();
  }

  int t = from;
  double xp[3] = {0.0, 0.0, 0.0};
  for (; t < n; ++t) {
    const bool last = t == n - 1;
    if (due(t)) {
      // ---- lists from the current positions (k_lists' tests; entries in
      // ascending order); to memory too when no later rebuild of this launch
      // replaces them.  Tasks of 64 beads against 32: an even share for the
      // waves where 64 against 64 left some with twice the others' (200 steps of
      // a 64-nt hairpin and its frame 2,344 -> 2,038 us; a ladder of 64 of them,
      // with its frames and exchange, 3,630 -> 3,334).
      const int nu = (nb + kUnit - 1) / kUnit;
      const bool keep = dyn || t + rebuild >= n;
      if (own)
        for (int d = 0; d < 3; ++d) { xp[d] = x[d * nb + tid]; x[d * nb + tid] = xc[d]; }
      __syncthreads();
      for (;;) {
        int k = take_task(&next[2]);
        if (k >= nqt * nqt + nbt * nu) break;
        if (k >= nqt * nqt) {
          // 64 beads against 32: the accept bits of each lane's bead
          k -= nqt * nqt;
          const int i = (k / nu) * kTile + lane, j0 = (k % nu) * kUnit, kend = min(kUnit, nb - j0);
          const int ic = i < nb ? i : 0;
          const double x0 = x[ic], x1 = x[nb + ic], x2 = x[2 * nb + ic];
          const int mi = (int)meta[ic], ui = mi >> 16, ti = mi & 0xFF, ci = (mi >> 8) & 0xFF;
          uint32_t m = 0;
          auto tests = [&](auto one) {
            constexpr bool ONE = decltype(one)::value;
#pragma unroll 8
            for (int q = 0; q < kend; ++q) {
              const int j = j0 + q, mj = (int)meta[j];
              const double d2 = sq3_separate(x[j] - x0, x[nb + j] - x1, x[2 * nb + j] - x2);
              const bool ok = exv_listed<ONE>(s, d2, i, ui, ti, ci, j, ONE ? ui : mj >> 16, mj & 0xFFFF, rl2);
              m |= (ok ? 1u : 0u) << q;
            }
          };
          if (s.nunit == 1) tests(std::true_type{});
          else tests(std::false_type{});
          if (i < nb) seg[(k % nu) * nb + i] = m;
          continue;
        }
        const int I = k / nqt, J = k % nqt, qi = I * kTile + lane, jt = J * kTile;
        if (J < I && !keep) continue;
        const int bi = qi < nq ? qb[qi] : 0, kend = min(kTile, nq - jt);
        const double xi[3] = {x[bi], x[nb + bi], x[2 * nb + bi]};
        uint64_t m = 0;
#pragma unroll 4
        for (int q = 0; q < kend; ++q) {
          const int bj = qb[jt + q];
          double dv[3];
          pair_vec(s, x[bj], x[nb + bj], x[2 * nb + bj], xi, true, dv);
          const bool ok = jt + q != qi && sq3_exact(dv[0], dv[1], dv[2]) < s.ele_rl2;
          m |= (uint64_t)(ok ? 1 : 0) << q;
        }
        if (qi >= nq) m = 0;
        if (J >= I) mask[ele_task_index(I, J, nqt) * kTile + lane] = m;
        if (keep && qi < nq) {
          uint32_t *row = P.qmask + s.moff + (int64_t)qi * s.mwords;
          row[2 * J] = (uint32_t)m;
          if (2 * J + 1 < s.mwords) row[2 * J + 1] = (uint32_t)(m >> 32);
        }
      }
      for (int k = tid; k < nhb; k += T) {
        const int b0 = hbm[k], b1 = hbm[nhb + k];
        const double dv[3] = {__dadd_rn(x[b0], -x[b1]), __dadd_rn(x[nb + b0], -x[nb + b1]),
                              __dadd_rn(x[2 * nb + b0], -x[2 * nb + b1])};
        inl[k] = (uint8_t)hb_listed(s, dv, hbp[k]);
        if (keep) P.hb_inlist[s.hoff + k] = inl[k];
      }
      __syncthreads();
      if (own)
        for (int d = 0; d < 3; ++d) x[d * nb + tid] = xp[d];
      if (tid == 0) next[2] = 0;
      for (int k = tid; k < nb * nu; k += T) {
        const int i = k % nb, sg = k / nb;
        int m = 0;
        for (int q = 0; q < sg; ++q) m += __popc(seg[q * nb + i]);
        uint32_t bits = seg[k];
        const int tot = m + __popc(bits);
        for (; bits; bits &= bits - 1u, ++m) {
          const int j = sg * kUnit + (int)__builtin_ctz(bits);
          if (m < rows) list[m * nb + i] = (uint16_t)(j | (int)spec[j] << 10);
          if ((keep || m >= rows) && m < P.nb_cap) P.nb[(size_t)m * N + s.off + i] = (uint32_t)(s.off + j);
        }
        if (sg == nu - 1) {
          nbc[i] = (uint16_t)tot;
          if (keep) P.nb_cnt[s.off + i] = tot;
          if (tot > P.nb_cap) {
            atomicMax(&over, (unsigned)tot);
            atomicMax(&P.counters[5], (unsigned long long)tot);
          }
        }
      }
      __syncthreads();
      if (over) break;   // (no thread writes it before the next rebuild)
      if (dyn) {
        ++nfire;
        for (int d = 0; d < 3; ++d) ds[d] = dl[d];
      }
    }
    // ---- the terms
    auto hb_task = [&](int q0) {
      const int q = q0 + lane;
      if (q >= nhb) return;
      const int m6[6] = {hbm[q], hbm[nhb + q], hbm[2 * nhb + q], hbm[3 * nhb + q], hbm[4 * nhb + q], hbm[5 * nhb + q]};
      double fo[18], ene = 0.0;
      int st = 0;
      if (inl[q]) {
        double nat[6], cf[7];
        for (int k = 0; k < 6; ++k) nat[k] = hbp[k * nhb + q];
        for (int k = 0; k < 7; ++k) cf[k] = hbp[(6 + k) * nhb + q];
        st = hbond_eval(s, lx, lx, m6, nat, cf, fo, &ene);
      }
      if (!st) for (int k = 0; k < 18; ++k) fo[k] = 0.0;
      for (int k = 0; k < 18; ++k) hslot[18 * q + k] = (float)fo[k];
      if (vlim) {
        stat[q] = (uint8_t)st;
        hene[q] = ene;
        if (st)
          for (int k = 0; k < 6; ++k)
            if (hbsite[6 * q + k] != 0xFFFF) atomicAdd(&scnt[hbsite[6 * q + k]], 1);
      } else if (last) {
        P.hb_status[s.hoff + q] = (uint8_t)st;
        P.hb_ene[s.hoff + q] = ene;
      }
    };
    auto st_task = [&](int k0) {
      const int k = k0 + lane;
      if (k >= nst) return;
      int m7[7];
      double nat[3], cf[4], fo[21];
      for (int q = 0; q < 7; ++q) m7[q] = stm[q * nst + k];
      for (int q = 0; q < 3; ++q) nat[q] = stp[q * nst + k];
      for (int q = 0; q < 4; ++q) cf[q] = stp[(3 + q) * nst + k];
      stack_eval(lx, m7, nat, cf, fo);
      float *o = slot + 3 * (lb_st + 7 * k);
      for (int q = 0; q < 21; ++q) o[q] = (float)fo[q];
    };
    if (vlim) {
      for (;;) {
        const int k = take_task(&next[0]);
        if (k >= nfirst) break;
        if (k < t_hb) hb_task(k * kTile);
        else st_task((k - t_hb) * kTile);
      }
      __syncthreads();
      if (w == 0) {
        bool any = false;
        for (int k = lane; k < s.nsite; k += kTile) any = any || hb.excess(k);
        if (__any(any)) ndel += (unsigned)hbond_valence_wave(P, s, step0 + (uint64_t)t, lane, hb);
        // the counts of the next step start at zero
        wave_sync();
        for (int k = lane; k < s.nsite; k += kTile) scnt[k] = 0;
        if (last)
          for (int q = lane; q < nhb; q += kTile) {
            P.hb_status[s.hoff + q] = stat[q];
            P.hb_ene[s.hoff + q] = hene[q];
          }
      }
    }
    for (;;) {
      int k = take_task(&next[1]);
      if (k >= nrest) break;
      if (k < np) {
        int I, J;
        chunk_pair(k, nqt, I, J);
        const int qi = I * kTile + lane, c = stage_at(lane, dir);
        const bool val = qi < nq;
        const double x0 = val ? je[I].x[c] : -kFar, x1 = val ? je[I].y[c] : -kFar, x2 = val ? je[I].z[c] : -kFar;
        const int nj = nq - J * kTile < kTile ? nq - J * kTile : kTile;
        double F[3], G[3];
        const uint64_t m64 = mask[k * kTile + lane];
        const uint32_t nc = s.ele_form == 0
            ? ele_pair_sums<0>(s, I == J, nj, val, m64, x0, x1, x2, qic[qi], dir, &je[J], F, G)
            : ele_pair_sums<1>(s, I == J, nj, val, m64, x0, x1, x2, qic[qi], dir, &je[J], F, G);
        double *o = pp + (size_t)k * (6 * kTile) + lane;
        for (int d = 0; d < 3; ++d) { o[d * kTile] = F[d]; o[(3 + d) * kTile] = G[d]; }
        clamp_ele += nc;
        continue;
      }
      k -= np;
      if (!vlim) {
        if (k < t_hb) { hb_task(k * kTile); continue; }
        k -= t_hb;
        if (k < t_st) { st_task(k * kTile); continue; }
        k -= t_st;
      }
      if (k < nbt) {
        const int i = k * kTile + lane;
        if (i < nb) {
          double gs[3];
          gauss3(P.seed, s.key, step0 + (uint64_t)t, (uint32_t)i, gs);
          for (int d = 0; d < 3; ++d) gn[d * nb + i] = gs[d];
        }
        continue;
      }
      k -= nbt;
      if (k < 2 * nbt) {
        // half h of the neighbour groups of 64 beads: groups k mod 4 = h and
        // h + 2, as exv_bead takes them
        const int h = k & 1, i = (k >> 1) * kTile + lane;
        if (i < nb) {
          const double xi[3] = {x[i], x[nb + i], x[2 * nb + i]};
          const float4 fi = xf[i];
          const int cnt = nbc[i], half = (cnt >> 3) * 4 + min(max((cnt & 7) - 4 * h, 0), 4);   // its entries
          const SpPair *tab = sptab + (int)spec[i] * s.nspecies;
          double E[2][3] = {};
          // entry q of the half
          auto entry = [&](int q) {
            const int m = (q >> 2) * 8 + 4 * h + (q & 3);
            if (m < rows) return (int)list[m * nb + i];
            const int j = (int)(P.nb[(size_t)m * N + s.off + i] & kIdxMask) - s.off;
            return j | (int)spec[j] << 10;
          };
          // sifted in FP32, 32 entries at a time (eight records' reads under
          // way: the cases of the list build's comment 2,361 -> 2,344 and 3,678 ->
          // 3,612 us), as in exv_bead; the pairs that may touch then in FP64
          const bool local = __all(cnt <= rows);   // no list past the rows in LDS
          for (int q0 = 0; q0 < half; q0 += 32) {
            uint32_t near = 0;
            auto sift = [&](auto at) {
              for (int q = q0; q < min(q0 + 32, half); q += 8) {
                float4 f[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) f[u] = xf[at(min(q + u, half - 1)) & 1023];
                uint32_t b = 0;
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                  const float v0 = f[u].x - fi.x, v1 = f[u].y - fi.y, v2 = f[u].z - fi.z;
                  const bool far = v0 * v0 + v1 * v1 + v2 * v2 > s.exv_near2;
                  b |= far ? 0u : 1u << u;
                }
                near |= (half - q < 8 ? b & ((1u << (half - q)) - 1u) : b) << (q - q0);
              }
            };
            if (local) sift([&](int q) { return (int)list[((q >> 2) * 8 + 4 * h + (q & 3)) * nb + i]; });
            else sift(entry);
            for (; near; near &= near - 1) {
              const int q = q0 + (int)__builtin_ctz(near), en = entry(q), j = en & 1023;
              const double v[3] = {x[j] - xi[0], x[nb + j] - xi[1], x[2 * nb + j] - xi[2]};
              const double d2 = dot3(v, v);
              const SpPair tp = tab[en >> 10];
              if (d2 > tp.dij2) continue;
              const bool cl = q & 4 ? exv_contact(s.exv_a, tp.dij, tp.coef, v, d2, E[1])
                                    : exv_contact(s.exv_a, tp.dij, tp.coef, v, d2, E[0]);
              if (cl && i < j) ++clamp_exv;
            }
          }
          for (int d = 0; d < 3; ++d) e[(3 * h + d) * nb + i] = E[0][d] + E[1][d];
        }
        continue;
      }
      k -= 2 * nbt;
      if (k < t_ba) {
        const int q = k * kTile + lane;
        if (q < nba) {
          double fo[9];
          angle_eval(lx, bam[q], bam[nba + q], bam[2 * nba + q], bap[q], bap[nba + q], fo);
          float *o = slot + 3 * (lb_ba + 3 * q);
          for (int u = 0; u < 9; ++u) o[u] = (float)fo[u];
        }
        continue;
      }
      k -= t_ba;
      const int q = k * kTile + lane;
      if (q < nbd) {
        double fo[6];
        bond_eval(lx, bdm[q], bdm[nbd + q], bdp[q], bdp[nbd + q], fo);
        float *o = slot + 6 * q;
        for (int u = 0; u < 6; ++u) o[u] = (float)fo[u];
      }
    }
    __syncthreads();
    // ---- sums and integration, one thread per bead
    if (tid == 0) { next[0] = 0; next[1] = 0; }
    double d2 = -1.0;   // squared displacement since the last rebuild, before this update
    if (own) {
      double S[3] = {0.0, 0.0, 0.0}, Q[3] = {0.0, 0.0, 0.0};
      const int k1 = incoff[tid + 1];
      for (int k = incoff[tid]; k < k1; ++k) {
        const float *sl = slot + 3 * inc[k];
        S[0] += (double)sl[0]; S[1] += (double)sl[1]; S[2] += (double)sl[2];
      }
      const int q = qidx[tid];
      if (q >= 0) {
        const int C = q / kTile, lc = q % kTile;
        for (int I = 0; I < nqt; ++I) {
          const int ta = I <= C ? I : C, tb = I <= C ? C : I;
          const double *o = pp + ele_task_index(ta, tb, nqt) * (6 * kTile) + (I < C ? 3 * kTile : 0) + lc;
          Q[0] += o[0]; Q[1] += o[kTile]; Q[2] += o[2 * kTile];
        }
      }
      double dx[3];
      for (int d = 0; d < 3; ++d) {
        const double F = (S[d] + Q[d]) + (e[d * nb + tid] + e[(3 + d) * nb + tid]);
        xc[d] = x[d * nb + tid];
        dx[d] = langevin_update(lr, rcm, P.tstep2, 1, F, gn[d * nb + tid], v[d], a[d]);
        xp[d] = __dadd_rn(xc[d], dx[d]);
        x[d * nb + tid] = xp[d];
        if (last) P.f[(size_t)d * N + g] = F;
      }
      xf[tid] = near_pos(xp[0], xp[1], xp[2], spec[tid]);
      if (q >= 0) {
        EleWave &E = je[q / kTile];
        const int c = stage_at(q % kTile, dir);
        E.x[c] = xp[0]; E.y[c] = xp[1]; E.z[c] = xp[2];
        E.x[c + kTile] = xp[0]; E.y[c + kTile] = xp[1]; E.z[c + kTile] = xp[2];
      }
      if (dyn) {
#pragma clang fp contract(off)
        d2 = ds[0] * ds[0] + ds[1] * ds[1] + ds[2] * ds[2];
        for (int d = 0; d < 3; ++d) { ds[d] = ds[d] + dx[d]; dl[d] = dx[d]; }
      }
    }
    if (dyn && w < nbt) {
      double m1, m2;
      top2_wave(d2, m1, m2);
      if (lane == 0) { top[w][0] = m1; top[w][1] = m2; }
    }
    __syncthreads();
  }
  // ---- the state back: at the end of the launch, or (t < n) before the step
  // whose rebuild overflowed, in the buffers of the launch's start
  const int cw = t == n ? ce : cu;
  if (own) {
    P.xf[cw][g] = near_pos(xc[0], xc[1], xc[2], spec[tid]);
    P.xf[cw ^ 1][g] = xf[tid];
  }
  if (own)
    for (int d = 0; d < 3; ++d) {
      const size_t o = (size_t)d * N + g;
      const double nx = x[d * nb + tid];
      P.x[cw][o] = xc[d];
      P.x[cw ^ 1][o] = nx;
      P.v[o] = v[d];
      P.a[o] = a[d];
      if (dyn) { P.dxyz[o] = ds[d]; P.dlast[o] = dl[d]; }
    }
  if (dyn && w < nbt) {
    if (lane == 0) { P.ttop[2 * (s.bt0 + w)] = top[w][0]; P.ttop[2 * (s.bt0 + w) + 1] = top[w][1]; }
    double p[3];
    for (int d = 0; d < 3; ++d) { const double p0 = __shfl(xc[d], 0); p[d] = own ? xc[d] : p0; }
    tile_boxes(p[0], p[1], p[2], &P.bbox[s.bt0 + w], &P.sbox[4 * (s.bt0 + w)]);
  }
  if (clamp_exv) atomicAdd(&P.counters[0], (unsigned long long)clamp_exv);
  if (lane == 0 && clamp_ele) atomicAdd(&P.counters[1], (unsigned long long)clamp_ele);
  if (tid == 0) {
    P.win_at[isys] = (base + (uint64_t)t) << 1 | (uint64_t)cw;
    if (ndel) atomicAdd(&P.counters[2], (unsigned long long)ndel);
    if (nfire) atomicAdd(&P.counters[3], (unsigned long long)nfire);
  }
}

// The systems that a k_window launch has left ahead of *stepbase put back to
// it (positions into buffer cu), for a run that cannot be resumed.
__global__ __launch_bounds__(kWinThreads) void k_window_back(DevPtrs P, const int32_t *wsys, const double *back,
                                                             int cu) {
  const int isys = wsys[blockIdx.x], i = (int)threadIdx.x, N = P.ntot;
  const DSys &s = P.sys[isys];
  if ((P.win_at[isys] >> 1) <= *P.stepbase || i >= s.nmp) return;
  const int g = s.off + i;
  for (int d = 0; d < 3; ++d) {
    P.x[cu][(size_t)d * N + g] = back[(size_t)d * N + g];
    P.v[(size_t)d * N + g] = back[(size_t)(3 + d) * N + g];
    P.a[(size_t)d * N + g] = back[(size_t)(6 + d) * N + g];
  }
  P.xf[cu][g] = near_pos(back[g], back[(size_t)N + g], back[2 * (size_t)N + g], P.species[g]);
}

// st_status of the consecutive stacks [s0, s0 + ns) at the given
// coordinates (force_dtrna_stack_nlocal.F90:83-92 via stack_on), for output.
__global__ __launch_bounds__(256) void k_stack_status(DevPtrs P, const double *X, const double *PX, int s0, int ns,
                                                      int32_t *out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < ns) out[k] = stack_on(P, X, PX, s0 + k) ? 1 : 0;
}

// The step counter: by steps at once after a captured run of steps or a
// k_window launch, one step per eager step; with its whole-batch list
// rebuilds and its completed steps where its kernels do not count them
// (rebuilds, completed).  A stopped run does not advance it (the host reads
// it to know where to resume).
__global__ void k_advance(uint64_t *stepbase, uint64_t by, uint64_t rebuilds, uint64_t completed,
                          unsigned long long *counters) {
  if (threadIdx.x == 0 && blockIdx.x == 0 && counters[5] == 0ull) {
    *stepbase += by; counters[4] += by; counters[3] += rebuilds; counters[6] += completed;
  }
}

// ------------------------------------------------------------------ energies
// energy_sumup.F90:149-529.  A system's terms are shared out over
// energy_parts blocks (tis_dev.h), and k_energy_sum adds the blocks' sums in
// a fixed order; the split depends on the system alone, so its energies do
// not depend on what else is evaluated.
// Bound: FP64 VALU (a square root, an exponential and a division per
// electrostatic pair).  With one block per system and one thread per charge
// row the largest system set the time, each row's loads following its bit
// tests one by one.  The pairs are taken by chunk pair now: the lane's charge
// of chunk J and its row's list bits in registers, row by row through lane
// reads, so the inner loop has no load; at four waves per SIMD (the compiler's
// own 179 VGPRs left two: 146 us).  The batch call of 576 systems (237,111
// beads, its copy to the host included): 557 -> 116 us.
constexpr int kEBlock = 256;
constexpr int kNE = kEnergyTerms;  // bond angle stack tstack hbond thbond exv ele velo

// sums of the block's kNE values per thread, thread k gets sum k
__device__ inline double block_sums(const double (&e)[kNE], double (*red)[kNE]) {
  const int t = threadIdx.x, w = t / kTile;
#pragma unroll
  for (int k = 0; k < kNE; ++k) {
    double v = e[k];
#pragma unroll
    for (int off = kTile / 2; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if ((t & (kTile - 1)) == 0) red[w][k] = v;
  }
  __syncthreads();
  double r = 0.0;
  if (t < kNE)
    for (int q = 0; q < kEBlock / kTile; ++q) r += red[q][t];
  return r;
}

// Electrostatic pair energies of wave w of nw over system s: the chunk pairs
// (I <= J) in task order, 64 rows each, in nw runs of consecutive rows.  A
// pair counts once, by its lower charge (qj > qi).
// Debye-Hueckel (energy_ele_DH.F90:33-100), plain Coulomb
// (energy_ele_coulomb.F90:55-66), the Ewald real-space term
// (energy_ele_coulomb_ewld.F90:126-138).
__device__ inline double ele_energy(const DevPtrs &P, const DSys &s, const double *Y, int w, int nw, int unit_mode,
                                    int ua, int ub) {
  const int lane = threadIdx.x & (kTile - 1);
  const int n = P.ntot;
  const int64_t nrow = (int64_t)s.nqt * (s.nqt + 1) / 2 * kTile;
  const int64_t r0 = nrow * w / nw, r1 = nrow * (w + 1) / nw;
  const double cut2 = s.ele_form == 0 ? s.dh_ecut2 : s.cl_cut2;
  double e = 0.0;
  int I = 0;
  int64_t first = 0;   // chunk pairs before row I of them
  while (I + 1 < s.nqt && r0 / kTile >= first + (s.nqt - I)) { first += s.nqt - I; ++I; }
  int J = I + (int)(r0 / kTile - first);
  for (int64_t p = r0 / kTile; p * kTile < r1; ++p) {
    const int ra = (int)max((int64_t)0, r0 - p * kTile), rb = (int)min((int64_t)kTile, r1 - p * kTile);
    // lane l: charge l of chunk I with its list bits against chunk J, and
    // charge l of chunk J
    const int qi = I * kTile + lane, qj = J * kTile + lane;
    double xi[3] = {0, 0, 0}, xj[3] = {0, 0, 0}, ci = 0.0, cj = 0.0;
    uint64_t m64 = 0;
    int ui = 0, uj = 0;
    if (qi < s.nq) {
      const int g = P.qbead[s.qoff + qi];
      ld3(Y, n, g, xi);
      ci = P.charge[g];
      ui = P.unit[g];
      const uint32_t *row = P.qmask + s.moff + (int64_t)qi * s.mwords;
      m64 = row[2 * J];
      if (2 * J + 1 < s.mwords) m64 |= (uint64_t)row[2 * J + 1] << 32;
    }
    if (qj < s.nq) {
      const int g = P.qbead[s.qoff + qj];
      ld3(Y, n, g, xj);
      cj = P.charge[g];
      uj = P.unit[g];
    }
    if (I == J) m64 &= lane < kTile - 1 ? ~0ull << (lane + 1) : 0ull;
    const uint32_t mlo = (uint32_t)m64, mhi = (uint32_t)(m64 >> 32);
    for (int r = ra; r < rb; ++r) {
      const uint64_t row = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)mlo, r) |
                           (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)mhi, r) << 32;
      if (row == 0) continue;
      if (unit_mode && __builtin_amdgcn_readlane(ui, r) != ua) continue;
      bool on = (row >> lane) & 1u;
      if (unit_mode) on = on && uj == ub;
      // (every lane read stands before the branch: lane r may be off behind it)
      const double cr = at_lane(ci, r);
      double v[3] = {xj[0] - at_lane(xi[0], r), xj[1] - at_lane(xi[1], r), xj[2] - at_lane(xi[2], r)};
      if (s.periodic) {
        const int c = on ? (int)P.qmirror[s.mioff + (int64_t)(I * kTile + r) * s.nq + qj] : 26;
        for (int d = 0; d < 3; ++d) v[d] += mirror_shift(s, c, d);
      }
      const double d2 = dot3(v, v);
      if (!on || d2 > cut2) continue;
      const double d1 = sqrt(d2);
      const double cij = (cr * cj) * s.ele_coef;
      if (s.ele_form == 0) e += cij / d1 * exp(-d1 * s.rcdist);
      else if (s.ele_form == 1) e += cij * (1.0 / d1 - s.cl_rcinv);
      else e += cij * erfc(s.ew_alpha * d1) / d1;
    }
    if (++J == s.nqt) { ++I; J = I; }
  }
  return e;
}

// One block per task (system, part of its nparts): task ids[blockIdx.x], or
// t0 + blockIdx.x without ids; the sums of task k go to part[k].
// unit_mode 1: block (x, y) is part x of gridDim.x of the system of task t0
// and sums only the terms whose unit pair, taken as energy_sumup.F90's terms
// take it, is (y mod nunit, y / nunit): raw energy_unit entries (the Ewald
// terms add none, as in energy_ele_coulomb_ewld.F90:168-170); their sums go to
// part[y gridDim.x + x].
__global__ __launch_bounds__(kEBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_energy(DevPtrs P, const double *X, const double *PX,
                                                    const EwTask *tasks, const int32_t *ids, int t0, double *part,
                                                    int unit_mode) {
  __shared__ double red[kEBlock / kTile][kNE];
  const int task = ids ? ids[blockIdx.x] : t0 + (unit_mode ? 0 : (int)blockIdx.x);
  const EwTask tk = tasks[task];
  const DSys s = P.sys[tk.sys];
  const int tp = unit_mode ? (int)blockIdx.x : tk.a, np = unit_mode ? (int)gridDim.x : tk.b;
  const int t = tp * kEBlock + (int)threadIdx.x, nt = np * kEBlock;   // this thread of the system's
  const int n = P.ntot;
  const int ua = unit_mode ? (int)blockIdx.y % s.nunit : 0, ub = unit_mode ? (int)blockIdx.y / s.nunit : 0;
  auto take = [&](int gi, int gj) { return !unit_mode || (P.unit[gi] == ua && P.unit[gj] == ub); };
  double e[kNE];
  for (int k = 0; k < kNE; ++k) e[k] = 0.0;
  // bonds (energy_bond.F90:39-57)
  for (int b = s.boff + t; b < s.boff + s.nbd; b += nt) {
    if (!take(P.bd_mp[2 * b], P.bd_mp[2 * b + 1])) continue;
    double v[3];
    vsub(X, n, P.bd_mp[2 * b + 1], P.bd_mp[2 * b], v);
    double dd = sqrt(dot3(v, v)) - P.bd_nat[b];
    e[0] += P.bd_coef[b] * (dd * dd);
  }
  // angles (energy_bangle.F90:36-52)
  for (int a = s.aoff + t; a < s.aoff + s.nba; a += nt) {
    if (!take(P.ba_mp[3 * a], P.ba_mp[3 * a + 1])) continue;
    double v21[3], v32[3];
    vsub(X, n, P.ba_mp[3 * a + 1], P.ba_mp[3 * a], v21);
    vsub(X, n, P.ba_mp[3 * a + 2], P.ba_mp[3 * a + 1], v32);
    double ct = -dot3(v32, v21) / sqrt(dot3(v21, v21) * dot3(v32, v32));
    ct = ct > 1.0 ? 1.0 : (ct < -1.0 ? -1.0 : ct);
    double dba = acos(ct) - P.ba_nat[a];
    e[1] += P.ba_coef[a] * (dba * dba);
  }
  // consecutive stacks (energy_dtrna_stack.F90:85-160)
  for (int st = s.soff + t; st < s.soff + s.nst; st += nt) {
    if (!take(P.st_mp[7 * st], P.st_mp[7 * st])) continue;
    if (!stack_on(P, X, PX, st)) continue;
    const int32_t *m7 = P.st_mp + 7 * st;
    const double *nat = P.st_nat + 3 * st, *cf = P.st_coef + 4 * st;
    double v21[3], v34[3], v54[3], v56[3], v76[3], m[3], nn[3];
    vsub(X, n, m7[1], m7[0], v21); vsub(X, n, m7[2], m7[3], v34); vsub(X, n, m7[4], m7[3], v54);
    vsub(X, n, m7[4], m7[5], v56); vsub(X, n, m7[6], m7[5], v76);
    double dd = sqrt(dot3(v21, v21)) - nat[0];
    double ediv = 1.0 + cf[1] * dd * dd;
    cross3(v34, v54, m); cross3(v54, v56, nn);
    double dph = wrap_pi(atan2(dot3(v34, nn) * sqrt(dot3(v54, v54)), dot3(m, nn)) - nat[1]);
    ediv += cf[2] * dph * dph;
    cross3(v76, v56, m);
    for (int d = 0; d < 3; ++d) nn[d] = -nn[d];
    dph = wrap_pi(atan2(dot3(v76, nn) * sqrt(dot3(v56, v56)), dot3(m, nn)) - nat[2]);
    ediv += cf[3] * dph * dph;
    e[2] += cf[0] / ediv;
  }
  // tertiary stacks (energy_dtrna_stack_nlocal.F90:55-230)
  for (int k = s.toff + t; k < s.toff + s.ntst; k += nt) {
    if (!take(P.tst_mp[6 * k], P.tst_mp[6 * k + 1])) continue;
    const int32_t *m6 = P.tst_mp + 6 * k;
    const double *nat = P.tst_nat + 6 * k, *cf = P.tst_coef + 7 * k;
    const double *Y = s.periodic ? PX : X;
    double v12[3], v13[3], v53[3], v42[3], v46[3], c4212[3], c1213[3], m[3], nn[3];
    vsub(Y, n, m6[0], m6[1], v12); vsub(Y, n, m6[0], m6[2], v13); vsub(Y, n, m6[4], m6[2], v53);
    vsub(Y, n, m6[3], m6[1], v42); vsub(Y, n, m6[3], m6[5], v46);
    if (s.periodic) { pbneighbor(s, v12); pbneighbor(s, v13); pbneighbor(s, v53); pbneighbor(s, v42); pbneighbor(s, v46); }
    double a12 = sqrt(dot3(v12, v12)), dd = a12 - nat[0];
    double ediv = 1.0 + cf[1] * dd * dd;
    double a13 = sqrt(dot3(v13, v13));
    double da = acos(dot3(v13, v12) / (a13 * a12)) - nat[1];
    ediv += cf[2] * da * da;
    double a42 = sqrt(dot3(v42, v42));
    da = acos(dot3(v12, v42) / (a12 * a42)) - nat[2];
    ediv += cf[3] * da * da;
    cross3(v42, v12, c4212); cross3(v12, v13, c1213);
    double dph = wrap_pi(atan2(dot3(v42, c1213) * a12, dot3(c4212, c1213)) - nat[3]);
    ediv += cf[4] * dph * dph;
    cross3(v53, v13, m);
    for (int d = 0; d < 3; ++d) nn[d] = -c1213[d];
    dph = wrap_pi(atan2(dot3(v53, nn) * a13, dot3(m, nn)) - nat[4]);
    ediv += cf[5] * dph * dph;
    for (int d = 0; d < 3; ++d) m[d] = -c4212[d];
    cross3(v42, v46, nn);
    dph = wrap_pi(atan2(dot3(v12, nn) * a42, dot3(m, nn)) - nat[5]);
    ediv += cf[6] * dph * dph;
    e[3] += cf[0] / ediv;
  }
  // hbonds: energies of the last force evaluation (energy_dtrna_hbond15.F90:119-148)
  for (int h = s.hoff + t; h < s.hoff + s.nhb; h += nt)
    if (P.hb_inlist[h] && P.hb_status[h] && take(P.hb_mp[6 * h], P.hb_mp[6 * h + 1]))
      e[P.hb_tert[h] ? 5 : 4] += P.hb_ene[h];
  // excluded volume, each pair once by its lower bead
  // (energy_exv_dt15.F90:60-116): the entries of four neighbours, then their
  // beads, are loaded together
  {
    const double *Y = s.periodic ? PX : X;
    const double a = s.exv_a;
    for (int li = t; li < s.nmp; li += nt) {
      const int g = s.off + li;
      if (unit_mode && P.unit[g] != ua) continue;
      double xi[3];
      ld3(Y, n, g, xi);
      const int cnt = min(P.nb_cnt[g], P.nb_cap);
      const SpPair *tab = P.sptab + s.sptab + (int)P.species[g] * s.nspecies;
      for (int m0 = 0; m0 < cnt; m0 += 4) {
        uint32_t ent[4];
        double y[4][3];
        SpPair tp[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) ent[u] = P.nb[(size_t)min(m0 + u, cnt - 1) * n + g];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int j = (int)(ent[u] & kIdxMask);
          ld3(Y, n, j, y[u]);
          tp[u] = tab[P.species[j]];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int j = (int)(ent[u] & kIdxMask);
          if (m0 + u >= cnt || j < g) continue;
          double v[3] = {y[u][0] - xi[0], y[u][1] - xi[1], y[u][2] - xi[2]};
          if (s.periodic) {
            const int c = (int)(ent[u] >> kMirrorShift);
            for (int d = 0; d < 3; ++d) v[d] += mirror_shift(s, c, d);
          }
          double dist = sqrt(dot3(v, v));
          if (dist > tp[u].dij || !take(g, j)) continue;
          dist = dist + a - tp[u].dij;
          if (dist > s.exv_inf) {
            double r = a / dist, r2 = r * r, r6 = r2 * r2 * r2;
            e[6] += ((double)P.exv_eps[g] * (double)P.exv_eps[j]) * (r6 * r6 - 2.0 * r6 + 1.0);
          } else {
            e[6] += kHighEnergy;
          }
        }
      }
    }
  }
  if (s.ele_form == 0 || s.ele_form == 1 || (s.ele_form == 2 && !unit_mode))
    e[7] += ele_energy(P, s, s.periodic ? PX : X, __builtin_amdgcn_readfirstlane(t / kTile), nt / kTile, unit_mode, ua,
                       ub);
  // Ewald Fourier sum (energy_ele_coulomb_ewld.F90:70-90) from the partial
  // structure factors of the last k_ewald_sk pass, plus the self term
  if (s.ele_form == 2 && !unit_mode) {
    for (int k = t; k < s.nk; k += nt) {
      double sc = 0.0, ss = 0.0;
      for (int c = 0; c < s.nqc; ++c) {
        const double *ps = P.psk + s.psk_off + 2 * ((int64_t)c * s.nk + k);
        sc += ps[0]; ss += ps[1];
      }
      e[7] += s.ele_coef * P.ewc[s.ewk0 + k] * (sc * sc + ss * ss);
    }
    if (t == 0) e[7] += s.ew_self;
  }
  // kinetic (energy_kinetic.F90:33-44)
  for (int li = t; li < s.nmp; li += nt) {
    int g = s.off + li;
    if (!take(g, g)) continue;
    double v[3] = {P.v[g], P.v[n + g], P.v[2 * n + g]};
    e[8] += 0.5 * P.mass[g] * dot3(v, v);
  }
  const double tot = block_sums(e, red);
  const size_t slot = unit_mode ? (size_t)blockIdx.y * gridDim.x + blockIdx.x : (size_t)task;
  if ((int)threadIdx.x < kNE) part[slot * kNE + threadIdx.x] = tot;
}

// The parts of entry k (tasks [first[i], first[i + 1]) with i = pos[k], or k0
// + k without pos; unit_parts > 0: the unit_parts parts of block row
// blockIdx.y) added in a fixed order into the 25 E_TYPE slots of out[k]; TOTAL
// excludes VELO.
__global__ __launch_bounds__(kTile) void k_energy_sum(const int32_t *first, const int32_t *pos, int k0,
                                                      const double *part, double *out, int unit_parts) {
  const int i = pos ? pos[blockIdx.x] : k0 + (int)blockIdx.x, t = (int)threadIdx.x;
  const int np = unit_parts ? unit_parts : first[i + 1] - first[i];
  const double *p = part + (unit_parts ? (size_t)blockIdx.y * np : (size_t)first[i]) * kNE;
  // lane l adds parts l, l + 64, ..; then the lanes' sums
  double tot[kNE];
#pragma unroll
  for (int k = 0; k < kNE; ++k) tot[k] = 0.0;
  for (int q = t; q < np; q += kTile)
#pragma unroll
    for (int k = 0; k < kNE; ++k) tot[k] += p[(size_t)q * kNE + k];
#pragma unroll
  for (int k = 0; k < kNE; ++k)
#pragma unroll
    for (int off = kTile / 2; off > 0; off >>= 1) tot[k] += __shfl_xor(tot[k], off);
  double *o = out + ((size_t)blockIdx.x * gridDim.y + blockIdx.y) * 25;
  if (t >= 25) return;
  // E_TYPE slots of the kNE sums
  double v = 0.0;
  switch (t) {
    case 0:   // in slot order
      v = ((((((tot[0] + tot[1]) + tot[7]) + tot[2]) + tot[4]) + tot[6]) + tot[3]) + tot[5];
      break;
    case 1: v = tot[8]; break;
    case 2: v = tot[0]; break;
    case 3: v = tot[1]; break;
    case 7: v = tot[7]; break;
    case 15: v = tot[2]; break;
    case 16: v = tot[4]; break;
    case 17: v = tot[6]; break;
    case 18: v = tot[3]; break;
    case 19: v = tot[5]; break;
    default: break;
  }
  o[t] = v;
}

// ------------------------------------------------------------------ labels
// Replica exchange: system isys[k] takes the temperature-dependent
// coefficients of label lab[k] (charges, stack U0, descriptor fields and the
// Langevin noise amplitude c1 of time_integral_pre.F90:163-164, as the
// refresh of time_integral_post.F90:264-370 does) and, with vscale, has its
// velocities scaled (simu_replica_exchange.F90:272-300).  One block per
// entry; the descriptor is written after every lane has read it.
__global__ __launch_bounds__(256) void k_label_apply(DevPtrs P, LabelDev L, const int32_t *isys, const int32_t *lab,
                                                     const double *vscale) {
#pragma clang fp contract(off)
  const int k = blockIdx.x;
  const int is = isys[k], lb = lab[k];
  const DSys t = P.sys[is];
  const DSys src = L.sys[lb];
  const int n = P.ntot;
  double *charge = const_cast<double *>(P.charge);
  double *stc = const_cast<double *>(P.st_coef);
  const double f = vscale ? vscale[k] : 1.0;
  for (int q = threadIdx.x; q < t.nlc; q += blockDim.x) {
    LangClass &c = P.lcls[t.lc0 + q];
    if (P.tstep > 0.0) c.r[0] = sqrt(2.0 * c.fric * kBoltzKcalMol * src.tempk / (P.tstep * c.mass));
  }
  for (int i = threadIdx.x; i < t.nmp; i += blockDim.x) {
    const int g = t.off + i;
    charge[g] = L.q[L.qoff[lb] + i];
    if (vscale)
      for (int d = 0; d < 3; ++d) P.v[(size_t)d * n + g] *= f;
  }
  for (int q = threadIdx.x; q < t.nst; q += blockDim.x) stc[4 * (size_t)(t.soff + q)] = L.u0[L.u0off[lb] + q];
  __syncthreads();
  if (threadIdx.x == 0) {
    DSys d = t;
    copy_t_fields(d, src);
    const_cast<DSys *>(P.sys)[is] = d;
  }
}

}  // namespace tis
