// Forward dynamics of the primal rollouts (gfx950): the Go2 step of spi_dyn.h with every leg
// eliminated in closed form in its hip frame.  Same model, contact law and integrator as
// spi_dyn.h in two thirds of its instructions: a rollout lane is bound by VALU issue, so the
// algebra is what its time consists of (3,546 FLOP per sub-interval against 5,293; vector
// instructions 3,424 -> 2,222 by the counters).
//
// What the leg's structure gives (hip axis x; thigh and calf axes both y; the thigh's origin
// lies on its own axis through the hip origin O, so every y offset can be absorbed into the
// links' constants):
//   * Thigh and calf stay in planes of the hip frame: their constants are rotated about y once
//     (angles q2 and q2 + q3) and nothing else in the leg needs a rotation.
//   * Mass on a joint's axis moves the same with either neighbour, so each link's mass, axial
//     first moment and axial second moment are handed to its parent at compile time
//     (leg_constants, base_with_legs).  The links left over have no mass, h = (hx, 0, hz) and
//     no S_yy (hip: h = (0, hy, hz), no S_xx); S is the second moment, sum of m p p^T.
//   * The legs' composite inertias need no articulated recursion: a 3 x 3 elimination (calf,
//     thigh, hip) of the joint rows leaves the leg's inertia at O with an empty n_x row and an
//     n_y row of the hip link alone.
//   * Velocity products: the composite leg moves with the hip's field a(p) = a_O + A p; a spin
//     s about the y axis through a point adds (k px, 2 s (wx px + wz pz), k pz), with
//     k = -s (2 wy + s), at p from that point.  No per-link velocity or force is formed, and
//     with the base's proper acceleration dv/dt + w x v - g as the unknown, none depends on v.
// Measured on 4096 candidates x 256 segments x H 20 (rollout_cost_kernel): 31.6 -> 23.2 ms by the
// algebra, -> 16.8 ms with two waves per SIMD (end_leg below, LaneLds in spi_kernels.hip).  Error
// of the costs against 64 bits: 2.2e-6 before, 2.0e-6 after.
#pragma once
#include "spi_dyn.h"

namespace SPI_DYN_NS {

// Type of the legs' constants: that of the arithmetic where it is a builtin one.
template <class T> struct LegConst { using type = float; };
template <> struct LegConst<double> { using type = double; };
using LegReal = LegConst<Real>::type;

// Constants of one leg in its hip frame at O.  Thigh and calf: p, q = (Sxx +- Szz) / 2 and the
// products of S about their axis (a 2 marks twice the value), h the first moment; hip link: see
// above.
template <class T> struct LegC {
  T rx, ry, sx, sy, dz;                     // hip origin in the base and its signs, calf axis below O
  T cp, cp2, cq2, cxz2, cxy, cyz, chx, chz, ci;   // calf; ci = 1 / cp2, its inverse joint inertia
  T tcp, tq2, txz2, txy, tyz, thx, thz;           // thigh, with the calf's axial mass; tcp = tp + cp
  T d2;                                           // 2 (tp + cp) - 2 cp2: thigh pivot at n3 = 0
  T hhy, hhz, hyy, hzz, hxy, hxz, hyz;      // hip link, with the thigh's axial mass
  T fx, fy, fz;                             // foot sphere centre in the calf (y from O)
};

// Mass, first and second moments about a point.
struct MassMoments { double m, hx, hy, hz, xx, yy, zz, xy, xz, yz; };
constexpr MassMoments link_moments(int b, double oy) {   // folded body b (1..12), origin moved by -oy along y
  const double m = SPI_LINK_MASS[b - 1];
  const double x = SPI_LINK_COM[3 * (b - 1)], y = SPI_LINK_COM[3 * (b - 1) + 1] + oy, z = SPI_LINK_COM[3 * (b - 1) + 2];
  const double* I = &SPI_LINK_INERTIA[6 * (b - 1)];
  const double t = 0.5 * (I[0] + I[1] + I[2]);
  return MassMoments{m, m * x, m * y, m * z, t - I[0] + m * x * x, t - I[1] + m * y * y, t - I[2] + m * z * z,
                     -I[3] + m * x * y, -I[4] + m * x * z, -I[5] + m * y * z};
}
// Leg l: its three links after the regrouping, and what its hip axis hands to the base
// (moments about the base origin).
struct LegMass { MassMoments calf, thigh, hip, base; double rx, ry, dz; };
constexpr LegMass leg_mass(int l) {
  const double* o = &SPI_JOINT_ORIGIN[9 * l];
  LegMass r{};
  r.rx = o[0]; r.ry = o[1]; r.dz = o[8];
  r.calf = link_moments(3 + 3 * l, o[4]);
  r.thigh = link_moments(2 + 3 * l, o[4]);
  r.hip = link_moments(1 + 3 * l, 0.0);
  const double m = r.calf.m, y = r.calf.hy, yy = r.calf.yy;         // on the calf axis, at (0, ., dz)
  r.thigh.m += m; r.thigh.hy += y; r.thigh.hz += m * r.dz;
  r.thigh.yy += yy; r.thigh.yz += y * r.dz; r.thigh.zz += m * r.dz * r.dz;
  r.hip.m += r.thigh.m; r.hip.hy += r.thigh.hy; r.hip.yy += r.thigh.yy;   // on the thigh axis, through O
  const double M = r.hip.m, x = r.hip.hx, xx = r.hip.xx;            // on the hip axis, at r0 = (rx, ry, 0)
  r.base = MassMoments{M, M * r.rx + x, M * r.ry, 0.0, xx + 2.0 * x * r.rx + M * r.rx * r.rx, M * r.ry * r.ry, 0.0,
                       x * r.ry + M * r.rx * r.ry, 0.0, 0.0};
  return r;
}
template <class T> constexpr LegC<T> leg_c(int l) {
  const LegMass g = leg_mass(l);
  const double cp = 0.5 * (g.calf.xx + g.calf.zz), cq = 0.5 * (g.calf.xx - g.calf.zz);
  const double tp = 0.5 * (g.thigh.xx + g.thigh.zz), tq = 0.5 * (g.thigh.xx - g.thigh.zz);
  return LegC<T>{T(g.rx), T(g.ry), T(g.rx < 0 ? -1 : 1), T(g.ry < 0 ? -1 : 1), T(g.dz),
                 T(cp), T(2.0 * cp), T(2.0 * cq), T(2.0 * g.calf.xz), T(g.calf.xy), T(g.calf.yz), T(g.calf.hx),
                 T(g.calf.hz), T(0.5 / cp),
                 T(tp + cp), T(2.0 * tq), T(2.0 * g.thigh.xz), T(g.thigh.xy), T(g.thigh.yz), T(g.thigh.hx),
                 T(g.thigh.hz), T(2.0 * (tp + cp) - 4.0 * cp),
                 T(g.hip.hy), T(g.hip.hz), T(g.hip.yy), T(g.hip.zz), T(g.hip.xy), T(g.hip.xz), T(g.hip.yz),
                 T(SPI_FOOT_POS[3 * l]), T(SPI_FOOT_POS[3 * l + 1] + SPI_JOINT_ORIGIN[9 * l + 4]),
                 T(SPI_FOOT_POS[3 * l + 2])};
}

// The structure above: axes x, y, y; hip origin (x, y, 0), thigh (0, y, 0), calf (0, 0, z).
constexpr bool legs_are_planar() {
  for (int l = 0; l < 4; ++l) {
    if (SPI_JOINT_AXIS[3 * l] != 0 || SPI_JOINT_AXIS[3 * l + 1] != 1 || SPI_JOINT_AXIS[3 * l + 2] != 1) return false;
    const double* o = &SPI_JOINT_ORIGIN[9 * l];
    if (o[2] != 0.0 || o[3] != 0.0 || o[5] != 0.0 || o[6] != 0.0 || o[7] != 0.0) return false;
  }
  return true;
}
static_assert(legs_are_planar(), "the closed-form leg elimination assumes the Go2 leg structure");

// Base inertia with the legs' axial mass: what the functions below take as the base.
SPI_HD BaseInertia base_with_legs(const BaseInertia& b) {
  constexpr LegMass g0 = leg_mass(0), g1 = leg_mass(1), g2 = leg_mass(2), g3 = leg_mass(3);
#define SPI_LEGS(f) LegReal(g0.base.f + g1.base.f + g2.base.f + g3.base.f)
  constexpr LegReal m = SPI_LEGS(m), hx = SPI_LEGS(hx), hy = SPI_LEGS(hy), xx = SPI_LEGS(xx), yy = SPI_LEGS(yy),
                    xy = SPI_LEGS(xy);
#undef SPI_LEGS
  return BaseInertia{b.m + m, b.hx + hx, b.hy + hy, b.hz, b.ixx + yy, b.iyy + xx, b.izz + (xx + yy), b.ixy - xy,
                     b.ixz, b.iyz};
}

// 1 / (1 + 2^x): both tanh laws in one exponential and one reciprocal, with no sign handling:
// 1 - tanh(u) = 2 / (1 + 2^(2 u log2 e)).  Its absolute error is spi_tanh's.
SPI_HD Real spi_fall(Real x) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x));
#else
  return 1.0f / (1.0f + exp2f(x));
#endif
}
constexpr float kTwoLog2e = 2.8853900817779268f;
// tau - fric tanh(qd / v0) with inv = 2 log2(e) / v0.
SPI_HD Real joint_friction(Real tau, Real fric, Real qd, Real inv) {
  return (tau - fric) + 2.0f * fric * spi_fall(qd * inv);
}

// What the acceleration pass needs of a leg: the eliminated rows over their pivots (hip: n_y,
// n_z, f; thigh, calf: n_z, f_x, f_z), the multipliers, the bias accelerations, the hip angle.
struct LegElim {
  Real w1y, w1z, w1fx, w1fy, w1fz;
  Real w2z, w2fx, w2fz;
  Real w3z, w3fx, w3fz;
  Real l12, l13, l23;
  Real u1, u2, u3;
  Real c1, s1;
};

// Ends a leg: the sums into the base pass an empty asm, so this leg is finished before the next
// one begins.  Left alone, the compiler evaluates the four contact branches first and then all
// legs interleaved, whose temporaries together leave the 256 registers of two waves per SIMD.
SPI_HD void end_leg(ABI& I, F6& p) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("" : "+v"(I.A.xx), "+v"(I.A.yy), "+v"(I.A.zz), "+v"(I.A.xy), "+v"(I.A.xz), "+v"(I.A.yz),
                    "+v"(I.C.xx), "+v"(I.C.yy), "+v"(I.C.zz), "+v"(I.C.xy), "+v"(I.C.xz), "+v"(I.C.yz));
  asm volatile("" : "+v"(I.B.m00), "+v"(I.B.m01), "+v"(I.B.m02), "+v"(I.B.m10), "+v"(I.B.m11), "+v"(I.B.m12),
                    "+v"(I.B.m20), "+v"(I.B.m21), "+v"(I.B.m22), "+v"(p.n.x), "+v"(p.n.y), "+v"(p.n.z),
                    "+v"(p.f.x), "+v"(p.f.y), "+v"(p.f.z));
#endif
}

// What the four legs share of the base state.  Products with the hip origin's coordinates carry
// the sign-free |rx|, |ry| that all four legs have: a leg adds or subtracts them.
struct BaseMotion {
  V3 w, v;        // base twist, base coordinates
  V3 up;          // world z in base coordinates
  Real z;         // base height
  Real upx, upy;  // |rx| up.x, |ry| up.y
  V3 cx, cy;      // w x (w x .) of (|rx|, 0, 0) and (0, |ry|, 0)
  V3 wh;          // w x (w x h), h the base's first moment
};
constexpr LegReal kHipX = LegReal(SPI_JOINT_ORIGIN[0] < 0 ? -SPI_JOINT_ORIGIN[0] : SPI_JOINT_ORIGIN[0]);
constexpr LegReal kHipY = LegReal(SPI_JOINT_ORIGIN[1] < 0 ? -SPI_JOINT_ORIGIN[1] : SPI_JOINT_ORIGIN[1]);
constexpr bool hips_are_mirrored() {
  for (int l = 0; l < 4; ++l)
    for (int k = 0; k < 2; ++k)
      if (SPI_JOINT_ORIGIN[9 * l + k] != SPI_JOINT_ORIGIN[k] && SPI_JOINT_ORIGIN[9 * l + k] != -SPI_JOINT_ORIGIN[k])
        return false;
  return true;
}
static_assert(hips_are_mirrored(), "the legs share the hip coordinates' magnitudes");
SPI_HD BaseMotion base_motion(V3 w, V3 v, V3 up, Real z, const BaseInertia& B) {
  const Real xx = w.x * w.x, yy = w.y * w.y, zz = w.z * w.z, xy = w.x * w.y, xz = w.x * w.z, yz = w.y * w.z;
  const Real a = -(yy + zz), b = -(xx + zz), c = -(xx + yy);
  return BaseMotion{w, v, up, z, kHipX * up.x, kHipY * up.y, V3{kHipX * a, kHipX * xy, kHipX * xz},
                    V3{kHipY * xy, kHipY * b, kHipY * yz},
                    V3{a * B.hx + xy * B.hy + xz * B.hz, xy * B.hx + b * B.hy + yz * B.hz,
                       xz * B.hx + yz * B.hy + c * B.hz}};
}

// Joint angles' sine and cosine: the hardware's (1.2e-7 absolute), or exact to rounding.
template <bool EXACT> SPI_HD void joint_sincos(Real x, Real* s, Real* c) {
  if constexpr (EXACT) {
    *s = sinf(x);
    *c = cosf(x);
  } else {
    spi_sincos(x, s, c);
  }
}
// a b + c in one rounding, in this order whatever the build lets the compiler regroup.
SPI_HD Real spi_fma(Real a, Real b, Real c) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_fmaf(a, b, c);
#else
  return a * b + c;
#endif
}

// Contact force of the foot sphere in the hip frame and its moments: about O (x, z), about the
// thigh axis (y2) and the calf axis (y3).  The law of foot_contact (spi_dyn.h) with the normal
// and the tangential velocity taken along the ground normal n instead of in world axes.  The
// penetration is summed from the largest terms down: they cancel to the millimetre, and the
// stiffness turns each 1e-8 m of rounding into 5e-4 N.
// SKIP: lanes off the ground skip the block.  One rollout per lane, a wave holds candidates of one
// segment, whose foot is off the ground together (4096 x 256 x H 20 on one box: 16.3 ms, 17.1 without
// the branch); four lanes per rollout, a wave nearly always has a foot down and the skip only costs
// its zeroed results (256 x 64 x H 5: 131 us, 126 without).
struct FootLoad { V3 f; Real mx, mz, y2, y3; };
template <bool SKIP, class C>
SPI_HD FootLoad foot_load(const SpiSimArgs& a, const C& k, const BaseMotion& b, Real x1, Real wy, Real wz, Real sd2,
                          Real sd3, Real c1, Real s1, Real dx, Real dz, Real c3, Real s3) {
  constexpr LegReal rad = LegReal(SPI_FOOT_RADIUS[0]);
  const Real o(0.0f);
  FootLoad out{V3{o, o, o}, o, o, o, o};
  const V3 n = rotT<0>(b.up, c1, s1);
  const Real ex = c3 * k.fx + s3 * k.fz, ez = c3 * k.fz - s3 * k.fx;   // sphere centre from the calf axis
  const Real px = dx + ex, pz = dz + ez;
  const Real pen = -(spi_fma(n.z, pz, b.z - rad) + (n.x * px + n.y * k.fy + (k.sx * b.upx + k.sy * b.upy)));
  if (SKIP && !(pen > Real(0.0f))) return out;
  const Real qx = px - rad * n.x, qy = k.fy - rad * n.y, qz = pz - rad * n.z;   // contact point from O
  const Real gx = ex - rad * n.x, gz = ez - rad * n.z;                          // ... from the calf axis
  // velocity of that point of the calf: hip origin, hip rotation, the two spins about y
  V3 v{b.v.x - b.w.z * k.ry, b.v.y + b.w.z * k.rx, b.v.z + (b.w.x * k.ry - b.w.y * k.rx)};
  v = rotT<0>(v, c1, s1);
  const Real y2 = wy + sd2;
  v.x += y2 * qz - wz * qy + sd3 * gz;
  v.y += wz * qx - x1 * qz;
  v.z += x1 * qy - y2 * qx - sd3 * gx;
  const Real vn = v.x * n.x + v.y * n.y + v.z * n.z;
  const Real kpen = SKIP ? a.k_contact * pen : fmaxf(a.k_contact * pen, Real(1e-20f));
  Real fn = 2.0f * kpen * spi_fall(a.c_contact * kTwoLog2e * vn * spi_rcp(kpen));
  if (!SKIP) fn = pen > Real(0.0f) ? fn : o;   // and with it the friction cone and the force
  const V3 vt{v.x - vn * n.x, v.y - vn * n.y, v.z - vn * n.z};
  // min(c_t |vt|, mu fn) / |vt|; the 1e-30 (m/s)^2 keeps a foot at rest finite
  const Real inv = spi_rsqrt(vt.x * vt.x + vt.y * vt.y + vt.z * vt.z + Real(1e-30f));
  const Real sc = fminf(Real(a.c_tangent), a.mu * fn * inv);
  const V3 f{fn * n.x - sc * vt.x, fn * n.y - sc * vt.y, fn * n.z - sc * vt.z};
  out.f = f;
  out.mx = qy * f.z - qz * f.y;
  out.mz = qx * f.y - qy * f.x;
  out.y2 = qz * f.x - qx * f.z;
  out.y3 = gz * f.x - gx * f.z;
  return out;
}

// One leg: its articulated inertia and bias at the base origin (for the base solve, to be added
// to the base's own) and the record for leg_resolve.  q, qd, tau: hip, thigh, calf (tau after
// friction).  fout (optional): world contact force, R the base rotation.
template <bool SKIP, bool EXACT, class C>
SPI_HD void leg_eliminate(const SpiSimArgs& a, const C& k, const BaseMotion& b, const Real* q, const Real* qd,
                          const Real* tau, ABI& Iout, F6& pout, LegElim& e, const G3* R, Real* fout) {
  Real c1, s1, c2, s2, c3, s3;
  joint_sincos<EXACT>(q[0], &s1, &c1);
  joint_sincos<EXACT>(q[1], &s2, &c2);
  joint_sincos<EXACT>(q[1] + q[2], &s3, &c3);
  const Real sd1 = qd[0], sd2 = qd[1], sd3 = qd[2];

  // --- moments in the hip frame: calf about its axis (h, S), thigh + calf about O (g, T);
  // double angles as cos(2x) / 2 = c^2 - 1/2 and sin(2x) / 2 = c s
  const Real dx = k.dz * s2, dz = k.dz * c2;
  const Real Cc = c3 * c3 - 0.5f, Sc = c3 * s3, Ct = c2 * c2 - 0.5f, St = c2 * s2;
  const Real hx = k.chx * c3 + k.chz * s3, hz = k.chz * c3 - k.chx * s3;
  const Real gx = k.thx * c2 + k.thz * s2 + hx, gz = k.thz * c2 - k.thx * s2 + hz;
  const Real ct = k.cq2 * Cc + k.cxz2 * Sc;
  const Real Sxx = k.cp + ct, Szz = k.cp - ct, Sxz = k.cxz2 * Cc - k.cq2 * Sc;
  const Real Sxy = k.cxy * c3 + k.cyz * s3, Syz = k.cyz * c3 - k.cxy * s3;
  const Real tt = k.tq2 * Ct + k.txz2 * St + ct;
  const Real dxhx = dx * hx, dzhz = dz * hz;
  const Real Txx = 2.0f * dxhx + (k.tcp + tt), Tzz = 2.0f * dzhz + (k.tcp - tt);
  const Real Txz = k.txz2 * Ct - k.tq2 * St + Sxz + dx * hz + dz * hx;
  const Real Txy = k.txy * c2 + k.tyz * s2 + Sxy, Tyz = k.tyz * c2 - k.txy * s2 + Syz;
  // whole leg about O: h = (gx, hhy, Hz), Sxx = Txx, Syy = hyy
  const Real Hz = gz + k.hhz, Vzz = Tzz + k.hzz, Vxy = Txy + k.hxy, Vxz = Txz + k.hxz, Vyz = Tyz + k.hyz;

  // --- elimination of the joint rows, calf first (its pivot is a constant)
  const Real n3 = k.cp2 + dxhx + dzhz;           // calf row: n = (-Sxy, n3, -Syz), f = (hz, 0, -hx)
  const Real l23 = n3 * k.ci, l13 = -k.ci * Sxy;
  const Real w3z = -k.ci * Syz, w3fx = k.ci * hz, w3fz = -k.ci * hx;
  const Real D2 = k.d2 + 2.0f * n3 - l23 * n3;          // Txx + Tzz less the calf's share
  const Real H12 = l23 * Sxy - Txy;
  const Real F2z = l23 * Syz - Tyz, F2x = gz - l23 * hz, F2w = l23 * hx - gx;   // n_z, f_x, f_z
  const Real i2 = spi_rcp(D2);
  const Real l12 = H12 * i2;
  const Real w2z = F2z * i2, w2fx = F2x * i2, w2fz = F2w * i2;
  const Real D1 = k.hyy + Vzz + l13 * Sxy - l12 * H12;
  const LegReal F1y = -k.hxy;
  const Real F1z = l13 * Syz - Vxz - l12 * F2z;
  const Real F1x = -(l13 * hz) - l12 * F2x, F1v = -Hz, F1w = k.hhy + l13 * hx - l12 * F2w;   // f_x, f_y, f_z
  const Real i1 = spi_rcp(D1);
  const Real w1y = F1y * i1, w1z = F1z * i1, w1fx = F1x * i1, w1fy = F1v * i1, w1fz = F1w * i1;
  ABI I;
  const Real o(0.0f);
  I.A = S3{o, k.hzz - w1y * F1y, Txx + k.hyy + w3z * Syz - w2z * F2z - w1z * F1z, o, o, -k.hyz - w1y * F1z};
  I.B = G3{o, o, o,
           k.hhz - w1y * F1x, -(w1y * F1v), -(w1y * F1w),
           -k.hhy - w3z * hz - w2z * F2x - w1z * F1x, gx - w1z * F1v, w3z * hx - w2z * F2w - w1z * F1w};
  I.C = S3{-(w3fx * hz) - w2fx * F2x - w1fx * F1x, -(w1fy * F1v), w3fz * hx - w2fz * F2w - w1fz * F1w,
           -(w1fx * F1v), w3fx * hx - w2fx * F2w - w1fx * F1w, -(w1fy * F1w)};

  // --- velocity products: hip field A about O, spins of the thigh and calf on top
  const V3 w = rotT<0>(b.w, c1, s1);
  const Real x1 = w.x + sd1, x2 = x1 + sd1;
  const V3 aO = rotT<0>(V3{k.sx * b.cx.x + k.sy * b.cy.x, k.sx * b.cx.y + k.sy * b.cy.y, k.sx * b.cx.z + k.sy * b.cy.z},
                        c1, s1);
  const Real xx = x1 * x1, yy = w.y * w.y, zz = w.z * w.z;
  const Real Axx = -(yy + zz), Ayy = -(xx + zz), Azz = -(xx + yy);
  const Real Axy = w.y * x2, Axz = w.z * x2, Ayx = w.y * w.x, Azx = w.z * w.x, Ayz = w.y * w.z;   // Azy = Ayz
  const Real k2 = -(sd2 * (2.0f * w.y + sd2)), bx2 = 2.0f * (sd2 * x1), bz2 = 2.0f * (sd2 * w.z);
  const Real y2 = w.y + sd2;
  const Real k3 = -(sd3 * (2.0f * y2 + sd3)), bx3 = 2.0f * (sd3 * x1), bz3 = 2.0f * (sd3 * w.z);
  const Real f3y = bx3 * hx + bz3 * hz;
  const Real dA = Axx - Azz;
  const FootLoad fc = foot_load<SKIP>(a, k, b, x1, w.y, w.z, sd2, sd3, c1, s1, dx, dz, c3, s3);
  V3 f;
  const Real Bxx = Axx + k2, Bzz = Azz + k2;
  f.x = Bxx * gx + Axy * k.hhy + Axz * Hz + k3 * hx - fc.f.x;
  f.y = Ayx * gx + Ayy * k.hhy + Ayz * Hz + bx2 * gx + bz2 * gz + f3y - fc.f.y;
  f.z = Azx * gx + Ayz * k.hhy + Azz * k.hhz + Bzz * gz + k3 * hz - fc.f.z;
  const Real nx = k.hhy * aO.z - Hz * aO.y + Azx * Vxy + Ayz * (k.hyy - Vzz) + (Azz - Ayy) * Vyz - Ayx * Vxz +
                  (k2 * Tyz - bx2 * Txz - bz2 * Tzz) + (k3 * Syz - bx3 * Sxz - bz3 * Szz - dz * f3y) - fc.mx;
  const Real nz = gx * aO.y - k.hhy * aO.x + Ayx * Txx + (Ayy - Axx) * Vxy + Ayz * Vxz - Axy * k.hyy - Axz * Vyz +
                  (bx2 * Txx + bz2 * Txz - k2 * Txy) + (bx3 * Sxx + bz3 * Sxz - k3 * Sxy + dx * f3y) - fc.mz;
  const Real nyh = k.hhz * aO.x + dA * k.hxz + Axz * k.hzz + Axy * k.hyz - Ayz * k.hxy;   // hip link alone
  const Real n2 = gz * aO.x - gx * aO.z + dA * Txz + Axz * Tzz - Azx * Txx + Axy * Tyz - Ayz * Txy +
                  k3 * (dz * hx - dx * hz) - fc.y2;
  const Real acx = aO.x + Bxx * dx + Axz * dz, acz = aO.z + Azx * dx + Bzz * dz;
  const Real n3b = hz * acx - hx * acz + dA * Sxz + Axz * Szz - Azx * Sxx + Axy * Syz - Ayz * Sxy - fc.y3;

  const Real r3 = tau[2] - n3b, r2 = tau[1] - n2 - l23 * r3, r1 = tau[0] - nx - l13 * r3 - l12 * r2;
  const Real u3 = r3 * k.ci, u2 = r2 * i2, u1 = r1 * i1;
  F6 p;
  p.n = V3{tau[0], tau[1] + nyh + F1y * u1, nz - Syz * u3 + F2z * u2 + F1z * u1};
  p.f = V3{f.x + hz * u3 + F2x * u2 + F1x * u1, f.y + F1v * u1, f.z - hx * u3 + F2w * u2 + F1w * u1};
  e = LegElim{w1y, w1z, w1fx, w1fy, w1fz, w2z, w2fx, w2fz, w3z, w3fx, w3fz, l12, l13, l23, u1, u2, u3, c1, s1};
  const V3 r0{k.rx, k.ry, o};
  Iout = xtix<0>(I, r0, c1, s1);
  pout = xtf<0>(p, r0, c1, s1);
  if (fout) {
    const V3 fw = mul(*R, rot<0>(fc.f, c1, s1));
    fout[0] = fw.x; fout[1] = fw.y; fout[2] = fw.z;
  }
}

// Joint accelerations of a leg from the base's (a0: angular, proper linear).
template <class C> SPI_HD void leg_resolve(const C& k, const LegElim& e, const M6& a0, Real* qdd) {
  const V3 al = rotT<0>(a0.w, e.c1, e.s1);
  const V3 aO = rotT<0>(V3{a0.v.x - a0.w.z * k.ry, a0.v.y + a0.w.z * k.rx, a0.v.z + (a0.w.x * k.ry - a0.w.y * k.rx)},
                        e.c1, e.s1);
  const Real X1 = e.u1 - (e.w1y * al.y + e.w1z * al.z + e.w1fx * aO.x + e.w1fy * aO.y + e.w1fz * aO.z);
  const Real X2 = e.u2 - (e.w2z * al.z + e.w2fx * aO.x + e.w2fz * aO.z) - e.l12 * X1;
  qdd[0] = X1 - al.x;
  qdd[1] = X2 - al.y;
  qdd[2] = e.u3 - (e.w3z * al.z + e.w3fx * aO.x + e.w3fz * aO.z) - e.l13 * X1 - e.l23 * X2;
}

// Base inertia blocks and velocity product of the base (with the legs' axial mass).
SPI_HD void base_terms(const BaseInertia& B, const BaseMotion& b, ABI& I, F6& p) {
  const RBT<Real> rb{B.m, B.hx, B.hy, B.hz, B.ixx, B.iyy, B.izz, B.ixy, B.ixz, B.iyz};
  I = rb_abi(rb);
  p = F6{cross(b.w, mul(I.A, b.w)), b.wh};
}
// dv/dt of the base in base coordinates from its proper acceleration a0.
SPI_HD M6 base_rate(const M6& a0, V3 w, V3 v, V3 up, Real g) {
  return M6{a0.w, a0.v - cross(w, v) - g * up};
}

// The lane's parameters and joint torques, all in registers.
template <bool EXACT = false> struct LaneRegsT {
  static constexpr bool kSkip = false, kExact = EXACT;
  const LaneParams& lp;       // lp.base: base_with_legs()
  const Real* tau_motor;
  SPI_HD BaseInertia base() const { return lp.base; }
  SPI_HD void leg(int l, Real* tau, Real* fric) const {
#pragma unroll
    for (int k = 0; k < 3; ++k) tau[k] = tau_motor[3 * l + k];
    *fric = lp.fric[l];
  }
};
using LaneRegs = LaneRegsT<false>;

// forward_dynamics of spi_dyn.h by leg elimination.  P: base() the base inertia with the legs'
// axial mass, leg(l, tau, &friction) the leg's motor torques and joint friction, kSkip of foot_load, kExact of joint_sincos.
template <class P>
SPI_HD void forward_dynamics_elim(const SpiSimArgs& a, const P& par, const State& st, M6& acc0, Real* qdd,
                                  Real* foot_force) {
  const G3 R = quat_to_rot(st.qx, st.qy, st.qz, st.qw);
  const BaseInertia B = par.base();
  const BaseMotion b = base_motion(st.w, st.v, V3{R.m20, R.m21, R.m22}, st.p.z, B);
  constexpr LegC<LegReal> k0 = leg_c<LegReal>(0), k1 = leg_c<LegReal>(1), k2 = leg_c<LegReal>(2),
                          k3 = leg_c<LegReal>(3);
  ABI I;
  F6 p;
  base_terms(B, b, I, p);
  LegElim e[4];
#define SPI_ELIM(L, K)                                                                                        \
  {                                                                                                           \
    ABI t;                                                                                                    \
    F6 pt;                                                                                                    \
    Real tau[3], fric;                                                                                        \
    par.leg(L, tau, &fric);                                                                                   \
    for (int j = 0; j < 3; ++j)                                                                               \
      tau[j] = joint_friction(tau[j], fric, st.qd[3 * L + j], a.fric_vel_inv * kTwoLog2e);                    \
    leg_eliminate<P::kSkip, P::kExact>(a, K, b, st.q + 3 * L, st.qd + 3 * L, tau, t, pt, e[L], &R,                                 \
                  foot_force ? foot_force + 3 * L : nullptr);                                                 \
    abi_add(I, t);                                                                                            \
    p = F6{p.n + pt.n, p.f + pt.f};                                                                           \
    end_leg(I, p);                                                                                            \
  }
  SPI_ELIM(0, k0)
  SPI_ELIM(1, k1)
  SPI_ELIM(2, k2)
  SPI_ELIM(3, k3)
#undef SPI_ELIM
  const M6 a0 = solve_base(I, F6{-1.0f * p.n, -1.0f * p.f});
  leg_resolve(k0, e[0], a0, qdd);
  leg_resolve(k1, e[1], a0, qdd + 3);
  leg_resolve(k2, e[2], a0, qdd + 6);
  leg_resolve(k3, e[3], a0, qdd + 9);
  acc0 = base_rate(a0, st.w, st.v, b.up, a.gravity);
}

// physics_step of spi_dyn.h by leg elimination.
template <class P>
SPI_HD void physics_step_elim(const SpiSimArgs& a, const P& par, State& st, Real* foot_force) {
  const Real h = a.dt / Real(a.substeps);
  for (int k = 0; k < a.substeps; ++k) {
    M6 acc0;
    Real qdd[12];
    forward_dynamics_elim(a, par, st, acc0, qdd, foot_force);
    integrate(st, acc0, qdd, h);
  }
}

}  // namespace SPI_DYN_NS
