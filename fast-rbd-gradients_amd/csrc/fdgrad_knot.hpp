// Per-knot-point forward-dynamics gradient of the KUKA iiwa 14, register resident.
//
// One call computes, for one knot point, q, qd, u -> qdd, dqdd/dq, dqdd/dqd with
// the reference's results (plancherb1/fast-rbd-gradients); the steps:
//   1. sin/cos of q and the seven joint transforms  (dynamicsGradient.h:507-587)
//   2. the articulated-body recursion: the mass matrix's factors, or Minv
//      where it is an output or shared by lanes       (minv.h:423-478)
//   3. RNEA with qdd = 0 -> bias c                    (dynamicsGradient.h:619-683)
//   4. qdd = Minv (u - c)                             (dynamicsGradient.h:704)
//   5. RNEA with qdd: v, a, f                         (dynamicsGradient.h:893-895)
//   6. dtau/dq, dtau/dqd: from composite quantities in one lane, by a forward
//      and a backward sweep over the links per column in a lane group
//                                                     (dynamicsGradient.h:786-857)
//   7. dqdd/d(q,qd) = -Minv dtau/d(q,qd)              (dynamicsGradient.h:921)
// Every link index is a compile-time constant (static_for), so each joint's
// transform, inertia and offset are folded into straight-line code: structural
// zeros of E, r and I cost nothing when the file is compiled with
// -fno-signed-zeros -ffinite-math-only (these let x*0 and x+0 fold away).
// A lane group gives each lane run-time columns of its own
// (dtau_column_uniform).
//
// The file is plain C++17 when RBD_HD is empty, so the same arithmetic is also
// compiled for the host by the CPU test harness.
#pragma once
// The robot: the KUKA iiwa 14 unless the build names a header generated from a
// URDF by urdf_model.py (-DRBD_MODEL_HEADER='"model_NAME.hpp"').
#ifdef RBD_MODEL_HEADER
#include RBD_MODEL_HEADER
#else
#include "iiwa_model.hpp"
#endif
#include <type_traits>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define RBD_HD __host__ __device__
#else
#include <cmath>
#define RBD_HD
#endif
#define RBD_INLINE __attribute__((always_inline)) inline

namespace rbd {

template <int N> struct IC { static constexpr int value = N; };

// f(IC<B>), f(IC<B+1>), ..., f(IC<E-1>)
template <int B, int E, class F>
RBD_HD RBD_INLINE void static_for(F&& f) {
  if constexpr (B < E) { f(IC<B>{}); static_for<B + 1, E>(f); }
}
// f(IC<B-1>), f(IC<B-2>), ..., f(IC<E>)
template <int B, int E, class F>
RBD_HD RBD_INLINE void static_for_down(F&& f) {
  if constexpr (B > E) { f(IC<B - 1>{}); static_for_down<B - 1, E>(f); }
}

template <typename S> struct CS { S c, s; };

RBD_HD RBD_INLINE float fma_s(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
RBD_HD RBD_INLINE double fma_s(double a, double b, double c) { return __builtin_fma(a, b, c); }

// sin and cos without divergent branches.  The math library's take one path
// for ordinary arguments and another for huge ones, an if/else that lanes may
// split over; in kernels short of registers the compiler moved values that
// live across it into accumulation registers or scratch at the start of the
// block where the two paths meet, ahead of the instruction that turns the
// other lanes back on, so that with no lane on the rare path nothing was saved
// and garbage came back (in FP64-column kernels: wrong gradients in groups of
// 8 lanes, stores to garbage addresses).  Below, every lane takes one straight
// path, and a second one only if some lane of the wave is out of its range.
//
// r = x - k pi/2 in [-pi/4, pi/4], sin and cos of r by minimax polynomials in
// r^2 fitted for that range, quadrant k mod 4.
//
// FP32, |x| <= 512: pi/2 in three parts.  The first difference is exact; the
// second part has 15 bits, so that its product with k (9 bits) is exact too
// and what rounding r loses can be formed, and goes into the results with the
// third part as the low word lo.  Polynomial errors 3.6e-9 and 1e-10; the
// results are within 0.92 units in the last place.
template <typename S> constexpr S kSincosMax = sizeof(S) == 4 ? S(512) : S(65536);
RBD_HD RBD_INLINE void sincos_reduced(float x, float* s, float* c) {
  const float k = __builtin_rintf(x * 0.63661977236758134f);
  const float r1 = __builtin_fmaf(-k, 0x1.921fb6p+0f, x);
  const float r = __builtin_fmaf(-k, -0x1.777cp-25f, r1);
  // what rounding r lost, and the third part
  const float lo = __builtin_fmaf(-k, 0x1.a308d4p-41f, __builtin_fmaf(-k, -0x1.777cp-25f, r1 - r));
  const float z = r * r;
  float ps = __builtin_fmaf(z, -0x1.994b4p-13f, 0x1.110756p-7f);
  ps = __builtin_fmaf(z, ps, -0x1.555546p-3f);
  const float sr = r + __builtin_fmaf(r * z, ps, lo);
  float pc = __builtin_fmaf(z, 0x1.99ff42p-16f, -0x1.6c0c82p-10f);
  pc = __builtin_fmaf(z, pc, 0x1.55554ap-5f);
  const float hz = 0.5f * z, ca = 1.0f - hz;
  const float cr = ca + __builtin_fmaf(z * z, pc, __builtin_fmaf(-lo, r, (1.0f - ca) - hz));
  const unsigned q = unsigned(int(k));
  const bool swap = (q & 1u) != 0u;
  const float ss = swap ? cr : sr, cc = swap ? sr : cr;
  *s = (q & 2u) ? -ss : ss;
  *c = ((q + 1u) & 2u) ? -cc : cc;
}
// sin and cos of q pi/2 + r in FP64 (polynomial errors 3.5e-18 and 4.7e-20)
RBD_HD RBD_INLINE void sincos_quadrant(unsigned q, double r, double* s, double* c) {
  const double z = r * r;
  double ps = __builtin_fma(z, 0x1.5d92451b64143p-33, -0x1.ae5e63c6fd08dp-26);
  ps = __builtin_fma(z, ps, 0x1.71de3574b0c8ap-19);
  ps = __builtin_fma(z, ps, -0x1.a01a019c0e3efp-13);
  ps = __builtin_fma(z, ps, 0x1.111111110f861p-7);
  ps = __builtin_fma(z, ps, -0x1.5555555555549p-3);
  const double sr = __builtin_fma(r * z, ps, r);
  double pc = __builtin_fma(z, -0x1.8fadd03da3e34p-37, 0x1.1ee9ea6c52bd8p-29);
  pc = __builtin_fma(z, pc, -0x1.27e4f807d5628p-22);
  pc = __builtin_fma(z, pc, 0x1.a01a019caef23p-16);
  pc = __builtin_fma(z, pc, -0x1.6c16c16c15162p-10);
  pc = __builtin_fma(z, pc, 0x1.555555555554cp-5);
  const double cr = __builtin_fma(z, __builtin_fma(z, pc, -0.5), 1.0);
  const bool swap = (q & 1u) != 0u;
  const double ss = swap ? cr : sr, cc = swap ? sr : cr;
  *s = (q & 2u) ? -ss : ss;
  *c = ((q + 1u) & 2u) ? -cc : cc;
}
// FP64, |x| <= 65536: pi/2 in two parts (results within 2 units in the last
// place; every output is FP32)
RBD_HD RBD_INLINE void sincos_reduced(double x, double* s, double* c) {
  const double k = __builtin_rint(x * 0x1.45f306dc9c883p-1);
  const double r = __builtin_fma(-k, 0x1.1a62633145c07p-54, __builtin_fma(-k, 0x1.921fb54442d18p+0, x));
  sincos_quadrant(unsigned(int(k)), r, s, c);
}
// sin and cos of an FP32 angle of any size from 2^-7 up, by integer arithmetic
// (Payne and Hanek's reduction): with x = m 2^E, the bits of 2/pi from weight
// 2^(1 - E) on, as a 128-bit number W, give x 2/pi mod 4 = (m W mod 2^128)
// 2^-126: two bits of quadrant and 126 of fraction, of which an FP32 x cancels
// at most about 30.  For FP64 results (S) the fraction is taken in two words
// and multiplied by pi/2 in two, so that r is rounded once and the results stay
// within 2 units in the last place (1.50; one word of each: 2.53).
template <typename S>
RBD_HD RBD_INLINE void sincos_far(float x, double* s, double* c) {
  constexpr unsigned kTwoOverPi[9] = {0u, 0xa2f9836eu, 0x4e441529u, 0xfc2757d1u, 0xf534ddc0u, 0xdb629599u, 0x3c439041u, 0xfe5163abu, 0xdebbc561u};
  const unsigned bits = __builtin_bit_cast(unsigned, x);
  const unsigned m = (bits & 0x7fffffu) | 0x800000u;
  const int e = int((bits >> 23) & 255u) - 120;      // first bit of W, after 32 zero bits
  const unsigned p = unsigned(e < 0 ? 0 : e), word = p >> 5, shift = p & 31u;
  unsigned w[5];                                     // the five words that W lies in
  static_for<0, 5>([&](auto Jc) {
    constexpr int j = decltype(Jc)::value;
    w[j] = kTwoOverPi[j];
    static_for<1, 5>([&](auto Kc) {
      constexpr int k = decltype(Kc)::value;
      w[j] = word == unsigned(k) ? kTwoOverPi[j + k] : w[j];
    });
  });
  unsigned long long t = 0;
  unsigned limb[4];
  static_for_down<4, 0>([&](auto Jc) {
    constexpr int j = decltype(Jc)::value;
    const unsigned long long two = (static_cast<unsigned long long>(w[j]) << 32) | w[j + 1];
    t = static_cast<unsigned long long>(m) * unsigned(two >> (32u - shift)) + (t >> 32);
    limb[j] = unsigned(t);
  });
  const unsigned long long hi = (static_cast<unsigned long long>(limb[0]) << 32) | limb[1];
  const unsigned long long lo = (static_cast<unsigned long long>(limb[2]) << 32) | limb[3];
  const unsigned q = unsigned((hi + (1ull << 61)) >> 62);           // nearest quarter turn
  const long long whole = static_cast<long long>(hi - (static_cast<unsigned long long>(q) << 62));
  constexpr double half_pi = 0x1p-62 * 0x1.921fb54442d18p+0, half_pi_low = 0x1p-62 * 0x1.1a62633145c07p-54;
  double r;
  if constexpr (sizeof(S) == 8) {
    const double f = double(whole);
    const double low = double(whole - static_cast<long long>(f)) + double(lo) * 0x1p-64;
    r = __builtin_fma(f, half_pi, __builtin_fma(low, half_pi, f * half_pi_low));
  } else {
    r = (double(whole) + double(lo) * 0x1p-64) * half_pi;
  }
  const bool neg = (bits >> 31) != 0u;
  sincos_quadrant(neg ? 0u - q : q, neg ? -r : r, s, c);
}
// sin and cos of a joint angle x (an FP32 value in either type)
template <typename S>
RBD_HD RBD_INLINE void sincos_s(S x, S* s, S* c) {
#if defined(__HIP_DEVICE_COMPILE__)
  sincos_reduced(x, s, c);
  const bool far = !(__builtin_fabs(x) <= kSincosMax<S>);
  if (__ballot(far) != 0) {              // the same in every lane
    double sf, cf;
    sincos_far<S>(float(x), &sf, &cf);
    *s = far ? S(sf) : *s;
    *c = far ? S(cf) : *c;
  }
#else
  *s = std::sin(x); *c = std::cos(x);
#endif
}

// ---------------------------------------------------------------------------
// Joint transform of link K: T = [E 0; -E r^ E]
// ---------------------------------------------------------------------------
template <int K, int I, int J, typename S>
RBD_HD RBD_INLINE S Eij(const CS<S>& t) {
  constexpr S a = S(ecoef_c(K, I, J)), b = S(ecoef_s(K, I, J)), d = S(ecoef_1(K, I, J));
  return a * t.c + b * t.s + d;
}
// y = E x
template <int K, typename S>
RBD_HD RBD_INLINE void rot(const CS<S>& t, const S* x, S* y) {
  static_for<0, 3>([&](auto Ic) {
    constexpr int i = decltype(Ic)::value;
    y[i] = Eij<K, i, 0>(t) * x[0] + Eij<K, i, 1>(t) * x[1] + Eij<K, i, 2>(t) * x[2];
  });
}
// y = E^T x
template <int K, typename S>
RBD_HD RBD_INLINE void rot_t(const CS<S>& t, const S* x, S* y) {
  static_for<0, 3>([&](auto Jc) {
    constexpr int j = decltype(Jc)::value;
    y[j] = Eij<K, 0, j>(t) * x[0] + Eij<K, 1, j>(t) * x[1] + Eij<K, 2, j>(t) * x[2];
  });
}
template <int K, typename S> constexpr S roff(int i) { return S(kJointOffset[K][i]); }

// y = T x for a motion vector: [E w; E (u - r x w)]
template <int K, typename S>
RBD_HD RBD_INLINE void xmotion(const CS<S>& t, const S* x, S* y) {
  constexpr S rx = roff<K, S>(0), ry = roff<K, S>(1), rz = roff<K, S>(2);
  // u - r x w, each product subtracted on its own
  S d[3] = {x[3], x[4], x[5]};
  d[0] -= ry * x[2]; d[0] += rz * x[1];
  d[1] -= rz * x[0]; d[1] += rx * x[2];
  d[2] -= rx * x[1]; d[2] += ry * x[0];
  S y0[3], y1[3];
  rot<K>(t, x, y0);
  rot<K>(t, d, y1);
  y[0] = y0[0]; y[1] = y0[1]; y[2] = y0[2];
  y[3] = y1[0]; y[4] = y1[1]; y[5] = y1[2];
}
// y = T^T x + z for a force vector: [E^T n + r x (E^T f); E^T f] + z.  The
// angular rows add each product to the row on its own (one FMA each), starting
// from z.
template <int K, typename S>
RBD_HD RBD_INLINE void xforce_t_add(const CS<S>& t, const S* x, const S* z, S* y) {
  constexpr S rx = roff<K, S>(0), ry = roff<K, S>(1), rz = roff<K, S>(2);
  S fl[3];
  rot_t<K>(t, x + 3, fl);
  const S r[3] = {rx, ry, rz};
  static_for<0, 3>([&](auto Jc) {
    constexpr int j = decltype(Jc)::value;
    constexpr int j1 = (j + 1) % 3, j2 = (j + 2) % 3;
    S acc = z[j];
    acc += Eij<K, 0, j>(t) * x[0];
    acc += Eij<K, 1, j>(t) * x[1];
    acc += Eij<K, 2, j>(t) * x[2];
    acc += r[j1] * fl[j2];                    // (r x fl)_j
    acc -= r[j2] * fl[j1];
    y[j] = acc;
  });
  for (int j = 0; j < 3; ++j) y[3 + j] = z[3 + j] + fl[j];
}

// entry (R, C) of link K's spatial inertia, as a compile-time constant
template <typename S, int K, int R, int C>
constexpr S kInertia = S(inertia_entry(K, R, C));

// y (+)= I_K x, I_K the constant spatial inertia of link K
template <int K, bool ACC = false, typename S>
RBD_HD RBD_INLINE void imv(const S* x, S* y) {
  static_for<0, 6>([&](auto Rc) {
    constexpr int r = decltype(Rc)::value;
    S acc = kInertia<S, K, r, 0> * x[0];
    static_for<1, 6>([&](auto Cc) {
      constexpr int c = decltype(Cc)::value;
      acc += kInertia<S, K, r, c> * x[c];
    });
    y[r] = ACC ? y[r] + acc : acc;
  });
}
// A = I_K (for the host's check of the model's tables)
template <int K, typename S>
RBD_HD RBD_INLINE void iload(S A[6][6]) {
  static_for<0, 6>([&](auto Rc) {
    constexpr int r = decltype(Rc)::value;
    static_for<0, 6>([&](auto Cc) {
      constexpr int c = decltype(Cc)::value;
      A[r][c] = kInertia<S, K, r, c>;
    });
  });
}

// y (+)= x x* z  =  [w x za + u x zl ; w x zl]   (spatial force cross product).
// Accumulating, each product is added to y on its own (one FMA each) rather
// than summed first and added once: the same terms, one instruction fewer
// per component.
template <bool ACC = false, typename S>
RBD_HD RBD_INLINE void crf(const S* x, const S* z, S* y) {
  if (ACC) {
    S y0 = y[0], y1 = y[1], y2 = y[2], y3 = y[3], y4 = y[4], y5 = y[5];
    y0 += x[1] * z[2]; y0 -= x[2] * z[1]; y0 += x[4] * z[5]; y0 -= x[5] * z[4];
    y1 += x[2] * z[0]; y1 -= x[0] * z[2]; y1 += x[5] * z[3]; y1 -= x[3] * z[5];
    y2 += x[0] * z[1]; y2 -= x[1] * z[0]; y2 += x[3] * z[4]; y2 -= x[4] * z[3];
    y3 += x[1] * z[5]; y3 -= x[2] * z[4];
    y4 += x[2] * z[3]; y4 -= x[0] * z[5];
    y5 += x[0] * z[4]; y5 -= x[1] * z[3];
    y[0] = y0; y[1] = y1; y[2] = y2; y[3] = y3; y[4] = y4; y[5] = y5;
  } else {
    y[0] = x[1] * z[2] - x[2] * z[1] + x[4] * z[5] - x[5] * z[4];
    y[1] = x[2] * z[0] - x[0] * z[2] + x[5] * z[3] - x[3] * z[5];
    y[2] = x[0] * z[1] - x[1] * z[0] + x[3] * z[4] - x[4] * z[3];
    y[3] = x[1] * z[5] - x[2] * z[4];
    y[4] = x[2] * z[3] - x[0] * z[5];
    y[5] = x[0] * z[4] - x[1] * z[3];
  }
}

// ---------------------------------------------------------------------------
// The recursions below are written with every multiply-add explicit (fma_s),
// so that each kernel that inlines them computes bitwise the same values: left
// to the compiler, which product of a sum is fused differs from kernel to
// kernel.  Products with structural zeros still fold away.
// ---------------------------------------------------------------------------
// F of E = Z(q) F, Z = [c s 0; -s c 0; 0 0 1]: the joint's fixed rotation
template <int K>
RBD_HD constexpr double fixed_rot(int i, int j) {
  return i < 2 ? double(ecoef_c(K, i, j)) : double(ecoef_1(K, 2, j));
}
template <int K>
RBD_HD constexpr bool signed_permutation() {
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) {
      const double f = fixed_rot<K>(i, j);
      if (f != 0.0 && f != 1.0 && f != -1.0) return false;
    }
  return true;
}
template <typename S, int K, int I, int J> constexpr S kFixed = S(fixed_rot<K>(I, J));

// (F^T x)_J and (F x)_I
template <int K, int J, typename S>
RBD_HD RBD_INLINE S fixed_t(const S* x) {
  return fma_s(kFixed<S, K, 0, J>, x[0], fma_s(kFixed<S, K, 1, J>, x[1], kFixed<S, K, 2, J> * x[2]));
}
template <int K, int I, typename S>
RBD_HD RBD_INLINE S fixed(const S* x) {
  return fma_s(kFixed<S, K, I, 0>, x[0], fma_s(kFixed<S, K, I, 1>, x[1], kFixed<S, K, I, 2> * x[2]));
}
// Entry (I, J) of E = Rz(q)^T F.  Where F is no signed permutation, a rotation
// by E's entries (formed once per link and shared by all its rotations) takes 9
// instructions and one by F, then Rz, 13.  Synthetic arm: 128 knots 6.35 -> 6.05
// us, 2,500 knots 7.3 -> 6.7, 9,000 knots 10.5 -> 10.0; in one lane the entries
// cost registers (216 bytes of spills; 20,000 knots 15.4 -> 14.9 us, 2^20 knots
// 164 -> 173), and one form serves all mappings so that they round alike.
template <int K, int I, int J, typename S>
RBD_HD RBD_INLINE S rot_entry(const CS<S>& t) {
  if constexpr (I == 0) return fma_s(t.c, kFixed<S, K, 0, J>, t.s * kFixed<S, K, 1, J>);
  else if constexpr (I == 1) return fma_s(t.c, kFixed<S, K, 1, J>, -t.s * kFixed<S, K, 0, J>);
  else return kFixed<S, K, 2, J>;
}
// y = E x
template <int K, typename S>
RBD_HD RBD_INLINE void to_child(const CS<S>& t, const S* x, S* y) {
  if constexpr (!signed_permutation<K>()) {
    const S x0 = x[0], x1 = x[1], x2 = x[2];
    static_for<0, 3>([&](auto Ic) {
      constexpr int i = decltype(Ic)::value;
      y[i] = fma_s(rot_entry<K, i, 0>(t), x0, fma_s(rot_entry<K, i, 1>(t), x1, rot_entry<K, i, 2>(t) * x2));
    });
    return;
  }
  const S w0 = fixed<K, 0>(x), w1 = fixed<K, 1>(x), w2 = fixed<K, 2>(x);
  y[0] = fma_s(t.s, w1, t.c * w0);
  y[1] = fma_s(-t.s, w0, t.c * w1);
  y[2] = w2;
}
// y = E^T x, and y = E^T x + z
template <int K, typename S>
RBD_HD RBD_INLINE void to_parent(const CS<S>& t, const S* x, S* y) {
  if constexpr (!signed_permutation<K>()) {
    const S x0 = x[0], x1 = x[1], x2 = x[2];
    static_for<0, 3>([&](auto Jc) {
      constexpr int j = decltype(Jc)::value;
      y[j] = fma_s(rot_entry<K, 0, j>(t), x0, fma_s(rot_entry<K, 1, j>(t), x1, rot_entry<K, 2, j>(t) * x2));
    });
    return;
  }
  const S w[3] = {fma_s(-t.s, x[1], t.c * x[0]), fma_s(t.s, x[0], t.c * x[1]), x[2]};
  const S y0 = fixed_t<K, 0>(w), y1 = fixed_t<K, 1>(w), y2 = fixed_t<K, 2>(w);
  y[0] = y0; y[1] = y1; y[2] = y2;
}
template <int K, typename S>
RBD_HD RBD_INLINE void to_parent_add(const CS<S>& t, const S* x, const S* z, S* y) {
  if constexpr (signed_permutation<K>()) {
    // F^T (Z^T x + F z): the permuted z starts the sums, two adds fewer
    const S w[3] = {fma_s(-t.s, x[1], fma_s(t.c, x[0], fixed<K, 0>(z))),
                    fma_s(t.s, x[0], fma_s(t.c, x[1], fixed<K, 1>(z))), x[2] + fixed<K, 2>(z)};
    const S y0 = fixed_t<K, 0>(w), y1 = fixed_t<K, 1>(w), y2 = fixed_t<K, 2>(w);
    y[0] = y0; y[1] = y1; y[2] = y2;
  } else {
    const S x0 = x[0], x1 = x[1], x2 = x[2];
    static_for<0, 3>([&](auto Jc) {
      constexpr int j = decltype(Jc)::value;
      y[j] = fma_s(rot_entry<K, 0, j>(t), x0,
                   fma_s(rot_entry<K, 1, j>(t), x1, fma_s(rot_entry<K, 2, j>(t), x2, z[j])));
    });
  }
}
// y += r x f, r joint K's offset
template <int K, typename S>
RBD_HD RBD_INLINE void add_offset_cross(const S* f, S* y) {
  constexpr S rx = roff<K, S>(0), ry = roff<K, S>(1), rz = roff<K, S>(2);
  y[0] = fma_s(ry, f[2], fma_s(-rz, f[1], y[0]));
  y[1] = fma_s(rz, f[0], fma_s(-rx, f[2], y[1]));
  y[2] = fma_s(rx, f[1], fma_s(-ry, f[0], y[2]));
}
// x = T x for a motion vector (parent to child), in place
template <int K, typename S>
RBD_HD RBD_INLINE void move_motion(const CS<S>& t, const S* x, S* y) {
  constexpr S rx = roff<K, S>(0), ry = roff<K, S>(1), rz = roff<K, S>(2);
  const S d[3] = {fma_s(-ry, x[2], fma_s(rz, x[1], x[3])), fma_s(-rz, x[0], fma_s(rx, x[2], x[4])),
                  fma_s(-rx, x[1], fma_s(ry, x[0], x[5]))};
  S w[3];
  to_child<K>(t, x, w);
  to_child<K>(t, d, y + 3);
  y[0] = w[0]; y[1] = w[1]; y[2] = w[2];
}
// x = T^T x for a force vector (child to parent), in place
template <int K, typename S>
RBD_HD RBD_INLINE void move_force(const CS<S>& t, S* x) {
  to_parent<K>(t, x, x);
  to_parent<K>(t, x + 3, x + 3);
  add_offset_cross<K>(x + 3, x);
}
// z += T^T x
template <int K, typename S>
RBD_HD RBD_INLINE void add_moved_force(const CS<S>& t, const S* x, S* z) {
  S f[3];
  to_parent<K>(t, x + 3, f);
  to_parent_add<K>(t, x, z, z);
  add_offset_cross<K>(f, z);
  z[3] += f[0]; z[4] += f[1]; z[5] += f[2];
}
// y = I_K x, I_K the constant inertia of link K
template <int K, typename S>
RBD_HD RBD_INLINE void inertia_times(const S* x, S* y) {
  static_for<0, 6>([&](auto Rc) {
    constexpr int r = decltype(Rc)::value;
    S acc = kInertia<S, K, r, 0> * x[0];
    static_for<1, 6>([&](auto Cc) {
      constexpr int c = decltype(Cc)::value;
      acc = fma_s(kInertia<S, K, r, c>, x[c], acc);
    });
    y[r] = acc;
  });
}
// y += x x* z
template <typename S>
RBD_HD RBD_INLINE void add_force_cross(const S* x, const S* z, S* y) {
  y[0] = fma_s(x[1], z[2], fma_s(-x[2], z[1], fma_s(x[4], z[5], fma_s(-x[5], z[4], y[0]))));
  y[1] = fma_s(x[2], z[0], fma_s(-x[0], z[2], fma_s(x[5], z[3], fma_s(-x[3], z[5], y[1]))));
  y[2] = fma_s(x[0], z[1], fma_s(-x[1], z[0], fma_s(x[3], z[4], fma_s(-x[4], z[3], y[2]))));
  y[3] = fma_s(x[1], z[5], fma_s(-x[2], z[4], y[3]));
  y[4] = fma_s(x[2], z[3], fma_s(-x[0], z[5], y[4]));
  y[5] = fma_s(x[0], z[4], fma_s(-x[1], z[3], y[5]));
}

// Symmetric 3x3 matrices are stored as xx, xy, xz, yy, yz, zz.
RBD_HD constexpr int sym(int i, int j) { return (i == 0 || j == 0) ? i + j : i + j + 1; }
// products of a joint's sin and cos: cos^2 q, sin^2 q, sin 2q, cos 2q, sin(2q) / 2
template <typename S> struct DoubleAngle { S cc, ss, s2, c2, sc; };
template <typename S>
RBD_HD RBD_INLINE DoubleAngle<S> double_angle(const CS<S>& t) {
  const S ss = t.s * t.s, sc = t.c * t.s;
  return {t.c * t.c, ss, sc + sc, fma_s(S(-2), ss, S(1)), sc};
}
// A = E^T A E.  Where F is a signed permutation: the z rotation leaves the trace
// of the x-y block, so the block takes 7 operations instead of the 14 of two
// one-sided rotations.  SMALL_DIAGONAL: a diagonal entry may come out far below
// the other (the articulated inertia about a slender link's axis, the pivot),
// and as the difference of two large numbers it would keep their rounding
// error: its terms are summed instead (3 operations more).  Error of dqdd/dq in
// lane groups, FP32: 2.07e-7 against 2.14e-7 of its norm.  Other F: two
// one-sided rotations by E's entries, which also take fewer instructions than
// the z rotation and F on both sides (synthetic arm, dqdd/dq 4.37e-7 against
// 4.58e-7; 104 instructions fewer in a factorisation).
template <int K, bool SMALL_DIAGONAL, typename S>
RBD_HD RBD_INLINE void sym_to_parent(const CS<S>& t, const DoubleAngle<S>& q, S A[6]) {
  if constexpr (!signed_permutation<K>()) {
    S Y[3][3];                                   // A E
    static_for<0, 3>([&](auto Rc) {
      constexpr int r = decltype(Rc)::value;
      const S row[3] = {A[sym(r, 0)], A[sym(r, 1)], A[sym(r, 2)]};
      to_parent<K>(t, row, Y[r]);
    });
    static_for<0, 3>([&](auto Jc) {
      constexpr int j = decltype(Jc)::value;
      const S col[3] = {Y[0][j], Y[1][j], Y[2][j]};
      S y[3];
      to_parent<K>(t, col, y);
      for (int i = 0; i <= j; ++i) A[sym(i, j)] = y[i];
    });
    return;
  }
  const S d = A[3] - A[0];
  S b0, b3;
  if constexpr (SMALL_DIAGONAL) {
    b0 = fma_s(-q.s2, A[1], fma_s(q.ss, A[3], q.cc * A[0]));
    b3 = fma_s(q.s2, A[1], fma_s(q.ss, A[0], q.cc * A[3]));
  } else {
    const S e = fma_s(-q.s2, A[1], q.ss * d);
    b0 = A[0] + e;
    b3 = A[3] - e;
  }
  const S B[6] = {b0, fma_s(-q.sc, d, q.c2 * A[1]), fma_s(-t.s, A[4], t.c * A[2]),
                  b3, fma_s(t.s, A[2], t.c * A[4]), A[5]};
  static_for<0, 3>([&](auto Ic) {
    constexpr int i = decltype(Ic)::value;
    S col[3];                                    // column i of B F
    static_for<0, 3>([&](auto Rc) {
      constexpr int r = decltype(Rc)::value;
      const S row[3] = {B[sym(r, 0)], B[sym(r, 1)], B[sym(r, 2)]};
      col[r] = fixed_t<K, i>(row);
    });
    static_for<0, i + 1>([&](auto Jc) {
      constexpr int j = decltype(Jc)::value;
      A[sym(j, i)] = fixed_t<K, j>(col);
    });
  });
}
// A += g (2 (r.h) 1 - h r^T - r h^T)
template <typename S>
RBD_HD RBD_INLINE void add_sym_outer(S g, S rx, S ry, S rz, const S* h, S A[6]) {
  const S gx = g * rx, gy = g * ry, gz = g * rz;
  A[0] = fma_s(S(2) * gy, h[1], fma_s(S(2) * gz, h[2], A[0]));
  A[3] = fma_s(S(2) * gx, h[0], fma_s(S(2) * gz, h[2], A[3]));
  A[5] = fma_s(S(2) * gx, h[0], fma_s(S(2) * gy, h[1], A[5]));
  A[1] = fma_s(-gx, h[1], fma_s(-gy, h[0], A[1]));
  A[2] = fma_s(-gx, h[2], fma_s(-gz, h[0], A[2]));
  A[4] = fma_s(-gy, h[2], fma_s(-gz, h[1], A[4]));
}

// ---------------------------------------------------------------------------
// Arithmetic precision per phase.  Inputs and outputs are FP32 in every mode.
//   Minv  : the articulated-body recursion for Minv
//   Pivot : the pivots D_k = S^T IA_k S and 1/D_k inside it
//   Rnea  : bias RNEA, qdd and the RNEA with qdd
//   Col   : the derivative columns dtau/d(q,qd) and -Minv dtau
// ---------------------------------------------------------------------------
//   HW_TRIG: FP32 sin/cos from the hardware's v_sin_f32/v_cos_f32 (knot_sincos)
template <typename SMinv, typename SPivot, typename SRnea, typename SCol, bool HW_TRIG = false>
struct Precision {
  using Minv = SMinv; using Pivot = SPivot; using Rnea = SRnea; using Col = SCol;
  static constexpr bool kHwTrig = HW_TRIG;
};
using PrecFP32      = Precision<float, float, float, float>;     // all FP32
using PrecFP32HwTrig = Precision<float, float, float, float, true>;  // all FP32, hardware sin/cos
using PrecFP64Pivot = Precision<float, double, float, float>;    // FP64 pivots only
using PrecFP64Col   = Precision<float, float, float, double>;    // FP64 derivative columns
using PrecFP64      = Precision<double, double, double, double>; // all FP64

// Waves each SIMD keeps resident for the kernels of precision P.  With FP32
// RNEA and columns a knot's state fits in 256 registers per lane, so two waves
// share a SIMD: a wave issues at most one instruction every 4 cycles, so two
// issue twice as many (and each hides the other's latency); with FP64 columns
// it needs 320 to 500 and runs one.
template <class P>
constexpr int kWavesPerSimd = (sizeof(typename P::Col) == 4 && sizeof(typename P::Rnea) == 4) ? 2 : 1;

// sin/cos of a joint angle under precision P: sincos_s, or, with P::kHwTrig and
// an FP32 angle, the hardware's v_sin_f32/v_cos_f32 (whose argument is in
// revolutions).  The angle is first reduced to [-pi, pi] as
// x - k 2pi with 2pi split into two FP32 parts (exact to about 2^-40 |x|), so
// small and large angles keep their precision.  Measured on MI355X: a call of
// 128 knots 4.37 us against 4.49, 2^20 knots 100.0 against 101.2, and the largest
// relative output error over 2^20 random and stretched-arm poses 4.5e-5 instead
// of 1.7e-5.  The host build uses the math library's in both.
template <class P, typename S>
RBD_HD RBD_INLINE void knot_sincos(S x, S* s, S* c) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (P::kHwTrig && std::is_same<S, float>::value) {
    constexpr double kTwoPi = 6.283185307179586476925286766559;
    constexpr float kHi = float(kTwoPi);
    constexpr float kLo = float(kTwoPi - double(kHi));
    constexpr float kInv = float(1.0 / kTwoPi);
    const float k = __builtin_rintf(x * kInv);
    const float a = __builtin_fmaf(-k, kLo, __builtin_fmaf(-k, kHi, x));
    *s = __builtin_amdgcn_sinf(a * kInv);
    *c = __builtin_amdgcn_cosf(a * kInv);
    return;
  }
#endif
  sincos_s(x, s, c);
}

// ---------------------------------------------------------------------------
// The mass matrix in factors, M = L^T D L with L unit lower triangular, from the
// articulated-body recursion: D_k = S^T IA_k S, the pivots of computeMinv
// (minv.h:423-478), and L[k][j] = S_j^T (IA_k S / D_k moved to link j).  A
// right-hand side costs the 49 multiply-adds of a product with Minv, and the
// recursion has neither the F columns nor the forward pass that forming Minv
// takes (about 700 instructions against 1,300); factoring the joint-space
// matrix from composite inertias would take fewer still but doubled the error
// of dqdd/dq (4.7e-7 against 2.2e-7 in FP32).
// The pivots D_k and 1/D_k are formed in SP (FP64 in the pivot variant).
// ---------------------------------------------------------------------------
template <typename S> struct MassFactors {
  S L[NQ][NQ];     // [k][j], j < k
  S dinv[NQ];
};

// 1 / x of a pivot
RBD_HD RBD_INLINE float reciprocal(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const float r = __builtin_amdgcn_rcpf(x);      // within one unit in the last place; a Newton step
  return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
#else
  return 1.0f / x;
#endif
}
RBD_HD RBD_INLINE double reciprocal(double x) { return 1.0 / x; }

// T^T Ia T of a symmetric Ia = [A C; C^T N] whose row and column 2 are zero (a
// revolute joint about z): A = (xx, xy, yy), C rows 0 and 1, N all six.  The
// 3x3 blocks are rotated (A' = E^T A E, C' = E^T C E, N' = E^T N E), then
// translated: TR = C' + r^ N', TL = A' + r^ C'^T - TR r^, BR = N'.
// (Same product as the reference's ctransform_Ia_revolute, minv.h:221-386.)
template <int K, typename S>
RBD_HD RBD_INLINE void move_articulated(const CS<S>& t, const S a[3], const S c[2][3], const S n[6], S TL[6],
                                        S TR[3][3], S BR[6]) {
  const DoubleAngle<S> q = double_angle(t);
  TL[0] = a[0]; TL[1] = a[1]; TL[3] = a[2]; TL[2] = S(0); TL[4] = S(0); TL[5] = S(0);
  sym_to_parent<K, true>(t, q, TL);
  for (int i = 0; i < 6; ++i) BR[i] = n[i];
  sym_to_parent<K, true>(t, q, BR);
  S r0[3], r1[3], C[3][3];                       // C E, then E^T (C E)
  to_parent<K>(t, c[0], r0);
  to_parent<K>(t, c[1], r1);
  static_for<0, 3>([&](auto Jc) {
    constexpr int j = decltype(Jc)::value;
    const S col[3] = {r0[j], r1[j], S(0)};
    S y[3];
    to_parent<K>(t, col, y);
    C[0][j] = y[0]; C[1][j] = y[1]; C[2][j] = y[2];
    const S b[3] = {BR[sym(0, j)], BR[sym(1, j)], BR[sym(2, j)]};
    add_offset_cross<K>(b, y);
    TR[0][j] = y[0]; TR[1][j] = y[1]; TR[2][j] = y[2];
  });
  // (r^ C'^T)_ij = (r x C'_j)_i, (TR r^)_ij = -(r x TR_i)_j, rows of C' and TR
  static_for<0, 3>([&](auto Ic) {
    constexpr int i = decltype(Ic)::value;
    static_for<i, 3>([&](auto Jc) {
      constexpr int j = decltype(Jc)::value;
      constexpr int i1 = (i + 1) % 3, i2 = (i + 2) % 3, j1 = (j + 1) % 3, j2 = (j + 2) % 3;
      TL[sym(i, j)] = fma_s(roff<K, S>(i1), C[j][i2], fma_s(-roff<K, S>(i2), C[j][i1],
                      fma_s(roff<K, S>(j1), TR[i][j2], fma_s(-roff<K, S>(j2), TR[i][j1], TL[sym(i, j)]))));
    });
  });
}

template <typename S, typename SP>
RBD_HD RBD_INLINE void mass_factors(const CS<S>* t, MassFactors<S>& f) {
  // articulated inertia of link k: [A C; C^T N]
  S A[6], C[3][3], N[6];
  static_for<0, 3>([&](auto Ic) {
    constexpr int i = decltype(Ic)::value;
    static_for<0, 3>([&](auto Jc) {
      constexpr int j = decltype(Jc)::value;
      C[i][j] = kInertia<S, NQ - 1, i, 3 + j>;
      if constexpr (j >= i) {
        A[sym(i, j)] = kInertia<S, NQ - 1, i, j>;
        N[sym(i, j)] = kInertia<S, NQ - 1, 3 + i, 3 + j>;
      }
    });
  });
  SP pivot = SP(kInertia<S, NQ - 1, 2, 2>);
  static_for_down<NQ, 0>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    f.dinv[k] = S(reciprocal(pivot));
    if constexpr (k > 0) {
      const S U[6] = {A[2], A[4], A[5], C[2][0], C[2][1], C[2][2]};      // IA S
      S W[6];                                                              // U / D
      for (int i = 0; i < 6; ++i) W[i] = i == 2 ? S(1) : U[i] * f.dinv[k];
      // IA - U U^T / D
      const S a[3] = {fma_s(-U[0], W[0], A[0]), fma_s(-U[0], W[1], A[1]), fma_s(-U[1], W[1], A[3])};
      S c[2][3], n[6];
      static_for<0, 3>([&](auto Jc) {
        constexpr int j = decltype(Jc)::value;
        c[0][j] = fma_s(-U[0], W[3 + j], C[0][j]);
        c[1][j] = fma_s(-U[1], W[3 + j], C[1][j]);
        static_for<0, j + 1>([&](auto Ic) {
          constexpr int i = decltype(Ic)::value;
          n[sym(i, j)] = fma_s(-U[3 + i], W[3 + j], N[sym(i, j)]);
        });
      });
      S TL[6], TR[3][3], BR[6];
      move_articulated<k>(t[k], a, c, n, TL, TR, BR);
      static_for<0, 3>([&](auto Ic) {
        constexpr int i = decltype(Ic)::value;
        static_for<0, 3>([&](auto Jc) {
          constexpr int j = decltype(Jc)::value;
          C[i][j] = TR[i][j] + kInertia<S, k - 1, i, 3 + j>;
          if constexpr (j >= i) {
            A[sym(i, j)] = TL[sym(i, j)] + kInertia<S, k - 1, i, j>;
            N[sym(i, j)] = BR[sym(i, j)] + kInertia<S, k - 1, 3 + i, 3 + j>;
          }
        });
      });
      if constexpr (sizeof(SP) > sizeof(S)) {
        // the next pivot formed in SP from the same (rounded) terms; only
        // entry (2, 2) of this second transport is live, the rest is dead code
        const SP aw[3] = {SP(a[0]), SP(a[1]), SP(a[2])};
        SP cw[2][3], nw[6], TLw[6], TRw[3][3], BRw[6];
        for (int j = 0; j < 3; ++j) { cw[0][j] = SP(c[0][j]); cw[1][j] = SP(c[1][j]); }
        for (int i = 0; i < 6; ++i) nw[i] = SP(n[i]);
        const CS<SP> tw{SP(t[k].c), SP(t[k].s)};
        move_articulated<k>(tw, aw, cw, nw, TLw, TRw, BRw);
        pivot = SP(inertia_entry(k - 1, 2, 2)) + TLw[5];
      } else {
        pivot = SP(A[5]);
      }
      static_for_down<k + 1, 1>([&](auto Jc) {
        constexpr int j = decltype(Jc)::value;   // W from link j to link j - 1
        move_force<j>(t[j], W);
        f.L[k][j - 1] = W[2];
      });
    }
  });
}

// x = M^-1 x, or -M^-1 x (NEG, a derivative column).  The back substitution of a
// solve sums its products first and takes them from y_k / D_k in one
// multiply-add, whose product is not rounded: y_k / D_k is often far above the
// result, and with the sum started from it every step rounds at its size
// (error of qdd in FP32 7.1e-8 of its norm, so 4.9e-8).  A derivative column is
// started from it all the same: it gains little (dqdd/dq 2.03e-7, so 1.98e-7),
// and with the sum beside y_k the one-lane kernels are a register short (external
// forces at 150,001 knots 24.6 us, so 26.0).
template <bool NEG, typename S, typename SX>
RBD_HD RBD_INLINE void mass_solve(const MassFactors<S>& f, SX x[NQ]) {
  static_for_down<NQ, 1>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    static_for<0, k>([&](auto Jc) {
      constexpr int j = decltype(Jc)::value;
      x[j] = fma_s(-SX(f.L[k][j]), x[k], x[j]);
    });
  });
  if constexpr (NEG) {
    for (int k = 0; k < NQ; ++k) x[k] = -x[k] * SX(f.dinv[k]);
    static_for<1, NQ>([&](auto Kc) {
      constexpr int k = decltype(Kc)::value;
      static_for<0, k>([&](auto Jc) {
        constexpr int j = decltype(Jc)::value;
        x[k] = fma_s(-SX(f.L[k][j]), x[j], x[k]);
      });
    });
  } else {
    x[0] *= SX(f.dinv[0]);
    static_for<1, NQ>([&](auto Kc) {
      constexpr int k = decltype(Kc)::value;
      SX sum = SX(f.L[k][0]) * x[0];
      static_for<1, k>([&](auto Jc) {
        constexpr int j = decltype(Jc)::value;
        sum = fma_s(SX(f.L[k][j]), x[j], sum);
      });
      x[k] = fma_s(x[k], SX(f.dinv[k]), -sum);
    });
  }
}

// Column j of Minv from the factors: col[k] = Minv[k][j] for k <= j (the
// entries below are formed too far only to k = j when J is a constant, and
// left unspecified).  The forward sums of links k > j are exactly zero, so the
// run-time j of the lane groups gives bitwise the entries of a constant j.  The
// products are summed first, as in mass_solve (error of Minv in FP32 5.6e-8 of
// its norm, so 3.8e-8).
template <int J, typename S>
RBD_HD RBD_INLINE void minv_column(const MassFactors<S>& f, int j, S col[NQ]) {
  constexpr int top = J < 0 ? NQ : J + 1;        // rows to form
  S y[NQ];
  static_for_down<top, 0>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    S acc = (J < 0 ? k == j : k == J) ? S(1) : S(0);
    static_for_down<top, k + 1>([&](auto Ic) {
      constexpr int i = decltype(Ic)::value;
      acc = fma_s(-f.L[i][k], y[i], acc);
    });
    y[k] = acc;
  });
  static_for<0, top>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    if constexpr (k == 0) {
      col[0] = y[0] * f.dinv[0];
    } else {
      S sum = f.L[k][0] * col[0];
      static_for<1, k>([&](auto Ic) {
        constexpr int i = decltype(Ic)::value;
        sum = fma_s(f.L[k][i], col[i], sum);
      });
      col[k] = fma_s(y[k], f.dinv[k], -sum);
    }
  });
}

// Minv (upper triangle, Mi[r][c] for r <= c)
template <typename S>
RBD_HD RBD_INLINE void minv_from_factors(const MassFactors<S>& f, S Mi[NQ][NQ]) {
  static_for<0, NQ>([&](auto Jc) {
    constexpr int j = decltype(Jc)::value;
    S col[NQ];
    minv_column<j>(f, j, col);
    for (int r = 0; r <= j; ++r) Mi[r][j] = col[r];
  });
}
template <typename S, typename SP>
RBD_HD RBD_INLINE void compute_minv(const CS<S>* t, S Mi[NQ][NQ]) {
  MassFactors<S> f;
  mass_factors<S, SP>(t, f);
  minv_from_factors(f, Mi);
}
// Column j of Minv, for a lane that computes one column (entries k > j are
// left unspecified).
template <typename S, typename SP>
RBD_HD RBD_INLINE void compute_minv_column(const CS<S>* t, int j, S col[NQ]) {
  MassFactors<S> f;
  mass_factors<S, SP>(t, f);
  minv_column<-1>(f, j, col);
}

// ---------------------------------------------------------------------------
// RNEA forward pass (RNEA_fp, dynamicsGradient.h:619-659): v, a, f per link.
// The gravity trick sets the base acceleration to +g along z.
// ---------------------------------------------------------------------------
template <typename S>
RBD_HD RBD_INLINE void rnea_fwd(const CS<S>* t, const S* qd, const S* qdd, S gravity,
                                S v[NQ][6], S a[NQ][6], S f[NQ][6]) {
  static_for<0, NQ>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    if constexpr (k == 0) {
      for (int i = 0; i < 6; ++i) { v[0][i] = S(0); a[0][i] = S(0); }
      v[0][2] = qd[0];
      a[0][2] = qdd[0];
      const S g[3] = {S(0), S(0), gravity};
      S ga[3];
      rot<0>(t[0], g, ga);                   // T_0 [0,0,0,0,0,g] = [0; E g]
      a[0][3] = ga[0]; a[0][4] = ga[1]; a[0][5] = ga[2];
    } else {
      xmotion<k>(t[k], v[k - 1], v[k]);
      v[k][2] += qd[k];
      xmotion<k>(t[k], a[k - 1], a[k]);
      a[k][0] += v[k][1] * qd[k];            // + (v x S) qd
      a[k][1] -= v[k][0] * qd[k];
      a[k][3] += v[k][4] * qd[k];
      a[k][4] -= v[k][3] * qd[k];
      a[k][2] += qdd[k];
    }
    S Iv[6];
    imv<k>(v[k], Iv);
    imv<k>(a[k], f[k]);                      // f = I a + v x* I v
    crf<true>(v[k], Iv, f[k]);
  });
}

// RNEA backward pass (RNEA_bp, dynamicsGradient.h:661-670): f_{k-1} += T^T f_k
template <typename S>
RBD_HD RBD_INLINE void rnea_bwd(const CS<S>* t, S f[NQ][6]) {
  static_for_down<NQ, 1>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    S y[6];
    xforce_t_add<k>(t[k], f[k], f[k - 1], y);
    for (int i = 0; i < 6; ++i) f[k - 1][i] = y[i];
  });
}

// External forces (RNEA_fp's s_fext, dynamicsGradient.h:654-657): f_k -= fext_k
// with fext_k link k's spatial force in its own frame at fx[6k .. 6k+5].  The
// input accessor's fx is null (a compile-time constant in the plain kernels,
// so this folds away) unless the call passes forces.
template <class In, typename S>
RBD_HD RBD_INLINE void subtract_fext(const In& in, S f[NQ][6]) {
  if (in.fx)
    for (int k = 0; k < NQ; ++k)
      for (int i = 0; i < 6; ++i) f[k][i] -= S(in.fx[6 * k + i]);
}

// ---------------------------------------------------------------------------
// One derivative column.  Forward sweep (compute_vafdu, dynamicsGradient.h:786-829)
// from link c: at k == c the seed is dv = S, da = v_c x S for d/dqd, and
// dv = v_c x S, da = a_c x S for d/dq (the reference's (T v_{c-1}) x S and
// (v x S) qd + (T a_{c-1}) x S reduce to these because S x S = 0);
// for k > c: dv = T dv, da = T da + (dv x S) qd_k.  Then
// df_k = I da + dv x* (I v_k) + v_k x* (I dv).
// Backward sweep (compute_cdu, :831-857): g_{k-1} = df_{k-1} + T^T g_k, with the
// extra T^T (-(f_k x S)) at k == c for d/dq; dtau_k = g_k[2].
// ---------------------------------------------------------------------------
// Written per link instead of as a recursion in (dv, da): with
// D_c = 2 v_c x S and P_c = a_c x S + v_c x (v_c x S), both moved to link k,
//   d/dq_c:   df_k = I_k P_c + B_k D_c
//   d/dqd_c:  df_k = I_k D_c + 2 B_k S
// with B_k = ((v_k x*) I_k - I_k (v_k x) + (. x* h_k)) / 2, h_k = I_k v_k the
// momentum.  B maps [w; u] to [(Bs - n^ / 2) w; -p x w] with Bs symmetric and
// (n, p) the momentum, so it sees only the angular part of its argument: a
// column takes 65 instructions a link and seed in place of 120, and its
// largest error is about half (dqdd/dqd 4.9e-7 against 8.2e-7 of the norm).
// first moment of link K (mass times centre of mass)
template <int K>
RBD_HD constexpr double first_moment(int i) {
  return i == 0 ? inertia_entry(K, 2, 4) : (i == 1 ? inertia_entry(K, 0, 5) : inertia_entry(K, 1, 3));
}
// Bs of link K alone at velocity v
template <int K, typename S>
RBD_HD RBD_INLINE void body_bs(const S* v, S B[6]) {
  constexpr double xx = inertia_entry(K, 0, 0), xy = inertia_entry(K, 0, 1), xz = inertia_entry(K, 0, 2),
                   yy = inertia_entry(K, 1, 1), yz = inertia_entry(K, 1, 2), zz = inertia_entry(K, 2, 2);
  const S w0 = v[0], w1 = v[1], w2 = v[2];
  B[0] = fma_s(S(xz), w1, S(-xy) * w2);
  B[3] = fma_s(S(xy), w2, S(-yz) * w0);
  B[5] = fma_s(S(yz), w0, S(-xz) * w1);
  B[1] = fma_s(S(0.5 * (xx - yy)), w2, fma_s(S(0.5 * yz), w1, S(-0.5 * xz) * w0));
  B[2] = fma_s(S(0.5 * (zz - xx)), w1, fma_s(S(-0.5 * yz), w2, S(0.5 * xy) * w0));
  B[4] = fma_s(S(0.5 * (yy - zz)), w0, fma_s(S(0.5 * xz), w2, S(-0.5 * xy) * w1));
  add_sym_outer<S>(S(0.5), S(first_moment<K>(0)), S(first_moment<K>(1)), S(first_moment<K>(2)), v + 3, B);
}

// D = 2 v x S (entries 2 and 5 are zero) and P = a x S + v x (v x S)
template <typename S>
RBD_HD RBD_INLINE void motion_pair(const S* v, const S* a, S D[6], S P[6]) {
  D[0] = v[1] + v[1]; D[1] = -(v[0] + v[0]); D[2] = S(0);
  D[3] = v[4] + v[4]; D[4] = -(v[3] + v[3]); D[5] = S(0);
  P[0] = fma_s(v[2], v[0], a[1]);
  P[1] = fma_s(v[2], v[1], -a[0]);
  P[2] = fma_s(-v[0], v[0], -(v[1] * v[1]));
  P[3] = fma_s(v[2], v[3], fma_s(v[5], v[0], a[4]));
  P[4] = fma_s(v[2], v[4], fma_s(v[5], v[1], -a[3]));
  P[5] = fma_s(D[1], v[3], -(D[0] * v[4]));
}

// What a column needs of each link besides its transform: Bs, P and D.  In FP32
// they are stored (a lane of a group runs up to four columns); in FP64, where
// they would take 280 registers more and the kernels spill, they are formed
// again from v and a in each column.
template <typename S, bool STORED = sizeof(S) == 4>
struct LinkTerms {
  S b[NQ][6], P[NQ][6], D[NQ][6];
  template <int K> RBD_HD RBD_INLINE void set(const S* v, const S* a) {
    body_bs<K>(v, b[K]);
    motion_pair(v, a, D[K], P[K]);
  }
  template <int K> RBD_HD RBD_INLINE void get(S bk[6], S Dk[6], S Pk[6]) const {
    for (int i = 0; i < 6; ++i) { bk[i] = b[K][i]; Dk[i] = D[K][i]; Pk[i] = P[K][i]; }
  }
  RBD_HD RBD_INLINE void forget() {}
};
template <typename S>
struct LinkTerms<S, false> {
  S v[NQ][6], a[NQ][6];
  template <int K> RBD_HD RBD_INLINE void set(const S* vk, const S* ak) {
    for (int i = 0; i < 6; ++i) { v[K][i] = vk[i]; a[K][i] = ak[i]; }
  }
  template <int K> RBD_HD RBD_INLINE void get(S bk[6], S Dk[6], S Pk[6]) const {
    body_bs<K>(v[K], bk);
    motion_pair(v[K], a[K], Dk, Pk);
  }
  // between two columns of a lane: keeps the compiler from holding the first
  // column's terms for the second
  RBD_HD RBD_INLINE void forget() {
#if defined(__HIP_DEVICE_COMPILE__)
    for (int k = 0; k < NQ; ++k)
      for (int i = 0; i < 6; ++i) asm volatile("" : "+v"(v[k][i]));
#endif
  }
};

template <typename S>
struct PhaseC {
  CS<S> t[NQ];
  LinkTerms<S> link;
  S n[NQ][3], p[NQ][3];   // momentum of each link
  S nfxs[NQ][4];   // -(f_k x S) -> (-f1, f0, -f4, f3)
  S Mi[NQ][NQ];    // upper triangle of Minv
};

// tau[c] += x for a run-time c without indexing a register array
template <typename S>
RBD_HD RBD_INLINE void add_on_diagonal(S tau[NQ], int c, S x) {
  static_for<0, NQ>([&](auto Rc) {
    constexpr int r = decltype(Rc)::value;
    tau[r] += (r == c) ? x : S(0);
  });
}

// out[r] = (Minv x)[r] (NEG: negated), Minv upper-stored
template <bool NEG, typename S, typename SX>
RBD_HD RBD_INLINE void minv_times(const S Mi[NQ][NQ], const SX x[NQ], SX out[NQ]) {
  static_for<0, NQ>([&](auto Rc) {
    constexpr int r = decltype(Rc)::value;
    SX acc = SX(0);
    static_for<0, NQ>([&](auto Cc) {
      constexpr int c = decltype(Cc)::value;
      acc += SX(r <= c ? Mi[r][c] : Mi[c][r]) * x[c];
    });
    out[r] = NEG ? -acc : acc;
  });
}

// dtau of one derivative column for lane-parallel use: the column c and its
// kind (dq) may differ from lane to lane while every lane executes the same
// instructions.  The moved vectors x (6) and w (the angular part that B sees)
// start at zero and stay zero until k == c, where the seed replaces them by
// select; the zero df_k for k < c then adds exactly nothing in the backward
// sweep.
template <typename S>
RBD_HD RBD_INLINE void dtau_column_uniform(const PhaseC<S>& P, int c, bool dq, S tau[NQ]) {
  S x[6], w[3], df[NQ][6];
  for (int i = 0; i < 6; ++i) x[i] = S(0);
  for (int i = 0; i < 3; ++i) w[i] = S(0);
  static_for<0, NQ>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    if constexpr (k > 0) {
      move_motion<k>(P.t[k], x, x);
      to_child<k>(P.t[k], w, w);
    }
    S b[6], Dk[6], Pk[6];
    P.link.template get<k>(b, Dk, Pk);
    const bool seed = (k == c);
    for (int i = 0; i < 6; ++i) x[i] = seed ? (dq ? Pk[i] : Dk[i]) : x[i];
    for (int i = 0; i < 3; ++i) w[i] = seed ? (dq ? Dk[i] : (i == 2 ? S(2) : S(0))) : w[i];
    inertia_times<k>(x, df[k]);
    const S* n = P.n[k]; const S* p = P.p[k];
    // += [(Bs - n^ / 2) w; -p x w], n^ w / 2 = n x w / 2
    const S h[3] = {S(0.5) * w[0], S(0.5) * w[1], S(0.5) * w[2]};
    df[k][0] = fma_s(b[0], w[0], fma_s(b[1], w[1], fma_s(b[2], w[2], fma_s(n[2], h[1], fma_s(-n[1], h[2], df[k][0])))));
    df[k][1] = fma_s(b[1], w[0], fma_s(b[3], w[1], fma_s(b[4], w[2], fma_s(n[0], h[2], fma_s(-n[2], h[0], df[k][1])))));
    df[k][2] = fma_s(b[2], w[0], fma_s(b[4], w[1], fma_s(b[5], w[2], fma_s(n[1], h[0], fma_s(-n[0], h[1], df[k][2])))));
    df[k][3] = fma_s(p[2], w[1], fma_s(-p[1], w[2], df[k][3]));
    df[k][4] = fma_s(p[0], w[2], fma_s(-p[2], w[0], df[k][4]));
    df[k][5] = fma_s(p[1], w[0], fma_s(-p[0], w[1], df[k][5]));
  });
  S g[6];
  for (int i = 0; i < 6; ++i) g[i] = df[NQ - 1][i];
  static_for_down<NQ, 1>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    tau[k] = g[2];
    const bool extra = dq && (k == c);
    g[0] += extra ? P.nfxs[k][0] : S(0); g[1] += extra ? P.nfxs[k][1] : S(0);
    g[3] += extra ? P.nfxs[k][2] : S(0); g[4] += extra ? P.nfxs[k][3] : S(0);
    add_moved_force<k>(P.t[k], g, df[k - 1]);
    for (int i = 0; i < 6; ++i) g[i] = df[k - 1][i];
  });
  tau[0] = g[2];
}

// Phase-C inputs from v, a (with qdd), f (after the backward pass) and Minv.
template <typename SC, typename SR, typename SM>
RBD_HD RBD_INLINE void make_phase_c(PhaseC<SC>& P, const CS<SC>* t, const SR v[NQ][6], const SR a[NQ][6],
                                    const SR f[NQ][6], const SM Mi[NQ][NQ]) {
  for (int k = 0; k < NQ; ++k) P.t[k] = t[k];
  for (int r = 0; r < NQ; ++r)
    for (int c = r; c < NQ; ++c) P.Mi[r][c] = SC(Mi[r][c]);
  static_for<0, NQ>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    SC vk[6], ak[6], h[6];
    for (int i = 0; i < 6; ++i) { vk[i] = SC(v[k][i]); ak[i] = SC(a[k][i]); }
    inertia_times<k>(vk, h);
    for (int i = 0; i < 3; ++i) { P.n[k][i] = h[i]; P.p[k][i] = h[3 + i]; }
    P.link.template set<k>(vk, ak);
    P.nfxs[k][0] = -SC(f[k][1]); P.nfxs[k][1] = SC(f[k][0]); P.nfxs[k][2] = -SC(f[k][4]); P.nfxs[k][3] = SC(f[k][3]);
  });
}

// ---------------------------------------------------------------------------
// All derivative columns in one lane, from composite quantities.
//
// In df_k above only I_k and B_k depend on the link, so the backward sweep's
// sum over the links from c on is a product with their composite inertia IC_c
// and composite B_c.  Both composites are a few numbers: IC six and three
// (its mass is a constant), B six and the composite momentum.  Going from the
// tip to the base, link c gives
//   rows j <= c of column c:  S_j . (IC P + B D + S x* f) and S_j . (IC D + 2 B S),
//   columns j < c of row c:   (IC S) . P_j + (B^T S) . D_j and (IC S) . D_j + 2 (B^T S) . S_j
// where the four force vectors (the last a pure couple) are moved down the
// links j < c.  That is 21 moves of three and a half vectors in place of the
// thirteen columns' sweeps over up to seven links forward and back (2,300
// instructions against 3,700; Singh, Russell and Wensing, "Efficient
// analytical derivatives of rigid-body dynamics using spatial vector
// algebra", 2022, give the world-frame form).
// ---------------------------------------------------------------------------
// mass of the links from K on
template <int K>
RBD_HD constexpr double composite_mass() {
  double m = 0.0;
  for (int j = K; j < NQ; ++j) m += inertia_entry(j, 3, 3);
  return m;
}
template <typename S> struct Composite {
  S i[6], h[3];    // composite inertia: about the link's origin, first moment
  S b[6];          // Bs
  S n[3], p[3];    // momentum
  S f[6];          // force on the link from the links from here on
};

// Link K joins the composite, which moves from link K + 1's frame to its own.
// f_given: the force on the link (the reference's split layout) instead of
// the composite's own sum.
template <int K, bool F_GIVEN, class In, typename S>
RBD_HD RBD_INLINE void composite_step(const In& in, const CS<S>* t, const S* v, const S* a, Composite<S>& c) {
  S h[6], B[6];
  inertia_times<K>(v, h);
  body_bs<K>(v, B);
  S f[6];
  if constexpr (F_GIVEN) {
    for (int i = 0; i < 6; ++i) f[i] = S(in.f(K, i));
  } else {
    inertia_times<K>(a, f);
    add_force_cross(v, h, f);
    if (in.fx)
      for (int i = 0; i < 6; ++i) f[i] -= S(in.fx[6 * K + i]);
  }
  if constexpr (K == NQ - 1) {
    static_for<0, 3>([&](auto Ic) {
      constexpr int i = decltype(Ic)::value;
      static_for<i, 3>([&](auto Jc) {
        constexpr int j = decltype(Jc)::value;
        c.i[sym(i, j)] = kInertia<S, K, i, j>;
      });
      c.h[i] = S(first_moment<K>(i));
      c.n[i] = h[i];
      c.p[i] = h[3 + i];
    });
    for (int i = 0; i < 6; ++i) { c.b[i] = B[i]; c.f[i] = f[i]; }
  } else {
    constexpr int u = K + 1;
    constexpr double r[3] = {kJointOffset[u][0], kJointOffset[u][1], kJointOffset[u][2]};
    constexpr double m = composite_mass<u>();
    constexpr double rr = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
    const DoubleAngle<S> q = double_angle(t[u]);
    // inertia about the new origin: i + 2 (r.h) 1 - h r^T - r h^T + m (r.r 1 - r r^T), then the link's own
    to_parent<u>(t[u], c.h, c.h);
    sym_to_parent<u, false>(t[u], q, c.i);
    add_sym_outer<S>(S(1), S(r[0]), S(r[1]), S(r[2]), c.h, c.i);
    static_for<0, 3>([&](auto Ic) {
      constexpr int i = decltype(Ic)::value;
      constexpr double hk = m * r[i] + first_moment<K>(i);
      c.h[i] += S(hk);
      static_for<i, 3>([&](auto Jc) {
        constexpr int j = decltype(Jc)::value;
        constexpr double ik = inertia_entry(K, i, j) + m * ((i == j ? rr : 0.0) - r[i] * r[j]);
        c.i[sym(i, j)] += S(ik);
      });
    });
    // Bs likewise with the momentum p in h's place; the momentum moves as a force
    to_parent<u>(t[u], c.p, c.p);
    sym_to_parent<u, false>(t[u], q, c.b);
    add_sym_outer<S>(S(0.5), S(r[0]), S(r[1]), S(r[2]), c.p, c.b);
    for (int i = 0; i < 6; ++i) c.b[i] += B[i];
    to_parent_add<u>(t[u], c.n, h, c.n);
    add_offset_cross<u>(c.p, c.n);
    for (int i = 0; i < 3; ++i) c.p[i] += h[3 + i];
    if constexpr (!F_GIVEN) add_moved_force<u>(t[u], c.f, f);
    for (int i = 0; i < 6; ++i) c.f[i] = f[i];
  }
}

// The columns from the tip's to the base's: emit(IC<c>, dtau/dq_c, dtau/dqd_c)
// (the d/dq column 0 is identically zero: rotation about the gravity axis).
template <bool F_GIVEN = false, class In, typename S, class Emit>
RBD_HD RBD_INLINE void derivative_columns(const In& in, const CS<S>* t, const S v[NQ][6], const S a[NQ][6],
                                          Emit&& emit) {
  S tq[NQ][NQ], td[NQ][NQ];        // dtau/dq, dtau/dqd: [row][column]
  Composite<S> c;
  static_for_down<NQ, 0>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    constexpr S m = S(composite_mass<k>());
    composite_step<k, F_GIVEN>(in, t, v[k], a[k], c);
    const S b01 = fma_s(S(0.5), c.n[2], c.b[1]), b10 = fma_s(S(-0.5), c.n[2], c.b[1]);
    const S b02 = fma_s(S(-0.5), c.n[1], c.b[2]), b20 = fma_s(S(0.5), c.n[1], c.b[2]);
    const S b12 = fma_s(S(0.5), c.n[0], c.b[4]), b21 = fma_s(S(-0.5), c.n[0], c.b[4]);
    S D[6], P[6];
    motion_pair(v[k], a[k], D, P);
    S is[6] = {c.i[2], c.i[4], c.i[5], -c.h[1], c.h[0], S(0)};       // IC S
    S bs[3] = {b20, b21, c.b[5]};                                    // B^T S
    S g[6], gd[6];                                                    // IC P + B D + S x* f, IC D + 2 B S
    gd[0] = fma_s(c.i[0], D[0], fma_s(c.i[1], D[1], fma_s(-c.h[2], D[4], S(2) * b02)));
    gd[1] = fma_s(c.i[1], D[0], fma_s(c.i[3], D[1], fma_s(c.h[2], D[3], S(2) * b12)));
    gd[2] = fma_s(c.i[2], D[0], fma_s(c.i[4], D[1], fma_s(c.h[0], D[4], fma_s(-c.h[1], D[3], S(2) * c.b[5]))));
    gd[3] = fma_s(m, D[3], fma_s(c.h[2], D[1], S(-2) * c.p[1]));
    gd[4] = fma_s(m, D[4], fma_s(-c.h[2], D[0], S(2) * c.p[0]));
    gd[5] = fma_s(c.h[1], D[0], -(c.h[0] * D[1]));
    td[k][k] = gd[2];
    if constexpr (k > 0) {
      g[0] = fma_s(c.i[0], P[0], fma_s(c.i[1], P[1], fma_s(c.i[2], P[2], fma_s(c.h[1], P[5], fma_s(-c.h[2], P[4],
             fma_s(c.b[0], D[0], fma_s(b01, D[1], -c.f[1])))))));
      g[1] = fma_s(c.i[1], P[0], fma_s(c.i[3], P[1], fma_s(c.i[4], P[2], fma_s(c.h[2], P[3], fma_s(-c.h[0], P[5],
             fma_s(b10, D[0], fma_s(c.b[3], D[1], c.f[0])))))));
      g[2] = fma_s(c.i[2], P[0], fma_s(c.i[4], P[1], fma_s(c.i[5], P[2], fma_s(c.h[0], P[4], fma_s(-c.h[1], P[3],
             fma_s(b20, D[0], b21 * D[1]))))));
      g[3] = fma_s(m, P[3], fma_s(c.h[2], P[1], fma_s(-c.h[1], P[2], fma_s(c.p[2], D[1], -c.f[4]))));
      g[4] = fma_s(m, P[4], fma_s(c.h[0], P[2], fma_s(-c.h[2], P[0], fma_s(-c.p[2], D[0], c.f[3]))));
      g[5] = fma_s(m, P[5], fma_s(c.h[1], P[0], fma_s(-c.h[0], P[1], fma_s(c.p[1], D[0], -(c.p[0] * D[1])))));
      tq[k][k] = g[2];
      static_for_down<k + 1, 1>([&](auto Uc) {
        constexpr int u = decltype(Uc)::value, j = u - 1;             // from link u to link j
        move_force<u>(t[u], g);
        move_force<u>(t[u], gd);
        move_force<u>(t[u], is);
        to_parent<u>(t[u], bs, bs);
        tq[j][k] = g[2];
        td[j][k] = gd[2];
        if constexpr (j > 0 || F_GIVEN) {
          S Dj[6], Pj[6];
          motion_pair(v[j], a[j], Dj, Pj);
          td[k][j] = fma_s(is[0], Dj[0], fma_s(is[1], Dj[1], fma_s(is[3], Dj[3], fma_s(is[4], Dj[4], S(2) * bs[2]))));
          if constexpr (j > 0)
            tq[k][j] = fma_s(is[0], Pj[0], fma_s(is[1], Pj[1], fma_s(is[2], Pj[2], fma_s(is[3], Pj[3],
                       fma_s(is[4], Pj[4], fma_s(is[5], Pj[5], fma_s(bs[0], Dj[0], bs[1] * Dj[1])))))));
        } else {
          // link 0 only turns, D_0 = 0; where the velocities are given they may
          // be those of an arm on a moving base
          td[k][0] = S(2) * bs[2];
        }
      });
    }
    S cq[NQ], cd[NQ];
    static_for<0, NQ>([&](auto Rc) {
      constexpr int r = decltype(Rc)::value;
      if constexpr (k > 0) cq[r] = tq[r][k];
      else cq[r] = S(0);
      cd[r] = td[r][k];
    });
    emit(Kc, cq, cd);
  });
}

// Link velocities and accelerations in one lane (RNEA_fp's recursions,
// dynamicsGradient.h:619-659); qdd null: zero joint accelerations.
template <typename S>
RBD_HD RBD_INLINE void link_motion(const CS<S>* t, const S* qd, const S* qdd, S gravity, S v[NQ][6], S a[NQ][6]) {
  static_for<0, NQ>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    if constexpr (k == 0) {
      for (int i = 0; i < 6; ++i) { v[0][i] = S(0); a[0][i] = S(0); }
      v[0][2] = qd[0];
      const S g[3] = {S(0), S(0), gravity};
      to_child<0>(t[0], g, a[0] + 3);              // T_0 [0,0,0,0,0,g] = [0; E g]
    } else {
      move_motion<k>(t[k], v[k - 1], v[k]);
      v[k][2] += qd[k];
      move_motion<k>(t[k], a[k - 1], a[k]);
      a[k][0] = fma_s(v[k][1], qd[k], a[k][0]);    // + (v x S) qd
      a[k][1] = fma_s(-v[k][0], qd[k], a[k][1]);
      a[k][3] = fma_s(v[k][4], qd[k], a[k][3]);
      a[k][4] = fma_s(-v[k][3], qd[k], a[k][4]);
    }
    if (qdd) a[k][2] += qdd[k];
  });
}
// a += the accelerations that qdd adds
template <typename S>
RBD_HD RBD_INLINE void add_joint_accelerations(const CS<S>* t, const S* qdd, S a[NQ][6]) {
  S d[6] = {S(0), S(0), qdd[0], S(0), S(0), S(0)};
  a[0][2] += qdd[0];
  static_for<1, NQ>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    move_motion<k>(t[k], d, d);
    d[2] += qdd[k];
    for (int i = 0; i < 6; ++i) a[k][i] += d[i];
  });
}
// Link forces and joint torques of a motion, from the tip (RNEA_bp,
// dynamicsGradient.h:661-670): sink(IC<k>, the force on link k), its entry 2 the torque
template <class In, typename S, class Sink>
RBD_HD RBD_INLINE void link_forces(const In& in, const CS<S>* t, const S v[NQ][6], const S a[NQ][6], Sink&& sink) {
  S f[6];
  static_for_down<NQ, 0>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    S h[6], b[6];
    inertia_times<k>(v[k], h);
    inertia_times<k>(a[k], b);
    add_force_cross(v[k], h, b);
    if (in.fx)
      for (int i = 0; i < 6; ++i) b[i] -= S(in.fx[6 * k + i]);
    if constexpr (k < NQ - 1) add_moved_force<k + 1>(t[k + 1], f, b);
    for (int i = 0; i < 6; ++i) f[i] = b[i];
    sink(Kc, f);
  });
}

// The columns' last step and their stores: times -Minv through the factors of
// M, times a given -Minv (upper triangle), or none (the inverse-dynamics
// gradient itself, the reference's cdu).
template <typename S> struct TimesMassInverse {
  const MassFactors<S>& f;
  template <typename SX> RBD_HD RBD_INLINE void operator()(SX x[NQ]) const { mass_solve<true>(f, x); }
};
template <typename S> struct TimesMinv {
  const S (*Mi)[NQ];
  template <typename SX> RBD_HD RBD_INLINE void operator()(SX x[NQ]) const {
    SX y[NQ];
    static_for<0, NQ>([&](auto Rc) {
      constexpr int r = decltype(Rc)::value;
      SX acc = -SX(Mi[0][r]) * x[0];
      static_for<1, NQ>([&](auto Cc) {
        constexpr int c = decltype(Cc)::value;
        acc = fma_s(-SX(r <= c ? Mi[r][c] : Mi[c][r]), x[c], acc);
      });
      y[r] = acc;
    });
    for (int r = 0; r < NQ; ++r) x[r] = y[r];
  }
};
struct TimesNothing {
  template <typename SX> RBD_HD RBD_INLINE void operator()(SX*) const {}
};
template <bool F_GIVEN = false, class In, typename S, class Times, class Out>
RBD_HD RBD_INLINE void gradient_columns(const In& in, const CS<S>* t, const S v[NQ][6], const S a[NQ][6],
                                        float damping, const Times& times, Out& out) {
  derivative_columns<F_GIVEN>(in, t, v, a, [&](auto Cc, S* cq, S* cd) {
    constexpr int c = decltype(Cc)::value;
    cd[c] += S(damping);
    times(cd);
    if constexpr (c > 0) times(cq);
    static_for<0, NQ>([&](auto Rc) {
      constexpr int r = decltype(Rc)::value;
      out.dq(r, c, float(cq[r]));
    });
    static_for<0, NQ>([&](auto Rc) {
      constexpr int r = decltype(Rc)::value;
      out.dqd(r, c, float(cd[r]));
    });
  });
}

// Lane roles when one knot is spread over a group of kLanesPerKnotGroup lanes:
// role j < 7: d/dqd column j; 7 <= j < 13: d/dq column j - 6; j == 13: qdd and
// the zero d/dq column 0; j >= 14: no stores.
constexpr int kLanesPerKnotGroup = 16;
constexpr int kRoleQdd = 13;

// One derivative column for lane role `role` of a knot group and its store
// (MINV as in gradient_columns).
template <bool MINV = true, typename SC, class Out>
RBD_HD RBD_INLINE void gradient_column_lane(const PhaseC<SC>& P, float damping, int role, Out& out) {
  const bool dq = role >= NQ;
  const int c = dq ? role - (NQ - 1) : role;
  SC tau[NQ], col[NQ];
  dtau_column_uniform(P, c, dq, tau);
  add_on_diagonal(tau, dq ? -1 : c, SC(damping));
  if constexpr (MINV) minv_times<true>(P.Mi, tau, col);
  else for (int r = 0; r < NQ; ++r) col[r] = tau[r];
  if (role < NQ) {
    for (int r = 0; r < NQ; ++r) out.dqd(r, c, float(col[r]));
  } else if (role < 2 * NQ - 1) {
    for (int r = 0; r < NQ; ++r) out.dq(r, c, float(col[r]));
  }
}

// Largest of two scalar types
template <typename A, typename B>
using Wider = typename std::conditional<(sizeof(A) >= sizeof(B)), A, B>::type;

// ---------------------------------------------------------------------------
// Accessors.  In: q(i), qd(i), u(i) [, qdd(i), minv(r, c) in the reference-
// compatible mode].  Out: qdd(i, x), dq(r, c, x), dqd(r, c, x).  All FP32.
// ---------------------------------------------------------------------------

// Run-time model options (the reference's compile-time VEL_DAMPING and MPC_MODE),
// and the bound on the two-wave mapping's LDS handoff waits.
struct Options {
  float damping = 0.0f;               // joint viscous damping: 0.5 with VEL_DAMPING (dynamicsGradient.h:680,840)
  float gravity = float(kGravity);    // 0 in MPC_MODE (dynamicsGradient.h:635-637)
  // A handoff wait polls its flag at most handoff_spins + 1 times, with a
  // short sleep between polls (2^24 sleeps of 64 cycles: about half a second);
  // a negative value makes every wait give up at once.  A wait that gives up
  // writes 1 to *fault, a word the host can read (null: nowhere), and the
  // kernel carries on and exits normally; its results are then invalid.
  unsigned* fault = nullptr;
  int handoff_spins = 1 << 24;
};

// The bounded wait of a handoff, for any poll and pause: true when poll()
// returned true within spins + 1 polls; false at once for spins < 0.
template <class Poll, class Pause>
RBD_HD RBD_INLINE bool bounded_wait(Poll&& poll, Pause&& pause, int spins) {
  if (spins < 0) return false;
  for (int spin = 0;; ++spin) {
    if (poll()) return true;
    if (spin >= spins) return false;
    pause();
  }
}

// sin/cos type of the full path: computed once in the widest arithmetic type
template <class P>
using KnotTrig = Wider<typename P::Minv, Wider<typename P::Rnea, typename P::Col>>;

// sin/cos of a knot's joints in one lane, in type ST
template <class P, typename ST, class In>
RBD_HD RBD_INLINE void knot_trig_in(P, const In& in, CS<ST> tw[NQ]) {
  for (int k = 0; k < NQ; ++k) {
    ST s, c;
    knot_sincos<P>(ST(in.q(k)), &s, &c);
    tw[k] = CS<ST>{c, s};
  }
}
template <class P, class In>
RBD_HD RBD_INLINE void knot_trig(const In& in, CS<KnotTrig<P>> tw[NQ]) { knot_trig_in(P{}, in, tw); }

// The same for a knot's lane group: lane role j < 7 computes the sin/cos of
// q_j alone and the group's lanes read all seven from each other by
// shuffles, instead of every lane computing all seven (a sincos is about 100
// instructions).  The values are those of knot_trig; the host build, which
// runs the lane roles one after another, calls knot_trig.
template <class P, class In>
RBD_HD RBD_INLINE void knot_trig_group(const In& in, int role, CS<KnotTrig<P>> tw[NQ]) {
#if defined(__HIP_DEVICE_COMPILE__)
  using ST = KnotTrig<P>;
  ST s, c;
  knot_sincos<P>(ST(in.q(role < NQ ? role : 0)), &s, &c);
  for (int k = 0; k < NQ; ++k) tw[k] = CS<ST>{__shfl(c, k, kLanesPerKnotGroup), __shfl(s, k, kLanesPerKnotGroup)};
#else
  (void)role;
  knot_trig<P>(in, tw);
#endif
}

// Steps 2-5 of the full path, given sin/cos and Minv: bias RNEA, qdd = Minv
// (u - c), RNEA with qdd; fills the phase-C inputs and qdd.
template <class P, class In>
RBD_HD RBD_INLINE void phase_a_after_minv(const In& in, const Options& opt, const CS<KnotTrig<P>> tw[NQ],
                                          const typename P::Minv Mi[NQ][NQ], PhaseC<typename P::Col>& PC,
                                          typename P::Rnea qdd[NQ]) {
  using SR = typename P::Rnea; using SC = typename P::Col;
  CS<SR> tr[NQ]; CS<SC> tc[NQ];
  SR qd[NQ], u[NQ];
  for (int k = 0; k < NQ; ++k) {
    tr[k] = CS<SR>{SR(tw[k].c), SR(tw[k].s)}; tc[k] = CS<SC>{SC(tw[k].c), SC(tw[k].s)};
    qd[k] = SR(in.qd(k));
    u[k] = SR(in.u(k));
  }
  // bias: RNEA with qdd = 0
  SR v[NQ][6], a[NQ][6], f[NQ][6];
  const SR zero[NQ] = {SR(0), SR(0), SR(0), SR(0), SR(0), SR(0), SR(0)};
  rnea_fwd(tr, qd, zero, SR(opt.gravity), v, a, f);
  subtract_fext(in, f);
  rnea_bwd(tr, f);
  SR bias[NQ];
  for (int k = 0; k < NQ; ++k) bias[k] = u[k] - f[k][2] - SR(opt.damping) * qd[k];
  minv_times<false>(Mi, bias, qdd);
  // RNEA with qdd, added incrementally: a += da, f += bwd(I da), da_k = T da_{k-1} + S qdd_k
  {
    SR dA[6] = {SR(0), SR(0), qdd[0], SR(0), SR(0), SR(0)};
    SR dF[NQ][6];
    static_for<0, NQ>([&](auto Kc) {
      constexpr int k = decltype(Kc)::value;
      if constexpr (k > 0) {
        SR y[6];
        xmotion<k>(tr[k], dA, y);
        for (int i = 0; i < 6; ++i) dA[i] = y[i];
        dA[2] += qdd[k];
      }
      for (int i = 0; i < 6; ++i) a[k][i] += dA[i];
      imv<k>(dA, dF[k]);
    });
    rnea_bwd(tr, dF);
    for (int k = 0; k < NQ; ++k)
      for (int i = 0; i < 6; ++i) f[k][i] += dF[k][i];
  }
  make_phase_c(PC, tc, v, a, f, Mi);
}

// Steps 1 and 5 of the reference-compatible modes: qdd given, and with
// WITH_MINV the dense Minv too (otherwise PC.Mi is left zero and unused).
template <class P, bool WITH_MINV = true, class In>
RBD_HD RBD_INLINE void phase_a_given_qdd_minv(const In& in, const Options& opt, PhaseC<typename P::Col>& PC) {
  using SR = typename P::Rnea; using SC = typename P::Col;
  using ST = Wider<SR, SC>;
  CS<SR> tr[NQ]; CS<SC> tc[NQ];
  SR qd[NQ], qdd[NQ];
  CS<ST> tw[NQ];
  knot_trig_in(P{}, in, tw);
  for (int k = 0; k < NQ; ++k) {
    tr[k] = CS<SR>{SR(tw[k].c), SR(tw[k].s)}; tc[k] = CS<SC>{SC(tw[k].c), SC(tw[k].s)};
    qd[k] = SR(in.qd(k));
    qdd[k] = SR(in.qdd(k));
  }
  SC Mi[NQ][NQ];
  for (int r = 0; r < NQ; ++r)
    for (int c = r; c < NQ; ++c) {
      if constexpr (WITH_MINV) Mi[r][c] = SC(in.minv(r, c));
      else Mi[r][c] = SC(0);
    }
  SR v[NQ][6], a[NQ][6], f[NQ][6];
  rnea_fwd(tr, qd, qdd, SR(opt.gravity), v, a, f);
  subtract_fext(in, f);
  rnea_bwd(tr, f);
  make_phase_c(PC, tc, v, a, f, Mi);
}

// Output accessors that also want dqdd/du = Minv (dense) declare kMinv = true.
template <class Out, class = void> struct WantsMinv { static constexpr bool value = false; };
template <class Out> struct WantsMinv<Out, typename std::enable_if<Out::kMinv>::type> {
  static constexpr bool value = true;
};

// Those that want to know when Minv is complete, before anything else is
// stored, have a minv_done().
template <class Out, class = void> struct StagesMinv { static constexpr bool value = false; };
template <class Out> struct StagesMinv<Out, decltype(static_cast<const Out*>(nullptr)->minv_done())> {
  static constexpr bool value = true;
};

// column c of the symmetric Minv (upper-stored) to out.minv
template <class Out, typename S>
RBD_HD RBD_INLINE void store_minv_column(Out& out, const S Mi[NQ][NQ], int c) {
  static_for<0, NQ>([&](auto Rc) {
    constexpr int r = decltype(Rc)::value;
    S m = S(0);
    static_for<0, NQ>([&](auto Cc) {
      constexpr int cc = decltype(Cc)::value;
      m = (cc == c) ? (r <= cc ? Mi[r][cc] : Mi[cc][r]) : m;
    });
    out.minv(r, c, float(m));
  });
}

// sin/cos in the type S of a phase
template <typename S, typename ST>
RBD_HD RBD_INLINE void cast_trig(const CS<ST> tw[NQ], CS<S> t[NQ]) {
  for (int k = 0; k < NQ; ++k) t[k] = CS<S>{S(tw[k].c), S(tw[k].s)};
}

// Steps 1-4 of the full path in one lane: sin/cos, the factors of M, bias RNEA,
// qdd = M^-1 (u - c); v and a (the latter at qdd = 0) for the gradient.
template <class P, class In>
RBD_HD RBD_INLINE void knot_forward_dynamics(const In& in, const Options& opt, const CS<KnotTrig<P>> tw[NQ],
                                             MassFactors<typename P::Minv>& f, typename P::Rnea v[NQ][6],
                                             typename P::Rnea a[NQ][6], typename P::Rnea qdd[NQ]) {
  using SM = typename P::Minv; using SP = typename P::Pivot; using SR = typename P::Rnea;
  CS<SM> tm[NQ]; CS<SR> tr[NQ];
  cast_trig(tw, tm);
  cast_trig(tw, tr);
  mass_factors<SM, SP>(tm, f);
  SR qd[NQ];
  for (int k = 0; k < NQ; ++k) qd[k] = SR(in.qd(k));
  link_motion(tr, qd, static_cast<const SR*>(nullptr), SR(opt.gravity), v, a);
  link_forces(in, tr, v, a, [&](auto Kc, const SR* fk) {
    constexpr int k = decltype(Kc)::value;
    qdd[k] = fma_s(-SR(opt.damping), qd[k], SR(in.u(k)) - fk[2]);
  });
  mass_solve<false>(f, qdd);
}

// Minv (dense) to out.minv
template <class Out, typename S>
RBD_HD RBD_INLINE void store_minv(Out& out, const MassFactors<S>& f) {
  S Mi[NQ][NQ];
  minv_from_factors(f, Mi);
  static_for<0, NQ>([&](auto Cc) {
    constexpr int c = decltype(Cc)::value;
    static_for<0, NQ>([&](auto Rc) {
      constexpr int r = decltype(Rc)::value;
      out.minv(r, c, float(r <= c ? Mi[r][c] : Mi[c][r]));
    });
  });
}

// Full path for one knot in one lane.  P: arithmetic precision per phase.
template <class P = PrecFP32, class In, class Out>
RBD_HD RBD_INLINE void fdgrad_knot(const In& in, Out& out, const Options& opt) {
  using SM = typename P::Minv; using SR = typename P::Rnea; using SC = typename P::Col;
  CS<KnotTrig<P>> tw[NQ];
  knot_trig<P>(in, tw);
  MassFactors<SM> f;
  SR v[NQ][6], a[NQ][6], qdd[NQ];
  knot_forward_dynamics<P>(in, opt, tw, f, v, a, qdd);
  if constexpr (WantsMinv<Out>::value) {
    store_minv(out, f);
    if constexpr (StagesMinv<Out>::value) out.minv_done();
  }
  for (int r = 0; r < NQ; ++r) out.qdd(r, float(qdd[r]));
  CS<SR> tr[NQ];
  cast_trig(tw, tr);
  add_joint_accelerations(tr, qdd, a);
  const TimesMassInverse<SM> times{f};
  if constexpr (std::is_same<SR, SC>::value) {
    gradient_columns(in, tr, v, a, opt.damping, times, out);
  } else {
    CS<SC> tc[NQ];
    SC vc[NQ][6], ac[NQ][6];
    cast_trig(tw, tc);
    for (int k = 0; k < NQ; ++k)
      for (int i = 0; i < 6; ++i) { vc[k][i] = SC(v[k][i]); ac[k][i] = SC(a[k][i]); }
    gradient_columns(in, tc, vc, ac, opt.damping, times, out);
  }
}

// Forward dynamics only: qdd = FD(q, qd, u) and the dense Minv, one lane per
// knot (forwardDynamics with DENSE_MINV, dynamicsGradient.h:685-706, :936-939,
// with the bias RNEA at qdd = 0).
template <class P = PrecFP32, class In, class Out>
RBD_HD RBD_INLINE void fd_knot(const In& in, Out& out, const Options& opt) {
  using SM = typename P::Minv; using SR = typename P::Rnea;
  CS<KnotTrig<P>> tw[NQ];
  knot_trig<P>(in, tw);
  MassFactors<SM> f;
  SR v[NQ][6], a[NQ][6], qdd[NQ];
  knot_forward_dynamics<P>(in, opt, tw, f, v, a, qdd);
  for (int r = 0; r < NQ; ++r) out.qdd(r, float(qdd[r]));
  store_minv(out, f);
}

// Minv of a knot shared by its lane group: the packed upper triangle
// (upper_index), in LDS in the kernels.
constexpr int kMinvPacked = NQ * (NQ + 1) / 2;

// index of (r, c), r <= c, in the packed upper triangle
RBD_HD constexpr int upper_index(int r, int c) { return r * NQ - r * (r - 1) / 2 + (c - r); }

// Lanes of one wave see each other's LDS writes made before this point.  The
// fences order the LDS accesses of the wave (they cost no instruction); in the
// host build, which runs the lane roles of a stage one after another, there
// is nothing to do.
RBD_HD RBD_INLINE void wave_lds_sync() {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
#endif
}

// Lane-group stage 1: sin/cos (kept in tw for stage 2) and lane role's column
// of Minv (roles 0..6), its upper entries stored into the group's mi.
template <class P, class In>
RBD_HD RBD_INLINE void lanes_minv_stage(const In& in, int role, CS<KnotTrig<P>> tw[NQ], typename P::Minv* mi) {
  using SM = typename P::Minv; using SP = typename P::Pivot;
  knot_trig_group<P>(in, role, tw);
  CS<SM> tm[NQ];
  for (int k = 0; k < NQ; ++k) tm[k] = CS<SM>{SM(tw[k].c), SM(tw[k].s)};
  const int j = role < NQ ? role : NQ - 1;
  SM col[NQ];
  compute_minv_column<SM, SP>(tm, j, col);
  if (role < NQ)
    for (int k = 0; k < NQ; ++k)
      if (k <= j) mi[upper_index(k, j)] = col[k];
}

// Minv (upper triangle) from a group's packed mi
template <typename S>
RBD_HD RBD_INLINE void load_packed_minv(const S* mi, S Mi[NQ][NQ]) {
  static_for<0, NQ>([&](auto Rc) {
    constexpr int r = decltype(Rc)::value;
    static_for<r, NQ>([&](auto Cc) {
      constexpr int c = decltype(Cc)::value;
      Mi[r][c] = mi[upper_index(r, c)];
    });
  });
}

// Lane-group stage 2 (after every lane's stage 1): steps 2-5 with the shared
// Minv (identical values in every lane), then lane `role` computes one
// derivative column (steps 6-7) and stores it.
template <class P, class In, class Out>
RBD_HD RBD_INLINE void lanes_finish_stage(const In& in, Out& out, const Options& opt, int role,
                                          const CS<KnotTrig<P>> tw[NQ], const typename P::Minv* mi) {
  typename P::Minv Mi[NQ][NQ];
  load_packed_minv(mi, Mi);
  PhaseC<typename P::Col> PC;
  typename P::Rnea qdd[NQ];
  phase_a_after_minv<P>(in, opt, tw, Mi, PC, qdd);
  if (role == kRoleQdd) {
    for (int r = 0; r < NQ; ++r) out.qdd(r, float(qdd[r]));
    for (int r = 0; r < NQ; ++r) out.dq(r, 0, 0.0f);
  }
  if constexpr (WantsMinv<Out>::value)
    if (role < NQ) store_minv_column(out, PC.Mi, role);
  gradient_column_lane(PC, opt.damping, role, out);
}

// Full path for one knot spread over kLanesPerKnotGroup lanes of one wave:
// lanes 0..6 each compute one column of Minv and share it through the group's
// LDS slot mi (kMinvPacked values), then every lane runs steps 2-5 and one
// derivative column.  Device code only: the host build runs the two stages
// for every lane role in turn.
template <class P = PrecFP32, class In, class Out>
RBD_HD RBD_INLINE void fdgrad_knot_lanes(const In& in, Out& out, const Options& opt, int role,
                                         typename P::Minv* mi) {
  CS<KnotTrig<P>> tw[NQ];
  lanes_minv_stage<P>(in, role, tw, mi);
  wave_lds_sync();
  lanes_finish_stage<P>(in, out, opt, role, tw, mi);
}

// ---------------------------------------------------------------------------
// Two-wave latency mapping.  For one knot, one wave (M) runs the Minv
// recursion, lane j of the knot's group computing column j, while a second
// wave (R) runs the RNEA at qdd = 0 and all thirteen derivative columns with
// the bias accelerations and forces a_b, f_b; the two overlap instead of
// adding up.  The columns
// need a, f at the true qdd only in the d/dq seeds (a_c x S at link c) and the
// backward extra term (f_c at link c), in which a d/dq column is linear.  So
// with da = a - a_b and df = f - f_b, both linear in qdd:
//   dtau/dq_c = column(a_b, f_b) + column'(da_c x S, df_c)
// where column' is the sweep with v = 0 (no velocity terms, ~400
// instructions).  After M has Minv it forms qdd = Minv (u - c - damping qd),
// the chain da_k = T_k da_{k-1} + S qdd_k, dF_k = I_k da_k, df = RNEA
// backward pass of dF, and each d/dq lane's correction column'; R then adds
// the corrections and forms -Minv dtau.  Stage functions are per (knot, lane
// role); wave M runs M1a (its Minv column into LDS), M1b (the whole Minv back
// from LDS), waits for R1a's bias, runs M2 and signals; wave R runs R1a,
// signals, runs R1b, waits for M2, runs R2.  The critical path is the longer
// of M1 + M2 and R1, plus R2.
// ---------------------------------------------------------------------------

// Exchange between the waves for one knot (LDS in the kernel).
template <class P>
struct TwoWaveShared {
  typename P::Rnea bias[NQ];                        // u - c - damping qd (R1 -> M2)
  typename P::Minv mi[kMinvPacked];                 // upper Minv, packed (M1a -> M1b, R2)
  typename P::Col corr[kLanesPerKnotGroup][NQ];     // d/dq corrections by lane role (M2 -> R2)
};

// column'(da_c x S, df_c) for lane role's d/dq column c, uniform over lanes
// like dtau_column_uniform: dax[k] = (da_k x S) as (a1, -a0, a4, -a3),
// ndfx[k] = -(df_k x S) as (-f1, f0, -f4, f3).
template <typename S>
RBD_HD RBD_INLINE void dq_correction_uniform(const CS<S>* t, const S dax[NQ][4], const S ndfx[NQ][4], int c,
                                             S tau[NQ]) {
  S da[6], df[NQ][6];
  for (int i = 0; i < 6; ++i) da[i] = S(0);
  static_for<0, NQ>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    S pa[6];
    if constexpr (k > 0) {
      xmotion<k>(t[k], da, pa);
    } else {
      for (int i = 0; i < 6; ++i) pa[i] = S(0);
    }
    const S ax[6] = {dax[k][0], dax[k][1], S(0), dax[k][2], dax[k][3], S(0)};
    const bool seed = (k == c);
    for (int i = 0; i < 6; ++i) da[i] = seed ? ax[i] : pa[i];
    imv<k>(da, df[k]);
  });
  S g[6];
  for (int i = 0; i < 6; ++i) g[i] = df[NQ - 1][i];
  static_for_down<NQ, 1>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    tau[k] = g[2];
    const bool extra = (k == c);
    g[0] += extra ? ndfx[k][0] : S(0); g[1] += extra ? ndfx[k][1] : S(0);
    g[3] += extra ? ndfx[k][2] : S(0); g[4] += extra ? ndfx[k][3] : S(0);
    S y[6];
    xforce_t_add<k>(t[k], g, df[k - 1], y);
    for (int i = 0; i < 6; ++i) g[i] = y[i];
  });
  tau[0] = g[2];
}

// Wave R's state between its stages.
template <class P>
struct TwoWaveR {
  using SR = typename P::Rnea; using SC = typename P::Col;
  CS<SC> tc[NQ];
  SR qd[NQ], v[NQ][6], a[NQ][6], f[NQ][6];
};

// Stage R1a (wave R): RNEA at qdd = 0 and the bias into sh.
template <class P, class In>
RBD_HD RBD_INLINE void two_wave_r1a(const In& in, const Options& opt, int role, TwoWaveShared<P>& sh,
                                    TwoWaveR<P>& st) {
  using SR = typename P::Rnea; using SC = typename P::Col;
  CS<KnotTrig<P>> tw[NQ];
  knot_trig_group<P>(in, role, tw);
  CS<SR> tr[NQ];
  SR u[NQ];
  for (int k = 0; k < NQ; ++k) {
    tr[k] = CS<SR>{SR(tw[k].c), SR(tw[k].s)}; st.tc[k] = CS<SC>{SC(tw[k].c), SC(tw[k].s)};
    st.qd[k] = SR(in.qd(k));
    u[k] = SR(in.u(k));
  }
  const SR zero[NQ] = {SR(0), SR(0), SR(0), SR(0), SR(0), SR(0), SR(0)};
  rnea_fwd(tr, st.qd, zero, SR(opt.gravity), st.v, st.a, st.f);
  subtract_fext(in, st.f);
  rnea_bwd(tr, st.f);
  static_for<0, NQ>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    if (role == k) sh.bias[k] = u[k] - st.f[k][2] - SR(opt.damping) * st.qd[k];
  });
}

// Stage R1b (wave R): lane role's column with a_b, f_b (damping on the
// d/dqd diagonal) into tau_col.
template <class P>
RBD_HD RBD_INLINE void two_wave_r1b(const Options& opt, int role, const TwoWaveR<P>& st,
                                    typename P::Col tau_col[NQ]) {
  using SR = typename P::Rnea; using SC = typename P::Col;
  SR Mz[NQ][NQ];
  for (int r = 0; r < NQ; ++r)
    for (int c = 0; c < NQ; ++c) Mz[r][c] = SR(0);
  PhaseC<SC> PC;
  make_phase_c(PC, st.tc, st.v, st.a, st.f, Mz);
  const bool dq = role >= NQ;
  const int c = dq ? role - (NQ - 1) : role;
  dtau_column_uniform(PC, c, dq, tau_col);
  add_on_diagonal(tau_col, dq ? -1 : c, SC(opt.damping));
}

// sin/cos type of wave M (shared by its two stages)
template <class P>
using TwoWaveTrig = KnotTrig<P>;

// Stage M1a (wave M): sin/cos (kept for M2) and lane role's column of Minv
// (roles 0..6), its upper entries stored into sh.mi.
template <class P, class In>
RBD_HD RBD_INLINE void two_wave_m1a(const In& in, int role, CS<TwoWaveTrig<P>> tw[NQ], TwoWaveShared<P>& sh) {
  lanes_minv_stage<P>(in, role, tw, sh.mi);
}

// Stage M1b (wave M, after every lane's M1a): the whole upper Minv from sh.mi.
template <class P>
RBD_HD RBD_INLINE void two_wave_m1b(const TwoWaveShared<P>& sh, typename P::Minv Mi[NQ][NQ]) {
  load_packed_minv(sh.mi, Mi);
}

// Stage M2 (wave M, after R1): qdd (stored by lane role kRoleQdd), the
// qdd-dependent chain and lane role's d/dq correction into sh.
template <class P, class Out>
RBD_HD RBD_INLINE void two_wave_m2(int role, const CS<TwoWaveTrig<P>> tw[NQ], const typename P::Minv Mi[NQ][NQ],
                                   TwoWaveShared<P>& sh, Out& out) {
  using SR = typename P::Rnea; using SC = typename P::Col;
  CS<SR> tr[NQ]; CS<SC> tc[NQ];
  for (int k = 0; k < NQ; ++k) {
    tr[k] = CS<SR>{SR(tw[k].c), SR(tw[k].s)};
    tc[k] = CS<SC>{SC(tw[k].c), SC(tw[k].s)};
  }
  SR bias[NQ], qdd[NQ];
  for (int k = 0; k < NQ; ++k) bias[k] = sh.bias[k];
  minv_times<false>(Mi, bias, qdd);
  if (role == kRoleQdd)
    for (int r = 0; r < NQ; ++r) out.qdd(r, float(qdd[r]));
  // da_k = T_k da_{k-1} + S qdd_k, dF_k = I_k da_k, then the backward pass
  SR dA[NQ][6], dF[NQ][6];
  static_for<0, NQ>([&](auto Kc) {
    constexpr int k = decltype(Kc)::value;
    if constexpr (k == 0) {
      for (int i = 0; i < 6; ++i) dA[0][i] = SR(0);
    } else {
      xmotion<k>(tr[k], dA[k - 1], dA[k]);
    }
    dA[k][2] += qdd[k];
    imv<k>(dA[k], dF[k]);
  });
  rnea_bwd(tr, dF);
  SC dax[NQ][4], ndfx[NQ][4];
  for (int k = 0; k < NQ; ++k) {
    dax[k][0] = SC(dA[k][1]); dax[k][1] = -SC(dA[k][0]); dax[k][2] = SC(dA[k][4]); dax[k][3] = -SC(dA[k][3]);
    ndfx[k][0] = -SC(dF[k][1]); ndfx[k][1] = SC(dF[k][0]); ndfx[k][2] = -SC(dF[k][4]); ndfx[k][3] = SC(dF[k][3]);
  }
  SC corr[NQ];
  dq_correction_uniform(tc, dax, ndfx, role - (NQ - 1), corr);
  for (int r = 0; r < NQ; ++r) sh.corr[role][r] = corr[r];
}

// Stage R2 (wave R, after M2): corrections added, -Minv dtau, stores.
template <class P, class Out>
RBD_HD RBD_INLINE void two_wave_r2(int role, const TwoWaveShared<P>& sh, typename P::Col tau_col[NQ], Out& out) {
  using SC = typename P::Col;
  const bool dq = role >= NQ;
  const int c = dq ? role - (NQ - 1) : role;
  if (dq)
    for (int r = 0; r < NQ; ++r) tau_col[r] += sh.corr[role][r];
  SC Mi[NQ][NQ];
  static_for<0, NQ>([&](auto Rc) {
    constexpr int r = decltype(Rc)::value;
    static_for<r, NQ>([&](auto Cc) {
      constexpr int cc = decltype(Cc)::value;
      Mi[r][cc] = SC(sh.mi[upper_index(r, cc)]);
    });
  });
  SC col[NQ];
  minv_times<true>(Mi, tau_col, col);
  if (role < NQ) {
    for (int r = 0; r < NQ; ++r) out.dqd(r, c, float(col[r]));
  } else if (role < 2 * NQ - 1) {
    for (int r = 0; r < NQ; ++r) out.dq(r, c, float(col[r]));
  } else if (role == kRoleQdd) {
    for (int r = 0; r < NQ; ++r) out.dq(r, 0, 0.0f);
  }
}

// Reference-compatible mode (QDD_MINV_PASSED_IN, the reference's timed
// configuration; dynamicsGradientKernel, helpers_GPU/dynamicsGradient.cuh:1257-1291):
// qdd and a dense Minv are inputs; out is dqdd/dq, dqdd/dqd.  The upper triangle
// of the given Minv is read (the same matrix for the symmetric Minv that
// forwardDynamics produces).
template <class P, class In, class Out, class Times>
RBD_HD RBD_INLINE void gradient_given_qdd(const In& in, Out& out, const Options& opt, const Times& times) {
  using SR = typename P::Rnea; using SC = typename P::Col;
  CS<Wider<SR, SC>> tw[NQ];
  knot_trig_in(P{}, in, tw);
  CS<SR> tr[NQ];
  cast_trig(tw, tr);
  SR v[NQ][6], a[NQ][6], qd[NQ], qdd[NQ];
  for (int k = 0; k < NQ; ++k) { qd[k] = SR(in.qd(k)); qdd[k] = SR(in.qdd(k)); }
  link_motion(tr, qd, qdd, SR(opt.gravity), v, a);
  if constexpr (std::is_same<SR, SC>::value) {
    gradient_columns(in, tr, v, a, opt.damping, times, out);
  } else {
    CS<SC> tc[NQ];
    SC vc[NQ][6], ac[NQ][6];
    cast_trig(tw, tc);
    for (int k = 0; k < NQ; ++k)
      for (int i = 0; i < 6; ++i) { vc[k][i] = SC(v[k][i]); ac[k][i] = SC(a[k][i]); }
    gradient_columns(in, tc, vc, ac, opt.damping, times, out);
  }
}
template <class P = PrecFP32, class In, class Out>
RBD_HD RBD_INLINE void fdgrad_knot_given_qdd_minv(const In& in, Out& out, const Options& opt) {
  using SC = typename P::Col;
  SC Mi[NQ][NQ];
  for (int r = 0; r < NQ; ++r)
    for (int c = r; c < NQ; ++c) Mi[r][c] = SC(in.minv(r, c));
  gradient_given_qdd<P>(in, out, opt, TimesMinv<SC>{Mi});
}

// The same spread over a lane group.
template <class P = PrecFP32, class In, class Out>
RBD_HD RBD_INLINE void fdgrad_knot_given_qdd_minv_lanes(const In& in, Out& out, const Options& opt, int role) {
  PhaseC<typename P::Col> PC;
  phase_a_given_qdd_minv<P>(in, opt, PC);
  if (role == kRoleQdd)
    for (int r = 0; r < NQ; ++r) out.dq(r, 0, 0.0f);
  gradient_column_lane(PC, opt.damping, role, out);
}

// Inverse-dynamics gradient cdu = [dtau/dq | dtau/dqd] (98 per knot, the
// reference's "fused" GPU stage, dynamicsGradientKernel_fused,
// helpers_GPU/dynamicsGradient.cuh:1223-1255): q, qd, qdd given (u unused),
// RNEA at qdd, then the derivative sweeps; no Minv.
template <class P = PrecFP32, class In, class Out>
RBD_HD RBD_INLINE void id_gradient_knot(const In& in, Out& out, const Options& opt) {
  gradient_given_qdd<P>(in, out, opt, TimesNothing{});
}
template <class P = PrecFP32, class In, class Out>
RBD_HD RBD_INLINE void id_gradient_knot_lanes(const In& in, Out& out, const Options& opt, int role) {
  PhaseC<typename P::Col> PC;
  phase_a_given_qdd_minv<P, false>(in, opt, PC);
  if (role == kRoleQdd)
    for (int r = 0; r < NQ; ++r) out.dq(r, 0, 0.0f);
  gradient_column_lane<false>(PC, opt.damping, role, out);
}

// The same from precomputed v, a, f (the reference's "split" GPU stage,
// dynamicsGradientKernel_split, .cuh:1191-1221): in.v/a/f(k, i) are RNEA's
// link velocities, accelerations and forces, f after the backward pass.
template <class P, class In>
RBD_HD RBD_INLINE void phase_split(const In& in, PhaseC<typename P::Col>& PC) {
  using SC = typename P::Col;
  CS<SC> tc[NQ];
  SC v[NQ][6], a[NQ][6], f[NQ][6], Mi[NQ][NQ];
  knot_trig_in(P{}, in, tc);
  for (int k = 0; k < NQ; ++k) {
    for (int i = 0; i < 6; ++i) { v[k][i] = SC(in.v(k, i)); a[k][i] = SC(in.a(k, i)); f[k][i] = SC(in.f(k, i)); }
    for (int c2 = 0; c2 < NQ; ++c2) Mi[k][c2] = SC(0);
  }
  make_phase_c(PC, tc, v, a, f, Mi);
}
template <class P = PrecFP32, class In, class Out>
RBD_HD RBD_INLINE void id_gradient_split_knot(const In& in, Out& out, const Options& opt) {
  using SC = typename P::Col;
  CS<SC> tc[NQ];
  knot_trig_in(P{}, in, tc);
  SC v[NQ][6], a[NQ][6];
  for (int k = 0; k < NQ; ++k)
    for (int i = 0; i < 6; ++i) { v[k][i] = SC(in.v(k, i)); a[k][i] = SC(in.a(k, i)); }
  gradient_columns<true>(in, tc, v, a, opt.damping, TimesNothing{}, out);
}
template <class P = PrecFP32, class In, class Out>
RBD_HD RBD_INLINE void id_gradient_split_knot_lanes(const In& in, Out& out, const Options& opt, int role) {
  PhaseC<typename P::Col> PC;
  phase_split<P>(in, PC);
  if (role == kRoleQdd)
    for (int r = 0; r < NQ; ++r) out.dq(r, 0, 0.0f);
  gradient_column_lane<false>(PC, opt.damping, role, out);
}

// RNEA's v, a, f at (q, qd, qdd), f after the backward pass: what the
// reference's CPU "start" stage writes into the split layout
// (forwardDynamicsGradientSetup_forGPU, .cuh:1148-1157, with QDD_MINV_PASSED_IN).
template <class P = PrecFP32, class In, class Out>
RBD_HD RBD_INLINE void vaf_knot(const In& in, Out& out, const Options& opt) {
  using SR = typename P::Rnea;
  CS<SR> tr[NQ];
  SR qd[NQ], qdd[NQ];
  knot_trig_in(P{}, in, tr);
  for (int k = 0; k < NQ; ++k) {
    qd[k] = SR(in.qd(k));
    qdd[k] = SR(in.qdd(k));
  }
  SR v[NQ][6], a[NQ][6], f[NQ][6];
  rnea_fwd(tr, qd, qdd, SR(opt.gravity), v, a, f);
  subtract_fext(in, f);
  rnea_bwd(tr, f);
  for (int k = 0; k < NQ; ++k)
    for (int i = 0; i < 6; ++i) out.vaf(k, i, float(v[k][i]), float(a[k][i]), float(f[k][i]));
}

// The reference's CPU "finish" stage (forwardDynamicsGradientFinish_forGPU,
// .cuh:1168-1179; matMultSym, helpers_CPU/math.h:16-25): dqdd = -Minv cdu
// with the upper triangle of Minv (49, column-major) and cdu 98 per knot.
template <typename S = float, class In, class Out>
RBD_HD RBD_INLINE void finish_knot(const In& in, Out& out) {
  S Mi[NQ][NQ];
  for (int r = 0; r < NQ; ++r)
    for (int c = r; c < NQ; ++c) Mi[r][c] = S(in.minv(r, c));
  for (int c = 0; c < 2 * NQ; ++c) {
    S x[NQ], y[NQ];
    for (int r = 0; r < NQ; ++r) x[r] = S(in.cdu(r, c));
    minv_times<true>(Mi, x, y);
    for (int r = 0; r < NQ; ++r) out.dqdd(r, c, float(y[r]));
  }
}

// ---------------------------------------------------------------------------
// Memory layouts
// ---------------------------------------------------------------------------
constexpr int kInPerKnot = 21;     // q, qd, u
constexpr int kOutPerKnot = 105;   // qdd, dqdd/dq (col-major), dqdd/dqd
constexpr int kVolPerKnot = 77;    // q, qd, u, qdd, Minv dense (COMPLETELY_FUSED_VALS, .cuh:1145)
constexpr int kDqddPerKnot = 98;   // dqdd/dq, dqdd/dqd
constexpr int kFextPerSet = 42;    // external forces: 7 links x (moment, force) in the link frame
constexpr int kFusedPerKnot = 28;  // q, qd, u, qdd (FUSED_VALS, .cuh:1144)
constexpr int kSplitPerKnot = 154; // q, qd, u, qdd, v (42), a (42), f (42) (SPLIT_VALS, .cuh:1143)

// array-of-structures: one knot's values contiguous (the reference's knot<T> order)
struct InAoS {
  const float* p;
  const float* fx = nullptr;   // external link forces (42 floats) or null
  RBD_HD float q(int i) const { return p[i]; }
  RBD_HD float qd(int i) const { return p[NQ + i]; }
  RBD_HD float u(int i) const { return p[2 * NQ + i]; }
  RBD_HD float qdd(int i) const { return p[3 * NQ + i]; }
  RBD_HD float minv(int r, int c) const { return p[4 * NQ + r + NQ * c]; }
};
struct OutAoS {
  float* p;
  RBD_HD void qdd(int i, float x) const { p[i] = x; }
  RBD_HD void dq(int r, int c, float x) const { p[NQ + NQ * c + r] = x; }
  RBD_HD void dqd(int r, int c, float x) const { p[NQ + NQ * NQ + NQ * c + r] = x; }
};
// full-path output plus dqdd/du = Minv (dense, column-major, 49 per knot)
struct OutAoSMinv {
  static constexpr bool kMinv = true;
  float* p; float* m;
  RBD_HD void qdd(int i, float x) const { p[i] = x; }
  RBD_HD void dq(int r, int c, float x) const { p[NQ + NQ * c + r] = x; }
  RBD_HD void dqd(int r, int c, float x) const { p[NQ + NQ * NQ + NQ * c + r] = x; }
  RBD_HD void minv(int r, int c, float x) const { m[NQ * c + r] = x; }
};
// The WAFR baseline's gradient layout (time_GPU_WAFR.cu:18; finish_dqdd_v2,
// helpers_WAFR/dynamics_WAFR.cuh:2555-2579): per knot kWafrPerKnot floats,
// [dqdd/dq | dqdd/dqd | dqdd/du = Minv], each 7x7 column-major; qdd (7 per
// knot) to its own buffer when q is not null.
constexpr int kWafrPerKnot = 3 * NQ * NQ;
struct OutWafr {
  static constexpr bool kMinv = true;
  float* q; float* p;
  RBD_HD void qdd(int i, float x) const { if (q) q[i] = x; }
  RBD_HD void dq(int r, int c, float x) const { p[NQ * c + r] = x; }
  RBD_HD void dqd(int r, int c, float x) const { p[NQ * NQ + NQ * c + r] = x; }
  RBD_HD void minv(int r, int c, float x) const { p[2 * NQ * NQ + NQ * c + r] = x; }
};
// forward dynamics only: qdd (7 per knot) and Minv (49 per knot, dense column-major)
// an output accessor whose stores are dropped when `on` is false (lanes that
// only take part in a workgroup's barriers)
template <class Out>
struct OutMasked {
  Out o; bool on;
  RBD_HD void qdd(int i, float x) const { if (on) o.qdd(i, x); }
  RBD_HD void dq(int r, int c, float x) const { if (on) o.dq(r, c, x); }
  RBD_HD void dqd(int r, int c, float x) const { if (on) o.dqd(r, c, x); }
};
struct OutFD {
  float* qdd_p; float* minv_p;
  RBD_HD void qdd(int i, float x) const { qdd_p[i] = x; }
  RBD_HD void minv(int r, int c, float x) const { minv_p[NQ * c + r] = x; }
};
struct OutDqddAoS {   // 98 per knot, no qdd
  float* p;
  RBD_HD void qdd(int, float) const {}
  RBD_HD void dq(int r, int c, float x) const { p[NQ * c + r] = x; }
  RBD_HD void dqd(int r, int c, float x) const { p[NQ * NQ + NQ * c + r] = x; }
};
// structure-of-arrays: value i of knot k at p[i * ld + k]
// split layout: [q | qd | u | qdd | v | a | f], link k's 6-vectors at 6k
struct InSplit {
  const float* p;
  const float* fx = nullptr;
  RBD_HD float q(int i) const { return p[i]; }
  RBD_HD float qd(int i) const { return p[NQ + i]; }
  RBD_HD float v(int k, int i) const { return p[4 * NQ + 6 * k + i]; }
  RBD_HD float a(int k, int i) const { return p[10 * NQ + 6 * k + i]; }
  RBD_HD float f(int k, int i) const { return p[16 * NQ + 6 * k + i]; }
};
struct OutVaf {   // v, a, f into the split layout
  float* p;
  RBD_HD void vaf(int k, int i, float v, float a, float f) const {
    p[4 * NQ + 6 * k + i] = v; p[10 * NQ + 6 * k + i] = a; p[16 * NQ + 6 * k + i] = f;
  }
};
// finish stage: Minv (49, column-major, upper triangle read) and cdu (98) in, dqdd (98) out
struct InFinish {
  const float* m; const float* c;
  RBD_HD float minv(int r, int col) const { return m[r + NQ * col]; }
  RBD_HD float cdu(int r, int col) const { return c[r + NQ * col]; }
};
struct OutFinish {
  float* p;
  RBD_HD void dqdd(int r, int col, float x) const { p[r + NQ * col] = x; }
};
struct InSoA {
  const float* p; long ld;
  const float* fx = nullptr;   // external link forces (42 floats) or null
  RBD_HD float q(int i) const { return p[i * ld]; }
  RBD_HD float qd(int i) const { return p[(NQ + i) * ld]; }
  RBD_HD float u(int i) const { return p[(2 * NQ + i) * ld]; }
};
// A knot's 21 inputs already in registers: the one-lane kernels load them
// before anything else of a loop iteration, ahead of the stores they defer.
struct InRegs {
  float x[kInPerKnot];
  const float* fx = nullptr;
  RBD_HD float q(int i) const { return x[i]; }
  RBD_HD float qd(int i) const { return x[NQ + i]; }
  RBD_HD float u(int i) const { return x[2 * NQ + i]; }
};
struct OutSoA {
  float* p; long ld;
  RBD_HD void qdd(int i, float x) const { p[i * ld] = x; }
  RBD_HD void dq(int r, int c, float x) const { p[(NQ + NQ * c + r) * ld] = x; }
  RBD_HD void dqd(int r, int c, float x) const { p[(NQ + NQ * NQ + NQ * c + r) * ld] = x; }
};

}  // namespace rbd
