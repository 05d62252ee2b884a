// fft_common.h -- complex arithmetic and in-register DFT butterflies shared by the generic and
// the size-specialised Stockham FFT kernels.
#pragma once
#include "fhd_device.h"
#include "fhd_kernels.h"

namespace fhd {

FHD_DEV float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
FHD_DEV float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
FHD_DEV float2 cmul(float2 a, float2 b) {
  return make_float2(fmaf(a.x, b.x, -(a.y * b.y)), fmaf(a.x, b.y, a.y * b.x));
}
FHD_DEV float2 cconj(float2 a) { return make_float2(a.x, -a.y); }
FHD_DEV float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
// a * (s i), s = +-1
FHD_DEV float2 cmul_si(float2 a, float s) { return make_float2(-s * a.y, s * a.x); }

// t sqrt(1/2) and t sqrt(3)/2 with the constants' low parts: the rounded constants alone (2e-8 small)
// shrink every forward and inverse transform a little, which adds up over the steps of a run.
FHD_DEV float mul_r2(float t) { return fmaf(1.2101617e-8f, t, 0.70710678118654752440f * t); }
FHD_DEV float mul_r3(float t) { return fmaf(1.5543628e-8f, t, 0.86602540378443864676f * t); }
// a e^{s i pi/4} and a e^{s 3 i pi/4}
FHD_DEV float2 turn1(float2 a, float s) { return make_float2(mul_r2(fmaf(-s, a.y, a.x)), mul_r2(fmaf(s, a.x, a.y))); }
FHD_DEV float2 turn3(float2 a, float s) { return make_float2(mul_r2(fmaf(-s, a.y, -a.x)), mul_r2(fmaf(s, a.x, -a.y))); }

// a (p c + i s d) with (c, d) = (cos, sin) of pi/8, or exchanged (swap), and their low parts.
FHD_DEV float2 turn16(float2 a, float p, float s, bool swap) {
  const float c = 0.92387953251128675613f, d = 0.38268343236508977173f, cl = 2.8307490e-8f, dl = 6.2233509e-9f;
  const float u = p * (swap ? d : c), ul = p * (swap ? dl : cl), v = s * (swap ? c : d), vl = s * (swap ? cl : dl);
  return make_float2(fmaf(a.x, u, -(a.y * v)) + fmaf(a.x, ul, -(a.y * vl)),
                     fmaf(a.x, v, a.y * u) + fmaf(a.x, vl, a.y * ul));
}

// a (p + i s sqrt(3)/2) and a (s sqrt(3)/2 + i p)
FHD_DEV float2 turn6(float2 a, float p, float s) {
  return make_float2(fmaf(p, a.x, -s * mul_r3(a.y)), fmaf(p, a.y, s * mul_r3(a.x)));
}
FHD_DEV float2 turn12(float2 a, float s, float p) {
  return make_float2(fmaf(-p, a.y, s * mul_r3(a.x)), fmaf(p, a.x, s * mul_r3(a.y)));
}

// In-register DFTs with kernel e^{s 2 pi i / R}.
template <int R> struct Dft;
template <> struct Dft<2> {
  static FHD_DEV void run(float2* v, float) {
    float2 a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  }
};
template <> struct Dft<3> {
  static FHD_DEV void run(float2* v, float s) {
    float2 t = cadd(v[1], v[2]);
    float2 u = csub(v[1], v[2]);
    float2 m = make_float2(fmaf(-0.5f, t.x, v[0].x), fmaf(-0.5f, t.y, v[0].y));
    float2 r = cmul_si(make_float2(mul_r3(u.x), mul_r3(u.y)), s);
    v[0] = cadd(v[0], t);
    v[1] = cadd(m, r);
    v[2] = csub(m, r);
  }
};
template <> struct Dft<4> {
  static FHD_DEV void run(float2* v, float s) {
    float2 t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
    float2 t2 = cadd(v[1], v[3]), t3 = cmul_si(csub(v[1], v[3]), s);
    v[0] = cadd(t0, t2);
    v[2] = csub(t0, t2);
    v[1] = cadd(t1, t3);
    v[3] = csub(t1, t3);
  }
};
template <> struct Dft<6> {
  static FHD_DEV void run(float2* v, float s) {
    float2 e[3] = {v[0], v[2], v[4]}, o[3] = {v[1], v[3], v[5]};
    Dft<3>::run(e, s);
    Dft<3>::run(o, s);
    // w^k = e^{s 2 pi i k / 6}
    const float2 o1 = turn6(o[1], 0.5f, s), o2 = turn6(o[2], -0.5f, s);
    v[0] = cadd(e[0], o[0]);
    v[3] = csub(e[0], o[0]);
    v[1] = cadd(e[1], o1);
    v[4] = csub(e[1], o1);
    v[2] = cadd(e[2], o2);
    v[5] = csub(e[2], o2);
  }
};
template <> struct Dft<9> {
  static FHD_DEV void run(float2* v, float s) {
    // three 3-point transforms of every third element, twiddles e^{s 2 pi i b k / 9}, three more
    float2 y[3][3];
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      y[b][0] = v[b];
      y[b][1] = v[b + 3];
      y[b][2] = v[b + 6];
      Dft<3>::run(y[b], s);
    }
    const float c1 = 0.76604444311897803520f, s1 = 0.64278760968653932632f;  // 2 pi / 9
    const float c2 = 0.17364817766693034885f, s2 = 0.98480775301220805937f;  // 4 pi / 9
    const float c4 = -0.93969262078590838405f, s4 = 0.34202014332566873304f;  // 8 pi / 9
    y[1][1] = cmul(y[1][1], make_float2(c1, s * s1));
    y[1][2] = cmul(y[1][2], make_float2(c2, s * s2));
    y[2][1] = cmul(y[2][1], make_float2(c2, s * s2));
    y[2][2] = cmul(y[2][2], make_float2(c4, s * s4));
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      float2 t[3] = {y[0][k], y[1][k], y[2][k]};
      Dft<3>::run(t, s);
      v[k] = t[0];
      v[k + 3] = t[1];
      v[k + 6] = t[2];
    }
  }
};
template <> struct Dft<8> {
  static FHD_DEV void run(float2* v, float s) {
    float2 e[4] = {v[0], v[2], v[4], v[6]};
    float2 o[4] = {v[1], v[3], v[5], v[7]};
    Dft<4>::run(e, s);
    Dft<4>::run(o, s);
    // w^k = e^{s 2 pi i k / 8}
    float2 o1 = turn1(o[1], s);
    float2 o2 = cmul_si(o[2], s);
    float2 o3 = turn3(o[3], s);
    v[0] = cadd(e[0], o[0]);
    v[4] = csub(e[0], o[0]);
    v[1] = cadd(e[1], o1);
    v[5] = csub(e[1], o1);
    v[2] = cadd(e[2], o2);
    v[6] = csub(e[2], o2);
    v[3] = cadd(e[3], o3);
    v[7] = csub(e[3], o3);
  }
};

template <> struct Dft<12> {
  static FHD_DEV void run(float2* v, float s) {
    // four-point transforms of every third element, twiddles e^{s 2 pi i b k / 12}, three-point ones
    float2 y[3][4];
#pragma unroll
    for (int b = 0; b < 3; ++b) {
#pragma unroll
      for (int k = 0; k < 4; ++k) y[b][k] = v[b + 3 * k];
      Dft<4>::run(y[b], s);
    }
    y[1][1] = turn12(y[1][1], 1.0f, 0.5f * s);
    y[1][2] = turn6(y[1][2], 0.5f, s);
    y[1][3] = cmul_si(y[1][3], s);
    y[2][1] = turn6(y[2][1], 0.5f, s);
    y[2][2] = turn6(y[2][2], -0.5f, s);
    y[2][3] = make_float2(-y[2][3].x, -y[2][3].y);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float2 t[3] = {y[0][k], y[1][k], y[2][k]};
      Dft<3>::run(t, s);
      v[k] = t[0];
      v[k + 4] = t[1];
      v[k + 8] = t[2];
    }
  }
};

template <> struct Dft<16> {
  static FHD_DEV void run(float2* v, float s) {
    float2 e[8], o[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      e[k] = v[2 * k];
      o[k] = v[2 * k + 1];
    }
    Dft<8>::run(e, s);
    Dft<8>::run(o, s);
    // w^k = e^{s 2 pi i k / 16}
    const float2 t[8] = {o[0],
                         turn16(o[1], 1.0f, s, false),
                         turn1(o[2], s),
                         turn16(o[3], 1.0f, s, true),
                         cmul_si(o[4], s),
                         turn16(o[5], -1.0f, s, true),
                         turn3(o[6], s),
                         turn16(o[7], -1.0f, s, false)};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      v[k] = cadd(e[k], t[k]);
      v[k + 8] = csub(e[k], t[k]);
    }
  }
};

// The Fourier-space operator at one mode of the z pass (the transforms b0, b1, b2 of the three
// components, replaced by the solution's): the kept part of the stochastic stress divergence is
// added (Stokes limit), then shift to the staggered basis, project, apply the viscous or Stokes
// operator with the 1/N normalisation folded in, shift back.
FHD_DEV void solve_mode(const FftArgs& a, const Key& key, int kx, int ky, int z, float gx, float gy, float gz, float2 ex,
                        float2 ey, float2 ez, float2& b0, float2& b1, float2& b2) {
  if (a.knoise) {
    float2 nw[3];
    kspace_noise(key, kx, ky, z, a.g.mx, a.g.my, a.g.mz, a.knoise, a.kn_f4, a.kn_sqrt_half_n, gx, gy, gz, ex, ey, ez, nw);
    b0 = cadd(b0, nw[0]);
    b1 = cadd(b1, nw[1]);
    b2 = cadd(b2, nw[2]);
  }
  const float2 w0 = cmul(b0, cconj(ex));
  const float2 w1 = cmul(b1, cconj(ey));
  const float2 w2 = cmul(b2, cconj(ez));
  const float L = -fmaf(gz, gz, fmaf(gy, gy, gx * gx));
  if (kx == 0 && ky == 0 && z == 0) {
    const float keep = a.stokes ? 0.0f : a.inv_n;
    b0 = cscale(b0, keep);
    b1 = cscale(b1, keep);
    b2 = cscale(b2, keep);
  } else {
    const float iL = 1.0f / L;
    const float2 GW = make_float2(fmaf(gz, w2.x, fmaf(gy, w1.x, gx * w0.x)) * iL, fmaf(gz, w2.y, fmaf(gy, w1.y, gx * w0.y)) * iL);
    const float den = a.stokes ? (-a.eta * L) : fmaf(-a.cn_coef, L, 1.0f);
    const float sc = a.inv_n / den;
    // sc (b_a + e_a g_a GW): the unprojected part keeps its phase, so the shift there and back (|e|^2,
    // not quite 1) does not touch it
    const auto part = [&](float2 b, float2 e, float g) {
      const float2 q = cmul(e, make_float2(g * GW.x, g * GW.y));
      return cscale(cadd(b, q), sc);
    };
    b0 = part(b0, ex, gx);
    b1 = part(b1, ey, gy);
    b2 = part(b2, ez, gz);
  }
}

// Radix plan of the size-specialised kernels: 16s first, then 8, 4, 2, 3 (fewest LDS stages).
constexpr int plan_radix(int n, int st) {
  for (int i = 0;; ++i) {
    int r = (n % 16 == 0) ? 16 : (n % 8 == 0) ? 8 : (n % 4 == 0) ? 4 : (n % 2 == 0) ? 2 : (n % 3 == 0) ? 3 : 1;
    if (i == st || r == 1) return r;
    n /= r;
  }
}

// Explicit radix plans, 5 bits per stage from the first (0 ends the plan; plan 0 is the default
// above).  Those of 96 x 96 and 128 x 128 planes are square_plan's, or forced with FHD_PLAN_XY.
constexpr uint32_t plan2(int r0, int r1) { return (uint32_t)r0 | ((uint32_t)r1 << 5); }
constexpr uint32_t plan3(int r0, int r1, int r2) { return plan2(r0, r1) | ((uint32_t)r2 << 10); }
constexpr int plan_at(uint32_t plan, int n, int st) { return plan ? (int)((plan >> (5 * st)) & 31u) : plan_radix(n, st); }
// Candidate plans: index 0 is the default for every length; 48, 64, 96 and 128 have two more
// (for 48 and 96, other placements of the radix-3 stage).
constexpr uint32_t kPlan48[3] = {0u, plan2(3, 16), plan3(4, 4, 3)};
constexpr uint32_t kPlan64[3] = {0u, plan2(4, 16), plan2(8, 8)};
constexpr uint32_t kPlan96[3] = {0u, plan3(8, 4, 3), plan3(3, 8, 4)};
constexpr uint32_t kPlan128[3] = {0u, plan2(8, 16), plan3(4, 4, 8)};
constexpr uint32_t plan_choice(int n, int i) {
  return i == 0     ? 0u
         : n == 48  ? kPlan48[i]
         : n == 64  ? kPlan64[i]
         : n == 96  ? kPlan96[i]
         : n == 128 ? kPlan128[i]
                    : 0u;
}

}  // namespace fhd
