/*
 * transport_device.h -- FP32 device implementation of one electron step.
 *
 * Restates, for one GPU lane per electron, the per-step work of
 * MonteCarloSS::takeStep (gov/nist/microanalysis/NISTMonte/MonteCarloSS.cu:107-163)
 * and everything it calls.  Units: nm, eV; directions are unit vectors
 * (the reference keeps theta/phi; Electron::updateDirection, Electron.cu:111-131,
 * is the same rotation written in the electron's local frame).
 *
 * Geometry: every region shape is compiled into convex primitives and a
 * truth table.  The first boundary of the composite along a ray is found by
 * walking the primitives' entry/exit crossings in order and testing where
 * the composite's inside state changes.  This finds the same boundary as the
 * depth-counter walks of NormalIntersectionShape.cu:19-239 and
 * NormalUnionShape.cu:30-271 without their recursive re-queries.
 */
#ifndef MONSEL_TRANSPORT_DEVICE_H
#define MONSEL_TRANSPORT_DEVICE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/monsel_gpu.h"
#include "device_scene.h"
#include "phase_timing.h"

namespace monsel_dev {

#define MD __device__ __forceinline__

constexpr float kPI = 3.14159265358979323846f;
constexpr float kTwoPI = 6.28318530717958647692f;
constexpr float kInf = __builtin_huge_valf();
constexpr float kA0nm = 0.05291772083f;          /* Bohr radius (nm) */
constexpr float kA0nm2 = 0.05291772083f * 0.05291772083f;
constexpr float kMottLn50 = 3.9120230054281460f;    /* ln(50) */
constexpr float kMottInvParam = 60.0f / 5.9914645471079810f; /* 60 / ln(400) */
constexpr float kMaxNISTMott = 20000.0f;            /* eV */
constexpr float kEcharge = 1.60217653e-19f;         /* J per eV */

/* ----------------------------------------------------------- RNG ------- */

/* Square root, natural log and exponential straight from the hardware
 * instructions (v_sqrt_f32, v_log_f32, v_exp_f32: about 1 ulp; FP32
 * denormals are flushed in this code, so no rescaling is needed).  The
 * compiler's own expansions refine sqrt to correct rounding with a
 * reciprocal-root Newton step and scale log/exp around denormal ranges, some
 * ten instructions each, on the transport loop's critical path. */
MD float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
MD float flog(float x) { return __builtin_amdgcn_logf(x) * 0.693147180559945309f; }
MD float fexp(float x) { return __builtin_amdgcn_exp2f(x * 1.442695040888963407f); }

/* Holds wave-uniform values in scalar registers from here on: the loads that
 * feed several of them are then issued together and waited for once, instead
 * of each sinking to its first use behind a branch (a step waited for some 80
 * scalar loads one by one). */
MD void pin() {}
template <class T, class... Rest>
MD void pin(T& v, Rest&... rest) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+s"(v));
#endif
  pin(rest...);
}

/* a product that is not contracted into a following sum */
MD float fmul(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}

/* a / b as a times the hardware reciprocal: what the compiler's own division
 * gives for |b| <= 2^96 (beyond it rescales b around the reciprocal's flush
 * to zero: four more instructions for denominators no transport quantity
 * reaches).  The product is not contracted into a following sum. */
MD float fdiv(float a, float b) {
#pragma clang fp contract(off)
  return a * __builtin_amdgcn_rcpf(b);
}

/* Philox4x32-10 (Salmon et al., SC'11).  Counter words: (block, lineage lo,
 * lineage hi, primary index) under one fixed key; a job's seed enters
 * through the lineage of its primaries (splitmix64 of the seed), a
 * secondary's lineage is derived from its parent's. */
MD void philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0, uint32_t k1,
                      uint32_t& o0, uint32_t& o1, uint32_t& o2, uint32_t& o3) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    if (r > 0) {
      k0 += 0x9E3779B9u;
      k1 += 0xBB67AE85u;
    }
    /* each 32x32 -> 64-bit product is one v_mad_u64_u32 (a separate low
     * and high multiply would be two quarter-rate instructions) */
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
    const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
    const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
    uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
    c0 = n0;
    c1 = lo1;
    c2 = n2;
    c3 = lo0;
  }
  o0 = c0;
  o1 = c1;
  o2 = c2;
  o3 = c3;
}

MD uint64_t splitmix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

MD uint64_t child_lineage(uint64_t parent, uint32_t k) {
  return splitmix64(parent ^ (0x9E3779B97F4A7C15ull * (uint64_t)(k + 1)));
}

/* electron state held in registers */
struct Elec {
  float px, py, pz;
  float dx, dy, dz;
  float E;
  int region;
  uint32_t primary;
  uint32_t lin_lo, lin_hi;
  uint32_t job;
  uint32_t nchild;
  uint32_t steps;
  float safe;   /* lower bound on the distance to the nearest boundary findEndOfStep
                 * would test from here (own shape and children); 0 = unknown */
};

MD float u01(uint32_t x) { return (float)(x >> 9) * 1.1920928955078125e-07f + 5.9604644775390625e-08f; }

/* Uniforms per electron step: Philox blocks 2s and 2s+1 of the electron's
 * stream, s = its step count.  u[0] draws the free path, u[1] the mechanism
 * (or a barrier transmission); the scatter mechanism takes u[2], u[3], ...
 * in the order the reference's scatter() draws them (at most six). */
constexpr int kStepUniforms = 8;

/* u[0..3] from block 2s (drawn when the step starts) */
MD void step_uniforms_lo(const Elec& e, uint32_t k0, uint32_t k1, float* u) {
  uint32_t a0, a1, a2, a3;
  philox4x32_10(2u * e.steps, e.lin_lo, e.lin_hi, e.primary, k0, k1, a0, a1, a2, a3);
  u[0] = u01(a0);
  u[1] = u01(a1);
  u[2] = u01(a2);
  u[3] = u01(a3);
}

/* u[4..7] from block 2s+1, drawn only by a scatter event (s = the step
 * count before the step, `steps` has been advanced since) */
MD void step_uniforms_hi(const Elec& e, uint32_t k0, uint32_t k1, float* u) {
  uint32_t b0, b1, b2, b3;
  philox4x32_10(2u * (e.steps - 1u) + 1u, e.lin_lo, e.lin_hi, e.primary, k0, k1, b0, b1, b2, b3);
  u[4] = u01(b0);
  u[5] = u01(b1);
  u[6] = u01(b2);
  u[7] = u01(b3);
}

/* block reserved for the primary's initial position (never a step block) */
constexpr uint32_t kPrimaryBlock = 0xFFFFFFFFu;
constexpr uint32_t kPhiloxKey0 = 0x6D6F6E73u, kPhiloxKey1 = 0x656C3235u;

/* Lanes per block of every kernel that uses the per-lane LDS arrays below. */
constexpr int kLaneBlock = 256;

/* ----------------------------------------------------------- math ------ */

/* dot product, its rounding fixed whatever surrounds it */
MD float dot3(float ax, float ay, float az, float bx, float by, float bz) {
#pragma clang fp contract(off)
  return __builtin_fmaf(az, bz, __builtin_fmaf(ax, bx, ay * by));
}

/* Electron::updateDirection (Electron.cu:111-131) on a unit vector: deflect
 * by polar angle (ca = cos, sa = sin) and azimuth (cb, sb). */
MD void rotate_dir(float& dx, float& dy, float& dz, float ca, float sa, float cb, float sb) {
  float st2 = dx * dx + dy * dy;
  float cp = 1.f, sp = 0.f, st = 0.f;
  if (st2 > 0.f) {
    st = fsqrt(st2);
    float inv = 1.f / st;
    cp = dx * inv;
    sp = dy * inv;
  }
  float ct = dz;
  float xx = cb * ct * sa + ca * st;
  float yy = sa * sb;
  float nx = cp * xx - sp * yy;
  float ny = cp * yy + sp * xx;
  float nz = ca * ct - cb * sa * st;
  float inv = __builtin_amdgcn_rsqf(nx * nx + ny * ny + nz * nz);
  dx = nx * inv;
  dy = ny * inv;
  dz = nz * inv;
}

/* direction from polar/azimuth angles (Electron(parent, theta, phi, kE)) */
MD void dir_from_angles(float ct, float st, float cph, float sph, float& dx, float& dy, float& dz) {
  dx = st * cph;
  dy = st * sph;
  dz = ct;
}

/* Weights at t of the Lagrange cubic through unit-spaced nodes 0..3 (which
 * Neville's scheme in ULagrangeInterpolation.cu:5-33 evaluates). */
MD void lagrange4_w(float t, float& l0, float& l1, float& l2, float& l3) {
  float t1 = t - 1.f, t2 = t - 2.f, t3 = t - 3.f;
  l0 = -t1 * t2 * t3 * (1.f / 6.f);
  l1 = t * t2 * t3 * 0.5f;
  l2 = -t * t1 * t3 * 0.5f;
  l3 = t * t1 * t2 * (1.f / 6.f);
}

/* ULagrangeInterpolation::d1 index choice (ULagrangeInterpolation.cu:41-47). */
MD int u_index0(float reduced, int len) {
  int i0 = (int)reduced - 1;
  i0 = i0 < 0 ? 0 : i0;
  return i0 > len - 4 ? len - 4 : i0;
}

/* ------------------------------------------------- elastic (per element) */

/* BrowningEmpiricalCrossSection.cu:24-29 (nm^2); e in keV, re its root and
 * inv_re the root's reciprocal */
MD float browning_sigma(float num, float root, float inv, float e, float re, float inv_re) {
#pragma clang fp contract(off)
  return num * __builtin_amdgcn_rcpf(__builtin_fmaf(re, root, e) + inv * inv_re);
}

/* BrowningEmpiricalCrossSection.cu:31-45 -> cos(theta) */
MD float browning_cos(float z, float zp3, float EeV, float r1, float r2) {
  const float e = EeV * 1.0e-3f;
  const float r = fdiv(300.0f * e, z) + fdiv(zp3, 3.0e5f * e);
  const float alpha = fdiv(7.0e-3f, e);
  const bool screened = r1 <= fdiv(r, r + 1.f);
  return 1.0f - (screened ? fdiv(2.0f * alpha * r2, alpha - r2 + 1.f) : 2.0f * r2);
}

/* ScreenedRutherfordScatteringAngle.cu:24-39 (sigma nm^2, cos theta) */
MD float rutherford_sigma(const MONSEL_CS DElem& el, float EeV) {
  const float K1 = 7.670843088080456e-38f / 1.60217653e-19f * 1.0e18f;
  const float K2 = 5.44967975966321e-19f / 1.60217653e-19f;
  float zp = el.rz13;
  return fdiv(K1 * zp * (1.f + el.z), __builtin_fmaf(zp, K2 * zp, EeV));
}
MD float rutherford_cos(float rz23, float EeV, float r) {
  const float K = 5.44968e-19f / 1.60217653e-19f;
  float alpha = fdiv(K * rz23, EeV);
  /* alpha - r + 1 summed as (1 - r) + alpha: 1 - r is exact for r >= 1/2,
   * so the denominator keeps its relative precision when alpha and 1 - r are
   * both small (E >= 20 keV, r near 1) */
  return 1.f - fdiv(2.0f * alpha * r, (1.f - r) + alpha);
}

/* The hot tables: the cross-section nodes (Spwem, 61 floats) of the first
 * kLdsMott NIST Mott elements of a scene, which every step above 50 eV reads
 * for every element of its material, live in LDS; each kernel that evaluates
 * cross-sections copies them there at its start (stage_tables).  The
 * angle tables (61 x 201 per element, read once per elastic event) stay in
 * device memory. */
#ifndef MONSEL_LDS_MOTT_TABLES
#define MONSEL_LDS_MOTT_TABLES 16
#endif
constexpr int kLdsMott = MONSEL_LDS_MOTT_TABLES;
MD float* lds_spwem() {
  __shared__ float l_spwem[(kLdsMott > 0 ? kLdsMott : 1) * kMottNE];
  return l_spwem;
}
/* The search words of the inelastic tables (abscissae, guides and windows;
 * 12.8 KB for the dielectric model's four tables), in LDS as well where those
 * of all tables of the launch's scenes fit; else all are searched in device
 * memory. */
constexpr int kLdsNuWords = 1792;
MD unsigned long long* lds_nu_words() {
  __shared__ unsigned long long l_nu_words[kLdsNuWords];
  return l_nu_words;
}
/* every thread of the block calls it before any cross-section (TAB: or
 * inelastic table) */
template <bool TAB>
MD void stage_tables(const DevScene& S) {
  const int n = min(S.n_mott, kLdsMott) * kMottNE;
  float* l = lds_spwem();
  for (int i = threadIdx.x; i < n; i += blockDim.x) l[i] = S.mott_spwem[i];
  if constexpr (TAB) {
    if (S.n_nu_words <= kLdsNuWords)
      for (int i = threadIdx.x; i < S.n_nu_words; i += blockDim.x) lds_nu_words()[i] = S.nu_words[i];
  }
  __syncthreads();
}

/* NISTMottRS::totalCrossSection (NISTMottRS.cu:103-119), nm^2: the window
 * of the energy grid and its weights, shared by the elements of a material */
struct MottWindow {
  int i0;
  float l0, l1, l2, l3;
};
MD MottWindow mott_window(float EeV) {
  MottWindow w;
  const float red = (flog(EeV) - kMottLn50) * kMottInvParam;
  w.i0 = u_index0(red, kMottNE);
  lagrange4_w(red - (float)w.i0, w.l0, w.l1, w.l2, w.l3);
  return w;
}
MD float mott_sigma(const MottWindow& w, float f0, float f1, float f2, float f3) {
  return kA0nm2 * __builtin_fmaf(w.l3, f3, __builtin_fmaf(w.l2, f2, __builtin_fmaf(w.l1, f1, w.l0 * f0)));
}
MD float mott_table_sigma(const DevScene& S, int mott, const MottWindow& w) {
  float f0, f1, f2, f3;
  if (mott < kLdsMott) {
    const float* f = lds_spwem() + mott * kMottNE + w.i0;
    f0 = f[0];
    f1 = f[1];
    f2 = f[2];
    f3 = f[3];
  } else {
    const MONSEL_CS float* f = S.mott_spwem + mott * kMottNE + w.i0;
    f0 = f[0];
    f1 = f[1];
    f2 = f[2];
    f3 = f[3];
  }
  return mott_sigma(w, f0, f1, f2, f3);
}

/* The terms sigma_i * atoms_i of an elastic mechanism of at most kFewElem
 * elements (m.few) at energy EeV: c[i], 0 beyond the last element.  The same
 * arithmetic as elastic_terms, without its loops: one wave-uniform branch on
 * the element count, one on the energy. */
MD void elastic_terms_few(const DevScene& S, const MONSEL_CS DMech& m, float EeV, float* c) {
#pragma clang fp contract(off)
  const bool mott = m.kind == MONSEL_MECH_NISTMOTT_ELASTIC;
  const bool one = m.nelem == 1;
  const MONSEL_CS DFewElem& el = m.el;
  float n0 = el.natoms[0], n1 = el.natoms[1], n2 = el.natoms[2];
  float s0 = el.sfBrowning[0], s1 = el.sfBrowning[1], s2 = el.sfBrowning[2];
  float a0 = el.brNum[0], a1 = el.brNum[1], a2 = el.brNum[2];
  float b0 = el.brRoot[0], b1 = el.brRoot[1], b2 = el.brRoot[2];
  float d0 = el.brInv[0], d1 = el.brInv[1], d2 = el.brInv[2];
  float extrap = el.extrap;
  int t0 = el.spwem[0], t1 = el.spwem[1], t2 = el.spwem[2];
  pin(n0, n1, n2, s0, s1, s2, a0, a1, a2, b0, b1, b2, d0, d1, d2, extrap, t0, t1, t2);
  c[0] = c[1] = c[2] = 0.f;
  if (m.kind == MONSEL_MECH_BROWNING_ELASTIC || (mott && EeV < extrap)) {
    if (mott && m.method == 3) {
#pragma unroll
      for (int i = 0; i < kFewElem; ++i)
        if (i < m.nelem) {
          const MONSEL_CS DElem& q = S.elems[m.elem0 + i];
          c[i] = fdiv(q.mottAtMin * EeV, q.extrap) * q.natoms;
        }
    } else {
      const float e = EeV * 1.0e-3f;
      const float re = fsqrt(e);
      const float inv_re = __builtin_amdgcn_rcpf(re);
      auto term = [&](float num, float root, float inv, float sf, float n) {
        const float b = browning_sigma(num, root, inv, e, re, inv_re);
        return fmul(mott ? fmul(sf, b) : b, n);
      };
      c[0] = term(a0, b0, d0, s0, n0);
      if (!one) {
        c[1] = term(a1, b1, d1, s1, n1);
        c[2] = term(a2, b2, d2, s2, n2);
      }
    }
  } else if (mott && EeV < kMaxNISTMott) {
    const MottWindow w = mott_window(EeV);
    const float* f = lds_spwem() + w.i0;
    auto term = [&](int t, float n) { return fmul(mott_sigma(w, f[t], f[t + 1], f[t + 2], f[t + 3]), n); };
    c[0] = term(t0, n0);
    if (!one) {
      c[1] = term(t1, n1);
      c[2] = term(t2, n2);
    }
  } else {
#pragma unroll
    for (int i = 0; i < kFewElem; ++i)
      if (i < m.nelem) c[i] = rutherford_sigma(S.elems[m.elem0 + i], EeV) * S.elems[m.elem0 + i].natoms;
  }
}

/* The terms sigma_i * atoms_i of an elastic mechanism at energy EeV, given in
 * element order to f(i, term).  The elements of a mechanism share its kind
 * and extrapolation energy, so which formula holds depends on the energy
 * alone and what the elements share is formed once. */
template <class F>
MD void elastic_terms(const DevScene& S, const MONSEL_CS DMech& m, float EeV, F f) {
#pragma clang fp contract(off)
  const int n = m.nelem;
  if (n <= 0) return;
  const MONSEL_CS DElem* el = S.elems + m.elem0;
  const bool mott = m.kind == MONSEL_MECH_NISTMOTT_ELASTIC;
  const bool low = mott && EeV < el[0].extrap;
  if (m.kind == MONSEL_MECH_BROWNING_ELASTIC || low) {
    if (mott && el[0].method == 3) {
      for (int i = 0; i < n; ++i) f(i, fdiv(el[i].mottAtMin * EeV, el[i].extrap) * el[i].natoms);
    } else {
      const float e = EeV * 1.0e-3f;
      const float re = fsqrt(e);
      const float inv_re = __builtin_amdgcn_rcpf(re);
      for (int i = 0; i < n; ++i) {
        const float b = browning_sigma(el[i].brNum, el[i].brRoot, el[i].brInv, e, re, inv_re);
        f(i, (mott ? el[i].sfBrowning * b : b) * el[i].natoms);
      }
    }
  } else if (mott && EeV < kMaxNISTMott) {
    const MottWindow w = mott_window(EeV);
    for (int i = 0; i < n; ++i) f(i, mott_table_sigma(S, el[i].mott, w) * el[i].natoms);
  } else {
    for (int i = 0; i < n; ++i) f(i, rutherford_sigma(el[i], EeV) * el[i].natoms);
  }
}

/* NISTMottRS::randomScatteringAngle table branch: bicubic Lagrange on X1
 * over (ln E, U) (NISTMottRS.cu:134-150, ULagrangeInterpolation.cu:55-78) at
 * offset x1 of the tables;
 * returns cos(theta) clamped as the reference does. */
MD float mott_cos(const DevScene& S, int x1, float EeV, float u) {
  float rx = (flog(EeV) - kMottLn50) * kMottInvParam;
  int i0 = u_index0(rx, kMottNE);
  float ry = u * 200.0f;
  int j0 = u_index0(ry, kMottNQ);
  float wx0, wx1, wx2, wx3, wy0, wy1, wy2, wy3;
  lagrange4_w(rx - (float)i0, wx0, wx1, wx2, wx3);
  lagrange4_w(ry - (float)j0, wy0, wy1, wy2, wy3);
  const float* base = S.mott_x1 + (uint32_t)(x1 + i0 * kMottNQ + j0);
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float* row = base + i * kMottNQ;
    const float v = __builtin_fmaf(wy3, row[3], __builtin_fmaf(wy2, row[2], __builtin_fmaf(wy0, row[0], wy1 * row[1])));
    const float wx = i == 0 ? wx0 : (i == 1 ? wx1 : (i == 2 ? wx2 : wx3));
    q = __builtin_fmaf(wx, v, q);
  }
  float com = 1.0f - 2.0f * q * q;
  return com > -1.0f ? (com < 1.0f ? com : 1.0f) : -1.0f;
}

/* ------------------------------------------------------------- CSD ----- */

/* (1 + eps)^(-2/3) - 1 for eps >= 0: the Taylor series below 1e-3 (error
 * < 5e-13 relative), the hardware log2/exp2 above (relative error of the
 * result < 1e-4 there, where it is at least 6.7e-4 in size). */
MD float nieminen_factor(float eps) {
  const float series = eps * (-2.f / 3.f + eps * (5.f / 9.f - eps * (40.f / 81.f)));
  const float power = __builtin_amdgcn_exp2f(-(2.f / 3.f) * __builtin_amdgcn_logf(1.f + eps)) - 1.f;
  return eps < 1e-3f ? series : power;
}

/* A stopping-power record's head and its first three elements, 14 words read
 * together into scalar registers. */
struct CSDHead {
  int active, nce;
  float breakE, gamma15, minE;
  float r0, b0, k0, r1, b1, k1, r2, b2, k2;
};
MD CSDHead csd_head(const MONSEL_CS DCSD& c) {
  CSDHead h = {c.active,      c.nce,      c.breakE,   c.gamma15,      c.minE,     c.el[0].recipJ, c.el[0].beta,
               c.el[0].coef, c.el[1].recipJ, c.el[1].beta, c.el[1].coef, c.el[2].recipJ, c.el[2].beta, c.el[2].coef};
  pin(h.active, h.nce, h.breakE, h.gamma15, h.minE, h.r0, h.b0, h.k0, h.r1, h.b1, h.k1, h.r2, h.b2, h.k2);
  return h;
}

/* sum over the elements of coef ln(E / J + beta) */
MD float joy_luo_sum(const MONSEL_CS DCSD& c, const CSDHead& h, float kE) {
  float s = 0.f;
  auto term = [&](float recipJ, float beta, float coef) { s += coef * flog(recipJ * kE + beta); };
  term(h.r0, h.b0, h.k0);
  if (h.nce > 1) {
    /* slots beyond the last element add 0 */
    term(h.r1, h.b1, h.k1);
    term(h.r2, h.b2, h.k2);
    for (int i = 3; i < h.nce; ++i) term(c.el[i].recipJ, c.el[i].beta, c.el[i].coef);
  }
  return s;
}

/* JoyLuoNieminenCSD::compute (JoyLuoNieminenCSD.cu:91-121) with the
 * recursive halving of :154-159 as an explicit depth-first walk: bit d of
 * `pending` marks a second half at depth d.  Below breakE the Nieminen form
 * kE (1 + 1.5 gamma len kE^1.5)^(-2/3) - kE; above it the Joy-Luo loss,
 * halved while it exceeds 10% of the energy. */
MD float csd_compute_split(const MONSEL_CS DCSD& c, const CSDHead& h, float len, float kE);

/* The common case in straight-line code: one segment, no halving (the
 * first pass of csd_compute_split, with the same arithmetic). */
MD float csd_compute(const MONSEL_CS DCSD& c, float len, float kE) {
#pragma clang fp contract(off)
  const CSDHead h = csd_head(c);
  if (!h.active || h.nce == 0) return 0.f;
  if ((kE < h.minE) | (kE <= 0.f)) return 0.f;
  float dE;
  if (kE <= h.breakE) {
    dE = kE * nieminen_factor(h.gamma15 * len * kE * fsqrt(kE));
  } else {
    const float loss = fdiv(joy_luo_sum(c, h, kE) * len, kE);
    dE = -loss;
    if (loss > 0.1f * kE) dE = csd_compute_split(c, h, len, kE);
  }
  return dE;
}

MD float csd_compute_split(const MONSEL_CS DCSD& c, const CSDHead& h, float len, float kE) {
#pragma clang fp contract(off)
  float E = kE, total = 0.f;
  uint32_t pending = 0;
  int d = 0;
  for (int it = 0; it < 128; ++it) {
    const float seg = ldexpf(len, -d);
    float dE = 0.f;
    if (!((E < h.minE) | (E <= 0.f))) {
      if (E <= h.breakE) {
        dE = E * nieminen_factor(h.gamma15 * seg * E * fsqrt(E));
      } else {
        const float loss = fdiv(joy_luo_sum(c, h, E) * seg, E);
        if (loss > 0.1f * E && d < 30) {
          pending |= 1u << (d + 1);
          d += 1;
          continue;
        }
        dE = -loss;
      }
    }
    E += dE;
    total += dE;
    if (pending == 0) break;
    d = 31 - __clz(pending);
    pending &= ~(1u << d);
  }
  return total;
}

/* ------------------------------------------------------- NU tables ----- */

/* Non-uniform table interpolation, generic over the arithmetic type T:
 * float for the inelastic mean free path (a well-conditioned 1-D lookup),
 * double for the tabulated scatter, whose 3-D angle lookup in reference
 * mode extrapolates a cubic far outside its abscissae
 * (NULagrangeInterpolation.cu:236) with weights up to ~1e7, so that FP32
 * rounding of the table values would change the result. */
MD const double* nu_axis(const DevScene& S, const MONSEL_CS DNUAxis& a) { return (const double*)(S.nu_words + a.x); }

/* NULagrangeInterpolation::locate (NULagrangeInterpolation.cu:5-68) on an
 * ascending or descending grid: first index of the order+1 window. */
template <typename T>
MD int nu_locate(const double* xs64, int n, int order, T x) {
  const auto xs = [=](int i) { return (T)xs64[i]; };
  int lowlim = -1, uplim = n, maxindex = n - 1;
  bool asc = xs(maxindex) > xs(0);
  while (uplim - lowlim > 1) {
    int mid = (uplim + lowlim) >> 1;
    if ((x > xs(mid)) == asc) lowlim = mid;
    else uplim = mid;
  }
  if (lowlim < 0) return 0;
  if (uplim > maxindex) return maxindex - order;
  T xl = xs(lowlim), xu = xs(uplim);
  int first = lowlim, last = uplim;
  while ((last - first) < order && first > 0 && last < maxindex) {
    if ((((xl - xs(first - 1)) + xu) - xs(last + 1) >= (T)0) == asc) last += 1;
    else first -= 1;
  }
  if (last >= maxindex) return maxindex - order;
  if (first <= 0) return 0;
  return first;
}

/* Lagrange basis weights of the ORDER+1 abscissae xs[0..ORDER] at x: the
 * interpolant sum_i w_i f_i is the polynomial Neville's scheme
 * (NULagrangeInterpolation.cu:85-112) evaluates.  Weights are formed once
 * per axis and shared by every row of a multi-dimensional window. */
template <typename T, int ORDER>
MD void nu_weights(const double* xs, T x, T* w) {
  /* differences are taken in units of the window's span, so that products
   * of ORDER of them stay far from underflow whatever the grid's units
   * (energies in J are ~1e-17) */
  T xv[ORDER + 1];
#pragma unroll
  for (int i = 0; i <= ORDER; ++i) xv[i] = (T)xs[i];
  const T inv = (T)1 / (xv[ORDER] - xv[0]);
#pragma unroll
  for (int i = 0; i <= ORDER; ++i) {
    T num = 1, den = 1;
#pragma unroll
    for (int j = 0; j <= ORDER; ++j)
      if (j != i) {
        num *= (x - xv[j]) * inv;
        den *= (xv[i] - xv[j]) * inv;
      }
    w[i] = num / den;
  }
}

template <typename T, int ORDER>
MD T nu_dot(const T* w, const T* f) {
  T y = 0;
#pragma unroll
  for (int i = 0; i <= ORDER; ++i) y += w[i] * f[i];
  return y;
}

template <typename T, int ORDER>
MD T nu_poly(const double* xs, const T* f, T x) {
  T w[ORDER + 1];
  nu_weights<T, ORDER>(xs, x, w);
  return nu_dot<T, ORDER>(w, f);
}

/* NULagrangeInterpolation::d1 (:144-158). */
template <int ORDER>
MD float nu_d1(const DevScene& S, const MONSEL_CS DNUTable& t, float x0) {
  const double* xa = nu_axis(S, t.axis[0]);
  int i0 = nu_locate<float>(xa, t.axis[0].n, ORDER, x0);
  return nu_poly<float, ORDER>(xa + i0, (const float*)(S.nu_data + t.voff + i0), x0);
}

/* NULagrangeInterpolation::d2 (:169-192); values are an [na][nb] block. */
template <int ORDER>
MD double nu_d2(const DevScene& S, const MONSEL_CS DNUTable& t, double x0, double x1) {
  const double* xa = nu_axis(S, t.axis[0]);
  const double* xb = nu_axis(S, t.axis[1]);
  const double* f = (const double*)(S.nu_data64 + t.voff);
  const int nb = t.axis[1].n;
  int i0 = nu_locate<double>(xa, t.axis[0].n, ORDER, x0);
  int j0 = nu_locate<double>(xb, nb, ORDER, x1);
  double wb[ORDER + 1], y[ORDER + 1];
  nu_weights<double, ORDER>(xb + j0, x1, wb);
#pragma unroll
  for (int i = 0; i <= ORDER; ++i) y[i] = nu_dot<double, ORDER>(wb, f + (size_t)(i0 + i) * nb + j0);
  return nu_poly<double, ORDER>(xa + i0, y, x0);
}

/* NULagrangeInterpolation::d3 (:215-240); compat_d3 reproduces line 236
 * (outer abscissae taken from the start of the grid).  voff overrides the
 * value offset (the 4-D lookup walks 3-D slices). */
template <int ORDER>
MD double nu_d3(const DevScene& S, const MONSEL_CS DNUTable& t, int ax, int voff, double x0, double x1, double x2, bool compat_d3) {
  const double* xa = nu_axis(S, t.axis[ax]);
  const double* xb = nu_axis(S, t.axis[ax + 1]);
  const double* xc = nu_axis(S, t.axis[ax + 2]);
  const double* v = (const double*)(S.nu_data64 + voff);
  const int nb = t.axis[ax + 1].n, nc = t.axis[ax + 2].n;
  int i0 = nu_locate<double>(xa, t.axis[ax].n, ORDER, x0);
  int j0 = nu_locate<double>(xb, nb, ORDER, x1);
  int k0 = nu_locate<double>(xc, nc, ORDER, x2);
  double wb[ORDER + 1], wc[ORDER + 1], y[ORDER + 1];
  nu_weights<double, ORDER>(xb + j0, x1, wb);
  nu_weights<double, ORDER>(xc + k0, x2, wc);
#pragma unroll 1
  for (int i = 0; i <= ORDER; ++i) {
    double z[ORDER + 1];
    const double* blk = v + (size_t)(i0 + i) * nb * nc;
#pragma unroll 1
    for (int j = 0; j <= ORDER; ++j) {
      const double zj = nu_dot<double, ORDER>(wc, blk + (size_t)(j0 + j) * nc + k0);
#pragma unroll
      for (int q = 0; q <= ORDER; ++q)
        if (q == j) z[q] = zj;
    }
    const double yi = nu_dot<double, ORDER>(wb, z);
#pragma unroll
    for (int q = 0; q <= ORDER; ++q)
      if (q == i) y[q] = yi;
  }
  return nu_poly<double, ORDER>(compat_d3 ? xa : xa + i0, y, x0);
}

/* NULagrangeInterpolation::d4 (:259-306). */
template <int ORDER>
MD double nu_d4(const DevScene& S, const MONSEL_CS DNUTable& t, const double* x, bool compat_d3) {
  const double* xa = nu_axis(S, t.axis[0]);
  int i0 = nu_locate<double>(xa, t.axis[0].n, ORDER, x[0]);
  double y[ORDER + 1];
#pragma unroll
  for (int i = 0; i <= ORDER; ++i)
    y[i] = nu_d3<ORDER>(S, t, 1, t.voff + (i0 + i) * t.axis[1].n * t.axis[2].n * t.axis[3].n, x[1], x[2], x[3], compat_d3);
  return nu_poly<double, ORDER>(xa + i0, y, x[0]);
}

template <int ORDER>
MD double nu_interp_o(const DevScene& S, const MONSEL_CS DNUTable& t, const double* x, bool compat_d3) {
  if (t.dim == 2) return nu_d2<ORDER>(S, t, x[0], x[1]);
  if (t.dim == 3) return nu_d3<ORDER>(S, t, 0, t.voff, x[0], x[1], x[2], compat_d3);
  return nu_d4<ORDER>(S, t, x, compat_d3);
}

/* The lookups of the transport step: FP64 cubic in two and three dimensions,
 * FP32 linear in one, with the bits of nu_d2, nu_d3 and nu_d1 above.  Through
 * those, an axis took a bisection of seven dependent reads of device memory
 * and four more for the window, and a window nine double divisions; tabulated
 * scatter was 55 to 65 % of a step with it, and a bulk run of few primaries is
 * a chain of steps.  Here the axes of a lookup are searched together, in LDS,
 * from the bounds their guides give (mostly one probe each), the window of an
 * interval is a word beside them, and what the weights hold of the axis alone
 * comes in a DNUWindow.  Transport of 3001 primaries of 5 keV in Cu, with the
 * spread of small launches: 19.7 ms to 4.7; of 400,000 of 1 keV in Si 71 to 39. */
template <typename T, int A, class P>
MD void nu_search(P w, const MONSEL_CS DNUAxis* ax, const T* x, int* lo, int* first) {
  int up[A];
  bool more = false;
#pragma unroll
  for (int k = 0; k < A; ++k) {
    const double xk = (double)x[k];
    const double v = ax[k].log ? (double)__double2hiint(xk) : xk;
    const double h = fmin(fmax((v - ax[k].origin) * ax[k].scale, 0.), ax[k].last);
    const unsigned long long g = w[ax[k].guide + (xk == xk ? (int)h : 0)];
    lo[k] = (int)(unsigned int)g;
    up[k] = (int)(unsigned int)(g >> 32);
    more |= up[k] - lo[k] > 1;
  }
  bool asc[A];
#pragma unroll
  for (int k = 0; k < A; ++k) asc[k] = (ax[k].asc & (sizeof(T) == 8 ? 1 : 2)) != 0;
  while (more) {
    more = false;
#pragma unroll
    for (int k = 0; k < A; ++k) {
      const int mid = (up[k] + lo[k]) >> 1;
      const T xm = (T)__longlong_as_double((long long)w[ax[k].x + max(mid, 0)]);
      const bool above = (x[k] > xm) == asc[k], open = up[k] - lo[k] > 1;
      lo[k] = (open & above) ? mid : lo[k];
      up[k] = (open & !above) ? mid : up[k];
      more |= up[k] - lo[k] > 1;
    }
  }
#pragma unroll
  for (int k = 0; k < A; ++k) first[k] = (int)w[ax[k].first + lo[k]];
}

template <int A>
MD void nu_find(const DevScene& S, const MONSEL_CS DNUAxis* ax, const double* x, int* lo, int* first) {
  if (S.n_nu_words <= kLdsNuWords)
    nu_search<double, A>((const unsigned long long*)lds_nu_words(), ax, x, lo, first);
  else
    nu_search<double, A>(S.nu_words, ax, x, lo, first);
}

/* num / den, correctly rounded, from y = 1 / den correctly rounded (Markstein:
 * a quotient within one unit and its exact remainder; the first correction
 * brings the product within that unit, the second rounds it) */
MD double nu_quotient(double num, double den, double y) {
  double q = num * y;
  q = __builtin_fma(__builtin_fma(-den, q, num), y, q);
  q = __builtin_fma(__builtin_fma(-den, q, num), y, q);
  return __builtin_amdgcn_div_fixup(q, den, num);
}

/* nu_weights<double, 3> over the window of a record */
MD void nu_cubic_weights(const MONSEL_CS DNUWindow& r, double x, double* w) {
  double d[4], den[4], rden[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    d[j] = (x - r.x[j]) * r.inv;
    den[j] = r.den[j];
    rden[j] = r.rden[j];
  }
  w[0] = nu_quotient((d[1] * d[2]) * d[3], den[0], rden[0]);
  w[1] = nu_quotient((d[0] * d[2]) * d[3], den[1], rden[1]);
  w[2] = nu_quotient((d[0] * d[1]) * d[3], den[2], rden[2]);
  w[3] = nu_quotient((d[0] * d[1]) * d[2], den[3], rden[3]);
}

MD double nu_cubic2(const DevScene& S, const MONSEL_CS DNUTable& t, double x0, double x1) {
  const MONSEL_CS DNUAxis* ax = t.axis;
  const double x[2] = {x0, x1};
  int lo[2], first[2];
  nu_find<2>(S, ax, x, lo, first);
  const int nb = ax[1].n;
  const MONSEL_CS double* f = S.nu_data64 + t.voff + (size_t)first[0] * nb + first[1];
  double v[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) v[i][j] = f[(size_t)i * nb + j];
  double wa[4], wb[4], y[4];
  nu_cubic_weights(S.nu_recs[ax[1].rec + lo[1]], x1, wb);
  nu_cubic_weights(S.nu_recs[ax[0].rec + lo[0]], x0, wa);
#pragma unroll
  for (int i = 0; i < 4; ++i) y[i] = nu_dot<double, 3>(wb, v[i]);
  return nu_dot<double, 3>(wa, y);
}

MD double nu_cubic3(const DevScene& S, const MONSEL_CS DNUTable& t, double x0, double x1, double x2, bool compat_d3) {
  const MONSEL_CS DNUAxis* ax = t.axis;
  const double x[3] = {x0, x1, x2};
  int lo[3], first[3];
  nu_find<3>(S, ax, x, lo, first);
  const int nb = ax[1].n, nc = ax[2].n;
  const MONSEL_CS double* f = S.nu_data64 + t.voff + ((size_t)first[0] * nb + first[1]) * nc + first[2];
  double wa[4], wb[4], wc[4], y = 0.;
  nu_cubic_weights(S.nu_recs[ax[2].rec + lo[2]], x2, wc);
  nu_cubic_weights(S.nu_recs[ax[1].rec + lo[1]], x1, wb);
  nu_cubic_weights(S.nu_recs[ax[0].rec + (compat_d3 ? -1 : lo[0])], x0, wa);
  /* one outer point at a time: with the sixteen values of a point, or of two,
   * loaded together and the windows beside them the registers spill (9 % more
   * time for 400,000 primaries in Si) */
#pragma unroll 1
  for (int i = 0; i < 4; ++i) {
    double z[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      double v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = f[(size_t)j * nc + k];
      z[j] = nu_dot<double, 3>(wc, v);
    }
    y = __builtin_fma(wa[0], nu_dot<double, 3>(wb, z), y);
    wa[0] = wa[1];
    wa[1] = wa[2];
    wa[2] = wa[3];
    f += (size_t)nb * nc;
  }
  return y;
}

MD float nu_linear1(const DevScene& S, const MONSEL_CS DNUTable& t, float x) {
  const MONSEL_CS DNUAxis* ax = t.axis;
  int lo, first;
  if (S.n_nu_words <= kLdsNuWords)
    nu_search<float, 1>((const unsigned long long*)lds_nu_words(), ax, &x, &lo, &first);
  else
    nu_search<float, 1>(S.nu_words, ax, &x, &lo, &first);
  const int i0 = min(max(lo, 0), ax->n - 2);
  return nu_poly<float, 1>(nu_axis(S, *ax) + i0, (const float*)(S.nu_data + t.voff + i0), x);
}

/* NUTableInterpolation::interpolate (NUTableInterpolation.cu:98-115) in
 * the arithmetic the transport uses for that table's dimension: FP32 for
 * 1-D (mean free path), FP64 otherwise. */
MD double nu_interp(const DevScene& S, int table, int order, const double* x, bool compat_d3) {
  const MONSEL_CS DNUTable& t = S.nu[table];
  if (t.dim == 1) {
    const float xf = (float)x[0];
    if (order == 1) return nu_linear1(S, t, xf);
    return order == 2 ? nu_d1<2>(S, t, xf) : nu_d1<3>(S, t, xf);
  }
  if (order == 1) return nu_interp_o<1>(S, t, x, compat_d3);
  if (order == 2) return nu_interp_o<2>(S, t, x, compat_d3);
  if (t.dim == 2) return nu_cubic2(S, t, x[0], x[1]);
  if (t.dim == 3) return nu_cubic3(S, t, x[0], x[1], x[2], compat_d3);
  return nu_d4<3>(S, t, x, compat_d3);
}

/* ------------------------------------------------------ mechanisms ----- */

MD float elastic_rate(const DevScene& S, const MONSEL_CS DMech& m, float EeV) {
  float tot = 0.f;
  if (m.few) {
    float c[kFewElem];
    elastic_terms_few(S, m, EeV, c);
    tot = (c[0] + c[1]) + c[2];
  } else {
    elastic_terms(S, m, EeV, [&](int, float c) { tot += c; });
  }
  return tot;
}

/* ScatterMechanism::scatterRate (1/nm); TAB as for mech_scatter */
template <bool TAB = true>
MD float mech_rate(const DevScene& S, const MONSEL_CS DMech& m, float EeV) {
  int kind = m.kind;
  float p0 = m.p[0], p1 = m.p[1], p2 = m.p[2];
  pin(kind, p0, p1, p2);
  switch (kind) {
    case MONSEL_MECH_NISTMOTT_ELASTIC:
    case MONSEL_MECH_BROWNING_ELASTIC:
    case MONSEL_MECH_RUTHERFORD_ELASTIC:
      return elastic_rate(S, m, EeV);
    case MONSEL_MECH_FITTED_INELASTIC: /* FittedInelSM.cu:20-25 */
      if (EeV <= p0) return 0.f;
      return -csd_compute(m.csd, 0.1f, EeV) * 10.f * p2;
    case MONSEL_MECH_POLARON_TRAP: /* GanachaudMokraniPolaronTrapSM.cu:21-27 */
      if (EeV > p2) return 0.f;
      return p0 * fexp(-p1 * EeV);
    case MONSEL_MECH_PHONON: { /* GanachaudMokraniPhononInelasticSM.cu:46-72 */
      if (EeV < p0) return 0.f;
      const float x = fdiv(p0, EeV);
      const float temp = fsqrt(1.f - x);
      const bool small = x < 0.1f;
      const float rate = p1 * x * flog(fdiv(small ? 4.f : 1.f + temp, small ? x : 1.f - temp));
      return small || !(x >= 1.f) ? rate : 0.f;
    }
    case MONSEL_MECH_TABULATED_INELASTIC: if constexpr (TAB) { /* TabulatedInelasticSM.cu:436-459 */
      float kE = (EeV + m.p[TP_OFFSET]) * kEcharge;
      if (kE < m.p[TP_IIMFPDOM0]) return 0.f;
      return m.p[TP_RATEMULT] * nu_linear1(S, S.nu[m.table[0]], kE) * 1.0e-9f;
    }
  }
  return 0.f;
}

/* secondary produced by a scatter event (new Electron(*pe, theta, phi, E)
 * followed by an optional relative rotation) */
struct Spawn {
  uint32_t has; /* 0 or 1 (a bool kept across branches costs scalar mask merges) */
  float dx, dy, dz;
  float E;
};

/* TabulatedInelasticSM.cu:103-151 (energies in J) */
MD float e0_from_dispersion(float Eq, float deltaE) {
  if (Eq == 0.f) return deltaE;
  float x = Eq / deltaE;
  float y = 3.77300614251479e17f * Eq;
  float x13 = cbrtf(x);
  float x2 = x * x;
  float c1 = x2 * x2 * (27.f + (18.f * y) + (2.f * y * y));
  float c2 = x2 * (27.f + (4.f * y));
  float c3 = c2 - 27.f;
  float c4 = x2 * (3.f + y);
  float c6 = 1.f - x2;
  if (c3 > 0.f) {
    float tanPart = atan2f(3.f * c6 * sqrtf(3.f * c3 * c6), (18.f * c4) - c1 - 27.f);
    float trigPart = cosf(tanPart / 3.f);
    float prefactor = 2.f * x * sqrtf(y * (y - (c6 * (y + 6.f))));
    trigPart *= prefactor;
    return deltaE * sqrtf(((3.f - c4) + trigPart) / 3.f);
  }
  float c5 = cbrtf(-c1 + (18.f * c4) + (3.f * (-9.f + (c6 * sqrtf(-(3.f * c3 * c6))))));
  float term1 = -2.f * c4;
  float x23 = x13 * x13;
  float x43 = x * x13;
  float y13 = cbrtf(y);
  float y23 = y13 * y13;
  float x43y23 = x43 * y23;
  float two13 = 1.2599210498948732f;
  float term2 = -12.f * two13 * x43y23 * c6;
  float term3 = 2.f * two13 * x43y23 * x2 * y;
  float term23 = (term2 + term3) / c5;
  float term4 = two13 * two13 * x23 * y13 * c5;
  return deltaE * sqrtf((6.f + term1 + term23 + term4) / 6.f);
}

/* TabulatedInelasticSM::pickBE (:153-207), default branching ratios; J. */
MD double pick_be(const MONSEL_CS DMech& m, double Eq, double deltaE) {
  const int ncore = (int)m.q[TP_NCORE];
  if (ncore > 0 && deltaE <= m.q[TP_CORE0]) return 0.;
  const double eIon = m.q[TP_E0DISP] != 0. ? (double)e0_from_dispersion((float)Eq, (float)deltaE) : deltaE;
  int i = 0;
  while (i < ncore && m.q[TP_CORE0 + i] <= eIon) ++i;
  return i == 0 ? 0. : m.q[TP_CORE0 + i - 1];
}

MD void isotropic_dir(float u1, float u2, float& dx, float& dy, float& dz) {
  /* theta = acos(1 - 2 u1), phi = 2 pi u2 */
  float ct = 1.f - 2.f * u1;
  float st = fsqrt(fmaxf(0.f, 1.f - ct * ct));
  float sp, cp;
  __sincosf(kTwoPI * u2, &sp, &cp);
  dx = st * cp;
  dy = st * sp;
  dz = ct;
}

/* TabulatedInelasticSM::scatter (TabulatedInelasticSM.cu:209-434) in FP64,
 * in the reference's SI units (J); only the final rotations are FP32.  The
 * parameters come from DMech::q (J). */
MD Spawn tabulated_scatter(const DevScene& S, const MONSEL_CS DMech& m, Elec& e, const float* u) {
  Spawn se;
  se.has = 0u;
  const bool cd3 = (S.compat & MONSEL_COMPAT_D3_ABSCISSAE) != 0;
  const double J = 1.60217653e-19;
  const double kE0 = (double)e.E * J;
  const double kE = kE0 + m.q[TP_OFFSET];
  if (kE < m.q[TP_EIDOM0]) return se;
  const double rnd0 = u[2], rnd1 = u[3], rnd2 = u[4], rnd3 = u[5];
  double deltaE = kE * nu_cubic2(S, S.nu[m.table[1]], kE, rnd0);
  const double gap = m.q[TP_GAP], bandgap = m.q[TP_BANDGAP];
  if (deltaE < gap && deltaE > 0.95 * gap) deltaE = gap;
  const float d0x = e.dx, d0y = e.dy, d0z = e.dz;
  double theta = 0.;
  float sphi = 0.f, cphi = 1.f;
  const double offsetFermi = m.q[TP_OFFSETFERMI];
  if (deltaE >= bandgap) {
    double red = (deltaE - gap) / (kE - offsetFermi - 2. * gap);
    red = red > 1. ? 1. : (red < 0. ? 0. : red);
    theta = nu_cubic3(S, S.nu[m.table[2]], kE, red, rnd1, cd3);
    __sincosf(kTwoPI * (float)rnd2, &sphi, &cphi);
    float st, ct;
    sincosf((float)theta, &st, &ct);
    rotate_dir(e.dx, e.dy, e.dz, ct, st, cphi, sphi);
  }
  e.E = (float)((kE0 - deltaE) / J);
  if (deltaE < bandgap) return se;
  const double Eq = (2. * kE) - deltaE - (2. * sqrt(kE * (kE - deltaE)) * (double)cosf((float)theta));
  const double cb = m.q[TP_CB], minEgen = m.q[TP_MINEGEN], bEref = m.q[TP_BEREF];
  const double offset = m.q[TP_OFFSET];
  const int method = m.method;
  const double be = pick_be(m, Eq, deltaE);
  const double root = 2. * sqrt(offsetFermi * (offsetFermi + deltaE));
  const double sum = (2. * offsetFermi) + deltaE;
  /* the source of the SE's energy: a bound level, the band (method 3 where the
   * momentum transfer allows it) or the table; one lookup serves both methods */
  const bool bound = method == 1 || be > 0.;
  const bool band = !bound && method == 3 && (sum - root) <= Eq && Eq <= (sum + root);
  double energySE = (deltaE + bEref) - be;
  float thSE = 0.f;
  if (band) {
    /* simESEf (TabulatedInelasticSM.cu:87-101) */
    const double q = sqrt(Eq);
    const double kz = (deltaE - Eq) / 2. / q;
    const double kzf = kz + q;
    const double Ezq = kzf * kzf;
    double minE = (offsetFermi + bandgap) - Ezq;
    if (minE < 0.) minE = 0.;
    const double maxE = offsetFermi - (kz * kz);
    const double Exy = (minE * (1. - rnd3)) + (maxE * rnd3);
    const double ESEf = Exy + Ezq;
    thSE = acosf((float)(kzf / sqrt(ESEf)));
    energySE = ESEf - offset;
  } else if (!bound) {
    double e0 = nu_cubic2(S, S.nu[m.table[3]], deltaE, rnd3);
    if (e0 < m.q[TP_SE0RANGE0]) e0 = m.q[TP_SE0RANGE0];
    else if (e0 > m.q[TP_SE0RANGE1]) e0 = m.q[TP_SE0RANGE1];
    energySE = (deltaE + e0) - offset;
  }
  if (energySE + cb < minEgen) return se;
  if (method == 3 && !band) {
    isotropic_dir(u[6], u[7], se.dx, se.dy, se.dz);
  } else {
    /* SE direction relative to the PE's original direction: thetaSE = pi/2 -
     * theta, phiSE = phi + pi */
    float st, ct, sp = -sphi, cp = -cphi;
    sincosf((float)(0.5 * 3.14159265358979323846 - theta), &st, &ct);
    if (band) {
      /* TabulatedInelasticSM.cu:388-395: the q-vector direction (pi/2 - theta,
       * phi + pi) is deflected by (thSE, 2 pi U) in the PE frame, and the SE
       * is the PE's original direction rotated by the resulting angles. */
      float wx, wy, wz;
      dir_from_angles(ct, st, cp, sp, wx, wy, wz);
      float sp2, cp2, st2, ct2;
      __sincosf(kTwoPI * u[6], &sp2, &cp2);
      sincosf(thSE, &st2, &ct2);
      rotate_dir(wx, wy, wz, ct2, st2, cp2, sp2);
      const float wst = fsqrt(fmaxf(0.f, wx * wx + wy * wy));
      cp = 1.f;
      sp = 0.f;
      if (wst > 0.f) {
        cp = wx / wst;
        sp = wy / wst;
      }
      ct = wz;
      st = wst;
    }
    se.dx = d0x;
    se.dy = d0y;
    se.dz = d0z;
    rotate_dir(se.dx, se.dy, se.dz, ct, st, cp, sp);
  }
  se.has = 1u;
  se.E = (float)(energySE / J);
  return se;
}

/* The pick-th of three wave-uniform values.  They are held in scalar
 * registers first: left to itself the compiler selects among their addresses
 * and loads per lane. */
template <class T>
MD T of_three(int pick, T a, T b, T c) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm("" : "+s"(a), "+s"(b), "+s"(c));
#endif
  return pick == 0 ? a : (pick == 1 ? b : c);
}

/* A deflection of the electron's direction left for the end of the scatter:
 * polar angle by its cosine, azimuth by its uniform. */
struct Deflect {
  uint32_t has;
  float cos_polar, u_azimuth;
};

/* Electron::updateDirection by d */
MD void deflect(Elec& e, const Deflect& d) {
  const float ca = fminf(1.f, fmaxf(-1.f, d.cos_polar));
  const float sa = fsqrt(fmaxf(0.f, 1.f - ca * ca));
  float sb, cb;
  __sincosf(kTwoPI * d.u_azimuth, &sb, &cb);
  rotate_dir(e.dx, e.dy, e.dz, ca, sa, cb, sb);
}

/* ScatterMechanism::scatter of mechanism m (the same one on every active
 * lane).  `rate` is this mechanism's scatterRate at prevE, as summed when the
 * step's free path was drawn; esig, if given, holds the elastic mechanism's
 * first two terms if it has no more than kFewElem elements (lane stride
 * kLaneBlock); draw_hi(u) draws u[4..7].
 * A deflection of the primary is left in `de` for the caller, which applies
 * it once for every mechanism.  TAB = false leaves the tabulated mechanism
 * out of the code (its FP64 scatter sets the register budget of every kernel
 * that contains it); only for scenes without one. */
template <bool TAB = true, class Draw>
MD Spawn mech_scatter(const DevScene& S, const MONSEL_CS DMech& m, Elec& e, float prevE, float rate, bool& trapped,
                      float* u, Draw draw_hi, Deflect& de, const float* esig = nullptr) {
  Spawn se;
  se.has = 0u;
  switch (m.kind) {
    case MONSEL_MECH_NISTMOTT_ELASTIC:
    case MONSEL_MECH_BROWNING_ELASTIC:
    case MONSEL_MECH_RUTHERFORD_ELASTIC: { /* SelectableElasticSM.cu:49-67 */
      PT_BEGIN(t_el);
      /* first element whose running sum of sigma * atoms reaches u * rate
       * (the last if none does); the sum is re-formed in the order
       * elastic_rate formed it */
      const float r = u[2] * rate;
      const bool nist = m.kind == MONSEL_MECH_NISTMOTT_ELASTIC;
      int pick = 0;
      if (m.few) {
        if (m.nelem > 1) {
          float c[kFewElem];
          if (esig) {
            c[0] = esig[0];
            c[1] = esig[kLaneBlock];
          } else {
            elastic_terms_few(S, m, prevE, c);
          }
          const bool past0 = c[0] < r, past1 = past0 & (m.nelem > 2) & (c[0] + c[1] < r);
          pick = past1 ? 2 : (past0 ? 1 : 0);
        }
      } else {
        float cum = 0.f;
        elastic_terms(S, m, prevE, [&](int i, float c) {
          if (i < m.nelem - 1) {
            cum += c;
            if (pick == i && cum < r) pick = i + 1;
          }
        });
      }
      draw_hi(u);
      /* the polar angle takes one uniform (two for Browning), the azimuth
       * the next one (SelectableElasticSM.cu:62-64) */
      de.has = 1u;
      de.u_azimuth = u[4];
      if (m.kind == MONSEL_MECH_BROWNING_ELASTIC || (nist && prevE < m.extrap)) {
        float z, zp3;
        if (m.few) {
          z = of_three(pick, m.el.z[0], m.el.z[1], m.el.z[2]);
          zp3 = of_three(pick, m.el.zp3[0], m.el.zp3[1], m.el.zp3[2]);
        } else {
          z = S.elems[m.elem0 + pick].z;
          zp3 = S.elems[m.elem0 + pick].zp3;
        }
        de.cos_polar = browning_cos(z, zp3, prevE, u[3], u[4]);
        de.u_azimuth = u[5];
      } else if (nist && !(prevE >= kMaxNISTMott)) {
        const int x1 = m.few ? of_three(pick, m.el.x1[0], m.el.x1[1], m.el.x1[2])
                             : S.elems[m.elem0 + pick].mott * (kMottNE * kMottNQ);
        de.cos_polar = mott_cos(S, x1, prevE, u[3]);
      } else {
        de.cos_polar = rutherford_cos(S.elems[m.elem0 + pick].rz23, prevE, u[3]);
      }
      PT_END(PH_ELASTIC, t_el);
      return se;
    }
    case MONSEL_MECH_FITTED_INELASTIC: { /* FittedInelSM.cu:13-18 */
      PT_BEGIN(t_fi);
      float u_phi = u[2];
      float u_th = u[3];
      isotropic_dir(u_th, u_phi, se.dx, se.dy, se.dz);
      se.E = m.p[1];
      se.has = 1u;
      PT_END(PH_FITTED, t_fi);
      return se;
    }
    case MONSEL_MECH_POLARON_TRAP: { /* GanachaudMokraniPolaronTrapSM.cu:15-20 */
      PT_BEGIN(t_po);
      e.E = 0.f;
      trapped = true;
      PT_END(PH_POLARON, t_po);
      return se;
    }
    case MONSEL_MECH_PHONON: { /* GanachaudMokraniPhononInelasticSM.cu:19-44 */
      PT_BEGIN(t_ph);
      float kE0 = e.E;
      if (kE0 < m.p[0]) {
        PT_END(PH_PHONON, t_ph);
        return se;
      }
      float x = fdiv(m.p[0], kE0);
      const float r0 = u[2], r1 = u[3];
      float ct;
      /* x^a = 2^(a log2 x) for x > 0, on the hardware exp2/log2 */
      if (x < 0.1f)
        ct = 1.f + ((x * x) - __builtin_amdgcn_exp2f(
                                  __builtin_fmaf(2.f - 2.f * r0, __builtin_amdgcn_logf(x), 4.f * r0))) / 8.f;
      else {
        float root = fsqrt(1.f - x);
        float temp = __builtin_amdgcn_exp2f(
            r0 * __builtin_amdgcn_logf(fdiv((-2.f * (1.f + root)) + x, (-2.f * (1.f - root)) + x)));
        ct = temp + fdiv(((x - 2.f) * (temp - 1.f)) / 2.f, root);
      }
      de.has = 1u;
      de.cos_polar = ct;
      de.u_azimuth = r1;
      e.E = kE0 - m.p[0];
      PT_END(PH_PHONON, t_ph);
      return se;
    }
    case MONSEL_MECH_TABULATED_INELASTIC:
      if constexpr (TAB) {
        PT_BEGIN(t_tb);
        draw_hi(u);
        Spawn r = tabulated_scatter(S, m, e, u);
        PT_END(PH_TABULATED, t_tb);
        return r;
      }
      break;
  }
  return se;
}

/* --------------------------------------------------------- geometry ---- */

struct Interval {
  float tin, tout;
  int fin, fout; /* face codes: plane index, or -1 cap0 / -2 cap1 / -3 side */
};

/* NormalMultiPlaneShape.cu:26-38: whether a line within the plane of normal
 * (nx, ny, nz) counts as inside */
inline __host__ __device__ bool plane_tie_break(float nx, float ny, float nz) {
  if (nx < 0.f) return false;
  if (nx == 0.f) {
    if (ny < 0.f) return false;
    if (ny == 0.f && nz < 0.f) return false;
  }
  return true;
}

/* plane k of a multi-plane primitive (k may differ by lane) */
MD float4 prim_plane(const DevScene& S, const MONSEL_CS DPrim& pr, int k) {
  return k < kInlinePlanes ? pr.pl[k] : S.planes[pr.first_plane + k];
}

/* f(plane, k) for every plane of a wave-uniform multi-plane primitive; the
 * first four are loaded together (a slot beyond the last plane is 0) */
template <class F>
MD void for_planes(const DevScene& S, const MONSEL_CS DPrim& pr, F f) {
  float4 a = pr.pl[0], b = pr.pl[1], c = pr.pl[2], d = pr.pl[3];
  const int n = pr.n_planes;
  pin(a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, c.x, c.y, c.z, c.w, d.x, d.y, d.z, d.w);
  f(a, 0);
  if (n > 1) f(b, 1);
  if (n > 2) f(c, 2);
  if (n > 3) f(d, 3);
  for (int k = kInlinePlanes; k < n; ++k) f(S.planes[pr.first_plane + k], k);
}

/* Parameter interval of the line p + t d inside a convex primitive (empty
 * intervals come back with tin > tout).  The primitive is the same on every
 * active lane, so its kind and plane count branch uniformly; what differs by
 * lane is selected, not branched on. */
MD Interval prim_interval(const DevScene& S, const MONSEL_CS DPrim& pr, float px, float py, float pz, float dx, float dy,
                          float dz) {
  Interval iv;
  iv.tin = -kInf;
  iv.tout = kInf;
  iv.fin = iv.fout = -4;
  bool miss = false;
  if (pr.kind == PRIM_PLANES) {
    const int tie = pr.tie;
    auto plane = [&](const float4& pl, int k) {
      const float num = pl.x * px + pl.y * py + pl.z * pz - pl.w;
      const float den = pl.x * dx + pl.y * dy + pl.z * dz;
      const float t = fdiv(-num, den);
      /* parallel: inside the half space, or outside of it for good */
      const bool flat = den == 0.f;
      const bool in = (num < 0.f) | ((num == 0.f) & (((tie >> k) & 1) != 0));
      miss = miss | (flat & !in);
      const bool leaves = (den > 0.f) & (t < iv.tout);
      const bool enters = !flat & !(den > 0.f) & (t > iv.tin);
      iv.tout = leaves ? t : iv.tout;
      iv.fout = leaves ? k : iv.fout;
      iv.tin = enters ? t : iv.tin;
      iv.fin = enters ? k : iv.fin;
    };
    for_planes(S, pr, plane);
  } else if (pr.kind == PRIM_CYLINDER) {
    float wx = px - pr.e0[0], wy = py - pr.e0[1], wz = pz - pr.e0[2];
    float apar = wx * pr.ax[0] + wy * pr.ax[1] + wz * pr.ax[2];
    float dpar = dx * pr.ax[0] + dy * pr.ax[1] + dz * pr.ax[2];
    const float inv = __builtin_amdgcn_rcpf(dpar);
    const float t0 = -apar * inv, t1 = (pr.len - apar) * inv;
    const bool along = dpar > 0.f, flat = dpar == 0.f;
    const float sin_ = flat ? -kInf : (along ? t0 : t1), sout = flat ? kInf : (along ? t1 : t0);
    const int fsin = along ? -1 : -2, fsout = along ? -2 : -1;
    miss = flat & !((apar >= 0.f) & (apar <= pr.len));
    /* radial part from the components perpendicular to the axis */
    float qx = wx - apar * pr.ax[0], qy = wy - apar * pr.ax[1], qz = wz - apar * pr.ax[2];
    float vx = dx - dpar * pr.ax[0], vy = dy - dpar * pr.ax[1], vz = dz - dpar * pr.ax[2];
    float A = vx * vx + vy * vy + vz * vz;
    float B = qx * vx + qy * vy + qz * vz;
    float C = qx * qx + qy * qy + qz * qz - pr.r2;
    const bool slanted = A > 1e-12f;
    const float disc = B * B - A * C;
    miss = miss | (slanted ? disc < 0.f : C > 0.f);
    const float sq = fsqrt(disc);
    const float q = -(B + (B >= 0.f ? sq : -sq));
    const float ra = fdiv(q, A), rb = (q != 0.f) ? C * __builtin_amdgcn_rcpf(q) : ra;
    const float rin = slanted ? fminf(ra, rb) : -kInf, rout = slanted ? fmaxf(ra, rb) : kInf;
    const bool cap_in = sin_ >= rin, cap_out = sout <= rout;
    iv.tin = cap_in ? sin_ : rin;
    iv.fin = cap_in ? fsin : -3;
    iv.tout = cap_out ? sout : rout;
    iv.fout = cap_out ? fsout : -3;
  } else {
    float cx = px - pr.e0[0], cy = py - pr.e0[1], cz = pz - pr.e0[2];
    float B = cx * dx + cy * dy + cz * dz;
    float C = cx * cx + cy * cy + cz * cz - pr.r2;
    const float disc = B * B - C;
    miss = disc < 0.f;
    const float sq = fsqrt(disc);
    iv.tin = -B - sq;
    iv.tout = -B + sq;
    iv.fin = iv.fout = -3;
  }
  iv.tin = miss ? kInf : iv.tin;
  iv.tout = miss ? -kInf : iv.tout;
  return iv;
}

/* Outward normal of primitive face `f` at point q. */
MD void prim_normal(const DevScene& S, const MONSEL_CS DPrim& pr, int f, float qx, float qy, float qz, float& nx, float& ny,
                    float& nz) {
  if (pr.kind == PRIM_PLANES) {
    float4 pl = prim_plane(S, pr, f < 0 ? 0 : f);
    nx = pl.x;
    ny = pl.y;
    nz = pl.z;
    return;
  }
  if (pr.kind == PRIM_CYLINDER) {
    if (f == -1) { nx = -pr.ax[0]; ny = -pr.ax[1]; nz = -pr.ax[2]; return; }
    if (f == -2) { nx = pr.ax[0]; ny = pr.ax[1]; nz = pr.ax[2]; return; }
    float wx = qx - pr.e0[0], wy = qy - pr.e0[1], wz = qz - pr.e0[2];
    float apar = wx * pr.ax[0] + wy * pr.ax[1] + wz * pr.ax[2];
    wx -= apar * pr.ax[0];
    wy -= apar * pr.ax[1];
    wz -= apar * pr.ax[2];
    float inv = __builtin_amdgcn_rsqf(wx * wx + wy * wy + wz * wz);
    nx = wx * inv;
    ny = wy * inv;
    nz = wz * inv;
    return;
  }
  float wx = qx - pr.e0[0], wy = qy - pr.e0[1], wz = qz - pr.e0[2];
  float inv = __builtin_amdgcn_rsqf(wx * wx + wy * wy + wz * wz);
  nx = wx * inv;
  ny = wy * inv;
  nz = wz * inv;
}

MD bool prim_contains(const DevScene& S, const MONSEL_CS DPrim& pr, float px, float py, float pz) {
  if (pr.kind == PRIM_PLANES) {
    /* MultiPlaneShape.cu:23-27 for every plane */
    bool in = true;
    for_planes(S, pr, [&](const float4& pl, int) { in = in & (pl.x * px + pl.y * py + pl.z * pz - pl.w <= 0.f); });
    return in;
  }
  float wx = px - pr.e0[0], wy = py - pr.e0[1], wz = pz - pr.e0[2];
  if (pr.kind == PRIM_CYLINDER) {
    /* CylindricalShape.cu:41-45 */
    float u = fdiv(pr.axv[0] * wx + pr.axv[1] * wy + pr.axv[2] * wz, pr.len2);
    float rx = wx - u * pr.axv[0], ry = wy - u * pr.axv[1], rz = wz - u * pr.axv[2];
    return (u >= 0.f) & (u <= 1.f) & ((rx * rx + ry * ry + rz * rz) <= pr.r2);
  }
  return wx * wx + wy * wy + wz * wz <= pr.r2;
}

/* the shape's truth value for the primitives' inside bits; a shape of at most
 * five primitives has its table in one (scalar) word */
MD bool truth(const MONSEL_CS DShape& sh, uint32_t bits) {
  uint32_t word = sh.truth[0];
  if (sh.n_prims > 5) word = sh.truth[bits >> 5];
  return (word >> (bits & 31u)) & 1u;
}

/* max_k g_k over a convex primitive's constraints, g_k the signed distance
 * to constraint k (plane rows scaled by sdscale <= 1/|n|): <= 0 inside.
 * Its magnitude bounds the distance from p to the primitive's surface from
 * below -- inside, -max g_k is the distance to the nearest face; outside,
 * max g_k is at most the distance to the primitive.  `in` receives the
 * primitive's inside bit as prim_contains computes it.  Planes: the same row
 * values.  A sphere or cylinder: the sign of the result, except within a band
 * of 1e-5 of the magnitudes involved around the surface -- far wider than the
 * few ulps by which the two formulas can round apart -- where prim_contains
 * itself decides. */
MD float prim_gmax_in(const DevScene& S, const MONSEL_CS DPrim& pr, float px, float py, float pz, bool& in) {
  if (pr.kind == PRIM_PLANES) {
    float g = -kInf;
    bool all = true;
    for_planes(S, pr, [&](const float4& pl, int) {
      const float v = pl.x * px + pl.y * py + pl.z * pz - pl.w;
      g = fmaxf(g, v);
      all = all & (v <= 0.f);
    });
    in = all;
    return g * pr.sdscale;
  }
  const float wx = px - pr.e0[0], wy = py - pr.e0[1], wz = pz - pr.e0[2];
  const float r = fsqrt(pr.r2);
  float g, scale;
  if (pr.kind == PRIM_CYLINDER) {
    const float apar = wx * pr.ax[0] + wy * pr.ax[1] + wz * pr.ax[2];
    const float qx = wx - apar * pr.ax[0], qy = wy - apar * pr.ax[1], qz = wz - apar * pr.ax[2];
    const float q = fsqrt(qx * qx + qy * qy + qz * qz);
    g = fmaxf(q - r, fmaxf(-apar, apar - pr.len));
    scale = q + fabsf(apar) + pr.len + r;
  } else {
    const float w = fsqrt(wx * wx + wy * wy + wz * wz);
    g = w - r;
    scale = w + r;
  }
  in = g <= 0.f;
  if (fabsf(g) <= 1e-5f * scale) in = prim_contains(S, pr, px, py, pz);
  return g;
}

MD bool shape_contains(const DevScene& S, const MONSEL_CS DShape& sh, float px, float py, float pz) {
  uint32_t bits = 0;
  for (int k = 0; k < sh.n_prims; ++k)
    if (prim_contains(S, S.prims[sh.first_prim + k], px, py, pz)) bits |= 1u << k;
  return truth(sh, bits);
}

/* whether some active lane of the wave has p */
MD bool wave_any(bool p) { return __builtin_amdgcn_ballot_w64(p) != 0ull; }

struct ShapeHit {
  float t;      /* kInf if none within tmax */
  float nx, ny, nz;
};

/* First boundary of the composite shape along p + t d, 0 < t <= tmax: the
 * walk visits the primitives' crossings in increasing t, toggling their
 * inside bits, until the truth table changes value.  Each pass over the
 * primitives forms their intervals and finds the next crossing after tcur;
 * a segment that ends before the first one, or crosses the boundary there,
 * takes one pass.  A crossing that leaves the truth value takes another, of
 * the primitives that have a crossing left on the segment of some lane still
 * walking (all primitives again: a shape of 8 parts 5 to 30 % slower, 1.6 M
 * primaries on random ones 20 to 37 ms instead of 16 to 30).  Forming the
 * intervals again keeps them out of LDS (20 KB per block of 256 lanes), which
 * held the kernel to 4 waves per SIMD.  The normal is formed only when asked
 * for.  Requires the same shape on every active lane. */
MD ShapeHit shape_first(const DevScene& S, const MONSEL_CS DShape& sh, float px, float py, float pz, float dx,
                        float dy, float dz, float tmax, bool want_normal) {
  ShapeHit h;
  h.t = kInf;
  h.nx = h.ny = h.nz = 0.f;
  const int n = sh.n_prims;
  const MONSEL_CS DPrim* prims = S.prims + sh.first_prim;
  uint32_t bits = 0;
  float tcur = 0.f;
  uint32_t live = (1u << n) - 1u;   /* primitives the next pass visits (wave-uniform) */
  bool inside = false, open = true;
  /* primitive and face of the lowest two indices crossing at the hit */
  int k1 = 0, f1 = 0, k2 = -1, f2 = 0;
  PT_BEGIN(t_iv);
  for (int it = 0; it < 2 * n; ++it) {
    uint32_t mask = 0, within = 0;
    float tnext = kInf;
    for (uint32_t todo = live; todo; todo &= todo - 1u) {
      const int k = __ffs((int)todo) - 1;
      const Interval iv = prim_interval(S, prims[k], px, py, pz, dx, dy, dz);
      const bool empty = !(iv.tin < iv.tout);
      const float a = empty ? -kInf : iv.tin, b = empty ? -kInf : iv.tout;
      if (it == 0) bits |= (a <= 0.f) & (b > 0.f) ? 1u << k : 0u;
      const bool at_in = a > tcur;
      const float nk = at_in ? a : (b > tcur ? b : kInf);
      within |= nk <= tmax ? 1u << k : 0u;
      const bool nearer = nk < tnext, same = nk == tnext;
      if (want_normal && open) {
        const int f = at_in ? iv.fin : iv.fout;
        k2 = nearer ? -1 : (same & (k2 < 0) ? k : k2);
        f2 = k2 == k ? f : f2;
        k1 = nearer ? k : k1;
        f1 = nearer ? f : f1;
      }
      mask = nearer ? 1u << k : (same ? mask | (1u << k) : mask);
      tnext = nearer ? nk : tnext;
    }
    if (it == 0) inside = truth(sh, bits);
    open = open & (within != 0u);
    bits ^= open ? mask : 0u;
    const bool hit = open & (truth(sh, bits) != inside);
    h.t = hit ? tnext : h.t;
    open = open & !hit;
    tcur = tnext;
    if (!wave_any(open)) break;
    /* those with a crossing left on some open lane's segment */
    for (uint32_t todo = live; todo; todo &= todo - 1u) {
      const uint32_t bit = todo & (0u - todo);
      if (!wave_any(open & ((within & bit) != 0u))) live &= ~bit;
    }
  }
  PT_END(PH_GEOM_IV, t_iv);
  PT_BEGIN(t_wk);
  if (want_normal && h.t < kInf) {
    const float qx = px + h.t * dx, qy = py + h.t * dy, qz = pz + h.t * dz;
    float nx, ny, nz;
    prim_normal(S, prims[k1], f1, qx, qy, qz, nx, ny, nz);
    if (k2 >= 0) {
      /* simultaneous crossings: mean of the two lowest-index normals
       * (NormalIntersectionShape.cu:229-236) */
      float mx, my, mz;
      prim_normal(S, prims[k2], f2, qx, qy, qz, mx, my, mz);
      nx = 0.5f * (nx + mx);
      ny = 0.5f * (ny + my);
      nz = 0.5f * (nz + mz);
    }
    h.nx = nx;
    h.ny = ny;
    h.nz = nz;
  }
  PT_END(PH_GEOM_WALK, t_wk);
  return h;
}

/* Runs body(r) once for each value r that `key` has among the lanes with
 * `on`: r is wave-uniform (the loop runs over a uniform mask), so the scene
 * records it selects are read with scalar loads; the body runs with those
 * lanes active. */
template <class F>
MD void by_value(bool on, int key, F body) {
  unsigned long long todo = __builtin_amdgcn_ballot_w64(on);
  while (todo) {
    const int r0 = __builtin_amdgcn_readlane(key, __ffsll((long long)todo) - 1);
    const unsigned long long turn = __builtin_amdgcn_ballot_w64(key == r0) & todo;
    if (__builtin_amdgcn_inverse_ballot_w64(turn)) body(r0);
    todo &= ~turn;
  }
}

/* The region among r (which contains the point) and its descendants that
 * holds it: the descent of RegionBase::containingSubRegion. */
MD int descend(const DevScene& S, int r, float px, float py, float pz) {
  bool open = true;
  for (int guard = 0; guard < 64 && wave_any(open); ++guard) {
    int next = -1;
    by_value(open, r, [&](int r0) {
      const MONSEL_CS DRegion& rg = S.regions[r0];
      for (int c = 0; c < rg.n_children; ++c) {
        const MONSEL_CS DShape& ch = S.children[rg.first_child + c];
        const bool in = shape_contains(S, ch, px, py, pz);
        next = (next < 0) & in ? ch.region : next;
      }
    });
    open = open && next >= 0;
    r = open ? next : r;
  }
  return r;
}

/* RegionBase::containingSubRegion (RegionBase.cu:50-60) from region r (which
 * may differ by lane). */
MD int containing_sub_region(const DevScene& S, int r, float px, float py, float pz) {
  bool in = false;
  by_value(true, r, [&](int r0) { in = shape_contains(S, S.regions[r0].sh, px, py, pz); });
  return in ? descend(S, r, px, py, pz) : -1;
}

MD bool is_containing_region(const DevScene& S, int r, int target) {
  int a = S.regions[target].parent;
  while (a >= 0) {
    if (a == r) return true;
    a = S.regions[a].parent;
  }
  return false;
}

/* T'[S] = T[S ^ B] for the entries of an n-input truth table (n <= 5,
 * wave-uniform; B < 2^n) */
MD uint32_t xor_permute(uint32_t T, uint32_t B, int n) {
  if (B & 1u) T = ((T & 0x55555555u) << 1) | ((T >> 1) & 0x55555555u);
  if (n > 1 && (B & 2u)) T = ((T & 0x33333333u) << 2) | ((T >> 2) & 0x33333333u);
  if (n > 2 && (B & 4u)) T = ((T & 0x0F0F0F0Fu) << 4) | ((T >> 4) & 0x0F0F0F0Fu);
  if (n > 3 && (B & 8u)) T = ((T & 0x00FF00FFu) << 8) | ((T >> 8) & 0x00FF00FFu);
  if (n > 4 && (B & 16u)) T = (T << 16) | (T >> 16);
  return T;
}

/* Lower bound on the distance from p to the surface of shape sh.  Moving
 * less than the distance D_k to primitive k's surface cannot change k's
 * inside bit, so within distance D_k only the bits of the primitives with
 * D_j <= D_k can have flipped; the bound is the least D_k for which some
 * flip of those bits changes the shape's truth value.  Surfaces inside the
 * shape, or shared by primitives whose crossing does not matter, therefore
 * do not limit it.  With at most kMaxCstPrims primitives the test is on
 * bit masks: M[S] = truth(B ^ S) != truth(B) over the 32 flip sets S, and
 * the flip sets within a set F of primitives are the AND, over the
 * primitives b outside F, of the sets with bit b clear.  Larger shapes: the
 * nearest primitive surface. */
MD float shape_safety(const DevScene& S, const MONSEL_CS DShape& sh, float px, float py, float pz, bool& inside) {
  const int n = sh.n_prims;
  if (n == 1) {
    bool in;
    const float d = fabsf(prim_gmax_in(S, S.prims[sh.first_prim], px, py, pz, in));
    inside = truth(sh, in ? 1u : 0u);
    return truth(sh, 0u) != truth(sh, 1u) ? d : kInf;
  }
  if (n > kMaxCstPrims) {
    float d = kInf;
    uint32_t bits = 0;
    for (int k = 0; k < n; ++k) {
      bool in;
      d = fminf(d, fabsf(prim_gmax_in(S, S.prims[sh.first_prim + k], px, py, pz, in)));
      if (in) bits |= 1u << k;
    }
    inside = truth(sh, bits);
    return d;
  }
  float d[kMaxCstPrims];
  uint32_t bits = 0;
#pragma unroll
  for (int k = 0; k < kMaxCstPrims; ++k) {
    d[k] = kInf;
    if (k < n) {
      bool in;
      d[k] = fabsf(prim_gmax_in(S, S.prims[sh.first_prim + k], px, py, pz, in));
      if (in) bits |= 1u << k;
    }
  }
  const uint32_t Tp = xor_permute(sh.truth[0], bits, n);
  inside = (Tp & 1u) != 0u;   /* bit 0 of the permuted table is truth(bits) */
  const uint32_t M = Tp ^ (0u - (Tp & 1u));
  constexpr uint32_t kClear[kMaxCstPrims] = {0x55555555u, 0x33333333u, 0x0F0F0F0Fu, 0x00FF00FFu, 0x0000FFFFu};
  /* flip sets of primitives beyond n never occur */
  uint32_t exist = 0xFFFFFFFFu;
#pragma unroll
  for (int b = 0; b < kMaxCstPrims; ++b)
    if (b >= n) exist &= kClear[b];
  float best = kInf;
  /* the loops run over the n primitives only (n is wave-uniform) */
#pragma unroll
  for (int k = 0; k < kMaxCstPrims; ++k) {
    if (k < n) {
      uint32_t within = exist;
#pragma unroll
      for (int b = 0; b < kMaxCstPrims; ++b)
        if (b < n && b != k && !(d[b] <= d[k])) within &= kClear[b];
      if (M & within) best = fminf(best, d[k]);
    }
  }
  return best;
}

/* Lower bound on the distance from p to the surfaces findEndOfStep tests
 * from region r: r's shape and its children's shapes.  A step from p shorter
 * than this cannot end at a boundary.  0 when p is outside r's own shape by
 * the containment test of the step's start (shape_contains): such an
 * electron is relocated before its next step, as the reference relocates it
 * (MonteCarloSS.cu:107-115), so a bound measured from outside the shape
 * never lets it skip that test. */
MD float region_safety(const DevScene& S, int r, float px, float py, float pz) {
  const MONSEL_CS DRegion& rg = S.regions[r];
  bool inside;
  float d = shape_safety(S, rg.sh, px, py, pz, inside);
  if (!inside) return 0.f;
  for (int c = 0; c < rg.n_children; ++c) {
    bool in_child;
    d = fminf(d, shape_safety(S, S.children[rg.first_child + c], px, py, pz, in_child));
  }
  return d;
}

/* Result of RegionBase::findEndOfStep. */
struct StepEnd {
  float t;        /* distance moved (<= s) */
  int next;       /* next region; == current if no boundary; -1 left the chamber */
  bool boundary;
  float ownNx, ownNy, ownNz;   /* current shape's crossing normal (this step) */
  int winner;                  /* child region whose shape won, -1 = own shape */
  float winNx, winNy, winNz;
};

/* Displacement that carries a point across a boundary at coordinate scale |p|. */
MD float nudge_nm(float px, float py, float pz) {
  float m = fmaxf(fabsf(px), fmaxf(fabsf(py), fabsf(pz)));
  return 1.0e-3f + 4.0e-6f * m;
}

/* RegionBase::findEndOfStep (RegionBase.cu:74-119) on the ray p + t d,
 * 0 < t <= s.  A crossing of the chamber's own boundary leaves the chamber. */
MD StepEnd find_end_of_step(const DevScene& S, int r, float px, float py, float pz, float dx, float dy, float dz,
                            float s, bool want_normal) {
  StepEnd se;
  const MONSEL_CS DRegion& rg = S.regions[r];
  float t = kInf;
  int base = r;
  se.winner = -1;
  /* c = -1: the region's own shape; c >= 0: its children, each limited to
   * the nearest crossing found so far */
  for (int c = -1; c < rg.n_children; ++c) {
    const MONSEL_CS DShape& sh = c < 0 ? rg.sh : S.children[rg.first_child + c];
    const int reg = c < 0 ? r : sh.region;
    ShapeHit h = shape_first(S, sh, px, py, pz, dx, dy, dz, c < 0 ? s : fminf(s, t), want_normal);
    if (c < 0) {
      se.ownNx = se.winNx = h.nx;
      se.ownNy = se.winNy = h.ny;
      se.ownNz = se.winNz = h.nz;
      t = h.t;
      base = (t <= s && rg.parent >= 0) ? rg.parent : r;
    } else if (h.t <= s && h.t < t) {
      t = h.t;
      base = reg;
      se.winner = reg;
      se.winNx = h.nx;
      se.winNy = h.ny;
      se.winNz = h.nz;
    }
  }
  if (t <= s) {
    se.t = t;
    se.boundary = true;
    if (rg.parent < 0 && se.winner < 0) {
      se.next = -1; /* through the chamber wall */
      return se;
    }
    float qx = px + t * dx, qy = py + t * dy, qz = pz + t * dz;
    float dd = nudge_nm(qx, qy, qz);
    float ox = qx + dd * dx, oy = qy + dd * dy, oz = qz + dd * dz;
    int res = -1;
    PT_BEGIN(t_lo);
    /* up from the crossed shape's side until a region contains the point */
    bool up = base >= 0;
    for (int guard = 0; guard < 64 && wave_any(up); ++guard) {
      by_value(up, base, [&](int r0) {
        const MONSEL_CS DRegion& rb = S.regions[r0];
        if (shape_contains(S, rb.sh, ox, oy, oz)) {
          res = r0;
          up = false;
        } else {
          base = rb.parent;
          up = base >= 0;
        }
      });
    }
    if (res >= 0) res = descend(S, res, ox, oy, oz);
    PT_END(PH_GEOM_LOC, t_lo);
    se.next = res;
    return se;
  }
  se.t = s;
  se.boundary = false;
  se.next = r;
  return se;
}

}  // namespace monsel_dev

#endif
