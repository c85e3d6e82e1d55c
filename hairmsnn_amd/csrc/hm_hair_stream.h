// The hair BSDF of hm_hair_bsdf.h arranged for the batched device streams
// (hmsnn_hair_bsdf_eval_dev / _sample_dev).
//
// The streams are bound by vector instructions: one 40-byte query per lane
// ran 1320 of them per sample (0.99 of the SIMDs' issue cycles) where the
// memory traffic alone would take 60% of the time. Against the renderer's
// routines, whose operations every schedule has to repeat bit for bit:
//  - exp, log, reciprocal and square root go to the hardware instructions with
//    the argument's rounding carried along (the library's range handling is
//    not needed for the magnitudes here),
//  - atan2 and asin are short polynomials (least-squares fits in the relative
//    error, 3e-9 and 2e-8), and only the difference of the two azimuths is
//    taken, from one arc tangent,
//  - the longitudinal lobe's log(1 / a) / 2 and log(I0) become factors outside
//    its exponential, the azimuthal wrap one rounding in place
//    of a loop,
//  - the four lobes are unrolled (no value selects; the branch on a lobe's
//    variance is uniform).
//  - the sampler carries 1 - cos theta and both tails of the logistic's cdf,
//    whose roundings the library form divides by the lobes' variances.
// Error against FP64, 3 million queries of equal roughnesses 0.12 / 0.3 / 0.6,
// root mean square, before -> after: evaluated f (relative) 2.3e-6 -> 1.7e-6 /
// 1.2e-6 -> 9.0e-7 / 4.1e-7 -> 3.9e-7; sampled direction 9.7e-7 -> 1.7e-7 /
// 1.2e-6 -> 1.7e-7 / 9.9e-7 -> 2.0e-7; sampled f 7.7e-6 -> 5.7e-6 / 4.6e-6 ->
// 1.6e-6 / 1.5e-6 -> 5.4e-7. (The 2-norm over a whole batch's outputs, which
// its largest values of f decide, is level: 1.2e-6 on both sides for four
// million samples at roughness 0.3.) Four million evaluations 82 -> 48 us,
// samples 113 -> 74 us (88 bytes each: 3.1 -> 4.8 TB/s); 100,000 samples 6.8 ->
// 4.8 us; a thousand queries are the launch (4.4 to 4.9 us on both sides).
#pragma once

#include "hm_hair_bsdf.h"

#if defined(__HIPCC__)

namespace hm {

// 2^t from the hardware, the rounding of x * log2(e) added back (finite t: at
// -inf the rounding would be a difference of infinities).
HM_D float fast_exp(float x) {
  const float t = x * 1.44269504f;
  const float r = fmaf(x, 1.92596299e-8f, fmaf(x, 1.44269504f, -t));
  const float e = __builtin_amdgcn_exp2f(t);
  return fmaf(e, r * 0.693147181f, e);
}
// exp of -x that may be infinite or overflow in t: 0 from 104 on, as in FP32
// (the maximum keeps a NaN).
HM_D float fast_exp_down(float x) { return fast_exp(__builtin_elementwise_maximum(-x, -104.f)); }
HM_D float fast_log(float x) {
  const float l = __builtin_amdgcn_logf(x);
  return fmaf(l, 0.693147181f, l * -1.90465433e-9f);
}
HM_D float fast_rcp(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.f), r, r);
}
// sqrt(max(x, 0)).
HM_D float fast_sqrt(float x) { return __builtin_amdgcn_sqrtf(fmaxf(x, 0.f)); }
HM_D float fast_rsq(float x) {
  const float r = __builtin_amdgcn_rsqf(x);
  return fmaf(r * 0.5f, fmaf(-x * r, r, 1.f), r);
}

// Finite arguments, not both zero.
HM_D float fast_atan2(float y, float x) {
  const float ax = fabsf(x), ay = fabsf(y);
  const float mx = fmaxf(ax, ay), mn = fminf(ax, ay);
  // beyond tan(pi / 8): atan(t) = pi / 4 + atan((t - 1) / (t + 1))
  const bool far = mn > 0.414213562f * mx;
  const float num = far ? mn - mx : mn, den = far ? mn + mx : mx;
  const float r = __builtin_amdgcn_rcpf(den);
  float t = num * r;
  t = fmaf(fmaf(-t, den, num), r, t);
  const float z = t * t;
  float p = fmaf(z, -6.456608151e-02f, 1.074535552e-01f);
  p = fmaf(z, p, -1.426413289e-01f);
  p = fmaf(z, p, 1.999954678e-01f);
  p = fmaf(z, p, -3.333333180e-01f);
  float a = fmaf(t * z, p, t);
  a = far ? a + 0.785398163f : a;
  a = ay > ax ? 1.570796327f - a : a;
  a = x < 0.f ? 3.141592654f - a : a;
  return copysignf(a, y);
}

// phi_i - phi_o from the products of the two directions: one arc tangent and
// no rounding of either azimuth. A direction along the fibre (its azimuth is
// the library's, from the signs of its zeros) and components that are not
// finite or whose products could leave the range take the two azimuths.
HM_D float azimuth_between(V3 wo, V3 wi) {
  const float ro = fmaf(wo.y, wo.y, wo.z * wo.z), ri = fmaf(wi.y, wi.y, wi.z * wi.z);
  if (!(fminf(ro, ri) > 1e-12f && ro + ri < 1e12f)) return atan2f(wi.z, wi.y) - atan2f(wo.z, wo.y);
  return fast_atan2(fmaf(wi.z, wo.y, -(wi.y * wo.z)), fmaf(wi.y, wo.y, wi.z * wo.z));
}

// |x| <= 1 (NaN beyond, as asinf).
HM_D float fast_asin(float x) {
  const float ax = fabsf(x);
  const bool far = ax > 0.5f;
  const float z = far ? 0.5f - 0.5f * ax : ax * ax;
  const float s = far ? __builtin_amdgcn_sqrtf(z) : ax;
  float p = fmaf(z, 3.819634508e-02f, 2.649934400e-02f);
  p = fmaf(z, p, 4.500990536e-02f);
  p = fmaf(z, p, 7.498813171e-02f);
  p = fmaf(z, p, 1.666667273e-01f);
  const float a = fmaf(s * z, p, s);
  return copysignf(far ? fmaf(-2.f, a, 1.570796327f) : a, x);
}

// hair_prepare.
HM_D HairWo stream_prepare(const HairConsts& hc, V3 wo, float h, V3 sigma_a) {
  HairWo w;
  w.so = wo.x;
  w.co = fast_sqrt((1.f - w.so) * (1.f + w.so));
  w.phi_o = 0.f;  // (azimuths are taken relative to wo's)
  w.h = h;
  w.gamma_o = fast_asin(h);
  const float cos_gamma_o = fast_sqrt((1.f - h) * (1.f + h));
  const float sin_theta_t = w.so * (1.f / kEta);
  const float sin_gamma_t = h * w.co * fast_rsq((hc.eta - w.so) * (hc.eta + w.so));
  w.gamma_t = fast_asin(clampf(sin_gamma_t, -1.f, 1.f));
  const float fac = 2.f * fast_sqrt((1.f - sin_gamma_t) * (1.f + sin_gamma_t)) *
                    fast_rsq((1.f - sin_theta_t) * (1.f + sin_theta_t));
  const V3 T = v3(fast_exp_down(sigma_a.x * fac), fast_exp_down(sigma_a.y * fac), fast_exp_down(sigma_a.z * fac));
  const float xd = 1.f - w.co * cos_gamma_o;
  const float xd2 = xd * xd;
  const float F = hc.f0 + (1.f - hc.f0) * (xd2 * xd2 * xd);
  const float omf2 = (1.f - F) * (1.f - F);
  w.ap[0] = v3(F);
  w.ap[1] = omf2 * T;
  w.ap[2] = (omf2 * F) * (T * T);
  const V3 ft = F * T;
  w.ap[3] = w.ap[2] * ft * v3(fast_rcp(1.f - ft.x), fast_rcp(1.f - ft.y), fast_rcp(1.f - ft.z));
  float sum = 0.f;
#pragma unroll
  for (int p = 0; p < 4; ++p) sum += (w.ap[p].x + w.ap[p].y + w.ap[p].z) * (1.f / 3.f);
  w.inv_ap_sum = fast_rcp(sum);
  return w;
}

// M_p (hair_mp).
HM_D float stream_mp(const HairConsts& hc, int lobe, float ci, float co_t, float si, float so_t) {
  const float inv_v = hc.inv_v[lobe];
  const float a = ci * co_t * inv_v, b = si * so_t * inv_v;
  const float i0 = bessel_i0_series(a);
  if (hc.v[lobe] > 0.1f) return fast_exp(-b) * i0 * hc.mp_sinh_c[lobe];
  // a > 12: I0(a) ~ exp(a + 1 / 16a) / sqrt(2 pi a), and a - b - 1 / v is
  // -(1 - cos(theta_i + theta_o')) / v
  const bool big = a > 12.f;
  const float S = si * co_t + ci * so_t, C = ci * co_t - si * so_t;
  const float one_minus_c = C > 0.f ? S * S * fast_rcp(1.f + C) : 1.f - C;
  const float rs = fast_rsq(a);
  const float far = fmaf(-one_minus_c, inv_v, fmaf(0.0625f * rs, rs, -kHalfLog2Pi));
  return fast_exp((big ? far : -b - inv_v) + hc.mp_log_c[lobe]) * (big ? rs : i0);
}

// N_p (hair_np) at the azimuth difference phi: m half turns, odd or even as p
// is, wrap into [-pi, pi], pi taken in two parts.
HM_D float stream_np(const HairConsts& hc, float phi, int p, float gamma_o, float gamma_t) {
  const float c = fmaf(-2.f * (float)p, gamma_t, 2.f * gamma_o);
  const float m = (float)p + 2.f * rintf((phi + c) * (0.5f / kPi) - 0.5f * (float)p);
  const float dphi = fmaf(-m, 3.14159274f, phi) + fmaf(m, 8.74227766e-8f, c);
  const float e = fast_exp_down(fabsf(dphi) * hc.inv_s);
  const float d = 1.f + e;
  return e * (hc.inv_s * hc.trim_norm) * fast_rcp(d * d);
}

// hair_eval_fp.
HM_D FPdf stream_eval(const HairConsts& hc, const HairWo& w, V3 wo, V3 wi) {
  const float si = wi.x;
  const float ci = fast_sqrt((1.f - si) * (1.f + si));
  const float phi = azimuth_between(wo, wi);
  V3 f = v3(0.f);
  float pd = 0.f;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    float so_t, co_t;
    hair_tilt(hc, w, p, &so_t, &co_t);
    const float mp = stream_mp(hc, p, ci, fabsf(co_t), si, so_t);
    const float np = p < 3 ? stream_np(hc, phi, p, w.gamma_o, w.gamma_t) : 1.f / (2.f * kPi);
    const float mn = mp * np;
    f += (hc.gain[p] * mn) * w.ap[p];
    pd += mn * hair_ap_pdf(w, p);
  }
  return FPdf{f, pd};
}

// The lobe that u0 picks (disney_hair.cuh:300-305).
HM_D int pick_lobe(const HairWo& w, float u0) {
  const float q0 = hair_ap_pdf(w, 0), q1 = hair_ap_pdf(w, 1), q2 = hair_ap_pdf(w, 2);
  if (u0 < q0) return 0;
  u0 -= q0;
  if (u0 < q1) return 1;
  u0 -= q1;
  return u0 < q2 ? 2 : 3;
}

// hair_sample_dir. The lobe is the one hair_sample_dir picks for the same
// uniforms: the two sets of attenuations differ by a few roundings, and within
// 1e-5 of an edge between lobes (6 draws in 100,000) hair_prepare's are the
// ones that count.
HM_D V3 stream_sample_dir(const HairConsts& hc, const HairWo& w, V3 wo, V3 sigma_a, float u0, float u1, float u2,
                          float u3, int* lobe_out) {
  const float c0 = hair_ap_pdf(w, 0), c1 = c0 + hair_ap_pdf(w, 1), c2 = c1 + hair_ap_pdf(w, 2);
  const float gap = fminf(fminf(fabsf(u0 - c0), fabsf(u0 - c1)), fabsf(u0 - c2));
  int p = pick_lobe(w, u0);
  if (!(gap >= 1e-5f)) p = pick_lobe(hair_prepare(hc, wo, w.h, sigma_a), u0);
  float so_t, co_t;
  hair_tilt(hc, w, p, &so_t, &co_t);
  const float v = sel4(p, hc.vs[0], hc.vs[1], hc.vs[2], hc.vs[3]);
  const float inv_v = sel4(p, hc.inv_vs[0], hc.inv_vs[1], hc.inv_vs[2], hc.inv_vs[3]);
  const float e2 = fmaxf(u1, 1e-5f);
  // 1 - cos theta, not cos theta: its rounding next to 1 counts 1 / v in M_p
  const float omc = -v * fast_log(e2 + (1.f - e2) * fast_exp(-2.f * inv_v));
  const float sin_t = fast_sqrt(omc * (2.f - omc));
  const float si = fmaf(omc, so_t, -so_t) + sin_t * cos_small(2.f * kPi * u2) * co_t;
  const float ci = fast_sqrt((1.f - si) * (1.f + si));
  // trimmed-logistic inversion on the first three lobes, uniform on the
  // last; the cdf's range is symmetric about 1/2, so 1 - y comes without
  // cancellation
  const float y = u3 * hc.cdf_span + hc.cdf_lo, y1 = (1.f - u3) * hc.cdf_span + hc.cdf_lo;
  float x = -hc.s * fast_log(y1 * fast_rcp(y));
  x = clampf(x, -kPi, kPi);
  const float dphi = p < 3 ? fmaf(2.f * (float)p, w.gamma_t, -2.f * w.gamma_o) + x : 2.f * kPi * u3;
  float s, c;
  sincos_small(dphi, &s, &c);
  // wo's azimuth turned by dphi + p pi, one along the fibre from the signs of
  // its zeros
  const float ro = fmaf(wo.y, wo.y, wo.z * wo.z);
  float cy = wo.y * fast_rsq(ro), cz = wo.z * fast_rsq(ro);
  if (!(ro > 1e-12f && ro < 1e12f)) {
    const float phi_o = atan2f(wo.z, wo.y);
    cy = cosf(phi_o);
    cz = sinf(phi_o);
  }
  const float turn = p == 1 ? -ci : ci;
  *lobe_out = p;
  const V3 d = v3(si, turn * fmaf(cy, c, -(cz * s)), turn * fmaf(cz, c, cy * s));
  return d * fast_rsq(dot(d, d));
}

}  // namespace hm

#endif  // __HIPCC__
