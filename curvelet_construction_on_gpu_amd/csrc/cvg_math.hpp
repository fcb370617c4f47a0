// Correctly rounded (to within a ~2^-70 relative evaluation error) FP64 sin,
// cos and atan2 for the curve-bundle path, usable on the host and on gfx950.
//
// Why not the device libm: cpu_curvelet's decisions (direction filter, bundle
// branch, k_min/k_max comparisons) are built on glibc's sin/cos/atan2
// (cpu_curvelet.hpp:690,705,728-733; curvelet_utils.hpp:61,68).  glibc 2.35 is
// not correctly rounded for about 0.1-0.2% of arguments, and no other libm
// reproduces its misroundings; a correctly rounded result agrees with glibc on
// every argument where glibc itself is correctly rounded, which is the closest
// an independent implementation can get.
//
// Methods (all published, none taken from a vendor libm):
//   * error-free transformations: TwoSum (Knuth), FastTwoSum (Dekker) and
//     TwoProduct through a fused multiply-add;
//   * Cody-Waite argument reduction with pi/2 split into three doubles, the
//     products k*C1, k*C2 formed exactly as double-doubles;
//   * table-driven evaluation (Tang; Gal's accurate tables): sin/cos of i/128
//     and atan of i/64 stored as double-doubles, generated by
//     gen_trig_tables.py from 80-digit decimal arithmetic, with Taylor
//     polynomials for the small remainder;
//   * atan2 by octant reduction to atan(t), t in [0, 1], and the addition
//     formula atan(t) = atan(c) + atan((t - c)/(1 + t c)).
//   * Payne-Hanek reduction for |x| >= 2^20: the bits of 2/pi that matter
//     for x's exponent (a 256-bit window of a 1408-bit table) times x's
//     53-bit significand in exact integer arithmetic, the quadrant from the
//     product's integer part mod 4 and the remainder from its fraction.
// Special values follow C99 Annex F.
//
// Every function is a plain sequence of IEEE-754 double operations and fma,
// so the host and device builds give bitwise identical results when compiled
// without contraction (-ffp-contract=off).  The tables are passed in by
// pointer: device code hands in __constant__ or LDS copies, host code the
// static arrays below.
#ifndef CVG_MATH_HPP
#define CVG_MATH_HPP

#include <hip/hip_runtime.h>

#include <cmath>

#include "cvg_trig_tables.hpp"

#define CVG_HD __host__ __device__ inline

namespace cvg {

struct dd {
    double hi;
    double lo;
};

CVG_HD dd two_sum(double a, double b)
{
    const double s = a + b;
    const double bb = s - a;
    const double e = (a - (s - bb)) + (b - bb);
    return {s, e};
}

// Requires |a| >= |b| (or a == 0).
CVG_HD dd fast_two_sum(double a, double b)
{
    const double s = a + b;
    return {s, b - (s - a)};
}

CVG_HD dd two_prod(double a, double b)
{
    const double p = a * b;
    return {p, fma(a, b, -p)};
}

// 64 x 64 -> 128-bit unsigned product from 32-bit halves.
CVG_HD void mul_u64(unsigned long long a, unsigned long long b, unsigned long long *hi, unsigned long long *lo)
{
    const unsigned long long a0 = a & 0xffffffffULL, a1 = a >> 32, b0 = b & 0xffffffffULL, b1 = b >> 32;
    const unsigned long long p00 = a0 * b0, p01 = a0 * b1, p10 = a1 * b0, p11 = a1 * b1;
    const unsigned long long mid = (p00 >> 32) + (p01 & 0xffffffffULL) + (p10 & 0xffffffffULL);
    *lo = (mid << 32) | (p00 & 0xffffffffULL);
    *hi = p11 + (p01 >> 32) + (p10 >> 32) + (mid >> 32);
}

// Word j of 2/pi's binary expansion (2/pi = sum_j W[j] 2^(-64 (j + 1))),
// kept after the sin/cos rows of the table as two exact 32-bit halves.
CVG_HD unsigned long long two_over_pi_word(const double *tab, int j)
{
    const double *w = tab + 4 * CVG_SIN_ROWS + 2 * j;
    return (static_cast<unsigned long long>(w[0]) << 32) | static_cast<unsigned long long>(w[1]);
}

// 64 bits of 2/pi's expansion starting at fractional bit p (bit 1 is the
// first after the binary point; bits at p <= 0 are the integer part, 0).
CVG_HD unsigned long long two_over_pi_bits(const double *tab, int p)
{
    if (p + 63 <= 0) return 0ULL;
    if (p <= 0) return two_over_pi_word(tab, 0) >> (1 - p);
    const int j = (p - 1) >> 6, o = (p - 1) & 63;
    const unsigned long long a = two_over_pi_word(tab, j);
    return o == 0 ? a : (a << o) | (two_over_pi_word(tab, j + 1) >> (64 - o));
}

// Payne-Hanek: x = k (pi/2) + r for any finite |x| >= 2^20, r = rh + rl with
// |r| <= pi/4 to about 2^-104 relative.  |x| = m 2^e (m the 53-bit
// significand); the integer part of m 2^e (2/pi) mod 4 is the quadrant and
// only the bits of 2/pi from position e - 1 on reach it or the fraction: with
// F = frac(2^(e-2) (2/pi)) taken to 256 bits, frac(m F) = frac(|x| (2/pi) / 4)
// to within 2^-203.  The top 2 bits of that 256-bit fraction are k, the rest
// (254 bits) the fraction of a quadrant, recentred to [-1/2, 1/2), normalized
// and converted to a double-double, times pi/2.
CVG_HD int reduce_pio2_large(double x, const double *tab, double *rh, double *rl)
{
    const unsigned long long bits = static_cast<unsigned long long>(__builtin_bit_cast(long long, x));
    const int e = static_cast<int>((bits >> 52) & 0x7ff) - 1075;
    const unsigned long long m = (bits & 0xfffffffffffffULL) | (1ULL << 52);
    const int q = e - 2;
    unsigned long long w[4];
    for (int i = 0; i < 4; ++i) w[i] = two_over_pi_bits(tab, q + 1 + 64 * i);
    // (m * window) mod 2^256, most significant word first
    unsigned long long h[4], l[4];
    for (int i = 0; i < 4; ++i) mul_u64(m, w[i], &h[i], &l[i]);
    unsigned long long r[4];
    r[3] = l[3];
    r[2] = l[2] + h[3];
    unsigned long long c = r[2] < h[3] ? 1ULL : 0ULL;
    r[1] = l[1] + h[2];
    unsigned long long c1 = r[1] < h[2] ? 1ULL : 0ULL;
    r[1] += c;
    c1 += (r[1] < c) ? 1ULL : 0ULL;
    r[0] = l[0] + h[1] + c1;
    int k = static_cast<int>(r[0] >> 62);
    // the quadrant's fraction, 254 bits moved to the top
    unsigned long long f[4];
    f[0] = (r[0] << 2) | (r[1] >> 62);
    f[1] = (r[1] << 2) | (r[2] >> 62);
    f[2] = (r[2] << 2) | (r[3] >> 62);
    f[3] = r[3] << 2;
    const bool neg = (f[0] >> 63) != 0;  // fraction >= 1/2: the next quadrant, negative remainder
    if (neg) {
        k += 1;
        unsigned long long carry = 1ULL;
        for (int i = 3; i >= 0; --i) {
            f[i] = ~f[i] + carry;
            carry = (carry && f[i] == 0ULL) ? 1ULL : 0ULL;
        }
    }
    // normalize: |r| >= 2^-62 for every double, so 3 words hold 128 bits
    // beyond the leading one
    int lz = 0;
    while (f[0] == 0ULL && lz < 192) {
        f[0] = f[1];
        f[1] = f[2];
        f[2] = f[3];
        f[3] = 0ULL;
        lz += 64;
    }
    if (f[0] == 0ULL) {
        *rh = 0.0;
        *rl = 0.0;
    } else {
        const int z = __builtin_clzll(f[0]);
        if (z) {
            f[0] = (f[0] << z) | (f[1] >> (64 - z));
            f[1] = (f[1] << z) | (f[2] >> (64 - z));
        }
        lz += z;
        // g = 0.f0 f1 ... * 2^-lz: its first 106 bits as two exact doubles
        const double gh = static_cast<double>(f[0] >> 11) * 0x1p-53;
        const double gm = static_cast<double>(((f[0] & 0x7ffULL) << 42) | (f[1] >> 22)) * 0x1p-106;
        const dd g = fast_two_sum(gh, gm);
        // times pi/2, then the scale
        dd p = two_prod(g.hi, CVG_PIO2_HI);
        p.lo += g.hi * CVG_PIO2_LO + g.lo * CVG_PIO2_HI;
        p = fast_two_sum(p.hi, p.lo);
        const double sc = ldexp(1.0, -lz);
        *rh = (neg ? -p.hi : p.hi) * sc;
        *rl = (neg ? -p.lo : p.lo) * sc;
    }
    if (x < 0) {
        *rh = -*rh;
        *rl = -*rl;
        k = -k;
    }
    return k & 3;
}

// x = k (pi/2) + r with r = (*rh + *rl), |r| <= pi/4 (1 + 2^-50); k is
// exact below 2^20 and k mod 4 beyond (Payne-Hanek).  LARGE = false: the
// caller guarantees |x| < 2^20, and the Payne-Hanek code (and its registers)
// is left out.
template <bool LARGE = true>
CVG_HD int reduce_pio2(double x, const double *tab, double *rh, double *rl)
{
    if (LARGE && !(fabs(x) < 0x1p20)) return reduce_pio2_large(x, tab, rh, rl);
    const double k = rint(x * CVG_TWO_OVER_PI);
    const dd p1 = two_prod(k, CVG_PIO2_1);
    const double t = x - p1.hi;  // exact (Sterbenz), or x itself when k == 0
    const dd p2 = two_prod(k, CVG_PIO2_2);
    const double p3 = k * CVG_PIO2_3;
    const dd s1 = two_sum(t, -p1.lo);
    const dd s2 = two_sum(s1.hi, -p2.hi);
    const double lo = ((s1.lo + s2.lo) - p2.lo) - p3;
    const dd r = two_sum(s2.hi, lo);
    *rh = r.hi;
    *rl = r.lo;
    return static_cast<int>(k);
}

// sin and cos of r = rh + rl, |r| <= pi/4 (1 + 2^-50), each as an unevaluated
// sum hi + lo (|lo| << |hi|); hi + lo rounded is the correctly rounded result.
// The lo parts are accurate to about 2^-86 absolute (the roundings of the
// 2^-37-sized correction terms).  Null outputs are skipped.
CVG_HD void sincos_reduced_parts(double rh, double rl, const double *tab, dd *s_out, dd *c_out)
{
    const double fi = rint(rh * 128.0);
    const int i = static_cast<int>(fi);
    const double a = fi * 0x1p-7;
    const dd d = two_sum(rh - a, rl);  // rh - a is exact
    const int ai = i < 0 ? -i : i;
    const double sg = i < 0 ? -1.0 : 1.0;
    const double Sh = sg * tab[4 * ai + 0];
    const double Sl = sg * tab[4 * ai + 1];
    const double Ch = tab[4 * ai + 2];
    const double Cl = tab[4 * ai + 3];

    const dd z2 = two_prod(d.hi, d.hi);
    const double zh = z2.hi;
    const double zl = z2.lo + 2.0 * d.hi * d.lo;
    // cos(d) = 1 - z/2 + z^2 pc2(z);  sin(d) = d - d z/6 + d z^2 ps2(z)
    const double pc2 = 1.0 / 24.0 + zh * (-1.0 / 720.0 + zh * (1.0 / 40320.0));
    const double ps2 = 1.0 / 120.0 + zh * (-1.0 / 5040.0 + zh * (1.0 / 362880.0));

    if (s_out) {
        // sin(a + d) = S + C d - S z/2 + S z^2 pc2 - C d z/6 + C d z^2 ps2
        const dd p = two_prod(Ch, d.hi);
        const dd h1 = two_sum(Sh, p.hi);
        const dd q = two_prod(Sh, zh);
        const dd h2 = two_sum(h1.hi, -0.5 * q.hi);
        const dd w = two_prod(p.hi, zh);
        const dd u = two_prod(w.hi, CVG_MINUS_SIXTH_HI);
        const dd h3 = two_sum(h2.hi, u.hi);
        double t = (h1.lo + h2.lo) + h3.lo;
        t += ((p.lo + Sl) + Ch * d.lo) + Cl * d.hi;
        t += (-0.5 * q.lo - 0.5 * (Sh * zl + Sl * zh)) + Sh * zh * zh * pc2;
        t += (u.lo + w.hi * CVG_MINUS_SIXTH_LO) + w.lo * CVG_MINUS_SIXTH_HI;
        t += (((p.lo + Ch * d.lo) + Cl * d.hi) * zh + p.hi * zl) * CVG_MINUS_SIXTH_HI;
        t += p.hi * zh * zh * ps2;
        *s_out = {h3.hi, t};
    }
    if (c_out) {
        // cos(a + d) = C - S d - C z/2 + C z^2 pc2 + S d z/6 - S d z^2 ps2
        const dd p = two_prod(Sh, d.hi);
        const dd h1 = two_sum(Ch, -p.hi);
        const dd q = two_prod(Ch, zh);
        const dd h2 = two_sum(h1.hi, -0.5 * q.hi);
        const dd w = two_prod(p.hi, zh);
        const dd u = two_prod(w.hi, CVG_MINUS_SIXTH_HI);
        const dd h3 = two_sum(h2.hi, -u.hi);
        double t = (h1.lo + h2.lo) + h3.lo;
        t += ((Cl - p.lo) - Sh * d.lo) - Sl * d.hi;
        t += (-0.5 * q.lo - 0.5 * (Ch * zl + Cl * zh)) + Ch * zh * zh * pc2;
        t -= (u.lo + w.hi * CVG_MINUS_SIXTH_LO) + w.lo * CVG_MINUS_SIXTH_HI;
        t -= (((p.lo + Sh * d.lo) + Sl * d.hi) * zh + p.hi * zl) * CVG_MINUS_SIXTH_HI;
        t -= p.hi * zh * zh * ps2;
        *c_out = {h3.hi, t};
    }
}

CVG_HD void sincos_reduced(double rh, double rl, const double *tab, double *s_out, double *c_out)
{
    dd s, c;
    sincos_reduced_parts(rh, rl, tab, s_out ? &s : nullptr, c_out ? &c : nullptr);
    if (s_out) *s_out = s.hi + s.lo;
    if (c_out) *c_out = c.hi + c.lo;
}

// sin(r) (want_cos false) or cos(r) of r = rh + rl, |r| <= pi/4 (1 + 2^-50),
// with one branch-free evaluation: the sine expression of sincos_reduced
// applied to the table pair (S, C) = sin/cos(a) gives sin(a + d); applied to
// (C, -S) = sin/cos(a + pi/2) it gives cos(a + d), and every operation then
// is the negation-exact image of the cosine expression's, so the result has
// the same bits as sincos_reduced's cosine.  Lanes wanting sine and cosine no
// longer run both code paths.
CVG_HD double sin_or_cos_reduced(double rh, double rl, const double *tab, bool want_cos)
{
    const double fi = rint(rh * 128.0);
    const int i = static_cast<int>(fi);
    const double a = fi * 0x1p-7;
    const dd d = two_sum(rh - a, rl);  // rh - a is exact
    const int ai = i < 0 ? -i : i;
    const double sg = i < 0 ? -1.0 : 1.0;
    const double Sh0 = sg * tab[4 * ai + 0];
    const double Sl0 = sg * tab[4 * ai + 1];
    const double Ch0 = tab[4 * ai + 2];
    const double Cl0 = tab[4 * ai + 3];
    const double Sh = want_cos ? Ch0 : Sh0;
    const double Sl = want_cos ? Cl0 : Sl0;
    const double Ch = want_cos ? -Sh0 : Ch0;
    const double Cl = want_cos ? -Sl0 : Cl0;

    const dd z2 = two_prod(d.hi, d.hi);
    const double zh = z2.hi;
    const double zl = z2.lo + 2.0 * d.hi * d.lo;
    const double pc2 = 1.0 / 24.0 + zh * (-1.0 / 720.0 + zh * (1.0 / 40320.0));
    const double ps2 = 1.0 / 120.0 + zh * (-1.0 / 5040.0 + zh * (1.0 / 362880.0));

    const dd p = two_prod(Ch, d.hi);
    const dd h1 = two_sum(Sh, p.hi);
    const dd q = two_prod(Sh, zh);
    const dd h2 = two_sum(h1.hi, -0.5 * q.hi);
    const dd w = two_prod(p.hi, zh);
    const dd u = two_prod(w.hi, CVG_MINUS_SIXTH_HI);
    const dd h3 = two_sum(h2.hi, u.hi);
    double t = (h1.lo + h2.lo) + h3.lo;
    t += ((p.lo + Sl) + Ch * d.lo) + Cl * d.hi;
    t += (-0.5 * q.lo - 0.5 * (Sh * zl + Sl * zh)) + Sh * zh * zh * pc2;
    t += (u.lo + w.hi * CVG_MINUS_SIXTH_LO) + w.lo * CVG_MINUS_SIXTH_HI;
    t += (((p.lo + Ch * d.lo) + Cl * d.hi) * zh + p.hi * zl) * CVG_MINUS_SIXTH_HI;
    t += p.hi * zh * zh * ps2;
    return h3.hi + t;
}

template <bool LARGE = true>
CVG_HD double cr_sin(double x, const double *tab)
{
    const double ax = fabs(x);
    if (!(ax <= 0x1.fffffffffffffp+1023)) return x - x;  // NaN for NaN and infinities
    if (ax < 0x1p-26) return x;
    double rh, rl;
    const int k = reduce_pio2<LARGE>(x, tab, &rh, &rl);
    const double v = sin_or_cos_reduced(rh, rl, tab, (k & 1) != 0);
    return (k & 2) ? -v : v;
}

CVG_HD double cr_cos(double x, const double *tab)
{
    const double ax = fabs(x);
    if (!(ax <= 0x1.fffffffffffffp+1023)) return x - x;  // NaN for NaN and infinities
    if (ax < 0x1p-27) return 1.0;
    double rh, rl;
    const int k = reduce_pio2(x, tab, &rh, &rl);
    const double v = sin_or_cos_reduced(rh, rl, tab, (k & 1) == 0);
    return ((k + 1) & 2) ? -v : v;
}

// LARGE = false: the caller guarantees |x| < 2^20 (same results there).
template <bool LARGE = true>
CVG_HD void cr_sincos(double x, const double *tab, double *s, double *c)
{
    const double ax = fabs(x);
    if (!(ax <= 0x1.fffffffffffffp+1023)) {
        const double bad = x - x;  // NaN for NaN and infinities
        *s = bad;
        *c = bad;
        return;
    }
    if (ax < 0x1p-27) {
        *s = x;
        *c = 1.0;
        return;
    }
    if (ax < 0x1p-26) {
        *s = x;
        double rh, rl;
        reduce_pio2<LARGE>(x, tab, &rh, &rl);
        sincos_reduced(rh, rl, tab, nullptr, c);
        return;
    }
    double rh, rl;
    const int k = reduce_pio2<LARGE>(x, tab, &rh, &rl);
    double sr, cr;
    sincos_reduced(rh, rl, tab, &sr, &cr);
    switch (k & 3) {
    case 0: *s = sr; *c = cr; break;
    case 1: *s = cr; *c = -sr; break;
    case 2: *s = -sr; *c = -cr; break;
    default: *s = -cr; *c = sr; break;
    }
}

// sin and cos of x as double-doubles: s->hi and c->hi carry the bits of
// cr_sincos(x); s->lo and c->lo are the remainders (about 2^-86 absolute).
// LARGE = false: the caller guarantees |x| < 2^20.
template <bool LARGE = true>
CVG_HD void cr_sincos_dd(double x, const double *tab, dd *s, dd *c)
{
    const double ax = fabs(x);
    if (!(ax <= 0x1.fffffffffffffp+1023)) {
        const double bad = x - x;  // NaN for NaN and infinities
        *s = {bad, 0.0};
        *c = {bad, 0.0};
        return;
    }
    if (ax < 0x1p-27) {
        *s = {x, -(x * x * x) / 6.0};
        *c = {1.0, -0.5 * (x * x)};
        return;
    }
    double rh, rl;
    const int k = reduce_pio2<LARGE>(x, tab, &rh, &rl);
    dd sp, cp;
    sincos_reduced_parts(rh, rl, tab, &sp, &cp);
    const double sh = sp.hi + sp.lo, ch = cp.hi + cp.lo;
    dd sr = {sh, sp.lo - (sh - sp.hi)};
    const dd cr = {ch, cp.lo - (ch - cp.hi)};
    if (ax < 0x1p-26) sr = {x, -(x * x * x) / 6.0};  // cr_sincos's sine of such x is x
    switch (k & 3) {
    case 0: *s = sr; *c = cr; break;
    case 1: *s = cr; *c = {-sr.hi, -sr.lo}; break;
    case 2: *s = {-sr.hi, -sr.lo}; *c = {-cr.hi, -cr.lo}; break;
    default: *s = {-cr.hi, -cr.lo}; *c = sr; break;
    }
}

// sin(fl(a - b)) from sin and cos of a and b as double-doubles (cr_sincos_dd),
// by the subtraction formula (Ziv's strategy: a fast evaluation with an error
// bound, kept only when the bound settles the rounding).  With a - b = d + e
// exactly (d = fl(a - b), e the TwoSum remainder, required <= 2^-45):
//   sin(d) = sin(a - b) cos(e) - cos(a - b) sin(e)
//          = (sa cb - ca sb) - (ca cb + sa sb) e + O(e^2).
// The inputs' errors (<= 2^-86 each, values <= 1) give <= 2^-84 absolute; the
// double-double arithmetic and the dropped e^2 terms add < 2^-90.  The result
// is kept when every value within kErr = 2^-80 of the computed sum rounds to
// the same double, so it is then the correctly rounded sin(d).  Returns false
// (out unset) otherwise, and for d = 0, where the caller's cr_sin(d) gives the
// signed zero.
CVG_HD bool sin_of_difference(double a, double b, dd sa, dd ca, dd sb, dd cb, double *out)
{
    const dd r = two_sum(a, -b);
    const dd p1 = two_prod(sa.hi, cb.hi);
    const dd p2 = two_prod(ca.hi, sb.hi);
    const dd s = two_sum(p1.hi, -p2.hi);
    const double cross = (sa.hi * cb.lo + sa.lo * cb.hi) - (ca.hi * sb.lo + ca.lo * sb.hi);
    const double cosd = ca.hi * cb.hi + sa.hi * sb.hi;
    const double lo = ((s.lo + (p1.lo - p2.lo)) + cross) - cosd * r.lo;
    const dd v = two_sum(s.hi, lo);
    const double kErr = 0x1p-80;
    *out = v.hi;
    return r.hi != 0.0 && fabs(r.lo) <= 0x1p-45 && v.hi + (v.lo + kErr) == v.hi && v.hi + (v.lo - kErr) == v.hi;
}

// cr_sin(fl(a - b)): the subtraction formula where it settles the rounding,
// else the direct evaluation.  (No kernel uses the two: they are kept as
// diagnostics, cvg_math_eval's ops 8 and 9.)
CVG_HD double sin_difference(double a, double b, dd sa, dd ca, dd sb, dd cb, const double *tab)
{
    double v;
    return sin_of_difference(a, b, sa, ca, sb, cb, &v) ? v : cr_sin(a - b, tab);
}

// a - b for double-doubles whose difference is not much smaller than a.
CVG_HD dd dd_sub(double ah, double al, dd b)
{
    const dd s = two_sum(ah, -b.hi);
    return fast_two_sum(s.hi, (s.lo + al) - b.lo);
}

CVG_HD dd cr_atan2_dd(double y, double x, const double *atab);

CVG_HD double cr_atan2(double y, double x, const double *atab) { return cr_atan2_dd(y, x, atab).hi; }

// atan2(y, x) as a double-double: hi carries the bits of cr_atan2, lo the
// remainder (special values: lo = 0).
CVG_HD dd cr_atan2_dd(double y, double x, const double *atab)
{
    if (x != x || y != y) return {x + y, 0.0};
    const bool xneg = __builtin_signbit(x) != 0;
    const bool yneg = __builtin_signbit(y) != 0;
    const double ax = fabs(x);
    const double ay = fabs(y);
    if (ay == 0.0) return {xneg ? (yneg ? -CVG_PI_HI : CVG_PI_HI) : y, 0.0};
    if (ax == 0.0) return {yneg ? -CVG_PIO2_HI : CVG_PIO2_HI, 0.0};
    if (ax == INFINITY || ay == INFINITY) {
        double v;
        if (ax == INFINITY && ay == INFINITY)
            v = xneg ? CVG_3PIO4_HI : CVG_PIO4_HI;
        else if (ay == INFINITY)
            v = CVG_PIO2_HI;
        else
            v = xneg ? CVG_PI_HI : 0.0;
        return {yneg ? -v : v, 0.0};
    }
    const bool swap = ay > ax;
    double num = swap ? ax : ay;
    double den = swap ? ay : ax;
    int e;
    frexp(den, &e);
    den = ldexp(den, 1 - e);  // den in [1, 2)
    num = ldexp(num, 1 - e);
    const double th = num / den;
    const double tl = fma(-th, den, num) / den;

    // atan(t), t = th + tl in [0, 1]
    const double fi = rint(th * 64.0);
    const int i = static_cast<int>(fi);
    const double c = fi * 0x1p-6;
    dd u;
    if (i == 0) {
        u = {th, tl};
    } else {
        const dd N = two_sum(th - c, tl);  // th - c is exact
        const dd m = two_prod(th, c);
        const dd D0 = two_sum(1.0, m.hi);
        const dd D = fast_two_sum(D0.hi, (D0.lo + m.lo) + tl * c);
        const double uh = N.hi / D.hi;
        const dd pu = two_prod(uh, D.hi);
        const double rem = (((N.hi - pu.hi) - pu.lo) + N.lo) - uh * D.lo;
        u = {uh, rem / D.hi};
    }
    const double Ah = atab[2 * i];
    const double Al = atab[2 * i + 1];
    const dd v2 = two_prod(u.hi, u.hi);
    const double vh = v2.hi;
    const double vl = v2.lo + 2.0 * u.hi * u.lo;
    // atan(u) = u - u v/3 + u v^2 pa2(v)
    const double pa2 = 0.2 + vh * (-1.0 / 7.0 + vh * (1.0 / 9.0 + vh * (-1.0 / 11.0)));
    const dd g1 = two_sum(Ah, u.hi);
    const dd w = two_prod(u.hi, vh);
    const dd q = two_prod(w.hi, CVG_MINUS_THIRD_HI);
    const dd g2 = two_sum(g1.hi, q.hi);
    double t = ((g1.lo + g2.lo) + Al) + u.lo;
    t += (q.lo + w.hi * CVG_MINUS_THIRD_LO) + w.lo * CVG_MINUS_THIRD_HI;
    t += (u.lo * vh + u.hi * vl) * CVG_MINUS_THIRD_HI;
    t += u.hi * vh * vh * pa2;
    dd r = fast_two_sum(g2.hi, t);
    if (swap) r = dd_sub(CVG_PIO2_HI, CVG_PIO2_LO, r);
    if (xneg) r = dd_sub(CVG_PI_HI, CVG_PI_LO, r);
    return yneg ? dd{-r.hi, -r.lo} : r;
}

// To2Pi, curvelet_utils.hpp:25-46 (fmod is exact, so any exact fmod matches).
CVG_HD double wrap_two_pi(double angle)
{
    const double two_pi = 2.0 * 3.14159265358979323846;
    double a;
    if (angle >= two_pi)
        a = fmod(angle, two_pi);
    else if (angle < 0)
        a = two_pi + fmod(angle, two_pi);
    else
        a = angle;
    if (!(a >= 0 && a < two_pi)) a = 0;
    return a;
}

// ---------------------------------------------------------------------------
// binary32: the reference's float instantiation calls sinf, cosf, sincosf and
// atan2f (cpu_curvelet.hpp:690-733, curvelet_utils.hpp:61,68).  These return
// the correctly rounded float of the exact value: the double-double result
// (error far below the distance of any sin, cos or atan2 value of float
// arguments from a float rounding boundary) rounded once to float.
// ---------------------------------------------------------------------------

// hi + lo to the nearest float.  (float)hi is that float unless hi lies
// exactly halfway between two floats, where lo decides.
CVG_HD float round_dd_to_float(dd v)
{
    const float f = static_cast<float>(v.hi);
    if (v.lo == 0.0 || v.hi != v.hi || f == 0.0f) return f;
    const double fd = static_cast<double>(f);
    if (fd == v.hi || fabs(fd) == INFINITY) return f;
    // the float neighbour on hi's other side, and the midpoint between them
    unsigned bits;
    __builtin_memcpy(&bits, &f, sizeof(bits));
    const bool up = (v.hi > fd) == (f > 0.0f);  // away from zero in magnitude
    bits = up ? bits + 1u : bits - 1u;
    float g;
    __builtin_memcpy(&g, &bits, sizeof(g));
    const double mid = 0.5 * (fd + static_cast<double>(g));
    if (v.hi != mid) return f;
    // exactly halfway in double: the sign of lo says on which side the value lies
    return ((v.lo > 0.0) == (static_cast<double>(g) > fd)) ? g : f;
}

CVG_HD float cr_sinf(float x, const double *tab)
{
    dd s, c;
    cr_sincos_dd(static_cast<double>(x), tab, &s, &c);
    return round_dd_to_float(s);
}

CVG_HD float cr_cosf(float x, const double *tab)
{
    dd s, c;
    cr_sincos_dd(static_cast<double>(x), tab, &s, &c);
    return round_dd_to_float(c);
}

template <bool LARGE = true>
CVG_HD void cr_sincosf(float x, const double *tab, float *s, float *c)
{
    dd sd, cd;
    cr_sincos_dd<LARGE>(static_cast<double>(x), tab, &sd, &cd);
    *s = round_dd_to_float(sd);
    *c = round_dd_to_float(cd);
}

CVG_HD float cr_atan2f(float y, float x, const double *atab)
{
    return round_dd_to_float(cr_atan2_dd(static_cast<double>(y), static_cast<double>(x), atab));
}

// To2Pi<float>, curvelet_utils.hpp:25-46: 2 pi is T(2) * T(M_PI) in float,
// and fmodf is exact, so fmod of the (exact) double values matches it.
CVG_HD float wrap_two_pi_f(float angle)
{
    const float two_pi = 2.0f * static_cast<float>(3.14159265358979323846);
    float a;
    if (angle >= two_pi)
        a = static_cast<float>(fmod(static_cast<double>(angle), static_cast<double>(two_pi)));
    else if (angle < 0)
        a = two_pi + static_cast<float>(fmod(static_cast<double>(angle), static_cast<double>(two_pi)));
    else
        a = angle;
    if (!(a >= 0 && a < two_pi)) a = 0;
    return a;
}

// sqrtf: the double square root of a float, rounded to float, is the
// correctly rounded float square root (53 >= 2 x 24 + 2 bits).
CVG_HD float sqrt_f(float x) { return static_cast<float>(sqrt(static_cast<double>(x))); }

// Host copies of the tables (device code keeps its own __constant__ copies).
static const double kSinCosTableHost[CVG_SINCOS_TABLE_SIZE] = CVG_SINCOS_TABLE_INIT;
static const double kAtanTableHost[2 * CVG_ATAN_ROWS] = CVG_ATAN_TABLE_INIT;

}  // namespace cvg

#endif
