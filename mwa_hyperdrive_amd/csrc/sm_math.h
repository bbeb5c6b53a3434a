// FP64 sin/cos for the measurement-equation phases.
//
// The phases reach |x| ~ 1e4 rad, far inside the range where a Cody-Waite reduction
// with a two-part pi/2 and fused multiply-adds is exact to within one rounding:
//   k = rint(x * 2/pi),  r = fma(-k, P1, x) - k P2,  |r| <= pi/4 (1 + eps),
// P1 = pi/2 rounded to double, P2 = (pi/2 - P1) rounded to double (the third part,
// ~1.5e-33, changes r by less than 1e-28 for |k| < 1e5 and is dropped). Both constants
// and 2/pi were computed from a 78-digit pi (Machin's formula). On |r| <= pi/4 the Taylor
// series truncated after r^19 (sin) and r^20 (cos) leave remainders below 1e-19, so the
// result is limited by the Horner rounding (about 1 ulp). Arguments up to |x| = 1e9 keep
// the reduction error below 1e-16 absolute; the kernels' phases stay far below that.
#pragma once

#ifdef __HIPCC__
#define SM_HD __host__ __device__
#else
#define SM_HD
#endif

#include <cmath>

namespace sm {

SM_HD inline void fast_sincos(double x, double &s, double &c) {
    const double k = rint(x * 0.6366197723675814);
    double r = fma(-k, 1.5707963267948966, x);
    r = fma(-k, 6.123233995736766e-17, r);
    const double r2 = r * r;
    // sin r = r + r^3 (-1/3! + r^2 (1/5! - ...)), coefficients (-1)^n / (2n+1)!
    double ps = -8.22063524662433e-18;
    ps = fma(ps, r2, 2.8114572543455206e-15);
    ps = fma(ps, r2, -7.647163731819816e-13);
    ps = fma(ps, r2, 1.6059043836821613e-10);
    ps = fma(ps, r2, -2.505210838544172e-08);
    ps = fma(ps, r2, 2.7557319223985893e-06);
    ps = fma(ps, r2, -0.0001984126984126984);
    ps = fma(ps, r2, 0.008333333333333333);
    ps = fma(ps, r2, -0.16666666666666666);
    const double sn = fma(r * r2, ps, r);
    // cos r = 1 + r^2 (-1/2! + r^2 (1/4! - ...)), coefficients (-1)^n / (2n)!
    double pc = 4.110317623312165e-19;
    pc = fma(pc, r2, -1.5619206968586225e-16);
    pc = fma(pc, r2, 4.779477332387385e-14);
    pc = fma(pc, r2, -1.1470745597729725e-11);
    pc = fma(pc, r2, 2.08767569878681e-09);
    pc = fma(pc, r2, -2.755731922398589e-07);
    pc = fma(pc, r2, 2.48015873015873e-05);
    pc = fma(pc, r2, -0.001388888888888889);
    pc = fma(pc, r2, 0.041666666666666664);
    pc = fma(pc, r2, -0.5);
    const double cn = fma(r2, pc, 1.0);
    const int q = (int)(long long)k & 3;
    const double a = (q & 1) ? cn : sn;  // sin x = sin r, cos r, -sin r, -cos r for q = 0..3
    const double b = (q & 1) ? sn : cn;  // cos x = cos r, -sin r, -cos r, sin r
    s = (q & 2) ? -a : a;
    c = ((q + 1) & 2) ? -b : b;
}

// (sin, cos) of k pi / 32 for k = 0 .. 63, each rounded to nearest from a 300-bit evaluation.
#define SM_SINCOS32_TABLE \
    0.0, 1.0, 0.0980171403295606, 0.9951847266721969, \
    0.19509032201612828, 0.9807852804032304, 0.2902846772544624, 0.9569403357322088, \
    0.3826834323650898, 0.9238795325112867, 0.47139673682599764, 0.881921264348355, \
    0.5555702330196022, 0.8314696123025452, 0.6343932841636455, 0.773010453362737, \
    0.7071067811865476, 0.7071067811865476, 0.773010453362737, 0.6343932841636455, \
    0.8314696123025452, 0.5555702330196022, 0.881921264348355, 0.47139673682599764, \
    0.9238795325112867, 0.3826834323650898, 0.9569403357322088, 0.2902846772544624, \
    0.9807852804032304, 0.19509032201612828, 0.9951847266721969, 0.0980171403295606, \
    1.0, 0.0, 0.9951847266721969, -0.0980171403295606, \
    0.9807852804032304, -0.19509032201612828, 0.9569403357322088, -0.2902846772544624, \
    0.9238795325112867, -0.3826834323650898, 0.881921264348355, -0.47139673682599764, \
    0.8314696123025452, -0.5555702330196022, 0.773010453362737, -0.6343932841636455, \
    0.7071067811865476, -0.7071067811865476, 0.6343932841636455, -0.773010453362737, \
    0.5555702330196022, -0.8314696123025452, 0.47139673682599764, -0.881921264348355, \
    0.3826834323650898, -0.9238795325112867, 0.2902846772544624, -0.9569403357322088, \
    0.19509032201612828, -0.9807852804032304, 0.0980171403295606, -0.9951847266721969, \
    0.0, -1.0, -0.0980171403295606, -0.9951847266721969, \
    -0.19509032201612828, -0.9807852804032304, -0.2902846772544624, -0.9569403357322088, \
    -0.3826834323650898, -0.9238795325112867, -0.47139673682599764, -0.881921264348355, \
    -0.5555702330196022, -0.8314696123025452, -0.6343932841636455, -0.773010453362737, \
    -0.7071067811865476, -0.7071067811865476, -0.773010453362737, -0.6343932841636455, \
    -0.8314696123025452, -0.5555702330196022, -0.881921264348355, -0.47139673682599764, \
    -0.9238795325112867, -0.3826834323650898, -0.9569403357322088, -0.2902846772544624, \
    -0.9807852804032304, -0.19509032201612828, -0.9951847266721969, -0.0980171403295606, \
    -1.0, 0.0, -0.9951847266721969, 0.0980171403295606, \
    -0.9807852804032304, 0.19509032201612828, -0.9569403357322088, 0.2902846772544624, \
    -0.9238795325112867, 0.3826834323650898, -0.881921264348355, 0.47139673682599764, \
    -0.8314696123025452, 0.5555702330196022, -0.773010453362737, 0.6343932841636455, \
    -0.7071067811865476, 0.7071067811865476, -0.6343932841636455, 0.773010453362737, \
    -0.5555702330196022, 0.8314696123025452, -0.47139673682599764, 0.881921264348355, \
    -0.3826834323650898, 0.9238795325112867, -0.2902846772544624, 0.9569403357322088, \
    -0.19509032201612828, 0.9807852804032304, -0.0980171403295606, 0.9951847266721969

// FP64 sin/cos with a table-driven reduction (P. T. P. Tang, "Table-lookup algorithms for
// elementary functions and their error analysis", 10th IEEE Symposium on Computer Arithmetic,
// 1991): x = k pi/32 + r with |r| <= pi/64 (1 + eps), then
//   sin x = S_k cos r + C_k sin r,   cos x = C_k cos r - S_k sin r,
// where (S_k, C_k) = (sin, cos)(k pi/32) come from `tab` (SM_SINCOS32_TABLE, index k mod 64)
// and the Taylor series of sin r to r^9 and of cos r to r^8 leave remainders below 3e-20 at
// |r| = pi/64. The reduction is fast_sincos's with a two-part pi/32 (P1 = pi/32 rounded to
// double, P2 = the rest rounded to double, 32/pi rounded to double, all from a 300-bit pi).
// Nine polynomial terms instead of twenty and no quadrant selection, for one table read. In two
// steps: k and r of x, and sin and cos from them.
SM_HD inline double table_reduce(double x, double &k) {
    k = rint(x * 10.185916357881302);
    return fma(-k, 3.827021247335479e-18, fma(-k, 0.09817477042468103, x));
}

SM_HD inline void table_reduced_sincos(double k, double r, const double *tab, double &s, double &c) {
    const double r2 = r * r;
    // coefficients (-1)^n / (2n+1)! and (-1)^n / (2n)!
    double ps = 2.7557319223985893e-06;
    ps = fma(ps, r2, -0.0001984126984126984);
    ps = fma(ps, r2, 0.008333333333333333);
    ps = fma(ps, r2, -0.16666666666666666);
    const double sr = fma(r * r2, ps, r);
    double pc = 2.48015873015873e-05;
    pc = fma(pc, r2, -0.001388888888888889);
    pc = fma(pc, r2, 0.041666666666666664);
    pc = fma(pc, r2, -0.5);
    const double cr = fma(r2, pc, 1.0);
    const int i = (int)k & 63;  // k fits an int for |x| < 2e8, far beyond any phase here
    const double S = tab[2 * i], C = tab[2 * i + 1];
    s = fma(S, cr, C * sr);
    c = fma(C, cr, -(S * sr));
}

SM_HD inline void table_sincos(double x, const double *tab, double &s, double &c) {
    double k;
    const double r = table_reduce(x, k);
    table_reduced_sincos(k, r, tab, s, c);
}

// A factor in two doubles, hi + lo.
struct TwoDouble {
    double hi, lo;
};

// a / b in two doubles (exact to about 2^-105 of it).
SM_HD inline TwoDouble two_quotient(double a, double b) {
    const double hi = a / b;
    return {hi, fma(-hi, b, a) / b};
}

// sin and cos of x y with neither the product nor y rounded to one double: a phase of 1e4 rad
// rounded to one is off by up to 9e-13. Three instructions more than table_sincos(x * y.hi).
SM_HD inline void table_sincos_product(double x, TwoDouble y, const double *tab, double &s, double &c) {
    const double p = x * y.hi;
    const double lo = fma(x, y.lo, fma(x, y.hi, -p));
    double k;
    const double r = table_reduce(p, k);
    table_reduced_sincos(k, r + lo, tab, s, c);
}

// 2^(j / 64) for j = 0 .. 63, each rounded to nearest from a 60-digit evaluation.
#define SM_EXP64_TABLE \
    1.0, 1.0108892860517005, 1.0218971486541166, 1.0330248790212284, \
    1.0442737824274138, 1.0556451783605572, 1.0671404006768237, 1.0787607977571199, \
    1.0905077326652577, 1.102382583307841, 1.1143867425958924, 1.1265216186082418, \
    1.1387886347566916, 1.1511892299529827, 1.1637248587775775, 1.1763969916502812, \
    1.189207115002721, 1.202156731452703, 1.215247359980469, 1.22848053610687, \
    1.241857812073484, 1.255380757024691, 1.2690509571917332, 1.2828700160787783, \
    1.2968395546510096, 1.3109612115247644, 1.3252366431597413, 1.339667524053303, \
    1.3542555469368927, 1.3690024229745905, 1.383909881963832, 1.3989796725383112, \
    1.4142135623730951, 1.42961333839197, 1.4451808069770467, 1.460917794180647, \
    1.4768261459394993, 1.4929077282912648, 1.5091644275934228, 1.5255981507445384, \
    1.5422108254079407, 1.559004400237837, 1.5759808451078865, 1.593142151342267, \
    1.6104903319492543, 1.6280274218573478, 1.645755478153965, 1.6636765803267364, \
    1.681792830507429, 1.7001063537185235, 1.718619298122478, 1.7373338352737062, \
    1.7562521603732995, 1.7753764925265212, 1.7947090750031072, 1.8142521755003989, \
    1.8340080864093424, 1.8539791250833855, 1.8741676341103, 1.8945759815869656, \
    1.9152065613971474, 1.9360617934922943, 1.9571441241754002, 1.978456026387951

// FP64 e^x with a table-driven reduction (P. T. P. Tang, "Table-driven implementation of the
// exponential function in IEEE floating-point arithmetic", ACM TOMS 15, 1989):
// x = k ln2/64 + r with |r| <= ln2/128 (1 + eps), e^x = 2^(k >> 6) T[k mod 64] e^r with the
// Taylor series of e^r to r^5 (remainder below 4e-17). ln2/64 is split in two doubles, both and
// 64/ln2 rounded from 60 digits. Underflows to 0; x below -800 or above 700 is outside its range
// (a NaN gives NaN). About 17 instructions.
SM_HD inline double table_exp(double x, const double *tab) {
    const double k = rint(x * 92.33248261689366);
    double r = fma(-k, 0.010830424696249145, x);
    r = fma(-k, 3.623510646634843e-19, r);
    double p = 0.008333333333333333;
    p = fma(p, r, 0.041666666666666664);
    p = fma(p, r, 0.16666666666666666);
    p = fma(p, r, 0.5);
    p = fma(p * r, r, r);
    const int i = (int)k;
    const double t = tab[i & 63];
    return ldexp(fma(t, p, t), i >> 6);
}

// e^x for |x| <= 2e-3: the Taylor series to x^5 (remainder below 1e-19).
SM_HD inline double small_exp(double x) {
    double p = 0.008333333333333333;
    p = fma(p, x, 0.041666666666666664);
    p = fma(p, x, 0.16666666666666666);
    p = fma(p, x, 0.5);
    p = fma(p, x, 1.0);
    return fma(p, x, 1.0);
}

#ifdef __HIPCC__
// The device copy of SM_SINCOS32_TABLE for table_sincos, one per translation unit; 16-byte
// aligned, so a lane reads its (sin, cos) pair in one load.
[[maybe_unused]] static __device__ const double kSinCos32[128] __attribute__((aligned(16))) = {SM_SINCOS32_TABLE};
[[maybe_unused]] static __device__ const double kExp64[64] = {SM_EXP64_TABLE};
#endif

}  // namespace sm
