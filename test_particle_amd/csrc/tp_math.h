/*
 * tp_math.h -- project-written FP64 sine/cosine shared by the GPU kernels
 * and the CPU oracle.
 *
 * The reference tracer takes sin/cos from the system libm
 * (src/force_free.c:143-145, src/tracking.c:816-817, :853-854).  libm's
 * results are not reproducible on a GPU, and in the chaotic ABC field a
 * one-ulp difference grows over thousands of steps.  Both sides of the
 * parity test therefore evaluate this one routine, with the same IEEE
 * operations in the same order (fma where written, no other contraction),
 * which makes FP64 trajectories bitwise reproducible between host and
 * device.  Accuracy against libm is tested separately (within 2 ulp).
 *
 * Method:
 *   - Cody & Waite (1980) additive argument reduction by pi/2 with a
 *     three-part constant.  x - k*P1 is formed by one fma and is exact for
 *     |x| < 2^52 (the difference is a multiple of 2^-52 below 2 in
 *     magnitude); the P2/P3 terms are carried as a double-double (r, rlo)
 *     with Knuth's TwoSum and fma product errors.
 *   - Taylor series of sin (to r^17) and cos (to r^18) on |r| <= pi/4,
 *     evaluated by Horner's rule with fma; the series truncation error is
 *     below 2^-60 relative there.
 *   - cos uses 1 - r^2/2 split with its rounding error recovered, as in
 *     the classical kernel of Sun's fdlibm.
 * The constants are pi/2 split into doubles and 1/n!.
 */
#ifndef TP_MATH_H
#define TP_MATH_H

#include <math.h>
#include <stdint.h>
#include <string.h>

#if defined(__HIPCC__)
#define TP_HD __host__ __device__ __forceinline__
#else
#define TP_HD static inline
#endif

/* A polynomial coefficient.  On the GPU it is kept in scalar registers (the
 * empty asm hides its value): otherwise the compiler copies each one into
 * vector registers in front of a two-operand FMA that overwrites it. */
TP_HD double tp_const(double c)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm("" : "+s"(c));
#endif
    return c;
}

/* the same, not formed ahead of its use (of a loop around it) */
TP_HD double tp_const_here(double c)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(c));
#endif
    return c;
}

/* v with its sign flipped if the lowest bit of t is set */
TP_HD double tp_flip_by_low_bit(double v, double t)
{
#if defined(__HIP_DEVICE_COMPILE__)
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    u32x2 b = __builtin_bit_cast(u32x2, v);
    /* adding 2^31 to the high word flips its top bit (one v_lshl_add_u32) */
    b.y += __builtin_bit_cast(u32x2, t).x << 31;
    return __builtin_bit_cast(double, b);
#else
    uint64_t b, c;
    memcpy(&b, &v, sizeof(b));
    memcpy(&c, &t, sizeof(c));
    b ^= c << 63;
    memcpy(&v, &b, sizeof(v));
    return v;
#endif
}

TP_HD uint32_t tp_low_word(double t)
{
    uint64_t b;
    memcpy(&b, &t, sizeof(b));
    return (uint32_t)b;
}

/* v with the bits of mask flipped in its high word */
TP_HD double tp_flip_sign(double v, uint32_t mask)
{
#if defined(__HIP_DEVICE_COMPILE__)
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    u32x2 b = __builtin_bit_cast(u32x2, v);
    b.y ^= mask;
    return __builtin_bit_cast(double, b);
#else
    uint64_t b;
    memcpy(&b, &v, sizeof(b));
    b ^= (uint64_t)mask << 32;
    memcpy(&v, &b, sizeof(v));
    return v;
#endif
}

#define TP_2_OVER_PI 0x1.45f306dc9c883p-1
#define TP_PIO2_1    0x1.921fb54442d18p+0
#define TP_PIO2_2    0x1.1a62633145c07p-54
#define TP_PIO2_3   -0x1.f1976b7ed8fbcp-110

/* sin and cos of r + rlo, |r| <= pi/4 and a little */
TP_HD void tp_sincos_reduced(double r, double rlo, double *sp, double *cp)
{
    double z = r * r;
    /* sin(r) = r + r z Ps(z) */
    double ps = 0x1.952c77030ad4ap-49;                      /*  1/17! */
    ps = fma(ps, z, -0x1.ae7f3e733b81fp-41);                /* -1/15! */
    ps = fma(ps, z, 0x1.6124613a86d09p-33);                 /*  1/13! */
    ps = fma(ps, z, -0x1.ae64567f544e4p-26);                /* -1/11! */
    ps = fma(ps, z, 0x1.71de3a556c734p-19);                 /*  1/9!  */
    ps = fma(ps, z, -0x1.a01a01a01a01ap-13);                /* -1/7!  */
    ps = fma(ps, z, 0x1.1111111111111p-7);                  /*  1/5!  */
    ps = fma(ps, z, -0x1.5555555555555p-3);                 /* -1/3!  */
    *sp = r + fma(r * z, ps, rlo);
    /* cos(r) = 1 - z/2 + z^2 Pc(z) */
    double pc = 0x1.6827863b97d97p-53;                      /*  1/18! */
    pc = fma(pc, z, -0x1.ae7f3e733b81fp-45);                /* -1/16! */
    pc = fma(pc, z, 0x1.93974a8c07c9dp-37);                 /*  1/14! */
    pc = fma(pc, z, -0x1.1eed8eff8d898p-29);                /* -1/12! */
    pc = fma(pc, z, 0x1.27e4fb7789f5cp-22);                 /*  1/10! */
    pc = fma(pc, z, -0x1.a01a01a01a01ap-16);                /* -1/8!  */
    pc = fma(pc, z, 0x1.6c16c16c16c17p-10);                 /*  1/6!  */
    pc = fma(pc, z, -0x1.5555555555555p-5);                 /* -1/4!  */
    pc = -pc;                                               /* z^2 * (1/4! - ...) */
    double hz = 0.5 * z;
    double wc = 1.0 - hz;
    *cp = wc + (((1.0 - wc) - hz) + fma(z * z, pc, -r * rlo));
}

/* sin(x) and cos(x) together; NaN/Inf in give NaN out. */
TP_HD void tp_sincos(double x, double *sp, double *cp)
{
    /* k = rint(2x/pi); the quadrant k mod 4 is in the low bits of the sum that
     * rounds it (adding 1.5 2^52), or, where that sum has no room for k, comes
     * from k itself */
    double k;
    uint32_t q;
    if (fabs(x) < 0x1p50) {
        const double t = fma(x, TP_2_OVER_PI, 0x1.8p52);
        k = t - 0x1.8p52;
        q = tp_low_word(t);
    } else {
        k = rint(x * TP_2_OVER_PI);
        const double m = k - 4.0 * floor(k * 0.25);
        q = m == 1.0 ? 1u : (m == 2.0 ? 2u : (m == 3.0 ? 3u : 0u));
    }
    double r1 = fma(-k, TP_PIO2_1, x);          /* exact */
    double w = k * TP_PIO2_2;
    double werr = fma(k, TP_PIO2_2, -w);        /* k*P2 = w + werr exactly */
    /* TwoSum(r1, -w) */
    double r = r1 - w;
    double bb = r - r1;
    double rlo = (r1 - (r - bb)) + (-w - bb);
    rlo = rlo - werr;
    rlo = fma(-k, TP_PIO2_3, rlo);
    double s, c;
    tp_sincos_reduced(r, rlo, &s, &c);
    /* (s, c), (c, -s), (-s, -c), (-c, s) in quadrants 0 to 3: a swap and two
     * sign bits */
    const double so = tp_flip_sign(q & 1u ? c : s, (q & 2u) << 30);
    const double co = tp_flip_sign(q & 1u ? s : c, ((q + 1u) & 2u) << 30);
    *sp = so;
    *cp = co;
}

/* tp_sincos for angles that are small as a rule (a step's rotation): below
 * 0.75 the reduction gives k = 0, r = x and rlo = 0, and is left out with its
 * quadrants (same bits).  Wirz, 33,000 particles x 200 steps, tp_sincos / this:
 * MHD grid 748 / 723 us, PIC grid 712 / 684, its textbook gather on two slices
 * 845 / 823; 140,000 in the ABC field 1188 / 1144. */
TP_HD void tp_sincos_angle(double x, double *sp, double *cp)
{
    if (fabs(x) < 0.75) tp_sincos_reduced(x, 0.0, sp, cp);
    else tp_sincos(x, sp, cp);
}

TP_HD double tp_sin(double x)
{
    double s, c;
    tp_sincos(x, &s, &c);
    return s;
}

TP_HD double tp_cos(double x)
{
    double s, c;
    tp_sincos(x, &s, &c);
    return c;
}

/*
 * cos(x) alone, for sums over many modes: reduction by pi instead of pi/2,
 * then one even Taylor polynomial to r^22 (truncation < 4e-20 on
 * [-pi/2, pi/2]) and the sign (-1)^k.  Rounding x/pi by adding 1.5 2^52
 * leaves k = rint(x/pi) in the low bits of the sum, so the sign is its lowest
 * bit moved to the sign position: one integer operation, where comparing
 * k/2 with its floor takes five.  r = x - k pi with pi in two parts, the
 * first product exact by the same fma argument as above (|x| < 2^52); a
 * third part would move r by less than 2^-57 even there.  17 operations; the
 * comparison and the third part make it 22 and give the same bits (3e7
 * arguments in each of |x| < 1.5, 30, 1e3, 1e5, 1e9).  From 2^51 pi on the sum
 * has no room for k's lowest bit: a sum over modes whose phases can reach
 * TP_COS_PI_MAX takes tp_cos_pi.
 */
#define TP_COS_PI_MAX 7e15

typedef struct tp_cos_pi_consts {
    double inv_pi, round, pi_hi, pi_lo, c[10];
} tp_cos_pi_consts;

/* the constants, to be formed once ahead of a loop over modes */
TP_HD tp_cos_pi_consts tp_cos_pi_init(void)
{
    tp_cos_pi_consts q;
    q.inv_pi = tp_const(0x1.45f306dc9c883p-2);
    q.round = 0x1.8p52;
    q.pi_hi = tp_const(0x1.921fb54442d18p+1);
    q.pi_lo = tp_const(0x1.1a62633145c07p-53);
    q.c[0] = tp_const(0x1.0ce396db7f853p-70);               /*  1/22! */
    q.c[1] = tp_const(-0x1.e542ba4020225p-62);              /* -1/20! */
    q.c[2] = tp_const(0x1.6827863b97d97p-53);               /*  1/18! */
    q.c[3] = tp_const(-0x1.ae7f3e733b81fp-45);              /* -1/16! */
    q.c[4] = tp_const(0x1.93974a8c07c9dp-37);               /*  1/14! */
    q.c[5] = tp_const(-0x1.1eed8eff8d898p-29);              /* -1/12! */
    q.c[6] = tp_const(0x1.27e4fb7789f5cp-22);               /*  1/10! */
    q.c[7] = tp_const(-0x1.a01a01a01a01ap-16);              /* -1/8!  */
    q.c[8] = tp_const(0x1.6c16c16c16c17p-10);               /*  1/6!  */
    q.c[9] = tp_const(-0x1.5555555555555p-5);               /* -1/4!  */
    return q;
}

TP_HD double tp_cos_pi_with(double x, const tp_cos_pi_consts *q)
{
    const double t = fma(x, q->inv_pi, q->round);
    const double k = t - q->round;
    double r = fma(-k, q->pi_hi, x);                        /* exact */
    r = fma(-k, q->pi_lo, r);
    const double z = r * r;
    double p = fma(q->c[0], z, q->c[1]);
    p = fma(p, z, q->c[2]);
    p = fma(p, z, q->c[3]);
    p = fma(p, z, q->c[4]);
    p = fma(p, z, q->c[5]);
    p = fma(p, z, q->c[6]);
    p = fma(p, z, q->c[7]);
    p = fma(p, z, q->c[8]);
    p = fma(p, z, q->c[9]);
    p = fma(p, z, 0.5);
    return tp_flip_by_low_bit(fma(-z, p, 1.0), t);  /* 1 - z/2 + z^2/24 - ... */
}

/* the same for an argument of any size (NaN for NaN and infinities): from
 * TP_COS_PI_MAX on k is rounded by itself, pi has a third part and the parity
 * comes from k.  The constants are formed where they are used: beside a loop
 * that holds tp_cos_pi_with's there is no room for them. */
TP_HD double tp_cos_pi(double x)
{
    const int near = fabs(x) < TP_COS_PI_MAX;
    const double inv_pi = tp_const_here(0x1.45f306dc9c883p-2);
    const double t = fma(x, inv_pi, 0x1.8p52);
    const double k = near ? t - 0x1.8p52 : rint(x * inv_pi);
    double r = fma(-k, tp_const_here(0x1.921fb54442d18p+1), x);
    r = fma(-k, tp_const_here(0x1.1a62633145c07p-53), r);
    if (!near) r = fma(-k, tp_const_here(-0x1.f1976b7ed8fbcp-109), r);
    const double z = r * r;
    double p = tp_const_here(0x1.0ce396db7f853p-70);
    p = fma(p, z, tp_const_here(-0x1.e542ba4020225p-62));
    p = fma(p, z, tp_const_here(0x1.6827863b97d97p-53));
    p = fma(p, z, tp_const_here(-0x1.ae7f3e733b81fp-45));
    p = fma(p, z, tp_const_here(0x1.93974a8c07c9dp-37));
    p = fma(p, z, tp_const_here(-0x1.1eed8eff8d898p-29));
    p = fma(p, z, tp_const_here(0x1.27e4fb7789f5cp-22));
    p = fma(p, z, tp_const_here(-0x1.a01a01a01a01ap-16));
    p = fma(p, z, tp_const_here(0x1.6c16c16c16c17p-10));
    p = fma(p, z, tp_const_here(-0x1.5555555555555p-5));
    p = fma(p, z, 0.5);
    const double c = fma(-z, p, 1.0), half = k * 0.5;
    return near ? tp_flip_by_low_bit(c, t) : (half == floor(half) ? c : -c);
}

/*
 * Deterministic log2 / exp2 / pow for the adaptive stepper's controller
 * (step-size factors err^(1/(2k+1))).  Only reproducibility between host and
 * device matters there; accuracy is ~1e-15 relative.
 *   log2: frexp into [sqrt(1/2), sqrt(2)), ln m = 2 atanh(s) with
 *         s = (m-1)/(m+1), odd series to s^23;
 *   exp2: 2^y = 2^n e^(f ln 2) with n = rint(y), Taylor series to r^14.
 * Arguments: x > 0 finite (log2, pow); |y| < 1000 (exp2).
 */
TP_HD double tp_log2(double x)
{
    int e;
    double m = frexp(x, &e);
    if (m < 0x1.6a09e667f3bcdp-1) {   /* sqrt(1/2) */
        m = 2.0 * m;
        e = e - 1;
    }
    double s = (m - 1.0) / (m + 1.0);
    double s2 = s * s;
    double p = 0x1.642c8590b2164p-5;              /* 1/23 */
    p = fma(p, s2, 0x1.8618618618618p-5);         /* 1/21 */
    p = fma(p, s2, 0x1.af286bca1af28p-5);         /* 1/19 */
    p = fma(p, s2, 0x1.e1e1e1e1e1e1ep-5);         /* 1/17 */
    p = fma(p, s2, 0x1.1111111111111p-4);         /* 1/15 */
    p = fma(p, s2, 0x1.3b13b13b13b14p-4);         /* 1/13 */
    p = fma(p, s2, 0x1.745d1745d1746p-4);         /* 1/11 */
    p = fma(p, s2, 0x1.c71c71c71c71cp-4);         /* 1/9 */
    p = fma(p, s2, 0x1.2492492492492p-3);         /* 1/7 */
    p = fma(p, s2, 0x1.999999999999ap-3);         /* 1/5 */
    p = fma(p, s2, 0x1.5555555555555p-2);         /* 1/3 */
    double lnm = 2.0 * s + 2.0 * s * s2 * p;
    return (double)e + lnm * 0x1.71547652b82fep+0; /* 1/ln 2 */
}

TP_HD double tp_exp2(double y)
{
    double n = rint(y);
    double r = (y - n) * 0x1.62e42fefa39efp-1;    /* ln 2 */
    double p = 0x1.93974a8c07c9dp-37;              /* 1/14! */
    p = fma(p, r, 0x1.6124613a86d09p-33);          /* 1/13! */
    p = fma(p, r, 0x1.1eed8eff8d898p-29);          /* 1/12! */
    p = fma(p, r, 0x1.ae64567f544e4p-26);          /* 1/11! */
    p = fma(p, r, 0x1.27e4fb7789f5cp-22);          /* 1/10! */
    p = fma(p, r, 0x1.71de3a556c734p-19);          /* 1/9! */
    p = fma(p, r, 0x1.a01a01a01a01ap-16);          /* 1/8! */
    p = fma(p, r, 0x1.a01a01a01a01ap-13);          /* 1/7! */
    p = fma(p, r, 0x1.6c16c16c16c17p-10);          /* 1/6! */
    p = fma(p, r, 0x1.1111111111111p-7);           /* 1/5! */
    p = fma(p, r, 0x1.5555555555555p-5);           /* 1/4! */
    p = fma(p, r, 0x1.5555555555555p-3);           /* 1/3! */
    p = fma(p, r, 0.5);
    p = fma(p, r, 1.0);
    p = fma(p, r, 1.0);
    return ldexp(p, (int)n);
}

TP_HD double tp_pow(double x, double y)
{
    return tp_exp2(y * tp_log2(x));
}

/* x^e for an integer e >= 0 by repeated multiplication, left to right */
TP_HD double tp_powi(double x, int e)
{
    double r = 1.0;
    for (int i = 0; i < e; i++) r = r * x;
    return r;
}

#endif /* TP_MATH_H */
