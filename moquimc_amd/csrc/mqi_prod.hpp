// The step of the production transport kernels (MQI_EXACT=0), written out for
// the instruction count: the batched pass is bound by VALU issue, and a
// launch with fewer histories than lanes by the length of one wave's
// instruction stream, so both run at the rate of the instructions per step.
//
// Every value is the one that the expressions of the verification build gave
// when this build compiled them too: the same operations are rounded in the
// same order, with the fused multiply-adds spelled out (contraction is off
// here, so the code around an inlined call cannot change them).  What is left out is work whose result is known: range scaling of
// divisions and square roots whose operands are nowhere near the ends of the
// float range, products with the zeros and ones of a rotation's matrices, a
// conversion to double around an operation that is exact in float, a table
// index formed once per table.  The helpers are compared with IEEE results and
// with this build's own operations on the device (mqi_math_probe 10 - 18).
//
// Measured against the expressions: 2000-spot CT plan (512x512x200, dose and
// statistics) 437 -> 354 ms, 25-spot slab phantom (dose and LETd, 2.5e6
// histories) 49.6 -> 39.8 ms, one 200 MeV spot of 1e5 histories in water 7.57
// -> 6.11 ms, one launch per spot 138 -> 103 ms for 40 spots.
#ifndef MQI_PROD_HPP
#define MQI_PROD_HPP

#include "mqi_device.hpp"

namespace mqi_dev
{

// Thresholds that the formulas state in double, applied to floats: x < c is
// x < at_least(c), x <= c is x <= at_most(c) (no float lies between), without
// the conversion of x.
constexpr float at_least(double c) {   // the smallest float >= c, c > 0
    const float f = (float) c;
    return (double) f >= c ? f : __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, f) + 1u);
}
constexpr float at_most(double c) {    // the largest float <= c, c > 0
    const float f = (float) c;
    return (double) f <= c ? f : __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, f) - 1u);
}

// a / b as this build's float division gives it (hardware reciprocal, one
// multiplication), without the exponent handling the compiler wraps around
// it (8 instructions): bit for bit the same for operands and results within
// 2^-60 .. 2^60
MQI_DI float q_div(float a, float b) {
    MQI_NO_CONTRACT
    return a * __builtin_amdgcn_rcpf(b);
}
// the same for the square root (arguments of 2^-96 .. 2^60, and 0); the
// empty asm keeps the compiler from making one reciprocal square root, which
// rounds differently, of a division by it
MQI_DI float q_sqrt(float a) {
    float r = __builtin_amdgcn_sqrtf(a);
    asm("" : "+v"(r));
    return r;
}
// natural logarithm of a normal, positive, finite float, bit for bit logf of
// this build: the hardware's log2 times ln 2 as the sum of two floats, the
// low part and the rounding error of the product added on (the last fused
// multiply-add is what contraction makes of that addition: the error counts
// twice, half an ulp at most)
MQI_DI float q_log(float a) {
    MQI_NO_CONTRACT
    const float y  = __builtin_amdgcn_logf(a);
    const float hi = 0x1.62e42ep-1f, lo = 0x1.efa39ep-25f;   // ln 2 = hi + lo
    float       e  = __builtin_fmaf(y, hi, -(y * hi));
    e              = __builtin_fmaf(y, lo, e);
    return __builtin_fmaf(y, hi, e);
}
// correctly rounded a / b (the geometry) for |b| in 2^-13 .. 2^13 and a = 0 or
// |a| in 2^-60 .. 2^60: the reciprocal after one Newton-Raphson step, the
// quotient corrected by its residual, which a fused multiply-add gives exactly
// (P. W. Markstein, IBM J. Res. Dev. 34 (1990) 111); no range scaling
MQI_DI float r_div(float a, float b) {
    MQI_NO_CONTRACT
    float r = __builtin_amdgcn_rcpf(b);
    r       = __builtin_fmaf(__builtin_fmaf(-b, r, 1.0f), r, r);
    float q = a * r;
    q       = __builtin_fmaf(__builtin_fmaf(-b, q, a), r, q);
    return __builtin_fmaf(__builtin_fmaf(-b, q, a), r, q);
}
// the same in double, from a hardware reciprocal of half the digits: the
// correctly rounded a / b is d_quot(a, b, d_recip(b)) for operands within
// 2^-200 .. 2^200 (and a = 0)
MQI_DI double d_recip(double b) {
    MQI_NO_CONTRACT
    double r = __builtin_amdgcn_rcp(b);
    r        = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
    return __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
}
MQI_DI double d_quot(double a, double b, double r) {
    MQI_NO_CONTRACT
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}

// correctly rounded square root in double of a in 2^-700 .. 2^700:
// Goldschmidt's iteration on sqrt(a) and 1 / (2 sqrt(a)) together, from the
// hardware reciprocal square root, then two corrections by the residual
// (Markstein, as above); no range scaling
MQI_DI double d_sqrt(double a) {
    MQI_NO_CONTRACT
    const double y = __builtin_amdgcn_rsq(a);
    double       g = a * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g              = __builtin_fma(g, r, g);
    h              = __builtin_fma(h, r, h);
    g              = __builtin_fma(__builtin_fma(-g, g, a), h, g);
    return __builtin_fma(__builtin_fma(-g, g, a), h, g);
}

MQI_DI void q_normalize(v3& a) {   // normalize_fast
    MQI_NO_CONTRACT
    const float r = __builtin_amdgcn_rcpf(q_sqrt(a.x * a.x + a.y * a.y + a.z * a.z));
    a.x           = a.x * r;
    a.y           = a.y * r;
    a.z           = a.z * r;
}

// rotate_direction in two parts.  q_align: the matrix g that takes the z axis
// to d (Moller-Hughes) with the zeros of that axis multiplied out.  q_turn:
// the local direction (theta, phi), the z axis rotated about y and z, taken
// through it.  IEEE: divisions and square roots correctly rounded (post_poi,
// whose matrix serves all its daughters); YX: the order |d|^2 is summed in
// (x, y, z or y, x, z).
struct q_mat {
    float g0, g1, g2, g3, g4, g5, g6, g7, g8;
};
template<bool IEEE>
MQI_DI float p_div(float a, float b) {
    return IEEE ? r_div(a, b) : q_div(a, b);
}
template<bool IEEE>
MQI_DI float p_sqrt(float a) {
    return IEEE ? geo_sqrt(a) : q_sqrt(a);
}
template<bool IEEE, bool YX>
MQI_DI q_mat q_align(v3 d) {
    MQI_NO_CONTRACT
    const float xy = YX ? __builtin_fmaf(d.x, d.x, d.y * d.y) : __builtin_fmaf(d.y, d.y, d.x * d.x);
    const float c  = p_div<IEEE>(d.z, p_sqrt<IEEE>(__builtin_fmaf(d.z, d.z, xy)));
    q_mat       m;
    if (fminf(fabsf(c - 1.0f), fabsf(c + 1.0f)) < 1e-3f) {
        // d close to the axis: two reflections, through the bisector of x
        // and -z, U = (K, 0, -K), and through V = (1, 0, 0) - d normalised
        const float K = 0x1.6a09e6p-1f;
        v3          v = mk(1.0f - d.x, -d.y, -d.z);
        const float n = p_sqrt<IEEE>(v.x * v.x + v.y * v.y + v.z * v.z);
        v             = mk(p_div<IEEE>(v.x, n), p_div<IEEE>(v.y, n), p_div<IEEE>(v.z, n));
        const float dot_v  = __builtin_fmaf(v.z, v.z, __builtin_fmaf(v.x, v.x, v.y * v.y));
        const float dot_uv = __builtin_fmaf(v.z, -K, K * v.x);
        const float b      = p_div<IEEE>(2.0f, dot_v);
        const float a      = p_div<IEEE>(4.0f * dot_uv, 0x1.fffffep-1f * dot_v);
        const float b0 = v.x * b, b1 = v.y * b, b2 = v.z * b;
        const float a0 = v.x * a, a1 = v.y * a, a2 = v.z * a;
        m.g0 = __builtin_fmaf(K, a0, -(v.x * b0));
        m.g1 = -(v.y * b0);
        m.g2 = __builtin_fmaf(-K, a0, __builtin_fmaf(-v.z, b0, 1.0f));
        m.g3 = __builtin_fmaf(K, a1, -(v.x * b1));
        m.g4 = __builtin_fmaf(-v.y, b1, 1.0f);
        m.g5 = __builtin_fmaf(-K, a1, -(v.z * b1));
        m.g6 = __builtin_fmaf(K, a2, __builtin_fmaf(-v.x, b2, 1.0f));
        m.g7 = -(v.y * b2);
        m.g8 = __builtin_fmaf(-K, a2, -(v.z * b2));
    } else {
        const double dd = 1.0 - (double) (c * c);
        const float  h  = (float) d_quot(1.0 - (double) c, dd, d_recip(dd));
        const float  hx = d.x * h, hy = d.y * h;
        m.g0 = __builtin_fmaf(d.y, hy, c);
        m.g1 = m.g3 = -(d.x * hy);
        m.g2 = d.x;
        m.g4 = __builtin_fmaf(d.x, hx, c);
        m.g5 = d.y;
        m.g6 = -d.x;
        m.g7 = -d.y;
        m.g8 = c;
    }
    return m;
}
MQI_DI v3 q_turn(const q_mat& m, float theta, float phi) {
    MQI_NO_CONTRACT
    float st, ct, sp, cp;
    sincosf(theta, &st, &ct);
    sincosf(phi, &sp, &cp);
    v3 l = mk(cp * st, sp * st, ct);
    q_normalize(l);
    v3 o = mk(l.x * m.g0 + l.y * m.g1 + l.z * m.g2, l.x * m.g3 + l.y * m.g4 + l.z * m.g5,
              l.x * m.g6 + l.y * m.g7 + l.z * m.g8);
    q_normalize(o);
    return o;
}

// distance along one axis to the exit of voxel i (axis_in with its two
// directions as one: the edge ahead is e[i + 1] or e[i])
MQI_DI float axis_exit(float& dcomp, float p, const float* e, float sh, int i) {
    MQI_NO_CONTRACT
    const float tol = 1e-3f;
    const float d   = dcomp;
    const bool  neg = d < 0;
    const float q   = r_div((e[neg ? i : i + 1] + sh) - p, d);
    const bool  on  = fabsf(q) < tol && (!neg || i > 0);
    float       t   = on ? 1 / tol : q;
    if (!(d * d > 1e-7f)) {
        dcomp = 0;
        t     = __builtin_huge_valf();
    }
    return t;
}
MQI_DI float exit_distance(const grid_view& g, v3 p, v3& d, int& cx, int& cy, int& cz) {   // intersect_in
    const float tx = axis_exit(d.x, p.x, g.xe, g.sx, cx);
    const float ty = axis_exit(d.y, p.y, g.ye, g.sy, cy);
    const float tz = axis_exit(d.z, p.z, g.ze, g.sz, cz);
    const float u  = fminf(fminf(tx, ty), tz);
    if (u > 0) return u;
    cx = cy = cz = -1;
    return -1.0f;
}

// relativistic_quantities (mqi_relativistic_quantities.hpp:24-43) in float as
// far as a step needs them: beta^2 = Ek (Ek + 2 Mp) / Et^2 and p^2 = Ek (Ek +
// 2 Mp), without the cancellations of 1 - 1 / gamma^2 and Et^2 - Mp^2 at low
// energy
struct q_rel {
    float beta_sq, pp, Et_sq;   // pp = Ek (Ek + 2 Mp), the momentum squared
    float Et;
};
MQI_DI q_rel q_relq(float Ek) {
    MQI_NO_CONTRACT
    q_rel r;
    r.Et      = Ek + units::Mp;
    r.Et_sq   = r.Et * r.Et;
    r.pp      = Ek * (Ek + 2.0f * units::Mp);
    r.beta_sq = q_div(r.pp, r.Et_sq);
    return r;
}
MQI_DI float q_te_max(const q_rel& r) {
    MQI_NO_CONTRACT
    const float Me = 0.510998928f, MeMp = 0.510998928f / 938.272046f;
    const float gamma = q_div(r.Et, units::Mp);
    const float num   = (gamma * gamma) * ((2.0f * Me) * r.beta_sq);
    return q_div(num, __builtin_fmaf(gamma + gamma, MeMp, 1.0f) + MeMp * MeMp);
}

template<bool DBG>
MQI_DI float q_spr(float rho, float Ek) {   // spr
    MQI_NO_CONTRACT
    const float d = rho * 1000.0f;
    if (DBG) {
        if (fabsf(d - 1.0f) < at_least(1e-3)) return 1.0f;
    }
    if (d <= at_most(0.26)) {
        if (d < at_least(0.0012)) return 0.0f;
        return 0.8815f + q_div((d - 0.0012f) * (0.9925f - 0.8815f), 0.26f - 0.0012f);
    }
    const float  r0 = (float) __builtin_fma((double) Ek, -3.386e-5, 1.0123);
    const double pe = (double) MQ_POWF(Ek, -0.3421f) + 1.0;
    const double pr = (double) MQ_POWF(d, -0.7f) - 1.0;
    const float  r  = (float) __builtin_fma(pe * 0.291, pr, (double) r0);
    if (d >= at_least(0.9)) return r;
    return 0.9925f + q_div((d - 0.26f) * (r - 0.9925f), 0.9f - 0.26f);
}

template<bool DBG>
MQI_DI float q_radiation_length(float rho) {   // radiation_length
    MQI_NO_CONTRACT
    const float d = rho * 1000.0f;
    if (DBG) {
        if (fabsf(d - 1.0f) < at_least(1e-3)) return units::X0_water;
    }
    float f;
    if (d <= at_most(0.26))
        f = (float) __builtin_fma((double) d, 0.0085, 0.9857);
    else if (d <= at_most(0.9))
        f = (float) __builtin_fma((double) d, -0.2180, 1.0446);
    else
        f = __builtin_fmaf(q_log(d - 0.44f), 0.44f, 1.19f);
    return q_div(units::water_density * units::X0_water, d * 0.001f * f);
}

}   // namespace mqi_dev

#endif
