// Device-side helpers shared by the gfx950 kernels: numeric conventions and random streams.
//
// Numeric conventions (they are what make results reproducible against a CPU statement
// of the same arithmetic):
//   * every translation unit is built with -ffp-contract=off: a*b+c is two roundings
//     unless fmaf() is written out;
//   * fp32 sin/cos of an fp32 angle are the correctly rounded values, computed in fp64 and
//     rounded once;
//   * fp32 exp/log where an index or a branch depends on the last bit (action sampling, the PPO
//     ratio and its clip test) are the correctly rounded values as well;
//   * fp32 divide and sqrt are IEEE (hipcc default for gfx9).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define MRL_DEV __device__ __forceinline__

namespace mrl {

// The remainder r + tail of ax, finite and above 2^20, against multiples of pi / 2, and the multiple (Payne and Hanek's method,
// in integers): ax = M 2^E; the bits of 1 / (2 pi) from bit E on, times M, are the fraction of a turn, to 104 bits and
// more.
MRL_DEV void reduce_large(float ax, double &r, double &tail, int &q) {
    const uint32_t bits = __float_as_uint(ax), M = (bits & 0x7FFFFFu) | 0x800000u;
    const uint32_t at = (bits >> 23) - 150u + 32u, word = at >> 5, shift = at & 31u;   // (the first 32 bits: zeros for E < 0)
    constexpr uint32_t T[9] = {0x00000000u, 0x28BE60DBu, 0x9391054Au, 0x7F09D5F4u, 0x7D4D3770u, 0x36D8A566u, 0x4F10E410u, 0x7F9458EAu, 0xF7AEF158u};
    uint32_t t[5];
#pragma unroll
    for (int j = 0; j < 5; ++j) {
        t[j] = T[j];
#pragma unroll
        for (int i = 1; i < 5; ++i) t[j] = word == (uint32_t)i ? T[i + j] : t[j];
    }
    uint32_t w[4], p[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = (uint32_t)(((((uint64_t)t[j] << 32) | t[j + 1]) << shift) >> 32);
    uint64_t carry = 0;
#pragma unroll
    for (int j = 3; j >= 0; --j) {
        carry = (uint64_t)M * w[j] + carry;
        p[j] = (uint32_t)carry;
        carry >>= 32;
    }
    const uint32_t quarter = (p[0] + 0x20000000u) >> 30;
    const double high = (double)(int)(p[0] - (quarter << 30)) * 0x1p-32, low = (double)p[1] * 0x1p-64 + (double)p[2] * 0x1p-96;
    const double turn = high + low, off = low - (turn - high);
    const double two_pi = 6.283185307179586, rem = turn * two_pi;
    const double more = fma(turn, two_pi, -rem) + fma(turn, 2.4492935982947064e-16, off * two_pi);   // (2 pi in two pieces)
    r = rem + more;
    tail = more - (r - rem);
    q = (int)quarter;
}

// Sine and cosine of an fp32 angle, rounded once from Float64.  An env step takes a dozen of them in a row on the one
// wavefront that everything waits for, and a wavefront alone issues an instruction every six cycles whether it depends on
// the last one or not, so what counts is the number of instructions: the argument less k pi/2 (pi/2 in two pieces; the fma's
// product is exact), both polynomials of the remainder r, |r| <= pi/4 (interpolated at the Chebyshev points, off by less than
// 2^-55), and the quadrant's choice among the two rounded values.  237 cycles a call where the library's pair takes 441.
// Beyond 2^20 the remainder is carried in two pieces: the cosine of +-2.8616508e15 is 1.3e-9 of an ulp off the middle between
// two floats.  Compared with the rounded Float64 functions of a C library on every finite fp32 value: no difference.
struct SinCosK {
    double two_over_pi = 0.6366197723675814, half_pi = 1.5707963267948966, half_pi_lo = 6.123233995736766e-17;
    double s1 = -0.16666666666666666, s2 = 0.008333333333330936, s3 = -0.00019841269836740532, s4 = 2.7557316093198404e-06,
           s5 = -2.5051129896450185e-08, s6 = 1.5917988979397435e-10;
    double c1 = 0.041666666666666664, c2 = -0.0013888888888887389, c3 = 2.48015872987544e-05, c4 = -2.755731726587808e-07,
           c5 = 2.087614504941318e-09, c6 = -1.138254464534925e-11;
    // The constants in registers for as long as the caller keeps the struct: without, every use moves their halves into
    // scalar registers again, 30 instructions a call.  (Vector registers: the kernels that ask for it are short of
    // scalar ones, which would come and go through lanes of a vector register.)
    static MRL_DEV SinCosK held() {
        SinCosK k;
        asm volatile("" : "+v"(k.two_over_pi), "+v"(k.half_pi), "+v"(k.half_pi_lo), "+v"(k.s1), "+v"(k.s2), "+v"(k.s3),
                     "+v"(k.s4), "+v"(k.s5), "+v"(k.s6));
        asm volatile("" : "+v"(k.c1), "+v"(k.c2), "+v"(k.c3), "+v"(k.c4), "+v"(k.c5), "+v"(k.c6));
        return k;
    }
};
// of the angle q pi / 2 + r (+ tail), with x's sign
template <bool TAIL = false>
MRL_DEV void sincos_reduced(float x, double r, int q, const SinCosK &k, float &s, float &c, double tail = 0.0) {
    const double u = r * r;
    double ps = fma(k.s6, u, k.s5), pc = fma(k.c6, u, k.c5);
    ps = fma(ps, u, k.s4); pc = fma(pc, u, k.c4);
    ps = fma(ps, u, k.s3); pc = fma(pc, u, k.c3);
    ps = fma(ps, u, k.s2); pc = fma(pc, u, k.c2);
    ps = fma(ps, u, k.s1); pc = fma(pc, u, k.c1);
    const float fs = (float)(TAIL ? r + fma(r * u, ps, tail) : fma(r * u, ps, r));
    const float fc = (float)(TAIL ? 1.0 + fma(fma(u, pc, -0.5), u, -r * tail) : fma(fma(u, pc, -0.5), u, 1.0));
    const uint32_t a = __float_as_uint((q & 1) ? fc : fs), b = __float_as_uint((q & 1) ? fs : fc);
    s = __uint_as_float(a ^ ((uint32_t)(q & 2) << 30) ^ (__float_as_uint(x) & 0x80000000u));
    c = __uint_as_float(b ^ ((uint32_t)((q + 1) & 2) << 30));
}
MRL_DEV void sincos32(float x, float &s, float &c, const SinCosK &k = SinCosK{}) {
    const float ax = fabsf(x);
    const bool far = __any(ax > 0x1p20f);   // (beyond, pi / 2 in two pieces is too short)
    const double xd = (double)ax;
    const double n = __builtin_rint(xd * k.two_over_pi);
    sincos_reduced(x, fma(-n, k.half_pi_lo, fma(-n, k.half_pi, xd)), (int)n, k, s, c);
    if (__builtin_expect(far, 0)) {
        // (No branch on a lane's own value: at the end of one the compiler has been seen to save registers that live across
        // it before it widens the lane mask again; build.py looks for that.)
        const bool large = ax > 0x1p20f && ax < __builtin_inff();
        double r, tail;
        float ls, lc;
        int q;
        reduce_large(ax, r, tail, q);
        sincos_reduced<true>(x, r, q, k, ls, lc, tail);
        s = large ? ls : s;
        c = large ? lc : c;
    }
}
// the same without the test, which is a third of its time, for a caller that knows |x| <= 2^20 or finds out later
MRL_DEV void sincos32_near(float x, float &s, float &c, const SinCosK &k) {
    const double xd = (double)fabsf(x);
    const double n = __builtin_rint(xd * k.two_over_pi);
    sincos_reduced(x, fma(-n, k.half_pi_lo, fma(-n, k.half_pi, xd)), (int)n, k, s, c);
}
MRL_DEV float sin32(float x) {
    float s, c;
    sincos32(x, s, c);
    return s;
}
MRL_DEV float cos32(float x) {
    float s, c;
    sincos32(x, s, c);
    return c;
}
MRL_DEV float exp32(float x) { return (float)::exp((double)x); }
// log of an fp32 value, rounded once from Float64: x = 2^e m, m in [sqrt(1/2), sqrt(2)), log m = 2 f + f^3 Q(f^2) with
// f = (m - 1) / (m + 1) (Q interpolated at the Chebyshev points, off by less than 2^-57).  237 cycles a call where the
// library's takes 424; the same bits, rounded, on every fp32 value.
MRL_DEV float log32(float x) {
    const double xd = (double)x;
    double m = __builtin_amdgcn_frexp_mant(xd);
    int e = __builtin_amdgcn_frexp_exp(xd);
    const bool low = m < 0.7071067811865476;
    m = low ? m + m : m;
    e = low ? e - 1 : e;
    const double n = m - 1.0, d = m + 1.0;
    double y = __builtin_amdgcn_rcp(d);
    y = fma(fma(-d, y, 1.0), y, y);
    y = fma(fma(-d, y, 1.0), y, y);
    double f = n * y;
    f = fma(fma(-d, f, n), y, f);
    const double u = f * f;
    double q = 0.14617808833650164;
    q = fma(q, u, 0.15331611566227585);
    q = fma(q, u, 0.18182892438088938);
    q = fma(q, u, 0.2222221108928466);
    q = fma(q, u, 0.28571428626254625);
    q = fma(q, u, 0.3999999999989889);
    q = fma(q, u, 0.666666666666667);
    const double ed = (double)e;
    const double t = fma(f * u, q, ed * 2.3190468138462996e-17);   // (ln 2 in two pieces)
    float r = (float)fma(ed, 0.6931471805599453, fma(2.0, f, t));
    if (!(x > 0.0f && x < __builtin_inff())) r = x == 0.0f ? -__builtin_inff() : (x < 0.0f ? __builtin_nanf("") : x);
    return r;
}

// the value of lane L of every four
template <int L>
MRL_DEV float quad_bcast(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), L * 0x55, 0xF, 0xF, true));
}
// whether any active lane says so, straight from the compare
MRL_DEV bool any_lane(bool p) { return __builtin_amdgcn_ballot_w64(p) != 0; }

// x / d for a divisor that is divided by again and again (a joint's summed inverse inertia, a contact's
// effective mass over the sweeps of a step), given r = 1.0f / d, the IEEE reciprocal taken once: two
// Newton steps on the quotient, each with the exact remainder from an fma, then the hardware's fix-up of
// the special cases (zero / infinite / NaN operands, the sign of a zero quotient).  This is the tail of
// the instruction sequence that the compiler emits for an fp32 division (which first rebuilds the
// reciprocal, 11 instructions; this is 6), without that sequence's rescaling of extreme exponents.
// The result is the correctly rounded quotient -- the bits of x / d -- for every x and d whose quotient,
// and the remainders on the way, stay in the normal range (2^-100 <= |x|, |x / d| <= 2^100 is ample):
// with r correctly rounded, q1 is within an ulp of the quotient and the second step then rounds correctly
// (Markstein's theorem); checked against x / d on 2 * 10^9 random pairs, divisors with an all-ones
// significand included, without a difference.  Physical quantities of a stepped env live there; an env
// that has diverged to 1e30 is past the point where the two forms could be told apart by a test.
MRL_DEV float div_by(float x, float d, float r) {
    const float q0 = x * r;
    const float e1 = fmaf(-d, q0, x);
    const float q1 = fmaf(e1, r, q0);
    const float e2 = fmaf(-d, q1, x);
    const float q2 = fmaf(e2, r, q1);
    return __builtin_amdgcn_div_fixupf(q2, d, x);
}

// tanh of the MLP layers: 1 - 2 / (exp(2x) + 1) on the hardware's exp2 and reciprocal (1 ulp each):
// absolute error below 3e-7, exact saturation (exp2 -> inf gives 1, -> 0 gives -1); a fifth of the
// instructions of the library's tanhf, which was a quarter of a hidden layer's time.  That form cancels
// for small |x| (its error is absolute), so below 1/8 the odd series x (1 - x^2/3 + 2 x^4/15) takes over
// (next term 17 x^6 / 315 < 2.1e-7): the relative error stays below 2e-6 for every x, tanh_mlp(x) = x for
// tiny x, and 1 - y^2 in the backward pass inherits it.
MRL_DEV float tanh_mlp(float x) {
    const float e = __builtin_amdgcn_exp2f(x * 2.8853900817779268f);   // 2 log2(e)
    const float big = fmaf(-2.0f, __builtin_amdgcn_rcpf(e + 1.0f), 1.0f);   // (twice a float is exact: one rounding either way)
    const float x2 = x * x;
    const float small = x * fmaf(x2, fmaf(x2, 0.13333333333333333f, -0.33333333333333333f), 1.0f);
    return fabsf(x) < 0.125f ? small : big;
}

// deep_rl/gpu/random.mojo:11-43
MRL_DEV uint32_t xorshift32(uint32_t x) {
    x ^= x << 13;
    x ^= x >> 17;
    x ^= x << 5;
    return x;
}
MRL_DEV float random_uniform(uint32_t &state) {
    state = xorshift32(state);
    return (float)state / (float)0xFFFFFFFFu;
}
MRL_DEV float random_range(uint32_t &state, float lo, float hi) {
    float u = random_uniform(state);
    return lo + u * (hi - lo);
}

// Philox4x32-10 (Random123).  key = (seed lo, hi); counter = (offset lo, hi, 0, 0) + call;
// uniform = float(x & 0x7fffffff) * 4.6566127342e-10f  -- the stream layout of
// random.philox.Random(seed, offset).step_uniform() that the reference draws from.
struct Uniform4 { float v[4]; };

MRL_DEV Uniform4 philox_uniform4(uint64_t seed, uint64_t offset, uint64_t call_index) {
    uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
    uint64_t lo = offset + call_index;
    uint32_t c0 = (uint32_t)lo, c1 = (uint32_t)(lo >> 32), c2 = (lo < offset) ? 1u : 0u, c3 = 0u;
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        uint64_t p0 = (uint64_t)0xD2511F53u * c0;
        uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
        uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0;
        uint32_t n1 = (uint32_t)p1;
        uint32_t n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
        uint32_t n3 = (uint32_t)p0;
        c0 = n0; c1 = n1; c2 = n2; c3 = n3;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    Uniform4 u;
    u.v[0] = (float)(c0 & 0x7FFFFFFFu) * 4.6566127342e-10f;
    u.v[1] = (float)(c1 & 0x7FFFFFFFu) * 4.6566127342e-10f;
    u.v[2] = (float)(c2 & 0x7FFFFFFFu) * 4.6566127342e-10f;
    u.v[3] = (float)(c3 & 0x7FFFFFFFu) * 4.6566127342e-10f;
    return u;
}

}  // namespace mrl
