/*
 * libm_f32.h -- single-precision logf / sinf that reproduce the host C
 * library bit for bit on the inputs of NeMo's Gaussian RNG.
 *
 * NeMo's nrand() (src/nemo/RNG.cpp:25-33) calls the host's logf and sinf.
 * glibc >= 2.28 implements both with the algorithms published in ARM's
 * "optimized-routines" project (math/logf.c, math/sinf.c, math/sincosf.h,
 * math/logf_data.c, math/sincosf_data.c): a 16-entry table plus a degree-3
 * polynomial in double for logf, and a quadrant reduction plus even/odd
 * double polynomials for sinf. This file restates those algorithms in
 * double precision so they run on gfx950 FP64 and on the host alike.
 *
 * glibc rounds a double result to float once, at the end, so other orders of
 * the same double operations give the same float except where the double
 * lands within its last bits of a rounding boundary. The forms here are
 * shorter than the published ones and free of branches: Horner polynomials
 * with fma(), the quadrant found by adding 1.5 * 2^52 (its nearest integer
 * lands in the sum's low bits), one evaluation for small and reduced
 * arguments. Each was compared with the host libm on every input that
 * reaches it, with zero differences: logf at all x = m * 2^-24
 * (m = 0..2^24), sinf at every float |a| < 120 (2.2e9 values), which holds
 * the RNG's a = float(u) * 1.4629180792671596810513378043098e-9f.
 * tests/test_libm_f32.py repeats the check on the RNG's arguments and, for
 * sinf, on a sample of the wider domain with the floats around each
 * multiple of pi/2.
 *
 * logf is supported for x in [0, 1] only (no NaN / negative paths). sinf
 * takes every float: besides the RNG's arguments, the Kuramoto model feeds
 * it phase differences of either sign and whatever magnitude the coupling
 * produces, so the large-argument reduction (|a| >= 120, by integer
 * multiplication with 2/pi) is restated too. The wider domain is checked
 * against the host C library by tests/test_libm_f32.py and, on the device,
 * by the GPU libm tests.
 */
#ifndef NEMOSIM_LIBM_F32_H
#define NEMOSIM_LIBM_F32_H

#include <math.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define NEMO_HD __host__ __device__
#else
#define NEMO_HD
#endif

namespace nemo_libm {

NEMO_HD inline uint32_t f2u(float f) { union { float f; uint32_t u; } x; x.f = f; return x.u; }
NEMO_HD inline float u2f(uint32_t u) { union { float f; uint32_t u; } x; x.u = u; return x.f; }

/* 1/c and log(c) for the 16 sub-intervals of [0x3f330000, 2*0x3f330000) */
struct LogfEntry { double invc, logc; };

/* constexpr, so that clang makes the table available to device code too */
constexpr LogfEntry LOGF_TABLE[16] = {
	{ 0x1.661ec79f8f3bep+0, -0x1.57bf7808caadep-2 },
	{ 0x1.571ed4aaf883dp+0, -0x1.2bef0a7c06ddbp-2 },
	{ 0x1.49539f0f010bp+0, -0x1.01eae7f513a67p-2 },
	{ 0x1.3c995b0b80385p+0, -0x1.b31d8a68224e9p-3 },
	{ 0x1.30d190c8864a5p+0, -0x1.6574f0ac07758p-3 },
	{ 0x1.25e227b0b8eap+0, -0x1.1aa2bc79c81p-3 },
	{ 0x1.1bb4a4a1a343fp+0, -0x1.a4e76ce8c0e5ep-4 },
	{ 0x1.12358f08ae5bap+0, -0x1.1973c5a611cccp-4 },
	{ 0x1.0953f419900a7p+0, -0x1.252f438e10c1ep-5 },
	{ 0x1p+0, 0x0p+0 },
	{ 0x1.e608cfd9a47acp-1, 0x1.aa5aa5df25984p-5 },
	{ 0x1.ca4b31f026aap-1, 0x1.c5e53aa362eb4p-4 },
	{ 0x1.b2036576afce6p-1, 0x1.526e57720db08p-3 },
	{ 0x1.9c2d163a1aa2dp-1, 0x1.bc2860d22477p-3 },
	{ 0x1.886e6037841edp-1, 0x1.1058bc8a07ee1p-2 },
	{ 0x1.767dcf5534862p-1, 0x1.4043057b6ee09p-2 },
};

/* logf for x in [0, 1]: x = 2^k z with z in [OFF, 2 OFF); log(x) =
 * log1p(z/c - 1) + log(c) + k ln2, log1p by a degree-3 polynomial. */
NEMO_HD inline float logf_glibc(float x)
{
	const double A0 = -0x1.00ea348b88334p-2;
	const double A1 = 0x1.5575b0be00b6ap-2;
	const double A2 = -0x1.ffffef20a4123p-2;
	const double LN2 = 0x1.62e42fefa39efp-1;
	const uint32_t OFF = 0x3f330000u;

	const uint32_t ix = f2u(x);
	const uint32_t tmp = ix - OFF;
	const int i = int((tmp >> 19) & 15u);
	const int k = int32_t(tmp) >> 23;
	const uint32_t iz = ix - (tmp & 0xff800000u);
	const LogfEntry& e = LOGF_TABLE[i];
	const double r = fma(double(u2f(iz)), e.invc, -1.0);
	const double y0 = fma(double(k), LN2, e.logc);
	const double y = fma(A0 * r + A1, r, A2);   /* one constant per operation: see sinf_rng */
	const float v = float(fma(fma(y, r, 1.0), r, y0));
	return ix == 0u ? -__builtin_inff() : v;   /* log(1) comes out as +0 */
}

/* Sine and cosine of a reduced argument, |x| <= pi/4 */
NEMO_HD inline double sinf_poly_sin(double x, double x2)
{
	const double S1 = -0x1.555545995a603p-3;
	const double S2 = 0x1.1107605230bc4p-7;
	const double S3 = -0x1.994eb3774cf24p-13;
	return fma(x * x2, fma(x2, fma(x2, S3, S2), S1), x);
}

NEMO_HD inline double sinf_poly_cos(double x2)
{
	const double C1 = -0x1.ffffffd0c621cp-2;
	const double C2 = 0x1.55553e1068f19p-5;
	const double C3 = -0x1.6c087e89a359dp-10;
	const double C4 = 0x1.99343027bf8c3p-16;
	return fma(x2, fma(x2, fma(x2, fma(x2, C4, C3), C2), C1), 1.0);
}

/* sinf for |y| < 120: x = y - q pi/2 with q the nearest integer to 2y/pi
 * (0 for a small argument, which it leaves as it is), the sine or cosine of
 * x by q's lowest bit, negated by its next. Both polynomials are evaluated:
 * a wave's lanes need both, and 4 multiply-adds are less than a branch. An
 * argument below 2^-12 is its own sine (which also keeps the sign of 0). */
NEMO_HD inline float sinf_reduced(float y)
{
	const double INV_HPI = 0x1.45F306DC9C883p-1;
	const double HPI = 0x1.921FB54442D18p0;
	const double ROUND = 0x1.8p52;

	const double y64 = y;
	union { double d; uint64_t u; } t;
	t.d = fma(y64, INV_HPI, ROUND);
	const uint32_t q = uint32_t(t.u);
	const double x = fma(ROUND - t.d, HPI, y64);
	const double x2 = x * x;
	const double s = sinf_poly_sin(x, x2);
	const double c = sinf_poly_cos(x2);
	const uint32_t v = f2u(float((q & 1u) ? c : s)) ^ ((q & 2u) << 30);
	return __builtin_fabsf(y) < 0x1p-12f ? y : u2f(v);
}

/* sinf for the RNG's arguments, in [0, 2*pi + 1ulp]: sinf_reduced with at
 * most one constant per operation. gfx950 takes one scalar operand per vector
 * instruction, so a multiply-add of two constants keeps one of them in a
 * vector register pair, hoisted out of the step kernel's cycle loop, where it
 * spills. Compared with the host libm at every float in [0, 6.283186]
 * (1.09e9 values): zero differences. */
NEMO_HD inline float sinf_rng(float y)
{
	const double INV_HPI = 0x1.45F306DC9C883p-1;
	const double HPI = 0x1.921FB54442D18p0;
	const double ROUND = 0x1.8p52;
	const double S1 = -0x1.555545995a603p-3, S2 = 0x1.1107605230bc4p-7, S3 = -0x1.994eb3774cf24p-13;
	const double C1 = -0x1.ffffffd0c621cp-2, C2 = 0x1.55553e1068f19p-5, C3 = -0x1.6c087e89a359dp-10,
			C4 = 0x1.99343027bf8c3p-16;

	const double y64 = y;
	union { double d; uint64_t u; } t;
	t.d = y64 * INV_HPI + ROUND;
	const uint32_t q = uint32_t(t.u);
	const double x = fma(ROUND - t.d, HPI, y64);
	const double x2 = x * x;
	const double s = fma(x * x2, x2 * (x2 * S3 + S2) + S1, x);
	const double c = fma(x2, x2 * (x2 * (x2 * C4 + C3) + C2) + C1, 1.0);
	const uint32_t v = f2u(float((q & 1u) ? c : s)) ^ ((q & 2u) << 30);
	return y < 0x1p-12f ? y : u2f(v);
}

/* Bits of 2/pi: entry i is floor(2/pi * 2^(8(i+1))) mod 2^32, i.e. the
 * 32-bit window ending at byte i+1 of the binary expansion. The table is a
 * property of the number (tests/test_libm_f32.py recomputes it from pi with
 * integer arithmetic). */
constexpr uint32_t INV_PIO4_BITS[24] = {
	0xa2u, 0xa2f9u, 0xa2f983u, 0xa2f9836eu, 0xf9836e4eu, 0x836e4e44u, 0x6e4e4415u, 0x4e441529u,
	0x441529fcu, 0x1529fc27u, 0x29fc2757u, 0xfc2757d1u, 0x2757d1f5u, 0x57d1f534u, 0xd1f534ddu, 0xf534ddc0u,
	0x34ddc0dbu, 0xddc0db62u, 0xc0db6295u, 0xdb629599u, 0x6295993cu, 0x95993c43u, 0x993c4390u, 0x3c439041u,
};

/* Reduction of |a| >= 120 (the float's bits in xi, sign ignored) to
 * r in about [-pi/4, pi/4] and the quadrant n: the 24-bit significand times
 * a 96-bit window of 2/pi (chosen by the exponent) gives the product modulo
 * 4 as a 2.62 fixed-point number, exactly; n is its rounded integer part,
 * and the remainder, converted to double, is scaled by pi/2 * 2^-62. */
NEMO_HD inline double sinf_reduce_large(uint32_t xi, int* np)
{
	const uint32_t* w = &INV_PIO4_BITS[(xi >> 26) & 15u];
	const int shift = int((xi >> 23) & 7u);
	uint32_t m = ((xi & 0xffffffu) | 0x800000u) << shift;
	uint64_t hi = uint64_t(uint32_t(m * w[0]));           /* only its low 32 bits matter */
	uint64_t mid = uint64_t(m) * w[4];
	uint64_t lo = uint64_t(m) * w[8];
	uint64_t acc = ((lo >> 32) | (hi << 32)) + mid;
	uint64_t n = (acc + (uint64_t(1) << 61)) >> 62;
	acc -= n << 62;
	*np = int(n);
	return double(int64_t(acc)) * 0x1.921FB54442D18p-62;
}

/* sinf of any float: |a| < 120 by sinf_reduced; larger finite |a| by
 * sinf_reduce_large, whose sign rule takes the argument's sign in; NaN for
 * infinities and NaN. */
NEMO_HD inline float sinf_glibc(float y)
{
	if(__builtin_fabsf(y) < 120.0f) {
		return sinf_reduced(y);
	}
	const uint32_t yi = f2u(y);
	if(((yi >> 20) & 0x7ffu) >= ((f2u(__builtin_inff()) >> 20) & 0x7ffu)) {
		return (y - y) / (y - y);
	}
	int n = 0;
	const double x = sinf_reduce_large(yi, &n);
	const int m = n + int(yi >> 31);
	/* quadrant n picks the polynomial, m = n plus the argument's sign bit
	 * the sign */
	const double v = (n & 1) ? sinf_poly_cos(x * x) : sinf_poly_sin(x, x * x);
	const bool neg = (n & 1) ? (m & 2) != 0 : (((m & 3) == 1) || ((m & 3) == 2));
	return neg ? -float(v) : float(v);
}

/* The phase wrap of the Kuramoto model (src/nemo/cpu/plugins/Kuramoto.cpp:
 * 121, 150): fmodf by 2*pi rounded to float, then, for a negative phase,
 * 2*pi added in double -- the reference's expression mixes the float
 * remainder with the double constant 2.0f*M_PI -- and the sum rounded to
 * float. fmodf is exact, so any correct implementation gives the same
 * remainder. */
NEMO_HD inline float kuramoto_wrap(float phase)
{
	const double TWO_PI = 6.283185307179586;
	const float r = fmodf(phase, float(TWO_PI));
	return float(double(r) + (phase < 0.0f ? TWO_PI : 0.0));
}

} // namespace nemo_libm

#endif
