// Device-side tracking physics for gfx950.
//
// Every floating-point expression keeps the operation order of the reference
// function cited beside it (paths relative to the reference's source/), and
// the library is compiled with -ffp-contract=off, so each step is
// bit-reproducible against a CPU evaluation of the same expressions.
// Transcendentals are the float routines of this file (see "math").
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace nbl { namespace dev {

constexpr float EPS = 10.0f * 1.1920928955078125e-07f;  // config/data_types.h:55
constexpr float PI_F = 3.1415926535897932f;             // config/config.h:32
// Bounds on the two unbounded loops of the reference (octree cell walk,
// plasmon-decay rejection), so that every wave finishes.
constexpr uint32_t MAX_CELLS = 1000000u;
constexpr int MAX_REJECT = 1000;

// Special material indices (core/material_manager.h:77-86).
constexpr int MAT_NOP = -128, MAT_TERMINATOR = -127, MAT_DETECTOR = -126,
	MAT_DETECTOR_LT50 = -125, MAT_DETECTOR_GE50 = -124, MAT_VACUUM = -123,
	MAT_MIRROR = -122;

// Physics option bits (same values as NBL_PHYS_* in nebula.h).
constexpr uint32_t PH_EL_PHONON = 1u << 0, PH_EL_RECOIL = 1u << 1, PH_PN_SE = 1u << 2,
	PH_KI_OPTICAL = 1u << 3, PH_KI_SE = 1u << 4, PH_KI_INST = 1u << 5, PH_KI_MOMCONS = 1u << 6,
	PH_BI_QUANTUM = 1u << 7, PH_BI_REFRACT = 1u << 8, PH_BI_ABSORB = 1u << 9;

enum { ALIVE = 0, TERMINATED = 1, DETECTED = 2 };
enum { EV_NONE = 0, EV_INELASTIC = 1, EV_ELASTIC = 2, EV_INTERSECT = 3 };
// Particle flags.
constexpr uint32_t FL_PEND_INEL = 1u, FL_PEND_DET = 2u;
// The particle's step has been planned (its direction is the normalised one,
// the step is counted); FL_WALK: its walk has begun and is kept beside it.
constexpr uint32_t FL_PLANNED = 4u, FL_WALK = 8u;
// Bits 16..31 of a particle's flags: its world (geometry + material set) in
// a driver that tracks several scans at once.
constexpr uint32_t FL_WORLD_SHIFT = 16u, FL_WORLD_MASK = 0xffff0000u;

struct F3 { float x, y, z; };

// Lanes with p set.  (HIP's __ballot takes an int: a select and a compare more
// where p is not a compare's result.)
__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }

// ------------------------------------------------------------------ math --
// Float transcendentals built from IEEE float +, -, *, / and integer bit
// operations only, so that (compiled without FMA contraction) they give the
// same bits on the GPU and in a CPU evaluation.  Methods: exponent/mantissa
// split with log(1+f) = f - f^2/2 + s(f^2/2 + R(s^2)), s = f/(2+f), R the
// atanh series; Cody-Waite reduction by k ln2 or k pi/2 with split constants
// and Taylor polynomials; arctangent by reduction to |u| <= tan(pi/8) and a
// least-squares polynomial; cube root by a bit-level first guess and four
// Newton steps.  All within 2.5 ulp of the exact functions.
__device__ __forceinline__ float pf_nan() { return __uint_as_float(0x7fc00000u); }
__device__ __forceinline__ float pf_pow2(int k) { return __uint_as_float((uint32_t)(k + 127) << 23); }
constexpr float PF_P1 = 0x1.922p+0f, PF_P2 = -0x1.2aep-18f, PF_P3 = -0x1.de973ep-31f;
constexpr float PF_LN2_HI = 0x1.62e4p-1f, PF_LN2_LO = 0x1.7f7d1cp-20f, PF_INV_LN2 = 0x1.715476p+0f;
constexpr float PF_PI_HI = 0x1.921fb6p+1f, PF_PI_LO = -0x1.777a5cp-24f;
constexpr float PF_PI_2_HI = 0x1.921fb6p+0f, PF_PI_2_LO = -0x1.777a5cp-25f;
constexpr float PF_PI_4_HI = 0x1.921fb6p-1f, PF_PI_4_LO = -0x1.777a5cp-26f;
constexpr float PF_TWO_OVER_PI = 0x1.45f306p-1f, PF_TAN_PI_8 = 0x1.a8279ap-2f;

// Correctly rounded quotients and square roots for operands whose size is
// known: the compiler's division scales, refines and fixes up for every
// float (12 issue slots of the VALU, 16 for a square root), which the step
// kernel, bound by VALU issue, does 30 times a step.  A reciprocal of v_rcp's
// accuracy (1 ulp) refined once, a quotient from it and one fused correction
// (Markstein's theorem, IBM J. Res. Dev. 34, 1990) need 4 and 3 slots.
// Compared with / and sqrtf on every float in the stated ranges, and the
// quotients on 10^11 random pairs and on all numerators for the mantissas
// next to a power of two: the same bits.  With the short logarithm,
// exponential, phase and table index below and one Philox block a step instead
// of one more for boundary events, the step kernel issues 18 % fewer VALU
// instructions: 6 553 600 primaries of 300 eV 288 -> 277 ms, 100 of 1 keV in a
// slab 1.92 -> 1.75.  (What the tests repeat is whole steps, bit for bit, with
// operands in the ranges and outside them.)
//
// 1 / x, |x| in [2^-100, 2^100].
__device__ __forceinline__ float rcp_mid(float x)
{
	const float y = __builtin_amdgcn_rcpf(x);
	return __builtin_fmaf(__builtin_fmaf(-x, y, 1.0f), y, y);
}
// a / b from y = rcp_mid(b), for |a / b| and |a| in [2^-100, 2^100] or a = +0.
// (A smaller |a| gives a quotient within an ulp.)
__device__ __forceinline__ float div_by(float a, float b, float y)
{
	const float q = a * y;
	return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
}
__device__ __forceinline__ float div_mid(float a, float b) { return div_by(a, b, rcp_mid(b)); }
// In [2^-100, 2^100]?
__device__ __forceinline__ bool is_mid(float x) { return __float_as_uint(x) - 0x0d800000u <= 0x64000000u; }
// sqrt(x), x in [2^-100, 2^100] or 0.
__device__ __forceinline__ float sqrt_mid(float x)
{
	const float y = __builtin_amdgcn_rsqf(fmaxf(x, 0x1p-100f));
	const float g = x * y;
	return __builtin_fmaf(__builtin_fmaf(-g, g, x), 0.5f * y, g);
}
// 1 / sqrt(x), both operations rounded.  (Refining v_rsq instead of a new
// reciprocal misses where the root is next to a power of two: at unit vectors.)
__device__ __forceinline__ float rsqrt_ieee(float x)
{
	return is_mid(x) ? rcp_mid(sqrt_mid(x)) : 1.0f / sqrtf(x);
}

__device__ inline float pf_log(float x)
{
	if (x != x) return x;
	if (x < 0.0f) return pf_nan();
	if (x == 0.0f) return -__builtin_inff();
	uint32_t i = __float_as_uint(x);
	if (i >= 0x7f800000u) return x;
	int e = 0;
	if (i < 0x00800000u) { x = x * 0x1p25f; i = __float_as_uint(x); e = -25; }
	e += (int)(i >> 23) - 127;
	const uint32_t m = i & 0x007fffffu;
	if (m > 0x3504f3u) { i = m | 0x3f000000u; e += 1; }
	else i = m | 0x3f800000u;
	const float f = __uint_as_float(i) - 1.0f;
	const float s = f / (2.0f + f);
	const float z = s * s;
	const float R = z * (0x1.555556p-1f + z * (0x1.99999ap-2f + z * (0x1.24924ap-2f + z * 0x1.c71c72p-3f)));
	const float hfsq = 0.5f * f * f;
	const float l1p = f - (hfsq - s * (hfsq + R));
	const float fe = (float)e;
	return fe * PF_LN2_HI + (l1p + fe * PF_LN2_LO);
}

// pf_log of a normal positive float (a uniform draw among them): no special
// values, the same operations otherwise.
__device__ __forceinline__ float pf_log_normal(float x)
{
	uint32_t i = __float_as_uint(x);
	// the exponent, one more for mantissas above 0x3504f3
	const uint32_t u = i - 0x3f3504f4u;
	const float fe = (float)((int)u >> 23);
	const float f = __uint_as_float(i - (u & 0xff800000u)) - 1.0f;
	const float s = div_mid(f, 2.0f + f);
	const float z = s * s;
	const float R = z * (0x1.555556p-1f + z * (0x1.99999ap-2f + z * (0x1.24924ap-2f + z * 0x1.c71c72p-3f)));
	const float hfsq = 0.5f * f * f;
	const float l1p = f - (hfsq - s * (hfsq + R));
	return fe * PF_LN2_HI + (l1p + fe * PF_LN2_LO);
}
__device__ __forceinline__ float pf_log_fast(float x)
{
	return __builtin_expect(__float_as_uint(x) - 0x00800000u < 0x7f000000u, 1) ? pf_log_normal(x) : pf_log(x);
}

__device__ __forceinline__ float pf_exp_p(float r)
{
	return 0.5f + r * (0x1.555556p-3f + r * (0x1.555556p-5f + r * (0x1.111112p-7f
		+ r * (0x1.6c16c2p-10f + r * 0x1.a01a02p-13f))));
}

__device__ inline float pf_exp(float x)
{
	if (x != x) return x;
	if (x > 0x1.62e42ep+6f) return __builtin_inff();
	if (x < -0x1.9fe368p+6f) return 0.0f;
	const float kf = rintf(x * PF_INV_LN2);
	const int k = (int)kf;
	const float r = (x - kf * PF_LN2_HI) - kf * PF_LN2_LO;
	const float e = 1.0f + (r + (r * r) * pf_exp_p(r));
	if (k > 127) return (e * 0x1p127f) * pf_pow2(k - 127);
	if (k < -126) return (e * 0x1p-126f) * pf_pow2(k + 126);
	return e * pf_pow2(k);
}

// pf_exp, short for |x| <= 86 (the power of two is a normal float there)
__device__ __forceinline__ float pf_exp_short(float x)
{
	const float kf = rintf(x * PF_INV_LN2);
	const float r = (x - kf * PF_LN2_HI) - kf * PF_LN2_LO;
	return __builtin_amdgcn_ldexpf(1.0f + (r + (r * r) * pf_exp_p(r)), (int)kf);
}
__device__ __forceinline__ float pf_exp_fast(float x)
{
	return (fabsf(x) <= 86.0f) ? pf_exp_short(x) : pf_exp(x);
}

__device__ inline float pf_expm1(float x)
{
	if (x != x) return x;
	if (x > 0x1.62e42ep+6f) return __builtin_inff();
	if (x < -0x1.154246p+4f) return -1.0f;
	if (fabsf(x) < 0x1.62e430p-2f) {
		if (fabsf(x) < 0x1p-28f) return x;
		return x + (x * x) * pf_exp_p(x);
	}
	const float kf = rintf(x * PF_INV_LN2);
	const int k = (int)kf;
	const float r = (x - kf * PF_LN2_HI) - kf * PF_LN2_LO;
	const float em = r + (r * r) * pf_exp_p(r);
	if (k > 127) return ((em + 1.0f) * 0x1p127f) * 2.0f - 1.0f;
	const float t = pf_pow2(k);
	return em * t + (t - 1.0f);
}

__device__ inline float pf_cbrt(float x)
{
	if (x != x || x == 0.0f || fabsf(x) == __builtin_inff()) return x;
	float ax = fabsf(x);
	float post = 1.0f;
	if (ax < 0x1p-126f) { ax = ax * 0x1p24f; post = 0x1p-8f; }
	float y = __uint_as_float(__float_as_uint(ax) / 3u + 0x2a555555u);
#pragma unroll
	for (int it = 0; it < 4; ++it)
		y = (2.0f * y + ax / (y * y)) / 3.0f;
	y = y * post;
	return copysignf(y, x);
}

__device__ __forceinline__ float pf_sin_r(float r)
{
	const float z = r * r;
	return r + (r * z) * (-0x1.555556p-3f + z * (0x1.111112p-7f + z * (-0x1.a01a02p-13f
		+ z * (0x1.71de3ap-19f + z * -0x1.ae6456p-26f))));
}
__device__ __forceinline__ float pf_cos_r(float r)
{
	const float z = r * r;
	return 1.0f - (0.5f * z - (z * z) * (0x1.555556p-5f + z * (-0x1.6c16c2p-10f
		+ z * (0x1.a01a02p-16f + z * -0x1.27e4fcp-22f))));
}
__device__ __forceinline__ float pf_reduce(float x, int& q)
{
	const float kf = rintf(x * PF_TWO_OVER_PI);
	q = ((int)kf) & 3;
	return ((x - kf * PF_P1) - kf * PF_P2) - kf * PF_P3;
}
// sin and cos of the same argument (the reference calls sincos on the CPU
// as separate sin and cos, which give the same values as these)
__device__ inline void pf_sincos(float x, float& s, float& c)
{
	if (x != x || fabsf(x) == __builtin_inff()) { s = pf_nan(); c = pf_nan(); return; }
	int q;
	const float r = pf_reduce(x, q);
	const float sr = pf_sin_r(r), cr = pf_cos_r(r);
	switch (q) {
	case 0: s = sr; c = cr; break;
	case 1: s = cr; c = -sr; break;
	case 2: s = -sr; c = -cr; break;
	default: s = -cr; c = sr; break;
	}
}

// The same for x in [0, 2 pi]: the quadrant by selects and sign bits.
__device__ __forceinline__ void pf_sincos_phase(float x, float& s, float& c)
{
	const float kf = rintf(x * PF_TWO_OVER_PI);
	const uint32_t q = (uint32_t)(int)kf;
	const float r = ((x - kf * PF_P1) - kf * PF_P2) - kf * PF_P3;
	const float sr = pf_sin_r(r), cr = pf_cos_r(r);
	const bool odd = (q & 1u) != 0u;
	s = __uint_as_float(__float_as_uint(odd ? cr : sr) ^ ((q << 30) & 0x80000000u));
	c = __uint_as_float(__float_as_uint(odd ? sr : cr) ^ (((q + 1u) << 30) & 0x80000000u));
}

__device__ __forceinline__ float pf_atan_r(float u)
{
	const float z = u * u;
	return u + (u * z) * (-0x1.555556p-2f + z * (0x1.999982p-3f + z * (-0x1.248b8p-3f
		+ z * (0x1.c5adfep-4f + z * (-0x1.62ae6ep-4f + z * 0x1.a49afap-5f)))));
}
__device__ inline float pf_atan2(float y, float x)
{
	if (x != x || y != y) return x + y;
	const float ax = fabsf(x), ay = fabsf(y);
	const bool xneg = (__float_as_uint(x) >> 31) != 0;
	if (ay == 0.0f)
		return xneg ? copysignf(PF_PI_HI, y) : y;
	if (ax == 0.0f)
		return copysignf(PF_PI_2_HI, y);
	const float inf = __builtin_inff();
	if (ax == inf || ay == inf) {
		float a;
		if (ax == inf && ay == inf) a = xneg ? 3.0f * PF_PI_4_HI : PF_PI_4_HI;
		else if (ax == inf) a = xneg ? PF_PI_HI : 0.0f;
		else a = PF_PI_2_HI;
		return copysignf(a, y);
	}
	const bool swap = ay > ax;
	const float t = swap ? ax / ay : ay / ax;
	float a;
	if (t > PF_TAN_PI_8)
		a = PF_PI_4_HI + (pf_atan_r((t - 1.0f) / (t + 1.0f)) + PF_PI_4_LO);
	else
		a = pf_atan_r(t);
	if (swap) a = (PF_PI_2_HI - a) + PF_PI_2_LO;
	if (xneg) a = (PF_PI_HI - a) + PF_PI_LO;
	return copysignf(a, y);
}

__device__ __forceinline__ float m_log(float x) { return pf_log_fast(x); }
__device__ __forceinline__ float m_exp(float x) { return pf_exp_fast(x); }
__device__ __forceinline__ float m_expm1(float x) { return pf_expm1(x); }
__device__ __forceinline__ float m_cbrt(float x) { return pf_cbrt(x); }
__device__ __forceinline__ float m_atan2(float y, float x) { return pf_atan2(y, x); }

// common/scalar_math.h:16-25; float->int conversions follow the x86 CPU
// build for out-of-range and NaN inputs (INT_MIN).
__device__ __forceinline__ int clampi(int i, int lo, int hi) { return i < lo ? lo : (i > hi ? hi : i); }
__device__ __forceinline__ float clampr(float i, float lo, float hi) { return i < lo ? lo : (i > hi ? hi : i); }
__device__ __forceinline__ float fmin_std(float a, float b) { return (b < a) ? b : a; }
__device__ __forceinline__ float fmax_std(float a, float b) { return (a < b) ? b : a; }
__device__ __forceinline__ int to_int_x86(float f)
{
	return (f >= -2147483648.0f && f < 2147483648.0f) ? (int)f : (int)0x80000000;
}
__device__ __forceinline__ int floorr(float x) { return to_int_x86(floorf(x)); }
__device__ __forceinline__ int rintr(float x) { return to_int_x86(rintf(x)); }
__device__ __forceinline__ float saturater(float x) { return clampr(x, 0.0f, 1.0f); }

// common/vector_math.h
__device__ __forceinline__ F3 v_add(F3 a, F3 b) { return { a.x + b.x, a.y + b.y, a.z + b.z }; }
__device__ __forceinline__ F3 v_sub(F3 a, F3 b) { return { a.x - b.x, a.y - b.y, a.z - b.z }; }
__device__ __forceinline__ F3 v_mul(F3 a, float b) { return { a.x * b, a.y * b, a.z * b }; }
__device__ __forceinline__ F3 s_mul(float a, F3 b) { return { a * b.x, a * b.y, a * b.z }; }
__device__ __forceinline__ F3 cross(F3 a, F3 b)
{
	return { a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x };
}
__device__ __forceinline__ float dot(F3 a, F3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ float mag2(F3 a) { return a.x * a.x + a.y * a.y + a.z * a.z; }
// normalised(): a * (1/sqrt(a.a)) with IEEE sqrt and division.
__device__ __forceinline__ F3 normalised(F3 a)
{
	return v_mul(a, rsqrt_ieee(a.x * a.x + a.y * a.y + a.z * a.z));
}
// The same for a normalised vector (or NaN, or zero: then NaN, as above).
__device__ __forceinline__ F3 normalised_unit(F3 a)
{
	return v_mul(a, rcp_mid(sqrt_mid(a.x * a.x + a.y * a.y + a.z * a.z)));
}
// vector_math.h:171-186; phi in [0, 2 pi]
__device__ __forceinline__ F3 make_normal_vec(F3 dir, float phi)
{
	// cos and sin of the azimuth atan2(y, x) as x/r and y/r (equal up to
	// rounding; r = 0 takes the atan2 limits: cosine +-1 by the sign of x)
	const float r2 = dir.x * dir.x + dir.y * dir.y;
	float r, sin_az, cos_az;
	if (is_mid(r2)) {
		r = sqrt_mid(r2);
		const float y = rcp_mid(r);
		cos_az = div_by(dir.x, r, y);
		sin_az = div_by(dir.y, r, y);
	} else {
		r = sqrtf(r2);
		sin_az = 0.0f;
		cos_az = signbit(dir.x) ? -1.0f : 1.0f;
		if (r > 0.0f) {
			cos_az = dir.x / r;
			sin_az = dir.y / r;
		}
	}
	const F3 unit_v = { dir.z * cos_az, dir.z * sin_az, -r };
	const F3 unit_u = cross(unit_v, dir);
	float sin_phi, cos_phi;
	pf_sincos_phase(phi, sin_phi, cos_phi);
	return v_add(v_mul(unit_u, cos_phi), v_mul(unit_v, sin_phi));
}
// vector_math.h:194-206
__device__ inline F3 make_unit_vec(float cos_theta, float phi)
{
	float sin_phi, cos_phi;
	pf_sincos_phase(phi, sin_phi, cos_phi);
	cos_theta = clampr(cos_theta, -1.0f, 1.0f);
	const float sin_theta = sqrt_mid(1.0f - cos_theta * cos_theta);
	return { sin_theta * cos_phi, sin_theta * sin_phi, cos_theta };
}

// ------------------------------------------------------------------- RNG --
// Counter-based Philox4x32-10 (Salmon et al., SC'11): key = run seed,
// counter = (sid lo, sid hi, step, block of four draws).  A particle's draws
// depend only on (seed, sid, step, draw index), so trajectories are
// independent of scheduling and can be replayed.
struct Rng {
	uint32_t k0, k1, c0, c1, c2, idx;
	uint32_t b0, b1, b2, b3;
};

__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t k)
{
	uint32_t r;
	asm("v_bitop3_b32 %0, %1, %2, %3 bitop3:0x96" : "=v"(r) : "v"(a), "v"(b), "s"(k));
	return r;
}

__device__ __forceinline__ void philox4x32_10(uint32_t& c0, uint32_t& c1, uint32_t& c2, uint32_t& c3,
	uint32_t k0, uint32_t k1)
{
	// The keys are the run's seed, the same in every lane.  The empty
	// statement keeps the ten rounds' keys out of registers: computed ahead
	// of the step loop they were spilled and read back lane by lane (1 % of
	// the step kernel); each is one scalar addition.
	k0 = __builtin_amdgcn_readfirstlane(k0);
	k1 = __builtin_amdgcn_readfirstlane(k1);
	asm volatile("" : "+s"(k0), "+s"(k1));
#pragma unroll
	for (int r = 0; r < 10; ++r) {
		// one 64-bit product each (v_mad_u64_u32, as fast as either half),
		// and both XORs in one v_bitop3
		const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
		c0 = xor3((uint32_t)(p1 >> 32), c1, k0);
		c2 = xor3((uint32_t)(p0 >> 32), c3, k1);
		c1 = (uint32_t)p1;
		c3 = (uint32_t)p0;
		k0 += 0x9E3779B9u;
		k1 += 0xBB67AE85u;
	}
}

__device__ __forceinline__ void rng_start(Rng& r, uint32_t k0, uint32_t k1, uint64_t sid, uint32_t step)
{
	r.k0 = k0; r.k1 = k1;
	r.c0 = (uint32_t)sid; r.c1 = (uint32_t)(sid >> 32); r.c2 = step;
	r.idx = 0;
}

// Uniform in (0, 1]: ((w >> 8) + 1) * 2^-24, exact in float.
__device__ __forceinline__ float unit_of(uint32_t w)
{
	return __builtin_fmaf((float)(w >> 8), 0x1p-24f, 0x1p-24f);
}
__device__ __forceinline__ float rng_unit(Rng& r)
{
	const uint32_t i = r.idx & 3u;
	if (i == 0) {
		uint32_t a = r.c0, b = r.c1, c = r.c2, d = r.idx >> 2;
		philox4x32_10(a, b, c, d, r.k0, r.k1);
		r.b0 = a; r.b1 = b; r.b2 = c; r.b3 = d;
	}
	const uint32_t w = (i == 0) ? r.b0 : (i == 1) ? r.b1 : (i == 2) ? r.b2 : r.b3;
	r.idx++;
	return unit_of(w);
}

// The four draws a step's free paths and its elastic or boundary event take
// at most (two each), taken in turn; the event's are kept while it lasts.
struct Draws { uint32_t b0, b1, b2, b3; };
__device__ __forceinline__ Draws step_draws(uint32_t k0, uint32_t k1, uint64_t sid, uint32_t step)
{
	Draws d = { (uint32_t)sid, (uint32_t)(sid >> 32), step, 0u };
	philox4x32_10(d.b0, d.b1, d.b2, d.b3, k0, k1);
	return d;
}
__device__ __forceinline__ float rng_unit(Draws& d)
{
	const float u = unit_of(d.b0);
	d.b0 = d.b1;
	d.b1 = d.b2;
	d.b2 = d.b3;
	return u;
}

// Resume a stream at draw `idx` (re-running an event whose path draws were
// taken by an earlier launch).
__device__ __forceinline__ void rng_seek(Rng& r, uint32_t idx)
{
	const uint32_t blk = idx >> 2;
	uint32_t a = r.c0, b = r.c1, c = r.c2, d = blk;
	philox4x32_10(a, b, c, d, r.k0, r.k1);
	r.b0 = a; r.b1 = b; r.b2 = c; r.b3 = d;
	r.idx = idx;   // rng_unit recomputes the block if idx is a multiple of four
}

// common/util/random.h:56-84: phi = 2 pi U; uniform_vector draws phi first.
template <class R>
__device__ __forceinline__ float rng_phi(R& r) { return (2.0f * PI_F) * rng_unit(r); }
__device__ __forceinline__ F3 rng_uniform_vector(Rng& r)
{
	const float phi = rng_phi(r);
	const float ct = 2.0f * rng_unit(r) - 1.0f;
	return make_unit_vec(ct, phi);
}

// Stream id of a secondary electron: splitmix64 finaliser of the parent's
// (sid, step), top bit set.
__device__ __forceinline__ uint64_t se_sid(uint64_t parent_sid, uint32_t parent_step)
{
	uint64_t z = parent_sid * 0x9E3779B97F4A7C15ull + (uint64_t)parent_step + 1u;
	z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
	z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
	z ^= z >> 31;
	return z | 0x8000000000000000ull;
}

// ---------------------------------------------------------------- tables --
// topx, topy: the last interval's index (n - 2) as a float
struct Table1 { const float* d; int n; float xmin, xstep, topx; };
struct Table2 { const float* d; int nx, ny; float xmin, xstep, ymin, ystep, topx, topy; };
struct Table3 { const float* d; int nx, ny, nz; float xmin, xstep, ymin, ystep, zmin, zstep; };

// clampi(floorr(xi), 0, top) as a float: clamped before the conversion, and
// what to_int_x86 makes INT_MIN (a NaN, 2^31 and above) is index 0.
__device__ __forceinline__ float t_index(float xi, float top)
{
	const float f = __builtin_amdgcn_fmed3f(floorf(xi), 0.0f, top);
	return (xi < 2147483648.0f) ? f : 0.0f;
}
// Table values are in global memory (a pointer read from memory would
// otherwise be loaded from as a flat one).
using GFloat = const __attribute__((address_space(1))) float;

// a float4 at a multiple of 8 bytes
typedef float float4a8 __attribute__((ext_vector_type(4), aligned(8)));

// common/util/table_1D.inl:66-81
__device__ __forceinline__ float t1_get(const Table1& t, float x)
{
	const float xi = (x - t.xmin) * t.xstep;
	const float low = t_index(xi, t.topx);
	GFloat* p = (GFloat*)t.d + (int)low;
	const float lv = p[0], hv = p[1];
	const float frac = xi - low;
	return (1.0f - frac) * lv + frac * hv;
}

// common/util/table_2D.inl:73-94 (row-major [x][y])
__device__ __forceinline__ float t2_get(const Table2& t, float x, float y)
{
	const float xi = (x - t.xmin) * t.xstep;
	const float yi = (y - t.ymin) * t.ystep;
	const float lx = t_index(xi, t.topx), ly = t_index(yi, t.topy);
	GFloat* r0 = (GFloat*)t.d + ((size_t)(uint32_t)(int)lx * (uint32_t)t.ny + (uint32_t)(int)ly);
	GFloat* r1 = r0 + t.ny;
	const float v00 = r0[0], v10 = r1[0], v01 = r0[1], v11 = r1[1];
	const float fx = xi - lx, fy = yi - ly;
	return (1.0f - fx) * (1.0f - fy) * v00
		+ fx * (1.0f - fy) * v10
		+ (1.0f - fx) * fy * v01
		+ fx * fy * v11;
}

// common/util/table_2D.inl:96-114
__device__ __forceinline__ float t2_get_rounddown(const Table2& t, float x, float y)
{
	const float xi = (x - t.xmin) * t.xstep;
	const float yi = (y - t.ymin) * t.ystep;
	const int lx = clampi(floorr(xi), 0, t.nx - 1);
	const int ly = clampi(floorr(yi), 0, t.ny - 1);
	return t.d[(size_t)lx * t.ny + ly];
}
__device__ __forceinline__ float t2_get_nearest(const Table2& t, float x, float y)
{
	const float xi = (x - t.xmin) * t.xstep;
	const float yi = (y - t.ymin) * t.ystep;
	const int nx = clampi(rintr(xi), 0, t.nx - 1);
	const int ny = clampi(rintr(yi), 0, t.ny - 1);
	return t.d[(size_t)nx * t.ny + ny];
}

// common/util/table_3D.inl:78-121 ([x][y][z])
__device__ __forceinline__ float t3_get(const Table3& t, float x, float y, float z)
{
	const float xi = (x - t.xmin) * t.xstep;
	const float yi = (y - t.ymin) * t.ystep;
	const float zi = (z - t.zmin) * t.zstep;
	const int lx = clampi(floorr(xi), 0, t.nx - 2);
	const int ly = clampi(floorr(yi), 0, t.ny - 2);
	const int lz = clampi(floorr(zi), 0, t.nz - 2);
	const size_t sy = (size_t)t.nz, sx = (size_t)t.ny * t.nz;
	const float* p = t.d + (size_t)lx * sx + (size_t)ly * sy + lz;
	const float v000 = p[0], v001 = p[1];
	const float v010 = p[sy], v011 = p[sy + 1];
	const float v100 = p[sx], v101 = p[sx + 1];
	const float v110 = p[sx + sy], v111 = p[sx + sy + 1];
	const float fx = xi - (float)lx, fy = yi - (float)ly, fz = zi - (float)lz;
	return (1.0f - fx) * (1.0f - fy) * (1.0f - fz) * v000
		+ fx * (1.0f - fy) * (1.0f - fz) * v100
		+ (1.0f - fx) * fy * (1.0f - fz) * v010
		+ fx * fy * (1.0f - fz) * v110
		+ (1.0f - fx) * (1.0f - fy) * fz * v001
		+ fx * (1.0f - fy) * fz * v101
		+ (1.0f - fx) * fy * fz * v011
		+ fx * fy * fz * v111;
}
__device__ __forceinline__ float t3_get_rounddown(const Table3& t, float x, float y, float z)
{
	const float xi = (x - t.xmin) * t.xstep;
	const float yi = (y - t.ymin) * t.ystep;
	const float zi = (z - t.zmin) * t.zstep;
	const int lx = clampi(floorr(xi), 0, t.nx - 1);
	const int ly = clampi(floorr(yi), 0, t.ny - 1);
	const int lz = clampi(floorr(zi), 0, t.nz - 1);
	return t.d[((size_t)lx * t.ny + ly) * t.nz + lz];
}

// -------------------------------------------------------------- material --
struct Material {
	float barrier, phonon_loss, recoil_const, fermi, band_gap;
	// mean-free-path scales of the derivative estimator (1 = the tables)
	float el_scale, in_scale;
	int inel_model;
	Table1 el_imfp, in_imfp;
	Table2 el_icdf, in_icdf, ki_ion;
	Table3 pn_q, pn_ion;
	// For the step kernels (StepMat): (elastic, inelastic) of each entry of the
	// two mean-free-path tables where they share their energies, or null; and
	// rows lx and lx + 1 of el_icdf side by side.
	const float2* imfp2;
	const float2* el_icdf2;
};

// What a step other than an inelastic event needs of a material.  The step
// kernels keep it in LDS: a step read some 17 of these constants from global
// memory, and a load takes the texture unit as long when all lanes want one
// word as when they want 64 (16 cycles and more; the units of the CUs were
// busy 78 % of the step kernel's time).  At 104 bytes each, 64 of them take
// 6.7 KB; drivers with more run the general variants, which read global memory.
struct StepMat {
	float barrier, phonon_loss, recoil_const, el_scale, in_scale;
	struct { float xmin, xstep, topx; } el, in;
	struct { float xmin, xstep, ymin, ystep, topx, topy; } cdf;
	int ny;
	const float2* imfp2;        // or null: the two tables below
	const float2* icdf2;
	const float* el_imfp;
	const float* in_imfp;
};
constexpr int STEP_MATS = 64;   // materials a step kernel keeps in LDS
__device__ __forceinline__ void load_step_mat(StepMat& d, const Material& m)
{
	d.barrier = m.barrier;
	d.phonon_loss = m.phonon_loss;
	d.recoil_const = m.recoil_const;
	d.el_scale = m.el_scale;
	d.in_scale = m.in_scale;
	d.el = { m.el_imfp.xmin, m.el_imfp.xstep, m.el_imfp.topx };
	d.in = { m.in_imfp.xmin, m.in_imfp.xstep, m.in_imfp.topx };
	d.cdf = { m.el_icdf.xmin, m.el_icdf.xstep, m.el_icdf.ymin, m.el_icdf.ystep, m.el_icdf.topx, m.el_icdf.topy };
	d.ny = m.el_icdf.ny;
	d.imfp2 = m.imfp2;
	d.icdf2 = m.el_icdf2;
	d.el_imfp = m.el_imfp.d;
	d.in_imfp = m.in_imfp.d;
}
using GFloat2 = const __attribute__((address_space(1))) float2;

// Both logarithms of the inverse mean free paths at log energy x (t1_get)
__device__ __forceinline__ void log_imfps(const Material& m, float x, float& el, float& in)
{
	el = t1_get(m.el_imfp, x);
	in = t1_get(m.in_imfp, x);
}
// `same`: all tables share their energies (a uniform branch)
__device__ __forceinline__ void log_imfps(const StepMat& m, float x, float& el, float& in, bool same = false)
{
	const float xe = (x - m.el.xmin) * m.el.xstep;
	const float le = t_index(xe, m.el.topx), fe = xe - le;
	float e0, e1, i0, i1, fi;
	if (same || m.imfp2) {
		const float4a8 v = *(const __attribute__((address_space(1))) float4a8*)((GFloat2*)m.imfp2 + (int)le);
		e0 = v.x; i0 = v.y; e1 = v.z; i1 = v.w;
		fi = fe;
	} else {
		const float xn = (x - m.in.xmin) * m.in.xstep;
		const float ln = t_index(xn, m.in.topx);
		GFloat* p = (GFloat*)m.el_imfp + (int)le;
		GFloat* q = (GFloat*)m.in_imfp + (int)ln;
		e0 = p[0]; e1 = p[1]; i0 = q[0]; i1 = q[1];
		fi = xn - ln;
	}
	el = (1.0f - fe) * e0 + fe * e1;
	in = (1.0f - fi) * i0 + fi * i1;
}

// The elastic event's cosine (t2_get)
__device__ __forceinline__ float el_cosine(const Material& m, float x, float y) { return t2_get(m.el_icdf, x, y); }
__device__ __forceinline__ float el_cosine(const StepMat& m, float x, float y)
{
	const float xi = (x - m.cdf.xmin) * m.cdf.xstep;
	const float yi = (y - m.cdf.ymin) * m.cdf.ystep;
	const float lx = t_index(xi, m.cdf.topx), ly = t_index(yi, m.cdf.topy);
	// v00, v10, v01, v11
	const float4a8 v = *(const __attribute__((address_space(1))) float4a8*)((GFloat2*)m.icdf2
		+ ((size_t)(uint32_t)(int)lx * (uint32_t)m.ny + (uint32_t)(int)ly));
	const float fx = xi - lx, fy = yi - ly;
	return (1.0f - fx) * (1.0f - fy) * v.x
		+ fx * (1.0f - fy) * v.y
		+ (1.0f - fx) * fy * v.z
		+ fx * fy * v.w;
}

// -------------------------------------------------------------- geometry --
// Triangle as three float4: (r0.xyz, e1.x), (e1.yz, e2.xy), (e2.z, mat_in,
// mat_out, 0) with the materials stored as int bits.  (A 64-byte record that
// also holds e1 x e2 measured slower: the extra load costs more than the
// cross product it saves.)
struct Tri { F3 r0, e1, e2; int mat_in, mat_out; };

__device__ __forceinline__ Tri load_tri(const float4* t, int i)
{
	const float4 a = t[3 * i], b = t[3 * i + 1], c = t[3 * i + 2];
	Tri r;
	r.r0 = { a.x, a.y, a.z };
	r.e1 = { a.w, b.x, b.y };
	r.e2 = { b.z, b.w, c.x };
	r.mat_in = __float_as_int(c.y);
	r.mat_out = __float_as_int(c.z);
	return r;
}

// 40 bytes in a row, loaded as 8 and twice 16: 6 553 600 primaries of 300 eV
// on a grating 184 ms, 192 with `tri` and `safety` in a table of their own.
struct alignas(8) ScreenRec {
	int32_t tri;
	float safety;           // 0.9999 / (1.0001 |n| + 1e-5 ee)
	float r0[3], ee;        // ee: |e1|_1 |e2|_1
	float n[3];             // e1 x e2 as the triangle test computes it
	uint32_t mats;          // material_in | material_out as two int16
};

struct Geometry {
	const int* od;
	const float4* tris;
	// Screening record per entry of the octree table, filled at every position
	// that names a triangle.  Stored in list order, so the screen reads
	// neighbouring records for neighbouring pairs, without waiting for the
	// triangle index.
	const ScreenRec* scr;
	// The octree's cells, inner ones and leaves, numbered from 1 with the
	// eight children of a cell in a row (0: the root).  Of an inner cell,
	// cells[2 i] is its centre, with the roundings of the reference's descent,
	// and in integer bits its first child; of a leaf, cells[2 i] are its lower
	// walls as a ray meets them (EPS outside, in the reference's roundings) and
	// the negative start of its list in `od`, cells[2 i + 1] its upper walls
	// and the list's length.
	const float4* cells;
	// next[8 i + 2 axis + (0 or 1)]: the cell that a ray leaving leaf i
	// through its upper (0) or lower (1) wall of that axis enters, or an inner
	// cell that holds it; 0: none, the ray leaves the octree
	const uint32_t* next;
	// The cells of one level of the tree by position: start[(z << 2 b) + (y <<
	// b) + x], b = start_bits, with x = (pos - lo) * inv rounded down; a leaf
	// above that level fills its part.  A position closer than start_eps (in
	// these cells' widths) to one of their walls starts at the root instead.
	const uint32_t* start;
	F3 lo, inv;             // lo: the domain's lower walls, centre - halfsize
	F3 hi;                  // its upper walls
	float start_eps, start_n;   // start_n: 2^b
	uint32_t start_bits;
	F3 center, halfsize;
	float max_extent;
	int ntri;
	// Bound on the rounding of one move inside the domain (a position
	// update's error, summed over components, plus the safety's own
	// subtraction): 3e-7 x the domain's largest 1-norm + 1e-6 nm.
	float step_eps;
	float wall_eps;         // wall_safety's margin
};

// core/triangle.inl:7-28
__device__ __forceinline__ float intersect_ray(const Tri& t, F3 start, F3 dir)
{
	const F3 pvec = cross(dir, t.e2);
	const float det = dot(t.e1, pvec);
	if (fabsf(det) < EPS)
		return -1.0f;
	// |det| >= EPS; a numerator below 2^-100 leaves every comparison as it is
	const float y = rcp_mid(det);
	const F3 s = v_sub(start, t.r0);
	const float u = div_by(dot(s, pvec), det, y);
	if ((u < -EPS) || (u > 1.0f + EPS))
		return -1.0f;
	const F3 qvec = cross(s, t.e1);
	const float v = div_by(dot(dir, qvec), det, y);
	if ((v < -EPS) || (u + v > 1.0f + EPS))
		return -1.0f;
	const float tt = div_by(dot(t.e2, qvec), det, y);
	if (tt < 0.0f)
		return -1.0f;
	return tt;
}

// geometry/octree.inl:24-30
__device__ __forceinline__ bool in_domain(const Geometry& g, F3 p)
{
	return (p.x > g.lo.x) && (p.x < g.hi.x)
		&& (p.y > g.lo.y) && (p.y < g.hi.y)
		&& (p.z > g.lo.z) && (p.z < g.hi.z);
}

// Levels of the octree at most (the builder's limit).
constexpr int MAX_DEPTH = 21;

// The pieces of the cell walk of geometry/octree.inl:32-192.
//
// The reference finds every cell by a descent from the root, adding up the
// centre on the way, and its neighbour by flipping bits of a location code.
// Both depend on the cell alone, so they are tables here: a cell's centre and
// scale as that descent rounds them, and the cell a location code with its
// bits flipped names.  A walk starts from the cell that one level's grid names
// for its position and goes down the few levels that are left (comparing with
// the centres as the reference does), and a move to the next cell reads one
// entry.  (With descents of seven levels from the root for every walk and
// the centre added up again for every further cell: 6 553 600 primaries of
// 300 eV on a grating 294 ms, with the tables 288; 160 000 of 1 keV on contact
// holes 21.5 and 21.0; 2046 of 300 eV 1.72 and 1.68.)
//
// cell_start: the cell in which a walk from `p` begins its descent.
__device__ __forceinline__ uint32_t cell_start(const Geometry& g, F3 p)
{
	const float tx = (p.x - g.lo.x) * g.inv.x, ty = (p.y - g.lo.y) * g.inv.y, tz = (p.z - g.lo.z) * g.inv.z;
	const float fx = __builtin_amdgcn_fractf(tx), fy = __builtin_amdgcn_fractf(ty), fz = __builtin_amdgcn_fractf(tz);
	// near a wall, where the rounding of t could name the other side, and
	// outside the domain (also for a NaN): from the root
	const bool sure = (int)(tx >= 0.0f) & (int)(ty >= 0.0f) & (int)(tz >= 0.0f) & (int)(fmaxf(fmaxf(tx, ty), tz) < g.start_n)
		& (int)(fminf(fminf(fx, fy), fz) >= g.start_eps) & (int)(fmaxf(fmaxf(fx, fy), fz) <= 1.0f - g.start_eps);
	if (!sure)
		return 0u;
	return g.start[((((uint32_t)tz << g.start_bits) | (uint32_t)ty) << g.start_bits) | (uint32_t)tx];
}

// cell_find: the leaf that holds `cur`, from `cell` downwards, with its walls;
// returns the start of its triangle list and its length in `count`.
__device__ __forceinline__ int cell_find(const Geometry& g, F3 cur, uint32_t& cell, F3& lo, F3& hi, int& count)
{
	for (;;) {
		const float4 a = g.cells[2 * (size_t)cell];
		const int child = __float_as_int(a.w);
		if (child < 0) {
			const float4 b = g.cells[2 * (size_t)cell + 1];
			lo = { a.x, a.y, a.z };
			hi = { b.x, b.y, b.z };
			count = __float_as_int(b.w);
			return -child;
		}
		cell = (uint32_t)child + ((cur.x > a.x) ? 1u : 0u) + ((cur.y > a.y) ? 2u : 0u) + ((cur.z > a.z) ? 4u : 0u);
	}
}

// Distance to the cell wall the ray leaves through (target -1/-2/-3 for the
// x/y/z wall).
__device__ __forceinline__ void cell_exit(F3 cur, F3 dir, F3 lo, F3 hi, float& isect, int& target)
{
	const float nx = ((__float_as_int(dir.x) < 0) ? lo.x : hi.x) - cur.x,
		ny = ((__float_as_int(dir.y) < 0) ? lo.y : hi.y) - cur.y,
		nz = ((__float_as_int(dir.z) < 0) ? lo.z : hi.z) - cur.z;
	float tx = div_mid(nx, dir.x), ty = div_mid(ny, dir.y), tz = div_mid(nz, dir.z);
	if (!(fminf(fminf(fabsf(dir.x), fabsf(dir.y)), fabsf(dir.z)) >= 0x1p-90f)) {
		tx = nx / dir.x;
		ty = ny / dir.y;
		tz = nz / dir.z;
	}
	if ((tx < ty) && (tx < tz)) { isect = tx; target = -1; }
	else if ((ty < tx) && (ty < tz)) { isect = ty; target = -2; }
	else { isect = tz; target = -3; }
}

// Candidate test: octree.inl:128-138 skips triangles whose outgoing material
// is the current one, then core/triangle.inl gives the distance (or -1).
// (A separate 16-byte record with e1 x e2 and the materials, read before the
// triangle, measured 9% slower: the extra dependent load costs more than the
// cross product it saves.  Estimating the three quotients with one
// reciprocal and dividing only where the outcome is not certain kept every
// result but measured 3% slower in the wave-wide walk.)
__device__ __forceinline__ float cell_candidate(const Geometry& g, int ti, F3 cur, F3 dir, int ignore_mat)
{
	const Tri tri = load_tri(g.tris, ti);
	const int mat_out = (dot(cross(tri.e1, tri.e2), dir) < 0.0f) ? tri.mat_in : tri.mat_out;
	if (mat_out == ignore_mat)
		return -1.0f;
	return intersect_ray(tri, cur, dir);
}

// First stage of the wave-wide walk's candidate test, on the 32-byte
// screening record of the list entry: the material test of cell_candidate (the same e1 x e2,
// computed on the host with the same operations, so the same result) and a
// plane test that drops
// a pair only when its intersection distance cannot matter.  For the pair's
// float inputs (s = cur - r0, dir, e1, e2), Moller-Trumbore's t is
// t* = -(s . n) / (dir . n) with n = e1 x e2 in exact arithmetic, and
// f(x) = s . n + x (dir . n) is the plane value at distance x along the ray.
// The pair is dropped when f has one sign, by more than
// tol = 1e-3 (|s| + L) |e1||e2|, at both x = -m and x = L with
// m = 1e-2 (1 + |s|) and L = 1.01 to_go + m: then t* < -m or t* > L.
// (Lengths here are 1-norms, which bound the 2-norms from above: every
// margin only grows.)
// Rounding moves f by at most about 1e-5 (|s| + L) |e1||e2| (a few unit
// roundoffs times the terms' magnitudes), far inside tol.  Pairs whose ray
// is within |dir . n| < 1e-2 |e1||e2| of the plane always pass: elsewhere
// the computed determinant and numerator of intersect_ray are within
// 1e-4 |t*| + 1e-4 |s| of their exact quotient, so a dropped pair has
// computed t < 0 (cannot hit) or t > to_go + EPS.  Such a far result cannot
// change the running-minimum fold: taking it needs isect >= t - EPS > to_go,
// and from there the owner ends without a hit whatever it takes next (a
// candidate below to_go is taken in both folds and makes them equal again).
// Pairs that pass are tested in full (intersect_ray) in the second stage.
__device__ __forceinline__ float dot_fma(F3 a, F3 b) { return __builtin_fmaf(a.z, b.z, __builtin_fmaf(a.y, b.y, a.x * b.x)); }
__device__ __forceinline__ float norm1(F3 a) { return fabsf(a.x) + fabsf(a.y) + fabsf(a.z); }
// What both bounds need of a pair: e1 x e2, the materials, |e1|_1 |e2|_1 and
// the safety's factor, |s|_1 and s . n.
struct Screen { F3 nrm; uint32_t mats; float ee, rden, slen, d0; };
__device__ __forceinline__ Screen load_screen(const Geometry& g, uint32_t entry, F3 cur, int& tri)
{
	static_assert(sizeof(ScreenRec) == 40, "loaded in three parts");
	using Part = const __attribute__((address_space(1))) float4a8;
	using Head = const __attribute__((address_space(1))) int2;
	const char* rec = (const char*)(g.scr + entry);
	const int2 h = { ((Head*)rec)->x, ((Head*)rec)->y };
	const float4a8 a = *(Part*)(rec + 8), b = *(Part*)(rec + 24);
	tri = h.x;
	const F3 nrm = { b.x, b.y, b.z };
	const F3 sv = { cur.x - a.x, cur.y - a.y, cur.z - a.z };
	return { nrm, __float_as_uint(b.w), a.w, __int_as_float(h.y), norm1(sv), dot_fma(sv, nrm) };
}
__device__ __forceinline__ bool cell_may_hit(const Screen& s, F3 dir, int ignore_mat, float to_go)
{
	const float dn = dot(s.nrm, dir);
	const int mat_out = (dn < 0.0f) ? (int)(int16_t)(s.mats & 0xffffu) : (int)(int16_t)(s.mats >> 16);
	const float m = __builtin_fmaf(1e-2f, s.slen, 1e-2f);
	const float L = __builtin_fmaf(1.01f, to_go, m);
	const float fa = __builtin_fmaf(-m, dn, s.d0), fb = __builtin_fmaf(L, dn, s.d0);
	const float tol = 1e-3f * (s.slen + L) * s.ee;
	// (f is between fa and fb along the segment.)  All of it without branches:
	// the lanes of a wave hardly ever agree.
	const bool far = fminf(fa, fb) > tol || fmaxf(fa, fb) < -tol;
	return mat_out != ignore_mat && !(far && fabsf(dn) >= 1e-2f * s.ee);
}

// Safety of a walk's start point: a radius S such that any later ray of
// length d starting within distance r of `cur`, with r + d <= S, finds no
// hit in the walk (the walk returns "no hit" and the full free path), so
// that such a step can skip the walk with the same result.
//
// Triangle part, for one triangle of the start cell from its screening
// record: with s = cur - r0, n the exact e1 x e2 and t the computed
// intersect_ray distance of a ray from p' = cur + D (|D| <= r) along any
// unit direction, intersect_ray's numerator and determinant are the exact
// s'.n and -dir.n up to rounding errors of at most 1e-6 |s'|_1 |e1|_1 |e2|_1
// and 1e-6 |e1|_1 |e2|_1 (a few unit roundoffs of each product, with
// |dir|_1 <= sqrt(3)), and the record's n is within 2e-7 |e1|_1 |e2|_1 of
// the exact one.  Hence |t| >= (|s.n| - r |n| - err) / (|n| + err'), and
// |t| >= d holds whenever a - 2e-6 |s|_1 ee >= S (|n|~ (1 + 2e-6) + 3e-6 ee)
// with a = |s.n| as computed here, ee = |e1|_1 |e2|_1 and |n|~ >= |n| the
// record's norm rounded up (the terms in r double the error allowance,
// r <= S).  A computed t >= d (= the remaining free path) is never taken as
// a hit: the walk keeps the nearest t <= (cell exit + EPS) and reports a hit
// only below the free path.  The bound below keeps a further 1e-4 relative
// slack for its own rounding; its factor is made at upload, in 64 bits.
// Fused multiply-adds: their roundings are a part of those allowed for, here
// and in cell_may_hit's plane test; the material test keeps dot()'s order.
// Triangles skipped by the material or last-triangle tests count too: the
// direction and the last triangle change between steps.
__device__ __forceinline__ float pair_safety(const Screen& s)
{
	return __builtin_fmaf(-2e-6f * s.slen, s.ee, fabsf(s.d0)) * s.rden;
}

// Wall part: distance from `cur` to the walls of its leaf cell, less a margin
// that covers the rounding of cell_exit's exit distances (a few unit roundoffs
// of the coordinates' magnitudes: 4e-6 of the domain's largest 1-norm, and 1e-3
// nm, which holds the EPS by which the walls are outside): a segment that ends
// at least that far inside the cell is seen to end before the cell's exit.
__device__ __forceinline__ float wall_safety(const Geometry& g, F3 cur, F3 lo, F3 hi)
{
	const float a = fminf(fminf(cur.x - lo.x, cur.y - lo.y), cur.z - lo.z);
	const float b = fminf(fminf(hi.x - cur.x, hi.y - cur.y), hi.z - cur.z);
	return fminf(a, b) - g.wall_eps;
}

// The cell across wall `target` (-1/-2/-3); 0 means the ray left the octree.
__device__ __forceinline__ uint32_t cell_next(const Geometry& g, uint32_t cell, int target, F3 dir)
{
	const float d = target == -1 ? dir.x : target == -2 ? dir.y : dir.z;
	const uint32_t axis = (uint32_t)~target;
	return g.next[8 * (size_t)cell + (2u * axis + (__float_as_uint(d) >> 31))];
}

// geometry/octree.inl:32-192: walk from leaf to leaf; returns the
// hit triangle (or -1) and the distance.  One lane, one ray.
__device__ inline int propagate(const Geometry& g, F3 start, F3 dir, float distance,
	int ignore_tri, int ignore_mat, float& out_dist)
{
	const int* __restrict__ od = g.od;
	F3 cur = start;
	float to_go = distance;
	uint32_t cell = cell_start(g, start);
	uint32_t cells = 0;
	do {
		F3 lo, hi;
		int count;
		int index = cell_find(g, cur, cell, lo, hi, count);
		++cells;
		float isect;
		int target;
		cell_exit(cur, dir, lo, hi, isect, target);
		for (;;) {
			const int ti = od[index++];
			if (ti < 0)
				break;
			if (ti == ignore_tri)
				continue;
			const float t = cell_candidate(g, ti, cur, dir, ignore_mat);
			if ((t > 0.0f) && (t <= isect + EPS)) {
				isect = t;
				target = ti;
			}
		}
		if (isect >= to_go) {
			out_dist = distance;
			return -1;
		} else if (target >= 0) {
			out_dist = distance - to_go + isect;
			return target;
		}
		to_go -= isect;
		cur = v_add(cur, v_mul(dir, isect));
		cell = cell_next(g, cell, target, dir);
	} while (cell != 0u && cells < MAX_CELLS);
	out_dist = distance;
	return -1;
}

// Lane `src`'s value of a pointer.
__device__ __forceinline__ const void* shfl_ptr(const void* p, int src)
{
	const uint64_t v = (uint64_t)p;
	const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)v, src);
	const uint32_t hi = (uint32_t)__shfl((int)(uint32_t)(v >> 32), src);
	return (const void*)(((uint64_t)hi << 32) | lo);
}

// Lane `at / 4`'s value of v (every lane of the wave active).
__device__ __forceinline__ int lane_int(int at, int v) { return __builtin_amdgcn_ds_bpermute(at, v); }
__device__ __forceinline__ float lane_float(int at, float v)
{
	return __int_as_float(__builtin_amdgcn_ds_bpermute(at, __float_as_int(v)));
}

// Sum of v over lanes 0..lane; every lane of the wave must be active.  By
// DPP in the VALU (within rows of 16, then row 0's and 2's sums to rows 1 and
// 3, then the first half's to the second): six dependent trips through LDS
// less a cell than with __shfl_up, and fewer registers (the step kernel 7 %
// faster: 6 553 600 primaries at 300 eV 367 -> 341 ms).
__device__ __forceinline__ int wave_incl_sum(int v)
{
	v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1
	v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
	v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
	v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
	v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15
	v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31
	return v;
}

// Owner of pair base + lane in a round of the wave-wide walk: the last lane
// whose pairs start at or before it (excl = first pair of this lane's list,
// n = its length).  Each lane whose pairs start inside the chunk marks that
// position in `owner_at` (64 ints of LDS); position 0 holds the owner carried
// in from earlier (the last lane with excl <= base).  A running maximum by
// DPP (as in wave_incl_sum) carries each mark on to the next one.
__device__ __forceinline__ int chunk_owner(int base, int excl, int n, int* owner_at, int lane)
{
	const uint64_t before = ballot(excl <= base);
	const int o0 = 63 - (int)__builtin_clzll(before);
	owner_at[lane] = 0;
	__builtin_amdgcn_wave_barrier();
	const int e = excl - base;
	if (n > 0 && e > 0 && e < 64)
		owner_at[e] = lane + 1;
	__builtin_amdgcn_wave_barrier();
	int v = (lane == 0) ? o0 + 1 : owner_at[lane];
	v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));
	v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
	v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
	v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
	v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));
	v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));
	return v - 1;
}

// A ray on its way through the octree: where it has got to, what is left of
// its free path, its cell (or an inner one that holds it) and the cells it
// has been in.
struct Walk {
	F3 cur;
	float to_go;
	uint32_t cell;
	uint32_t cells;
};
__device__ __forceinline__ void walk_start(const Geometry& g, Walk& w, F3 start, float distance)
{
	w.cur = start;
	w.to_go = distance;
	w.cell = cell_start(g, start);
	w.cells = 0;
}
enum { WALK_ON = 0, WALK_END, WALK_HIT };

// A wave's particles and walks, a lane each, in LDS: a walk's candidate tests
// read other lanes' rays (three wide reads of LDS a pair, where fetching ten
// values across lanes takes ten narrow ones), and what a phase of a step does
// not need leaves its registers to the phase.
//
// This alone, with 6 waves per SIMD instead of 5 and 8 % fewer VALU
// instructions, changed nothing (254 -> 257 ms for 6 553 600 primaries of
// 300 eV): the step kernel then waited for its loads.  With the materials in
// LDS as well (StepMat), 35 % fewer loads: 244.
struct WaveMem {
	float4 cur[64];       // walk: position, what is left of the free path
	float4 dir[64];       // direction (normalised once the step is planned), material
	float4 pos[64];       // position, energy
	float4 evt[64];       // free path, log of the energy, the event's draws
	int2 last[64];        // last triangle; walk: first entry of the list less the lane's first pair
	uint64_t sid[64];
	uint32_t step[64];
	uint32_t cell[64];    // walk: its cell
	int owner[64];        // owner table
	int q_ti[64];         // queue of pairs: triangle, owner lane
	unsigned saf[64];     // safeties
	uint8_t q_own[64];
};
__device__ __forceinline__ F3 xyz(const float4& v) { return { v.x, v.y, v.z }; }
// Reads of LDS are not carried over this point in registers.
__device__ __forceinline__ void lds_again() { asm volatile("" ::: "memory"); }

// One cell of the same walk for the rays of a whole wave, with the candidate
// tests shared out over all 64 lanes.
//
// One lane walking its own cell's triangle list leaves most of the wave idle:
// lists differ in length, and the wave runs as long as the longest.  Here
// every walking lane enters its next cell and gets its list's length
// (cell_find); the (ray, candidate) pairs of all lists are numbered by a prefix
// sum over lanes and screened 64 at a time, one per lane, with the owning
// ray's origin and direction read from LDS (cell_may_hit: material
// test and a conservative plane test; about 9 % of the pairs pass on a
// grating scan).  The pairs that pass are queued in LDS in pair order and
// tested in full 64 at a time.  The results that can hit (t > 0) are then
// taken in queue order, which is each owner's list order, and each owner
// applies the reference's running-minimum rule to its own, so hit, distance
// and tie choices are those of `propagate`.  (Testing every pair in full
// took about 20 % more of the step kernel.)
//
// Every lane of the wave must call it (lanes with active == false take part
// in the shared tests only).  The rays are m.cur, m.dir, m.last and m.cell.
// Returns WALK_HIT (triangle `target` at distance m.cur.w - isect before the
// end of the free path), WALK_END (no hit) or WALK_ON (moved to the next
// cell).
//
// SAF: `safety` receives, from a walk's start cell, the safety of its start
// point: wall_safety of the cell, and pair_safety of every triangle listed
// there, minimised per owner (in other cells a value without meaning).
template <bool SAF>
__device__ __forceinline__ int walk_round(const Geometry& g, bool active, WaveMem& m, uint32_t& cells,
	float& safety, float& isect, int& target)
{
	const int lane = (int)__lane_id();
	int n = 0, off = 0;
	target = 0;
	isect = 0.0f;
	if (active) {
		F3 lo, hi;
		const F3 cur = xyz(m.cur[lane]), dir = xyz(m.dir[lane]);
		uint32_t cell = m.cell[lane];
		off = cell_find(g, cur, cell, lo, hi, n);
		m.cell[lane] = cell;
		++cells;
		cell_exit(cur, dir, lo, hi, isect, target);
		if (SAF)
			m.saf[lane] = __float_as_uint(fmaxf(wall_safety(g, cur, lo, hi), 0.0f));
	}
	const int incl = wave_incl_sum(n);
	const int excl = incl - n;
	m.last[lane].y = off - excl;  // pair p of this lane tests od[off - excl + p]
	const int total = __builtin_amdgcn_readlane(incl, 63);
	int qn = 0;   // queued pairs (wave-uniform)
	// Second stage: test the queued pairs in full and fold the results
	// that can hit, in queue order, into their owners' running minimum.
	auto flush = [&]() {
		__builtin_amdgcn_wave_barrier();
		int ti = -1, own = 0;
		float t = -1.0f;
		if (lane < qn) {
			ti = m.q_ti[lane];
			own = m.q_own[lane];
			t = intersect_ray(load_tri(g.tris, ti), xyz(m.cur[own]), xyz(m.dir[own]));
		}
		__builtin_amdgcn_wave_barrier();
		uint64_t hits = ballot(t > 0.0f);
		while (hits) {
			const int src = (int)__builtin_ctzll(hits);
			hits &= hits - 1ull;
			const float ts = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t), src));
			const int tis = __builtin_amdgcn_readlane(ti, src), os = __builtin_amdgcn_readlane(own, src);
			if (lane == os && ts <= isect + EPS) {
				isect = ts;
				target = tis;
			}
		}
	};
	for (int base = 0; base < total; base += 64) {
		lds_again();
		const int o = chunk_owner(base, excl, n, m.owner, lane);
		// (the lanes behind the last pair repeat it)
		const bool valid = base + lane < total;
		const float4 oc = m.cur[o], od = m.dir[o];
		const int2 ol = m.last[o];
		const uint32_t entry = (uint32_t)(ol.y + min(base + lane, total - 1));
		int ti;
		const Screen sc = load_screen(g, entry, xyz(oc), ti);
		const bool pass = valid && ti != ol.x && cell_may_hit(sc, xyz(od), __float_as_int(od.w), oc.w);
		if (SAF && valid)
			atomicMin(&m.saf[o], __float_as_uint(fmaxf(pair_safety(sc), 0.0f)));
		const uint64_t pm = ballot(pass);
		const int np = (int)__popcll(pm);
		if (qn + np > 64) {
			flush();
			qn = 0;
		}
		if (pass) {
			const int slot = qn + (int)__popcll(pm & ((1ull << lane) - 1ull));
			m.q_ti[slot] = ti;
			m.q_own[slot] = (uint8_t)o;
		}
		qn += np;
	}
	if (qn > 0)
		flush();
	lds_again();
	if (SAF)
		safety = __uint_as_float(m.saf[lane]);
	if (!active)
		return WALK_ON;
	const float4 c = m.cur[lane];
	if (isect >= c.w)
		return WALK_END;
	if (target >= 0)
		return WALK_HIT;
	const F3 dir = xyz(m.dir[lane]);
	const F3 cur = v_add(xyz(c), v_mul(dir, isect));
	m.cur[lane] = { cur.x, cur.y, cur.z, c.w - isect };
	const uint32_t next = cell_next(g, m.cell[lane], target, dir);
	m.cell[lane] = next;
	return (next != 0u && cells < MAX_CELLS) ? WALK_ON : WALK_END;
}

// The whole walk for the rays of a wave (every lane calls; lanes with walk ==
// false take part in the shared tests only).  The query hook's: the step
// kernels call walk_round themselves.
__device__ inline int propagate_wave(const Geometry& g, bool walk, F3 start, F3 dir, float distance,
	int ignore_tri, int ignore_mat, float& out_dist, WaveMem& m)
{
	const uint32_t lane = __lane_id();
	uint32_t cells = 0;
	m.cur[lane] = { start.x, start.y, start.z, distance };
	m.dir[lane] = { dir.x, dir.y, dir.z, __int_as_float(ignore_mat) };
	m.last[lane].x = ignore_tri;
	if (walk)
		m.cell[lane] = cell_start(g, start);
	out_dist = distance;
	int result = -1;
	while (ballot(walk) != 0ull) {
		float isect, safety;
		int target;
		const int r = walk_round<false>(g, walk, m, cells, safety, isect, target);
		if (walk && r != WALK_ON) {
			walk = false;
			if (r == WALK_HIT) {
				result = target;
				out_dist = distance - m.cur[lane].w + isect;
			}
		}
	}
	return result;
}

// The walk for lanes of different geometries (the multi-world kernels, 4
// waves per SIMD): the candidate tests read the owning lane's triangle
// tables, and every pair is tested in full; the screen's queue and second
// load measured slower there.
__device__ inline int propagate_wave_multi(const Geometry& g, bool walk, F3 start, F3 dir, float distance,
	int ignore_tri, int ignore_mat, float& out_dist, int* owner_at)
{
	out_dist = distance;
	const int lane = (int)__lane_id();
	Walk w = {};
	if (walk)
		walk_start(g, w, start, distance);
	int result = -1;
	bool active = walk;
	while (ballot(active) != 0ull) {
		int n = 0, off = 0, target = 0;
		float isect = 0.0f;
		if (active) {
			F3 lo, hi;
			off = cell_find(g, w.cur, w.cell, lo, hi, n);
			++w.cells;
			cell_exit(w.cur, dir, lo, hi, isect, target);
		}
		const int incl = wave_incl_sum(n);
		const int excl = incl - n;
		off -= excl;  // pair p of this lane tests od[off + p]
		const int total = __builtin_amdgcn_readlane(incl, 63);
		for (int base = 0; base < total; base += 64) {
			const int p = base + lane;
			const int o = chunk_owner(base, excl, n, owner_at, lane);
			const F3 oc = { __shfl(w.cur.x, o), __shfl(w.cur.y, o), __shfl(w.cur.z, o) };
			const F3 odir = { __shfl(dir.x, o), __shfl(dir.y, o), __shfl(dir.z, o) };
			const int oign_tri = __shfl(ignore_tri, o), oign_mat = __shfl(ignore_mat, o);
			const int ooff = __shfl(off, o);
			Geometry og = g;
			og.od = (const int*)shfl_ptr(g.od, o);
			og.tris = (const float4*)shfl_ptr(g.tris, o);
			float t = -1.0f;
			int ti = -1;
			if (p < total) {
				ti = og.od[ooff + p];
				if (ti != oign_tri)
					t = cell_candidate(og, ti, oc, odir, oign_mat);
			}
			// this lane's pairs within the chunk, lanes [lo, hi)
			uint64_t todo = 0;
			const uint64_t can_hit = ballot(t > 0.0f);
			if (active) {
				const int lo = max(excl - base, 0), hi = min(incl - base, 64);
				if (lo < hi) {
					const uint64_t upto = (hi == 64) ? ~0ull : ((1ull << hi) - 1ull);
					todo = can_hit & upto & ~((1ull << lo) - 1ull);
				}
			}
			while (ballot(todo != 0ull) != 0ull) {
				const int src = todo ? (int)__builtin_ctzll(todo) : lane;
				const float ts = __shfl(t, src);
				const int tis = __shfl(ti, src);
				if (todo) {
					if (ts <= isect + EPS) {
						isect = ts;
						target = tis;
					}
					todo &= todo - 1ull;
				}
			}
		}
		if (active) {
			if (isect >= w.to_go) {
				active = false;
			} else if (target >= 0) {
				out_dist = distance - w.to_go + isect;
				result = target;
				active = false;
			} else {
				w.to_go -= isect;
				w.cur = v_add(w.cur, v_mul(dir, isect));
				w.cell = cell_next(g, w.cell, target, dir);
				if (!(w.cell != 0u && w.cells < MAX_CELLS))
					active = false;
			}
		}
	}
	return result;
}

// -------------------------------------------------------------- physics --
struct Particle { F3 pos, dir; float E; };

// physics/full_penn.h:50-57 (same body in elastic.h:54-62); the mean free
// path is multiplied by the mechanism's scale (exact when it is 1).  logE is
// m_log(E), computed once per step for both mechanisms.
template <class R>
__device__ __forceinline__ float mech_sample_path(float log_imfp, float scale, R& rng, float& tau)
{
	const float imfp = m_exp(log_imfp);
	tau = (is_mid(imfp) ? rcp_mid(imfp) : 1.0f / imfp) * scale;
	return -tau * pf_log_normal(rng_unit(rng));
}

// What the derivative estimator needs from a step's free-path race: the
// scaled mean free paths, the winning mechanism (0 none, 1 inelastic,
// 2 elastic) and the distance travelled; also log(E) of the step, which
// the elastic event uses again (E does not change in between).
struct PathInfo { float tau_el, tau_in, dist; int type; float logE; };

// physics/kieft/elastic.h:67-115; logE = m_log(p.E)
template <class M, class R>
__device__ __forceinline__ void elastic_execute(const M& m, uint32_t fl, Particle& p, R& rng, float logE)
{
	Particle tp = p;
	float cos_theta, sin_theta;
	{
		const float x = logE;
		const float y = rng_unit(rng);
		cos_theta = clampr(el_cosine(m, x, y), -1.0f, 1.0f);
		sin_theta = sqrt_mid(1.0f - cos_theta * cos_theta);   // 0 or at least 2^-24
	}
	// the direction is the step's normalised one
	tp.dir = normalised_unit(tp.dir);
	const F3 normal_dir = normalised_unit(make_normal_vec(tp.dir, rng_phi(rng)));
	tp.dir = v_add(v_mul(tp.dir, cos_theta), v_mul(normal_dir, sin_theta));
	if (tp.E < 200.0f) {
		if (fl & PH_EL_PHONON)
			tp.E = tp.E - fmin_std(50e-3f, m.phonon_loss);
	} else {
		if (fl & PH_EL_RECOIL)
			tp.E = tp.E - m.recoil_const * (1.0f - cos_theta) * tp.E;
	}
	p = tp;
}

// physics/full_penn.h:62-288
__device__ inline bool penn_execute(const Material& m, uint32_t fl, Particle& p, Rng& rng, Particle& se)
{
	Particle tp = p;
	float omega;
	{
		const float x = m_log(tp.E);
		const float y = rng_unit(rng);
		omega = m_exp(t2_get(m.in_icdf, x, y));
	}
	float binding;
	{
		const float x = m_log(tp.E);
		const float y = m_log(omega / tp.E);
		const float z = rng_unit(rng);
		binding = t3_get_rounddown(m.pn_ion, x, y, z);
	}
	tp.dir = normalised(tp.dir);

	if (binding <= 0.0f) {
		if (omega > m.band_gap) {
			float q;
			{
				const float x = m_log(tp.E);
				const float y = omega / tp.E;
				const float z = rng_unit(rng);
				q = t3_get(m.pn_q, x, y, z);
			}
			const F3 prim_normal_dir = normalised(make_normal_vec(tp.dir, rng_phi(rng)));
			F3 q_dir, q_normal_dir;
			{
				const float c = clampr((omega + q * q) / (2.0f * sqrtf(tp.E) * q), -1.0f, 1.0f);
				const float s = sqrtf(1.0f - c * c);
				q_dir = normalised(v_add(v_mul(tp.dir, c), v_mul(prim_normal_dir, s)));
				q_normal_dir = normalised(make_normal_vec(q_dir, rng_phi(rng)));
			}
			const float cpf = clampr((2.0f * tp.E - omega - q * q) / (2.0f * sqrtf(tp.E * (tp.E - omega))), -1.0f, 1.0f);
			const float spf = sqrtf(1.0f - cpf * cpf);
			tp.E = tp.E - omega;
			tp.dir = v_add(v_mul(tp.dir, cpf), v_mul(prim_normal_dir, spf));
			p = tp;
			if (!(fl & PH_PN_SE))
				return false;
			Particle sp;
			sp.pos = tp.pos;
			const float k_fermi = sqrtf(m.fermi);
			const float k_fermi_omega = sqrtf(m.fermi + omega);
			if (q < k_fermi_omega - k_fermi) {
				// plasmon decay (:141-194)
				const float f = m.fermi / omega;
				float x;
				if (f < 0.1f) {
					const float U = m_cbrt(rng_unit(rng));
					x = f * U * U;
				} else {
					const float lower = fmax_std(0.0f, f - 1.0f);
					const float upper = f;
					const float d1 = upper - lower;
					const float d2 = upper * upper - lower * lower;
					const float alpha = d2 / (d1 + d2);
					int rounds = 0;
					do {
						const float U1 = rng_unit(rng);
						const float U2 = rng_unit(rng);
						x = (U1 < alpha) ? sqrtf(d2 * U2 + lower * lower) : d1 * U2 + lower;
					} while (rng_unit(rng) > sqrtf(x * x + x) / (x + 0.5f) && ++rounds < MAX_REJECT);
				}
				sp.E = x * omega + omega;
				sp.dir = rng_uniform_vector(rng);
			} else if (q < k_fermi_omega + k_fermi) {
				// single excitation (:195-222)
				const float ki_parr = (omega - q * q) / (2.0f * q);
				const float kf_parr = ki_parr + q;
				const float ki_perp_min_sq = fmax_std(0.0f, m.fermi - kf_parr * kf_parr);
				const float ki_perp_max_sq = m.fermi - ki_parr * ki_parr;
				const float ki_perp_sq = fmax_std(0.0f,
					ki_perp_min_sq + (ki_perp_max_sq - ki_perp_min_sq) * rng_unit(rng));
				const F3 ki = v_add(s_mul(ki_parr, q_dir), s_mul(sqrtf(ki_perp_sq), q_normal_dir));
				sp.E = mag2(ki) + omega;
				sp.dir = v_add(ki, s_mul(q, q_dir));
			} else {
				return false;
			}
			se = sp;
			return true;
		}
		tp.E = tp.E - omega;   // sub-band-gap loss (:234-242)
		p = tp;
		return false;
	}

	// inner-shell excitation (:245-287)
	const F3 normal_dir = normalised(make_normal_vec(tp.dir, rng_phi(rng)));
	const float K = tp.E - m.fermi + 2.0f * binding;
	const float dK = binding + omega;
	const float cos_theta = sqrtf(dK / K);
	const float sin_theta = sqrtf(1.0f - saturater(cos_theta * cos_theta));
	F3 sdir = v_add(v_mul(tp.dir, cos_theta), v_mul(normal_dir, sin_theta));
	sdir = normalised(sdir);
	sdir = v_add(sdir, s_mul(sqrtf(binding / dK), rng_uniform_vector(rng)));
	sdir = normalised(sdir);
	bool made = false;
	if (fl & PH_PN_SE) {
		se.E = m.fermi + omega - binding;
		se.pos = tp.pos;
		se.dir = sdir;
		made = true;
	}
	tp.E = tp.E - omega;
	tp.dir = v_sub(tp.dir, s_mul(cos_theta, sdir));
	p = tp;
	return made;
}

// physics/kieft/inelastic.h:68-206
__device__ inline bool kieft_execute(const Material& m, uint32_t fl, Particle& p, Rng& rng, Particle& se)
{
	Particle tp = p;
	float omega0;
	{
		const float x = m_log(tp.E);
		const float y = rng_unit(rng);
		omega0 = m_exp(t2_get(m.in_icdf, x, y));
	}
	float binding;
	{
		const float x = m_log(omega0);
		const float y = rng_unit(rng);
		binding = t2_get_rounddown(m.ki_ion, x, y);
	}
	float omega;
	{
		const float omega_max = 0.5f * (tp.E + omega0 - m.fermi);
		float omega_min = omega0;
		float w0 = fmin_std(omega0 - 1.0f, fmax_std(0.0f, binding) - m.fermi);
		if (tp.E > 2.0f * omega0) {
			omega_min = 0.5f * (tp.E + omega0 - sqrtf(tp.E * (tp.E - 2.0f * omega0)));
			w0 = omega0;
		}
		const float U = rng_unit(rng);
		if ((w0 > 0.0f) && (omega_min > w0) && (omega_min < omega_max)) {
			const float f_min = 1.0f / w0 * m_log((omega_min - w0) / omega_min);
			const float f_max = 1.0f / w0 * m_log((omega_max - w0) / omega_max);
			omega = -w0 / m_expm1(w0 * (f_min * (1.0f - U) + f_max * U));
		} else {
			omega = omega0 * omega_max / (omega0 * (1.0f - U) + omega_max * U);
		}
	}
	if (binding < 0.0f) {
		if (m.band_gap < 0.0f) {
			// metals: no special case in the reference
		} else if (omega0 > m.band_gap) {
			binding = m.band_gap;
		} else {
			if (fl & PH_KI_OPTICAL) {
				tp.E = tp.E - omega0;
				p = tp;
			}
			return false;
		}
	}
	binding = fmax_std(0.0f, binding);
	tp.dir = normalised(tp.dir);
	const F3 normal_dir = normalised(make_normal_vec(tp.dir, rng_phi(rng)));
	const float K = tp.E - m.fermi + 2.0f * binding;
	const float dK = binding + omega;
	const float cos_theta = sqrtf(dK / K);
	const float sin_theta = sqrtf(1.0f - saturater(cos_theta * cos_theta));
	F3 sdir = v_add(v_mul(tp.dir, cos_theta), v_mul(normal_dir, sin_theta));
	if (fl & PH_KI_INST) {
		sdir = normalised(sdir);
		sdir = v_add(sdir, s_mul(sqrtf(binding / dK), rng_uniform_vector(rng)));
	}
	sdir = normalised(sdir);
	bool made = false;
	if (fl & PH_KI_SE) {
		se.E = m.fermi + omega - binding;
		se.pos = tp.pos;
		se.dir = sdir;
		made = true;
	}
	tp.E = tp.E - omega;
	if (fl & PH_KI_MOMCONS)
		tp.dir = v_sub(tp.dir, s_mul(cos_theta, sdir));
	p = tp;
	return made;
}

// physics/boundary_intersect.h:38-155
//
// With `g` given, it receives d log p / d dU of the random choices made
// (transmission, reflection, absorption; 0 if none), and mi / mo the
// materials with dU = b(mo) - b(mi).
template <class M, class R>
__device__ __forceinline__ int boundary_execute(const M* mats, uint32_t fl, const Tri& tri,
	Particle& p, int& mat, R& rng, float* g = nullptr, int* g_mi = nullptr, int* g_mo = nullptr)
{
	if (g) *g = 0.0f;
	Particle tp = p;
	const F3 nd = normalised_unit(tp.dir);   // the step's normalised direction
	const F3 n = normalised(cross(tri.e1, tri.e2));
	const float cos_theta = dot(n, nd);
	int mi, mo;
	if (cos_theta > 0.0f) { mi = tri.mat_in; mo = tri.mat_out; }
	else { mi = tri.mat_out; mo = tri.mat_in; }
	switch (mo) {
	case MAT_DETECTOR:
		return DETECTED;
	case MAT_DETECTOR_LT50:
		return (tp.E < 50.0f) ? DETECTED : ALIVE;
	case MAT_DETECTOR_GE50:
		return (tp.E >= 50.0f) ? DETECTED : ALIVE;
	case MAT_TERMINATOR:
		return TERMINATED;
	case MAT_MIRROR:
		tp.dir = v_sub(nd, v_mul(s_mul(2.0f, n), cos_theta));
		p = tp;
		return ALIVE;
	case MAT_NOP:
		return ALIVE;
	default:
		break;
	}
	float dU = 0.0f;
	if (mi >= 0) dU = dU - mats[mi].barrier;
	if (mo >= 0) dU = dU + mats[mo].barrier;
	if (g) { *g_mi = mi; *g_mo = mo; }
	if (tp.E * cos_theta * cos_theta + dU > 0.0f) {
		const float ec2 = tp.E * cos_theta * cos_theta;
		const float s = sqrtf(1.0f + dU / ec2);
		const float T = (fl & PH_BI_QUANTUM) ? 4.0f * s / ((1.0f + s) * (1.0f + s)) : 1.0f;
		if (rng_unit(rng) < T) {
			// d log T / d dU
			if (g && (fl & PH_BI_QUANTUM) && T < 1.0f)
				*g = (1.0f - s) / (2.0f * s * s * (1.0f + s) * ec2);
			if (fl & PH_BI_REFRACT)
				tp.dir = v_add(v_sub(nd, v_mul(n, cos_theta)), v_mul(s_mul(s, n), cos_theta));
			tp.E = tp.E + dU;
			mat = mo;
			p = tp;
			return ALIVE;
		}
		// d log (1 - T) / d dU
		if (g && (fl & PH_BI_QUANTUM) && T < 1.0f)
			*g = 2.0f / (s * dU);
	}
	if (fl & PH_BI_ABSORB) {
		if (dU < 0.0f) {
			const float P = m_exp(1.0f + 0.5f * tp.E / dU);
			const bool absorbed = rng_unit(rng) < P;
			if (g && P < 1.0f)
				*g = *g + (absorbed ? -0.5f * tp.E / (dU * dU) : P * 0.5f * tp.E / (dU * dU * (1.0f - P)));
			if (absorbed)
				return TERMINATED;
		}
	}
	tp.dir = v_sub(nd, v_mul(s_mul(2.0f, n), cos_theta));
	p = tp;
	return ALIVE;
}

// --------------------------------------------------------------- a step --
struct State {
	Particle p;
	int mat, last_tri;
	uint32_t tag, step, flags;
	uint64_t sid;
	// Safety left of the particle's last walk: no triangle of that walk's
	// start cell and no wall of that cell lies within this distance of the
	// particle (the step kernel's walk skip); < 0 when unknown.
	float safe;
};

struct World {
	Geometry g;
	const Material* mats;
	int nmats;
	uint32_t flags;
	float threshold;
	uint32_t key0, key1;
};

// Geometry and materials of one world of a multi-scan driver.
struct WorldDesc {
	Geometry g;
	const Material* mats;
	int nmats;
};

// init (drivers/gpu/gpu_driver.inl:403-480) in two halves around the walk.
//
// step_plan: domain and energy checks and path sampling.  Returns ALIVE or
// TERMINATED; for ALIVE, `distance` and `type` are the free path and its
// mechanism (0 in vacuum), `nd` the normalised direction (the direction
// itself when the step was `planned` before, FL_PLANNED).
template <class M, class R>
__device__ __forceinline__ int step_plan(const World& W, const M* mats, const State& s, R& rng, F3& nd, float& distance,
	int& type, PathInfo& pinfo, bool planned = false)
{
	pinfo.type = 0;
	pinfo.logE = 0.0f;
	type = 0;
	if (!in_domain(W.g, s.p.pos))
		return TERMINATED;
	distance = W.g.max_extent;
	float tau_el = 0.0f, tau_in = 0.0f;
	if (s.mat >= 0) {
		const M& m = mats[s.mat];
		if (s.p.E < m.barrier + W.threshold)
			return TERMINATED;
		// core/scatter_list.h:101-107 with the reverse visiting order of
		// common/tuple.h:114-124: elastic first, strictly shorter wins.
		float dist = __builtin_inff();
		const float logE = m_log(s.p.E);
		pinfo.logE = logE;
		float log_el, log_in;
		log_imfps(m, logE, log_el, log_in);
		const float pe = mech_sample_path(log_el, m.el_scale, rng, tau_el);
		if (pe < dist) { type = 2; dist = pe; }
		const float pi = mech_sample_path(log_in, m.in_scale, rng, tau_in);
		if (pi < dist) { type = 1; dist = pi; }
		distance = dist;
	}
	nd = planned ? s.p.dir : normalised(s.p.dir);
	pinfo.tau_el = tau_el;
	pinfo.tau_in = tau_in;
	return ALIVE;
}

// The same without its special cases one by one: the short forms in a row and
// one check that their operands were in range (else step_plan).
template <class R>
__device__ __forceinline__ int step_plan_short(const World& W, const StepMat* mats, bool same, const State& s, R& rng,
	F3& nd, float& distance, int& type, PathInfo& pinfo, bool planned)
{
	pinfo.type = 0;
	pinfo.logE = 0.0f;
	pinfo.tau_el = pinfo.tau_in = 0.0f;
	type = 0;
	if (!in_domain(W.g, s.p.pos))
		return TERMINATED;
	distance = W.g.max_extent;
	const R rng0 = rng;
	const float m2 = s.p.dir.x * s.p.dir.x + s.p.dir.y * s.p.dir.y + s.p.dir.z * s.p.dir.z;
	nd = planned ? s.p.dir : v_mul(s.p.dir, rcp_mid(sqrt_mid(m2)));
	bool ok = planned || is_mid(m2);
	if (s.mat >= 0) {
		const StepMat& m = mats[s.mat];
		if (s.p.E < m.barrier + W.threshold)
			return TERMINATED;
		const float logE = pf_log_normal(s.p.E);
		pinfo.logE = logE;
		float log_el, log_in;
		log_imfps(m, logE, log_el, log_in, same);
		pinfo.tau_el = rcp_mid(pf_exp_short(log_el)) * m.el_scale;
		pinfo.tau_in = rcp_mid(pf_exp_short(log_in)) * m.in_scale;
		const float pe = -pinfo.tau_el * pf_log_normal(rng_unit(rng));
		const float pi = -pinfo.tau_in * pf_log_normal(rng_unit(rng));
		// normal energy, exponentials in [2^-100, 2^100] (or NaN)
		ok = ok && __float_as_uint(s.p.E) - 0x00800000u < 0x7f000000u && fmaxf(fabsf(log_el), fabsf(log_in)) <= 69.0f;
		// (as in step_plan: elastic first, strictly shorter wins)
		float dist = __builtin_inff();
		if (pe < dist) { type = 2; dist = pe; }
		if (pi < dist) { type = 1; dist = pi; }
		distance = dist;
	}
	if (!ok) {
		rng = rng0;
		return step_plan(W, mats, s, rng, nd, distance, type, pinfo, planned);
	}
	return ALIVE;
}

// step_move: after the walk, move to the hit or to the end of the free path
// and name the event; stores the normalised direction.
__device__ __forceinline__ void step_move(State& s, F3 nd, float distance, int type, int hit, float hd,
	int& event, PathInfo& pinfo)
{
	s.p.dir = nd;
	if (hit < 0) {
		s.p.pos = v_add(s.p.pos, v_mul(nd, distance));
		event = type;
	} else {
		s.p.pos = v_add(s.p.pos, v_mul(nd, hd));
		s.last_tri = hit;
		event = EV_INTERSECT;
	}
	pinfo.dist = (hit < 0) ? distance : hd;
	pinfo.type = (s.mat >= 0) ? type : 0;
}

// The whole init for one lane: domain and energy checks, path sampling,
// propagate, move.  Returns ALIVE or TERMINATED and the event; `hit` is the
// intersected triangle.
__device__ inline int step_init(const World& W, State& s, Rng& rng, int& event, int& hit, PathInfo& pinfo)
{
	event = EV_NONE;
	hit = -1;
	F3 nd;
	float distance;
	int type;
	if (step_plan(W, W.mats, s, rng, nd, distance, type, pinfo) != ALIVE)
		return TERMINATED;
	float hd;
	hit = propagate(W.g, s.p.pos, nd, distance, s.last_tri, s.mat, hd);
	step_move(s, nd, distance, type, hit, hd, event, pinfo);
	return ALIVE;
}

// The event chosen by init (gpu_driver.inl:482-566).  For inelastic events
// the new parent state and secondary are computed into `s`/`se`; the caller
// commits them.
__device__ inline int step_event(const World& W, State& s, Rng& rng, int event, int hit,
	Particle& se, bool& se_made, float* g = nullptr, int* g_mi = nullptr, int* g_mo = nullptr)
{
	se_made = false;
	if (event == EV_INTERSECT) {
		const Tri tri = load_tri(W.g.tris, hit);
		return boundary_execute(W.mats, W.flags, tri, s.p, s.mat, rng, g, g_mi, g_mo);
	}
	if (event == EV_NONE)
		return ALIVE;
	s.last_tri = -1;
	const Material& m = W.mats[s.mat];
	if (event == EV_ELASTIC) {
		elastic_execute(m, W.flags, s.p, rng, m_log(s.p.E));
		return ALIVE;
	}
	se_made = (m.inel_model == 0) ? penn_execute(m, W.flags, s.p, rng, se)
		: kieft_execute(m, W.flags, s.p, rng, se);
	return ALIVE;
}

// The events of a step other than inelastic scattering: boundary crossing
// and elastic scattering (and nothing for EV_NONE).  The tracking kernel
// sends inelastic events to their own kernel, so its code holds neither the
// inelastic models nor their register pressure.  logE is m_log(s.p.E)
// from the step's path sampling.
template <class M, class R>
__device__ __forceinline__ int step_event_elastic_or_boundary(const World& W, const M* mats, State& s, R& rng, int event,
	int hit, float logE, float* g = nullptr, int* g_mi = nullptr, int* g_mo = nullptr)
{
	if (event == EV_INTERSECT) {
		const Tri tri = load_tri(W.g.tris, hit);
		return boundary_execute(mats, W.flags, tri, s.p, s.mat, rng, g, g_mi, g_mo);
	}
	if (event == EV_ELASTIC) {
		s.last_tri = -1;
		elastic_execute(mats[s.mat], W.flags, s.p, rng, logE);
	}
	return ALIVE;
}

}} // namespace nbl::dev
