// Device-side building blocks of the batched propagator: field evaluation
// (uniform, Grid3f trilinear, plane waves) and the Boris / Cash-Karp steps.
//
// The FP64 functions follow the reference's operation order exactly (no
// contraction: the library is built with -ffp-contract=off), so that a lane
// reproduces CRPropa3's CPU result bit for bit:
//   Grid<Vector3f>::trilinearInterpolate   include/crpropa/Grid.h:540-582
//   periodicClamp / reflectiveClamp         include/crpropa/Grid.h:31-34,49-59
//   PlaneWaveTurbulence::getField           src/magneticField/turbulentField/PlaneWaveTurbulence.cpp:231-240
//   PropagationBP::dY                       src/module/PropagationBP.cpp:19-39
//   PropagationCK::dYdt / tryStep           src/module/PropagationCK.cpp:28-61
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "crp_crmath.h"

namespace crp {

constexpr double kCLight = 2.99792458e8; // include/crpropa/Units.h:64

struct V3 {
	double x, y, z;
};

__device__ __forceinline__ V3 v3(double x, double y, double z) {
	V3 r;
	r.x = x;
	r.y = y;
	r.z = z;
	return r;
}

// Cash-Karp tableau of src/module/PropagationCK.cpp:11-26 (textbook constants).
struct CK {
	static constexpr double a10 = 1. / 5.;
	static constexpr double a20 = 3. / 40., a21 = 9. / 40.;
	static constexpr double a30 = 3. / 10., a31 = -9. / 10., a32 = 6. / 5.;
	static constexpr double a40 = -11. / 54., a41 = 5. / 2., a42 = -70. / 27., a43 = 35. / 27.;
	static constexpr double a50 = 1631. / 55296., a51 = 175. / 512., a52 = 575. / 13824., a53 = 44275. / 110592.,
	                        a54 = 253. / 4096.;
	static constexpr double b0 = 37. / 378., b1 = 0., b2 = 250. / 621., b3 = 125. / 594., b4 = 0.,
	                        b5 = 512. / 1771.;
	static constexpr double s0 = 2825. / 27648., s1 = 0., s2 = 18575. / 48384., s3 = 13525. / 55296.,
	                        s4 = 277. / 14336., s5 = 1. / 4.;
};

// Vector3<T>::getR: sqrt((x*x + y*y) + z*z)
__device__ __forceinline__ double norm(const V3 &v) { return __builtin_sqrt((v.x * v.x + v.y * v.y) + v.z * v.z); }

// x / s, bit-identical to the IEEE division, from invs = RN(1/s) (one IEEE division shared by
// several quotients with the same divisor): q = x * invs is within one ulp of x/s, the FMA
// residual x - q*s is exact, and RN(q + residual * invs) is the correctly rounded quotient
// (Markstein's correction theorem; J.-M. Muller et al., Handbook of Floating-Point Arithmetic,
// division with an FMA).  The theorem assumes no underflow or overflow: magnitudes outside
// [2^-500, 2^500] (and 0, inf, NaN) take the IEEE division.
__device__ __forceinline__ double div_rn(double x, double s, double invs) {
	const double ax = __builtin_fabs(x), as = __builtin_fabs(s);
	if (!(ax > 0x1p-500 && ax < 0x1p500 && as > 0x1p-500 && as < 0x1p500))
		return x / s;
	const double q = x * invs;
	const double r = __builtin_fma(-q, s, x);
	return __builtin_fma(r, invs, q);
}

constexpr double kInvCLight = 1.0 / 299792458.0; // RN(1/c), folded by the compiler

// The quotient of div_rn without its range test, for callers that test several operands at once and take
// the tested form where one of them fails: the tests and their branches, one per quotient, are a third of a
// Boris step's instructions and keep loads and independent steps from overlapping.  x = 0 is right too (the
// sum would lose the sign of -0).
__device__ __forceinline__ double div_fast(double x, double s, double invs) {
	const double q = x * invs;
	const double r = __builtin_fma(-q, s, x);
	return __builtin_copysign(__builtin_fma(r, invs, q), q);
}

// RN(1/s) for s within [2^-500, 2^500] without the division's scaling and special cases: the hardware's
// approximation (better than 2^-20) and a third-order step give 1/s to less than an ulp, and one more step
// rounds it correctly unless the significand of s is all ones (Markstein; Handbook of Floating-Point
// Arithmetic, the reciprocal with an FMA); 1/(2^k (2 - 2^-52)) rounds to 2^-(k+1) (1 + 2^-52).
__device__ __forceinline__ double rcp_rn(double s) {
	const double r = __builtin_amdgcn_rcp(s);
	const double e = __builtin_fma(-s, r, 1.0);
	const double y = __builtin_fma(r, __builtin_fma(e, e, e), r);
	const int hi = __double2hiint(s);
	const bool ones = (hi & 0xfffff) == 0xfffff && __double2loint(s) == -1;
	const double z = __builtin_fma(__builtin_fma(-s, y, 1.0), y, y);
	return ones ? __hiloint2double(0x7fd00000 - (hi & 0x7ff00000), 1) : z;
}

// RN(1/s) for s near 1; `bad` is set for |1 - s| > 2^-45.  With e = 1 - s (exact), 1/s = 1 + e + e^2 + ...: for
// s > 1, 1 - |e| is a double and the rest too small to matter; for s < 1, e is a multiple of 2^-53 and where
// 1 + e is a tie the rest decides it upwards, which e (1 + 2^-50) does as well.
__device__ __forceinline__ double rcp_near_one(double s, bool &bad) {
	const double e = 1.0 - s;
	bad |= !(__builtin_fabs(e) <= 0x1p-45);
	return __builtin_fma(e, 1.0 + 0x1p-50, 1.0);
}

// RN(sqrt(d)) for d near 1; `bad` is set for |d - 1| > 2^-44.  With e = d - 1 (exact), sqrt(d) = 1 + e/2 - e^2/8
// + ...: 1 + e/2 is a double or halfway between two, and the rest, too small to matter otherwise, decides a tie
// downwards, as |e| 2^-52 taken off does.
__device__ __forceinline__ double sqrt_near_one(double d, bool &bad) {
	const double e = d - 1.0, ae = __builtin_fabs(e);
	bad |= !(ae <= 0x1p-44);
	return 1.0 + __builtin_fma(ae, -0x1p-52, 0.5 * e);
}

// every component zero or of magnitude within [2^-500, 2^500) (infinities and NaN pass: their exponent reads 0)
__device__ __forceinline__ bool in_div_range(const V3 &v) {
	const int a = __builtin_amdgcn_frexp_exp(v.x), b = __builtin_amdgcn_frexp_exp(v.y),
	          c = __builtin_amdgcn_frexp_exp(v.z);
	const int lo = min(min(a, b), c), hi = max(max(a, b), c);
	return lo > -500 && hi <= 500;
}

// v / s, component by component, with one range test
__device__ __forceinline__ V3 div3_rn(const V3 &v, double s, double invs) {
	V3 r = v3(div_fast(v.x, s, invs), div_fast(v.y, s, invs), div_fast(v.z, s, invs));
	if (!(s > 0x1p-500 && s < 0x1p500 && in_div_range(v)))
		r = v3(v.x / s, v.y / s, v.z / s);
	return r;
}

// A trivially copyable value read from immutable device memory through the constant address space,
// so that wave-uniform reads become scalar loads.
template <class T> __device__ __forceinline__ T ld_const(const T *p) {
	static_assert(sizeof(T) % 4 == 0, "ld_const: size must be a multiple of 4");
	typedef __attribute__((address_space(4))) const uint32_t cu32;
	cu32 *src = (cu32 *)p;
	T out;
	uint32_t *dst = reinterpret_cast<uint32_t *>(&out);
#pragma unroll
	for (unsigned i = 0; i < sizeof(T) / 4; i++)
		dst[i] = src[i];
	return out;
}

// u / |u|, one range test
__device__ __forceinline__ V3 unit_rn(const V3 &u) {
	const double n = norm(u), invn = rcp_rn(n);
	V3 r = v3(div_fast(u.x, n, invn), div_fast(u.y, n, invn), div_fast(u.z, n, invn));
	if (!(n > 0x1p-500 && n < 0x1p500 && in_div_range(u)))
		r = v3(u.x / n, u.y / n, u.z / n);
	return r;
}

// ---------------------------------------------------------------- fields
// Parameters as the host computes them from the reference's field objects.
struct GridDesc {
	const float *values; // AoS float3 per point, index (ix*Ny + iy)*Nz + iz
	int nx, ny, nz;
	int reflective, clip;
	double gridOrigin[3]; // origin + spacing/2 (Grid.h:225-228)
	double spacing[3];
	double origin[3], edge[3]; // clipVolume box: origin, origin + N*spacing (Grid.h:320-327)
	double invSpacing[3];      // RN(1/spacing), computed on the host
	double invN[3];            // 1/N per axis, for the division-free periodic wrap
	int fastDiv;               // spacing within [2^-300, 2^300]: its reciprocal may stand for the division
	int interp;                // GridInterp: Grid::setInterpolationType (Grid.h:24-28, 255-264)
};

// Interpolation types of Grid::interpolate (include/crpropa/Grid.h:24-28, 318-335), numbered as
// the C ABI's crp_grid_interpolation
enum GridInterp { kInterpTrilinear = 0, kInterpTricubic = 1, kInterpNearest = 2 };

// Plane-wave mode tables, one record per mode, read through the constant address space so that
// the compiler loads them with scalar (SMEM) loads into SGPRs: every lane of a wave evaluates the
// same mode at the same time, so one scalar load serves the wave and the VALU instructions take the
// mode's values as scalar operands.  The tables are immutable while kernels run.
struct PwMode64 {    // FP64 path: k, beta, kappa, xi*A (xi*A is the first product of getField)
	double k, beta, kx, ky, kz, ax, ay, az;
};
struct PwModeMixed { // mixed path: phase in turns = p . kt + bt (FP64), amplitude xi*A in FP32
	double ktx, kty, ktz, bt;
	float ax, ay, az, pad;
};
typedef __attribute__((address_space(4))) const PwMode64 PwMode64Const;
typedef __attribute__((address_space(4))) const PwModeMixed PwModeMixedConst;

struct PlaneWaveDesc {
	int nm;
	const PwMode64 *m64;   // [nm]
	const PwModeMixed *mm; // [nm]
	double reach;          // mixed path: |x| + |y| + |z| below which every phase is below 2^18 turns
};

struct FieldUniform {
	double b[3];
	__device__ __forceinline__ V3 eval(const V3 &) const { return v3(b[0], b[1], b[2]); }
	__device__ __forceinline__ float3 evalf(const V3 &) const { return make_float3((float)b[0], (float)b[1], (float)b[2]); }
};

struct FieldNone {
	__device__ __forceinline__ V3 eval(const V3 &) const { return v3(0.0, 0.0, 0.0); }
	__device__ __forceinline__ float3 evalf(const V3 &) const { return make_float3(0.f, 0.f, 0.f); }
};

// ---------------------------------------------------------------- mixed-precision grid helpers
// Cell index and fraction of a periodic axis without integer division: the
// position in cells is formed with a multiply by 1/spacing (FP64), wrapped
// with floor() in FP64, then the fraction goes to FP32.
__device__ __forceinline__ void periodic_cell_fast(double x, int n, double invn, int &lo, float &frac) {
	double fl = __builtin_floor(x);
	frac = (float)(x - fl);
	double w = fl - (double)n * __builtin_floor(fl * invn);
	int i = (int)w;
	i = i >= n ? i - n : (i < 0 ? i + n : i);
	lo = i;
}

__device__ __forceinline__ float3 trilinear_f32(const float *v, float fx, float fy, float fz) {
	// v: 24 floats, corners in the order of Grid.h:572-579
	const float gx = 1.f - fx, gy = 1.f - fy, gz = 1.f - fz;
	const float w0 = gx * gy * gz, w1 = fx * gy * gz, w2 = gx * fy * gz, w3 = gx * gy * fz;
	const float w4 = fx * gy * fz, w5 = gx * fy * fz, w6 = fx * fy * gz, w7 = fx * fy * fz;
	float b[3];
#pragma unroll
	for (int a = 0; a < 3; a++) {
		float s = v[a] * w0;
		s = __builtin_fmaf(v[3 + a], w1, s);
		s = __builtin_fmaf(v[6 + a], w2, s);
		s = __builtin_fmaf(v[9 + a], w3, s);
		s = __builtin_fmaf(v[12 + a], w4, s);
		s = __builtin_fmaf(v[15 + a], w5, s);
		s = __builtin_fmaf(v[18 + a], w6, s);
		s = __builtin_fmaf(v[21 + a], w7, s);
		b[a] = s;
	}
	return make_float3(b[0], b[1], b[2]);
}

// x / s rounded exactly like the IEEE division the reference performs, without a division:
// q = x * RN(1/s) is within one ulp of x/s, the FMA residual x - q*s is exact, and
// RN(q + residual * RN(1/s)) is the correctly rounded quotient when nothing underflows or
// overflows (Markstein's correction theorem; J.-M. Muller et al., Handbook of Floating-Point
// Arithmetic, the chapter on division with an FMA).  Magnitudes outside [2^-500, 2^500] (and
// 0, inf, NaN) take the IEEE division.
__device__ __forceinline__ double div_cr(double x, double s, double invs, int fast) {
	const double ax = __builtin_fabs(x);
	if (!(fast && ax > 0x1p-500 && ax < 0x1p500))
		return x / s;
	const double q = x * invs;
	const double r = __builtin_fma(-q, s, x);
	return __builtin_fma(r, invs, q);
}

// ((i % n) + n) % n (Grid.h:31-34) without an integer division: floor(i * (1/n)) is within one
// of floor(i/n) for |i| <= 2^31, the remainder is corrected into [0, n).  The remainder lies within
// (-n, 2n), so 32-bit arithmetic modulo 2^32 forms it (n < 2^30).
__device__ __forceinline__ int wrap_index(int i, int n, double invn) {
	const int q = (int)__builtin_floor((double)i * invn);
	int r = (int)((unsigned)i - (unsigned)q * (unsigned)n);
	r += (r < 0) ? n : 0;
	r -= (r >= n) ? n : 0;
	return r;
}

__device__ __forceinline__ void periodic_clamp(double x, int n, double invn, int &lo, int &hi, double &frac) {
	double fl = __builtin_floor(x);
	lo = wrap_index((int)fl, n, invn);
	hi = (lo + 1 == n) ? 0 : lo + 1;
	frac = x - fl;
}

// reflectiveClamp's loop (Grid.h:49-59) without its passes: mirrored at -1/2 once, moved by a multiple of the
// period 2n and mirrored at n - 1/2 once, x lies in [-1/2, n - 1/2] where the loop ends.  Below 2^50 every
// one of these operations is exact (a result is a multiple of the operand's last bit and no larger), as the
// loop's are, and two points of [-1/2, n - 1/2] are never images of each other, so the bits agree.  The
// multiple can come out one too large where x + 1/2 rounds up to it: x then lies just outside, which the
// caller tests.
__device__ __forceinline__ double mirror_fold(double x, int n, double invn) {
	const double dn = (double)n, p = 2 * dn;
	x = (x < -0.5) ? -x - 1 : x;
	x = __builtin_fma(-__builtin_floor((x + 0.5) * (0.5 * invn)), p, x);
	return (x > dn - 0.5) ? p - x - 1 : x;
}

__device__ __forceinline__ void reflective_clamp(double x, int n, double invn, int &lo, int &hi, double &frac) {
	if ((x < -0.5) || (x > (n - 0.5))) { // most positions are inside, and a wave of them takes none of this
		if (__builtin_fabs(x) < 0x1p50)
			x = mirror_fold(x, n, invn);
		while ((x < -0.5) || (x > (n - 0.5)))
			x = 2 * n * (x > (n - 0.5)) - x - 1;
	}
	double fl = __builtin_floor(x);
	lo = (int)fl;
	hi = lo + (lo < n - 1);
	if (x < 0) {
		lo = 0;
		hi = 0;
	}
	frac = x - fl;
}

// one axis of a trilinear cell in a straight line, periodic or reflective; `bad` where reflective_clamp has
// to be asked
__device__ __forceinline__ void clamp_fast(double x, int n, double invn, bool refl, int &lo, int &hi, double &frac,
                                           bool &bad) {
	if (refl) { // the same for every lane
		bad |= !(__builtin_fabs(x) < 0x1p50);
		x = mirror_fold(x, n, invn);
		bad |= !(x >= -0.5 && x <= n - 0.5);
	}
	const double fl = __builtin_floor(x);
	const int i = (int)fl, w = wrap_index(i, n, invn);
	lo = refl ? min(max(i, 0), n - 1) : w;
	hi = refl ? min(max(i + 1, 0), n - 1) : (w + 1 == n ? 0 : w + 1);
	frac = x - fl;
}

// ---------------------------------------------------------------- tricubic and nearest neighbour
// crpropa::round (include/crpropa/Grid.h:61-63): r + 0.5 is rounded before the floor (so 0.5 - 2^-54
// goes up), unlike the C library's round
__device__ __forceinline__ double round_sym(double r) {
	return (r > 0.0) ? __builtin_floor(r + 0.5) : __builtin_ceil(r - 0.5);
}

// reflectiveBoundary (Grid.h:36-41) without its loop: each pass maps the index to its mirror image
// at the nearer face, and the images repeat with period 2n, so the loop ends at i mod 2n folded
// onto [0, n).  Every int maps into [0, n).
__device__ __forceinline__ int reflect_index(int i, int n) {
	const int p = 2 * n;
	int m = i % p;
	m += (m < 0) ? p : 0;
	return (m < n) ? m : p - 1 - m;
}

// fmod(x, n), which is x itself for |x| < n: most positions lie within a box of the origin, and the loop of
// the general case is left to the others
__device__ __attribute__((noinline)) inline double fmod_far(double x, double n) { return __builtin_fmod(x, n); }
__device__ __forceinline__ double fmod_near(double x, double n) { return __builtin_fabs(x) < n ? x : fmod_far(x, n); }

// Grid::closestValue (include/crpropa/Grid.h:383-405): flat index of the grid point nearest to p,
// mirrored (reflective) or wrapped (periodic) into the grid
__device__ inline size_t grid_closest(const GridDesc &g, const V3 &p) {
	const double rx = div_cr(p.x - g.gridOrigin[0], g.spacing[0], g.invSpacing[0], g.fastDiv);
	const double ry = div_cr(p.y - g.gridOrigin[1], g.spacing[1], g.invSpacing[1], g.fastDiv);
	const double rz = div_cr(p.z - g.gridOrigin[2], g.spacing[2], g.invSpacing[2], g.fastDiv);
	int ix, iy, iz;
	if (g.reflective) {
		ix = reflect_index((int)round_sym(rx), g.nx);
		iy = reflect_index((int)round_sym(ry), g.ny);
		iz = reflect_index((int)round_sym(rz), g.nz);
	} else {
		// fmod(r, n) lies in (-n, n), its rounding in [-n, n]: (i + n * (i < 0)) % n is one correction each way
		ix = (int)round_sym(fmod_near(rx, (double)g.nx));
		iy = (int)round_sym(fmod_near(ry, (double)g.ny));
		iz = (int)round_sym(fmod_near(rz, (double)g.nz));
		ix += (ix < 0) ? g.nx : 0;
		iy += (iy < 0) ? g.ny : 0;
		iz += (iz < 0) ? g.nz : 0;
		ix -= (ix >= g.nx) ? g.nx : 0;
		iy -= (iy >= g.ny) ? g.ny : 0;
		iz -= (iz >= g.nz) ? g.nz : 0;
	}
	// a non-finite position converts to indices outside the grid: read point 0 instead of faulting
	if ((unsigned)ix >= (unsigned)g.nx || (unsigned)iy >= (unsigned)g.ny || (unsigned)iz >= (unsigned)g.nz)
		ix = iy = iz = 0;
	return ((size_t)ix * g.ny + iy) * g.nz + iz;
}

// CubicInterpolate (include/crpropa/Grid.h:436-456), one lane of the SSE code in FP32; t, t^2 and t^3
// are formed in double by the caller and rounded to float once each
__device__ __forceinline__ float cubic_f32(float p0, float p1, float p2, float p3, float t, float t2, float t3) {
	const float term = (0.5f * p2 - 0.5f * p0) * t;
	const float term2 = ((p0 + 2.f * p2) - (2.5f * p1 + 0.5f * p3)) * t2;
	const float term3 = ((1.5f * p1 + 0.5f * p3) - (0.5f * p0 + 1.5f * p2)) * t3;
	return ((term3 + term2) + term) + p1;
}

// CubicInterpolateScalar (include/crpropa/Grid.h:499-501) in FP64, left to right
__device__ __forceinline__ double cubic_f64(double p0, double p1, double p2, double p3, double t) {
	return (((((-0.5 * p0 + 1.5 * p1) - 1.5 * p2) + 0.5 * p3) * t * t * t +
	         (((p0 - 2.5 * p1) + p2 * 2) - 0.5 * p3) * t * t) +
	        (-0.5 * p0 + 0.5 * p2) * t) +
	       p1;
}

// neighbour index i of one axis through periodicGet / reflectiveGet (Grid.h:346-358)
__device__ __forceinline__ int cubic_index(int i, int n, double invn, int reflective) {
	return reflective ? reflect_index(i, n) : wrap_index(i, n, invn);
}

// unit-grid position of p: the reference's r = (pos - gridOrigin) / spacing, iX0 = floor(r),
// fX = r - iX0 (Grid.h:461-472)
__device__ __forceinline__ void cubic_origin(const GridDesc &g, const V3 &p, int i0[3], double f[3]) {
	const double r[3] = {div_cr(p.x - g.gridOrigin[0], g.spacing[0], g.invSpacing[0], g.fastDiv),
	                     div_cr(p.y - g.gridOrigin[1], g.spacing[1], g.invSpacing[1], g.fastDiv),
	                     div_cr(p.z - g.gridOrigin[2], g.spacing[2], g.invSpacing[2], g.fastDiv)};
#pragma unroll
	for (int a = 0; a < 3; a++) {
		i0[a] = (int)__builtin_floor(r[a]);
		f[a] = r[a] - (double)i0[a];
	}
}

// Grid<Vector3f>::tricubicInterpolate (include/crpropa/Grid.h:459-492): cubics along z for each of
// the 16 (x, y) neighbours, along y for each of the 4 x neighbours, then along x; the x, y and z
// components are independent lanes.  The result is FP32, widened to double as getField returns it.
__device__ inline V3 grid_tricubic(const GridDesc &g, const V3 &p) {
	int i0[3];
	double f[3];
	cubic_origin(g, p, i0, f);
	float t[3], t2[3], t3[3];
#pragma unroll
	for (int a = 0; a < 3; a++) {
		t[a] = (float)f[a];
		t2[a] = (float)(f[a] * f[a]);
		t3[a] = (float)(f[a] * f[a] * f[a]);
	}
	int Z[4];
	size_t Y[4];
#pragma unroll
	for (int d = 0; d < 4; d++) {
		Z[d] = cubic_index(i0[2] - 1 + d, g.nz, g.invN[2], g.reflective);
		Y[d] = (size_t)cubic_index(i0[1] - 1 + d, g.ny, g.invN[1], g.reflective) * g.nz;
	}
	float vx[4][3];
#pragma unroll
	for (int a = 0; a < 4; a++) {
		const size_t X = (size_t)cubic_index(i0[0] - 1 + a, g.nx, g.invN[0], g.reflective) * g.ny * g.nz;
		float vy[4][3];
#pragma unroll
		for (int b = 0; b < 4; b++) {
			const float *q0 = g.values + 3 * (X + Y[b] + Z[0]), *q1 = g.values + 3 * (X + Y[b] + Z[1]);
			const float *q2 = g.values + 3 * (X + Y[b] + Z[2]), *q3 = g.values + 3 * (X + Y[b] + Z[3]);
#pragma unroll
			for (int l = 0; l < 3; l++)
				vy[b][l] = cubic_f32(q0[l], q1[l], q2[l], q3[l], t[2], t2[2], t3[2]);
		}
#pragma unroll
		for (int l = 0; l < 3; l++)
			vx[a][l] = cubic_f32(vy[0][l], vy[1][l], vy[2][l], vy[3][l], t[1], t2[1], t3[1]);
	}
	float b[3];
#pragma unroll
	for (int l = 0; l < 3; l++)
		b[l] = cubic_f32(vx[0][l], vx[1][l], vx[2][l], vx[3][l], t[0], t2[0], t3[0]);
	return v3((double)b[0], (double)b[1], (double)b[2]);
}

// Grid<float>::tricubicInterpolate(double, ...) (include/crpropa/Grid.h:504-536): the same loops in
// FP64 over the float values; Grid::interpolate narrows the result to float
__device__ inline float scalar_grid_tricubic(const GridDesc &g, const V3 &p) {
	int i0[3];
	double f[3];
	cubic_origin(g, p, i0, f);
	int Z[4];
	size_t Y[4];
#pragma unroll
	for (int d = 0; d < 4; d++) {
		Z[d] = cubic_index(i0[2] - 1 + d, g.nz, g.invN[2], g.reflective);
		Y[d] = (size_t)cubic_index(i0[1] - 1 + d, g.ny, g.invN[1], g.reflective) * g.nz;
	}
	double vx[4];
#pragma unroll
	for (int a = 0; a < 4; a++) {
		const size_t X = (size_t)cubic_index(i0[0] - 1 + a, g.nx, g.invN[0], g.reflective) * g.ny * g.nz;
		double vy[4];
#pragma unroll
		for (int b = 0; b < 4; b++) {
			const float *q = g.values + X + Y[b];
			vy[b] = cubic_f64(q[Z[0]], q[Z[1]], q[Z[2]], q[Z[3]], f[2]);
		}
		vx[a] = cubic_f64(vy[0], vy[1], vy[2], vy[3], f[1]);
	}
	return (float)cubic_f64(vx[0], vx[1], vx[2], vx[3], f[0]);
}

// Grid::interpolate (Grid.h:329-332) for the tricubic and nearest-neighbour types, after the clip
// test: inline in the kernels of FieldGridAny (which read nothing else), out of line for the field
// types that read such grids beside others (JF12's turbulent grid, decorator leaves)
__device__ __forceinline__ V3 grid_eval_other_inline(const GridDesc &g, const V3 &p) {
	if (g.interp == kInterpNearest) {
		const float *c = g.values + 3 * grid_closest(g, p);
		return v3((double)c[0], (double)c[1], (double)c[2]);
	}
	return grid_tricubic(g, p);
}
__device__ __attribute__((noinline)) V3 grid_eval_other(const GridDesc &g, const V3 &p) {
	return grid_eval_other_inline(g, p);
}

__device__ __forceinline__ float scalar_grid_other_inline(const GridDesc &g, const V3 &p) {
	if (g.interp == kInterpNearest)
		return g.values[grid_closest(g, p)];
	return scalar_grid_tricubic(g, p);
}
__device__ __attribute__((noinline)) float scalar_grid_other(const GridDesc &g, const V3 &p) {
	return scalar_grid_other_inline(g, p);
}

// p in units of the spacing from the first point: the reference's (pos - gridOrigin) / spacing, with one
// range test for the three.  Fast: without the division, `bad` set where it is needed.  A quotient of magnitude
// below 2^-500 need not be rounded right (fastDiv: the spacing is within [2^-300, 2^300]): only its sign
// reaches the cell, and the position within the cell rounds to 0 or 1 all the same.
template <bool Fast>
__device__ __forceinline__ void grid_position(const GridDesc &g, const V3 &p, double &rx, double &ry, double &rz,
                                              bool *bad) {
	const double dx = p.x - g.gridOrigin[0], dy = p.y - g.gridOrigin[1], dz = p.z - g.gridOrigin[2];
	const double qx = dx * g.invSpacing[0], qy = dy * g.invSpacing[1], qz = dz * g.invSpacing[2];
	rx = __builtin_fma(__builtin_fma(-qx, g.spacing[0], dx), g.invSpacing[0], qx);
	ry = __builtin_fma(__builtin_fma(-qy, g.spacing[1], dy), g.invSpacing[1], qy);
	rz = __builtin_fma(__builtin_fma(-qz, g.spacing[2], dz), g.invSpacing[2], qz);
	const double far = __builtin_fmax(__builtin_fmax(__builtin_fabs(dx), __builtin_fabs(dy)), __builtin_fabs(dz));
	const bool slow = !(far < 0x1p500 && g.fastDiv);
	if (Fast) {
		*bad |= slow;
	} else if (slow) {
		rx = dx / g.spacing[0];
		ry = dy / g.spacing[1];
		rz = dz / g.spacing[2];
	}
}

struct FieldGrid {
	GridDesc g;

	// the corners' values in the order of Grid.h:572-579
	__device__ __forceinline__ V3 sum(int x0, int x1, int y0, int y1, int z0, int z1, double fx, double fy,
	                                  double fz) const {
		// weights narrowed to float (Vector3<float>::operator*(float))
		const float wx0 = (float)fx, wy0 = (float)fy, wz0 = (float)fz;
		const float wx1 = (float)(1 - fx), wy1 = (float)(1 - fy), wz1 = (float)(1 - fz);
		const size_t sy = (size_t)g.nz, sx = (size_t)g.ny * g.nz;
		const size_t bx0 = (size_t)x0 * sx, bx1 = (size_t)x1 * sx;
		const size_t by0 = (size_t)y0 * sy, by1 = (size_t)y1 * sy;
		const float *v = g.values;
		const float *c0 = v + 3 * (bx0 + by0 + z0);
		const float *c1 = v + 3 * (bx1 + by0 + z0);
		const float *c2 = v + 3 * (bx0 + by1 + z0);
		const float *c3 = v + 3 * (bx0 + by0 + z1);
		const float *c4 = v + 3 * (bx1 + by0 + z1);
		const float *c5 = v + 3 * (bx0 + by1 + z1);
		const float *c6 = v + 3 * (bx1 + by1 + z0);
		const float *c7 = v + 3 * (bx1 + by1 + z1);
		float b[3];
#pragma unroll
		for (int a = 0; a < 3; a++) {
			float s = 0.0f;
			s += ((c0[a] * wx1) * wy1) * wz1;
			s += ((c1[a] * wx0) * wy1) * wz1;
			s += ((c2[a] * wx1) * wy0) * wz1;
			s += ((c3[a] * wx1) * wy1) * wz0;
			s += ((c4[a] * wx0) * wy1) * wz0;
			s += ((c5[a] * wx1) * wy0) * wz0;
			s += ((c6[a] * wx0) * wy0) * wz1;
			s += ((c7[a] * wx0) * wy0) * wz0;
			b[a] = s;
		}
		return v3((double)b[0], (double)b[1], (double)b[2]);
	}
	__device__ __forceinline__ bool outside(const V3 &p) const {
		if (!g.clip)
			return false;
		bool in = (p.x >= g.origin[0]) && (p.x <= g.edge[0]);
		in &= (p.y >= g.origin[1]) && (p.y <= g.edge[1]);
		in &= (p.z >= g.origin[2]) && (p.z <= g.edge[2]);
		return !in;
	}
	__device__ __forceinline__ V3 eval(const V3 &p) const {
		if (outside(p))
			return v3(0.0, 0.0, 0.0);
		double rx, ry, rz;
		grid_position<false>(g, p, rx, ry, rz, nullptr);
		int x0, x1, y0, y1, z0, z1;
		double fx, fy, fz;
		if (g.reflective) {
			reflective_clamp(rx, g.nx, g.invN[0], x0, x1, fx);
			reflective_clamp(ry, g.ny, g.invN[1], y0, y1, fy);
			reflective_clamp(rz, g.nz, g.invN[2], z0, z1, fz);
		} else {
			periodic_clamp(rx, g.nx, g.invN[0], x0, x1, fx);
			periodic_clamp(ry, g.ny, g.invN[1], y0, y1, fy);
			periodic_clamp(rz, g.nz, g.invN[2], z0, z1, fz);
		}
		return sum(x0, x1, y0, y1, z0, z1, fx, fy, fz);
	}
	// eval's straight line: the same value wherever it leaves `bad` alone
	__device__ __forceinline__ V3 eval_fast(const V3 &p, bool &bad) const {
		double rx, ry, rz, fx, fy, fz;
		grid_position<true>(g, p, rx, ry, rz, &bad);
		int x0, x1, y0, y1, z0, z1;
		const bool refl = g.reflective != 0;
		clamp_fast(rx, g.nx, g.invN[0], refl, x0, x1, fx, bad);
		clamp_fast(ry, g.ny, g.invN[1], refl, y0, y1, fy, bad);
		clamp_fast(rz, g.nz, g.invN[2], refl, z0, z1, fz, bad);
		const V3 b = sum(x0, x1, y0, y1, z0, z1, fx, fy, fz);
		return outside(p) ? v3(0.0, 0.0, 0.0) : b;
	}
	__device__ __forceinline__ const FieldGrid &lane_field() const { return *this; }

	// mixed precision: reference index arithmetic, FP32 weights and fused sum
	__device__ __forceinline__ float3 evalf(const V3 &p) const {
		if (g.clip) {
			bool in = (p.x >= g.origin[0]) && (p.x <= g.edge[0]);
			in &= (p.y >= g.origin[1]) && (p.y <= g.edge[1]);
			in &= (p.z >= g.origin[2]) && (p.z <= g.edge[2]);
			if (!in)
				return make_float3(0.f, 0.f, 0.f);
		}
		double rx = (p.x - g.gridOrigin[0]) * g.invSpacing[0];
		double ry = (p.y - g.gridOrigin[1]) * g.invSpacing[1];
		double rz = (p.z - g.gridOrigin[2]) * g.invSpacing[2];
		int x0, x1, y0, y1, z0, z1;
		double fx, fy, fz;
		if (g.reflective) {
			reflective_clamp(rx, g.nx, g.invN[0], x0, x1, fx);
			reflective_clamp(ry, g.ny, g.invN[1], y0, y1, fy);
			reflective_clamp(rz, g.nz, g.invN[2], z0, z1, fz);
		} else {
			periodic_clamp(rx, g.nx, g.invN[0], x0, x1, fx);
			periodic_clamp(ry, g.ny, g.invN[1], y0, y1, fy);
			periodic_clamp(rz, g.nz, g.invN[2], z0, z1, fz);
		}
		const size_t sy = (size_t)g.nz, sx = (size_t)g.ny * g.nz;
		const size_t X[2] = {(size_t)x0 * sx, (size_t)x1 * sx}, Yo[2] = {(size_t)y0 * sy, (size_t)y1 * sy};
		const int Z[2] = {z0, z1};
		const int cx[8] = {0, 1, 0, 0, 1, 0, 1, 1}, cy[8] = {0, 0, 1, 0, 0, 1, 1, 1}, cz[8] = {0, 0, 0, 1, 1, 1, 0, 1};
		float v[24];
#pragma unroll
		for (int k = 0; k < 8; k++) {
			const float *c = g.values + 3 * (X[cx[k]] + Yo[cy[k]] + Z[cz[k]]);
			v[3 * k] = c[0];
			v[3 * k + 1] = c[1];
			v[3 * k + 2] = c[2];
		}
		return trilinear_f32(v, (float)fx, (float)fy, (float)fz);
	}
};

// Grid<float>::interpolate + trilinearInterpolate (Grid.h:318-335, 540-582) with T = float: each
// corner value times the double weights in double, and every b += term rounds the double sum to
// float.  `g.values` holds one float per point.
__device__ __forceinline__ float scalar_grid_eval(const GridDesc &g, const V3 &p) {
	if (g.clip) {
		bool in = (p.x >= g.origin[0]) && (p.x <= g.edge[0]);
		in &= (p.y >= g.origin[1]) && (p.y <= g.edge[1]);
		in &= (p.z >= g.origin[2]) && (p.z <= g.edge[2]);
		if (!in)
			return 0.f;
	}
	const double rx = div_cr(p.x - g.gridOrigin[0], g.spacing[0], g.invSpacing[0], g.fastDiv);
	const double ry = div_cr(p.y - g.gridOrigin[1], g.spacing[1], g.invSpacing[1], g.fastDiv);
	const double rz = div_cr(p.z - g.gridOrigin[2], g.spacing[2], g.invSpacing[2], g.fastDiv);
	int x0, x1, y0, y1, z0, z1;
	double fx, fy, fz;
	if (g.reflective) {
		reflective_clamp(rx, g.nx, g.invN[0], x0, x1, fx);
		reflective_clamp(ry, g.ny, g.invN[1], y0, y1, fy);
		reflective_clamp(rz, g.nz, g.invN[2], z0, z1, fz);
	} else {
		periodic_clamp(rx, g.nx, g.invN[0], x0, x1, fx);
		periodic_clamp(ry, g.ny, g.invN[1], y0, y1, fy);
		periodic_clamp(rz, g.nz, g.invN[2], z0, z1, fz);
	}
	const double gx = 1 - fx, gy = 1 - fy, gz = 1 - fz;
	const size_t sy = (size_t)g.nz, sx = (size_t)g.ny * g.nz;
	const size_t bx0 = (size_t)x0 * sx, bx1 = (size_t)x1 * sx, by0 = (size_t)y0 * sy, by1 = (size_t)y1 * sy;
	const float *v = g.values;
	float b = 0.f;
	b = (float)((double)b + (((double)v[bx0 + by0 + z0] * gx) * gy) * gz);
	b = (float)((double)b + (((double)v[bx1 + by0 + z0] * fx) * gy) * gz);
	b = (float)((double)b + (((double)v[bx0 + by1 + z0] * gx) * fy) * gz);
	b = (float)((double)b + (((double)v[bx0 + by0 + z1] * gx) * gy) * fz);
	b = (float)((double)b + (((double)v[bx1 + by0 + z1] * fx) * gy) * fz);
	b = (float)((double)b + (((double)v[bx0 + by1 + z1] * gx) * fy) * fz);
	b = (float)((double)b + (((double)v[bx1 + by1 + z0] * fx) * fy) * gz);
	b = (float)((double)b + (((double)v[bx1 + by1 + z1] * fx) * fy) * fz);
	return b;
}

// mixed precision: reciprocal spacing, FP32 weights, fused sum
__device__ __forceinline__ float scalar_grid_evalf(const GridDesc &g, const V3 &p) {
	if (g.clip) {
		bool in = (p.x >= g.origin[0]) && (p.x <= g.edge[0]);
		in &= (p.y >= g.origin[1]) && (p.y <= g.edge[1]);
		in &= (p.z >= g.origin[2]) && (p.z <= g.edge[2]);
		if (!in)
			return 0.f;
	}
	const double rx = (p.x - g.gridOrigin[0]) * g.invSpacing[0];
	const double ry = (p.y - g.gridOrigin[1]) * g.invSpacing[1];
	const double rz = (p.z - g.gridOrigin[2]) * g.invSpacing[2];
	int x0, x1, y0, y1, z0, z1;
	double fx, fy, fz;
	if (g.reflective) {
		reflective_clamp(rx, g.nx, g.invN[0], x0, x1, fx);
		reflective_clamp(ry, g.ny, g.invN[1], y0, y1, fy);
		reflective_clamp(rz, g.nz, g.invN[2], z0, z1, fz);
	} else {
		periodic_clamp(rx, g.nx, g.invN[0], x0, x1, fx);
		periodic_clamp(ry, g.ny, g.invN[1], y0, y1, fy);
		periodic_clamp(rz, g.nz, g.invN[2], z0, z1, fz);
	}
	const float wx = (float)fx, wy = (float)fy, wz = (float)fz, vx = 1.f - wx, vy = 1.f - wy, vz = 1.f - wz;
	const size_t sy = (size_t)g.nz, sx = (size_t)g.ny * g.nz;
	const size_t bx0 = (size_t)x0 * sx, bx1 = (size_t)x1 * sx, by0 = (size_t)y0 * sy, by1 = (size_t)y1 * sy;
	const float *v = g.values;
	float b = v[bx0 + by0 + z0] * (vx * vy * vz);
	b = __builtin_fmaf(v[bx1 + by0 + z0], wx * vy * vz, b);
	b = __builtin_fmaf(v[bx0 + by1 + z0], vx * wy * vz, b);
	b = __builtin_fmaf(v[bx0 + by0 + z1], vx * vy * wz, b);
	b = __builtin_fmaf(v[bx1 + by0 + z1], wx * vy * wz, b);
	b = __builtin_fmaf(v[bx0 + by1 + z1], vx * wy * wz, b);
	b = __builtin_fmaf(v[bx1 + by1 + z0], wx * wy * vz, b);
	b = __builtin_fmaf(v[bx1 + by1 + z1], wx * wy * wz, b);
	return b;
}

// Periodic Grid3f read through a cell-major corner table: cell (i,j,k) holds
// the 8 corner values of the reference's corner order (Grid.h:572-579) as 24
// floats, padded to 128 bytes, so one evaluation reads one aligned line
// instead of eight scattered 12-byte points.  Same values, same arithmetic
// as FieldGrid (bit-identical results).
constexpr int kCellFloats = 32;

struct FieldGridCells {
	GridDesc g;
	const float *cells; // [nx*ny*nz][32]

	__device__ __forceinline__ bool outside(const V3 &p) const {
		if (!g.clip)
			return false;
		bool in = (p.x >= g.origin[0]) && (p.x <= g.edge[0]);
		in &= (p.y >= g.origin[1]) && (p.y <= g.edge[1]);
		in &= (p.z >= g.origin[2]) && (p.z <= g.edge[2]);
		return !in;
	}
	// the cell of a position and the position within it; Fast: without the divisions' range tests, `bad` is
	// set where they are needed
	template <bool Fast = false>
	__device__ __forceinline__ size_t cell(const V3 &p, double &fx, double &fy, double &fz, bool *bad = nullptr) const {
		double rx, ry, rz;
		grid_position<Fast>(g, p, rx, ry, rz, bad);
		int x0, x1, y0, y1, z0, z1;
		periodic_clamp(rx, g.nx, g.invN[0], x0, x1, fx);
		periodic_clamp(ry, g.ny, g.invN[1], y0, y1, fy);
		periodic_clamp(rz, g.nz, g.invN[2], z0, z1, fz);
		return ((size_t)x0 * g.ny + y0) * g.nz + z0;
	}
	// mixed precision: reciprocal spacing, division-free periodic wrap
	__device__ __forceinline__ size_t cellf(const V3 &p, float &fx, float &fy, float &fz) const {
		int x0, y0, z0;
		periodic_cell_fast((p.x - g.gridOrigin[0]) * g.invSpacing[0], g.nx, 1.0 / g.nx, x0, fx);
		periodic_cell_fast((p.y - g.gridOrigin[1]) * g.invSpacing[1], g.ny, 1.0 / g.ny, y0, fy);
		periodic_cell_fast((p.z - g.gridOrigin[2]) * g.invSpacing[2], g.nz, 1.0 / g.nz, z0, fz);
		return ((size_t)x0 * g.ny + y0) * g.nz + z0;
	}
	// the sum over the corners of Grid.h:572-579
	static __device__ __forceinline__ V3 sum(const float4 *c, double fx, double fy, double fz) {
		const float wx0 = (float)fx, wy0 = (float)fy, wz0 = (float)fz;
		const float wx1 = (float)(1 - fx), wy1 = (float)(1 - fy), wz1 = (float)(1 - fz);
		const float4 q0 = c[0], q1 = c[1], q2 = c[2], q3 = c[3], q4 = c[4], q5 = c[5];
		const float v[24] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w, q2.x, q2.y, q2.z, q2.w,
		                     q3.x, q3.y, q3.z, q3.w, q4.x, q4.y, q4.z, q4.w, q5.x, q5.y, q5.z, q5.w};
		float b[3];
#pragma unroll
		for (int a = 0; a < 3; a++) {
			float s = 0.0f;
			s += ((v[0 + a] * wx1) * wy1) * wz1;
			s += ((v[3 + a] * wx0) * wy1) * wz1;
			s += ((v[6 + a] * wx1) * wy0) * wz1;
			s += ((v[9 + a] * wx1) * wy1) * wz0;
			s += ((v[12 + a] * wx0) * wy1) * wz0;
			s += ((v[15 + a] * wx1) * wy0) * wz0;
			s += ((v[18 + a] * wx0) * wy0) * wz1;
			s += ((v[21 + a] * wx0) * wy0) * wz0;
			b[a] = s;
		}
		return v3((double)b[0], (double)b[1], (double)b[2]);
	}
	static __device__ __forceinline__ float3 sumf(const float4 *c, float fx, float fy, float fz) {
		const float4 q0 = c[0], q1 = c[1], q2 = c[2], q3 = c[3], q4 = c[4], q5 = c[5];
		const float v[24] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w, q2.x, q2.y, q2.z, q2.w,
		                     q3.x, q3.y, q3.z, q3.w, q4.x, q4.y, q4.z, q4.w, q5.x, q5.y, q5.z, q5.w};
		return trilinear_f32(v, fx, fy, fz);
	}

	__device__ __forceinline__ V3 eval(const V3 &p) const {
		if (outside(p))
			return v3(0.0, 0.0, 0.0);
		double fx, fy, fz;
		const size_t c = cell(p, fx, fy, fz);
		return sum(reinterpret_cast<const float4 *>(cells + kCellFloats * c), fx, fy, fz);
	}
	// eval's straight line: the same value wherever it leaves `bad` alone
	__device__ __forceinline__ V3 eval_fast(const V3 &p, bool &bad) const {
		double fx, fy, fz;
		const size_t c = cell<true>(p, fx, fy, fz, &bad);
		const V3 b = sum(reinterpret_cast<const float4 *>(cells + kCellFloats * c), fx, fy, fz);
		return outside(p) ? v3(0.0, 0.0, 0.0) : b;
	}
	__device__ __forceinline__ const FieldGridCells &lane_field() const { return *this; }
	__device__ __forceinline__ float3 evalf(const V3 &p) const {
		if (outside(p))
			return make_float3(0.f, 0.f, 0.f);
		float fx, fy, fz;
		const size_t c = cellf(p, fx, fy, fz);
		return sumf(reinterpret_cast<const float4 *>(cells + kCellFloats * c), fx, fy, fz);
	}
};

// Reduced storage for the mixed path: each periodic cell holds its 8 corner
// vectors as FP16 values normalised by the FP32 scale of the 8^3-point brick
// that contains the cell (max |component| over the brick and its +1 faces),
// followed by that scale: 48 + 4 bytes, padded to one 64-byte sector.
constexpr int kCell16Bytes = 64;

struct FieldGridCells16 {
	GridDesc g;
	const unsigned char *cells16; // [nx*ny*nz][64]

	__device__ __forceinline__ V3 eval(const V3 &p) const {
		float3 b = evalf(p);
		return v3(b.x, b.y, b.z);
	}

	__device__ __forceinline__ float3 evalf(const V3 &p) const {
		if (g.clip) {
			bool in = (p.x >= g.origin[0]) && (p.x <= g.edge[0]);
			in &= (p.y >= g.origin[1]) && (p.y <= g.edge[1]);
			in &= (p.z >= g.origin[2]) && (p.z <= g.edge[2]);
			if (!in)
				return make_float3(0.f, 0.f, 0.f);
		}
		int x0, y0, z0;
		float fx, fy, fz;
		periodic_cell_fast((p.x - g.gridOrigin[0]) * g.invSpacing[0], g.nx, 1.0 / g.nx, x0, fx);
		periodic_cell_fast((p.y - g.gridOrigin[1]) * g.invSpacing[1], g.ny, 1.0 / g.ny, y0, fy);
		periodic_cell_fast((p.z - g.gridOrigin[2]) * g.invSpacing[2], g.nz, 1.0 / g.nz, z0, fz);
		const size_t cidx = ((size_t)x0 * g.ny + y0) * g.nz + z0;
		const uint4 *c = reinterpret_cast<const uint4 *>(cells16 + (size_t)kCell16Bytes * cidx);
		const uint4 a0 = c[0], a1 = c[1], a2 = c[2], a3 = c[3];
		const unsigned int w[13] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w, a2.x, a2.y, a2.z, a2.w, a3.x};
		float v[24];
#pragma unroll
		for (int k = 0; k < 12; k++) {
			const unsigned int u = w[k];
			v[2 * k] = __half2float(__ushort_as_half((unsigned short)(u & 0xffffu)));
			v[2 * k + 1] = __half2float(__ushort_as_half((unsigned short)(u >> 16)));
		}
		const float scale = __uint_as_float(w[12]);
		float3 b = trilinear_f32(v, fx, fy, fz);
		return make_float3(b.x * scale, b.y * scale, b.z * scale);
	}
};

// ModulatedMagneticFieldGrid::getField (src/magneticField/MagneticFieldGrid.cpp:51-55): the Grid3f
// value widened to double times the Grid1f modulation widened to double
template <class G> struct FieldModulated {
	G grid;
	GridDesc mod;
	__device__ __forceinline__ V3 eval(const V3 &p) const {
		const double m = (double)scalar_grid_eval(mod, p);
		const V3 b = grid.eval(p);
		return v3(b.x * m, b.y * m, b.z * m);
	}
	__device__ __forceinline__ float3 evalf(const V3 &p) const {
		const float m = scalar_grid_evalf(mod, p);
		const float3 b = grid.evalf(p);
		return make_float3(b.x * m, b.y * m, b.z * m);
	}
};

__device__ __forceinline__ bool in_clip_box(const GridDesc &g, const V3 &p) {
	bool in = (p.x >= g.origin[0]) && (p.x <= g.edge[0]);
	in &= (p.y >= g.origin[1]) && (p.y <= g.edge[1]);
	in &= (p.z >= g.origin[2]) && (p.z <= g.edge[2]);
	return in;
}

// Grid::interpolate (include/crpropa/Grid.h:318-335) for every interpolation type: trilinear in
// line, tricubic and nearest neighbour after the clip test (in line when Inline, else out of line)
template <bool Inline = false>
__device__ __forceinline__ V3 grid_interpolate(const GridDesc &g, const V3 &p) {
	if (g.interp == kInterpTrilinear)
		return FieldGrid{g}.eval(p);
	if (g.clip && !in_clip_box(g, p))
		return v3(0.0, 0.0, 0.0);
	return Inline ? grid_eval_other_inline(g, p) : grid_eval_other(g, p);
}

template <bool Inline = false>
__device__ __forceinline__ float scalar_grid_interpolate(const GridDesc &g, const V3 &p) {
	if (g.interp == kInterpTrilinear)
		return scalar_grid_eval(g, p);
	if (g.clip && !in_clip_box(g, p))
		return 0.f;
	return Inline ? scalar_grid_other_inline(g, p) : scalar_grid_other(g, p);
}

// MagneticFieldGrid and ModulatedMagneticFieldGrid (src/magneticField/MagneticFieldGrid.cpp:5-55)
// whose Grid3f or Grid1f is read tricubic or nearest-neighbour (Grid::setInterpolationType).  Its own
// field type, so that the trilinear kernels keep their register allocation.  The mixed path reads
// trilinear grids as FieldGrid::evalf does and the other types with the FP64 path's code, whose
// result is a float already.
struct FieldGridAny {
	GridDesc g;
	GridDesc mod; // the Grid1f modulation when `modulated`
	int modulated;

	__device__ __forceinline__ V3 eval(const V3 &p) const {
		const V3 b = grid_interpolate<true>(g, p);
		if (!modulated)
			return b;
		const double m = (double)scalar_grid_interpolate<true>(mod, p);
		return v3(b.x * m, b.y * m, b.z * m);
	}
	__device__ __forceinline__ float3 evalf(const V3 &p) const {
		float3 b;
		if (g.interp == kInterpTrilinear) {
			b = FieldGrid{g}.evalf(p);
		} else {
			const V3 d = grid_interpolate<true>(g, p);
			b = make_float3((float)d.x, (float)d.y, (float)d.z);
		}
		if (!modulated)
			return b;
		const float m = mod.interp == kInterpTrilinear ? scalar_grid_evalf(mod, p) : scalar_grid_interpolate<true>(mod, p);
		return make_float3(b.x * m, b.y * m, b.z * m);
	}
};

// Fields of which a group of lanes evaluates one position together: the lanes of a group (aligned, this
// many) hold the same particle
template <class F> struct LaneGroup {
	static constexpr int value = 1;
};

// the value of lane K of the quad
template <int K> __device__ __forceinline__ int quad_lane(int v) {
	return __builtin_amdgcn_mov_dpp(v, K * 0x55, 0xf, 0xf, true);
}
template <int K> __device__ __forceinline__ float quad_lane(float v) {
	return __int_as_float(quad_lane<K>(__float_as_int(v)));
}
// v[k] of lane j <- v[j] of lane k
__device__ __forceinline__ void quad_transpose(float v[4], bool odd, bool high) {
	constexpr int swap1 = 0xb1, swap2 = 0x4e; // quad_perm [1,0,3,2] and [2,3,0,1]
#pragma unroll
	for (int i = 0; i < 4; i += 2) {
		const float a = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v[i]), swap1, 0xf, 0xf, true));
		const float b = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v[i + 1]), swap1, 0xf, 0xf, true));
		v[i] = odd ? b : v[i];
		v[i + 1] = odd ? v[i + 1] : a;
	}
#pragma unroll
	for (int i = 0; i < 2; i++) {
		const float a = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v[i]), swap2, 0xf, 0xf, true));
		const float b = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v[i + 2]), swap2, 0xf, 0xf, true));
		v[i] = high ? b : v[i];
		v[i + 2] = high ? v[i + 2] : a;
	}
}

// A Grid3f read tricubic, four lanes to a particle (the same operations as grid_tricubic, so the same bits).
// One lane's 64 points lie in 16 rows of four; a load in which every lane reads a point of its own row costs
// the address unit a cycle a lane, 4096 cycles a wave for 64 particles, and one particle a lane leaves one
// wave of 330 registers on a SIMD.  Here the four lanes of a quad read the four points of a row together
// (48 bytes, one or two lines), and the quad shares the cubics: lane j takes the z-cubics of row y_j of
// every plane, the y-cubics of plane x_j, and all four the last one; values change lanes by DPP.
struct FieldTricubic {
	GridDesc g;

	template <bool Fast> __device__ __forceinline__ V3 value(const V3 &p, bool *bad) const {
		const int j = __lane_id() & 3;
		const bool odd = j & 1, high = j & 2;
		double r[3];
		grid_position<Fast>(g, p, r[0], r[1], r[2], bad);
		int own[3];
		float t[3], t2[3], t3[3];
#pragma unroll
		for (int a = 0; a < 3; a++) {
			const int i0 = (int)__builtin_floor(r[a]);
			const double f = r[a] - (double)i0;
			t[a] = (float)f;
			t2[a] = (float)(f * f);
			t3[a] = (float)(f * f * f);
			own[a] = i0 - 1 + j; // this lane's neighbour on the axis
		}
		const unsigned zo = (unsigned)cubic_index(own[2], g.nz, g.invN[2], g.reflective);
		const int yo = (int)((unsigned)cubic_index(own[1], g.ny, g.invN[1], g.reflective) * (unsigned)g.nz);
		const int xo = (int)((unsigned)cubic_index(own[0], g.nx, g.invN[0], g.reflective) * (unsigned)g.ny * (unsigned)g.nz);
		const unsigned Y[4] = {(unsigned)quad_lane<0>(yo), (unsigned)quad_lane<1>(yo), (unsigned)quad_lane<2>(yo),
		                       (unsigned)quad_lane<3>(yo)};
		const unsigned X[4] = {(unsigned)quad_lane<0>(xo), (unsigned)quad_lane<1>(xo), (unsigned)quad_lane<2>(xo),
		                       (unsigned)quad_lane<3>(xo)};
		float v[4][4][3]; // plane, row, component: this lane's point
#pragma unroll
		for (int a = 0; a < 4; a++)
#pragma unroll
			for (int b = 0; b < 4; b++) {
				const unsigned off = 12u * (X[a] + Y[b] + zo); // below 4 GiB (grid_tricubic_fits)
				const float *q = reinterpret_cast<const float *>(reinterpret_cast<const char *>(g.values) + off);
#pragma unroll
				for (int l = 0; l < 3; l++)
					v[a][b][l] = q[l];
			}
		float vx[3];
#pragma unroll
		for (int l = 0; l < 3; l++) {
			float w[4]; // plane a: row y_j after its z-cubic
#pragma unroll
			for (int a = 0; a < 4; a++) {
				float z[4] = {v[a][0][l], v[a][1][l], v[a][2][l], v[a][3][l]};
				quad_transpose(z, odd, high);
				w[a] = cubic_f32(z[0], z[1], z[2], z[3], t[2], t2[2], t3[2]);
			}
			quad_transpose(w, odd, high); // rows of plane x_j
			vx[l] = cubic_f32(w[0], w[1], w[2], w[3], t[1], t2[1], t3[1]);
		}
		float b[3];
#pragma unroll
		for (int l = 0; l < 3; l++)
			b[l] = cubic_f32(quad_lane<0>(vx[l]), quad_lane<1>(vx[l]), quad_lane<2>(vx[l]), quad_lane<3>(vx[l]), t[0],
			                 t2[0], t3[0]);
		return v3((double)b[0], (double)b[1], (double)b[2]);
	}
	__device__ __forceinline__ bool outside(const V3 &p) const { return g.clip && !in_clip_box(g, p); }
	__device__ __forceinline__ V3 eval(const V3 &p) const {
		if (outside(p))
			return v3(0.0, 0.0, 0.0);
		return value<false>(p, nullptr);
	}
	__device__ __forceinline__ V3 eval_fast(const V3 &p, bool &bad) const {
		const V3 b = value<true>(p, &bad);
		return outside(p) ? v3(0.0, 0.0, 0.0) : b;
	}
	__device__ __forceinline__ const FieldTricubic &lane_field() const { return *this; }
	__device__ __forceinline__ float3 evalf(const V3 &p) const {
		const V3 b = eval(p);
		return make_float3((float)b.x, (float)b.y, (float)b.z);
	}
};
template <> struct LaneGroup<FieldTricubic> {
	static constexpr int value = 4;
};

// A periodic Grid3f read tricubic through a table of row pairs: entry (x, y, z) holds the points z .. z + 3 of
// rows y and y + 1 (wrapped) as 24 floats in a 128-byte line, so the 64 points come from 8 lines instead of the
// 21.5 that 16 rows of 48 bytes touch; where a batch fills the chip the rate of line requests bounds it.  A run
// builds the table for itself (the grid may be the caller's memory and change between runs).
struct FieldTricubicTable {
	GridDesc g;
	const float *rows; // [nx*ny*nz][32]

	__device__ __forceinline__ V3 value(const V3 &p) const {
		double r[3];
		grid_position<false>(g, p, r[0], r[1], r[2], nullptr);
		int i0[3];
		float t[3], t2[3], t3[3];
#pragma unroll
		for (int a = 0; a < 3; a++) {
			i0[a] = (int)__builtin_floor(r[a]);
			const double f = r[a] - (double)i0[a];
			t[a] = (float)f;
			t2[a] = (float)(f * f);
			t3[a] = (float)(f * f * f);
		}
		const size_t z = (size_t)wrap_index(i0[2] - 1, g.nz, g.invN[2]);
		const size_t y0 = (size_t)wrap_index(i0[1] - 1, g.ny, g.invN[1]) * g.nz + z;
		const size_t y1 = (size_t)wrap_index(i0[1] + 1, g.ny, g.invN[1]) * g.nz + z;
		float vx[4][3];
#pragma unroll
		for (int a = 0; a < 4; a++) {
			const size_t x = (size_t)wrap_index(i0[0] - 1 + a, g.nx, g.invN[0]) * g.ny * g.nz;
			float w[4][3];
#pragma unroll
			for (int h = 0; h < 2; h++) {
				const float4 *c = reinterpret_cast<const float4 *>(rows + 32 * (x + (h ? y1 : y0)));
				const float4 q0 = c[0], q1 = c[1], q2 = c[2], q3 = c[3], q4 = c[4], q5 = c[5];
				const float v[24] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w, q2.x, q2.y, q2.z, q2.w,
				                     q3.x, q3.y, q3.z, q3.w, q4.x, q4.y, q4.z, q4.w, q5.x, q5.y, q5.z, q5.w};
#pragma unroll
				for (int l = 0; l < 3; l++) {
					w[2 * h][l] = cubic_f32(v[l], v[3 + l], v[6 + l], v[9 + l], t[2], t2[2], t3[2]);
					w[2 * h + 1][l] = cubic_f32(v[12 + l], v[15 + l], v[18 + l], v[21 + l], t[2], t2[2], t3[2]);
				}
			}
#pragma unroll
			for (int l = 0; l < 3; l++)
				vx[a][l] = cubic_f32(w[0][l], w[1][l], w[2][l], w[3][l], t[1], t2[1], t3[1]);
		}
		float b[3];
#pragma unroll
		for (int l = 0; l < 3; l++)
			b[l] = cubic_f32(vx[0][l], vx[1][l], vx[2][l], vx[3][l], t[0], t2[0], t3[0]);
		return v3((double)b[0], (double)b[1], (double)b[2]);
	}
	__device__ __forceinline__ bool outside(const V3 &p) const { return g.clip && !in_clip_box(g, p); }
	__device__ __forceinline__ V3 eval(const V3 &p) const {
		if (outside(p))
			return v3(0.0, 0.0, 0.0);
		return value(p);
	}
	__device__ __forceinline__ float3 evalf(const V3 &p) const {
		const V3 b = eval(p);
		return make_float3((float)b.x, (float)b.y, (float)b.z);
	}
};

struct FieldPlaneWave {
	PlaneWaveDesc w;

	// B = sum_i (xi_i A_i) cos(k_i (x . kappa_i) + beta_i), accumulated in mode order
	// (PlaneWaveTurbulence.cpp:231-240), with the correctly rounded cos; `tab` is crp_turn_tab or a copy
	__device__ __forceinline__ V3 sum(const V3 &p, const double *tab) const {
		double bx = 0.0, by = 0.0, bz = 0.0;
		PwMode64Const *m = (PwMode64Const *)w.m64;
		const int nm = w.nm;
#pragma unroll 2
		for (int i = 0; i < nm; i++) {
			const double kx = m[i].kx, ky = m[i].ky, kz = m[i].kz;
			double z_ = (p.x * kx + p.y * ky) + p.z * kz;
			double c = crp_cos_cr_turn(m[i].k * z_ + m[i].beta, tab);
			bx += m[i].ax * c;
			by += m[i].ay * c;
			bz += m[i].az * c;
		}
		return v3(bx, by, bz);
	}
	__device__ __forceinline__ V3 eval(const V3 &p) const { return sum(p, crp_turn_tab); }

	// mixed precision: phase in turns in FP64 (positions span many wavelengths), its fractional part
	// evaluated with the hardware cosine (v_cos_f32 computes cos(2 pi x)); amplitudes and the sum in FP32
	__device__ __forceinline__ float3 evalf(const V3 &p) const {
		float bx = 0.f, by = 0.f, bz = 0.f;
		PwModeMixedConst *m = (PwModeMixedConst *)w.mm;
		const int nm = w.nm;
#pragma unroll 4
		for (int i = 0; i < nm; i++) {
			const double t = __builtin_fma(p.x, m[i].ktx, __builtin_fma(p.y, m[i].kty, __builtin_fma(p.z, m[i].ktz, m[i].bt)));
			const float c = __builtin_amdgcn_cosf((float)__builtin_amdgcn_fract(t));
			bx = __builtin_fmaf(m[i].ax, c, bx);
			by = __builtin_fmaf(m[i].ay, c, by);
			bz = __builtin_fmaf(m[i].az, c, bz);
		}
		return make_float3(bx, by, bz);
	}
};

// Fields whose evaluation is one computation of all 64 lanes: callers reach it with the whole wave converged
template <class F> struct WaveField {
	static constexpr bool value = false;
};

// FieldPlaneWave with the cosine's table in LDS
struct FieldPlaneWaveLds : FieldPlaneWave {
	const double *tab;
	__device__ __forceinline__ V3 eval(const V3 &p) const { return sum(p, tab); }
};

// The mixed path's mode loop in a propagation kernel.  A vector instruction reads one scalar pair, so the
// phase's start value (the bias) comes from LDS, read by all lanes at once, instead of two moves a mode; it
// carries 1.5 x 2^20, after which the low word of the phase is its fraction in units of 2^-32 turns, rounded
// there (2^-33 turns; FP32 fractions have 2^-25), and a conversion and a product replace the FP64 fraction
// and its narrowing.  Positions whose phases leave 2^18 turns take FieldPlaneWave's loop.  Bound by vector
// issue: 46.6 cycles a mode and wave against 58.6.
struct FieldPlaneWaveMix : FieldPlaneWave {
	static constexpr int kModesMax = 2048; // 16 KB of LDS
	static constexpr double kBias = 1.5 * 1048576.0;
	const double *bias; // bt + kBias in LDS

	__device__ __forceinline__ float3 evalf(const V3 &p) const {
		if (!(__builtin_fabs(p.x) + __builtin_fabs(p.y) + __builtin_fabs(p.z) < w.reach))
			return FieldPlaneWave::evalf(p);
		float bx = 0.f, by = 0.f, bz = 0.f;
		PwModeMixedConst *m = (PwModeMixedConst *)w.mm;
		const int nm = w.nm;
#pragma unroll 8
		for (int i = 0; i < nm; i++) {
			const double t = __builtin_fma(p.z, m[i].ktz, __builtin_fma(p.y, m[i].kty, __builtin_fma(p.x, m[i].ktx, bias[i])));
			const float c = __builtin_amdgcn_cosf((float)__double2loint(t) * 0x1p-32f);
			bx = __builtin_fmaf(m[i].ax, c, bx);
			by = __builtin_fmaf(m[i].ay, c, by);
			bz = __builtin_fmaf(m[i].az, c, bz);
		}
		return make_float3(bx, by, bz);
	}
};

// The field a propagation kernel evaluates for its argument: `make` is called once by every thread of
// the workgroup; `lds` are lds_bytes() of dynamic LDS.  The FP64 plane waves copy the cosine's 12 KB table
// to LDS: 64 lanes read 64 entries of it per mode, which as global loads would be up to 128 line requests per
// mode and wave.  The mode loop is bound by FP64 issue: 65 vector instructions a mode with this table against
// about 230 with the octant table and its selection; 2^18 particles x 300 steps x 256 modes in 52.7 ms
// against 147.5.
template <class F, bool MIX> struct KernelField {
	typedef F type;
	static size_t lds_bytes(const F &, int) { return 0; }
	static __device__ __forceinline__ type make(const F &f, char *) { return f; }
};
template <> struct KernelField<FieldPlaneWave, false> {
	typedef FieldPlaneWaveLds type;
	static size_t lds_bytes(const FieldPlaneWave &, int) { return 2 * CRP_TURN_ENTRIES * sizeof(double); }
	static __device__ __forceinline__ type make(const FieldPlaneWave &f, char *lds) {
		double *const tab = reinterpret_cast<double *>(lds);
		for (int i = threadIdx.x; i < 2 * CRP_TURN_ENTRIES; i += blockDim.x)
			tab[i] = crp_turn_tab[i];
		__syncthreads();
		type r;
		r.w = f.w;
		r.tab = tab;
		return r;
	}
};
template <> struct KernelField<FieldPlaneWave, true> {
	typedef FieldPlaneWaveMix type;
	static size_t lds_bytes(const FieldPlaneWave &f, int) {
		return f.w.nm <= type::kModesMax ? f.w.nm * sizeof(double) : 0;
	}
	static __device__ __forceinline__ type make(const FieldPlaneWave &f, char *lds) {
		double *const bias = reinterpret_cast<double *>(lds);
		type r;
		r.w = f.w;
		r.bias = bias;
		if (f.w.nm > type::kModesMax) {
			r.w.reach = 0;
			return r;
		}
		for (int i = threadIdx.x; i < f.w.nm; i += blockDim.x)
			bias[i] = f.w.mm[i].bt + type::kBias;
		__syncthreads();
		return r;
	}
};

// FieldGridCells whose cell lines are gathered by the wave together.  A lane that reads its own line does
// it in six 16-byte loads, and each of them translates an address for every lane: once the table outgrows
// the reach of the first-level translation cache (about 3 GB) all six miss, and random lines come at
// 1.3e10/s.  Here eight lanes read one line in one load, piece by piece, straight into LDS, and eight
// loads serve the wave's 64 lines: one translation per line, 4.6e10 lines/s at 17 GB; below the cliff
// both ways reach the same 5.3e10/s, and the lane's own loads need no LDS (measured, 96 bytes per line).
// 512^3, 2^20 particles: an adaptive Cash-Karp step 224 us against 699, a fixed one 122 against 482, Boris 156 and
// 49 against 365 and 92.
// Lane 8g + j loads piece j ^ p of the line of lane 8g + p in load p, so that the eight lanes of a group
// find their pieces in eight different 16-byte columns of LDS when they read them back.
struct FieldGridCellsWave : FieldGridCells {
	static constexpr int kLdsPerWave = 8 * 1024;
	char *lds; // the wave's 8 KB

	template <int P> __device__ __forceinline__ void load(unsigned c, int lane) const {
		const unsigned line = (unsigned)__builtin_amdgcn_ds_swizzle((int)c, 0x18 | (P << 5)); // lane 8g + P's
		const int piece = (lane & 7) ^ P;
		if (piece < 6) // 96 of a line's 128 bytes hold corners
			__builtin_amdgcn_global_load_lds(
			    (const __attribute__((address_space(1))) void *)(cells + (size_t)kCellFloats * line + 4 * piece),
			    (__attribute__((address_space(3))) void *)(lds + P * 1024), 16, 0, 0);
	}
	// the six pieces of this lane's line; every lane of the wave calls it, with a cell of the table
	__device__ __forceinline__ void gather(size_t cidx, float4 q[6]) const {
		const int lane = __lane_id();
		const unsigned c = (unsigned)cidx;
		load<0>(c, lane); load<1>(c, lane); load<2>(c, lane); load<3>(c, lane);
		load<4>(c, lane); load<5>(c, lane); load<6>(c, lane); load<7>(c, lane);
		asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the lines are in LDS
		const int p = lane & 7;
		const char *r = lds + p * 1024 + (lane >> 3) * 128;
#pragma unroll
		for (int i = 0; i < 6; i++)
			q[i] = *reinterpret_cast<const float4 *>(r + ((i ^ p) << 4));
		asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // and read before the next gather overwrites them
	}
	__device__ __forceinline__ V3 eval(const V3 &p) const {
		double fx, fy, fz;
		float4 q[6];
		gather(cell(p, fx, fy, fz), q);
		const V3 b = sum(q, fx, fy, fz);
		return outside(p) ? v3(0.0, 0.0, 0.0) : b;
	}
	__device__ __forceinline__ V3 eval_fast(const V3 &p, bool &bad) const {
		double fx, fy, fz;
		float4 q[6];
		gather(cell<true>(p, fx, fy, fz, &bad), q);
		const V3 b = sum(q, fx, fy, fz);
		return outside(p) ? v3(0.0, 0.0, 0.0) : b;
	}
	__device__ __forceinline__ float3 evalf(const V3 &p) const {
		float fx, fy, fz;
		float4 q[6];
		gather(cellf(p, fx, fy, fz), q);
		const float3 b = sumf(q, fx, fy, fz);
		return outside(p) ? make_float3(0.f, 0.f, 0.f) : b;
	}
};
template <> struct WaveField<FieldGridCellsWave> {
	static constexpr bool value = true;
};
// the argument a kernel is launched with for FieldGridCellsWave
struct FieldGridCellsBig : FieldGridCells {};
template <bool MIX> struct KernelField<FieldGridCellsBig, MIX> {
	typedef FieldGridCellsWave type;
	static size_t lds_bytes(const FieldGridCellsBig &, int block) { return (size_t)type::kLdsPerWave * (block / 64); }
	static __device__ __forceinline__ type make(const FieldGridCellsBig &f, char *lds) {
		type r;
		static_cast<FieldGridCells &>(r) = f;
		r.lds = lds + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * type::kLdsPerWave;
		return r;
	}
};

// ---------------------------------------------------------------- mixed-precision steps
__device__ __forceinline__ float3 f3(float x, float y, float z) { return make_float3(x, y, z); }
__device__ __forceinline__ float3 cross3(const float3 &a, const float3 &b) {
	return f3(a.y * b.z - b.y * a.z, a.z * b.x - b.z * a.x, a.x * b.y - b.x * a.y);
}
__device__ __forceinline__ float dot3(const float3 &a, const float3 &b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ float3 unit3(const float3 &a) {
	const float r = __builtin_amdgcn_rsqf(dot3(a, a));
	return f3(a.x * r, a.y * r, a.z * r);
}

// Boris step with FP32 field and rotation, FP64 position drift.  coef =
// (q/2/m) * step / c formed in FP64 by the caller (t = B * coef).
template <class F>
__device__ __forceinline__ void bp_dy_mixed(const F &field, V3 &pos, float3 &dir, double step, float coef) {
	const double hs = step * 0.5;
	pos = v3(pos.x + (double)dir.x * hs, pos.y + (double)dir.y * hs, pos.z + (double)dir.z * hs);
	const float3 B = field.evalf(pos);
	const float3 t = f3(B.x * coef, B.y * coef, B.z * coef);
	const float sf = 2.f / (1.f + dot3(t, t));
	const float3 s = f3(t.x * sf, t.y * sf, t.z * sf);
	const float3 c1 = cross3(dir, t);
	const float3 vh = f3(dir.x + c1.x, dir.y + c1.y, dir.z + c1.z);
	const float3 c2 = cross3(vh, s);
	dir = f3(dir.x + c2.x, dir.y + c2.y, dir.z + c2.z);
	pos = v3(pos.x + (double)dir.x * hs, pos.y + (double)dir.y * hs, pos.z + (double)dir.z * hs);
}

// Cash-Karp trial with FP32 direction stages and field, FP64 positions and
// FP64 error accumulation.  Q = q c^2 / E (per particle); h = step / c.
struct YM {
	V3 x;
	float3 u;
};

// The field at a Cash-Karp trial's start.  A rejected trial is retried from the same state with a
// smaller step (src/module/PropagationCK.cpp:99-126), so the retry's first stage reads the same field
// value again; the adaptive kernels keep it for the retries instead of reading the grid (same bits).
// CkB0Store<true> serves fields whose FP64 evaluation is an FP32 value widened (the trilinear Grid3f
// readers): it keeps the value in three floats, three registers fewer; CkB0f is the mixed path's.
template <class F> struct FloatValuedField {
	static constexpr bool value = false;
};
template <> struct FloatValuedField<FieldGridCells> {
	static constexpr bool value = true;
};
template <> struct FloatValuedField<FieldGrid> {
	static constexpr bool value = true;
};
template <> struct FloatValuedField<FieldTricubicTable> {
	static constexpr bool value = true;
};
template <> struct FloatValuedField<FieldTricubic> {
	static constexpr bool value = true;
};
template <> struct FloatValuedField<FieldGridCellsWave> {
	static constexpr bool value = true;
};
template <bool F32> struct CkB0Store;
template <> struct CkB0Store<false> {
	V3 B;
	bool have;
	__device__ __forceinline__ V3 get() const { return B; }
	__device__ __forceinline__ void put(const V3 &b) { B = b; have = true; }
};
template <> struct CkB0Store<true> {
	float3 B;
	bool have;
	__device__ __forceinline__ V3 get() const { return v3((double)B.x, (double)B.y, (double)B.z); }
	__device__ __forceinline__ void put(const V3 &b) {
		B = make_float3((float)b.x, (float)b.y, (float)b.z);
		have = true;
	}
};
struct CkB0f {
	float3 B;
	bool have;
};

template <class F>
__device__ __forceinline__ void ck_dydt_mixed(const F &field, const YM &y, float Q, float3 &n, float3 &du,
                                              CkB0f *b0 = nullptr) {
	n = unit3(y.u);                 // velocity / c
	float3 B;
	if (WaveField<F>::value && b0) { // the whole wave evaluates while any lane needs it
		if (__ballot(!b0->have)) {
			const float3 e = field.evalf(y.x);
			if (!b0->have)
				b0->B = e;
			b0->have = true;
		}
		B = b0->B;
	} else if (b0 && b0->have) {
		B = b0->B;
	} else {
		B = field.evalf(y.x);
		if (b0) {
			b0->B = B;
			b0->have = true;
		}
	}
	const float3 c = cross3(n, B);
	du = f3(c.x * Q, c.y * Q, c.z * Q);
}

template <class F>
__device__ __forceinline__ void ck_trystep_mixed(const F &field, const YM &y, double h, float Q, YM &out, double &errU,
                                                 CkB0f *b0 = nullptr) {
	constexpr double cA[6][5] = {{0, 0, 0, 0, 0},
	                             {CK::a10, 0, 0, 0, 0},
	                             {CK::a20, CK::a21, 0, 0, 0},
	                             {CK::a30, CK::a31, CK::a32, 0, 0},
	                             {CK::a40, CK::a41, CK::a42, CK::a43, 0},
	                             {CK::a50, CK::a51, CK::a52, CK::a53, CK::a54}};
	constexpr double cB[6] = {CK::b0, CK::b1, CK::b2, CK::b3, CK::b4, CK::b5};
	constexpr double cE[6] = {CK::b0 - CK::s0, CK::b1 - CK::s1, CK::b2 - CK::s2,
	                          CK::b3 - CK::s3, CK::b4 - CK::s4, CK::b5 - CK::s5};
	const double ch = kCLight * h; // position step per unit of velocity/c
	const float hf = (float)h;
	float3 kn[6], ku[6];
	double ex = 0, ey = 0, ez = 0;
	out = y;
#pragma unroll
	for (int i = 0; i < 6; i++) {
		YM yn = y;
#pragma unroll
		for (int j = 0; j < i; j++) {
			const double ax = cA[i][j] * ch;
			const float au = (float)cA[i][j] * hf;
			yn.x = v3(yn.x.x + (double)kn[j].x * ax, yn.x.y + (double)kn[j].y * ax, yn.x.z + (double)kn[j].z * ax);
			yn.u = f3(__builtin_fmaf(ku[j].x, au, yn.u.x), __builtin_fmaf(ku[j].y, au, yn.u.y),
			          __builtin_fmaf(ku[j].z, au, yn.u.z));
		}
		ck_dydt_mixed(field, yn, Q, kn[i], ku[i], i == 0 ? b0 : nullptr);
		if (cB[i] != 0.0) {
			const double bx = cB[i] * ch;
			const float bu = (float)cB[i] * hf;
			out.x = v3(out.x.x + (double)kn[i].x * bx, out.x.y + (double)kn[i].y * bx, out.x.z + (double)kn[i].z * bx);
			out.u = f3(__builtin_fmaf(ku[i].x, bu, out.u.x), __builtin_fmaf(ku[i].y, bu, out.u.y),
			           __builtin_fmaf(ku[i].z, bu, out.u.z));
		}
		const double eh = cE[i] * h;
		ex += (double)ku[i].x * eh;
		ey += (double)ku[i].y * eh;
		ez += (double)ku[i].z * eh;
	}
	errU = __builtin_sqrt((ex * ex + ey * ey) + ez * ez);
}

// ---------------------------------------------------------------- Boris push
struct Y {
	V3 x, u;
};

// Fields with eval_fast, whose values are FP32 numbers widened: their FP64 steps run without range tests and
// are repeated with them where one would have failed
template <class F> struct FastField {
	static constexpr bool value = false;
};
template <> struct FastField<FieldGridCells> {
	static constexpr bool value = true;
};
template <> struct FastField<FieldGrid> {
	static constexpr bool value = true;
};
template <> struct FastField<FieldTricubic> {
	static constexpr bool value = true;
};
template <> struct FastField<FieldGridCellsWave> {
	static constexpr bool value = true;
};

// Whether bp_dy_fast's quotients stay where div_fast is exact: nonzero field components are within
// [2^-149, 2^128], so with these bounds B q/2 / m * step / c is 0 or within [2^-399, 2^390]
__device__ __forceinline__ bool bp_in_range(double q, double m, double step) {
	const double aq = __builtin_fabs(q);
	return aq > 0x1p-100 && aq < 0x1p20 && m > 0x1p-150 && m < 0x1p60 && step > 0x1p-60 && step < 0x1p120;
}

// bp_dy below in one straight line; `bad` is set where its result may differ
template <class F>
__device__ __forceinline__ Y bp_dy_fast(const F &field, const V3 &pos0, const V3 &dir, double step, double q, double m,
                                        double invm, bool &bad) {
	V3 pos = v3(pos0.x + (dir.x * step) / 2., pos0.y + (dir.y * step) / 2., pos0.z + (dir.z * step) / 2.);
	V3 B = field.eval_fast(pos, bad);
	V3 t = v3(div_fast(div_fast((B.x * q) / 2, m, invm) * step, kCLight, kInvCLight),
	          div_fast(div_fast((B.y * q) / 2, m, invm) * step, kCLight, kInvCLight),
	          div_fast(div_fast((B.z * q) / 2, m, invm) * step, kCLight, kInvCLight));
	double tt = (t.x * t.x + t.y * t.y) + t.z * t.z;
	double den = 1 + tt;
	bad |= !(den < 0x1p100); // NaN and infinities too
	const double invden = rcp_rn(den);
	V3 s = v3(div_fast(t.x * 2, den, invden), div_fast(t.y * 2, den, invden), div_fast(t.z * 2, den, invden));
	V3 vh = v3(dir.x + (dir.y * t.z - t.y * dir.z), dir.y + (dir.z * t.x - t.z * dir.x),
	           dir.z + (dir.x * t.y - t.x * dir.y));
	V3 d = v3(dir.x + (vh.y * s.z - s.y * vh.z), dir.y + (vh.z * s.x - s.z * vh.x),
	          dir.z + (vh.x * s.y - s.x * vh.y));
	Y out;
	out.x = v3(pos.x + (d.x * step) / 2., pos.y + (d.y * step) / 2., pos.z + (d.z * step) / 2.);
	out.u = d;
	return out;
}

// u / |u| twice, as setDirection(getUnitVector()) does
__device__ __forceinline__ V3 unit_twice_tested(const V3 &u) {
	const double n1 = norm(u), i1 = 1 / n1;
	const V3 u1 = v3(div_rn(u.x, n1, i1), div_rn(u.y, n1, i1), div_rn(u.z, n1, i1));
	const double n2 = norm(u1), i2 = 1 / n2;
	return v3(div_rn(u1.x, n2, i2), div_rn(u1.y, n2, i2), div_rn(u1.z, n2, i2));
}
// in one straight line; `bad` is set where it may differ.  Rotated: |u| is 1 to a few ulps, as a Boris rotation
// leaves it.  Components of u of magnitude 2^-400 and more, or 0, keep both divisions in range.
template <bool Rotated> __device__ __forceinline__ V3 unit_twice_fast(const V3 &u, bool &bad) {
	const double d1 = (u.x * u.x + u.y * u.y) + u.z * u.z;
	const double n1 = Rotated ? sqrt_near_one(d1, bad) : __builtin_sqrt(d1);
	const double i1 = Rotated ? rcp_near_one(n1, bad) : rcp_rn(n1);
	const V3 u1 = v3(div_fast(u.x, n1, i1), div_fast(u.y, n1, i1), div_fast(u.z, n1, i1));
	const double n2 = sqrt_near_one((u1.x * u1.x + u1.y * u1.y) + u1.z * u1.z, bad);
	const double i2 = rcp_near_one(n2, bad); // 1 to an ulp or two
	if (!Rotated)
		bad |= !(n1 > 0x1p-80 && n1 < 0x1p80);
	bad |= min(min(__builtin_amdgcn_frexp_exp(u.x), __builtin_amdgcn_frexp_exp(u.y)), __builtin_amdgcn_frexp_exp(u.z)) < -400;
	return v3(div_fast(u1.x, n2, i2), div_fast(u1.y, n2, i2), div_fast(u1.z, n2, i2));
}
__device__ __forceinline__ V3 unit_twice(const V3 &u) {
	bool bad = false;
	V3 d = unit_twice_fast<false>(u, bad);
	if (bad)
		d = unit_twice_tested(u);
	return d;
}

// PropagationBP::dY (src/module/PropagationBP.cpp:19-39)
// (divisions as div_rn with shared reciprocals: invm = RN(1/m) from the caller)
template <class F>
__device__ __forceinline__ Y bp_dy(const F &field, const V3 &pos0, const V3 &dir, double step, double q, double m,
                                  double invm) {
	V3 pos = v3(pos0.x + (dir.x * step) / 2., pos0.y + (dir.y * step) / 2., pos0.z + (dir.z * step) / 2.);
	V3 B = field.eval(pos);
	V3 t = v3(div_rn(div_rn((B.x * q) / 2, m, invm) * step, kCLight, kInvCLight),
	          div_rn(div_rn((B.y * q) / 2, m, invm) * step, kCLight, kInvCLight),
	          div_rn(div_rn((B.z * q) / 2, m, invm) * step, kCLight, kInvCLight));
	double tt = (t.x * t.x + t.y * t.y) + t.z * t.z;
	double den = 1 + tt;
	const double invden = 1 / den;
	V3 s = v3(div_rn(t.x * 2, den, invden), div_rn(t.y * 2, den, invden), div_rn(t.z * 2, den, invden));
	V3 vh = v3(dir.x + (dir.y * t.z - t.y * dir.z), dir.y + (dir.z * t.x - t.z * dir.x),
	           dir.z + (dir.x * t.y - t.x * dir.y));
	V3 d = v3(dir.x + (vh.y * s.z - s.y * vh.z), dir.y + (vh.z * s.x - s.z * vh.x),
	          dir.z + (vh.x * s.y - s.x * vh.y));
	Y out;
	out.x = v3(pos.x + (d.x * step) / 2., pos.y + (d.y * step) / 2., pos.z + (d.z * step) / 2.);
	out.u = d;
	return out;
}

// ---------------------------------------------------------------- Cash-Karp
// PropagationCK::dYdt (src/module/PropagationCK.cpp:51-61); qcE = (q*c)/E
template <class F>
__device__ __forceinline__ Y ck_dydt(const F &field, const Y &y, double qcE,
                                     CkB0Store<FloatValuedField<F>::value> *b0 = nullptr) {
	Y d;
	const V3 v = unit_rn(y.u);
	d.x = v3(v.x * kCLight, v.y * kCLight, v.z * kCLight);
	V3 B;
	if (WaveField<F>::value && b0) { // the whole wave evaluates while any lane needs it
		if (__ballot(!b0->have)) {
			const V3 e = field.eval(y.x);
			if (!b0->have)
				b0->put(e);
			b0->have = true;
		}
		B = b0->get();
	} else if (b0 && b0->have) {
		B = b0->get();
	} else {
		B = field.eval(y.x);
		if (b0)
			b0->put(B);
	}
	d.u = v3((d.x.y * B.z - B.y * d.x.z) * qcE, (d.x.z * B.x - B.z * d.x.x) * qcE,
	         (d.x.x * B.y - B.x * d.x.y) * qcE);
	return d;
}

// y_n += (k * a) * h, component-wise over x and u
__device__ __forceinline__ void axpy(Y &yn, const Y &k, double a, double h) {
	yn.x.x += (k.x.x * a) * h;
	yn.x.y += (k.x.y * a) * h;
	yn.x.z += (k.x.z * a) * h;
	yn.u.x += (k.u.x * a) * h;
	yn.u.y += (k.u.y * a) * h;
	yn.u.z += (k.u.z * a) * h;
}

// PropagationCK::tryStep (src/module/PropagationCK.cpp:28-49).  Returns the
// new phase point in `out` and the error estimate in `err`.
template <class F>
__device__ __forceinline__ void ck_trystep_err(const F &field, const Y &y, double h, double qcE, Y &out, Y &err,
                                               CkB0Store<FloatValuedField<F>::value> *b0 = nullptr) {
	err.x = v3(0.0, 0.0, 0.0);
	err.u = v3(0.0, 0.0, 0.0);
	out = y;
	const double e0 = CK::b0 - CK::s0, e1 = CK::b1 - CK::s1, e2 = CK::b2 - CK::s2, e3 = CK::b3 - CK::s3,
	             e4 = CK::b4 - CK::s4, e5 = CK::b5 - CK::s5;
	Y k0, k1, k2, k3, k4, k5, yn;
	k0 = ck_dydt(field, y, qcE, b0);
	axpy(out, k0, CK::b0, h);
	axpy(err, k0, e0, h);
	yn = y;
	axpy(yn, k0, CK::a10, h);
	k1 = ck_dydt(field, yn, qcE);
	axpy(out, k1, CK::b1, h);
	axpy(err, k1, e1, h);
	yn = y;
	axpy(yn, k0, CK::a20, h);
	axpy(yn, k1, CK::a21, h);
	k2 = ck_dydt(field, yn, qcE);
	axpy(out, k2, CK::b2, h);
	axpy(err, k2, e2, h);
	yn = y;
	axpy(yn, k0, CK::a30, h);
	axpy(yn, k1, CK::a31, h);
	axpy(yn, k2, CK::a32, h);
	k3 = ck_dydt(field, yn, qcE);
	axpy(out, k3, CK::b3, h);
	axpy(err, k3, e3, h);
	yn = y;
	axpy(yn, k0, CK::a40, h);
	axpy(yn, k1, CK::a41, h);
	axpy(yn, k2, CK::a42, h);
	axpy(yn, k3, CK::a43, h);
	k4 = ck_dydt(field, yn, qcE);
	axpy(out, k4, CK::b4, h);
	axpy(err, k4, e4, h);
	yn = y;
	axpy(yn, k0, CK::a50, h);
	axpy(yn, k1, CK::a51, h);
	axpy(yn, k2, CK::a52, h);
	axpy(yn, k3, CK::a53, h);
	axpy(yn, k4, CK::a54, h);
	k5 = ck_dydt(field, yn, qcE);
	axpy(out, k5, CK::b5, h);
	axpy(err, k5, e5, h);
}

// the same with only |err.u|, the quantity the step control reads
template <class F>
__device__ __forceinline__ void ck_trystep(const F &field, const Y &y, double h, double qcE, Y &out, double &errU,
                                           CkB0Store<FloatValuedField<F>::value> *b0 = nullptr) {
	Y err;
	ck_trystep_err(field, y, h, qcE, out, err, b0);
	errU = norm(err.u);
}

} // namespace crp
