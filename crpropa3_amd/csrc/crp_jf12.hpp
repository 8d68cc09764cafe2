// JF12Field on the device (included by crp_kernels.hip): the Jansson-Farrar 2012 Galactic field,
// src/magneticField/JF12Field.cpp:230-346, in the reference's FP64 operation order with the
// correctly rounded exp, atan2, sin and cos of crp_crmath.h; pow(x, 2.) is x * x, as GCC compiles
// the reference.
#pragma once

#include "crp_device.hpp"
#include "crpropa3_amd.h"

namespace crp {

// include/crpropa/Units.h: parsec = 648000 / pi * au, kiloparsec = 1e3 parsec
constexpr double kJKpc = 1e3 * (648000 / 3.14159265358979323846 * 149597870700.0);
constexpr double kJPi = 3.14159265358979323846;

// exp and atan2 for the arguments that their quick phases leave open
static __device__ __attribute__((noinline)) double jf12_exp(double x) { return crp_exp_rn(x); }
static __device__ __attribute__((noinline)) double jf12_atan2(double y, double x) { return crp_atan2_rn(y, x); }
// four exponentials side by side, one copy of the code
struct Exp4 {
	double a, b, c, d;
};
static __device__ __attribute__((noinline)) Exp4 jf12_exp4(double a, double b, double c, double d) {
	const double x[4] = {a, b, c, d};
	double v[4];
	bool ok[4];
#pragma unroll
	for (int i = 0; i < 4; i++)
		ok[i] = crp_exp_quick(x[i], &v[i]) && x[i] >= -708.0 && x[i] <= 708.0;
#pragma unroll
	for (int i = 0; i < 4; i++)
		if (!ok[i])
			v[i] = jf12_exp(x[i]);
	return Exp4{v[0], v[1], v[2], v[3]};
}

// Grid<float>::closestValue (include/crpropa/Grid.h:383-405): nearest point, reflective or periodic
__device__ __forceinline__ float scalar_grid_closest(const GridDesc &g, const V3 &p) { return g.values[grid_closest(g, p)]; }

struct FieldJF12 {
	crp_jf12_params p;
	GridDesc striated; // Grid1f, one float per point (use_striated)
	GridDesc turbulent; // Grid3f (use_turbulent)

	// pow(x, 2.) as the reference's build evaluates it: GCC rewrites the call as x * x
	__device__ __forceinline__ static double sq(double x) { return x * x; }

	// JF12Field::logisticFunction (JF12Field.cpp:188-190): 1 / (1 + exp(logistic_arg))
	__device__ __forceinline__ static double logistic_arg(double x, double x0, double w) {
		return -2. * (__builtin_fabs(x) - x0) / w;
	}

	// What an evaluation takes from the position: the transcendental functions of every part, each correctly
	// rounded.  The azimuth, its sine and cosine and the eight exponentials that most positions read are formed
	// side by side, whether or not this one reads all of them: a batch has about one wave to a SIMD, where every
	// instruction waits for the one before.  The angle inside rc and the other two windings are left to the
	// positions that have them.
	enum { E_DISK, E_HALO, E_HALO_R, E_X, E_TURB_DISK, E_TURB_R, E_TURB_HALO, E_ARM, E_COUNT };
	struct Geo {
		double d, r, rn, rc, rp;
		double sinPhi, cosPhi, sinThetaX, cosThetaX;
		double e[E_COUNT];
	};
	__device__ __forceinline__ Geo geo(const V3 &pos) const {
		Geo g;
		const double z = pos.z, az = __builtin_fabs(z);
		g.d = norm(pos);
		g.r = __builtin_sqrt(pos.x * pos.x + pos.y * pos.y);
		// X field (:252-300): rp and the angle inside rc
		g.rc = p.r_xc + az / p.tan_theta_x0;
		const bool inner = g.r < g.rc;
		g.rp = inner ? g.r * p.r_xc / g.rc : g.r - az / p.tan_theta_x0;
		// azimuth (Vector3::getPhi, include/crpropa/Vector3.h:136-142) and theta_X
		const double eps = 2.2250738585072014e-308; // numeric_limits<double>::min()
		const bool axis = __builtin_fabs(pos.x) < eps && __builtin_fabs(pos.y) < eps;
		const double tx = g.r - g.rp;
		double phi = 0, theta = 0;
		const bool okPhi = pos.x == pos.x && pos.y == pos.y && pos.x != 0 && pos.y != 0 && crp_atan2_quick(pos.y, pos.x, &phi);
		if (!okPhi && !axis)
			phi = jf12_atan2(pos.y, pos.x);
		if (axis)
			phi = 0.0;
		const bool useTheta = p.use_x && inner && g.r * g.r + z * z > 1 * kJKpc * kJKpc;
		if (useTheta)
			theta = z == 0 ? kJPi / 2. : jf12_atan2(az, tx);
		// exponentials
		double x[E_COUNT];
		x[E_DISK] = logistic_arg(z, p.h_disk, p.w_disk);
		x[E_HALO] = -az / p.z0;
		x[E_HALO_R] = logistic_arg(g.r, z >= 0 ? p.r_north : p.r_south, p.w_halo);
		x[E_X] = -g.rp / p.r_x;
		x[E_TURB_DISK] = p.use_turbulent ? -0.5 * sq(z / p.z_disk_turb) : 0.0;
		x[E_TURB_R] = p.use_turbulent ? -g.r / p.r_halo_turb : 0.0;
		x[E_TURB_HALO] = p.use_turbulent ? -0.5 * sq(z / p.z_halo_turb) : 0.0;
		x[E_ARM] = -(phi - kJPi) / p.tan90_minus_pitch;
		const Exp4 e0 = jf12_exp4(x[0], x[1], x[2], x[3]), e1 = jf12_exp4(x[4], x[5], x[6], x[7]);
		const double e[E_COUNT] = {e0.a, e0.b, e0.c, e0.d, e1.a, e1.b, e1.c, e1.d};
#pragma unroll
		for (int i = 0; i < E_COUNT; i++)
			g.e[i] = e[i];
		const bool okP = crp_sincos_turn(phi, &g.sinPhi, &g.cosPhi);
		g.sinThetaX = g.cosThetaX = 0;
		if (useTheta) {
			const crp_dd sc = crp_sincos_cr(theta);
			g.sinThetaX = sc.hi;
			g.cosThetaX = sc.lo;
		}
		if (!okP) {
			const crp_dd sc = crp_sincos_cr(phi);
			g.sinPhi = sc.hi;
			g.cosPhi = sc.lo;
		}
		// radius where the arm through (r, phi) crosses the negative x-axis, tried for three windings
		g.rn = g.r * g.e[E_ARM];
		if (g.rn > p.r_arms[7])
			g.rn = g.r * jf12_exp(-(phi + kJPi) / p.tan90_minus_pitch);
		if (g.rn > p.r_arms[7])
			g.rn = g.r * jf12_exp(-(phi + 3 * kJPi) / p.tan90_minus_pitch);
		return g;
	}

	// JF12Field::getRegularField with getDiskField, getToroidalHaloField, getXField (:192-300)
	__device__ __forceinline__ V3 regular(const V3 &pos, const Geo &gm) const {
		double bx = 0, by = 0, bz = 0;
		if (gm.d < 20 * kJKpc) {
			const double r = gm.r;
			const double sinPhi = gm.sinPhi, cosPhi = gm.cosPhi;
			const double z = pos.z;
			const double lfDisk = 1. / (1. + gm.e[E_DISK]);
			// disk
			double dx = 0, dy = 0;
			if (p.use_disk) {
				if (r > 3 * kJKpc) {
					double bMag = 0;
					if (r < 5 * kJKpc) {
						bMag = p.b_ring * (5 * kJKpc / r) * (1 - lfDisk);
						dx += -bMag * sinPhi;
						dy += bMag * cosPhi;
					} else {
						const double rn = gm.rn;
						for (int i = 7; i >= 0; i--)
							if (rn < p.r_arms[i])
								bMag = p.b_disk[i];
						bMag *= (5 * kJKpc / r) * (1 - lfDisk);
						dx += bMag * (p.sin_pitch * cosPhi - p.cos_pitch * sinPhi);
						dy += bMag * (p.sin_pitch * sinPhi + p.cos_pitch * cosPhi);
					}
				}
			}
			bx += dx;
			by += dy;
			bz += 0.0;
			// toroidal halo
			double hx = 0, hy = 0;
			if (p.use_toroidal_halo && (r * r + z * z > 1 * kJKpc * kJKpc)) {
				double bMagH = gm.e[E_HALO] * lfDisk;
				const double lfR = 1. / (1. + gm.e[E_HALO_R]);
				if (z >= 0)
					bMagH *= p.b_north * (1 - lfR);
				else
					bMagH *= p.b_south * (1 - lfR);
				hx += -bMagH * sinPhi;
				hy += bMagH * cosPhi;
			}
			bx += hx;
			by += hy;
			bz += 0.0;
			// X field
			double xx = 0, xy = 0, xz = 0;
			if (p.use_x && (r * r + z * z > 1 * kJKpc * kJKpc)) {
				double bMagX, sinThetaX, cosThetaX;
				const double rc = gm.rc, rp = gm.rp;
				if (r < rc) {
					bMagX = p.b_x * gm.e[E_X] * sq(p.r_xc / rc);
					sinThetaX = gm.sinThetaX;
					cosThetaX = gm.cosThetaX;
				} else {
					bMagX = p.b_x * gm.e[E_X] * (rp / r);
					sinThetaX = p.sin_theta_x0;
					cosThetaX = p.cos_theta_x0;
				}
				const double zsign = z < 0 ? -1 : 1;
				xx += zsign * bMagX * cosThetaX * cosPhi;
				xy += zsign * bMagX * cosThetaX * sinPhi;
				xz += bMagX * sinThetaX;
			}
			bx += xx;
			by += xy;
			bz += xz;
		}
		return v3(bx, by, bz);
	}

	// JF12Field::getTurbulentStrength (:307-331)
	__device__ __forceinline__ double turbulent_strength(const Geo &gm) const {
		if (gm.d > 20 * kJKpc)
			return 0;
		const double r = gm.r;
		double bDisk = 0;
		if (r < 5 * kJKpc) {
			bDisk = p.b_disk_turb5;
		} else {
			for (int i = 7; i >= 0; i--)
				if (gm.rn < p.r_arms[i])
					bDisk = p.b_disk_turb[i];
			bDisk *= (5 * kJKpc) / r;
		}
		bDisk *= gm.e[E_TURB_DISK];
		const double bHalo = p.b_halo_turb * gm.e[E_TURB_R] * gm.e[E_TURB_HALO];
		return __builtin_sqrt(sq(bDisk) + sq(bHalo));
	}

	// JF12Field::getField (:337-346) with the model read by three sections (jf12_eval); the turbulent term is
	// Vector3f * (float)strength in float, and every part ends 20 kpc from the centre (:230-231, 307-308).
	// AnyInterp: the turbulent grid may be read tricubic or nearest-neighbour (Grid::interpolate).
	template <bool AnyInterp, class M>
	static __device__ __forceinline__ V3 sum_parts(const V3 &pos, M &&model) {
		const bool in = !(norm(pos) > 20 * kJKpc);
		Geo gm;
		V3 r = v3(0, 0, 0);
		float strength = 0.f;
		if (in) {
			{
				const FieldJF12 f = model();
				gm = f.geo(pos);
			}
			const FieldJF12 f = model();
			if (f.p.use_striated || f.p.use_regular)
				r = f.regular(pos, gm);
			if (f.p.use_turbulent)
				strength = (float)f.turbulent_strength(gm);
		}
		double bx = 0, by = 0, bz = 0;
		const FieldJF12 f = model();
		if (f.p.use_turbulent) {
			const V3 g = AnyInterp ? grid_interpolate(f.turbulent, pos) : FieldGrid{f.turbulent}.eval(pos);
			bx += (double)((float)g.x * strength);
			by += (double)((float)g.y * strength);
			bz += (double)((float)g.z * strength);
		}
		if (f.p.use_striated) {
			const double s = 1. + f.p.sqrt_beta * (double)scalar_grid_closest(f.striated, pos);
			bx += r.x * s;
			by += r.y * s;
			bz += r.z * s;
		} else if (f.p.use_regular) {
			bx += r.x;
			by += r.y;
			bz += r.z;
		}
		return v3(bx, by, bz);
	}
	template <bool AnyInterp> __device__ __forceinline__ V3 eval_impl(const V3 &pos) const {
		return sum_parts<AnyInterp>(pos, [&]() { return *this; });
	}
	// Out of line: one copy serves the six stages of a Cash-Karp step.
	__device__ __attribute__((noinline)) V3 eval(const V3 &pos) const { return eval_impl<false>(pos); }
	__device__ float3 evalf(const V3 &pos) const {
		const V3 b = eval(pos);
		return make_float3((float)b.x, (float)b.y, (float)b.z);
	}
	// the same with a turbulent grid of any interpolation type; its own copy, so that the trilinear
	// one keeps its register allocation
	__device__ __attribute__((noinline)) V3 eval_any(const V3 &pos) const { return eval_impl<true>(pos); }
};

// JF12Field whose turbulent Grid3f is read tricubic or nearest-neighbour
struct FieldJF12Any {
	FieldJF12 f;
	__device__ __forceinline__ V3 eval(const V3 &pos) const { return f.eval_any(pos); }
	__device__ __forceinline__ float3 evalf(const V3 &pos) const {
		const V3 b = f.eval_any(pos);
		return make_float3((float)b.x, (float)b.y, (float)b.z);
	}
};

// The same fields in the propagation kernels, which read the model's hundred parameters from device memory
// through scalar loads.  As a kernel argument the model was copied to scratch, since its out-of-line
// evaluation takes an address, and every parameter came back as a 64-lane scratch load.
template <bool AnyInterp>
static __device__ __attribute__((noinline)) V3 jf12_eval(const FieldJF12 *model, const V3 pos) {
	const uint64_t a = (uint64_t)model; // the same in every lane
	const uint64_t u = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a) |
	                   (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32)) << 32;
	return FieldJF12::sum_parts<AnyInterp>(pos, [&]() {
		uint64_t v = u; // each section loads what it reads: all at once, most of it would be spilled
		asm volatile("" : "+s"(v));
		return ld_const((const FieldJF12 *)v);
	});
}
template <bool AnyInterp> struct FieldJF12Ref {
	const FieldJF12 *model;
	__device__ __forceinline__ V3 eval(const V3 &pos) const { return jf12_eval<AnyInterp>(model, pos); }
	__device__ __forceinline__ float3 evalf(const V3 &pos) const {
		const V3 b = eval(pos);
		return make_float3((float)b.x, (float)b.y, (float)b.z);
	}
};

} // namespace crp
