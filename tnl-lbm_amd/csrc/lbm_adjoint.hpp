// Adjoint (transposed Jacobian) of one A-B lattice step with the default
// cumulant collision, for the gradient of an objective with respect to the
// state and to the inflow velocity.
//
// The reference's adjoint (col_srt_adjoint.h, streaming_AB.h:246-281,
// bc.h:295-398) is for the SRT operator; this one is derived for the default
// cumulant (col_cum.h:13-511).  Key structure: the post-collision state of
// the default cumulant depends on the pre-collision populations only through
// ten raw moments (m0, j, Pi): rho and u, the second-order central moments
// (the only relaxed cumulants), and the 4th/6th-order products built from
// them.  So J^T lam = M^T (dG/dM)^T lam with M the constant 10 x 27 moment
// matrix, and (dG/dM)^T lam is one reverse sweep through the backward
// central-moment chain (27 columns of 3) and a few dozen scalar products --
// about the cost of the forward collision, so the adjoint step stays bound
// by memory traffic.
#pragma once

#include "lbm_step.hpp"

namespace lbm {

template <typename real>
struct AdjCum
{
	static constexpr int NMOM = 10;
	static LBM_DEV void raw_moments(const real* f, real* m) { raw_moments10(f, m); }

	// The backward central-moment transform of one column (k0, k1, k2) along an
	// axis of velocity v is f = V^-1 S(v) k: the shift of the central moments to
	// raw ones, m = S(v) k with
	//   m0 = k0,  m1 = k1 + v k0,  m2 = k2 + 2 v k1 + v^2 k0,
	// then f_-+ = (m2 -+ m1) / 2, f_0 = m0 - m2.  Its transpose takes
	// (lm, lz, lp) to (l0, l1, l2).
	static LBM_DEV void bwd_adj(real v, real lm, real lz, real lp, real& l0, real& l1, real& l2)
	{
		const real d = (real) 0.5 * (lp - lm);
		l2 = (real) 0.5 * (lp + lm) - lz;
		const real t = v * l2 + d;
		l0 = v * t + lz;
		l1 = v * l2 + t;
	}

	// (d f_out / d f_in)^T lam for the collision, from the raw moments of the
	// pre-collision populations, which are all the Jacobian of the default
	// cumulant depends on.  The result is mu = M^T l: `l` holds the ten
	// cotangents of the raw moments in the order of raw_moments10, and
	// for_each_mu spreads them over the populations.  rho_fixed: the caller
	// has replaced rho by 1 before the collision (OUTFLOW_RIGHT,
	// bc.h:191-194): the 4th/6th-order products then divide by 1 while u and
	// the trace keep the actual mass.  lam may be held in a narrower type than
	// the arithmetic (float fields, double sweep).
	//
	// The velocity's cotangent needs no forward recomputation of the chain:
	// S(v) = exp(v N) with N k = (0, k0, 2 k1), so d/dv of a column's output is
	// the transform applied to N k, the transforms along different axes
	// commute, and
	//   d/dv_a <lam, f_out> = <lK, N_a K>
	// with K the post-collision central moments and lK = lam pulled back
	// through all three passes.  That leaves one array of 27 values live (the
	// recomputed intermediate populations of the two earlier passes, 54
	// doubles, set the register count before) and half the operations.
	template <typename L>
	static LBM_DEV void vjp_m(const real* m, const L* lam, real Fx, real Fy, real Fz, real omega1, bool rho_fixed, real* l)
	{
		const real hx = (real) 0.5 * Fx, hy = (real) 0.5 * Fy, hz = (real) 0.5 * Fz;
		const real m0 = m[0];
		const real rv = (real) 1 / m0;
		const real vx = (m[1] + hx) * rv, vy = (m[2] + hy) * rv, vz = (m[3] + hz) * rv;
		// ---- the collision's central moments (m0 u - j = F/2 throughout) --------
		const real rk = rho_fixed ? (real) 1 : rv;
		const real om = (real) 1 - omega1;
		const real third = (real) (1.0 / 3.0);
		real a, b, c, s, p, qq;
		{
			const real k200 = m[4] - vx * (m[1] - hx), k020 = m[5] - vy * (m[2] - hy), k002 = m[6] - vz * (m[3] - hz);
			const real E33 = om * (k200 - k020), E34 = om * (k200 - k002);
			a = third * (E33 + E34 + m0);
			b = third * (-(real) 2 * E33 + E34 + m0);
			c = third * (E33 - (real) 2 * E34 + m0);
			s = om * (m[7] - vx * m[2] + vy * hx);
			p = om * (m[8] - vx * m[3] + vz * hx);
			qq = om * (m[9] - vy * m[3] + vz * hy);
		}
		const real ks211 = (a * qq + (real) 2 * p * s) * rk, ks121 = (b * p + (real) 2 * s * qq) * rk,
				   ks112 = (c * s + (real) 2 * qq * p) * rk;
		const real ks220 = (b * a + (real) 2 * s * s) * rk, ks022 = (c * b + (real) 2 * qq * qq) * rk,
				   ks202 = (a * c + (real) 2 * p * p) * rk;
		// the schedule keeps these three phases apart (moments, the passes over
		// lam, the products' reverse): mixed, their live values spill
		__builtin_amdgcn_sched_barrier(0);
		// ---- lam through the three passes, z first: cotangents lK[i][j][k] of K ---
		real lK[3][3][3];
#pragma unroll
		for (int i = 0; i < 3; i++)
#pragma unroll
			for (int j = 0; j < 3; j++)
				bwd_adj(vz, (real) lam[qidx(i, j, 0)], (real) lam[qidx(i, j, 1)], (real) lam[qidx(i, j, 2)], lK[i][j][0], lK[i][j][1],
						lK[i][j][2]);
#pragma unroll
		for (int i = 0; i < 3; i++)
#pragma unroll
			for (int k = 0; k < 3; k++)
				bwd_adj(vy, lK[i][0][k], lK[i][1][k], lK[i][2][k], lK[i][0][k], lK[i][1][k], lK[i][2][k]);
#pragma unroll
		for (int j = 0; j < 3; j++)
#pragma unroll
			for (int k = 0; k < 3; k++)
				bwd_adj(vx, lK[0][j][k], lK[1][j][k], lK[2][j][k], lK[0][j][k], lK[1][j][k], lK[2][j][k]);
		// d/dv_a: <lK, N_a K> over the columns whose K is not identically zero
		real lvx = lK[1][0][0] * m0 + lK[1][1][0] * hy + lK[1][0][1] * hz + lK[1][2][0] * b + lK[1][1][1] * qq + lK[1][0][2] * c
				 + lK[1][2][2] * ks022
				 + (real) 2 * (lK[2][0][0] * hx + lK[2][1][0] * s + lK[2][0][1] * p + lK[2][2][1] * ks121 + lK[2][1][2] * ks112);
		real lvy = lK[0][1][0] * m0 + lK[1][1][0] * hx + lK[0][1][1] * hz + lK[2][1][0] * a + lK[1][1][1] * p + lK[0][1][2] * c
				 + lK[2][1][2] * ks202
				 + (real) 2 * (lK[0][2][0] * hy + lK[1][2][0] * s + lK[0][2][1] * qq + lK[2][2][1] * ks211 + lK[1][2][2] * ks112);
		real lvz = lK[0][0][1] * m0 + lK[1][0][1] * hx + lK[0][1][1] * hy + lK[2][0][1] * a + lK[1][1][1] * s + lK[0][2][1] * b
				 + lK[2][2][1] * ks220
				 + (real) 2 * (lK[0][0][2] * hz + lK[1][0][2] * p + lK[0][1][2] * qq + lK[2][1][2] * ks211 + lK[1][2][2] * ks121);
		__builtin_amdgcn_sched_barrier(0);
		// ---- the products' reverse sweep ---------------------------------------
		// (the first-order inputs hx, hy, hz are constants: post-collision
		// k_100 = -(j_x - m0 u_x) = F_x / 2 identically)
		real lm0 = lK[0][0][0];
		real la = lK[2][0][0], lb = lK[0][2][0], lc = lK[0][0][2];
		real ls = lK[1][1][0], lp = lK[1][0][1], lqq = lK[0][1][1];
		real lks220 = lK[2][2][0], lks211 = lK[2][1][1], lks121 = lK[1][2][1], lks202 = lK[2][0][2], lks112 = lK[1][1][2];
		real lks022 = lK[0][2][2];
		const real lks222 = lK[2][2][2];
		// ks222 = Y1 rk - Y2 rk^2; lr collects rk d/d(rk) of the products
		const real Y1 = a * ks022 + b * ks202 + c * ks220 + (real) 4 * (qq * ks211 + p * ks121 + s * ks112);
		const real Y2 = (real) 16 * s * p * qq + (real) 4 * (p * p * b + qq * qq * a + s * s * c) + (real) 2 * a * b * c;
		const real lY1 = lks222 * rk, lY2 = -lY1 * rk;
		real lr = lY1 * Y1 + (real) 2 * lY2 * Y2;
		la += lY1 * ks022; lks022 += lY1 * a;
		lb += lY1 * ks202; lks202 += lY1 * b;
		lc += lY1 * ks220; lks220 += lY1 * c;
		lqq += (real) 4 * lY1 * ks211; lks211 += (real) 4 * lY1 * qq;
		lp += (real) 4 * lY1 * ks121;  lks121 += (real) 4 * lY1 * p;
		ls += (real) 4 * lY1 * ks112;  lks112 += (real) 4 * lY1 * s;
		ls += lY2 * ((real) 16 * p * qq + (real) 8 * s * c);
		lp += lY2 * ((real) 16 * s * qq + (real) 8 * p * b);
		lqq += lY2 * ((real) 16 * s * p + (real) 8 * qq * a);
		lb += lY2 * ((real) 4 * p * p + (real) 2 * a * c);
		la += lY2 * ((real) 4 * qq * qq + (real) 2 * b * c);
		lc += lY2 * ((real) 4 * s * s + (real) 2 * a * b);
		// ks_xyz = X_xyz rk
		lr += lks211 * ks211 + lks121 * ks121 + lks112 * ks112 + lks220 * ks220 + lks022 * ks022 + lks202 * ks202;
		const real l211 = lks211 * rk, l121 = lks121 * rk, l112 = lks112 * rk;
		const real l220 = lks220 * rk, l022 = lks022 * rk, l202 = lks202 * rk;
		la += l211 * qq; lqq += l211 * a; lp += (real) 2 * l211 * s; ls += (real) 2 * l211 * p;
		lb += l121 * p; lp += l121 * b; ls += (real) 2 * l121 * qq; lqq += (real) 2 * l121 * s;
		lc += l112 * s; ls += l112 * c; lqq += (real) 2 * l112 * p; lp += (real) 2 * l112 * qq;
		lb += l220 * a; la += l220 * b; ls += (real) 4 * l220 * s;
		lc += l022 * b; lb += l022 * c; lqq += (real) 4 * l022 * qq;
		la += l202 * c; lc += l202 * a; lp += (real) 4 * l202 * p;
		// a, b, c <- E33, E34, m0
		const real lE33 = third * (la - (real) 2 * lb + lc);
		const real lE34 = third * (la + lb - (real) 2 * lc);
		lm0 += third * (la + lb + lc);
		const real lk200 = om * (lE33 + lE34), lk020 = -om * lE33, lk002 = -om * lE34;
		const real lk110 = om * ls, lk101 = om * lp, lk011 = om * lqq;
		// rk = 1 / m0 unless the caller fixed rho
		lm0 -= rho_fixed ? (real) 0 : lr * rk;
		// central moments <- raw moments, velocity, mass (m0 u - j = F/2)
		lvx += (real) 2 * hx * lk200 + hy * lk110 + hz * lk101;
		lvy += (real) 2 * hy * lk020 + hx * lk110 + hz * lk011;
		lvz += (real) 2 * hz * lk002 + hx * lk101 + hy * lk011;
		const real tx = vx * lk200, ty = vy * lk020, tz = vz * lk002;
		lm0 += vx * (tx + vy * lk110 + vz * lk101) + vy * (ty + vz * lk011) + vz * tz;
		// u = (j + F/2) / m0
		const real ux = lvx * rv, uy = lvy * rv, uz = lvz * rv;
		const real ljx = ux - (real) 2 * tx - vy * lk110 - vz * lk101;
		const real ljy = uy - (real) 2 * ty - vx * lk110 - vz * lk011;
		const real ljz = uz - (real) 2 * tz - vx * lk101 - vy * lk011;
		lm0 -= ux * vx + uy * vy + uz * vz;
		l[0] = lm0; l[1] = ljx; l[2] = ljy; l[3] = ljz; l[4] = lk200; l[5] = lk020; l[6] = lk002; l[7] = lk110; l[8] = lk101;
		l[9] = lk011;
	}

	// mu = M^T l, the raw moments being linear in the populations: put(q, mu_q)
	// for every q, by (c_x, c_y) columns of one base and one z-odd part.
	template <typename Put>
	static LBM_DEV void for_each_mu(const real* l, Put&& put)
	{
#pragma unroll
		for (int i = 0; i < 3; i++)
#pragma unroll
			for (int j = 0; j < 3; j++) {
				real e = l[0], o = l[3];
				if (i != 1) {
					e += i == 2 ? l[4] + l[1] : l[4] - l[1];
					o += i == 2 ? l[8] : -l[8];
				}
				if (j != 1) {
					e += j == 2 ? l[5] + l[2] : l[5] - l[2];
					o += j == 2 ? l[9] : -l[9];
				}
				if (i != 1 && j != 1)
					e += i == j ? l[7] : -l[7];
				const real ez = e + l[6];
				put(qidx(i, j, 0), ez - o);
				put(qidx(i, j, 1), e);
				put(qidx(i, j, 2), ez + o);
			}
	}

	// gradient with respect to u of sum_q lam_q feq_q(1, u), feq = D3Q27_EQ_INV_CUM
	template <int c>
	static LBM_DEV real phi(real v)
	{
		if constexpr (c == 0)
			return (real) 3 * v * v - (real) 2;
		else if constexpr (c > 0)
			return (real) 3 * v * v + (real) 3 * v + (real) 1;
		else
			return (real) 3 * v * v - (real) 3 * v + (real) 1;
	}
	template <int c>
	static LBM_DEV real dphi(real v)
	{
		return (real) 6 * v + (real) (3 * c);
	}
	template <int q, typename L>
	static LBM_DEV void eq_grad_q(const L* lam, real vx, real vy, real vz, real& gx, real& gy, real& gz)
	{
		constexpr int nz = (CX[q] != 0) + (CY[q] != 0) + (CZ[q] != 0);
		constexpr double coef = nz == 0 ? -1.0 / 27.0 : nz == 1 ? 1.0 / 54.0 : nz == 2 ? -1.0 / 108.0 : 1.0 / 216.0;
		const real w = (real) coef * (real) lam[q];
		const real px = phi<CX[q]>(vx), py = phi<CY[q]>(vy), pz = phi<CZ[q]>(vz);
		gx += w * dphi<CX[q]>(vx) * py * pz;
		gy += w * px * dphi<CY[q]>(vy) * pz;
		gz += w * px * py * dphi<CZ[q]>(vz);
	}
	template <int q = 0, typename L>
	static LBM_DEV void eq_grad(const L* lam, real vx, real vy, real vz, real& gx, real& gy, real& gz)
	{
		if constexpr (q < 27) {
			eq_grad_q<q>(lam, vx, vy, vz, gx, gy, gz);
			eq_grad<q + 1>(lam, vx, vy, vz, gx, gy, gz);
		}
	}
};

// adjoint arrays of one step
struct AdjPtrs
{
	const void* lam_next;  // adjoint of the state the forward step wrote (27 XYZ)
	void* lam;             // adjoint of the state the forward step read (27 XYZ, output)
	double* grad;          // d/d(inflow velocity), 3 x (Y Z) indexed Y z + y, accumulated; or null
	const void* tape;      // raw moments recorded by the forward step (tape_index layout), or null
};

// One thread per site.  Pass SPECIAL = false writes, for every site and q, the
// site's contribution to the slot it would pull from under periodic wrapping
// (that map is a bijection, so every output slot is written exactly once:
// plain stores, no clearing); slots that the site really pulls from somewhere
// else (array-edge clamps of non-periodic sites, OUTFLOW_RIGHT's pull from
// x-1, NOTHING sites that pull nothing) get 0 there.  Pass SPECIAL = true then
// adds those contributions to the slots actually pulled, atomically.
// The faces of the box [0,X)x[0,Y)x[0,Z), each site once: x faces whole,
// then the y faces of the interior x, then the z faces of the interior x and
// y.  Only face sites can pull from a source other than the periodic wrap
// (non-periodic neighbour indices clamp at the array edge), and OUTFLOW_RIGHT
// belongs on the x = X-1 face.
inline uint64_t shell_count(int64_t X, int64_t Y, int64_t Z)
{
	const uint64_t fx = X > 1 ? 2 : 1, fy = Y > 1 ? 2 : 1, fz = Z > 1 ? 2 : 1;
	const uint64_t ix = X > 2 ? X - 2 : 0, iy = Y > 2 ? Y - 2 : 0;
	return fx * Y * Z + ix * fy * Z + ix * iy * fz;
}

LBM_DEV bool shell_coords(const StepArgs& A, int64_t& x, int64_t& z, int64_t& y)
{
	uint64_t i = (uint64_t) blockIdx.x * blockDim.x + threadIdx.x;
	const uint64_t X = A.X, Y = A.Y, Z = A.Z;
	const uint64_t fx = X > 1 ? 2 : 1, fy = Y > 1 ? 2 : 1, fz = Z > 1 ? 2 : 1;
	const uint64_t ix = X > 2 ? X - 2 : 0, iy = Y > 2 ? Y - 2 : 0;
	const uint64_t n1 = fx * Y * Z, n2 = ix * fy * Z, n3 = ix * iy * fz;
	if (i < n1) {
		const uint64_t r = i % (Y * Z);
		x = i / (Y * Z) ? (int64_t) X - 1 : 0;
		z = (int64_t) (r / Y);
		y = (int64_t) (r % Y);
		return true;
	}
	i -= n1;
	if (i < n2) {
		const uint64_t r = i % (fy * Z);
		x = 1 + (int64_t) (i / (fy * Z));
		z = (int64_t) (r / fy);
		y = r % fy ? (int64_t) Y - 1 : 0;
		return true;
	}
	i -= n2;
	if (i < n3) {
		const uint64_t r = i % (iy * fz);
		x = 1 + (int64_t) (i / (iy * fz));
		y = 1 + (int64_t) (r / fz);
		z = r % fz ? (int64_t) Z - 1 : 0;
		return true;
	}
	return false;
}

// Whether the periodic-wrap slot of direction q differs from the slot the
// site really pulls from, as a bit per direction.  Per axis a pull towards -1
// or +1 is irregular where the wrap and the clamp differ (a non-periodic site
// on that face of the box); OUTFLOW_RIGHT pulls c_x = 0 and -1 from x - 1.
constexpr uint32_t dir_mask(int axis, int c)
{
	uint32_t m = 0;
	for (int q = 0; q < 27; q++)
		if ((axis == 0 ? CX[q] : axis == 1 ? CY[q] : CZ[q]) == c)
			m |= 1u << q;
	return m;
}
LBM_DEV uint32_t irregular_pulls(bool per, bool right, int32_t x, int32_t y, int32_t z, int32_t X, int32_t Y, int32_t Z)
{
	uint32_t m = 0;
	if (! per) {
		m |= x == 0 && X > 1 ? dir_mask(0, 1) : 0;
		m |= x == X - 1 && X > 1 && ! right ? dir_mask(0, -1) : 0;
		m |= y == 0 && Y > 1 ? dir_mask(1, 1) : 0;
		m |= y == Y - 1 && Y > 1 ? dir_mask(1, -1) : 0;
		m |= z == 0 && Z > 1 ? dir_mask(2, 1) : 0;
		m |= z == Z - 1 && Z > 1 ? dir_mask(2, -1) : 0;
	}
	if (right) {
		m |= x > 0 ? dir_mask(0, 0) : 0;
		m |= X > 2 || x < X - 1 ? dir_mask(0, -1) : 0;
	}
	return m;
}

// rank of q among the directions with its c_y
constexpr int y_rank(int q)
{
	int k = 0;
	for (int r = 0; r < q; r++)
		k += CY[r] == CY[q];
	return k;
}

// Wall sites of the y faces.  A y face is strided in memory, so the second pass
// touches a cache line for every one of a wall's nine irregular pulls, reading and
// adding (with them 32 us in a 256x96x96 duct, float fields, without 16; the first
// pass 145 and 134).  The slots meant are those
// that the site one row in owns, and it is the next lane: the wall hands its nine
// values to that lane through LDS, and the second pass leaves the wall out.  That
// is done where the wall's pulls are irregular in y alone, the site one row in is
// an ordinary one, and both are in one wave.
LBM_DEV bool inner_xz(const StepArgs& A, int64_t x, int64_t z)
{
	return A.Y >= 3 && x > 0 && x < A.X - 1 && z > 0 && z < A.Z - 1;
}
LBM_DEV bool collides(int16_t gi)
{
	return gi == GEO_FLUID || gi == GEO_PERIODIC;
}
// whether the wall (x, y, z) hands them over; lane: its lane in the first pass
LBM_DEV bool wall_gives(const StepArgs& A, int64_t x, int64_t y, int64_t z, uint32_t lane, int16_t before, int16_t after)
{
	return inner_xz(A, x, z) && ((y == 0 && lane < 63 && collides(after)) || (y == A.Y - 1 && lane > 0 && collides(before)));
}

// SPECIAL = false: every site, plain stores to the slots it owns under the
// periodic wrap (0 for slots whose true reader is elsewhere).  SPECIAL = true:
// the face sites only, atomic adds of those contributions to their true
// sources, after the first pass.
//
// P32: one x plane of a population array holds at most 4 GiB.  A block lies in
// one x plane in every mapping, so the first pass addresses a slot as a
// wave-uniform base (array, direction and x plane) plus a 32-bit per-lane
// offset within the plane.
//
// Bound: HBM, then FP64 issue (about 500 FP64 instructions a site).  Four
// waves per SIMD (at most 128 VGPRs; from an FP64 state, whose 27 pulled values
// meet the 27 of lambda, three): 256x96x96 duct, float fields and recording,
// 164 -> 145 us (134 with the walls handed over, 4.5 TB/s) against the sweep that recomputed the chain's
// intermediate populations at 256 VGPRs and two waves.
template <int ST, bool SPECIAL, int TAPE = 0, bool P32 = false>
__global__ void __launch_bounds__(256, (TAPE == 0 && ST == TNL_LBM_STORE_F64) ? 3 : 4) k_adjoint_ab(const StepArgs A, const AdjPtrs P)
{
	using S = Storage<ST>;
	using real = typename S::real;
	using elem = typename S::elem;
	using D = AdjCum<real>;
	// lambda in the element type where it is narrower than the arithmetic
	// (float fields with a double sweep): fewer registers
	using lreal = std::conditional_t<(sizeof(elem) < sizeof(real)), elem, real>;
	int64_t x, z, y;
	if (SPECIAL ? ! shell_coords(A, x, z, y) : ! block_coords(A, x, z, y))
		return;
	const int64_t s0 = (x * A.Zs + z) * A.Ys + y;
	const int16_t gi = A.map ? A.map[s0] : (int16_t) GEO_PERIODIC;
	const bool per = gi == GEO_PERIODIC;
	const uint32_t irregular = gi == GEO_NOTHING ? (1u << 27) - 1
												 : irregular_pulls(per, gi == GEO_OUTFLOW_RIGHT, (int32_t) x, (int32_t) y, (int32_t) z,
																   (int32_t) A.X, (int32_t) A.Y, (int32_t) A.Z);
	if (SPECIAL && (gi == GEO_NOTHING || irregular == 0))
		return;
	// the slot of direction q at (xs, ys, zs); xs is wave-uniform in the first
	// pass except for the pulls
	auto slot_at = [&](auto* base, int q, int64_t xs, int64_t ys, int64_t zs) {
		if constexpr (P32 && ! SPECIAL)
			return at(base + (q * A.XYZ + xs * A.Zs * A.Ys), (uint32_t) zs * (uint32_t) A.Ys + (uint32_t) ys);
		else
			return base + (q * A.XYZ + (xs * A.Zs + zs) * A.Ys + ys);
	};
	const elem* __restrict__ Ln = (const elem*) P.lam_next;
	elem* __restrict__ L = (elem*) P.lam;
	if (SPECIAL && (gi == GEO_WALL || gi == GEO_INFLOW)) {
		// bounce-back: mu_q = lam_next[opp(q)], read only for the irregular directions
		// (the face sites are one per cache line here); inflow: mu = 0
		if (gi == GEO_WALL) {
			if ((y == 0 || y == A.Y - 1) && inner_xz(A, x, z)) {
				const uint32_t lane = ((A.lin ? (uint32_t) z * (uint32_t) A.Y : 0u) + (uint32_t) y) & 63u;
				const int16_t in = A.map[y == 0 ? s0 + 1 : s0 - 1];
				if (wall_gives(A, x, y, z, lane, in, in))
					return;
			}
			const Nb NX = neighbours<false>(x, A.X, 0, false, false);
			const Nb NY = neighbours<false>(y, A.Y, 0, false, false);
			const Nb NZ = neighbours<false>(z, A.Z, 0, false, false);
#pragma unroll
			for (int q = 0; q < 27; q++)
				if ((irregular >> q) & 1u)
					atomicAdd(slot_at(L, q, NX[-CX[q]], NY[-CY[q]], NZ[-CZ[q]]), (elem) S::ld(Ln + opp(q) * A.XYZ + s0));
		}
		return;
	}
	const bool on_shell = x == 0 || x == A.X - 1 || y == 0 || y == A.Y - 1 || z == 0 || z == A.Z - 1;
	// an irregular pull away from the faces (OUTFLOW_RIGHT inside the box) has no fix-up: poison it
	const bool unsupported = gi != GEO_NOTHING && irregular != 0 && ! on_shell;

	lreal lam[27];
#pragma unroll
	for (int q = 0; q < 27; q++)
		lam[q] = (lreal) S::ld(slot_at(Ln, q, x, y, z));
	// what the walls of the y faces hand to the next lane (wall_gives)
	__shared__ lreal given[SPECIAL ? 1 : 9][SPECIAL ? 1 : 256];
	bool from_before = false, from_after = false;
	if constexpr (! SPECIAL) {
		const uint32_t lane = threadIdx.x & 63u;
		const int16_t before = (int16_t) __shfl_up((int) gi, 1), after = (int16_t) __shfl_down((int) gi, 1);
		const bool inner = inner_xz(A, x, z) && collides(gi);
		from_before = inner && y == 1 && lane > 0 && before == GEO_WALL;
		from_after = inner && y == A.Y - 2 && lane < 63 && after == GEO_WALL;
		if (gi == GEO_WALL && wall_gives(A, x, y, z, lane, before, after)) {
#pragma unroll
			for (int q = 0; q < 27; q++)
				if (CY[q] != 0 && (CY[q] > 0) == (y == 0))
					given[y_rank(q)][threadIdx.x] = lam[opp(q)];
		}
		// (one wave: its LDS accesses are in order; the compiler must keep them so)
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
		__builtin_amdgcn_wave_barrier();
	}
	// raw moments of the pulled populations: from the state, or recorded by the
	// forward step (read at every site, used where the forward step wrote them)
	Nb PX, NY, NZ;
	if (SPECIAL || TAPE == 0) {
		PX = neighbours<false>(x, A.X, 0, false, per);
		NY = neighbours<false>(y, A.Y, 0, false, per);
		NZ = neighbours<false>(z, A.Z, 0, false, per);
		if (gi == GEO_OUTFLOW_RIGHT)
			PX.p = PX.o = PX.m;
	}
	real m[D::NMOM];
	if constexpr (TAPE == 0) {
		const elem* F = (const elem*) A.df0;
		real f[27];
#pragma unroll
		for (int q = 0; q < 27; q++)
			f[q] = S::ld(F + (q * A.XYZ + (PX[-CX[q]] * A.Zs + NZ[-CZ[q]]) * A.Ys + NY[-CY[q]]));
		D::raw_moments(f, m);
	}
	else {
		using TT = std::conditional_t<TAPE == 2, double, float>;
		const TT* tp = (const TT*) P.tape;
#pragma unroll
		for (int k = 0; k < D::NMOM; k++)
			m[k] = (real) tp[tape_index(k, s0)];
	}

	const Nb WX = neighbours<false>(x, A.X, 0, false, true);
	const Nb WY = neighbours<false>(y, A.Y, 0, false, true);
	const Nb WZ = neighbours<false>(z, A.Z, 0, false, true);
	// mu_q of this site to its slot: a plain store in the first pass (0 where
	// the true reader is elsewhere), an atomic add in the second
	auto put = [&](int q, real v) {
		const bool irr = (irregular >> q) & 1u;
		if constexpr (SPECIAL) {
			if (irr)
				atomicAdd(slot_at(L, q, PX[-CX[q]], NY[-CY[q]], NZ[-CZ[q]]), (elem) v);
		}
		else
			S::st(slot_at(L, q, WX[-CX[q]], WY[-CY[q]], WZ[-CZ[q]]), irr && ! unsupported ? (real) 0 : v);
	};
	if ((gi == GEO_FLUID || gi == GEO_PERIODIC || gi == GEO_OUTFLOW_RIGHT) && ! unsupported) {
		real l[D::NMOM];
		D::vjp_m(m, lam, (real) A.fx, (real) A.fy, (real) A.fz, (real) A.omega1, gi == GEO_OUTFLOW_RIGHT, l);
		if (! SPECIAL && irregular == 0) {
			real wb[9], wa[9];
#pragma unroll
			for (int k = 0; k < 9; k++)
				wb[k] = wa[k] = 0;
			if (from_before)
#pragma unroll
				for (int k = 0; k < 9; k++)
					wb[k] = (real) given[k][threadIdx.x - 1];
			if (from_after)
#pragma unroll
				for (int k = 0; k < 9; k++)
					wa[k] = (real) given[k][threadIdx.x + 1];
			D::for_each_mu(l, [&](int q, real v) {
				const real w = CY[q] > 0 ? v + wb[y_rank(q)] : CY[q] < 0 ? v + wa[y_rank(q)] : v;
				S::st(slot_at(L, q, WX[-CX[q]], WY[-CY[q]], WZ[-CZ[q]]), w);
			});
		}
		else
			D::for_each_mu(l, put);
	}
	else if (gi == GEO_WALL && ! unsupported) {
#pragma unroll
		for (int q = 0; q < 27; q++)
			put(q, (real) lam[opp(q)]);
	}
	else if (gi == GEO_OUTFLOW_EQ && ! unsupported) {
		// f_out = feq(1, u(f_in)), u = (j + F/2) / m0
		const real rv = (real) 1 / m[0];
		const real ux = (m[1] + (real) 0.5 * (real) A.fx) * rv, uy = (m[2] + (real) 0.5 * (real) A.fy) * rv,
				   uz = (m[3] + (real) 0.5 * (real) A.fz) * rv;
		real gx = 0, gy = 0, gz = 0;
		D::eq_grad(lam, ux, uy, uz, gx, gy, gz);
#pragma unroll
		for (int q = 0; q < 27; q++)
			put(q, (gx * ((real) CX[q] - ux) + gy * ((real) CY[q] - uy) + gz * ((real) CZ[q] - uz)) * rv);
	}
	else {
		if (gi == GEO_INFLOW && ! unsupported && ! SPECIAL && P.grad) {
			const int64_t iy = A.Y * z + y;
			const real ux = (real) inflow_component(A, 0, iy);
			const real uy = (real) inflow_component(A, 1, iy);
			const real uz = (real) inflow_component(A, 2, iy);
			real gx = 0, gy = 0, gz = 0;
			D::eq_grad(lam, ux, uy, uz, gx, gy, gz);
			const int64_t n = A.Y * A.Z;
			atomicAdd(P.grad + iy, (double) gx);
			atomicAdd(P.grad + n + iy, (double) gy);
			atomicAdd(P.grad + 2 * n + iy, (double) gz);
		}
		// inlet sites (f_out does not depend on the state) and NOTHING sites: 0;
		// a geometry code without an adjoint, or an irregular pull without a
		// fix-up, makes the result unusable, visibly
		const bool none = gi == GEO_NOTHING || (gi == GEO_INFLOW && ! unsupported);
		const real v = none ? (real) 0 : (real) __builtin_nan("");
#pragma unroll
		for (int q = 0; q < 27; q++)
			put(q, v);
	}
}

// ===========================================================================
// Adjoint of the D3Q7 part of one coupled A-B step (ade_site), for a given
// velocity field: the passive scalar does not act on the flow, and the D3Q7
// collision is linear in the populations for a given u (SRT, MRT and CLBM
// relax moments whose equilibria are linear in phi), so
//   lambda <- C(u)^T lambda_next scattered back along the pull,
//   dJ/dS  += sum_q w_q lambda_next_q at the sites that collide.
// C(u)^T is applied directly (Ade7::collide_adjoint: each operator is the
// identity or a multiple of it plus a few rank-one terms).
// ===========================================================================
struct AdeAdjArgs
{
	const void* u;          // vx, vy, vz planes (XYZ each) of the step's velocity, macro_real
	const void* lam_next;   // 7 XYZ of the compute type
	void* lam;              // 7 XYZ, output
	double* grad_source;    // XYZ, accumulated, or null
	const int16_t* map;     // D3Q7 codes, or null (all periodic)
	const void* diff;       // per-site diffusivity (macro_real) or null
	double D;
	int32_t collision;
};

template <int ST, bool SPECIAL>
__global__ void __launch_bounds__(256) k_ade_adjoint_ab(const StepArgs A, const AdeAdjArgs P)
{
	using K = Ade7<ST>;
	using real = typename K::real;
	int64_t x, z, y;
	if (SPECIAL ? ! shell_coords(A, x, z, y) : ! block_coords(A, x, z, y))
		return;
	const int64_t s0 = (x * A.Zs + z) * A.Ys + y;
	// the pull uses the NSE site's periodicity, as in the coupled kernel
	const int16_t gn = A.map ? A.map[s0] : (int16_t) GEO_PERIODIC;
	const bool per = gn == GEO_PERIODIC;
	const int16_t ga = P.map ? P.map[s0] : (int16_t) A_PERIODIC;
	const Nb NX = neighbours<false>(x, A.X, 0, false, per);
	const Nb NY = neighbours<false>(y, A.Y, 0, false, per);
	const Nb NZ = neighbours<false>(z, A.Z, 0, false, per);
	Nb PX = NX;
	if (ga == A_OUTFLOW_RIGHT)
		PX.p = PX.o = NX.m;
	const Nb WX = neighbours<false>(x, A.X, 0, false, true);
	const Nb WY = neighbours<false>(y, A.Y, 0, false, true);
	const Nb WZ = neighbours<false>(z, A.Z, 0, false, true);
	auto sidx = [&](int64_t xs, int64_t ys, int64_t zs) { return (xs * A.Zs + zs) * A.Ys + ys; };
	uint32_t irregular = 0;
#pragma unroll
	for (int q = 0; q < 7; q++) {
		const bool same = PX[-CX[q]] == WX[-CX[q]] && NY[-CY[q]] == WY[-CY[q]] && NZ[-CZ[q]] == WZ[-CZ[q]];
		if (ga == A_NOTHING || ! same)
			irregular |= 1u << q;
	}
	if (SPECIAL && (ga == A_NOTHING || irregular == 0))
		return;
	const real* Ln = (const real*) P.lam_next;
	real* L = (real*) P.lam;
	if (SPECIAL && (ga == A_WALL || ga == A_INFLOW)) {
#pragma unroll
		for (int q = 0; q < 7; q++)
			if (ga == A_WALL && ((irregular >> q) & 1u))
				atomicAdd(L + q * A.XYZ + sidx(PX[-CX[q]], NY[-CY[q]], NZ[-CZ[q]]), Ln[opp(q) * A.XYZ + s0]);
		return;
	}
	const bool on_shell = x == 0 || x == A.X - 1 || y == 0 || y == A.Y - 1 || z == 0 || z == A.Z - 1;
	const bool unsupported = ga != A_NOTHING && irregular != 0 && ! on_shell;
	real mu[7];
	if (ga == A_NOTHING || unsupported) {
		const real v = unsupported ? (real) __builtin_nan("") : (real) 0;
#pragma unroll
		for (int q = 0; q < 7; q++)
			mu[q] = v;
	}
	else {
		real lam[7];
#pragma unroll
		for (int q = 0; q < 7; q++)
			lam[q] = Ln[q * A.XYZ + s0];
		switch (ga) {
			case A_FLUID:
			case A_PERIODIC:
			case A_SOLID:
			case A_OUTFLOW_RIGHT:
				{
					auto macro_at = [&](const void* p, int64_t i) -> real {
						return A.macro_f64 ? (real) ((const double*) p)[i] : (real) ((const float*) p)[i];
					};
					const real vx = macro_at(P.u, s0), vy = macro_at(P.u, A.XYZ + s0), vz = macro_at(P.u, 2 * A.XYZ + s0);
					const real D = P.diff ? macro_at(P.diff, s0) : (real) P.D;
					K::collide_adjoint(P.collision, lam, mu, vx, vy, vz, D);
					if (! SPECIAL && P.grad_source) {
						real g = 0;
#pragma unroll
						for (int q = 0; q < 7; q++)
							g += (real) w7(q) * lam[q];
						P.grad_source[s0] += (double) g;
					}
					break;
				}
			case A_WALL:
#pragma unroll
				for (int q = 0; q < 7; q++)
					mu[q] = lam[opp(q)];
				break;
			case A_INFLOW:
#pragma unroll
				for (int q = 0; q < 7; q++)
					mu[q] = 0;
				break;
			default:
#pragma unroll
				for (int q = 0; q < 7; q++)
					mu[q] = (real) __builtin_nan("");
				break;
		}
	}
	if (! SPECIAL) {
#pragma unroll
		for (int q = 0; q < 7; q++) {
			const real v = (irregular >> q) & 1u && ! unsupported ? (real) 0 : mu[q];
			L[q * A.XYZ + sidx(WX[-CX[q]], WY[-CY[q]], WZ[-CZ[q]])] = v;
		}
	}
	else {
#pragma unroll
		for (int q = 0; q < 7; q++)
			if ((irregular >> q) & 1u)
				atomicAdd(L + q * A.XYZ + sidx(PX[-CX[q]], NY[-CY[q]], NZ[-CZ[q]]), mu[q]);
	}
}

// the D3Q7 adjoint step (built in lbm_adjoint.hip)
int launch_ade_adjoint(const tnl_lbm_config* cfg, const StepArgs& A, const AdeAdjArgs& P, unsigned threads,
					   unsigned grid, hipStream_t st);

// both passes of one adjoint step (built in lbm_adjoint.hip); tape_kind 0:
// Jacobian from the state df0, 1: from a float tape, 2: from a double tape
int launch_adjoint(const tnl_lbm_config* cfg, const StepArgs& A, const AdjPtrs& P, int tape_kind, unsigned threads,
				   unsigned grid, hipStream_t st);
// one A-B step of the default cumulant that records the raw moments in A.tape
int launch_record(const tnl_lbm_config* cfg, const StepArgs& A, int tape_kind, unsigned threads, unsigned grid,
				  hipStream_t st);
// the same with F32 storage and a float recording, pulling from the FP64
// populations A.df0 (256x96x96 duct: 217 us, against 185 for the conversion of
// the state and 137 for the step on it)
int launch_record_from_f64(const StepArgs& A, unsigned threads, unsigned grid, hipStream_t st);

}  // namespace lbm
