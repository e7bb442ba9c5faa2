// Device side of the D3Q27 step shared by the library's translation units:
// kernel arguments, the periodic A-A fast kernel, the general (map + BC)
// kernel, the coupled NSE + ADE kernel, initialisation / transfer /
// reduction kernels, and the launch template.  See lbm_d3q27.hip for the
// design notes and the C ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "lbm_ade.hpp"
#include "lbm_device.hpp"

namespace lbm {

// host-side error reporting (defined in lbm_d3q27.hip)
int hip_check(hipError_t e, const char* what);

// Whether the kernels that can address a population array of at most 4 GiB
// as a per-direction base plus a 32-bit offset may do so; false while
// tnl_lbm_set_wide_addressing(1) holds (defined in lbm_d3q27.hip).
bool narrow_slots_allowed();

// a population array of XYZ elements of `elem` bytes takes 32-bit slot offsets
inline bool narrow_slots(int64_t XYZ, size_t elem)
{
	return narrow_slots_allowed() && (uint64_t) XYZ * elem <= (1ull << 32);
}

// ---------------------------------------------------------------------------
struct StepArgs
{
	void* df0;
	void* df1;
	void* macro;
	const int16_t* map;
	int64_t XYZ;
	int64_t X, Y, Z;     // sizes without overlaps
	int64_t ox, oy, oz;  // overlaps
	int64_t Ys, Zs;      // stored extents Y+2oy, Z+2oz
	uint64_t plane_bytes;  // XYZ * sizeof(element): byte stride between population planes
	float rs[4], invr[4];  // fixed-point form per direction class: R_n / 32767 and 1 / R_n
	// fixed-point form per weight class n = |c_q|^2 (w_n = (2/3)^(3-n) / 6^n):
	// decode w_n R / 32767, encode 1 / (w_n R) times the fast collision's
	// 2^-n output factor
	float cls_sc[4], cls_inv[4];
	int32_t offx, offy, offz;
	int32_t nx, ny, nz;
	uint32_t nyb;      // y segments per row (linear mapping: blocks per x plane)
	uint32_t nblocks;  // logical blocks
	uint32_t group, span;  // which logical blocks belong to one XCD (block_of)
	int32_t backwards;  // the blocks in falling order
	int32_t lin;       // linear y-z mapping (see linearize)
	// the even A-A step over one contiguous range of stored sites (flat_range)
	int32_t flat;
	int64_t flat0, nflat;  // its first site and length
	int32_t even;
	int32_t out_macro;
	int32_t macro_f64;
	int32_t dist_x, dist_y, dist_z;
	double omega1;
	double nu;  // lbmViscosity (MRT_LES and KBC use it directly)
	double fx, fy, fz;
	double inflow[3];
	const void* prof[3];  // inflow profiles: double arrays, or float where prof_f32
	int32_t prof_f32;
	const void* force;  // per-site force: 3 planes of macro elements (macro_f64), or null
	void* tape;  // moment recording of the A-B step (10 planes of XYZ), or null
	// a launch over one row list (tnl_lbm_classify_rows): the listed (x, z)
	// rows of the box, each entry x << 16 | z; null = the box itself
	const uint32_t* rows;
	uint32_t nrows;
	// host side: the three lists of a full-box step (classes 0, 1, 2 one
	// after another), or null
	const uint32_t* lists;
	int64_t list_count[3];
	int32_t others;  // listed launches: the sites of other codes than the plain ones only
};

enum : int16_t
{
	GEO_FLUID = 0, GEO_WALL, GEO_INFLOW, GEO_INFLOW_LEFT, GEO_INFLOW_BB_LEFT, GEO_INFLOW_EQ_LEFT, GEO_OUTFLOW_EQ,
	GEO_OUTFLOW_RIGHT, GEO_OUTFLOW_RIGHT_INTERP, GEO_PERIODIC, GEO_NOTHING, GEO_SYM_TOP, GEO_SYM_BOTTOM, GEO_SYM_LEFT,
	GEO_SYM_RIGHT, GEO_SYM_BACK, GEO_SYM_FRONT
};


// the codes of most sites: collide and stream, or bounce back
LBM_DEV bool plain(int16_t gi)
{
	return gi == GEO_FLUID || gi == GEO_PERIODIC || gi == GEO_WALL;
}
LBM_DEV bool plain_scalar(int16_t ga)
{
	return ga == A_FLUID || ga == A_PERIODIC || ga == A_WALL;
}

constexpr int NXCD = 8;

// Workgroups go to the XCDs in turn.  Groups of 2^A.group consecutive logical
// blocks belong to one XCD, so that its L2 serves the lines that neighbouring
// waves share, and the groups go to the XCDs in turn, so that all of them work
// on one range of each population plane.  With an eighth of the grid for each XCD
// the step streamed through 8 ranges of 27 (A-B: 54) planes at once, on most
// sizes at 5 to 20% less bandwidth.  Steps in one process on one buffer, an
// eighth each / groups of 1 / 8 / 32 / 256 blocks: 48x320x320 FP64 slab 964 / 803 /
// 794 / 789 / 817 us; 256x96x96 mixed gradient 15.1 / 12.5 / 12.3 / 12.3 / 12.5 ms;
// 301x417x333 F32_DEV box 4359 / - / 3498 / 3477 / 3480 us; 512^3 FP64 box 18.95 /
// 22.9 / 19.05 / 18.90 / 18.81 ms (singly, the XCDs fetch each other's lines).
// (block_of: groups of 2^group blocks with span = 2^group; one run of `span` blocks
// for each XCD with group = 31)
__host__ __device__ __forceinline__ uint32_t block_of(uint32_t b, uint32_t group, uint32_t span)
{
	const uint32_t k = b / NXCD;
	return ((k >> group) * NXCD + b % NXCD) * span + (k & ((1u << group) - 1u));
}
LBM_DEV uint32_t logical_block(const StepArgs& A)
{
	const uint32_t L = block_of(blockIdx.x, A.group, A.span);
	return A.backwards && L < A.nblocks ? A.nblocks - 1u - L : L;
}
// bytes of the step's population arrays
inline uint64_t population_bytes(const StepArgs& A)
{
	return (A.df1 ? 54u : 27u) * A.plane_bytes;
}
constexpr uint64_t LLC_BYTES = 256ull << 20;  // last-level cache
// Whether steps that run in alternating order find enough of the arrays in the
// last-level cache: five times its size at most.
inline bool alternating(uint64_t bytes)
{
	return bytes <= 5 * LLC_BYTES;
}
// A-B arrays with planes of exactly 8 or 16 MiB (128^3 FP32 and FP64, 256^2 x 64 and
// 128 F16): the same range of all 54 planes meets in the same memory channels, so a
// step whose XCDs work side by side on one range waits for those.  An eighth of the
// grid to each XCD and hints instead.  Two steps, side by side / so: 128^3 FP64 354 /
// 337 us, MRT 365 / 339, FP32 187 / 180; 64x256x256 F16 197 / 181; coupled 128^3 FP64
// 460 / 439.  (32 MiB planes 658 / 687, 12 and 20 MiB 266 / 285 and 436 / 474, 15.875
// MiB 377 / 427, 4 MiB within the cache.)
inline bool planes_meet(const StepArgs& A)
{
	return A.df1 && (A.plane_bytes == 8ull << 20 || A.plane_bytes == 16ull << 20);
}
// The grid for A.nblocks logical blocks.  Smaller groups where there would be
// fewer than 16 for each XCD: the last ones keep one XCD busy alone (128x64x64,
// groups of 1024: 208 us a pair of steps, of 32: 90).
//
// Where the arrays fit half the last-level cache, an eighth of the grid to each XCD
// instead, in one order: its L2 then still holds (a part of) what it stepped before,
// and no range of memory is short of bandwidth.  A pair of steps, eighths / groups:
// 48^3 FP64 25 / 30 us; F16 70^3 28 / 34; beyond the L2 caches' 32 MB F32 A-B duct
// 50x60x55 (36 MB) 26.5 / 32, F32 box 70^3 (37) 31 / 35, FP64 A-B 61x77x53 (108)
// 43.6 / 45.4; from there to the cache's size equal.  Runs of the same length for all
// XCDs: with powers of two, some of them idle (48x61x53 FP64 coupled A-A 57 us and
// 45, 30x300x30 F16 32 and 26).
//
// Where they do not, but are no more than some times the last-level cache, odd
// steps run through the blocks backwards: they begin where the step before ended,
// with what that cache still holds, while in one order each step evicts what it
// would need next.  One process and buffer, without / with: 189x233x43 FP64 A-A duct
// 370 / 302 us, 262x85x95 FP64 coupled 561 / 477, 301x187x129 F16 channel 398 / 362,
// 243x205x157 F32_DEV box 682 / 625, 150x90x96 FP64 A-B duct 220 / 201.
inline uint32_t padded_blocks(StepArgs& A, uint32_t group = 5)
{
	if (population_bytes(A) <= LLC_BYTES / 2 || planes_meet(A)) {
		A.backwards = 0;
		A.group = 31;
		A.span = (A.nblocks + NXCD - 1) / NXCD;
		return NXCD * A.span;
	}
	A.backwards = ! A.even && alternating(population_bytes(A));
	while (group > 0 && ((uint64_t) NXCD << group) * 16 > A.nblocks)
		group--;
	A.group = group;
	A.span = 1u << group;
	const uint32_t whole = (uint32_t) NXCD << group;
	return (A.nblocks + whole - 1) / whole * whole;
}

// One x plane of a population array of `elem`-byte elements takes 32-bit offsets.
// plane_fits alone decides for the kernels that have no other form (lean, linear odd
// step): the addressing switch chooses between the forms of one kernel only.
inline bool plane_fits(const StepArgs& A, size_t elem)
{
	return (uint64_t) A.Ys * (uint64_t) A.Zs * elem <= (1ull << 32);
}
inline bool narrow_planes(const StepArgs& A, size_t elem)
{
	return narrow_slots_allowed() && plane_fits(A, elem);
}

// per-site force of MACRO::computeForcing (kernels.h:103): added to the
// homogeneous force of copyQuantities (macro.h:80-86) in the arithmetic of
// the collision
template <typename real>
LBM_DEV void add_site_force(const StepArgs& A, int64_t s, real& Fx, real& Fy, real& Fz)
{
	if (A.macro_f64) {
		const double* F = (const double*) A.force;
		Fx += (real) F[s];
		Fy += (real) F[A.XYZ + s];
		Fz += (real) F[2 * A.XYZ + s];
	}
	else {
		const float* F = (const float*) A.force;
		Fx += (real) F[s];
		Fy += (real) F[A.XYZ + s];
		Fz += (real) F[2 * A.XYZ + s];
	}
}

// component k of the inflow velocity at profile index i = Y z + y
// (NSE_Data_InflowProfile::vel_*, lbm_data.h:104-125; the constant of
// NSE_Data_ConstInflow where no profile is given)
LBM_DEV double inflow_component(const StepArgs& A, int k, int64_t i)
{
	if (! A.prof[k])
		return A.inflow[k];
	return A.prof_f32 ? (double) static_cast<const float*>(A.prof[k])[i] : static_cast<const double*>(A.prof[k])[i];
}

// logical block -> (x, z, y segment) with XCD-aware remapping
// LIN = false: whole rows only (x and z stay uniform per block, as the
// periodic kernel's scalar addressing needs)
// LIST: a launch over a row list (A.rows); a compile-time choice, since
// coordinates that may come from either source are per-lane values in both
// (the coupled kernel's registers rose from 109 to 133 with a run-time one)
template <bool LIN = true, bool LIST = false>
LBM_DEV bool block_coords(const StepArgs& A, int64_t& x, int64_t& z, int64_t& y)
{
	const uint32_t L = logical_block(A);
	if (L >= A.nblocks)
		return false;
	if constexpr (LIST) {
		// a row list: whole rows per block, or the listed rows' sites one
		// after another (linear mapping)
		uint32_t k, yy;
		if (LIN && A.lin) {
			const uint32_t i = L * blockDim.x + threadIdx.x;
			k = i / (uint32_t) A.ny;
			if (k >= A.nrows)
				return false;
			yy = i % (uint32_t) A.ny;
		}
		else {
			k = L / A.nyb;
			yy = (L % A.nyb) * blockDim.x + threadIdx.x;
			if (yy >= (uint32_t) A.ny)
				return false;
		}
		const uint32_t r = A.rows[k];
		x = (int64_t) (r >> 16);
		z = (int64_t) (r & 0xffffu);
		y = (int64_t) yy;
		return x < A.X && z < A.Z;
	}
	if (LIN && A.lin) {
		// consecutive lanes walk the y-z plane of one x, row after row
		const uint32_t i = (L % A.nyb) * blockDim.x + threadIdx.x;
		x = A.offx + (int64_t) (L / A.nyb);
		if (i >= (uint32_t) A.ny * (uint32_t) A.nz)
			return false;
		z = A.offz + (int64_t) (i / (uint32_t) A.ny);
		y = A.offy + (int64_t) (i % (uint32_t) A.ny);
		return true;
	}
	const uint32_t yb = L % A.nyb;
	const uint32_t t = L / A.nyb;
	z = A.offz + (int64_t) (t % (uint32_t) A.nz);
	x = A.offx + (int64_t) (t / (uint32_t) A.nz);
	y = A.offy + (int64_t) yb * blockDim.x + threadIdx.x;
	return y < A.offy + A.ny;
}

// the box's sites with the mapping chosen at compile time
template <bool LIN>
LBM_DEV bool box_coords(const StepArgs& A, int64_t& x, int64_t& z, int64_t& y)
{
	const uint32_t L = logical_block(A);
	if (L >= A.nblocks)
		return false;
	if constexpr (LIN) {
		const uint32_t i = (L % A.nyb) * blockDim.x + threadIdx.x;
		x = A.offx + (int64_t) (L / A.nyb);
		z = A.offz + (int64_t) (i / (uint32_t) A.ny);
		y = A.offy + (int64_t) (i % (uint32_t) A.ny);
		return i < (uint32_t) A.ny * (uint32_t) A.nz;
	}
	const uint32_t t = L / A.nyb;
	z = A.offz + (int64_t) (t % (uint32_t) A.nz);
	x = A.offx + (int64_t) (t / (uint32_t) A.nz);
	y = A.offy + (int64_t) (L % A.nyb) * blockDim.x + threadIdx.x;
	return y < A.offy + A.ny;
}

template <typename E>
LBM_DEV E* at(E* base, uint32_t i)
{
	// uniform 64-bit base + 32-bit per-lane byte offset (global saddr form)
	return (E*) ((char*) base + (uint32_t) (i * (uint32_t) sizeof(E)));
}

template <typename real>
LBM_DEV void write_macro(const StepArgs& A, int64_t s, real rho, real vx, real vy, real vz)
{
	if (A.macro_f64) {
		double* m = (double*) A.macro;
		m[s] = rho;
		m[A.XYZ + s] = vx;
		m[2 * A.XYZ + s] = vy;
		m[3 * A.XYZ + s] = vz;
	}
	else {
		float* m = (float*) A.macro;
		m[s] = (float) rho;
		m[A.XYZ + s] = (float) vx;
		m[2 * A.XYZ + s] = (float) vy;
		m[3 * A.XYZ + s] = (float) vz;
	}
}

// COLL::collision after computeDensityAndVelocity, in the reference's operation order
template <int ST, int COLL>
LBM_DEV void collide(typename Storage<ST>::real* f, typename Storage<ST>::real rho, typename Storage<ST>::real vx,
					 typename Storage<ST>::real vy, typename Storage<ST>::real vz, const StepArgs& A,
					 typename Storage<ST>::real Fx, typename Storage<ST>::real Fy, typename Storage<ST>::real Fz)
{
	using P = Phys<ST>;
	using real = typename Storage<ST>::real;
	const real omega1 = (real) A.omega1;
	if constexpr (Storage<ST>::dev)
		P::cumulant(f, rho, vx, vy, vz, omega1);
	else if constexpr (COLL == TNL_LBM_COLL_CUM)
		P::template cumulant<false, false>(f, rho, vx, vy, vz, omega1);
	else if constexpr (COLL == TNL_LBM_COLL_CUM_2017)
		P::template cumulant<true, false>(f, rho, vx, vy, vz, omega1);
	else if constexpr (COLL == TNL_LBM_COLL_CUM_2017_ANTIALIAS)
		P::template cumulant<true, true>(f, rho, vx, vy, vz, omega1);
	else if constexpr (COLL == TNL_LBM_COLL_MRT_LES)
		P::mrt(f, rho, vx, vy, vz, (real) A.nu);
	else {
		// KBC_N1..N4 = 4..7, KBC_C1..C4 = 8..11: shear part D, D+T, D+Q, D+T+Q
		constexpr int k = (COLL - TNL_LBM_COLL_KBC_N1) % 4;
		constexpr bool central = COLL >= TNL_LBM_COLL_KBC_C1;
		P::template kbc<central, k == 1 || k == 3, k >= 2>(f, rho, vx, vy, vz, (real) A.nu, Fx, Fy, Fz);
	}
}

// ===========================================================================
// Fast path: A-A pattern, every site GEO_PERIODIC (no map).
// Even step (streaming_AA.h:81-84, 16-45): read own slots, write opposite.
// Odd step (streaming_AA.h:86-115, 46-75): pull from r - c_q (opposite
// slot), push to r + c_q (same slot).
// Addresses: base + plane[q] (kernel argument, scalar) + row (scalar) + y
// (per lane), one vector add per access.  The even step streams with
// nontemporal hints; so do the odd step's accesses in the site's own y,
// while its +-1 shifted rows share cache lines between neighbouring waves
// and keep the default policy.
// ===========================================================================
template <int ST, int COLL>
constexpr bool fast_collision = std::is_same<typename Storage<ST>::real, float>::value && COLL == TNL_LBM_COLL_CUM;

// Collision slot of the streaming-only measurement kernel
// (tnl_lbm_d3q27_stream_only): the identity, so that the periodic kernels
// move the populations of free streaming with the step's own loads, stores
// and addressing, and time the memory traffic of the access pattern alone.
constexpr int COLL_STREAM_ONLY = 1000;

// number of non-zero components of c_q (the weight class of q)
constexpr int ncls(int q)
{
	return (CX[q] != 0) + (CY[q] != 0) + (CZ[q] != 0);
}

// Factor applied to a post-collision value before its (non-fixed-point)
// store: the fast collision leaves population q scaled by 2^n(q).
template <int ST, int COLL>
constexpr float out_factor(int q)
{
	return fast_collision<ST, COLL> ? FastCum<Storage<ST>::dev>::unscale(q) : 1.0f;
}

template <int ST, int COLL>
LBM_DEV void collide_site(typename Storage<ST>::real* f, const StepArgs& A, typename Storage<ST>::real Fx,
						  typename Storage<ST>::real Fy, typename Storage<ST>::real Fz, typename Storage<ST>::real& rho,
						  typename Storage<ST>::real& vx, typename Storage<ST>::real& vy, typename Storage<ST>::real& vz)
{
	using real = typename Storage<ST>::real;
	if constexpr (COLL == COLL_STREAM_ONLY) {
		rho = vx = vy = vz = 0;
	}
	else if constexpr (fast_collision<ST, COLL>) {
		FastCum<Storage<ST>::dev>::collide(f, Fx, Fy, Fz, (real) A.omega1, true, rho, vx, vy, vz);
	}
	else {
		Phys<ST>::density_velocity(f, Fx, Fy, Fz, rho, vx, vy, vz);
		collide<ST, COLL>(f, rho, vx, vy, vz, A, Fx, Fy, Fz);
	}
}
template <int ST, int COLL>
LBM_DEV void collide_site(typename Storage<ST>::real* f, const StepArgs& A, typename Storage<ST>::real& rho,
						  typename Storage<ST>::real& vx, typename Storage<ST>::real& vy, typename Storage<ST>::real& vz)
{
	using real = typename Storage<ST>::real;
	collide_site<ST, COLL>(f, A, (real) A.fx, (real) A.fy, (real) A.fz, rho, vx, vy, vz);
}

// Full-way bounce-back (bc.h:201-221) of loaded populations, times the power of
// two that encode_all takes off again.
template <int ST, int COLL>
LBM_DEV void bounce_back(typename Storage<ST>::real* f)
{
	using real = typename Storage<ST>::real;
#pragma unroll
	for (int q = 1; q < 27; q += 2) {
		const real t = f[q] * (real) (1.0f / out_factor<ST, COLL>(q));
		f[q] = f[q + 1] * (real) (1.0f / out_factor<ST, COLL>(q));
		f[q + 1] = t;
	}
}

// Post-collision populations to their stored form: put(q, element) in turn
// (the fixed-point form converts two per instruction).
template <int ST, int COLL, typename Put>
LBM_DEV void encode_all(const typename Storage<ST>::real* f, const StepArgs& A, Put&& put)
{
	using S = Storage<ST>;
	using elem = typename S::elem;
	if constexpr (S::fixed) {
#pragma unroll
		for (int q = 0; q < 27; q += 2) {
			const int q1 = q + 1 < 27 ? q + 1 : q;
			const auto r = __builtin_amdgcn_cvt_pknorm_i16(f[q] * A.cls_inv[ncls(q)], f[q1] * A.cls_inv[ncls(q1)]);
			put(q, (elem) r[0]);
			if (q + 1 < 27)
				put(q1, (elem) r[1]);
		}
	}
	else {
#pragma unroll
		for (int q = 0; q < 27; q++) {
			elem v;
			S::st(&v, f[q] * out_factor<ST, COLL>(q));
			put(q, v);
		}
	}
}

// Keeps `p` in scalar registers and makes everything derived from it depend
// on `v`: the store addresses are then formed after the collision instead of
// being hoisted above it (which would keep 27 scalar pairs live and spill).
template <bool PIN, typename T>
LBM_DEV char* after(char* p, const T& v)
{
	if constexpr (PIN) {
		auto g = (__attribute__((address_space(1))) char*) p;
		asm volatile("" : "+s"(g) : "v"(v));
		return (char*) g;
	}
	return p;
}

// Build-time tuning knobs (defaults are the measured best on MI355X):
//  LBM_NT_EVEN   bitmask over storage forms: nontemporal hints on the even
//                step, where every wave's access covers whole lines
//  LBM_PIN_ADDR  bitmask over storage forms: scalar base pointers, even step
//  LBM_NT_ODD    bitmask over storage forms: nontemporal hints on the odd
//                step's accesses within the site's own y (c_y = 0); the +-1
//                shifted rows share lines with the neighbouring wave through
//                L2 and keep the default policy (with hints they measured 40%
//                slower)
//  LBM_PIN_ODD   bitmask over storage forms: scalar base pointers, odd step
//                (F16 / BF16 odd step at 512^3, one allocation: -3.8% / -1.3%
//                time; HBM writes above the algorithmic bytes +2.8% -> +0.8% /
//                +5.2% -> +1.7%)
//  LBM_WAVES_F64 minimum waves per SIMD requested for the FP64 kernels
#ifndef LBM_NT_EVEN
#define LBM_NT_EVEN 0x3f
#endif
#ifndef LBM_PIN_ADDR
#define LBM_PIN_ADDR 0x3f
#endif
#ifndef LBM_NT_ODD
#define LBM_NT_ODD 0x3f
#endif
//  LBM_NT_GENERAL bitmask over storage forms: the same hints in the map kernel
#ifndef LBM_NT_GENERAL
#define LBM_NT_GENERAL 0x3f
#endif
#ifndef LBM_PIN_ODD
#define LBM_PIN_ODD 0x3f
#endif
//  LBM_TPB_FP32  block size of the periodic odd step for the FP32-compute forms
//                where the row length is a multiple of it: a 512-site row in
//                one block keeps 7 of its 8 wave boundaries, whose +-1 shifted
//                lines the neighbouring waves share, on one CU (measured +0.6
//                to +1.2 points at 512^3); and of the even step's flat range
#ifndef LBM_TPB_FP32
#define LBM_TPB_FP32 512
#endif
#ifndef LBM_WAVES_F64
#define LBM_WAVES_F64 1
#endif
//  LBM_PAIR_EVEN bitmask over the 2-byte storage forms: two sites per lane
//                on the even step (k_aa_even_pair)
#ifndef LBM_PAIR_EVEN
#define LBM_PAIR_EVEN 0x38
#endif
#ifndef LBM_MAXWAVES_F64
#define LBM_MAXWAVES_F64 3
#endif

// Pins a wave-uniform pointer (base + plane + row) in scalar registers, so
// that each access is one global load/store with a scalar base and a 32-bit
// per-lane offset; left to itself the compiler adds the shared per-lane part
// first and then pays a 64-bit vector add per access.
// (The pinned copy is a global-address-space pointer: a plain pointer that
// has passed through the asm would make every access a flat one.)
template <bool PIN>
LBM_DEV char* sptr(char* p)
{
	if constexpr (PIN) {
		auto g = (__attribute__((address_space(1))) char*) p;
		asm volatile("" : "+s"(g));
		return (char*) g;
	}
	return p;
}

// The arrays of the directions in turn: two scalar additions each, where the
// multiples of the stride, formed afresh for every access so as not to stay live,
// took six: 548 -> 378 scalar instructions a wave, coupled 256^3 F16 1009 -> 986 us for
// two steps, equal where HBM alone bounds the step.
template <typename E, bool PIN = true>
struct Planes
{
	char* p;
	uint64_t pb;
	LBM_DEV Planes(const void* base, uint64_t stride) : p((char*) base), pb(stride) {}
	LBM_DEV E* next()
	{
		E* r = (E*) p;
		p = sptr<PIN>(p + pb);
		return r;
	}
};

// Site of a lane of the even step: the stored offset of its block's row or
// range (wave-uniform) and its own offset from there.  The even step moves
// nothing between sites, so where the launch covers whole rows and columns of
// a lattice without y and z overlaps, its sites are one contiguous range of
// every population plane (A.flat): blocks take it in order, every wave is
// full whatever the row length, and the planes' alignment alone decides
// whether a wave's accesses cover whole lines.  `per` sites per lane.
LBM_DEV bool even_site(const StepArgs& A, uint32_t per, uint64_t& row, uint32_t& yl)
{
	const uint32_t L = logical_block(A);
	if (L >= A.nblocks)
		return false;
	if (A.flat) {
		const uint64_t first = (uint64_t) L * (blockDim.x * per);
		row = (uint64_t) A.flat0 + first;
		yl = threadIdx.x * per;
		return first + yl < (uint64_t) A.nflat;
	}
	const uint32_t t = L / A.nyb;
	const int64_t z = A.offz + (int64_t) (t % (uint32_t) A.nz);
	const int64_t x = A.offx + (int64_t) (t / (uint32_t) A.nz);
	const uint32_t i = ((L % A.nyb) * blockDim.x + threadIdx.x) * per;
	row = (uint64_t) (((x + A.ox) * A.Zs + (z + A.oz)) * A.Ys);
	yl = (uint32_t) (A.offy + A.oy) + i;
	return i < (uint32_t) A.ny;
}

// NTE: nontemporal hints, taken where every wave's accesses cover whole 128-byte
// lines (even_launch).  A partial line written with the hint goes to memory by
// itself instead of meeting its other half in L2: (301, 187, 129) F64 985 us
// with the hints and 707 without, F32 (200, 100, 400) 578 and 303; with whole
// lines they gain 2% (F64) to 10% (F16) at 512^3.
// MAP: the step of a lattice with a geometry map, at its plain sites (FLUID,
// PERIODIC and WALL; sites of any other code are left to the general kernel).
// A wall site's even step is the identity: the bounce-back swaps q and opp(q)
// and the store swaps them back.  Waves of walls alone leave theirs; in other
// waves the walls store what they loaded, since a gap would leave partial lines.

// (no map: a box with a force field alone, every site PERIODIC)
LBM_DEV int16_t code_at(const StepArgs& A, int64_t s)
{
	return A.map ? A.map[s] : (int16_t) GEO_PERIODIC;
}
// whether the site collides (a wall keeps its populations)
LBM_DEV bool even_active(const StepArgs& A, int64_t s)
{
	const int16_t gi = code_at(A, s);
	return gi == GEO_FLUID || gi == GEO_PERIODIC;
}
LBM_DEV void wall_macro(const StepArgs& A, int64_t s, bool f64)
{
	if (A.out_macro && code_at(A, s) == GEO_WALL) {
		if (f64)
			write_macro(A, s, 1.0, 0.0, 0.0, 0.0);
		else
			write_macro(A, s, 1.0f, 0.0f, 0.0f, 0.0f);
	}
}

template <int ST, int COLL, bool NTE, bool MAP = false>
__global__ void __launch_bounds__(ST == TNL_LBM_STORE_F64 ? 256 : LBM_TPB_FP32)
__attribute__((amdgpu_waves_per_eu(ST == TNL_LBM_STORE_F64 ? LBM_WAVES_F64 : 1, ST == TNL_LBM_STORE_F64 ? LBM_MAXWAVES_F64 : 8)))
k_aa_even(const StepArgs A)
{
	using S = Storage<ST>;
	using real = typename S::real;
	using elem = typename S::elem;
	constexpr uint32_t E = sizeof(elem);
	constexpr bool NT = NTE && ((LBM_NT_EVEN >> ST) & 1);
	constexpr bool PIN = (LBM_PIN_ADDR >> ST) & 1;
	uint64_t first;
	uint32_t yl;
	if (! even_site(A, 1, first, yl))
		return;
	bool wall = false;
	if constexpr (MAP) {
		const int16_t gi = code_at(A, (int64_t) first + yl);
		wall = gi == GEO_WALL;
		const bool moves = gi == GEO_FLUID || gi == GEO_PERIODIC;
		const uint64_t any = __ballot(moves);
		if (! (moves || (wall && any))) {
			wall_macro(A, (int64_t) first + yl, ST == TNL_LBM_STORE_F64);
			return;
		}
	}
	char* __restrict__ df = (char*) A.df0;
	const uint64_t pb = A.plane_bytes;
	const uint64_t row = first * E;
	const uint32_t yb = yl * E;
	real f[27];
#pragma unroll
	for (int q = 0; q < 27; q++) {
		const elem* p = (const elem*) (sptr<PIN>(df + ((uint64_t) q * pb + row)) + yb);
		const elem v = NT ? ld_nt(p) : *p;
		f[q] = S::ld(&v, A.cls_sc[ncls(q)]);
	}
	real rho = 1, vx = 0, vy = 0, vz = 0;
	if constexpr (MAP) {
		real Fx = (real) A.fx, Fy = (real) A.fy, Fz = (real) A.fz;
		if (A.force)
			add_site_force(A, (int64_t) first + yl, Fx, Fy, Fz);
		if (wall)
			bounce_back<ST, COLL>(f);
		if (! wall)
			collide_site<ST, COLL>(f, A, Fx, Fy, Fz, rho, vx, vy, vz);
	}
	else
		collide_site<ST, COLL>(f, A, rho, vx, vy, vz);
	char* out = after<PIN>(df, f[26]);
	uint32_t ob = yb;
	if constexpr (MAP)
		asm volatile("" : "+v"(ob));  // in this block, for the scalar-base form
	encode_all<ST, COLL>(f, A, [&](int q, elem e) {
		elem* p = (elem*) (sptr<PIN>(out + ((uint64_t) opp(q) * pb + row)) + ob);
		if (NT)
			st_nt(p, e);
		else
			*p = e;
	});
	if (A.out_macro)
		write_macro(A, (int64_t) first + yl, rho, vx, vy, vz);
}

// LIN: consecutive lanes walk the y-z plane of one x, row after row, so that a
// row length that is not a multiple of the wave still fills every wave; x
// stays wave-uniform, z becomes a per-lane row offset.  Otherwise a block is a
// segment of one row and the row offsets are scalars.
// NTO: nontemporal hints on the c_y = 0 accesses.
template <int ST, int COLL, bool NTO, bool LIN>
__global__ void __launch_bounds__(ST == TNL_LBM_STORE_F64 ? 256 : LBM_TPB_FP32)
__attribute__((amdgpu_waves_per_eu(ST == TNL_LBM_STORE_F64 ? LBM_WAVES_F64 : 1, ST == TNL_LBM_STORE_F64 ? LBM_MAXWAVES_F64 : 8)))
k_aa_odd(const StepArgs A)
{
	using S = Storage<ST>;
	using real = typename S::real;
	using elem = typename S::elem;
	constexpr uint32_t E = sizeof(elem);
	constexpr bool PIN_ODD = (LBM_PIN_ODD >> ST) & 1;
	constexpr bool NT_ODD = NTO && ((LBM_NT_ODD >> ST) & 1);
	int64_t x, z, y;
	if (! box_coords<LIN>(A, x, z, y))
		return;
	char* __restrict__ df = (char*) A.df0;
	const uint64_t pb = A.plane_bytes;
	real f[27];
	const uint32_t yl = (uint32_t) (y + A.oy);
	// periodic neighbours (kernelInitIndices, kernels.h:21-28)
	const int64_t xp = (! A.dist_x && x == A.X - 1) ? 0 : x + 1;
	const int64_t xm = (! A.dist_x && x == 0) ? A.X - 1 : x - 1;
	const int64_t zp = (! A.dist_z && z == A.Z - 1) ? 0 : z + 1;
	const int64_t zm = (! A.dist_z && z == 0) ? A.Z - 1 : z - 1;
	const uint32_t ypl = (uint32_t) (((! A.dist_y && y == A.Y - 1) ? 0 : y + 1) + A.oy);
	const uint32_t yml = (uint32_t) (((! A.dist_y && y == 0) ? A.Y - 1 : y - 1) + A.oy);
	const int64_t xs[3] = {xm + A.ox, x + A.ox, xp + A.ox};
	const int64_t zs[3] = {zm + A.oz, z + A.oz, zp + A.oz};
	const uint32_t ys[3] = {yml * E, yl * E, ypl * E};
	// scalar part and per-lane part of a slot's byte offset in its plane
	// (LIN: one x plane holds at most 4 GiB, odd_launch)
	uint64_t xrow[3];
	uint32_t zrow[3];
#pragma unroll
	for (int k = 0; k < 3; k++) {
		xrow[k] = (uint64_t) (xs[k] * A.Zs * A.Ys) * E;
		zrow[k] = (uint32_t) zs[k] * (uint32_t) A.Ys * E;
	}
	auto slot_of = [&](char* plane, int cx, int cy, int cz) {
		if constexpr (LIN)
			return (elem*) (sptr<PIN_ODD>(plane + xrow[1 + cx]) + (zrow[1 + cz] + ys[1 + cy]));
		else {
			const uint64_t row = (uint64_t) ((xs[1 + cx] * A.Zs + zs[1 + cz]) * A.Ys) * E;
			return (elem*) (sptr<PIN_ODD>(plane + row) + ys[1 + cy]);
		}
	};
	// The 2-byte forms in rows take the arrays in order: where the last-level cache or
	// a fast allocation serves them, their issue bounds the step (one odd step, pairs'
	// order / this: 256x256x64 F16 82 / 76 us, 256x256x100 134 / 129, 1024x512x512 I16
	// 5050 / 4990; 512^3 F16, both steps, 4986 / 4835); on slower allocations of large
	// boxes it is up to 1.2% slower (200x512x300 F16 628 / 635, 512^3 2870 / 2895).  The
	// wider forms, which HBM bounds alone, and the linear mapping keep the pairs'
	// order, up to 0.7% faster there.
	constexpr bool WALK = ! LIN && E == 2;
	Planes<char, PIN_ODD> in(df, pb);
#pragma unroll
	for (int k = 0; k < 27; k++) {
		const int q = WALK ? opp(k) : k;
		const elem* p = slot_of(WALK ? in.next() : df + (uint64_t) opp(q) * pb, -CX[q], -CY[q], -CZ[q]);
		if (NT_ODD && CY[q] == 0) {
			const elem v = ld_nt(p);
			f[q] = S::ld(&v, A.cls_sc[ncls(q)]);
		}
		else
			f[q] = S::ld(p, A.cls_sc[ncls(q)]);
	}
	real rho, vx, vy, vz;
	collide_site<ST, COLL>(f, A, rho, vx, vy, vz);
	Planes<char, PIN_ODD> out(after<PIN_ODD>(df, f[26]), pb);
	encode_all<ST, COLL>(f, A, [&](int q, elem v) {
		elem* p = slot_of(WALK ? out.next() : out.p + (uint64_t) q * pb, CX[q], CY[q], CZ[q]);
		if (NT_ODD && CY[q] == 0)
			st_nt(p, v);
		else
			*p = v;
	});
	if (A.out_macro)
		write_macro(A, (xs[1] * A.Zs + zs[1]) * A.Ys + yl, rho, vx, vy, vz);
}

// ===========================================================================
// Paired even step for the 2-byte storage forms (the A-A even step above).
// Each lane updates the two sites y, y + 1 of a row (y even) and moves both
// through one aligned 4-byte access per population, site y in the low half:
// half the memory instructions per site.  The host uses it where Y, oy, offy,
// ny and XYZ are even.  (The odd step keeps one site per lane: its +-1
// shifted pairs would need 2-byte aligned 4-byte accesses, which measured
// slower than the single 2-byte accesses they replace.)
// ===========================================================================
template <int ST, int COLL>
struct PairCodec
{
	using S = Storage<ST>;
	using elem = typename S::elem;
	static_assert(sizeof(elem) == 2, "pairs of 2-byte elements");
	static LBM_DEV float get(uint32_t h, int q, const StepArgs& A)
	{
		if constexpr (S::fixed)
			return (float) (int16_t) (uint16_t) h * A.cls_sc[ncls(q)];
		else
			return (float) __builtin_bit_cast(elem, (uint16_t) h);
	}
	static LBM_DEV uint32_t put(float v, int q, const StepArgs& A)
	{
		if constexpr (S::fixed)
			return (uint16_t) __builtin_amdgcn_cvt_pknorm_i16(v * A.cls_inv[ncls(q)], 0.0f)[0];
		else
			return __builtin_bit_cast(uint16_t, (elem) (v * out_factor<ST, COLL>(q)));
	}
	// forms whose conversion packs two values at once
	static constexpr bool PACK2 = S::fixed || std::is_same<elem, __bf16>::value;
	// the value the conversion takes, and the packed pair (lo = site y)
	static LBM_DEV float scaled(float v, int q, const StepArgs& A)
	{
		if constexpr (S::fixed)
			return v * A.cls_inv[ncls(q)];
		else
			return v * out_factor<ST, COLL>(q);
	}
	static LBM_DEV uint32_t pack2(float lo, float hi)
	{
		if constexpr (S::fixed)
			return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pknorm_i16(lo, hi));
		else {
			typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
			const bf16x2 v = {(__bf16) lo, (__bf16) hi};
			return __builtin_bit_cast(uint32_t, v);
		}
	}
};

// Collides the pair held in w[] in place: site s (low halves), then s + 1.
// For the float forms site s's outputs replace the low halves while the
// high halves still hold site s + 1's inputs, so one packed array serves
// both sites (binary16 writes a half and keeps the other in one
// instruction).
// (MAP: a site that does not collide, `lo` or `hi` false, writes no macros here)
template <int ST, int COLL, bool MAP = false>
LBM_DEV void collide_pair(uint32_t* w, const StepArgs& A, int64_t s, bool lo = true, bool hi = true)
{
	using C = PairCodec<ST, COLL>;
	float f[27];
	float rho, vx, vy, vz;
	auto site = [&](int64_t i, bool on) {
		float Fx = (float) A.fx, Fy = (float) A.fy, Fz = (float) A.fz;
		if (MAP && A.force)
			add_site_force(A, i, Fx, Fy, Fz);
		collide_site<ST, COLL>(f, A, Fx, Fy, Fz, rho, vx, vy, vz);
		if (A.out_macro && (! MAP || on))
			write_macro(A, i, rho, vx, vy, vz);
	};
	if constexpr (C::PACK2) {
		// I16 and BF16 convert two values per instruction: site s's scaled
		// outputs wait as floats, in the registers its decoded inputs held,
		// and one conversion packs both sites, with no per-half merges
		// (I16: 1001 -> 947 VALU per pair).
		float a[27];
#pragma unroll
		for (int q = 0; q < 27; q++)
			f[q] = C::get(w[q] & 0xffffu, q, A);
		site(s, lo);
#pragma unroll
		for (int q = 0; q < 27; q++)
			a[q] = C::scaled(f[q], q, A);
#pragma unroll
		for (int q = 0; q < 27; q++)
			f[q] = C::get(w[q] >> 16, q, A);
		site(s + 1, hi);
#pragma unroll
		for (int q = 0; q < 27; q++)
			w[q] = C::pack2(a[q], C::scaled(f[q], q, A));
		return;
	}
#pragma unroll
	for (int q = 0; q < 27; q++)
		f[q] = C::get(w[q] & 0xffffu, q, A);
	site(s, lo);
#pragma unroll
	for (int q = 0; q < 27; q++)
		w[q] = (w[q] & 0xffff0000u) | C::put(f[q], q, A);
#pragma unroll
	for (int q = 0; q < 27; q++)
		f[q] = C::get(w[q] >> 16, q, A);
	site(s + 1, hi);
#pragma unroll
	for (int q = 0; q < 27; q++)
		w[q] = (w[q] & 0xffffu) | (C::put(f[q], q, A) << 16);
}

// MAP as in k_aa_even: a lane with one site that collides stores that half.
template <int ST, int COLL, bool NTE, bool MAP = false>
__global__ void __launch_bounds__(256) k_aa_even_pair(const StepArgs A)
{
	constexpr bool NT = NTE && ((LBM_NT_EVEN >> ST) & 1);
	constexpr bool PIN = (LBM_PIN_ADDR >> ST) & 1;
	uint64_t first;
	uint32_t yl;  // sites yl, yl + 1 from `first` on
	if (! even_site(A, 2, first, yl))
		return;
	char* __restrict__ df = (char*) A.df0;
	const uint64_t pb = A.plane_bytes;
	const uint64_t row = first * 2;
	const uint32_t yb = yl * 2;
	bool lo = true, hi = true;
	if constexpr (MAP) {
		lo = even_active(A, (int64_t) first + yl);
		hi = even_active(A, (int64_t) first + yl + 1);
		if (! lo && ! hi) {
			wall_macro(A, (int64_t) first + yl, false);
			wall_macro(A, (int64_t) first + yl + 1, false);
			return;
		}
	}
	uint32_t w[27];
#pragma unroll
	for (int q = 0; q < 27; q++) {
		const uint32_t* p = (const uint32_t*) (sptr<PIN>(df + ((uint64_t) q * pb + row)) + yb);
		w[q] = NT ? __builtin_nontemporal_load(p) : *p;
	}
	collide_pair<ST, COLL, MAP>(w, A, (int64_t) (row / 2) + yl, lo, hi);
	if constexpr (MAP) {
		if (! (lo && hi)) {
			// one plain site of the pair: its half only
			wall_macro(A, (int64_t) first + yl + (lo ? 1 : 0), false);
			uint32_t ob = lo ? yb : yb + 2;
			asm volatile("" : "+v"(ob));
#pragma unroll
			for (int q = 0; q < 27; q++)
				*(uint16_t*) (sptr<PIN>(after<PIN>(df, w[q]) + ((uint64_t) opp(q) * pb + row)) + ob)
					= (uint16_t) (lo ? w[q] : w[q] >> 16);
			return;
		}
	}
	// The stores use the loads' lane offset, kept opaque: when the compiler
	// sees the two equal it shares 64-bit lane pointers between loads and
	// stores and drops both out of the scalar-base (saddr) form.  Each store's
	// base is pinned after its value is final (one base after the last value
	// left 64-bit vector adds on every store).
	uint32_t ob = yb;
	asm volatile("" : "+v"(ob));
#pragma unroll
	for (int q = 0; q < 27; q++) {
		uint32_t* p = (uint32_t*) ((char*) sptr<PIN>(after<PIN>(df, w[q]) + ((uint64_t) opp(q) * pb + row)) + ob);
		if (NT)
			__builtin_nontemporal_store(w[q], p);
		else
			*p = w[q];
	}
}

// ===========================================================================
// General path: geometry map + D3Q27_BC_All, A-A or A-B.
// ===========================================================================
struct Nb
{
	int64_t m, o, p;  // storage coordinates (overlap-shifted) of c = -1, 0, +1
	LBM_DEV int64_t operator[](int c) const { return c < 0 ? m : (c > 0 ? p : o); }
};

// kernelInitIndices (kernels.h:5-57).  A-A indices of non-periodic sites
// that would leave the stored array wrap instead (the reference reads
// outside its allocation there).
template <bool AA>
LBM_DEV Nb neighbours(int64_t c, int64_t n, int64_t o, bool dist, bool periodic)
{
	int64_t p, m;
	if (periodic) {
		p = (! dist && c == n - 1) ? 0 : c + 1;
		m = (! dist && c == 0) ? n - 1 : c - 1;
	}
	else if (AA) {
		p = c + 1 < n + o ? c + 1 : 0;
		m = c - 1 >= -o ? c - 1 : n - 1;
	}
	else {
		p = c + 1 < n - 1 + o ? c + 1 : n - 1 + o;
		m = c - 1 > -o ? c - 1 : -o;
	}
	return Nb{m + o, c + o, p + o};
}

// Moment recording layout: blocks of 64 consecutive sites, each holding its
// 10 moments as 10 runs of 64 values, so that one wave writes (and the
// adjoint reads) one contiguous 2560-element stretch instead of 10 planes.
__host__ __device__ inline int64_t tape_index(int k, int64_t s)
{
	return ((s >> 6) * 10 + k) * 64 + (s & 63);
}

// The raw moments m0, j, Pi of 27 populations, in one summation order shared
// by the step's moment recording and the adjoint that reads it back.
template <typename real>
LBM_DEV void raw_moments10(const real* f, real* m)
{
	real m0 = 0, jx = 0, jy = 0, jz = 0, Pxx = 0, Pyy = 0, Pzz = 0, Pxy = 0, Pxz = 0, Pyz = 0;
#pragma unroll
	for (int q = 0; q < 27; q++) {
		const real v = f[q];
		m0 += v;
		if (CX[q]) { jx += CX[q] > 0 ? v : -v; Pxx += v; }
		if (CY[q]) { jy += CY[q] > 0 ? v : -v; Pyy += v; }
		if (CZ[q]) { jz += CZ[q] > 0 ? v : -v; Pzz += v; }
		if (CX[q] * CY[q]) Pxy += CX[q] * CY[q] > 0 ? v : -v;
		if (CX[q] * CZ[q]) Pxz += CX[q] * CZ[q] > 0 ? v : -v;
		if (CY[q] * CZ[q]) Pyz += CY[q] * CZ[q] > 0 ? v : -v;
	}
	m[0] = m0; m[1] = jx; m[2] = jy; m[3] = jz; m[4] = Pxx; m[5] = Pyy; m[6] = Pzz; m[7] = Pxy; m[8] = Pxz; m[9] = Pyz;
}

// Slot q of the site at storage coordinates (xs, ys, zs), and of site s:
// with O32, the array of direction q as a wave-uniform base, pinned in scalar
// registers, plus a 32-bit per-lane byte offset formed in 32-bit arithmetic;
// else a 64-bit address per lane.
template <bool O32, typename E>
LBM_DEV E* slot(E* base, int q, const StepArgs& A, int64_t xs, int64_t ys, int64_t zs)
{
	if constexpr (O32) {
		const uint32_t i = ((uint32_t) xs * (uint32_t) A.Zs + (uint32_t) zs) * (uint32_t) A.Ys + (uint32_t) ys;
		return at((E*) sptr<true>((char*) (base + q * A.XYZ)), i);
	}
	else
		return base + q * A.XYZ + (xs * A.Zs + zs) * A.Ys + ys;
}
template <bool O32, typename E>
LBM_DEV E* slot0(E* base, int q, const StepArgs& A, int64_t s)
{
	if constexpr (O32)
		return at((E*) sptr<true>((char*) (base + q * A.XYZ)), (uint32_t) s);
	else
		return base + q * A.XYZ + s;
}

// O32: every population array holds under 4 GiB (XYZ * element size <= 2^32,
// checked on the host), so a population slot is a wave-uniform base (the
// array of direction q, pinned in scalar registers) plus a 32-bit per-lane
// byte offset. The site index is then formed in 32-bit arithmetic and each
// access is one scalar-base load or store, in place of a 64-bit address per
// lane and access.
//
// LISTED: the launch covers a list of rows; with A.others it steps their sites of
// other codes only, the plain ones belonging to the lean kernels.
//
// NTG: nontemporal hints on the A-B streams no other wave touches in this step
// (the site's own slots, and the pulls with c_y = 0; the +-1 shifted rows share
// cache lines with the neighbouring wave), where rows start on lines and the
// last-level cache holds too little of the arrays (hint_streams): 256^3 F16 +2%, F32 +3%;
// rows off the lines 301x187x129 F16 282 us with them and 187 without, arrays
// within the cache 128x64x64 FP64 48.6 and 41.
template <int ST, int COLL, int PATTERN, int TAPE = 0, bool O32 = false, bool LISTED = false, bool NTG = false>
struct General
{
	using S = Storage<ST>;
	using real = typename S::real;
	using elem = typename S::elem;
	using pulled = typename Pulled<ST>::elem;
	using P = Phys<ST>;
	static constexpr bool AA = PATTERN == TNL_LBM_PATTERN_AA;
	static constexpr int EQK = eq_kind_of(COLL);
	static constexpr bool FAST = fast_collision<ST, COLL>;

	static constexpr bool NT = NTG && (ST == STORE_F32_FROM_F64 || ((LBM_NT_GENERAL >> ST % 32) & 1));
	static LBM_DEV real ldq(const pulled* p, float sc, bool nt)
	{
		if (nt) {
			const pulled v = ld_nt(p);
			return S::ld(&v, sc);
		}
		return S::ld(p, sc);
	}
	static LBM_DEV void stq(elem* p, real v, float inv, bool nt)
	{
		if (nt) {
			elem e;
			S::st(&e, v, inv);
			st_nt(p, e);
		}
		else
			S::st(p, v, inv);
	}

	static LBM_DEV int64_t sidx(const StepArgs& A, int64_t xs, int64_t ys, int64_t zs)
	{
		return (xs * A.Zs + zs) * A.Ys + ys;
	}
	template <typename E>
	static LBM_DEV E* pq(E* base, int q, const StepArgs& A, int64_t xs, int64_t ys, int64_t zs)
	{
		return slot<O32>(base, q, A, xs, ys, zs);
	}
	template <typename E>
	static LBM_DEV E* pq0(E* base, int q, const StepArgs& A, int64_t s0)
	{
		return slot0<O32>(base, q, A, s0);
	}

	static LBM_DEV void set_eq(real* f, real rho, real vx, real vy, real vz)
	{
#pragma unroll
		for (int q = 0; q < 27; q++)
			f[q] = eq_q(q, rho, vx, vy, vz);
	}
	static LBM_DEV real eq_q(int q, real rho, real vx, real vy, real vz)
	{
		// q is a compile-time constant after unrolling
		switch (q) {
#define EQC(Q) case Q: return P::template eq<EQK, Q>(rho, vx, vy, vz);
			EQC(0) EQC(1) EQC(2) EQC(3) EQC(4) EQC(5) EQC(6) EQC(7) EQC(8) EQC(9) EQC(10) EQC(11) EQC(12) EQC(13)
			EQC(14) EQC(15) EQC(16) EQC(17) EQC(18) EQC(19) EQC(20) EQC(21) EQC(22) EQC(23) EQC(24) EQC(25) EQC(26)
#undef EQC
		}
		return 0;
	}

	static LBM_DEV void inflow(const StepArgs& A, int64_t y, int64_t z, real& vx, real& vy, real& vz)
	{
		// NSE_Data_ConstInflow / NSE_Data_InflowProfile::inflow (lbm_data.h:85-132)
		const int64_t i = A.Y * z + y;
		vx = (real) inflow_component(A, 0, i);
		vy = (real) inflow_component(A, 1, i);
		vz = (real) inflow_component(A, 2, i);
	}

	static LBM_DEV void site(const StepArgs& A, int64_t x, int64_t y, int64_t z)
	{
		real vx, vy, vz;
		Nb NX, NY, NZ;
		site(A, x, y, z, vx, vy, vz, NX, NY, NZ);
	}

	// full-way bounce-back (bc.h:201-221)
	static LBM_DEV void bounce_back(real* f, real& rho, real& vx, real& vy, real& vz)
	{
		rho = 1;
		vx = vy = vz = 0;
#pragma unroll
		for (int q = 1; q < 27; q += 2) {
			const real t = f[q];
			f[q] = f[q + 1];
			f[q + 1] = t;
		}
	}

	// one site; returns the pre-collision velocity and the neighbour indices
	// (the coupled kernel drives the ADE step with them, kernels.h:152-176)
	static LBM_DEV void site(const StepArgs& A, int64_t x, int64_t y, int64_t z, real& ovx, real& ovy, real& ovz, Nb& NX,
							 Nb& NY, Nb& NZ)
	{
		const int64_t s0 = sidx(A, x + A.ox, y + A.oy, z + A.oz);
		const int16_t gi = A.map ? __builtin_nontemporal_load(A.map + s0) : (int16_t) GEO_PERIODIC;
		if (LISTED && A.others && plain(gi))
			return;
		const bool per = gi == GEO_PERIODIC;
		NX = neighbours<AA>(x, A.X, A.ox, A.dist_x, per);
		NY = neighbours<AA>(y, A.Y, A.oy, A.dist_y, per);
		NZ = neighbours<AA>(z, A.Z, A.oz, A.dist_z, per);
		real Fx = (real) A.fx, Fy = (real) A.fy, Fz = (real) A.fz;
		if (A.force)
			add_site_force(A, s0, Fx, Fy, Fz);
		real f[27];
		real rho = 1, vx = 0, vy = 0, vz = 0;
		const pulled* __restrict__ cur = (const pulled*) A.df0;

		if (gi != GEO_NOTHING) {
			// pull location (bc.h:72-74); OUTFLOW_RIGHT pulls as if located at x-1
			Nb PX = NX;
			if (gi == GEO_OUTFLOW_RIGHT)
				PX.p = PX.o = NX.m;
			if (gi == GEO_OUTFLOW_RIGHT_INTERP) {
				// streamingInterpRight (streaming_AB.h:446-478)
				const real cs = (real) 0.5773502691896257;
#pragma unroll
				for (int q = 0; q < 27; q++) {
					const int64_t yy = NY[-CY[q]], zz = NZ[-CZ[q]];
					if (CX[q] < 0)
						f[q] = cs * S::ld(cur + q * A.XYZ + sidx(A, NX.m, yy, zz), fx_sc(q, A.rs)) + ((real) 1 - cs) * S::ld(cur + q * A.XYZ + sidx(A, NX.o, yy, zz), fx_sc(q, A.rs));
					else
						f[q] = S::ld(cur + q * A.XYZ + sidx(A, CX[q] > 0 ? NX.m : NX.o, yy, zz), fx_sc(q, A.rs));
				}
			}
			else if (AA && A.even) {
#pragma unroll
				for (int q = 0; q < 27; q++)
					f[q] = ldq(pq(cur, q, A, PX.o, NY.o, NZ.o), fx_sc(q, A.rs), NT);
			}
			else if (AA) {
#pragma unroll
				for (int q = 0; q < 27; q++)
					f[q] = ldq(pq(cur, opp(q), A, PX[-CX[q]], NY[-CY[q]], NZ[-CZ[q]]), fx_sc(opp(q), A.rs),
							   NT && CY[q] == 0);
			}
			else {
#pragma unroll
				for (int q = 0; q < 27; q++)
					f[q] = ldq(pq(cur, q, A, PX[-CX[q]], NY[-CY[q]], NZ[-CZ[q]]), fx_sc(q, A.rs), NT && CY[q] == 0);
			}

			// the raw moments of the pulled populations, recorded after the step's own stores
			using TT = std::conditional_t<TAPE == 2, double, float>;
			TT tm[10];
			const bool rec = TAPE != 0 && (gi == GEO_FLUID || gi == GEO_PERIODIC || gi == GEO_OUTFLOW_RIGHT || gi == GEO_OUTFLOW_EQ);
			if constexpr (TAPE != 0) {
				real m[10];
				raw_moments10(f, m);
#pragma unroll
				for (int k = 0; k < 10; k++)
					tm[k] = (TT) m[k];
			}
			const real rest = S::dev ? (real) 1 : (real) 0;
			switch (gi) {
				case GEO_INFLOW:
					inflow(A, y, z, vx, vy, vz);
					rho = 1;
					set_eq(f, rho, vx, vy, vz);
					break;
				case GEO_INFLOW_LEFT:
					if constexpr (! S::dev) {
						// moment-based inflow (bc.h:91-142)
						inflow(A, y, z, vx, vy, vz);
						rho = (real) 1 / (1 - vx)
							* ((f[zzz] + (((f[zpp] + f[zmm]) + (f[zpm] + f[zmp])) + ((f[zpz] + f[zmz]) + (f[zzp] + f[zzm]))))
							   + 2 * (f[mzz] + (((f[mpp] + f[mmm]) + (f[mpm] + f[mmp])) + ((f[mpz] + f[mmz]) + (f[mzp] + f[mzm])))));
						const real n1o3 = (real) (1.0 / 3.0), n1o9 = (real) (1.0 / 9.0);
						const real m100 = rho * vx, m010 = rho * vy, m001 = rho * vz, m011 = rho * (vy * vz);
						const real m020 = n1o3 * rho + rho * (vy * vy);
						const real m002 = n1o3 * rho + rho * (vz * vz);
						const real m021 = n1o3 * rho * vz + rho * ((vy * vy) * vz);
						const real m012 = n1o3 * rho * vy + rho * (vy * (vz * vz));
						const real m022 = n1o9 * rho + n1o3 * rho * (vy * vy + vz * vz) + rho * (vy * vy) * (vz * vz);
						f[pzz] = m100 + (m022 - (m020 + m002)) + f[mzz]
							   + (((f[zpp] + f[zmm]) + (f[zpm] + f[zmp])) + ((f[zzp] + f[zzm]) + (f[zpz] + f[zmz])))
							   + 2 * (((f[mpp] + f[mmm]) + (f[mpm] + f[mmp])) + ((f[mpz] + f[mmz]) + (f[mzp] + f[mzm])));
						f[ppz] = (real) 0.5 * ((m020 - m022) + (-m012 + m010)) - (f[mpz] + f[zpz]);
						f[pmz] = (real) 0.5 * ((m020 - m022) + (m012 - m010)) - (f[mmz] + f[zmz]);
						f[pzp] = (real) 0.5 * ((m002 - m022) + (-m021 + m001)) - (f[mzp] + f[zzp]);
						f[pzm] = (real) 0.5 * ((m002 - m022) + (m021 - m001)) - (f[mzm] + f[zzm]);
						f[ppp] = (real) 0.25 * ((m022 + m011) + (m021 + m012)) - (f[mpp] + f[zpp]);
						f[ppm] = (real) 0.25 * ((m022 - m011) + (-m021 + m012)) - (f[mpm] + f[zpm]);
						f[pmp] = (real) 0.25 * ((m022 - m011) + (m021 - m012)) - (f[mmp] + f[zmp]);
						f[pmm] = (real) 0.25 * ((m022 + m011) + (-m021 - m012)) - (f[mmm] + f[zmm]);
					}
					else
						P::density_velocity(f, Fx, Fy, Fz, rho, vx, vy, vz);
					break;
				case GEO_INFLOW_BB_LEFT:
					{
						// bc.h:143-165 (pull scheme): reads unstreamed own slots
						inflow(A, y, z, vx, vy, vz);
						const real k2 = (real) 2 * (real) 3;
						const int64_t so = sidx(A, NX.o, NY.o, NZ.o);
						f[pzz] = S::ld(cur + mzz * A.XYZ + so, fx_sc(mzz, A.rs)) - k2 * (real) (2.0 / 27.0) * rho * (-vx);
						f[ppz] = S::ld(cur + mmz * A.XYZ + so, fx_sc(mmz, A.rs)) - k2 * (real) (1.0 / 54.0) * rho * (-vx - vy);
						f[pmz] = S::ld(cur + mpz * A.XYZ + so, fx_sc(mpz, A.rs)) - k2 * (real) (1.0 / 54.0) * rho * (-vx + vy);
						f[pzp] = S::ld(cur + mzm * A.XYZ + so, fx_sc(mzm, A.rs)) - k2 * (real) (1.0 / 54.0) * rho * (-vx - vz);
						f[pzm] = S::ld(cur + mzp * A.XYZ + so, fx_sc(mzp, A.rs)) - k2 * (real) (1.0 / 54.0) * rho * (-vx + vz);
						f[ppp] = S::ld(cur + mmm * A.XYZ + so, fx_sc(mmm, A.rs)) - k2 * (real) (1.0 / 216.0) * rho * (-vx - vy - vz);
						f[ppm] = S::ld(cur + mmp * A.XYZ + so, fx_sc(mmp, A.rs)) - k2 * (real) (1.0 / 216.0) * rho * (-vx - vy + vz);
						f[pmp] = S::ld(cur + mpm * A.XYZ + so, fx_sc(mpm, A.rs)) - k2 * (real) (1.0 / 216.0) * rho * (-vx + vy - vz);
						f[pmm] = S::ld(cur + mpp * A.XYZ + so, fx_sc(mpp, A.rs)) - k2 * (real) (1.0 / 216.0) * rho * (-vx + vy + vz);
						P::density_velocity(f, Fx, Fy, Fz, rho, vx, vy, vz);
						break;
					}
				case GEO_INFLOW_EQ_LEFT:
					// bc.h:166-185 (deviation storage: the known-direction weights sum to 1)
					inflow(A, y, z, vx, vy, vz);
					rho = (real) 1 / (1 - vx)
						* ((rest + (f[zzz] + (((f[zpp] + f[zmm]) + (f[zpm] + f[zmp])) + ((f[zpz] + f[zmz]) + (f[zzp] + f[zzm])))))
						   + 2 * (f[mzz] + (((f[mpp] + f[mmm]) + (f[mpm] + f[mmp])) + ((f[mpz] + f[mmz]) + (f[mzp] + f[mzm])))));
					set_eq(f, rho, vx, vy, vz);
					break;
				case GEO_OUTFLOW_EQ:
					P::density_velocity(f, Fx, Fy, Fz, rho, vx, vy, vz);
					rho = 1;
					set_eq(f, rho, vx, vy, vz);
					break;
				case GEO_OUTFLOW_RIGHT:
					P::density_velocity(f, Fx, Fy, Fz, rho, vx, vy, vz);
					rho = 1;
					break;
				case GEO_OUTFLOW_RIGHT_INTERP:
					P::density_velocity(f, Fx, Fy, Fz, rho, vx, vy, vz);
#pragma unroll
					for (int q = 0; q < 27; q++)
						f[q] += eq_q(q, (real) 1, vx, vy, vz) - eq_q(q, rho, vx, vy, vz);
					rho = 1;
					break;
				case GEO_WALL:
					bounce_back(f, rho, vx, vy, vz);
					break;
				case GEO_SYM_TOP:
				case GEO_SYM_BOTTOM:
				case GEO_SYM_LEFT:
				case GEO_SYM_RIGHT:
				case GEO_SYM_BACK:
				case GEO_SYM_FRONT:
					{
						// bc.h:222-293
						const int axis = (gi == GEO_SYM_TOP || gi == GEO_SYM_BOTTOM) ? 2 : (gi == GEO_SYM_LEFT || gi == GEO_SYM_RIGHT) ? 0 : 1;
						const int sgn = (gi == GEO_SYM_BOTTOM || gi == GEO_SYM_LEFT || gi == GEO_SYM_BACK) ? 1 : -1;
#pragma unroll
						for (int q = 0; q < 27; q++) {
							const int c = axis == 0 ? CX[q] : axis == 1 ? CY[q] : CZ[q];
							if (c == sgn) {
								const int mq = axis == 0 ? qidx(1 - sgn, CY[q] + 1, CZ[q] + 1)
											 : axis == 1 ? qidx(CX[q] + 1, 1 - sgn, CZ[q] + 1)
														 : qidx(CX[q] + 1, CY[q] + 1, 1 - sgn);
								real src = 0;
#pragma unroll
								for (int r = 0; r < 27; r++)
									if (r == mq)
										src = f[r];
								f[q] = src;
							}
						}
						P::density_velocity(f, Fx, Fy, Fz, rho, vx, vy, vz);
						break;
					}
				default:
					// the fast FP32 collision sums its own moments at plain collided sites
					if (! (FAST && (gi == GEO_FLUID || gi == GEO_PERIODIC)))
						P::density_velocity(f, Fx, Fy, Fz, rho, vx, vy, vz);
					break;
			}
			// doCollision (bc.h:406-412)
			const bool do_coll = gi == GEO_FLUID || gi == GEO_PERIODIC || gi == GEO_OUTFLOW_RIGHT || gi == GEO_OUTFLOW_RIGHT_INTERP
							  || gi == GEO_INFLOW_LEFT || gi == GEO_INFLOW_BB_LEFT;
			if constexpr (FAST) {
				// FP32 forms, default cumulant: the raw-moment formulation (as the periodic kernel)
				// wherever rho and u are the site's own; the boundary codes that replace them keep
				// the reference chain
				if (gi == GEO_FLUID || gi == GEO_PERIODIC) {
					using FC = FastCum<S::dev>;
					FC::collide(f, Fx, Fy, Fz, (real) A.omega1, true, rho, vx, vy, vz);
#pragma unroll
					for (int q = 0; q < 27; q++)
						f[q] *= FC::unscale(q);
				}
				else if (do_coll)
					collide<ST, COLL>(f, rho, vx, vy, vz, A, Fx, Fy, Fz);
			}
			else if (do_coll)
				collide<ST, COLL>(f, rho, vx, vy, vz, A, Fx, Fy, Fz);
			// postCollision streaming
			if (AA && A.even) {
				elem* __restrict__ out = (elem*) A.df0;
#pragma unroll
				for (int q = 0; q < 27; q++)
					stq(pq0(out, opp(q), A, s0), f[q], fx_inv(opp(q), A.invr), NT);
			}
			else if (AA) {
				elem* __restrict__ out = (elem*) A.df0;
#pragma unroll
				for (int q = 0; q < 27; q++)
					stq(pq(out, q, A, NX[CX[q]], NY[CY[q]], NZ[CZ[q]]), f[q], fx_inv(q, A.invr), NT && CY[q] == 0);
			}
			else {
				elem* __restrict__ out = (elem*) A.df1;
#pragma unroll
				for (int q = 0; q < 27; q++)
					stq(pq0(out, q, A, s0), f[q], fx_inv(q, A.invr), NT);
			}
			if constexpr (TAPE != 0) {
				if (rec) {
					TT* __restrict__ tp = (TT*) A.tape;
#pragma unroll
					for (int k = 0; k < 10; k++)
						__builtin_nontemporal_store(tm[k], tp + tape_index(k, s0));
				}
			}
		}
		if (A.out_macro)
			write_macro(A, s0, rho, vx, vy, vz);
		ovx = vx;
		ovy = vy;
		ovz = vz;
	}
};

// The FP64 default cumulant needs ~170 VGPRs here: asking for 3 waves per SIMD
// (<= 168) costs at most 2 spilled registers; the alternative operators keep
// their registers.
template <int ST, int COLL, int PATTERN, int TAPE = 0, bool O32 = false, bool LISTED = false, bool NTG = false>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(COLL == TNL_LBM_COLL_CUM ? 3 : 1, 8))) k_general(const StepArgs A)
{
	int64_t x, z, y;
	if (! block_coords<true, LISTED>(A, x, z, y))
		return;
	General<ST, COLL, PATTERN, TAPE, O32, LISTED, NTG>::site(A, x, y, z);
}

// ===========================================================================
// Coupled NSE + ADE: cudaLBMKernel<NSE,ADE> (kernels.h:114-196)
// ===========================================================================
// The D3Q7 inputs of one site: its code, the 7 pulled populations, the
// diffusivity and the source.  Loaded before the D3Q27 update of the same
// site, so that their latency overlaps it (the compiler cannot move them above
// the D3Q27 stores by itself).
template <int ST>
struct AdeIn
{
	int16_t gi;
	typename Storage<ST>::real f[7];
	typename Storage<ST>::real D, S;
};

// src(k, ...): the k-th load, population from(k) pulled here
template <int ST, bool LEAN, typename From, typename Src>
LBM_DEV void ade_load(const StepArgs& A, const AdeArgs& B, int64_t s0, int16_t gi, From from, Src&& src, AdeIn<ST>& in)
{
	using K = Ade7<ST>;
	using real = typename K::real;
	in.gi = gi;
	auto macro_at = [&](const void* p) -> real {
		return A.macro_f64 ? (real) ((const double*) p)[s0] : (real) ((const float*) p)[s0];
	};
	// D3Q7_MACRO_Default::copyQuantities (d3q7/macro.h:38-42)
	in.D = B.diff ? macro_at(B.diff) : (real) B.D;
	in.S = B.source ? macro_at(B.source) : (real) 0;
	const real pr = (real) B.phi_ref, isc = (real) 1 / (real) B.scale;
	if (LEAN || gi != A_NOTHING) {
#pragma unroll
		for (int k = 0; k < 7; k++)
			in.f[from(k)] = src(k, pr, isc);
	}
}

// one pulled population: nontemporal where `nt`
template <int ST>
LBM_DEV typename Storage<ST>::real ade_get(const typename Storage<ST>::elem* p, int qs, typename Storage<ST>::real pr,
										   typename Storage<ST>::real isc, bool nt)
{
	if (nt) {
		const auto v = ld_nt(p);
		return Ade7<ST>::ld(&v, qs, pr, isc);
	}
	return Ade7<ST>::ld(p, qs, pr, isc);
}
template <int ST>
LBM_DEV void ade_put(typename Storage<ST>::elem* p, int qs, typename Storage<ST>::real v, typename Storage<ST>::real pr,
					 typename Storage<ST>::real sc, bool nt)
{
	if (nt) {
		typename Storage<ST>::elem e;
		Ade7<ST>::st(&e, qs, v, pr, sc);
		st_nt(p, e);
	}
	else
		Ade7<ST>::st(p, qs, v, pr, sc);
}

// boundary codes and collision of the loaded populations: f post-collision,
// returns phi.  LEAN: the plain codes only.
template <int ST, bool LEAN>
LBM_DEV typename Storage<ST>::real ade_update(const AdeArgs& B, const AdeIn<ST>& in, typename Storage<ST>::real vx,
											  typename Storage<ST>::real vy, typename Storage<ST>::real vz,
											  typename Storage<ST>::real* f)
{
	using K = Ade7<ST>;
	using real = typename K::real;
	const int16_t gi = in.gi;
	real phi = 0;
#pragma unroll
	for (int q = 0; q < 7; q++)
		f[q] = in.f[q];
	if constexpr (LEAN) {
		phi = K::density(f);
		if (gi == A_WALL)
			K::bounce_back(f);
	}
	else switch (gi) {
		case A_INFLOW:
			phi = (real) B.inflow_phi;
			K::set_eq(f, phi, vx, vy, vz);
			break;
		case A_WALL:
			phi = K::density(f);
			K::bounce_back(f);
			break;
		case A_SYM_TOP: f[zzm] = f[zzp]; phi = K::density(f); break;
		case A_SYM_BOTTOM: f[zzp] = f[zzm]; phi = K::density(f); break;
		case A_SYM_LEFT: f[pzz] = f[mzz]; phi = K::density(f); break;
		case A_SYM_RIGHT: f[mzz] = f[pzz]; phi = K::density(f); break;
		case A_SYM_BACK: f[zpz] = f[zmz]; phi = K::density(f); break;
		case A_SYM_FRONT: f[zmz] = f[zpz]; phi = K::density(f); break;
		default: phi = K::density(f); break;
	}
	if (LEAN ? gi != A_WALL : (gi == A_FLUID || gi == A_PERIODIC || gi == A_SOLID || gi == A_OUTFLOW_RIGHT)) {
		K::collide(B.collision, f, phi, vx, vy, vz, in.D);
		if (B.source) {
#pragma unroll
			for (int q = 0; q < 7; q++)
				f[q] += (real) w7(q) * in.S;
		}
	}
	return phi;
}

template <int ST>
LBM_DEV void write_phi(const StepArgs& A, const AdeArgs& B, int64_t s0, typename Storage<ST>::real phi)
{
	if (A.out_macro && B.macro) {
		if (A.macro_f64)
			((double*) B.macro)[s0] = phi;
		else
			((float*) B.macro)[s0] = (float) phi;
	}
}

// LISTED, NTG as in General; a site is plain where both of its codes are
template <int ST, int COLL, int PATTERN, bool O32 = false, bool LISTED = false, bool NTG = false>
__global__ void __launch_bounds__(256) k_nse_ade(const StepArgs A, const AdeArgs B)
{
	using K = Ade7<ST>;
	using real = typename K::real;
	using elem = typename K::elem;
	int64_t x, z, y;
	if (! block_coords<true, LISTED>(A, x, z, y))
		return;
	constexpr bool AA = PATTERN == TNL_LBM_PATTERN_AA;
	constexpr bool NT = NTG && ((LBM_NT_GENERAL >> ST) & 1);
	const int64_t s0 = ((x + A.ox) * A.Zs + (z + A.oz)) * A.Ys + (y + A.oy);
	const int16_t gn = A.map ? A.map[s0] : (int16_t) GEO_PERIODIC;
	const int16_t ga = B.map ? B.map[s0] : (int16_t) A_PERIODIC;
	if (LISTED && A.others && plain(gn) && plain_scalar(ga))
		return;
	// neighbours as General::site forms them (periodic wrap for PERIODIC-coded sites)
	const bool per = gn == GEO_PERIODIC;
	const Nb NX = neighbours<AA>(x, A.X, A.ox, A.dist_x, per);
	const Nb NY = neighbours<AA>(y, A.Y, A.oy, A.dist_y, per);
	const Nb NZ = neighbours<AA>(z, A.Z, A.oz, A.dist_z, per);
	Nb PX = NX;
	if (ga == A_OUTFLOW_RIGHT)
		PX.p = PX.o = NX.m;
	AdeIn<ST> in;
	const elem* cur = (const elem*) B.df0;
	ade_load<ST, false>(A, B, s0, ga, [](int q) { return q; },
				 [&](int q, real pr, real isc) {
					 if (AA && B.even)
						 return ade_get<ST>(slot0<O32>(cur, q, A, s0), q, pr, isc, NT);
					 const int qs = AA ? opp(q) : q;
					 return ade_get<ST>(slot<O32>(cur, qs, A, PX[-CX[q]], NY[-CY[q]], NZ[-CZ[q]]), qs, pr, isc, NT && CY[q] == 0);
				 },
				 in);
	real vx, vy, vz;
	Nb GX, GY, GZ;
	General<ST, COLL, PATTERN, 0, O32, false, NTG>::site(A, x, y, z, vx, vy, vz, GX, GY, GZ);
	real phi = 0;
	if (ga != A_NOTHING) {
		real f[7];
		phi = ade_update<ST, false>(B, in, vx, vy, vz, f);
		elem* out = (elem*) (AA ? B.df0 : B.df1);
		const real pr = (real) B.phi_ref, sc = (real) B.scale;
#pragma unroll
		for (int q = 0; q < 7; q++) {
			if (AA && B.even)
				ade_put<ST>(slot0<O32>(out, opp(q), A, s0), opp(q), f[q], pr, sc, NT);
			else if (AA)
				ade_put<ST>(slot<O32>(out, q, A, NX[CX[q]], NY[CY[q]], NZ[CZ[q]]), q, f[q], pr, sc, NT && CY[q] == 0);
			else
				ade_put<ST>(slot0<O32>(out, q, A, s0), q, f[q], pr, sc, NT);
		}
	}
	write_phi<ST>(A, B, s0, phi);
}

// ===========================================================================
// Lean kernels: the plain sites (FLUID, PERIODIC, WALL) of a box with a
// geometry map, flow alone (A-A odd step, A-B step) or coupled (all three).
// The sites of any other code are skipped; a launch of the general kernels
// over the rows that hold them (LISTED) steps those before.
//
// A kernel's registers are the maximum over all of its paths, so the rarely
// taken boundary codes cost every site of the general kernels their occupancy
// (F16 A-B: 97 VGPRs with all 17 codes, 48 with these).  Beyond that, a block
// lies in one x plane (LIN) or in one row, so x (and z) are wave-uniform and a
// slot is a scalar base plus a 32-bit per-lane offset; per-lane coordinates
// cost about 150 VALU instructions a site.  Only the choice between the
// periodic wrap and the clamp at a face depends on the site's code: where the
// two differ, the lanes of either kind run in turn.
// Bound: HBM.  Both steps, against the list kernels with per-lane coordinates:
// 256^3 with z walls A-A F16 816 -> 710 us, F32 1484 -> 1368, FP64 2934 ->
// 2761; A-B 301x187x129 F16 571 -> 363 (rows off the lines); coupled A-A 256^3
// F16 1074 -> 985; coupled A-B aligned: equal (4.9 TB/s).
// ===========================================================================
constexpr int LEAN_EVEN = 0, LEAN_ODD = 1, LEAN_AB = 2;

template <bool LIN>
struct Stencil
{
	uint64_t xoff[3];       // sites before the x plane of -1, 0, +1 (wave-uniform)
	uint32_t zs[3], zr[3];  // stored z: wave-uniform, or (LIN) the z row's per-lane offset in its plane
	uint32_t ys[3];         // stored y, per lane
	// Called in the basic block of each group of accesses: a lane offset that is
	// extended to 64 bits in another block leaves the scalar-base form.
	LBM_DEV void local()
	{
#pragma unroll
		for (int c = 0; c < 3; c++) {
			asm volatile("" : "+v"(ys[c]));
			if constexpr (LIN)
				asm volatile("" : "+v"(zr[c]));
		}
	}
	// the site's own stored index
	LBM_DEV int64_t own(const StepArgs& A) const
	{
		int64_t s = (int64_t) xoff[1] + (LIN ? zr[1] : zs[1] * (uint32_t) A.Ys) + ys[1];
		asm volatile("" : "+v"(s));
		return s;
	}
	// slot of the direction whose array `base` is
	template <typename E>
	LBM_DEV E* slot(E* base, const StepArgs& A, int cx, int cy, int cz) const
	{
		if constexpr (LIN)
			return at((E*) sptr<true>((char*) base + xoff[1 + cx] * sizeof(E)), zr[1 + cz] + ys[1 + cy]);
		else
			return at((E*) sptr<true>((char*) base + (xoff[1 + cx] + (uint64_t) (zs[1 + cz] * (uint32_t) A.Ys)) * sizeof(E)), ys[1 + cy]);
	}
};

// neighbours<AA> of a per-lane coordinate in 32 bits (extents below 2^30)
template <bool AA>
LBM_DEV void neighbours32(uint32_t* r, int32_t c, int32_t n, int32_t o, bool dist, bool periodic)
{
	const int32_t pw = (! dist && c == n - 1) ? 0 : c + 1, mw = (! dist && c == 0) ? n - 1 : c - 1;
	const int32_t pc = AA ? (c + 1 < n + o ? c + 1 : 0) : (c + 1 < n - 1 + o ? c + 1 : n - 1 + o);
	const int32_t mc = AA ? (c - 1 >= -o ? c - 1 : n - 1) : (c - 1 > -o ? c - 1 : -o);
	r[0] = (uint32_t) ((periodic ? mw : mc) + o);
	r[1] = (uint32_t) (c + o);
	r[2] = (uint32_t) ((periodic ? pw : pc) + o);
}

// A wave-uniform value the compiler may not form ahead of this point: the scalar
// bases of 27 directions, hoisted out of a loop or above the collision, would
// spill.
template <typename T>
LBM_DEV T here(T v)
{
	asm volatile("" : "+s"(v));
	return v;
}
template <int ST, int MODE, bool LIN, bool NTG, bool ADE>
LBM_DEV void lean_site(const StepArgs& A, const AdeArgs& B)
{
	using S = Storage<ST>;
	using real = typename S::real;
	using elem = typename S::elem;
	constexpr int COLL = TNL_LBM_COLL_CUM;
	constexpr bool AA = MODE != LEAN_AB;
	constexpr bool NT = NTG && ((LBM_NT_GENERAL >> ST) & 1);
	int64_t x, z, y;
	if (! box_coords<LIN>(A, x, z, y))
		return;
	const int64_t s0 = ((x + A.ox) * A.Zs + (z + A.oz)) * A.Ys + (y + A.oy);
	const int16_t gi = A.map ? A.map[s0] : (int16_t) GEO_PERIODIC;
	const int16_t ga = ADE && B.map ? B.map[s0] : (int16_t) A_PERIODIC;
	const bool per = gi == GEO_PERIODIC, wall = gi == GEO_WALL;
	const bool mine = plain(gi) && plain_scalar(ga);
	const Nb XW = neighbours<AA>(x, A.X, A.ox, A.dist_x, true), XC = neighbours<AA>(x, A.X, A.ox, A.dist_x, false);
	const Nb ZW = neighbours<AA>(z, A.Z, A.oz, A.dist_z, true), ZC = neighbours<AA>(z, A.Z, A.oz, A.dist_z, false);
	bool same = MODE == LEAN_EVEN || (XW.m == XC.m && XW.p == XC.p);
	if (! LIN && MODE != LEAN_EVEN)
		same = same && ZW.m == ZC.m && ZW.p == ZC.p;
	auto kind = [&](const Nb& NX, const Nb& NZ) __attribute__((always_inline)) {
		Stencil<LIN> N;
		const uint64_t pb = here(A.plane_bytes);
		const uint64_t plane = (uint64_t) (A.Zs * A.Ys);
		N.xoff[0] = NX.m * plane;
		N.xoff[1] = NX.o * plane;
		N.xoff[2] = NX.p * plane;
		// (formed here: the offsets of both kinds would stay live)
		int32_t yl = (int32_t) y;
		asm volatile("" : "+v"(yl));
		neighbours32<AA>(N.ys, yl, (int32_t) A.Y, (int32_t) A.oy, A.dist_y, per);
		if constexpr (LIN) {
			int32_t zl = (int32_t) z;
			asm volatile("" : "+v"(zl));
			neighbours32<AA>(N.zr, zl, (int32_t) A.Z, (int32_t) A.oz, A.dist_z, per);
#pragma unroll
			for (int c = 0; c < 3; c++)
				N.zr[c] *= (uint32_t) A.Ys;
		}
		else {
			N.zs[0] = (uint32_t) NZ.m;
			N.zs[1] = (uint32_t) NZ.o;
			N.zs[2] = (uint32_t) NZ.p;
		}
		// Array k holds what population from(k) pulls here and population to(k)
		// pushes; their slots in it.
		constexpr auto from = [](int k) { return MODE == LEAN_ODD ? opp(k) : k; };
		constexpr auto to = [](int k) { return MODE == LEAN_EVEN ? opp(k) : k; };
		auto src = [&](const elem* base, int k) {
			if constexpr (MODE == LEAN_EVEN)
				return N.slot(base, A, 0, 0, 0);
			else
				return N.slot(base, A, -CX[from(k)], -CY[from(k)], -CZ[from(k)]);
		};
		auto dst = [&](elem* base, int k) {
			if constexpr (MODE == LEAN_ODD)
				return N.slot(base, A, CX[k], CY[k], CZ[k]);
			else
				return N.slot(base, A, 0, 0, 0);
		};
		AdeIn<ST> in;
		N.local();
		if constexpr (ADE) {
			Planes<const elem> acur(here((char*) B.df0), pb);
			ade_load<ST, true>(A, B, N.own(A), ga, from,
							   [&](int k, real pr, real isc) {
								   return ade_get<ST>(src(acur.next(), k), k, pr, isc, NT && (MODE == LEAN_EVEN || CY[k] == 0));
							   },
							   in);
			N.local();
		}
		real f[27];
		Planes<const elem> cur(here((char*) A.df0), pb);
#pragma unroll
		for (int k = 0; k < 27; k++) {
			const elem* p = src(cur.next(), k);
			const elem v = NT && (MODE == LEAN_EVEN || CY[k] == 0) ? ld_nt(p) : *p;
			f[from(k)] = S::ld(&v, A.cls_sc[ncls(k)]);
		}
		real rho = 1, vx = 0, vy = 0, vz = 0;
		real Fx = (real) here(A.fx), Fy = (real) here(A.fy), Fz = (real) here(A.fz);
		if (A.force)
			add_site_force(A, N.own(A), Fx, Fy, Fz);
		if (wall)
			bounce_back<ST, COLL>(f);
		if (! wall)
			collide_site<ST, COLL>(f, A, Fx, Fy, Fz, rho, vx, vy, vz);
		Planes<elem> out(after<true>((char*) (AA ? A.df0 : A.df1), f[26]), here(A.plane_bytes));
		N.local();
		real o[27];
#pragma unroll
		for (int k = 0; k < 27; k++)
			o[k] = f[to(k)];
		encode_all<ST, COLL>(o, A, [&](int k, elem e) {
			elem* p = dst(out.next(), k);
			if (NT && (MODE != LEAN_ODD || CY[k] == 0))
				st_nt(p, e);
			else
				*p = e;
		});
		if (A.out_macro)
			write_macro(A, N.own(A), rho, vx, vy, vz);
		if constexpr (ADE) {
			real g[7];
			const real phi = ade_update<ST, true>(B, in, vx, vy, vz, g);
			const real pr = (real) B.phi_ref, sc = (real) B.scale;
			Planes<elem> aout(after<true>((char*) (AA ? B.df0 : B.df1), g[6]), here(A.plane_bytes));
			N.local();
#pragma unroll
			for (int k = 0; k < 7; k++)
				ade_put<ST>(dst(aout.next(), k), k, g[to(k)], pr, sc, NT && (MODE != LEAN_ODD || CY[k] == 0));
			write_phi<ST>(A, B, N.own(A), phi);
		}
	};
	if (mine && (same || per))
		kind(XW, ZW);
	if (! same && mine && ! per)
		kind(XC, ZC);
}

template <int ST, int MODE, bool LIN, bool NTG>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(ST == TNL_LBM_STORE_F64 ? 3 : 4, 8)))
k_lean(const StepArgs A)
{
	lean_site<ST, MODE, LIN, NTG, false>(A, AdeArgs{});
}
template <int ST, int MODE, bool LIN, bool NTG>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(ST == TNL_LBM_STORE_F64 ? 3 : 4, 8)))
k_lean_ade(const StepArgs A, const AdeArgs B)
{
	lean_site<ST, MODE, LIN, NTG, true>(A, B);
}

template <int ST>
__global__ void k_ade_set_equilibrium(void* df0, void* df1, int ncopies, int64_t XYZ, int64_t n, const void* phi,
									  int phi_f64, double phi0, double pr, double sc)
{
	using K = Ade7<ST>;
	const int64_t s = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
	if (s >= n)
		return;
	const double p = phi ? (phi_f64 ? ((const double*) phi)[s] : (double) ((const float*) phi)[s]) : phi0;
	typename K::real f[7];
	K::set_eq(f, (typename K::real) p, 0, 0, 0);
	for (int k = 0; k < ncopies; k++) {
		auto* out = (typename K::elem*) (k == 0 ? df0 : df1);
#pragma unroll
		for (int q = 0; q < 7; q++)
			K::st(out + q * XYZ + s, q, f[q], (typename K::real) pr, (typename K::real) sc);
	}
}

template <int ST>
__global__ void k_ade_export(const void* df, double* out, int64_t XYZ, int64_t n, double pr, double sc)
{
	using K = Ade7<ST>;
	const int64_t s = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
	if (s >= n)
		return;
#pragma unroll
	for (int q = 0; q < 7; q++)
		out[q * XYZ + s] = (double) K::ld((const typename K::elem*) df + q * XYZ + s, q, (typename K::real) pr,
										  (typename K::real) 1 / (typename K::real) sc);
}

// ===========================================================================
// Row classification for the row-list launches (tnl_lbm_classify_rows)
// ===========================================================================
// One wave per interior (x, z) row, row i = x * Z + z: class 1 when every
// code of the row is FLUID or PERIODIC (D3Q27 and, with amap, D3Q7), 2 when
// WALL sites occur as well, 0 otherwise.  A null map is all PERIODIC.
static __global__ void __launch_bounds__(256) k_classify_rows(const int16_t* map, const int16_t* amap, int64_t X, int64_t Y,
													   int64_t Z, int64_t ox, int64_t oy, int64_t oz, int64_t Ys, int64_t Zs,
													   uint8_t* cls)
{
	const int64_t i = ((int64_t) blockIdx.x * blockDim.x + threadIdx.x) >> 6;  // uniform per wave
	if (i >= X * Z)
		return;
	const int64_t x = i / Z, z = i % Z;
	const int64_t base = ((x + ox) * Zs + (z + oz)) * Ys + oy;
	bool other = false, wall = false;
	for (int64_t y = threadIdx.x & 63; y < Y; y += 64) {
		if (map) {
			const int16_t c = map[base + y];
			wall |= c == GEO_WALL;
			other |= ! (c == GEO_FLUID || c == GEO_PERIODIC || c == GEO_WALL);
		}
		if (amap) {
			const int16_t c = amap[base + y];
			wall |= c == A_WALL;
			other |= ! (c == A_FLUID || c == A_PERIODIC || c == A_WALL);
		}
	}
	const uint64_t o = __ballot(other), w = __ballot(wall);
	if ((threadIdx.x & 63) == 0)
		cls[i] = o ? 0 : (w ? 2 : 1);
}

// The three row lists from the classes, in one workgroup so that each list
// keeps increasing row order: counts first, then every chunk of 1024 rows
// places its rows of each class after those of the earlier chunks.
static __global__ void __launch_bounds__(1024) k_row_lists(const uint8_t* cls, uint32_t n, uint32_t Z, uint32_t* rows,
													uint32_t* counts)
{
	__shared__ uint32_t part[16][3];
	__shared__ uint32_t off[3];
	const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
	uint32_t c3[3] = {0, 0, 0};
	for (uint32_t i = t; i < n; i += 1024) {
		const uint8_t c = cls[i];
		c3[0] += c == 0;
		c3[1] += c == 1;
		c3[2] += c == 2;
	}
	for (int k = 0; k < 3; k++) {
		uint32_t v = c3[k];
		for (int d = 32; d >= 1; d >>= 1)
			v += __shfl_xor(v, d);
		if (lane == 0)
			part[wave][k] = v;
	}
	__syncthreads();
	if (t == 0) {
		uint32_t tot[3] = {0, 0, 0};
		for (int w = 0; w < 16; w++)
			for (int k = 0; k < 3; k++)
				tot[k] += part[w][k];
		for (int k = 0; k < 3; k++)
			counts[k] = tot[k];
		off[0] = 0;
		off[1] = tot[0];
		off[2] = tot[0] + tot[1];
	}
	__syncthreads();
	const uint64_t below = (lane == 0) ? 0 : (~0ull >> (64 - lane));
	for (uint32_t c0 = 0; c0 < n; c0 += 1024) {
		const uint32_t i = c0 + t;
		const int c = i < n ? (int) cls[i] : -1;
		uint64_t m[3];
		for (int k = 0; k < 3; k++) {
			m[k] = __ballot(c == k);
			if (lane == 0)
				part[wave][k] = (uint32_t) __popcll(m[k]);
		}
		__syncthreads();
		if (c >= 0) {
			uint32_t pos = off[c];
			for (uint32_t w = 0; w < wave; w++)
				pos += part[w][c];
			const uint64_t mc = c == 0 ? m[0] : (c == 1 ? m[1] : m[2]);
			pos += (uint32_t) __popcll(mc & below);
			rows[pos] = ((i / Z) << 16) | (i % Z);
		}
		__syncthreads();
		if (t < 3) {
			uint32_t add = 0;
			for (int w = 0; w < 16; w++)
				add += part[w][t];
			off[t] += add;
		}
		__syncthreads();
	}
}

// ===========================================================================
// Initialisation, transfer and reduction kernels
// ===========================================================================
struct FieldArgs
{
	void* df[2];
	int ncopies;
	int64_t XYZ;
	int64_t nsites;  // stored sites incl. overlaps
	const double* rho;
	const double* vx;
	const double* vy;
	const double* vz;
	double c[4];
	float rs[4], invr[4];
};

template <int ST, int EQK>
__global__ void k_set_equilibrium(const FieldArgs A)
{
	using S = Storage<ST>;
	using real = typename S::real;
	const int64_t s = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
	if (s >= A.nsites)
		return;
	const real rho = (real) (A.rho ? A.rho[s] : A.c[0]);
	const real vx = (real) (A.vx ? A.vx[s] : A.c[1]);
	const real vy = (real) (A.vy ? A.vy[s] : A.c[2]);
	const real vz = (real) (A.vz ? A.vz[s] : A.c[3]);
	real f[27];
	// one operator per equilibrium kind
	constexpr int coll = EQK == 0 ? TNL_LBM_COLL_CUM : EQK == 1 ? TNL_LBM_COLL_MRT_LES : TNL_LBM_COLL_KBC_N2;
	General<ST, coll, TNL_LBM_PATTERN_AA>::set_eq(f, rho, vx, vy, vz);
	for (int k = 0; k < A.ncopies; k++) {
		auto* out = (typename S::elem*) A.df[k];
#pragma unroll
		for (int q = 0; q < 27; q++)
			S::st(out + q * A.XYZ + s, f[q], fx_inv(q, A.invr));
	}
}

struct MacroArgs
{
	float rs[4], invr[4];
	const void* df;
	void* macro;
	int macro_f64;
	int64_t XYZ;
	int64_t X, Y, Z, ox, oy, oz, Ys, Zs;
	int32_t dist_x, dist_y, dist_z;  // gradient reduction: neighbours from the overlaps, not wrapped
};

// LBM_BLOCK::computeInitialMacro (lbm_block.hpp:281-305); forces zeroed
template <int ST>
__global__ void k_compute_macro(const MacroArgs A)
{
	using S = Storage<ST>;
	using real = typename S::real;
	const int64_t n = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
	if (n >= A.X * A.Y * A.Z)
		return;
	const int64_t y = n % A.Y, t = n / A.Y, z = t % A.Z, x = t / A.Z;
	const int64_t s = ((x + A.ox) * A.Zs + (z + A.oz)) * A.Ys + (y + A.oy);
	real f[27];
#pragma unroll
	for (int q = 0; q < 27; q++)
		f[q] = S::ld((const typename S::elem*) A.df + q * A.XYZ + s, fx_sc(q, A.rs));
	real rho, vx, vy, vz;
	Phys<ST>::density_velocity(f, 0, 0, 0, rho, vx, vy, vz);
	if (A.macro_f64) {
		double* m = (double*) A.macro;
		m[s] = rho; m[A.XYZ + s] = vx; m[2 * A.XYZ + s] = vy; m[3 * A.XYZ + s] = vz;
	}
	else {
		float* m = (float*) A.macro;
		m[s] = rho; m[A.XYZ + s] = vx; m[2 * A.XYZ + s] = vy; m[3 * A.XYZ + s] = vz;
	}
}

template <int ST, int Q, bool EXPORT>
__global__ void k_transfer(void* df, double* buf, int64_t XYZ, int64_t nsites, const FixedRange R)
{
	using S = Storage<ST>;
	const int64_t s = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
	if (s >= nsites)
		return;
	auto* p = (typename S::elem*) df;
#pragma unroll
	for (int q = 0; q < Q; q++) {
		const double w = S::dev ? (Q == 27 ? w27(q) : (q == 0 ? 0.25 : 0.125)) : 0.0;
		if constexpr (EXPORT)
			buf[q * XYZ + s] = (double) S::ld(p + q * XYZ + s, fx_sc(q, R.rs)) + w;
		else
			S::st(p + q * XYZ + s, (typename S::real) (buf[q * XYZ + s] - w), fx_inv(q, R.invr));
	}
}

// FP64 reductions over the macro field: deterministic two-pass block sums
constexpr int RED_N = 6;
constexpr int RED_BLOCKS = 1024;
constexpr unsigned RED_THREADS = 256;

// v[0..N) summed over the block, in thread 0: shuffles within each wave, the
// waves' sums through LDS (blocks of up to 16 whole waves)
template <int N>
__device__ void block_sum(double* v)
{
	__shared__ double sh[16][N];
	const unsigned t = threadIdx.x;
#pragma unroll
	for (int i = 0; i < N; i++)
		for (int d = 32; d >= 1; d >>= 1)
			v[i] += __shfl_xor(v[i], d);
	if ((t & 63) == 0)
#pragma unroll
		for (int i = 0; i < N; i++)
			sh[t >> 6][i] = v[i];
	__syncthreads();
	if (t == 0)
		for (unsigned w = 1; w < blockDim.x / 64; w++)
#pragma unroll
			for (int i = 0; i < N; i++)
				v[i] += sh[w][i];
}

static __global__ void __launch_bounds__(RED_THREADS) k_reduce_macro(const MacroArgs A, double* partial)
{
	double v[RED_N] = {0, 0, 0, 0, 0, 0};
	const int64_t N = A.X * A.Y * A.Z;
	for (int64_t n = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; n < N; n += (int64_t) gridDim.x * blockDim.x) {
		const int64_t y = n % A.Y, t = n / A.Y, z = t % A.Z, x = t / A.Z;
		const int64_t s = ((x + A.ox) * A.Zs + (z + A.oz)) * A.Ys + (y + A.oy);
		double rho, vx, vy, vz;
		if (A.macro_f64) {
			const double* m = (const double*) A.macro;
			rho = m[s]; vx = m[A.XYZ + s]; vy = m[2 * A.XYZ + s]; vz = m[3 * A.XYZ + s];
		}
		else {
			const float* m = (const float*) A.macro;
			rho = m[s]; vx = m[A.XYZ + s]; vy = m[2 * A.XYZ + s]; vz = m[3 * A.XYZ + s];
		}
		const double u2 = vx * vx + vy * vy + vz * vz;
		v[0] += rho;
		v[1] += rho * u2;
		v[2] += (rho != rho) ? 1.0 : 0.0;
		v[3] += (rho - 1.0) * (rho - 1.0);
		v[4] += u2;
		v[5] += 1.0;
	}
	block_sum<RED_N>(v);
	if (threadIdx.x == 0)
#pragma unroll
		for (int i = 0; i < RED_N; i++)
			partial[blockIdx.x * RED_N + i] = v[i];
}

// Velocity-gradient reductions of sim_4.cu:282-300: with the central
// differences G_ab = (v_a(r + e_b) - v_a(r - e_b)) / 2 of computeGradVel
// (sim_4.cu:20-60; periodic wrap on an axis that is not distributed, the
// overlap layer on one that is), per block:
//   [0] sum rho |G|^2       (the enstrophy integrand of sim_4.cu:284-298)
//   [1] sum rho |curl v|^2  (computeVorticity, sim_4.cu:62-82)
//
// A lane owns one (y, z) column of a segment of `len` x planes and walks it, the
// velocities at x - 1 and x in registers, so that a plane is fetched once a
// segment; the y and z neighbours of a plane are the columns of the same block
// and of the next ones, found in L1 and (blocks of an XCD being consecutive) its
// L2.  Item = (segment, 256 columns).  192^3 FP64:
// 99 us with all 18 neighbours of a site loaded for it and its coordinates divided
// out of its index, 66 to 83 us so (2.8 to 3.4 TB/s; the slower after a step that
// leaves dirty lines in the last-level cache).  Bound: the latency of the loads.
// as many blocks as run at once at 74 VGPRs, six waves per SIMD (at 64 VGPRs, eight
// waves, it spills: 106 us against 79)
constexpr int GRAD_BLOCKS = 1536;
struct GradShape
{
	uint64_t tiles, items;
	int64_t len;
};
inline GradShape grad_shape(const MacroArgs& A)
{
	GradShape g;
	g.tiles = ((uint64_t) A.Y * (uint64_t) A.Z + RED_THREADS - 1) / RED_THREADS;
	const int64_t most = g.tiles >= (uint64_t) GRAD_BLOCKS ? 1 : (int64_t) ((uint64_t) GRAD_BLOCKS / g.tiles);
	const int64_t nseg = most < A.X ? most : A.X;
	g.len = (A.X + nseg - 1) / nseg;
	g.items = g.tiles * (uint64_t) ((A.X + g.len - 1) / g.len);
	return g;
}

// Off: type of a byte offset within an x plane (32 bits where it holds at most
// 4 GiB: scalar bases and one register per neighbour)
template <typename T, typename Off>
static __global__ void __launch_bounds__(RED_THREADS) k_reduce_gradients(const MacroArgs A, const GradShape S, double* partial)
{
	double v[2] = {0, 0};
	const uint64_t plane = (uint64_t) A.Zs * (uint64_t) A.Ys;
	// consecutive items on one XCD (GRAD_BLOCKS is a multiple of their number)
	for (uint64_t L = (blockIdx.x % NXCD) * (gridDim.x / NXCD) + blockIdx.x / NXCD; L < S.items; L += gridDim.x) {
		const uint64_t seg = L / S.tiles, i = (L % S.tiles) * RED_THREADS + threadIdx.x;
		if (i >= (uint64_t) A.Y * (uint64_t) A.Z)
			continue;
		const int64_t z = (int64_t) (i / (uint64_t) A.Y), y = (int64_t) (i % (uint64_t) A.Y);
		const int64_t yp = (! A.dist_y && y == A.Y - 1) ? 0 : y + 1, ym = (! A.dist_y && y == 0) ? A.Y - 1 : y - 1;
		const int64_t zp = (! A.dist_z && z == A.Z - 1) ? 0 : z + 1, zm = (! A.dist_z && z == 0) ? A.Z - 1 : z - 1;
		auto off = [&](int64_t zz, int64_t yy) { return (Off) (((zz + A.oz) * A.Ys + (yy + A.oy)) * (int64_t) sizeof(T)); };
		const Off o = off(z, y), oyp = off(z, yp), oym = off(z, ym), ozp = off(zp, y), ozm = off(zm, y);
		// field k of the x plane `base` sites into the array
		auto get = [&](int k, uint64_t base, Off at) {
			return *(const T*) ((const char*) ((const T*) A.macro + (k * A.XYZ + (int64_t) base)) + at);
		};
		const int64_t x0 = (int64_t) seg * S.len, x1 = x0 + S.len < A.X ? x0 + S.len : A.X;
		const int64_t before = (! A.dist_x && x0 == 0) ? A.X - 1 : x0 - 1;
		T vm[3], vc[3];
#pragma unroll
		for (int a = 0; a < 3; a++) {
			vm[a] = get(1 + a, (uint64_t) (before + A.ox) * plane, o);
			vc[a] = get(1 + a, (uint64_t) (x0 + A.ox) * plane, o);
		}
		for (int64_t x = x0; x < x1; x++) {
			const int64_t xp = (! A.dist_x && x == A.X - 1) ? 0 : x + 1;
			const uint64_t here = (uint64_t) (x + A.ox) * plane, next = (uint64_t) (xp + A.ox) * plane;
			T n[3][5];
#pragma unroll
			for (int a = 0; a < 3; a++) {
				n[a][0] = get(1 + a, next, o);
				n[a][1] = get(1 + a, here, oyp);
				n[a][2] = get(1 + a, here, oym);
				n[a][3] = get(1 + a, here, ozp);
				n[a][4] = get(1 + a, here, ozm);
			}
			const double rho = get(0, here, o);
			// all 16 loads in flight before the first is used
			__builtin_amdgcn_sched_barrier(0);
			double G[3][3];  // G[a][b] = d v_a / d x_b
#pragma unroll
			for (int a = 0; a < 3; a++) {
				G[a][0] = 0.5 * ((double) n[a][0] - (double) vm[a]);
				G[a][1] = 0.5 * ((double) n[a][1] - (double) n[a][2]);
				G[a][2] = 0.5 * ((double) n[a][3] - (double) n[a][4]);
				vm[a] = vc[a];
				vc[a] = n[a][0];
			}
			double g2 = 0;
#pragma unroll
			for (int a = 0; a < 3; a++)
#pragma unroll
				for (int b = 0; b < 3; b++)
					g2 += G[a][b] * G[a][b];
			const double wx = G[2][1] - G[1][2], wy = G[0][2] - G[2][0], wz = G[1][0] - G[0][1];
			v[0] += rho * g2;
			v[1] += rho * (wx * wx + wy * wy + wz * wz);
		}
	}
	block_sum<2>(v);
	if (threadIdx.x == 0) {
		partial[blockIdx.x * 2] = v[0];
		partial[blockIdx.x * 2 + 1] = v[1];
	}
}

// the sums of ROWS blocks to `out` (device memory, or host memory mapped into
// the device)
template <int N, int ROWS>
static __global__ void __launch_bounds__(1024) k_reduce_final(const double* partial, double* out)
{
	double v[N] = {};
	for (int r = threadIdx.x; r < ROWS; r += 1024)
#pragma unroll
		for (int i = 0; i < N; i++)
			v[i] += partial[r * N + i];
	block_sum<N>(v);
	if (threadIdx.x == 0)
#pragma unroll
		for (int i = 0; i < N; i++)
			out[i] = v[i];
}

// ===========================================================================
// Host side: validation and dispatch
// ===========================================================================
// Kernels that compute every lane's coordinates (k_general, k_nse_ade, the
// adjoint) can take the y-z plane of one x as one linear range, so that a row
// length that is not a multiple of the block (Y = 96, say) still fills every
// wave.  (k_aa_odd and k_lean choose between the two mappings at compile time.)
inline void linearize(StepArgs& A, unsigned& threads, unsigned& grid)
{
	if (A.nx == 0 || A.ny % (int32_t) threads == 0)
		return;
	threads = 256;
	const uint64_t plane = (uint64_t) A.ny * (uint64_t) A.nz;
	A.nyb = (uint32_t) ((plane + threads - 1) / threads);
	A.nblocks = A.nyb * (uint32_t) A.nx;  // no larger than the row mapping's count
	const uint32_t padded = padded_blocks(A);
	A.lin = 1;
	grid = padded;
}

// Launch shape over one row list of a full-box launch: whole rows per block
// where the row length is a multiple of the block, else the listed rows'
// sites one after another, as linearize does for the box.
inline void list_shape(StepArgs& A, const uint32_t* rows, uint32_t nrows, unsigned& threads, unsigned& grid)
{
	A.rows = rows;
	A.nrows = nrows;
	threads = A.ny > 128 ? 256 : (A.ny > 64 ? 128 : 64);
	if (A.ny % (int32_t) threads == 0) {
		A.lin = 0;
		A.nyb = (uint32_t) A.ny / threads;
		A.nblocks = A.nyb * nrows;
	}
	else {
		threads = 256;
		A.lin = 1;
		A.nyb = 1;
		A.nblocks = (uint32_t) (((uint64_t) nrows * (uint64_t) A.ny + threads - 1) / threads);
	}
	const uint32_t padded = padded_blocks(A);
	grid = padded;
}

// Whether a step finds a part of `planes` population planes in the last-level
// cache, where the step before it left them; nontemporal accesses give that up
// (300x50x300 F16, 243 MB: 204 us for the two steps with them, 153 without; with
// alternating order 128^3 FP64, 453 MB, 312 and 293; 48x320x320 FP64 slab, 1.1 GB,
// 811 and 791; 192^3 FP64, 1.5 GB, equal; 256^3 F32, 1.8 GB, 1286 and 1316).
// The rule takes a lattice to step alone.  Where other work between its steps takes
// the cache, it costs what it gains and more: two lattices stepped in turn, two steps
// of each, with hints / without: 128^3 F32 331 / 372 us, FP64 668 / 742, 160^3 FP64
// 1344 / 1402, 256x256x100 F16 542 / 595, 256x256x200 F16 1090 / 1148 (alone 152 / 141,
// 318 / 297, 653 / 621, 257 / 248, 528 / 501; in turn by two steps as alone).
inline bool cache_resident(const StepArgs& A, uint64_t planes = 27)
{
	return alternating(planes * A.plane_bytes) && ! planes_meet(A);
}
// Whether a step over `planes` population planes in all hints the streams that
// no other wave touches: rows and planes start on lines, and the last-level cache
// holds too little of the arrays.
inline bool hint_streams(const StepArgs& A, uint64_t planes, size_t elem)
{
	return ! cache_resident(A, planes) && A.plane_bytes % 128 == 0 && (uintptr_t) A.df0 % 128 == 0
		&& (uintptr_t) A.df1 % 128 == 0 && (uint64_t) A.Ys * elem % 128 == 0;
}

// Launch shape of an even A-A step with `per` sites per lane: the contiguous
// range where the box covers whole rows and columns of a lattice without y and
// z overlaps, else rows.  Returns whether to use nontemporal hints: where every
// wave's accesses cover whole lines (the planes and each wave's first site
// start on a 128-byte line) and the last-level cache holds too little of the arrays.
inline bool even_shape(StepArgs& A, uint32_t per, unsigned most, unsigned& threads, unsigned& grid, size_t elem)
{
	const bool planes = A.plane_bytes % 128 == 0 && (uintptr_t) A.df0 % 128 == 0 && ! cache_resident(A);
	bool whole;
	if (A.oy == 0 && A.oz == 0 && A.ny == A.Y && A.nz == A.Z) {
		A.flat = 1;
		A.flat0 = (A.offx + A.ox) * A.Y * A.Z;
		A.nflat = (int64_t) A.nx * A.Y * A.Z;
		// smaller blocks where there would be fewer than eight for each CU
		threads = most;
		while (threads > 64 && (uint64_t) A.nflat < (uint64_t) threads * per * 2048)
			threads /= 2;
		A.nblocks = (uint32_t) ((A.nflat + (int64_t) threads * per - 1) / (threads * per));
		whole = planes && (uint64_t) A.flat0 * elem % 128 == 0;
	}
	else {
		const uint32_t n = (uint32_t) A.ny / per;
		threads = n > 128 ? 256 : (n > 64 ? 128 : 64);
		A.nyb = (n + threads - 1) / threads;
		A.nblocks = A.nyb * (uint32_t) A.nz * (uint32_t) A.nx;  // no more blocks than one lane per site needs
		whole = planes && (uint64_t) A.Ys * elem % 128 == 0 && (uint64_t) (A.oy + A.offy) * elem % 128 == 0;
	}
	// Groups of 256 blocks for the 2-byte forms on planes of a power of two from 128 MiB
	// on, which meet in the same channels: groups of 32 / 256, us, 512^3 F16 2532 / 2419,
	// I16 2440 / 2289, 512x512x256 F16 1222 / 1165, 1024x512x512 I16 4811 / 4605.  Other
	// sizes are equal or slower so: 512x256x256 F16 585 / 598, 450x448x448 1722 / 1824,
	// 640x320x320 1362 / 1397, 301x187x129 159 / 159.
	const bool pow2 = A.plane_bytes >= 128ull << 20 && (A.plane_bytes & (A.plane_bytes - 1)) == 0;
	const uint32_t padded = padded_blocks(A, elem == 2 && pow2 ? 8 : 5);
	grid = padded;
	return whole;
}

// Whether rows in which walls and other sites may meet are common (class 2, an
// eighth of the rows or more): the pairs of such rows would be split
inline bool mixed_rows(const StepArgs& A)
{
	return A.list_count[2] * 8 > A.X * A.Z;
}

template <int ST, int COLL, bool MAP = false>
int even_launch(const StepArgs& A0, hipStream_t st)
{
	constexpr size_t E = sizeof(typename Storage<ST>::elem);
	StepArgs A = A0;
	unsigned threads = 0, grid = 0;
	if constexpr (E == 2 && ((LBM_PAIR_EVEN >> ST) & 1)) {
		// pairs must start at even stored offsets of every plane
		// (the fixed-point form takes them in even rows only: in odd rows its
		// stored integers stay those of the one-site kernel, whose fused
		// operations round 1 in 10^4 of them to the neighbouring unit)
		const bool flat = ! Storage<ST>::fixed && A.oy == 0 && A.oz == 0 && A.ny == A.Y && A.nz == A.Z;
		const int64_t odd = flat ? ((A.offx + A.ox) * A.Y * A.Z) | (A.nx * A.Y * A.Z) : A.ny | A.offy | A.oy | A.Y;
		if (! ((odd | A.XYZ) & 1) && ! ((uintptr_t) A.df0 & 3) && ! (MAP && mixed_rows(A))) {
			if (even_shape(A, 2, 256, threads, grid, E))
				hipLaunchKernelGGL((k_aa_even_pair<ST, COLL, true, MAP>), dim3(grid), dim3(threads), 0, st, A);
			else
				hipLaunchKernelGGL((k_aa_even_pair<ST, COLL, false, MAP>), dim3(grid), dim3(threads), 0, st, A);
			return hip_check(hipGetLastError(), "step launch");
		}
	}
	if (even_shape(A, 1, ST == TNL_LBM_STORE_F64 ? 256 : LBM_TPB_FP32, threads, grid, E))
		hipLaunchKernelGGL((k_aa_even<ST, COLL, true, MAP>), dim3(grid), dim3(threads), 0, st, A);
	else
		hipLaunchKernelGGL((k_aa_even<ST, COLL, false, MAP>), dim3(grid), dim3(threads), 0, st, A);
	return hip_check(hipGetLastError(), "step launch");
}

// The odd step: rows of whole blocks, else the linear mapping, whose waves are
// all full (even and odd step together: 320^3 FP64 5.26 -> 4.63 ms, 512x30x512
// F32 1042 -> 557 us, with the even step's flat range; where rows are whole
// blocks the scalar row offsets win, 512^3 F16 2.46 against 2.52 ms).
template <int ST, int COLL, bool NTO>
void odd_launch(const StepArgs& A0, unsigned threads, unsigned grid, hipStream_t st)
{
	StepArgs A = A0;
	if (A.ny % (int32_t) threads && plane_fits(A, sizeof(typename Storage<ST>::elem))) {
		threads = 256;
		const uint64_t plane = (uint64_t) A.ny * (uint64_t) A.nz;
		while (threads > 64 && plane * (uint64_t) A.nx < (uint64_t) threads * 2048)
			threads /= 2;
		A.nyb = (uint32_t) ((plane + threads - 1) / threads);
		A.nblocks = A.nyb * (uint32_t) A.nx;
		const uint32_t padded = padded_blocks(A);
		hipLaunchKernelGGL((k_aa_odd<ST, COLL, NTO, true>), dim3(padded), dim3(threads), 0, st, A);
		return;
	}
	if (ST != TNL_LBM_STORE_F64 && LBM_TPB_FP32 > 256 && A.ny % LBM_TPB_FP32 == 0) {
		threads = LBM_TPB_FP32;
		A.nyb = (uint32_t) A.ny / LBM_TPB_FP32;
		A.nblocks = A.nyb * (uint32_t) A.nz * (uint32_t) A.nx;  // fewer blocks than at 256
		grid = padded_blocks(A);
	}
	hipLaunchKernelGGL((k_aa_odd<ST, COLL, NTO, false>), dim3(grid), dim3(threads), 0, st, A);
}

// The map-free periodic A-A kernels
template <int ST, int COLL>
int launch_periodic(const StepArgs& A, unsigned threads, unsigned grid, hipStream_t st)
{
	if (A.even)
		return even_launch<ST, COLL>(A, st);
	// nontemporal hints on the c_y = 0 accesses where rows start on lines, as
	// in even_shape (301x187x129 FP64, both steps: 1428 us with them, 1377
	// without; 512^3: 18.79 and 18.96 ms)
	if (hint_streams(A, 27, sizeof(typename Storage<ST>::elem)))
		odd_launch<ST, COLL, true>(A, threads, grid, st);
	else
		odd_launch<ST, COLL, false>(A, threads, grid, st);
	return hip_check(hipGetLastError(), "step launch");
}

inline bool lists_cover(const StepArgs& A)
{
	return A.lists && A.list_count[0] + A.list_count[1] + A.list_count[2] == A.X * A.Z;
}

// In place, a site whose code pulls from another site's slots (OUTFLOW_RIGHT, and
// OUTFLOW_RIGHT_INTERP, from column x - 1) reads them as they were before the step
// if the rows that hold other codes are stepped first: in one launch the two sites
// race, and after it such a site reads the step's results.  So the A-A steps of the
// deviation forms and the coupled ones step those rows first, with the lean kernels
// or without (in_turn).  (FP64 and F32 flow steps go through one launch.)
inline bool in_order(const StepArgs& A, bool dev_or_coupled, int pattern)
{
	return dev_or_coupled && pattern == TNL_LBM_PATTERN_AA && A.list_count[0] > 0 && A.list_count[0] < A.X * A.Z;
}

// Whether a full-box launch with row lists takes the lean kernels: x planes
// within 32-bit offsets, and few rows with other codes (each of those is read
// again by the general kernel; from an eighth of the rows on, that launch costs
// what the lean one saves).  Steps that keep the order need two launches
// anyhow: up to a quarter.  A-A F16 128x128 rows, flow / coupled, us for two
// steps, lean and in turn: 64 planes, a fifth of the rows 74 / 89 and 78 / 111,
// half 91 / 108 and 81 / 109 (in one launch, out of order, 68 / 93 and 68 / 97).
inline bool lean_split(const StepArgs& A, size_t elem, bool ordered)
{
	return lists_cover(A) && plane_fits(A, elem) && A.list_count[0] * (ordered ? 4 : 8) <= A.X * A.Z;
}

// The rows that hold other codes in one launch of the general kernel, then the rest
// in another.  go(shape, threads, grid) makes a launch.
template <typename Go>
int in_turn(const StepArgs& A, Go&& go)
{
	const int64_t first = A.list_count[0];
	const int64_t rest = A.X * A.Z - first;
	for (int k = 0; k < 2; k++) {
		StepArgs B = A;
		unsigned threads = 0, grid = 0;
		list_shape(B, A.lists + (k ? first : 0), (uint32_t) (k ? rest : first), threads, grid);
		if (int rc = go(B, threads, grid))
			return rc;
	}
	return 0;
}

// Launch shape of a lean kernel: rows of whole blocks with hints, else the
// linear mapping without.  go(shape, threads, grid, lin).
template <typename Go>
void lean_shape(const StepArgs& A0, uint64_t planes, size_t elem, Go&& go)
{
	StepArgs A = A0;
	A.rows = nullptr;
	unsigned threads = A.ny > 128 ? 256 : (A.ny > 64 ? 128 : 64);
	const bool lin = A.ny % (int32_t) threads || ! hint_streams(A, planes, elem);
	if (lin) {
		const uint64_t plane = (uint64_t) A.ny * (uint64_t) A.nz;
		threads = 256;
		while (threads > 64 && plane * (uint64_t) A.nx < (uint64_t) threads * 2048)
			threads /= 2;
		A.nyb = (uint32_t) ((plane + threads - 1) / threads);
		A.nblocks = A.nyb * (uint32_t) A.nx;
	}
	else {
		A.nyb = (uint32_t) A.ny / threads;
		A.nblocks = A.nyb * (uint32_t) A.nz * (uint32_t) A.nx;
	}
	const uint32_t padded = padded_blocks(A);
	go(A, threads, padded, lin);
}

template <int ST, int MODE>
void lean_launch(const StepArgs& A, hipStream_t st)
{
	lean_shape(A, MODE == LEAN_AB ? 54 : 27, sizeof(typename Storage<ST>::elem),
			   [&](const StepArgs& C, unsigned t, unsigned g, bool lin) {
				   if (lin)
					   hipLaunchKernelGGL((k_lean<ST, MODE, true, false>), dim3(g), dim3(t), 0, st, C);
				   else
					   hipLaunchKernelGGL((k_lean<ST, MODE, false, true>), dim3(g), dim3(t), 0, st, C);
			   });
}

// One launch of the map kernel
template <int ST, int COLL, bool LISTED>
void launch_general(int pattern, const StepArgs& B, unsigned threads, unsigned grid, hipStream_t st)
{
	constexpr bool two = sizeof(typename Storage<ST>::elem) == 2;
	// 2-byte forms: 32-bit slot offsets where a population array is under
	// 4 GiB (F16 384^3 channel: A-A 1821 -> 1430 us, 139 -> 106 VGPRs;
	// A-B -2%; neutral for the 4- and 8-byte forms, which keep 64-bit)
	const bool o32 = two && narrow_slots(B.XYZ, sizeof(typename Storage<ST>::elem));
	const bool nt = ! LISTED && pattern == TNL_LBM_PATTERN_AB && hint_streams(B, 54, sizeof(typename Storage<ST>::elem));
	auto go = [&](auto oc) {
		constexpr bool O32 = decltype(oc)::value;
		if (pattern == TNL_LBM_PATTERN_AA)
			hipLaunchKernelGGL((k_general<ST, COLL, TNL_LBM_PATTERN_AA, 0, O32, LISTED>), dim3(grid), dim3(threads), 0, st, B);
		else if (! nt)
			hipLaunchKernelGGL((k_general<ST, COLL, TNL_LBM_PATTERN_AB, 0, O32, LISTED>), dim3(grid), dim3(threads), 0, st, B);
		else if constexpr (! LISTED)
			hipLaunchKernelGGL((k_general<ST, COLL, TNL_LBM_PATTERN_AB, 0, O32, false, true>), dim3(grid), dim3(threads), 0, st, B);
	};
	if constexpr (two) {
		if (o32) {
			go(std::true_type{});
			return;
		}
	}
	go(std::false_type{});
}

template <int ST, int COLL>
int launch_step(const tnl_lbm_config* cfg, const StepArgs& A, unsigned threads, unsigned grid, hipStream_t st)
{
	// the map-free periodic kernels take the homogeneous force only
	if (! A.map && ! A.force && cfg->pattern == TNL_LBM_PATTERN_AA)
		return launch_periodic<ST, COLL>(A, threads, grid, st);
	// The rows that hold other codes (in_order says why first), then the lean
	// kernels for the plain sites.
	// FP64 and F32 take them where there are no such rows: their map kernel is bound
	// by HBM, and the second launch costs more than it gains (A-A ducts, two steps,
	// with it / in one launch: FP64 24^3 28 / 22 us, 64^3 56 / 51, 160x128x128 396 /
	// 386; F32 24^3 26 / 19, 200x131x128 272 / 256).
	if constexpr (COLL == TNL_LBM_COLL_CUM) {
		constexpr bool DEV = Storage<ST>::dev;
		const bool ordered = in_order(A, DEV, cfg->pattern);
		if (lean_split(A, sizeof(typename Storage<ST>::elem), ordered) && (DEV || A.list_count[0] == 0)) {
			if constexpr (DEV) {
				if (A.list_count[0] > 0) {
					StepArgs B = A;
					B.others = 1;
					list_shape(B, A.lists, (uint32_t) A.list_count[0], threads, grid);
					launch_general<ST, COLL, true>(cfg->pattern, B, threads, grid, st);
					if (int rc = hip_check(hipGetLastError(), "step launch"))
						return rc;
				}
			}
			if (cfg->pattern == TNL_LBM_PATTERN_AB)
				lean_launch<ST, LEAN_AB>(A, st);
			else if (! A.even)
				lean_launch<ST, LEAN_ODD>(A, st);
			else
				return even_launch<ST, COLL, true>(A, st);
			return hip_check(hipGetLastError(), "step launch");
		}
		if constexpr (DEV) {
			if (ordered && lists_cover(A))
				return in_turn(A, [&](const StepArgs& B, unsigned t, unsigned g) {
					launch_general<ST, COLL, true>(cfg->pattern, B, t, g, st);
					return hip_check(hipGetLastError(), "step launch");
				});
		}
	}
	StepArgs B = A;
	linearize(B, threads, grid);
	launch_general<ST, COLL, false>(cfg->pattern, B, threads, grid, st);
	return hip_check(hipGetLastError(), "step launch");
}

// launches of the alternative operators (MRT_LES, KBC), built in lbm_alt.hip
int launch_alt(const tnl_lbm_config* cfg, const StepArgs& A, unsigned threads, unsigned grid, hipStream_t st);

}  // namespace lbm
