/*
 * FP64 tree walks, a lane or a team of lanes per active particle,
 * reproducing the reference's per-particle decisions and summation order:
 *   k_walk64        Gravity_Tree_Acceleration (Gravity/tree_accel.c:32-394):
 *                   top-node loop, gravity_tree_walk (relative criterion +
 *                   "inside" test) or gravity_tree_walk_BH, interact()
 *   k_walk64_ewald  Gravity_Tree_Periodic (Gravity/tree_periodic.c:23-450)
 *                   with Ewald_Correction (Gravity/periodic.c:35-113)
 * Opening decisions use the same FP64 expressions in the same order as the
 * reference, so the interaction set and P.Cost are identical; the build is
 * compiled without FP contraction so every product and sum rounds once.
 * Lanes of a wavefront are PH neighbours whose walks visit nearly the same
 * nodes, so the wavefront walks in lockstep (see k_walk64): node and
 * particle records are loaded once per wavefront through the scalar cache.
 */
#include "tdv_internal.h"
#include "tdv_device.h"
#include <climits>

struct WalkParams {
	int ntop, vs, compat, periodic, use_bh;
	double G, theta_bh, theta_bh2, alpha_rel, eps2, eps3, box, boxhalf;
	double dom_size, box2ewald;
};

/* Periodic_Nearest (periodic.c:62-80) */
__device__ __forceinline__ double wrap(double d, const WalkParams &w)
{
	if (!w.periodic)
		return d;
	if (d > w.boxhalf)
		d -= w.box;
	else if (d < -w.boxhalf)
		d += w.box;
	return d;
}

struct Acc {
	double x, y, z;
	int cost;                        /* interactions */
};

/* sum of P.Cost over the launch: one atomic per wavefront */
__device__ __forceinline__ void count_interactions(int cost,
		unsigned long long *counter)
{
	unsigned long long v = (unsigned long long)cost;
	for (int d = 32; d >= 1; d >>= 1)
		v += __shfl_xor(v, d, 64);
	if ((threadIdx.x & 63) == 0 && v)
		atomicAdd(counter, v);
}

/* the factor of an interaction, interact (Gravity/tree_accel.c:362-394):
 * Dehnen K1 kernel, h < 0 */
__device__ __forceinline__ double kernel_fac(double m, double r2,
		const WalkParams &w)
{
	double fac = w.G * m;
	if (r2 < w.eps2) {
		const double u2 = r2 / w.eps2;
		fac *= (175 - u2 * (294 - u2 * 135)) / (16 * w.eps3);
	} else {
		bool ok;
		double r_inv = inv_sqrt(r2, &ok);
		if (!ok)
			r_inv = 1 / sqrt(r2);
		fac *= r_inv * r_inv * r_inv;
	}
	return fac;
}

__device__ __forceinline__ void interact(Acc &a, double m, double dx,
		double dy, double dz, double r2, const WalkParams &w)
{
	const double fac = kernel_fac(m, r2, w);
	a.x += fac * dx;
	a.y += fac * dy;
	a.z += fac * dz;
	a.cost++;
}

/* ---- lane teams -----------------------------------------------------------
 *
 * L lanes work for one particle: a bundle's particles are dealt out to them
 * L at a time, each lane forms one particle's contribution, and the team's
 * lanes then all add the L contributions in particle order, taken from one
 * another by DPP, so the sums round exactly as one lane's would.  A walk is
 * one long chain of interactions per particle; with one lane each, a few
 * thousand particles are a few wavefronts that leave most SIMDs idle and
 * have nothing to hide an interaction's latency behind. */
template <int ctrl>
__device__ __forceinline__ double dpp_f64(double v)
{
	const uint64_t u = (uint64_t)__double_as_longlong(v);
	const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, ctrl, 0xf,
			0xf, false);
	const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), ctrl, 0xf,
			0xf, false);
	return __longlong_as_double((long long)((uint64_t)(uint32_t)hi << 32
			| (uint32_t)lo));
}

/* the value of the team's lane S: quad_perm(S, S, S, S) in teams of 4,
 * row_newbcast S in teams of 16 (a DPP row) */
template <int L, int S>
__device__ __forceinline__ double team_lane(double v)
{
	return dpp_f64<L == 4 ? S * 0x55 : 0x150 + S>(v);
}

/* a += the contributions of the team's lanes S .. S + 3, in lane order (a
 * lane without one holds zeros, which change no sum) */
template <int L, int S>
__device__ __forceinline__ void team_add4(Acc &a, double x, double y, double z)
{
	a.x += team_lane<L, S>(x);
	a.y += team_lane<L, S>(y);
	a.z += team_lane<L, S>(z);
	a.x += team_lane<L, S + 1>(x);
	a.y += team_lane<L, S + 1>(y);
	a.z += team_lane<L, S + 1>(z);
	a.x += team_lane<L, S + 2>(x);
	a.y += team_lane<L, S + 2>(y);
	a.z += team_lane<L, S + 2>(z);
	a.x += team_lane<L, S + 3>(x);
	a.y += team_lane<L, S + 3>(y);
	a.z += team_lane<L, S + 3>(z);
}

/* a += the first `count` (uniform) of the team's contributions */
template <int L>
__device__ __forceinline__ void team_add(Acc &a, double x, double y, double z,
		bool hit, int count)
{
	team_add4<L, 0>(a, x, y, z);
	if constexpr (L == 16) {
		if (count > 4)
			team_add4<L, 4>(a, x, y, z);
		if (count > 8)
			team_add4<L, 8>(a, x, y, z);
		if (count > 12)
			team_add4<L, 12>(a, x, y, z);
	}
	const uint64_t hits = __ballot(hit) >> (threadIdx.x & 63 & ~(L - 1));
	a.cost += __popcll(hits & ((1ull << L) - 1));
}

/* The factors of U interactions with r2 > 0 (kernel_fac): the roots and
 * divisions, which are most of an interaction, as independent chains */
template <int U>
__device__ __forceinline__ void kernel_facs(double (&fac)[U],
		const double (&m)[U], const double (&r2)[U], const WalkParams &w)
{
	bool all = true;
#pragma unroll
	for (int u = 0; u < U; u++) {
		bool ok;
		const double r_inv = inv_sqrt(r2[u], &ok);
		fac[u] = w.G * m[u];
		fac[u] *= r_inv * r_inv * r_inv;
		all = all && ok && !(r2[u] < w.eps2);
	}
	if (!all) {
#pragma unroll
		for (int u = 0; u < U; u++)
			fac[u] = kernel_fac(m[u], r2[u], w);
	}
}

/* P-P with U particles of a uniform range, in the reference's order */
template <int U>
__device__ __forceinline__ void pp_batch(Acc &a, const double4 (&q)[U],
		double px, double py, double pz, const WalkParams &w)
{
	double dx[U], dy[U], dz[U], r2[U], m[U], fac[U];
	bool self = false;
#pragma unroll
	for (int u = 0; u < U; u++) {
		dx[u] = wrap(q[u].x - px, w);
		dy[u] = wrap(q[u].y - py, w);
		dz[u] = wrap(q[u].z - pz, w);
		r2[u] = dx[u] * dx[u] + dy[u] * dy[u] + dz[u] * dz[u];
		m[u] = q[u].w;
		self = self || r2[u] == 0;
	}
	if (self) {
#pragma unroll
		for (int u = 0; u < U; u++)
			if (r2[u] != 0)
				interact(a, m[u], dx[u], dy[u], dz[u], r2[u], w);
		return;
	}
	kernel_facs<U>(fac, m, r2, w);
#pragma unroll
	for (int u = 0; u < U; u++) {
		a.x += fac[u] * dx[u];
		a.y += fac[u] * dy[u];
		a.z += fac[u] * dz[u];
	}
	a.cost += U;
}

/* P-P with the particles [first, last) for the lanes with `on` (a team's
 * alike), in the reference's order; the range is the wavefront's, so one
 * lane per particle loads uniformly */
template <int L>
__device__ __forceinline__ void pp_range_on(Acc &a, const double4 *pm,
		int first, int last, double px, double py, double pz, bool on,
		const WalkParams &w)
{
	if constexpr (L == 1) {
		int j = first;
		for (; j + 4 <= last; j += 4) {
			const double4 q[4] = { pm[j], pm[j + 1], pm[j + 2], pm[j + 3] };
			if (on)
				pp_batch<4>(a, q, px, py, pz, w);
		}
		for (; j < last; j++) {
			const double4 q[1] = { pm[j] };
			if (on)
				pp_batch<1>(a, q, px, py, pz, w);
		}
	} else {
		const int sub = threadIdx.x & (L - 1);
		double4 n = pm[min(first + sub, last - 1)];
		for (int j = first; j < last; j += L) {
			const double4 q = n;
			n = pm[min(j + L + sub, last - 1)];
			if (!on)
				continue;
			const double dx = wrap(q.x - px, w), dy = wrap(q.y - py, w),
					dz = wrap(q.z - pz, w);
			const double r2 = dx * dx + dy * dy + dz * dz;
			const bool hit = j + sub < last && r2 != 0;
			const double m[1] = { q.w }, d2[1] = { hit ? r2 : 1.0 };
			double fac[1];
			kernel_facs<1>(fac, m, d2, w);
			team_add<L>(a, hit ? fac[0] * dx : 0.0, hit ? fac[0] * dy : 0.0,
					hit ? fac[0] * dz : 0.0, hit, last - j);
		}
	}
}

/* min of v and the value DPP control `ctrl` moves into this lane (INT_MAX
 * where nothing arrives) */
template <int ctrl, int rows>
__device__ __forceinline__ int dpp_min(int v)
{
	const int o = __builtin_amdgcn_update_dpp(INT_MAX, v, ctrl, rows, 0xf,
			false);
	return o < v ? o : v;
}

/* The wavefront's minimum, in registers: a prefix minimum by DPP (row_shr
 * 1, 2, 4, 8 within rows of 16, row_bcast 15 and 31 across rows) leaves
 * it in lane 63.  Every lane of the wavefront takes part. */
__device__ __forceinline__ int wave_min(int v)
{
	v = dpp_min<0x111, 0xf>(v);
	v = dpp_min<0x112, 0xf>(v);
	v = dpp_min<0x114, 0xf>(v);
	v = dpp_min<0x118, 0xf>(v);
	v = dpp_min<0x142, 0xa>(v);
	v = dpp_min<0x143, 0xc>(v);
	return __builtin_amdgcn_readlane(v, 63);
}

/* A team of L lanes per active particle, taking exactly the reference's
 * walk: its own decisions, its own interactions in its own order.  The
 * wavefront walks in lockstep: each lane keeps the next node of its walk,
 * the wavefront takes the smallest of them (walks only move forward in
 * the depth-first array), loads that node once through the scalar cache,
 * and the lanes whose next node it is act on it; the others wait.  PH
 * neighbours' walks share most nodes, so the wavefront visits little more
 * than one walk's nodes, without the per-lane gathers and divergent
 * branches of independent loops. */
/* Bound by instruction latency and, in the tail, by the longest walks.  With
 * the periodic switch a constant and the short inverse root (inv_sqrt) the
 * Hernquist sphere of 65536 takes 2.5 ms instead of 3.0, 14000 particles 1.2
 * instead of 1.5, the box of 64^3 126 instead of 157.  Two particles per
 * lane and turn gained nothing (and 24 registers more), nor did loading a
 * node's three records at once. */
template <int L, bool PERIODIC>
__global__ void __launch_bounds__(256) k_walk64(int nact,
		const int *__restrict__ active, const double4 *__restrict__ pm,
		const double *__restrict__ last_acc, TopNodes T,
		const double4 *__restrict__ na, const double4 *__restrict__ nb,
		const int4 *__restrict__ nc, WalkParams w, double *__restrict__ ax,
		double *__restrict__ ay, double *__restrict__ az,
		double *__restrict__ gx, double *__restrict__ gy,
		double *__restrict__ gz, double *__restrict__ cost, int npart_total,
		unsigned *err, unsigned long long *counter)
{
	w.periodic = PERIODIC;               /* a constant */
	const int gid = (int)((blockIdx.x * blockDim.x + threadIdx.x) / L);
	const bool live = gid < nact;
	const int ip = live ? active[gid] : 0;
	const double4 p = pm[ip];
	const double fac = last_acc[ip] / w.G * w.alpha_rel;
	Acc a = { 0, 0, 0, 0 };

	for (int j = 0; j < w.ntop; j++) {
		/* interact_with_topnode, Gravity/tree_accel.c:137-176 */
		const double nSize = w.dom_size / ((double)(1ull << T.level[j]));
		bool walk = false;
		if (live) {
			const double dx = (double)T.pos[3 * j] - p.x;
			const double dy = (double)T.pos[3 * j + 1] - p.y;
			const double dz = (double)T.pos[3 * j + 2] - p.z;
			const bool inside = fabs(dx) < 0.6 * nSize && fabs(dy) < 0.6 * nSize
					&& fabs(dz) < 0.6 * nSize;
			walk = inside;
			if (!inside) {
				const double rx = wrap((double)T.com[3 * j] - p.x, w);
				const double ry = wrap((double)T.com[3 * j + 1] - p.y, w);
				const double rz = wrap((double)T.com[3 * j + 2] - p.z, w);
				const double r2 = rx * rx + ry * ry + rz * rz;
				const double m = (double)T.mass[j];
				const bool open = w.use_bh ? (nSize * nSize > r2 * w.theta_bh)
						: (m * nSize * nSize > r2 * r2 * fac);
				if (open)
					walk = true;
				else
					interact(a, m, rx, ry, rz, r2, w);
			}
		}
		if (!__any(walk))
			continue;
		if (T.npart[j] <= w.vs) {
			/* interact_with_topnode_particles, tree_accel.c:183-203 */
			const int f = w.compat ? T.target[j] : T.first[j];
			if (f < 0 || f + T.npart[j] > npart_total) {
				if (walk)
					atomicOr(err, TDV_EBIT_RANGE);
				continue;
			}
			pp_range_on<L>(a, pm, f, f + T.npart[j], p.x, p.y, p.z, walk, w);
			continue;
		}
		/* gravity_tree_walk(_BH), Gravity/tree_accel.c:211-353 */
		const int start = T.target[j], term = T.term[j];
		int next = walk ? start : INT_MAX;
		for (;;) {
			const int node = wave_min(next);
			if (node == INT_MAX)
				break;
			if (node < start || node > term) {  /* never for a valid tree */
				atomicOr(err, TDV_EBIT_RANGE);
				break;
			}
			const bool mine = next == node;
			const int4 c = nc[node];
			if (c.x == 0) {                     /* the terminator */
				if (node == start)
					atomicOr(err, TDV_EBIT_RANGE);
				if (mine)
					next = INT_MAX;
				continue;
			}
			if (c.x < 0) {
				const int f = -c.x - 1;
				if (f + c.y > npart_total) {
					atomicOr(err, TDV_EBIT_RANGE);
					break;
				}
				pp_range_on<L>(a, pm, f, f + c.y, p.x, p.y, p.z, mine, w);
				if (mine)
					next = node + 1;
				continue;
			}
			const double4 A = na[node];
			const double4 B = nb[node];
			if (!mine)
				continue;
			const double rx = wrap(A.x - p.x, w), ry = wrap(A.y - p.y, w),
					rz = wrap(A.z - p.z, w);
			const double r2 = rx * rx + ry * ry + rz * rz;
			const double m = A.w;
			const double s = B.w;
			bool open;
			if (w.use_bh) {
				open = s * s > r2 * w.theta_bh;
			} else {
				open = m * s * s > r2 * r2 * fac;
				if (!open) {
					const double sx = wrap(B.x - p.x, w),
							sy = wrap(B.y - p.y, w), sz = wrap(B.z - p.z, w);
					open = fabs(sx) < 0.6 * s && fabs(sy) < 0.6 * s
							&& fabs(sz) < 0.6 * s;
				}
			}
			if (open) {
				next = node + 1;
			} else {
				interact(a, m, rx, ry, rz, r2, w);
				next = node + c.x;
			}
		}
	}
	/* add_recv_to, Gravity/tree_accel.c:110-129 */
	const bool mine = live && (threadIdx.x & (L - 1)) == 0;
	if (mine) {
		ax[ip] = ax[ip] + a.x;
		ay[ip] = ay[ip] + a.y;
		az[ip] = az[ip] + a.z;
		gx[ip] = a.x;
		gy[ip] = a.y;
		gz[ip] = a.z;
		cost[ip] = (double)a.cost;
	}
	count_interactions(mine ? a.cost : 0, counter);
}

__device__ __forceinline__ void ewald_cube(Acc &a, const double *tab,
		double dx, double dy, double dz, double m, const WalkParams &w)
{
	double f[3];
	ewald_corr_rows(tab, dx, dy, dz, w.box2ewald, f);
	a.x += w.G * m * f[0];
	a.y += w.G * m * f[1];
	a.z += w.G * m * f[2];
	a.cost++;
}

/* as pp_range_on, with the Ewald correction of each pair.  One lane per
 * particle takes one pair at a time: with two gathers in flight it held 170
 * registers instead of 102, two wavefronts per SIMD instead of four, and the
 * walk of 256^3 particles took 1077 ms instead of 978. */
template <int L>
__device__ __forceinline__ void ewald_pp_range_on(Acc &a, const double *tab,
		const double4 *pm, int first, int last, double px, double py,
		double pz, bool on, const WalkParams &w)
{
	if constexpr (L == 1) {
		for (int j = first; j < last; j++) {
			const double4 q = pm[j];
			if (!on)
				continue;
			const double dx = wrap(q.x - px, w), dy = wrap(q.y - py, w),
					dz = wrap(q.z - pz, w);
			if (dx != 0 && dy != 0 && dz != 0)
				ewald_cube(a, tab, dx, dy, dz, q.w, w);
		}
	} else {
		const int sub = threadIdx.x & (L - 1);
		double4 n = pm[min(first + sub, last - 1)];
		for (int j = first; j < last; j += L) {
			const double4 q = n;
			n = pm[min(j + L + sub, last - 1)];
			if (!on)
				continue;
			const double dx = wrap(q.x - px, w), dy = wrap(q.y - py, w),
					dz = wrap(q.z - pz, w);
			const bool hit = j + sub < last && dx != 0 && dy != 0 && dz != 0;
			double f[3];
			ewald_corr_rows(tab, dx, dy, dz, w.box2ewald, f);
			team_add<L>(a, hit ? w.G * q.w * f[0] : 0.0,
					hit ? w.G * q.w * f[1] : 0.0,
					hit ? w.G * q.w * f[2] : 0.0, hit, last - j);
		}
	}
}

/* Gravity_Tree_Periodic by lane teams, in lockstep as k_walk64 */
template <int L>
__global__ void __launch_bounds__(256) k_walk64_ewald(int nact,
		const int *__restrict__ active, const double4 *__restrict__ pm,
		const double *__restrict__ last_acc, TopNodes T,
		const double4 *__restrict__ na, const double4 *__restrict__ nb,
		const int4 *__restrict__ nc, const double *__restrict__ tab,
		WalkParams w, double *__restrict__ ax, double *__restrict__ ay,
		double *__restrict__ az, double *__restrict__ gx,
		double *__restrict__ gy, double *__restrict__ gz,
		double *__restrict__ cost, int npart_total, unsigned *err,
		unsigned long long *counter)
{
	w.periodic = 1;                      /* a constant */
	const int gid = (int)((blockIdx.x * blockDim.x + threadIdx.x) / L);
	const bool live = gid < nact;
	const int ip = live ? active[gid] : 0;
	const double4 p = pm[ip];
	const double fac = last_acc[ip] / w.G * w.alpha_rel;
	Acc a = { 0, 0, 0, 0 };

	for (int j = 0; j < w.ntop; j++) {
		/* interact_with_topnode, Gravity/tree_periodic.c:112-177 */
		const double s = w.dom_size / (double)(1ull << T.level[j]);
		bool walk = false;
		if (live) {
			bool want_open = false;
			const double rx = wrap((double)T.com[3 * j] - p.x, w);
			const double ry = wrap((double)T.com[3 * j + 1] - p.y, w);
			const double rz = wrap((double)T.com[3 * j + 2] - p.z, w);
			const double r2 = rx * rx + ry * ry + rz * rz;
			if (w.use_bh) {
				if (s * s > r2 * w.theta_bh)
					want_open = true;
			} else {
				const double m = (double)T.mass[j];
				if (m * s * s > r2 * r2 * fac)
					want_open = true;
			}
			if (fabs(p.x - (double)T.pos[3 * j]) < 0.6 * s
					&& fabs(p.y - (double)T.pos[3 * j + 1]) < 0.6 * s
					&& fabs(p.z - (double)T.pos[3 * j + 2]) < 0.6 * s)
				want_open = true;
			/* a node that wants opening is walked only when it straddles
			 * the half box or is larger than 0.2 box; otherwise the
			 * correction of its centre of mass is used */
			if (want_open) {
				const double lim = 0.5 * (w.box - s);
				walk = fabs(rx) > lim || fabs(ry) > lim || fabs(rz) > lim
						|| s > 0.2 * w.box;
			}
			if (!walk)
				ewald_cube(a, tab, rx, ry, rz, (double)T.mass[j], w);
		}
		if (!__any(walk))
			continue;
		if (T.npart[j] <= w.vs) {
			const int f = w.compat ? T.target[j] : T.first[j];
			if (f < 0 || f + T.npart[j] > npart_total) {
				if (walk)
					atomicOr(err, TDV_EBIT_RANGE);
				continue;
			}
			ewald_pp_range_on<L>(a, tab, pm, f, f + T.npart[j], p.x, p.y, p.z,
					walk, w);
			continue;
		}
		/* gravity_tree_walk_ewald(_BH), Gravity/tree_periodic.c:216-422 */
		const int start = T.target[j];
		const int end = start + nc[start].x;
		if (end != T.term[j]) {
			if (walk)
				atomicOr(err, TDV_EBIT_RANGE);
			continue;
		}
		int next = walk ? start : INT_MAX;
		for (;;) {
			const int node = wave_min(next);
			if (node == INT_MAX)
				break;
			if (node < start || node >= end) {   /* never for a valid tree */
				atomicOr(err, TDV_EBIT_RANGE);
				break;
			}
			const bool mine = next == node;
			const int4 c = nc[node];
			if (c.x < 0) {
				const int f = -c.x - 1;
				if (f + c.y > npart_total) {
					atomicOr(err, TDV_EBIT_RANGE);
					break;
				}
				ewald_pp_range_on<L>(a, tab, pm, f, f + c.y, p.x, p.y, p.z, mine,
						w);
				if (mine)
					next = node + 1 == end ? INT_MAX : node + 1;
				continue;
			}
			const double4 A = na[node];
			const double4 B = nb[node];
			if (!mine)
				continue;
			const double dx = wrap(A.x - p.x, w), dy = wrap(A.y - p.y, w),
					dz = wrap(A.z - p.z, w);
			const double d2 = dx * dx + dy * dy + dz * dz;
			const double m = A.w;
			const double ns = B.w;
			const double sx = B.x - p.x, sy = B.y - p.y, sz = B.z - p.z;
			bool open = w.use_bh ? (ns * ns > d2 * w.theta_bh2)
					: (m * ns * ns > d2 * d2 * fac);
			if (!open && fabs(sx) < 0.6 * ns && fabs(sy) < 0.6 * ns
					&& fabs(sz) < 0.6 * ns)
				open = true;
			int to;
			if (open) {
				const double lim = 0.5 * (w.box - ns);
				if (fabs(wrap(sx, w)) > lim || fabs(wrap(sy, w)) > lim
						|| fabs(wrap(sz, w)) > lim || ns > 0.2 * w.box)
					to = node + 1;
				else
					to = -1;
			} else {
				to = -1;
			}
			if (to < 0) {
				ewald_cube(a, tab, dx, dy, dz, m, w);
				to = node + c.x;
			}
			next = to == end ? INT_MAX : to;
		}
	}
	/* add_recv_to, Gravity/tree_periodic.c:91-110 */
	const bool mine = live && (threadIdx.x & (L - 1)) == 0;
	if (mine) {
		ax[ip] = ax[ip] + a.x;
		ay[ip] = ay[ip] + a.y;
		az[ip] = az[ip] + a.z;
		gx[ip] = gx[ip] + a.x;
		gy[ip] = gy[ip] + a.y;
		gz[ip] = gz[ip] + a.z;
		cost[ip] = cost[ip] + (double)a.cost;
	}
	count_interactions(mine ? a.cost : 0, counter);
}

static WalkParams walk_params(const tdv_context *c, int use_bh)
{
	WalkParams w;
	w.ntop = c->ntop;
	w.vs = c->par.vector_size;
	w.compat = c->par.compat;
	w.periodic = c->par.periodic;
	w.use_bh = use_bh;
	w.G = c->par.gravity;
	w.theta_bh = c->par.theta_bh;
	w.theta_bh2 = c->par.theta_bh * c->par.theta_bh;
	w.alpha_rel = c->par.alpha_rel;
	w.eps2 = c->Epsilon2;
	w.eps3 = c->Epsilon3;
	w.box = c->par.boxsize;
	w.boxhalf = c->par.boxsize / 2.0;
	w.dom_size = c->dom_size;
	w.box2ewald = 2 * TDV_NE / c->par.boxsize;
	return w;
}

/* Lanes per particle and threads per workgroup.  Teams buy wavefronts and
 * idle less in the lockstep (fewer particles per wavefront to wait for);
 * they pay with L instead of one addition per component for each of the
 * wavefront's pairs, and with L lanes that test every node alike.
 *
 * Newton walk, ms for teams of 1, 4 and 16: Hernquist 8192: 1.35, 0.88,
 * 0.79; 14000: 1.83, 1.21, 1.48; 30000: 2.35, 1.91, 2.42; 65536: 2.48, 2.50,
 * 3.84; 10^6: 15.2, 15.1, 26.5; periodic box 24^3: 3.79, 1.96, 2.47; 40^3:
 * 16.7, 17.8, 32.5; 64^3: 126, 191, 393.  So teams of 4 up to three quarters
 * of a wavefront per SIMD with one lane each (49152 particles), of 16 up to
 * 10240.  A wavefront per workgroup spreads few of them over more CUs; the
 * large walks keep four neighbours on one CU, which share its scalar cache
 * (64^3: 182 ms apart, 157 together, then).
 *
 * Ewald walk, ms for one lane, teams of 4 and of 16: box of 20^3: 4.97, 2.00,
 * 1.65; 24^3: 8.32, 3.62, 3.69; 32^3: 21.1, 13.2, 14.7; of 10^6 uniform
 * particles 10000: 12.1, 5.6 (one, 4).  It is bound by pairs where its walk
 * reaches the bundles, by the node tests where the tree is deeper than that,
 * and teams pay only for pairs.  With 98304 particles (a wavefront and a half
 * per SIMD with one lane each) and fewer, idle SIMDs outweigh that and teams
 * of 4 lost in no box.  With more the tree's size decides, over up to 131072
 * nodes teams of 4 (one lane, 4): 110^3 218, 133; 128^3 (70784 nodes) 349,
 * 248; uniform 10^6 113, 72; clustered 2^20 (98940) 20.5, 11.1, 1.3e6
 * (129705) 13.5, 9.3; and beyond one lane: clustered 1.5e6 (152597) 5.4, 8.8,
 * 2^23 14.6, 43.2; uniform 3e6 48, 141; 144^3 120, 170; 256^3 978, 1093.
 * (All with alpha 0.005.  0.001: clustered 2^20 30, 18; 128^3 2890, 3010.
 * 0.02: 4.3, 5.3; 216, 123; uniform 10^6 54, 35.)  The Barnes-Hut walk and
 * relative walks of a looser criterion, which stay above the bundles, take
 * one lane there: Barnes-Hut, 110^3 1606, 1620; clustered 2^20 558, 837, 6e6
 * 3834, 6131; uniform 10^7 322, 1125; alpha 0.1, clustered 2^20 1.7, 3.5,
 * uniform 10^6 8.8, 16.8. */
struct Walk64Shape {
	int team, block;
};

#define TDV_W64_TEAM16 10240
#define TDV_W64_TEAM4 49152
#define TDV_W64_EWALD_TEAM4 98304
#define TDV_W64_EWALD_NODES 131072
#define TDV_W64_EWALD_ALPHA 0.02
#define TDV_W64_TEAM_MAX (1 << 28)       /* thread numbers within 32 bits */

static Walk64Shape newton_shape(int nact)
{
	if (nact <= TDV_W64_TEAM16)
		return { 16, 64 };
	if (nact <= TDV_W64_TEAM4)
		return { 4, 64 };
	return { 1, 256 };
}

static Walk64Shape ewald_shape(int nact, size_t nnodes, const WalkParams &w)
{
	if (nact <= TDV_W64_TEAM16)
		return { 16, 64 };
	if (nact <= TDV_W64_EWALD_TEAM4 || (!w.use_bh
			&& w.alpha_rel <= TDV_W64_EWALD_ALPHA
			&& nnodes <= TDV_W64_EWALD_NODES && nact <= TDV_W64_TEAM_MAX))
		return { 4, 64 };
	return { 1, 64 };
}

int tdv_walk64(tdv_context *c, int use_bh)
{
	if (!c->nactive)
		return 0;
	const WalkParams w = walk_params(c, use_bh);
	const Walk64Shape sh = newton_shape(c->nactive);
	const int L = sh.team;
	auto kern = w.periodic
			? (L == 16 ? k_walk64<16, true> : L == 4 ? k_walk64<4, true>
				: k_walk64<1, true>)
			: (L == 16 ? k_walk64<16, false> : L == 4 ? k_walk64<4, false>
				: k_walk64<1, false>);
	hipLaunchKernelGGL(kern, dim3(tdv_blocks((size_t)c->nactive * L, sh.block)),
			dim3(sh.block), 0, c->stream, c->nactive, c->active, c->pm, c->last_acc,
			c->top, c->node_a, c->node_b, c->node_c, w, c->acc[0], c->acc[1],
			c->acc[2], c->gacc[0], c->gacc[1], c->gacc[2], c->cost, (int)c->n,
			c->d_err, c->d_count);
	return tdv_check(c, hipGetLastError(), "k_walk64");
}

int tdv_walk64_ewald(tdv_context *c, int use_bh)
{
	if (!c->nactive)
		return 0;
	if (!c->have_ewald)
		return tdv_fail(c, TDV_ERR_ARG, "periodic walk without an Ewald table");
	const WalkParams w = walk_params(c, use_bh);
	const Walk64Shape sh = ewald_shape(c->nactive, c->nnodes, w);
	const int L = sh.team;
	auto kern = L == 16 ? k_walk64_ewald<16> : L == 4 ? k_walk64_ewald<4>
			: k_walk64_ewald<1>;
	hipLaunchKernelGGL(kern, dim3(tdv_blocks((size_t)c->nactive * L, sh.block)),
			dim3(sh.block), 0, c->stream, c->nactive, c->active, c->pm, c->last_acc,
			c->top, c->node_a, c->node_b, c->node_c, c->ewald_rows, w,
			c->acc[0], c->acc[1], c->acc[2], c->gacc[0], c->gacc[1],
			c->gacc[2], c->cost, (int)c->n, c->d_err, c->d_count + 1);
	return tdv_check(c, hipGetLastError(), "k_walk64_ewald");
}

/* safe_last_accel, accel.c:28-43 */
__global__ void k_safe_last_accel(int nact, const int *__restrict__ active,
		double *__restrict__ ax, double *__restrict__ ay,
		double *__restrict__ az, double *__restrict__ last)
{
	const int g = blockIdx.x * blockDim.x + threadIdx.x;
	if (g >= nact)
		return;
	const int i = active[g];
	last[i] = sqrt(ax[i] * ax[i] + ay[i] * ay[i] + az[i] * az[i]);
	ax[i] = 0;
	ay[i] = 0;
	az[i] = 0;
}

void tdv_launch_safe_last_accel(tdv_context *c)
{
	if (!c->nactive)
		return;
	hipLaunchKernelGGL(k_safe_last_accel,
			dim3(tdv_blocks((size_t)c->nactive, 256)), dim3(256), 0, c->stream,
			c->nactive, c->active, c->acc[0], c->acc[1], c->acc[2],
			c->last_acc);
}

__global__ void k_ewald_correction_batch(size_t n, const double *__restrict__ dr,
		double *__restrict__ f, const double *__restrict__ tab, double b2e)
{
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	double r[3];
	ewald_corr_rows(tab, dr[3 * i], dr[3 * i + 1], dr[3 * i + 2], b2e, r);
	f[3 * i] = r[0];
	f[3 * i + 1] = r[1];
	f[3 * i + 2] = r[2];
}

void tdv_launch_ewald_correction(tdv_context *c, size_t n, const double *dr,
		double *f)
{
	hipLaunchKernelGGL(k_ewald_correction_batch, dim3(tdv_blocks(n, 256)),
			dim3(256), 0, c->stream, n, dr, f, c->ewald_rows,
			2 * TDV_NE / c->par.boxsize);
}
