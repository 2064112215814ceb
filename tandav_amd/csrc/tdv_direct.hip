/*
 * FP64 direct summation for sampled target particles -- the engine's form of
 * Gravity_Forcetest (Gravity/forcetest.c:24-174): for each target, the sum
 * over every other particle of the path's own pairwise kernel (K1 with the
 * negative softening length, Gravity/tree_accel.c:362-394), plus, on
 * periodic runs, the tabulated Ewald correction of every pair (nearest image
 * + Ewald_Correction, Gravity/periodic.c:35-113).  The sources are cut into
 * parts, one workgroup per target and part; lanes stride over a part's
 * sources, the sums meet in a block reduction and the parts' sums are added
 * in part order.  Used to state the acceleration error of the walks.
 */
#include "tdv_internal.h"
#include "tdv_device.h"
#include <algorithm>

/* Two workgroups per CU keep the table's gathers busy, which bound a pair
 * (more of them only spread the sources' separations over more of the table:
 * 512 targets in 64^3 particles took 3.0 ms in one part each, 3.1 in two);
 * with fewer targets than that the sources are cut into parts of at least
 * TDV_DIRECT_MIN (16 targets 1.56 -> 0.15 ms, 100 targets 1.72 -> 0.95 ms). */
#define TDV_DIRECT_BLOCKS 512
#define TDV_DIRECT_MIN 2048

__device__ __forceinline__ double dwrap(double d, double box, double half)
{
	if (d > half)
		d -= box;
	else if (d < -half)
		d += box;
	return d;
}

/* Periodic sums are bound by the table's lines: the separations of 64
 * neighbouring sources lie in some hundred cells, 27 KB of the rows' lines,
 * each used once (46 KB of the components' own tables: those took 0.40 ms
 * for 512 targets in 31^3 particles, the rows 0.34).  The next two sources
 * are loaded and both gathers are in flight while a pair's sum is formed:
 * 512 targets in 64^3 particles 2.3 ms.  (With `periodic` an argument the
 * compiler keeps 120 registers instead of 178 and waits for one gather
 * before the other: 2.5.  Copying the cells to LDS first took 6.1, its
 * latency bare with the few wavefronts that fit.)  Isolated sums are bound by
 * the FP64 arithmetic of a pair: 600 targets in 10^6 particles 1.4 ms. */
template <bool PERIODIC>
__global__ void __launch_bounds__(256) k_direct(int nt,
		const int *__restrict__ idx, const double4 *__restrict__ pm, int n,
		double box, double G, double eps2, double eps3,
		const double *__restrict__ rows, double b2e, int chunk,
		double *__restrict__ out)
{
	constexpr int U = PERIODIC ? 2 : 1;
	__shared__ double red[3][256];
	const int t = blockIdx.x;
	if (t >= nt)
		return;
	/* this part's sources; its sums go to row blockIdx.y of out */
	const int first = (int)blockIdx.y * chunk;
	const int last = n - first < chunk ? n : first + chunk;
	const int i = idx[t];
	const double4 p = pm[i];
	const double half = box / 2.0;
	double ax = 0, ay = 0, az = 0;
	double4 next[U];
#pragma unroll
	for (int u = 0; u < U; u++)
		next[u] = pm[min(first + (int)threadIdx.x + 256 * u, last - 1)];
	for (int j = first + threadIdx.x; j < last; j += 256 * U) {
		double dx[U], dy[U], dz[U], m[U], f[U][3];
#pragma unroll
		for (int u = 0; u < U; u++) {
			dx[u] = next[u].x - p.x;
			dy[u] = next[u].y - p.y;
			dz[u] = next[u].z - p.z;
			m[u] = G * next[u].w;
			next[u] = pm[min(j + 256 * (U + u), last - 1)];
			if (PERIODIC) {
				dx[u] = dwrap(dx[u], box, half);
				dy[u] = dwrap(dy[u], box, half);
				dz[u] = dwrap(dz[u], box, half);
				ewald_corr_rows(rows, dx[u], dy[u], dz[u], b2e, f[u]);
			}
		}
#pragma unroll
		for (int u = 0; u < U; u++) {
			const double r2 = dx[u] * dx[u] + dy[u] * dy[u] + dz[u] * dz[u];
			if (j + 256 * u >= last || j + 256 * u == i || r2 == 0)
				continue;
			bool ok;
			const double ri = inv_sqrt(r2, &ok);
			double g = ri * ri * ri;
			if (!ok || r2 < eps2) {
				/* rare; free to, the compiler evaluates both cases for
				 * every pair (600 targets in 10^6 isolated particles 2.9
				 * ms) */
				asm volatile("");
				if (r2 < eps2) {
					const double u2 = r2 / eps2;
					g = (175 - u2 * (294 - u2 * 135)) / (16 * eps3);
				} else {
					const double rs = 1 / sqrt(r2);
					g = rs * rs * rs;
				}
			}
			const double fac = m[u] * g;
			ax += fac * dx[u];
			ay += fac * dy[u];
			az += fac * dz[u];
			if (PERIODIC) {
				ax += m[u] * f[u][0];
				ay += m[u] * f[u][1];
				az += m[u] * f[u][2];
			}
		}
	}
	red[0][threadIdx.x] = ax;
	red[1][threadIdx.x] = ay;
	red[2][threadIdx.x] = az;
	__syncthreads();
	for (int s = blockDim.x / 2; s > 0; s >>= 1) {
		if ((int)threadIdx.x < s)
			for (int d = 0; d < 3; d++)
				red[d][threadIdx.x] += red[d][threadIdx.x + s];
		__syncthreads();
	}
	if (threadIdx.x == 0)
		for (int d = 0; d < 3; d++)
			out[3 * ((size_t)blockIdx.y * nt + t) + d] = red[d][0];
}

__global__ void k_direct_parts(int n3, int nparts,
		const double *__restrict__ part, double *__restrict__ out)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n3)
		return;
	double s = part[i];
	for (int k = 1; k < nparts; k++)
		s += part[(size_t)k * n3 + i];
	out[i] = s;
}

int tdv_direct_sum(tdv_context *c, int nt, const int *idx_dev, double *out_dev)
{
	if (nt <= 0)
		return 0;
	if (c->par.periodic && !c->have_ewald)
		return tdv_fail(c, TDV_ERR_ARG, "direct sum without an Ewald table");
	/* parts, their sums in the sort's scratch (cap words, free here) */
	const size_t n = c->n;
	size_t parts = std::min({ (size_t)(TDV_DIRECT_BLOCKS / nt),
		n / TDV_DIRECT_MIN, c->cap / (3 * (size_t)nt) });
	if (parts < 1)
		parts = 1;
	const int chunk = (int)((n + parts - 1) / parts);
	parts = (n + chunk - 1) / chunk;
	double *sums = parts > 1 ? reinterpret_cast<double *>(c->sk[0]) : out_dev;
	auto kern = c->par.periodic ? k_direct<true> : k_direct<false>;
	hipLaunchKernelGGL(kern, dim3(nt, (unsigned)parts), dim3(256), 0,
			c->stream, nt, idx_dev, c->pm, (int)n, c->par.boxsize,
			c->par.gravity, c->Epsilon2, c->Epsilon3, c->ewald_rows,
			2 * TDV_NE / (c->par.periodic ? c->par.boxsize : 1.0), chunk,
			sums);
	if (parts > 1)
		hipLaunchKernelGGL(k_direct_parts, dim3(tdv_blocks(3 * (size_t)nt,
				256)), dim3(256), 0, c->stream, 3 * nt, (int)parts, sums,
				out_dev);
	return tdv_check(c, hipGetLastError(), "k_direct");
}
