/*
 * PH keys, the key sort, gathers and the device-wide scan.
 *
 * Keys: one lane per particle runs Skilling's transform (peano.c:122-195)
 * and writes the standard 128-bit key.  Reversed keys (peano.c:203-276) are
 * the triplet permutation of the standard key, produced after the sort.
 *
 * Sort: LSD radix sort, 8-bit digits, over the high 64 key bits with a
 * 32-bit payload (the original index), 8 passes of histogram -> scan ->
 * stable scatter (few tiles: the scatter sums the histograms itself; one
 * tile: all passes in one workgroup's LDS).  Runs of equal high words are then ordered by the low
 * word; equal full keys raise TDV_ERR_DUP_KEYS (the reference's quicksort
 * is unstable, sort.c:253-341, so only unique keys have a defined order).
 * Traffic per pass: 12 B read (histogram) + 12 B read + 12 B written.
 */
#include "tdv_internal.h"
#include "tdv_device.h"

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <mutex>

#define RS_THREADS 256
#define RS_ITEMS (TDV_SORT_TILE / RS_THREADS)
#define RS_TILE TDV_SORT_TILE
#define RS_BINS 256
#define RS_WAVES (RS_THREADS / 64)

/* ------------------------------------------------------------------------ */
/* keys                                                                      */
/* ------------------------------------------------------------------------ */

__global__ void __launch_bounds__(256) k_peano_keys(size_t n,
		const double *__restrict__ x, const double *__restrict__ y,
		const double *__restrict__ z, double o0, double o1, double o2,
		double fac, uint64_t *__restrict__ out, int reversed)
{
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	uint64_t lo, hi;
	peano_key_words(x[i], y[i], z[i], o0, o1, o2, fac, reversed, &lo, &hi);
	out[2 * i] = lo;
	out[2 * i + 1] = hi;
}

void tdv_launch_keys(tdv_context *c, size_t n, const double *x,
		const double *y, const double *z, const double o[3], double size,
		uint64_t *out, int reversed)
{
	if (!n)
		return;
	const double fac = (double)(1ull << 63) / size;
	hipLaunchKernelGGL(k_peano_keys, dim3(tdv_blocks(n, 256)), dim3(256), 0,
			c->stream, n, x, y, z, o[0], o[1], o[2], fac, out, reversed);
}

/* reversed key from a standard key: level k (1..41) triplet moves from
 * bits [128-3k, 130-3k] to [3k, 3k+2]; level 42 keeps its two low bits at
 * 126..127; level 0 is 000 */
__global__ void k_reverse_keys(size_t n, const uint64_t *__restrict__ in,
		uint64_t *__restrict__ out)
{
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	const Key2 k = load_key(in, i);
	uint64_t lo = 0, hi = 0;
#pragma unroll 6
	for (int L = 1; L <= 42; L++) {
		const uint64_t t = key_triplet(k, L);
		const int p = 3 * L;
		if (p >= 64)
			hi |= t << (p - 64);
		else if (p <= 61)
			lo |= t << p;
		else {
			lo |= t << p;
			hi |= t >> (64 - p);
		}
	}
	store_key(out, i, Key2{ lo, hi });
}

void tdv_launch_reverse_keys(tdv_context *c, size_t n, const uint64_t *in,
		uint64_t *out)
{
	if (!n)
		return;
	hipLaunchKernelGGL(k_reverse_keys, dim3(tdv_blocks(n, 256)), dim3(256), 0,
			c->stream, n, in, out);
}

/* ------------------------------------------------------------------------ */
/* device-wide exclusive scan of u32 (out has n+1 entries, out[n] = total)   */
/* ------------------------------------------------------------------------ */

#define SC_THREADS 256
#define SC_ITEMS 4
#define SC_TILE (SC_THREADS * SC_ITEMS)

__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *tot,
		uint32_t *sh)
{
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	uint32_t inc = v;
#pragma unroll
	for (int d = 1; d < 64; d <<= 1) {
		uint32_t t = __shfl_up(inc, d, 64);
		if (lane >= d)
			inc += t;
	}
	if (lane == 63)
		sh[w] = inc;
	__syncthreads();
	uint32_t wbase = 0, all = 0;
	for (int q = 0; q < (int)(blockDim.x >> 6); q++) {
		if (q < w)
			wbase += sh[q];
		all += sh[q];
	}
	__syncthreads();
	*tot = all;
	return wbase + inc - v;
}

__global__ void __launch_bounds__(SC_THREADS) k_scan_reduce(
		const uint32_t *__restrict__ in, size_t n, uint32_t *__restrict__ part)
{
	__shared__ uint32_t sh[SC_THREADS / 64];
	const size_t base = (size_t)blockIdx.x * SC_TILE + threadIdx.x * SC_ITEMS;
	uint32_t s = 0;
	for (int k = 0; k < SC_ITEMS; k++)
		if (base + k < n)
			s += in[base + k];
	uint32_t tot;
	block_excl_scan(s, &tot, sh);
	if (threadIdx.x == 0)
		part[blockIdx.x] = tot;
}

__global__ void __launch_bounds__(SC_THREADS) k_scan_partials(
		uint32_t *__restrict__ part, size_t np, uint32_t *__restrict__ total)
{
	__shared__ uint32_t sh[SC_THREADS / 64];
	uint32_t carry = 0;
	for (size_t b = 0; b < np; b += SC_THREADS) {
		const size_t i = b + threadIdx.x;
		const uint32_t v = i < np ? part[i] : 0;
		uint32_t tot;
		const uint32_t e = block_excl_scan(v, &tot, sh);
		if (i < np)
			part[i] = carry + e;
		carry += tot;
	}
	if (threadIdx.x == 0)
		*total = carry;
}

__global__ void __launch_bounds__(SC_THREADS) k_scan_down(
		const uint32_t *__restrict__ in, size_t n,
		const uint32_t *__restrict__ part, uint32_t *__restrict__ out)
{
	__shared__ uint32_t sh[SC_THREADS / 64];
	const size_t base = (size_t)blockIdx.x * SC_TILE + threadIdx.x * SC_ITEMS;
	uint32_t v[SC_ITEMS];
	uint32_t s = 0;
	for (int k = 0; k < SC_ITEMS; k++) {
		v[k] = base + k < n ? in[base + k] : 0;
		s += v[k];
	}
	uint32_t tot;
	uint32_t e = block_excl_scan(s, &tot, sh) + part[blockIdx.x];
	for (int k = 0; k < SC_ITEMS; k++) {
		if (base + k < n)
			out[base + k] = e;
		e += v[k];
	}
}

/* exclusive scan on stream s with the block partials in part
 * ((n + SC_TILE - 1) / SC_TILE + 1 entries); errors go to c (may be NULL) */
static int scan_u32(tdv_context *c, hipStream_t s, uint32_t *part,
		const uint32_t *in, uint32_t *out, size_t n)
{
	const size_t nb = (n + SC_TILE - 1) / SC_TILE;
	if (nb == 0) {
		TDV_HIP(c, hipMemsetAsync(out, 0, sizeof(uint32_t), s));
		return 0;
	}
	hipLaunchKernelGGL(k_scan_reduce, dim3((unsigned)nb), dim3(SC_THREADS), 0,
			s, in, n, part);
	hipLaunchKernelGGL(k_scan_partials, dim3(1), dim3(SC_THREADS), 0, s, part,
			nb, out + n);
	hipLaunchKernelGGL(k_scan_down, dim3((unsigned)nb), dim3(SC_THREADS), 0,
			s, in, n, part, out);
	return tdv_check(c, hipGetLastError(), "scan");
}

int tdv_scan_u32(tdv_context *c, const uint32_t *in, uint32_t *out, size_t n)
{
	return scan_u32(c, c->stream, c->scan_part, in, out, n);
}

/* ------------------------------------------------------------------------ */
/* LSD radix sort of u64 keys with a u32 payload                             */
/* ------------------------------------------------------------------------ */

/* key source: pass 0 may read the high words of 128-bit keys (stride 2) */
__device__ __forceinline__ uint64_t rs_load(const uint64_t *k, size_t i,
		int stride, int off)
{
	return k[i * stride + off];
}

/* The tile workgroup b of nb takes.  Workgroups go to the 8 XCDs in turn
 * (b to XCD b mod 8); numbering the tiles so that each XCD takes one
 * contiguous range of them keeps neighbouring tiles' histogram and offset
 * entries (4 bytes apart, digit-major) and the digit runs they write side
 * by side in one XCD's L2, where they had been partial lines of eight
 * L2s, each written back or fetched on its own. */
__device__ __forceinline__ unsigned rs_tile(unsigned b, unsigned nb)
{
	const unsigned q = nb / 8, r = nb % 8, x = b % 8, i = b / 8;
	return x < r ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
}

/* BY_TILE: the counts of a tile side by side (the scatter sums them), else
 * digit-major for the device-wide scan */
template <bool BY_TILE>
__global__ void __launch_bounds__(RS_THREADS) k_rs_hist(
		const uint64_t *__restrict__ keys, int stride, int off, size_t n,
		int shift, uint32_t *__restrict__ hist, unsigned nblocks)
{
	__shared__ uint32_t h[RS_BINS];
	h[threadIdx.x] = 0;
	__syncthreads();
	const unsigned tile = rs_tile(blockIdx.x, nblocks);
	const size_t base = (size_t)tile * RS_TILE;
	/* every load issued before the first is used: unconditional loads of
	 * an index clamped into [0, n) (n >= 1), the count only when i < n */
	uint64_t kk[RS_ITEMS];
#pragma unroll
	for (int it = 0; it < RS_ITEMS; it++) {
		const size_t i = base + (size_t)it * RS_THREADS + threadIdx.x;
		kk[it] = rs_load(keys, i < n ? i : n - 1, stride, off);
	}
#pragma unroll
	for (int it = 0; it < RS_ITEMS; it++) {
		const size_t i = base + (size_t)it * RS_THREADS + threadIdx.x;
		if (i < n)
			atomicAdd(&h[(unsigned)(kk[it] >> shift) & 255u], 1u);
	}
	__syncthreads();
	hist[BY_TILE ? (size_t)tile * RS_BINS + threadIdx.x
			: (size_t)threadIdx.x * nblocks + tile] = h[threadIdx.x];
}

/* exclusive prefix sum over the 256 digits of the first four waves' v
 * (thread d holds digit d's), every thread of the workgroup taking part */
__device__ __forceinline__ uint32_t rs_digit_scan(uint32_t v,
		uint32_t *wsum)
{
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	uint32_t x = v;
#pragma unroll
	for (int o = 1; o < 64; o <<= 1) {
		const uint32_t y = __shfl_up(x, o, 64);
		if (lane >= o)
			x += y;
	}
	if (lane == 63 && w < 4)
		wsum[w] = x;
	__syncthreads();
	uint32_t before = 0;
	for (int q = 0; q < w && q < 4; q++)
		before += wsum[q];
	return before + x - v;
}

/* A workgroup's tile of THREADS x ITEMS keys in LDS */
template <int THREADS, int ITEMS>
struct RsShared {
	uint32_t wcnt[THREADS / 64][RS_BINS];
	uint32_t dstart[RS_BINS];            /* digit's first slot in the tile */
	uint32_t wsum[4];
	uint64_t skey[THREADS * ITEMS];
	uint32_t sval[THREADS * ITEMS];
};

/* The tile's keys sorted by one digit into LDS: every key's rank among the
 * tile's keys of its digit (stable: waves, items and lanes in input order),
 * then the digits' runs one after the other.  Wave w's item it of lane l is
 * the tile's key (w ITEMS + it) 64 + l; the first nvalid keys count. */
template <int THREADS, int ITEMS>
__device__ __forceinline__ void rs_sort_tile(RsShared<THREADS, ITEMS> &sh,
		const uint64_t (&kk)[ITEMS], const uint32_t (&vv)[ITEMS], int nvalid,
		int shift)
{
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	for (int q = threadIdx.x; q < THREADS / 64 * RS_BINS; q += THREADS)
		sh.wcnt[q / RS_BINS][q % RS_BINS] = 0;
	__syncthreads();
	uint32_t rk[ITEMS];
	const uint64_t lt = (1ull << lane) - 1;
#pragma unroll
	for (int it = 0; it < ITEMS; it++) {
		const bool valid = (w * ITEMS + it) * 64 + lane < nvalid;
		const unsigned d = (unsigned)(kk[it] >> shift) & 255u;
		uint64_t peers = __ballot(valid);
#pragma unroll
		for (int b = 0; b < 8; b++) {
			const uint64_t bal = __ballot((d >> b) & 1u);
			peers &= ((d >> b) & 1u) ? bal : ~bal;
		}
		const uint32_t below = (uint32_t)__popcll(peers & lt);
		const int leader = peers ? (__ffsll((unsigned long long)peers) - 1) : 0;
		uint32_t old = 0;
		if (valid && below == 0)
			old = atomicAdd(&sh.wcnt[w][d], (uint32_t)__popcll(peers));
		old = __shfl(old, leader, 64);
		rk[it] = old + below;
	}
	__syncthreads();
	/* per digit: the waves' exclusive prefix, and the tile's count, whose
	 * exclusive scan over the digits places each digit's run in the tile */
	uint32_t cnt = 0;
	if (threadIdx.x < RS_BINS)
		for (int q = 0; q < THREADS / 64; q++) {
			const uint32_t t = sh.wcnt[q][threadIdx.x];
			sh.wcnt[q][threadIdx.x] = cnt;
			cnt += t;
		}
	const uint32_t start = rs_digit_scan(cnt, sh.wsum);
	if (threadIdx.x < RS_BINS)
		sh.dstart[threadIdx.x] = start;
	__syncthreads();
#pragma unroll
	for (int it = 0; it < ITEMS; it++)
		if ((w * ITEMS + it) * 64 + lane < nvalid) {
			const unsigned d = (unsigned)(kk[it] >> shift) & 255u;
			const uint32_t slot = sh.dstart[d] + sh.wcnt[w][d] + rk[it];
			sh.skey[slot] = kk[it];
			sh.sval[slot] = vv[it];
		}
	__syncthreads();
}

/* One LSD pass's scatter of a tile of RS_TILE keys: the tile sorted by
 * digit in LDS, then written out in that order, so consecutive threads
 * store consecutive positions of a digit's run (one run of ~16 keys per
 * digit and tile) instead of every lane a key of its own digit somewhere
 * else.  BY_TILE: where a tile's runs go is summed here from all tiles'
 * counts (thread d digit d's), else read from the scanned histogram. */
template <bool BY_TILE>
__global__ void __launch_bounds__(RS_THREADS) k_rs_scatter(
		const uint64_t *__restrict__ kin, int stride, int off,
		const uint32_t *__restrict__ vin, uint64_t *__restrict__ kout,
		uint32_t *__restrict__ vout, size_t n, int shift,
		const uint32_t *__restrict__ hscan, unsigned nblocks)
{
	__shared__ RsShared<RS_THREADS, RS_ITEMS> sh;
	__shared__ uint32_t binoff[RS_BINS];
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	const unsigned tile = rs_tile(blockIdx.x, nblocks);
	const size_t tile0 = (size_t)tile * RS_TILE;
	const size_t base = tile0 + (size_t)w * 64 * RS_ITEMS;
	uint64_t kk[RS_ITEMS];
	uint32_t vv[RS_ITEMS];
	/* all of the wave's loads in flight at once: unconditional, at an
	 * index clamped into [0, n) (n >= 1); what lies past n is not used */
#pragma unroll
	for (int it = 0; it < RS_ITEMS; it++) {
		const size_t i = base + (size_t)it * 64 + lane;
		kk[it] = rs_load(kin, i < n ? i : n - 1, stride, off);
	}
	if (vin) {
#pragma unroll
		for (int it = 0; it < RS_ITEMS; it++) {
			const size_t i = base + (size_t)it * 64 + lane;
			vv[it] = vin[i < n ? i : n - 1];
		}
	} else {
#pragma unroll
		for (int it = 0; it < RS_ITEMS; it++)
			vv[it] = (uint32_t)(base + (size_t)it * 64 + lane);
	}
	if (BY_TILE) {
		uint32_t before = 0, all = 0;
#pragma unroll 8
		for (unsigned t = 0; t < nblocks; t++) {
			const uint32_t h = hscan[(size_t)t * RS_BINS + threadIdx.x];
			before += t < tile ? h : 0;
			all += h;
		}
		binoff[threadIdx.x] = rs_digit_scan(all, sh.wsum) + before;
	} else {
		binoff[threadIdx.x] = hscan[(size_t)threadIdx.x * nblocks + tile];
	}
	const int nvalid = n - tile0 < (size_t)RS_TILE ? (int)(n - tile0)
			: RS_TILE;
	__syncthreads();
	rs_sort_tile<RS_THREADS, RS_ITEMS>(sh, kk, vv, nvalid, shift);
	for (int j = threadIdx.x; j < nvalid; j += RS_THREADS) {
		const uint64_t k = sh.skey[j];
		const unsigned d = (unsigned)(k >> shift) & 255u;
		const uint32_t pos = binoff[d] + ((uint32_t)j - sh.dstart[d]);
		if (pos < n) {                       /* always, by construction */
			kout[pos] = k;
			vout[pos] = sh.sval[j];
		}
	}
}

/* All passes of up to RS_TILE keys in one workgroup: each pass sorts the
 * tile by its digit in LDS and reads it back in that order.  A launch costs
 * more than a pass of so few keys (a 4096-particle step 1.11 -> 0.95 ms). */
#define RS1_THREADS 1024
#define RS1_ITEMS (RS_TILE / RS1_THREADS)
static_assert(RS1_THREADS * RS1_ITEMS == RS_TILE, "one tile");

__global__ void __launch_bounds__(RS1_THREADS) k_rs_one_tile(
		const uint64_t *__restrict__ kin, int stride, int off,
		const uint32_t *__restrict__ vin, uint64_t *__restrict__ kout,
		uint32_t *__restrict__ vout, int n)
{
	__shared__ RsShared<RS1_THREADS, RS1_ITEMS> sh;
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	const int base = w * 64 * RS1_ITEMS + lane;
	uint64_t kk[RS1_ITEMS];
	uint32_t vv[RS1_ITEMS];
#pragma unroll
	for (int it = 0; it < RS1_ITEMS; it++) {
		const int i = base + it * 64;
		kk[it] = rs_load(kin, (size_t)(i < n ? i : n - 1), stride, off);
		vv[it] = vin ? vin[i < n ? i : n - 1] : (uint32_t)i;
	}
	for (int shift = 0; shift < 64; shift += 8) {
		rs_sort_tile<RS1_THREADS, RS1_ITEMS>(sh, kk, vv, n, shift);
#pragma unroll
		for (int it = 0; it < RS1_ITEMS; it++) {
			const int i = base + it * 64;
			kk[it] = sh.skey[i < n ? i : n - 1];
			vv[it] = sh.sval[i < n ? i : n - 1];
		}
		__syncthreads();
	}
#pragma unroll
	for (int it = 0; it < RS1_ITEMS; it++) {
		const int i = base + it * 64;
		if (i < n) {
			kout[i] = kk[it];
			vout[i] = vv[it];
		}
	}
}

/* the buffers a key sort works in: a context's own, or the no-allocation
 * entry point's static scratch */
struct SortWork {
	hipStream_t stream;
	uint64_t *sk[2];             /* n keys each */
	uint32_t *sv[2];             /* n payloads each */
	uint32_t *hist;              /* hist_cap digit counts */
	size_t hist_cap;
	uint32_t *scan_part;         /* scan block partials */
	unsigned *d_err;             /* TDV_EBIT_* flags */
	uint64_t *hi_tmp;            /* n words: the tie fallback's high words */
	uint32_t *p_tmp;             /* n: the tie fallback's first order */
	uint32_t *order;             /* n: the order while the keys are read */
	bool no_sync;                /* no read back, no fallback (the tie flag
	                                stays in d_err for the caller) */
};

static SortWork context_work(tdv_context *c, const uint32_t *perm_out)
{
	SortWork w;
	w.stream = c->stream;
	for (int b = 0; b < 2; b++) {
		w.sk[b] = c->sk[b];
		w.sv[b] = c->sv[b];
	}
	w.hist = c->hist;
	w.hist_cap = c->hist_cap;
	w.scan_part = c->scan_part;
	w.d_err = c->d_err;
	w.hi_tmp = reinterpret_cast<uint64_t *>(c->tmp_f64);
	w.p_tmp = c->perm == perm_out ? reinterpret_cast<uint32_t *>(c->lohi)
			: c->perm;
	w.order = c->perm == perm_out ? c->perm : c->sv[1];
	w.no_sync = false;
	return w;
}

/* Up to this many tiles the scatter sums the tiles' counts itself: two
 * launches a pass instead of five.  The sum reads 1 KiB per tile and
 * workgroup; with more tiles the scan's three launches are cheaper. */
#define RS_SUM_TILES 64

/* sorts n u64 keys (read with stride/offset, e.g. the high words of 128-bit
 * keys) carrying payload vin (NULL = original index): the sorted keys into
 * w.sk[*res], the payload into vout */
static int radix_sort_u64(tdv_context *c, const SortWork &w, size_t n,
		const uint64_t *keys, int stride, int off, const uint32_t *vin,
		uint32_t *vout, int *res)
{
	const unsigned nb = (unsigned)((n + RS_TILE - 1) / RS_TILE);
	const size_t hn = (size_t)nb * RS_BINS;
	if (hn + 1 > w.hist_cap)
		return tdv_fail(c, TDV_ERR_ARG, "radix sort histogram too small");
	if (nb == 1) {
		hipLaunchKernelGGL(k_rs_one_tile, dim3(1), dim3(RS1_THREADS), 0,
				w.stream, keys, stride, off, vin, w.sk[0], vout, (int)n);
		*res = 0;
		return tdv_check(c, hipGetLastError(), "radix sort");
	}
	const bool by_tile = nb <= RS_SUM_TILES;
	const uint64_t *kin = keys;
	const uint32_t *vi = vin;
	int s = stride, o = off, cur = 0;
	for (int pass = 0; pass < 8; pass++) {
		const int shift = 8 * pass;
		uint32_t *vo = pass == 7 ? vout : w.sv[cur];
		if (by_tile) {
			hipLaunchKernelGGL(k_rs_hist<true>, dim3(nb), dim3(RS_THREADS), 0,
					w.stream, kin, s, o, n, shift, w.hist, nb);
			hipLaunchKernelGGL(k_rs_scatter<true>, dim3(nb),
					dim3(RS_THREADS), 0, w.stream, kin, s, o, vi, w.sk[cur],
					vo, n, shift, w.hist, nb);
		} else {
			hipLaunchKernelGGL(k_rs_hist<false>, dim3(nb), dim3(RS_THREADS),
					0, w.stream, kin, s, o, n, shift, w.hist, nb);
			TDV_TRY(scan_u32(c, w.stream, w.scan_part, w.hist, w.hist, hn));
			hipLaunchKernelGGL(k_rs_scatter<false>, dim3(nb),
					dim3(RS_THREADS), 0, w.stream, kin, s, o, vi, w.sk[cur],
					vo, n, shift, w.hist, nb);
		}
		kin = w.sk[cur];
		vi = w.sv[cur];
		s = 1;
		o = 0;
		cur ^= 1;
	}
	*res = cur ^ 1;
	return tdv_check(c, hipGetLastError(), "radix sort");
}

/* One stable pass over the low 8 bits of n u64 keys with the keys' indices
 * as payload: work items in key order (the FP32 walk's groups by expected
 * cost), in index order within a key */
int tdv_radix_pass8(tdv_context *c, size_t n, const uint64_t *keys,
		uint64_t *kout, uint32_t *order)
{
	const unsigned nb = (unsigned)((n + RS_TILE - 1) / RS_TILE);
	const size_t hn = (size_t)nb * RS_BINS;
	if (hn + 1 > c->hist_cap)
		return tdv_fail(c, TDV_ERR_ARG, "radix pass histogram too small");
	hipLaunchKernelGGL(k_rs_hist<true>, dim3(nb), dim3(RS_THREADS), 0,
			c->stream, keys, 1, 0, n, 0, c->hist, nb);
	hipLaunchKernelGGL(k_rs_scatter<true>, dim3(nb), dim3(RS_THREADS), 0,
			c->stream, keys, 1, 0, nullptr, kout, order, n, 0, c->hist, nb);
	return tdv_check(c, hipGetLastError(), "radix pass");
}

/* order runs of equal high words by the low word; flag duplicate keys */
__global__ void k_fix_ties(size_t n, const uint64_t *__restrict__ shi,
		uint32_t *__restrict__ perm, const uint64_t *__restrict__ keys,
		unsigned *err)
{
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	const uint64_t h = shi[i];
	if (i > 0 && shi[i - 1] == h)
		return;                          /* not a run start */
	if (i + 1 >= n || shi[i + 1] != h)
		return;                          /* run of one */
	size_t e = i + 1;
	while (e + 1 < n && shi[e + 1] == h)
		e++;
	if (e - i + 1 > 4096) {
		atomicOr(err, TDV_EBIT_TIES);
		return;
	}
	for (size_t r = i + 1; r <= e; r++) {   /* insertion sort by low word */
		const uint32_t pv = perm[r];
		const uint64_t lv = keys[2 * (size_t)pv];
		size_t t = r;
		while (t > i && keys[2 * (size_t)perm[t - 1]] > lv) {
			perm[t] = perm[t - 1];
			t--;
		}
		perm[t] = pv;
	}
	for (size_t r = i + 1; r <= e; r++)
		if (keys[2 * (size_t)perm[r]] == keys[2 * (size_t)perm[r - 1]])
			atomicOr(err, TDV_EBIT_DUP);
}

/* gather the high words of 128-bit keys by a permutation */
__global__ void k_gather_hi(size_t n, const uint32_t *__restrict__ perm,
		const uint64_t *__restrict__ keys, uint64_t *__restrict__ out)
{
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		out[i] = keys[2 * (size_t)perm[i] + 1];
}

__global__ void k_check_dups(size_t n, const uint32_t *__restrict__ perm,
		const uint64_t *__restrict__ keys, unsigned *err)
{
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i == 0 || i >= n)
		return;
	const size_t a = perm[i - 1], b = perm[i];
	if (keys[2 * a] == keys[2 * b] && keys[2 * a + 1] == keys[2 * b + 1])
		atomicOr(err, TDV_EBIT_DUP);
}

/* Qsort_Index's order of unique 128-bit keys (2n words) into perm_out:
 * the high words radix-sorted, runs of equal high words ordered by the low
 * word; runs longer than 4096 switch to a full 128-bit LSD sort.  Duplicate
 * keys set TDV_EBIT_DUP in w.d_err.  Reads w.d_err back (a stream
 * synchronisation) to choose the fallback. */
static int sort_keys_work(tdv_context *c, const SortWork &w, size_t n,
		const uint64_t *keys, uint32_t *perm_out)
{
	if (n == 0)
		return 0;
	int res;
	TDV_TRY(radix_sort_u64(c, w, n, keys, 2, 1, nullptr, w.order, &res));
	hipLaunchKernelGGL(k_fix_ties, dim3(tdv_blocks(n, 256)), dim3(256), 0,
			w.stream, n, w.sk[res], w.order, keys, w.d_err);
	if (w.no_sync) {
		if (w.order != perm_out)
			TDV_HIP(c, hipMemcpyAsync(perm_out, w.order,
					n * sizeof(uint32_t), hipMemcpyDeviceToDevice, w.stream));
		return tdv_check(c, hipGetLastError(), "sort");
	}
	unsigned e = 0;
	TDV_HIP(c, hipMemcpyAsync(&e, w.d_err, sizeof(e), hipMemcpyDeviceToHost,
			w.stream));
	TDV_HIP(c, hipStreamSynchronize(w.stream));
	if (e & TDV_EBIT_TIES) {
		/* long runs of equal high words: full 128-bit LSD sort, low word
		 * first (8 passes), then the high words in that order (8 passes) */
		TDV_HIP(c, hipMemsetAsync(w.d_err, 0, sizeof(unsigned), w.stream));
		int r1;
		TDV_TRY(radix_sort_u64(c, w, n, keys, 2, 0, nullptr, w.p_tmp, &r1));
		hipLaunchKernelGGL(k_gather_hi, dim3(tdv_blocks(n, 256)), dim3(256), 0,
				w.stream, n, w.p_tmp, keys, w.hi_tmp);
		TDV_TRY(radix_sort_u64(c, w, n, w.hi_tmp, 1, 0, w.p_tmp, w.order,
				&res));
		hipLaunchKernelGGL(k_check_dups, dim3(tdv_blocks(n, 256)), dim3(256), 0,
				w.stream, n, w.order, keys, w.d_err);
	}
	if (w.order != perm_out)
		TDV_HIP(c, hipMemcpyAsync(perm_out, w.order, n * sizeof(uint32_t),
				hipMemcpyDeviceToDevice, w.stream));
	return tdv_check(c, hipGetLastError(), "sort");
}

/* defer: the tie flag stays in d_err for the caller, no fallback */
int tdv_sort_device(tdv_context *c, size_t n, const uint64_t *keys,
		uint32_t *perm_out, bool defer)
{
	SortWork w = context_work(c, perm_out);
	w.no_sync = defer;
	return sort_keys_work(c, w, n, keys, perm_out);
}

/* perm = first, then perm */
__global__ void k_compose(size_t n, const uint32_t *__restrict__ first,
		uint32_t *__restrict__ perm)
{
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		perm[i] = first[perm[i]];
}

void tdv_launch_compose(tdv_context *c, size_t n, const uint32_t *first,
		uint32_t *perm)
{
	hipLaunchKernelGGL(k_compose, dim3(tdv_blocks(n, 256)), dim3(256), 0,
			c->stream, n, first, perm);
}

/* ------------------------------------------------------------------------ */
/* the key sort without allocation: a static scratch array per device      */
/* ------------------------------------------------------------------------ */

/* byte offsets of the work buffers in the scratch array, for
 * TDV_NOALLOC_MAX_KEYS keys (each 256-byte aligned) */
#define NA_N ((size_t)TDV_NOALLOC_MAX_KEYS)
#define NA_ALIGN(x) (((x) + 255) & ~(size_t)255)
#define NA_HIST_CAP (((NA_N + RS_TILE - 1) / RS_TILE) * RS_BINS + 1)
#define NA_PART_CAP (NA_HIST_CAP / SC_TILE + 2)
#define NA_SK0 ((size_t)0)
#define NA_SK1 (NA_SK0 + NA_ALIGN(NA_N * 8))
#define NA_SV0 (NA_SK1 + NA_ALIGN(NA_N * 8))
#define NA_SV1 (NA_SV0 + NA_ALIGN(NA_N * 4))
#define NA_HI (NA_SV1 + NA_ALIGN(NA_N * 4))
#define NA_PT (NA_HI + NA_ALIGN(NA_N * 8))
#define NA_HIST (NA_PT + NA_ALIGN(NA_N * 4))
#define NA_PART (NA_HIST + NA_ALIGN(NA_HIST_CAP * 4))
#define NA_ERR (NA_PART + NA_ALIGN(NA_PART_CAP * 4))
#define NA_BYTES (NA_ERR + 256)

/* one copy per GPU, held until the process ends; every call on a GPU uses
 * that GPU's copy, so calls that overlap on one GPU race */
static __device__ __align__(256) unsigned char scratch[NA_BYTES];

#define NA_MAX_DEVICES 64
static std::mutex na_mutex;
static unsigned char *na_ptr[NA_MAX_DEVICES];

/* the device address of this GPU's scratch (host code never passes the
 * array's own name: on the host it is not the device address) */
static int noalloc_scratch(int dev, unsigned char **out)
{
	std::lock_guard<std::mutex> lock(na_mutex);
	if (!na_ptr[dev]) {
		void *p = nullptr;
		if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess
				|| !p) {
			(void)hipGetLastError();
			return TDV_ERR_HIP;
		}
		na_ptr[dev] = static_cast<unsigned char *>(p);
	}
	*out = na_ptr[dev];
	return 0;
}

extern "C" int tdv_sort_keys_noalloc(size_t n, const uint64_t *keys,
		uint32_t *perm_out, void *stream)
{
	if (n > NA_N)
		return TDV_ERR_ARG;
	if (n == 0)
		return 0;
	if (!keys || !perm_out)
		return TDV_ERR_ARG;
	int dev = -1;
	if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= NA_MAX_DEVICES) {
		(void)hipGetLastError();
		return TDV_ERR_HIP;
	}
	unsigned char *base = nullptr;
	TDV_TRY(noalloc_scratch(dev, &base));
	SortWork w;
	w.stream = static_cast<hipStream_t>(stream);
	w.sk[0] = reinterpret_cast<uint64_t *>(base + NA_SK0);
	w.sk[1] = reinterpret_cast<uint64_t *>(base + NA_SK1);
	w.sv[0] = reinterpret_cast<uint32_t *>(base + NA_SV0);
	w.sv[1] = reinterpret_cast<uint32_t *>(base + NA_SV1);
	w.hi_tmp = reinterpret_cast<uint64_t *>(base + NA_HI);
	w.p_tmp = reinterpret_cast<uint32_t *>(base + NA_PT);
	w.order = w.sv[1];
	w.hist = reinterpret_cast<uint32_t *>(base + NA_HIST);
	w.hist_cap = NA_HIST_CAP;
	w.scan_part = reinterpret_cast<uint32_t *>(base + NA_PART);
	w.d_err = reinterpret_cast<unsigned *>(base + NA_ERR);
	w.no_sync = false;
	/* the previous call's flags stay in the array: clear them */
	if (hipMemsetAsync(w.d_err, 0, sizeof(unsigned), w.stream) != hipSuccess) {
		(void)hipGetLastError();
		return TDV_ERR_HIP;
	}
	TDV_TRY(sort_keys_work(nullptr, w, n, keys, perm_out));
	unsigned e = 0;
	if (hipMemcpyAsync(&e, w.d_err, sizeof(e), hipMemcpyDeviceToHost, w.stream)
			!= hipSuccess || hipStreamSynchronize(w.stream) != hipSuccess) {
		(void)hipGetLastError();
		return TDV_ERR_HIP;
	}
	if (e & TDV_EBIT_DUP)
		return TDV_ERR_DUP_KEYS;
	if (e & TDV_EBIT_TIES)
		return TDV_ERR_TIES;
	return 0;
}

/* ------------------------------------------------------------------------ */
/* gathers                                                                   */
/* ------------------------------------------------------------------------ */

template <typename T>
__global__ void k_gather(size_t n, const uint32_t *__restrict__ perm,
		const T *__restrict__ in, T *__restrict__ out)
{
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		out[i] = in[perm[i]];
}

void tdv_launch_gather_f64(tdv_context *c, size_t n, const uint32_t *perm,
		const double *in, double *out)
{
	hipLaunchKernelGGL(k_gather<double>, dim3(tdv_blocks(n, 256)), dim3(256),
			0, c->stream, n, perm, in, out);
}

void tdv_launch_gather_i32(tdv_context *c, size_t n, const uint32_t *perm,
		const int *in, int *out)
{
	hipLaunchKernelGGL(k_gather<int>, dim3(tdv_blocks(n, 256)), dim3(256), 0,
			c->stream, n, perm, in, out);
}

/* ---- the reorder (reorder_collisionless_particles, peano.c:50-82) --------
 *
 * Every column gathered by the sort's order.  A kernel takes several columns
 * per pass over the order, each into a spare buffer of its size that then
 * changes places with the column; the first also writes the walk's packed
 * records.  One kernel per column, the 32-bit ones copied back, took 28
 * launches and 40% more traffic. */
struct Cols3 {
	double *in[3], *out[3];
};

struct Cols5 {
	int *in[5], *out[5];
};

__global__ void k_reorder_pos(size_t n, const uint32_t *__restrict__ perm,
		const ulonglong2 *__restrict__ kin, ulonglong2 *__restrict__ kout,
		Cols3 c, const double *__restrict__ m, double4 *__restrict__ pm,
		unsigned *__restrict__ err, unsigned clear)
{
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i == 0)
		*err &= ~clear;
	if (i >= n)
		return;
	const uint32_t p = perm[i];
	const ulonglong2 k = kin[p];
	const double4 q = make_double4(c.in[0][p], c.in[1][p], c.in[2][p], m[p]);
	kout[i] = k;
	c.out[0][i] = q.x;
	c.out[1][i] = q.y;
	c.out[2][i] = q.z;
	pm[i] = q;
}

/* perm NULL: copied in place order (a captured step's way back) */
__global__ void k_reorder_f64(size_t n, const uint32_t *__restrict__ perm,
		Cols3 c)
{
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	const size_t p = perm ? perm[i] : i;
	const double a = c.in[0][p], b = c.in[1][p], d = c.in[2][p];
	c.out[0][i] = a;
	c.out[1][i] = b;
	c.out[2][i] = d;
}

__global__ void k_reorder_i32(size_t n, const uint32_t *__restrict__ perm,
		Cols5 c)
{
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	const size_t p = perm ? perm[i] : i;
	int v[5];
#pragma unroll
	for (int q = 0; q < 5; q++)
		v[q] = c.in[q][p];
#pragma unroll
	for (int q = 0; q < 5; q++)
		c.out[q][i] = v[q];
}

/* The particle columns, the key (key_tmp -> key) and pm in the order perm;
 * the error bits `clear` are dropped.  The spare buffers are the sort's and
 * the build's scratch, free here and of the columns' size.  A captured step
 * copies back instead of changing places, so each replay finds its columns
 * where they were. */
void tdv_launch_reorder(tdv_context *c, unsigned clear)
{
	const size_t n = c->n;
	const dim3 grid(tdv_blocks(n, 256)), block(256);
	double *spare[3] = { c->tmp_f64, reinterpret_cast<double *>(c->sk[0]),
		reinterpret_cast<double *>(c->sk[1]) };
	double **cols[5][3] = { { &c->pos[0], &c->pos[1], &c->pos[2] },
		{ &c->vel[0], &c->vel[1], &c->vel[2] },
		{ &c->acc[0], &c->acc[1], &c->acc[2] },
		{ &c->gacc[0], &c->gacc[1], &c->gacc[2] },
		{ &c->mass, &c->last_acc, &c->cost } };
	for (int g = 0; g < 5; g++) {
		Cols3 k;
		for (int q = 0; q < 3; q++) {
			k.in[q] = *cols[g][q];
			k.out[q] = spare[q];
		}
		if (g == 0)
			hipLaunchKernelGGL(k_reorder_pos, grid, block, 0, c->stream, n,
					c->perm, reinterpret_cast<const ulonglong2 *>(c->key_tmp),
					reinterpret_cast<ulonglong2 *>(c->key), k, c->mass, c->pm,
					c->d_err, clear);
		else
			hipLaunchKernelGGL(k_reorder_f64, grid, block, 0, c->stream, n,
					c->perm, k);
		for (int q = 0; q < 3; q++)
			if (c->graph_mode) {
				std::swap(k.in[q], k.out[q]);
			} else {
				*cols[g][q] = k.out[q];
				spare[q] = k.in[q];
			}
		if (c->graph_mode)
			hipLaunchKernelGGL(k_reorder_f64, grid, block, 0, c->stream, n,
					(const uint32_t *)nullptr, k);
	}
	c->tmp_f64 = spare[0];
	c->sk[0] = reinterpret_cast<uint64_t *>(spare[1]);
	c->sk[1] = reinterpret_cast<uint64_t *>(spare[2]);
	const Cols5 g = { { c->tree_parent, c->time_bin,
		reinterpret_cast<int *>(c->id), reinterpret_cast<int *>(c->it_drift),
		reinterpret_cast<int *>(c->it_kick) },
		{ c->cnt, c->lohi, reinterpret_cast<int *>(c->minpack),
		reinterpret_cast<int *>(c->sv[0]),
		reinterpret_cast<int *>(c->sv[1]) } };
	hipLaunchKernelGGL(k_reorder_i32, grid, block, 0, c->stream, n, c->perm,
			g);
	if (c->graph_mode) {
		Cols5 k;
		for (int q = 0; q < 5; q++) {
			k.in[q] = g.out[q];
			k.out[q] = g.in[q];
		}
		hipLaunchKernelGGL(k_reorder_i32, grid, block, 0, c->stream, n,
				(const uint32_t *)nullptr, k);
		return;
	}
	c->tree_parent = g.out[0];
	c->time_bin = g.out[1];
	c->id = reinterpret_cast<uint32_t *>(g.out[2]);
	c->it_drift = reinterpret_cast<uint32_t *>(g.out[3]);
	c->it_kick = reinterpret_cast<uint32_t *>(g.out[4]);
	c->cnt = g.in[0];
	c->lohi = g.in[1];
	c->minpack = reinterpret_cast<uint32_t *>(g.in[2]);
	c->sv[0] = reinterpret_cast<uint32_t *>(g.in[3]);
	c->sv[1] = reinterpret_cast<uint32_t *>(g.in[4]);
}

__global__ void k_pack_pm(size_t n, const double *__restrict__ x,
		const double *__restrict__ y, const double *__restrict__ z,
		const double *__restrict__ m, double4 *__restrict__ pm)
{
	const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		pm[i] = make_double4(x[i], y[i], z[i], m[i]);
}

void tdv_launch_pack_pm(tdv_context *c)
{
	if (!c->n)
		return;
	hipLaunchKernelGGL(k_pack_pm, dim3(tdv_blocks(c->n, 256)), dim3(256), 0,
			c->stream, c->n, c->pos[0], c->pos[1], c->pos[2], c->mass, c->pm);
}

/* ------------------------------------------------------------------------ */
/* non-periodic domain (domain.c:751-847, select.c:19-80)                    */
/* ------------------------------------------------------------------------ */

/* order-preserving u64 image of a double, and back */
__device__ __forceinline__ uint64_t f64_orderkey(double x)
{
	const uint64_t u = (uint64_t)__double_as_longlong(x);
	return (u >> 63) ? ~u : (u | (1ull << 63));
}

__host__ __device__ inline uint64_t f64_from_orderkey(uint64_t u)
{
	return (u >> 63) ? (u & ~(1ull << 63)) : ~u;
}

/* The k-th smallest of each of the three coordinates by radix selection: a
 * pass counts the next digit of the keys that share the prefix found so
 * far, and the last workgroup to finish extends the prefix by the digit
 * whose bin holds the k-th.  Six passes over 24 bytes per particle and one
 * launch each for all three; sorting each coordinate to read one element
 * took 24 radix passes of five launches, 1.1 ms of a 65,536-particle step.
 * Leaves the counters cleared for the next pass. */
#define SEL_BITS 11
#define SEL_BINS TDV_SELECT_BINS
#define SEL_THREADS 256
static_assert(SEL_BINS == 1 << SEL_BITS, "bins of a digit");

__global__ void k_select_init(SelectState *st, uint64_t k)
{
	for (int i = threadIdx.x; i < 3 * SEL_BINS; i += blockDim.x)
		st->hist[i] = 0;
	if (threadIdx.x < 3) {
		st->prefix[threadIdx.x] = 0;
		st->k[threadIdx.x] = k;
	}
	if (threadIdx.x == 0) {
		st->done = 0;
		st->maxd = 0;
	}
}

__global__ void __launch_bounds__(SEL_THREADS) k_select_pass(size_t n,
		const double *__restrict__ x, const double *__restrict__ y,
		const double *__restrict__ z, int shift, int bits, SelectState *st)
{
	__shared__ unsigned h[3 * SEL_BINS];
	__shared__ unsigned wsum[SEL_THREADS / 64];
	__shared__ unsigned last;
	const int tid = threadIdx.x;
	for (int i = tid; i < 3 * SEL_BINS; i += SEL_THREADS)
		h[i] = 0;
	const double *col[3] = { x, y, z };
	uint64_t prefix[3];
	for (int d = 0; d < 3; d++)
		prefix[d] = st->prefix[d];
	__syncthreads();
	const int above = shift + bits;      /* the prefix's lowest bit */
	const unsigned mask = (1u << bits) - 1;
	for (size_t i = (size_t)blockIdx.x * SEL_THREADS + tid; i < n;
			i += (size_t)gridDim.x * SEL_THREADS)
#pragma unroll
		for (int d = 0; d < 3; d++) {
			const uint64_t u = f64_orderkey(col[d][i]);
			if (above >= 64 || (u >> above) == prefix[d])
				atomicAdd(&h[d * SEL_BINS + ((unsigned)(u >> shift) & mask)],
						1u);
		}
	__syncthreads();
	for (int i = tid; i < 3 * SEL_BINS; i += SEL_THREADS)
		if (h[i])
			atomicAdd(&st->hist[i], h[i]);
	__threadfence();                     /* the counts before the ticket */
	__syncthreads();
	if (tid == 0)
		last = atomicAdd(&st->done, 1u) == gridDim.x - 1;
	__syncthreads();
	if (!last)
		return;
	/* the last workgroup: every count is in; read past this XCD's L2 */
	constexpr int PER = SEL_BINS / SEL_THREADS;
	for (int d = 0; d < 3; d++) {
		unsigned c[PER], sum = 0;
#pragma unroll
		for (int u = 0; u < PER; u++) {
			unsigned *p = &st->hist[d * SEL_BINS + tid * PER + u];
			c[u] = __hip_atomic_load(p, __ATOMIC_RELAXED,
					__HIP_MEMORY_SCOPE_AGENT);
			sum += c[u];
		}
		unsigned tot;
		const unsigned before = block_excl_scan(sum, &tot, wsum);
		const uint64_t k = st->k[d];
		__syncthreads();                 /* k read by all before it changes */
		if (k >= before && k < (uint64_t)before + sum) {
			unsigned b = before;
			int u = 0;
			while (k >= (uint64_t)b + c[u])
				b += c[u++];
			st->k[d] = k - b;
			st->prefix[d] = prefix[d] << bits | (unsigned)(tid * PER + u);
		}
	}
	__syncthreads();
	for (int i = tid; i < 3 * SEL_BINS; i += SEL_THREADS)
		st->hist[i] = 0;
	if (tid == 0)
		st->done = 0;
}

/* the largest distance on an axis from the centre just found */
__global__ void k_max_dist(size_t n, const double *__restrict__ x,
		const double *__restrict__ y, const double *__restrict__ z,
		SelectState *st)
{
	double c[3];
	for (int d = 0; d < 3; d++)
		c[d] = __longlong_as_double((long long)f64_from_orderkey(
				st->prefix[d]));
	/* non-negative doubles order like their bit patterns */
	unsigned long long b = 0;
	for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
			i += (size_t)gridDim.x * blockDim.x) {
		const unsigned long long v = (unsigned long long)__double_as_longlong(
				fmax(fmax(fabs(x[i] - c[0]), fabs(y[i] - c[1])),
				fabs(z[i] - c[2])));
		b = v > b ? v : b;
	}
	for (int d = 32; d >= 1; d >>= 1) {
		unsigned long long o = __shfl_xor(b, d, 64);
		b = o > b ? o : b;
	}
	if ((threadIdx.x & 63) == 0)
		atomicMax(&st->maxd, b);
}

int tdv_domain_nonperiodic(tdv_context *c)
{
	const size_t n = c->n;
	if (n < 3)
		return tdv_fail(c, TDV_ERR_ARG, "non-periodic domain needs 3 particles");
	/* Select(n>>1, n, data) orders data[1..n-1] and returns position n>>1 of
	 * that 1-based range, i.e. the ((n>>1)-1)-th smallest of data[1..n-1] */
	const size_t m = n - 1, k = (n >> 1) - 1;
	SelectState *st = c->select;
	const unsigned grid = (unsigned)std::min((size_t)tdv_blocks(m, 1024),
			(size_t)512);
	hipLaunchKernelGGL(k_select_init, dim3(1), dim3(1024), 0, c->stream, st,
			(uint64_t)k);
	for (int above = 64; above > 0; ) {
		const int bits = above < SEL_BITS ? above : SEL_BITS;
		above -= bits;
		hipLaunchKernelGGL(k_select_pass, dim3(grid), dim3(SEL_THREADS), 0,
				c->stream, m, c->pos[0] + 1, c->pos[1] + 1, c->pos[2] + 1,
				above, bits, st);
	}
	hipLaunchKernelGGL(k_max_dist, dim3(grid), dim3(SEL_THREADS), 0,
			c->stream, n, c->pos[0], c->pos[1], c->pos[2], st);
	TDV_HIP(c, hipGetLastError());
	SelectState h;
	TDV_HIP(c, hipMemcpyAsync(&h, st, offsetof(SelectState, k),
			hipMemcpyDeviceToHost, c->stream));
	TDV_HIP(c, hipStreamSynchronize(c->stream));
	for (int d = 0; d < 3; d++) {
		const uint64_t u = f64_from_orderkey(h.prefix[d]);
		memcpy(&c->dom_center[d], &u, 8);
	}
	double maxd;
	memcpy(&maxd, &h.maxd, 8);
	c->dom_size = 2.001 * maxd;
	for (int d = 0; d < 3; d++)
		c->dom_origin[d] = c->dom_center[d] - 0.5 * c->dom_size;
	return 0;
}
