/* Data-parallel building blocks of the pipeline: exclusive scan, a stable
 * LSD radix sort used for ordered binning (tile lists, per-pixel fragment
 * lists), fills. */
#include "kernels.h"

#include <algorithm>

namespace srp {
namespace lib {

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_CHUNK = SCAN_THREADS * SCAN_ITEMS;
static_assert(SCAN_ITEMS == 8, "k_scan_blocks loads a thread's values as two 16-byte vectors");

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_local(uint32_t* data, size_t n, uint32_t* sums)
{
	__shared__ uint32_t sh[SCAN_THREADS];
	const uint32_t t = threadIdx.x;
	const size_t base = (size_t) blockIdx.x * SCAN_CHUNK + (size_t) t * SCAN_ITEMS;
	uint32_t v[SCAN_ITEMS];
	uint32_t sum = 0;
#pragma unroll
	for (int j = 0; j < SCAN_ITEMS; j++)
	{
		const size_t i = base + j;
		v[j] = (i < n) ? data[i] : 0u;
		sum += v[j];
	}
	sh[t] = sum;
	__syncthreads();
	for (uint32_t off = 1; off < SCAN_THREADS; off <<= 1)
	{
		const uint32_t x = (t >= off) ? sh[t - off] : 0u;
		__syncthreads();
		sh[t] += x;
		__syncthreads();
	}
	uint32_t run = sh[t] - sum;
#pragma unroll
	for (int j = 0; j < SCAN_ITEMS; j++)
	{
		const size_t i = base + j;
		if (i < n) data[i] = run;
		run += v[j];
	}
	if (t == SCAN_THREADS - 1)
		sums[blockIdx.x] = sh[t];
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_add(uint32_t* data, size_t n, const uint32_t* sums)
{
	const uint32_t add = sums[blockIdx.x];
	const size_t base = (size_t) blockIdx.x * SCAN_CHUNK;
	for (int j = 0; j < SCAN_ITEMS; j++)
	{
		const size_t i = base + (size_t) j * SCAN_THREADS + threadIdx.x;
		if (i < n) data[i] += add;
	}
}

__global__ void k_copy1(const uint32_t* src, uint32_t* dst) { *dst = *src; }

void copyU32(const uint32_t* src, uint32_t* dst, hipStream_t s)
{
	hipLaunchKernelGGL(k_copy1, dim3(1), dim3(1), 0, s, src, dst);
}

static void scanLevel(uint32_t* data, size_t n, uint32_t* total, uint32_t* scratch, hipStream_t s)
{
	const size_t nb = (n + SCAN_CHUNK - 1) / SCAN_CHUNK;
	uint32_t* sums = scratch;
	hipLaunchKernelGGL(k_scan_local, dim3((uint32_t) nb), dim3(SCAN_THREADS), 0, s, data, n, sums);
	if (nb == 1)
	{
		hipLaunchKernelGGL(k_copy1, dim3(1), dim3(1), 0, s, sums, total);
		return;
	}
	scanLevel(sums, nb, total, scratch + nb, s);
	hipLaunchKernelGGL(k_scan_add, dim3((uint32_t) nb), dim3(SCAN_THREADS), 0, s, data, n, sums);
}

void scanExclusive(uint32_t* data, size_t n, uint32_t* total, ScanScratch& scratch, hipStream_t s)
{
	if (n == 0)
	{
		fillU32(total, 0u, 1, s);
		return;
	}
	size_t need = 0;
	for (size_t m = n; m > 1; m = (m + SCAN_CHUNK - 1) / SCAN_CHUNK)
		need += (m + SCAN_CHUNK - 1) / SCAN_CHUNK;
	need += 2;
	if (need > scratch.cap)
	{
		if (scratch.buf) hipFree(scratch.buf);
		scratch.cap = need * 2;
		hipMalloc(&scratch.buf, scratch.cap * sizeof(uint32_t));
	}
	scanLevel(data, n, total, scratch.buf, s);
}

/* Two-launch exclusive scan of up to a few equal-length arrays (grid.y
 * selects the array): block-local scans and block totals, then each block
 * adds the sum of the totals before it (summed redundantly per block, which
 * is cheaper than a third launch while there are at most a few thousand
 * blocks).  The last block writes the array's grand total. */
__global__ __launch_bounds__(SCAN_THREADS) void k_scan_blocks(uint32_t* base, size_t stride, size_t n, uint32_t* sums,
                                                              unsigned long long* sums64, uint32_t nb)
{
	uint32_t* data = base + (size_t) blockIdx.y * stride;
	__shared__ uint32_t waveTot[SCAN_THREADS / 64];
	__shared__ unsigned long long waveSum[SCAN_THREADS / 64];
	const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
	const size_t b0 = (size_t) blockIdx.x * SCAN_CHUNK + (size_t) t * SCAN_ITEMS;
	/* this thread's SCAN_ITEMS consecutive values: two 16-byte loads when
	 * they are all there and aligned (the arrays of one launch start at
	 * arbitrary word offsets) */
	const bool vec = b0 + SCAN_ITEMS <= n && (reinterpret_cast<uintptr_t>(data + b0) & 15u) == 0;
	uint32_t v[SCAN_ITEMS];
	if (vec)
	{
		const uint4 a = *reinterpret_cast<const uint4*>(data + b0);
		const uint4 b = *reinterpret_cast<const uint4*>(data + b0 + 4);
		v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
		v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
	}
	else
	{
#pragma unroll
		for (int j = 0; j < SCAN_ITEMS; j++)
			v[j] = (b0 + j < n) ? data[b0 + j] : 0u;
	}
	uint32_t sum = 0;
	unsigned long long wide = 0;
#pragma unroll
	for (int j = 0; j < SCAN_ITEMS; j++)
	{
		sum += v[j];
		wide += v[j];
	}
	/* inclusive scan of the threads' sums within the wave, then across the
	 * block's waves.  (The block's sum may wrap: the offsets below are
	 * exact only while the array's total fits 32 bits, which the caller
	 * checks; the 64-bit sums are exact.) */
	uint32_t incl = sum;
#pragma unroll
	for (int off = 1; off < 64; off <<= 1)
	{
		const uint32_t x = __shfl_up(incl, off);
		if ((int) lane >= off) incl += x;
	}
	for (int off = 32; off > 0; off >>= 1)
		wide += __shfl_xor(wide, off);
	if (lane == 63u)
	{
		waveTot[wave] = incl;
		waveSum[wave] = wide;
	}
	__syncthreads();
	uint32_t run = incl - sum;
	for (uint32_t w = 0; w < wave; w++)
		run += waveTot[w];
#pragma unroll
	for (int j = 0; j < SCAN_ITEMS; j++)
	{
		const uint32_t x = v[j];
		v[j] = run;
		run += x;
	}
	if (vec)
	{
		*reinterpret_cast<uint4*>(data + b0) = make_uint4(v[0], v[1], v[2], v[3]);
		*reinterpret_cast<uint4*>(data + b0 + 4) = make_uint4(v[4], v[5], v[6], v[7]);
	}
	else
	{
#pragma unroll
		for (int j = 0; j < SCAN_ITEMS; j++)
			if (b0 + j < n) data[b0 + j] = v[j];
	}
	if (t == SCAN_THREADS - 1)
	{
		uint32_t bs = 0;
		unsigned long long w = 0;
		for (int k = 0; k < SCAN_THREADS / 64; k++)
		{
			bs += waveTot[k];
			w += waveSum[k];
		}
		sums[(size_t) blockIdx.y * nb + blockIdx.x] = bs;
		sums64[(size_t) blockIdx.y * nb + blockIdx.x] = w;
	}
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_finish(uint32_t* base, size_t stride, size_t n,
                                                              const uint32_t* sums, const unsigned long long* sums64,
                                                              uint32_t nb, uint32_t* totals,
                                                              unsigned long long* totals64)
{
	uint32_t* data = base + (size_t) blockIdx.y * stride;
	const uint32_t* s = sums + (size_t) blockIdx.y * nb;
	__shared__ uint32_t red[SCAN_THREADS / 64];
	const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
	uint32_t acc = 0;
	for (uint32_t k = t; k < blockIdx.x; k += SCAN_THREADS) acc += s[k];
	for (int off = 32; off > 0; off >>= 1)
		acc += __shfl_xor(acc, off);
	if (lane == 0)
		red[wave] = acc;
	__syncthreads();
	uint32_t add = 0;
	for (int w = 0; w < SCAN_THREADS / 64; w++)
		add += red[w];
	const size_t b0 = (size_t) blockIdx.x * SCAN_CHUNK;
	if (add)
		for (int j = 0; j < SCAN_ITEMS; j++)
		{
			const size_t i = b0 + (size_t) j * SCAN_THREADS + t;
			if (i < n) data[i] += add;
		}
	if (blockIdx.x == nb - 1)
	{
		if (t == 0)
			totals[blockIdx.y] = add + s[blockIdx.x];
		if (totals64)
		{
			/* the array's exact total (the last block reduces every block's) */
			__shared__ unsigned long long red64[SCAN_THREADS / 64];
			const unsigned long long* s64 = sums64 + (size_t) blockIdx.y * nb;
			unsigned long long acc64 = 0;
			for (uint32_t k = t; k < nb; k += SCAN_THREADS) acc64 += s64[k];
			for (int off = 32; off > 0; off >>= 1)
				acc64 += __shfl_xor(acc64, off);
			if (lane == 0)
				red64[wave] = acc64;
			__syncthreads();
			if (t == 0)
			{
				unsigned long long tot = 0;
				for (int w = 0; w < SCAN_THREADS / 64; w++)
					tot += red64[w];
				totals64[blockIdx.y] = tot;
			}
		}
	}
}

/* Exact (64-bit) sum of n u32 values added into *out (zeroed by the caller). */
__global__ __launch_bounds__(SCAN_THREADS) void k_sum64(const uint32_t* data, size_t n, unsigned long long* out)
{
	unsigned long long acc = 0;
	for (size_t i = (size_t) blockIdx.x * SCAN_THREADS + threadIdx.x; i < n; i += (size_t) gridDim.x * SCAN_THREADS)
		acc += data[i];
	for (int off = 32; off > 0; off >>= 1)
		acc += __shfl_xor(acc, off);
	if ((threadIdx.x & 63u) == 0 && acc)
		atomicAdd(out, acc);
}

void scanExclusiveMulti(uint32_t* base, size_t stride, int nArrays, size_t n, uint32_t* totals, ScanScratch& scratch,
                        hipStream_t s, unsigned long long* totals64)
{
	if (n == 0)
	{
		fillU32(totals, 0u, (size_t) nArrays, s);
		if (totals64)
			fillU32(reinterpret_cast<uint32_t*>(totals64), 0u, (size_t) nArrays * 2, s);
		return;
	}
	const size_t nb = (n + SCAN_CHUNK - 1) / SCAN_CHUNK;
	if (nb > 8192)
	{
		if (totals64)
		{
			fillU32(reinterpret_cast<uint32_t*>(totals64), 0u, (size_t) nArrays * 2, s);
			const size_t blocks = (n + SCAN_THREADS - 1) / SCAN_THREADS;
			const uint32_t g = (uint32_t) (blocks < 2048 ? blocks : 2048);
			for (int a = 0; a < nArrays; a++)
				hipLaunchKernelGGL(k_sum64, dim3(g), dim3(SCAN_THREADS), 0, s, base + (size_t) a * stride, n,
				                   totals64 + a);
		}
		for (int a = 0; a < nArrays; a++)
			scanExclusive(base + (size_t) a * stride, n, totals + a, scratch, s);
		return;
	}
	scanReserve(scratch, n, nArrays);
	const dim3 grid((uint32_t) nb, (uint32_t) nArrays);
	hipLaunchKernelGGL(k_scan_blocks, grid, dim3(SCAN_THREADS), 0, s, base, stride, n, scratch.buf, scratch.buf64,
	                   (uint32_t) nb);
	hipLaunchKernelGGL(k_scan_finish, grid, dim3(SCAN_THREADS), 0, s, base, stride, n, scratch.buf, scratch.buf64,
	                   (uint32_t) nb, totals, totals64);
}

/* Tile ranges of a list sorted by tile: [start, end) per tile; tiles that
 * received nothing keep start == end == 0 (set by the caller's fill).  A
 * thread takes EACH items: four from one load where the list is long, one
 * where it is short and the threads few.  us with one and with four, traced:
 * 37 k items 2.2 and 3.4, 350 k 2.6 and 3.7, 0.75 M and 1.4 M 5.3 and 5.3,
 * 3.0 M 6.6 and 5.8, 7.4 M 11.7 and 9.1, 18 M 24 and 17, 74 M 111 and 69. */
constexpr size_t TB_LONG_FROM = (size_t) 4 << 20;

template <int EACH>
__global__ __launch_bounds__(256) void k_tile_bounds(const uint32_t* keys, size_t n, const uint32_t* nDev,
                                                     uint32_t* start, uint32_t* end)
{
	if (nDev && *nDev < n) n = *nDev;
	const size_t i = ((size_t) blockIdx.x * 256u + threadIdx.x) * EACH;
	if (i >= n) return;
	uint32_t k[EACH + 2];   /* items i - 1 .. i + EACH */
	k[0] = i ? keys[i - 1] : 0u;
	if (EACH == 4 && i + EACH <= n)
	{
		const uint4 v = *reinterpret_cast<const uint4*>(keys + i);
		k[1] = v.x;
		k[EACH > 1 ? 2 : 1] = v.y;
		k[EACH > 1 ? 3 : 1] = v.z;
		k[EACH > 1 ? 4 : 1] = v.w;
	}
	else
	{
#pragma unroll
		for (int q = 0; q < EACH; q++)
			k[1 + q] = i + (size_t) q < n ? keys[i + (size_t) q] : 0u;
	}
	k[EACH + 1] = i + EACH < n ? keys[i + EACH] : 0u;
#pragma unroll
	for (int q = 0; q < EACH; q++)
		if (i + (size_t) q < n)
		{
			const size_t at = i + (size_t) q;
			if (at == 0 || k[q] != k[q + 1]) start[k[q + 1]] = (uint32_t) at;
			if (at + 1 == n || k[q + 2] != k[q + 1]) end[k[q + 1]] = (uint32_t) (at + 1);
		}
}

void tileBounds(const uint32_t* keys, size_t n, uint32_t* start, uint32_t* end, hipStream_t s, const uint32_t* nDev)
{
	if (n > TB_LONG_FROM)
		hipLaunchKernelGGL(k_tile_bounds<4>, dim3((uint32_t) ((n + 1023) / 1024)), dim3(256), 0, s, keys, n, nDev, start, end);
	else if (n)
		hipLaunchKernelGGL(k_tile_bounds<1>, dim3((uint32_t) ((n + 255) / 256)), dim3(256), 0, s, keys, n, nDev, start, end);
}

/* ------------------------------------------------------------ radix sort */

constexpr int RS_THREADS = 256;
constexpr int RS_SLICES = 2;     /* slices of RS_THREADS items ranked per round */
constexpr int RS_CHUNK = 1024;   /* items per block: more blocks than CUs for the 1080p mesh's ~350 k pairs
                                   (measured: 4096 0.234 ms/frame, 2048 0.223, 1024 0.219) */
/* A sort of more than RS_LONG_FROM items takes whole rounds of
 * RS_LONG_ROUND items a block (k_radix_scatter_long), some RS_LONG_BLOCKS
 * blocks of at most RS_LONG_CHUNK: enough to fill the chip several times
 * over, and few enough digit counts to scan.  Kernel time of two passes over
 * the tile pairs of large triangles, us with the short sort's blocks and with
 * these: 1.05 M items 73 and 51, 1.5 M 88 and 53, 2 M 110 and 55, 4 M 184 and
 * 84, 8 M 345 and 135, 40 M 1,549 and 570.  (300 k: 36 and 44, fused passes
 * and not.)  1,024 and 4,096 blocks: within the noise up to 8 M, 245 and 236
 * against 221 at 16 M, 587 and 563 against 570 at 40 M. */
constexpr int RS_LONG_ROUND = 4096;
constexpr int RS_LONG_CHUNK = 32768;
constexpr int RS_LONG_BLOCKS = 2048;
constexpr size_t RS_LONG_FROM = (size_t) 1 << 20;

/* The block size a sort of n items uses (identical for its reservation). */
inline uint32_t rsChunk(size_t n)
{
	if (n <= RS_LONG_FROM)
		return (uint32_t) RS_CHUNK;
	const size_t rounds = (n / RS_LONG_BLOCKS + RS_LONG_ROUND - 1) / RS_LONG_ROUND;
	return (uint32_t) std::min<size_t>(rounds * RS_LONG_ROUND, RS_LONG_CHUNK);
}

/* Up to this many blocks, each scatter block sums the per-block digit counts
 * itself (reading all of them from L2) instead of a separate scan over them:
 * two launches per pass fewer, at nBlocks KiB of L2 reads per block. */
constexpr uint32_t RS_FUSED_MAX_BLOCKS = 512;

/* Up to RS_FUSED_MAX_BLOCKS blocks, the digit counts are also summed per
 * group of RS_GROUP consecutive blocks (grp[group * 256 + digit], atomics),
 * so that a scatter block finds its offsets from the group rows and at most
 * RS_GROUP - 1 block rows.  The groups' sums are zero when a pass starts:
 * the last scatter block of each pass to read them clears them (and the
 * pass's counter of such blocks, grp[RS_GROUP_WORDS]). */
constexpr uint32_t RS_GROUP = 16;
constexpr uint32_t RS_GROUP_WORDS = RS_FUSED_MAX_BLOCKS / RS_GROUP * 256u;

/* Digit counts of one block of `chunk` keys, written at
 * hist[digit * digitStride + block * blockStride]; with grp, also added to
 * the block's group row.  A thread has RS_HIST_AHEAD keys in flight. */
constexpr int RS_HIST_AHEAD = 4;
__global__ __launch_bounds__(RS_THREADS) void k_radix_hist(const uint32_t* keys, size_t n, const uint32_t* nDev,
                                                           uint32_t shift, uint32_t* hist, uint32_t digitStride,
                                                           uint32_t blockStride, uint32_t chunk, uint32_t* grp)
{
	if (nDev && *nDev < n) n = *nDev;
	__shared__ uint32_t h[256];
	const uint32_t t = threadIdx.x;
	h[t] = 0;
	__syncthreads();
	const size_t begin = (size_t) blockIdx.x * chunk;
	const size_t end = (begin + chunk < n) ? begin + chunk : n;
	for (size_t i = begin + t; i < end; i += RS_THREADS * RS_HIST_AHEAD)
	{
		uint32_t k[RS_HIST_AHEAD];
#pragma unroll
		for (int q = 0; q < RS_HIST_AHEAD; q++)
			k[q] = i + (size_t) q * RS_THREADS < end ? keys[i + (size_t) q * RS_THREADS] : 0u;
#pragma unroll
		for (int q = 0; q < RS_HIST_AHEAD; q++)
			if (i + (size_t) q * RS_THREADS < end)
				atomicAdd(&h[(k[q] >> shift) & 255u], 1u);
	}
	__syncthreads();
	hist[(size_t) t * digitStride + (size_t) blockIdx.x * blockStride] = h[t];
	if (grp && h[t])
		atomicAdd(grp + (blockIdx.x / RS_GROUP) * 256u + t, h[t]);
}

/* Stable scatter: items keep their input order within a digit.  Each tile
 * of 256 items ranks its items per digit with wave ballots, then by wave.
 * FUSED: hist holds raw block-major counts (hist[block * 256 + digit]), grp
 * their sums per group of blocks, and the block finds its digits' offsets
 * itself; otherwise hist holds the exclusive scan of the digit-major
 * counts. */
template <bool FUSED>
__global__ __launch_bounds__(RS_THREADS) void k_radix_scatter(const uint32_t* keysIn, const uint32_t* valsIn,
                                                              uint32_t* keysOut, uint32_t* valsOut, size_t n,
                                                              const uint32_t* nDev, uint32_t shift, const uint32_t* hist,
                                                              uint32_t nBlocks, uint32_t chunk, uint32_t* grp)
{
	if (nDev && *nDev < n) n = *nDev;
	/* blocks past the device count (a capacity-sized grid) have nothing to
	 * place; whole blocks leave together, before any barrier */
	if ((size_t) blockIdx.x * chunk >= n)
		return;
	/* hist rows of blocks past the count are zero: not read */
	const uint32_t usedBlocks = (uint32_t) ((n + chunk - 1) / chunk);
	__shared__ uint32_t running[256];
	__shared__ uint32_t sliceCnt[RS_SLICES * 4][256];
	__shared__ uint32_t tileTotal[256];
	__shared__ bool lastReader;
	uint32_t (*waveCnt)[256] = sliceCnt;   /* the offsets prologue's per-wave sums */
	const uint32_t t = threadIdx.x;
	const uint32_t lane = t & 63u, wave = t >> 6;
	if (FUSED)
	{
		/* Digit t: items of all blocks (total) and of the blocks before
		 * this one (before), from the group rows and then the block rows
		 * of this block's group before it.  Wave w reads every fourth row,
		 * a lane four digits at once; the four waves' sums meet in LDS. */
		__shared__ uint32_t befCnt[4][256];
		const uint32_t d4 = 4u * lane;
		const uint32_t myGroup = blockIdx.x / RS_GROUP;
		const uint32_t nGroups = (usedBlocks + RS_GROUP - 1) / RS_GROUP;
		uint32_t tot[4] = {0u, 0u, 0u, 0u}, bef[4] = {0u, 0u, 0u, 0u};
		for (uint32_t g = wave; g < nGroups; g += 4u)
		{
			const uint4 v = *reinterpret_cast<const uint4*>(grp + (size_t) g * 256u + d4);
			const uint32_t vv[4] = {v.x, v.y, v.z, v.w};
			const uint32_t take = (g < myGroup) ? ~0u : 0u;
#pragma unroll
			for (int k = 0; k < 4; k++)
			{
				tot[k] += vv[k];
				bef[k] += vv[k] & take;
			}
		}
		for (uint32_t b = myGroup * RS_GROUP + wave; b < blockIdx.x; b += 4u)
		{
			const uint4 v = *reinterpret_cast<const uint4*>(hist + (size_t) b * 256u + d4);
			bef[0] += v.x;
			bef[1] += v.y;
			bef[2] += v.z;
			bef[3] += v.w;
		}
#pragma unroll
		for (int k = 0; k < 4; k++)
		{
			waveCnt[wave][d4 + k] = tot[k];
			befCnt[wave][d4 + k] = bef[k];
		}
		__syncthreads();
		const uint32_t total = waveCnt[0][t] + waveCnt[1][t] + waveCnt[2][t] + waveCnt[3][t];
		const uint32_t before = befCnt[0][t] + befCnt[1][t] + befCnt[2][t] + befCnt[3][t];
		/* exclusive scan of the totals over the 256 digits */
		uint32_t incl = total;
		for (int off = 1; off < 64; off <<= 1)
		{
			const uint32_t v = __shfl_up(incl, off);
			if ((int) lane >= off) incl += v;
		}
		if (lane == 63u)
			tileTotal[wave] = incl;
		__syncthreads();   /* also: every total read before waveCnt is reused below */
		uint32_t waveBase = 0;
		for (uint32_t w = 0; w < wave; w++)
			waveBase += tileTotal[w];
		running[t] = waveBase + incl - total + before;
		/* Every group row this block reads has been read (the sums above
		 * are done); the block that finishes reading last clears the rows
		 * and the counter for the next pass. */
		if (t == 0)
			lastReader = atomicAdd(grp + RS_GROUP_WORDS, 1u) == usedBlocks - 1u;
		__syncthreads();
	}
	else
		running[t] = hist[(size_t) t * nBlocks + blockIdx.x];
	const size_t begin = (size_t) blockIdx.x * chunk;
	const size_t end = (begin + chunk < n) ? begin + chunk : n;
	const uint64_t ltMask = (lane == 0) ? 0ull : ((~0ull) >> (64u - lane));
	/* Rounds of RS_SLICES slices of RS_THREADS items; item order is slice,
	 * then wave, then lane, and so is the order of the per-(slice, wave)
	 * digit counts summed below. */
	for (size_t base = begin; base < end; base += (size_t) RS_SLICES * RS_THREADS)
	{
		for (int k = 0; k < RS_SLICES * 4; k++) sliceCnt[k][t] = 0;
		__syncthreads();
		uint32_t key[RS_SLICES], val[RS_SLICES], d[RS_SLICES], rank[RS_SLICES];
		bool valid[RS_SLICES];
#pragma unroll
		for (int sl = 0; sl < RS_SLICES; sl++)
		{
			const size_t i = base + (size_t) sl * RS_THREADS + t;
			valid[sl] = i < end;
			key[sl] = 0; val[sl] = 0; d[sl] = 0;
			if (valid[sl])
			{
				key[sl] = keysIn[i];
				val[sl] = valsIn ? valsIn[i] : (uint32_t) i;
				d[sl] = (key[sl] >> shift) & 255u;
			}
		}
#pragma unroll
		for (int sl = 0; sl < RS_SLICES; sl++)
		{
			uint64_t peers = __ballot(valid[sl]);
#pragma unroll
			for (int b = 0; b < 8; b++)
			{
				const bool bit = (d[sl] >> b) & 1u;
				const uint64_t m = __ballot(bit);
				peers &= bit ? m : ~m;
			}
			rank[sl] = (uint32_t) __popcll(peers & ltMask);
			if (valid[sl] && rank[sl] == 0)
				sliceCnt[sl * 4 + wave][d[sl]] = (uint32_t) __popcll(peers);
		}
		__syncthreads();
		{
			uint32_t sum = 0;
			for (int k = 0; k < RS_SLICES * 4; k++)
			{
				const uint32_t c = sliceCnt[k][t];
				sliceCnt[k][t] = sum;
				sum += c;
			}
			tileTotal[t] = sum;
		}
		__syncthreads();
#pragma unroll
		for (int sl = 0; sl < RS_SLICES; sl++)
			if (valid[sl])
			{
				const uint32_t dst = running[d[sl]] + sliceCnt[sl * 4 + wave][d[sl]] + rank[sl];
				keysOut[dst] = key[sl];
				valsOut[dst] = val[sl];
			}
		__syncthreads();
		running[t] += tileTotal[t];
	}
	if (FUSED && lastReader)
	{
		const uint32_t nGroups = (usedBlocks + RS_GROUP - 1) / RS_GROUP;
		for (uint32_t i = t; i < nGroups * 256u; i += RS_THREADS)
			grp[i] = 0u;
		if (t == 0)
			grp[RS_GROUP_WORDS] = 0u;
	}
}

/* The scatter of a long sort (hist: the exclusive scan of the digit-major
 * counts).  A round's 4,096 items are put in digit order in LDS first, so
 * that they leave in runs of sixteen a digit on average, whole lines where
 * one item at a time would write each line in pieces, from several rounds,
 * with more lines open than the L2s hold.  A wave ranks 1,024 consecutive
 * items, 64 at a time, as k_tile_sort does.
 * The binning of a 1920x1080 mix, 73 M pairs a pass: 1,200 us with the short
 * rounds' scatter, 440 so (550 where the digits are the tiles' low bits). */
constexpr int RS_LONG_EACH = RS_LONG_ROUND / RS_THREADS;

__global__ __launch_bounds__(RS_THREADS) void k_radix_scatter_long(const uint32_t* __restrict__ keysIn,
                                                                   const uint32_t* __restrict__ valsIn,
                                                                   uint32_t* __restrict__ keysOut,
                                                                   uint32_t* __restrict__ valsOut, size_t n,
                                                                   const uint32_t* nDev, uint32_t shift,
                                                                   const uint32_t* __restrict__ hist, uint32_t nBlocks,
                                                                   uint32_t chunk)
{
	if (nDev && *nDev < n) n = *nDev;
	const size_t begin = (size_t) blockIdx.x * chunk;
	if (begin >= n)
		return;
	__shared__ uint32_t sortedKey[RS_LONG_ROUND], sortedVal[RS_LONG_ROUND];
	__shared__ uint32_t cnt[4][256];
	__shared__ uint32_t placeOf[256];   /* digit: its first output place less its first place in the round */
	__shared__ uint32_t waveSum[4];
	const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
	const uint64_t below = (1ull << lane) - 1ull;
	const size_t end = (begin + chunk < n) ? begin + chunk : n;
	uint32_t running = hist[(size_t) t * nBlocks + blockIdx.x];   /* digit t's next output place */
	for (size_t base = begin; base < end; base += RS_LONG_ROUND)
	{
		const uint32_t have = (uint32_t) (end - base < (size_t) RS_LONG_ROUND ? end - base : (size_t) RS_LONG_ROUND);
		const uint32_t first = wave * (RS_LONG_ROUND / 4) + lane;
		uint32_t key[RS_LONG_EACH], val[RS_LONG_EACH], place[RS_LONG_EACH];
#pragma unroll
		for (int k = 0; k < RS_LONG_EACH; k++)
		{
			const uint32_t i = first + 64u * (uint32_t) k;
			key[k] = i < have ? keysIn[base + i] : 0u;
			val[k] = valsIn ? (i < have ? valsIn[base + i] : 0u) : (uint32_t) (base + i);
		}
#pragma unroll
		for (int d = 0; d < 4; d++)
			cnt[wave][lane + 64u * (uint32_t) d] = 0u;
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
		for (int k = 0; k < RS_LONG_EACH; k++)
		{
			const bool valid = first + 64u * (uint32_t) k < have;
			const uint32_t d = (key[k] >> shift) & 255u;
			uint64_t peers = __ballot(valid);
#pragma unroll
			for (int b = 0; b < 8; b++)
			{
				const bool bit = (d >> b) & 1u;
				const uint64_t m = __ballot(bit);
				peers &= bit ? m : ~m;
			}
			const uint32_t rank = (uint32_t) __popcll(peers & below);
			const uint32_t before = cnt[wave][d];
			place[k] = before + rank;
			__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
			if (valid && rank == 0)
				cnt[wave][d] = before + (uint32_t) __popcll(peers);
			__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
		}
		__syncthreads();
		uint32_t sum = 0, c[4];
#pragma unroll
		for (int w = 0; w < 4; w++)
		{
			c[w] = sum;
			sum += cnt[w][t];
		}
		uint32_t incl = sum;
#pragma unroll
		for (uint32_t off = 1; off < 64; off <<= 1)
		{
			const uint32_t v = __shfl_up(incl, off);
			if (lane >= off) incl += v;
		}
		if (lane == 63u)
			waveSum[wave] = incl;
		__syncthreads();
		uint32_t at = incl - sum;   /* digit t's first place in the round */
		for (uint32_t w = 0; w < wave; w++)
			at += waveSum[w];
#pragma unroll
		for (int w = 0; w < 4; w++)
			cnt[w][t] = at + c[w];
		placeOf[t] = running - at;
		running += sum;
		__syncthreads();
#pragma unroll
		for (int k = 0; k < RS_LONG_EACH; k++)
			if (first + 64u * (uint32_t) k < have)
			{
				const uint32_t p = cnt[wave][(key[k] >> shift) & 255u] + place[k];
				sortedKey[p] = key[k];
				sortedVal[p] = val[k];
			}
		__syncthreads();
#pragma unroll
		for (int k = 0; k < RS_LONG_EACH; k++)
		{
			const uint32_t p = t + RS_THREADS * (uint32_t) k;
			if (p < have)
			{
				const uint32_t key1 = sortedKey[p];
				const uint32_t dst = placeOf[(key1 >> shift) & 255u] + p;
				keysOut[dst] = key1;
				valsOut[dst] = sortedVal[p];
			}
		}
		/* the next round's first writes of cnt are each wave's to its own
		 * row, which since the last barrier only that wave reads; its writes
		 * of the sorted items follow this round's reads by three barriers */
	}
}

/* Scratch of a multi-array scan of nArrays x n values, allocated now. */
void scanReserve(ScanScratch& sc, size_t n, int nArrays)
{
	if (n == 0)
		return;
	const size_t nb = (n + SCAN_CHUNK - 1) / SCAN_CHUNK;
	size_t need;
	if (nb > 8192)
	{
		need = 2;
		for (size_t m = n; m > 1; m = (m + SCAN_CHUNK - 1) / SCAN_CHUNK)
			need += (m + SCAN_CHUNK - 1) / SCAN_CHUNK;
	}
	else
		need = nb * (size_t) nArrays + 2;
	if (need > sc.cap)
	{
		if (sc.buf) hipFree(sc.buf);
		sc.cap = need * 2;
		hipMalloc(&sc.buf, sc.cap * sizeof(uint32_t));
	}
	if (nb <= 8192 && need > sc.cap64)
	{
		if (sc.buf64) hipFree(sc.buf64);
		sc.cap64 = need * 2;
		hipMalloc(&sc.buf64, sc.cap64 * sizeof(unsigned long long));
	}
}

void radixSortReserve(SortScratch& sc, size_t n)
{
	if (n <= 1)
		return;
	const uint32_t chunk = rsChunk(n);
	const uint32_t nBlocks = (uint32_t) ((n + chunk - 1) / chunk);
	if (n > sc.cap)
	{
		if (sc.keys) hipFree(sc.keys);
		if (sc.vals) hipFree(sc.vals);
		sc.cap = n + n / 2;
		hipMalloc(&sc.keys, sc.cap * sizeof(uint32_t));
		hipMalloc(&sc.vals, sc.cap * sizeof(uint32_t));
	}
	const size_t histN = (size_t) 256 * nBlocks;
	if (histN + 1 > sc.histCap)
	{
		if (sc.hist) hipFree(sc.hist);
		sc.histCap = (histN + 1) * 2;
		hipMalloc(&sc.hist, sc.histCap * sizeof(uint32_t));
	}
	if (nBlocks > RS_FUSED_MAX_BLOCKS || chunk != (uint32_t) RS_CHUNK)
		scanReserve(sc.scan, histN, 1);
	else if (!sc.grp)
	{
		/* zeroed once (a copy, complete on return); every fused pass leaves
		 * it zero again */
		static const uint32_t zeros[RS_GROUP_WORDS + 1] = {};
		hipMalloc(&sc.grp, sizeof(zeros));
		hipMemcpy(sc.grp, zeros, sizeof(zeros), hipMemcpyHostToDevice);
	}
}

void radixSort(uint32_t* keys, uint32_t* vals, size_t n, int bits, SortScratch& sc,
               uint32_t** outKeys, uint32_t** outVals, hipStream_t s, const uint32_t* nDev, bool index)
{
	*outKeys = keys;
	*outVals = vals;
	if (n <= 1 || bits <= 0)
	{
		if (index)
			iota(vals, n, s);
		return;
	}
	const uint32_t chunk = rsChunk(n);
	const uint32_t nBlocks = (uint32_t) ((n + chunk - 1) / chunk);
	radixSortReserve(sc, n);
	const size_t histN = (size_t) 256 * nBlocks;
	uint32_t* kIn = keys;
	uint32_t* vIn = vals;
	uint32_t* kOut = sc.keys;
	uint32_t* vOut = sc.vals;
	const bool fused = nBlocks <= RS_FUSED_MAX_BLOCKS && chunk == (uint32_t) RS_CHUNK;
	for (int shift = 0; shift < bits; shift += 8)
	{
		const uint32_t* from = index && shift == 0 ? nullptr : vIn;
		if (fused)
		{
			hipLaunchKernelGGL(k_radix_hist, dim3(nBlocks), dim3(RS_THREADS), 0, s, kIn, n, nDev, (uint32_t) shift,
			                   sc.hist, 1u, 256u, chunk, sc.grp);
			hipLaunchKernelGGL(k_radix_scatter<true>, dim3(nBlocks), dim3(RS_THREADS), 0, s, kIn, from, kOut, vOut, n,
			                   nDev, (uint32_t) shift, sc.hist, nBlocks, chunk, sc.grp);
		}
		else
		{
			hipLaunchKernelGGL(k_radix_hist, dim3(nBlocks), dim3(RS_THREADS), 0, s, kIn, n, nDev, (uint32_t) shift,
			                   sc.hist, nBlocks, 1u, chunk, (uint32_t*) nullptr);
			scanExclusiveMulti(sc.hist, histN, 1, histN, sc.hist + histN, sc.scan, s);
			if (chunk == (uint32_t) RS_CHUNK)
				hipLaunchKernelGGL(k_radix_scatter<false>, dim3(nBlocks), dim3(RS_THREADS), 0, s, kIn, from, kOut, vOut,
				                   n, nDev, (uint32_t) shift, sc.hist, nBlocks, chunk, (uint32_t*) nullptr);
			else
				hipLaunchKernelGGL(k_radix_scatter_long, dim3(nBlocks), dim3(RS_THREADS), 0, s, kIn, from, kOut, vOut, n,
				                   nDev, (uint32_t) shift, sc.hist, nBlocks, chunk);
		}
		uint32_t* tk = kIn; kIn = kOut; kOut = tk;
		uint32_t* tv = vIn; vIn = vOut; vOut = tv;
	}
	*outKeys = kIn;
	*outVals = vIn;
}

/* Stable sort by tile of up to TS_MAX_ITEMS items by one block, and the
 * tiles' ranges: sorted[i] = the value of the item at place i, start/end of
 * every tile that received one.  Inside, an item is one word, tile << 16 | index, so
 * its radix passes (8 bits each) stay in LDS.  A wave ranks consecutive
 * items, 64 at a time, in order; a digit's places are ordered by wave, then
 * within the wave.
 *
 * A small draw's sort was five launches of 4-5 us each whatever they sorted
 * (two histograms, two scatters, the ranges): 21.5 us for the pairs of a
 * 576-triangle object at 1280x720, 8.5 us in this one.  TS_MAX_ITEMS is what
 * the items and places of a thread keep in registers (16 rounds) with the
 * items in 64 KB of LDS; above it the passes spread over the chip. */
constexpr int TS_THREADS = 1024;
constexpr int TS_WAVES = TS_THREADS / 64;
constexpr int TS_ROUNDS = (int) (TS_MAX_ITEMS / TS_THREADS);

__global__ __launch_bounds__(TS_THREADS) void k_tile_sort(const uint32_t* __restrict__ keys,
                                                          const uint32_t* __restrict__ vals, uint32_t cap,
                                                          const uint32_t* __restrict__ nDev, int bits,
                                                          uint32_t* __restrict__ sorted, uint32_t* __restrict__ start,
                                                          uint32_t* __restrict__ end)
{
	__shared__ uint32_t item[TS_MAX_ITEMS];
	__shared__ uint32_t cnt[TS_WAVES][256];
	__shared__ uint32_t digitSum[4];
	const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
	const uint32_t n = *nDev < cap ? *nDev : cap;
	const uint64_t below = (1ull << lane) - 1ull;
	/* a wave's share: whole rounds of 64 */
	const uint32_t rounds = (n + TS_THREADS - 1u) / TS_THREADS;
	const uint32_t first = wave * rounds * 64u + lane;
	uint32_t it[TS_ROUNDS], place[TS_ROUNDS];
#pragma unroll
	for (int k = 0; k < TS_ROUNDS; k++)
	{
		const uint32_t i = first + 64u * (uint32_t) k;
		it[k] = ((uint32_t) k < rounds && i < n) ? (keys[i] << 16 | i) : 0u;
	}
	for (int shift = 16; shift < 16 + bits; shift += 8)
	{
		for (int d = (int) lane; d < 256; d += 64)
			cnt[wave][d] = 0u;
		__syncthreads();
#pragma unroll
		for (int k = 0; k < TS_ROUNDS; k++)
			if ((uint32_t) k < rounds)
			{
				const bool valid = first + 64u * (uint32_t) k < n;
				const uint32_t d = (it[k] >> shift) & 255u;
				uint64_t peers = __ballot(valid);
#pragma unroll
				for (int b = 0; b < 8; b++)
				{
					const bool bit = (d >> b) & 1u;
					const uint64_t m = __ballot(bit);
					peers &= bit ? m : ~m;
				}
				const uint32_t rank = (uint32_t) __popcll(peers & below);
				const uint32_t before = cnt[wave][d];
				place[k] = before + rank;
				__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
				if (valid && rank == 0)
					cnt[wave][d] = before + (uint32_t) __popcll(peers);
				__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
			}
		__syncthreads();
		/* digit t: its places start after every smaller digit's, wave by wave */
		if (t < 256u)
		{
			uint32_t sum = 0;
#pragma unroll
			for (int w = 0; w < TS_WAVES; w++)
			{
				const uint32_t c = cnt[w][t];
				cnt[w][t] = sum;
				sum += c;
			}
			uint32_t incl = sum;
#pragma unroll
			for (uint32_t off = 1; off < 64; off <<= 1)
			{
				const uint32_t v = __shfl_up(incl, off);
				if (lane >= off) incl += v;
			}
			if (lane == 63u)
				digitSum[wave] = incl;
			const uint32_t ex = incl - sum;
#pragma unroll
			for (int w = 0; w < TS_WAVES; w++)
				cnt[w][t] += ex;
		}
		__syncthreads();
#pragma unroll
		for (int k = 0; k < TS_ROUNDS; k++)
			if ((uint32_t) k < rounds && first + 64u * (uint32_t) k < n)
			{
				const uint32_t d = (it[k] >> shift) & 255u;
				uint32_t at = cnt[wave][d] + place[k];
				for (uint32_t q = 0; q < (d >> 6); q++)
					at += digitSum[q];
				item[at] = it[k];
			}
		__syncthreads();
#pragma unroll
		for (int k = 0; k < TS_ROUNDS; k++)
		{
			const uint32_t i = first + 64u * (uint32_t) k;
			if ((uint32_t) k < rounds && i < n)
				it[k] = item[i];
		}
	}
	if (bits <= 0)
	{
#pragma unroll
		for (int k = 0; k < TS_ROUNDS; k++)
		{
			const uint32_t i = first + 64u * (uint32_t) k;
			if ((uint32_t) k < rounds && i < n)
				item[i] = it[k];
		}
		__syncthreads();
	}
#pragma unroll
	for (int k = 0; k < TS_ROUNDS; k++)
	{
		const uint32_t i = first + 64u * (uint32_t) k;
		if ((uint32_t) k < rounds && i < n)
		{
			const uint32_t tile = it[k] >> 16;
			sorted[i] = vals[it[k] & 0xFFFFu];
			if (i == 0 || item[i - 1] >> 16 != tile) start[tile] = i;
			if (i + 1 == n || item[i + 1] >> 16 != tile) end[tile] = i + 1;
		}
	}
}

void tileSort(const uint32_t* keys, const uint32_t* vals, size_t cap, int bits, uint32_t* sorted, uint32_t* start,
              uint32_t* end, hipStream_t s, const uint32_t* nDev)
{
	if (cap)
		hipLaunchKernelGGL(k_tile_sort, dim3(1), dim3(TS_THREADS), 0, s, keys, vals, (uint32_t) cap, nDev, bits, sorted,
		                   start, end);
}

/* ------------------------------------------------------------------ fills */

__global__ void k_fill_u32(uint32_t* p, uint32_t v, size_t n)
{
	const size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
	const size_t stride = (size_t) gridDim.x * blockDim.x;
	for (size_t k = i; k < n; k += stride) p[k] = v;
}

__global__ void k_fill_u8(uint8_t* p, uint8_t v, size_t n)
{
	const size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
	const size_t stride = (size_t) gridDim.x * blockDim.x;
	for (size_t k = i; k < n; k += stride) p[k] = v;
}

__global__ void k_iota(uint32_t* p, size_t n)
{
	const size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
	const size_t stride = (size_t) gridDim.x * blockDim.x;
	for (size_t k = i; k < n; k += stride) p[k] = (uint32_t) k;
}

static dim3 fillGrid(size_t n)
{
	size_t b = (n + 255) / 256;
	if (b > 4096) b = 4096;
	if (b == 0) b = 1;
	return dim3((uint32_t) b);
}

void fillU32(uint32_t* p, uint32_t v, size_t n, hipStream_t s)
{
	if (n) hipLaunchKernelGGL(k_fill_u32, fillGrid(n), dim3(256), 0, s, p, v, n);
}

void fillU8(uint8_t* p, uint8_t v, size_t n, hipStream_t s)
{
	if (n) hipLaunchKernelGGL(k_fill_u8, fillGrid(n), dim3(256), 0, s, p, v, n);
}

/* Colour, depth and stencil fills of one framebuffer in one launch (a null
 * array is left alone). */
__global__ void k_fill_fb(uint32_t* color, uint32_t cv, uint32_t* depth, uint32_t dv, uint8_t* stencil, uint8_t sv, size_t n)
{
	const size_t i0 = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
	const size_t stride = (size_t) gridDim.x * blockDim.x;
	for (size_t i = i0; i < n; i += stride)
	{
		if (color) color[i] = cv;
		if (depth) depth[i] = dv;
	}
	/* stencil bytes four at a time, then the tail */
	const size_t n4 = n / 4;
	const uint32_t sv4 = (uint32_t) sv * 0x01010101u;
	if (stencil)
	{
		uint32_t* s4 = reinterpret_cast<uint32_t*>(stencil);
		for (size_t i = i0; i < n4; i += stride) s4[i] = sv4;
		for (size_t i = n4 * 4 + i0; i < n; i += stride) stencil[i] = sv;
	}
}

void fillFramebuffer(uint32_t* color, uint32_t cv, uint32_t* depth, uint32_t dv, uint8_t* stencil, uint8_t sv, size_t n,
                     hipStream_t s)
{
	if (n) hipLaunchKernelGGL(k_fill_fb, fillGrid(n), dim3(256), 0, s, color, cv, depth, dv, stencil, sv, n);
}

/* Up to three arrays copied in one launch, between device memory and pinned
 * host memory (the host's lines pass over the link as the lanes read or
 * write them, sixteen bytes each).  A thread has COPY_AHEAD of them in
 * flight: the link's latency is some 2 us.  The link bounds it: 18.7 MB of a
 * 1920x1080 framebuffer in 341 us (54.7 GB/s, what one large copy reaches).
 * Three copy calls in its place cost a launch each and, where the runtime
 * gives a copy to a DMA engine, a wait between queues: a synchronous draw of
 * 256x256 pixels took 162 us with them, 120 with one launch each way. */
constexpr int COPY_AHEAD = 4;

__global__ __launch_bounds__(256) void k_copy_arrays(CopyArrays c)
{
	const uint64_t u0 = c.bytes[0] / 16, u1 = u0 + c.bytes[1] / 16, u2 = u1 + c.bytes[2] / 16;
	const uint64_t stride = (uint64_t) gridDim.x * 256u;
	for (uint64_t u = (uint64_t) blockIdx.x * 256u + threadIdx.x; u < u2; u += stride * COPY_AHEAD)
	{
		uint4 v[COPY_AHEAD];
		uint4* to[COPY_AHEAD];
#pragma unroll
		for (int k = 0; k < COPY_AHEAD; k++)
		{
			const uint64_t at = u + stride * (uint64_t) k;
			const int a = at < u0 ? 0 : (at < u1 ? 1 : 2);
			const uint64_t i = at - (a == 0 ? 0u : (a == 1 ? u0 : u1));
			const void* src = a == 0 ? c.src[0] : (a == 1 ? c.src[1] : c.src[2]);
			void* dst = a == 0 ? c.dst[0] : (a == 1 ? c.dst[1] : c.dst[2]);
			to[k] = srpGlobal(static_cast<uint4*>(dst)) + i;
			if (at < u2)
				v[k] = srpGlobal(static_cast<const uint4*>(src))[i];
		}
#pragma unroll
		for (int k = 0; k < COPY_AHEAD; k++)
			if (u + stride * (uint64_t) k < u2)
				*to[k] = v[k];
	}
	/* the last bytes of each array */
	if (blockIdx.x == 0 && threadIdx.x < 16u)
	{
#pragma unroll
		for (int a = 0; a < 3; a++)
		{
			const uint64_t n = c.bytes[a], at = n - n % 16u + threadIdx.x;
			if (at < n)
				static_cast<uint8_t*>(c.dst[a])[at] = static_cast<const uint8_t*>(c.src[a])[at];
		}
	}
}

void copyArrays(const CopyArrays& c, hipStream_t s)
{
	const uint64_t units = c.bytes[0] / 16 + c.bytes[1] / 16 + c.bytes[2] / 16;
	if (c.bytes[0] + c.bytes[1] + c.bytes[2] == 0)
		return;
	const uint64_t b = (units + 256 * COPY_AHEAD - 1) / (256 * COPY_AHEAD);
	hipLaunchKernelGGL(k_copy_arrays, dim3((uint32_t) (b < 1 ? 1 : (b > 1024 ? 1024 : b))), dim3(256), 0, s, c);
}

/* A small block of words written to the device from the launch's own
 * arguments (uploadSmall). */
struct SmallBlock
{
	uint4 w[UPLOAD_SMALL_BYTES / 16];
};

__global__ __launch_bounds__(UPLOAD_SMALL_BYTES / 16) void k_upload(SmallBlock b, uint4* dst, uint32_t quads)
{
	if (threadIdx.x < quads)
		srpGlobal(dst)[threadIdx.x] = b.w[threadIdx.x];
}

void uploadSmall(void* dst, const void* src, size_t bytes, hipStream_t s)
{
	SmallBlock b;
	memcpy(b.w, src, bytes);
	hipLaunchKernelGGL(k_upload, dim3(1), dim3(UPLOAD_SMALL_BYTES / 16), 0, s, b, static_cast<uint4*>(dst),
	                   (uint32_t) ((bytes + 15) / 16));
}

/* Block b fills framebuffer d, the last descriptor with firstBlock <= b,
 * with the blocks from its firstBlock to the next one's. */
__global__ void k_fill_many(const FillDesc* desc, uint32_t nDesc, uint32_t blocks)
{
	uint32_t a = 0, z = nDesc;
	while (z - a > 1)
	{
		const uint32_t m = (a + z) >> 1;
		if (desc[m].firstBlock <= blockIdx.x) a = m;
		else z = m;
	}
	const FillDesc D = desc[a];
	const uint32_t nb = ((a + 1 < nDesc) ? desc[a + 1].firstBlock : blocks) - D.firstBlock;
	const size_t i0 = (size_t) (blockIdx.x - D.firstBlock) * blockDim.x + threadIdx.x;
	const size_t stride = (size_t) nb * blockDim.x;
	for (size_t i = i0; i < D.n; i += stride)
	{
		if (D.color) D.color[i] = D.colorValue;
		if (D.depth) D.depth[i] = D.depthValue;
		if (D.stencil) D.stencil[i] = (uint8_t) D.stencilValue;
	}
}

uint32_t fillBlocksFor(size_t n)
{
	const size_t b = (n + 1023) / 1024;
	return (uint32_t) (b < 1 ? 1 : (b > 1024 ? 1024 : b));
}

void fillFramebuffers(const FillDesc* desc, uint32_t nDesc, uint32_t blocks, hipStream_t s)
{
	if (nDesc && blocks)
		hipLaunchKernelGGL(k_fill_many, dim3(blocks), dim3(256), 0, s, desc, nDesc, blocks);
}

void iota(uint32_t* p, size_t n, hipStream_t s)
{
	if (n) hipLaunchKernelGGL(k_iota, fillGrid(n), dim3(256), 0, s, p, n);
}

__global__ void k_publish(const uint32_t* totals, uint32_t* hostCopy, uint32_t seq)
{
	publish(totals, hostCopy, seq);
}

void launchPublish(const uint32_t* totals, uint32_t* hostCopy, uint32_t seq, hipStream_t s)
{
	hipLaunchKernelGGL(k_publish, dim3(1), dim3(1), 0, s, totals, hostCopy, seq);
}


}  // namespace lib
}  // namespace srp
