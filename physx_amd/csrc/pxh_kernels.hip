// HIP kernels of the rigid-body step for gfx950 (wave64). One lane per body,
// pair or constraint; all arrays are structure-of-arrays in HBM so a wave's
// loads are coalesced float4 rows.
//
// Stage map (reference stage -> kernels here):
//   shape bounds (updateTransformCacheAndBoundArrayLaunch)  k_bounds
//   broadphase (gpubroadphase/src/CUDA/broadphase.cu)        k_scene_grid, k_keys, radix sort, k_row_start,
//                                                            k_gather_sorted, k_sweep<count|write>
//   narrowphase (cudaSphere.cu, cudaBox.cu, cudaGJKEPA.cu)  k_np_pairs, k_np_planes
//   partitioning (PxgIncrementalPartition, host in ref)     k_con_build, k_color_min, k_color_pick, colour sort
//   pre-integration (preIntegrationTGS.cu)                  k_preintegrate
//   contact prep (constraintBlockPrepTGS.cu)                k_prep
//   solve (solverMultiBlockTGS.cu solveBlockUnified)        k_solve
//   integration (integrationTGS.cu)                         k_integrate, k_finalize
#include "pxh_kernels.h"
#include "pxh_launch.h"
#include <hip/hip_ext.h>
#include "pxh_np.h"
#include "pxh_convex.h"
#include "pxh_joint.h"
#include "pxh_mesh.h"

#include <algorithm>
#include <type_traits>

namespace pxh {

// ---------------------------------------------------------------------------
// wave / block scans
// ---------------------------------------------------------------------------
PXH_D uint32_t waveInclScan(uint32_t v)
{
	const int lane = threadIdx.x & 63;
#pragma unroll
	for (int o = 1; o < 64; o <<= 1)
	{
		const uint32_t t = __shfl_up(v, o, 64);
		if (lane >= o)
			v += t;
	}
	return v;
}

// exclusive scan over the block (blockDim.x <= 1024, multiple of 64); returns
// the exclusive prefix, writes the block total
PXH_D uint32_t blockExclScan(uint32_t v, uint32_t* sh, uint32_t& total)
{
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
	const uint32_t inc = waveInclScan(v);
	if (lane == 63)
		sh[wave] = inc;
	__syncthreads();
	if (threadIdx.x < 64)
	{
		const uint32_t w = threadIdx.x < nw ? sh[threadIdx.x] : 0u;
		const uint32_t wi = waveInclScan(w);
		if (threadIdx.x < nw)
			sh[threadIdx.x] = wi - w;
		if (threadIdx.x == nw - 1)
			sh[32] = wi;
	}
	__syncthreads();
	const uint32_t r = sh[wave] + inc - v;
	total = sh[32];
	__syncthreads();
	return r;
}

// Exclusive scan in two launches: the sums of 4,096-element tiles, then every
// tile adds up the sums before it and scans its own elements; an array of one
// tile needs the second launch alone. Bound by launches and their latency at
// the step's sizes: 11 us on average at 262k bodies, where three launches and a
// second pass over the data took 13. Adding up grows with the square of the
// tiles, so past SUMS_DIRECT of them the sums are scanned first (adding up and
// scanning: 4,096 tiles 42 / 44 us, 8,192 tiles 90 / 71, 32,768 tiles 715 / 378; the
// constraint list's 1,024-slot tiles: 4,096 25 / 26 us, 8,192 49 / 41, 65,536 940 / 324).
constexpr int SUMS_DIRECT = 4096;
constexpr int SCAN_THREADS = 256, SCAN_ITEMS = 16, SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

// sum over the block; every thread gets it (sh: 8 entries)
PXH_D uint32_t blockSum(uint32_t v, uint32_t* sh)
{
#pragma unroll
	for (int o = 32; o > 0; o >>= 1)
		v += __shfl_xor(v, o, 64);
	if ((threadIdx.x & 63) == 0)
		sh[threadIdx.x >> 6] = v;
	__syncthreads();
	uint32_t t = 0;
	for (int w = 0; w < int(blockDim.x >> 6); w++)
		t += sh[w];
	__syncthreads();
	return t;
}

__global__ void __launch_bounds__(SCAN_THREADS) k_scan_sums(const uint32_t* data, int64_t n, uint32_t* sums)
{
	__shared__ uint32_t sh[8];
	const int64_t base = int64_t(blockIdx.x) * SCAN_TILE;
	uint32_t v = 0;
#pragma unroll
	for (int k = 0; k < SCAN_ITEMS; k++)
	{
		const int64_t g = base + k * SCAN_THREADS + threadIdx.x;
		v += g < n ? data[g] : 0u;
	}
	v = blockSum(v, sh);
	if (threadIdx.x == 0)
		sums[blockIdx.x] = v;
}

// what the tiles before this one hold: the tile's entry of scanned sums, or their
// sum, added up here (sh: 8 entries; its barriers also publish LDS)
template <bool SCANNED> PXH_D uint32_t tilesBefore(const uint32_t* sums, uint32_t* sh)
{
	if constexpr (SCANNED)
	{
		__syncthreads();
		return sums[blockIdx.x];
	}
	else
	{
		uint32_t before = 0;
		for (int t = threadIdx.x; t < int(blockIdx.x); t += int(blockDim.x))
			before += sums[t];
		return blockSum(before, sh);
	}
}

// in-place exclusive scan of each tile, offset by the sums of the tiles before it
template <bool SCANNED>
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_tiles(uint32_t* data, int64_t n, const uint32_t* sums)
{
	__shared__ uint32_t sh[33];
	__shared__ uint32_t tile[SCAN_TILE + SCAN_TILE / 32];   // a word of padding every 32: no bank conflicts
	auto at = [](int i) { return i + (i >> 5); };
	const int64_t base = int64_t(blockIdx.x) * SCAN_TILE;
#pragma unroll
	for (int k = 0; k < SCAN_ITEMS; k++)
	{
		const int i = k * SCAN_THREADS + threadIdx.x;
		tile[at(i)] = base + i < n ? data[base + i] : 0u;
	}
	const uint32_t before = tilesBefore<SCANNED>(sums, sh);
	uint32_t loc[SCAN_ITEMS];
	uint32_t sum = 0;
#pragma unroll
	for (int k = 0; k < SCAN_ITEMS; k++)
	{
		loc[k] = tile[at(threadIdx.x * SCAN_ITEMS + k)];
		sum += loc[k];
	}
	uint32_t total;
	uint32_t pre = before + blockExclScan(sum, sh, total);
#pragma unroll
	for (int k = 0; k < SCAN_ITEMS; k++)
	{
		tile[at(threadIdx.x * SCAN_ITEMS + k)] = pre;
		pre += loc[k];
	}
	__syncthreads();
#pragma unroll
	for (int k = 0; k < SCAN_ITEMS; k++)
	{
		const int i = k * SCAN_THREADS + threadIdx.x;
		if (base + i < n)
			data[base + i] = tile[at(i)];
	}
}

// ---------------------------------------------------------------------------
// LSD radix sort of (u64 key, u32 value), 8-bit digits, stable
// ---------------------------------------------------------------------------
// A key is two fields, the low lowBits bits of its low word below its high
// word; the digits run over the two fields joined, so the unused bits between
// them cost no pass.
//
// Up to RS_SMALL keys: one launch, one workgroup keeps the keys in registers
// through every pass. Up to RS_DIRECT tiles of 4,096: two launches a pass, the
// digit counts of the tiles and the scatter, in which each tile adds up the counts
// of all tiles itself, so no scan runs between. Past that, since the adding up
// grows with the square of the tiles, the counts are laid out digit by digit and
// scanned between the two.
// A key's rank in its wave comes from eight ballots (the lanes with its digit).
// Bound by launches and latency. 262,144 broadphase keys (51 bits, seven passes):
// 92 us back to back, where a count, a scan of three launches and a bit-by-bit split
// a pass took 219 in the step. One workgroup against tiles: 4,096 keys 34 / 67 us,
// 8,192 keys 59 / 76 (of 16 bits 19 / 22). Adding up against scanning: 256 tiles
// 128 / 155 us, 512 tiles 225 / 198, 4,096 tiles 5.3 / 1.1 ms.
constexpr int RS_THREADS = 1024, RS_ITEMS = 4, RS_TILE = RS_THREADS * RS_ITEMS;
constexpr int RS_SMALL_THREADS = 1024, RS_SMALL_ITEMS = 8, RS_SMALL = RS_SMALL_THREADS * RS_SMALL_ITEMS;
constexpr int RS_DIRECT = 384;
int radix_tile() { return RS_TILE; }

PXH_D uint32_t rsDigit(uint64_t key, int lowBits, int shift)
{
	const uint64_t low = lowBits >= 32 ? (key & 0xFFFFFFFFull) : (key & ((1ull << lowBits) - 1ull));
	return uint32_t((((key >> 32) << lowBits) | low) >> shift) & 0xFFu;
}

// the lanes of the wave that are valid and hold digit d
PXH_D uint64_t rsPeers(uint32_t d, bool valid)
{
	uint64_t m = __ballot(valid);
#pragma unroll
	for (int b = 0; b < 8; b++)
	{
		const bool one = d >> b & 1u;
		const uint64_t v = __ballot(one);
		m &= one ? v : ~v;
	}
	return m;
}

// where the counts of digit d of tile b lie: tile by tile, or digit by digit for a scan
template <bool SCANNED> PXH_D int64_t rsCount(int d, int b, int nblocks)
{
	return SCANNED ? int64_t(d) * nblocks + b : int64_t(b) * 256 + d;
}

template <bool SCANNED>
__global__ void __launch_bounds__(RS_THREADS) k_rs_hist(const uint64_t* keys, int n, int lowBits, int shift,
                                                        uint32_t* hist, int nblocks)
{
	__shared__ uint32_t cnt[256];
	if (threadIdx.x < 256)
		cnt[threadIdx.x] = 0;
	__syncthreads();
	const int base = blockIdx.x * RS_TILE;
#pragma unroll
	for (int k = 0; k < RS_ITEMS; k++)
	{
		const int g = base + k * RS_THREADS + threadIdx.x;
		if (g < n)
			atomicAdd(&cnt[rsDigit(keys[g], lowBits, shift)], 1u);
	}
	__syncthreads();
	if (threadIdx.x < 256)
		hist[rsCount<SCANNED>(threadIdx.x, blockIdx.x, nblocks)] = cnt[threadIdx.x];
}

template <bool SCANNED>
__global__ void __launch_bounds__(RS_THREADS) k_rs_scatter(const uint64_t* kin, const uint32_t* vin, uint64_t* kout,
                                                           uint32_t* vout, int n, int lowBits, int shift,
                                                           const uint32_t* hist, int nblocks)
{
	constexpr int WAVES = RS_THREADS / 64, PARTS = RS_THREADS / 256;
	__shared__ uint32_t cnt[WAVES][256];
	__shared__ uint32_t part[PARTS][2][256];
	__shared__ uint32_t start[256], shift0[256];
	__shared__ uint32_t sh[33];
	__shared__ uint64_t xk[RS_TILE];
	__shared__ uint32_t xv[RS_TILE];
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	// item k of the wave: 64 keys in order, the wave's items one after the other
	const int base = blockIdx.x * RS_TILE + w * (64 * RS_ITEMS) + lane;
	uint64_t key[RS_ITEMS];
	uint32_t val[RS_ITEMS];
#pragma unroll
	for (int k = 0; k < RS_ITEMS; k++)
	{
		const int g = base + 64 * k;
		key[k] = g < n ? kin[g] : 0ull;
		val[k] = g < n ? vin[g] : 0u;
	}
	for (int i = lane; i < 256; i += 64)
		cnt[w][i] = 0u;
	// this digit's count over all tiles and over the tiles before this one,
	// every PARTS-th tile to each part of the block
	if constexpr (!SCANNED)
	{
		const int d = threadIdx.x & 255, p = threadIdx.x >> 8;
		uint32_t all = 0, before = 0;
#pragma unroll 8
		for (int b = p; b < nblocks; b += PARTS)
		{
			const uint32_t c = hist[rsCount<false>(d, b, nblocks)];
			all += c;
			before += b < int(blockIdx.x) ? c : 0u;
		}
		part[p][0][d] = all;
		part[p][1][d] = before;
	}
	// ranks among the wave's earlier keys of the same digit; a wave's LDS
	// accesses keep their order, and only it uses its counters here
	uint32_t rank[RS_ITEMS];
	volatile uint32_t* mine = cnt[w];
#pragma unroll
	for (int k = 0; k < RS_ITEMS; k++)
	{
		const uint32_t d = rsDigit(key[k], lowBits, shift);
		const bool valid = base + 64 * k < n;
		const uint64_t m = rsPeers(d, valid);
		const uint32_t lower = uint32_t(__popcll(m & ((1ull << lane) - 1ull)));
		const uint32_t had = mine[d];
		rank[k] = had + lower;
		if (valid && lower == 0)
			mine[d] = had + uint32_t(__popcll(m));
	}
	__syncthreads();
	// the digit's first place in the output and in this tile's sorted order
	{
		const int d = threadIdx.x & 255;
		uint32_t own = 0, total = 0, before = 0;
		if (threadIdx.x < 256)
		{
#pragma unroll
			for (int i = 0; i < WAVES; i++)
			{
				const uint32_t c = cnt[i][d];
				cnt[i][d] = own;
				own += c;
			}
			if constexpr (SCANNED)
				before = hist[rsCount<true>(d, blockIdx.x, nblocks)];
			else
			{
#pragma unroll
				for (int p = 0; p < PARTS; p++)
				{
					total += part[p][0][d];
					before += part[p][1][d];
				}
			}
		}
		uint32_t sum;
		const uint32_t local = blockExclScan(own, sh, sum);
		const uint32_t pre = SCANNED ? 0u : blockExclScan(total, sh, sum);
		if (threadIdx.x < 256)
		{
			start[d] = local;
			shift0[d] = pre + before - local;
		}
	}
	__syncthreads();
	// through LDS in sorted order, so the keys of a digit leave side by side
#pragma unroll
	for (int k = 0; k < RS_ITEMS; k++)
		if (base + 64 * k < n)
		{
			const uint32_t d = rsDigit(key[k], lowBits, shift);
			const uint32_t at = start[d] + cnt[w][d] + rank[k];
			xk[at] = key[k];
			xv[at] = val[k];
		}
	__syncthreads();
	const int live = min(RS_TILE, n - int(blockIdx.x) * RS_TILE);
#pragma unroll
	for (int k = 0; k < RS_ITEMS; k++)
	{
		const int at = k * RS_THREADS + threadIdx.x;
		if (at < live)
		{
			const uint64_t x = xk[at];
			const uint32_t dst = shift0[rsDigit(x, lowBits, shift)] + uint32_t(at);
			kout[dst] = x;
			vout[dst] = xv[at];
		}
	}
}

// every pass of up to 1,024 * ITEMS keys in one workgroup
template <int ITEMS>
__global__ void __launch_bounds__(RS_SMALL_THREADS) k_rs_small(uint64_t* keys, uint32_t* vals, int n, int lowBits,
                                                               int bits)
{
	constexpr int WAVES = RS_SMALL_THREADS / 64;
	__shared__ uint32_t cnt[WAVES][256];
	__shared__ uint32_t start[256];
	__shared__ uint32_t sh[33];
	__shared__ uint64_t xk[RS_SMALL_THREADS * ITEMS];
	__shared__ uint32_t xv[RS_SMALL_THREADS * ITEMS];
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	const int base = w * (64 * ITEMS) + lane;
	uint64_t key[ITEMS];
	uint32_t val[ITEMS];
#pragma unroll
	for (int k = 0; k < ITEMS; k++)
	{
		const int g = base + 64 * k;
		key[k] = g < n ? keys[g] : 0ull;
		val[k] = g < n ? vals[g] : 0u;
	}
	for (int shift = 0; shift < bits; shift += 8)
	{
		for (int i = lane; i < 256; i += 64)
			cnt[w][i] = 0u;
		uint32_t rank[ITEMS];
		volatile uint32_t* mine = cnt[w];
#pragma unroll
		for (int k = 0; k < ITEMS; k++)
		{
			const uint32_t d = rsDigit(key[k], lowBits, shift);
			const bool valid = base + 64 * k < n;
			const uint64_t m = rsPeers(d, valid);
			const uint32_t lower = uint32_t(__popcll(m & ((1ull << lane) - 1ull)));
			const uint32_t had = mine[d];
			rank[k] = had + lower;
			if (valid && lower == 0)
				mine[d] = had + uint32_t(__popcll(m));
		}
		__syncthreads();
		uint32_t total = 0;
		if (threadIdx.x < 256)
		{
#pragma unroll
			for (int i = 0; i < WAVES; i++)
			{
				const uint32_t c = cnt[i][threadIdx.x];
				cnt[i][threadIdx.x] = total;
				total += c;
			}
		}
		uint32_t sum;
		const uint32_t pre = blockExclScan(total, sh, sum);
		if (threadIdx.x < 256)
			start[threadIdx.x] = pre;
		__syncthreads();
#pragma unroll
		for (int k = 0; k < ITEMS; k++)
			if (base + 64 * k < n)
			{
				const uint32_t d = rsDigit(key[k], lowBits, shift);
				const uint32_t at = start[d] + cnt[w][d] + rank[k];
				xk[at] = key[k];
				xv[at] = val[k];
			}
		__syncthreads();
#pragma unroll
		for (int k = 0; k < ITEMS; k++)
			if (base + 64 * k < n)
			{
				key[k] = xk[base + 64 * k];
				val[k] = xv[base + 64 * k];
			}
	}
#pragma unroll
	for (int k = 0; k < ITEMS; k++)
		if (base + 64 * k < n)
		{
			keys[base + 64 * k] = key[k];
			vals[base + 64 * k] = val[k];
		}
}

// ---------------------------------------------------------------------------
// bounds and broadphase
// ---------------------------------------------------------------------------

// a body's shape bounds, centre - w to centre + w (Gu::computeBounds,
// geomutils/src/GuBounds.cpp:354-395)
PXH_D void shapeBounds(int i, const float4* pos, const float4* rot, const float4* geom, const HullSet& hs, f3& mn,
                       f3& mx)
{
	const float4 g = geom[i];
	f3 p = mk(pos[i]);
	f3 w;
	if (int(g.w) == GEOM_SPHERE)
		w = mk(g.x, g.x, g.x);
	else if (int(g.w) == GEOM_CAPSULE)
	{
		// computeCapsuleBounds (geomutils/include/GuBounds.h:54-62)
		const m33 R = qmat(mkq(rot[i]));
		w = mk(fabsf(R.c0.x) * g.y + g.x, fabsf(R.c0.y) * g.y + g.x, fabsf(R.c0.z) * g.y + g.x);
	}
	else
	{
		const m33 R = qmat(mkq(rot[i]));
		f3 e = mk(g.x, g.y, g.z);
		if (int(g.w) == GEOM_CONVEXMESH)
		{
			// hull bounds: the local box rotated about the pose
			// (geomutils/src/GuBounds.cpp:136-140 transformNoEmptyTest)
			const int h = int(g.x);
			e = mk(hs.be[h]);
			p = mmul(R, mk(hs.bc[h])) + p;
		}
		const f3 c0 = R.c0 * e.x, c1 = R.c1 * e.y, c2 = R.c2 * e.z;
		w = mk(fabsf(c0.x) + fabsf(c1.x) + fabsf(c2.x), fabsf(c0.y) + fabsf(c1.y) + fabsf(c2.y),
		       fabsf(c0.z) + fabsf(c1.z) + fabsf(c2.z));
	}
	mn = p - w;
	mx = p + w;
}

// shape bounds plus the broadphase's contact-distance inflation
// (lowlevelaabb/src/BpBroadPhaseABP.cpp:1187-1192)
// The step's first launch over the bodies also clears what its colouring keeps
// per body and its few device words.
__global__ void k_bounds(int n, const float4* pos, const float4* rot, const float4* geom, HullSet hs, float co,
                         float4* bmin, float4* bmax, ColorState cs)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < STEP_WORDS)
		cs.words[i] = 0u;
	if (i >= n)
		return;
	cs.mask[i] = 0ull;
	cs.need[i] = 0u;
	cs.next[i] = 0u;
	f3 mn, mx;
	shapeBounds(i, pos, rot, geom, hs, mn, mx);
	bmin[i] = make_float4(mn.x - co, mn.y - co, mn.z - co, geom[i].w);
	bmax[i] = make_float4(mx.x + co, mx.y + co, mx.z + co, 0.0f);
}

// Per-world row grid for the sweep: rows are (y,z) cells no smaller than the
// widest inflated box, so overlapping boxes sit in the same or adjacent rows.
// Pass 1 reduces each world's centre range and widest box with order-
// preserving integer atomics (one per wave when the wave holds one world).
PXH_D float decode_float(uint32_t u) { return __uint_as_float((u & 0x80000000u) ? (u ^ 0x80000000u) : ~u); }

// Bodies are read side by side, sixteen to a lane; a block of one world reduces
// in LDS and makes one set of atomics, a wave over several worlds one set for
// each of them. Bound by the atomics on one world's five words: 262,144 bodies
// take 12 us in 64 blocks, 19 us in 256.
constexpr int GRID_ITEMS = 16;

struct GridRange
{
	uint32_t v[5];   // lowest / highest centre y, lowest / highest centre z, widest box
};
PXH_D void gridMerge(GridRange& a, const GridRange& b)
{
	a.v[0] = min(a.v[0], b.v[0]); a.v[1] = max(a.v[1], b.v[1]);
	a.v[2] = min(a.v[2], b.v[2]); a.v[3] = max(a.v[3], b.v[3]);
	a.v[4] = max(a.v[4], b.v[4]);
}
// every lane gets the wave's range
PXH_D GridRange gridWave(GridRange a)
{
#pragma unroll
	for (int o = 1; o < 64; o <<= 1)
	{
		GridRange b;
#pragma unroll
		for (int k = 0; k < 5; k++)
			b.v[k] = __shfl_xor(a.v[k], o, 64);
		gridMerge(a, b);
	}
	return a;
}
PXH_D void gridAtomic(uint32_t* w, const GridRange& a)
{
	atomicMin(&w[0], a.v[0]); atomicMax(&w[1], a.v[1]); atomicMin(&w[2], a.v[2]); atomicMax(&w[3], a.v[3]);
	atomicMax(&w[4], a.v[4]);
}

__global__ void __launch_bounds__(256) k_grid_reduce(int n, const float4* bmin, const float4* bmax, const int* scene,
                                                      uint32_t* acc)
{
	__shared__ GridRange red[4];
	const int base = blockIdx.x * 256 * GRID_ITEMS;
	const int blockLast = min(n, base + 256 * GRID_ITEMS) - 1;
	const int lane = threadIdx.x & 63;
	const GridRange none = {{0xFFFFFFFFu, 0u, 0xFFFFFFFFu, 0u, 0u}};
	auto load = [&](int i, GridRange& r) {
		const float4 a = bmin[i], b = bmax[i];
		const uint32_t cy = encode_float(0.5f * (a.y + b.y)), cz = encode_float(0.5f * (a.z + b.z));
		r = {{cy, cy, cz, cz, encode_float(fmaxf(b.y - a.y, b.z - a.z))}};
	};
	if (scene[base] == scene[blockLast])
	{
		// one world in the whole block (bodies are ordered by world)
		GridRange t = none;
#pragma unroll 4
		for (int k = 0; k < GRID_ITEMS; k++)
		{
			const int i = base + k * 256 + threadIdx.x;
			if (i < n)
			{
				GridRange r;
				load(i, r);
				gridMerge(t, r);
			}
		}
		t = gridWave(t);
		if (lane == 0)
			red[threadIdx.x >> 6] = t;
		__syncthreads();
		if (threadIdx.x == 0)
		{
			for (int k = 1; k < 4; k++)
				gridMerge(t, red[k]);
			gridAtomic(acc + 5 * int64_t(scene[base]), t);
		}
		return;
	}
	for (int k = 0; k < GRID_ITEMS; k++)
	{
		const int i = base + k * 256 + threadIdx.x;
		GridRange own = none;
		int world = -1;
		if (i < n)
		{
			load(i, own);
			world = scene[i];
		}
		uint64_t todo = __ballot(world >= 0);
		while (todo)
		{
			const int lead = __ffsll((unsigned long long)todo) - 1;
			const int w = __shfl(world, lead);
			const bool mine = world == w;
			todo &= ~__ballot(mine);
			const GridRange r = gridWave(mine ? own : none);
			if (lane == lead)
				gridAtomic(acc + 5 * int64_t(w), r);
		}
	}
}

__global__ void k_grid_init(int nScenes, uint32_t* acc)
{
	const int s = blockIdx.x * blockDim.x + threadIdx.x;
	if (s < nScenes)
	{
		acc[5 * s + 0] = 0xFFFFFFFFu; acc[5 * s + 1] = 0u;
		acc[5 * s + 2] = 0xFFFFFFFFu; acc[5 * s + 3] = 0u;
		acc[5 * s + 4] = 0u;
	}
}

// Each world's rows are capped by its slice of rowOff (the host sizes the row
// table up front, so no count comes back before the sort): the cell grows
// until ny * nz fits. Cells only need to be at least as wide as the widest
// box; wider cells give the same pairs with longer sweeps.
PXH_D void gridCells(const GridRange& w, int64_t cap, float4& gf, int2& gi)
{
	const bool empty = w.v[0] == 0xFFFFFFFFu && w.v[1] == 0u;
	const float ly = empty ? 0.0f : decode_float(w.v[0]), hy = empty ? 0.0f : decode_float(w.v[1]);
	const float lz = empty ? 0.0f : decode_float(w.v[2]), hz = empty ? 0.0f : decode_float(w.v[3]);
	const float wm = empty ? 0.0f : decode_float(w.v[4]);
	float cell = wm * 1.01f + 1e-6f;
	cell = fmaxf(cell, fmaxf(hy - ly, hz - lz) * (1.0f / 1000.0f));
	int ny = 1, nz = 1;
	for (int it = 0; it < 96; it++)
	{
		ny = max(1, min(int((hy - ly) / cell) + 1, 1024));
		nz = max(1, min(int((hz - lz) / cell) + 1, 1024));
		if (int64_t(ny) * nz <= cap)
			break;
		cell *= 1.25f;
	}
	if (int64_t(ny) * nz > cap)
	{
		ny = 1;
		nz = 1;
		cell = fmaxf(cell, fmaxf(hy - ly, hz - lz) + 1.0f);
	}
	gf = make_float4(ly, lz, 1.0f / cell, cell);
	gi = make_int2(ny, nz);
}

__global__ void k_grid_finish(int nScenes, const uint32_t* acc, float4* gridF, int2* gridI, const uint32_t* rowOff)
{
	const int s = blockIdx.x * blockDim.x + threadIdx.x;
	if (s >= nScenes)
		return;
	GridRange w;
	for (int k = 0; k < 5; k++)
		w.v[k] = acc[5 * int64_t(s) + k];
	gridCells(w, int64_t(rowOff[s + 1] - rowOff[s]), gridF[s], gridI[s]);
}

// row table of a single world with cap rows
__global__ void k_row_off_single(uint32_t* rowOff, uint32_t cap)
{
	if (threadIdx.x == 0 && blockIdx.x == 0)
	{
		rowOff[0] = 0u;
		rowOff[1] = cap;
	}
}

PXH_D uint64_t sweepKey(float4 a, float4 b, float4 gf, int2 gi, uint32_t rowOff)
{
	const float cy = 0.5f * (a.y + b.y), cz = 0.5f * (a.z + b.z);
	const int iy = min(max(int(floorf((cy - gf.x) * gf.z)), 0), gi.x - 1);
	const int iz = min(max(int(floorf((cz - gf.y) * gf.z)), 0), gi.y - 1);
	const uint32_t row = rowOff + uint32_t(iz * gi.x + iy);
	return (uint64_t(row) << 32) | encode_float(a.x);
}

__global__ void k_keys(int n, const float4* bmin, const float4* bmax, const int* scene, const float4* gridF,
                       const int2* gridI, const uint32_t* rowOff, uint64_t* keys, uint32_t* vals)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	const int s = scene[i];
	keys[i] = sweepKey(bmin[i], bmax[i], gridF[s], gridI[s], rowOff[s]);
	vals[i] = uint32_t(i);
}

// Grid and sweep keys of worlds that one workgroup each can take (the launch
// has a workgroup a world): the range, the cells and the keys in one launch
// without atomics, for k_grid_init, k_grid_reduce, k_grid_finish and k_keys.
__global__ void __launch_bounds__(1024) k_world_grid(const int* bodyStart, const float4* bmin, const float4* bmax,
                                                     float4* gridF, int2* gridI, const uint32_t* rowOff,
                                                     uint64_t* keys, uint32_t* vals)
{
	__shared__ GridRange red[16];
	__shared__ float4 sF;
	__shared__ int2 sI;
	const int w = blockIdx.x;
	const int b0 = bodyStart[w], b1 = bodyStart[w + 1];
	GridRange t = {{0xFFFFFFFFu, 0u, 0xFFFFFFFFu, 0u, 0u}};
#pragma unroll 4
	for (int i = b0 + int(threadIdx.x); i < b1; i += int(blockDim.x))
	{
		const float4 a = bmin[i], b = bmax[i];
		const uint32_t cy = encode_float(0.5f * (a.y + b.y)), cz = encode_float(0.5f * (a.z + b.z));
		const GridRange r = {{cy, cy, cz, cz, encode_float(fmaxf(b.y - a.y, b.z - a.z))}};
		gridMerge(t, r);
	}
	t = gridWave(t);
	if ((threadIdx.x & 63) == 0)
		red[threadIdx.x >> 6] = t;
	__syncthreads();
	const uint32_t ro = rowOff[w];
	if (threadIdx.x == 0)
	{
		for (int k = 1; k < int(blockDim.x >> 6); k++)
			gridMerge(t, red[k]);
		float4 gf;
		int2 gi;
		gridCells(t, int64_t(rowOff[w + 1] - ro), gf, gi);
		sF = gf;
		sI = gi;
		gridF[w] = gf;
		gridI[w] = gi;
	}
	__syncthreads();
	const float4 gf = sF;
	const int2 gi = sI;
#pragma unroll 4
	for (int i = b0 + int(threadIdx.x); i < b1; i += int(blockDim.x))
	{
		keys[i] = sweepKey(bmin[i], bmax[i], gf, gi, ro);
		vals[i] = uint32_t(i);
	}
}

__global__ void k_gather_sorted(int n, const uint32_t* sortedVals, const float4* bmin, const float4* bmax,
                                float4* smin, float4* smax)
{
	const int s = blockIdx.x * blockDim.x + threadIdx.x;
	if (s >= n)
		return;
	const uint32_t i = sortedVals[s];
	smin[s] = bmin[i];
	float4 b = bmax[i];
	b.w = __uint_as_float(i);
	smax[s] = b;
}

// rowStart[r] = first sorted position of row r; rowStart[totalRows] = n.
// Keys past totalRows count as totalRows (rowStart has totalRows + 2 entries).
// Lane s fills the rows from the previous key's row (exclusive) to its own, a
// long run of empty rows with its whole wave (one lane alone took 38 us where
// worlds leave hundreds of rows empty); the rows after the last key have a lane
// each.
// Where the host reads the starts, rowStart is host memory, and the step's words
// go along; copies of a few words cost 3 us each on the stream.
__global__ void __launch_bounds__(256) k_row_start(int n, const uint64_t* sortedKeys, uint32_t* rowStart,
                                                   uint32_t totalRows, const uint32_t* words, uint32_t* hostWords)
{
	const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (words && t < STEP_WORDS)
		hostWords[t] = words[t];
	const int64_t last = int64_t(min(uint32_t(sortedKeys[n - 1] >> 32), totalRows));
	if (t > last && t <= int64_t(totalRows))
		rowStart[t] = uint32_t(n);
	int64_t r = 0, from = 1;   // rows [from, r] start at t
	if (t < n)
	{
		r = int64_t(min(uint32_t(sortedKeys[t] >> 32), totalRows));
		from = t == 0 ? 0 : int64_t(min(uint32_t(sortedKeys[t - 1] >> 32), totalRows)) + 1;
	}
	const int lane = threadIdx.x & 63;
	const bool longRun = r - from >= 4;
	uint64_t todo = __ballot(longRun);
	while (todo)
	{
		const int lead = __ffsll((unsigned long long)todo) - 1;
		todo &= todo - 1;
		const int64_t f = __shfl(from, lead), e = __shfl(r, lead), v = __shfl(t, lead);
		for (int64_t k = f + lane; k <= e; k += 64)
			rowStart[k] = uint32_t(v);
	}
	if (!longRun)
		for (int64_t k = from; k <= r; k++)
			rowStart[k] = uint32_t(t);
}

__global__ void k_fill_u32(uint32_t* p, int64_t n, uint32_t v)
{
	const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i < n)
		p[i] = v;
}

// pair class from the two geometry types, spheres and capsules counting as
// round shapes: 0 round-round, 1 round-box, 2 box-box, 3 round-convex,
// 4 box-convex, 5 convex-convex
PXH_D int pairClass(int t0, int t1)
{
	const int nc = (t0 == GEOM_CONVEXMESH) + (t1 == GEOM_CONVEXMESH);
	const int nb = (t0 == GEOM_BOX) + (t1 == GEOM_BOX);
	return nc == 0 ? nb : (nc == 2 ? 5 : 3 + nb);
}

// Sweep of the sorted rows: lane s (body i) reports each overlapping body j in
// its own and the 8 neighbouring rows whose (minX, index) sorts after its own,
// so every pair is found exactly once. The overlap test is the reference ABP's
// inclusive test on inflated bounds (BpBroadPhaseABP.cpp:2246-2262, :2474).
// WRITE=false counts pairs per class into counts[cls*n + s]; WRITE=true writes
// them at the scanned offsets.
//
// Broadphase group filter (Bp::groupFiltering, lowlevelaabb/include/BpFiltering.h:99-109):
// boxes of equal groups never pair; otherwise bit (type0 * 8 + type1) of lut,
// type = group & 7 (BpFilter's 7 x 7 table, lowlevelaabb/src/BpFiltering.cpp,
// in an 8 x 8 bit mask; all bits set: only equal groups are filtered)
PXH_D bool groupsPair(int g0, int g1, uint64_t lut)
{
	return g0 != g1 && ((lut >> ((g0 & 7) * 8 + (g1 & 7))) & 1ull);
}

// G lanes share a body, each taking 9 / G of the nine rows in order, so a body's
// pairs keep their places: one lane for all nine rows is a chain of nine binary
// searches and scans. launch_sweep has the rule and its figures. With G > 1 the
// write pass first counts again the pairs of the lanes that have a later lane to
// place (with one huge box the whole grid is one row and nobody has: 30,000 boxes
// 22.7 ms, 33.4 when every lane counted, 29.6 with one lane a body; 131,072 boxes
// 64, 94 and 70).
// CLASSES: pair classes that can occur (1: the standalone broadphase's boxes, 3:
// no convex hulls, 6).
constexpr int SWEEP_THREADS = 256;
template <bool WRITE, int G, int CLASSES>
__global__ void __launch_bounds__(SWEEP_THREADS) k_sweep(int n, const uint64_t* sortedKeys, const float4* smin,
                                                         const float4* smax, const int* scene, const int* group,
                                                         uint64_t groupLut, const int2* gridI, const uint32_t* rowOff,
                                                         const uint32_t* rowStart, uint32_t* counts,
                                                         const uint32_t* offsets, uint2* pairs, uint32_t pairCap)
{
	constexpr int PER = 63 / G, ROWS = 9 / G;   // bodies of a wave (its last lane idles), rows of a lane
	const int lane = threadIdx.x & 63;
	const int slot = lane / G, sub = lane - slot * G;
	const int s = (blockIdx.x * (SWEEP_THREADS / 64) + (threadIdx.x >> 6)) * PER + slot;
	const bool live = slot < PER && s < n;
	const int at = live ? s : n - 1;
	const uint64_t key = sortedKeys[at];
	const float4 a0 = smin[at], a1 = smax[at];
	const uint32_t i = __float_as_uint(a1.w);
	const int ti = int(a0.w);
	const int sc = scene[i];
	const int gi_ = group ? group[i] : -1;
	const int2 gi = gridI[sc];
	const uint32_t r = uint32_t(key >> 32);
	const uint32_t ro = rowOff[sc];
	const int lr = int(r - ro);
	const int cy = lr % gi.x, cz = lr / gi.x;
	uint32_t lo[ROWS], hi[ROWS];
#pragma unroll
	for (int q = 0; q < ROWS; q++)
	{
		const int row = sub * ROWS + q;
		const int z = cz + row / 3 - 1, y = cy + row % 3 - 1;
		lo[q] = hi[q] = 0u;
		if (!live || z < 0 || z >= gi.y || y < 0 || y >= gi.x)
			continue;
		const uint32_t rr = ro + uint32_t(z * gi.x + y);
		uint32_t l = rowStart[rr];
		hi[q] = rowStart[rr + 1];
		if (rr == r)
			l = uint32_t(s) + 1u;
		else
		{
			// first position whose (minX key, body index) follows ours
			uint32_t h = hi[q];
			while (l < h)
			{
				const uint32_t m = (l + h) >> 1;
				const uint64_t km = sortedKeys[m];
				const bool after = (uint32_t(km) > uint32_t(key)) ||
				                   (uint32_t(km) == uint32_t(key) && __float_as_uint(smax[m].w) > i);
				if (after) h = m;
				else l = m + 1;
			}
		}
		lo[q] = l;
	}
	uint32_t cnt[CLASSES];
#pragma unroll
	for (int c = 0; c < CLASSES; c++)
		cnt[c] = 0u;
	// the candidates of this lane's rows: found(class, body index, its type)
	auto visit = [&](auto found) {
#pragma unroll
		for (int q = 0; q < ROWS; q++)
			for (uint32_t j = lo[q]; j < hi[q]; j++)
			{
				const float4 b0 = smin[j];
				if (b0.x > a1.x)
					break;
				const float4 b1 = smax[j];
				if (b1.y < a0.y || a1.y < b0.y || b1.z < a0.z || a1.z < b0.z)
					continue;
				const uint32_t jj = __float_as_uint(b1.w);
				if (group && !groupsPair(gi_, group[jj], groupLut))
					continue;
				const int tj = int(b0.w);
				found(CLASSES == 1 ? 0 : pairClass(ti, tj), jj, tj);
			}
	};
	bool counted = true;
	if constexpr (WRITE && G > 1)
	{
		// a lane's count places the pairs of the body's later lanes only
		bool has = false;
#pragma unroll
		for (int q = 0; q < ROWS; q++)
			has |= lo[q] < hi[q];
		counted = ((__ballot(has) >> lane >> 1) & ((1ull << (G - 1 - sub)) - 1ull)) != 0ull;
	}
	if (counted)
		visit([&](int cls, uint32_t, int) {
#pragma unroll
			for (int c = 0; c < CLASSES; c++)
				cnt[c] += cls == c ? 1u : 0u;
		});
	if (!WRITE)
	{
		// the scan's last entry (its total) starts as zero
		if (live && sub == 0 && s == 0)
			counts[int64_t(CLASSES) * n] = 0u;
#pragma unroll
		for (int c = 0; c < CLASSES; c++)
		{
			uint32_t sum = 0;
#pragma unroll
			for (int k = 0; k < G; k++)
				sum += __shfl(cnt[c], min(slot * G + k, 63));
			if (live && sub == 0)
				counts[int64_t(c) * n + s] = sum;
		}
		return;
	}
	// the lane's first place in each class: the body's, and its earlier rows' pairs
	uint32_t off[CLASSES];
#pragma unroll
	for (int c = 0; c < CLASSES; c++)
	{
		uint32_t inc = cnt[c];
#pragma unroll
		for (int d = 1; d < G; d <<= 1)
		{
			const uint32_t t = __shfl_up(inc, d);
			if (sub >= d)
				inc += t;
		}
		off[c] = (live ? offsets[int64_t(c) * n + s] : 0u) + inc - cnt[c];
	}
	visit([&](int cls, uint32_t jj, int tj) {
		// shape order of the reference's contact managers: the lower
		// geometry type first (contact-method table order); two
		// shapes of one type put the later-added body first
		// (shouldSwapBodies, simulationcontroller/src/ScNPhaseCore.cpp:182-249)
		uint32_t pa, pb;
		if (ti != tj) { pa = ti < tj ? i : jj; pb = ti < tj ? jj : i; }
		else { pa = max(i, jj); pb = min(i, jj); }
		// pairs past the buffer's capacity are counted, not written
#pragma unroll
		for (int c = 0; c < CLASSES; c++)
			if (cls == c)
			{
				if (off[c] < pairCap)
					pairs[off[c]] = make_uint2(pa, pb);
				off[c]++;
			}
	});
}

// ---------------------------------------------------------------------------
// narrowphase
// ---------------------------------------------------------------------------
PXH_D void storeContacts(int slot, const Contacts& c, int cnt, float4* ctN, float4* ctP)
{
	ctN[slot] = make_float4(c.n.x, c.n.y, c.n.z, __int_as_float(cnt));
	// at most four points; fixed indices keep them in registers
#pragma unroll
	for (int k = 0; k < 4; k++)
		if (k < cnt)
			ctP[4 * int64_t(slot) + k] = make_float4(c.p[k].x, c.p[k].y, c.p[k].z, c.sep[k]);
}

// appends value to out where take, at the count *total (one atomic a block;
// the order is left to chance, which nothing that reads the lists depends on)
PXH_D void blockAppend(bool take, int value, int* out, uint32_t* total)
{
	__shared__ uint32_t waveCnt[16], blockBase;
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
	const uint64_t m = __ballot(take);
	if (lane == 0)
		waveCnt[w] = uint32_t(__popcll(m));
	__syncthreads();
	if (threadIdx.x < 64)
	{
		const uint32_t c = lane < nw ? waveCnt[lane] : 0u;
		uint32_t sum = c;
		for (int off = 1; off < 16; off <<= 1)
		{
			const uint32_t o = __shfl_up(sum, off);
			sum += lane >= off ? o : 0u;
		}
		if (lane < nw)
			waveCnt[lane] = sum - c;
		if (lane == nw - 1)
			blockBase = sum ? atomicAdd(total, sum) : 0u;
	}
	__syncthreads();
	if (take)
		out[blockBase + waveCnt[w] + uint32_t(__popcll(m & ((1ull << lane) - 1ull)))] = value;
	__syncthreads();
}

// Kernels whose items are long serial chains with branches of their own (joint
// rows, a wave's pairs one after the other) fill a wave only as far as the chip is
// full: a wave of 64 such lanes runs every branch of every lane one after the
// other, while most compute units idle. THIN_BLOCKS waves take `lanes` items
// each at a time, one until there are more items than waves.
constexpr int THIN_BLOCKS = 4096;
__host__ __device__ inline int thinLanes(uint32_t count)
{
	int l = 1;
	while (l < 64 && uint32_t(l) * THIN_BLOCKS < count)
		l *= 2;
	return l;
}
// item of this lane for i = 0, 1, ...: false where it has none; loops end at the
// same i for the whole wave
#define PXH_THIN_LOOP(q, count)                                                                                    \
	for (uint32_t lanes_ = uint32_t(thinLanes(count)), base_ = blockIdx.x * lanes_, q = base_ + threadIdx.x;       \
	     base_ < uint32_t(count); base_ += gridDim.x * lanes_, q = base_ + threadIdx.x)                            \
		if (threadIdx.x < lanes_ && q < uint32_t(count))
static inline int thinGrid(int64_t most) { return int(std::min<int64_t>(std::max<int64_t>(most, 1), THIN_BLOCKS)); }

// Body-body pairs; the shape order is the reference contact-method table's
// (lower geometry type first), so body a of a sphere-box pair is the sphere.
// Lanes past the pair count on the device (*dP) have no pair; pair p fills slot
// slotBase + p. One wave per workgroup: its box manifolds take 9 KB of LDS, and
// the box pairs that clipping leaves without a point share the wave
// (boxBoxEdgeWave), so no lane leaves before that. Bound by the longest lane of a
// wave: with that search in one lane and the manifolds in scratch memory the
// settled 262k sphere/box bin took 513 us, a 4,096-box pile 202 us; now 136 and 28.
constexpr int NP_THREADS = 64;
__global__ void __launch_bounds__(NP_THREADS) k_np_pairs(int cap, const uint32_t* dP, const uint32_t* dConvex,
                                                         int slotBase, const uint2* pairs, const float4* pos,
                                                         const float4* rot, const float4* geom, float cd, float tol,
                                                         float4* ctN, float4* ctP)
{
	__shared__ float4 points[3 * BOX_MAX_POINTS * NP_THREADS / 4];
	const int p = blockIdx.x * NP_THREADS + threadIdx.x;
	const bool live = p < cap && uint32_t(p) < *dConvex && uint32_t(p) < *dP;
	if (!__any(live))
		return;
	float4 g0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), g1 = g0;
	xf x0, x1;
	x0.p = mk(0.0f, 0.0f, 0.0f); x0.q = mkq(make_float4(0.0f, 0.0f, 0.0f, 1.0f));
	x1 = x0;
	Contacts c;
	c.count = 0;
	int cnt = 0;
	if (live)
	{
		const uint2 ab = pairs[p];
		g0 = geom[ab.x];
		g1 = geom[ab.y];
		const int t0 = int(g0.w), t1 = int(g1.w);
		x0.p = mk(pos[ab.x]);
		x1.p = mk(pos[ab.y]);
		if (t0 == GEOM_SPHERE && t1 == GEOM_SPHERE)
			cnt = sphereSphere(g0.x, x0.p, g1.x, x1.p, cd, c);
		else
		{
			if (t0 != GEOM_SPHERE)
				x0.q = mkq(rot[ab.x]);
			x1.q = mkq(rot[ab.y]);
			if (t0 == GEOM_SPHERE && t1 == GEOM_CAPSULE)
				cnt = sphereCapsule(g0.x, x0.p, g1.x, g1.y, x1, cd, c);
			else if (t0 == GEOM_SPHERE)
				cnt = sphereBox(g0.x, x0.p, mk(g1.x, g1.y, g1.z), x1, cd, c);
			else if (t1 == GEOM_CAPSULE)
				cnt = capsuleCapsule(g0.x, g0.y, x0, g1.x, g1.y, x1, cd, c);
			else if (t0 == GEOM_CAPSULE)
				cnt = capsulePoly<true>(g0.x, g0.y, x0, boxPoly(mk(g1.x, g1.y, g1.z)), x1, cd, tol, 0, c);
			else
				cnt = boxBoxFace(mk(g0.x, g0.y, g0.z), x0, mk(g1.x, g1.y, g1.z), x1, cd, tol, BoxPoints{reinterpret_cast<float*>(points) + threadIdx.x}, c);
		}
	}
	boxBoxEdgeWave(cnt == BOXBOX_EDGE, mk(g0.x, g0.y, g0.z), x0, mk(g1.x, g1.y, g1.z), x1, cd, c, cnt);
	if (live)
		storeContacts(slotBase + p, c, cnt, ctN, ctP);
}

// Body-plane pairs (every body against every plane of its world; a plane's
// bounds are unbounded so the broadphase always reports these pairs). The body
// is constraint body a; normals point from the plane to the body.
__global__ void __launch_bounds__(NP_THREADS) k_np_planes(int Q, int slotBase, const int* qBody, const int* qPlane,
                                                          const float4* pos, const float4* rot, const float4* geom,
                                                          const float4* planes, float cd, float4* ctN, float4* ctP)
{
	__shared__ float4 points[8 * NP_THREADS];
	const int q = blockIdx.x * NP_THREADS + threadIdx.x;
	if (q >= Q)
		return;
	const int i = qBody[q];
	const float4 g = geom[i];
	if (int(g.w) == GEOM_CONVEXMESH)
		return;
	const float4 pl = planes[qPlane[q]];
	Contacts c;
	c.count = 0;
	int cnt;
	if (int(g.w) == GEOM_SPHERE)
		cnt = spherePlane(g.x, mk(pos[i]), mk(pl), pl.w, cd, c);
	else
	{
		xf x;
		x.p = mk(pos[i]); x.q = mkq(rot[i]);
		if (int(g.w) == GEOM_CAPSULE)
			cnt = planeCapsule(mk(pl), pl.w, g.x, g.y, x, cd, c);
		else
			cnt = planeBox(mk(pl), pl.w, mk(g.x, g.y, g.z), x, cd, points + threadIdx.x, c);
		c.n = -c.n;
	}
	storeContacts(slotBase + q, c, cnt, ctN, ctP);
}

// Convex pairs: the class segments from *dConvex to *dP hold them. Sphere- and
// capsule-convex pairs, and the box- and convex-convex pairs whose bounding
// spheres come within the contact distance and that a few support steps don't
// show to be farther apart, go to their lists, the others get their empty
// contact slot here. Two lists of cap entries after two counts: 0 pairs to
// search (k_np_convex_wave and k_np_convex_finish), 1 round pairs
// (k_np_round_convex). Three of four pairs of a rubble pile don't touch; the
// steps take 8 lanes of a pair where the search takes a wave: of 8,192 hulls'
// 89,000 pairs, 7 us without and 37 with them, for 386 and 276 us of search.
PXH_D uint32_t* cvxEntries(uint32_t* list, int cap, int which) { return list + 2 + int64_t(which) * cap; }
PXH_D const uint32_t* cvxEntries(const uint32_t* list, int cap, int which) { return list + 2 + int64_t(which) * cap; }
constexpr int APART_BLOCK = 512;
__global__ void __launch_bounds__(APART_BLOCK) k_np_convex(int cap, const uint32_t* dP, const uint32_t* dConvex,
                            int slotBase, const uint2* pairs, const float4* pos, const float4* rot, const float4* geom,
                            HullSet hs, float cd, float4* ctN, uint32_t* list)
{
	constexpr uint32_t PAIRS = APART_BLOCK / APART_LANES;
	const uint32_t end = min(*dP, uint32_t(cap));
	const int sub = threadIdx.x % APART_LANES;
	for (uint32_t p0 = *dConvex + blockIdx.x * PAIRS; p0 < end; p0 += gridDim.x * PAIRS)
	{
		const uint32_t p = p0 + threadIdx.x / APART_LANES;
		bool round = false, search = false;
		if (p < end)
		{
			const uint2 ab = pairs[p];
			const float4 g0 = geom[ab.x], g1 = geom[ab.y];
			const int t0 = int(g0.w);
			round = t0 == GEOM_SPHERE || t0 == GEOM_CAPSULE;
			if (!round)
			{
				xf x0, x1;
				x0.p = mk(pos[ab.x]); x0.q = mkq(rot[ab.x]);
				x1.p = mk(pos[ab.y]); x1.q = mkq(rot[ab.y]);
				const float r0 = t0 == GEOM_BOX ? sqrtf(g0.x * g0.x + g0.y * g0.y + g0.z * g0.z) : hs.be[int(g0.x)].w;
				const float r1 = hs.be[int(g1.x)].w;
				const f3 d = x1.p - x0.p;
				const float reach = r0 + r1 + cd;
				search = dot(d, d) <= reach * reach;
				if (search)
				{
					const Poly B = hullPoly(hs, int(g1.x));
					const mxf aToB = mxfOf(xinvmul(x1, x0));
					const Poly A = t0 == GEOM_BOX ? boxPoly(mk(g0.x, g0.y, g0.z)) : hullPoly(hs, int(g0.x));
					// pairs within rounding, or within what planes lie off their
					// polygons' vertices (which the search also measures to), stay
					search = !convexApart(A, aToB, B, cd + 1e-5f * reach + 4.0f * (A.slack + B.slack), sub);
				}
				if (!search && sub == 0)
					ctN[slotBase + int(p)] = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(0));
			}
		}
		blockAppend(search && sub == 0, int(p), reinterpret_cast<int*>(cvxEntries(list, cap, 0)), list);
		blockAppend(round && sub == 0, int(p), reinterpret_cast<int*>(cvxEntries(list, cap, 1)), list + 1);
	}
}

// sphere- and capsule-convex pairs of list 1, a wave per pair that its bounding
// spheres do not settle; waves take thinLanes pairs at a time. Beyond the bounding
// spheres no face or edge is near enough, but planes of merged faces meet outside
// their vertices (1.5 cm off the radius of a blade a metre long), and inside all
// planes is a contact, so a lane looks at those. A lane's chain over a hull's faces
// and edges bound them: the pairs of 2,116 mixed bodies on a terrain took 86 us in a
// lane each, 13 so.
__global__ void __launch_bounds__(64) k_np_round_convex(int cap, int slotBase, const uint2* pairs, const float4* pos,
                                                        const float4* rot, const float4* geom, HullSet hs, float cd,
                                                        float tol, float4* ctN, float4* ctP, const uint32_t* list)
{
	const int lane = threadIdx.x;
	const uint32_t count = min(list[1], uint32_t(cap)), lanes = uint32_t(thinLanes(count));
	for (uint32_t base = blockIdx.x * lanes; base < count; base += gridDim.x * lanes)
	{
		const bool live = uint32_t(lane) < lanes && base + lane < count;
		const int p = live ? int(cvxEntries(list, cap, 1)[base + lane]) : 0;
		bool near = false;
		if (live)
		{
			const uint2 ab = pairs[p];
			const float4 g0 = geom[ab.x];
			const f3 d = mk(pos[ab.y]) - mk(pos[ab.x]);
			const int hull = int(geom[ab.y].x);
			const float core = g0.x + (int(g0.w) == GEOM_CAPSULE ? g0.y : 0.0f);
			const float reach = (core + hs.be[hull].w + cd + 4.0f * __int_as_float(hs.info2[hull].w)) * 1.00001f;
			near = !(dot(d, d) > reach * reach);
			if (!near)
			{
				xf x0, x1;
				x0.p = mk(pos[ab.x]); x0.q = mkq(rot[ab.x]);
				x1.p = mk(pos[ab.y]); x1.q = mkq(rot[ab.y]);
				f3 e0 = xtransinv(x1, x0.p), e1 = e0;
				if (int(g0.w) == GEOM_CAPSULE)
				{
					const mxf aToB = mxfOf(xinvmul(x1, x0));
					const f3 ext = mmul(aToB.r, mk(g0.y, 0.0f, 0.0f));
					e0 = aToB.p + ext;
					e1 = aToB.p - ext;
				}
				near = !planesKeepOut(hullPoly(hs, hull), e0, e1);
			}
			if (!near)
				ctN[slotBase + p] = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(0));
		}
		for (uint64_t m = __ballot(near); m != 0ull; m &= m - 1ull)
		{
			const int pp = laneOf(p, __ffsll((unsigned long long)m) - 1);
			const uint2 ab = pairs[pp];
			const float4 g0 = geom[ab.x], g1 = geom[ab.y];
			xf x0, x1;
			x0.p = mk(pos[ab.x]); x0.q = mkq(rot[ab.x]);
			x1.p = mk(pos[ab.y]); x1.q = mkq(rot[ab.y]);
			const Poly B = hullPoly(hs, int(g1.x));
			Contacts c;
			c.count = 0;
			const int cnt = int(g0.w) == GEOM_SPHERE ? sphereConvexWave(g0.x, x0.p, B, x1, cd, lane, c)
			                                         : capsulePoly<false>(g0.x, g0.y, x0, B, x1, cd, tol, lane, c);
			if (lane == 0)
				storeContacts(slotBase + pp, c, cnt, ctN, ctP);
		}
	}
}

// Box- and convex-convex pairs, separation phase: one wavefront per pair
// (grid-stride over the search list k_np_convex wrote) finds the closest
// features or the minimum translation and stores (dist, n), cA, cB at
// wit[3p .. 3p+2]; bound by vector instructions (half of its time at 386 us),
// so what it saves are pairs, edges and lanes without a result: 542 us at 8,192
// hulls of 24 points before crossing arcs were listed and closest features
// bounded, 386 after, 276 with k_np_convex's steps, 261 with B's arcs laid out.
// The contact phase looks at every searched pair's distance
// (a list of the touching ones, an atomic on one word for each, cost 32 us of
// 574 at 8,192 hulls). Polytopes past the LDS limits are searched by lane 0
// alone.
constexpr int CVX_WAVES = 4;
__global__ void __launch_bounds__(64 * CVX_WAVES, 4)   // at least 4 waves per SIMD
k_np_convex_wave(int cap, const uint2* pairs, const float4* pos, const float4* rot, const float4* geom, HullSet hs,
                 float cd, float4* wit, const uint32_t* list)
{
	__shared__ CvxLds lds[CVX_WAVES];
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	const uint32_t n = min(list[0], uint32_t(cap));
	for (uint32_t i = blockIdx.x * CVX_WAVES + w; i < n; i += gridDim.x * CVX_WAVES)
	{
		const uint32_t p = cvxEntries(list, cap, 0)[i];
		const uint2 ab = pairs[p];
		const float4 g0 = geom[ab.x], g1 = geom[ab.y];
		const int t0 = int(g0.w);
		float4 sep = make_float4(2.0f * cd + 1.0f, 1.0f, 0.0f, 0.0f);
		f3 cA = mk(0.0f, 0.0f, 0.0f), cB = cA;
		xf x0, x1;
		x0.p = mk(pos[ab.x]); x0.q = mkq(rot[ab.x]);
		x1.p = mk(pos[ab.y]); x1.q = mkq(rot[ab.y]);
		const Poly B = hullPoly(hs, int(g1.x));
		const Poly A = t0 == GEOM_BOX ? boxPoly(mk(g0.x, g0.y, g0.z)) : hullPoly(hs, int(g0.x));
		if (fitsWave(A, B))
			convexSeparationWave(A, x0, B, x1, cd, lds[w], lane, sep, cA, cB);
		else if (lane == 0)
		{
			const mxf aToB = mxfOf(xinvmul(x1, x0));
			f3 n = mk(1.0f, 0.0f, 0.0f);
			polySeparation(A, aToB, B, cd, sep.x, n, cA, cB);
			sep.y = n.x; sep.z = n.y; sep.w = n.z;
		}
		if (lane == 0)
		{
			wit[3 * int64_t(p)] = sep;
			if (sep.x <= cd)
			{
				wit[3 * int64_t(p) + 1] = f4(cA, 0.0f);
				wit[3 * int64_t(p) + 2] = f4(cB, 0.0f);
			}
		}
	}
}

// Box- and convex-convex pairs, contact phase: 16 lanes per touching pair of the
// search list (witness polygons, clipping, reduction); the others get their empty
// slot. The list order does not matter, pair p fills slot slotBase + p. Bound by a
// pair's chain of dependent loads and steps: for 20,600 touching pairs of 8,192
// hulls 107 us in a lane each, 90 in a wave each, 43 so (a terrain's few pairs
// 42, 13 and 19: a wave that takes one group only still needs 18).
__global__ void __launch_bounds__(64) k_np_convex_finish(int cap, int slotBase, const uint2* pairs, const float4* pos,
                                                         const float4* rot, const float4* geom, HullSet hs, float cd,
                                                         float tol, const float4* wit, const uint32_t* list,
                                                         float4* ctN, float4* ctP)
{
	__shared__ ContactLds lds[64 / GROUP];
	const int gl = threadIdx.x % GROUP, group = threadIdx.x / GROUP;
	const uint32_t count = min(list[0], uint32_t(cap));
	for (uint32_t q = blockIdx.x * (64 / GROUP) + group; q < count; q += gridDim.x * (64 / GROUP))
	{
		const int p = int(cvxEntries(list, cap, 0)[q]);
		const float4 sep = wit[3 * int64_t(p)];
		if (!(sep.x <= cd))
		{
			if (gl == 0)
				ctN[slotBase + p] = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(0));
			continue;
		}
		const uint2 ab = pairs[p];
		const float4 g0 = geom[ab.x], g1 = geom[ab.y];
		xf x0, x1;
		x0.p = mk(pos[ab.x]); x0.q = mkq(rot[ab.x]);
		x1.p = mk(pos[ab.y]); x1.q = mkq(rot[ab.y]);
		const Poly B = hullPoly(hs, int(g1.x));
		const Poly A = int(g0.w) == GEOM_BOX ? boxPoly(mk(g0.x, g0.y, g0.z)) : hullPoly(hs, int(g0.x));
		convexContactsGroup(A, x0, B, x1, sep.x, mk(sep.y, sep.z, sep.w), mk(wit[3 * int64_t(p) + 1]),
		                    mk(wit[3 * int64_t(p) + 2]), cd, tol, lds[group], gl, int64_t(slotBase) + p, ctN, ctP);
	}
}

// Body-plane pairs of convex bodies (the others are left to k_np_planes), a wave
// per hull that its bounding sphere does not keep off the plane; the hull is
// constraint body a, so normals point from the plane to the hull.
__global__ void __launch_bounds__(64) k_np_planes_convex(int Q, int slotBase, const int* qBody, const int* qPlane,
                                                         const float4* pos, const float4* rot, const float4* geom,
                                                         const float4* planes, HullSet hs, float cd, float tol,
                                                         float4* ctN, float4* ctP)
{
	__shared__ ContactLds L;
	const int lane = threadIdx.x, lanes = thinLanes(uint32_t(Q));
	for (int base = blockIdx.x * lanes; base < Q; base += gridDim.x * lanes)
	{
		const int q = base + lane;
		bool near = false;
		if (lane < lanes && q < Q)
		{
			const int i = qBody[q];
			const float4 g = geom[i];
			if (int(g.w) == GEOM_CONVEXMESH)
			{
				const float4 pl = planes[qPlane[q]];
				const f3 x = mk(pos[i]);
				const float r = hs.be[int(g.x)].w;
				// the margin is well above the rounding of a vertex's own distance
				const float slack = 1e-5f * (fabsf(x.x) + fabsf(x.y) + fabsf(x.z) + fabsf(pl.w) + r);
				near = !(dot(mk(pl), x) + pl.w > r * sqrtf(dot(mk(pl), mk(pl))) + cd + slack);
				if (!near)
					ctN[slotBase + q] = f4(mk(pl), __int_as_float(0));
			}
		}
		for (uint64_t m = __ballot(near); m != 0ull; m &= m - 1ull)
		{
			const int qq = base + __ffsll((unsigned long long)m) - 1;
			const int i = qBody[qq];
			const float4 pl = planes[qPlane[qq]];
			xf x;
			x.p = mk(pos[i]); x.q = mkq(rot[i]);
			planeConvexWave(mk(pl), pl.w, hullPoly(hs, int(geom[i].x)), x, cd, tol, L, lane, int64_t(slotBase) + qq, ctN,
			                ctP);
		}
	}
}

// Contact data of the last step, one 128-byte record per constraint in
// constraint order (row o of the colour order holds constraint order[o]):
// body0, body1 (or -1 - plane), contact count | normal (shape1 -> shape0) |
// 4 x (point, separation) | 4 applied normal impulses | 0. Lane 0 stores the
// number of records written.
__global__ void k_copy_contacts(int C, int maxPairs, const int* order, const int* conA, const int* conB,
                                const int* conSlot, const float4* ctN, const float4* ctP, const float* nF,
                                float4* out, uint32_t* nbPairs)
{
	const int o = blockIdx.x * blockDim.x + threadIdx.x;
	if (o == 0 && nbPairs)
		*nbPairs = uint32_t(min(C, maxPairs));
	if (o >= C)
		return;
	const int c = order[o];
	if (c >= maxPairs)
		return;
	const int slot = conSlot[c];
	const float4 n = ctN[slot];
	const int cnt = __float_as_int(n.w);
	float4* r = out + 8 * int64_t(c);
	r[0] = make_float4(__int_as_float(conA[c]), __int_as_float(conB[c]), __int_as_float(cnt), 0.0f);
	r[1] = make_float4(n.x, n.y, n.z, 0.0f);
	float f[4];
	for (int k = 0; k < 4; k++)
	{
		r[2 + k] = k < cnt ? ctP[4 * int64_t(slot) + k] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		f[k] = k < cnt ? nF[int64_t(k) * C + o] : 0.0f;
	}
	r[6] = make_float4(f[0], f[1], f[2], f[3]);
	r[7] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// slots: [0, Q) body-plane pairs, then body pairs up to the device count *dP
// slots: body-plane [0, Q), body pairs [Q, pairEnd) up to the count on the
// device, body-mesh patches [pairEnd, S)
PXH_D bool liveSlot(int s, int Q, int pairEnd, const uint32_t* dP)
{
	return s < Q || s >= pairEnd || uint32_t(s - Q) < *dP;
}

// flags of the touching slots and their sums over CON_TILE-slot tiles (smaller
// than the scan's: a thread that built up to sixteen constraints one after the
// other took 20 us at 20,011 bodies)
constexpr int CON_THREADS = 256, CON_ITEMS = 4, CON_TILE = CON_THREADS * CON_ITEMS;
__global__ void __launch_bounds__(CON_THREADS) k_touch_flags(int S, int Q, int pairEnd, const uint32_t* dP,
                                                             const float4* ctN, uint32_t* flags, uint32_t* sums)
{
	__shared__ uint32_t sh[8];
	const int base = blockIdx.x * CON_TILE;
	uint32_t v = 0;
#pragma unroll
	for (int k = 0; k < CON_ITEMS; k++)
	{
		const int s = base + k * CON_THREADS + threadIdx.x;
		if (s < S)
		{
			const uint32_t f = liveSlot(s, Q, pairEnd, dP) && __float_as_int(ctN[s].w) > 0 ? 1u : 0u;
			flags[s] = f;
			v += f;
		}
	}
	v = blockSum(v, sh);
	if (threadIdx.x == 0)
		sums[blockIdx.x] = v;
}
// Pair identity across steps, world-relative so it survives changes to other
// worlds: world (16 bits) | local index of a (24 bits) | local index of b or
// 0x800000 | plane index (24 bits).
PXH_D uint64_t worldPairKey(int w, uint32_t la, uint32_t lb)
{
	const uint32_t b24 = (lb & 0x80000000u) ? (0x800000u | (lb & 0x7FFFFFu)) : (lb & 0x7FFFFFu);
	return (uint64_t(uint32_t(w) & 0xFFFFu) << 48) | (uint64_t(la & 0xFFFFFFu) << 24) | b24;
}

// constraint list: touching pair slots in slot order, with the scene-local
// ordering key used by the colouring
// Each tile of slots adds up the counts of the tiles before it and scans its
// own flags; the last one leaves the pair and constraint counts (and whether
// the mesh candidates overflowed) in the host's words, which saves the copies.
PXH_D void buildConstraint(int s, int c, int Q, int pairEnd, const uint2* pairs, const int* qBody, const int* qPlane,
                           const int* meshBody, int nPlanes, const int* local, const int* planeLocal, const int* world,
                           const int* worldTag, int* conA, int* conB, int* conSlot, uint64_t* conKey,
                           uint64_t* conPKey, int* conColor)
{
	int a, b;
	uint32_t la, lb;
	if (s >= pairEnd)
	{
		// a mesh patch: static index plane count + patch, local id 0x400000 + patch
		const int k = s - pairEnd, p = k % MESH_MAXP;
		a = meshBody[k / MESH_MAXP];
		b = -1 - (nPlanes + p);
		la = uint32_t(local[a]);
		lb = 0x80000000u | (0x400000u + uint32_t(p));
	}
	else if (s >= Q)
	{
		const uint2 ab = pairs[s - Q];
		a = int(ab.x); b = int(ab.y);
		la = uint32_t(local[a]); lb = uint32_t(local[b]);
	}
	else
	{
		a = qBody[s];
		const int pl = qPlane[s];
		b = -1 - pl;
		la = uint32_t(local[a]);
		lb = 0x80000000u | uint32_t(planeLocal[pl]);
	}
	conA[c] = a;
	conB[c] = b;
	conSlot[c] = s;
	conKey[c] = mix64((uint64_t(la) << 32) | lb);
	conPKey[c] = worldPairKey(worldTag[world[a]], la, lb);
	conColor[c] = b >= 0 ? -1 : -2;  // -2: body-plane, placed after the body-body rounds
}

template <bool SCANNED>
__global__ void __launch_bounds__(CON_THREADS) k_con_build(
    int S, int Q, int pairEnd, const uint32_t* dP, const uint32_t* flags, const uint32_t* sums, const uint2* pairs,
    const int* qBody, const int* qPlane, const int* meshBody, int nPlanes, const int* local, const int* planeLocal,
    const int* world, const int* worldTag, const uint32_t* overflow, int* conA, int* conB, int* conSlot,
    uint64_t* conKey, uint64_t* conPKey, int* conColor, uint32_t* hostCounts)
{
	__shared__ uint32_t sh[33];
	__shared__ uint32_t waveSum[CON_ITEMS][CON_THREADS / 64];
	const int base = blockIdx.x * CON_TILE;
	const uint32_t before = tilesBefore<SCANNED>(sums, sh);
	// slot k * CON_THREADS + thread of the tile: its place among the wave's flags
	// of row k, then the waves before it
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	uint32_t mine = 0;   // bit k: slot k of this thread touches
	uint32_t rank[CON_ITEMS];
#pragma unroll
	for (int k = 0; k < CON_ITEMS; k++)
	{
		const int s = base + k * CON_THREADS + threadIdx.x;
		const bool f = s < S && flags[s] != 0u;
		const uint64_t m = __ballot(f);
		rank[k] = uint32_t(__popcll(m & ((1ull << lane) - 1ull)));
		mine |= f ? 1u << k : 0u;
		if (lane == 0)
			waveSum[k][w] = uint32_t(__popcll(m));
	}
	__syncthreads();
	uint32_t run = before;
#pragma unroll
	for (int k = 0; k < CON_ITEMS; k++)
	{
		uint32_t at = run;
#pragma unroll
		for (int i = 0; i < CON_THREADS / 64; i++)
		{
			at += i < w ? waveSum[k][i] : 0u;
			run += waveSum[k][i];
		}
		if (mine >> k & 1u)
			buildConstraint(base + k * CON_THREADS + threadIdx.x, int(at + rank[k]), Q, pairEnd, pairs, qBody, qPlane,
			                meshBody, nPlanes, local, planeLocal, world, worldTag, conA, conB, conSlot, conKey, conPKey,
			                conColor);
	}
	if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0)
	{
		hostCounts[0] = *dP;
		hostCounts[1] = run;
		hostCounts[2] = overflow ? *overflow : 0u;
	}
}

// ---------------------------------------------------------------------------
// colouring: a body-body constraint joins colour r when its key is the minimum
// over the uncoloured constraints of both its bodies (deterministic, and a
// function of each world's own content); body-plane constraints then follow
// every colour of their body's body-body constraints
// ---------------------------------------------------------------------------
__global__ void k_fill_u64(uint64_t* p, int64_t n, uint64_t v)
{
	const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i < n)
		p[i] = v;
}

// Colouring kernels run over the list of the still-uncoloured (body-body)
// constraints, list[i] for i below the count *mDev on the device, which m
// bounds. They loop grid-stride so the grid can be sized for the bound while few
// constraints remain.
PXH_D int listCount(int m, const uint32_t* mDev) { return min(m, int(*mDev)); }
#define PXH_GRID_STRIDE(i, count) \
	for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < (count); i += gridDim.x * blockDim.x)

__global__ void k_color_reset(int m, const uint32_t* mDev, const int* list, const int* conA, const int* conB,
                              unsigned long long* best)
{
	const int mm = listCount(m, mDev);
	PXH_GRID_STRIDE(i, mm)
	{
		const int c = list[i];
		best[conA[c]] = ~0ull;
		best[conB[c]] = ~0ull;
	}
}

__global__ void k_color_min(int m, const uint32_t* mDev, const int* list, const int* conA, const int* conB,
                            const uint64_t* conKey, const int* conColor, unsigned long long* best)
{
	const int mm = listCount(m, mDev);
	PXH_GRID_STRIDE(i, mm)
	{
		const int c = list[i];
		if (conColor[c] != -1)
			continue;
		const unsigned long long k = conKey[c];
		atomicMin(&best[conA[c]], k);
		atomicMin(&best[conB[c]], k);
	}
}

// A local minimum takes the smallest colour used by neither of its bodies
// (first fit on 64-bit per-body colour masks; colours past 63 fall back to
// one colour per round, 64 + round, and raise the bodies' `next`, the first
// colour past them). Minima of one round share no body, so their mask updates
// never race with each other's reads.
__global__ void k_color_pick(int m, const uint32_t* mDev, const int* list, int round, const int* conA,
                             const int* conB, const uint64_t* conKey, int* conColor, const unsigned long long* best,
                             unsigned long long* nextBest, ColorState cs)
{
	unsigned long long* mask = cs.mask;
	const int mm = listCount(m, mDev);
	PXH_GRID_STRIDE(i, mm)
	{
		const int c = list[i];
		if (conColor[c] != -1)
			continue;
		const unsigned long long k = conKey[c];
		const int a = conA[c], b = conB[c];
		nextBest[a] = ~0ull;
		nextBest[b] = ~0ull;
		if (best[a] == k && best[b] == k)
		{
			const unsigned long long used = mask[a] | mask[b];
			const int col = used == ~0ull ? 64 + round : __ffsll((long long)~used) - 1;
			conColor[c] = col;
			if (col < 64)
			{
				atomicOr(&mask[a], 1ull << col);
				atomicOr(&mask[b], 1ull << col);
			}
			else
			{
				atomicMax(&cs.next[a], uint32_t(col + 1));
				atomicMax(&cs.next[b], uint32_t(col + 1));
			}
		}
	}
}

// the constraints of the list that the rounds left uncoloured, as the next list
__global__ void __launch_bounds__(256) k_color_left(int m, const uint32_t* mDev, const int* list, const int* conColor,
                                                    int* out, uint32_t* left, uint32_t* ran, uint32_t rounds)
{
	const int mm = listCount(m, mDev);
	if (blockIdx.x == 0 && threadIdx.x == 0)
		*ran = rounds;
	for (int base = blockIdx.x * 256; base < mm; base += gridDim.x * 256)
	{
		const int i = base + threadIdx.x;
		const int c = i < mm ? list[i] : 0;
		blockAppend(i < mm && conColor[c] == -1, c, out, left);
	}
}

// Up to `rounds` colouring rounds of a short list (at most `limit`; else it only
// says so, *ran = 0) in one workgroup, ending when nothing is left; the same
// rounds as k_color_reset / min / pick. A settled step leaves a few hundred new
// constraints, for which eight rounds were 24 launches and 55 us; this takes 9 us
// on a 20,011-body bin. best holds two arrays of n: a round's picks clear the next round's
// minima. The minima and masks change in L2 by atomics and are read there
// (agent-scope loads), since the first-level cache may hold older lines.
PXH_D unsigned long long loadAgent(const unsigned long long* p)
{
	return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
PXH_D void storeAgent(unsigned long long* p, unsigned long long v)
{
	__hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// every memory operation of the wave done, then the block's barrier
PXH_D void blockPhase()
{
	__atomic_signal_fence(__ATOMIC_SEQ_CST);
	__builtin_amdgcn_s_waitcnt(0);
	__syncthreads();
}
constexpr int ROUND_THREADS = 1024;
__global__ void __launch_bounds__(ROUND_THREADS) k_color_rounds(const uint32_t* mDev, int limit, const int* list,
                                                                int firstRound, int rounds, int n, const int* conA,
                                                                const int* conB, const uint64_t* conKey, int* conColor,
                                                                unsigned long long* best, ColorState cs, int* out,
                                                                uint32_t* left, uint32_t* ran)
{
	const int m = int(*mDev);
	if (m > limit)
	{
		if (threadIdx.x == 0)
		{
			*left = uint32_t(m);
			*ran = 0u;
		}
		return;
	}
	for (int i = threadIdx.x; i < m; i += ROUND_THREADS)
	{
		const int c = list[i];
		storeAgent(&best[conA[c]], ~0ull);
		storeAgent(&best[conB[c]], ~0ull);
	}
	blockPhase();
	bool open = m > 0;
	for (int r = 0; r < rounds && open; r++)
	{
		unsigned long long* cur = best + (r & 1) * int64_t(n);
		unsigned long long* nxt = best + ((r + 1) & 1) * int64_t(n);
		for (int i = threadIdx.x; i < m; i += ROUND_THREADS)
		{
			const int c = list[i];
			if (conColor[c] != -1)
				continue;
			const unsigned long long k = conKey[c];
			atomicMin(&cur[conA[c]], k);
			atomicMin(&cur[conB[c]], k);
		}
		blockPhase();
		int more = 0;
		for (int i = threadIdx.x; i < m; i += ROUND_THREADS)
		{
			const int c = list[i];
			if (conColor[c] != -1)
				continue;
			const unsigned long long k = conKey[c];
			const int a = conA[c], b = conB[c];
			if (loadAgent(&cur[a]) == k && loadAgent(&cur[b]) == k)
			{
				const unsigned long long used = loadAgent(&cs.mask[a]) | loadAgent(&cs.mask[b]);
				const int col = used == ~0ull ? 64 + firstRound + r : __ffsll((long long)~used) - 1;
				conColor[c] = col;
				if (col < 64)
				{
					atomicOr(&cs.mask[a], 1ull << col);
					atomicOr(&cs.mask[b], 1ull << col);
				}
				else
				{
					atomicMax(&cs.next[a], uint32_t(col + 1));
					atomicMax(&cs.next[b], uint32_t(col + 1));
				}
			}
			else
				more = 1;
			storeAgent(&nxt[a], ~0ull);
			storeAgent(&nxt[b], ~0ull);
		}
		blockPhase();
		open = __syncthreads_or(more) != 0;
	}
	if (threadIdx.x == 0)
	{
		*left = 0u;
		*ran = uint32_t(rounds);
	}
	blockPhase();
	for (int base = 0; open && base < m; base += ROUND_THREADS)
	{
		const int i = base + threadIdx.x;
		const int c = i < m ? list[i] : 0;
		blockAppend(i < m && conColor[c] == -1, c, out, left);
	}
}

// Colour masks of the bodies that need theirs: those of a constraint still to be
// coloured and those with a body-plane constraint (k_con_prev marks them). Most
// constraints of a settled pile touch neither and make no atomic.
__global__ void k_color_mask(int C, const int* conA, const int* conB, const int* conColor, ColorState cs)
{
	const int c = blockIdx.x * blockDim.x + threadIdx.x;
	if (c >= C)
		return;
	const int col = conColor[c];
	if (col < 0)
		return;   // body-plane or not coloured yet; a carried colour is below 64
	const int a = conA[c], b = conB[c];
	if (cs.need[a])
		atomicOr(&cs.mask[a], 1ull << col);
	if (cs.need[b])
		atomicOr(&cs.mask[b], 1ull << col);
}

// Body-plane and body-mesh constraints go after every colour of their body's
// body-body constraints, one colour each in constraint order (the reference
// places static constraints at maxSolverNormalProgress + k:
// lowleveldynamics/src/DyConstraintPartition.cpp:168-179, 604-616). The last
// colour of a body is the top bit of its mask, or past 63 its `next`. k counts the
// body's static constraints before c: its plane constraints lead the list beside
// each other (slots are body-major, the bodies ascending), its mesh patches end it,
// also beside each other, with the body pairs between; where a world has planes
// and a mesh, a patch finds its body's plane constraints by bisection.
PXH_D int constraintColor(int c, const int* conA, const int* conB, int nPlanes, const ColorState& cs, int* conColor)
{
	auto plane = [&](int e) { return conB[e] < 0 && -1 - conB[e] < nPlanes; };
	if (conB[c] >= 0)
		return conColor[c];
	const int a = conA[c];
	const bool patch = !plane(c);
	int k = 0;
	for (int e = c - 1; e >= 0 && conA[e] == a && conB[e] < 0 && plane(e) != patch; e--)
		k++;
	if (patch && nPlanes > 0)
	{
		int lo = 0, hi = c;
		while (lo < hi)
		{
			const int m = (lo + hi) >> 1;
			if (plane(m) && conA[m] < a)
				lo = m + 1;
			else
				hi = m;
		}
		for (; lo < c && plane(lo) && conA[lo] == a; lo++)
			k++;
	}
	const unsigned long long m = cs.mask[a];
	const int next = max(int(cs.next[a]), m ? 64 - __clzll((long long)m) : 0);
	conColor[c] = next + k;
	return next + k;
}

// open-addressing table of the previous step's pair keys -> row (keys are
// unique; the table has at least twice as many slots as keys)
PXH_D uint32_t patchSlot(uint64_t key, uint32_t mask) { return uint32_t(mix64(key)) & mask; }

// an entry is the key and its row side by side, so a probe touches one line;
// the whole table starts at ~0 (no key has that value)
__global__ void k_patch_insert(int m, const uint64_t* keys, unsigned long long* table, uint32_t mask)
{
	const int o = blockIdx.x * blockDim.x + threadIdx.x;
	if (o >= m)
		return;
	const unsigned long long key = keys[o];
	uint32_t slot = patchSlot(key, mask);
	for (uint32_t probe = 0; probe <= mask; probe++)
	{
		if (atomicCAS(&table[2 * int64_t(slot)], ~0ull, key) == ~0ull)
		{
			table[2 * int64_t(slot) + 1] = (unsigned long long)(o);
			return;
		}
		slot = (slot + 1) & mask;
	}
}

PXH_D int patchFind(const PatchIO& io, uint64_t key)
{
	if (!io.table)
		return -1;
	uint32_t slot = patchSlot(key, io.tableMask);
	for (uint32_t probe = 0; probe <= io.tableMask; probe++)
	{
		const ulonglong2 e = io.table[slot];
		if (e.x == key)
			return int(e.y);
		if (e.x == ~0ull)
			return -1;
		slot = (slot + 1) & io.tableMask;
	}
	return -1;
}


// A body-body constraint that existed in the previous step keeps its colour
// (below 64): those constraints were coloured together then, so they never
// share a colour at a body now. The reference GPU solver keeps its partitions
// from step to step the same way (gpusolver/src/PxgConstraintPartition.cpp:1940).
// Lists the others and marks the bodies whose masks the colouring reads.
__global__ void __launch_bounds__(256) k_con_prev(int C, const int* conA, const int* conB, const int* conSlot,
                                                  PatchIO io, int* conColor, ColorState cs, int* list)
{
	const int c = blockIdx.x * blockDim.x + threadIdx.x;
	bool open = false;
	if (c < C)
	{
		const int a = conA[c], b = conB[c];
		const uint64_t pkey = io.conPKey[c];
		const int po = patchFind(io, pkey);
		if (io.prevRow)
			io.prevRow[c] = po;
		io.conRec[2 * int64_t(c)] = make_int4(a, b, conSlot[c], po);
		io.conRec[2 * int64_t(c) + 1] = make_int4(int(uint32_t(pkey)), int(uint32_t(pkey >> 32)), 0, 0);
		if (b < 0)
			cs.need[a] = 1u;
		else
		{
			const int pc = po >= 0 ? io.prevColor[po] : -1;
			if (pc >= 0 && pc < 64)
				conColor[c] = pc;
			else
			{
				open = true;
				cs.need[a] = 1u;
				cs.need[b] = 1u;
			}
		}
	}
	blockAppend(open, c, list, cs.words + STEP_OPEN);
}

// colour-ordered constraint list by a stable radix sort of (colour, index)
// A constraint not coloured yet (-1, when the rounds have not finished) sorts
// to colour `limit`, past every real colour.
__global__ void k_color_keys(int C, const int* conA, const int* conB, int nPlanes, int* conColor, ColorState cs,
                             uint32_t limit, uint64_t* keys, uint32_t* vals)
{
	const int c = blockIdx.x * blockDim.x + threadIdx.x;
	if (c < C)
	{
		const int col = constraintColor(c, conA, conB, nPlanes, cs, conColor);
		const uint32_t k = col < 0 ? limit : min(uint32_t(col), limit);
		keys[c] = (uint64_t(k) << 32) | uint32_t(c);
		vals[c] = uint32_t(c);
	}
}
// rows ordered by (world, colour): key world * CB + colour, CB = limit + 1; the
// largest colour in the step's words (one atomic a block)
__global__ void __launch_bounds__(256) k_color_keys_world(int C, const int* conA, const int* conB, int nPlanes,
                                                          int* conColor, ColorState cs, const int* bodyWorld,
                                                          uint32_t limit, uint64_t* keys, uint32_t* vals)
{
	__shared__ int red[4];
	const int c = blockIdx.x * blockDim.x + threadIdx.x;
	int top = 0;
	if (c < C)
	{
		const int col = constraintColor(c, conA, conB, nPlanes, cs, conColor);
		const uint32_t k = col < 0 ? limit : min(uint32_t(col), limit);
		const uint64_t w = uint64_t(bodyWorld[conA[c]]);
		keys[c] = ((w * (limit + 1) + k) << 32) | uint32_t(c);
		vals[c] = uint32_t(c);
		top = max(col, 0);
	}
#pragma unroll
	for (int o = 1; o < 64; o <<= 1)
		top = max(top, __shfl_xor(top, o));
	if ((threadIdx.x & 63) == 0)
		red[threadIdx.x >> 6] = top;
	__syncthreads();
	if (threadIdx.x == 0)
	{
		top = max(max(red[0], red[1]), max(red[2], red[3]));
		// most blocks stay below the maximum that others have left
		if (uint32_t(top) > __hip_atomic_load(&cs.words[STEP_TOP], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
			atomicMax(&cs.words[STEP_TOP], uint32_t(top));
	}
}

// ---------------------------------------------------------------------------
// solver
// ---------------------------------------------------------------------------

// bodyCoreComputeUnconstrainedVelocity (lowleveldynamics/src/DyBodyCoreIntegrator.h:40-75)
// + copyToSolverBodyDataStep (lowleveldynamics/src/DyTGSDynamics.cpp:154-242)
__global__ void k_preintegrate(int n, const float4* pos, const float4* rot, const float4* lin, const float4* ang,
                               const float4* invI, float3 gdt, float linDampDt, float angDampDt, float maxLinSq,
                               float maxAngSq, int pgs, float4* vel, float4* svP, float4* svDQ, float4* svI0,
                               float4* svI1, float4* svOrigLin, float4* rec, float dt, float4* extLin, float4* extAng,
                               float4* prevLin, float4* prevAng, const uint32_t* sleepFlags)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	const float4 l = lin[i];
	f3 lv = mk(l);
	f3 av = mk(ang[i]);
	// velocities before the step, for the acceleration reads
	if (prevLin)
	{
		prevLin[i] = f4(lv, 0.0f);
		prevAng[i] = f4(av, 0.0f);
	}
	// external accelerations (forces and torques set through the Direct GPU
	// API) change the velocities first, then gravity (BodySim::updateForces,
	// simulationcontroller/src/ScBodySim.cpp:656-713, before
	// bodyCoreComputeUnconstrainedVelocity); they last one step
	if (extLin)
	{
		const float4 el = extLin[i], ea = extAng[i];
		if (el.x != 0.0f || el.y != 0.0f || el.z != 0.0f)
			lv = lv + mk(el) * dt;
		if (ea.x != 0.0f || ea.y != 0.0f || ea.z != 0.0f)
			av = av + mk(ea) * dt;
		extLin[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		extAng[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	}
	// sleeping bodies are not in the solver: no gravity, velocities stay zero
	if (!sleepFlags || !(sleepFlags[i] & SLEEP_ASLEEP))
		lv = lv + mk(gdt.x, gdt.y, gdt.z);
	const float ld = 1.0f - linDampDt, ad = 1.0f - angDampDt;
	lv = lv * (ld >= 0.0f ? ld : 0.0f);
	av = av * (ad >= 0.0f ? ad : 0.0f);
	const float l2 = dot(lv, lv);
	if (l2 > maxLinSq) lv = lv * sqrtf(maxLinSq / l2);
	const float a2 = dot(av, av);
	if (a2 > maxAngSq) av = av * sqrtf(maxAngSq / a2);
	const m33 R = qmat(mkq(rot[i]));
	const float4 ii = invI[i];
	const f3 si = mk(sqrtf(ii.x), sqrtf(ii.y), sqrtf(ii.z));
	const f3 sI = mk(si.x == 0.0f ? 0.0f : 1.0f / si.x, si.y == 0.0f ? 0.0f : 1.0f / si.y,
	                 si.z == 0.0f ? 0.0f : 1.0f / si.z);
	m33 A, B;
	A.c0 = R.c0 * si.x; A.c1 = R.c1 * si.y; A.c2 = R.c2 * si.z;
	B.c0 = R.c0 * sI.x; B.c1 = R.c1 * sI.y; B.c2 = R.c2 * sI.z;
	const m33 Rt = mtrans(R);
	const m33 S = mmm(A, Rt);
	const m33 SI = mmm(B, Rt);
	float4* v = vel + 4 * int64_t(i);
	if (pgs)
	{
		// PGS solves for velocity changes from the pre-integrated velocities,
		// kept in the record's second half (copyToSolverBodyData,
		// lowleveldynamics/src/DyRigidBodyToSolverBody.cpp:37-113)
		v[0] = make_float4(0.0f, 0.0f, 0.0f, l.w);
		v[1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		v[2] = f4(lv, 0.0f);
		v[3] = f4(av, 0.0f);
	}
	else
	{
		v[0] = f4(lv, l.w);
		v[1] = f4(mmul(SI, av), 0.0f);
		v[2] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		v[3] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	}
	svP[i] = pos[i];
	svDQ[i] = make_float4(0.0f, 0.0f, 0.0f, 1.0f);
	// symmetric sqrt inverse inertia: (xx yy zz xy) (xz yz)
	const float4 i0 = make_float4(S.c0.x, S.c1.y, S.c2.z, S.c1.x);
	const float4 i1 = make_float4(S.c2.x, S.c2.y, 0.0f, 0.0f);
	svI0[i] = i0;
	svI1[i] = i1;
	svOrigLin[i] = f4(lv, 0.0f);
	float4* r = rec + PREP_REC * int64_t(i);
	const float4 p = pos[i];
	r[0] = make_float4(p.x, p.y, p.z, l.w);
	r[1] = rot[i];
	r[2] = i0;
	r[3] = i1;
	r[4] = f4(lv, 0.0f);
	r[5] = f4(av, 0.0f);
}

PXH_D m33 loadSym(float4 a, float4 b)
{
	m33 m;
	m.c0 = mk(a.x, a.w, b.x);
	m.c1 = mk(a.w, a.y, b.y);
	m.c2 = mk(b.x, b.y, a.z);
	return m;
}

// Friction patch of the constraint at row o (constraint c, bodies a, b,
// normal n, frames f0/f1, contact points cp/cs): the previous step's patch of
// this pair is kept when it is unbroken, has anchors, its body normals still
// agree, no anchor drifted apart along the normal, and its world normal
// matches this step's normal (getFrictionPatches, correlatePatches,
// growPatches: lowleveldynamics/src/DyContactPrepShared.h:53-127,
// DyFrictionCorrelation.cpp:136-316). Writes the patch for the next step and
// returns the anchor count, the anchors in pa0/pa1 (body space). Shared by the
// TGS and PGS preparation.
PXH_D int frictionPatch(int o, int c, int po, uint64_t pkey, f3 n, const xf& f0, const xf& f1, const f3 (&cp)[4],
                        const float (&cs)[4], int cnt, float restDist, float frictionOffsetThreshold,
                        const PatchIO& io, f3 (&pa0)[2], f3 (&pa1)[2])
{
	// friction patch: the previous step's patch of this pair is kept when it is
	// unbroken, has anchors, its body normals still agree, no anchor drifted
	// apart along the normal, and its world normal matches this step's normal
	f3 pn0, pn1;
	int nKept = 0;
	{
		bool kept = false;
		if (po >= 0 && !io.prevBroken[po])
		{
			const float4 q0 = io.prev[6 * int64_t(po) + 0];
			const int pc = __float_as_int(q0.w);
			if (pc != 0)
			{
				const float4 q1 = io.prev[6 * int64_t(po) + 1];
				pn0 = mk(q0); pn1 = mk(q1);
				pa0[0] = mk(io.prev[6 * int64_t(po) + 2]); pa0[1] = mk(io.prev[6 * int64_t(po) + 3]);
				pa1[0] = mk(io.prev[6 * int64_t(po) + 4]); pa1[1] = mk(io.prev[6 * int64_t(po) + 5]);
				const xf b10 = xinvmul(f0, f1);
				if (dot(pn0, qrot(b10.q, pn1)) > 0.999f)
				{
					bool separated = false;
#pragma unroll
					for (int j = 0; j < 2; j++)
						if (j < pc && !(fabsf(dot(pa0[j] - xtrans(b10, pa1[j]), pn0)) < io.corrDist))
							separated = true;
					if (!separated && !(dot(n, qrot(f0.q, pn0)) < 0.999f))
					{
						kept = true;
						nKept = pc;
					}
				}
			}
		}
		if (!kept)
		{
			pn0 = qrotinv(f0.q, n);
			pn1 = qrotinv(f1.q, n);
		}
	}
	// anchors: two kept anchors stay unless closer than half the diagonal of
	// this step's contact bounds; one kept anchor is completed from the
	// contacts; otherwise up to two points closer than the offset threshold
	if (nKept == 2)
	{
		f3 mn = cp[0], mx = cp[0];
#pragma unroll
		for (int j = 1; j < 4; j++)
		{
			if (j >= cnt)
				break;
			mn = mk(fminf(mn.x, cp[j].x), fminf(mn.y, cp[j].y), fminf(mn.z, cp[j].z));
			mx = mk(fmaxf(mx.x, cp[j].x), fmaxf(mx.y, cp[j].y), fmaxf(mx.z, cp[j].z));
		}
		const f3 dg = mx - mn, da = pa0[0] - pa0[1];
		if (!(dot(da, da) * 4.0f >= dot(dg, dg)))
			nKept = 0;
	}
	int nAnch = nKept;
	if (nKept != 2)
	{
		f3 wa0 = mk(0, 0, 0), wa1 = mk(0, 0, 0);
		nAnch = 0;
		if (nKept == 1)
		{
			wa0 = xtrans(f0, pa0[0]);
			nAnch = 1;
		}
		float pd2 = 0.0f;
		const float thr = frictionOffsetThreshold + restDist;
#pragma unroll
		for (int j = 0; j < 4; j++)
		{
			if (j >= cnt || !(cs[j] < thr))
				continue;
			const f3 wp = cp[j];
			if (nAnch == 0) { wa0 = wp; nAnch = 1; }
			else if (nAnch == 1)
			{
				const f3 d = wp - wa0;
				pd2 = dot(d, d);
				if (pd2 > 1e-8f) { wa1 = wp; nAnch = 2; }
			}
			else
			{
				const f3 e0 = wp - wa0, e1 = wp - wa1;
				const float d0 = dot(e0, e0), d1 = dot(e1, e1);
				if (d0 > d1) { if (d0 > pd2) { wa1 = wp; pd2 = d0; } }
				else if (d1 > pd2) { wa0 = wp; pd2 = d1; }
			}
		}
		if (nKept == 0 && nAnch > 0)
		{
			pa0[0] = xtransinv(f0, wa0);
			pa1[0] = xtransinv(f1, wa0);
		}
		if (nAnch == 2)
		{
			pa0[1] = xtransinv(f0, wa1);
			pa1[1] = xtransinv(f1, wa1);
		}
		if (nAnch == 0)
		{
			pa0[0] = mk(0, 0, 0);
			pa1[0] = pa0[0];
		}
		if (nAnch < 2)
		{
			pa0[1] = mk(0, 0, 0);
			pa1[1] = pa0[1];
		}
	}
	io.curKey[o] = pkey;
	io.curColor[o] = io.conColor[c];
	io.cur[6 * int64_t(o) + 0] = f4(pn0, __int_as_float(nAnch));
	io.cur[6 * int64_t(o) + 1] = f4(pn1, 0.0f);
	io.cur[6 * int64_t(o) + 2] = f4(pa0[0], 0.0f);
	io.cur[6 * int64_t(o) + 3] = f4(pa0[1], 0.0f);
	io.cur[6 * int64_t(o) + 4] = f4(pa1[0], 0.0f);
	io.cur[6 * int64_t(o) + 5] = f4(pa1[1], 0.0f);
	return nAnch;
}

PXH_D void prepBody(int o, int C, const int* order, const float4* ctN, const float4* ctP, const float4* rec,
                    float invStepDt, float scale, float restDist, float frictionOffsetThreshold, Rows& rows,
                    const PatchIO& io, uint32_t& nCntOut, uint32_t& nDynOut, uint32_t& nFricOut);

// Per-block sums of four per-thread counts (256-thread blocks) stored at
// partial[4 * block]: no atomics on shared counters from every wave (with
// thousands of waves those serialise); k_sum_counters adds the blocks up.
PXH_D void blockCounters4(uint32_t v0, uint32_t v1, uint32_t v2, uint32_t v3, unsigned long long* partial)
{
	__shared__ uint32_t red[4][4];
	const uint32_t s0 = waveInclScan(v0), s1 = waveInclScan(v1), s2 = waveInclScan(v2), s3 = waveInclScan(v3);
	const int w = threadIdx.x >> 6;
	if ((threadIdx.x & 63) == 63)
	{
		red[w][0] = s0; red[w][1] = s1; red[w][2] = s2; red[w][3] = s3;
	}
	__syncthreads();
	if (threadIdx.x < 4)
	{
		unsigned long long t = 0;
		for (int k = 0; k < int(blockDim.x >> 6); k++)
			t += red[k][threadIdx.x];
		partial[4 * int64_t(blockIdx.x) + threadIdx.x] = t;
	}
}

// counters[k] = sum over blocks of partial[4 * block + k] (one block)
__global__ void __launch_bounds__(256) k_sum_counters(int nBlocks, const unsigned long long* partial,
                                                      unsigned long long* counters)
{
	__shared__ unsigned long long red[4][256];
	unsigned long long t[4] = {0, 0, 0, 0};
	for (int b = threadIdx.x; b < nBlocks; b += blockDim.x)
		for (int k = 0; k < 4; k++)
			t[k] += partial[4 * int64_t(b) + k];
	for (int k = 0; k < 4; k++)
		red[k][threadIdx.x] = t[k];
	__syncthreads();
	for (int o = 128; o > 0; o >>= 1)
	{
		if (threadIdx.x < o)
			for (int k = 0; k < 4; k++)
				red[k][threadIdx.x] += red[k][threadIdx.x + o];
		__syncthreads();
	}
	if (threadIdx.x < 4)
		counters[threadIdx.x] = red[threadIdx.x][0];
}

// Contact rows of one constraint at its colour-ordered position o
// (setupFinalizeSolverConstraints / constructContactConstraintStep,
//  lowleveldynamics/src/DyTGSContactPrep.cpp:310-404, 426-812; friction patches
//  getFrictionPatches / correlatePatches / growPatches, DyContactPrepShared.h:53-127,
//  DyFrictionCorrelation.cpp:136-316)
__global__ void k_prep(int C, const int* order, const float4* ctN, const float4* ctP, const float4* rec,
                       float invStepDt, float scale, float restDist, float frictionOffsetThreshold, Rows rows,
                       PatchIO io, unsigned long long* counters)
{
	const int o = blockIdx.x * blockDim.x + threadIdx.x;
	// per-step counters: contact points, friction rows, dynamic-dynamic constraints
	uint32_t myCnt = 0, myFric = 0, myDyn = 0;
	prepBody(o, C, order, ctN, ctP, rec, invStepDt, scale, restDist, frictionOffsetThreshold, rows, io, myCnt, myDyn,
	         myFric);
	blockCounters4(myCnt, myFric, myDyn, myDyn ? myFric : 0u, counters);
}

PXH_D void prepBody(int o, int C, const int* order, const float4* ctN, const float4* ctP, const float4* rec,
                    float invStepDt, float scale, float restDist, float frictionOffsetThreshold, Rows& rows,
                    const PatchIO& io, uint32_t& nCntOut, uint32_t& nDynOut, uint32_t& nFricOut)
{
	if (o >= C)
		return;
	const int c = order[o];
	const int4 cr = io.conRec[2 * int64_t(c)], ck = io.conRec[2 * int64_t(c) + 1];
	const int a = cr.x, b = cr.y, slot = cr.z, po = cr.w;
	const uint64_t pkey = (uint64_t(uint32_t(ck.y)) << 32) | uint32_t(ck.x);
	const float4 nn = ctN[slot];
	const int cnt = __float_as_int(nn.w);
	const f3 n = mk(nn);
	const bool dynB = b >= 0;
	nCntOut = uint32_t(cnt);
	nDynOut = dynB ? 1u : 0u;
	const float4* ra4 = rec + PREP_REC * int64_t(a);
	const float4 pa4 = ra4[0];
	const m33 Sa = loadSym(ra4[2], ra4[3]);
	const f3 linA = mk(ra4[4]);
	m33 Sb;
	Sb.c0 = mk(0, 0, 0); Sb.c1 = Sb.c0; Sb.c2 = Sb.c0;
	float invMassB = 0.0f;
	xf f0, f1;
	f0.p = mk(pa4); f0.q = mkq(ra4[1]);
	f1.p = mk(0, 0, 0); f1.q.x = 0; f1.q.y = 0; f1.q.z = 0; f1.q.w = 1;
	f3 linB = mk(0, 0, 0);
	if (dynB)
	{
		const float4* rb4 = rec + PREP_REC * int64_t(b);
		const float4 pb4 = rb4[0];
		Sb = loadSym(rb4[2], rb4[3]);
		invMassB = pb4.w;
		f1.p = mk(pb4); f1.q = mkq(rb4[1]);
		linB = mk(rb4[4]);
	}
	const float invMassA = pa4.w;
	const float nlen2 = dot(n, n);
	const float imn0 = invMassA * nlen2, imn1 = -invMassB * nlen2;
	const float invDtp8 = invStepDt * scale;
	// loops run to the fixed bound 4 with guards so the point arrays stay in
	// registers (a loop to cnt would index them dynamically, in scratch)
	f3 cp[4];
	float cs[4];
#pragma unroll
	for (int k = 0; k < 4; k++)
	{
		cp[k] = mk(0, 0, 0);
		cs[k] = 0.0f;
		if (k >= cnt)
			continue;
		const float4 q = ctP[4 * int64_t(slot) + k];
		cp[k] = mk(q);
		cs[k] = q.w;
		const f3 ra = cp[k] - f0.p, rb = cp[k] - f1.p;
		const f3 raXnI = mmul(Sa, cross(ra, n)), rbXnI = mmul(Sb, cross(rb, n));
		const float unit = (imn0 + dot(raXnI, raXnI)) + (dot(rbXnI, rbXnI) - imn1);
		const float pen = q.w - restDist;
		const float recip = unit > 0.0f ? 1.0f / unit : 0.0f;
		rows.nA[k * int64_t(C) + o] = f4(raXnI, pen);
		// the bias coefficient is -invStepDt for a separated point, else -invStepDt*scale:
		// the sign of the stored reciprocal response carries that choice
		rows.nB[k * int64_t(C) + o] = f4(rbXnI, pen > 0.0f ? -recip : recip);
		rows.nF[k * int64_t(C) + o] = 0.0f;
	}
	f3 pa0[2], pa1[2];
	const int nAnch =
	    frictionPatch(o, c, po, pkey, n, f0, f1, cp, cs, cnt, restDist, frictionOffsetThreshold, io, pa0, pa1);
	nFricOut = uint32_t(2 * nAnch);
	(void)invDtp8;
	rows.hI[o] = make_int4(a, b, cnt | ((2 * nAnch) << 8), 0);
	rows.hF[o] = make_float4(n.x, n.y, n.z, 0.0f);
	if (nAnch == 0)
		return;
	const f3 lvr = linA - linB;
	const f3 fb = (0.70710678f > fabsf(n.x)) ? mk(0.0f, -n.z, n.y) : mk(-n.y, n.x, 0.0f);
	f3 t0 = lvr - n * dot(n, lvr);
	t0 = dot(t0, t0) > 0.0001f ? t0 : fb;
	t0 = normalize(t0);
	const f3 t1 = normalize(cross(n, t0));
	const f3 relTr = f0.p - f1.p;
#pragma unroll
	for (int j = 0; j < 2; j++)
	{
		if (j >= nAnch)
			break;
		const f3 ra = qrot(f0.q, pa0[j]), rb = qrot(f1.q, pa1[j]);
		const f3 err = (ra - rb) + relTr;
		for (int d = 0; d < 2; d++)
		{
			const f3 t = d == 0 ? t0 : t1;
			const f3 raXnI = mmul(Sa, cross(ra, t)), rbXnI = mmul(Sb, cross(rb, t));
			const float unit = (imn0 + dot(raXnI, raXnI)) + (dot(rbXnI, rbXnI) - imn1);
			const int r = 2 * j + d;
			rows.fT[r * int64_t(C) + o] = f4(t, dot(err, t));
			rows.fA[r * int64_t(C) + o] = f4(raXnI, unit > 0.0f ? scale / unit : 0.0f);
			if (dynB)
				rows.fB[r * int64_t(C) + o] = f4(rbXnI, 0.0f);
			rows.fF[r * int64_t(C) + o] = 0.0f;
		}
	}
}

// one colour: each lane solves one constraint (solveContact /
// solveDynamicContactsStep, lowleveldynamics/src/DyTGSContactPrep.cpp:1490-1843);
// 64-lane blocks spread a colour over all CUs. A short colour is bound by its
// chain: arguments, row header, rows and bodies together, some 700 instructions
// of one wave, stores. So all arguments come before anything depends on them,
// and the rows' loads are issued ahead of the bodies': a colour of 4,400 rows
// took 5.9 us with the bodies first and an early exit, and takes 4.7 (the step
// of a 20,011-body bin 1.43 -> 1.22 ms; 262,144 bodies 3.60 -> 3.49).
constexpr int SOLVE_THREADS = 64;

// Body velocity records: the scene's array, or a world's records
// in LDS, whose first body is `base`).
struct VelPlain
{
	float4* v;
	int base;
	PXH_D void load(int body, float4 (&r)[4]) const
	{
		const float4* p = v + 4 * int64_t(body - base);
		r[0] = p[0]; r[1] = p[1]; r[2] = p[2]; r[3] = p[3];
	}
	PXH_D void store(int body, float4 lin, float4 ang) const
	{
		float4* p = v + 4 * int64_t(body - base);
		p[0] = lin;
		p[1] = ang;
	}
	// the substeps' summed linear and angular motion
	PXH_D void storeMoved(int body, float4 lin, float4 ang) const
	{
		float4* p = v + 4 * int64_t(body - base);
		p[2] = lin;
		p[3] = ang;
	}
};

// with the bodies' turn over the substeps, which the joint rows read
struct VelTurn : VelPlain
{
	const float4* dq;
	PXH_D float4 turn(int body) const { return dq[body]; }
};

// one TGS contact row's data but for its bodies
struct TgsRow
{
	int4 hi;
	float4 hf;
	float4 nA[4], nB[4], fT[4], fA[4], fB[4];
	float nFc[4], fFc[4];
};
PXH_D void loadTgsRow(int o, int C, const Rows& rows, TgsRow& r)
{
	r.hi = rows.hI[o];
	r.hf = rows.hF[o];
	const int cnt = r.hi.z & 0xFF, nF = r.hi.z >> 8;
	const bool dynB = r.hi.y >= 0;
#pragma unroll
	for (int k = 0; k < 4; k++)
	{
		const int64_t ri = k * int64_t(C) + o;
		if (k < cnt)
		{
			r.nA[k] = rows.nA[ri]; r.nB[k] = rows.nB[ri]; r.nFc[k] = rows.nF[ri];
		}
		if (k < nF)
		{
			r.fT[k] = rows.fT[ri]; r.fA[k] = rows.fA[ri]; r.fFc[k] = rows.fF[ri];
			r.fB[k] = dynB ? rows.fB[ri] : make_float4(0, 0, 0, 0);
		}
	}
}

// One TGS contact row o; the arithmetic is the same wherever the velocity
// records are.
template <class Vel>
__device__ __forceinline__ void solveTgsRow(int o, int C, const Rows& rows, TgsRow& row, const Vel& vel, float minPen,
                                            float muS, float muD, float invStepDt, float biasScale, float scale,
                                            uint32_t* broken)
{
	const int4 hi = row.hi;
	const float4 hf = row.hf;
	const int cnt = hi.z & 0xFF, nF = hi.z >> 8;
	const bool dynB = hi.y >= 0;
	float4 va[4], vb[4];
	vel.load(hi.x, va);
	if (dynB)
		vel.load(hi.y, vb);
	else
		vb[0] = vb[1] = vb[2] = vb[3] = make_float4(0, 0, 0, 0);
	const float4 la4 = va[0], aa4 = va[1], dla4 = va[2], am04 = va[3];
	const float4 lb4 = vb[0], ab4 = vb[1], dlb4 = vb[2], am14 = vb[3];
	const float4(&nA)[4] = row.nA, (&nB)[4] = row.nB, (&fT)[4] = row.fT, (&fA)[4] = row.fA, (&fB)[4] = row.fB;
	float(&nFc)[4] = row.nFc, (&fFc)[4] = row.fFc;
	const f3 n = mk(hf);
	const float invMassA = la4.w, invMassB = lb4.w;
	f3 l0 = mk(la4), a0 = mk(aa4), l1 = mk(lb4), a1 = mk(ab4);
	const f3 am0 = mk(am04), am1 = mk(am14);
	const f3 rel = mk(dla4) - mk(dlb4);
	const f3 nim0 = n * invMassA, nim1 = n * invMassB;
	const float dv = dot(rel, n);
	const float biasSep = -invStepDt, biasPen = -invStepDt * scale;
	float acc = 0.0f;
#pragma unroll
	for (int k = 0; k < 4; k++)
	{
		if (k >= cnt)
			break;
		const f3 raXnI = mk(nA[k]), rbXnI = mk(nB[k]);
		const float rs = nB[k].w;
		const float recip = fabsf(rs);
		const float biasCoef = rs < 0.0f ? biasSep : biasPen;
		const float dang = dot(am0, raXnI) - dot(am1, rbXnI);
		const float sep = fmaxf(minPen, nA[k].w + (dv + dang));
		const float bias = fminf(1e32f, biasCoef * sep);
		const f3 v0 = mulv(l0, n) + mulv(a0, raXnI);
		const f3 v1 = mulv(l1, n) + mulv(a1, rbXnI);
		const f3 dvv = v0 - v1;
		const float nv = dvv.x + dvv.y + dvv.z;
		const float lambda = bias * recip - nv * recip;
		const float af = nFc[k];
		const float nf = fminf(af + fmaxf(lambda, -af), 1e32f);
		const float df = nf - af;
		l0 = nim0 * df + l0;
		l1 = l1 - nim1 * df;
		a0 = raXnI * df + a0;
		a1 = a1 - rbXnI * df;
		nFc[k] = nf;
		acc = acc + nf;
	}
	bool anyClamp = false;
	if (nF)
	{
		const float maxF = muS * acc, maxD = muD * acc;
		const float fscale = nF == 4 ? 0.5f : 1.0f;
#pragma unroll
		for (int i = 0; i < 4; i += 2)
		{
			if (i >= nF)
				break;
			float ti[2];
#pragma unroll
			for (int d = 0; d < 2; d++)
			{
				const f3 t = mk(fT[i + d]), raI = mk(fA[i + d]), rbI = mk(fB[i + d]);
				const float dvf = (dot(raI, am0) - dot(rbI, am1)) + dot(t, rel);
				const float bias = (fT[i + d].w + dvf) * biasScale;
				const f3 v0 = mulv(l0, t) + mulv(a0, raI);
				const f3 v1 = mulv(l1, t) + mulv(a1, rbI);
				const f3 dd = v0 - v1;
				const float nv = dd.x + dd.y + dd.z;
				const float vm = fA[i + d].w;
				ti[d] = (fFc[i + d] - bias * vm) - nv * vm;
			}
			const float tot = sqrtf(ti[0] * ti[0] + ti[1] * ti[1]);
			const bool clamp = tot > fscale * maxF;
			const float tc = clamp ? fminf(fscale * maxD, tot) : tot;
			const float ratio = tot > 0.0f ? tc / tot : 0.0f;
			const float n0 = ti[0] * ratio, n1 = ti[1] * ratio;
			const float d0 = n0 - fFc[i], d1 = n1 - fFc[i + 1];
			const f3 t0 = mk(fT[i]), t1 = mk(fT[i + 1]);
			l0 = (t0 * invMassA) * d0 + ((t1 * invMassA) * d1 + l0);
			l1 = (l1 - (t1 * invMassB) * d1) - (t0 * invMassB) * d0;
			a0 = mk(fA[i]) * d0 + (mk(fA[i + 1]) * d1 + a0);
			a1 = (a1 - mk(fB[i + 1]) * d1) - mk(fB[i]) * d0;
			fFc[i] = n0;
			fFc[i + 1] = n1;
			anyClamp |= clamp;
		}
	}
	// the broken flag of the friction patch is the last pass's clamp state
	// (DyTGSContactPrep.cpp:1837, 1907)
	if (broken)
		broken[o] = anyClamp ? 1u : 0u;
#pragma unroll
	for (int k = 0; k < 4; k++)
	{
		const int64_t ri = k * int64_t(C) + o;
		if (k < cnt)
			rows.nF[ri] = nFc[k];
		if (k < nF)
			rows.fF[ri] = fFc[k];
	}
	vel.store(hi.x, f4(l0, invMassA), f4(a0, 0.0f));
	if (dynB)
		vel.store(hi.y, f4(l1, invMassB), f4(a1, 0.0f));
}

__global__ void __launch_bounds__(SOLVE_THREADS) k_solve(int begin, int end, int C, Rows rows, float4* vel,
                                                          float minPen, float muS, float muD, float invStepDt,
                                                          float biasScale, float scale, uint32_t* broken)
{
	// lanes past the colour's end load its last row and leave after the loads, so
	// the kernel's arguments come in one scalar load before the first row's
	const int own = begin + blockIdx.x * SOLVE_THREADS + threadIdx.x;
	const int o = min(own, end - 1);
	TgsRow row;
	loadTgsRow(o, C, rows, row);
	if (own >= end)
		return;
	solveTgsRow(o, C, rows, row, VelPlain{vel, 0}, minPen, muS, muD, invStepDt, biasScale, scale, broken);
}

// ---------------------------------------------------------------------------
// PGS (DynamicsContext, lowleveldynamics/src/DyDynamics.cpp; DySolverControl.cpp)
// Rows (PGS use): hI.w = dynamic friction (scaled for the anchor count, float
// bits), hF.w = static friction (scaled); nA = raXnI | biased error; nB =
// rbXnI | velocity multiplier; unbiased error in its own array; fT = t |
// bias - target velocity; fA = raXnI | velocity multiplier; fB = rbXnI |
// -target velocity.
// ---------------------------------------------------------------------------

// setupFinalizeSolverConstraints (lowleveldynamics/src/DyContactPrep.cpp:49-357)
// with constructContactConstraint (DyContactPrepShared.h:298-393)
__global__ void k_prep_pgs(int C, const int* order, const float4* ctN, const float4* ctP, const float4* rec,
                           float invDt, float muS,
                           float muD, float restDist, float frictionOffsetThreshold, Rows rows, float* rowsU,
                           PatchIO io, unsigned long long* counters)
{
	const int o = blockIdx.x * blockDim.x + threadIdx.x;
	uint32_t myCnt = 0, myFric = 0, myDyn = 0;
	if (o < C)
	{
		const int c = order[o];
		const int4 cr = io.conRec[2 * int64_t(c)], ck = io.conRec[2 * int64_t(c) + 1];
		const int a = cr.x, b = cr.y, slot = cr.z, po = cr.w;
		const uint64_t pkey = (uint64_t(uint32_t(ck.y)) << 32) | uint32_t(ck.x);
		const float4 nn = ctN[slot];
		const int cnt = __float_as_int(nn.w);
		const f3 n = mk(nn);
		const bool dynB = b >= 0;
		myCnt = uint32_t(cnt);
		myDyn = dynB ? 1u : 0u;
		const float4* ra4 = rec + PREP_REC * int64_t(a);
		const float4 pa4 = ra4[0];
		const m33 Sa = loadSym(ra4[2], ra4[3]);
		m33 Sb;
		Sb.c0 = mk(0, 0, 0); Sb.c1 = Sb.c0; Sb.c2 = Sb.c0;
		xf f0, f1;
		f0.p = mk(pa4); f0.q = mkq(ra4[1]);
		f1.p = mk(0, 0, 0); f1.q.x = 0; f1.q.y = 0; f1.q.z = 0; f1.q.w = 1;
		const float invMassA = pa4.w;
		const f3 v0 = mk(ra4[4]), w0 = mk(ra4[5]);
		float invMassB = 0.0f;
		f3 v1 = mk(0, 0, 0), w1 = mk(0, 0, 0);
		if (dynB)
		{
			const float4* rb4 = rec + PREP_REC * int64_t(b);
			const float4 pb4 = rb4[0];
			Sb = loadSym(rb4[2], rb4[3]);
			invMassB = pb4.w;
			v1 = mk(rb4[4]);
			w1 = mk(rb4[5]);
			f1.p = mk(pb4); f1.q = mkq(rb4[1]);
		}
		const float nl2 = dot(n, n);
		const float imn0 = invMassA * nl2, imn1 = -invMassB * nl2;
		const float invDtp8 = invDt * 0.8f;
		const float norVel = (n.x * v0.x - n.x * v1.x) + (n.y * v0.y - n.y * v1.y) + (n.z * v0.z - n.z * v1.z);
		f3 cp[4];
		float cs[4];
#pragma unroll
		for (int k = 0; k < 4; k++)
		{
			cp[k] = mk(0, 0, 0);
			cs[k] = 0.0f;
			if (k >= cnt)
				continue;
			const float4 q = ctP[4 * int64_t(slot) + k];
			cp[k] = mk(q);
			cs[k] = q.w;
			const f3 ra = cp[k] - f0.p, rb = cp[k] - f1.p;
			const f3 raXn = cross(ra, n), rbXn = cross(rb, n);
			const float vrel = norVel + (dot(raXn, w0) - dot(rbXn, w1));
			const f3 raXnI = mmul(Sa, raXn), rbXnI = mmul(Sb, rbXn);
			const float unit = (imn0 + dot(raXnI, raXnI)) + (dot(rbXnI, rbXnI) - imn1);
			const float pen = q.w - restDist;
			const float target = 0.0f - vrel;
			const float recip = unit > 0.0f ? 1.0f / unit : 0.0f;
			const float penScaled = pen >= 0.0f ? pen * invDt : pen * invDtp8;
			const float scaledBias = recip * fmaxf(-1e32f, penScaled);
			const int64_t ri = k * int64_t(C) + o;
			rows.nA[ri] = f4(raXnI, target * recip + -scaledBias);
			rows.nB[ri] = f4(rbXnI, recip);
			rowsU[ri] = target * recip + -fmaxf(scaledBias, 0.0f);
			rows.nF[ri] = 0.0f;
		}
		f3 pa0[2], pa1[2];
		const int nAnch =
		    frictionPatch(o, c, po, pkey, n, f0, f1, cp, cs, cnt, restDist, frictionOffsetThreshold, io, pa0, pa1);
		myFric = uint32_t(2 * nAnch);
		const float fc = nAnch == 2 ? 0.5f : 1.0f;
		rows.hI[o] = make_int4(a, b, cnt | ((2 * nAnch) << 8), __float_as_int(muD * fc));
		rows.hF[o] = make_float4(n.x, n.y, n.z, muS * fc);
		if (nAnch > 0)
		{
			const f3 lvr = v0 - v1;
			const f3 fb = (0.70710678f > fabsf(n.x)) ? mk(0.0f, -n.z, n.y) : mk(-n.y, n.x, 0.0f);
			f3 t0 = lvr - n * dot(n, lvr);
			t0 = dot(t0, t0) > 0.0001f ? t0 : fb;
			t0 = normalize(t0);
			const f3 t1 = cross(n, t0);
#pragma unroll
			for (int j = 0; j < 2; j++)
			{
				if (j >= nAnch)
					break;
				const f3 ra = qrot(f0.q, pa0[j]), rb = qrot(f1.q, pa1[j]);
				const f3 err = (ra + f0.p) - (rb + f1.p);
#pragma unroll
				for (int d = 0; d < 2; d++)
				{
					const f3 t = d == 0 ? t0 : t1;
					const f3 raXn = cross(ra, t), rbXn = cross(rb, t);
					const f3 raXnI = mmul(Sa, raXn), rbXnI = mmul(Sb, rbXn);
					const float resp = (invMassA + dot(raXnI, raXnI)) + (dot(rbXnI, rbXnI) - -invMassB);
					const float vrel = (dot(t, v0) + dot(raXn, w0)) - (dot(t, v1) + dot(rbXn, w1));
					const float target = 0.0f - vrel;
					const float bias = dot(t, err) * invDt;
					const int64_t ri = (2 * j + d) * int64_t(C) + o;
					rows.fT[ri] = f4(t, bias - target);
					rows.fA[ri] = f4(raXnI, resp > 0.0f ? 0.8f / resp : 0.0f);
					rows.fB[ri] = f4(rbXnI, 0.0f - target);
					rows.fF[ri] = 0.0f;
				}
			}
		}
	}
	blockCounters4(myCnt, myFric, myDyn, myDyn ? myFric : 0u, counters);
}

// one colour of PGS (solveContact, lowleveldynamics/src/DySolverConstraints.cpp:221-371;
// normal rows solveDynamicContacts, DySolverConstraintsShared.h:49-105) on the
// velocity changes in vel[4i], vel[4i+1]. velocityPass: rows concluded after the
// last position pass use their unbiased error and friction without bias
// (concludeContact, DySolverConstraints.cpp:508-549).
struct PgsRow
{
	int4 hi;
	float4 hf;
	float4 nA[4], nB[4], fT[4], fA[4], fB[4];
	float nFc[4], fFc[4], err[4];
};
PXH_D void loadPgsRow(int o, int C, const Rows& rows, const float* rowsU, bool doFriction, bool velocityPass, PgsRow& r)
{
	r.hi = rows.hI[o];
	r.hf = rows.hF[o];
	const int cnt = r.hi.z & 0xFF, nF = doFriction ? r.hi.z >> 8 : 0;
#pragma unroll
	for (int k = 0; k < 4; k++)
	{
		const int64_t ri = k * int64_t(C) + o;
		if (k < cnt)
		{
			r.nA[k] = rows.nA[ri]; r.nB[k] = rows.nB[ri]; r.nFc[k] = rows.nF[ri];
			r.err[k] = velocityPass ? rowsU[ri] : r.nA[k].w;
		}
		if (k < nF)
		{
			r.fT[k] = rows.fT[ri]; r.fA[k] = rows.fA[ri]; r.fB[k] = rows.fB[ri]; r.fFc[k] = rows.fF[ri];
		}
	}
}

// (only the first half of a record is used: the compiler drops the other loads)
template <class Vel>
__device__ __forceinline__ void solvePgsRow(int o, int C, const Rows& rows, PgsRow& row, const Vel& vel,
                                            bool doFriction, bool velocityPass, uint32_t* broken)
{
	const int4 hi = row.hi;
	const float4 hf = row.hf;
	const int cnt = hi.z & 0xFF, nF = doFriction ? hi.z >> 8 : 0;
	const bool dynB = hi.y >= 0;
	float4 va[4], vb[4];
	vel.load(hi.x, va);
	if (dynB)
		vel.load(hi.y, vb);
	else
		vb[0] = vb[1] = make_float4(0, 0, 0, 0);
	const float4 la4 = va[0], aa4 = va[1], lb4 = vb[0], ab4 = vb[1];
	const float4(&nA)[4] = row.nA, (&nB)[4] = row.nB, (&fT)[4] = row.fT, (&fA)[4] = row.fA, (&fB)[4] = row.fB;
	float(&nFc)[4] = row.nFc, (&fFc)[4] = row.fFc;
	const float(&err)[4] = row.err;
	const f3 n = mk(hf);
	const float invMassA = la4.w, invMassB = lb4.w;
	f3 l0 = mk(la4), a0 = mk(aa4), l1 = mk(lb4), a1 = mk(ab4);
	const f3 dl0 = n * invMassA, dl1 = n * invMassB;
	float acc = 0.0f;
#pragma unroll
	for (int k = 0; k < 4; k++)
	{
		if (k >= cnt)
			break;
		const f3 raXnI = mk(nA[k]), rbXnI = mk(nB[k]);
		const f3 v0 = mulv(l0, n) + mulv(a0, raXnI);
		const f3 v1 = mulv(l1, n) + mulv(a1, rbXnI);
		const f3 dv = v0 - v1;
		const float nv = dv.x + dv.y + dv.z;
		const float af = nFc[k];
		const float d0 = fmaxf(err[k] - nv * nB[k].w, -af);
		const float nf = fminf(af + d0, 1e32f);
		const float df = nf - af;
		l0 = dl0 * df + l0;
		l1 = l1 - dl1 * df;
		a0 = raXnI * df + a0;
		a1 = a1 - rbXnI * df;
		nFc[k] = nf;
		acc = acc + nf;
	}
	bool anyClamp = false;
	if (nF)
	{
		const float maxF = hf.w * acc, maxD = __int_as_float(hi.w) * acc;
#pragma unroll
		for (int r = 0; r < 4; r++)
		{
			if (r >= nF)
				break;
			const f3 t = mk(fT[r]), raI = mk(fA[r]), rbI = mk(fB[r]);
			const f3 v0 = mulv(l0, t) + mulv(a0, raI);
			const f3 v1 = mulv(l1, t) + mulv(a1, rbI);
			const f3 dv = v0 - v1;
			const float nv = dv.x + dv.y + dv.z;
			const float vm = fA[r].w;
			const float af = fFc[r];
			const float tmp = af - (velocityPass ? fB[r].w : fT[r].w) * vm;
			const float total = tmp - nv * vm;
			const bool clamp = fabsf(total) > maxF;
			const float tc = fminf(maxD, fmaxf(-maxD, total));
			const float nf = clamp ? tc : total;
			anyClamp |= clamp;
			const float df = nf - af;
			l0 = (t * invMassA) * df + l0;
			l1 = l1 - (t * invMassB) * df;
			a0 = raI * df + a0;
			a1 = a1 - rbI * df;
			fFc[r] = nf;
		}
	}
	if (broken)
		broken[o] = anyClamp ? 1u : 0u;
#pragma unroll
	for (int k = 0; k < 4; k++)
	{
		const int64_t ri = k * int64_t(C) + o;
		if (k < cnt)
			rows.nF[ri] = nFc[k];
		if (k < nF)
			rows.fF[ri] = fFc[k];
	}
	vel.store(hi.x, f4(l0, invMassA), f4(a0, 0.0f));
	if (dynB)
		vel.store(hi.y, f4(l1, invMassB), f4(a1, 0.0f));
}

__global__ void __launch_bounds__(SOLVE_THREADS) k_solve_pgs(int begin, int end, int C, Rows rows,
                                                              const float* rowsU, float4* vel, int doFriction,
                                                              int velocityPass, uint32_t* broken)
{
	const int own = begin + blockIdx.x * SOLVE_THREADS + threadIdx.x;
	const int o = min(own, end - 1);
	PgsRow row;
	loadPgsRow(o, C, rows, rowsU, doFriction != 0, velocityPass != 0, row);
	if (own >= end)
		return;
	solvePgsRow(o, C, rows, row, VelPlain{vel, 0}, doFriction != 0, velocityPass != 0, broken);
}

// velocity changes after the position passes move the bodies (saveMotionVelocities,
// lowleveldynamics/src/DySolverCore.cpp:40-55)
__global__ void k_pgs_save_motion(int n, const float4* vel, float4* motionLin, float4* motionAng)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	motionLin[i] = vel[4 * int64_t(i)];
	motionAng[i] = vel[4 * int64_t(i) + 1];
}

// updateWakeCounter without stabilization and the readiness it reports
// (lowleveldynamics/src/DySleep.cpp:173-235) for body i after its step: ml,
// ma its motion velocities (world frame), q its new orientation, invMass and
// invI (mass-space inverse inertia) its mass properties
PXH_D void sleepCheck(const SleepState& ss, int i, float dt, f3 ml, f3 ma, qt q, float invMass, float4 invI)
{
	const float resetTime = 20.0f * 0.02f;
	float wc = ss.wc[i];
	if (wc < resetTime * 0.5f || wc < dt)
	{
		const f3 I = mk(invI.x > 0.0f ? 1.0f / invI.x : 1.0f, invI.y > 0.0f ? 1.0f / invI.y : 1.0f,
		                invI.z > 0.0f ? 1.0f / invI.z : 1.0f);
		const f3 l = mk(ss.accL[i]) + ml;
		const f3 a = mk(ss.accA[i]) + qrotinv(q, ma);
		const float im = invMass == 0.0f ? 1.0f : invMass;
		const float angular = (a.x * a.x * I.x + a.y * a.y * I.y + a.z * a.z * I.z) * im;
		const float linear = l.x * l.x + l.y * l.y + l.z * l.z;
		const float energy = 0.5f * (angular + linear);
		const float cluster = float(1 + ss.counted[i]);
		const float threshold = cluster * ss.threshold;
		if (energy >= threshold)
		{
			// woken by its own motion: filter reset, new wake counter; from a
			// zero counter (eACTIVATE_THIS_FRAME) no longer ready for sleep
			ss.accL[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
			ss.accA[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
			const float factor = threshold == 0.0f ? 2.0f : fminf(energy / threshold, 2.0f);
			ss.wc[i] = factor * 0.5f * resetTime + dt * (cluster - 1.0f);
			if (wc == 0.0f)
				ss.flags[i] &= ~SLEEP_READY;
			return;
		}
		ss.accL[i] = f4(l, 0.0f);
		ss.accA[i] = f4(a, 0.0f);
	}
	wc = fmaxf(wc - dt, 0.0f);
	ss.wc[i] = wc;
	if (wc == 0.0f)
	{
		// eDEACTIVATE_THIS_FRAME: ready for sleep, filter reset
		ss.flags[i] |= SLEEP_READY;
		ss.accL[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		ss.accA[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	}
}

// integrateCore (lowleveldynamics/src/DyBodyCoreIntegrator.h:83-175): poses
// from the motion velocities, body velocities from the final changes; the
// sleep check on the motion velocities (DyDynamics.cpp:1403-1420)
__global__ void k_pgs_finalize(int n, float dt, float4* pos, float4* rot, float4* lin, float4* ang,
                               const float4* invI, const float4* vel, const float4* motionLin,
                               const float4* motionAng, const float4* svI0, const float4* svI1, SleepState ss)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	if (ss.flags && (ss.flags[i] & SLEEP_ASLEEP))
		return;   // sleeping: pose and zero velocities kept
	const float4* v = vel + 4 * int64_t(i);
	const f3 vD = mk(v[2]), wD = mk(v[3]);
	const m33 S = loadSym(svI0[i], svI1[i]);
	const f3 lm = vD + mk(motionLin[i]);
	pos[i] = f4(mk(pos[i]) + lm * dt, pos[i].w);
	f3 am = wD + mmul(S, mk(motionAng[i]));
	float w = dot(am, am);
	if (w != 0.0f)
	{
		w = sqrtf(w);
		if (w > 1e7f)
		{
			am = normalize(am) * 1e7f;
			w = 1e7f;
		}
		const float hv = dt * w * 0.5f;
		float s, c;
		sincosf(hv, &s, &c);
		s /= w;
		const f3 pqr = am * s;
		qt qv; qv.x = pqr.x; qv.y = pqr.y; qv.z = pqr.z; qv.w = 0.0f;
		const qt q0 = mkq(rot[i]);
		qt res = qmul(qv, q0);
		res.x += q0.x * c; res.y += q0.y * c; res.z += q0.z * c; res.w += q0.w * c;
		rot[i] = f4(qnormalize(res));
	}
	const float4 l = v[0];
	lin[i] = f4(vD + mk(l), l.w);
	ang[i] = f4(wD + mmul(S, mk(v[1])), 0.0f);
	if (ss.flags)
		sleepCheck(ss, i, dt, lm, am, mkq(rot[i]), l.w, invI[i]);
}

// integrateCoreStep (lowleveldynamics/src/DyTGSDynamics.cpp:1403-1476) of
// body i
template <class Vel>
__device__ __forceinline__ void integrateBodyTGS(int i, float dt, const Vel& vel, float4* svP, float4* svDQ,
                                                 const float4* svI0, const float4* svI1)
{
	float4 v[4];
	vel.load(i, v);
	const f3 lv = mk(v[0]);
	const f3 av = mk(v[1]);
	const f3 delta = lv * dt;
	const f3 amv = mmul(loadSym(svI0[i], svI1[i]), av);
	const float w2 = dot(amv, amv);
	svP[i] = f4(mk(svP[i]) + delta, 0.0f);
	if (w2 != 0.0f)
	{
		const float w = sqrtf(w2);
		const float half = dt * w * 0.5f;
		float s, q;
		sincosf(half, &s, &q);
		s /= w;
		const f3 pqr = amv * s;
		qt qv; qv.x = pqr.x; qv.y = pqr.y; qv.z = pqr.z; qv.w = 0.0f;
		const qt dq = mkq(svDQ[i]);
		qt res = qmul(qv, dq);
		res.x += dq.x * q; res.y += dq.y * q; res.z += dq.z * q; res.w += dq.w * q;
		svDQ[i] = f4(qnormalize(res));
	}
	vel.storeMoved(i, f4(mk(v[2]) + delta, 0.0f), f4(mk(v[3]) + av * dt, 0.0f));
}

__global__ void k_integrate(int n, float dt, float4* vel, float4* svP, float4* svDQ, const float4* svI0,
                            const float4* svI1)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	integrateBodyTGS(i, dt, VelPlain{vel, 0}, svP, svDQ, svI0, svI1);
}

// ---------------------------------------------------------------------------
// joints (pxh_joint.h)
// ---------------------------------------------------------------------------
// jointed bodies do not collide (PxConstraintFlag::eCOLLISION_ENABLED is off
// by default, physx/include/PxConstraint.h): their pair slots lose their
// contacts before the constraint list is built
// Body-mesh narrowphase of one body of a world with a mesh in a lane (k-th of
// meshBody): candidate triangles through the mesh's tree (depth-first nodes,
// each with the index after its subtree), taken in triangle order, then the
// patches of pxh_mesh.h into slots slotBase + k * MESH_MAXP + patch (deepest
// first; empty slots count 0). More than MESH_MAX_TRIS candidates set
// *overflow and leave the body without mesh contacts.
PXH_D void meshContactsOf(int k, const int* meshBody, const int* world, const int4* worldMesh,
                                                MeshSet M, const float4* pos, const float4* rot, const float4* geom,
                                                HullSet hs, float cd, int slotBase, float4* ctN, float4* ctP,
                                                uint32_t* overflow)
{
	const int i = meshBody[k];
	const int base = slotBase + k * MESH_MAXP;
	for (int p = 0; p < MESH_MAXP; p++)
		ctN[base + p].w = __int_as_float(0);
	const int4 wm = worldMesh[world[i]];
	if (wm.x < 0)
		return;
	f3 mn, mx;
	shapeBounds(i, pos, rot, geom, hs, mn, mx);
	mn = mn - mk(cd, cd, cd);
	mx = mx + mk(cd, cd, cd);
	int idx[MESH_MAX_TRIS];
	int nc = 0;
	for (int nd = wm.x; nd < wm.x + wm.y;)
	{
		const float4 lo = M.nodeLo[nd], hi = M.nodeHi[nd];
		const int4 info = M.nodeInfo[nd];
		if (lo.x > mx.x || mn.x > hi.x || lo.y > mx.y || mn.y > hi.y || lo.z > mx.z || mn.z > hi.z)
		{
			nd = info.z;
			continue;
		}
		for (int j = 0; j < info.y; j++)
		{
			const int t = M.leafTri[info.x + j];
			const float4 tl = M.lo[t], th = M.hi[t];
			if (tl.x > mx.x || mn.x > th.x || tl.y > mx.y || mn.y > th.y || tl.z > mx.z || mn.z > th.z)
				continue;
			if (nc == MESH_MAX_TRIS)
			{
				atomicOr(overflow, 1u);
				return;
			}
			idx[nc++] = t;
		}
		nd++;
	}
	if (nc == 0)
		return;
	for (int a = 1; a < nc; a++)   // triangle order
	{
		const int x = idx[a];
		int b = a - 1;
		while (b >= 0 && idx[b] > x)
		{
			idx[b + 1] = idx[b];
			b--;
		}
		idx[b + 1] = x;
	}
	MPatches P;
	P.np = 0;
	const float4 g = geom[i];
	const int type = int(g.w);
	xf x;
	x.p = mk(pos[i]);
	x.q = mkq(rot[i]);
	if (type == GEOM_SPHERE || type == GEOM_CAPSULE)
	{
		MeshCache C;
		MeshDef def[MESH_MAX_TRIS];
		if (type == GEOM_SPHERE)
			meshSphere(M, idx, nc, x.p, g.x, cd, C, def, P);
		else
		{
			const f3 tmp = qrot(x.q, mk(1.0f, 0.0f, 0.0f)) * g.y;
			meshCapsule(M, idx, nc, x.p + tmp, x.p - tmp, x.p, g.x, cd, C, def, P);
		}
	}
	else
		meshPoly(M, idx, nc, type == GEOM_CONVEXMESH ? hullPoly(hs, int(g.x)) : boxPoly(mk(g.x, g.y, g.z)), x, cd, P);
	int order[MESH_NPATCH];
	for (int a = 0; a < P.np; a++)
	{
		int b = a - 1;
		while (b >= 0 && P.p[order[b]].maxPen > P.p[a].maxPen)
		{
			order[b + 1] = order[b];
			b--;
		}
		order[b + 1] = a;
	}
	const int keep = P.np < MESH_MAXP ? P.np : MESH_MAXP;
	for (int a = 0; a < keep; a++)
	{
		MPatch& q = P.p[order[a]];
		int cnt = meshReduce4(q.c, q.count, q.n);
		if (type == GEOM_SPHERE)
		{
			int d = 0;
			for (int j = 1; j < cnt; j++)
				if (q.c[d].s > q.c[j].s) d = j;
			q.c[0] = q.c[d];
			cnt = 1;
		}
		ctN[base + a] = f4(q.n, __int_as_float(cnt));
		for (int j = 0; j < cnt; j++)
			ctP[4 * int64_t(base + a) + j] = f4(q.c[j].p, q.c[j].s);
	}
}

// The same over a wave per body (pxh_mesh.h): every body but those a wave can't
// hold, which go to rest (a count, then their k).
__global__ void __launch_bounds__(64) k_np_mesh_wave(int nMB, const int* meshBody, const int* world,
                                                     const int4* worldMesh, MeshSet M, const float4* pos,
                                                     const float4* rot, const float4* geom, HullSet hs, float cd,
                                                     int slotBase, float4* ctN, float4* ctP, uint32_t* overflow,
                                                     uint32_t* rest)
{
	__shared__ MeshLds L;
	const int lane = threadIdx.x;
	for (int k = blockIdx.x; k < nMB; k += gridDim.x)
	{
		const int i = meshBody[k];
		const int base = slotBase + k * MESH_MAXP;
		const int4 wm = worldMesh[world[i]];
		int nc = 0;
		if (wm.x >= 0)
		{
			f3 mn, mx;
			shapeBounds(i, pos, rot, geom, hs, mn, mx);
			nc = meshCandidates(M, wm.x, wm.y, mn - mk(cd, cd, cd), mx + mk(cd, cd, cd), L, lane);
		}
		if (nc > MESH_MAX_TRIS)
		{
			if (lane == 0)
				atomicOr(overflow, 1u);
			nc = 0;
		}
		MeshWave P;
		P.init(lane);
		int type = GEOM_SPHERE;
		bool done = true;
		if (nc > 0)
		{
			const float4 g = geom[i];
			type = int(g.w);
			xf x;
			x.p = mk(pos[i]);
			x.q = mkq(rot[i]);
			if (type == GEOM_SPHERE || type == GEOM_CAPSULE)
			{
				const f3 tmp = qrot(x.q, mk(1.0f, 0.0f, 0.0f)) * g.y;
				done = nc <= 64;
				if (done && type == GEOM_SPHERE)
					meshRoundWave<false>(M, L.idx, nc, x.p, x.p, x.p, g.x, cd, lane, P);
				else if (done)
					meshRoundWave<true>(M, L.idx, nc, x.p + tmp, x.p - tmp, x.p, g.x, cd, lane, P);
			}
			else
				done = meshPolyWave(M, nc, type == GEOM_CONVEXMESH ? hullPoly(hs, int(g.x)) : boxPoly(mk(g.x, g.y, g.z)),
				                    x, cd, L, lane, P);
		}
		if (done)
		{
			// patches by their least separation, the first among equals
			int rank = 0;
			for (int j = 0; j < P.np; j++)
			{
				const float v = laneOf(P.maxPen, j * (MESH_PC + 1));
				rank += v < P.maxPen || (v == P.maxPen && j < P.patch);
			}
			const int keep = P.np < MESH_MAXP ? P.np : MESH_MAXP;
			for (int a = 0; a < MESH_MAXP; a++)
			{
				const uint64_t m = __ballot(a < keep && P.patch < P.np && rank == a);
				if (m == 0ull)
				{
					if (lane == 0)
						ctN[base + a].w = __int_as_float(0);
					continue;
				}
				const int l0 = firstLane(m);
				int cnt = P.reduce4(l0, laneOf(P.count, l0)), from = l0;
				if (type == GEOM_SPHERE)
				{
					for (int j = 1; j < cnt; j++)
						if (laneOf(P.s, from) > laneOf(P.s, l0 + j)) from = l0 + j;
					cnt = 1;
				}
				if (lane == l0)
					ctN[base + a] = f4(P.n, __int_as_float(cnt));
				if (lane >= from && lane < from + cnt)
					ctP[4 * int64_t(base + a) + lane - from] = f4(P.p, P.s);
			}
		}
		else if (lane == 0)
			rest[1 + atomicAdd(rest, 1u)] = uint32_t(k);
		waveSync();
	}
}

__global__ void __launch_bounds__(64) k_np_mesh_rest(const uint32_t* rest, const int* meshBody, const int* world,
                                                     const int4* worldMesh, MeshSet M, const float4* pos,
                                                     const float4* rot, const float4* geom, HullSet hs, float cd,
                                                     int slotBase, float4* ctN, float4* ctP, uint32_t* overflow)
{
	PXH_THIN_LOOP(q, rest[0])
		meshContactsOf(int(rest[1 + q]), meshBody, world, worldMesh, M, pos, rot, geom, hs, cd, slotBase, ctN, ctP,
		               overflow);
}

// whether the bodies of a pair are joined: its (lower, higher) key is among
// the sorted joint keys
PXH_D bool pairJointed(uint2 ab, const uint64_t* keys, int nKeys)
{
	const uint32_t lo = ab.x < ab.y ? ab.x : ab.y, hi = ab.x < ab.y ? ab.y : ab.x;
	const uint64_t k = (uint64_t(lo) << 32) | hi;
	int a = 0, b = nKeys;
	while (a < b)
	{
		const int m = (a + b) >> 1;
		if (keys[m] < k)
			a = m + 1;
		else
			b = m;
	}
	return a < nKeys && keys[a] == k;
}

__global__ void k_joint_filter(int cap, int Q, const uint32_t* dP, const uint2* pairs, const uint64_t* keys, int nKeys,
                               float4* ctN)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= cap || uint32_t(i) >= *dP)
		return;
	if (pairJointed(pairs[i], keys, nKeys))
		ctN[Q + i].w = __int_as_float(0);
}

// ---------------------------------------------------------------------------
// sleeping. The observable order of the reference CPU pipeline
// (simulationcontroller/src/ScPipeline.cpp:1472-1776, lowlevel/software/src/
// PxsIslandSim.cpp:1630-1720): the narrowphase runs on every pair; a touching
// pair of an awake and a sleeping body wakes the sleeping body's island; an
// island whose bodies were all ready for sleep after the last step sleeps
// before the solve; the solve and integration skip sleeping bodies.
// ---------------------------------------------------------------------------
PXH_D bool asleepBody(const uint32_t* flags, uint32_t i) { return (flags[i] & SLEEP_ASLEEP) != 0u; }

__global__ void k_sleep_count_init(int n, SleepState ss)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		ss.counted[i] = ss.jcount[i];   // each joint counts (BodySim::onConstraintAttach, ScBodySim.h:159)
}

// Interactions a body counts: broadphase pairs that are not filtered out
// (ScShapeInteraction.cpp:84-93, ScPipeline.cpp:1222-1228) and planes whose
// bounds its inflated bounds overlap: the half-space behind the plane when its
// normal is a coordinate axis, else the whole space (computePlaneBounds,
// geomutils/src/GuBounds.cpp:210-250), inflated by the plane's contact offset.
__global__ void k_sleep_count(int Q, int cap, const uint32_t* dP, const uint2* pairs, const int* qBody,
                              const int* qPlane, const float4* planes, const float4* bmin, const float4* bmax, float co,
                              const uint64_t* keys, int nKeys, int nMB, const int* meshBody, const int* world,
                              const float4* meshLo, const float4* meshHi, SleepState ss)
{
	const int s = blockIdx.x * blockDim.x + threadIdx.x;
	if (s >= Q + cap)
	{
		// a mesh whose broadphase bounds (its world bounds inflated by its
		// contact offset) overlap the body's
		const int k = s - Q - cap;
		if (k >= nMB)
			return;
		const int i = meshBody[k];
		const float4 lo = meshLo[world[i]], hi = meshHi[world[i]], a = bmin[i], b = bmax[i];
		if (!(lo.x - co > b.x || a.x > hi.x + co || lo.y - co > b.y || a.y > hi.y + co || lo.z - co > b.z ||
		      a.z > hi.z + co))
			atomicAdd(&ss.counted[i], 1);
		return;
	}
	if (s < Q)
	{
		const int i = qBody[s];
		const float4 pl = planes[qPlane[s]];
		const float ax = fabsf(pl.x), ay = fabsf(pl.y), az = fabsf(pl.z);
		const float e = 1e-6f, one = 1.0f - e;
		int axis = -1;
		if (ax > one && ay < e && az < e) axis = 0;
		else if (ax < e && ay > one && az < e) axis = 1;
		else if (ax < e && ay < e && az > one) axis = 2;
		bool counted = true;
		if (axis >= 0)
		{
			const float4 lo4 = bmin[i], hi4 = bmax[i];
			const float lo = axis == 0 ? lo4.x : axis == 1 ? lo4.y : lo4.z;
			const float hi = axis == 0 ? hi4.x : axis == 1 ? hi4.y : hi4.z;
			const float c = axis == 0 ? pl.x : axis == 1 ? pl.y : pl.z;
			counted = c > 0.0f ? lo <= -pl.w + co : hi >= pl.w - co;
		}
		if (counted)
			atomicAdd(&ss.counted[i], 1);
		return;
	}
	const int k = s - Q;
	if (k >= cap || uint32_t(k) >= *dP)
		return;
	const uint2 ab = pairs[k];
	if (nKeys > 0 && pairJointed(ab, keys, nKeys))
		return;   // jointed bodies: the pair is filtered out, no interaction
	atomicAdd(&ss.counted[ab.x], 1);
	atomicAdd(&ss.counted[ab.y], 1);
}

// a touching pair of an awake and a sleeping body names the sleeping body's
// island (setEdgesConnected, secondPassIslandGen: ScPipeline.cpp:1726-1776)
__global__ void k_sleep_wake_mark(int Q, int cap, const uint32_t* dP, const uint2* pairs, const float4* ctN,
                                  SleepState ss)
{
	const int k = blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= cap || uint32_t(k) >= *dP || __float_as_int(ctN[Q + k].w) <= 0)
		return;
	const uint2 ab = pairs[k];
	const bool sa = asleepBody(ss.flags, ab.x), sb = asleepBody(ss.flags, ab.y);
	if (sa != sb)
		ss.wakeIsl[ss.isl[sa ? ab.x : ab.y]] = 1u;
}

// bodies of named islands wake (wakeObjectsUp), keeping their wake counter,
// not ready for sleep (IslandSim::activateNode, PxsIslandSim.cpp:400-432)
__global__ void k_sleep_wake_apply(int n, SleepState ss)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n && asleepBody(ss.flags, i) && ss.wakeIsl[ss.isl[i]])
		ss.flags[i] = 0u;
}

// pairs of sleeping bodies lose their contacts (inactive contact managers)
__global__ void k_sleep_drop(int Q, int cap, const uint32_t* dP, const uint2* pairs, const int* qBody, int nMB,
                             const int* meshBody, float4* ctN, const uint32_t* flags)
{
	const int s = blockIdx.x * blockDim.x + threadIdx.x;
	if (s >= Q + cap)
	{
		const int k = s - Q - cap;
		if (k < nMB * MESH_MAXP && asleepBody(flags, meshBody[k / MESH_MAXP]))
			ctN[s].w = __int_as_float(0);
		return;
	}
	if (s < Q)
	{
		if (asleepBody(flags, qBody[s]))
			ctN[s].w = __int_as_float(0);
		return;
	}
	const int k = s - Q;
	if (k >= cap || uint32_t(k) >= *dP)
		return;
	const uint2 ab = pairs[k];
	if (asleepBody(flags, ab.x) && asleepBody(flags, ab.y))
		ctN[s].w = __int_as_float(0);
}

__global__ void k_sleep_isl_init(int n, SleepState ss)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
	{
		ss.parent[i] = i;
		ss.notReady[i] = 0u;
		ss.wakeIsl[i] = 0u;
	}
}

// Island union-find over the body indices, roots the smallest index of their
// tree. Parents only ever move to smaller indices, so a stale read is still an
// ancestor; roots are linked only by compare-and-swap, and path halving writes
// only to non-roots.
PXH_D int islFind(int* par, int x)
{
	int cur = par[x];
	if (cur == x)
		return x;
	int prev = x, next;
	while (cur > (next = par[cur]))
	{
		par[prev] = next;
		prev = cur;
		cur = next;
	}
	return cur;
}

PXH_D void islUnion(int* par, int a, int b)
{
	int ra = islFind(par, a), rb = islFind(par, b);
	while (ra != rb)
	{
		if (ra < rb)
		{
			const int t = ra;
			ra = rb;
			rb = t;
		}
		// link the larger root under the smaller one
		const int old = atomicCAS(&par[ra], ra, rb);
		if (old == ra)
			return;
		ra = islFind(par, old);
		rb = islFind(par, rb);
	}
}

// touching body pairs (both awake after the wake-up) and joints of two awake
// bodies join islands
__global__ void k_sleep_union(int Q, int cap, const uint32_t* dP, const uint2* pairs, const float4* ctN, int J,
                              const int4* jInfo, SleepState ss)
{
	const int s = blockIdx.x * blockDim.x + threadIdx.x;
	if (s < cap)
	{
		if (uint32_t(s) < *dP && __float_as_int(ctN[Q + s].w) > 0)
		{
			const uint2 ab = pairs[s];
			islUnion(ss.parent, int(ab.x), int(ab.y));
		}
		return;
	}
	const int j = s - cap;
	if (j >= J)
		return;
	const int4 ji = jInfo[j];
	if (ji.y >= 0 && ji.z >= 0 && !asleepBody(ss.flags, ji.y) && !asleepBody(ss.flags, ji.z))
		islUnion(ss.parent, ji.y, ji.z);
}

// awake bodies take their island's label; a body not ready for sleep keeps
// its island awake
__global__ void k_sleep_label(int n, SleepState ss)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n || asleepBody(ss.flags, i))
		return;
	const int r = islFind(ss.parent, i);
	ss.isl[i] = r;
	if (!(ss.flags[i] & SLEEP_READY))
		ss.notReady[r] = 1u;
}

// islands whose bodies are all ready go to sleep, velocities zeroed
// (IslandSim::processLostEdges deactivation, PxsIslandSim.cpp:1690-1720;
// BodySim::deactivate, ScBodySim.cpp:469-490)
__global__ void k_sleep_deactivate(int n, SleepState ss, float4* lin, float4* ang)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n || asleepBody(ss.flags, i) || ss.notReady[ss.isl[i]])
		return;
	ss.flags[i] |= SLEEP_ASLEEP;
	lin[i] = make_float4(0.0f, 0.0f, 0.0f, lin[i].w);
	ang[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

PXH_D void wakeBody(const SleepState& ss, uint32_t i);

__global__ void k_sleep_wake_bodies(int k, const int* bodies, SleepState ss)
{
	const int j = blockIdx.x * blockDim.x + threadIdx.x;
	if (j < k)
		wakeBody(ss, uint32_t(bodies[j]));
}

__global__ void k_sleep_read(int n, SleepState ss, float* wc, int* asleep)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
	{
		wc[i] = ss.wc[i];
		asleep[i] = asleepBody(ss.flags, i) ? 1 : 0;
	}
}

PXH_D xf bodyPose(int i, const float4* pos, const float4* rot)
{
	xf t;
	if (i < 0)
	{
		t.q.x = t.q.y = t.q.z = 0.0f;
		t.q.w = 1.0f;
		t.p = mk(0.0f, 0.0f, 0.0f);
		return t;
	}
	t.q = mkq(rot[i]);
	t.p = mk(pos[i]);
	return t;
}

PXH_D m33 bodySqrtInvI(int i, const float4* svI0, const float4* svI1)
{
	if (i < 0)
	{
		m33 z;
		z.c0 = z.c1 = z.c2 = mk(0.0f, 0.0f, 0.0f);
		return z;
	}
	return loadSym(svI0[i], svI1[i]);
}

PXH_D xf jointFrame(const float4* f)
{
	xf t;
	t.p = mk(f[0]);
	t.q = mkq(f[1]);
	return t;
}

// a joint whose bodies all sleep is out of the solve
PXH_D bool jointAsleep(int4 ji, const uint32_t* sleepFlags)
{
	return sleepFlags && (ji.y < 0 || (sleepFlags[ji.y] & SLEEP_ASLEEP)) &&
	       (ji.z < 0 || (sleepFlags[ji.z] & SLEEP_ASLEEP));
}

PXH_D void prepJointOf(int j, const int4* info, const float4* frame, const float4* param, const float4* pos,
                             const float4* rot, const float4* vel, const float4* rec, const float4* svI0,
                             const float4* svI1, float stepDt, float invStepDt, float invDt, float erp,
                             float lengthScale, float4* head, float4* rows, const uint32_t* sleepFlags)
{
	const int4 ji = info[j];
	if (jointAsleep(ji, sleepFlags))
		return;
	const xf bA = bodyPose(ji.y, pos, rot), bB = bodyPose(ji.z, pos, rot);
	const m33 sI0 = bodySqrtInvI(ji.y, svI0, svI1), sI1 = bodySqrtInvI(ji.z, svI0, svI1);
	const float im0 = ji.y >= 0 ? vel[4 * int64_t(ji.y)].w : 0.0f;
	const float im1 = ji.z >= 0 ? vel[4 * int64_t(ji.z)].w : 0.0f;
	// the bodies' velocities at the start of the solve (world frame)
	const f3 zero = mk(0.0f, 0.0f, 0.0f);
	const f3 v0 = ji.y >= 0 ? mk(rec[PREP_REC * int64_t(ji.y) + 4]) : zero;
	const f3 w0 = ji.y >= 0 ? mk(rec[PREP_REC * int64_t(ji.y) + 5]) : zero;
	const f3 v1 = ji.z >= 0 ? mk(rec[PREP_REC * int64_t(ji.z) + 4]) : zero;
	const f3 w1 = ji.z >= 0 ? mk(rec[PREP_REC * int64_t(ji.z) + 5]) : zero;
	const float4* jp = param + JOINT_PARAM * int64_t(j);
	prepJoint(ji.x, jp[0], jp[1], jp[2], bA, bB, jointFrame(frame + 4 * int64_t(j)),
	          jointFrame(frame + 4 * int64_t(j) + 2), sI0, sI1, im0, im1, v0, w0, v1, w1, stepDt, invStepDt, invDt,
	          erp, lengthScale, head + JOINT_HEAD * int64_t(j), rows + JOINT_ROWS * int64_t(j));
}

__global__ void __launch_bounds__(64) k_joint_prep(int J, const int4* info, const float4* frame, const float4* param,
                                                   const float4* pos, const float4* rot, const float4* vel,
                                                   const float4* rec, const float4* svI0, const float4* svI1,
                                                   float stepDt, float invStepDt, float invDt, float erp,
                                                   float lengthScale, float4* head, float4* rows,
                                                   const uint32_t* sleepFlags)
{
	PXH_THIN_LOOP(j, J)
		prepJointOf(int(j), info, frame, param, pos, rot, vel, rec, svI0, svI1, stepDt, invStepDt, invDt, erp,
		            lengthScale, head, rows, sleepFlags);
}

template <class Vel>
__device__ __forceinline__ void solveJointOf(int j, const int4* info, const float4* head, float4* rows, const Vel& vel,
                                             const float4* svI0, const float4* svI1, float elapsed, bool conclude,
                                             const uint32_t* sleepFlags)
{
	const int4 ji = info[j];
	if (jointAsleep(ji, sleepFlags))
		return;
	const int a = ji.y, b = ji.z;
	f3 l0 = mk(0.0f, 0.0f, 0.0f), a0 = l0, dl0 = l0, da0 = l0, l1 = l0, a1 = l0, dl1 = l0, da1 = l0;
	qt q0, q1;
	q0.x = q0.y = q0.z = 0.0f; q0.w = 1.0f;
	q1 = q0;
	float w0 = 0.0f, w1 = 0.0f;
	float4 v[4];
	if (a >= 0)
	{
		vel.load(a, v);
		l0 = mk(v[0]); w0 = v[0].w; a0 = mk(v[1]); dl0 = mk(v[2]); da0 = mk(v[3]);
		q0 = mkq(vel.turn(a));
	}
	if (b >= 0)
	{
		vel.load(b, v);
		l1 = mk(v[0]); w1 = v[0].w; a1 = mk(v[1]); dl1 = mk(v[2]); da1 = mk(v[3]);
		q1 = mkq(vel.turn(b));
	}
	const m33 sI0 = bodySqrtInvI(a, svI0, svI1), sI1 = bodySqrtInvI(b, svI0, svI1);
	const float4* h = head + JOINT_HEAD * int64_t(j);
	solveJoint(__float_as_int(h[8].x), h, rows + JOINT_ROWS * int64_t(j), l0, a0, dl0, da0,
	           q0, sI0, l1, a1, dl1, da1, q1, sI1, elapsed, conclude);
	if (a >= 0)
		vel.store(a, f4(l0, w0), f4(a0, 0.0f));
	if (b >= 0)
		vel.store(b, f4(l1, w1), f4(a1, 0.0f));
}

__global__ void k_joint_solve(int begin, int end, const int4* info, const float4* head, float4* rows, float4* vel,
                              const float4* svDQ, const float4* svI0, const float4* svI1, float elapsed, int conclude,
                              const uint32_t* sleepFlags)
{
	const int j = begin + blockIdx.x * blockDim.x + threadIdx.x;
	if (j >= end)
		return;
	solveJointOf(j, info, head, rows, VelTurn{{vel, 0}, svDQ}, svI0, svI1, elapsed, conclude != 0, sleepFlags);
}

// A world's velocities in LDS, 32 bytes a body; the substeps' summed motion,
// which only the integration writes, stays in the scene's array. Half the LDS of
// whole records, so twice the worlds run at a time.
struct VelWorld
{
	float4* lds;
	float4* v;
	const float4* dq;
	int base;
	PXH_D void load(int body, float4 (&r)[4]) const
	{
		const float4* p = lds + 2 * (body - base);
		const float4* g = v + 4 * int64_t(body);
		r[2] = g[2]; r[3] = g[3];
		r[0] = p[0]; r[1] = p[1];
	}
	PXH_D void store(int body, float4 lin, float4 ang) const
	{
		float4* p = lds + 2 * (body - base);
		p[0] = lin;
		p[1] = ang;
	}
	PXH_D void storeMoved(int body, float4 lin, float4 ang) const
	{
		v[4 * int64_t(body) + 2] = lin;
		v[4 * int64_t(body) + 3] = ang;
	}
	PXH_D float4 turn(int body) const { return dq[body]; }
};

// Every iteration of independent worlds (the batched form and small scenes).
// Persistent workgroups take worlds from a queue
// ordered by size (largest first); a workgroup keeps its world's velocities in
// LDS (worlds of at most ldsBodies bodies; larger ones work on the scene's
// array), then for every iteration solves the world's joints by colour and its
// contacts by colour in order, one barrier between colours, and moves the bodies
// (TGS) or keeps their motion (PGS), as the launches for all worlds at once do.
// Rows are ordered by (world, colour): segStart[w * CB + c] is the first row of
// colour c of world w. Every wave leaves once the queue is empty. Same
// arithmetic in the same order as the per-colour path (cf. solveWholeIslandTGS,
// gpusolver/src/CUDA/solverMultiBlockTGS.cu:1686, which runs a small island in
// one block).
//
// Bound by the chain of colours: a row's data streams past while its bodies stay
// in LDS, so the next colour's rows are loaded before the barrier (a thread
// takes the same rows in every iteration, and their impulses are its own), and
// the non-empty colours' starts are listed in LDS once. The prefetch holds about
// 240 registers, two waves a SIMD; held to three it spills and takes 1,400 us
// where this takes 770 (8,192 worlds; 957 without the prefetch at three). 301
// worlds: 179 us against 247.
template <int THREADS, bool PGS, bool JOINTS>
__global__ void __launch_bounds__(THREADS, 2) k_solve_worlds(int nWorlds, const int* worldOrder, uint32_t* queueHead,
                                                          const int* bodyStart, const uint32_t* segStart, int CB, int C,
                                                          Rows rows, const float* rowsU, SolverBodies sb, int posIters,
                                                          int iters, float stepDt, float muS, float muD,
                                                          float invStepDt, float biasScale, float scale,
                                                          uint32_t* broken, int ldsBodies, WorldJoints J)
{
	extern __shared__ float4 lds[];
	uint32_t* list = reinterpret_cast<uint32_t*>(lds + 2 * ldsBodies);   // CB + 1
	__shared__ int sWorld, sColors;
	const int tid = threadIdx.x;
	for (;;)
	{
		if (tid == 0)
		{
			const uint32_t q = atomicAdd(queueHead, 1u);
			sWorld = q < uint32_t(nWorlds) ? worldOrder[q] : -1;
		}
		__syncthreads();
		const int w = sWorld;
		if (w < 0)
			return;
		const int b0 = bodyStart[w], nb = bodyStart[w + 1] - b0;
		const bool inLds = nb <= ldsBodies;
		if (inLds)
			for (int i = tid; i < 2 * nb; i += THREADS)
				lds[i] = sb.vel[4 * int64_t(b0 + (i >> 1)) + (i & 1)];
		if (tid < 64)
		{
			const uint32_t* seg = segStart + int64_t(w) * CB;
			int k = 0;
			for (int c = tid; c - tid < CB; c += 64)
			{
				const uint32_t s = c < CB ? seg[c] : 0u, e = c < CB ? seg[c + 1] : 0u;
				const uint64_t m = __ballot(s < e);
				if (s < e)
					list[k + __popcll(m & ((1ull << tid) - 1ull))] = s;
				k += __popcll(m);
			}
			if (tid == 0)
			{
				list[k] = seg[CB];
				sColors = k;
			}
		}
		__syncthreads();
		const int colors = sColors;
		auto solve = [&](const auto& vel) {
			typename std::conditional<PGS, PgsRow, TgsRow>::type row;
			auto load = [&](int o, int it) {
				if constexpr (PGS)
					loadPgsRow(o, C, rows, rowsU, it >= posIters || posIters - it <= 3, it >= posIters, row);
				else
					loadTgsRow(o, C, rows, row);
			};
			if (colors > 0 && list[0] + tid < list[1])
				load(int(list[0]) + tid, 0);
			for (int it = 0; it < iters; it++)
			{
				const bool posIter = it < posIters;
				uint32_t* brk = it == iters - 1 ? broken : nullptr;
				if constexpr (JOINTS)
					for (int c = 0; c < J.colors; c++)
					{
						const int* jseg = J.seg + int64_t(w) * (J.colors + 1);
						const float elapsed = stepDt * float(min(it, posIters));
						for (int k = jseg[c] + tid; k < jseg[c + 1]; k += THREADS)
							solveJointOf(J.order[k], J.info, J.head, J.rows, vel, sb.i0, sb.i1, elapsed, it == posIters - 1,
							             J.sleepFlags);
						__syncthreads();
					}
				for (int c = 0; c < colors; c++)
				{
					const int e = int(list[c + 1]);
					for (int o = int(list[c]) + tid; o < e;)
					{
						if constexpr (PGS)
							solvePgsRow(o, C, rows, row, vel, !posIter || posIters - it <= 3, !posIter, brk);
						else
							solveTgsRow(o, C, rows, row, vel, posIter ? -3.402823466e+38f : 0.0f, muS, muD, invStepDt,
							            biasScale, scale, brk);
						o += THREADS;
						if (o < e)
							load(o, it);
					}
					const int nc = c + 1 < colors ? c + 1 : 0;
					if (list[nc] + tid < list[nc + 1])
						load(int(list[nc]) + tid, nc ? it : it + 1);
					__syncthreads();
				}
				if constexpr (PGS)
				{
					if (it == posIters - 1)
					{
						for (int i = b0 + tid; i < b0 + nb; i += THREADS)
						{
							float4 v[4];
							vel.load(i, v);
							sb.p[i] = v[0];
							sb.dq[i] = v[1];
						}
						__syncthreads();   // the velocity passes change what is saved here
					}
				}
				else if (posIter)
				{
					for (int i = b0 + tid; i < b0 + nb; i += THREADS)
						integrateBodyTGS(i, stepDt, vel, sb.p, sb.dq, sb.i0, sb.i1);
					__syncthreads();
				}
			}
		};
		if (inLds)
		{
			solve(VelWorld{lds, sb.vel, sb.dq, b0});
			__syncthreads();
			for (int i = tid; i < 2 * nb; i += THREADS)
				sb.vel[4 * int64_t(b0 + (i >> 1)) + (i & 1)] = lds[i];
		}
		else
			solve(VelTurn{{sb.vel, 0}, sb.dq});
		__syncthreads();
	}
}


// copyBackBodies (lowleveldynamics/src/DyTGSDynamics.cpp:1549-1580), with
// the sleep check on the step's mean velocities (DyTGSDynamics.cpp:1561, 1577)
__global__ void k_finalize(int n, float dt, float4* pos, float4* rot, float4* lin, float4* ang, const float4* invI,
                           const float4* vel, const float4* svP, const float4* svDQ, const float4* svI0,
                           const float4* svI1, SleepState ss)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	if (ss.flags && (ss.flags[i] & SLEEP_ASLEEP))
		return;   // sleeping: pose and zero velocities kept
	const qt q = qnormalize(qmul(mkq(svDQ[i]), mkq(rot[i])));
	rot[i] = f4(q);
	pos[i] = svP[i];
	const float4* v = vel + 4 * int64_t(i);
	const float4 l = v[0];
	lin[i] = l;
	const m33 S = loadSym(svI0[i], svI1[i]);
	ang[i] = f4(mmul(S, mk(v[1])), 0.0f);
	if (ss.flags)
	{
		const float invDt = 1.0f / dt;
		sleepCheck(ss, i, dt, mk(v[2]) * invDt, mmul(S, mk(v[3]) * invDt), q, l.w, invI[i]);
	}
}

// ---------------------------------------------------------------------------
// Direct GPU API gather/scatter (updateBodiesAndShapes.cu:999-1253)
// ---------------------------------------------------------------------------
// what: PxRigidDynamicGPUAPIReadType (0 pose, 1 linear velocity, 2 angular
// velocity, 3 linear acceleration, 4 angular acceleration: the velocity change
// of the last step over its dt, getRigidDynamicLinearAcceleration,
// gpusimulationcontroller/src/CUDA/updateBodiesAndShapes.cu:1063-1106)
__global__ void k_get_data(int n, const uint32_t* idx, int what, const float4* pos, const float4* rot,
                           const float4* lin, const float4* ang, const float4* prevLin, const float4* prevAng,
                           float invDt, float* out)
{
	const int k = blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= n)
		return;
	const uint32_t i = idx ? idx[k] : uint32_t(k);
	if (what == 0)
	{
		const float4 q = rot[i], p = pos[i];
		float* o = out + 7 * int64_t(k);
		o[0] = q.x; o[1] = q.y; o[2] = q.z; o[3] = q.w; o[4] = p.x; o[5] = p.y; o[6] = p.z;
	}
	else if (what <= 2)
	{
		const float4 v = what == 1 ? lin[i] : ang[i];
		float* o = out + 3 * int64_t(k);
		o[0] = v.x; o[1] = v.y; o[2] = v.z;
	}
	else
	{
		const f3 a = (what == 3 ? mk(lin[i]) - mk(prevLin[i]) : mk(ang[i]) - mk(prevAng[i])) * invDt;
		float* o = out + 3 * int64_t(k);
		o[0] = a.x; o[1] = a.y; o[2] = a.z;
	}
}

// what: PxRigidDynamicGPUAPIWriteType (0 pose, 1 linear velocity, 2 angular
// velocity, 3 force, 4 torque). A force becomes the linear acceleration
// F / m, a torque the angular acceleration I_world^-1 tau with the body's
// current orientation (PxForceMode::eFORCE, NpRigidBodyTemplate.h:507-528;
// setRigidDynamicForce / setRigidDynamicTorque, updateBodiesAndShapes.cu:1229-1278)
// PxRigidDynamic::wakeUp (BodyCore::wakeUp with the scene's wake counter
// reset value, 20 * 0.02 s): awake now, not ready for sleep; the rest of a
// sleeping body's island wakes at the next step (IslandSim::activateNode)
PXH_D void wakeBody(const SleepState& ss, uint32_t i)
{
	ss.wc[i] = 20.0f * 0.02f;
	const uint32_t f = ss.flags[i];
	ss.flags[i] = 0u;
	if (f & SLEEP_ASLEEP)
		ss.wakeIsl[ss.isl[i]] = 1u;
}

__global__ void k_set_data(int n, const uint32_t* idx, int what, float4* pos, float4* rot, float4* lin, float4* ang,
                           const float4* invI, float4* extLin, float4* extAng, const float* in, SleepState ss)
{
	const int k = blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= n)
		return;
	const uint32_t i = idx ? idx[k] : uint32_t(k);
	if (what == 0)
	{
		const float* s = in + 7 * int64_t(k);
		rot[i] = make_float4(s[0], s[1], s[2], s[3]);
		pos[i] = make_float4(s[4], s[5], s[6], 0.0f);
		if (ss.flags)
			wakeBody(ss, i);   // autowake of setGlobalPose
		return;
	}
	const float* s = in + 3 * int64_t(k);
	const f3 v = mk(s[0], s[1], s[2]);
	// velocities always wake the body, forces and torques when nonzero
	// (autowake of setLinearVelocity / addForce)
	if (ss.flags && (what <= 2 || v.x != 0.0f || v.y != 0.0f || v.z != 0.0f))
		wakeBody(ss, i);
	if (what == 1)
		lin[i] = make_float4(v.x, v.y, v.z, lin[i].w);
	else if (what == 2)
		ang[i] = make_float4(v.x, v.y, v.z, 0.0f);
	else if (what == 3)
		extLin[i] = f4(v * lin[i].w, 0.0f);
	else
	{
		// R diag(invI) R^T (Cm::transformInertiaTensor)
		const m33 R = qmat(mkq(rot[i]));
		const float4 ii = invI[i];
		m33 A;
		A.c0 = R.c0 * ii.x; A.c1 = R.c1 * ii.y; A.c2 = R.c2 * ii.z;
		extAng[i] = f4(mmul(mmm(A, mtrans(R)), v), 0.0f);
	}
}

// ---------------------------------------------------------------------------
// standalone broadphase: found/lost pairs between consecutive pair sets, both
// sorted by (id0, id1) (BpBroadPhase.h:159-185 created/deleted semantics)
// ---------------------------------------------------------------------------
// canonical pair key (lower index first)
PXH_D uint64_t pkey(uint2 p) { return (uint64_t(min(p.x, p.y)) << 32) | max(p.x, p.y); }

// pair keys in the caller's handle space (ids[box], or the box index)
__global__ void k_pair_keys(int P, const uint2* pairs, const uint32_t* ids, uint64_t* keys, uint32_t* vals)
{
	const int p = blockIdx.x * blockDim.x + threadIdx.x;
	if (p < P)
	{
		uint2 q = pairs[p];
		if (ids)
			q = make_uint2(ids[q.x], ids[q.y]);
		keys[p] = pkey(q);
		vals[p] = uint32_t(p);
	}
}

// flag[i] = 1 if key a[i] is absent from sorted b
__global__ void k_set_diff_flags(int na, const uint64_t* a, int nb, const uint64_t* b, uint32_t* flag)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= na)
		return;
	const uint64_t k = a[i];
	int l = 0, h = nb;
	while (l < h)
	{
		const int m = (l + h) >> 1;
		if (b[m] < k) l = m + 1;
		else h = m;
	}
	flag[i] = (l < nb && b[l] == k) ? 0u : 1u;
}

// touch events (prepareLostFoundPairs_Stage1, gpunarrowphase/src/CUDA/cudaGJKEPA.cu:1468):
// a constraint without a row in the previous step starts touching; the
// previous rows it finds are marked, the unmarked ones stopped touching
__global__ void k_found_flags(int C, const int* prevRow, uint32_t* found, uint32_t* matched)
{
	const int c = blockIdx.x * blockDim.x + threadIdx.x;
	if (c >= C)
		return;
	const int po = prevRow ? prevRow[c] : -1;
	found[c] = po < 0 ? 1u : 0u;
	if (po >= 0)
		matched[po] = 1u;
}
__global__ void k_lost_flags(int R, const uint32_t* matched, uint32_t* lost)
{
	const int r = blockIdx.x * blockDim.x + threadIdx.x;
	if (r < R)
		lost[r] = matched[r] ? 0u : 1u;
}

__global__ void k_compact_keys(int na, const uint64_t* a, const uint32_t* flag, const uint32_t* scanned, uint2* out)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < na && flag[i])
		out[scanned[i]] = make_uint2(uint32_t(a[i] >> 32), uint32_t(a[i]));
}


// batched immediate-mode contacts (PxGenerateContacts on a fresh cache)
__global__ void __launch_bounds__(NP_THREADS) k_np_immediate(int n, const int* type0, const float* geom0,
                                                             const float* pose0, const int* type1, const float* geom1,
                                                             const float* pose1, float cd, float tol, float* out,
                                                             int* counts)
{
	__shared__ float4 points[3 * BOX_MAX_POINTS * NP_THREADS / 4];
	// lanes past the last pair repeat it (they help the wave's box searches) and store nothing
	const int own = blockIdx.x * NP_THREADS + threadIdx.x;
	const int k = min(own, n - 1);
	const int t0 = type0[k], t1 = type1[k];
	const float* g0 = geom0 + 4 * int64_t(k);
	const float* g1 = geom1 + 4 * int64_t(k);
	const float* q0 = pose0 + 7 * int64_t(k);
	const float* q1 = pose1 + 7 * int64_t(k);
	xf x0, x1;
	x0.p = mk(q0[0], q0[1], q0[2]); x0.q.x = q0[3]; x0.q.y = q0[4]; x0.q.z = q0[5]; x0.q.w = q0[6];
	x1.p = mk(q1[0], q1[1], q1[2]); x1.q.x = q1[3]; x1.q.y = q1[4]; x1.q.z = q1[5]; x1.q.w = q1[6];
	Contacts c;
	c.count = 0;
	int cnt = -1;
	if (t0 == GEOM_SPHERE && t1 == GEOM_SPHERE)
		cnt = sphereSphere(g0[0], x0.p, g1[0], x1.p, cd, c);
	else if (t0 == GEOM_SPHERE && t1 == GEOM_PLANE)
	{
		const f3 pn = qrot(x1.q, mk(1.0f, 0.0f, 0.0f));
		cnt = spherePlane(g0[0], x0.p, pn, -dot(pn, x1.p), cd, c);
	}
	else if (t0 == GEOM_SPHERE && t1 == GEOM_BOX)
		cnt = sphereBox(g0[0], x0.p, mk(g1[0], g1[1], g1[2]), x1, cd, c);
	else if (t0 == GEOM_PLANE && t1 == GEOM_BOX)
	{
		const f3 pn = qrot(x0.q, mk(1.0f, 0.0f, 0.0f));
		cnt = planeBox(pn, -dot(pn, x0.p), mk(g1[0], g1[1], g1[2]), x1, cd, points + threadIdx.x, c);
	}
	else if (t0 == GEOM_BOX && t1 == GEOM_BOX)
		cnt = boxBoxFace(mk(g0[0], g0[1], g0[2]), x0, mk(g1[0], g1[1], g1[2]), x1, cd, tol, BoxPoints{reinterpret_cast<float*>(points) + threadIdx.x}, c);
	else if (t0 == GEOM_SPHERE && t1 == GEOM_CAPSULE)
		cnt = sphereCapsule(g0[0], x0.p, g1[0], g1[1], x1, cd, c);
	else if (t0 == GEOM_CAPSULE && t1 == GEOM_CAPSULE)
		cnt = capsuleCapsule(g0[0], g0[1], x0, g1[0], g1[1], x1, cd, c);
	else if (t0 == GEOM_PLANE && t1 == GEOM_CAPSULE)
	{
		const f3 pn = qrot(x0.q, mk(1.0f, 0.0f, 0.0f));
		cnt = planeCapsule(pn, -dot(pn, x0.p), g1[0], g1[1], x1, cd, c);
	}
	else if (t0 == GEOM_CAPSULE && t1 == GEOM_BOX)
		cnt = capsulePoly<true>(g0[0], g0[1], x0, boxPoly(mk(g1[0], g1[1], g1[2])), x1, cd, tol, 0, c);
	boxBoxEdgeWave(cnt == BOXBOX_EDGE, mk(g0[0], g0[1], g0[2]), x0, mk(g1[0], g1[1], g1[2]), x1, cd, c, cnt);
	if (own >= n)
		return;
	counts[k] = cnt;
#pragma unroll
	for (int i = 0; i < 4; i++)
	{
		if (i >= cnt)
			break;
		float* o = out + (4 * int64_t(k) + i) * 8;
		o[0] = c.p[i].x; o[1] = c.p[i].y; o[2] = c.p[i].z; o[3] = c.sep[i];
		o[4] = c.n.x; o[5] = c.n.y; o[6] = c.n.z; o[7] = 0.0f;
	}
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static inline int nblk(int64_t n, int t) { return int((n + t - 1) / t); }

void launch_scan(uint32_t* data, int64_t n, uint32_t* tmp, hipStream_t st)
{
	// tmp must hold scan_tmp_size(n) entries
	if (n <= 0)
		return;
	const int nb = nblk(n, SCAN_TILE);
	if (nb > 1)
		k_scan_sums<<<nb, SCAN_THREADS, 0, st>>>(data, n, tmp);
	if (nb > SUMS_DIRECT)
	{
		launch_scan(tmp, nb, tmp + nb, st);
		k_scan_tiles<true><<<nb, SCAN_THREADS, 0, st>>>(data, n, tmp);
	}
	else
		k_scan_tiles<false><<<nb, SCAN_THREADS, 0, st>>>(data, n, tmp);
}

int64_t scan_tmp_size(int64_t n)
{
	const int64_t nb = (std::max<int64_t>(n, 0) + SCAN_TILE - 1) / SCAN_TILE;
	return nb + 1 + (nb > SUMS_DIRECT ? scan_tmp_size(nb) : 0);
}
int64_t con_tmp_size(int64_t slots)
{
	const int64_t nb = slots / CON_TILE + 1;
	return nb + scan_tmp_size(nb);
}

int64_t radix_tmp_size(int n) { return scan_tmp_size(int64_t(256) * nblk(n, RS_TILE)); }
bool radix_result_in_alt(int n, int bits) { return n > RS_SMALL && ((bits + 7) / 8) % 2 == 1; }

void launch_radix_sort(uint64_t* keys, uint32_t* vals, uint64_t* keys2, uint32_t* vals2, int n, int lowBits,
                       int highBits, uint32_t* hist, uint32_t* scanTmp, hipStream_t st, bool& resultInAlt)
{
	resultInAlt = false;
	const int bits = lowBits + highBits;
	if (n <= 0 || bits <= 0)
		return;
	if (n <= RS_SMALL)
	{
		if (n <= RS_SMALL_THREADS)
			k_rs_small<1><<<1, RS_SMALL_THREADS, 0, st>>>(keys, vals, n, lowBits, bits);
		else if (n <= 2 * RS_SMALL_THREADS)
			k_rs_small<2><<<1, RS_SMALL_THREADS, 0, st>>>(keys, vals, n, lowBits, bits);
		else if (n <= 4 * RS_SMALL_THREADS)
			k_rs_small<4><<<1, RS_SMALL_THREADS, 0, st>>>(keys, vals, n, lowBits, bits);
		else
			k_rs_small<8><<<1, RS_SMALL_THREADS, 0, st>>>(keys, vals, n, lowBits, bits);
		return;
	}
	const int nb = nblk(n, RS_TILE);   // radix_result_in_alt says where the result lands
	uint64_t* ka = keys;
	uint32_t* va = vals;
	uint64_t* kb = keys2;
	uint32_t* vb = vals2;
	for (int shift = 0; shift < bits; shift += 8)
	{
		if (nb > RS_DIRECT)
		{
			k_rs_hist<true><<<nb, RS_THREADS, 0, st>>>(ka, n, lowBits, shift, hist, nb);
			launch_scan(hist, int64_t(256) * nb, scanTmp, st);
			k_rs_scatter<true><<<nb, RS_THREADS, 0, st>>>(ka, va, kb, vb, n, lowBits, shift, hist, nb);
		}
		else
		{
			k_rs_hist<false><<<nb, RS_THREADS, 0, st>>>(ka, n, lowBits, shift, hist, nb);
			k_rs_scatter<false><<<nb, RS_THREADS, 0, st>>>(ka, va, kb, vb, n, lowBits, shift, hist, nb);
		}
		uint64_t* tk = ka; ka = kb; kb = tk;
		uint32_t* tv = va; va = vb; vb = tv;
		resultInAlt = !resultInAlt;
	}
}

#define PXH_LAUNCH(kernel, n, ...) \
	do { if ((n) > 0) kernel<<<nblk((n), 256), 256, 0, st>>>(__VA_ARGS__); } while (0)

void launch_bounds(int n, const float4* pos, const float4* rot, const float4* geom, const HullSet& hs, float co,
                   float4* bmin, float4* bmax, ColorState cs, hipStream_t st)
{
	PXH_LAUNCH(k_bounds, n, n, pos, rot, geom, hs, co, bmin, bmax, cs);
}
// Worlds of up to 8,192 bodies take a workgroup each (in one world, against four
// launches: 4,096 bodies 6.4 / 10.4 us, 8,192 8.7 / 10.6, 12,288 11.4 / 10.7); a
// larger world takes the launches over all bodies, whose blocks spread over the chip.
constexpr int WORLD_GRID_MAX = 8192;
void launch_scene_grid(int n, int nScenes, int maxWorldBodies, const int* bodyStart, const int* scene,
                       const float4* bmin, const float4* bmax, uint32_t* acc, float4* gridF, int2* gridI,
                       const uint32_t* rowOff, uint64_t* keys, uint32_t* vals, hipStream_t st)
{
	if (maxWorldBodies <= WORLD_GRID_MAX)
	{
		int threads = 64;
		while (threads < 1024 && 2 * threads < maxWorldBodies)
			threads *= 2;
		if (nScenes > 0)
			k_world_grid<<<nScenes, threads, 0, st>>>(bodyStart, bmin, bmax, gridF, gridI, rowOff, keys, vals);
		return;
	}
	PXH_LAUNCH(k_grid_init, nScenes, nScenes, acc);
	if (n > 0)
		k_grid_reduce<<<nblk(n, 256 * GRID_ITEMS), 256, 0, st>>>(n, bmin, bmax, scene, acc);
	PXH_LAUNCH(k_grid_finish, nScenes, nScenes, acc, gridF, gridI, rowOff);
	PXH_LAUNCH(k_keys, n, n, bmin, bmax, scene, gridF, gridI, rowOff, keys, vals);
}
void launch_row_off_single(uint32_t* rowOff, uint32_t cap, hipStream_t st)
{
	k_row_off_single<<<1, 64, 0, st>>>(rowOff, cap);
}
void launch_gather_sorted(int n, const uint32_t* sv, const float4* bmin, const float4* bmax, float4* smin,
                          float4* smax, hipStream_t st)
{
	PXH_LAUNCH(k_gather_sorted, n, n, sv, bmin, bmax, smin, smax);
}
void launch_row_start(int n, const uint64_t* sk, uint32_t* rowStart, uint32_t totalRows, hipStream_t st,
                      const uint32_t* words, uint32_t* hostWords)
{
	const int64_t rows = int64_t(totalRows) + 1;
	if (n == 0)
		PXH_LAUNCH(k_fill_u32, rows, rowStart, rows, 0u);
	else
		PXH_LAUNCH(k_row_start, std::max<int64_t>(n, rows), n, sk, rowStart, totalRows, words, hostWords);
}
template <int G, int CLASSES>
static void sweepPass(bool write, int n, const uint64_t* sk, const float4* smin, const float4* smax, const int* scene,
                      const int* group, uint64_t groupLut, const int2* gridI, const uint32_t* rowOff,
                      const uint32_t* rowStart, uint32_t* counts, const uint32_t* offsets, uint2* pairs,
                      uint32_t pairCap, hipStream_t st)
{
	const int blocks = nblk(n, (SWEEP_THREADS / 64) * (63 / G));
	if (write)
		k_sweep<true, G, CLASSES><<<blocks, SWEEP_THREADS, 0, st>>>(n, sk, smin, smax, scene, group, groupLut, gridI,
		                                                          rowOff, rowStart, counts, offsets, pairs, pairCap);
	else
		k_sweep<false, G, CLASSES><<<blocks, SWEEP_THREADS, 0, st>>>(n, sk, smin, smax, scene, group, groupLut, gridI,
		                                                           rowOff, rowStart, counts, offsets, pairs, pairCap);
}
void launch_sweep(bool write, int classes, int n, const uint64_t* sk, const float4* smin, const float4* smax,
                  const int* scene, const int* group, uint64_t groupLut, const int2* gridI, const uint32_t* rowOff,
                  const uint32_t* rowStart, uint32_t* counts, const uint32_t* offsets, uint2* pairs, uint32_t pairCap,
                  hipStream_t st)
{
	if (n <= 0)
		return;
	auto pass = [&](auto lanes) {
		constexpr int G = decltype(lanes)::value;
		if (classes == 1)
			sweepPass<G, 1>(write, n, sk, smin, smax, scene, group, groupLut, gridI, rowOff, rowStart, counts, offsets,
			                pairs, pairCap, st);
		else if (classes == PAIR_CLASS_FIRST_CONVEX)
			sweepPass<G, PAIR_CLASS_FIRST_CONVEX>(write, n, sk, smin, smax, scene, group, groupLut, gridI, rowOff,
			                                      rowStart, counts, offsets, pairs, pairCap, st);
		else
			sweepPass<G, PAIR_CLASSES>(write, n, sk, smin, smax, scene, group, groupLut, gridI, rowOff, rowStart, counts,
			                           offsets, pairs, pairCap, st);
	};
	// nine lanes a body while the chip has room for them; beyond, the loads of
	// the write pass's second look at each row cost more than the shorter chains
	// save (both passes, nine lanes against one: 4,096 boxes 22 / 83 us, 20,011
	// bodies 44 / 150, 100,003 boxes 80 / 126, 262,144 bodies 339 / 269)
	if (n <= 131072)
		pass(std::integral_constant<int, 9>());
	else
		pass(std::integral_constant<int, 1>());
}
void launch_np_pairs(int cap, const uint32_t* dP, const uint32_t* dConvex, int slotBase, const uint2* pairs,
                     const float4* pos, const float4* rot, const float4* geom, float cd, float tol, float4* ctN,
                     float4* ctP, hipStream_t st)
{
	if (cap > 0)
		k_np_pairs<<<nblk(cap, NP_THREADS), NP_THREADS, 0, st>>>(cap, dP, dConvex, slotBase, pairs, pos, rot, geom, cd,
		                                                        tol, ctN, ctP);
}
void launch_np_convex(int cap, const uint32_t* dP, const uint32_t* dConvex, int slotBase, const uint2* pairs,
                      const float4* pos, const float4* rot, const float4* geom, const HullSet& hs, float cd, float tol,
                      float4* wit, uint32_t* list, float4* ctN, float4* ctP, hipStream_t st)
{
	if (cap <= 0)
		return;
	k_fill_u32<<<1, 64, 0, st>>>(list, 2, 0u);
	// grid-stride: enough waves to fill the chip several times over
	k_np_convex<<<strideBlocks(cap, APART_BLOCK / APART_LANES, 2048), APART_BLOCK, 0, st>>>(
	    cap, dP, dConvex, slotBase, pairs, pos, rot, geom, hs, cd, ctN, list);
	k_np_convex_wave<<<strideBlocks(cap, CVX_WAVES, 8192), 64 * CVX_WAVES, 0, st>>>(cap, pairs, pos, rot, geom, hs, cd,
	                                                                              wit, list);
	k_np_round_convex<<<thinGrid(cap), 64, 0, st>>>(cap, slotBase, pairs, pos, rot, geom, hs, cd, tol, ctN, ctP, list);
	k_np_convex_finish<<<strideBlocks(cap, 64 / GROUP, 16384), 64, 0, st>>>(cap, slotBase, pairs, pos, rot, geom, hs, cd,
	                                                                      tol, wit, list, ctN, ctP);
}
void launch_np_planes_convex(int Q, int slotBase, const int* qBody, const int* qPlane, const float4* pos,
                             const float4* rot, const float4* geom, const float4* planes, const HullSet& hs, float cd,
                             float tol, float4* ctN, float4* ctP, hipStream_t st)
{
	if (Q > 0)
		k_np_planes_convex<<<thinGrid(Q), 64, 0, st>>>(Q, slotBase, qBody, qPlane, pos, rot, geom, planes, hs, cd, tol,
		                                               ctN, ctP);
}
void launch_np_planes(int Q, int slotBase, const int* qBody, const int* qPlane, const float4* pos, const float4* rot,
                      const float4* geom, const float4* planes, float cd, float4* ctN, float4* ctP, hipStream_t st)
{
	if (Q > 0)
		k_np_planes<<<nblk(Q, NP_THREADS), NP_THREADS, 0, st>>>(Q, slotBase, qBody, qPlane, pos, rot, geom, planes, cd,
		                                                        ctN, ctP);
}
void launch_copy_contacts(int C, int maxPairs, const int* order, const int* conA, const int* conB, const int* conSlot,
                          const float4* ctN, const float4* ctP, const float* nF, float4* out, uint32_t* nbPairs,
                          hipStream_t st)
{
	const int n = std::max(C, 1);
	k_copy_contacts<<<nblk(n, 256), 256, 0, st>>>(C, maxPairs, order, conA, conB, conSlot, ctN, ctP, nF, out, nbPairs);
}
void launch_joint_filter(int cap, int Q, const uint32_t* dP, const uint2* pairs, const uint64_t* jointKeys, int nKeys,
                         float4* ctN, hipStream_t st)
{
	if (nKeys > 0)
		PXH_LAUNCH(k_joint_filter, cap, cap, Q, dP, pairs, jointKeys, nKeys, ctN);
}
void launch_sleep_count(int n, int Q, int cap, const uint32_t* dP, const uint2* pairs, const int* qBody,
                        const int* qPlane, const float4* planes, const float4* bmin, const float4* bmax, float co,
                        const uint64_t* jointKeys, int nKeys, int nMB, const int* meshBody, const int* world,
                        const float4* meshLo, const float4* meshHi, SleepState ss, hipStream_t st)
{
	PXH_LAUNCH(k_sleep_count_init, n, n, ss);
	PXH_LAUNCH(k_sleep_count, Q + cap + nMB, Q, cap, dP, pairs, qBody, qPlane, planes, bmin, bmax, co, jointKeys,
	           nKeys, nMB, meshBody, world, meshLo, meshHi, ss);
}
void launch_sleep_wake(int n, int Q, int cap, const uint32_t* dP, const uint2* pairs, const int* qBody, int nMB,
                       const int* meshBody, float4* ctN, SleepState ss, hipStream_t st)
{
	PXH_LAUNCH(k_sleep_wake_mark, cap, Q, cap, dP, pairs, ctN, ss);
	PXH_LAUNCH(k_sleep_wake_apply, n, n, ss);
	PXH_LAUNCH(k_sleep_drop, Q + cap + nMB * MESH_MAXP, Q, cap, dP, pairs, qBody, nMB, meshBody, ctN, ss.flags);
}
void launch_sleep_islands(int n, int Q, int cap, const uint32_t* dP, const uint2* pairs, const int* qBody, int nMB,
                          const int* meshBody, float4* ctN, int J, const int4* jInfo, float4* lin, float4* ang,
                          SleepState ss, hipStream_t st)
{
	PXH_LAUNCH(k_sleep_isl_init, n, n, ss);
	PXH_LAUNCH(k_sleep_union, cap + J, Q, cap, dP, pairs, ctN, J, jInfo, ss);
	PXH_LAUNCH(k_sleep_label, n, n, ss);
	PXH_LAUNCH(k_sleep_deactivate, n, n, ss, lin, ang);
	PXH_LAUNCH(k_sleep_drop, Q + cap + nMB * MESH_MAXP, Q, cap, dP, pairs, qBody, nMB, meshBody, ctN, ss.flags);
}
void launch_np_mesh(int nMB, const int* meshBody, const int* world, const int4* worldMesh, const MeshSet& M,
                    const float4* pos, const float4* rot, const float4* geom, const HullSet& hs, float cd,
                    int slotBase, float4* ctN, float4* ctP, uint32_t* state, hipStream_t st)
{
	if (nMB <= 0)
		return;
	uint32_t* rest = state + 1;
	k_fill_u32<<<1, 64, 0, st>>>(state, 2, 0u);
	k_np_mesh_wave<<<std::min(nMB, 8192), 64, 0, st>>>(nMB, meshBody, world, worldMesh, M, pos, rot, geom, hs, cd,
	                                                   slotBase, ctN, ctP, state, rest);
	k_np_mesh_rest<<<thinGrid(nMB), 64, 0, st>>>(rest, meshBody, world, worldMesh, M, pos, rot, geom, hs, cd, slotBase,
	                                             ctN, ctP, state);
}
void launch_sleep_wake_bodies(int k, const int* bodies, SleepState ss, hipStream_t st)
{
	PXH_LAUNCH(k_sleep_wake_bodies, k, k, bodies, ss);
}
void launch_sleep_read(int n, SleepState ss, float* wc, int* asleep, hipStream_t st)
{
	PXH_LAUNCH(k_sleep_read, n, n, ss, wc, asleep);
}
void launch_joint_prep(int J, const int4* info, const float4* frame, const float4* param, const float4* pos,
                       const float4* rot, SolverBodies sb, float stepDt, float invStepDt, float invDt, float erp,
                       float lengthScale, float4* head, float4* rows, const uint32_t* sleepFlags, hipStream_t st)
{
	if (J > 0)
		k_joint_prep<<<thinGrid(J), 64, 0, st>>>(J, info, frame, param, pos, rot, sb.vel, sb.rec, sb.i0, sb.i1, stepDt,
		                                         invStepDt, invDt, erp, lengthScale, head, rows, sleepFlags);
}
void launch_joint_solve(int begin, int end, const int4* info, const float4* head, float4* rows, SolverBodies sb,
                        float elapsed, bool conclude, const uint32_t* sleepFlags, hipStream_t st)
{
	if (end <= begin)
		return;
	k_joint_solve<<<nblk(end - begin, 64), 64, 0, st>>>(begin, end, info, head, rows, sb.vel, sb.dq, sb.i0, sb.i1,
	                                                     elapsed, conclude ? 1 : 0, sleepFlags);
}
void launch_con_build(int S, int Q, int pairEnd, const uint32_t* dP, const float4* ctN, uint32_t* flags,
                      uint32_t* scanTmp, const uint2* pairs, const int* qBody, const int* qPlane, const int* meshBody,
                      int nPlanes, const int* local, const int* planeLocal, const int* world, const int* worldTag,
                      const uint32_t* overflow, int* conA, int* conB, int* conSlot, uint64_t* conKey,
                      uint64_t* conPKey, int* conColor, uint32_t* hostCounts, hipStream_t st)
{
	const int nb = std::max(nblk(S, CON_TILE), 1);
	k_touch_flags<<<nb, CON_THREADS, 0, st>>>(S, Q, pairEnd, dP, ctN, flags, scanTmp);
	const bool scanned = nb > SUMS_DIRECT;
	if (scanned)
		launch_scan(scanTmp, nb, scanTmp + nb, st);
	auto kernel = scanned ? k_con_build<true> : k_con_build<false>;
	kernel<<<nb, CON_THREADS, 0, st>>>(S, Q, pairEnd, dP, flags, scanTmp, pairs, qBody, qPlane, meshBody, nPlanes, local,
	                                   planeLocal, world, worldTag, overflow, conA, conB, conSlot, conKey, conPKey,
	                                   conColor, hostCounts);
}

__global__ void k_gather4(int n, const int* idx, const uint32_t* in, uint32_t* out)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		out[i] = in[idx[i]];
}
__global__ void k_gather16(int n, const int* idx, const float4* in, float4* out)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		out[i] = in[idx[i]];
}
void launch_gather(int n, const int* idx, const void* in, void* out, int bytes, hipStream_t st)
{
	if (bytes == 16)
		PXH_LAUNCH(k_gather16, n, n, idx, static_cast<const float4*>(in), static_cast<float4*>(out));
	else
		PXH_LAUNCH(k_gather4, n, n, idx, static_cast<const uint32_t*>(in), static_cast<uint32_t*>(out));
}
// colouring launches are grid-stride over at most 1024 blocks
static int colorBlocks(int m) { return std::max(1, std::min(nblk(m, 256), 1024)); }
void launch_color_rounds(int m, const uint32_t* mDev, const int* list, int firstRound, int rounds, int n,
                         const int* conA, const int* conB, const uint64_t* conKey, int* conColor, uint64_t* best,
                         ColorState cs, int* out, uint32_t* left, uint32_t* ran, bool oneBlock, hipStream_t st)
{
	unsigned long long* bst = reinterpret_cast<unsigned long long*>(best);
	if (oneBlock)
	{
		k_color_rounds<<<1, ROUND_THREADS, 0, st>>>(mDev, COLOR_SHORT_LIST, list, firstRound, rounds, n, conA, conB,
		                                            conKey, conColor, bst, cs, out, left, ran);
		return;
	}
	const int g = colorBlocks(m);
	k_color_reset<<<g, 256, 0, st>>>(m, mDev, list, conA, conB, bst);
	for (int r = 0; r < rounds; r++)
	{
		unsigned long long* cur = bst + (r & 1) * int64_t(n);
		unsigned long long* nxt = bst + ((r + 1) & 1) * int64_t(n);
		k_color_min<<<g, 256, 0, st>>>(m, mDev, list, conA, conB, conKey, conColor, cur);
		k_color_pick<<<g, 256, 0, st>>>(m, mDev, list, firstRound + r, conA, conB, conKey, conColor, cur, nxt, cs);
	}
	k_fill_u32<<<1, 64, 0, st>>>(left, 1, 0u);
	k_color_left<<<g, 256, 0, st>>>(m, mDev, list, conColor, out, left, ran, uint32_t(rounds));
}
void launch_color_mask(int C, const int* conA, const int* conB, const int* conColor, ColorState cs, hipStream_t st)
{
	PXH_LAUNCH(k_color_mask, C, C, conA, conB, conColor, cs);
}
void launch_patch_table(int m, const uint64_t* keys, ulonglong2* table, uint32_t mask, hipStream_t st)
{
	PXH_LAUNCH(k_fill_u64, 2 * int64_t(mask) + 2, reinterpret_cast<uint64_t*>(table), 2 * int64_t(mask) + 2, ~0ull);
	PXH_LAUNCH(k_patch_insert, m, m, keys, reinterpret_cast<unsigned long long*>(table), mask);
}
void launch_con_prev(int C, const int* conA, const int* conB, const int* conSlot, PatchIO io, int* conColor,
                     ColorState cs, int* list, hipStream_t st)
{
	PXH_LAUNCH(k_con_prev, C, C, conA, conB, conSlot, io, conColor, cs, list);
}
void launch_color_keys(int C, const int* conA, const int* conB, int nPlanes, int* conColor, ColorState cs,
                       uint32_t limit, uint64_t* keys, uint32_t* vals, hipStream_t st)
{
	PXH_LAUNCH(k_color_keys, C, C, conA, conB, nPlanes, conColor, cs, limit, keys, vals);
}
void launch_preintegrate(int n, const float4* pos, const float4* rot, const float4* lin, const float4* ang,
                         const float4* invI, float3 gdt, float linDampDt, float angDampDt, float maxLinSq,
                         float maxAngSq, bool pgs, SolverBodies sb, float dt, float4* extLin, float4* extAng,
                         float4* prevLin, float4* prevAng, const uint32_t* sleepFlags, hipStream_t st)
{
	PXH_LAUNCH(k_preintegrate, n, n, pos, rot, lin, ang, invI, gdt, linDampDt, angDampDt, maxLinSq, maxAngSq, pgs ? 1 : 0, sb.vel,
	           sb.p, sb.dq, sb.i0, sb.i1, sb.origLin, sb.rec, dt, extLin, extAng, prevLin, prevAng, sleepFlags);
}
void launch_prep(int C, const int* order, const int* conA, const int* conB, const int* conSlot, const float4* ctN,
                 const float4* ctP, const float4* pos, const float4* rot, SolverBodies sb, float invStepDt,
                 float scale, float restDist, float fot, Rows rows, PatchIO patches, unsigned long long* counters,
                 unsigned long long* hostCounters, hipStream_t st)
{
	(void)pos;
	(void)rot;
	(void)conA;
	(void)conB;
	(void)conSlot;
	PXH_LAUNCH(k_prep, C, C, order, ctN, ctP, sb.rec, invStepDt, scale, restDist, fot, rows, patches, counters);
	k_sum_counters<<<1, 256, 0, st>>>(nblk(C, 256), counters, hostCounters);
}
void launch_solve(int begin, int end, int C, Rows rows, SolverBodies sb, float minPen, float muS, float muD,
                  float invStepDt, float biasScale, float scale, uint32_t* broken, hipStream_t st, hipEvent_t evStart,
                  hipEvent_t evStop)
{
	if (end <= begin)
		return;
	const dim3 grid(nblk(end - begin, SOLVE_THREADS)), block(SOLVE_THREADS);
	if (evStart)
		hipExtLaunchKernelGGL(k_solve, grid, block, 0, st, evStart, evStop, 0, begin, end, C, rows, sb.vel, minPen,
		                      muS, muD, invStepDt, biasScale, scale, broken);
	else
		k_solve<<<grid, block, 0, st>>>(begin, end, C, rows, sb.vel, minPen, muS, muD, invStepDt, biasScale, scale,
		                                broken);
}
void launch_color_keys_world(int C, const int* conA, const int* conB, int nPlanes, int* conColor, ColorState cs,
                             const int* bodyWorld, uint32_t limit, uint64_t* keys, uint32_t* vals, hipStream_t st)
{
	PXH_LAUNCH(k_color_keys_world, C, C, conA, conB, nPlanes, conColor, cs, bodyWorld, limit, keys, vals);
}
void launch_fill_u32(uint32_t* p, int64_t n, uint32_t v, hipStream_t st)
{
	PXH_LAUNCH(k_fill_u32, n, p, n, v);
}
template <int THREADS, bool PGS, bool JOINTS>
static void solveWorlds(int grid, size_t shm, uint32_t* queueHead, hipStream_t st, hipEvent_t evStart,
                        hipEvent_t evStop, int nWorlds, const int* worldOrder, const int* bodyStart,
                        const uint32_t* segStart, int CB, int C, const Rows& rows, const float* rowsU,
                        const SolverBodies& sb, int posIters, int iters, float stepDt, float muS, float muD,
                        float invStepDt, float biasScale, float scale, uint32_t* broken, int ldsBodies,
                        const WorldJoints& joints)
{
	auto kernel = k_solve_worlds<THREADS, PGS, JOINTS>;
	if (evStart)
		hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(THREADS), shm, st, evStart, evStop, 0, nWorlds, worldOrder,
		                      queueHead, bodyStart, segStart, CB, C, rows, rowsU, sb, posIters, iters, stepDt, muS, muD,
		                      invStepDt, biasScale, scale, broken, ldsBodies, joints);
	else
		kernel<<<grid, THREADS, shm, st>>>(nWorlds, worldOrder, queueHead, bodyStart, segStart, CB, C, rows, rowsU, sb,
		                                   posIters, iters, stepDt, muS, muD, invStepDt, biasScale, scale, broken,
		                                   ldsBodies, joints);
}
void launch_solve_worlds(int workgroups, int nWorlds, int maxWorldBodies, const int* worldOrder, uint32_t* queueHead,
                         const int* bodyStart, const uint32_t* segStart, int CB, int C, Rows rows, const float* rowsU,
                         SolverBodies sb, int posIters, int iters, float stepDt, float muS, float muD,
                         float invStepDt, float biasScale, float scale, uint32_t* broken, int ldsBodies,
                         const WorldJoints& joints, hipStream_t st, hipEvent_t evStart, hipEvent_t evStop)
{
	if (nWorlds <= 0)
		return;
	int dev = 0, cus = 256;
	(void)hipGetDevice(&dev);
	(void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
	// One wave a world while the worlds fill the chip (their colours rarely have
	// more than 64 rows), four where they do not: 301 worlds of up to 512 bodies
	// step in 602 us with one and in 530 with four, 8,192 worlds in 2.26 and 2.77 ms.
	const int threads = nWorlds < 4 * cus && maxWorldBodies > 64 ? 256 : 64;
	ldsBodies = std::min(ldsBodies, WORLD_LDS_BODIES);
	const size_t shm = sizeof(float4) * 2 * size_t(ldsBodies) + sizeof(uint32_t) * (size_t(CB) + 1);
	// as many as run at a time: by LDS (160 KB a compute unit) and registers (8 waves)
	const int perCu = std::max(1, std::min(int(163840 / (shm + 64)), 512 / threads));
	const int grid = std::min(workgroups > 0 ? workgroups : perCu * cus, nWorlds);
	// the queue starts at zero (a fill kernel, no memset packet)
	k_fill_u32<<<1, 64, 0, st>>>(queueHead, 1, 0u);
	auto run = [&](auto t, auto pgs, auto j) {
		solveWorlds<decltype(t)::value, decltype(pgs)::value, decltype(j)::value>(
		    grid, shm, queueHead, st, evStart, evStop, nWorlds, worldOrder, bodyStart, segStart, CB, C, rows, rowsU, sb,
		    posIters, iters, stepDt, muS, muD, invStepDt, biasScale, scale, broken, ldsBodies, joints);
	};
	auto kind = [&](auto t) {
		if (rowsU)
			run(t, std::true_type(), std::false_type());
		else if (joints.colors > 0)
			run(t, std::false_type(), std::true_type());
		else
			run(t, std::false_type(), std::false_type());
	};
	if (threads == 256)
		kind(std::integral_constant<int, 256>());
	else
		kind(std::integral_constant<int, 64>());
}

void launch_prep_pgs(int C, const int* order, const int* conA, const int* conB, const int* conSlot,
                     const float4* ctN, const float4* ctP, const float4* pos, const float4* rot, SolverBodies sb,
                     float invDt, float muS, float muD, float restDist, float fot, Rows rows, float* rowsU,
                     PatchIO patches, unsigned long long* counters, unsigned long long* hostCounters, hipStream_t st)
{
	(void)pos;
	(void)rot;
	(void)conA;
	(void)conB;
	(void)conSlot;
	PXH_LAUNCH(k_prep_pgs, C, C, order, ctN, ctP, sb.rec, invDt, muS, muD, restDist, fot, rows, rowsU, patches,
	           counters);
	k_sum_counters<<<1, 256, 0, st>>>(nblk(C, 256), counters, hostCounters);
}
void launch_solve_pgs(int begin, int end, int C, Rows rows, const float* rowsU, SolverBodies sb, bool doFriction,
                      bool velocityPass, uint32_t* broken, hipStream_t st, hipEvent_t evStart, hipEvent_t evStop)
{
	if (end <= begin)
		return;
	const dim3 grid(nblk(end - begin, SOLVE_THREADS)), block(SOLVE_THREADS);
	if (evStart)
		hipExtLaunchKernelGGL(k_solve_pgs, grid, block, 0, st, evStart, evStop, 0, begin, end, C, rows, rowsU, sb.vel,
		                      doFriction ? 1 : 0, velocityPass ? 1 : 0, broken);
	else
		k_solve_pgs<<<grid, block, 0, st>>>(begin, end, C, rows, rowsU, sb.vel, doFriction ? 1 : 0,
		                                    velocityPass ? 1 : 0, broken);
}
void launch_pgs_save_motion(int n, SolverBodies sb, hipStream_t st)
{
	PXH_LAUNCH(k_pgs_save_motion, n, n, sb.vel, sb.p, sb.dq);
}
void launch_pgs_finalize(int n, float dt, float4* pos, float4* rot, float4* lin, float4* ang, const float4* invI,
                         SolverBodies sb, SleepState ss, hipStream_t st)
{
	PXH_LAUNCH(k_pgs_finalize, n, n, dt, pos, rot, lin, ang, invI, sb.vel, sb.p, sb.dq, sb.i0, sb.i1, ss);
}
void launch_integrate(int n, float dt, SolverBodies sb, hipStream_t st)
{
	PXH_LAUNCH(k_integrate, n, n, dt, sb.vel, sb.p, sb.dq, sb.i0, sb.i1);
}
void launch_finalize(int n, float dt, float4* pos, float4* rot, float4* lin, float4* ang, const float4* invI,
                     SolverBodies sb, SleepState ss, hipStream_t st)
{
	PXH_LAUNCH(k_finalize, n, n, dt, pos, rot, lin, ang, invI, sb.vel, sb.p, sb.dq, sb.i0, sb.i1, ss);
}
void launch_get_data(int n, const uint32_t* idx, int what, const float4* pos, const float4* rot, const float4* lin,
                     const float4* ang, const float4* prevLin, const float4* prevAng, float invDt, float* out,
                     hipStream_t st)
{
	PXH_LAUNCH(k_get_data, n, n, idx, what, pos, rot, lin, ang, prevLin, prevAng, invDt, out);
}
void launch_set_data(int n, const uint32_t* idx, int what, float4* pos, float4* rot, float4* lin, float4* ang,
                     const float4* invI, float4* extLin, float4* extAng, const float* in, SleepState ss,
                     hipStream_t st)
{
	PXH_LAUNCH(k_set_data, n, n, idx, what, pos, rot, lin, ang, invI, extLin, extAng, in, ss);
}
void launch_touch_events(int C, const int* prevRow, int R, uint32_t* found, uint32_t* matched, uint32_t* lost,
                         hipStream_t st)
{
	PXH_LAUNCH(k_fill_u32, int64_t(R) + 1, matched, int64_t(R) + 1, 0u);
	PXH_LAUNCH(k_found_flags, C, C, prevRow, found, matched);
	PXH_LAUNCH(k_lost_flags, R, R, matched, lost);
}
void launch_pair_keys(int P, const uint2* pairs, const uint32_t* ids, uint64_t* keys, uint32_t* vals, hipStream_t st)
{
	PXH_LAUNCH(k_pair_keys, P, P, pairs, ids, keys, vals);
}
void launch_set_diff(int na, const uint64_t* a, int nb, const uint64_t* b, uint32_t* flag, hipStream_t st)
{
	PXH_LAUNCH(k_set_diff_flags, na, na, a, nb, b, flag);
}
void launch_compact_keys(int na, const uint64_t* a, const uint32_t* flag, const uint32_t* scanned, uint2* out,
                         hipStream_t st)
{
	PXH_LAUNCH(k_compact_keys, na, na, a, flag, scanned, out);
}

void launch_np_immediate(int n, const int* type0, const float* geom0, const float* pose0, const int* type1,
                         const float* geom1, const float* pose1, float cd, float tol, float* out, int* counts,
                         hipStream_t st)
{
	if (n > 0)
		k_np_immediate<<<nblk(n, NP_THREADS), NP_THREADS, 0, st>>>(n, type0, geom0, pose0, type1, geom1, pose1, cd, tol,
		                                                           out, counts);
}

__global__ void k_bp_inflate(int n, const float* bounds, const float* dist, const uint32_t* groups, float4* bmin,
                             float4* bmax, int* scene, int* group, int* bodyStart)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i == 0)
	{
		bodyStart[0] = 0;
		bodyStart[1] = n;
	}
	if (i >= n)
		return;
	const float* b = bounds + 6 * int64_t(i);
	const float d = dist ? dist[i] : 0.0f;
	// geometry type slot unused by the standalone broadphase (all pairs class 2)
	bmin[i] = make_float4(b[0] - d, b[1] - d, b[2] - d, float(GEOM_BOX));
	bmax[i] = make_float4(b[3] + d, b[4] + d, b[5] + d, 0.0f);
	scene[i] = 0;
	group[i] = groups ? int(groups[i]) : i;
}

void launch_bp_inflate(int n, const float* bounds, const float* dist, const uint32_t* groups, float4* bmin,
                       float4* bmax, int* scene, int* group, int* bodyStart, hipStream_t st)
{
	k_bp_inflate<<<nblk(n > 0 ? n : 1, 256), 256, 0, st>>>(n, bounds, dist, groups, bmin, bmax, scene, group,
	                                                       bodyStart);
}

}  // namespace pxh
