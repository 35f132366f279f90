/*
 * BVH builds on the device (linear BVH and PLOC), written into the 4-wide or
 * 8-wide node records of lrh_layout.h.  The per-element steps are
 * lrh_lbvh.h's (shared with the CPU emulation); here they run as kernels:
 *   1. leaf boxes and the bounds of their centres;
 *   2. 63-bit Morton codes over a cube of cells, sorted with the triangle id
 *      as value by a stable LSD radix sort (8-bit digits: per-tile digit
 *      counts, an exclusive scan of each digit's row of the [digit][tile]
 *      table, a scatter that ranks equal digits in index order with wave
 *      ballots, stages the tile in LDS in sorted order and writes each digit's
 *      run coalesced), then checked to be in order;
 *   3. a binary tree over the sorted leaves: the radix tree (LBVH) or
 *      agglomerative clustering in rounds of mutual nearest neighbours
 *      within 16 places (PLOC), brought into the radix tree's form;
 *   4. boxes bottom-up -- LBVH: nodes ordered by the length of their common
 *      prefix, a launch per length (runs of short ones in one block); PLOC: as
 *      the clusters merge -- and surface-area costs, which decide whether a
 *      node of at most maxLeaf triangles becomes one leaf;
 *   5. breadth-first collapse into 4- or 8-wide nodes, child slots from an
 *      exclusive scan, so the node order is deterministic; level sizes stay on
 *      the device, the host looks at them once per few levels;
 *   6. triangle records in leaf order, bit for bit the host records.
 * Every kernel runs a bounded amount of work: no block waits on another
 * (the sort and the scans are sequences of kernels, not decoupled
 * look-back), every search loop has a step bound, and a violated
 * precondition sets a bit of an error word (or fails a host check of a
 * count read back) that the host reports as an error instead of going on.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <stdexcept>
#include <string>
#include <type_traits>
#include <vector>

#include "lrh_devnode.h"
#include "lrh_gpubuild.h"
#include "lrh_layout.h"
#include "lrh_lbvh.h"

namespace {

using namespace lrhlbvh;

#define GB_CHECK(x)                                                                                   \
	do {                                                                                              \
		const hipError_t e_ = (x);                                                                    \
		if (e_ != hipSuccess) throw std::runtime_error(std::string("device build: ") + hipGetErrorString(e_)); \
	} while (0)

__global__ void k_fill(uint32_t *p, uint32_t n, uint32_t v) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n) p[i] = v;
}

// 1. leaf boxes and centre bounds: a grid-stride loop, the bounds reduced
// in registers, across the wave by lane exchanges and across the block in
// LDS, one partial result a block (six atomics a block to the same line
// bounded the kernel: 105 us for 2.29M triangles, now 38 and 5 for the
// reduction).  A vertex index outside its mesh sets the error and is not
// followed; the host looks at the error before anything else reads vertices,
// so meshes need no pass over their indices on the host first.
constexpr uint32_t kPrimBlocks = 2048;
__device__ __forceinline__ uint32_t minU(uint32_t a, uint32_t b) { return a < b ? a : b; }
__device__ __forceinline__ uint32_t maxU(uint32_t a, uint32_t b) { return a > b ? a : b; }

__global__ __launch_bounds__(256) void k_prims(const float *__restrict__ verts, const uint32_t *__restrict__ tris,
		const uint32_t *__restrict__ tbase, const uint32_t *__restrict__ vbase, uint32_t nMeshes, uint32_t n,
		GBox *__restrict__ boxes, uint32_t *__restrict__ partial, uint32_t *err) {
	uint32_t mn[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, mx[3] = {0u, 0u, 0u};
	for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
		// the wave's first triangle's mesh is most lanes' mesh
		uint32_t m = meshOf(tbase, nMeshes, (uint32_t)__builtin_amdgcn_readfirstlane((int)i));
		if (i >= tbase[m + 1]) m = meshOf(tbase, nMeshes, i);
		const uint32_t v0 = vbase[m], nv = vbase[m + 1] - v0;
		float p[3][3];
		bool bad = false;
		for (int c = 0; c < 3; ++c) {
			const uint32_t v = tris[3 * (size_t)i + c];
			bad |= v >= nv;
			for (int k = 0; k < 3; ++k) p[c][k] = v < nv ? verts[3 * ((size_t)v0 + v) + k] : 0.f;
		}
		if (bad) atomicOr(err, kErrIndex);
		const GBox b = boxOf(p);
		boxes[i] = b;
		for (int k = 0; k < 3; ++k) {
			const uint32_t c = lrhdev::fkey(b.lo[k] + b.hi[k]);
			mn[k] = minU(mn[k], c);
			mx[k] = maxU(mx[k], c);
		}
	}
	for (int k = 0; k < 3; ++k)
		for (int o = 32; o > 0; o >>= 1) {
			mn[k] = minU(mn[k], (uint32_t)__shfl_xor((int)mn[k], o));
			mx[k] = maxU(mx[k], (uint32_t)__shfl_xor((int)mx[k], o));
		}
	__shared__ uint32_t smin[4][3], smax[4][3];
	const uint32_t wave = threadIdx.x >> 6;
	if ((threadIdx.x & 63u) == 0)
		for (int k = 0; k < 3; ++k) {
			smin[wave][k] = mn[k];
			smax[wave][k] = mx[k];
		}
	__syncthreads();
	if (threadIdx.x < 3) {
		const uint32_t k = threadIdx.x;
		uint32_t a = smin[0][k], b = smax[0][k];
		for (uint32_t w = 1; w < blockDim.x / 64; ++w) {
			a = minU(a, smin[w][k]);
			b = maxU(b, smax[w][k]);
		}
		partial[6 * blockIdx.x + k] = a;
		partial[6 * blockIdx.x + 3 + k] = b;
	}
}

// the blocks' partial bounds to one, a wave per bound
__global__ __launch_bounds__(384) void k_bounds(const uint32_t *partial, uint32_t nBlocks, uint32_t *cb) {
	const uint32_t k = threadIdx.x >> 6, lane = threadIdx.x & 63u;
	uint32_t v = k < 3 ? 0xffffffffu : 0u;
#pragma unroll 8
	for (uint32_t b = lane; b < nBlocks; b += 64) {
		const uint32_t x = partial[6 * b + k];
		v = k < 3 ? minU(v, x) : maxU(v, x);
	}
	for (int o = 32; o > 0; o >>= 1) {
		const uint32_t x = (uint32_t)__shfl_xor((int)v, o);
		v = k < 3 ? minU(v, x) : maxU(v, x);
	}
	if (lane == 0) cb[k] = v;
}

// 2. Morton codes of the box centres
__global__ void k_morton(const GBox *boxes, uint32_t n, const uint32_t *cbIn, uint64_t *keys, uint32_t *vals) {
	__shared__ uint32_t cb[6];
	if (threadIdx.x < 6) cb[threadIdx.x] = cbIn[threadIdx.x];
	__syncthreads();
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n) return;
	keys[i] = mortonKey(boxes[i], cb);
	vals[i] = i;
}

// ---- radix sort pass: per-tile digit counts, table [digit][tile] ----
// tiles of kSortTile keys, or of kSortTileSmall up to kSortSmall keys: there
// the large tiles leave compute units without a block, and a tile's eight
// rounds run one after another (the scatter of 50,000 keys: 12.8 us, now 6)
constexpr uint32_t kSortTileSmall = 512, kSortSmall = 512 * 1024;
uint32_t sortTiles(uint32_t n) {
	const uint32_t tile = n <= kSortSmall ? kSortTileSmall : kSortTile;
	return (uint32_t)(((uint64_t)n + tile - 1) / tile);
}

template <uint32_t TILE>
__global__ __launch_bounds__(kSortBlock) void k_sortCount(const uint64_t *keys, uint32_t n, uint32_t shift,
		uint32_t nTiles, uint32_t *table) {
	__shared__ uint32_t cnt[256];
	cnt[threadIdx.x] = 0;
	__syncthreads();
	const uint64_t base = (uint64_t)blockIdx.x * TILE;
	for (uint32_t j = threadIdx.x; j < TILE; j += kSortBlock) {
		const uint64_t idx = base + j;
		if (idx < n) atomicAdd(&cnt[digitOf(keys[idx], shift)], 1u);
	}
	__syncthreads();
	table[(size_t)threadIdx.x * nTiles + blockIdx.x] = cnt[threadIdx.x];
}

// ---- radix sort pass: stable scatter.  A tile is taken in rounds of 256
// consecutive keys, one per thread in index order; a key's place within the
// tile is its digit's start in the tile (a scan of the tile's digit counts)
// + the tile's earlier keys of that digit (earlier rounds) + the earlier
// waves' keys of that digit in this round + its rank among the lanes of its
// wave with the same digit (ballots over the eight digit bits).  Keys and
// values are first placed in LDS in that order, then written out in place
// order, so consecutive threads write consecutive addresses of one digit's
// run (its global start from the scanned [digit][tile] table). ----
template <uint32_t TILE>
__global__ __launch_bounds__(kSortBlock) void k_sortScatter(const uint64_t *keysIn, const uint32_t *valsIn, uint32_t n,
		uint32_t shift, uint32_t nTiles, const uint32_t *offsets, const uint32_t *totals, uint64_t *keysOut,
		uint32_t *valsOut, uint32_t *err) {
	constexpr uint32_t kWaves = kSortBlock / 64;
	__shared__ uint32_t run[256];
	__shared__ uint32_t wcnt[kWaves][256];
	__shared__ uint32_t off[256];    // global start of each digit's run for this tile
	__shared__ uint32_t start[256];  // each digit's start within the tile
	__shared__ uint32_t base[256];   // each digit's start in the whole output
	__shared__ uint64_t sKey[TILE];
	__shared__ uint32_t sVal[TILE];
	const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63u;
	const uint64_t tile0 = (uint64_t)blockIdx.x * TILE;
	const uint32_t tileN = (uint32_t)((n - tile0) < TILE ? (n - tile0) : TILE);
	// the tile's digit counts, scanned to starts
	run[tid] = 0;
	for (uint32_t w = 0; w < kWaves; ++w) wcnt[w][tid] = 0;
	off[tid] = offsets[(size_t)tid * nTiles + blockIdx.x];
	const uint32_t total = totals[tid];
	base[tid] = total;
	__syncthreads();
	for (uint32_t j = tid; j < tileN; j += kSortBlock) atomicAdd(&run[digitOf(keysIn[tile0 + j], shift)], 1u);
	__syncthreads();
	start[tid] = run[tid];
	__syncthreads();
	for (uint32_t o = 1; o < 256; o <<= 1) {  // inclusive scans (Hillis-Steele)
		const uint32_t add = tid >= o ? start[tid - o] : 0u, add2 = tid >= o ? base[tid - o] : 0u;
		__syncthreads();
		start[tid] += add;
		base[tid] += add2;
		__syncthreads();
	}
	start[tid] -= run[tid];  // exclusive
	off[tid] += base[tid] - total;
	run[tid] = 0;
	__syncthreads();
	const uint64_t lanesBelow = (1ull << lane) - 1ull;
	for (uint32_t r = 0; r < TILE / kSortBlock; ++r) {
		const uint32_t j = r * kSortBlock + tid;
		const bool valid = j < tileN;
		const uint64_t key = valid ? keysIn[tile0 + j] : 0ull;
		const uint32_t val = valid ? valsIn[tile0 + j] : 0u;
		const uint32_t dg = valid ? digitOf(key, shift) : 0u;
		uint64_t same = __ballot(valid);
		for (uint32_t b = 0; b < 8; ++b) {
			const bool bit = (dg >> b) & 1u;
			const uint64_t m = __ballot(bit);
			same &= bit ? m : ~m;
		}
		const uint32_t rank = (uint32_t)__popcll(same & lanesBelow);
		if (valid && rank == 0) wcnt[wave][dg] = (uint32_t)__popcll(same);
		__syncthreads();
		if (valid) {
			uint32_t before = run[dg];
			for (uint32_t w = 0; w < wave; ++w) before += wcnt[w][dg];
			const uint32_t p = start[dg] + before + rank;
			if (p < TILE) {
				sKey[p] = key;
				sVal[p] = val;
			} else {
				atomicOr(err, kErrUnsorted);  // a place outside the tile: never written
			}
		}
		__syncthreads();
		uint32_t add = 0;
		for (uint32_t w = 0; w < kWaves; ++w) {
			add += wcnt[w][tid];
			wcnt[w][tid] = 0;
		}
		run[tid] += add;
		__syncthreads();
	}
	// out in place order: one digit's run is contiguous in the tile and in
	// the output
	for (uint32_t p = tid; p < tileN; p += kSortBlock) {
		const uint64_t key = sKey[p];
		const uint32_t dg = digitOf(key, shift);
		const uint32_t pos = off[dg] + (p - start[dg]);
		if (pos < n) {
			keysOut[pos] = key;
			valsOut[pos] = sVal[p];
		} else {
			atomicOr(err, kErrUnsorted);
		}
	}
}

// exclusive scan of each digit's row of the [digit][tile] table, a block per
// digit, and the row's total; the scatter adds the digits' starts, so a pass
// is three launches (five when the whole table was scanned as one array)
__global__ __launch_bounds__(256) void k_scanRows(uint32_t *table, uint32_t nTiles, uint32_t *totals) {
	constexpr uint32_t kPer = 8;
	__shared__ uint32_t part[256];
	uint32_t *row = table + (size_t)blockIdx.x * nTiles;
	uint32_t carry = 0;
	for (uint32_t t0 = 0; t0 < nTiles; t0 += 256 * kPer) {
		const uint32_t b = t0 + threadIdx.x * kPer;
		uint32_t v[kPer], sum = 0;
		for (uint32_t k = 0; k < kPer; ++k) {
			v[k] = b + k < nTiles ? row[b + k] : 0u;
			sum += v[k];
		}
		part[threadIdx.x] = sum;
		__syncthreads();
		for (uint32_t o = 1; o < 256; o <<= 1) {
			const uint32_t add = threadIdx.x >= o ? part[threadIdx.x - o] : 0u;
			__syncthreads();
			part[threadIdx.x] += add;
			__syncthreads();
		}
		uint32_t run = carry + part[threadIdx.x] - sum;
		for (uint32_t k = 0; k < kPer; ++k) {
			if (b + k < nTiles) row[b + k] = run;
			run += v[k];
		}
		carry += part[255];
		__syncthreads();
	}
	if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// exclusive prefix of v over the 256 threads of a block; `sum` gets the total
__device__ __forceinline__ uint32_t blockPrefix(uint32_t v, uint32_t *lds /* 4 */, uint32_t &sum) {
	uint32_t incl = v;
	for (int o = 1; o < 64; o <<= 1) {
		const uint32_t x = (uint32_t)__shfl_up((int)incl, o);
		if ((int)(threadIdx.x & 63u) >= o) incl += x;
	}
	if ((threadIdx.x & 63u) == 63u) lds[threadIdx.x >> 6] = incl;
	__syncthreads();
	uint32_t before = 0;
	sum = 0;
	for (uint32_t w = 0; w < 4; ++w) {
		if (w < (threadIdx.x >> 6)) before += lds[w];
		sum += lds[w];
	}
	return before + incl - v;
}

// exclusive scan of n values in place by one block of 1024 threads, eight
// values a thread and turn; returns the total to every thread
__device__ uint32_t scanByBlock(uint32_t *v, uint32_t n, uint32_t *lds /* 16 */) {
	constexpr uint32_t kPer = 8;
	uint32_t carry = 0;
	for (uint32_t t0 = 0; t0 < n; t0 += 1024 * kPer) {
		const uint32_t b = t0 + threadIdx.x * kPer;
		uint32_t x[kPer], sum = 0;
		for (uint32_t k = 0; k < kPer; ++k) {
			x[k] = b + k < n ? v[b + k] : 0u;
			sum += x[k];
		}
		uint32_t incl = sum;
		for (int o = 1; o < 64; o <<= 1) {
			const uint32_t y = (uint32_t)__shfl_up((int)incl, o);
			if ((int)(threadIdx.x & 63u) >= o) incl += y;
		}
		if ((threadIdx.x & 63u) == 63u) lds[threadIdx.x >> 6] = incl;
		__syncthreads();
		uint32_t run = carry + incl - sum, all = 0;
		for (uint32_t w = 0; w < 16; ++w) {
			if (w < (threadIdx.x >> 6)) run += lds[w];
			all += lds[w];
		}
		for (uint32_t k = 0; k < kPer; ++k) {
			if (b + k < n) v[b + k] = run;
			run += x[k];
		}
		carry += all;
		__syncthreads();
	}
	return carry;
}

__global__ void k_checkSorted(const uint64_t *keys, uint32_t n, uint32_t *err) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i + 1 < n && keys[i] > keys[i + 1]) atomicOr(err, kErrUnsorted);
}

// 3. binary radix tree.  digits: 127 - the length of the node's common prefix
// (at most 64 key bits and 32 of position), so a node's children have smaller
// digits than it.  A node without a key range (codes out of order) sets the
// error and becomes two leaves, so that nothing after it reads out of bounds
// before the host sees the error.
constexpr uint32_t kDigits = 128;
__global__ void k_radixTree(const uint64_t *keys, uint32_t n, uint32_t *left, uint32_t *right, uint32_t *first,
		uint32_t *last, uint64_t *digits, uint32_t *ids, uint32_t *err) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i + 1 >= n) return;
	uint32_t lc, rc, lo, hi;
	if (!radixNode(keys, n, i, lc, rc, lo, hi)) {
		atomicOr(err, kErrRange);
		lc = kLeafBit | i;
		rc = kLeafBit | (i + 1);
		lo = i;
		hi = i + 1;
	}
	left[i] = lc;
	right[i] = rc;
	first[i] = lo;
	last[i] = hi;
	const int d = delta(keys, n, lo, hi);
	digits[i] = (uint64_t)(kDigits - 1u - (uint32_t)(d < 0 ? 0 : d > 127 ? 127 : d));
	ids[i] = i;
}

// 4. the first place of each digit in the sorted order
__global__ void k_digitStarts(const uint32_t *totals, uint32_t *out, uint32_t *host) {
	__shared__ uint32_t v[256];
	const uint32_t d = threadIdx.x;
	v[d] = totals[d];
	__syncthreads();
	for (uint32_t o = 1; o < 256; o <<= 1) {
		const uint32_t add = d >= o ? v[d - o] : 0u;
		__syncthreads();
		v[d] += add;
		__syncthreads();
	}
	if (d <= kDigits) out[d] = host[d] = v[d] - totals[d];
}

__global__ void k_leafBoxes(const GBox *boxes, const uint32_t *vals, uint32_t n, GBox *leafBox) {
	const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
	if (j >= n) return;
	const uint32_t v = vals[j];
	leafBox[j] = boxes[v < n ? v : 0u];  // (a failed sort's values are reported later)
}

// what the collapse compares: a node's area, or -1 if it becomes a leaf (an
// area is zero or more, but for boxes of NaN vertices, which may come out
// inverted and must not read as a leaf)
__device__ __forceinline__ float nodeKey(uint32_t leaf, float area) {
	return leaf ? -1.f : area == -1.f ? 0.f : area;
}

// box, surface-area cost and leaf decision of node x
__device__ __forceinline__ void boxNode(uint32_t x, const uint32_t *left, const uint32_t *right, const uint32_t *first,
		const uint32_t *last, const GBox *leafBox, uint32_t maxLeaf, float ci, GBox *nodeBox, float *cost, float *key) {
	const uint32_t l = left[x], r = right[x];
	const GBox a = (l & kLeafBit) ? leafBox[l & ~kLeafBit] : nodeBox[l];
	const GBox b = (r & kLeafBit) ? leafBox[r & ~kLeafBit] : nodeBox[r];
	const GBox u = unionBox(a, b);
	const float cl = (l & kLeafBit) ? areaOf(a) : cost[l];
	const float cr = (r & kLeafBit) ? areaOf(b) : cost[r];
	uint32_t lf;
	cost[x] = nodeCost(areaOf(u), cl, cr, last[x] - first[x] + 1u, maxLeaf, ci, lf);
	key[x] = nodeKey(lf, areaOf(u));
	nodeBox[x] = u;
}

// the nodes of one digit: the children's are done by earlier launches
__global__ void k_boxLevel(const uint32_t *order, uint32_t cnt, const uint32_t *left, const uint32_t *right,
		const uint32_t *first, const uint32_t *last, const GBox *leafBox, uint32_t maxLeaf, float ci, GBox *nodeBox,
		float *cost, float *key) {
	const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
	if (e < cnt) boxNode(order[e], left, right, first, last, leafBox, maxLeaf, ci, nodeBox, cost, key);
}

// the nodes of digits [d0, d1), each a few, by one block with a barrier after
// each digit: a launch per digit of a handful of nodes costs its launch (a
// 2.3M-triangle tree has 50 digits, half of them below 2,048 nodes)
constexpr uint32_t kSmallLevel = 2048;
__global__ __launch_bounds__(1024) void k_boxSmallLevels(const uint32_t *order, const uint32_t *starts, uint32_t d0,
		uint32_t d1, const uint32_t *left, const uint32_t *right, const uint32_t *first, const uint32_t *last,
		const GBox *leafBox, uint32_t maxLeaf, float ci, GBox *nodeBox, float *cost, float *key) {
	for (uint32_t d = d0; d < d1; ++d) {
		for (uint32_t e = starts[d] + threadIdx.x; e < starts[d + 1]; e += 1024)
			boxNode(order[e], left, right, first, last, leafBox, maxLeaf, ci, nodeBox, cost, key);
		__syncthreads();
	}
}

// 3'. clustering (PLOC): clusters start as the sorted leaves
struct PlocState;
__global__ void k_plocInit(const GBox *boxes, const uint32_t *vals, uint32_t n, uint32_t *cid, GBox *cbox,
		GBox *leafBox, PlocState *st) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < 4) reinterpret_cast<uint32_t *>(st)[i] = i == 0 ? n : 0u;
	if (i >= n) return;
	const uint32_t v = vals[i];
	const GBox b = boxes[v < n ? v : 0u];  // (a failed sort's values are reported later)
	leafBox[i] = b;
	cid[i] = kLeafBit | i;
	cbox[i] = b;
}

// a round's state, written by the round before: clusters, next node, whether
// the round pairs places 2k, 2k+1 (one that merged fewer than 1/64 of the
// clusters is followed by such a forced round)
struct PlocState {
	uint32_t nc, nodeBase, forced, pad;
};

// clusters of at most this many are finished by one block
constexpr uint32_t kPlocTail = 2048;
constexpr uint32_t kPlocMaxRounds = 4096;

// the kernels of a round run on an upper bound of clusters that the host
// knows; the state's count ends them, and a count at or below kPlocTail
// leaves the rest to the tail
__device__ __forceinline__ PlocState plocRound(const PlocState *st, uint32_t r) {
	PlocState s = st[r];
	if (s.nc <= kPlocTail) s.nc = 0;
	return s;
}

// The nearest neighbour of cluster i within kPlocRadius places: the smallest
// merged area, of equal areas the first pair by (lower, upper) place, so the
// first of all pairs is mutual and every round merges.  By L neighbouring
// lanes, each with every L-th place: of equal areas the lowest place wins, which
// is the order of the pairs (a pair with a lower place comes first by its lower
// end or, above i, by its upper)
template <uint32_t L, class BoxAt>
__device__ __forceinline__ uint32_t plocNearestLanes(const BoxAt &box, uint32_t nc, uint32_t i, uint32_t sub) {
	float best = INFINITY;
	uint32_t arg = kNone;
	if (i < nc) {
		const uint32_t lo = i > kPlocRadius ? i - kPlocRadius : 0u;
		const uint32_t hi = (nc - 1u - i > kPlocRadius) ? i + kPlocRadius : nc - 1u;
		const GBox ci = box(i);
		for (uint32_t j = lo + sub; j <= hi; j += L) {
			if (j == i) continue;
			const float a = mergedArea(ci, box(j));
			if (a < best || arg == kNone) {
				best = a;
				arg = j;
			}
		}
	}
	for (uint32_t o = L / 2; o > 0; o >>= 1) {
		const float a = __shfl_xor(best, (int)o);
		const uint32_t g = (uint32_t)__shfl_xor((int)arg, (int)o);
		if (a < best || (a == best && g < arg)) {
			best = a;
			arg = g;
		}
	}
	return arg == kNone ? i : arg;
}

// nearest neighbours of a tile of 256/L clusters, their boxes and the
// kPlocRadius on either side staged in LDS (each box is read by 2r+1 threads);
// L lanes a cluster.  A lane a cluster leaves a chain of 32 LDS reads and few
// waves to hide it up to kPlocSplit clusters, where four share it (50,000
// clusters: 12 us a round, now 5).
constexpr uint32_t kPlocSplit = 256 * 1024;
template <uint32_t L>
__global__ __launch_bounds__(256) void k_plocNearest(const GBox *cbox, const PlocState *st, uint32_t r, uint32_t *nn) {
	constexpr uint32_t kTile = 256 / L;
	constexpr uint32_t kSpan = kTile + 2 * kPlocRadius;
	__shared__ float tile[kSpan * 6];
	const uint32_t t0 = blockIdx.x * kTile;
	const PlocState s = plocRound(st, r);
	const uint32_t nc = s.forced ? 0u : s.nc;
	if (t0 >= nc) return;
	const int64_t base = (int64_t)t0 - kPlocRadius;  // cluster of tile entry 0
	const float *src = reinterpret_cast<const float *>(cbox);
	for (uint32_t k = threadIdx.x; k < kSpan * 6; k += 256) {
		const int64_t j = base + k / 6;
		tile[k] = (j >= 0 && j < (int64_t)nc) ? src[j * 6 + k % 6] : 0.f;
	}
	__syncthreads();
	const uint32_t i = t0 + threadIdx.x / L;
	const GBox *lds = reinterpret_cast<const GBox *>(tile);
	const uint32_t x = plocNearestLanes<L>([&](uint32_t j) -> const GBox & { return lds[(int64_t)j - base]; }, nc, i,
			threadIdx.x % L);
	if (i < nc && threadIdx.x % L == 0) nn[i] = x;
}

// partners and each cluster's place among the survivors and among the new
// nodes, within its block: lead (the lower place of a pair, a new node) counts
// in the upper half, keep (the place survives) in the lower
__global__ __launch_bounds__(256) void k_plocMark(const uint32_t *nn, const PlocState *st, uint32_t r, uint32_t *prefix,
		uint32_t *leadSums, uint32_t *keepSums) {
	const PlocState s = plocRound(st, r);
	if (blockIdx.x * 256u >= s.nc) return;
	__shared__ uint32_t lds[4];
	const uint32_t i = blockIdx.x * 256u + threadIdx.x;
	uint32_t v = 0;
	if (i < s.nc) {
		const uint32_t j = plocPartner(nn, s.nc, i, s.forced != 0);
		v = (j != kNone && i < j ? 0x10000u : 0u) + (j != kNone && i > j ? 0u : 1u);
	}
	uint32_t sum;
	const uint32_t p = blockPrefix(v, lds, sum);
	if (i < s.nc) prefix[i] = p;
	if (threadIdx.x == 0) {
		leadSums[blockIdx.x] = sum >> 16;
		keepSums[blockIdx.x] = sum & 0xffffu;
	}
}

// block sums to block starts, and the next round's state
__global__ __launch_bounds__(1024) void k_plocScan(uint32_t *leadSums, uint32_t *keepSums, PlocState *st, uint32_t r,
		uint32_t ni, PlocState *host, uint32_t *err) {
	__shared__ uint32_t lds[16];
	const PlocState s = plocRound(st, r);
	if (s.nc == 0) {
		if (threadIdx.x == 0) st[r + 1] = *host = st[r];
		return;
	}
	const uint32_t nb = (s.nc + 255u) / 256u;
	const uint32_t merged = scanByBlock(leadSums, nb, lds);
	const uint32_t kept = scanByBlock(keepSums, nb, lds);
	if (threadIdx.x == 0) {
		PlocState t = {kept, s.nodeBase + merged, !s.forced && (uint64_t)merged * 64u < s.nc ? 1u : 0u, 0u};
		if (merged == 0 || merged > s.nc / 2 || kept != s.nc - merged || t.nodeBase > ni) {
			atomicOr(err, kErrCluster);
			t = {0u, s.nodeBase, 0u, 0u};
		}
		st[r + 1] = *host = t;
	}
}

// the arrays of the clustering's binary tree (nodes in the order they are made)
struct PlocTree {
	uint32_t *left, *right, *count;
	GBox *box;
	float *cost, *key;
	const GBox *leafBox;
	uint32_t maxLeaf;
	float ci;
};

// node x of children l and r (older nodes or leaves): box, leaves, cost and
// leaf decision
__device__ __forceinline__ void plocMake(const PlocTree &T, uint32_t x, uint32_t l, uint32_t r, const GBox &u) {
	const uint32_t c = plocSize(l, T.count) + plocSize(r, T.count);
	const float cl = (l & kLeafBit) ? areaOf(T.leafBox[l & ~kLeafBit]) : T.cost[l];
	const float cr = (r & kLeafBit) ? areaOf(T.leafBox[r & ~kLeafBit]) : T.cost[r];
	uint32_t lf;
	T.left[x] = l;
	T.right[x] = r;
	T.box[x] = u;
	T.count[x] = c;
	T.cost[x] = nodeCost(areaOf(u), cl, cr, c, T.maxLeaf, T.ci, lf);
	T.key[x] = nodeKey(lf, areaOf(u));
}

__global__ __launch_bounds__(256) void k_plocApply(const uint32_t *nn, const PlocState *st, uint32_t r,
		const uint32_t *cid, const GBox *cbox, const uint32_t *prefix, const uint32_t *leadSums,
		const uint32_t *keepSums, uint32_t ni, uint32_t *outCid, GBox *outBox, PlocTree T) {
	const PlocState s = plocRound(st, r);
	const uint32_t i = blockIdx.x * 256u + threadIdx.x;
	if (i >= s.nc || st[r + 1].nc == 0) return;
	const uint32_t j = plocPartner(nn, s.nc, i, s.forced != 0);
	if (j != kNone && i > j) return;  // merged into its lower partner
	const uint32_t o = keepSums[blockIdx.x] + (prefix[i] & 0xffffu);
	if (j != kNone) {
		const uint32_t node = s.nodeBase + leadSums[blockIdx.x] + (prefix[i] >> 16);
		const GBox u = unionBox(cbox[i], cbox[j]);
		if (node < ni) plocMake(T, node, cid[i], cid[j], u);
		outCid[o] = node;
		outBox[o] = u;
	} else {
		outCid[o] = cid[i];
		outBox[o] = cbox[i];
	}
}

// The last kPlocTail clusters by one block, all their rounds in LDS with
// barriers: 46 rounds of a 50,000-triangle mesh were 46 times six launches
// and a wait for the host, most of them for a few hundred clusters.  Each
// thread has two clusters; a round is the one of the kernels above, its
// neighbour search with more lanes a cluster as clusters get fewer (the tail of
// 50,000 triangles: 283 us, now 196).
template <uint32_t L>
__device__ __forceinline__ void plocTailNearest(const GBox *box, uint32_t nc, uint32_t *nn) {
	for (uint32_t b = 0; b < nc; b += 1024 / L) {
		const uint32_t i = b + threadIdx.x / L;
		const uint32_t x = plocNearestLanes<L>([&](uint32_t j) -> const GBox & { return box[j]; }, nc, i, threadIdx.x % L);
		if (i < nc && threadIdx.x % L == 0) nn[i] = x;
	}
}
__global__ __launch_bounds__(1024) void k_plocTail(PlocState *st, uint32_t r0, uint32_t ni, const uint32_t *cidIn,
		const GBox *cboxIn, PlocTree T, uint32_t *rounds, uint32_t *err) {
	__shared__ GBox box[kPlocTail];
	__shared__ uint32_t cid[kPlocTail], nn[kPlocTail];
	__shared__ uint32_t wsum[16];
	PlocState s = st[r0];
	uint32_t r = r0;
	if (s.nc > kPlocTail) {
		if (threadIdx.x == 0) atomicOr(err, kErrCluster);
		return;
	}
	for (uint32_t i = threadIdx.x; i < s.nc; i += 1024) {
		box[i] = cboxIn[i];
		cid[i] = cidIn[i];
	}
	__syncthreads();
	const uint32_t i0 = 2u * threadIdx.x;
	while (s.nc > 1 && r < kPlocMaxRounds) {
		if (!s.forced) {
			if (s.nc <= 256) plocTailNearest<16>(box, s.nc, nn);
			else if (s.nc <= 1024) plocTailNearest<4>(box, s.nc, nn);
			else plocTailNearest<1>(box, s.nc, nn);
		}
		__syncthreads();
		// this thread's two places: their partners and flags, scanned over the block
		uint32_t part[2], v[2], sum = 0;
		for (uint32_t k = 0; k < 2; ++k) {
			const uint32_t i = i0 + k;
			part[k] = i < s.nc ? plocPartner(nn, s.nc, i, s.forced != 0) : kNone;
			v[k] = i >= s.nc ? 0u : (part[k] != kNone && i < part[k] ? 0x10000u : 0u) + (part[k] != kNone && i > part[k] ? 0u : 1u);
			sum += v[k];
		}
		uint32_t incl = sum;
		for (int o = 1; o < 64; o <<= 1) {
			const uint32_t x = (uint32_t)__shfl_up((int)incl, o);
			if ((int)(threadIdx.x & 63u) >= o) incl += x;
		}
		if ((threadIdx.x & 63u) == 63u) wsum[threadIdx.x >> 6] = incl;
		__syncthreads();
		uint32_t at = incl - sum, all = 0;
		for (uint32_t w = 0; w < 16; ++w) {
			if (w < (threadIdx.x >> 6)) at += wsum[w];
			all += wsum[w];
		}
		const uint32_t merged = all >> 16, kept = all & 0xffffu;
		const bool bad = merged == 0 || kept != s.nc - merged || s.nodeBase + merged > ni;
		GBox nb[2];
		uint32_t nid[2], to[2] = {kNone, kNone};
		for (uint32_t k = 0; k < 2 && !bad; ++k) {
			const uint32_t i = i0 + k, j = part[k];
			if (i >= s.nc || (j != kNone && i > j)) {
				at += v[k];
				continue;
			}
			to[k] = at & 0xffffu;
			if (j != kNone) {
				nid[k] = s.nodeBase + (at >> 16);
				nb[k] = unionBox(box[i], box[j]);
				plocMake(T, nid[k], cid[i], cid[j], nb[k]);
			} else {
				nid[k] = cid[i];
				nb[k] = box[i];
			}
			at += v[k];
		}
		__syncthreads();
		if (bad) {
			if (threadIdx.x == 0) atomicOr(err, kErrCluster);
			break;
		}
		for (uint32_t k = 0; k < 2; ++k)
			if (to[k] != kNone) {
				box[to[k]] = nb[k];
				cid[to[k]] = nid[k];
			}
		s.forced = !s.forced && merged * 64u < s.nc ? 1u : 0u;
		s.nodeBase += merged;
		s.nc = kept;
		++r;
		if (threadIdx.x == 0) st[r] = s;
		__syncthreads();
	}
	if (threadIdx.x == 0) {
		*rounds = r;
		if (s.nc != 1 || s.nodeBase != ni) atomicOr(err, kErrCluster);
	}
}

// first leaf place of each subtree, top down; leafFirst: the place of each
// sorted leaf
__device__ __forceinline__ void plocFirst(uint32_t x, const uint32_t *left, const uint32_t *right, const uint32_t *count,
		uint32_t *first, uint32_t *leafFirst) {
	const uint32_t f = first[x], l = left[x], r = right[x];
	const uint32_t fr = f + plocSize(l, count);
	if (l & kLeafBit) leafFirst[l & ~kLeafBit] = f; else first[l] = f;
	if (r & kLeafBit) leafFirst[r & ~kLeafBit] = fr; else first[r] = fr;
}

// the nodes of one round (their parents are younger)
__global__ void k_plocFirst(uint32_t b, uint32_t e, const uint32_t *left, const uint32_t *right, const uint32_t *count,
		uint32_t *first, uint32_t *leafFirst) {
	const uint32_t x = b + blockIdx.x * blockDim.x + threadIdx.x;
	if (x < e) plocFirst(x, left, right, count, first, leafFirst);
}

// rounds r1-1 down to r0 by one block (the tail's, below the root)
__global__ __launch_bounds__(1024) void k_plocFirstTail(const PlocState *st, uint32_t r0, uint32_t r1, uint32_t ni,
		const uint32_t *left, const uint32_t *right, const uint32_t *count, uint32_t *first, uint32_t *leafFirst) {
	if (threadIdx.x == 0) first[ni - 1] = 0u;  // the root
	__syncthreads();
	for (uint32_t r = r1; r-- > r0;) {
		for (uint32_t x = st[r].nodeBase + threadIdx.x; x < st[r + 1].nodeBase; x += 1024)
			plocFirst(x, left, right, count, first, leafFirst);
		__syncthreads();
	}
}

// the clustering's tree in the radix tree's form: internal node x becomes
// n-2-x (root 0), leaves their places; leaf values and boxes in place order
__global__ void k_plocFinish(uint32_t n, const uint32_t *left, const uint32_t *right, const uint32_t *count,
		const uint32_t *first, const GBox *nodeBox, const float *key, const uint32_t *leafFirst,
		const uint32_t *vals, const GBox *leafBoxIn, uint32_t *left2, uint32_t *right2, uint32_t *first2,
		uint32_t *last2, GBox *nodeBox2, float *key2, uint32_t *vals2, GBox *leafBox2) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n) return;
	const uint32_t p = leafFirst[i];
	vals2[p] = vals[i];
	leafBox2[p] = leafBoxIn[i];
	if (i + 1 >= n) return;  // n - 1 internal nodes
	const uint32_t y = n - 2 - i;
	auto remap = [&](uint32_t c) { return (c & kLeafBit) ? (kLeafBit | leafFirst[c & ~kLeafBit]) : n - 2 - c; };
	left2[y] = remap(left[i]);
	right2[y] = remap(right[i]);
	first2[y] = first[i];
	last2[y] = first[i] + count[i] - 1;
	nodeBox2[y] = nodeBox[i];
	key2[y] = key[i];
}

// 5. the breadth-first collapse, level by level.  A level's count and first
// node are written on the device by the level before, so several levels are
// launched on upper bounds between two looks of the host.
struct Level {
	uint32_t nf, base;
};

// 5a. children of each frontier node (its two, then the largest that is not a
// leaf opened until there are W; from the nodes' keys, so the areas of the
// candidates stay in registers and each opened child costs one read of its
// children and one of their keys), and how many become inner nodes, summed
// over the block
template <int W>
__global__ __launch_bounds__(256) void k_expand(const uint32_t *frontier, const Level *lv, uint32_t l, uint32_t nInner,
		const uint32_t *left, const uint32_t *right, const float *key, uint32_t *kids, uint32_t *prefix, uint32_t *sums,
		uint32_t *err) {
	const uint32_t nf = lv[l].nf;
	if (blockIdx.x * 256u >= nf) return;
	__shared__ uint32_t lds[4];
	const uint32_t e = blockIdx.x * 256u + threadIdx.x;
	uint32_t inner = 0;
	if (e < nf) {
		const uint32_t b = frontier[e];
		uint32_t ch[W];
		float a[W];
#pragma unroll
		for (int k = 0; k < W; ++k) {
			ch[k] = kNone;
			a[k] = -1.f;
		}
		auto keyOf = [key](uint32_t c) { return (c & kLeafBit) ? -1.f : key[c]; };
		if (b < nInner) {
			ch[0] = left[b];
			ch[1] = right[b];
			a[0] = keyOf(ch[0]);
			a[1] = keyOf(ch[1]);
			for (int nch = 2; nch < W; ++nch) {
				int pick = -1;
				float best = -1.f;
				uint32_t c = 0;
#pragma unroll
				for (int k = 0; k < W; ++k)
					if (a[k] > best) {
						best = a[k];
						pick = k;
						c = ch[k];
					}
				if (pick < 0) break;
				const uint32_t cl = left[c], cr = right[c];
				const float al = keyOf(cl), ar = keyOf(cr);
#pragma unroll
				for (int k = W - 1; k > 0; --k)
					if (k > pick + 1) {
						ch[k] = ch[k - 1];
						a[k] = a[k - 1];
					}
#pragma unroll
				for (int k = 0; k < W; ++k) {
					if (k == pick) {
						ch[k] = cl;
						a[k] = al;
					}
					if (k == pick + 1) {
						ch[k] = cr;
						a[k] = ar;
					}
				}
			}
		} else
			atomicOr(err, kErrExpand);  // not an internal node
#pragma unroll
		for (int k = 0; k < W; ++k) {
			// a child that stays a node has its area as key, zero or more (or a NaN's)
			const bool leaf = ch[k] == kNone || (ch[k] & kLeafBit) || a[k] == -1.f;
			kids[(size_t)W * e + k] = ch[k];
			inner += leaf ? 0u : 1u;
		}
	}
	uint32_t sum;
	const uint32_t p = blockPrefix(inner, lds, sum);
	if (e < nf) prefix[e] = p;
	if (threadIdx.x == 0) sums[blockIdx.x] = sum;
}

// 5b. block sums to block starts, and the next level (none, with the error
// set, if its nodes would not fit)
__global__ __launch_bounds__(1024) void k_levelScan(uint32_t *sums, Level *lv, uint32_t l, uint32_t capNodes,
		uint32_t *host, uint32_t *err) {
	__shared__ uint32_t lds[16];
	const Level v = lv[l];
	const uint32_t total = scanByBlock(sums, (v.nf + 255u) / 256u, lds);
	if (threadIdx.x == 0) {
		Level n = {total, v.base + v.nf};
		if ((uint64_t)n.base + n.nf > capNodes) {
			atomicOr(err, kErrExpand);
			n.nf = 0;
		}
		lv[l + 1] = n;
		host[0] = n.nf;
		host[1] = n.base;
		if (v.nf) host[2] = l + 1;  // levels with nodes
	}
}

// 5c. the level's wide nodes, W lanes each; inner children get slots after
// the level
template <int W, class Node>
__global__ __launch_bounds__(256) void k_emit(const Level *lv, uint32_t l, const uint32_t *kids, const uint32_t *prefix,
		const uint32_t *sums, const uint32_t *first, const uint32_t *last, const float *key, const GBox *leafBox,
		const GBox *nodeBox, Node *nodes, uint32_t *next) {
	const Level v = lv[l];
	const uint32_t t = blockIdx.x * 256u + threadIdx.x;
	const uint32_t e = t / W;
	const int c = (int)(t % W);
	if (e >= v.nf || lv[l + 1].base != v.base + v.nf) return;
	const uint32_t kid = kids[(size_t)W * e + c];
	const bool some = kid != kNone;
	const bool tri = some && (kid & kLeafBit);
	const bool leaf = tri || (some && key[kid] == -1.f);
	const uint32_t lane = threadIdx.x & 63u, shift = lane & ~(uint32_t)(W - 1);
	const uint32_t innerMask = (uint32_t)(__ballot(some && !leaf) >> shift) & ((1u << W) - 1u);
	const int n = __popc((uint32_t)(__ballot(some) >> shift) & ((1u << W) - 1u));
	GBox b;
	for (int k = 0; k < 3; ++k) { b.lo[k] = INFINITY; b.hi[k] = -INFINITY; }
	uint32_t ref = LRH_CHILD_EMPTY;
	if (some) b = tri ? leafBox[kid & ~kLeafBit] : nodeBox[kid];
	if (leaf)
		ref = tri ? leafRef(kid & ~kLeafBit, 1u) : leafRef(first[kid], last[kid] - first[kid] + 1u);
	else if (some && lv[l + 1].nf) {
		const uint32_t slot = sums[e / 256u] + prefix[e] + (uint32_t)__popc(innerMask & ((1u << c) - 1u));
		ref = v.base + v.nf + slot;
		next[slot] = kid;
	}
	Node *out = nodes + v.base + e;
	if constexpr (std::is_same<Node, lrh_node4f>::value)
		lrhdev::floatNodeLanes(b, c, n, ref, out);
	else
		lrhdev::quantizeNodeLanes<W>(b, c, n, ref, out);
}

__global__ void k_rootLevel(uint32_t *frontier, Level *lv, uint32_t *host) {
	if (threadIdx.x != 0 || blockIdx.x != 0) return;
	frontier[0] = 0u;
	lv[0] = {1u, 0u};
	host[0] = 1u;
	host[1] = host[2] = 0u;
}

// a scene of at most maxLeaf triangles: one node with one leaf
__global__ void k_smallRoot(const GBox *leafBox, uint32_t n, uint32_t layout, void *nodes) {
	if (threadIdx.x != 0 || blockIdx.x != 0) return;
	GBox b;
	for (int k = 0; k < 3; ++k) {
		b.lo[k] = INFINITY;
		b.hi[k] = -INFINITY;
	}
	for (uint32_t i = 0; i < n; ++i)
		for (int k = 0; k < 3; ++k) {
			b.lo[k] = minT(b.lo[k], leafBox[i].lo[k]);
			b.hi[k] = maxT(b.hi[k], leafBox[i].hi[k]);
		}
	uint32_t ref[kMaxWide];
	for (int k = 0; k < kMaxWide; ++k) ref[k] = k ? LRH_CHILD_EMPTY : leafRef(0, n);
	if (layout == 0)
		lrhdev::quantizeNode(&b, 1, ref, reinterpret_cast<lrh_node4q *>(nodes));
	else if (layout == 2)
		lrhdev::quantizeNode8(&b, 1, ref, reinterpret_cast<lrh_node8q *>(nodes));
	else
		lrhdev::floatNode(&b, 1, ref, reinterpret_cast<lrh_node4f *>(nodes));
}

__global__ void k_identity(const GBox *boxes, uint32_t n, uint32_t *vals, GBox *leafBox) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n) return;
	vals[i] = i;
	leafBox[i] = boxes[i];
}

// 6. triangle records in leaf order
__global__ void k_records(const float *verts, const uint32_t *tris, const uint32_t *tbase, const uint32_t *vbase,
		uint32_t nMeshes, const uint32_t *vals, uint32_t n, lrh_tri *recs, uint32_t *invPerm) {
	const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
	if (j >= n) return;
	const uint32_t i = vals[j];
	recs[j] = triRecord(verts, tris, tbase, vbase, nMeshes, i);
	invPerm[i] = j;
}

// the build's scratch arrays, carved from chunks of at least 256 MiB (an
// array above that is a chunk of its own) and released together at the end:
// the clustering's rounds ask for hundreds of small scan arrays, and a
// device allocation and release each would cost more than the kernels
struct Scratch {
	static constexpr size_t kChunk = size_t(256) << 20;
	const LrhGpuAlloc &a;
	std::vector<std::pair<void *, size_t>> held;
	char *cur = nullptr;
	size_t left = 0;
	// LRH_BUILD_PINNED bytes of pinned host memory that kernels write and the
	// host reads after a wait (word 0: error, 1: rounds, 4-6: the collapse's
	// level, 128+: digit starts)
	uint32_t *pin = nullptr;
	explicit Scratch(const LrhGpuAlloc &al) : a(al), pin(static_cast<uint32_t *>(al.pinned(al.ctx))) {}
	template <class T>
	T *get(size_t count) {
		const size_t bytes = (std::max<size_t>(count * sizeof(T), 16) + 255) & ~size_t(255);
		if (bytes > left) {
			const size_t chunk = std::max(bytes, kChunk);
			void *p = a.alloc(a.ctx, chunk);
			held.push_back({p, chunk});
			if (bytes == chunk) return static_cast<T *>(p);  // a chunk of its own; the current one stays
			cur = static_cast<char *>(p);
			left = chunk;
		}
		T *r = reinterpret_cast<T *>(cur);
		cur += bytes;
		left -= bytes;
		return r;
	}
	~Scratch() {
		for (auto &h : held) a.release(a.ctx, h.first, h.second);
		a.unpin(a.ctx, pin);
	}
};

inline unsigned grid(size_t n, unsigned b) { return (unsigned)((n + b - 1) / b); }

// one stable pass of the radix sort over the eight bits from `shift`
void sortPass(const uint64_t *kIn, const uint32_t *vIn, uint32_t n, uint32_t shift, uint32_t *table, uint32_t *totals,
		uint64_t *kOut, uint32_t *vOut, uint32_t *err, hipStream_t st) {
	const uint32_t tiles = sortTiles(n);
	const bool small = n <= kSortSmall;
	hipLaunchKernelGGL(small ? k_sortCount<kSortTileSmall> : k_sortCount<kSortTile>, dim3(tiles), dim3(kSortBlock), 0, st,
			kIn, n, shift, tiles, table);
	hipLaunchKernelGGL(k_scanRows, dim3(256), dim3(256), 0, st, table, tiles, totals);
	hipLaunchKernelGGL(small ? k_sortScatter<kSortTileSmall> : k_sortScatter<kSortTile>, dim3(tiles), dim3(kSortBlock), 0,
			st, kIn, vIn, n, shift, tiles, table, totals, kOut, vOut, err);
	GB_CHECK(hipGetLastError());
}

// waits for the stream (and the readbacks queued before) and returns the
// error word
uint32_t readError(Scratch &S, const uint32_t *err, hipStream_t st) {
	GB_CHECK(hipMemcpyAsync(S.pin, err, 4, hipMemcpyDeviceToHost, st));
	GB_CHECK(hipStreamSynchronize(st));
	return S.pin[0];
}

std::string errorText(uint32_t e) {
	std::string s = "device build: ";
	if (e & kErrUnsorted) s += "sorted Morton codes out of order; ";
	if (e & kErrRange) s += "radix tree node without a key range (codes not in order); ";
	if (e & kErrExpand) s += "collapse reached a non-internal node, or more nodes than the tree can have; ";
	if (e & kErrIndex) s += "vertex index out of range; ";
	if (e & kErrCluster) s += "clustering round without a consistent merge count; ";
	return s;
}

// Boxes, costs and leaf decisions of the radix tree's nodes bottom-up with a
// kernel boundary between levels instead of a fenced walk per leaf (a walk
// publishes each box to the other XCDs' caches by an agent-scope fence,
// which writes back and invalidates L2 on every step).  A node's common
// prefix is shorter than its children's, so nodes go by the length of their
// prefix, which the radix tree knows, one launch per length from the longest
// (depths would be fewer levels, but took seven rounds of pointer jumping);
// runs of lengths with few nodes go to one block.  (The build of 2.29M
// triangles, 8-wide, went from 2,450 to 1,575 us by this, the scan of a sort
// pass in one launch, and a collapse that does not stop for the host after
// each level.)
void boxesByPrefix(Scratch &S, const GBox *boxes, const uint32_t *vals, uint32_t n, const uint32_t *left,
		const uint32_t *right, const uint32_t *first, const uint32_t *last, const uint64_t *digits, const uint32_t *ids,
		uint32_t maxLeaf, float ci, hipStream_t st, uint32_t *err, GBox *leafBox, GBox *nodeBox, float *key) {
	const uint32_t ni = n - 1, tiles = sortTiles(ni);
	uint32_t *order = S.get<uint32_t>(ni), *starts = S.get<uint32_t>(256), *totals = S.get<uint32_t>(256);
	uint64_t *digitsOut = S.get<uint64_t>(ni);
	uint32_t *table = S.get<uint32_t>((size_t)256 * tiles);
	float *cost = S.get<float>(ni);
	sortPass(digits, ids, ni, 0u, table, totals, digitsOut, order, err, st);
	hipLaunchKernelGGL(k_digitStarts, dim3(1), dim3(256), 0, st, totals, starts, S.pin + 128);
	hipLaunchKernelGGL(k_leafBoxes, dim3(grid(n, 256)), dim3(256), 0, st, boxes, vals, n, leafBox);
	GB_CHECK(hipGetLastError());
	if (const uint32_t e = readError(S, err, st)) throw std::runtime_error(errorText(e));
	uint32_t off[kDigits + 1];
	std::copy(S.pin + 128, S.pin + 128 + kDigits + 1, off);
	for (uint32_t d = 0; d < kDigits; ++d)
		if (off[d + 1] < off[d]) throw std::runtime_error("device build: prefix table out of order");
	if (off[0] != 0 || off[kDigits] != ni) throw std::runtime_error("device build: radix tree nodes not all in the table");
	for (uint32_t d = 0; d < kDigits;) {
		const uint32_t cnt = off[d + 1] - off[d];
		if (cnt > kSmallLevel) {
			hipLaunchKernelGGL(k_boxLevel, dim3(grid(cnt, 256)), dim3(256), 0, st, order + off[d], cnt, left, right, first,
					last, leafBox, maxLeaf, ci, nodeBox, cost, key);
			++d;
			continue;
		}
		uint32_t d1 = d + 1;
		while (d1 < kDigits && off[d1 + 1] - off[d1] <= kSmallLevel) ++d1;
		if (off[d1] > off[d])
			hipLaunchKernelGGL(k_boxSmallLevels, dim3(1), dim3(1024), 0, st, order, starts, d, d1, left, right, first, last,
					leafBox, maxLeaf, ci, nodeBox, cost, key);
		d = d1;
	}
	GB_CHECK(hipGetLastError());
}

// The clustering's binary tree over the n >= 2 sorted leaves, written in the
// radix tree's form (left / right / first / last / nodeBox, root 0, leaf
// places contiguous per subtree); vals and leafBox are repointed to the
// leaves in place order.  Each round: nearest neighbours, the merge and keep
// flags scanned, then the pairs merged and the clusters compacted.  A round
// that merges fewer than 1/64 of the clusters is followed by a forced round
// that pairs places 2k, 2k+1, so the number of rounds is bounded by the size
// alone.  (Natural rounds merge a third of the clusters at first and a tenth
// or less near the top, where boxes overlap; forcing there would cost tree
// quality.)  Rounds find their sizes on the device; the host looks at them
// every kPlocBatch rounds, to shrink the grids and to stop.  What bounds a
// build of some ten thousand triangles is launches and waits: 50,000 triangles
// went from 2,690 us (six launches and a wait a round) to 1,205.
void plocTree(Scratch &S, const GBox *boxes, uint32_t n, uint32_t maxLeaf, float ci, hipStream_t st, uint32_t *err,
		uint32_t *&vals, GBox *&leafBox, uint32_t *left, uint32_t *right, uint32_t *first, uint32_t *last, GBox *nodeBox,
		float *key, uint32_t *roundsOut) {
	constexpr uint32_t kPlocBatch = 6;
	const uint32_t ni = n - 1;
	uint32_t *cidA = S.get<uint32_t>(n), *cidB = S.get<uint32_t>(n), *nn = S.get<uint32_t>(n), *prefix = S.get<uint32_t>(n);
	GBox *cboxA = S.get<GBox>(n), *cboxB = S.get<GBox>(n);
	uint32_t *leadSums = S.get<uint32_t>(grid(n, 256)), *keepSums = S.get<uint32_t>(grid(n, 256));
	PlocState *state = S.get<PlocState>(kPlocMaxRounds + 1);
	PlocTree T = {S.get<uint32_t>(ni), S.get<uint32_t>(ni), S.get<uint32_t>(ni), S.get<GBox>(ni), S.get<float>(ni),
			S.get<float>(ni), leafBox, maxLeaf, ci};
	hipLaunchKernelGGL(k_plocInit, dim3(grid(n, 256)), dim3(256), 0, st, boxes, vals, n, cidA, cboxA, leafBox, state);
	GB_CHECK(hipGetLastError());
	std::vector<PlocState> host(kPlocMaxRounds + 1);
	host[0] = {n, 0u, 0u, 0u};
	PlocState *seen = reinterpret_cast<PlocState *>(S.pin + 8);
	uint32_t r = 0, ub = n;
	while (ub > kPlocTail) {
		for (uint32_t k = 0; k < kPlocBatch; ++k, ++r) {
			if (r >= kPlocMaxRounds) throw std::runtime_error("device build: clustering did not converge");
			if (ub <= kPlocSplit)
				hipLaunchKernelGGL(k_plocNearest<4>, dim3(grid(ub, 64)), dim3(256), 0, st, cboxA, state, r, nn);
			else
				hipLaunchKernelGGL(k_plocNearest<1>, dim3(grid(ub, 256)), dim3(256), 0, st, cboxA, state, r, nn);
			hipLaunchKernelGGL(k_plocMark, dim3(grid(ub, 256)), dim3(256), 0, st, nn, state, r, prefix, leadSums, keepSums);
			hipLaunchKernelGGL(k_plocScan, dim3(1), dim3(1024), 0, st, leadSums, keepSums, state, r, ni, seen + k, err);
			hipLaunchKernelGGL(k_plocApply, dim3(grid(ub, 256)), dim3(256), 0, st, nn, state, r, cidA, cboxA, prefix,
					leadSums, keepSums, ni, cidB, cboxB, T);
			GB_CHECK(hipGetLastError());
			std::swap(cidA, cidB);
			std::swap(cboxA, cboxB);
		}
		if (const uint32_t e = readError(S, err, st)) throw std::runtime_error(errorText(e));
		std::copy_n(seen, kPlocBatch, host.begin() + (r - kPlocBatch + 1));
		ub = host[r].nc;
	}
	// the rounds after the count fell to the tail's changed nothing but the
	// buffers' roles: the clusters are where the last real round put them
	uint32_t r0 = r;
	while (r0 > 0 && host[r0 - 1].nc <= kPlocTail && host[r0 - 1].nc == host[r0].nc) --r0;
	if ((r - r0) & 1u) {
		std::swap(cidA, cidB);
		std::swap(cboxA, cboxB);
	}
	hipLaunchKernelGGL(k_plocTail, dim3(1), dim3(1024), 0, st, state, r0, ni, cidA, cboxA, T, S.pin + 1, err);
	if (const uint32_t e = readError(S, err, st)) throw std::runtime_error(errorText(e));
	const uint32_t r1 = S.pin[1];
	*roundsOut = r1;
	// first places, newest round first
	uint32_t *firstP = S.get<uint32_t>(ni), *leafFirst = S.get<uint32_t>(n);
	hipLaunchKernelGGL(k_plocFirstTail, dim3(1), dim3(1024), 0, st, state, r0, r1, ni, T.left, T.right, T.count, firstP,
			leafFirst);
	for (uint32_t k = r0; k-- > 0;) {
		const uint32_t b = host[k].nodeBase, e = host[k + 1].nodeBase;
		if (e > b)
			hipLaunchKernelGGL(k_plocFirst, dim3(grid(e - b, 256)), dim3(256), 0, st, b, e, T.left, T.right, T.count, firstP,
					leafFirst);
	}
	uint32_t *vals2 = S.get<uint32_t>(n);
	GBox *leafBox2 = S.get<GBox>(n);
	hipLaunchKernelGGL(k_plocFinish, dim3(grid(n, 256)), dim3(256), 0, st, n, T.left, T.right, T.count, firstP, T.box,
			T.key, leafFirst, vals, leafBox, left, right, first, last, nodeBox, key, vals2, leafBox2);
	GB_CHECK(hipGetLastError());
	vals = vals2;
	leafBox = leafBox2;
}

}  // namespace

void lrhGpuBuildBVH(const LrhGpuBuildIn &in, const LrhGpuAlloc &a, hipStream_t st, LrhGpuBuildOut *out) {
	const uint32_t n = in.nTris;
	if (n == 0) throw std::runtime_error("device build: empty scene");
	if (n > 0x7fffffffu) throw std::runtime_error("device build: at most 2^31-1 triangles");
	if (in.maxLeaf < 1 || in.maxLeaf > LRH_LEAF_MAX) throw std::runtime_error("device build: maxLeaf must be 1..8");
	if (!(in.travCost >= 0.f) || !std::isfinite(in.travCost))
		throw std::runtime_error("device build: travCost must be finite and >= 0");
	if (in.layout > 2) throw std::runtime_error("device build: layout must be 0, 1 or 2");
	const size_t nodeSz = in.layout == 0 ? sizeof(lrh_node4q) : in.layout == 2 ? sizeof(lrh_node8q) : sizeof(lrh_node4f);
	const int width = in.layout == 2 ? 8 : 4;
	Scratch S(a);
	hipEvent_t e0, e1;
	GB_CHECK(hipEventCreate(&e0));
	GB_CHECK(hipEventCreate(&e1));
	GB_CHECK(hipEventRecord(e0, st));

	uint32_t *err = S.get<uint32_t>(1);
	hipLaunchKernelGGL(k_fill, dim3(1), dim3(64), 0, st, err, 1u, 0u);
	uint32_t *tbase = S.get<uint32_t>(in.nMeshes + 1), *vbase = S.get<uint32_t>(in.nMeshes + 1);
	GB_CHECK(hipMemcpyAsync(tbase, in.meshTriBase, (in.nMeshes + 1) * 4, hipMemcpyHostToDevice, st));
	GB_CHECK(hipMemcpyAsync(vbase, in.meshVertBase, (in.nMeshes + 1) * 4, hipMemcpyHostToDevice, st));
	GBox *boxes = S.get<GBox>(n);
	uint32_t *cb = S.get<uint32_t>(6);
	const uint32_t primBlocks = std::min<uint32_t>(grid(n, 256), kPrimBlocks);
	uint32_t *partial = S.get<uint32_t>(6 * primBlocks);
	hipLaunchKernelGGL(k_prims, dim3(primBlocks), dim3(256), 0, st, in.verts, in.tris, tbase, vbase, in.nMeshes, n,
			boxes, partial, err);
	hipLaunchKernelGGL(k_bounds, dim3(1), dim3(384), 0, st, partial, primBlocks, cb);
	GB_CHECK(hipGetLastError());

	uint32_t *vals = S.get<uint32_t>(n);
	GBox *leafBox = S.get<GBox>(n);
	// output buffers (owned by the caller from here on)
	const size_t capNodes = std::max<uint32_t>(n > 1 ? n - 1 : 1, 1);
	void *nodes = a.alloc(a.ctx, capNodes * nodeSz);
	uint32_t nodeCount = 0, depth = 0;
	auto allocRecords = [&]() {
		if (out->tris) return;
		out->triBytes = (size_t)n * sizeof(lrh_tri);
		out->tris = a.alloc(a.ctx, out->triBytes);
		out->invPermBytes = (size_t)n * 4;
		out->invPerm = static_cast<uint32_t *>(a.alloc(a.ctx, out->invPermBytes));
	};
	try {
		if (n <= in.maxLeaf) {
			hipLaunchKernelGGL(k_identity, dim3(grid(n, 256)), dim3(256), 0, st, boxes, n, vals, leafBox);
			hipLaunchKernelGGL(k_smallRoot, dim3(1), dim3(64), 0, st, leafBox, n, in.layout, nodes);
			GB_CHECK(hipGetLastError());
			if (const uint32_t e = readError(S, err, st)) throw std::runtime_error(errorText(e));
			nodeCount = 1;
		} else {
			uint64_t *keys = S.get<uint64_t>(n), *keysB = S.get<uint64_t>(n);
			uint32_t *valsB = S.get<uint32_t>(n);
			hipLaunchKernelGGL(k_morton, dim3(grid(n, 256)), dim3(256), 0, st, boxes, n, cb, keys, vals);
			GB_CHECK(hipGetLastError());
			// stable LSD radix sort, 8 passes of 8 bits; an even number of
			// passes leaves the result in keys / vals
			uint32_t *table = S.get<uint32_t>((size_t)256 * sortTiles(n)), *totals = S.get<uint32_t>(256);
			uint64_t *kIn = keys, *kOut = keysB;
			uint32_t *vIn = vals, *vOut = valsB;
			for (uint32_t shift = 0; shift < 64; shift += 8) {
				sortPass(kIn, vIn, n, shift, table, totals, kOut, vOut, err, st);
				std::swap(kIn, kOut);
				std::swap(vIn, vOut);
			}
			hipLaunchKernelGGL(k_checkSorted, dim3(grid(n, 256)), dim3(256), 0, st, keys, n, err);
			GB_CHECK(hipGetLastError());
			allocRecords();  // (while the sort runs)

			const uint32_t ni = n - 1;
			uint32_t *left = S.get<uint32_t>(ni), *right = S.get<uint32_t>(ni), *first = S.get<uint32_t>(ni),
					 *last = S.get<uint32_t>(ni);
			GBox *nodeBox = S.get<GBox>(ni);
			float *key = S.get<float>(ni);
			if (in.method == 1) {
				plocTree(S, boxes, n, in.maxLeaf, in.travCost, st, err, vals, leafBox, left, right, first, last, nodeBox, key,
						&out->plocRounds);
			} else {
				// the sorted keys' other buffers hold the digits and ids
				hipLaunchKernelGGL(k_radixTree, dim3(grid(ni, 256)), dim3(256), 0, st, keys, n, left, right, first, last, keysB,
						valsB, err);
				GB_CHECK(hipGetLastError());
				boxesByPrefix(S, boxes, vals, n, left, right, first, last, keysB, valsB, in.maxLeaf, in.travCost, st, err,
						leafBox, nodeBox, key);
			}

			// breadth-first collapse: level frontiers of binary node ids; a level
			// has at most `width` times the nodes of the one before, which the host
			// knows after each batch of levels
			constexpr uint32_t kMaxLevels = 160;
			uint32_t *fA = S.get<uint32_t>(ni), *fB = S.get<uint32_t>(ni);
			uint32_t *kids = S.get<uint32_t>((size_t)width * ni), *prefix = S.get<uint32_t>(ni),
					 *sums = S.get<uint32_t>(grid(ni, 256));
			Level *lv = S.get<Level>(kMaxLevels + 1);
			hipLaunchKernelGGL(k_rootLevel, dim3(1), dim3(64), 0, st, fA, lv, S.pin + 4);
			uint32_t nf = 1, l = 0;
			while (nf) {
				// down to a level that may hold 4,096 nodes at first, then two at a time
				const uint32_t batch = l == 0 ? (width == 8 ? 5u : 7u) : 2u;
				uint64_t ub = nf;
				for (uint32_t k = 0; k < batch; ++k, ++l, ub = std::min<uint64_t>(ub * width, ni)) {
					if (l >= kMaxLevels) throw std::runtime_error("device build: collapse deeper than any valid tree");
					const dim3 ge(grid(ub, 256)), gm(grid(ub * width, 256)), b(256);
					if (width == 8)
						hipLaunchKernelGGL(k_expand<8>, ge, b, 0, st, fA, lv, l, ni, left, right, key, kids, prefix, sums, err);
					else
						hipLaunchKernelGGL(k_expand<4>, ge, b, 0, st, fA, lv, l, ni, left, right, key, kids, prefix, sums, err);
					hipLaunchKernelGGL(k_levelScan, dim3(1), dim3(1024), 0, st, sums, lv, l, (uint32_t)capNodes, S.pin + 4, err);
					if (in.layout == 2)
						hipLaunchKernelGGL((k_emit<8, lrh_node8q>), gm, b, 0, st, lv, l, kids, prefix, sums, first, last, key,
								leafBox, nodeBox, static_cast<lrh_node8q *>(nodes), fB);
					else if (in.layout == 1)
						hipLaunchKernelGGL((k_emit<4, lrh_node4f>), gm, b, 0, st, lv, l, kids, prefix, sums, first, last, key,
								leafBox, nodeBox, static_cast<lrh_node4f *>(nodes), fB);
					else
						hipLaunchKernelGGL((k_emit<4, lrh_node4q>), gm, b, 0, st, lv, l, kids, prefix, sums, first, last, key,
								leafBox, nodeBox, static_cast<lrh_node4q *>(nodes), fB);
					GB_CHECK(hipGetLastError());
					std::swap(fA, fB);
				}
				if (const uint32_t e = readError(S, err, st)) throw std::runtime_error(errorText(e));
				nf = S.pin[4];
			}
			depth = S.pin[6];
			const uint32_t levelBase = S.pin[5];
			nodeCount = levelBase;
		}
		// triangle records in leaf order
		allocRecords();
		hipLaunchKernelGGL(k_records, dim3(grid(n, 256)), dim3(256), 0, st, in.verts, in.tris, tbase, vbase,
				in.nMeshes, vals, n, static_cast<lrh_tri *>(out->tris), out->invPerm);
		GB_CHECK(hipGetLastError());
		// right-size the node array
		out->nodeBytes = (size_t)nodeCount * nodeSz;
		out->nodes = a.alloc(a.ctx, out->nodeBytes);
		GB_CHECK(hipMemcpyAsync(out->nodes, nodes, out->nodeBytes, hipMemcpyDeviceToDevice, st));
		GB_CHECK(hipEventRecord(e1, st));
		GB_CHECK(hipStreamSynchronize(st));
	} catch (...) {
		(void)hipStreamSynchronize(st);  // nothing in flight may still use what is released below
		a.release(a.ctx, nodes, capNodes * nodeSz);
		if (out->tris) a.release(a.ctx, out->tris, out->triBytes);
		if (out->invPerm) a.release(a.ctx, out->invPerm, out->invPermBytes);
		if (out->nodes) a.release(a.ctx, out->nodes, out->nodeBytes);
		out->tris = out->nodes = nullptr;
		out->invPerm = nullptr;
		(void)hipEventDestroy(e0);
		(void)hipEventDestroy(e1);
		throw;
	}
	a.release(a.ctx, nodes, capNodes * nodeSz);
	float ms = 0.f;
	(void)hipEventElapsedTime(&ms, e0, e1);
	(void)hipEventDestroy(e0);
	(void)hipEventDestroy(e1);
	out->nodeCount = nodeCount;
	out->root = 0;
	out->maxDepth = depth ? depth - 1 : 0;
	out->kernelMs = ms;
}
