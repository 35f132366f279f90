/*
 * gfx950 traversal kernels of the HIP intersection device.
 *
 * One lane = one ray, wave64, persistent grid.  Per wave, a ballot over idle
 * lanes takes ray tickets from its block's pool and hands them out by lane
 * rank, so lanes whose ray terminated are refilled while the others keep
 * traversing (the reference launches one thread per ray with no refill,
 * include/luxrays/accelerators/bvh.cl:228-260).
 *
 * Traversal is ordered (children sorted by entry distance) over 4-wide or
 * 8-wide nodes, with a per-lane stack whose top `ldsDepth` entries live in LDS and
 * deeper entries spill to a global scratch array (lrh_stack.h); popped entries
 * whose entry distance is above the current hit's, widened, are dropped
 * without a fetch.  The reference walks a skip-pointer array in memory order
 * instead (bvh.cl:136-217, src/luxrays/accelerators/bvhaccel.cpp:184-257); both
 * visit a superset of the boxes containing the closest hit, so the closest hit
 * is the same up to ties at equal t.  Which of two hits at equal t a ray
 * reports is fixed by the scene and the ray: every kernel here visits alike.
 *
 * The triangle test is Triangle::Intersect
 * (include/luxrays/core/geometry/triangle.h:55-89) with every operation
 * rounded as written (the file builds with -ffp-contract=off and correctly
 * rounded division) and the acceptance rule of BVHAccel::Intersect
 * (bvhaccel.cpp:173, 232-233): a hit is kept iff mint <= t < best, best
 * starting at maxt.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lrh_layout.h"
#include "lrh_kernels.h"
#include "lrh_motion_dev.h"
#include "lrh_rcp.h"
#include "lrh_stack.h"

#define LRH_SENTINEL 0xfffffffeu
#define DEVI __device__ __forceinline__

namespace {

using Stack = lrhstack::Stack<uint2>;
using lrhstack::drainPop;
using lrhstack::drainPush;
using lrhstack::overfull;
using lrhstack::pop;

DEVI float asf(uint32_t u) { return __uint_as_float(u); }
DEVI uint32_t asu(float f) { return __float_as_uint(f); }

// Reciprocal of a direction component for the box tests: a zero component
// becomes +-1e-20 so slab products stay finite.  The hardware estimate and one
// Newton step give the division's value with eight instructions less, for
// every ray and, in two-level scenes, on entering and on leaving an object
// (moving instances by division, then by the estimate alone 1,365 and 1,320
// us; the step, later, 1,230 -> 1,236).  The estimate flushes results below the
// normal range, so huge components are divided.
DEVI float safeRcp(float d) {
	const float dd = fabsf(d) < 1e-20f ? copysignf(1e-20f, d) : d;
	return lrhRefineRcp(dd, __builtin_amdgcn_rcpf(dd));
}

DEVI float byteF(uint32_t w, int c) {
	// compiles to v_cvt_f32_ubyteN
	return (float)((w >> (8 * c)) & 0xffu);
}

struct LocalRay {
	float ox, oy, oz, dx, dy, dz;
	float ix, iy, iz;     // 1/d
	float nx, ny, nz;     // -o/d
};

DEVI void setupRay(LocalRay &r) {
	r.ix = safeRcp(r.dx);
	r.iy = safeRcp(r.dy);
	r.iz = safeRcp(r.dz);
	if (fmaxf(fmaxf(fabsf(r.dx), fabsf(r.dy)), fabsf(r.dz)) > 1e30f) {
		if (fabsf(r.dx) > 1e30f) r.ix = 1.0f / r.dx;
		if (fabsf(r.dy) > 1e30f) r.iy = 1.0f / r.dy;
		if (fabsf(r.dz) > 1e30f) r.iz = 1.0f / r.dz;
	}
	r.nx = -r.ox * r.ix;
	r.ny = -r.oy * r.iy;
	r.nz = -r.oz * r.iz;
}

// Matrix * Point with the projective divide and Matrix * Vector
// (include/luxrays/core/geometry/matrix4x4op.h:31-59), rounded as written.
DEVI void xfRay(const float *M, const float wo[3], const float wd[3], LocalRay &r) {
	const float x = wo[0], y = wo[1], z = wo[2];
	float px = M[0] * x + M[1] * y + M[2] * z + M[3];
	float py = M[4] * x + M[5] * y + M[6] * z + M[7];
	float pz = M[8] * x + M[9] * y + M[10] * z + M[11];
	const float w = M[12] * x + M[13] * y + M[14] * z + M[15];
	if (w != 1.f) {
		const float inv = 1.f / w;
		px = inv * px; py = inv * py; pz = inv * pz;
	}
	r.ox = px; r.oy = py; r.oz = pz;
	const float a = wd[0], b = wd[1], c = wd[2];
	r.dx = M[0] * a + M[1] * b + M[2] * c;
	r.dy = M[4] * a + M[5] * b + M[6] * c;
	r.dz = M[8] * a + M[9] * b + M[10] * c;
	setupRay(r);
}

// ---- motion sampling: MotionSystem::Sample picks the segment
// (src/luxrays/core/geometry/motionsystem.cpp:340-346), lrhSegSample
// evaluates it (InterpolatedTransform::Sample, :89-159) ----
__device__ __forceinline__ void motionSample(const lrh_motion *mot, const lrh_motion_seg *segs, const float *times,
		float time, float M[16]) {
	// upper_bound(times, time), clamped to the last key; the record's
	// inline key times serve systems of up to LRH_MOTION_INLINE_TIMES keys
	const uint4 a = reinterpret_cast<const uint4 *>(mot)[0];
	const uint4 b = reinterpret_cast<const uint4 *>(mot)[1];
	// both halves of the record in one wait
	uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
	for (int k = 0; k < 8; ++k) asm volatile("" : "+v"(w[k]));
	const uint32_t n = w[1];
	uint32_t idx = 0;
	if (n <= LRH_MOTION_INLINE_TIMES) {
		const float tk[4] = {__uint_as_float(w[4]), __uint_as_float(w[5]), __uint_as_float(w[6]),
				__uint_as_float(w[7])};
#pragma unroll
		for (uint32_t k = 0; k < 4; ++k)
			if (idx == k && k < n && !(time < tk[k])) idx = k + 1;
	} else {
		const float *tk = times + w[0];
		while (idx < n && !(time < tk[idx])) ++idx;
	}
	if (idx > n - 1) idx = n - 1;
	lrhSegSample(segs[w[2] + idx], time, M);
}

// ---- node tests: up to 4 children -> (entry distance, child ref) ----
// The slab interval is widened conservatively on its far side only, by 2^-19
// of |t| and with the current hit's distance in it: what a hit at t needs is
// entry <= exit with both off by up to 2^-20 of |t|, and the same of entry
// and best, so one widening of min(exit, best) serves where one on each side
// was two instructions per child.  Adding a multiple of |t| is wider for
// either sign of t, which a scale by 1 + eps is not (negative mint).
constexpr float kWiden = 1.0f / 524288.0f;
DEVI float widen(float t) { return fmaf(fabsf(t), kWiden, t); }

DEVI void testNodeQ(const lrh_node4q *__restrict__ nodes, uint32_t idx, const LocalRay &r, float mint, float best,
		float t[4], uint32_t c[4]) {
	const uint4 *p = reinterpret_cast<const uint4 *>(nodes + idx);
	const uint4 q0 = p[0], q1 = p[1], q2 = p[2], q3 = p[3];
	const float sx = asf((q0.w & 0xffu) << 23), sy = asf(((q0.w >> 8) & 0xffu) << 23),
			sz = asf(((q0.w >> 16) & 0xffu) << 23);
	const float Ax = sx * r.ix, Ay = sy * r.iy, Az = sz * r.iz;
	const float Bx = fmaf(asf(q0.x), r.ix, r.nx), By = fmaf(asf(q0.y), r.iy, r.ny), Bz = fmaf(asf(q0.z), r.iz, r.nz);
	const uint32_t nX = r.ix >= 0.f ? q1.x : q1.y, fX = r.ix >= 0.f ? q1.y : q1.x;
	const uint32_t nY = r.iy >= 0.f ? q1.z : q1.w, fY = r.iy >= 0.f ? q1.w : q1.z;
	const uint32_t nZ = r.iz >= 0.f ? q2.x : q2.y, fZ = r.iz >= 0.f ? q2.y : q2.x;
	c[0] = q2.z; c[1] = q2.w; c[2] = q3.x; c[3] = q3.y;
#pragma unroll
	for (int k = 0; k < 4; ++k) {
		const float tnx = fmaf(byteF(nX, k), Ax, Bx), tfx = fmaf(byteF(fX, k), Ax, Bx);
		const float tny = fmaf(byteF(nY, k), Ay, By), tfy = fmaf(byteF(fY, k), Ay, By);
		const float tnz = fmaf(byteF(nZ, k), Az, Bz), tfz = fmaf(byteF(fZ, k), Az, Bz);
		const float a = fmaxf(fmaxf(fmaxf(tnx, tny), tnz), mint), b = widen(fminf(fminf(fminf(tfx, tfy), tfz), best));
		// empty slots hold inverted boxes; one that still passes (a far node
		// whose inverted extent is below the widening) is dropped when its
		// LRH_CHILD_EMPTY reference is taken or popped
		t[k] = (a <= b) ? a : INFINITY;
	}
}

// 8-wide quantized node: six 16-byte loads (origin and scales, the three
// axes' bytes, eight child references)
DEVI void testNode8Q(const lrh_node8q *__restrict__ nodes, uint32_t idx, const LocalRay &r, float mint, float best,
		float t[8], uint32_t c[8]) {
	const uint4 *p = reinterpret_cast<const uint4 *>(nodes + idx);
	const uint4 q0 = p[0], q1 = p[1], q2 = p[2], q3 = p[3], q4 = p[4], q5 = p[5];
	const float sx = asf((q0.w & 0xffu) << 23), sy = asf(((q0.w >> 8) & 0xffu) << 23),
			sz = asf(((q0.w >> 16) & 0xffu) << 23);
	const float Ax = sx * r.ix, Ay = sy * r.iy, Az = sz * r.iz;
	const float Bx = fmaf(asf(q0.x), r.ix, r.nx), By = fmaf(asf(q0.y), r.iy, r.ny), Bz = fmaf(asf(q0.z), r.iz, r.nz);
	const bool px = r.ix >= 0.f, py = r.iy >= 0.f, pz = r.iz >= 0.f;
	const uint32_t nX[2] = {px ? q1.x : q1.z, px ? q1.y : q1.w}, fX[2] = {px ? q1.z : q1.x, px ? q1.w : q1.y};
	const uint32_t nY[2] = {py ? q2.x : q2.z, py ? q2.y : q2.w}, fY[2] = {py ? q2.z : q2.x, py ? q2.w : q2.y};
	const uint32_t nZ[2] = {pz ? q3.x : q3.z, pz ? q3.y : q3.w}, fZ[2] = {pz ? q3.z : q3.x, pz ? q3.w : q3.y};
	c[0] = q4.x; c[1] = q4.y; c[2] = q4.z; c[3] = q4.w;
	c[4] = q5.x; c[5] = q5.y; c[6] = q5.z; c[7] = q5.w;
#pragma unroll
	for (int k = 0; k < 8; ++k) {
		const int w = k >> 2, b = k & 3;
		const float tnx = fmaf(byteF(nX[w], b), Ax, Bx), tfx = fmaf(byteF(fX[w], b), Ax, Bx);
		const float tny = fmaf(byteF(nY[w], b), Ay, By), tfy = fmaf(byteF(fY[w], b), Ay, By);
		const float tnz = fmaf(byteF(nZ[w], b), Az, Bz), tfz = fmaf(byteF(fZ[w], b), Az, Bz);
		const float a = fmaxf(fmaxf(fmaxf(tnx, tny), tnz), mint), bb = widen(fminf(fminf(fminf(tfx, tfy), tfz), best));
		t[k] = (a <= bb) ? a : INFINITY;
	}
}

DEVI void testNodeF(const lrh_node4f *__restrict__ nodes, uint32_t idx, const LocalRay &r, float mint, float best,
		float t[4], uint32_t c[4]) {
	const float4 *p = reinterpret_cast<const float4 *>(nodes + idx);
	const float4 lx = p[0], hx = p[1], ly = p[2], hy = p[3], lz = p[4], hz = p[5];
	const uint4 cc = reinterpret_cast<const uint4 *>(p)[6];
	c[0] = cc.x; c[1] = cc.y; c[2] = cc.z; c[3] = cc.w;
	const float LX[4] = {lx.x, lx.y, lx.z, lx.w}, HX[4] = {hx.x, hx.y, hx.z, hx.w};
	const float LY[4] = {ly.x, ly.y, ly.z, ly.w}, HY[4] = {hy.x, hy.y, hy.z, hy.w};
	const float LZ[4] = {lz.x, lz.y, lz.z, lz.w}, HZ[4] = {hz.x, hz.y, hz.z, hz.w};
	const bool sx = r.ix >= 0.f, sy = r.iy >= 0.f, sz = r.iz >= 0.f;
#pragma unroll
	for (int k = 0; k < 4; ++k) {
		const float tnx = fmaf(sx ? LX[k] : HX[k], r.ix, r.nx), tfx = fmaf(sx ? HX[k] : LX[k], r.ix, r.nx);
		const float tny = fmaf(sy ? LY[k] : HY[k], r.iy, r.ny), tfy = fmaf(sy ? HY[k] : LY[k], r.iy, r.ny);
		const float tnz = fmaf(sz ? LZ[k] : HZ[k], r.iz, r.nz), tfz = fmaf(sz ? HZ[k] : LZ[k], r.iz, r.nz);
		const float a = fmaxf(fmaxf(fmaxf(tnx, tny), tnz), mint), b = widen(fminf(fminf(fminf(tfx, tfy), tfz), best));
		t[k] = (a <= b) ? a : INFINITY;  // empty slots: lo = +inf, hi = -inf
	}
}

// Children as (entry distance, reference) in one double: the distance's bits
// are its high word, so doubles order as the distances do (INFINITY's bits are
// those of a finite double, and no distance is a NaN), and a comparator is one
// v_min_f64 and one v_max_f64, each issued in 4 cycles like any fp32 minimum,
// where comparing and exchanging two registers takes one compare and four
// selects of 4 cycles each.  Equal distances order by reference.  Of hits at
// the same distance the first one tested is reported, so every kernel and the
// drain visit a closest ray's children in this order (and an any-hit ray's in
// the network's): its hit is then its own, whatever launch it is part of.
DEVI double key64(float t, uint32_t c) { return __hiloint2double((int)asu(t), (int)c); }
DEVI float keyT(double k) { return asf((uint32_t)__double2hiint(k)); }
DEVI uint32_t keyC(double k) { return (uint32_t)__double2loint(k); }
DEVI void kswap(double &a, double &b) {
	double lo, hi;
	asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
	asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
	a = lo;
	b = hi;
}

DEVI void cswap(float &ta, uint32_t &ca, float &tb, uint32_t &cb) {
	const bool s = tb < ta;
	const float t0 = s ? tb : ta, t1 = s ? ta : tb;
	const uint32_t c0 = s ? cb : ca, c1 = s ? ca : cb;
	ta = t0; tb = t1; ca = c0; cb = c1;
}

// Triangle::Intersect on one record, rounded as written: true if the ray
// hits it at mint <= t < best
DEVI bool testTri(const lrh_tri *__restrict__ rec, const LocalRay &r, float mint, float best, float &t, float &b1,
		float &b2, uint32_t &triIndex, uint32_t &meshIndex) {
	const uint4 *tp = reinterpret_cast<const uint4 *>(rec);
	const uint4 a = tp[0], b = tp[1], c = tp[2];
	const float p0x = asf(a.x), p0y = asf(a.y), p0z = asf(a.z);
	const float e1x = asf(a.w), e1y = asf(b.x), e1z = asf(b.y);
	const float e2x = asf(b.z), e2y = asf(b.w), e2z = asf(c.x);
	const float s1x = (r.dy * e2z) - (r.dz * e2y);
	const float s1y = (r.dz * e2x) - (r.dx * e2z);
	const float s1z = (r.dx * e2y) - (r.dy * e2x);
	const float div = s1x * e1x + s1y * e1y + s1z * e1z;
	const float inv = 1.f / div;
	const float ddx = r.ox - p0x, ddy = r.oy - p0y, ddz = r.oz - p0z;
	b1 = (ddx * s1x + ddy * s1y + ddz * s1z) * inv;
	const float s2x = (ddy * e1z) - (ddz * e1y);
	const float s2y = (ddz * e1x) - (ddx * e1z);
	const float s2z = (ddx * e1y) - (ddy * e1x);
	b2 = (r.dx * s2x + r.dy * s2y + r.dz * s2z) * inv;
	const float b0 = 1.f - b1 - b2;
	t = (e2x * s2x + e2y * s2y + e2z * s2z) * inv;
	triIndex = c.y;
	meshIndex = c.z;
	return (div != 0.f) && !(b1 < 0.f) && !(b2 < 0.f) && !(b0 < 0.f) &&
			!(t < mint) && (t < best);
}

// sorting networks: 5 comparators for four entries, 19 for eight
DEVI void sort4(float t[4], uint32_t c[4]) {
	cswap(t[0], c[0], t[1], c[1]);
	cswap(t[2], c[2], t[3], c[3]);
	cswap(t[0], c[0], t[2], c[2]);
	cswap(t[1], c[1], t[3], c[3]);
	cswap(t[1], c[1], t[2], c[2]);
}
DEVI void sort4Closest(float t[4], uint32_t c[4]) {
	double k[4];
#pragma unroll
	for (int i = 0; i < 4; ++i) k[i] = key64(t[i], c[i]);
	kswap(k[0], k[1]);
	kswap(k[2], k[3]);
	kswap(k[0], k[2]);
	kswap(k[1], k[3]);
	kswap(k[1], k[2]);
#pragma unroll
	for (int i = 0; i < 4; ++i) { t[i] = keyT(k[i]); c[i] = keyC(k[i]); }
}
DEVI void sort8(float t[8], uint32_t c[8]) {
	cswap(t[0], c[0], t[2], c[2]); cswap(t[1], c[1], t[3], c[3]);
	cswap(t[4], c[4], t[6], c[6]); cswap(t[5], c[5], t[7], c[7]);
	cswap(t[0], c[0], t[4], c[4]); cswap(t[1], c[1], t[5], c[5]);
	cswap(t[2], c[2], t[6], c[6]); cswap(t[3], c[3], t[7], c[7]);
	cswap(t[0], c[0], t[1], c[1]); cswap(t[2], c[2], t[3], c[3]);
	cswap(t[4], c[4], t[5], c[5]); cswap(t[6], c[6], t[7], c[7]);
	cswap(t[2], c[2], t[4], c[4]); cswap(t[3], c[3], t[5], c[5]);
	cswap(t[1], c[1], t[4], c[4]); cswap(t[3], c[3], t[6], c[6]);
	cswap(t[1], c[1], t[2], c[2]); cswap(t[3], c[3], t[4], c[4]);
	cswap(t[5], c[5], t[6], c[6]);
}
DEVI void sort8Closest(float t[8], uint32_t c[8]) {
	double k[8];
#pragma unroll
	for (int i = 0; i < 8; ++i) k[i] = key64(t[i], c[i]);
	kswap(k[0], k[2]); kswap(k[1], k[3]); kswap(k[4], k[6]); kswap(k[5], k[7]);
	kswap(k[0], k[4]); kswap(k[1], k[5]); kswap(k[2], k[6]); kswap(k[3], k[7]);
	kswap(k[0], k[1]); kswap(k[2], k[3]); kswap(k[4], k[5]); kswap(k[6], k[7]);
	kswap(k[2], k[4]); kswap(k[3], k[5]); kswap(k[1], k[4]); kswap(k[3], k[6]);
	kswap(k[1], k[2]); kswap(k[3], k[4]); kswap(k[5], k[6]);
#pragma unroll
	for (int i = 0; i < 8; ++i) { t[i] = keyT(k[i]); c[i] = keyC(k[i]); }
}

DEVI bool push(Stack &s, uint32_t ref, float t, uint32_t *err) {
	return lrhstack::push(s, make_uint2(ref, asu(t)), [err]() { atomicOr(err, 1u); });
}

// ---- ray tickets ----
// A launch hands out its first rays by lane (waveRays to each wave) and the
// rest through counters in memory.  Atomics on one address from all eight
// XCDs take 11.4 ns each, whatever the number of waves, and when all waves
// come at once, for their second ray or to learn that there is none, the last
// waits 80 us; on eight addresses they take 1.9 ns.  So the blocks form eight
// groups (blockIdx modulo eight, as they are dealt to the XCDs), each with a
// counter of its own and every eighth unit of 256 rays, and a block's waves
// go there for a chunk that they divide through a pool in LDS.
// (2,073,600 rays, one counter and an atomic for each refill -> a pool -> and
// eight counters: camera rays 662 -> 395 -> 368 us; 500,001 shadow rays 300 ->
// 188 -> 140; 921,600 in a room 219 -> 145, a sixth of them live 200 -> 123.)
constexpr uint32_t kUnit = 256u;
struct TicketPool {
	unsigned long long range;  // low half: next ticket, high half: end of the chunk
	uint32_t fetching;         // 1: a wave of the block is replacing the chunk; 2: the counter is past the group's last
};

struct Tickets {
	uint32_t b0, n0, b1, n1;  // n0 tickets from b0, then n1 from b1
	bool exhausted;           // nothing is left in the counter (or, for this wave, in the pool)
};

// tickets of group g beyond the `first` rays handed out by lane (the last
// unit may run past the launch's rays)
DEVI uint32_t groupTickets(uint32_t g, uint32_t groups, uint32_t first, uint32_t nRays) {
	if (first >= nRays) return 0u;
	const uint32_t units = (nRays - first + kUnit - 1u) / kUnit;
	return units > g ? (units - g + groups - 1u) / groups * kUnit : 0u;
}

// the ray of ticket x of group g
DEVI uint32_t rayOf(uint32_t x, uint32_t g, uint32_t groups, uint32_t first) {
	return first + ((x / kUnit) * groups + g) * kUnit + x % kUnit;
}

// takes up to n tickets from the pool: the first one in `base`
DEVI uint32_t poolTake(TicketPool &pool, uint32_t n, uint32_t &base, uint32_t &end) {
	const unsigned long long old = __hip_atomic_fetch_add(&pool.range, (unsigned long long)n, __ATOMIC_RELAXED,
			__HIP_MEMORY_SCOPE_WORKGROUP);
	base = (uint32_t)old;
	end = (uint32_t)(old >> 32);
	return base < end ? (end - base < n ? end - base : n) : 0u;
}

// Tickets for a wave's n idle lanes, by its lane `leader`.  A wave that finds
// the pool empty takes what it still needs from the counter; if no other
// wave of its block is doing so it also takes a chunk for the pool.  Only the
// holder of `fetching` replaces the chunk, after it has found the pool empty
// while holding it, so no ticket is lost; nobody waits for it.  The chunk is
// a share of what was left at the block's last visit, so that the launch
// ends evenly: large reservations to the end cost 13%.  A wave stops asking
// once the counter is past the group's last ticket, and its block's other
// waves with it; a chunk that a wave has not seen then belongs to the wave
// that took it, which asks again.
DEVI Tickets takeTickets(TicketPool &pool, uint32_t *counter, uint32_t n, uint32_t total, uint32_t blocks,
		uint32_t leader) {
	uint32_t b0 = 0, n0 = 0, b1 = 0, n1 = 0, over = 0;
	if (__lane_id() == leader) {
		uint32_t end;
		n0 = poolTake(pool, n, b0, end);
		const uint32_t rest = n - n0;
		if (rest) {
			uint32_t chunk = 0, held = 0u;
			__hip_atomic_compare_exchange_strong(&pool.fetching, &held, 1u, __ATOMIC_ACQUIRE, __ATOMIC_RELAXED,
					__HIP_MEMORY_SCOPE_WORKGROUP);
			const bool mine = held == 0u;
			over = held == 2u ? 1u : 0u;
			if (mine) {
				// another wave may have put a chunk there meanwhile
				n1 = poolTake(pool, rest, b1, end);
				chunk = (total - (end < total ? end : total)) / blocks;
				chunk = chunk < 256u ? chunk : 256u;
				if (chunk < 16u) chunk = 0;
			}
			if (n1 == 0 && !over) {
				b1 = atomicAdd(counter, rest + chunk);
				n1 = rest;
				over = b1 + rest >= total ? 1u : 0u;
				if (mine && chunk) {
					const uint32_t a = b1 + rest, e = a + chunk < total ? a + chunk : total;
					__hip_atomic_store(&pool.range, ((unsigned long long)e << 32) | a, __ATOMIC_RELAXED,
							__HIP_MEMORY_SCOPE_WORKGROUP);
				}
			}
			if (mine) __hip_atomic_store(&pool.fetching, over ? 2u : 0u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
		}
	}
	Tickets t;
	t.b0 = (uint32_t)__builtin_amdgcn_readlane((int)b0, (int)leader);
	t.n0 = (uint32_t)__builtin_amdgcn_readlane((int)n0, (int)leader);
	t.b1 = (uint32_t)__builtin_amdgcn_readlane((int)b1, (int)leader);
	t.n1 = (uint32_t)__builtin_amdgcn_readlane((int)n1, (int)leader);
	t.exhausted = __builtin_amdgcn_readlane((int)over, (int)leader) != 0;
	return t;
}

constexpr uint32_t kNoRay = 0xffffffffu;
// Stack entries a lane pops in one pass: a lane whose entries all lie behind
// its hit goes on popping in the next pass instead of holding up the wave
// (no limit / 1 / 2 / 3: bounce rays over 26.2M triangles 600 / 603 / 603 /
// 600 us, over 2.1M 174 / 165 / 168 / 168, a soup 871 / 895 / 863 / 863, moving
// instances 1,292 / 1,311 / 1,238 / 1,244).
constexpr uint32_t kMaxPops = 2;
constexpr uint32_t kMaxSteps = 1u << 24;  // per-ray guard against corrupt trees

}  // namespace

// Per-lane view of the scene and buffers a ray belongs to.  In a plain trace
// every field comes from the launch parameters (uniform, kept in SGPRs); in a
// batched trace each lane loads its item's descriptor when it takes a ray.
struct SceneView {
	const void *nodes;
	const lrh_tri *tris;
	const lrh_inst *insts;
	const float *xforms;
	const lrh_motion *motions;
	const lrh_motion_seg *segs;
	const float *times;
	lrh_hit_rec *hits;
	uint32_t root;
	uint32_t flags;  // LRH_ITEM_ANY | LRH_ITEM_TWO
};

// ---- the drain: once no tickets are left and a wave holds at most 64 / W
// rays, W lanes take each of them, a lane per child of a node and per
// triangle of a leaf (W = the width of the nodes) ----
// At the end of a launch every wave waits for its longest ray with the
// other lanes idle, and its passes cost as much for one ray as for 64.  Shared
// by W lanes a pass takes about a fifth of the vector instructions, with the
// same order of visits and the same arithmetic, so the same hits.
template <int CTRL>
DEVI uint32_t dpp(uint32_t x) {
	return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
}
constexpr int kXor1 = 0xb1, kXor2 = 0x4e, kXor3 = 0x1b, kHalfMirror = 0x141;  // quad_perm, row_half_mirror

// how many of the group's W keys (key64) are below this lane's
template <int CTRL>
DEVI double dppKey(double k) {
	return __hiloint2double((int)dpp<CTRL>((uint32_t)__double2hiint(k)), (int)dpp<CTRL>((uint32_t)__double2loint(k)));
}
template <int W>
DEVI uint32_t groupRank(double key) {
	uint32_t n = (dppKey<kXor1>(key) < key) + (dppKey<kXor2>(key) < key) + (dppKey<kXor3>(key) < key);
	if (W == 8) {
		const double m = dppKey<kHalfMirror>(key);
		n += (m < key) + (dppKey<kXor1>(m) < key) + (dppKey<kXor2>(m) < key) + (dppKey<kXor3>(m) < key);
	}
	return n;
}

// One layer of a sorting network across the lanes of a group: the lanes of
// `part` exchange with their partner (its entry: ot, oc), those of `low`
// keep the nearer entry; equal ones stay, as in cswap.
template <uint32_t PART, uint32_t LOW>
DEVI void layer(uint32_t lane, float &t, uint32_t &ref, float ot, uint32_t oc) {
	const bool low = (LOW >> lane) & 1u, part = (PART >> lane) & 1u;
	const bool s = part && (low ? ot < t : t < ot);
	t = s ? ot : t;
	ref = s ? oc : ref;
}

// sort4 / sort8 across the lanes of a group, lane k with entry k: any-hit rays
// report the first blocker they meet, so equal distances must come out in
// the network's order here too
template <int W>
DEVI void groupSort(uint32_t lane, float &t, uint32_t &ref) {
	auto T = [&t](auto f) { return asf(f(asu(t))); };
	auto x1 = [](uint32_t x) { return dpp<kXor1>(x); };
	auto x2 = [](uint32_t x) { return dpp<kXor2>(x); };
	auto x3 = [](uint32_t x) { return dpp<kXor3>(x); };
	if (W == 4) {
		layer<0xf, 0x5>(lane, t, ref, T(x1), x1(ref));
		layer<0xf, 0x3>(lane, t, ref, T(x2), x2(ref));
		layer<0x6, 0x2>(lane, t, ref, T(x3), x3(ref));
		return;
	}
	auto x7 = [](uint32_t x) { return dpp<kHalfMirror>(x); };
	auto x4 = [](uint32_t x) { return dpp<kXor3>(dpp<kHalfMirror>(x)); };
	auto x5 = [](uint32_t x) { return dpp<kXor2>(dpp<kHalfMirror>(x)); };
	auto x6 = [](uint32_t x) { return dpp<kXor1>(dpp<kHalfMirror>(x)); };
	layer<0xff, 0x33>(lane, t, ref, T(x2), x2(ref));
	layer<0xff, 0x0f>(lane, t, ref, T(x4), x4(ref));
	layer<0xff, 0x55>(lane, t, ref, T(x1), x1(ref));
	layer<0x3c, 0x0c>(lane, t, ref, T(x6), x6(ref));  // (2,4) (3,5)
	layer<0x5a, 0x0a>(lane, t, ref, T(x5), x5(ref));  // (1,4) (3,6)
	const bool mid = lane == 3 || lane == 4;          // (1,2) (3,4) (5,6)
	const float t3 = T(x3), t7 = T(x7);
	const uint32_t r3 = x3(ref), r7 = x7(ref);
	layer<0x7e, 0x2a>(lane, t, ref, mid ? t7 : t3, mid ? r7 : r3);
}

// the group's smallest float, to all its lanes
template <int W>
DEVI float groupMin(float x) {
	x = fminf(x, asf(dpp<kXor1>(asu(x))));
	x = fminf(x, asf(dpp<kXor2>(asu(x))));
	if (W == 8) x = fminf(x, asf(dpp<kHalfMirror>(asu(x))));
	return x;
}

DEVI void waveFence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

template <int LAYOUT, bool TWO, bool ANY, int BATCH>
DEVI void drain(const LrhTraceParams &P, Stack &st, SceneView &v, LocalRay &r, float wo[3], float wd[3], float mint,
		float best, float time, float hb1, float hb2, uint32_t hTri, uint32_t hMesh, uint32_t cur, float curT,
		uint32_t obj, bool inInst, uint32_t rid) {
	constexpr uint32_t W = LAYOUT == 2 ? 8u : 4u;
	const uint32_t lane = __lane_id();
	const uint32_t c = lane & (W - 1u), group = lane / W;
	// group g takes the g-th live ray: its registers from the lane that held
	// it, its stack where it is
	uint64_t live = __ballot(rid != kNoRay);
	const uint32_t nLive = (uint32_t)__popcll(live);
	uint32_t src = lane;
	for (uint32_t g = 0; g < nLive; ++g) {
		const uint32_t l = (uint32_t)__ffsll((long long)live) - 1u;
		live &= live - 1u;
		if (group == g) src = l;
	}
	auto shu = [src](uint32_t x) { return (uint32_t)__shfl((int)x, (int)src); };
	auto shf = [&](float x) { return asf(shu(asu(x))); };
	auto shp = [&](auto *x) {
		const uint64_t a = (uint64_t)x;
		return (decltype(x))(((uint64_t)shu((uint32_t)(a >> 32)) << 32) | shu((uint32_t)a));
	};
	r.ox = shf(r.ox); r.oy = shf(r.oy); r.oz = shf(r.oz);
	r.dx = shf(r.dx); r.dy = shf(r.dy); r.dz = shf(r.dz);
	r.ix = shf(r.ix); r.iy = shf(r.iy); r.iz = shf(r.iz);
	r.nx = shf(r.nx); r.ny = shf(r.ny); r.nz = shf(r.nz);
	mint = shf(mint); best = shf(best); hb1 = shf(hb1); hb2 = shf(hb2); curT = shf(curT);
	hTri = shu(hTri); hMesh = shu(hMesh); cur = shu(cur);
	if (TWO) {
		for (int k = 0; k < 3; ++k) { wo[k] = shf(wo[k]); wd[k] = shf(wd[k]); }
		time = shf(time);
		obj = shu(obj);
		inInst = shu(inInst ? 1u : 0u) != 0u;
	}
	if (BATCH) {
		v.nodes = shp(v.nodes);
		v.tris = shp(v.tris);
		v.hits = shp(v.hits);
		v.flags = shu(v.flags);
		if (TWO) {
			v.insts = shp(v.insts);
			v.xforms = shp(v.xforms);
			v.motions = shp(v.motions);
			v.segs = shp(v.segs);
			v.times = shp(v.times);
		}
	}
	st.sp = shu(st.sp);
	st.lane = (st.lane & ~63u) + src;
	const uint32_t taken = shu(rid);  // (every exchange with all lanes active)
	rid = group < nLive ? taken : kNoRay;
	const bool two = TWO && (v.flags & LRH_ITEM_TWO);
	const bool anyq = ANY && (BATCH == LRH_BATCH || (v.flags & LRH_ITEM_ANY));
	const bool leader = c == 0;
	const auto full = [err = P.error]() { atomicOr(err, 1u); };
	waveFence();
	for (uint32_t steps = 0; __ballot(rid != kNoRay); ++steps) {
		if (rid == kNoRay) continue;
		bool done = false;
		while (cur == LRH_CHILD_EMPTY && st.sp) {
			const uint2 e = drainPop(st, leader);
			waveFence();
			cur = e.x;
			curT = asf(e.y);
			if (TWO && cur == LRH_SENTINEL) {
				r.ox = wo[0]; r.oy = wo[1]; r.oz = wo[2];
				r.dx = wd[0]; r.dy = wd[1]; r.dz = wd[2];
				setupRay(r);
				inInst = false;
				cur = LRH_CHILD_EMPTY;
			} else if (!(curT <= widen(best)))
				cur = LRH_CHILD_EMPTY;
		}
		if (cur != LRH_CHILD_EMPTY && !(cur & LRH_CHILD_LEAF)) {
			float tnx, tfx, tny, tfy, tnz, tfz;
			uint32_t child;
			if (LAYOUT == 1) {
				const char *nb = reinterpret_cast<const char *>(reinterpret_cast<const lrh_node4f *>(v.nodes) + cur) + 4 * c;
				const uint32_t x = r.ix >= 0.f ? 0u : 16u, y = r.iy >= 0.f ? 32u : 48u, z = r.iz >= 0.f ? 64u : 80u;
				auto f = [nb](uint32_t off) { return *reinterpret_cast<const float *>(nb + off); };
				tnx = fmaf(f(x), r.ix, r.nx); tfx = fmaf(f(x ^ 16u), r.ix, r.nx);
				tny = fmaf(f(y), r.iy, r.ny); tfy = fmaf(f(y ^ 16u), r.iy, r.ny);
				tnz = fmaf(f(z), r.iz, r.nz); tfz = fmaf(f(z ^ 16u), r.iz, r.nz);
				child = *reinterpret_cast<const uint32_t *>(nb + 96);
			} else {
				// the bounds' words of this child: lo and hi of an axis are `far` bytes apart
				constexpr uint32_t far = W, axis = 2 * W;
				const char *nb = reinterpret_cast<const char *>(v.nodes) + (size_t)cur * (LAYOUT == 2 ? 128u : 64u);
				const uint4 q0 = *reinterpret_cast<const uint4 *>(nb);
				const uint32_t o = 16u + (c & 4u);
				const uint32_t x = o ^ (r.ix >= 0.f ? 0u : far), y = (o + axis) ^ (r.iy >= 0.f ? 0u : far),
						z = (o + 2 * axis) ^ (r.iz >= 0.f ? 0u : far);
				auto u = [nb](uint32_t off) { return *reinterpret_cast<const uint32_t *>(nb + off); };
				const uint32_t wnx = u(x), wfx = u(x ^ far), wny = u(y), wfy = u(y ^ far), wnz = u(z), wfz = u(z ^ far);
				child = u((LAYOUT == 2 ? 64u : 40u) + 4u * c);
				const uint32_t sh = 8u * (c & 3u);
				auto q = [sh](uint32_t w) { return (float)((w >> sh) & 0xffu); };
				const float sx = asf((q0.w & 0xffu) << 23), sy = asf(((q0.w >> 8) & 0xffu) << 23),
						sz = asf(((q0.w >> 16) & 0xffu) << 23);
				const float Ax = sx * r.ix, Ay = sy * r.iy, Az = sz * r.iz;
				const float Bx = fmaf(asf(q0.x), r.ix, r.nx), By = fmaf(asf(q0.y), r.iy, r.ny),
						Bz = fmaf(asf(q0.z), r.iz, r.nz);
				tnx = fmaf(q(wnx), Ax, Bx); tfx = fmaf(q(wfx), Ax, Bx);
				tny = fmaf(q(wny), Ay, By); tfy = fmaf(q(wfy), Ay, By);
				tnz = fmaf(q(wnz), Az, Bz); tfz = fmaf(q(wfz), Az, Bz);
			}
			const float a = fmaxf(fmaxf(fmaxf(tnx, tny), tnz), mint), b = widen(fminf(fminf(fminf(tfx, tfy), tfz), best));
			// (INFINITY is a miss, as in the tests by lane: a hit's key lies below every miss's)
			const bool hit = a <= b && a < INFINITY && child != LRH_CHILD_EMPTY;
			const uint32_t n = (uint32_t)__popc((uint32_t)(__ballot(hit) >> (lane & ~(W - 1u))) & ((1u << W) - 1u));
			if (anyq) {
				float t = hit ? a : INFINITY;
				groupSort<W>(c, t, child);
				drainPush(st, c < n, st.sp + (n - 1u - c), st.sp + n, make_uint2(child, asu(t)), full);
			} else {
				const uint32_t rank = groupRank<W>(key64(hit ? a : INFINITY, child));
				drainPush(st, hit, st.sp + (n - 1u - rank), st.sp + n, make_uint2(child, asu(a)), full);
			}
			if (__ballot(st.sp + n > st.depth)) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");  // spilled entries written by other lanes
			st.sp += n;
			waveFence();
			cur = LRH_CHILD_EMPTY;
			if (n) {
				const uint2 e = drainPop(st, leader);
				waveFence();
				cur = e.x;
				curT = asf(e.y);
			}
		}
		if (!done && cur != LRH_CHILD_EMPTY && (cur & LRH_CHILD_LEAF)) {
			const uint32_t start = cur & LRH_LEAF_START_MASK, cnt = ((cur >> LRH_LEAF_START_BITS) & 7u) + 1u;
			cur = LRH_CHILD_EMPTY;
			if (two && !inInst) {
				const lrh_inst in = v.insts[start];
				if (in.kind == 1u) {
					xfRay(v.xforms + 16 * (size_t)in.index, wo, wd, r);
				} else if (in.kind == 2u) {
					float M[16];
					motionSample(v.motions + in.index, v.segs, v.times, time, M);
					xfRay(M, wo, wd, r);
				}
				obj = in.object;
				inInst = true;
				drainPush(st, leader, st.sp, st.sp + 1u, make_uint2(LRH_SENTINEL, asu(-INFINITY)), full);
				if (st.sp >= st.depth) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
				++st.sp;
				waveFence();
				cur = in.root;
				curT = -INFINITY;
			} else {
				for (uint32_t k = 0; k < cnt && !done; k += W) {
					float t = 0.f, b1 = 0.f, b2 = 0.f;
					uint32_t triIndex = 0, meshIndex = 0;
					const bool ok = k + c < cnt &&
							testTri(v.tris + start + k + c, r, mint, best, t, b1, b2, triIndex, meshIndex);
					const uint64_t oks = __ballot(ok);
					const uint32_t mine = (uint32_t)(oks >> (lane & ~(W - 1u))) & ((1u << W) - 1u);
					if (mine) {
						// the record the sequential test would keep: the nearest, of equal ones
						// the first; an any-hit ray's first
						const float tm = groupMin<W>(ok ? t : INFINITY);
						const uint32_t first = (uint32_t)(__ballot(ok && (anyq || t == tm)) >> (lane & ~(W - 1u))) &
								((1u << W) - 1u);
						const int w = (int)((lane & ~(W - 1u)) + (uint32_t)__ffs((int)first) - 1u);
						best = __shfl(t, w);
						hb1 = __shfl(b1, w);
						hb2 = __shfl(b2, w);
						hTri = (uint32_t)__shfl((int)triIndex, w);
						hMesh = two ? obj : (uint32_t)__shfl((int)meshIndex, w);
						done = anyq;
					}
				}
			}
		}
		if ((steps & 255u) == 255u) {  // (neither in a valid tree; an entry without room has set the error)
			if (leader && steps > kMaxSteps) atomicOr(P.error, 2u);
			done = done || steps > kMaxSteps || overfull(st);
		}
		if (done || (cur == LRH_CHILD_EMPTY && st.sp == 0)) {
			if (leader) {
				lrh_hit_rec *h = v.hits + rid;
				h->t = best;
				h->b1 = hb1;
				h->b2 = hb2;
				h->meshIndex = hMesh;
				h->triangleIndex = hTri;
			}
			rid = kNoRay;
		}
	}
}

template <int LAYOUT, bool TWO, bool ANY, bool COUNT, int BATCH, bool DRAIN>
__device__ __forceinline__ void traceBody(const LrhTraceParams &P) {
	extern __shared__ uint2 ldsStack[];  // [ldsDepth][blockDim] stack; batched: then item starts
	const uint32_t lane = __lane_id();
	Stack st;
	st.lds = ldsStack;
	st.spill = P.spill;
	st.shift = 31u - (uint32_t)__clz((int)blockDim.x);
	st.lane = threadIdx.x;
	st.gstride = P.nLanes;
	st.glane0 = blockIdx.x * blockDim.x;
	st.mask = P.ldsDepth - 1;
	st.depth = P.ldsDepth;
	st.spillDepth = P.spillDepth;
	st.sp = 0;

	uint32_t *itemStart = nullptr;
	if (BATCH) {
		itemStart = reinterpret_cast<uint32_t *>(ldsStack + (size_t)P.ldsDepth * blockDim.x);
		for (uint32_t i = threadIdx.x; i <= P.nItems; i += blockDim.x) itemStart[i] = P.itemStart[i];
	}
	__shared__ TicketPool pool;
	if (threadIdx.x == 0) {
		pool.range = 0;
		pool.fetching = 0;
	}
	__syncthreads();
	// tickets handed out by lane, without a counter: `waveRays` to each wave
	const uint32_t nStatic = gridDim.x * (blockDim.x >> 6) * P.waveRays;

	SceneView v;
	v.nodes = P.nodes;
	v.tris = P.tris;
	v.insts = P.insts;
	v.xforms = P.xforms;
	v.motions = P.motions;
	v.segs = P.segs;
	v.times = P.times;
	v.hits = P.hits;
	v.root = P.root;
	v.flags = (ANY && !BATCH ? LRH_ITEM_ANY : 0u) | (TWO ? LRH_ITEM_TWO : 0u);

	uint32_t rid = kNoRay;  // ray index within its buffer
	LocalRay r;
	float wo[3], wd[3];
	float mint = 0.f, best = 0.f, time = 0.f, hb1 = 0.f, hb2 = 0.f;
	uint32_t hTri = LRH_NULL_INDEX, hMesh = LRH_NULL_INDEX, cur = LRH_CHILD_EMPTY, obj = 0, steps = 0;
	float curT = 0.f;
	bool inInst = false;
	// (a grid of fewer blocks than groups is one group)
	const uint32_t tGroups = gridDim.x < LRH_GROUPS ? 1u : LRH_GROUPS;
	const uint32_t tGroup = blockIdx.x % tGroups, tBlocks = (gridDim.x - tGroup + tGroups - 1u) / tGroups;
	const uint32_t tTotal = groupTickets(tGroup, tGroups, nStatic, P.nRays);
	uint32_t *const tCounter = P.counter + tGroup * LRH_COUNTER_STRIDE;
	bool first = true, exhausted = tTotal == 0;
	// rays a wave hands to the drain (without one it goes on ray by lane)
	constexpr uint32_t kDrainRays = !DRAIN ? 0u : LAYOUT == 2 ? 8u : 16u;
	// COUNT variant only: per lane node tests / primitive tests / rays; per
	// wave passes, live lanes summed over passes, passes with a node test,
	// passes with a leaf test, refills
	uint32_t cNode = 0, cPrim = 0, cRay = 0, cPass = 0, cLive = 0, cNodePass = 0, cLeafPass = 0, cRefill = 0;
	uint32_t cObj = 0, cXf = 0, cMot = 0;  // per lane: object entries, through a matrix, through a motion system


	for (;;) {
		// the ray record a lane takes this pass
		uint4 ldA = make_uint4(0u, 0u, 0u, 0u), ldB = make_uint4(0u, 0u, 0u, 0u);
		uint32_t ldTime = 0u, ldFlags = 0u;
		bool loading = false;
		// ---- refill: idle lanes take tickets when fewer than `refill` lanes are live ----
		uint32_t ticket = P.nRays;  // none
		if (first) {
			first = false;
			if (lane < P.waveRays) ticket = ((st.glane0 + st.lane) >> 6) * P.waveRays + lane;
		} else if (!exhausted) {
			const uint64_t idle = __ballot(rid == kNoRay);
			const uint32_t nIdle = (uint32_t)__popcll(idle);
			if (64u - nIdle < P.refill) {
				if (COUNT) ++cRefill;
				const Tickets tk = takeTickets(pool, tCounter, nIdle, tTotal, tBlocks, (uint32_t)__ffsll((long long)idle) - 1u);
				exhausted = tk.exhausted;
				const uint32_t rank = (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
				if (rid == kNoRay && rank < tk.n0 + tk.n1)
					ticket = rayOf(rank < tk.n0 ? tk.b0 + rank : tk.b1 + (rank - tk.n0), tGroup, tGroups, nStatic);
			}
		}
		if (ticket < P.nRays) {
			uint32_t local = ticket;
			const lrh_ray_rec *rays = P.rays;
			if (BATCH) {
				// item of this ticket: the last item whose start is <= ticket
				uint32_t lo = 0, hi = P.nItems;
				while (hi - lo > 1) {
					const uint32_t mid = (lo + hi) >> 1;
					if (itemStart[mid] <= ticket) lo = mid; else hi = mid;
				}
				const LrhBatchDesc &d = P.items[lo];
				local = ticket - itemStart[lo];
				rays = d.rays;
				v.nodes = d.nodes;
				v.tris = d.tris;
				v.insts = d.insts;
				v.xforms = d.xforms;
				v.motions = d.motions;
				v.segs = d.segs;
				v.times = d.times;
				v.hits = d.hits;
				v.root = d.root;
				v.flags = d.flags & (TWO ? (LRH_ITEM_ANY | LRH_ITEM_TWO) : LRH_ITEM_ANY);
			}
			const uint4 *rp = reinterpret_cast<const uint4 *>(rays + local);
			rid = local;
			ldA = rp[0];
			ldB = rp[1];
			const uint2 c2 = reinterpret_cast<const uint2 *>(rp + 2)[0];
			ldTime = c2.x;
			ldFlags = c2.y;
			loading = true;
			cur = LRH_CHILD_EMPTY;
			st.sp = 0;
		}
		// ---- set up the rays taken this pass ----
		if (loading) {
			loading = false;
			if (ldFlags & 1u) {  // RAY_FLAGS_MASKED: skipped, hit record untouched
				rid = kNoRay;
			} else {
				r.ox = asf(ldA.x); r.oy = asf(ldA.y); r.oz = asf(ldA.z);
				r.dx = asf(ldA.w); r.dy = asf(ldB.x); r.dz = asf(ldB.y);
				if (TWO) {
					wo[0] = r.ox; wo[1] = r.oy; wo[2] = r.oz;
					wd[0] = r.dx; wd[1] = r.dy; wd[2] = r.dz;
				}
				mint = asf(ldB.z);
				best = asf(ldB.w);
				time = asf(ldTime);
				setupRay(r);
				hb1 = 0.f; hb2 = 0.f;
				hTri = LRH_NULL_INDEX; hMesh = LRH_NULL_INDEX;
				// a NaN origin or direction component makes every triangle test
				// fail (the divisor or the distance is NaN), while every box
				// would be entered: the ray misses without a traversal
				const bool nanRay = isnan(r.ox) || isnan(r.oy) || isnan(r.oz) || isnan(r.dx) || isnan(r.dy) ||
						isnan(r.dz);
				cur = nanRay ? LRH_CHILD_EMPTY : v.root;
				curT = -INFINITY;
				inInst = false;
				steps = 0;
				if (COUNT) ++cRay;
			}
		}
		const uint64_t liveNow = __ballot(rid != kNoRay);
		if (!liveNow) {
			if (exhausted) break;
			continue;
		}
		if constexpr (DRAIN) {
			if (exhausted && (uint32_t)__popcll(liveNow) <= kDrainRays) {
				drain<LAYOUT, TWO, ANY, BATCH>(P, st, v, r, wo, wd, mint, best, time, hb1, hb2, hTri, hMesh, cur, curT, obj,
						inInst, rid);
				break;
			}
		}
		// passes until fewer than `refill` lanes are live (after the last
		// ticket: until the drain takes the rest)
		const uint32_t minLive = exhausted ? kDrainRays + 1u : P.refill;
		do {
		if (COUNT) {
			++cPass;
			cLive += (uint32_t)__popcll(__ballot(rid != kNoRay));
		}

		// ---- node phase: one node test per lane and pass ----
		bool done = false, tested = false;
		if (rid != kNoRay) {
			for (uint32_t pops = 0;;) {
				if (cur == LRH_CHILD_EMPTY) {
					if (st.sp == 0 || pops++ == kMaxPops) break;
					const uint2 e = pop(st);
					cur = e.x;
					curT = asf(e.y);
					if (TWO && cur == LRH_SENTINEL) {
						// leaving an object's tree: back to the world-space ray
						r.ox = wo[0]; r.oy = wo[1]; r.oz = wo[2];
						r.dx = wd[0]; r.dy = wd[1]; r.dz = wd[2];
						setupRay(r);
						inInst = false;
						cur = LRH_CHILD_EMPTY;
					} else if (!(curT <= widen(best))) {
						cur = LRH_CHILD_EMPTY;  // entry not before the current hit
					}
					if (cur == LRH_CHILD_EMPTY) continue;
				}
				if (cur & LRH_CHILD_LEAF) break;
				if (++steps > kMaxSteps) {
					atomicOr(P.error, 2u);
					done = true;
					break;
				}
				if (COUNT) {
					++cNode;
					tested = true;
				}
				if (LAYOUT == 2) {
					float t8[8];
					uint32_t c8[8];
					testNode8Q(reinterpret_cast<const lrh_node8q *>(v.nodes), cur, r, mint, best, t8, c8);
					// an any-hit ray reports the first blocker it meets: its order is kept to the
					// network's.  In a batch of both kinds each ray takes its own sort: 899 us for
					// 3.9M rays, where one network whose comparators also compare a closest ray's
					// references takes 944 (and the network alone, with no order of ties, 889).
					if (ANY && (BATCH != LRH_BATCH_MIXED || (v.flags & LRH_ITEM_ANY))) sort8(t8, c8);
					else sort8Closest(t8, c8);
					bool ok = true;
					// sorted: the lanes that push entry k also push k-1..1; a
					// position no lane of the wave reaches is skipped as a whole
#pragma unroll
					for (int k = 7; k >= 1; --k)
						if (__ballot(t8[k] != INFINITY))
							if (t8[k] != INFINITY) ok = ok && push(st, c8[k], t8[k], P.error);
					if (t8[0] != INFINITY) {
						cur = c8[0];
						curT = t8[0];
					} else
						cur = LRH_CHILD_EMPTY;
					if (!ok) done = true;
					break;
				}
				float t4[4];
				uint32_t c4[4];
				if (LAYOUT == 0)
					testNodeQ(reinterpret_cast<const lrh_node4q *>(v.nodes), cur, r, mint, best, t4, c4);
				else
					testNodeF(reinterpret_cast<const lrh_node4f *>(v.nodes), cur, r, mint, best, t4, c4);
				if (ANY && (BATCH != LRH_BATCH_MIXED || (v.flags & LRH_ITEM_ANY))) sort4(t4, c4);
				else sort4Closest(t4, c4);
				bool ok = true;
				if (t4[3] != INFINITY) ok = ok && push(st, c4[3], t4[3], P.error);
				if (t4[2] != INFINITY) ok = ok && push(st, c4[2], t4[2], P.error);
				if (t4[1] != INFINITY) ok = ok && push(st, c4[1], t4[1], P.error);
				if (t4[0] != INFINITY) {
					cur = c4[0];
					curT = t4[0];
				} else
					cur = LRH_CHILD_EMPTY;
				if (!ok) done = true;
				break;
			}
		}

		// ---- leaf phase ----
		const bool atLeaf = rid != kNoRay && !done && cur != LRH_CHILD_EMPTY &&
				(cur & LRH_CHILD_LEAF);
		if (COUNT) {
			cNodePass += __ballot(tested) ? 1u : 0u;
			cLeafPass += __ballot(atLeaf) ? 1u : 0u;
		}
		if (atLeaf) {
			const bool two = TWO && (v.flags & LRH_ITEM_TWO);
			const bool anyq = ANY && (BATCH == LRH_BATCH || (v.flags & LRH_ITEM_ANY));
			const uint32_t start = cur & LRH_LEAF_START_MASK;
			uint32_t cnt = ((cur >> LRH_LEAF_START_BITS) & 7u) + 1u;
			cur = LRH_CHILD_EMPTY;
			if (!two && cnt > P.leafTris) {
				// test leafTris triangles now and keep the rest of the leaf for
				// the next pass: a wave then never loops over the longest leaf
				// of its lanes while the others wait
				cur = LRH_CHILD_LEAF | ((cnt - P.leafTris - 1u) << LRH_LEAF_START_BITS) | (start + P.leafTris);
				cnt = P.leafTris;
			}
			if (COUNT) cPrim += cnt;
			if (two && !inInst) {
				// root leaf: enter the object's tree in its local space
				const lrh_inst in = v.insts[start];
				if (COUNT) {
					++cObj;
					cXf += in.kind == 1u ? 1u : 0u;
					cMot += in.kind == 2u ? 1u : 0u;
				}
				if (in.kind == 1u) {
					xfRay(v.xforms + 16 * (size_t)in.index, wo, wd, r);
				} else if (in.kind == 2u) {
					float M[16];
					motionSample(v.motions + in.index, v.segs, v.times, time, M);
					xfRay(M, wo, wd, r);
				}
				obj = in.object;
				inInst = true;
				if (push(st, LRH_SENTINEL, -INFINITY, P.error)) {
					cur = in.root;
					curT = -INFINITY;
				} else
					done = true;
			} else {
				for (uint32_t k = 0; k < cnt; ++k) {
					float t, b1, b2;
					uint32_t triIndex, meshIndex;
					if (testTri(v.tris + start + k, r, mint, best, t, b1, b2, triIndex, meshIndex)) {
						best = t;
						hb1 = b1;
						hb2 = b2;
						hTri = triIndex;
						hMesh = two ? obj : meshIndex;
						if (anyq) {
							done = true;
							break;
						}
					}
				}
			}
		}
		if (rid != kNoRay && (done || (cur == LRH_CHILD_EMPTY && st.sp == 0))) {
			lrh_hit_rec *h = v.hits + rid;
			h->t = best;
			h->b1 = hb1;
			h->b2 = hb2;
			h->meshIndex = hMesh;
			h->triangleIndex = hTri;
			rid = kNoRay;
			cur = LRH_CHILD_EMPTY;
		}
		} while ((uint32_t)__popcll(__ballot(rid != kNoRay)) >= minLive);
	}
	if (COUNT) {
		unsigned long long a = cNode, b = cPrim, c = cRay, e = cObj, f = cXf, g = cMot;
		for (int o = 32; o > 0; o >>= 1) {
			a += __shfl_xor(a, o);
			b += __shfl_xor(b, o);
			c += __shfl_xor(c, o);
			e += __shfl_xor(e, o);
			f += __shfl_xor(f, o);
			g += __shfl_xor(g, o);
		}
		if (lane == 0) {
			// wave counters are uniform: lane 0 adds them once per wave
			atomicAdd(P.stats + 0, a);
			atomicAdd(P.stats + 1, b);
			atomicAdd(P.stats + 2, c);
			atomicAdd(P.stats + 3, (unsigned long long)cPass);
			atomicAdd(P.stats + 4, (unsigned long long)cLive);
			atomicAdd(P.stats + 5, (unsigned long long)cNodePass);
			atomicAdd(P.stats + 6, (unsigned long long)cLeafPass);
			atomicAdd(P.stats + 7, (unsigned long long)cRefill);
			if (TWO) {
				atomicAdd(P.stats + 8, e);
				atomicAdd(P.stats + 9, f);
				atomicAdd(P.stats + 10, g);
			}
		}
	}
	// the last block of a group to finish rewinds its counters for the next
	// launch (a group that never used them has nothing to rewind; every block's
	// own additions have returned before its barrier)
	if (tTotal == 0) return;
	__syncthreads();
	if (threadIdx.x == 0) {
		uint32_t *done = tCounter + LRH_GROUPS * LRH_COUNTER_STRIDE;
		if (atomicAdd(done, 1u) == tBlocks - 1u) {
			atomicExch(tCounter, 0u);
			atomicExch(done, 0u);
		}
	}
}

// Single-level traces are built for 7 waves per SIMD (at most 72 VGPRs),
// batched ones over 8-wide nodes (per-lane item view) for 5: at 6 the loop
// spills (a batch of 3.9M rays 1,032 us, at 5 983 us).
template <int LAYOUT, bool ANY, bool COUNT, int BATCH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(7))) void lrh_trace_kernel(LrhTraceParams P) {
	traceBody<LAYOUT, false, ANY, COUNT, BATCH, !COUNT>(P);
}

template <bool ANY, int BATCH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void lrh_trace8b_kernel(LrhTraceParams P) {
	traceBody<2, false, ANY, false, BATCH, true>(P);
}

// Two-level traces inline the motion sample, which reads its motion record
// and the hot part of its segment with all loads in flight at once.  Over
// 64-byte nodes they are built for 6 waves per SIMD (80 VGPRs, 8 spilled: 3%
// faster than 5 and 90 on moving instances), over 8-wide nodes for 5 (94
// VGPRs; at 6 it spills 10), batched 8-wide ones for 4 (at 5 it spills 37).
// With the drain, which holds a second motion sample, the loop spills; so
// a launch that the drain is a small part of goes without.
template <int LAYOUT, bool ANY, bool COUNT, int BATCH>
__global__ __launch_bounds__(256) void lrh_trace2_kernel(LrhTraceParams P) {
	traceBody<LAYOUT, true, ANY, COUNT, BATCH, false>(P);
}

template <bool ANY, int BATCH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(BATCH ? 4 : 5))) void lrh_trace28_kernel(
		LrhTraceParams P) {
	traceBody<2, true, ANY, false, BATCH, false>(P);
}

template <bool ANY>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void lrh_trace2q_kernel(LrhTraceParams P) {
	traceBody<0, true, ANY, false, 0, false>(P);
}

template <int LAYOUT, bool ANY>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void lrh_trace2_drain_kernel(LrhTraceParams P) {
	traceBody<LAYOUT, true, ANY, false, 0, true>(P);
}

__global__ void lrh_reset_kernel(uint32_t *p, uint32_t n) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n) p[i] = 0u;
}

// ---------------------------------------------------------------------------
// host-side launch table
// ---------------------------------------------------------------------------
typedef void (*KernelFn)(LrhTraceParams);

template <int L, bool A, int B>
static const void *batchKernelOf(bool two) {
	if (L == 2)
		return two ? (const void *)&lrh_trace28_kernel<A, B> : (const void *)&lrh_trace8b_kernel<A, B>;
	return two ? (const void *)&lrh_trace2_kernel<L == 2 ? 0 : L, A, false, B>
			: (const void *)&lrh_trace_kernel<L == 2 ? 0 : L, A, false, B>;
}

template <int L, bool A>
static const void *kernelOf(bool two, bool count, int batch, bool drain) {
	if (batch == LRH_BATCH_MIXED) return batchKernelOf<L, true, LRH_BATCH_MIXED>(two);
	if (batch) return batchKernelOf<L, A, LRH_BATCH>(two);
	if (!two) return count ? (const void *)&lrh_trace_kernel<L, A, true, 0> : (const void *)&lrh_trace_kernel<L, A, false, 0>;
	if (count) return (const void *)&lrh_trace2_kernel<L, A, true, 0>;
	if (drain) return (const void *)&lrh_trace2_drain_kernel<L, A>;
	if (L == 0) return (const void *)&lrh_trace2q_kernel<A>;
	if (L == 2) return (const void *)&lrh_trace28_kernel<A, 0>;
	return (const void *)&lrh_trace2_kernel<1, A, false, 0>;
}

// The counting variants are not offered for batches and have no drain.
static const void *kernelPtr(int layout, bool two, bool any, bool count, int batch, bool drain) {
	switch (layout * 2 + (any ? 1 : 0)) {
	case 0: return kernelOf<0, false>(two, count, batch, drain);
	case 1: return kernelOf<0, true>(two, count, batch, drain);
	case 2: return kernelOf<1, false>(two, count, batch, drain);
	case 3: return kernelOf<1, true>(two, count, batch, drain);
	case 4: return kernelOf<2, false>(two, count, batch, drain);
	case 5: return kernelOf<2, true>(two, count, batch, drain);
	default: return nullptr;
	}
}

hipError_t lrhLaunchReset(uint32_t *p, uint32_t n, hipStream_t s) {
	hipLaunchKernelGGL(lrh_reset_kernel, dim3((n + 63) / 64), dim3(64), 0, s, p, n);
	return hipGetLastError();
}

hipError_t lrhOccupancy(int layout, bool two, bool any, int batch, bool drain, int block, size_t lds,
		int *blocksPerCU) {
	const void *k = kernelPtr(layout, two, any, false, batch, drain);
	if (!k) return hipErrorInvalidDeviceFunction;
	return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocksPerCU, k, block, lds);
}

hipError_t lrhLaunchTrace(int layout, bool two, bool any, bool count, int batch, bool drain, dim3 grid, dim3 block,
		size_t lds, hipStream_t s, const LrhTraceParams &P) {
	void *args[] = {(void *)&P};
	const void *k = kernelPtr(layout, two, any, count, batch, drain);
	if (!k) return hipErrorInvalidDeviceFunction;
	return hipLaunchKernel(k, grid, block, args, lds, s);
}
