/*
 * Device helpers shared by the device-side tree code (the linear BVH build
 * and the two-level root refit): boxes, MachineEpsilon, ordered float keys
 * for atomic min/max, and the 4-wide node writers with the host builder's
 * outward-rounded quantization (lrh_build.cpp quantize / toFloatNode).
 */
#ifndef LRH_DEVNODE_H
#define LRH_DEVNODE_H

#include <stdint.h>

#include <cmath>
#include <cstring>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define LRH_DN __host__ __device__
#else
#define LRH_DN
#endif

#include "lrh_layout.h"

namespace lrhdev {

// float <-> bits on either side (the host build is the CPU emulation of the
// device tree code)
LRH_DN inline uint32_t bitsOf(float f) {
#if defined(__HIP_DEVICE_COMPILE__)
	return __float_as_uint(f);
#else
	uint32_t u;
	std::memcpy(&u, &f, 4);
	return u;
#endif
}
LRH_DN inline float fromBits(uint32_t u) {
#if defined(__HIP_DEVICE_COMPILE__)
	return __uint_as_float(u);
#else
	float f;
	std::memcpy(&f, &u, 4);
	return f;
#endif
}

struct GBox {
	float lo[3], hi[3];
};

LRH_DN inline float minT(float a, float b) { return a < b ? a : b; }  // utils.h Min
LRH_DN inline float maxT(float a, float b) { return a > b ? a : b; }  // utils.h Max

// MachineEpsilon::E (include/luxrays/core/epsilon.h:50-94)
LRH_DN inline float machineEps(float v) {
	const float n = fromBits(bitsOf(v) + 0x80u);
	const float e = fabsf(n - v);
	return e > 1e-5f ? (e < 1e-1f ? e : 1e-1f) : 1e-5f;
}

// ordered keys so unsigned min/max order floats
LRH_DN inline uint32_t fkey(float f) {
	const uint32_t u = bitsOf(f);
	return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
LRH_DN inline float unkey(uint32_t k) {
	return fromBits((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

LRH_DN inline float expScale(uint32_t e) { return fromBits(e << 23); }
LRH_DN inline float decodeQ(float org, uint32_t q, float s) { return org + (float)q * s; }

// exponent byte of one axis of a quantized node over [o, hi]: the smallest
// power of two whose 255 steps from o reach hi
LRH_DN inline int axisExp(float o, float hi) {
	const float ext = hi - o;
	int e2 = -126;
	if (ext > 0.f) frexpf(ext / 255.f, &e2);
	int e = e2 + 127;
	if (e < 1) e = 1;
	while (e < 254 && decodeQ(o, 255, expScale((uint32_t)e)) < hi) ++e;
	return e;
}

// a child's bounds on one axis as steps of s from o, rounded outward (the
// rule of the host builder's quantize)
LRH_DN inline uint8_t axisLo(float lo, float o, float s) {
	long q = (long)floorf((lo - o) / s);
	if (q < 0) q = 0;
	if (q > 255) q = 255;
	while (q > 0 && decodeQ(o, (uint32_t)q, s) > lo) --q;
	return (uint8_t)q;
}
LRH_DN inline uint8_t axisHi(float hi, float o, float s) {
	long q = (long)ceilf((hi - o) / s);
	if (q < 0) q = 0;
	if (q > 255) q = 255;
	while (q < 255 && decodeQ(o, (uint32_t)q, s) < hi) ++q;
	return (uint8_t)q;
}

// W-wide quantized node (lrh_node4q, lrh_node8q): the host builder's
// outward rounding
template <int W, class Node>
LRH_DN inline void quantizeNodeW(const GBox *cb, int n, const uint32_t *child, Node *out) {
	Node q;
	GBox pb;
	for (int k = 0; k < 3; ++k) {
		pb.lo[k] = INFINITY;
		pb.hi[k] = -INFINITY;
	}
	for (int c = 0; c < n; ++c)
		for (int k = 0; k < 3; ++k) {
			pb.lo[k] = minT(pb.lo[k], cb[c].lo[k]);
			pb.hi[k] = maxT(pb.hi[k], cb[c].hi[k]);
		}
	uint8_t *qlo[3] = {q.qlo_x, q.qlo_y, q.qlo_z};
	uint8_t *qhi[3] = {q.qhi_x, q.qhi_y, q.qhi_z};
	uint8_t *ex[3] = {&q.ex, &q.ey, &q.ez};
	for (int k = 0; k < 3; ++k) {
		const float o = pb.lo[k];
		q.org[k] = o;
		const int e = axisExp(o, pb.hi[k]);
		const float s = expScale((uint32_t)e);
		*ex[k] = (uint8_t)e;
		for (int c = 0; c < W; ++c) {
			// empty slot: inverted box
			qlo[k][c] = c < n ? axisLo(cb[c].lo[k], o, s) : 255;
			qhi[k][c] = c < n ? axisHi(cb[c].hi[k], o, s) : 0;
		}
	}
	q.nchild = (uint8_t)n;
	for (int c = 0; c < W; ++c) q.child[c] = child[c];
	for (auto &x : q.pad) x = 0;
	*out = q;
}

LRH_DN inline void quantizeNode(const GBox *cb, int n, const uint32_t child[4], lrh_node4q *out) {
	quantizeNodeW<4>(cb, n, child, out);
}

LRH_DN inline void quantizeNode8(const GBox *cb, int n, const uint32_t child[8], lrh_node8q *out) {
	quantizeNodeW<8>(cb, n, child, out);
}

LRH_DN inline void floatNode(const GBox *cb, int n, const uint32_t child[4], lrh_node4f *out) {
	lrh_node4f f;
	for (int c = 0; c < 4; ++c) {
		const bool v = c < n;
		f.lo_x[c] = v ? cb[c].lo[0] : INFINITY;
		f.lo_y[c] = v ? cb[c].lo[1] : INFINITY;
		f.lo_z[c] = v ? cb[c].lo[2] : INFINITY;
		f.hi_x[c] = v ? cb[c].hi[0] : -INFINITY;
		f.hi_y[c] = v ? cb[c].hi[1] : -INFINITY;
		f.hi_z[c] = v ? cb[c].hi[2] : -INFINITY;
		f.child[c] = child[c];
		f.pad[c] = 0;
	}
	*out = f;
}

#if defined(__HIPCC__)
// Union of the boxes of the first n of W neighbouring lanes (lane c, 0..W-1,
// with box c), to all of them: the sequential writers' fold by minT and maxT.
// Min and max of numbers are exact in any order; a NaN (a triangle of NaN
// vertices) hides the boxes before it from the fold and is kept only from
// the last place, and zeros of either sign are equal, so a wave that holds
// one takes the boxes in order.
template <int W>
__device__ inline GBox unionLanes(const GBox &b, int c, int n) {
	bool inOrder = false;
	for (int k = 0; k < 3; ++k) inOrder |= c < n && !(fabsf(b.lo[k]) > 0.f && fabsf(b.hi[k]) > 0.f);
	GBox u;
	if (__ballot(inOrder)) {
		for (int k = 0; k < 3; ++k) {
			u.lo[k] = INFINITY;
			u.hi[k] = -INFINITY;
			for (int j = 0; j < W; ++j) {
				const float lo = __shfl(b.lo[k], j, W), hi = __shfl(b.hi[k], j, W);
				u.lo[k] = j < n ? minT(u.lo[k], lo) : u.lo[k];
				u.hi[k] = j < n ? maxT(u.hi[k], hi) : u.hi[k];
			}
		}
		return u;
	}
	for (int k = 0; k < 3; ++k) {
		u.lo[k] = c < n ? b.lo[k] : INFINITY;
		u.hi[k] = c < n ? b.hi[k] : -INFINITY;
		for (int o = W / 2; o > 0; o >>= 1) {
			u.lo[k] = fminf(__shfl_xor(u.lo[k], o), u.lo[k]);
			u.hi[k] = fmaxf(__shfl_xor(u.hi[k], o), u.hi[k]);
		}
	}
	return u;
}

// The same node written by W neighbouring lanes of a wave, lane c (0..W-1)
// with child c: one lane per child instead of one thread per node, whose
// children's roundings (a division and a few compares each, six per child)
// would run one after another.  All W lanes call it together; lane c < n has
// the child's box and reference, the others pass any box and
// LRH_CHILD_EMPTY.  Returns the union of the boxes to all of them.
template <int W, class Node>
__device__ inline GBox quantizeNodeLanes(const GBox &b, int c, int n, uint32_t child, Node *out) {
	const GBox u = unionLanes<W>(b, c, n);
	uint8_t *const qlo[3] = {out->qlo_x, out->qlo_y, out->qlo_z};
	uint8_t *const qhi[3] = {out->qhi_x, out->qhi_y, out->qhi_z};
	for (int k = 0; k < 3; ++k) {
		const float o = u.lo[k];
		const int e = axisExp(o, u.hi[k]);
		const float s = expScale((uint32_t)e);
		qlo[k][c] = c < n ? axisLo(b.lo[k], o, s) : 255;
		qhi[k][c] = c < n ? axisHi(b.hi[k], o, s) : 0;
		if (c == 0) {
			out->org[k] = o;
			(&out->ex)[k] = (uint8_t)e;
		}
	}
	out->child[c] = child;
	constexpr int kPads = (int)(sizeof(out->pad) / 4);
	if (c < kPads) out->pad[c] = 0;
	if (c == 0) out->nchild = (uint8_t)n;
	return u;
}

// the fp32 node (lrh_node4f) by four lanes, likewise
__device__ inline GBox floatNodeLanes(const GBox &b, int c, int n, uint32_t child, lrh_node4f *out) {
	const bool some = c < n;
	out->lo_x[c] = some ? b.lo[0] : INFINITY; out->lo_y[c] = some ? b.lo[1] : INFINITY; out->lo_z[c] = some ? b.lo[2] : INFINITY;
	out->hi_x[c] = some ? b.hi[0] : -INFINITY; out->hi_y[c] = some ? b.hi[1] : -INFINITY; out->hi_z[c] = some ? b.hi[2] : -INFINITY;
	out->child[c] = child;
	out->pad[c] = 0;
	return unionLanes<4>(b, c, n);
}
#endif

}  // namespace lrhdev

#endif
