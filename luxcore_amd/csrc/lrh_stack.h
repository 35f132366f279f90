/*
 * The traversal stack of a ray: its top `depth` entries live in a ring in LDS
 * (one column per lane), deeper ones in a spill array in memory, `spillDepth`
 * to a lane.  While a lane has its ray to itself it pushes and pops one entry
 * at a time; in the drain a group of lanes shares a ray and pushes a node's
 * children at once, a lane each, into the column the ray has had so far.
 * Nothing is written or read outside the two arrays.  A single push is
 * refused where it would pass `depth + spillDepth`; a shared one leaves out
 * what has no room, and pops then repeat entries until the ray is ended for
 * being overfull. (Also compiled for the host, where
 * a test holds it against a plain stack.)
 */
#ifndef LRH_STACK_H
#define LRH_STACK_H

#include <stddef.h>
#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define LRH_ST __device__ __forceinline__
#else
#define LRH_ST inline
#endif

namespace lrhstack {

// Entry: two 32-bit words (uint2)
template <class Entry>
struct Stack {
	Entry *lds;
	Entry *spill;
	uint32_t shift;     // log2 of blockDim
	uint32_t lane;      // threadIdx / global lane
	uint32_t gstride;
	uint32_t glane0;    // of thread 0: the spill column is glane0 + lane
	uint32_t mask;      // ldsDepth - 1
	uint32_t depth;     // ldsDepth
	uint32_t spillDepth;
	uint32_t sp;
};

template <class Entry>
LRH_ST Entry &ringAt(const Stack<Entry> &s, uint32_t place) {
	return s.lds[((place & s.mask) << s.shift) + s.lane];
}

template <class Entry>
LRH_ST Entry &spillAt(const Stack<Entry> &s, uint32_t k) {
	return s.spill[(size_t)k * s.gstride + s.glane0 + s.lane];
}

// more entries than the arrays hold
template <class Entry>
LRH_ST bool overfull(const Stack<Entry> &s) {
	return s.sp > s.depth + s.spillDepth;
}

// false, after full(), where there is no room
template <class Entry, class Full>
LRH_ST bool push(Stack<Entry> &s, const Entry &v, const Full &full) {
	Entry *e = &ringAt(s, s.sp);
	if (s.sp >= s.depth) {
		const uint32_t k = s.sp - s.depth;
		if (k >= s.spillDepth) {
			full();
			return false;
		}
		spillAt(s, k) = *e;
	}
	*e = v;
	++s.sp;
	return true;
}

template <class Entry>
LRH_ST Entry pop(Stack<Entry> &s) {
	--s.sp;
	Entry *e = &ringAt(s, s.sp);
	const Entry v = *e;
	if (s.sp >= s.depth) *e = spillAt(s, s.sp - s.depth);
	return v;
}

// A lane's part of a shared push, if it has one: its entry to place `i` of the
// ray's stack (places sp .. top - 1, one lane each).  The ring ends up with
// the top `depth` places; what they displace and what lies below them goes to
// the spill array, or nowhere, after full(), beyond it.  sp is the caller's to
// advance.
template <class Entry, class Full>
LRH_ST void drainPush(const Stack<Entry> &s, bool has, uint32_t i, uint32_t top, const Entry &v, const Full &full) {
	if (!has) return;
	if (i + s.depth < top) {
		if (i < s.spillDepth) spillAt(s, i) = v;
		else full();
		return;
	}
	Entry *e = &ringAt(s, i);
	int old = (int)i - (int)s.depth;  // the place this ring slot holds: below sp
	if (old >= (int)s.sp) old -= (int)s.depth;
	if (old >= 0) {
		if ((uint32_t)old < s.spillDepth) spillAt(s, (uint32_t)old) = *e;
		else full();
	}
	*e = v;
}

// pops the top entry, for all lanes of the group (the leader refills the ring)
template <class Entry>
LRH_ST Entry drainPop(Stack<Entry> &s, bool leader) {
	--s.sp;
	Entry *e = &ringAt(s, s.sp);
	const Entry v = *e;
	const uint32_t k = s.sp - s.depth;  // (wraps, and is skipped, while all entries are in the ring)
	if (k < s.spillDepth && leader) *e = spillAt(s, k);
	return v;
}

}  // namespace lrhstack

#endif
