/*
 * Ray generation on either side of a trace, for the served path-tracing
 * sessions: pinhole camera rays, and from a wavefront's hits the next
 * cosine-weighted bounce (with Russian roulette) plus one shadow ray toward a
 * 1x1 area light.  They play the part of SLG's AdvancePaths micro-kernels that
 * generate the camera and next-vertex rays
 * (include/slg/engines/pathoclbase/kernels/pathoclbase_kernels_micro.cl:
 * 723-844, 1045-1075), reduced to what a synthetic session needs.
 *
 * The shading step (lrh_shade, and lrh_shade_batch for several wavefronts in
 * one launch) consumes hits as SLG's hit-consumption and direct-light
 * micro-kernels do, reduced to Lambertian surfaces and triangle lights.
 *
 * Terminated paths become masked rays (RAY_FLAGS_MASKED), so a wavefront
 * keeps its size and the tracer skips them; a path that ended before the
 * previous step is not touched again (its slots are masked already).
 * Random numbers are a hash of
 * (session seed, pixel, bounce, dimension): a session's rays do not depend on
 * what else is in flight.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lrh_layout.h"
#include "lrh_paths.h"

namespace {

__device__ __forceinline__ uint32_t pcg(uint32_t v) {
	const uint32_t s = v * 747796405u + 2891336453u;
	const uint32_t w = ((s >> ((s >> 28u) + 4u)) ^ s) * 277803737u;
	return (w >> 22u) ^ w;
}

__device__ __forceinline__ float rnd(uint64_t seed, uint32_t pixel, uint32_t bounce, uint32_t dim) {
	const uint32_t h = pcg((uint32_t)seed ^ pcg((uint32_t)(seed >> 32) ^ pcg(pixel ^ pcg(bounce * 16u + dim))));
	return (float)(h >> 8) * (1.0f / 16777216.0f);
}

// MachineEpsilon::E of a point (include/luxrays/core/epsilon.h:50-94)
__device__ __forceinline__ float epsE(float v) {
	const float n = __uint_as_float(__float_as_uint(v) + 0x80u);
	const float e = fabsf(n - v);
	return e > 1e-5f ? (e < 1e-1f ? e : 1e-1f) : 1e-5f;
}

__device__ __forceinline__ void writeMasked(lrh_ray_rec *r) {
	r->ox = r->oy = r->oz = 0.f;
	r->dx = 0.f; r->dy = 0.f; r->dz = 1.f;
	r->mint = 0.f; r->maxt = 0.f; r->time = 0.f;
	r->flags = 1u;
	r->pad[0] = r->pad[1] = 0.f;
}

// The 48-byte records of a wave's lanes (those in `mask`) to consecutive
// places, through the wave's 3 KiB of LDS: stored by their own lanes, each of
// the three store instructions of a record wrote a third of 24 lines, here
// eight whole lines (the three steps of 921,600 paths: 242 us, 196 with
// this, 179 with the loads of a step issued together as well; their bytes at
// the rate of a large copy: 174).  Called by the whole wave.
struct __attribute__((aligned(4))) Quarter {  // (a caller's records are aligned to their floats)
	uint32_t w[4];
};
template <class Rec>
__device__ __forceinline__ void storeRecords(uint4 *lds, Rec *dst, const Rec &r, uint64_t mask) {
	static_assert(sizeof(Rec) == 48, "three 16-byte parts");
	const uint32_t lane = threadIdx.x & 63u;
	uint32_t w[12];
	__builtin_memcpy(w, &r, 48);
	for (int k = 0; k < 3; ++k) lds[3 * lane + k] = make_uint4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
	__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
	__builtin_amdgcn_wave_barrier();
	for (uint32_t k = 0; k < 3; ++k) {
		const uint32_t c = k * 64 + lane;
		const uint4 v = lds[c];
		if ((mask >> (c / 3)) & 1ull) reinterpret_cast<Quarter *>(dst)[c] = Quarter{{v.x, v.y, v.z, v.w}};
	}
	__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
	__builtin_amdgcn_wave_barrier();
}

__global__ __launch_bounds__(256) void lrh_camera_kernel(LrhCameraParams C, lrh_ray_rec *rays) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	const uint32_t n = C.width * C.height;
	const uint32_t x = i % C.width, y = i / C.width;
	const float px = ((float)x + 0.5f) / (float)C.width * 2.f - 1.f;
	const float py = 1.f - ((float)y + 0.5f) / (float)C.height * 2.f;
	float d[3];
	for (int k = 0; k < 3; ++k) d[k] = C.fwd[k] + px * C.tw * C.right[k] + py * C.th * C.up[k];
	const float inv = 1.f / sqrtf(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
	lrh_ray_rec r;
	r.ox = C.eye[0]; r.oy = C.eye[1]; r.oz = C.eye[2];
	r.dx = d[0] * inv; r.dy = d[1] * inv; r.dz = d[2] * inv;
	r.mint = C.mint;
	r.maxt = INFINITY;
	r.time = 0.f;
	r.flags = 0u;
	r.pad[0] = r.pad[1] = 0.f;
	__shared__ uint4 stage[4][192];
	storeRecords(stage[threadIdx.x >> 6], rays + (i - (threadIdx.x & 63u)), r, __ballot(i < n));
}

// one bounce of ray i; returns the number of live rays it wrote (0..2)
__device__ uint32_t bounceOne(const LrhBounceParams &P, uint32_t i) {
	const lrh_ray_rec ray = P.rays[i];
	const lrh_hit_rec hit = P.hits[i];
	uint32_t live = 0;
	lrh_ray_rec *next = P.next + i;
	lrh_ray_rec *shadow = P.shadow ? P.shadow + i : nullptr;
	if ((ray.flags & 1u) || hit.meshIndex >= P.nMeshes ||
			hit.triangleIndex >= P.meshTriBase[hit.meshIndex + 1] - P.meshTriBase[hit.meshIndex]) {
		writeMasked(next);
		if (shadow) writeMasked(shadow);
		return 0;
	}
	const uint32_t rec = P.invPerm[P.meshTriBase[hit.meshIndex] + hit.triangleIndex];
	const lrh_tri tr = P.tris[rec];
	// geometric normal, facing the incoming ray
	float n[3] = {tr.e1[1] * tr.e2[2] - tr.e1[2] * tr.e2[1], tr.e1[2] * tr.e2[0] - tr.e1[0] * tr.e2[2],
			tr.e1[0] * tr.e2[1] - tr.e1[1] * tr.e2[0]};
	const float nl = sqrtf(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
	const float s = (n[0] * ray.dx + n[1] * ray.dy + n[2] * ray.dz > 0.f ? -1.f : 1.f) / fmaxf(nl, 1e-30f);
	for (int k = 0; k < 3; ++k) n[k] *= s;
	const float p[3] = {ray.ox + ray.dx * hit.t, ray.oy + ray.dy * hit.t, ray.oz + ray.dz * hit.t};
	const float eps = fmaxf(epsE(p[0]), fmaxf(epsE(p[1]), epsE(p[2])));
	const uint32_t pix = P.pixelBase + i;
	// Russian roulette from bounce rrStart on
	const bool alive = P.bounce < P.rrStart || rnd(P.seed, pix, P.bounce, 2) < P.rrSurvive;
	if (alive) {
		// cosine-weighted direction around n (Malley), branchless basis (Duff et al. 2017)
		const float u1 = rnd(P.seed, pix, P.bounce, 0), u2 = rnd(P.seed, pix, P.bounce, 1);
		const float r = sqrtf(u1), phi = 6.2831853f * u2;
		const float lx = r * cosf(phi), ly = r * sinf(phi), lz = sqrtf(fmaxf(0.f, 1.f - u1));
		const float sg = n[2] >= 0.f ? 1.f : -1.f;
		const float a = -1.f / (sg + n[2]);
		const float b = n[0] * n[1] * a;
		const float t0[3] = {1.f + sg * n[0] * n[0] * a, sg * b, -sg * n[0]};
		const float t1[3] = {b, sg + n[1] * n[1] * a, -n[1]};
		float d[3];
		for (int k = 0; k < 3; ++k) d[k] = lx * t0[k] + ly * t1[k] + lz * n[k];
		const float dl = 1.f / sqrtf(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
		lrh_ray_rec o;
		o.ox = p[0]; o.oy = p[1]; o.oz = p[2];
		o.dx = d[0] * dl; o.dy = d[1] * dl; o.dz = d[2] * dl;
		o.mint = eps;
		o.maxt = INFINITY;
		o.time = ray.time;
		o.flags = 0u;
		o.pad[0] = o.pad[1] = 0.f;
		*next = o;
		++live;
	} else
		writeMasked(next);
	if (shadow) {
		const float lx = P.light[0] + rnd(P.seed, pix, P.bounce, 3) - 0.5f;
		const float ly = P.light[1] + rnd(P.seed, pix, P.bounce, 4) - 0.5f;
		const float v[3] = {lx - p[0], ly - p[1], P.light[2] - p[2]};
		const float dist = sqrtf(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
		lrh_ray_rec o;
		o.ox = p[0]; o.oy = p[1]; o.oz = p[2];
		o.dx = v[0] / dist; o.dy = v[1] / dist; o.dz = v[2] / dist;
		o.mint = eps;
		o.maxt = dist - 2.f * eps;
		o.time = ray.time;
		o.flags = dist > 4.f * eps ? 0u : 1u;
		o.pad[0] = o.pad[1] = 0.f;
		*shadow = o;
		live += o.flags ? 0u : 1u;
	}
	return live;
}

// ---- one shading step (see lrh_shade in lrhip.h) ----
__device__ __forceinline__ void cosineDir(const float n[3], float u1, float u2, float d[3]) {
	// cosine-weighted direction around n (Malley), branchless basis (Duff et al. 2017)
	const float r = sqrtf(u1), phi = 6.2831853f * u2;
	const float lx = r * cosf(phi), ly = r * sinf(phi), lz = sqrtf(fmaxf(0.f, 1.f - u1));
	const float sg = n[2] >= 0.f ? 1.f : -1.f;
	const float a = -1.f / (sg + n[2]);
	const float b = n[0] * n[1] * a;
	const float t0[3] = {1.f + sg * n[0] * n[0] * a, sg * b, -sg * n[0]};
	const float t1[3] = {b, sg + n[1] * n[1] * a, -n[1]};
	float v[3];
	for (int k = 0; k < 3; ++k) v[k] = lx * t0[k] + ly * t1[k] + lz * n[k];
	const float dl = 1.f / sqrtf(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
	for (int k = 0; k < 3; ++k) d[k] = v[k] * dl;
}

struct ShadeOut {
	LrhPath path;
	lrh_ray_rec next, shadow;
	uint32_t live;
	bool write;
};

__device__ __forceinline__ void shadeOne(const LrhShadeParams &P, uint32_t i, ShadeOut &O) {
	O.live = 0;
	O.write = false;
	LrhPath &path = O.path;
	path = P.paths[i];
	const lrh_ray_rec ray = P.rays[i];
	lrh_hit_rec hit = P.hits[i];
	const bool pending = path.dl[0] != 0.f || path.dl[1] != 0.f || path.dl[2] != 0.f;
	// a path already ended when the previous step ran (pad = 1) and with no
	// light pending: that step and the one that ended it masked its slots of
	// both ray buffers and of the shadow buffer, so there is nothing to do
	if (!path.alive && path.pad && !pending) return;
	O.write = true;
	writeMasked(&O.next);
	writeMasked(&O.shadow);
	// (keeps the hit's load up here, beside the path's: three dependent waits
	// on memory were four)
	asm volatile("" : "+v"(hit.meshIndex), "+v"(hit.triangleIndex), "+v"(hit.t));
	// the previous step's shadow ray: its light counts if nothing blocked it
	if (P.shadowHits && pending && P.shadowHits[i].meshIndex == 0xffffffffu)
		for (int k = 0; k < 3; ++k) path.rad[k] = path.rad[k] + path.dl[k];
	for (int k = 0; k < 3; ++k) path.dl[k] = 0.f;
	if (!path.alive) {
		path.pad = 1u;
		return;
	}
	if ((ray.flags & 1u) || hit.meshIndex >= P.nMeshes ||
			hit.triangleIndex >= P.meshTriBase[hit.meshIndex + 1] - P.meshTriBase[hit.meshIndex]) {
		path.alive = 0u;
		return;
	}
	LrhMaterial m;
	if (hit.meshIndex < P.nMaterials)
		m = P.materials[hit.meshIndex];
	else
		for (int k = 0; k < 3; ++k) m.kd[k] = m.le[k] = 0.f;
	const uint32_t rec = P.invPerm[P.meshTriBase[hit.meshIndex] + hit.triangleIndex];
	const lrh_tri tr = P.tris[rec];
	float n[3] = {tr.e1[1] * tr.e2[2] - tr.e1[2] * tr.e2[1], tr.e1[2] * tr.e2[0] - tr.e1[0] * tr.e2[2],
			tr.e1[0] * tr.e2[1] - tr.e1[1] * tr.e2[0]};
	const float nl = sqrtf(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
	const float s = (n[0] * ray.dx + n[1] * ray.dy + n[2] * ray.dz > 0.f ? -1.f : 1.f) / fmaxf(nl, 1e-30f);
	for (int k = 0; k < 3; ++k) n[k] *= s;
	const float p[3] = {ray.ox + ray.dx * hit.t, ray.oy + ray.dy * hit.t, ray.oz + ray.dz * hit.t};
	const float eps = fmaxf(epsE(p[0]), fmaxf(epsE(p[1]), epsE(p[2])));
	const uint32_t pix = P.pixelBase + i;
	const uint32_t depth = path.depth;
	if (depth == 0)  // a light seen directly
		for (int k = 0; k < 3; ++k) path.rad[k] = path.rad[k] + path.thr[k] * m.le[k];
	const bool diffuse = m.kd[0] > 0.f || m.kd[1] > 0.f || m.kd[2] > 0.f;
	if (P.nLights && diffuse) {
		const float u0 = rnd(P.seed, pix, depth, 3), u1 = rnd(P.seed, pix, depth, 4), u2 = rnd(P.seed, pix, depth, 5);
		uint32_t j = (uint32_t)(u0 * (float)P.nLights);
		if (j > P.nLights - 1) j = P.nLights - 1;
		const LrhLightTri L = P.lights[j];
		const float su = sqrtf(u1), a = su * (1.f - u2), b = su * u2;
		float w[3];
		for (int k = 0; k < 3; ++k) w[k] = (L.p0[k] + a * L.e1[k] + b * L.e2[k]) - p[k];
		const float d2 = w[0] * w[0] + w[1] * w[1] + w[2] * w[2];
		const float dist = sqrtf(d2);
		float wn[3];
		for (int k = 0; k < 3; ++k) wn[k] = w[k] / dist;
		const float ln[3] = {L.e1[1] * L.e2[2] - L.e1[2] * L.e2[1], L.e1[2] * L.e2[0] - L.e1[0] * L.e2[2],
				L.e1[0] * L.e2[1] - L.e1[1] * L.e2[0]};
		const float lnl = sqrtf(ln[0] * ln[0] + ln[1] * ln[1] + ln[2] * ln[2]);
		const float cosS = n[0] * wn[0] + n[1] * wn[1] + n[2] * wn[2];
		const float cosL = fabsf(ln[0] * wn[0] + ln[1] * wn[1] + ln[2] * wn[2]) / lnl;
		if (cosS > 0.f && cosL > 0.f && dist > 4.f * eps) {
			// uniform light pick (1/n) and point (1/area): 1/pdf = n * area
			const float g = ((cosS * cosL) * (0.5f * lnl * (float)P.nLights)) / d2 * 0.31830988f;
			for (int k = 0; k < 3; ++k) path.dl[k] = path.thr[k] * m.kd[k] * L.le[k] * g;
			lrh_ray_rec o;
			o.ox = p[0]; o.oy = p[1]; o.oz = p[2];
			o.dx = wn[0]; o.dy = wn[1]; o.dz = wn[2];
			o.mint = eps;
			o.maxt = dist - 2.f * eps;
			o.time = ray.time;
			o.flags = 0u;
			o.pad[0] = o.pad[1] = 0.f;
			O.shadow = o;
			++O.live;
		}
	}
	const uint32_t depth1 = depth + 1;
	bool alive = depth1 < P.maxDepth && diffuse;
	if (alive && depth1 >= P.rrDepth) {
		if (rnd(P.seed, pix, depth, 2) < P.rrSurvive)
			for (int k = 0; k < 3; ++k) path.thr[k] = path.thr[k] / P.rrSurvive;
		else
			alive = false;
	}
	if (alive) {
		float d[3];
		cosineDir(n, rnd(P.seed, pix, depth, 0), rnd(P.seed, pix, depth, 1), d);
		// Lambertian: f cos / pdf = kd for cosine-weighted directions
		for (int k = 0; k < 3; ++k) path.thr[k] = path.thr[k] * m.kd[k];
		lrh_ray_rec o;
		o.ox = p[0]; o.oy = p[1]; o.oz = p[2];
		o.dx = d[0]; o.dy = d[1]; o.dz = d[2];
		o.mint = eps;
		o.maxt = INFINITY;
		o.time = ray.time;
		o.flags = 0u;
		o.pad[0] = o.pad[1] = 0.f;
		O.next = o;
		++O.live;
	}
	path.depth = depth1;
	path.alive = alive ? 1u : 0u;
}

__device__ __forceinline__ void countLive(uint32_t *counter, uint32_t live) {
	// one atomic per wave
	unsigned long long v = live;
	for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
	if (counter && __lane_id() == 0 && v) atomicAdd(counter, (uint32_t)v);
}

__global__ void lrh_bounce_kernel(LrhBounceParams P) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	uint32_t live = 0;
	if (i < P.count) live = bounceOne(P, i);
	countLive(P.liveCount, live);
}

__device__ __forceinline__ uint32_t shadeWave(const LrhShadeParams &P, uint32_t i) {
	__shared__ uint4 stage[4][192];
	ShadeOut O;
	O.live = 0;
	O.write = false;
	if (i < P.count) shadeOne(P, i, O);
	const uint64_t mask = __ballot(O.write);
	if (!mask) return 0;
	const uint32_t first = i - (threadIdx.x & 63u);
	uint4 *lds = stage[threadIdx.x >> 6];
	storeRecords(lds, P.next + first, O.next, mask);
	storeRecords(lds, P.shadow + first, O.shadow, mask);
	storeRecords(lds, P.paths + first, O.path, mask);
	return O.live;
}

__global__ __launch_bounds__(256) void lrh_shade_kernel(LrhShadeParams P) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	const uint32_t live = shadeWave(P, i);
	countLive(P.liveCount, live);
}

__global__ __launch_bounds__(256) void lrh_shade_batch_kernel(LrhShadeBatchArgs A) {
	// the item of this block (uniform over the block: scalar loads of the
	// kernel arguments)
	uint32_t k = 0;
	while (k + 1 < A.n && blockIdx.x >= A.blockStart[k + 1]) ++k;
	const LrhShadeParams &P = A.p[k];
	const uint32_t i = (blockIdx.x - A.blockStart[k]) * blockDim.x + threadIdx.x;
	const uint32_t live = shadeWave(P, i);
	countLive(P.liveCount, live);
}

__global__ __launch_bounds__(256) void lrh_paths_init_kernel(LrhPath *paths, uint32_t count) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	LrhPath p;
	for (int k = 0; k < 3; ++k) {
		p.thr[k] = 1.f;
		p.rad[k] = 0.f;
		p.dl[k] = 0.f;
	}
	p.depth = 0u;
	p.alive = 1u;
	p.pad = 0u;
	__shared__ uint4 stage[4][192];
	storeRecords(stage[threadIdx.x >> 6], paths + (i - (threadIdx.x & 63u)), p, __ballot(i < count));
}

}  // namespace

hipError_t lrhLaunchCamera(const LrhCameraParams &C, lrh_ray_rec *rays, hipStream_t s) {
	const uint32_t n = C.width * C.height;
	hipLaunchKernelGGL(lrh_camera_kernel, dim3((n + 255) / 256), dim3(256), 0, s, C, rays);
	return hipGetLastError();
}

hipError_t lrhLaunchPathsInit(LrhPath *paths, uint32_t count, hipStream_t s) {
	hipLaunchKernelGGL(lrh_paths_init_kernel, dim3((count + 255) / 256), dim3(256), 0, s, paths, count);
	return hipGetLastError();
}

hipError_t lrhLaunchShade(const LrhShadeParams &P, hipStream_t s) {
	hipLaunchKernelGGL(lrh_shade_kernel, dim3((P.count + 255) / 256), dim3(256), 0, s, P);
	return hipGetLastError();
}

hipError_t lrhLaunchShadeBatch(const LrhShadeBatchArgs &A, hipStream_t s) {
	if (A.n == 0 || A.n > (uint32_t)kShadeBatchMax) return hipErrorInvalidValue;
	hipLaunchKernelGGL(lrh_shade_batch_kernel, dim3(A.blockStart[A.n]), dim3(256), 0, s, A);
	return hipGetLastError();
}

hipError_t lrhLaunchBounce(const LrhBounceParams &P, hipStream_t s) {
	hipLaunchKernelGGL(lrh_bounce_kernel, dim3((P.count + 255) / 256), dim3(256), 0, s, P);
	return hipGetLastError();
}
