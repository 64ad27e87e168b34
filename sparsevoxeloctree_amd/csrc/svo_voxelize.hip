// Mesh voxelization into the reference's fragment list (Voxelizer, src/Voxelizer.cpp:5-179), as
// compute kernels instead of the geometry-shader + conservative-raster pipeline.
//
//   per triangle (shader/voxelizer.geom:21-54): dominant axis of the face normal, swizzled
//     projection, pixel AABB and voxel depth range, exactly as the geometry shader computes them;
//   coverage (conservative rasterization, src/Voxelizer.cpp:112-127): pixel (i,j) is covered when
//     the closed triangle, with vertices snapped to 1/256 pixel, meets the half-open pixel square
//     [i,i+1) x [j,j+1).  A closed triangle and a half-open square are disjoint exactly when the
//     square's or the triangle's own sides separate them, so the covered pixels of the AABB are
//     those inside three half-planes A_k i + B_k j >= C_k with integer coefficients, one per edge
//     (RowPlanes); every row's covered pixels form one span, found with exact double arithmetic;
//   per pixel (shader/voxelizer.frag:17-44): depth of the triangle's plane at the pixel centre,
//     clamps to [0,res-1] and to the depth range, swizzle back, fragment packing.
// Two passes like the reference's count-only + fill draws: vox_count writes the per-triangle count,
// a device scan turns counts into offsets, vox_fill writes each triangle's fragments at its offset
// (triangle order, row-major inside a triangle).  Both passes cover a batch of scenes in one launch
// (segment tables, svo_batch.hpp): the triangles of all scenes form one index space, and every
// scene's fragments land in its own list.
//
// Scene normalisation (src/Scene.cpp:62-99) runs here too: bounding-box reduction + transform.
#include <cstring>
#include <string>
#include <vector>

#include "svo_batch.hpp"
#include "svo_device.hpp"
#include "svo_runtime.hpp"
#include "svo_scan.hpp"

namespace svo {
namespace {

constexpr int kThreads = 256;

// |pixel coordinates| below this are RowPlanes' (2^30 in 1/256 pixels).
constexpr float kMaxPixel = 4194304.0f;

// A triangle as the geometry shader sees it.
struct TriBase {
	bool degenerate;
	uint32_t axis;
	uint32_t dr0, dr1;
	uint32_t a0, a1, a2, a3; // AABB
	float px[3], py[3], pz0;
	float dzdx, dzdy; // plane of the projected triangle (pixel units, depth in [0,1])
};

// What a fragment needs of its triangle: the plane, the depth range with res - 1 folded in, the shifts
// of i, j and depth in the packed word (0 for the volume's x, 12 for y, 24 for z; one byte each).
struct FragTri {
	float px0, py0, pz0, dzdx, dzdy, fres;
	uint32_t zmin, zmax, shifts, colour;
};

// Any triangle, in 64-bit integers: the general form of RowPlanes, for coordinates from kMaxPixel on.
struct Setup {
	bool empty;
	int32_t ilo, ihi, jlo, jhi; // pixel rectangle: AABB ∩ snapped bbox ∩ [0, res)
	int64_t X[3], Y[3];         // snapped vertices
};

__device__ __forceinline__ f3 project(f3 v, uint32_t axis) { // voxelizer.geom:15-19
	f3 r = axis == 0 ? f3{v.y, v.z, v.x} : (axis == 1 ? f3{v.z, v.x, v.y} : v);
	r.z = (r.z + 1.0f) * 0.5f;
	return r;
}

__device__ __forceinline__ int64_t imin64(int64_t a, int64_t b) { return a < b ? a : b; }
__device__ __forceinline__ int64_t imax64(int64_t a, int64_t b) { return a < b ? b : a; }

__device__ __forceinline__ void tri_base(const float *__restrict__ tri, uint64_t t, uint32_t res, TriBase &s) {
	const float *p = tri + 9 * t;
	f3 p0{p[0], p[1], p[2]}, p1{p[3], p[4], p[5]}, p2{p[6], p[7], p[8]};
	f3 e1{p1.x - p0.x, p1.y - p0.y, p1.z - p0.z}, e2{p2.x - p0.x, p2.y - p0.y, p2.z - p0.z};
	f3 n = cross3(e1, e2); // voxelizer.geom:29
	float wx = fabsf(n.x), wy = fabsf(n.y), wz = fabsf(n.z);
	s.axis = (wx > wy && wx > wz) ? 0u : (wy > wz ? 1u : 2u);
	s.degenerate = (n.x == 0.0f && n.y == 0.0f && n.z == 0.0f);
	f3 q0 = project(p0, s.axis), q1 = project(p1, s.axis), q2 = project(p2, s.axis);
	const float fres = (float)res;
	// voxelizer.geom:40-43
	float mnx = gmin(q0.x, gmin(q1.x, q2.x)), mny = gmin(q0.y, gmin(q1.y, q2.y));
	float mxx = gmax(q0.x, gmax(q1.x, q2.x)), mxy = gmax(q0.y, gmax(q1.y, q2.y));
	s.a0 = f2u_sat((mnx + 1.0f) * 0.5f * fres);
	s.a1 = f2u_sat((mny + 1.0f) * 0.5f * fres);
	s.a2 = f2u_sat((mxx + 1.0f) * 0.5f * fres);
	s.a3 = f2u_sat((mxy + 1.0f) * 0.5f * fres);
	s.dr0 = f2u_sat(gmin(q0.z, gmin(q1.z, q2.z)) * fres);
	s.dr1 = f2u_sat(gmax(q0.z, gmax(q1.z, q2.z)) * fres);
	s.px[0] = (q0.x + 1.0f) * 0.5f * fres;
	s.px[1] = (q1.x + 1.0f) * 0.5f * fres;
	s.px[2] = (q2.x + 1.0f) * 0.5f * fres;
	s.py[0] = (q0.y + 1.0f) * 0.5f * fres;
	s.py[1] = (q1.y + 1.0f) * 0.5f * fres;
	s.py[2] = (q2.y + 1.0f) * 0.5f * fres;
	s.pz0 = q0.z;
	float ax = s.px[1] - s.px[0], ay = s.py[1] - s.py[0], az = q1.z - q0.z;
	float bx = s.px[2] - s.px[0], by = s.py[2] - s.py[0], bz = q2.z - q0.z;
	float nx = ay * bz - az * by, ny = az * bx - ax * bz, nz = ax * by - ay * bx;
	s.dzdx = 0.0f;
	s.dzdy = 0.0f;
	if (nz != 0.0f) {
		s.dzdx = -nx / nz;
		s.dzdy = -ny / nz;
	}
}

// NaN is not below kMaxPixel
__device__ __forceinline__ bool pixels_ok(const TriBase &t) {
	bool ok = true;
#pragma unroll
	for (int k = 0; k < 3; ++k)
		ok = ok && fabsf(t.px[k]) < kMaxPixel && fabsf(t.py[k]) < kMaxPixel;
	return ok;
}

// Depth clamps (voxelizer.frag:21-22): min(max(min(z, res - 1), dr0), dr1) with dr0 <= dr1 is z clamped
// to [dr0, max(dr0, min(res - 1, dr1))].
__device__ __forceinline__ FragTri frag_tri(const TriBase &b, uint32_t res, uint32_t rgb) {
	return FragTri{b.px[0], b.py[0], b.pz0, b.dzdx, b.dzdy, (float)res,
	               b.dr0, umax32(b.dr0, umin32(res - 1u, b.dr1)),
	               b.axis == 0u ? 0x00180cu : b.axis == 1u ? 0x0c0018u : 0x180c00u, rgb & 0x00ffffffu};
}

__device__ void tri_setup(const TriBase &b, uint32_t res, Setup &s) {
	int64_t *X = s.X, *Y = s.Y;
#pragma unroll
	for (int k = 0; k < 3; ++k) {
		X[k] = (int64_t)__builtin_rintf(b.px[k] * 256.0f);
		Y[k] = (int64_t)__builtin_rintf(b.py[k] * 256.0f);
	}
	int64_t xmn = imin64(X[0], imin64(X[1], X[2])), xmx = imax64(X[0], imax64(X[1], X[2]));
	int64_t ymn = imin64(Y[0], imin64(Y[1], Y[2])), ymx = imax64(Y[0], imax64(Y[1], Y[2]));
	int64_t ilo = imax64((int64_t)b.a0, xmn >> 8), ihi = imin64(imin64((int64_t)b.a2, (int64_t)res - 1), xmx >> 8);
	int64_t jlo = imax64((int64_t)b.a1, ymn >> 8), jhi = imin64(imin64((int64_t)b.a3, (int64_t)res - 1), ymx >> 8);
	s.empty = b.degenerate || imax64(ilo, 0) > imax64(ihi, -1) || imax64(jlo, 0) > imax64(jhi, -1);
	s.ilo = (int32_t)imin64(imax64(ilo, 0), res);
	s.ihi = (int32_t)imax64(ihi, -1);
	s.jlo = (int32_t)imin64(imax64(jlo, 0), res);
	s.jhi = (int32_t)imax64(jhi, -1);
}

// Exact floor(a / b) for b > 0: the double quotient is within one of it wherever it matters (a
// quotient inside the pixel grid), and the integer remainder corrects it.
__device__ __forceinline__ int64_t floor_div(int64_t a, int64_t b) {
	int64_t q = (int64_t)floor((double)a / (double)b);
	const int64_t r = a - q * b;
	q -= r < 0 ? 1 : 0;
	q += r >= b ? 1 : 0;
	return q;
}

// Covered pixels of row j: [i0, i1] (empty when i0 > i1).  Edge k admits lo <= sx i + sy j <= hi with
// (sx, sy) = 256 times its normal; one edge at a time, as few registers as possible.
__device__ __forceinline__ void row_span(const Setup &s, int32_t j, int32_t &i0, int32_t &i1) {
	int64_t lo = s.ilo, hi = s.ihi;
	int64_t ax = s.X[0], ay = s.Y[0], bx = s.X[1], by = s.Y[1], cx = s.X[2], cy = s.Y[2];
#pragma unroll 1
	for (int k = 0; k < 3; ++k) {
		const int64_t A = by - ay, B = ax - bx;
		const int64_t ce = A * ax + B * ay, cc = A * cx + B * cy;
		const int64_t tlo = imin64(ce, cc), thi = imax64(ce, cc);
		const bool lo_att = A >= 0 && B >= 0, hi_att = A <= 0 && B <= 0;
		const int64_t sx = A * 256, sy = B * 256;
		const int64_t off_lo = (A < 0 ? sx : 0) + (B < 0 ? sy : 0);
		const int64_t width = (sx < 0 ? -sx : sx) + (sy < 0 ? -sy : sy);
		const int64_t syj = sy * (int64_t)j;
		const int64_t nlo = (hi_att ? tlo : tlo + 1) - off_lo - width - syj;
		const int64_t nhi = (lo_att ? thi : thi - 1) - off_lo - syj;
		if (sx != 0) {
			lo = imax64(lo, -floor_div(sx > 0 ? -nlo : nhi, sx > 0 ? sx : -sx));
			hi = imin64(hi, floor_div(sx > 0 ? nhi : -nlo, sx > 0 ? sx : -sx));
		} else if (nlo > 0 || nhi < 0) {
			hi = -1;
		}
		const int64_t tx = ax, ty = ay;
		ax = bx, ay = by;
		bx = cx, by = cy;
		cx = tx, cy = ty;
	}
	if (lo > hi) {
		i0 = 1;
		i1 = 0;
	} else {
		i0 = (int32_t)lo;
		i1 = (int32_t)hi;
	}
}

__device__ __forceinline__ int32_t lane_of(int32_t v, uint32_t l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ uint64_t lane_of(uint64_t u, uint32_t l) {
	const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((uint32_t)u, l);
	const uint32_t h = (uint32_t)__builtin_amdgcn_readlane((uint32_t)(u >> 32), l);
	return a | ((uint64_t)h << 32);
}
__device__ __forceinline__ double lane_of(double v, uint32_t l) {
	return __longlong_as_double((long long)lane_of((uint64_t)__double_as_longlong(v), l));
}

// 1 / a within 2^-51 of its value: two Newton steps from the instruction's 23 bits or more.
__device__ __forceinline__ double reciprocal(double a) {
	double x = __builtin_amdgcn_rcp(a);
	x = fma(fma(-a, x, 1.0), x, x);
	return fma(fma(-a, x, 1.0), x, x);
}

// The covered spans of a triangle's rows, from three half-planes A i + B j >= C.  The vertices are
// put in the order in which the triangle lies on the positive side of every edge; then an edge from
// (x, y) covers the pixels whose square reaches it:
//     256 (A i + B j) >= A x + B y + (corner attained ? 0 : 1) - 256 (max(A, 0) + max(B, 0)).
// The A of the three edges sum to 0, so rows are mirrored (i -> -i) where needed to have one upper
// bound of i (A < 0) and two lower ones (A >= 0), and the vertices rotated to have it last.  With
// M = B j - C the bounds are i <= floor(M / |A|) and i >= -floor(M / |A|), and
//     floor(M / |A|) = round((M + 1/2 - |A| / 2) / |A|),
// two fused multiply-adds and no conversion when the second adds 1.5 * 2^52, which leaves the rounded
// integer in the low word.  C is exact in 64 bits (|x|, |y| < 2^30).  Where the bound lies within the
// pixel grid, |M| < 2^45 is exact in double; what is rounded stays 1/(2 |A|) away from a tie, more than
// the 2^-51 |M / |A|| by which the reciprocal can err, so the result is exact.  Further out it only has
// to stay there: a line moves |B / A| pixels a row, at most the width in 1/256 pixels, and a side of a
// row lies less than the height + 1 rows from the vertices.  So where the width times the height (its
// whole rows + 2) is below 2^29 bounds fit the word (`near`); else they are clamped.  A = 0 bounds the
// rows only, by nothing that the snapped bounding box does not.  A triangle that is a segment or a
// point after snapping gets its line's both sides.
// Doubles rather than 32- or 64-bit integers: v_fma_f64 runs at the rate of an integer add here.
struct RowPlanes {
	double iv[3], b[3], d[3];
	int32_t ilo, ihi; // mirrored if mir
	int32_t jlo, jhi;
	bool mir, near;

	// false (and no rows) if a coordinate is kMaxPixel or more, or not a number
	__device__ __forceinline__ bool init(const TriBase &t, uint32_t res) {
		jlo = 0;
		jhi = -1;
		near = true;
		if (!pixels_ok(t))
			return t.degenerate;
		int32_t x[3], y[3];
#pragma unroll
		for (int k = 0; k < 3; ++k) {
			x[k] = (int32_t)__builtin_rintf(t.px[k] * 256.0f);
			y[k] = (int32_t)__builtin_rintf(t.py[k] * 256.0f);
		}
		const int32_t xmn = min(x[0], min(x[1], x[2])), xmx = max(x[0], max(x[1], x[2]));
		const int32_t ymn = min(y[0], min(y[1], y[2])), ymx = max(y[0], max(y[1], y[2]));
		const int32_t i0 = max((int32_t)t.a0, xmn >> 8), i1 = min(min((int32_t)t.a2, (int32_t)res - 1), xmx >> 8);
		const int32_t j0 = max((int32_t)t.a1, ymn >> 8), j1 = min(min((int32_t)t.a3, (int32_t)res - 1), ymx >> 8);
		if (t.degenerate || i0 > i1)
			return true;
		jlo = j0;
		jhi = j1;
		const int64_t area = (int64_t)(y[1] - y[0]) * (x[2] - x[0]) - (int64_t)(x[1] - x[0]) * (y[2] - y[0]);
		if (area == 0) {
			// on a line: its ends P and Q, as the edges P Q, Q Q (which bounds nothing) and Q P
			const bool flat = ymn == ymx;
			int32_t p = 0, q = 0;
#pragma unroll
			for (int k = 1; k < 3; ++k) {
				const int32_t vk = flat ? x[k] : y[k];
				p = vk < (flat ? pick(x, p) : pick(y, p)) ? k : p;
				q = vk > (flat ? pick(x, q) : pick(y, q)) ? k : q;
			}
			const int32_t xp = pick(x, p), yp = pick(y, p), xq = pick(x, q), yq = pick(y, q);
			x[0] = xp, y[0] = yp;
			x[1] = x[2] = xq, y[1] = y[2] = yq;
			mir = false;
		} else {
			if (area < 0) {
				const int32_t tx = x[1], ty = y[1];
				x[1] = x[2], y[1] = y[2];
				x[2] = tx, y[2] = ty;
			}
			const int32_t a0 = y[1] - y[0], a1 = y[2] - y[1], a2 = y[0] - y[2];
			mir = (a0 > 0) + (a1 > 0) + (a2 > 0) == 1;
			const bool u0 = mir ? a0 > 0 : a0 < 0, u1 = mir ? a1 > 0 : a1 < 0;
			const int32_t x0 = x[0], x1 = x[1], x2 = x[2], y0 = y[0], y1 = y[1], y2 = y[2];
			x[0] = u0 ? x1 : u1 ? x2 : x0, y[0] = u0 ? y1 : u1 ? y2 : y0;
			x[1] = u0 ? x2 : u1 ? x0 : x1, y[1] = u0 ? y2 : u1 ? y0 : y1;
			x[2] = u0 ? x0 : u1 ? x1 : x2, y[2] = u0 ? y0 : u1 ? y1 : y2;
		}
		ilo = mir ? -i1 : i0;
		ihi = mir ? -i0 : i1;
		near = (float)(xmx - xmn) * (float)(((ymx - ymn) >> 8) + 2) < 536870912.0f;
#pragma unroll
		for (int k = 0; k < 3; ++k) {
			const int32_t A = y[(k + 1) % 3] - y[k], B = x[k] - x[(k + 1) % 3];
			const int64_t r = (int64_t)A * x[k] + (int64_t)B * y[k] + (A <= 0 && B <= 0 ? 255 : 256);
			const double a = (double)(A < 0 ? -A : A);
			b[k] = A == 0 ? 0.0 : (double)B;
			d[k] = A == 0 ? 1073741824.0 : 0.5 - 0.5 * a - (double)((r >> 8) - max(A, 0) - max(B, 0));
			iv[k] = A == 0 ? 1.0 : reciprocal(a);
			iv[k] = k == 2 ? iv[k] : -iv[k];
		}
		return true;
	}
	static __device__ __forceinline__ int32_t pick(const int32_t *v, int32_t k) {
		return k == 0 ? v[0] : k == 1 ? v[1] : v[2];
	}
	template <bool kNear> __device__ __forceinline__ int32_t bound(int k, double j) const {
		const double magic = 6755399441055744.0, m = fma(b[k], j, d[k]);
		const double q = kNear ? fma(m, iv[k], magic) : fmin(fmax(m * iv[k], -1073741824.0), 1073741824.0) + magic;
		return (int32_t)(uint32_t)__double_as_longlong(q);
	}
	// number of covered pixels of row j, and the first one
	template <bool kNear> __device__ __forceinline__ int32_t span(int32_t j, int32_t &i0) const {
		const double dj = (double)j;
		const int32_t lo = max(max(bound<kNear>(0, dj), bound<kNear>(1, dj)), ilo), hi = min(bound<kNear>(2, dj), ihi);
		i0 = mir ? -hi : lo;
		return max(hi - lo + 1, 0);
	}
	template <bool kNear> __device__ __forceinline__ uint32_t count(int32_t j) const {
		int32_t i0;
		return (uint32_t)span<kNear>(j, i0);
	}
	__device__ __forceinline__ RowPlanes of_lane(uint32_t l) const {
		RowPlanes w;
#pragma unroll
		for (int k = 0; k < 3; ++k) {
			w.iv[k] = lane_of(iv[k], l);
			w.b[k] = lane_of(b[k], l);
			w.d[k] = lane_of(d[k], l);
		}
		w.ilo = lane_of(ilo, l);
		w.ihi = lane_of(ihi, l);
		w.jlo = lane_of(jlo, l);
		w.jhi = lane_of(jhi, l);
		w.mir = lane_of((int32_t)mir, l) != 0;
		return w;
	}
};

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
	for (int d = 32; d; d >>= 1)
		v += (uint32_t)__shfl_xor((int)v, d, 64);
	return v;
}
// LDS that a wave alone uses: its stores before are seen by its loads after
__device__ __forceinline__ void wave_sync() {
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
}

__global__ void vox_zero_counter(uint32_t *c) { c[0] = 0u; }

// Count pass: a lane walks its triangle's rows.  A few tall triangles in a wave of flat ones are
// instead taken by the whole wave, a row per lane; so are those in the general form that can cover a
// pixel, after the others (in a loop of its own: it needs the registers).  `general` lists the latter, [0] is their number.
// Bound by VALU issue (1.0 busy with slivers, a third of it the triangles' setup): 990,800 triangles
// of a room at 2^10 65 -> 22 us, 8.0M with slivers at 2^12 465 -> 108 us, against 64-bit integers with
// a division per edge side; 870 triangles of 500 rows 56 -> 7 us by the wave-wide walk.
constexpr int32_t kTallRows = 32;

__global__ void __launch_bounds__(kThreads)
    vox_count(const VoxSeg *__restrict__ segs, const uint64_t *__restrict__ tbeg, uint32_t S, uint64_t T,
              uint64_t *__restrict__ counts, uint32_t *__restrict__ general, uint32_t per) {
	const uint32_t lane = threadIdx.x & 63u;
	const uint64_t first = ((uint64_t)blockIdx.x * (kThreads / 64) + (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * per;
	const uint64_t stride = (uint64_t)gridDim.x * (kThreads / 64) * per;
	uint32_t hint = 0;
	bool again = false;
	for (uint64_t base = first; base < T; base += stride) {
		const bool in = lane < per && base + lane < T;
		const uint64_t t = in ? base + lane : base;
		const float *xyz;
		uint64_t tl;
		uint32_t level;
		with_seg<64u>(tbeg, S, hint, base, t, [&](uint32_t sg) {
			xyz = segs[sg].xyz;
			level = segs[sg].level;
			tl = t - tbeg[sg];
		});
		TriBase tri;
		tri_base(xyz, tl, 1u << level, tri);
		RowPlanes rp;
		const bool wild = !rp.init(tri, 1u << level) && in;
		const int32_t rows = in ? rp.jhi - rp.jlo + 1 : 0;
		// a tall triangle's share of the wave costs what about six rows of the lanes' walk cost
		const int32_t tall_rows = per == 64u ? kTallRows : 8;
		bool tall = rows > tall_rows;
		const bool far = rows > 0 && !rp.near;
		int32_t most = 0, n = 0;
		for (uint64_t m = __ballot(tall); m; m &= m - 1u, ++n)
			most = max(most, lane_of(rows, (uint32_t)__ffsll((unsigned long long)m) - 1u));
		tall = far || (tall && n * 6 < most - tall_rows);
		uint32_t c = 0;
		if (!tall && in)
			for (int32_t j = rp.jlo; j <= rp.jhi; ++j)
				c += rp.count<true>(j);
		for (uint64_t m = __ballot(tall); m; m &= m - 1u) {
			const uint32_t l = (uint32_t)__ffsll((unsigned long long)m) - 1u;
			const RowPlanes w = rp.of_lane(l);
			uint32_t wc = 0;
			for (int32_t j = w.jlo + (int32_t)lane; j <= w.jhi; j += 64)
				wc += w.count<false>(j);
			wc = wave_sum(wc);
			c = lane == l ? wc : c;
		}
		again |= __ballot(wild) != 0u;
		if (in && !wild)
			counts[t] = c;
	}
	if (!again)
		return;
	for (uint64_t base = first; base < T; base += stride) {
		// those that cannot cover a pixel are done here
		bool covers = false;
		if (lane < per && base + lane < T) {
			const uint64_t t = base + lane;
			const uint32_t sg = S == 1u ? 0u : seg_find(tbeg, S, t);
			const uint32_t res = 1u << segs[sg].level;
			TriBase tri;
			tri_base(segs[sg].xyz, t - tbeg[sg], res, tri);
			if (!pixels_ok(tri) && !tri.degenerate) {
				Setup s;
				tri_setup(tri, res, s);
				covers = !s.empty;
				if (s.empty)
					counts[t] = 0u;
			}
		}
		for (uint64_t m = __ballot(covers); m; m &= m - 1u) {
			const uint64_t t = base + (uint32_t)__ffsll((unsigned long long)m) - 1u;
			const uint32_t sg = S == 1u ? 0u : seg_find(tbeg, S, t);
			const uint32_t res = 1u << segs[sg].level;
			TriBase tri;
			tri_base(segs[sg].xyz, t - tbeg[sg], res, tri);
			Setup s;
			tri_setup(tri, res, s);
			uint32_t c = 0;
			for (int32_t j = s.jlo + (int32_t)lane; j <= s.jhi; j += 64) {
				int32_t i0, i1;
				row_span(s, j, i0, i1);
				c += (uint32_t)(i1 - i0 + 1);
			}
			c = wave_sum(c);
			if (lane == 0u) {
				counts[t] = c;
				if (c)
					general[1 + atomicAdd(&general[0], 1u)] = (uint32_t)t;
			}
		}
	}
}

// Scene s: first fragment and fragment count from the scanned offsets (total = all fragments), also into
// the host's copy of the descriptors (out, pinned memory) when there is one.
__device__ __forceinline__ void vox_seg_total(VoxSeg *segs, const uint64_t *tbeg, uint32_t s, uint64_t T,
                                              const uint64_t *offsets, const uint64_t *total, VoxSeg *out) {
	const uint64_t b = tbeg[s] < T ? offsets[tbeg[s]] : *total;
	const uint64_t e = tbeg[s + 1u] < T ? offsets[tbeg[s + 1u]] : *total;
	VoxSeg g = segs[s];
	g.frag_begin = b;
	g.F = e - b;
	segs[s].frag_begin = g.frag_begin;
	segs[s].F = g.F;
	if (out)
		out[s] = g;
}
__global__ void vox_seg_totals(VoxSeg *segs, const uint64_t *__restrict__ tbeg, uint32_t S, uint64_t T,
                               const uint64_t *__restrict__ offsets, const uint64_t *__restrict__ total, VoxSeg *out) {
	const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
	if (s < S)
		vox_seg_total(segs, tbeg, s, T, offsets, total, out);
}

// One fragment: depth at the pixel centre, clamps, swizzle back (voxelizer.frag:17-25) and packing
// (voxelizer.frag:38-42: x | y << 12 | z << 24, (z >> 8) << 28 | rgb).
__device__ __forceinline__ uint64_t make_frag(const FragTri &s, uint32_t i, uint32_t j) {
	const float dy = s.dzdy * (((float)(int32_t)j + 0.5f) - s.py0);
	const float zc = s.pz0 + (s.dzdx * (((float)(int32_t)i + 0.5f) - s.px0) + dy);
	const uint32_t z = umin32(umax32(f2u_sat(zc * s.fres), s.zmin), s.zmax);
	const uint32_t sj = s.shifts >> 8, sz = s.shifts >> 16;
	const uint32_t lo = i << (s.shifts & 31u) | j << (sj & 31u) | z << (sz & 31u);
	const uint32_t vz = sz == 24u ? z : (s.shifts & 255u) == 24u ? i : j;
	return (uint64_t)(((vz << 20u) & 0xf0000000u) | s.colour) << 32 | lo;
}
// a fragment list as a place in global memory, also where the address comes from LDS
using FragOut = __attribute__((address_space(1))) uint64_t;

// Fill (triangle order, row-major inside a triangle), split by work: triangle t costs kTriCost plus
// one per fragment, so it owns the keys from K(t) = offsets[t] + kTriCost t on, and a wave takes the
// work of `unit` consecutive keys, which may be many triangles or a small part of one.  Triangles are
// taken in groups of 64, one per lane: a group of at most `unit` keys by the wave that has its first
// key, a larger one by all that have a part of it, each its fragments.  The group's fragments are laid
// end to end, kWin of them per window: the lanes walk the rows and leave each row's {triangle, i, j} in
// LDS at its first fragment's place; then a lane per fragment finds its row by the heads at or below
// its place and its triangle's parameters in LDS, and writes: even work and whole lines, whatever the
// triangles' shapes.  Rows are walked a triangle per lane, or, where a window holds few triangles (tall
// ones, or of many fragments), a row per lane.
// Bound by VALU issue (0.7 busy in a room, 1.0 with slivers; per 64 fragments 46 instructions, and 25
// per row of the tallest triangle of a window): 35M fragments of a room at 2^10 245 -> 116 us, 173M with slivers at 2^12
// 1472 -> 560 us, 32 mixed scenes 990 -> 396 us, against a triangle per lane writing its own fragments
// and a block per triangle above 128 of them; where few triangles hold most (room of 220,848 at 2^11,
// 54M fragments) 659 -> 153 us.  Windows of 512 / 1024: 598 / 576 us with slivers, 404 / 415 the batch.
// Offsets are global over the batch; fend = {the batch's fragment total, the fill limit}: a triangle
// whose fragments end past the limit is not written (the limit is the total, or 0 when a captured
// plan found a fragment count above its list's capacity).
constexpr uint32_t kWin = 768;
constexpr uint32_t kTriCost = 8;
// Units: 48 waves per CU (twice what it holds) or more, for an even end, and at least 256 keys for the
// search and the group's setup; above 4096 the last waves run alone (870 triangles, 20,631 fragments:
// 256 / 1024 / 4096 12 / 14 / 28 us; slivers: 2048 / 4096 668 / 576 us; room: 4096 / 8192 139 / 159 us).
constexpr uint32_t kMinUnit = 256, kMaxUnit = 4096;

// Last group of 64 triangles whose keys begin at or below key.
__device__ __forceinline__ uint64_t key_group(const uint64_t *__restrict__ offsets, uint64_t groups, uint64_t key,
                                              uint32_t lane) {
	uint64_t lo = 0, hi = groups;
	while (hi - lo > 1u) {
		const uint64_t step = (hi - lo + 63u) / 64u, g = lo + lane * step, t = 64u * (g < hi ? g : lo);
		const uint64_t m = __ballot(g < hi && offsets[t] + kTriCost * t <= key);
		lo += ((uint32_t)__popcll(m) - 1u) * step; // lane 0's holds
		hi = lo + step < hi ? lo + step : hi;
	}
	return lo;
}

__global__ void __launch_bounds__(kThreads, 6)
    vox_fill(const VoxSeg *__restrict__ segs, const uint64_t *__restrict__ tbeg, uint32_t S, uint64_t T,
             const uint64_t *__restrict__ offsets, const uint32_t *__restrict__ general,
             const uint64_t *__restrict__ fend, uint32_t unit) {
	__shared__ uint32_t s_head[kThreads / 64][kWin]; // row heads: 1 << 31 | lane << 24 | j << 12 | i - place (12 bits); 0: none
	__shared__ uint4 s_tri[kThreads / 64][64][3];
	const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	uint32_t *head = s_head[wave];
	uint4(*par)[3] = s_tri[wave];
	for (uint32_t q = lane; q < kWin; q += 64u)
		head[q] = 0u;
	const uint64_t Ftot = fend[0], lim = fend[1];
	if (lim == 0u)
		return;
	const uint64_t keys = Ftot + kTriCost * T;
	const uint64_t waves = (uint64_t)gridDim.x * (kThreads / 64);
	for (uint64_t key = ((uint64_t)blockIdx.x * (kThreads / 64) + wave) * unit; key < keys; key += waves * unit) {
		const uint64_t key_end = key + unit;
		uint64_t t0 = 64u * key_group(offsets, (T + 63u) / 64u, key, lane);
		uint32_t hint = S == 1u ? 0u : seg_find(tbeg, S, t0);
		for (bool more = true; more; t0 += 64u) {
			const bool in = t0 + lane < T;
			const uint64_t t = in ? t0 + lane : T - 1u;
			const uint64_t k = offsets[t];
			const uint64_t kend = (t + 1 < T) ? offsets[t + 1] : Ftot;
			const uint64_t kb = k + kTriCost * (t + 1u); // key of its first fragment
			const uint64_t gb = lane_of(kb, 0u) - kTriCost, ge = lane_of(kb + (kend - k), 63u); // the group's keys
			more = t0 + 64u < T && ge < key_end;
			const bool whole = ge - gb <= unit;
			if (whole && gb < key)
				continue;
			// its fragments to write: [skip, skip + c)
			const uint64_t from = whole ? gb : key, to = whole ? ge : key_end;
			const uint32_t skip = kb < from ? (uint32_t)(from - kb) : 0u;
			const uint64_t ke = kb + (kend - k) < to ? kb + (kend - k) : to;
			uint32_t c = in && kend <= lim && ke > kb + skip ? (uint32_t)(ke - kb) - skip : 0u;
			if (!__any(c != 0u))
				continue;
			const float *xyz;
			const uint32_t *rgb;
			uint2 *frags;
			uint64_t tl, fb; // fb: offsets are global over the batch
			uint32_t level;
			with_seg<64u>(tbeg, S, hint, t0, t, [&](uint32_t sg) {
				const VoxSeg &g = segs[sg];
				xyz = g.xyz;
				rgb = g.rgb;
				frags = g.frags;
				fb = g.frag_begin;
				level = g.level;
				tl = t - tbeg[sg];
			});
			RowPlanes rp;
			TriBase tri;
			tri_base(xyz, tl, 1u << level, tri);
			if (!rp.init(tri, 1u << level))
				c = 0u; // in the general list
			uint32_t incl = c;
#pragma unroll
			for (int d = 1; d < 64; d <<= 1) {
				const uint32_t o = (uint32_t)__shfl_up((int)incl, (unsigned)d, 64);
				if ((int)lane >= d)
					incl += o;
			}
			const uint32_t N = (uint32_t)lane_of((int32_t)incl, 63u);
			// places of the batch's fragments: [0, N); the next row starts at p, its triangle ends at pend
			const int32_t pend = (int32_t)incl;
			int32_t p = (int32_t)(incl - c) - (int32_t)skip;
			{
				const FragTri ft = frag_tri(tri, 1u << level, rgb[tl]);
				const uint64_t out = (uint64_t)(uintptr_t)(frags + (k - fb)) - (int64_t)p * (int64_t)sizeof(uint2);
				par[lane][0] = make_uint4(fbits(ft.px0), fbits(ft.py0), fbits(ft.pz0), fbits(ft.dzdx));
				par[lane][1] = make_uint4(fbits(ft.dzdy), fbits(ft.fres), ft.zmin, ft.zmax);
				par[lane][2] = make_uint4(ft.shifts, ft.colour, (uint32_t)out, (uint32_t)(out >> 32));
			}
			int32_t j = rp.jlo;
			const int32_t rows = rp.jhi - j + 1;
			const bool tall = !rp.near || rows > kTallRows || (rows > 12 && c + skip >= 128u);
			const uint32_t mark = 0x80000000u | lane << 24;
			uint32_t last = 0u; // lane 0: the newest head before the step
			for (int32_t w0 = 0; w0 < (int32_t)N; w0 += (int32_t)kWin) {
				const int32_t wend = c ? min(w0 + (int32_t)kWin, pend) : p;
				// a row of no fragments leaves its head to the next row's; rows before the unit do so at 0
				if (!tall) {
					for (; p < wend && j <= rp.jhi; ++j) {
						int32_t i0;
						const int32_t n = rp.span<true>(j, i0);
						head[max(p, w0) - w0] = mark | (uint32_t)j << 12 | ((uint32_t)(i0 - p) & 4095u);
						p += n;
					}
					if (p < wend) { // never: the rows hold the fragments counted
						head[max(p, w0) - w0] = mark;
						p = pend;
					}
				}
				for (uint64_t m = __ballot(tall && p < wend); m; m &= m - 1u) {
					const uint32_t l = (uint32_t)__ffsll((unsigned long long)m) - 1u;
					const RowPlanes w = rp.of_lane(l);
					const int32_t le = lane_of(pend, l), lw = lane_of(wend, l);
					int32_t lj = lane_of(j, l), lp = lane_of(p, l);
					while (lp < lw) {
						int32_t i0 = 0, n = 0;
						if (lj + (int32_t)lane <= w.jhi)
							n = w.span<false>(lj + (int32_t)lane, i0);
						else if (lj + (int32_t)lane == w.jhi + 1 || (lane == 0u && lj > w.jhi))
							n = le; // never used, as above
						int32_t end = n;
#pragma unroll
						for (int d = 1; d < 64; d <<= 1) {
							const int32_t o = __shfl_up(end, (unsigned)d, 64);
							if ((int)lane >= d)
								end += o;
						}
						end = min(end + lp, le);
						const int32_t before = __shfl_up(end, 1u, 64), beg = lane ? before : lp;
						const int32_t at = max(beg, w0);
						if (beg < lw && end > at)
							head[at - w0] = 0x80000000u | l << 24 | ((uint32_t)(lj + (int32_t)lane) & 4095u) << 12 |
							                ((uint32_t)(i0 - beg) & 4095u);
						// rows that begin in this window or before it are done
						const uint32_t done = (uint32_t)__popcll(__ballot(beg < lw));
						lp = lane_of(end, done - 1u);
						lj += (int32_t)done;
					}
					j = lane == l ? lj : j;
					p = lane == l ? lp : p;
				}
				wave_sync();
				for (uint32_t q = 0; q < kWin && (uint32_t)w0 + q < N; q += 64u) {
					const uint32_t at = (uint32_t)w0 + q + lane;
					uint32_t h = head[q + lane];
					head[q + lane] = 0u;
					const uint64_t m = __ballot(h != 0u) | 1u;
					h = h ? h : last;
					const uint64_t below = m & (~0ull >> (63u - lane));
					const uint32_t row = (uint32_t)__shfl((int)h, 63 - __clzll((long long)below), 64);
					const uint32_t top = (uint32_t)lane_of((int32_t)h, 63u - (uint32_t)__clzll((long long)m));
					last = lane == 0u ? top : 0u;
					if (at < N) {
						const uint4 *tp = par[(row >> 24) & 63u];
						const uint4 f0 = tp[0], f1 = tp[1], f2 = tp[2];
						const FragTri ft{bitsf(f0.x), bitsf(f0.y), bitsf(f0.z), bitsf(f0.w), bitsf(f1.x),
						                 bitsf(f1.y), f1.z, f1.w, f2.x, f2.y};
						FragOut *out = (FragOut *)(uintptr_t)(f2.z | (uint64_t)f2.w << 32);
						out[at] = make_frag(ft, (row + at) & 4095u, (row >> 12) & 4095u);
					}
				}
				wave_sync();
			}
		}
	}
	// the triangles in the general form, a wave each, 64 rows at a time
	const uint32_t ngen = general[0];
	for (uint64_t g = (uint64_t)blockIdx.x * (kThreads / 64) + wave; g < ngen; g += waves) {
		const uint64_t t = general[1 + g];
		if (t >= T)
			continue;
		uint64_t k = offsets[t];
		const uint64_t kend = (t + 1 < T) ? offsets[t + 1] : Ftot;
		if (kend > lim)
			continue;
		const uint32_t sg = S == 1u ? 0u : seg_find(tbeg, S, t);
		const uint64_t tl = t - tbeg[sg];
		const uint32_t res = 1u << segs[sg].level;
		TriBase tri;
		tri_base(segs[sg].xyz, tl, res, tri);
		Setup s;
		tri_setup(tri, res, s);
		if (s.empty)
			continue;
		const FragTri ft = frag_tri(tri, res, segs[sg].rgb[tl]);
		FragOut *frags = (FragOut *)(uintptr_t)(segs[sg].frags - segs[sg].frag_begin);
		for (int32_t j0 = s.jlo; j0 <= s.jhi && k < kend; j0 += 64) {
			int32_t i0 = 1, i1 = 0;
			if (j0 + (int32_t)lane <= s.jhi)
				row_span(s, j0 + (int32_t)lane, i0, i1);
			for (int32_t r = 0; r < 64 && k < kend; ++r) {
				const int32_t a = lane_of(i0, (uint32_t)r), b = lane_of(i1, (uint32_t)r);
				for (int32_t i = a + (int32_t)lane; i <= b; i += 64)
					if (k + (uint32_t)(i - a) < kend)
						frags[k + (uint32_t)(i - a)] = make_frag(ft, (uint32_t)i, (uint32_t)(j0 + r));
				k += (uint32_t)(b - a + 1);
			}
		}
	}
}

struct CountSrc {
	static constexpr int kItems = 4;
	const uint64_t *counts;
	uint64_t n;
	__device__ uint64_t size() const { return n; }
	__device__ uint32_t operator()(uint64_t i) const { return (uint32_t)counts[i]; }
};
struct TotalCommit {
	uint64_t *total;
	__device__ void operator()(uint64_t t) const { *total = t; }
};
struct OffsetDst {
	uint64_t *offsets;
	__device__ bool active() const { return true; }
	__device__ void operator()(uint64_t i, uint64_t k, uint32_t) const { offsets[i] = k; }
};

struct SegTotals { // vox_seg_totals after a scan of one block
	VoxSeg *segs;
	const uint64_t *tbeg;
	uint32_t S;
	uint64_t T;
	const uint64_t *offsets, *total;
	VoxSeg *out;
	__device__ void operator()() const {
		if (threadIdx.x < S)
			vox_seg_total(segs, tbeg, threadIdx.x, T, offsets, total, out);
	}
};
static_assert(kMaxBatch <= kOneThreads, "a scene per thread");

// ---- normalisation (src/Scene.cpp:62-99) -------------------------------------------------------
// Per-block bounding box of the vertices -> parts[6 * b].
__global__ void __launch_bounds__(kThreads) norm_bbox(const float *__restrict__ xyz, uint64_t nverts, float *parts) {
	float mn[3] = {3.402823466e+38f, 3.402823466e+38f, 3.402823466e+38f};
	float mx[3] = {-3.402823466e+38f, -3.402823466e+38f, -3.402823466e+38f};
	const uint64_t stride = (uint64_t)gridDim.x * kThreads;
	for (uint64_t v = (uint64_t)blockIdx.x * kThreads + threadIdx.x; v < nverts; v += stride) {
#pragma unroll
		for (int c = 0; c < 3; ++c) {
			float p = xyz[3 * v + c];
			mn[c] = mn[c] < p ? mn[c] : p;
			mx[c] = p < mx[c] ? mx[c] : p;
		}
	}
	__shared__ float s[6][kThreads];
#pragma unroll
	for (int c = 0; c < 3; ++c) {
		s[c][threadIdx.x] = mn[c];
		s[3 + c][threadIdx.x] = mx[c];
	}
	__syncthreads();
	for (int w = kThreads / 2; w > 0; w >>= 1) {
		if ((int)threadIdx.x < w) {
#pragma unroll
			for (int c = 0; c < 3; ++c) {
				float a = s[c][threadIdx.x], b = s[c][threadIdx.x + w];
				s[c][threadIdx.x] = a < b ? a : b;
				float x = s[3 + c][threadIdx.x], y = s[3 + c][threadIdx.x + w];
				s[3 + c][threadIdx.x] = y < x ? x : y;
			}
		}
		__syncthreads();
	}
	if (threadIdx.x < 6)
		parts[6 * blockIdx.x + threadIdx.x] = s[threadIdx.x][0];
}

// Combines the per-block boxes and computes {center.xyz, inv_extent} into out[4].
__global__ void norm_params(const float *parts, uint32_t nparts, float *out) {
	if (threadIdx.x != 0)
		return;
	float mn[3] = {3.402823466e+38f, 3.402823466e+38f, 3.402823466e+38f};
	float mx[3] = {-3.402823466e+38f, -3.402823466e+38f, -3.402823466e+38f};
	for (uint32_t b = 0; b < nparts; ++b)
		for (int c = 0; c < 3; ++c) {
			float a = parts[6 * b + c], x = parts[6 * b + 3 + c];
			mn[c] = mn[c] < a ? mn[c] : a;
			mx[c] = x < mx[c] ? mx[c] : x;
		}
	float ex = mx[0] - mn[0], ey = mx[1] - mn[1], ez = mx[2] - mn[2];
	float extent = gmax(ex, gmax(ey, ez)) * 0.5f;
	out[0] = (mx[0] + mn[0]) * 0.5f;
	out[1] = (mx[1] + mn[1]) * 0.5f;
	out[2] = (mx[2] + mn[2]) * 0.5f;
	out[3] = 1.0f / extent;
}

__global__ void __launch_bounds__(kThreads) norm_apply(float *xyz, uint64_t nverts, const float *params) {
	const float cx = params[0], cy = params[1], cz = params[2], inv = params[3];
	const uint64_t stride = (uint64_t)gridDim.x * kThreads;
	for (uint64_t v = (uint64_t)blockIdx.x * kThreads + threadIdx.x; v < nverts; v += stride) {
		xyz[3 * v + 0] = (xyz[3 * v + 0] - cx) * inv;
		xyz[3 * v + 1] = (xyz[3 * v + 1] - cy) * inv;
		xyz[3 * v + 2] = (xyz[3 * v + 2] - cz) * inv;
	}
}

uint32_t grid_for(uint64_t items, const svo_ctx *ctx) {
	uint64_t g = (items + kThreads - 1) / kThreads;
	uint64_t cap = (uint64_t)ctx->cu_count * 64u; // 64 blocks per CU: more loads in flight than the CU holds at once
	if (g > cap)
		g = cap;
	return (uint32_t)(g ? g : 1);
}

// vox_count: 64 triangles per wave, fewer where that would leave SIMDs without a wave (then a wave's
// other lanes help with its tall triangles).
hipError_t launch_count(svo_ctx *ctx, const VoxBatch *vb) {
	const uint64_t T = vb->Ttot, want = (T + ctx->cu_count * 16u - 1) / (ctx->cu_count * 16u);
	const uint32_t per = want < 64u ? (uint32_t)want : 64u;
	const uint64_t blocks = (T + per * (kThreads / 64) - 1) / (per * (kThreads / 64)), cap = (uint64_t)ctx->cu_count * 64u;
	return launch(ctx, "vox_count", vox_count, dim3((uint32_t)(blocks < cap ? blocks : cap)), dim3(kThreads), 0,
	              (const VoxSeg *)vb->segs, (const uint64_t *)vb->tbeg, vb->S, T, vb->offsets, vb->general, per);
}

// vox_fill over T triangles with at most Fcap fragments.
hipError_t launch_fill(svo_ctx *ctx, const VoxBatch *vb, uint64_t Fcap) {
	const uint64_t keys = Fcap + kTriCost * vb->Ttot;
	const uint64_t fill = (uint64_t)ctx->cu_count * 48u;
	uint32_t unit = kMinUnit;
	while (unit < kMaxUnit && unit * fill < keys)
		unit *= 2u;
	const uint64_t blocks = (keys + (uint64_t)unit * (kThreads / 64) - 1) / ((uint64_t)unit * (kThreads / 64));
	const uint64_t cap = (uint64_t)ctx->cu_count * 64u;
	return launch(ctx, "vox_fill", vox_fill, dim3((uint32_t)(blocks < cap ? blocks : cap)), dim3(kThreads), 0,
	              (const VoxSeg *)vb->segs, (const uint64_t *)vb->tbeg, vb->S, vb->Ttot, (const uint64_t *)vb->offsets,
	              (const uint32_t *)vb->general, (const uint64_t *)vb->fend, unit);
}

} // namespace

int normalize_scene(svo_ctx *ctx, svo_scene *scene) {
	const uint64_t nverts = scene->T * 3u;
	if (nverts == 0)
		return SVO_OK;
	// parts: 6 floats per block + 4 result floats, carved out of the scan scratch (2 * kScanBlocks u64)
	float *parts = reinterpret_cast<float *>(ctx->d_scan_parts);
	const uint32_t blocks = 256; // 256 * 6 + 4 floats < 2 * kScanBlocks * 2 floats
	float *params = parts + 6 * blocks;
	hipError_t e;
	ctx->t_normalize.start(ctx->stream);
	if ((e = launch(ctx, "norm_bbox", norm_bbox, dim3(blocks), dim3(kThreads), 0, (const float *)scene->xyz, nverts,
	                parts)) != hipSuccess)
		return hip_check(ctx, e, "norm_bbox");
	if ((e = launch(ctx, "norm_params", norm_params, dim3(1), dim3(64), 0, (const float *)parts, blocks, params)) !=
	    hipSuccess)
		return hip_check(ctx, e, "norm_params");
	if ((e = launch(ctx, "norm_apply", norm_apply, dim3(grid_for(nverts, ctx)), dim3(kThreads), 0, scene->xyz, nverts,
	                (const float *)params)) != hipSuccess)
		return hip_check(ctx, e, "norm_apply");
	ctx->t_normalize.stop(ctx->stream);
	return SVO_OK;
}

void vox_batch_release(svo_ctx *ctx, VoxBatch *vb) {
	for (void *p : {(void *)vb->segs, (void *)vb->offsets}) // tbeg and general live in segs' allocation
		ctx->pool->free(p);
	vb->segs = nullptr;
	vb->tbeg = nullptr;
	vb->fend = nullptr;
	vb->offsets = nullptr;
	vb->general = nullptr;
}

namespace {
// Counts -> offsets, the sum into total, the scenes' first fragments and counts (out: see vox_seg_total).
hipError_t vox_scan(svo_ctx *ctx, const VoxBatch *vb, uint64_t *total, VoxSeg *out) {
	const uint64_t T = vb->Ttot;
	const uint32_t S = vb->S;
	const CountSrc src{vb->offsets, T};
	hipError_t e;
	if (T <= kScanOne)
		return launch(ctx, "vox_scan", scan_one<CountSrc, OffsetDst, TotalCommit, NoStep, SegTotals>, dim3(1),
		              dim3(kOneThreads), 0, src, OffsetDst{vb->offsets}, TotalCommit{total}, NoStep{},
		              SegTotals{vb->segs, vb->tbeg, S, T, vb->offsets, total, out});
	if ((e = launch(ctx, "vox_scan_reduce", scan_reduce<CountSrc>, dim3(kScanBlocks), dim3(kScanThreads), 0, src,
	                ctx->d_scan_parts)) != hipSuccess ||
	    (e = launch(ctx, "vox_scan_down", scan_down<CountSrc, OffsetDst, TotalCommit>, dim3(kScanBlocks),
	                dim3(kScanThreads), 0, src, OffsetDst{vb->offsets}, (const uint64_t *)ctx->d_scan_parts,
	                TotalCommit{total})) != hipSuccess)
		return e;
	return launch(ctx, "vox_seg_totals", vox_seg_totals, dim3(div_up(S, 64)), dim3(64), 0, vb->segs,
	              (const uint64_t *)vb->tbeg, S, T, (const uint64_t *)vb->offsets, (const uint64_t *)total, out);
}
} // namespace

// Count pass over a batch + scan + one read-back of every scene's F + allocation of the lists
// (Voxelizer::count_and_create_fragment_list, src/Voxelizer.cpp:134-179).
int voxelize_count_batch(svo_ctx *ctx, svo_fraglist *const *fls, uint32_t S, VoxBatch *vb) {
	if (S == 0)
		return SVO_OK;
	if (S > kMaxBatch)
		return set_error(ctx, SVO_ERR_INVALID_ARGUMENT, "batch larger than 1024 scenes");
	vb->S = S;
	vb->h_segs.assign(S, VoxSeg{});
	vb->h_tbeg.assign(S + 1, 0);
	uint64_t T = 0;
	for (uint32_t s = 0; s < S; ++s) {
		const svo_scene *sc = fls[s]->scene;
		VoxSeg &g = vb->h_segs[s];
		g.xyz = sc->xyz;
		g.rgb = sc->rgb;
		g.T = sc->T;
		g.level = fls[s]->level;
		vb->h_tbeg[s] = T;
		T += sc->T;
	}
	vb->h_tbeg[S] = T;
	vb->Ttot = T;
	if (T > 0xFFFFFFFFull)
		return set_error(ctx, SVO_ERR_OVERFLOW, "more than 2^32-1 triangles in one voxelize call");
	Pool *pool = ctx->pool;
	hipError_t e;
	// descriptors, triangle begins (+ the fill's {total, limit}) and the general list share one
	// allocation, so one copy uploads the tables and clears the list's count
	const size_t seg_bytes = (sizeof(VoxSeg) * S + 255) & ~size_t(255);
	const size_t tbeg_bytes = (sizeof(uint64_t) * (S + 3) + 255) & ~size_t(255);
	if (pool->alloc((void **)&vb->segs, seg_bytes + tbeg_bytes + sizeof(uint32_t) * (T + 1)) != hipSuccess ||
	    pool->alloc((void **)&vb->offsets, sizeof(uint64_t) * (T ? T : 1)) != hipSuccess)
		return set_error(ctx, SVO_ERR_OUT_OF_MEMORY, "count-pass allocation failed");
	vb->tbeg = reinterpret_cast<uint64_t *>(reinterpret_cast<uint8_t *>(vb->segs) + seg_bytes);
	vb->fend = vb->tbeg + S + 1;
	vb->general = reinterpret_cast<uint32_t *>(reinterpret_cast<uint8_t *>(vb->segs) + seg_bytes + tbeg_bytes);
	{
		std::vector<uint8_t> tables(seg_bytes + tbeg_bytes + sizeof(uint32_t), 0);
		std::memcpy(tables.data(), vb->h_segs.data(), sizeof(VoxSeg) * S);
		std::memcpy(tables.data() + seg_bytes, vb->h_tbeg.data(), sizeof(uint64_t) * (S + 1));
		if (int rc = upload_table(ctx, vb->segs, tables.data(), tables.size()))
			return rc; // general[0] = 0 came with the tables
	}
	uint64_t *total = ctx->d_scan_parts + 2 * kScanBlocks;
	VoxSeg *out = nullptr;
	if (S <= kReadbackScenes && !(out = static_cast<VoxSeg *>(readback_slot(ctx, sizeof(VoxSeg) * S))))
		return SVO_ERR_INVALID_ARGUMENT;
	ctx->t_count.start(ctx->stream);
	if (T > 0 && (e = launch_count(ctx, vb)) != hipSuccess)
		return hip_check(ctx, e, "vox_count");
	if ((e = vox_scan(ctx, vb, total, out)) != hipSuccess) // without triangles: every count 0
		return hip_check(ctx, e, "vox_scan");
	ctx->t_count.stop(ctx->stream);
	if (int rc = out ? readback_wait(ctx, vb->h_segs.data(), out, sizeof(VoxSeg) * S)
	                 : download_table(ctx, vb->h_segs.data(), vb->segs, sizeof(VoxSeg) * S))
		return rc;
	uint64_t Ftot = 0;
	for (uint32_t s = 0; s < S; ++s) {
		VoxSeg &g = vb->h_segs[s];
		if (g.F > 0xFFFFFFFFull)
			return set_error(ctx, SVO_ERR_OVERFLOW, "more than 2^32-1 fragments in scene " + std::to_string(s));
		svo_fraglist *fl = fls[s];
		fl->F = g.F;
		if (pool->alloc((void **)&fl->frags, sizeof(uint32_t) * 2 * (g.F ? g.F : 1)) != hipSuccess)
			return set_error(ctx, SVO_ERR_OUT_OF_MEMORY, "fragment list allocation failed");
		g.frags = reinterpret_cast<uint2 *>(fl->frags);
		Ftot += g.F;
	}
	// the descriptors with their lists, and the fill's {total, limit} = {Ftot, Ftot}
	std::vector<uint8_t> tables(seg_bytes + tbeg_bytes, 0);
	std::memcpy(tables.data(), vb->h_segs.data(), sizeof(VoxSeg) * S);
	vb->h_tbeg.push_back(Ftot);
	vb->h_tbeg.push_back(Ftot);
	std::memcpy(tables.data() + seg_bytes, vb->h_tbeg.data(), sizeof(uint64_t) * (S + 3));
	vb->h_tbeg.resize(S + 1);
	return upload_table(ctx, vb->segs, tables.data(), tables.size());
}

// Fill pass of a counted batch (CmdVoxelize, src/Voxelizer.cpp:166-179).
int voxelize_fill_batch(svo_ctx *ctx, VoxBatch *vb) {
	const uint64_t T = vb->Ttot;
	const uint32_t S = vb->S;
	uint64_t Ftot = 0;
	for (uint32_t s = 0; s < S; ++s)
		Ftot += vb->h_segs[s].F;
	hipError_t e;
	ctx->t_fill.start(ctx->stream);
	if (T > 0 && Ftot > 0) {
		if ((e = launch_fill(ctx, vb, Ftot)) != hipSuccess)
			return hip_check(ctx, e, "vox_fill");
	}
	ctx->t_fill.stop(ctx->stream);
	return SVO_OK;
}

// Tables of a captured plan's voxelize pass: the lists are allocated by the plan at their
// capacities, so the descriptors (scene buffers, list pointers, levels) never change; F and
// frag_begin are rewritten by every count pass.
int voxelize_plan_init(svo_ctx *ctx, VoxBatch *vb, svo_fraglist *const *fls, uint32_t S) {
	vb->S = S;
	vb->h_segs.assign(S, VoxSeg{});
	vb->h_tbeg.assign(S + 1, 0);
	uint64_t T = 0;
	for (uint32_t s = 0; s < S; ++s) {
		VoxSeg &g = vb->h_segs[s];
		g.xyz = fls[s]->scene->xyz;
		g.rgb = fls[s]->scene->rgb;
		g.T = fls[s]->scene->T;
		g.level = fls[s]->level;
		g.frags = reinterpret_cast<uint2 *>(fls[s]->frags);
		vb->h_tbeg[s] = T;
		T += g.T;
	}
	vb->h_tbeg[S] = T;
	vb->Ttot = T;
	if (T == 0 || T > 0xFFFFFFFFull)
		return set_error(ctx, SVO_ERR_INVALID_ARGUMENT, "a captured plan needs 1 to 2^32-1 triangles in all");
	const size_t seg_bytes = (sizeof(VoxSeg) * S + 255) & ~size_t(255);
	const size_t tbeg_bytes = (sizeof(uint64_t) * (S + 3) + 255) & ~size_t(255);
	if (ctx->pool->alloc((void **)&vb->segs, seg_bytes + tbeg_bytes + sizeof(uint32_t) * (T + 1)) != hipSuccess ||
	    ctx->pool->alloc((void **)&vb->offsets, sizeof(uint64_t) * T) != hipSuccess)
		return set_error(ctx, SVO_ERR_OUT_OF_MEMORY, "plan voxelize allocation failed");
	vb->tbeg = reinterpret_cast<uint64_t *>(reinterpret_cast<uint8_t *>(vb->segs) + seg_bytes);
	vb->fend = vb->tbeg + S + 1;
	vb->general = reinterpret_cast<uint32_t *>(reinterpret_cast<uint8_t *>(vb->segs) + seg_bytes + tbeg_bytes);
	std::vector<uint8_t> tables(seg_bytes + tbeg_bytes, 0);
	std::memcpy(tables.data(), vb->h_segs.data(), sizeof(VoxSeg) * S);
	std::memcpy(tables.data() + seg_bytes, vb->h_tbeg.data(), sizeof(uint64_t) * (S + 1));
	return upload_table(ctx, vb->segs, tables.data(), tables.size());
}

// Count pass of a plan: general list cleared by a kernel (the pass may be captured, so no
// memset), counts, scan into offsets and fend[0] = total, per-scene F and frag_begin.
hipError_t voxelize_plan_count(svo_ctx *ctx, VoxBatch *vb) {
	hipError_t e;
	if ((e = launch(ctx, "vox_zero", vox_zero_counter, dim3(1), dim3(1), 0, vb->general)) != hipSuccess ||
	    (e = launch_count(ctx, vb)) != hipSuccess)
		return e;
	return vox_scan(ctx, vb, vb->fend, nullptr);
}

// Fill pass of a plan: writes nothing when fend[1] (set between the passes) is 0.
hipError_t voxelize_plan_fill(svo_ctx *ctx, VoxBatch *vb, uint64_t Fcap) { return launch_fill(ctx, vb, Fcap); }

} // namespace svo
