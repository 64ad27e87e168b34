// Octree construction (OctreeBuilder::CmdBuild, src/OctreeBuilder.cpp:142-210) for a batch of
// scenes: every kernel covers all scenes of the batch in one launch (segment tables, svo_batch.hpp).
//
// The canonical breadth-first node order (child blocks in ascending parent word index) is the
// Morton order of the node prefixes at every depth: a block's 8 children sit in slot order
// x | y << 1 | z << 2 and blocks follow their parents.  So the whole internal structure follows
// from which prefixes are occupied, and the build works on occupancy bitmaps instead of one
// fragment pass per level:
//
// Reference pass              -> here
//   octree_tag_node.comp      -> bm_group: each tile of consecutive fragments is grouped by depth-(L-1)
//   (levels 1..L-1)              node ("runs"), and every run's node is marked in bitmap B[L-1];
//                                bm_reduce ORs each byte of B[d+1] (8 children) into one bit of B[d],
//                                d = L-2..1
//   octree_alloc_node.comp    -> one exclusive scan over the set-bit counts of all bitmaps' 8-word
//                                chunks (stored by bm_reduce while it reads them)
//                                (rank of every occupied node among its depth = its block among
//                                the allocated children blocks); child pointer = 8 * (first block
//                                of depth + rank)
//   octree_modify_arg.comp    -> bm_levels: per-depth counts -> first block of every depth, the
//                                leaf blocks and W = (counter + 1) * 8
//   octree_init_node.comp     -> bm_write_blocks writes every block whole (pointers and zeros)
//   octree_tag_node.comp      -> tag_runs: leaf block ("bin") of each run = rank of its depth-(L-1)
//   (level L) + leaf CAS fold    node; count per bin, scan, scatter_runs into per-bin buckets;
//                                build_fold and build_fold_lists sort each bucket in fragment order and
//                                fold the 8 leaves of the block in that order (the reference's order
//                                is whatever its atomics produce), writing the leaf block whole.
// The node words are identical to the reference's pass structure run with a serial allocator.
//
// Batch layout: the scenes' fragment tiles, bitmap words and leaf blocks each form one index space
// (begin tables tbeg, dw/dr per depth, bbeg).  Every depth's bitmap starts on an 8-word boundary;
// the rank array R holds one entry per 8-word chunk (set bits of all bitmaps before the chunk), so
// it is 1/8 of the bitmaps' size, and a node's rank is its chunk's entry plus the popcounts of the
// chunk's words before it.  Every rank is a difference of two R-based counts of the same scene,
// so modular uint32 arithmetic stays exact.
#include <algorithm>
#include <cstring>
#include <vector>
#include <string>

#include "svo_batch.hpp"
#include "svo_device.hpp"
#include "svo_runtime.hpp"
#include "svo_scan.hpp"

namespace svo {
namespace {

constexpr int kThreads = 256;
constexpr uint32_t kLdsBucket = 2048; // largest bucket sorted in LDS
constexpr uint32_t kRegBucket = 16;   // leaf blocks up to this size: one thread each (build_fold)
constexpr uint32_t kPairBucket = 32;  // up to this size: half a wave each (build_fold_lists)
constexpr uint32_t kWaveBucket = 64;  // up to this size: a wave each (build_fold_lists)
constexpr uint32_t kWideBucket = 512; // up to this size: one wave each, sorted in LDS (build_fold_lists)

// Effective voxel coordinate seen by the reference's descent: the coordinate's bits, saturating
// at res-1 for coordinates >= res (shader/octree_tag_node.comp:18-30).
__device__ __forceinline__ void decode_frag(uint2 fr, uint32_t res, uint32_t &x, uint32_t &y, uint32_t &z) {
	x = fr.x & 0xfffu;
	y = (fr.x >> 12u) & 0xfffu;
	z = (fr.x >> 24u) | ((fr.y >> 28u) << 8u);
	x = umin32(x, res - 1u);
	y = umin32(y, res - 1u);
	z = umin32(z, res - 1u);
}

// Every third bit, for 12-bit inputs (36-bit output).
__device__ __forceinline__ uint64_t spread3(uint32_t v) {
	uint64_t x = v & 0xfffu;
	x = (x | (x << 16)) & 0x0000FF0000FFull;
	x = (x | (x << 8)) & 0x00F00F00F00Full;
	x = (x | (x << 4)) & 0x0C30C30C30C3ull;
	x = (x | (x << 2)) & 0x249249249249ull;
	return x;
}

// Every third bit, for 10-bit inputs.
__device__ __forceinline__ uint32_t spread3_10(uint32_t x) {
	x = (x | x << 16) & 0x030000FFu;
	x = (x | x << 8) & 0x0300F00Fu;
	x = (x | x << 4) & 0x030C30C3u;
	return (x | x << 2) & 0x09249249u;
}

// Inclusive sum over the lanes of a wave, by data-parallel moves (no LDS).
__device__ __forceinline__ uint32_t wave_incl_sum(uint32_t v) {
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true); // row_shr 1
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true); // row_shr 2
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true); // row_shr 4
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true); // row_shr 8
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false); // lane 15 of a row to rows 1, 3
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false); // lane 31 to rows 2, 3
	return v;
}

// Morton code of a leaf: the child slots (x | y << 1 | z << 2) of depths 1..L, depth 1 highest.
__device__ __forceinline__ uint64_t morton(uint32_t x, uint32_t y, uint32_t z) {
	return spread3(x) | (spread3(y) << 1) | (spread3(z) << 2);
}

__device__ __forceinline__ uint64_t frag_key(uint2 f) { return ((uint64_t)f.x << 32) | f.y; }

// Set bits of the words of an 8-word chunk before word j (< 8), and word j (one 32-byte load).
__device__ __forceinline__ uint32_t chunk_before(const uint32_t *__restrict__ chunk, uint32_t j, uint32_t &word) {
	const uint4 *c = reinterpret_cast<const uint4 *>(chunk);
	const uint4 a = c[0], b = c[1];
	const uint32_t v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
	uint32_t r = 0u, cur = v[0];
#pragma unroll
	for (uint32_t t = 0; t < 8u; ++t) {
		r += t < j ? (uint32_t)__popc(v[t]) : 0u;
		cur = t == j ? v[t] : cur;
	}
	word = cur;
	return r;
}

// Set bits of the bitmaps before word w (a global word index) and the word itself: the rank of
// w's 8-word chunk plus the popcounts of the chunk's words before w.
__device__ __forceinline__ uint32_t bits_before(const uint32_t *__restrict__ B, const uint32_t *__restrict__ R,
                                                uint64_t w, uint32_t &word) {
	return R[w >> 3] + chunk_before(B + (w & ~7ull), (uint32_t)(w & 7u), word);
}

// Clears the bitmaps and the raw flags (one per scene, then one for all), and writes the batch's tables when they fit a kernel
// argument (words = 0: they are there already).
__global__ void __launch_bounds__(kThreads) bm_zero(uint32_t *B, uint64_t n, uint32_t *raw, uint32_t S, uint32_t *dst,
                                                    uint32_t words, SmallTable t) {
	if (blockIdx.x == 0u && threadIdx.x < words)
		dst[threadIdx.x] = t.w[threadIdx.x];
	const uint64_t stride = (uint64_t)gridDim.x * kThreads;
	for (uint64_t i = (uint64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride)
		B[i] = 0u;
	if (blockIdx.x == 0u)
		for (uint32_t s = threadIdx.x; s <= S; s += kThreads)
			raw[s] = 0u;
}

// Order of a leaf block's fragments in 32 bits: child slot | raw-coordinate flags | rgb.  The fold goes
// leaf by leaf in ascending fragment order, and the fragments of one leaf differ in their raw
// coordinates only where the descent saturates (res and above meet res - 1): at most one step above
// for a voxelized scene, so a flag per axis orders them as the packed words do (z's low byte, y, x;
// the low byte of res is below that of res - 1 from 2^8 on).  A raw coordinate above res (a list from
// the host, or a scene reaching out of the cube) does not fit, and neither do bits 24..27 of the second
// word, which the packing leaves unused but a list from the host may hold and the order counts: kRawKey,
// and its scene's keys become fragment indices (BuildSeg::raw), compared by the fragments they name.
constexpr uint32_t kRawKey = 0xFFFFFFFFu;

// x, y, z: the effective coordinates (decode_frag).  A raw coordinate exceeds its effective one by 1 where
// it saturates at res, by more above res.
__device__ __forceinline__ uint32_t leaf_key(uint2 f, uint32_t res, uint32_t x, uint32_t y, uint32_t z) {
	const uint32_t dx = (f.x & 0xfffu) - x, dy = ((f.x >> 12u) & 0xfffu) - y,
	               dz = ((f.x >> 24u) | ((f.y >> 28u) << 8u)) - z;
	const uint32_t slot = (x & 1u) | (y & 1u) << 1u | (z & 1u) << 2u;
	const uint32_t flags = dx | dy << 1u | (dz ^ (res >= 256u ? 1u : 0u)) << 2u;
	const uint32_t key = slot << 27u | flags << 24u | (f.y & 0xffffffu);
	return umax32(umax32(dx, dy), dz) > 1u || (f.y & 0x0f000000u) != 0u ? kRawKey : key;
}

// ---- tiles and runs ------------------------------------------------------------------------------
// Fragments come in raster order, so consecutive ones lie in few leaf blocks: a tile of kTile = 1024
// holds about 270 distinct ones (a room at 2^10; 160 for spheres at 2^9, 400 with random slivers at
// 2^12).  So a tile's fragments are grouped by leaf block once, into "runs", and everything that is
// random access happens per run: marking, rank lookups, bin counts, bucket places.  Per fragment only
// a 4-byte key moves, in tile order (whole lines) and from there to its bucket (a run at a time).
// Against marking, tagging and scattering whole fragments one by one (same order: room at 2^10 / slivers
// at 2^12 / 32 mixed scenes): 752 / 4688 / 2573 us -> 454 / 3804 / 1190 us for the three passes.  Larger
// tiles have hardly fewer runs (4096: -4%), and groups of tiles per XCD measured no different.
//   keys[t * kTile ..]   leaf_keys of tile t (or fragment indices), run after run
//   heads[t * 16 ..]     bit i: key i starts a run
//   runs[t * kTile ..]   per run {node P low, P's bit 32 << 31 | first key}, then {bin, place - first key}
//   nrun[t]              its runs
constexpr uint32_t kTile = 1024;
constexpr uint32_t kU = kTile / kThreads;
constexpr uint32_t kHeads = kTile / 64u;
constexpr uint32_t kLines = 256;    // LDS table: groups of 16 neighbouring nodes (2 bits of x, one of y and z)
constexpr uint32_t kLineStride = 9; // words of two counters per group, padded against bank conflicts
constexpr uint32_t kProbes = 32;
constexpr uint32_t kEmpty = 0xFFFFFFFFu;
static_assert(kLines == kThreads, "one thread per group in the scan");

// Home slot of a group in the tile's table: the low 3 bits of its Morton index (y0 z0 x0) under a hash of
// the rest.  So the groups of a 2x2x2 cube are neighbours in the table and their runs in the tile, and
// tag_runs counts them in common lines: room at 2^10 / slivers at 2^12 / 32 mixed scenes, tag_runs
// 132 / 1340 / 276 -> 102 / 1078 / 213 us, while bm_group pays 173 / 1351 / 493 -> 182 / 1460 / 517.  5 or 6
// Morton bits give tag_runs 3 us more and cost 8 here.
__device__ __forceinline__ uint32_t group_slot(uint32_t line) {
	const uint32_t rest = line & ~(1u | 1u << 9u | 1u << 19u);
	return ((rest * 2654435761u) >> 24u & (kLines - 8u)) | (line >> 9u & 1u) | (line >> 18u & 2u) | (line << 2u & 4u);
}

// One block per tile.  Every fragment finds its group of 16 nodes in an LDS hash table and takes a
// place in its node's counter; a scan over the counters turns them into offsets, so the runs come out
// group by group in Morton order inside (neighbouring lanes of tag_runs then count in one 64-byte
// line).  A fragment that finds no group in kProbes probes becomes a run of its own at the tile's end
// (random slivers at 2^12 touch 152 groups on average, 288 at most).  Each group marks its nodes with
// one load and, only if bits are missing, one atomic.  Bound by VALU issue (0.9 busy in a room) and LDS
// atomics, at 8 waves per SIMD.  35M fragments in a room / 180M with slivers at 2^12 / 100M of 32 mixed
// scenes: 192 / 1436 / 587 us, -> 180 / 1388 / 548 with packed sums, 32-bit Morton codes and scans by
// data-parallel moves, -> 173 / 1351 / 493 with the group read before the compare-and-swap
// (and see group_slot).  kIndex: a second pass (blocks of bm_write_blocks) that only rewrites the keys
// (and their order) of the raw scenes' tiles as fragment indices.
template <bool kIndex>
__device__ __forceinline__ void group_tile(const uint64_t tile, const BuildSeg *__restrict__ segs,
                                           const uint64_t *__restrict__ tbeg, uint32_t S, uint32_t *B,
                                           uint32_t *__restrict__ keys, uint64_t *__restrict__ heads,
                                           uint2 *__restrict__ runs, uint32_t *__restrict__ nrun, uint32_t *raw) {
	__shared__ uint32_t s_line[kLines], s_node[kLines]; // group key, Morton index of the group
	__shared__ uint32_t s_n[kLines * kLineStride];      // per node 16 bits: fragments, then the first key
	__shared__ uint32_t s_key[kTile];
	__shared__ uint32_t s_head[kTile / 32u], s_before[kTile / 32u];
	__shared__ uint32_t s_wave[kThreads / 64u], s_over;
	if (tile >= tbeg[S] || (kIndex && raw[S] == 0u))
		return;
	const uint32_t sc = S == 1u ? 0u : seg_find(tbeg, S, tile);
	const BuildSeg &g = segs[sc];
	if (kIndex && !g.raw)
		return; // block-uniform
	const uint32_t L = g.L, res = 1u << L;
	const uint64_t first = (tile - tbeg[sc]) * kTile;
	const uint32_t n = g.F - first < kTile ? (uint32_t)(g.F - first) : kTile;
	const uint2 *frags = g.frags + first;
	for (uint32_t i = threadIdx.x; i < kLines * kLineStride; i += kThreads)
		s_n[i] = 0u;
	s_line[threadIdx.x] = kEmpty;
	if (threadIdx.x < kTile / 32u)
		s_head[threadIdx.x] = 0u;
	if (threadIdx.x == 0u)
		s_over = 0u;
	uint2 fr[kU];
#pragma unroll
	for (uint32_t u = 0; u < kU; ++u) {
		const uint32_t i = threadIdx.x + u * kThreads;
		fr[u] = i < n ? frags[i] : make_uint2(0u, 0u);
	}
	__syncthreads();
	// counter of the fragment's node (group * 16 + node; kEmpty: a run of its own) and place in its run
	uint32_t at[kU], place[kU], key[kU];
	bool wide = false;
#pragma unroll
	for (uint32_t u = 0; u < kU; ++u) {
		at[u] = kEmpty;
		place[u] = 0u;
		if (threadIdx.x + u * kThreads >= n)
			continue;
		uint32_t x, y, z;
		decode_frag(fr[u], res, x, y, z);
		key[u] = leaf_key(fr[u], res, x, y, z);
		wide |= key[u] == kRawKey;
		const uint32_t line = (x >> 3u) | (y >> 2u) << 9u | (z >> 2u) << 19u;
		const uint32_t sub = (x >> 1u & 1u) | (y & 2u) | (z << 1u & 4u) | (x << 1u & 8u);
		uint32_t h = group_slot(line);
		for (uint32_t probe = 0; probe < kProbes; ++probe) {
			uint32_t old = __hip_atomic_load(&s_line[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
			if (old == kEmpty) // lanes of one group read in one go; atomics on one word go one after another
				old = atomicCAS(&s_line[h], kEmpty, line);
			if (old == kEmpty || old == line) {
				at[u] = h * 16u + sub;
				break;
			}
			h = (h + 1u) & (kLines - 1u);
		}
		const uint32_t sh = (sub & 1u) * 16u;
		place[u] = at[u] != kEmpty ? atomicAdd(&s_n[h * kLineStride + (sub >> 1u)], 1u << sh) >> sh & 0xffffu
		                           : atomicAdd(&s_over, 1u);
	}
	// only until the flag is seen: atomics on one address go one after another, and a wave in two may hold
	// such a fragment (3M fragments at 2^10, one in 100 raw: both passes 184 -> 80 us)
	if (!kIndex && __any(wide) && (threadIdx.x & 63u) == 0u &&
	    __hip_atomic_load(&raw[sc], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u) {
		atomicOr(&raw[sc], 1u);
		atomicOr(&raw[S], 1u);
	}
	__syncthreads();
	// first keys of the groups' nodes (thread h owns group h), marking
	uint32_t v[8], halves = 0u, mask = 0u;
#pragma unroll
	for (uint32_t c = 0; c < 8u; ++c) {
		v[c] = s_n[threadIdx.x * kLineStride + c];
		halves += v[c]; // a half sums up to kTile at most
		mask |= umin32(v[c] & 0xffffu, 1u) << (2u * c) | umin32(v[c] >> 16u, 1u) << (2u * c + 1u);
	}
	const uint32_t sum = (halves & 0xffffu) + (halves >> 16u);
	if (mask) {
		const uint32_t line = s_line[threadIdx.x];
		// the group's Morton index: the node's bits above the 4 of its place in the group (x0 y0 z0 x1)
		const uint32_t gn = spread3_10(line >> 9u & 0x3ffu) | spread3_10(line >> 19u & 0x3ffu) << 1u |
		                    spread3_10(line & 0x1ffu) << 2u;
		s_node[threadIdx.x] = gn;
		if (!kIndex && L > 1u) {
			uint32_t *word = B + g.bm + g.off[L - 1u] + (gn >> 1u);
			const uint32_t bits = mask << (16u * (gn & 1u));
			if ((*word & bits) != bits) // a stale cached word only costs a redundant atomic
				atomicOr(word, bits);
		}
	}
	const uint32_t incl = wave_incl_sum(sum);
	if ((threadIdx.x & 63u) == 63u)
		s_wave[threadIdx.x >> 6] = incl;
	__syncthreads();
	uint32_t run = incl - sum, grouped = 0u;
#pragma unroll
	for (uint32_t w = 0; w < kThreads / 64u; ++w) {
		run += w < (threadIdx.x >> 6) ? s_wave[w] : 0u;
		grouped += s_wave[w];
	}
	if (mask) {
#pragma unroll
		for (uint32_t c = 0; c < 8u; ++c) {
			const uint32_t next = run + (v[c] & 0xffffu);
			s_n[threadIdx.x * kLineStride + c] = run | next << 16u;
			run = next + (v[c] >> 16u);
		}
	}
	__syncthreads();
	// keys to their places, run heads
#pragma unroll
	for (uint32_t u = 0; u < kU; ++u) {
		const uint32_t i = threadIdx.x + u * kThreads;
		if (i >= n)
			continue;
		uint32_t p = grouped;
		if (at[u] != kEmpty)
			p = s_n[(at[u] >> 4u) * kLineStride + (at[u] >> 1u & 7u)] >> (at[u] & 1u) * 16u & 0xffffu;
		const bool head = at[u] == kEmpty || place[u] == 0u;
		p += place[u];
		s_key[p] = kIndex ? (uint32_t)(first + i) : key[u];
		if (head)
			atomicOr(&s_head[p >> 5u], 1u << (p & 31u));
		place[u] = head ? p : kEmpty; // from here on: the run's first key, at its head
	}
	__syncthreads();
	if (threadIdx.x < 64u) { // run heads before each 32 keys
		const uint32_t c = threadIdx.x < kTile / 32u ? (uint32_t)__popc(s_head[threadIdx.x]) : 0u;
		const uint32_t p = wave_incl_sum(c);
		if (threadIdx.x < kTile / 32u)
			s_before[threadIdx.x] = p - c;
		if (threadIdx.x == kTile / 32u - 1u)
			nrun[tile] = p;
	}
	for (uint32_t i = threadIdx.x; i < n; i += kThreads)
		keys[tile * kTile + i] = s_key[i];
	if (threadIdx.x < kHeads)
		heads[tile * kHeads + threadIdx.x] = (uint64_t)s_head[2u * threadIdx.x + 1u] << 32 | s_head[2u * threadIdx.x];
	__syncthreads();
#pragma unroll
	for (uint32_t u = 0; u < kU; ++u) {
		const uint32_t i = threadIdx.x + u * kThreads, p = place[u];
		if (i >= n || p == kEmpty)
			continue;
		const uint32_t r = s_before[p >> 5u] + (uint32_t)__popc(s_head[p >> 5u] & ((1u << (p & 31u)) - 1u));
		uint64_t P;
		if (at[u] != kEmpty) {
			P = (uint64_t)s_node[at[u] >> 4u] << 4 | (at[u] & 15u);
		} else {
			uint32_t x, y, z;
			decode_frag(frags[i], res, x, y, z);
			P = morton(x, y, z) >> 3;
			if (!kIndex && L > 1u)
				atomicOr(B + g.bm + g.off[L - 1u] + (P >> 5), 1u << (uint32_t)(P & 31u));
		}
		runs[tile * kTile + r] = make_uint2((uint32_t)P, (uint32_t)(P >> 32) << 31u | p);
	}
}

__global__ void __launch_bounds__(kThreads)
    bm_group(const BuildSeg *__restrict__ segs, const uint64_t *__restrict__ tbeg, uint32_t S, uint32_t *B,
             uint32_t *__restrict__ keys, uint64_t *__restrict__ heads, uint2 *__restrict__ runs,
             uint32_t *__restrict__ nrun, uint32_t *raw) {
	group_tile<false>(blockIdx.x, segs, tbeg, S, B, keys, heads, runs, nrun, raw);
}

// Bit q of B[d] = OR of byte q of B[d+1] (node q occupied iff one of its 8 children is); items are
// the words of B[d] of the scenes that have B[d+1] (begin table dr).  Word w of B[d] is made from
// chunk w of B[d+1], so the same thread also stores that chunk's set-bit count into R, which the
// rank scan then turns into ranks in place (the bitmaps are not read again for it).
__global__ void __launch_bounds__(kThreads)
    bm_reduce(const BuildSeg *__restrict__ segs, const uint64_t *__restrict__ dr, uint32_t S, uint64_t n, uint32_t d,
              uint32_t *B, uint32_t *R) {
	const uint64_t stride = (uint64_t)gridDim.x * kThreads;
	uint32_t hint = 0;
	for (uint64_t base = (uint64_t)blockIdx.x * kThreads; base < n; base += stride) {
		const uint64_t i = base + threadIdx.x;
		if (i >= n)
			continue;
		with_seg<kThreads>(dr, S, hint, base, i, [&](uint32_t s) {
			const BuildSeg &g = segs[s];
			const uint64_t w = i - dr[s];
			// the children of word w's 32 nodes: the 8-word chunk 8w of B[d+1] (B[d+1] is padded to
			// whole chunks; a padding word of a small B[d] may have no chunk)
			uint32_t bits = 0u;
			if (8u * w < g.off[d + 2u] - g.off[d + 1u]) {
				const uint4 *c = reinterpret_cast<const uint4 *>(B + g.bm + g.off[d + 1u] + 8u * w);
				const uint4 a = c[0], b = c[1];
				const uint32_t v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
				uint32_t pop = 0u;
#pragma unroll
				for (uint32_t k = 0; k < 8u; ++k) {
					uint32_t x = v[k] | (v[k] >> 4u); // bit 8q of x: byte q of v[k] is nonzero
					x |= x >> 2u;
					x |= x >> 1u;
					bits |= ((x & 1u) | ((x >> 7u) & 2u) | ((x >> 14u) & 4u) | ((x >> 21u) & 8u)) << (4u * k);
					pop += (uint32_t)__popc(v[k]);
				}
				R[((g.bm + g.off[d + 1u]) >> 3) + w] = pop;
			}
			B[g.bm + g.off[d] + w] = bits;
		});
	}
}

// The small depths d = min(L-2, kTopDepth) .. 1 of one scene per block: what one bm_reduce launch
// per depth does, with B[d] (at most 8^kTopDepth / 32 = 1024 words) kept in LDS from one depth to
// the next.  Also stores the set-bit count of B[1]'s one chunk (word 0; the padding words are zero)
// for every scene with L > 1.
constexpr uint32_t kTopDepth = 5;
constexpr uint32_t kTopWords = 1u << (3u * kTopDepth - 5u);

template <uint32_t kT> __device__ __forceinline__ void reduce_top(const BuildSeg &g, uint32_t *B, uint32_t *R) {
	__shared__ uint32_t s_b[2][kTopWords]; // B[d+1] of the previous depth, B[d]
	const uint32_t L = g.L;
	if (L <= 1u)
		return; // no bitmaps
	const uint32_t d0 = L - 2u < kTopDepth ? L - 2u : kTopDepth;
	uint32_t cur = 0u; // s_b[cur] holds B[d+1] below depth d0
	for (uint32_t d = d0; d >= 1u; --d) {
		const uint32_t nw = (uint32_t)(g.off[d + 1u] - g.off[d]);      // words of B[d], padded
		const uint32_t nc = (uint32_t)(g.off[d + 2u] - g.off[d + 1u]); // words of B[d+1], padded
		for (uint32_t w = threadIdx.x; w < nw; w += kT) {
			uint32_t bits = 0u;
			if (8u * w < nc) {
				uint32_t v[8];
				if (d == d0) {
					const uint4 *c = reinterpret_cast<const uint4 *>(B + g.bm + g.off[d + 1u] + 8u * w);
					const uint4 a = c[0], b = c[1];
					v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
				} else {
#pragma unroll
					for (uint32_t k = 0; k < 8u; ++k)
						v[k] = s_b[cur][8u * w + k];
				}
				uint32_t pop = 0u;
#pragma unroll
				for (uint32_t k = 0; k < 8u; ++k) {
					uint32_t x = v[k] | (v[k] >> 4u); // bit 8q of x: byte q of v[k] is nonzero
					x |= x >> 2u;
					x |= x >> 1u;
					bits |= ((x & 1u) | ((x >> 7u) & 2u) | ((x >> 14u) & 4u) | ((x >> 21u) & 8u)) << (4u * k);
					pop += (uint32_t)__popc(v[k]);
				}
				R[((g.bm + g.off[d + 1u]) >> 3) + w] = pop;
			}
			B[g.bm + g.off[d] + w] = bits;
			s_b[cur ^ 1u][w] = bits;
		}
		__syncthreads();
		cur ^= 1u;
	}
	if (threadIdx.x == 0u)
		R[g.bm >> 3] = (uint32_t)__popc(d0 >= 1u ? s_b[cur][0] : B[g.bm]);
}
__global__ void __launch_bounds__(kThreads) bm_reduce_top(const BuildSeg *__restrict__ segs, uint32_t *B, uint32_t *R) {
	reduce_top<kThreads>(segs[blockIdx.x], B, R);
}

// Set bits of 8-word chunk i, as stored by rank_top and bm_reduce.
struct ChunkCounts {
	static constexpr int kItems = 4;
	const uint32_t *R;
	uint64_t n; // chunks
	__device__ uint64_t size() const { return n; }
	__device__ uint32_t operator()(uint64_t i) const { return R[i]; }
};
struct RankTotal {
	uint32_t *R;
	uint64_t n;
	__device__ void operator()(uint64_t t) const { R[n] = (uint32_t)t; }
};
struct RankDst {
	uint32_t *R;
	__device__ bool active() const { return true; }
	__device__ void operator()(uint64_t i, uint64_t k, uint32_t) const { R[i] = (uint32_t)k; }
};

// Scene s: per-depth node counts -> first block of every depth (fb[0] = 0 is the root block, fb[1] = 1),
// the leaf blocks and W (src/OctreeBuilder.cpp:212-214: W = (counter + 1) * 8); also into the host's
// copy of the descriptors (out, pinned memory) when there is one.
struct Levels {
	BuildSeg *segs;
	uint32_t S;
	const uint32_t *R, *raw;
	uint64_t cap;
	BuildSeg *out;
	__device__ void scene(uint32_t s) const {
		BuildSeg &o = segs[s];
		const uint32_t L = o.L;
		const uint32_t *Rs = R + (o.bm >> 3); // every depth starts a chunk
		uint64_t first = 1;
		o.fb[0] = 0u;
		o.fb[1] = 1u;
		uint64_t nlast = 1; // nodes at depth L-1 (the root when L == 1)
		for (uint32_t d = 1; d < L; ++d) {
			const uint64_t nd = (uint32_t)(Rs[o.off[d + 1u] >> 3] - Rs[o.off[d] >> 3]);
			first += nd;
			o.fb[d + 1u] = (uint32_t)(first < 0xFFFFFFFFull ? first : 0xFFFFFFFFull);
			nlast = nd;
		}
		o.W = 8u * first;
		o.overflow = 8u * first > cap ? 1u : 0u;
		o.nbins = nlast;
		o.raw = raw[s];
		if (out)
			out[s] = o;
	}
	__device__ void operator()() const {
		if (threadIdx.x < S)
			scene(threadIdx.x);
	}
};
static_assert(kMaxBatch <= kOneThreads, "a scene per thread");
__global__ void bm_levels(Levels levels) {
	const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
	if (s < levels.S)
		levels.scene(s);
}
struct ReduceTop { // bm_reduce_top of a batch of one scene
	const BuildSeg *segs;
	uint32_t *B, *R;
	__device__ void operator()() const {
		reduce_top<kOneThreads>(segs[0], B, R);
		__threadfence_block(); // the scan reads R
	}
};

// The 8 words of the block of one depth-(d-1) parent: pointers to the blocks of its occupied
// children (bits of its byte in B[d]), zeros otherwise; r = rank of its first child among depth d.
__device__ __forceinline__ void store_parent_block(uint32_t *oct, uint64_t block, uint32_t byte, uint32_t fbd,
                                                   uint32_t r) {
	uint32_t wd[8];
#pragma unroll
	for (uint32_t t = 0; t < 8u; ++t) {
		const bool set = (byte >> t) & 1u;
		wd[t] = set ? (0x80000000u | ((fbd + r) << 3u)) : 0u;
		r += set ? 1u : 0u;
	}
	uint4 *dst = reinterpret_cast<uint4 *>(oct + 8u * block);
	dst[0] = make_uint4(wd[0], wd[1], wd[2], wd[3]);
	dst[1] = make_uint4(wd[4], wd[5], wd[6], wd[7]);
}

// Position of the n-th (from 0) set bit of v (n < popc(v)).
__device__ __forceinline__ uint32_t nth_bit(uint32_t v, uint32_t n) {
	uint32_t pos = 0u;
#pragma unroll
	for (uint32_t half = 16u; half >= 1u; half >>= 1) {
		const uint32_t c = (uint32_t)__popc(v & ((1u << half) - 1u));
		if (n >= c) {
			n -= c;
			pos += half;
			v >>= half;
		}
	}
	return pos;
}

// Blocks of every depth d >= 2 (the children of depth-(d-1) nodes), in one launch: every occupied
// parent's block (the parent's rank among depth d-1) is written whole.  Items are the words of
// B[d-1] of the scenes with L > d, depth after depth (begin table pw: segment k = (d - 2) S + s), so
// the scan covers the parents' bitmaps, 8x smaller than the children's.  A wave whose 64 words lie
// in one segment works cooperatively: the lanes' popcounts are prefix-summed, and lane k of each
// round writes the wave's k-th occupied parent, so every lane has work and the 64 blocks of a round
// are contiguous.  A wave across a segment boundary walks each word's set bits in its own lane.
// Block 0 also writes the root block of every scene with L > 1 (its 8 words point to the depth-1
// blocks of the occupied children, the bits of B[1]).  The same launch clears the nb leaf-block
// counters of tag_runs and the three counts of the fold's work lists.  All that by the first `grid`
// blocks; with kGroup (a scene may be raw) the others group the raw scenes' tiles again, which depends
// on nothing here: as a launch of its own that costs every plan replay 2 us.
template <bool kGroup>
__global__ void __launch_bounds__(kThreads)
    bm_write_blocks(const BuildSeg *__restrict__ segs, const uint64_t *__restrict__ pw, uint32_t M, uint32_t S,
                    const uint32_t *__restrict__ B, const uint32_t *__restrict__ R, uint32_t *cnt,
                    const uint64_t *__restrict__ nbp, uint32_t *list, uint32_t grid, const uint64_t *__restrict__ tbeg,
                    uint32_t scenes, uint32_t *__restrict__ keys, uint64_t *__restrict__ heads,
                    uint2 *__restrict__ runs, uint32_t *__restrict__ nrun, uint32_t *raw) {
	if (kGroup && blockIdx.x >= grid) {
		group_tile<true>(blockIdx.x - grid, segs, tbeg, scenes, nullptr, keys, heads, runs, nrun, raw);
		return;
	}
	const uint64_t n = pw[M], nb = *nbp;
	const uint32_t lane = threadIdx.x & 63u;
	const uint64_t stride = (uint64_t)grid * kThreads;
	for (uint64_t i = (uint64_t)blockIdx.x * kThreads + threadIdx.x; i < nb; i += stride)
		cnt[i] = 0u;
	if (blockIdx.x == 0u) {
		if (threadIdx.x < 3u)
			list[threadIdx.x] = 0u;
		for (uint32_t s = threadIdx.x; s < S; s += kThreads) {
			const BuildSeg &g = segs[s];
			if (g.L > 1u) // L == 1: the root block holds the leaves (build_fold)
				store_parent_block(g.words, 0u, B[g.bm + g.off[1]] & 0xffu, g.fb[1], 0u);
		}
	}
	// the 64 words from w0 on of segment ku, word w0 + lane being v
	auto wave_words = [&](uint32_t ku, uint64_t w0, uint32_t v) {
		const uint32_t d = 2u + ku / S;
		const BuildSeg &g = segs[ku % S];
		const uint64_t offp = g.bm + g.off[d - 1u], offc = g.bm + g.off[d]; // both start chunks
		const uint32_t c = (uint32_t)__popc(v);
		if (__ballot(v != 0u) == 0ull)
			return; // most waves of a sparse level
		const uint32_t incl = wave_incl_sum(c), excl = incl - c;
		const uint32_t T = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
		uint32_t first = 0u; // rank of the wave's first parent among depth d-1
		if (lane == 0u) {
			uint32_t dummy;
			first = bits_before(B, R, offp + w0, dummy) - R[offp >> 3];
		}
		const uint64_t blk0 = (uint64_t)g.fb[d - 1u] + __shfl(first, 0, 64);
		const uint32_t fbd = g.fb[d];
		// children of depth d before this word's 8-word chunk of B[d] (read only for occupied
		// words: an empty padding word of a small B[d-1] may have no chunk)
		const uint32_t rc = v != 0u ? R[(offc >> 3) + w0 + lane] - R[offc >> 3] : 0u;
		for (uint32_t t0 = 0; t0 < T; t0 += 64u) {
			const uint32_t j = t0 + lane; // the wave's j-th occupied parent
			uint32_t o = 0u; // owner lane: the last with excl <= j
#pragma unroll
			for (uint32_t step = 32u; step >= 1u; step >>= 1) {
				const uint32_t e = __shfl(excl, (int)(o + step), 64);
				o = e <= j ? o + step : o;
			}
			const uint32_t vo = __shfl(v, (int)o, 64), eo = __shfl(excl, (int)o, 64), ro = __shfl(rc, (int)o, 64);
			if (j < T) {
				const uint32_t b = nth_bit(vo, j - eo); // the parent's bit in the owner's word
				uint32_t cv; // the owner's chunk of B[d]: its word b / 4 holds the parent's byte
				const uint32_t before = chunk_before(B + offc + 8u * (w0 + o), b >> 2u, cv);
				const uint32_t sh = 8u * (b & 3u);
				const uint32_t r = ro + before + (uint32_t)__popc(cv & ((1u << sh) - 1u));
				store_parent_block(g.words, blk0 + j, (cv >> sh) & 0xffu, fbd, r);
			}
		}
	};
	// word i of segment k
	auto lane_word = [&](uint32_t k, uint64_t i) {
		const uint32_t d = 2u + k / S;
		const BuildSeg &g = segs[k % S];
		const uint64_t w = i - pw[k];
		const uint64_t offp = g.bm + g.off[d - 1u], offc = g.bm + g.off[d]; // both start chunks
		uint32_t v;
		const uint32_t rp = bits_before(B, R, offp + w, v);
		if (v == 0u)
			return;
		const uint32_t fbd = g.fb[d];
		uint64_t block = (uint64_t)g.fb[d - 1u] + (rp - R[offp >> 3]); // first parent's block
		// the 32 parents' children bytes are the 8-word chunk offc + 8w; parents not in v have zero
		// bytes, so a running count gives every child its rank
		const uint4 *cc = reinterpret_cast<const uint4 *>(B + offc + 8u * w);
		const uint4 c0 = cc[0], c1 = cc[1];
		uint32_t r = R[(offc >> 3) + w] - R[offc >> 3];
		while (v) {
			const uint32_t b = (uint32_t)__ffs(v) - 1u, j = b >> 2u;
			v &= v - 1u;
			uint32_t cv = c0.x;
			cv = j == 1u ? c0.y : cv;
			cv = j == 2u ? c0.z : cv;
			cv = j == 3u ? c0.w : cv;
			cv = j == 4u ? c1.x : cv;
			cv = j == 5u ? c1.y : cv;
			cv = j == 6u ? c1.z : cv;
			cv = j == 7u ? c1.w : cv;
			const uint32_t byte = (cv >> (8u * (b & 3u))) & 0xffu;
			store_parent_block(g.words, block, byte, fbd, r);
			r += (uint32_t)__popc(byte);
			++block;
		}
	};
	// A wave takes 256 words at a time, four loads in flight, where the grid has that many for every wave:
	// most words of a large batch or level are empty, and their waves only wait for the load (32 mixed
	// scenes 296 -> 131 us, slivers at 2^12 758 -> 729).  Else 64, which spreads the occupied words (room at
	// 2^10 34 us, 82 with 256).
	constexpr uint32_t kV = 4;
	const uint32_t per = n >= kV * stride ? kV : 1u;
	uint32_t hint = 0;
	for (uint64_t base = (uint64_t)blockIdx.x * kThreads * per; base < n; base += stride * per) {
		const uint64_t i0 = base + (uint64_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * 64u * per;
		if (i0 >= n)
			continue; // wave-uniform
		uint32_t k0 = 0u;
		with_seg<kThreads * kV>(pw, M, hint, base, i0, [&](uint32_t t) { k0 = t; });
		k0 = __builtin_amdgcn_readfirstlane(k0);
		if (i0 + 64u * per <= pw[k0 + 1u]) {
			const uint64_t w0 = i0 - pw[k0];
			const uint32_t *words = B + segs[k0 % S].bm + segs[k0 % S].off[1u + k0 / S] + w0 + lane;
			uint32_t v[kV] = {words[0], 0u, 0u, 0u};
			if (per == kV) {
#pragma unroll
				for (uint32_t q = 1; q < kV; ++q)
					v[q] = words[64u * q];
			}
#pragma unroll 1
			for (uint32_t q = 0; q < per; ++q)
				wave_words(k0, w0 + 64u * q, q == 0u ? v[0] : q == 1u ? v[1] : q == 2u ? v[2] : v[3]);
			continue;
		}
#pragma unroll 1
		for (uint32_t q = 0; q < per; ++q) { // a segment ends here
			const uint64_t i = i0 + 64u * q + lane;
			const uint32_t k = i < n ? seg_walk(pw, M, hint, i) : kEmpty;
			const uint32_t first = __builtin_amdgcn_readfirstlane(k);
			if (first == kEmpty)
				break; // the wave is past the end (lane 0 holds its first item)
			if (__all(k == first || k == kEmpty)) {
				const uint64_t w0 = (i - lane) - pw[first];
				const BuildSeg &g = segs[first % S];
				wave_words(first, w0, k != kEmpty ? B[g.bm + g.off[1u + first / S] + w0 + lane] : 0u);
			} else if (k != kEmpty) {
				lane_word(k, i);
			}
		}
	}
}

// Leaf block ("bin") of every run: the rank of its depth-(L-1) node, offset by the scene's first bin, and
// the run's place in the bin's bucket, from per-bin counters.  A wave takes a tile's runs 64 at a time;
// neighbouring lanes hold neighbouring nodes, so their counters share 64-byte lines and the L1 sends
// one request per line (device-coherent atomics are done at the memory side, and each request stalls
// the L2 for the reads behind it).  Bound by those requests, 17 a nanosecond: 9.4M runs of a room make
// 1.76M of them and take 102 us.
__global__ void __launch_bounds__(kThreads)
    tag_runs(const BuildSeg *__restrict__ segs, const uint64_t *__restrict__ tbeg, uint32_t S,
             const uint32_t *__restrict__ B, const uint32_t *__restrict__ R, uint2 *__restrict__ runs,
             const uint32_t *__restrict__ nrun, uint32_t *cnt) {
	constexpr uint32_t kPer = kThreads / 64u, kV = 4; // tiles per block, runs per lane and trip
	const uint32_t lane = threadIdx.x & 63u;
	const uint64_t tile = (uint64_t)blockIdx.x * kPer + (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	if (tile >= tbeg[S])
		return;
	const uint32_t sc = S == 1u ? 0u : seg_find(tbeg, S, tile);
	const BuildSeg &g = segs[sc];
	const uint64_t w0 = g.bm + (g.L > 1u ? g.off[g.L - 1u] : 0u); // the depth's first word starts a chunk
	const uint32_t bin0 = (uint32_t)g.bin_begin - (g.L > 1u ? R[w0 >> 3] : 0u);
	const uint64_t first = (tile - tbeg[sc]) * kTile;
	const uint32_t keys = g.F - first < kTile ? (uint32_t)(g.F - first) : kTile, n = nrun[tile];
	uint2 *rt = runs + tile * kTile;
	for (uint32_t i0 = 0; i0 < n; i0 += 64u * kV) {
		uint32_t bin[kV], len[kV];
		uint2 r[kV];
		uint32_t end[kV];
#pragma unroll
		for (uint32_t v = 0; v < kV; ++v) {
			const uint32_t i = i0 + v * 64u + lane;
			r[v] = i < n ? rt[i] : make_uint2(0u, 0u);
			end[v] = i + 1u < n ? rt[i + 1u].y : keys;
		}
#pragma unroll
		for (uint32_t v = 0; v < kV; ++v) {
			bin[v] = bin0;
			len[v] = (end[v] & 0x7fffffffu) - (r[v].y & 0x7fffffffu);
			if (g.L > 1u && i0 + v * 64u + lane < n) {
				const uint64_t P = (uint64_t)(r[v].y >> 31u) << 32 | r[v].x;
				uint32_t word;
				bin[v] += bits_before(B, R, w0 + (P >> 5), word);
				bin[v] += (uint32_t)__popc(word & ((1u << (uint32_t)(P & 31u)) - 1u));
			}
		}
#pragma unroll
		for (uint32_t v = 0; v < kV; ++v)
			if (i0 + v * 64u + lane < n)
				r[v] = make_uint2(bin[v], atomicAdd(&cnt[bin[v]], len[v]) - (r[v].y & 0x7fffffffu));
#pragma unroll
		for (uint32_t v = 0; v < kV; ++v)
			if (i0 + v * 64u + lane < n)
				rt[i0 + v * 64u + lane] = r[v];
	}
}

// Every key to its place in its bin's bucket (aux[j] = first slot of bin j), a wave per tile.  The wave
// first turns the tile's runs into slots in LDS, with the keys already on their way, so a tile costs
// three dependent loads; then lane i finds key i's run by the heads at or below it, and the lanes of a
// run write neighbouring slots.  Bound by latency and part-line writes: 35M keys in 122 us (190 us with
// every lane loading its key's run and bin offset itself).
__global__ void __launch_bounds__(kThreads)
    scatter_runs(const BuildSeg *__restrict__ segs, const uint64_t *__restrict__ tbeg, uint32_t S,
                 const uint32_t *__restrict__ keys, const uint64_t *__restrict__ heads,
                 const uint2 *__restrict__ runs, const uint32_t *__restrict__ nrun, const uint32_t *__restrict__ aux,
                 uint32_t *__restrict__ bucket) {
	constexpr uint32_t kPer = kThreads / 64u, kV = 4; // tiles per block, runs per lane and trip
	__shared__ uint32_t s_slot[kPer][kTile];          // run r: slot of key i of the run, less i
	const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const uint64_t upto = (2ull << lane) - 1ull; // heads at or below the lane
	const uint64_t tile = (uint64_t)blockIdx.x * kPer + wave;
	if (tile >= tbeg[S])
		return; // no block barrier follows
	const uint32_t sc = S == 1u ? 0u : seg_find(tbeg, S, tile);
	const uint64_t first = (tile - tbeg[sc]) * kTile, F = segs[sc].F;
	const uint32_t n = F - first < kTile ? (uint32_t)(F - first) : kTile, nr = nrun[tile];
	const uint2 *rt = runs + tile * kTile;
	const uint64_t *ht = heads + tile * kHeads;
	uint32_t *slot = s_slot[wave];
	uint32_t key[kHeads];
#pragma unroll
	for (uint32_t v = 0; v < kHeads; ++v)
		key[v] = v * 64u + lane < n ? keys[tile * kTile + v * 64u + lane] : 0u;
	for (uint32_t i0 = 0; i0 < nr; i0 += 64u * kV) {
		uint2 r[kV];
		uint32_t a[kV];
#pragma unroll
		for (uint32_t v = 0; v < kV; ++v)
			r[v] = i0 + v * 64u + lane < nr ? rt[i0 + v * 64u + lane] : make_uint2(0u, 0u);
#pragma unroll
		for (uint32_t v = 0; v < kV; ++v)
			a[v] = i0 + v * 64u + lane < nr ? aux[r[v].x] : 0u;
#pragma unroll
		for (uint32_t v = 0; v < kV; ++v)
			if (i0 + v * 64u + lane < nr)
				slot[i0 + v * 64u + lane] = a[v] + r[v].y;
	}
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
	uint32_t before = 0u; // runs that start before these 64 keys
#pragma unroll
	for (uint32_t v = 0; v < kHeads; ++v) {
		const uint32_t i = v * 64u + lane;
		const uint64_t h = ht[v]; // the last tile's heads are zero past its end
		if (i < n)
			bucket[slot[before + (uint32_t)__popcll(h & upto) - 1u] + i] = key[v];
		before += (uint32_t)__popcll(h);
	}
}

// The leaf a fragment key belongs to inside its block (child slot at depth L).
__device__ __forceinline__ uint32_t key_slot(uint64_t key, uint32_t res) {
	uint32_t x, y, z;
	decode_frag(make_uint2((uint32_t)(key >> 32), (uint32_t)key), res, x, y, z);
	return (x & 1u) | ((y & 1u) << 1u) | ((z & 1u) << 2u);
}

__device__ __forceinline__ void store_block(uint32_t *oct, uint64_t block, const uint32_t (&w)[8]) {
	uint4 *dst = reinterpret_cast<uint4 *>(oct + 8u * block);
	dst[0] = make_uint4(w[0], w[1], w[2], w[3]);
	dst[1] = make_uint4(w[4], w[5], w[6], w[7]);
}

// Work lists of leaf blocks too large for build_fold: list[0..2] = mid, big and wide counts; mid
// blocks (17..64 fragments) at list[3 ..], big ones (> 512) at list[3 + cap ..], wide ones
// (65..512) at list[3 + 2 cap ..] (each list holds at most Ftot / 17).  The mid list is long, and atomics on
// one address go one after another (12 ns each): the block appends to it once a step, 57,000 -> 14,000
// atomics and build_fold 712 -> 452 us for 32 mixed scenes.  This is for the big and wide ones: every
// lane of the wave calls it (the appends are aggregated per wave).
__device__ __forceinline__ void push_bins(uint32_t *list, uint64_t cap, uint32_t j, bool wide, bool big) {
	const uint32_t qb = wave_append(&list[1], big), qw = wave_append(&list[2], wide);
	if (big && qb < cap)
		list[3u + cap + qb] = j;
	if (wide && qw < cap)
		list[3u + 2u * cap + qw] = j;
}

// Octree block of global leaf block j (scene s): the scene's first leaf block + j's rank.
struct LeafTarget {
	uint32_t *oct;
	uint64_t block;
	uint32_t res;
	const uint2 *raw; // a raw scene's fragments, else null
};
__device__ __forceinline__ LeafTarget leaf_target(const BuildSeg &g, const uint64_t *bbeg, uint32_t s, uint32_t j) {
	const uint32_t L = g.L;
	return LeafTarget{g.words, (uint64_t)(L == 1u ? 0u : g.fb[L - 1u]) + (j - bbeg[s]), 1u << L, g.raw ? g.frags : nullptr};
}

__device__ __forceinline__ void cmp_swap(uint32_t &x, uint32_t &y) {
	const uint32_t lo = umin32(x, y), hi = umax32(x, y);
	x = lo;
	y = hi;
}
__device__ __forceinline__ void cmp_swap(uint64_t &x, uint64_t &y) {
	const bool less = y < x;
	const uint64_t lo = less ? y : x, hi = less ? x : y;
	x = lo;
	y = hi;
}

// The reference's running average of one leaf (octree_tag_node.comp:43-57), channels as floats: the
// n-th fragment (from 0, weight min(n, 63)) gives floor((avg * n + c) / (n + 1)).  The numerator is below
// 2^14 and the divisor at most 64, so (numerator + 1/2) / divisor is at least 1/128 away from an
// integer, and a reciprocal off by a few ulp gives the exact floor.
struct LeafMean {
	float r, g, b, n;
	__device__ __forceinline__ void clear() { r = g = b = n = 0.0f; }
	__device__ __forceinline__ void add(uint32_t rgb) {
		const float w = n + 1.0f, inv = __builtin_amdgcn_rcpf(w), half = 0.5f * inv;
		r = __builtin_floorf(__builtin_fmaf(__builtin_fmaf(r, n, (float)(rgb & 0xffu)), inv, half));
		g = __builtin_floorf(__builtin_fmaf(__builtin_fmaf(g, n, (float)(rgb >> 8u & 0xffu)), inv, half));
		b = __builtin_floorf(__builtin_fmaf(__builtin_fmaf(b, n, (float)(rgb >> 16u & 0xffu)), inv, half));
		n = __builtin_fminf(w, 63.0f);
	}
	__device__ __forceinline__ void load(uint32_t word) { // a leaf's word, or 0
		r = (float)(word & 0xffu);
		g = (float)(word >> 8u & 0xffu);
		b = (float)(word >> 16u & 0xffu);
		n = (float)(word >> 24u & 0x3fu);
	}
	__device__ __forceinline__ uint32_t word() const {
		uint32_t v = __builtin_amdgcn_cvt_pk_u8_f32(r, 0u, 0u);
		v = __builtin_amdgcn_cvt_pk_u8_f32(g, 1u, v);
		v = __builtin_amdgcn_cvt_pk_u8_f32(b, 2u, v);
		return __builtin_amdgcn_cvt_pk_u8_f32(n + 192.0f, 3u, v); // 0xC0 | n
	}
};

// Ascending sort of 4, 8 or 16 keys in registers (5, 19 or 63 comparators).
template <uint32_t kN, class Key> __device__ __forceinline__ void sort_small(Key (&k)[kN]) {
	if (kN == 4) {
		cmp_swap(k[0], k[1]), cmp_swap(k[2], k[3]), cmp_swap(k[0], k[2]), cmp_swap(k[1], k[3]);
		cmp_swap(k[1], k[2]);
	} else if (kN == 8) {
		cmp_swap(k[0], k[1]), cmp_swap(k[2], k[3]), cmp_swap(k[4], k[5]), cmp_swap(k[6], k[7]);
		cmp_swap(k[0], k[2]), cmp_swap(k[1], k[3]), cmp_swap(k[4], k[6]), cmp_swap(k[5], k[7]);
		cmp_swap(k[1], k[2]), cmp_swap(k[5], k[6]), cmp_swap(k[0], k[4]), cmp_swap(k[3], k[7]);
		cmp_swap(k[1], k[5]), cmp_swap(k[2], k[6]);
		cmp_swap(k[1], k[4]), cmp_swap(k[3], k[6]);
		cmp_swap(k[2], k[4]), cmp_swap(k[3], k[5]);
		cmp_swap(k[3], k[4]);
	} else { // Batcher odd-even merge sort of 16
		cmp_swap(k[0], k[1]), cmp_swap(k[2], k[3]), cmp_swap(k[0], k[2]), cmp_swap(k[1], k[3]);
		cmp_swap(k[1], k[2]), cmp_swap(k[4], k[5]), cmp_swap(k[6], k[7]), cmp_swap(k[4], k[6]);
		cmp_swap(k[5], k[7]), cmp_swap(k[5], k[6]), cmp_swap(k[0], k[4]), cmp_swap(k[2], k[6]);
		cmp_swap(k[2], k[4]), cmp_swap(k[1], k[5]), cmp_swap(k[3], k[7]), cmp_swap(k[3], k[5]);
		cmp_swap(k[1], k[2]), cmp_swap(k[3], k[4]), cmp_swap(k[5], k[6]), cmp_swap(k[8], k[9]);
		cmp_swap(k[10], k[11]), cmp_swap(k[8], k[10]), cmp_swap(k[9], k[11]), cmp_swap(k[9], k[10]);
		cmp_swap(k[12], k[13]), cmp_swap(k[14], k[15]), cmp_swap(k[12], k[14]), cmp_swap(k[13], k[15]);
		cmp_swap(k[13], k[14]), cmp_swap(k[8], k[12]), cmp_swap(k[10], k[14]), cmp_swap(k[10], k[12]);
		cmp_swap(k[9], k[13]), cmp_swap(k[11], k[15]), cmp_swap(k[11], k[13]), cmp_swap(k[9], k[10]);
		cmp_swap(k[11], k[12]), cmp_swap(k[13], k[14]), cmp_swap(k[0], k[8]), cmp_swap(k[4], k[12]);
		cmp_swap(k[4], k[8]), cmp_swap(k[2], k[10]), cmp_swap(k[6], k[14]), cmp_swap(k[6], k[10]);
		cmp_swap(k[2], k[4]), cmp_swap(k[6], k[8]), cmp_swap(k[10], k[12]), cmp_swap(k[1], k[9]);
		cmp_swap(k[5], k[13]), cmp_swap(k[5], k[9]), cmp_swap(k[3], k[11]), cmp_swap(k[7], k[15]);
		cmp_swap(k[7], k[11]), cmp_swap(k[3], k[5]), cmp_swap(k[7], k[9]), cmp_swap(k[11], k[13]);
		cmp_swap(k[1], k[2]), cmp_swap(k[3], k[4]), cmp_swap(k[5], k[6]), cmp_swap(k[7], k[8]);
		cmp_swap(k[9], k[10]), cmp_swap(k[11], k[12]), cmp_swap(k[13], k[14]);
	}
}

// A leaf block of a raw scene (keys = fragment indices): whole fragments sorted in registers, each folded
// into its leaf's word in w (one word per child slot, stride kThreads, 0 before).  Takes more registers
// than the keys do, so build_fold<true> is a launch of its own, made when a scene may be raw.  Bound
// by the gather of the fragments: 157,700 triangles of a room reaching half out of the cube at 2^10
// 1245 -> 165 us for both launches, 3M fragments at 2^10 458 -> 48 us, 100,000 at 2^6 260 -> 21 us, against
// repeated minima over the bucket in the one kernel, which fetch every fragment again for each.
template <uint32_t kN>
__device__ __forceinline__ void fold_whole(const uint32_t *b, const uint2 *frags, uint32_t n, uint32_t res, uint32_t *w) {
	uint64_t k[kN];
#pragma unroll
	for (uint32_t a = 0; a < kN; ++a)
		k[a] = a < n ? frag_key(frags[b[a]]) : ~0ull;
	sort_small<kN>(k);
#pragma unroll
	for (uint32_t a = 0; a < kN; ++a)
		if (a < n) {
			uint32_t *leaf = w + key_slot(k[a], res) * kThreads;
			LeafMean mean;
			mean.load(*leaf);
			mean.add((uint32_t)k[a]);
			*leaf = mean.word();
		}
}

// One thread per leaf block with at most 16 fragments: leaf_keys sorted in registers (5-, 19- or
// 63-comparator networks of v_min / v_max, +inf padding), then folded in that order, each leaf's word
// going to the thread's LDS column; the whole block is written, empty leaves as 0.  Each block of
// threads first orders its 256 leaf blocks by size class in LDS, so that most waves run a single
// network; the next 256 sizes and bucket positions are loaded a step ahead.  kRaw: the blocks of raw
// scenes (fold_whole), else all others and the lists.  Bound by the latency of its loads (7 waves per
// SIMD): 7.2M leaf blocks of a room at 2^10 279 -> 133 us, 62M with slivers at 2^12 1578 -> 893 us, against
// whole fragments, 64-bit comparators, leaf words in registers and integer division.  Staging the
// buckets in LDS instead of each thread reading its own: 192 and 1211 us.
template <uint32_t kN> __device__ __forceinline__ void fold_small(const uint32_t *b, uint32_t n, uint32_t *w) {
	uint32_t k[kN];
#pragma unroll
	for (uint32_t a = 0; a < kN; ++a)
		k[a] = a < n ? b[a] : kRawKey;
	sort_small<kN>(k);
	LeafMean leaf;
	leaf.clear();
	uint32_t slot = 8u;
#pragma unroll
	for (uint32_t a = 0; a < kN; ++a)
		if (a < n) {
			const uint32_t s = k[a] >> 27u;
			if (s != slot)
				leaf.clear();
			slot = s;
			leaf.add(k[a]);
			w[s * kThreads] = leaf.word();
		}
}

template <bool kRaw>
__global__ void __launch_bounds__(kThreads, kRaw ? 5 : 7)
    build_fold(const BuildSeg *__restrict__ segs, const uint64_t *__restrict__ bbeg, uint32_t S,
               const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ aux, const uint32_t *__restrict__ bucket,
               const uint32_t *__restrict__ raw, uint32_t *list, uint64_t cap) {
	if (kRaw && raw[S] == 0u)
		return;
	const uint64_t nbins = bbeg[S];
	constexpr uint32_t kWaves = kThreads / 64;
	__shared__ uint32_t s_bin[kThreads], s_n[kThreads];
	__shared__ uint32_t s_cls[kWaves][5], s_mid;
	__shared__ uint32_t s_leaf[8 * kThreads]; // the threads' leaf words, by child slot
	__shared__ uint32_t s_at[kThreads];       // first slot of the bin's bucket
	const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
	const uint64_t below = (1ull << lane) - 1ull;
	const uint64_t stride = (uint64_t)gridDim.x * kThreads;
	uint32_t hint = 0, next_n = 0u, next_slot = 0u; // loaded one step ahead
	auto ahead = [&](uint64_t at) {
		if (at + threadIdx.x < nbins) {
			next_n = cnt[at + threadIdx.x];
			next_slot = aux[at + threadIdx.x];
		}
	};
	ahead((uint64_t)blockIdx.x * kThreads);
	for (uint64_t base = (uint64_t)blockIdx.x * kThreads; base < nbins; base += stride) {
		const uint64_t jj = base + threadIdx.x;
		const uint32_t n = next_n, slot0 = next_slot;
		uint32_t cls = 5; // classes: <= 4, <= 8, <= 16 fragments; for the mid list <= 32, <= 64; 5 = neither
		if (base + stride < nbins)
			ahead(base + stride);
		if (jj < nbins) {
			cls = n <= 4u ? 0u : n <= 8u ? 1u : n <= kRegBucket ? 2u : n <= kPairBucket ? 3u : n <= kWaveBucket ? 4u : 5u;
		}
		if constexpr (!kRaw) {
			const bool rest = jj < nbins && cls == 5u;
			push_bins(list, cap, (uint32_t)jj, rest && n <= kWideBucket, rest && n > kWideBucket);
		}
		uint64_t mine = 0u; // the wave's lanes of the same class
#pragma unroll
		for (uint32_t c = 0; c < 5u; ++c) {
			const uint64_t m = __ballot(cls == c);
			mine = cls == c ? m : mine;
			if (lane == c)
				s_cls[wave][c] = (uint32_t)__popcll(m);
		}
		__syncthreads();
		uint32_t pos = 0, total = 0, mids = 0;
#pragma unroll
		for (uint32_t c = 0; c < 5u; ++c)
#pragma unroll
			for (uint32_t v = 0; v < kWaves; ++v) {
				const uint32_t k = s_cls[v][c];
				pos += (c < cls || (c == cls && v < wave)) ? k : 0u;
				(c < 3u ? total : mids) += k;
			}
		pos += (uint32_t)__popcll(mine & below);
		uint32_t first = 0u; // of the step's places in the mid list; used after the fold
		if (!kRaw && threadIdx.x == 0u && mids)
			first = atomicAdd(&list[0], mids);
		if (cls < 3u) {
			s_bin[pos] = (uint32_t)jj;
			s_n[pos] = n;
			s_at[pos] = slot0;
		}
		__syncthreads();
		if (threadIdx.x < total) {
			const uint32_t j = s_bin[threadIdx.x], nj = s_n[threadIdx.x];
			LeafTarget t;
			with_seg<kThreads>(bbeg, S, hint, base, j, [&](uint32_t s) { t = leaf_target(segs[s], bbeg, s, j); });
			if ((t.raw != nullptr) == kRaw) {
				uint32_t *w = s_leaf + threadIdx.x;
#pragma unroll
				for (uint32_t c = 0; c < 8u; ++c)
					w[c * kThreads] = 0u;
				const uint32_t *b = bucket + s_at[threadIdx.x];
				if (nj <= 4u)
					kRaw ? fold_whole<4>(b, t.raw, nj, t.res, w) : fold_small<4>(b, nj, w);
				else if (nj <= 8u)
					kRaw ? fold_whole<8>(b, t.raw, nj, t.res, w) : fold_small<8>(b, nj, w);
				else
					kRaw ? fold_whole<16>(b, t.raw, nj, t.res, w) : fold_small<16>(b, nj, w);
				uint32_t words[8];
#pragma unroll
				for (uint32_t c = 0; c < 8u; ++c)
					words[c] = w[c * kThreads];
				store_block(t.oct, t.block, words);
			}
		}
		if (threadIdx.x == 0u)
			s_mid = first;
		__syncthreads();
		if (!kRaw && (cls == 3u || cls == 4u) && s_mid + pos - total < cap)
			list[3u + s_mid + pos - total] = (uint32_t)jj;
	}
}

// Index pair (a, b), a < b, of comparator t at distance jj of a bitonic merge to k, in the form whose
// comparators all put the minimum at the lower index, so keys past the end behave as +infinity padding.
__device__ __forceinline__ void bitonic_pair(uint32_t t, uint32_t k, uint32_t jj, uint32_t &a, uint32_t &b) {
	const uint32_t blk = t / jj, off = t % jj;
	const bool flip = jj == (k >> 1); // first step of a merge
	a = flip ? blk * k + off : blk * 2u * jj + off;
	b = flip ? blk * k + k - 1u - off : a + jj;
}

// Folds keys [beg, end) of one leaf, ascending; rgb(i) = colour of key i.
template <class Rgb> __device__ __forceinline__ uint32_t fold_run(uint32_t beg, uint32_t end, Rgb rgb) {
	if (beg >= end)
		return 0u;
	LeafMean leaf;
	leaf.clear();
	for (uint32_t i = beg; i < end; ++i)
		leaf.add(rgb(i));
	return leaf.word();
}

// xor-shuffle by a power of two inside the wave: data-parallel moves where they reach, else LDS permutes.
template <uint32_t kD> __device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
	if constexpr (kD == 1u)
		return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xf, 0xf, true); // quad_perm 1 0 3 2
	else if constexpr (kD == 2u)
		return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xf, 0xf, true); // quad_perm 2 3 0 1
	else if constexpr (kD <= 16u)
		return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, (int)(kD << 10 | 0x1fu)); // xor within 32 lanes
	else
		return (uint32_t)__shfl_xor((int)v, (int)kD, 64);
}
// Steps d = kD .. 1 of a bitonic merge: bit[b] is all ones in the lanes with bit b of their id set, dir
// likewise in the lanes that sort downwards.  The median of (own, other, 0 or ~0) is their minimum or
// maximum, so a step is an exclusive or, a move and a v_med3.
template <uint32_t kB> __device__ __forceinline__ void wave_merge(uint32_t &key, const uint32_t (&bit)[6], uint32_t dir) {
	const uint32_t other = lane_xor<1u << kB>(key), bound = dir ^ bit[kB];
	key = umax32(umin32(key, other), umin32(umax32(key, other), bound));
	if constexpr (kB > 0u)
		wave_merge<kB - 1u>(key, bit, dir);
}
// Ascending bitonic sort of the keys of each half wave, or of the wave.
template <bool kHalves> __device__ __forceinline__ void wave_sort(uint32_t &key, const uint32_t (&bit)[6]) {
	wave_merge<0>(key, bit, bit[1]);
	wave_merge<1>(key, bit, bit[2]);
	wave_merge<2>(key, bit, bit[3]);
	wave_merge<3>(key, bit, bit[4]);
	wave_merge<4>(key, bit, kHalves ? 0u : bit[5]);
	if constexpr (!kHalves)
		wave_merge<5>(key, bit, 0u);
}

// Leaf blocks of 17..64 fragments: a wave takes 8 at a time (bins, n, at: numbers, sizes and bucket
// positions, `count` of them), sorts one after another (two side by side up to 32 fragments) so that every
// leaf's fragments are consecutive and ascending, and then folds the 64 leaves, one per lane.  A raw
// scene's block sorts (slot, whole fragment) pairs.  col: 8 x 64 words of LDS; t: where leaf block
// lane / 8 goes.  Bound by VALU: one block per wave, its runs folded by 8 lanes, and a step of the sort as
// an LDS permute, a minimum, a maximum and a select took 520 us for the listed blocks of 32 mixed scenes
// (100M fragments), this takes 150.
__device__ __forceinline__ void fold_mid(const uint32_t *n, const uint32_t *at, uint32_t count, uint32_t *col,
                                         const uint32_t *__restrict__ bucket, const LeafTarget &t) {
	const uint32_t lane = threadIdx.x & 63u, leaf = lane & 7u, mine = lane >> 3;
	const uint64_t raws = __ballot(t.raw != nullptr);
	uint32_t bit[6];
#pragma unroll
	for (uint32_t b = 0; b < 6u; ++b)
		bit[b] = 0u - (lane >> b & 1u);
	uint32_t beg = 0u, len = 0u;
	// the keys of one block are in the wave (sorted; lanes past its end: no slot): colours to LDS, run of
	// each leaf to its lane
	auto runs = [&](uint32_t item, uint32_t key, uint32_t slot) {
		col[item * 64u + lane] = key & 0xffffffu;
#pragma unroll
		for (uint32_t u = 0; u < 8u; ++u) {
			const uint64_t m = __ballot(slot == u);
			if (mine == item && leaf == u) {
				beg = m ? (uint32_t)__ffsll((unsigned long long)m) - 1u : 0u;
				len = (uint32_t)__popcll(m);
			}
		}
	};
#pragma unroll 1
	for (uint32_t i = 0; i < count; i += 2u) {
		const bool two = i + 1u < count;
		const uint32_t n0 = (uint32_t)__builtin_amdgcn_readfirstlane(n[i]),
		               n1 = two ? (uint32_t)__builtin_amdgcn_readfirstlane(n[i + 1u]) : 0u;
		const bool raw0 = raws >> (8u * i) & 1u, raw1 = two && (raws >> (8u * i + 8u) & 1u);
		if (umax32(n0, n1) <= kPairBucket && !raw0 && !raw1) {
			const uint32_t half = lane >> 5, l = lane & 31u, item = i + half;
			const bool have = l < (half ? n1 : n0);
			uint32_t key = have ? bucket[at[item] + l] : kRawKey;
			wave_sort<true>(key, bit);
			const uint32_t slot = key >> 27u;
			col[(i + half) * 64u + l] = key & 0xffffffu;
#pragma unroll
			for (uint32_t u = 0; u < 8u; ++u) {
				const uint64_t both = __ballot(slot == u);
				const uint32_t m = (mine & 1u) ? (uint32_t)(both >> 32) : (uint32_t)both;
				if ((mine & ~1u) == i && leaf == u) {
					beg = m ? (uint32_t)__ffs((int)m) - 1u : 0u;
					len = (uint32_t)__popc(m);
				}
			}
			continue;
		}
#pragma unroll 1
		for (uint32_t k = 0; k < (two ? 2u : 1u); ++k) {
			const uint32_t item = i + k, ni = k ? n1 : n0;
			uint32_t key = lane < ni ? bucket[at[item] + lane] : kRawKey;
			if (!(k ? raw1 : raw0)) {
				wave_sort<false>(key, bit);
				runs(item, key, key >> 27u);
				continue;
			}
			const uint32_t res = (uint32_t)__shfl((int)t.res, (int)(8u * item), 64);
			const uint2 *frags = reinterpret_cast<const uint2 *>(
			    __shfl((unsigned long long)reinterpret_cast<uintptr_t>(t.raw), (int)(8u * item), 64));
			uint64_t whole = ~0ull;
			uint32_t slot = 8u;
			if (lane < ni) {
				whole = frag_key(frags[key]);
				slot = key_slot(whole, res);
			}
#pragma unroll 1
			for (uint32_t q = 2; q <= 64u; q <<= 1)
#pragma unroll 1
				for (uint32_t d = q >> 1; d > 0u; d >>= 1) {
					const uint64_t ok = __shfl_xor(whole, (int)d, 64);
					const uint32_t os = __shfl_xor(slot, (int)d, 64);
					const bool other_less = os < slot || (os == slot && ok < whole);
					const bool take_min = ((lane & q) == 0u) == ((lane & d) == 0u);
					const bool take_other = take_min == other_less;
					whole = take_other ? ok : whole;
					slot = take_other ? os : slot;
				}
			runs(item, (uint32_t)whole, slot);
		}
	}
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
	if (mine < count)
		t.oct[8u * t.block + leaf] = fold_run(beg, beg + len, [&](uint32_t i) { return col[mine * 64u + i]; });
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
}

// Leaf blocks of 17..64 fragments from the list, 8 per wave and trip.  Blocks blk of nblk of the list
// launch; s_col, s_item: 512 and 16 words of LDS per wave.
__device__ void fold_mid_blocks(uint32_t blk, uint32_t nblk, const BuildSeg *__restrict__ segs,
                                const uint64_t *__restrict__ bbeg, uint32_t S, const uint32_t *__restrict__ cnt,
                                const uint32_t *__restrict__ aux, const uint32_t *__restrict__ bucket,
                                const uint32_t *list, uint64_t cap, uint32_t *s_col, uint32_t *s_item) {
	constexpr uint32_t kWaves = kThreads / 64;
	const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
	uint32_t *n = s_item + wave * 16u, *at = n + 8u;
	uint64_t count = list[0];
	if (count > cap)
		count = cap;
	// up to 8 per wave; fewer where the list is short, so that more waves share it
	const uint64_t waves = (uint64_t)nblk * kWaves, share = (count + waves - 1u) / waves;
	const uint32_t take = share >= 8u ? 8u : share > 2u ? (uint32_t)(share + 1u) & ~1u : 2u;
	for (uint64_t base = take * ((uint64_t)blk * kWaves + wave); base < count; base += take * waves) {
		const uint32_t m = (uint32_t)(count - base < take ? count - base : take), mine = lane >> 3;
		const uint32_t j = list[3u + base + (mine < m ? mine : 0u)]; // of leaf block lane / 8
		if (mine < m && (lane & 7u) == 0u) {
			n[mine] = cnt[j];
			at[mine] = aux[j];
		}
		__builtin_amdgcn_wave_barrier();
		__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
		const uint32_t s = S == 1u ? 0u : seg_find(bbeg, S, j);
		fold_mid(n, at, m, s_col + wave * 512u, bucket, leaf_target(segs[s], bbeg, s, j));
	}
}

// Bitonic sort of n (<= m = 2^p) keys by kStep lanes (one wave, or the block); step(a, b) leaves the
// smaller of keys a and b at a, sync() separates the stages.
template <uint32_t kStep, class Step, class Sync>
__device__ __forceinline__ void bitonic(uint32_t n, uint32_t m, uint32_t lane, Step step, Sync sync) {
	for (uint32_t k = 2; k <= m; k <<= 1)
		for (uint32_t jj = k >> 1; jj > 0; jj >>= 1) {
			for (uint32_t q = lane; q < m / 2u; q += kStep) {
				uint32_t a, b;
				bitonic_pair(q, k, jj, a, b);
				if (b < n)
					step(a, b);
			}
			sync();
		}
}

template <class Key> __device__ __forceinline__ void order_keys(Key *keys, uint32_t x, uint32_t y) {
	const Key kx = keys[x], ky = keys[y];
	if (ky < kx)
		keys[x] = ky, keys[y] = kx;
}

// Sorts the n keys of one leaf block in LDS and finds the runs of its 8 leaves: s_beg / s_end[slot].
// keys32: leaf_keys (or, of a raw scene, fragment indices on entry); keys64, slots: a raw scene's
// whole fragments.  Called by kStep lanes.
template <uint32_t kStep, class Sync>
__device__ __forceinline__ void sort_leaves(uint32_t n, uint32_t lane, const LeafTarget &t,
                                            const uint32_t *__restrict__ b, uint64_t *keys64, uint8_t *slots,
                                            uint32_t *s_beg, uint32_t *s_end, Sync sync) {
	uint32_t *keys32 = reinterpret_cast<uint32_t *>(keys64);
	uint32_t m = 1u;
	while (m < n)
		m <<= 1;
	if (lane < 8u)
		s_beg[lane] = s_end[lane] = 0u;
	if (t.raw) {
		for (uint32_t i = lane; i < n; i += kStep) {
			const uint64_t key = frag_key(t.raw[b[i]]);
			keys64[i] = key;
			slots[i] = (uint8_t)key_slot(key, t.res);
		}
		sync();
		bitonic<kStep>(
		    n, m, lane,
		    [&](uint32_t x, uint32_t y) {
			    const uint64_t kx = keys64[x], ky = keys64[y];
			    const uint8_t sx = slots[x], sy = slots[y];
			    if (sy < sx || (sy == sx && ky < kx)) {
				    keys64[x] = ky, keys64[y] = kx;
				    slots[x] = sy, slots[y] = sx;
			    }
		    },
		    sync);
	} else {
		for (uint32_t i = lane; i < n; i += kStep)
			keys32[i] = b[i];
		sync();
		bitonic<kStep>(n, m, lane, [&](uint32_t x, uint32_t y) { order_keys(keys32, x, y); }, sync);
	}
	auto slot_of = [&](uint32_t i) { return t.raw ? (uint32_t)slots[i] : keys32[i] >> 27u; };
	for (uint32_t i = lane; i < n; i += kStep) {
		const uint32_t sl = slot_of(i);
		if (i == 0u || slot_of(i - 1u) != sl)
			s_beg[sl] = i;
		if (i + 1u == n || slot_of(i + 1u) != sl)
			s_end[sl] = i + 1u;
	}
	sync();
	if (lane < 8u)
		t.oct[8u * t.block + lane] = fold_run(s_beg[lane], s_end[lane], [&](uint32_t i) {
			return (t.raw ? (uint32_t)keys64[i] : keys32[i]) & 0xffffffu;
		});
	sync();
}

// Leaf blocks of 65..512 fragments, one wave each, sorted in the wave's LDS (no block barriers: the
// wave's LDS accesses are ordered between stages by wave barriers).  Blocks blk of nblk of the list
// launch; s_keys / s_slots: kWideBucket entries per wave.
__device__ void fold_wide_blocks(uint32_t blk, uint32_t nblk, const BuildSeg *__restrict__ segs,
                                 const uint64_t *__restrict__ bbeg, uint32_t S, const uint32_t *__restrict__ cnt,
                                 const uint32_t *__restrict__ aux, const uint32_t *__restrict__ bucket,
                                 const uint32_t *list, uint64_t cap, uint64_t *s_keys, uint8_t *s_slots,
                                 uint32_t (*s_beg)[8], uint32_t (*s_end)[8]) {
	constexpr uint32_t kWaves = kThreads / 64;
	const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
	uint64_t count = list[2];
	if (count > cap)
		count = cap;
	for (uint64_t base = (uint64_t)blk * kWaves; base < count; base += (uint64_t)nblk * kWaves) {
		const uint64_t item = base + wave;
		if (item >= count)
			break; // wave-uniform; no block barrier follows
		const uint32_t j = list[3u + 2u * cap + item];
		const uint32_t s = S == 1u ? 0u : seg_find(bbeg, S, j);
		const LeafTarget t = leaf_target(segs[s], bbeg, s, j);
		sort_leaves<64u>(cnt[j], lane, t, bucket + aux[j], s_keys + wave * kWideBucket, s_slots + wave * kWideBucket,
		                 s_beg[wave], s_end[wave], [] {
			                 __builtin_amdgcn_wave_barrier();
			                 __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
		                 });
	}
}

// Leaf blocks of more than 512 fragments, one block each.  Up to kLdsBucket fragments: sorted in LDS.
// Beyond (rare): the keys are sorted in place in the bucket and each of 8 lanes folds its slot's run;
// a raw scene's whole fragments are sorted in spare (8 bytes per bucket entry), and each lane walks all
// of them, taking those of its slot.  Blocks blk of nblk of the list launch; s_keys / s_slots:
// kLdsBucket entries for the block.
__device__ void fold_big_blocks(uint32_t blk, uint32_t nblk, const BuildSeg *__restrict__ segs,
                                const uint64_t *__restrict__ bbeg, uint32_t S, const uint32_t *__restrict__ cnt,
                                const uint32_t *__restrict__ aux, uint32_t *bucket, uint64_t *spare,
                                const uint32_t *list, uint64_t cap, uint64_t *s_keys, uint8_t *s_slots,
                                uint32_t *s_beg, uint32_t *s_end) {
	uint64_t count = list[1];
	if (count > cap)
		count = cap;
	for (uint64_t item = blk; item < count; item += nblk) {
		const uint32_t j = list[3u + cap + item];
		const uint32_t n = cnt[j];
		const uint32_t s = S == 1u ? 0u : seg_find(bbeg, S, j);
		const LeafTarget t = leaf_target(segs[s], bbeg, s, j);
		uint32_t *b = bucket + aux[j];
		if (n <= kLdsBucket) {
			sort_leaves<kThreads>(n, threadIdx.x, t, b, s_keys, s_slots, s_beg, s_end, [] { __syncthreads(); });
		} else {
			uint32_t m = 1;
			while (m < n)
				m <<= 1;
			uint64_t *whole = spare + aux[j]; // a raw scene's
			if (t.raw) {
				for (uint32_t i = threadIdx.x; i < n; i += kThreads)
					whole[i] = frag_key(t.raw[b[i]]);
				__syncthreads();
			}
			if (t.raw)
				bitonic<kThreads>(
				    n, m, threadIdx.x, [&](uint32_t x, uint32_t y) { order_keys(whole, x, y); }, [] { __syncthreads(); });
			else
				bitonic<kThreads>(
				    n, m, threadIdx.x, [&](uint32_t x, uint32_t y) { order_keys(b, x, y); }, [] { __syncthreads(); });
			if (threadIdx.x < 8u && !t.raw) {
				auto first = [&](uint32_t key) { // index of the first key not below
					uint32_t lo = 0u, hi = n;
					while (lo < hi) {
						const uint32_t mid = lo + (hi - lo) / 2u;
						lo = b[mid] < key ? mid + 1u : lo;
						hi = b[mid] < key ? hi : mid;
					}
					return lo;
				};
				const uint32_t beg = first(threadIdx.x << 27u), end = first((threadIdx.x + 1u) << 27u);
				t.oct[8u * t.block + threadIdx.x] = fold_run(beg, end, [&](uint32_t i) { return b[i]; });
			} else if (threadIdx.x < 8u) {
				LeafMean leaf;
				leaf.clear();
				bool any = false;
				for (uint32_t i = 0; i < n; ++i) {
					const uint64_t key = whole[i];
					if (key_slot(key, t.res) == threadIdx.x) {
						leaf.add((uint32_t)key);
						any = true;
					}
				}
				t.oct[8u * t.block + threadIdx.x] = any ? leaf.word() : 0u;
			}
		}
		__syncthreads();
	}
}

// The fold's three work lists in one launch: blocks [0, g_mid) take the 17..64-fragment leaf blocks,
// the next g_wide the 65..512-fragment ones, the rest the larger ones.  Each role is block-uniform,
// so the big role's block barriers are safe; the LDS is shared between the roles.
__global__ void __launch_bounds__(kThreads)
    build_fold_lists(const BuildSeg *__restrict__ segs, const uint64_t *__restrict__ bbeg, uint32_t S,
                     const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ aux, uint32_t *bucket,
                     uint64_t *spare, const uint32_t *list, uint64_t cap, uint32_t g_mid, uint32_t g_wide) {
	constexpr uint32_t kWaves = kThreads / 64;
	static_assert(kWaves * kWideBucket == kLdsBucket, "the wide and big roles share the key arrays");
	__shared__ uint64_t s_keys[kLdsBucket];
	__shared__ uint8_t s_slots[kLdsBucket];
	__shared__ uint32_t s_beg[kWaves][8], s_end[kWaves][8], s_item[kWaves * 16];
	if (blockIdx.x < g_mid)
		fold_mid_blocks(blockIdx.x, g_mid, segs, bbeg, S, cnt, aux, bucket, list, cap,
		                reinterpret_cast<uint32_t *>(s_keys), s_item);
	else if (blockIdx.x < g_mid + g_wide)
		fold_wide_blocks(blockIdx.x - g_mid, g_wide, segs, bbeg, S, cnt, aux, bucket, list, cap, s_keys, s_slots, s_beg,
		                 s_end);
	else
		fold_big_blocks(blockIdx.x - g_mid - g_wide, gridDim.x - g_mid - g_wide, segs, bbeg, S, cnt, aux, bucket,
		                spare, list, cap, s_keys, s_slots, s_beg[0], s_end[0]);
}

// ---- scan plumbing for the bin offsets ---------------------------------------------------------
struct BinCounts {
	static constexpr int kItems = 4;
	const uint32_t *cnt;
	const uint64_t *n; // the batch's leaf blocks, in device memory (bbeg[S])
	__device__ uint64_t size() const { return *n; }
	__device__ uint32_t operator()(uint64_t i) const { return cnt[i]; }
};
struct BinOffsets {
	uint32_t *aux;
	__device__ bool active() const { return true; }
	__device__ void operator()(uint64_t i, uint64_t k, uint32_t) const { aux[i] = (uint32_t)k; }
};

// Blocks for a grid-stride loop over items (kThreads per block and trip), at most per_cu per CU:
// more blocks than the CU holds at once keep more loads in flight (64 per CU measured best for
// most passes; kernels that set up an LDS table per block want fewer, pure streams more).
uint32_t grid_for(uint64_t items, svo_ctx *ctx, uint32_t per_cu = 64u) {
	uint64_t g = (items + kThreads - 1) / kThreads;
	const uint64_t cap = (uint64_t)ctx->cu_count * per_cu;
	if (g > cap)
		g = cap;
	return (uint32_t)(g ? g : 1);
}

// Word offsets of B[1..L-1] inside one scene's bitmaps; off[L] = the scene's bitmap words.  Every
// depth starts an 8-word rank chunk (the padding words stay zero).
void levels_for(uint32_t L, uint64_t *off) {
	uint64_t o = 0;
	for (uint32_t d = 1; d <= L; ++d) {
		off[d] = o;
		if (d < L) {
			const uint64_t bits = 1ull << (3u * d);
			o += ((bits < 32u ? 1u : bits / 32u) + 7u) & ~7ull;
		}
	}
}

uint64_t big_capacity(uint64_t F) { return F / (kRegBucket + 1u) + 1u; }

// tiles: whole tiles of F fragments; the tile arrays of `tiles` tiles, one allocation.
uint64_t tiles_of(uint64_t F) { return (F + kTile - 1u) / kTile; }
hipError_t alloc_tiles(Pool *pool, BuildBatch &bb) {
	const uint64_t t = bb.tiles ? bb.tiles : 1u;
	const hipError_t e = pool->alloc((void **)&bb.runs, t * (kTile * (sizeof(uint2) + sizeof(uint32_t)) +
	                                                         kHeads * sizeof(uint64_t) + sizeof(uint32_t)));
	bb.heads = reinterpret_cast<uint64_t *>(bb.runs + t * kTile);
	bb.keys = reinterpret_cast<uint32_t *>(bb.heads + t * kHeads);
	bb.nrun = bb.keys + t * kTile;
	return e;
}

// tables: the batch's, to be written first (nullptr: they are in place); out: pinned copy of the
// descriptors for the host, or nullptr.
int structure_phase(svo_ctx *ctx, BuildBatch &bb, const std::vector<uint8_t> *tables, BuildSeg *out) {
	const uint32_t S = bb.S;
	hipError_t e;
	const size_t bytes = tables ? tables->size() : 0;
	const bool small = bytes > 0 && SmallTable::fits(bytes);
	if (bytes > 0 && !small)
		if (int rc = upload_table(ctx, bb.segs, tables->data(), bytes))
			return rc;
	static_assert(kThreads >= SmallTable::kWords, "a word per thread");
	if ((e = launch(ctx, "bm_zero", bm_zero, dim3(grid_for(bb.TW, ctx)), dim3(kThreads), 0, bb.bm, bb.TW, bb.raw, S,
	                reinterpret_cast<uint32_t *>(bb.segs), small ? (uint32_t)(bytes / 4u) : 0u,
	                small ? SmallTable(tables->data(), bytes) : SmallTable())) != hipSuccess)
		return hip_check(ctx, e, "bm_zero");
	if (bb.tiles > 0 && (e = launch(ctx, "bm_group", bm_group, dim3((uint32_t)bb.tiles), dim3(kThreads), 0,
	                                (const BuildSeg *)bb.segs, bb.tbeg(), S, bb.bm, bb.keys, bb.heads, bb.runs,
	                                bb.nrun, bb.raw)) != hipSuccess)
		return hip_check(ctx, e, "bm_group");
	const Levels levels{bb.segs, S, bb.rk, bb.raw, 1ull << 30, out};
	if (bb.TW > 0) {
		for (uint32_t d = bb.maxL >= 3 ? bb.maxL - 2 : 0; d > kTopDepth; --d) {
			const uint64_t n = bb.h_index[(3 + kMaxLevel + d) * (uint64_t)(S + 1) + S];
			if (n > 0 && (e = launch(ctx, "bm_reduce", bm_reduce, dim3(grid_for(n, ctx)), dim3(kThreads), 0,
			                         (const BuildSeg *)bb.segs, bb.index + (3 + kMaxLevel + d) * (uint64_t)(S + 1), S, n,
			                         d, bb.bm, bb.rk)) != hipSuccess)
				return hip_check(ctx, e, "bm_reduce");
		}
		// exclusive scan of the chunk counts, in place (each item is read and written by one thread)
		const ChunkCounts src{bb.rk, bb.TW / 8u};
		const RankDst dst{bb.rk};
		const RankTotal total{bb.rk, bb.TW / 8u};
		const bool one = src.n <= kScanOne;
		if (one && S == 1u) {
			e = launch(ctx, "rank", scan_one<ChunkCounts, RankDst, RankTotal, ReduceTop, Levels>, dim3(1),
			           dim3(kOneThreads), 0, src, dst, total, ReduceTop{bb.segs, bb.bm, bb.rk}, levels);
			return e == hipSuccess ? SVO_OK : hip_check(ctx, e, "rank");
		}
		if ((e = launch(ctx, "bm_reduce_top", bm_reduce_top, dim3(S), dim3(kThreads), 0, (const BuildSeg *)bb.segs,
		                bb.bm, bb.rk)) != hipSuccess)
			return hip_check(ctx, e, "bm_reduce_top");
		if (one) {
			e = launch(ctx, "rank", scan_one<ChunkCounts, RankDst, RankTotal, NoStep, Levels>, dim3(1),
			           dim3(kOneThreads), 0, src, dst, total, NoStep{}, levels);
			return e == hipSuccess ? SVO_OK : hip_check(ctx, e, "rank");
		}
		if ((e = launch(ctx, "rank_reduce", scan_reduce<ChunkCounts>, dim3(kScanBlocks), dim3(kScanThreads), 0, src,
		                ctx->d_scan_parts)) != hipSuccess)
			return hip_check(ctx, e, "rank_reduce");
		if ((e = launch(ctx, "rank_down", scan_down<ChunkCounts, RankDst, RankTotal>, dim3(kScanBlocks),
		                dim3(kScanThreads), 0, src, dst, (const uint64_t *)ctx->d_scan_parts, total)) != hipSuccess)
			return hip_check(ctx, e, "rank_down");
	}
	if ((e = launch(ctx, "bm_levels", bm_levels, dim3(div_up(S, 64)), dim3(64), 0, levels)) != hipSuccess)
		return hip_check(ctx, e, "bm_levels");
	return SVO_OK;
}

// maybe_raw: a scene may be raw (a plan's replay cannot know): its tiles are grouped again, its leaf blocks
// folded by a launch of their own.
int node_phase(svo_ctx *ctx, BuildBatch &bb, bool maybe_raw) {
	const uint32_t S = bb.S;
	const BuildSeg *segs = bb.segs;
	hipError_t e;
	{
		// with maxL == 1 there are no parent words and no root blocks to write (the bitmaps are empty)
		const uint32_t M = bb.pw_segs();
		const uint64_t n = bb.maxL > 1u ? bb.h_index[bb.pw_at() + M] : 0u; // parent words of all depths >= 2
		const uint32_t grid = grid_for(std::max(n, bb.nbins), ctx);
		if ((e = launch(ctx, "bm_write_blocks", maybe_raw ? bm_write_blocks<true> : bm_write_blocks<false>,
		                dim3(grid + (maybe_raw ? (uint32_t)bb.tiles : 0u)), dim3(kThreads), 0, segs, bb.pw(), M,
		                bb.maxL > 1u ? S : 0u, (const uint32_t *)bb.bm, (const uint32_t *)bb.rk, bb.cnt,
		                bb.bbeg() + S, bb.list, grid, bb.tbeg(), S, bb.keys, bb.heads, bb.runs, bb.nrun,
		                bb.raw)) != hipSuccess)
			return hip_check(ctx, e, "bm_write_blocks");
	}
	const uint32_t gT = div_up(bb.tiles, kThreads / 64u);
	if (bb.tiles > 0 && (e = launch(ctx, "tag_runs", tag_runs, dim3(gT), dim3(kThreads), 0, segs, bb.tbeg(), S,
	                                (const uint32_t *)bb.bm, (const uint32_t *)bb.rk, bb.runs,
	                                (const uint32_t *)bb.nrun, bb.cnt)) != hipSuccess)
		return hip_check(ctx, e, "tag_runs");
	BinCounts bc{bb.cnt, bb.bbeg() + S};
	const BinOffsets offsets{bb.aux};
	if (bb.nbins <= kScanOne) {
		if ((e = launch(ctx, "bin_offsets", scan_one<BinCounts, BinOffsets, NoCommit, NoStep, NoStep>, dim3(1),
		                dim3(kOneThreads), 0, bc, offsets, NoCommit{}, NoStep{}, NoStep{})) != hipSuccess)
			return hip_check(ctx, e, "bin_offsets");
	} else if ((e = launch(ctx, "bin_reduce", scan_reduce<BinCounts>, dim3(kScanBlocks), dim3(kScanThreads), 0, bc,
	                       ctx->d_scan_parts)) != hipSuccess ||
	           (e = launch(ctx, "bin_offsets", scan_down<BinCounts, BinOffsets>, dim3(kScanBlocks), dim3(kScanThreads),
	                       0, bc, offsets, (const uint64_t *)ctx->d_scan_parts, NoCommit{})) != hipSuccess) {
		return hip_check(ctx, e, "bin_offsets");
	}
	if (bb.tiles > 0 && (e = launch(ctx, "scatter_runs", scatter_runs, dim3(gT), dim3(kThreads), 0, segs, bb.tbeg(), S,
	                                (const uint32_t *)bb.keys, (const uint64_t *)bb.heads, (const uint2 *)bb.runs,
	                                (const uint32_t *)bb.nrun, (const uint32_t *)bb.aux, bb.bucket)) != hipSuccess)
		return hip_check(ctx, e, "scatter_runs");
	const uint64_t cap = big_capacity(bb.Ftot);
	for (int raw = 0; raw <= (maybe_raw ? 1 : 0); ++raw)
		if ((e = launch(ctx, "build_fold", raw ? build_fold<true> : build_fold<false>, dim3(grid_for(bb.nbins, ctx)),
		                dim3(kThreads), 0, segs, bb.bbeg(), S, (const uint32_t *)bb.cnt, (const uint32_t *)bb.aux,
		                (const uint32_t *)bb.bucket, (const uint32_t *)bb.raw, bb.list, cap)) != hipSuccess)
			return hip_check(ctx, e, "build_fold");
	// the roles' loops take any number of blocks: no more than the fragments can fill with listed leaf
	// blocks (17, 65 and 513 fragments at least), a wave or a block each
	constexpr uint64_t kWaves = kThreads / 64u;
	const uint32_t cu = (uint32_t)ctx->cu_count;
	const uint32_t g_mid = (uint32_t)std::min<uint64_t>(cu * 8u, bb.Ftot / (17u * 2u * kWaves) + 1u),
	               g_wide = (uint32_t)std::min<uint64_t>(cu * 8u, bb.Ftot / (65u * kWaves) + 1u),
	               g_big = (uint32_t)std::min<uint64_t>(cu * 2u, bb.Ftot / 513u + 1u);
	if ((e = launch(ctx, "build_fold_lists", build_fold_lists, dim3(g_mid + g_wide + g_big), dim3(kThreads), 0, segs,
	                bb.bbeg(), S, (const uint32_t *)bb.cnt, (const uint32_t *)bb.aux, bb.bucket,
	                reinterpret_cast<uint64_t *>(bb.runs), (const uint32_t *)bb.list, cap, g_mid, g_wide)) != hipSuccess)
		return hip_check(ctx, e, "build_fold_lists");
	return SVO_OK;
}

} // namespace

uint64_t build_bitmap_words(uint32_t L) {
	uint64_t off[16] = {};
	levels_for(L, off);
	return off[L];
}

void build_batch_release(svo_ctx *ctx, BuildBatch *bb) {
	for (void *p : {(void *)bb->segs, (void *)bb->bm, (void *)bb->rk, (void *)bb->cnt, (void *)bb->aux,
	                (void *)bb->runs, (void *)bb->bucket, (void *)bb->list}) // index lives in segs' allocation
		ctx->pool->free(p);
	bb->segs = nullptr;
	bb->index = nullptr;
	bb->bm = bb->rk = bb->raw = bb->cnt = bb->aux = bb->keys = bb->nrun = bb->bucket = bb->list = nullptr;
	bb->runs = nullptr;
	bb->heads = nullptr;
}

namespace {

// Host layout of a build batch of S scenes with F[s] fragments at level L[s]: descriptors (bitmap
// offsets), tile begins, per-depth bitmap word tables and the block writer's parent words.
void batch_layout(BuildBatch &bb, uint32_t S, const uint2 *const *frags, const uint64_t *F, const uint32_t *L) {
	bb.S = S;
	bb.h_segs.assign(S, BuildSeg{});
	const uint64_t stride = S + 1;
	bb.h_index.assign(bb.pw_at() + bb.pw_segs() + 1, 0);
	uint64_t *tbeg = bb.h_index.data();
	for (uint32_t s = 0; s < S; ++s) {
		BuildSeg &g = bb.h_segs[s];
		g.frags = frags[s];
		g.F = F[s];
		g.L = L[s];
		g.bm = bb.TW;
		levels_for(g.L, g.off);
		bb.TW += g.off[g.L];
		tbeg[s] = bb.tiles;
		bb.tiles += tiles_of(g.F);
		bb.Ftot += g.F;
		bb.maxL = std::max(bb.maxL, g.L);
	}
	tbeg[S] = bb.tiles;
	// per-depth begin tables: dw[d] over scenes with B[d] (L > d), dr[d] over scenes with B[d+1] (L > d+1)
	for (uint32_t d = 1; d <= kMaxLevel; ++d) {
		uint64_t *dw = bb.h_index.data() + (2 + d) * stride, *dr = bb.h_index.data() + (3 + kMaxLevel + d) * stride;
		uint64_t aw = 0, ar = 0;
		for (uint32_t s = 0; s < S; ++s) {
			const BuildSeg &g = bb.h_segs[s];
			dw[s] = aw;
			dr[s] = ar;
			const uint64_t words = g.L > d ? g.off[d + 1] - g.off[d] : 0;
			aw += words;
			ar += g.L > d + 1 ? words : 0;
		}
		dw[S] = aw;
		dr[S] = ar;
	}
	// parent words of the block writer: B[d-1] of the scenes with L > d, for d = 2..kMaxLevel-1
	uint64_t *pw = bb.h_index.data() + bb.pw_at(), a = 0;
	for (uint32_t d = 2; d < kMaxLevel; ++d)
		for (uint32_t s = 0; s < S; ++s) {
			const BuildSeg &g = bb.h_segs[s];
			*pw++ = a;
			a += g.L > d ? g.off[d] - g.off[d - 1] : 0;
		}
	*pw = a;
}

// Descriptors and begin tables in one device allocation, so each upload is one copy.
size_t seg_table_bytes(uint32_t S) { return (sizeof(BuildSeg) * S + 255) & ~size_t(255); }

std::vector<uint8_t> batch_tables(const BuildBatch &bb) {
	const size_t seg_bytes = seg_table_bytes(bb.S), idx_bytes = sizeof(uint64_t) * bb.h_index.size();
	std::vector<uint8_t> tables(seg_bytes + idx_bytes);
	std::memcpy(tables.data(), bb.h_segs.data(), sizeof(BuildSeg) * bb.S);
	std::memcpy(tables.data() + seg_bytes, bb.h_index.data(), idx_bytes);
	return tables;
}

int upload_batch_tables(svo_ctx *ctx, const BuildBatch &bb) {
	const std::vector<uint8_t> tables = batch_tables(bb);
	return upload_table(ctx, bb.segs, tables.data(), tables.size());
}

} // namespace

// The whole build of S octrees: structure phase, one read-back of every scene's W and leaf-block
// count, allocation of the octrees, node phase.  Scratch goes back to the pool at the end; the pool
// hands it only to later work on this stream, so no wait is needed for the node phase to finish.
int build_batch(svo_ctx *ctx, svo_octree *const *octs, uint32_t S) {
	if (S == 0)
		return SVO_OK;
	if (S > kMaxBatch)
		return set_error(ctx, SVO_ERR_INVALID_ARGUMENT, "batch larger than 1024 scenes");
	BuildBatch bb;
	const uint64_t stride = S + 1;
	{
		std::vector<const uint2 *> frags(S);
		std::vector<uint64_t> F(S);
		std::vector<uint32_t> L(S);
		for (uint32_t s = 0; s < S; ++s) {
			const svo_fraglist *fl = octs[s]->src;
			frags[s] = reinterpret_cast<const uint2 *>(fl->frags);
			F[s] = fl->F;
			L[s] = fl->level;
		}
		batch_layout(bb, S, frags.data(), F.data(), L.data());
	}
	if (bb.Ftot > 0xFFFFFFFEull)
		return set_error(ctx, SVO_ERR_OVERFLOW, "a build batch holds at most 2^32-2 fragments; split the batch");
	const uint64_t Fa = bb.Ftot ? bb.Ftot : 1;
	const uint64_t cap = big_capacity(bb.Ftot);
	Pool *pool = ctx->pool;
	int rc = SVO_OK;
	const size_t seg_bytes = seg_table_bytes(S), idx_bytes = sizeof(uint64_t) * bb.h_index.size();
	if (pool->alloc((void **)&bb.segs, seg_bytes + idx_bytes) != hipSuccess ||
	    pool->alloc((void **)&bb.bm, sizeof(uint32_t) * (bb.TW ? bb.TW : 1)) != hipSuccess ||
	    pool->alloc((void **)&bb.rk, sizeof(uint32_t) * (bb.TW / 8u + 2 + S)) != hipSuccess ||
	    alloc_tiles(pool, bb) != hipSuccess || pool->alloc((void **)&bb.bucket, sizeof(uint32_t) * Fa) != hipSuccess ||
	    pool->alloc((void **)&bb.list, sizeof(uint32_t) * (3 + 3 * cap)) != hipSuccess)
		rc = set_error(ctx, SVO_ERR_OUT_OF_MEMORY, "octree build allocation failed");
	// structure phase: bitmaps + ranks decide every W exactly; one read-back sizes the octrees
	BuildSeg *out = nullptr;
	if (!rc && S <= kReadbackScenes && !(out = static_cast<BuildSeg *>(readback_slot(ctx, sizeof(BuildSeg) * S))))
		rc = SVO_ERR_INVALID_ARGUMENT;
	if (!rc) {
		bb.index = reinterpret_cast<uint64_t *>(reinterpret_cast<uint8_t *>(bb.segs) + seg_bytes);
		bb.raw = bb.rk + bb.TW / 8u + 1;
		const std::vector<uint8_t> tables = batch_tables(bb);
		ctx->t_build.start(ctx->stream);
		rc = structure_phase(ctx, bb, &tables, out);
		ctx->t_build.stop(ctx->stream);
	}
	if (!rc)
		rc = out ? readback_wait(ctx, bb.h_segs.data(), out, sizeof(BuildSeg) * S)
		         : download_table(ctx, bb.h_segs.data(), bb.segs, sizeof(BuildSeg) * S);
	if (!rc)
		for (uint32_t s = 0; s < S; ++s)
			if (bb.h_segs[s].overflow) {
				rc = set_error(ctx, SVO_ERR_OVERFLOW,
				               "octree " + std::to_string(s) + " needs more than 2^30 words (30-bit child pointers)");
				break;
			}
	uint64_t *bbeg = bb.h_index.data() + stride;
	if (!rc) {
		for (uint32_t s = 0; s < S; ++s) {
			BuildSeg &g = bb.h_segs[s];
			svo_octree *o = octs[s];
			o->W = o->cap = g.W; // (counter + 1) * 8, src/OctreeBuilder.cpp:212-214
			if (pool->alloc((void **)&o->words, sizeof(uint32_t) * g.W) != hipSuccess) {
				rc = set_error(ctx, SVO_ERR_OUT_OF_MEMORY, "octree allocation failed");
				break;
			}
			g.words = o->words;
			g.bin_begin = bb.nbins;
			bbeg[s] = bb.nbins;
			bb.nbins += g.nbins;
		}
		bbeg[S] = bb.nbins;
	}
	if (!rc && (pool->alloc((void **)&bb.cnt, sizeof(uint32_t) * (bb.nbins ? bb.nbins : 1)) != hipSuccess ||
	            pool->alloc((void **)&bb.aux, sizeof(uint32_t) * (bb.nbins ? bb.nbins : 1)) != hipSuccess))
		rc = set_error(ctx, SVO_ERR_OUT_OF_MEMORY, "octree build allocation failed");
	if (!rc)
		rc = upload_batch_tables(ctx, bb);
	if (!rc) {
		ctx->t_build2.start(ctx->stream);
		bool raw = false;
		for (const BuildSeg &g : bb.h_segs)
			raw |= g.raw != 0u;
		rc = node_phase(ctx, bb, raw);
		ctx->t_build2.stop(ctx->stream);
	}
	build_batch_release(ctx, &bb);
	return rc;
}

// ---- captured plans: voxelize + build of a fixed set of scenes with the counts kept on the device
namespace {

constexpr uint32_t kPlanThreads = kMaxBatch; // the check kernels take one scene per thread

// Exclusive prefix of one value per thread over the block; total = the sum.  Every thread calls it.
__device__ __forceinline__ uint64_t plan_excl(uint64_t v, uint64_t &total) {
	__shared__ uint64_t s_wave[kPlanThreads / 64];
	const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
	uint64_t incl = v;
#pragma unroll
	for (uint32_t d = 1; d < 64u; d <<= 1) {
		const uint64_t t = __shfl_up(incl, d, 64);
		incl += lane >= d ? t : 0u;
	}
	if (lane == 63u)
		s_wave[wave] = incl;
	__syncthreads();
	uint64_t below = 0;
	total = 0;
	for (uint32_t w = 0; w < kPlanThreads / 64; ++w) {
		below += w < wave ? s_wave[w] : 0u;
		total += s_wave[w];
	}
	return below + incl - v;
}

// Between the voxelize count and fill passes: the scenes' fragment counts become the build's
// tile begins.  A count above its list's capacity sets status bit 1 and empties the batch: fill limit
// and every tile begin 0, so no later pass reads or writes a list past its end.  Also restores the
// block writer's parent-word total, which the node check of the previous run may have cleared.
// out = {status, F[S], W[S]}.
__global__ void __launch_bounds__(kPlanThreads)
    plan_check_frags(const VoxSeg *__restrict__ vsegs, BuildSeg *bsegs, uint64_t *tbeg, uint32_t S,
                     const uint64_t *__restrict__ fcap, uint64_t *fend, uint64_t *pw_total, uint64_t pw_value,
                     uint64_t *out) {
	const uint32_t s = threadIdx.x;
	uint64_t F = 0, tiles;
	int over = 0;
	if (s < S) {
		F = vsegs[s].F;
		over = F > fcap[s];
		out[1u + s] = F;
		out[1u + S + s] = 0u;
		bsegs[s].F = F;
	}
	over = __syncthreads_or(over);
	const uint64_t first = plan_excl((F + kTile - 1u) / kTile, tiles);
	if (s < S)
		tbeg[s] = over ? 0u : first;
	if (s == 0u) {
		fend[1] = over ? 0u : fend[0];
		tbeg[S] = over ? 0u : tiles;
		*pw_total = pw_value;
		out[0] = over ? 1u : 0u;
	}
}

// Between the structure and node phases: leaf-block begins (an exclusive scan of the scenes' leaf
// blocks) and W against each octree's capacity.  A W above its capacity (or above 2^30 words), or
// a fragment overflow found before, sets status bit 2 and empties the node phase: leaf blocks,
// tiles and parent words 0, so it writes nothing but the root blocks.
__global__ void __launch_bounds__(kPlanThreads)
    plan_check_nodes(BuildSeg *segs, uint64_t *bbeg, uint32_t S, const uint64_t *__restrict__ wcap, uint64_t *tbeg,
                     uint64_t *pw_total, uint64_t *out) {
	const uint32_t s = threadIdx.x;
	uint64_t nb = 0;
	int over = 0;
	if (s < S) {
		const BuildSeg &g = segs[s];
		nb = g.nbins;
		over = g.overflow || g.W > wcap[s];
		out[1u + S + s] = g.W;
	}
	over = __syncthreads_or(over) || out[0] != 0u;
	uint64_t total;
	const uint64_t excl = plan_excl(nb, total);
	if (s < S) {
		segs[s].bin_begin = over ? 0u : excl;
		bbeg[s] = over ? 0u : excl;
	}
	if (s == 0u) {
		bbeg[S] = over ? 0u : total;
		if (over) {
			tbeg[S] = 0u;
			*pw_total = 0u;
			out[0] |= 2u;
		}
	}
}

// The plan's passes in stream order; nothing waits on the host, so the sequence can be captured.
int plan_enqueue(svo_ctx *ctx, BuildPlan &p) {
	BuildBatch &bb = p.bb;
	const uint32_t S = p.S;
	uint64_t *pw_total = bb.index + bb.pw_at() + bb.pw_segs();
	hipError_t e;
	if ((e = voxelize_plan_count(ctx, &p.vb)) != hipSuccess)
		return hip_check(ctx, e, "plan voxelize count");
	if ((e = launch(ctx, "plan_check_frags", plan_check_frags, dim3(1), dim3(kPlanThreads), 0,
	                (const VoxSeg *)p.vb.segs, bb.segs, bb.index, S, (const uint64_t *)p.caps, p.vb.fend, pw_total,
	                p.pw_value, p.out)) != hipSuccess)
		return hip_check(ctx, e, "plan_check_frags");
	if ((e = voxelize_plan_fill(ctx, &p.vb, p.bb.Ftot)) != hipSuccess)
		return hip_check(ctx, e, "plan voxelize fill");
	if (int rc = structure_phase(ctx, bb, nullptr, nullptr))
		return rc;
	if ((e = launch(ctx, "plan_check_nodes", plan_check_nodes, dim3(1), dim3(kPlanThreads), 0, bb.segs,
	                bb.index + (S + 1), S, (const uint64_t *)p.caps + S, bb.index, pw_total, p.out)) != hipSuccess)
		return hip_check(ctx, e, "plan_check_nodes");
	return node_phase(ctx, bb, true);
}

} // namespace

int build_plan_init(svo_ctx *ctx, BuildPlan *p, const svo_scene *const *scenes, const uint32_t *levels, uint32_t S,
                    const uint64_t *fcap, const uint64_t *wcap) {
	p->S = S;
	Pool *pool = ctx->pool;
	uint64_t Fcap = 0, Bcap = 0;
	std::vector<uint64_t> caps(2 * (size_t)S);
	for (uint32_t s = 0; s < S; ++s) {
		const uint32_t L = levels[s];
		caps[s] = fcap[s] ? fcap[s] : 1u;
		caps[S + s] = std::max<uint64_t>((wcap[s] + 7u) & ~7ull, 8u);
		if (caps[S + s] > (1ull << 30))
			return set_error(ctx, SVO_ERR_OVERFLOW, "an octree capacity above 2^30 words (30-bit child pointers)");
		Fcap += caps[s];
		// leaf blocks: the root at level 1, else at most one per fragment and 8^(L-1)
		Bcap += L == 1u ? 1u : std::min<uint64_t>(caps[s], 1ull << (3u * (L - 1u)));
	}
	if (Fcap > 0xFFFFFFFEull)
		return set_error(ctx, SVO_ERR_OVERFLOW, "a plan holds at most 2^32-2 fragments of capacity; split it");
	p->fls.assign(S, nullptr);
	p->octs.assign(S, nullptr);
	for (uint32_t s = 0; s < S; ++s) {
		svo_fraglist *fl = p->fls[s] = new (std::nothrow) svo_fraglist();
		svo_octree *o = p->octs[s] = new (std::nothrow) svo_octree();
		if (!fl || !o)
			return SVO_ERR_OUT_OF_MEMORY;
		fl->ctx = o->ctx = ctx;
		fl->scene = scenes[s];
		fl->level = o->level = levels[s];
		o->cap = caps[S + s];
		if (pool->alloc((void **)&fl->frags, sizeof(uint32_t) * 2 * caps[s]) != hipSuccess ||
		    pool->alloc((void **)&o->words, sizeof(uint32_t) * o->cap) != hipSuccess)
			return set_error(ctx, SVO_ERR_OUT_OF_MEMORY, "plan list or octree allocation failed");
	}
	if (int rc = voxelize_plan_init(ctx, &p->vb, p->fls.data(), S))
		return rc;
	BuildBatch &bb = p->bb;
	{
		std::vector<const uint2 *> frags(S);
		for (uint32_t s = 0; s < S; ++s)
			frags[s] = reinterpret_cast<const uint2 *>(p->fls[s]->frags);
		batch_layout(bb, S, frags.data(), caps.data(), levels);
	}
	// host totals are capacities: they size the grids and scratch; the kernels read the counts
	bb.nbins = Bcap;
	for (uint32_t s = 0; s < S; ++s)
		bb.h_segs[s].words = p->octs[s]->words;
	p->pw_value = bb.h_index[bb.pw_at() + bb.pw_segs()];
	const size_t seg_bytes = seg_table_bytes(S), idx_bytes = sizeof(uint64_t) * bb.h_index.size();
	if (pool->alloc((void **)&bb.segs, seg_bytes + idx_bytes) != hipSuccess ||
	    pool->alloc((void **)&bb.bm, sizeof(uint32_t) * (bb.TW ? bb.TW : 1)) != hipSuccess ||
	    pool->alloc((void **)&bb.rk, sizeof(uint32_t) * (bb.TW / 8u + 2 + S)) != hipSuccess ||
	    alloc_tiles(pool, bb) != hipSuccess ||
	    pool->alloc((void **)&bb.bucket, sizeof(uint32_t) * Fcap) != hipSuccess ||
	    pool->alloc((void **)&bb.list, sizeof(uint32_t) * (3 + 3 * big_capacity(Fcap))) != hipSuccess ||
	    pool->alloc((void **)&bb.cnt, sizeof(uint32_t) * Bcap) != hipSuccess ||
	    pool->alloc((void **)&bb.aux, sizeof(uint32_t) * Bcap) != hipSuccess ||
	    pool->alloc((void **)&p->caps, sizeof(uint64_t) * 2 * S) != hipSuccess ||
	    pool->alloc((void **)&p->out, sizeof(uint64_t) * (1 + 2 * (size_t)S)) != hipSuccess)
		return set_error(ctx, SVO_ERR_OUT_OF_MEMORY, "plan build allocation failed");
	bb.index = reinterpret_cast<uint64_t *>(reinterpret_cast<uint8_t *>(bb.segs) + seg_bytes);
	bb.raw = bb.rk + bb.TW / 8u + 1;
	if (int rc = upload_batch_tables(ctx, bb))
		return rc;
	if (int rc = upload_table(ctx, p->caps, caps.data(), sizeof(uint64_t) * 2 * S))
		return rc;
	// results before the first run: status 0, no fragments, no words
	p->h_out.assign(1 + 2 * (size_t)S, 0);
	return upload_table(ctx, p->out, p->h_out.data(), sizeof(uint64_t) * p->h_out.size());
}

int build_plan_run(svo_ctx *ctx, BuildPlan *p) {
	hipError_t e = hipSuccess;
	int rc = SVO_OK;
	p->t_run.start(ctx->stream);
	if (p->use_graph) {
		if (!p->exec) {
			// profiler events stay out of the graph
			const bool prof = ctx->prof.enabled;
			ctx->prof.enabled = false;
			hipGraph_t g = nullptr;
			e = hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal);
			if (e == hipSuccess) {
				rc = plan_enqueue(ctx, *p);
				e = hipStreamEndCapture(ctx->stream, &g);
			}
			ctx->prof.enabled = prof;
			if (!rc && e == hipSuccess)
				e = hipGraphInstantiate(&p->exec, g, nullptr, nullptr, 0);
			if (g)
				(void)hipGraphDestroy(g);
			if (rc || e != hipSuccess) {
				p->exec = nullptr;
				return rc ? rc : hip_check(ctx, e, "plan capture");
			}
		}
		e = hipGraphLaunch(p->exec, ctx->stream);
	} else {
		rc = plan_enqueue(ctx, *p);
	}
	p->t_run.stop(ctx->stream);
	if (rc)
		return rc;
	if (e != hipSuccess)
		return hip_check(ctx, e, "plan launch");
	p->pending = true;
	return SVO_OK;
}

int build_plan_finish(svo_ctx *ctx, BuildPlan *p, uint64_t *F, uint64_t *W, double *ms) {
	if (int rc = download_table(ctx, p->h_out.data(), p->out, sizeof(uint64_t) * p->h_out.size()))
		return rc;
	if (ms)
		*ms = p->pending ? p->t_run.read() : 0.0;
	p->pending = false;
	const uint32_t S = p->S;
	const uint64_t status = p->h_out[0];
	for (uint32_t s = 0; s < S; ++s) {
		const uint64_t f = p->h_out[1 + s], w = p->h_out[1 + S + s];
		if (F)
			F[s] = f;
		if (W)
			W[s] = w;
		p->fls[s]->F = status & 1u ? 0u : f;
		p->fls[s]->filled = !(status & 1u);
		p->octs[s]->W = status ? 0u : w;
	}
	if (status & 1u)
		for (uint32_t s = 0; s < S; ++s)
			if (p->h_out[1 + s] > p->bb.h_segs[s].F)
				return set_error(ctx, SVO_ERR_OVERFLOW,
				                 "scene " + std::to_string(s) + " has " + std::to_string(p->h_out[1 + s]) +
				                     " fragments, above the plan's capacity of " +
				                     std::to_string(p->bb.h_segs[s].F));
	if (status)
		for (uint32_t s = 0; s < S; ++s)
			if (p->h_out[1 + S + s] > p->octs[s]->cap)
				return set_error(ctx, SVO_ERR_OVERFLOW,
				                 "octree " + std::to_string(s) + " needs " + std::to_string(p->h_out[1 + S + s]) +
				                     " words, above the plan's capacity of " + std::to_string(p->octs[s]->cap));
	if (status)
		return set_error(ctx, SVO_ERR_OVERFLOW, "a plan count passed its capacity");
	return SVO_OK;
}

void build_plan_release(svo_ctx *ctx, BuildPlan *p) {
	if (p->exec)
		(void)hipGraphExecDestroy(p->exec);
	p->exec = nullptr;
	if (p->pending)
		(void)hipStreamSynchronize(ctx->stream);
	p->pending = false;
	p->t_run.destroy();
	vox_batch_release(ctx, &p->vb);
	build_batch_release(ctx, &p->bb);
	ctx->pool->free(p->caps);
	ctx->pool->free(p->out);
	p->caps = p->out = nullptr;
	for (svo_fraglist *fl : p->fls)
		if (fl) {
			ctx->pool->free(fl->frags);
			delete fl;
		}
	for (svo_octree *o : p->octs)
		if (o) {
			ctx->pool->free(o->words);
			delete o;
		}
	p->fls.clear();
	p->octs.clear();
}

} // namespace svo
