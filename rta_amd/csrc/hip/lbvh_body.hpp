// Per-mesh bodies of the LBVH build stages (bbvh-cuda/lbvh-kernels.cu), as
// device functions over one mesh's base pointers.  The single-mesh kernels
// (lbvh.hip) and the batched kernels (batch.hip) both call them, so every
// mesh of a batch is built by exactly the single-mesh code.
#pragma once

#include "common.hpp"

namespace rta_hip {

constexpr int kInitBlock = 256;
constexpr int kTriWords = sizeof(rta_triangle) / 8;   // 13 x 8 bytes
constexpr float kBoundsInit = 100000000000.0f;        // lbvh-kernels.cu:519
constexpr int kBoundsBlock = 1024;
constexpr int kChunk = 1024;
constexpr int kSlots = 128;
constexpr int kMergeFan = 16;

// ---------------------------------------------------------- wave helpers

__device__ inline float wave_min(float v) {
	for (int off = kWave / 2; off > 0; off >>= 1) v = sel_min(v, __shfl_xor(v, off));
	return v;
}
__device__ inline float wave_max(float v) {
	for (int off = kWave / 2; off > 0; off >>= 1) v = sel_max(v, __shfl_xor(v, off));
	return v;
}

// ------------------------------------------------ stage 1: initTriangles

// One block of kInitBlock threads handles triangles [block*256, +256) of a
// mesh (26,624 contiguous bytes): a coalesced copy src -> scratch staged
// through LDS (16-byte words where aligned), then each thread forms its triangle's box
// (lbvh-kernels.cu:141-153) and centroid ((a+b)+c)/3.0f (lbvh-kernels.cu:
// 60-63) from LDS, and the block reduces its boxes into one partial box.
__device__ inline void init_triangles_block(rta_triangle *__restrict__ scratch,
                                            const rta_triangle *__restrict__ src,
                                            rta_aabb *__restrict__ boxes,
                                            rta_float3 *__restrict__ centers,
                                            rta_aabb *__restrict__ partial, int n, int block) {
	__shared__ __align__(16) uint2 words[kInitBlock * kTriWords];
	__shared__ float red[6][kInitBlock / kWave];

	const int tid = threadIdx.x;
	const long long base = (long long)block * kInitBlock;
	const int count = (int)((n - base) < kInitBlock ? (n - base) : kInitBlock);
	const int nwords = count * kTriWords;
	const uint2 *gsrc = reinterpret_cast<const uint2 *>(src + base);
	uint2 *gdst = reinterpret_cast<uint2 *>(scratch + base);
	// 16-byte words when both ends are 16-byte aligned (a mesh of a batch
	// may start at an odd triangle, 8 bytes off), then the odd last word
	const bool wide = ((reinterpret_cast<uintptr_t>(gsrc) | reinterpret_cast<uintptr_t>(gdst)) &
	                   15u) == 0u;
	int w0 = 0;
	if (wide) {
		const uint4 *s4 = reinterpret_cast<const uint4 *>(gsrc);
		uint4 *d4 = reinterpret_cast<uint4 *>(gdst);
		uint4 *l4 = reinterpret_cast<uint4 *>(words);
		const int n4 = nwords / 2;
		for (int w = tid; w < n4; w += kInitBlock) {
			uint4 v = s4[w];
			l4[w] = v;
			d4[w] = v;
		}
		w0 = 2 * n4;
	}
	for (int w = w0 + tid; w < nwords; w += kInitBlock) {
		uint2 v = gsrc[w];
		words[w] = v;
		gdst[w] = v;
	}
	__syncthreads();

	float mn[3] = {kBoundsInit, kBoundsInit, kBoundsInit};
	float mx[3] = {-kBoundsInit, -kBoundsInit, -kBoundsInit};
	if (tid < count) {
		const float *f = reinterpret_cast<const float *>(&words[tid * kTriWords]);
		float lo[3], hi[3], ce[3];
		for (int c = 0; c < 3; ++c) {
			float va = f[c], vb = f[3 + c], vc = f[6 + c];
			lo[c] = sel_min(sel_min(va, vb), vc);
			hi[c] = sel_max(sel_max(va, vb), vc);
			ce[c] = ((va + vb) + vc) / 3.0f;
			// a NaN box coordinate does not enter the scene box: with a NaN
			// operand the reference's MIN/MAX (reduce_max,
			// lbvh-kernels.cu:496-516) is neither associative nor
			// commutative, so its thrust::reduce result depends on the
			// reduction order; skipping NaNs makes the bounds the min/max
			// over the other coordinates in every order
			if (lo[c] == lo[c]) mn[c] = lo[c];
			if (hi[c] == hi[c]) mx[c] = hi[c];
		}
		rta_aabb b;
		b.min = {lo[0], lo[1], lo[2]};
		b.max = {hi[0], hi[1], hi[2]};
		boxes[base + tid] = b;
		centers[base + tid] = {ce[0], ce[1], ce[2]};
	}
	// block reduction of the boxes (min/max are exact; the order only
	// matters for the sign of a zero, which cannot change a Morton code)
	const int lane = tid % kWave, wv = tid / kWave;
	for (int c = 0; c < 3; ++c) {
		float a = wave_min(mn[c]);
		float b = wave_max(mx[c]);
		if (lane == 0) { red[c][wv] = a; red[3 + c][wv] = b; }
	}
	__syncthreads();
	if (tid == 0) {
		float r[6];
		for (int c = 0; c < 3; ++c) { r[c] = kBoundsInit; r[3 + c] = -kBoundsInit; }
		for (int w = 0; w < kInitBlock / kWave; ++w)
			for (int c = 0; c < 3; ++c) {
				r[c] = sel_min(r[c], red[c][w]);
				r[3 + c] = sel_max(r[3 + c], red[3 + c][w]);
			}
		rta_aabb p;
		p.min = {r[0], r[1], r[2]};
		p.max = {r[3], r[4], r[5]};
		*partial = p;
	}
}

// ----------------------------------------------- stage 2: voxel bounds

// One block of kBoundsBlock threads reduces a mesh's np partial boxes
// (calculateVoxelBounds, lbvh-kernels.cu:518-535).
__device__ inline void voxel_bounds_block(rta_aabb *__restrict__ bounds,
                                          const rta_aabb *__restrict__ partials, int np) {
	__shared__ float red[6][kBoundsBlock / kWave];
	float mn[3] = {kBoundsInit, kBoundsInit, kBoundsInit};
	float mx[3] = {-kBoundsInit, -kBoundsInit, -kBoundsInit};
	for (int i = threadIdx.x; i < np; i += kBoundsBlock) {
		rta_aabb p = partials[i];
		mn[0] = sel_min(mn[0], p.min.x); mn[1] = sel_min(mn[1], p.min.y); mn[2] = sel_min(mn[2], p.min.z);
		mx[0] = sel_max(mx[0], p.max.x); mx[1] = sel_max(mx[1], p.max.y); mx[2] = sel_max(mx[2], p.max.z);
	}
	const int lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
	for (int c = 0; c < 3; ++c) {
		float a = wave_min(mn[c]);
		float b = wave_max(mx[c]);
		if (lane == 0) { red[c][wv] = a; red[3 + c][wv] = b; }
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		float r[6];
		for (int c = 0; c < 3; ++c) { r[c] = kBoundsInit; r[3 + c] = -kBoundsInit; }
		for (int w = 0; w < kBoundsBlock / kWave; ++w)
			for (int c = 0; c < 3; ++c) {
				r[c] = sel_min(r[c], red[c][w]);
				r[3 + c] = sel_max(r[3 + c], red[3 + c][w]);
			}
		rta_aabb b;
		b.min = {r[0], r[1], r[2]};
		b.max = {r[3], r[4], r[5]};
		*bounds = b;
	}
}

// ------------------------------------------------ stage 3: Morton codes

// The code of a centroid.  d = GRIDSIZE/(max-min) is formed per thread with
// the same correctly rounded division the reference does once on the host
// (lbvh-kernels.cu:414-417), so every thread sees the identical d.
__device__ inline uint32_t morton_code(const rta_float3 &c, const rta_aabb &vb) {
	const float dx = 1024.0f / (vb.max.x - vb.min.x);
	const float dy = 1024.0f / (vb.max.y - vb.min.y);
	const float dz = 1024.0f / (vb.max.z - vb.min.z);
	const uint32_t x = f2u_rz_sat((c.x - vb.min.x) * dx);
	const uint32_t y = f2u_rz_sat((c.y - vb.min.y) * dy);
	const uint32_t z = f2u_rz_sat((c.z - vb.min.z) * dz);
	return morton_encode_10bit(x, y, z);
}

// the code of triangle i of a mesh
__device__ inline uint32_t morton_of(const rta_float3 *__restrict__ centers,
                                     const rta_aabb *__restrict__ bounds, int i) {
	return morton_code(centers[i], *bounds);
}

// ----------------------------------------- stage 5: Karras hierarchy

// The sorted codes of one mesh as the hierarchy searches read them:
// positions [lo, hi) from a copy in LDS, the rest from global memory.  Most
// probes of a node's searches fall within a few times its range length of
// the node, so a block that stages its own positions plus a halo on each
// side answers nearly all of them from LDS.
constexpr int kKarrasBlock = 256;
constexpr int kKarrasHalo = 256;   // 1024 measured slower: staging outweighs the probes saved
constexpr int kKarrasWindow = kKarrasBlock + 2 * kKarrasHalo;
struct CodeWindow {
	const uint32_t *__restrict__ codes;
	const uint32_t *lds;
	int lo, hi;
	__device__ uint32_t operator()(int j) const {
		return (j >= lo && j < hi) ? lds[j - lo] : codes[j];
	}
};

// Stages positions [base - halo, base + block + halo) of [0, n) in lds
// (kKarrasWindow words) when the block holds inner nodes (base < n - 1);
// every thread of the block must call it.
__device__ inline CodeWindow stage_codes(uint32_t *lds, const uint32_t *__restrict__ codes, int n,
                                         int base) {
	CodeWindow w{codes, lds, 0, 0};
	if (base >= n - 1) return w;
	w.lo = base - kKarrasHalo > 0 ? base - kKarrasHalo : 0;
	w.hi = base + kKarrasBlock + kKarrasHalo < n ? base + kKarrasBlock + kKarrasHalo : n;
	for (int j = w.lo + (int)threadIdx.x; j < w.hi; j += kKarrasBlock) lds[j - w.lo] = codes[j];
	__syncthreads();
	return w;
}

// Common prefix length of the augmented keys (code, position):
// clz(ci^cj), or 32+clz(i^j) for equal codes, -1 outside [0,n)
// (__cpl, lbvh-kernels.cu:84-92); ci is the code of position i.
__device__ inline int cpl(int i, uint32_t ci, int j, const CodeWindow &w, int n) {
	if (j < 0 || j >= n) return -1;
	const uint32_t cj = w(j);
	if (ci == cj) return __clz((int)((uint32_t)i ^ (uint32_t)j)) + 32;
	return __clz((int)(ci ^ cj));
}

// Node i of a mesh of n triangles (k::build_tree_karras, lbvh-kernels.cu:
// 186-256).  The direction/range/split searches are the reference's,
// including its ceil-halving split search that always runs in +1 direction
// from the lower end of the range.  Inner nodes also clear their visit
// counter and record their sorted range [from, to] for the bottom-up pass.
__device__ inline void karras_node(rta_node *__restrict__ nodes, uint32_t *__restrict__ parents,
                                   uint32_t *__restrict__ visit, uint2 *__restrict__ ranges,
                                   const CodeWindow &w, int n, int i) {
	uint2 *links = reinterpret_cast<uint2 *>(&nodes[i]);
	if (i >= n - 1) {
		// leaf: tris = i-(n-1), elems = 1, leaf bit clear
		*links = make_uint2(1u << 1, (uint32_t)(i - (n - 1)));
		return;
	}
	const uint32_t ci = w(i);
	int d = (cpl(i, ci, i + 1, w, n) - cpl(i, ci, i - 1, w, n)) >= 0 ? 1 : -1;
	const int cpl_min = cpl(i, ci, i - d, w, n);
	int l_max = 2;
	while (cpl(i, ci, i + l_max * d, w, n) > cpl_min) l_max *= 2;
	int l = 0;
	for (int t = l_max / 2; t >= 1; t /= 2)
		if (cpl(i, ci, i + (l + t) * d, w, n) > cpl_min) l += t;
	const int j = i + l * d;
	const int from = j < i ? j : i;
	const int to = j < i ? i : j;

	const uint32_t cfrom = w(from);
	const int cpl_node = cpl(from, cfrom, to, w, n);
	int s = 0;
	for (int t = (l / 2 + l % 2); t >= 1; t = (t / 2 + t % 2)) {
		if (cpl(from, cfrom, from + (s + t), w, n) > cpl_node) s += t;
		if (t <= 1) break;
	}
	const int mid = from + s;
	int left = mid, right = mid + 1;
	if (from == mid) left += n - 1;
	if (to == mid + 1) right += n - 1;
	*links = make_uint2(((uint32_t)left << 1) | 1u, (uint32_t)right);
	parents[left] = (uint32_t)i;
	parents[right] = (uint32_t)i;
	visit[i] = 0u;
	ranges[i] = make_uint2((uint32_t)from, (uint32_t)to);
}

// ----------------------------------------- stage 6: bottom-up boxes

// Bottom-up boxes (k::build_bounding_boxes_karras2, lbvh-kernels.cu:258-341),
// with the hierarchy of k::build_tree_karras (:186-256) emitted by the same
// climb.  The hierarchy is the binary radix tree of the augmented keys
// (code, position), which is unique, so it can be grown from the leaves: a
// completed node covering sorted positions [l, r] has its parent on the
// side of the longer common prefix with its neighbour -- split r (the node
// is the left child) when delta(r) > delta(l-1), else split l-1 (the right
// child), with delta(i) the common prefix length of positions i and i+1
// (cpl above) and delta(-1) = delta(n-1) = -1; two neighbours never tie.
// Karras numbering follows: the children of split s are nodes s and s+1
// (leaves when their range is one position), so a node's index is r as a
// left child, l as a right child, and 0 for the root.
//
// At each split the first arriving child stops and the second forms the
// parent: the union MIN(left, right) / MAX(left, right) with the
// reference's `(a<b)?a:b`, the whole 32-byte node, its range and (packed
// build) its pair record, and climbs on.  Merge rule: both children are
// leaves (original or merged) and their representative codes are equal
// (codes[s] == codes[s+1], i.e. delta(s) >= 32; `code == old` in the
// reference) -> the parent becomes one leaf with tris = min, elems = sum
// (lbvh-kernels.cu:302-330).  Deterministic form of the reference: a visit
// counter per split decides first/second arrival (the reference sums
// representative codes into the flag, so a first arrival with code 0 also
// stops the second thread, :288-291), and the union order is fixed (the
// reference leaves the sign of a zero to arrival order).
//
// Hierarchical schedule.  A subtree covers a contiguous range of sorted
// positions, so all communication inside a chunk of consecutive leaves
// stays in one workgroup:
//  level 1: a 1024-thread block owns 1024 leaves; the deltas, the visit
//           counters and the waiting children live in LDS; a climb stops
//           when its parent's split lies outside the chunk, and the
//           completed nodes whose parents stay incomplete form the chunk's
//           frontier (at most 2 per tree level, so <= 126 for depth <= 63);
//  level k: one block merges the frontiers of kMergeFan level-(k-1) chunks,
//           its visit counters and waiting children in LDS again (a table
//           keyed by split), until one block covers all leaves and reaches
//           the root.
// No step needs device-scope cache maintenance; results do not depend on
// the schedule.  A merge level of the 2.3 M-triangle terrain takes 18 us (35
// with a split table and scalar records), of an 82 k-triangle sphere 13 (25),
// of a 5 k-triangle one 10 (18).

__device__ inline rta_aabb union_lr(const rta_aabb &lb, const rta_aabb &rb) {
	rta_aabb u;
	u.min.x = sel_min(lb.min.x, rb.min.x);
	u.min.y = sel_min(lb.min.y, rb.min.y);
	u.min.z = sel_min(lb.min.z, rb.min.z);
	u.max.x = sel_max(lb.max.x, rb.max.x);
	u.max.y = sel_max(lb.max.y, rb.max.y);
	u.max.z = sel_max(lb.max.z, rb.max.z);
	return u;
}

// The traversal layout written by the build itself (rta_lbvh_build_packed):
// per inner node x a 64-byte child-pair record pairs[x] (both children's
// boxes SoA, their words -- (x << 1) | 1 for an inner child, first
// triangle << 1 for a leaf -- and their node ids), per triangle three
// float4 of tri4 (a, a - b, a - c; the w of the first is nonzero on the last
// triangle of a leaf), and flags bit 0 when some box coordinate leaves the
// exact-division range.  The same bytes as rta_bvh_pack over the finished
// nodes.  All pointers null: the plain build.
struct PackOut {
	rta_node_pair *pairs = nullptr;
	float4 *tri4 = nullptr;
	uint32_t *flags = nullptr;
};

__device__ inline bool box_fast(const rta_aabb &b) {
	return coord_fast_ok(b.min.x) && coord_fast_ok(b.min.y) && coord_fast_ok(b.min.z) &&
	       coord_fast_ok(b.max.x) && coord_fast_ok(b.max.y) && coord_fast_ok(b.max.z);
}

// pairs[x] from its children's boxes, words and ids; returns false when a
// box coordinate leaves the exact-division range
__device__ inline bool write_pair(rta_node_pair *pairs, uint32_t x, const rta_aabb &lb,
                                  const rta_aabb &rb, uint32_t lword, uint32_t rword, uint32_t lid,
                                  uint32_t rid) {
	rta_node_pair p;
	p.lo_x[0] = lb.min.x; p.lo_x[1] = rb.min.x;
	p.lo_y[0] = lb.min.y; p.lo_y[1] = rb.min.y;
	p.lo_z[0] = lb.min.z; p.lo_z[1] = rb.min.z;
	p.hi_x[0] = lb.max.x; p.hi_x[1] = rb.max.x;
	p.hi_y[0] = lb.max.y; p.hi_y[1] = rb.max.y;
	p.hi_z[0] = lb.max.z; p.hi_z[1] = rb.max.z;
	p.link[0] = lword; p.link[1] = rword;
	p.index[0] = lid; p.index[1] = rid;
	pairs[x] = p;
	return box_fast(lb) && box_fast(rb);
}

// a merge joins two leaves: the left one's last triangle no longer ends a
// leaf (the permute wrote every triangle as a leaf end)
__device__ inline void clear_leaf_end(float4 *tri4, uint32_t pos) {
	tri4[3 * (size_t)pos].w = 0.0f;
}

// delta(i): common prefix length of the augmented keys at sorted positions
// i and i+1, -1 outside [0, n-1)
__device__ inline int delta_at(const uint32_t *__restrict__ codes, long long i, int n) {
	if (i < 0 || i >= (long long)n - 1) return -1;
	const uint32_t a = codes[i], b = codes[i + 1];
	if (a == b) return __clz((int)((uint32_t)i ^ (uint32_t)(i + 1))) + 32;
	return __clz((int)(a ^ b));
}

// the whole node: link words and box, as two 16-byte stores
__device__ inline void store_node(rta_node *node, uint2 links, const rta_aabb &b) {
	uint4 *o = reinterpret_cast<uint4 *>(node);
	o[0] = make_uint4(links.x, links.y, __float_as_uint(b.min.x), __float_as_uint(b.min.y));
	o[1] = make_uint4(__float_as_uint(b.min.z), __float_as_uint(b.max.x), __float_as_uint(b.max.y),
	                  __float_as_uint(b.max.z));
}

// Bottom-up over E consecutive items of a mesh in one workgroup: the leaves
// of a chunk (level 1) or the frontier entries of some groups (above).  Item
// i covers the sorted positions [pos(i), pos(i + 1)); the items are adjacent
// and in order, so a node is a run of items [a, b] and a split is the
// boundary j between items j and j + 1.
//
// The climbs touch LDS only.  Every child arriving at a boundary writes its
// record (box, far item, delta there, leaf state: two 16-byte words) under
// that boundary and its side, then counts its arrival; the second arrival
// reads its sibling's record and climbs on with the parent.  Fences are
// LDS-only.  Afterwards each boundary whose two children arrived writes the
// parent's whole node, range and pair record from the two records, one
// boundary per thread; a node whose parent stays incomplete (its sibling
// reaches beyond the items) joins the frontier, which is written in order.
//
// A leaf holds the triangles of its range: a merge of leaves [l, s] and
// [s + 1, r] gives tris = l and elems = r - l + 1, so its state is one bit.
//
// What bounds it: the chain of dependent LDS round trips of the climbs and
// the instructions of waves with few lanes still climbing.
struct ClimbRecord {
	float4 lo;   // min.x, min.y, min.z, max.x
	float4 hi;   // max.y, max.z, far item, delta + 1 at the far end | inner << 8
};
constexpr uint32_t kArriveRight = 0x10000u;   // visit count of a right child (a left one adds 1)
constexpr uint32_t kNoFront = 0xffffffffu, kFrontInner = 0x80000000u;   // frontier marks
constexpr uint32_t kEntryInner = 0x10000u;    // frontier entry: an inner node
constexpr uint32_t kInnerBit = 0x100u;

template <int E>
struct ClimbShared {
	ClimbRecord rec[2][E];       // per side (0: the left child) and boundary
	uint32_t visit[E];           // arrivals per boundary; then the frontier
	int8_t delta[E + 4];         // delta at the start of item i; [items]: at the end
	uint32_t wave_count[16];
};

// One item, before the climb.
struct ClimbItem {
	rta_aabb box;
	bool inner;
};

// The climb of item i.
template <int E>
__device__ inline void climb(ClimbShared<E> &sh, int i, int items, const ClimbItem &it) {
	rta_aabb box = it.box;
	bool inner = it.inner;
	int a = i, b = i;
	int dl = sh.delta[i], dr = sh.delta[i + 1];
	for (int level = 0; level < 128; ++level) {
		if (dl < 0 && dr < 0) break;      // the root of the mesh
		const bool left = dr > dl;        // the left child of boundary b, else the right of a - 1
		// the sibling lies beyond the items: an edge record (boundary items - 1
		// is never formed here, its slots take the last and the first node)
		const bool edge = left ? b + 1 == items : a == 0;
		const int j = edge ? items - 1 : (left ? b : a - 1);
		ClimbRecord &mine = sh.rec[left ? 0 : 1][j];
		mine.lo = make_float4(box.min.x, box.min.y, box.min.z, box.max.x);
		mine.hi = make_float4(box.max.y, box.max.z, __uint_as_float((uint32_t)(left ? a : b)),
		                      __uint_as_float((uint32_t)((left ? dl : dr) + 1) |
		                                      (inner ? kInnerBit : 0u)));
		__builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
		const uint32_t old = atomicAdd(&sh.visit[j], left ? 1u : kArriveRight);
		if (edge || old == 0u) break;     // else the sibling forms the parent
		__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
		const ClimbRecord sib = sh.rec[left ? 1 : 0][j];
		const rta_aabb sbox = {{sib.lo.x, sib.lo.y, sib.lo.z}, {sib.lo.w, sib.hi.x, sib.hi.y}};
		const int far = (int)__float_as_uint(sib.hi.z);
		const uint32_t meta = __float_as_uint(sib.hi.w);
		const int dfar = (int)(meta & 0xffu) - 1, ds = left ? dr : dl;
		// both leaves and equal codes at the boundary: one leaf
		inner = inner || (meta & kInnerBit) != 0u || ds < 32;
		box = left ? union_lr(box, sbox) : union_lr(sbox, box);
		if (left) { b = far; dr = dfar; }
		else { a = far; dl = dfar; }
	}
}

// After the climbs of all items and a barrier: thread t takes boundaries (and
// frontier items) t, t + threads, ...  All threads of the block call it.
// Returns the frontier's size.
template <int E, int THREADS, class Pos>
__device__ inline uint32_t emit_nodes(ClimbShared<E> &sh, int items, const Pos &pos,
                                      rta_node *__restrict__ nodes, uint2 *__restrict__ ranges,
                                      uint4 *__restrict__ slots, int n, const PackOut &pk) {
	const int t = threadIdx.x;
	const uint32_t leaf0 = (uint32_t)(n - 1);
	constexpr int kPer = E / THREADS;
	static_assert(E % THREADS == 0 && THREADS % kWave == 0 && THREADS <= 16 * kWave, "whole rounds");
	bool slow = false;
	uint32_t v[kPer];
#pragma unroll
	for (int k = 0; k < kPer; ++k) {
		const int j = t + k * THREADS;
		v[k] = j < items ? sh.visit[j] : 0u;
		if (j + 1 >= items || v[k] != 1u + kArriveRight) continue;
		const ClimbRecord L = sh.rec[0][j], R = sh.rec[1][j];
		const int a = (int)__float_as_uint(L.hi.z), b = (int)__float_as_uint(R.hi.z);
		const uint32_t lm = __float_as_uint(L.hi.w), rm = __float_as_uint(R.hi.w);
		const uint32_t l = pos(a), s = pos(j + 1) - 1u, r = pos(b + 1) - 1u;
		const int dl = (int)(lm & 0xffu), dr = (int)(rm & 0xffu), ds = sh.delta[j + 1];
		const rta_aabb lb = {{L.lo.x, L.lo.y, L.lo.z}, {L.lo.w, L.hi.x, L.hi.y}};
		const rta_aabb rb = {{R.lo.x, R.lo.y, R.lo.z}, {R.lo.w, R.hi.x, R.hi.y}};
		const bool linner = (lm & kInnerBit) != 0u, rinner = (rm & kInnerBit) != 0u;
		const bool merge = ds >= 32 && !linner && !rinner;
		// the node's index: r as a left child, l as a right child or the root
		const uint32_t x = dr > dl ? r : l;
		const uint32_t lid = l == s ? leaf0 + s : s, rid = r == s + 1u ? leaf0 + r : s + 1u;
		store_node(&nodes[x], merge ? make_uint2((r - l + 1u) << 1, l) : make_uint2((lid << 1) | 1u, rid),
		           union_lr(lb, rb));
		ranges[x] = make_uint2(l, r);
		if (merge) {
			if (pk.tri4) clear_leaf_end(pk.tri4, s);
		} else if (pk.pairs) {
			const uint32_t lw = linner ? (s << 1) | 1u : l << 1;
			const uint32_t rw = rinner ? ((s + 1u) << 1) | 1u : (s + 1u) << 1;
			if (!write_pair(pk.pairs, x, lb, rb, lw, rw, lid, rid)) slow = true;
		}
	}
	if (pk.flags && __syncthreads_or(slow) && t == 0) atomicOr(pk.flags, 1u);
	__syncthreads();
	// The frontier, by first item: nodes that are the only arrival at their
	// boundary, and the edge records.
#pragma unroll
	for (int k = 0; k < kPer; ++k) sh.visit[t + k * THREADS] = kNoFront;
	__syncthreads();
#pragma unroll
	for (int k = 0; k < kPer; ++k) {
		const int j = t + k * THREADS;
		const bool edge = j + 1 == items;
		if (v[k] == 0u || (!edge && v[k] == 1u + kArriveRight)) continue;
		if (v[k] & 1u) {
			const float4 hi = sh.rec[0][j].hi;
			sh.visit[__float_as_uint(hi.z)] =
			    (uint32_t)j | (__float_as_uint(hi.w) & kInnerBit ? kFrontInner : 0u);
		}
		if (v[k] & kArriveRight) {
			const float4 hi = sh.rec[1][j].hi;
			sh.visit[edge ? 0 : j + 1] =
			    __float_as_uint(hi.z) | (__float_as_uint(hi.w) & kInnerBit ? kFrontInner : 0u);
		}
	}
	__syncthreads();
	uint32_t total = 0;
#pragma unroll
	for (int k = 0; k < kPer; ++k) {
		const int a = t + k * THREADS;
		const uint32_t f = a < items ? sh.visit[a] : kNoFront;
		const uint64_t has = __ballot(f != kNoFront);
		const int wave = t / kWave;
		if (__lane_id() == 0) sh.wave_count[wave] = (uint32_t)__popcll(has);
		__syncthreads();
		uint32_t before = total, all = 0;
		for (int w = 0; w < THREADS / kWave; ++w) {
			const uint32_t c = sh.wave_count[w];
			before += w < wave ? c : 0u;
			all += c;
		}
		__syncthreads();
		total += all;
		if (f == kNoFront) continue;
		const uint32_t rank = before + (uint32_t)__popcll(has & ((1ull << __lane_id()) - 1ull));
		const int b = (int)(f & ~kFrontInner);
		const uint32_t l = pos(a), r = pos(b + 1) - 1u;
		const int dl = sh.delta[a], dr = sh.delta[b + 1];
		const uint32_t x = l == r ? leaf0 + l : (dr > dl ? r : l);
		if (slots && rank < (uint32_t)kSlots)
			slots[rank] = make_uint4(x, l, r, (uint32_t)(dl + 1) | ((uint32_t)(dr + 1) << 8) |
			                                      (f & kFrontInner ? kEntryInner : 0u));
	}
	return total;
}

// Level 1 for leaves [chunk*kChunk, +kChunk) of a mesh: every leaf's node,
// every node completed inside the chunk, and the frontier in slots[0..kSlots)
// with its size in *count.
__device__ inline void bottom_up_chunk(rta_node *__restrict__ nodes,
                                       const rta_aabb *__restrict__ boxes,
                                       const uint32_t *__restrict__ codes,
                                       const uint32_t *__restrict__ indices,
                                       uint2 *__restrict__ ranges,
                                       uint4 *__restrict__ slots, uint32_t *__restrict__ count,
                                       uint32_t *__restrict__ status, int n, int chunk,
                                       PackOut pk = PackOut{}) {
	__shared__ ClimbShared<kChunk> sh;
	const int t = threadIdx.x;
	const uint32_t base = (uint32_t)chunk * kChunk;
	const int items = (int)min((uint32_t)kChunk, (uint32_t)n - base);
	ClimbItem it{{}, false};
	if (t < items) {
		const uint32_t k = base + t;
		it.box = boxes[indices[k]];
		store_node(&nodes[(uint32_t)(n - 1) + k], make_uint2(1u << 1, k), it.box);
	}
	sh.visit[t] = 0;
	for (int i = t; i <= items; i += kChunk)
		sh.delta[i] = (int8_t)delta_at(codes, (long long)base + i - 1, n);
	__syncthreads();
	if (t < items) climb(sh, t, items, it);
	__syncthreads();
	const uint32_t total = emit_nodes<kChunk, kChunk>(
	    sh, items, [&](int i) { return base + (uint32_t)i; }, nodes, ranges, slots, n, pk);
	if (t == 0) {
		if (total > (uint32_t)kSlots) atomicOr(status, (uint32_t)RTA_LBVH_FRONTIER_OVERFLOW);
		*count = min(total, (uint32_t)kSlots);
	}
}

// Level k >= 2 for one mesh: merges the frontier slots of the ng chunks of
// the previous level starting at in_slots/in_counts (kSlots entries per
// chunk, in order); the new frontier goes to out_slots / *out_count when
// given (the last level has none).
constexpr int kMergeThreads = 1024;
constexpr int kMergeEntries = kMergeFan * kSlots;
__device__ inline void bottom_up_merge(rta_node *__restrict__ nodes, uint2 *__restrict__ ranges,
                                       const uint4 *__restrict__ in_slots,
                                       const uint32_t *__restrict__ in_counts, int ng,
                                       uint4 *__restrict__ out_slots,
                                       uint32_t *__restrict__ out_count,
                                       uint32_t *__restrict__ status, int n,
                                       PackOut pk = PackOut{}) {
	__shared__ ClimbShared<kMergeEntries> sh;
	__shared__ uint32_t pos[kMergeEntries + 1];
	constexpr int kPer = kMergeEntries / kMergeThreads;
	static_assert(kMergeFan <= kWave, "group counts in one wave");
	const int t = threadIdx.x;
	// every wave finds the groups' first items by itself
	const int lane = __lane_id();
	const uint32_t mine = lane < ng ? min(in_counts[lane], (uint32_t)kSlots) : 0u;
	uint32_t upto = mine;
	for (int off = 1; off < kMergeFan; off <<= 1) {
		const uint32_t y = __shfl_up(upto, off);
		if (lane >= off) upto += y;
	}
	const int items = (int)__shfl(upto, kMergeFan - 1);
	const uint32_t first = upto - mine;
	ClimbItem it[kPer];
#pragma unroll
	for (int k = 0; k < kPer; ++k) {
		const int i = t + k * kMergeThreads;
		sh.visit[i] = 0;
		// the last group that starts at or before item i
		int g = 0;
		for (int step = kMergeFan / 2; step > 0; step >>= 1)
			if (__shfl(first, g + step) <= (uint32_t)i && g + step < ng) g += step;
		const uint32_t before = __shfl(first, g);
		if (i < items) {
			const uint4 e = in_slots[(size_t)g * kSlots + ((uint32_t)i - before)];
			pos[i] = e.y;
			sh.delta[i] = (int8_t)((int)(e.w & 0xffu) - 1);
			if (i == items - 1) {
				pos[items] = e.z + 1u;
				sh.delta[items] = (int8_t)((int)((e.w >> 8) & 0xffu) - 1);
			}
			it[k].inner = (e.w & kEntryInner) != 0u;
			it[k].box = nodes[e.x].box;
		}
	}
	__syncthreads();
	for (int k = 0; k < kPer; ++k) {
		const int i = t + k * kMergeThreads;
		if (i < items) climb(sh, i, items, it[k]);
	}
	__syncthreads();
	const uint32_t total = emit_nodes<kMergeEntries, kMergeThreads>(
	    sh, items, [&](int i) { return pos[i]; }, nodes, ranges, out_slots, n, pk);
	if (t == 0) {
		if (total > (out_slots ? (uint32_t)kSlots : 0u))
			atomicOr(status, (uint32_t)RTA_LBVH_FRONTIER_OVERFLOW);
		if (out_count) *out_count = min(total, (uint32_t)kSlots);
	}
}

// -------------------------------------------------- stage 7: permute

// out[i] = scratch[indices[i]] (invert_triangle_permutation_cuda,
// lbvh-kernels.cu:557-578) for the kPermuteBlock triangles of one block,
// as 13 * kPermuteBlock consecutive 8-byte output words: word w comes from
// word w % 13 of triangle indices[block * kPermuteBlock + w / 13].  Every
// store of a wave is contiguous and each scattered source record is read
// by 13 neighbouring lanes.  All threads of the block must call it.
constexpr int kPermuteBlock = 256;
constexpr int kVertexWords = 5;   // the 36 bytes of a, b, c lie in words 0..4
__device__ inline void permute_block(rta_triangle *__restrict__ out,
                                     const rta_triangle *__restrict__ scratch,
                                     const uint32_t *__restrict__ indices, int n, int block,
                                     float4 *__restrict__ tri4 = nullptr) {
	__shared__ uint32_t src[kPermuteBlock];
	__shared__ uint2 verts[kPermuteBlock][kVertexWords];
	const int t = threadIdx.x;
	const int base = block * kPermuteBlock;
	const int count = min(kPermuteBlock, n - base);
	if (t < count) src[t] = indices[base + t];
	__syncthreads();
	const uint2 *s = reinterpret_cast<const uint2 *>(scratch);
	uint2 *d = reinterpret_cast<uint2 *>(out + base);
	const int nwords = count * kTriWords;
	uint2 v[kTriWords];
#pragma unroll
	for (int k = 0; k < kTriWords; ++k) {
		const int w = t + k * kPermuteBlock;
		if (w < nwords) {
			const int r = w / kTriWords;
			v[k] = s[(size_t)src[r] * kTriWords + (w - r * kTriWords)];
		}
	}
#pragma unroll
	for (int k = 0; k < kTriWords; ++k) {
		const int w = t + k * kPermuteBlock;
		if (w < nwords) d[w] = v[k];
	}
	if (tri4) {
		// the vertex words of each triangle, gathered in LDS, give its three
		// tri4 records (a, a - b, a - c; every triangle first marked as the
		// end of a leaf, the bottom-up pass clears the marks that collapses
		// make interior)
#pragma unroll
		for (int k = 0; k < kTriWords; ++k) {
			const int w = t + k * kPermuteBlock;
			if (w < nwords) {
				const int r = w / kTriWords, c = w - r * kTriWords;
				if (c < kVertexWords) verts[r][c] = v[k];
			}
		}
		__syncthreads();
		if (t < count) {
			const float *f = reinterpret_cast<const float *>(&verts[t][0]);
			const float ax = f[0], ay = f[1], az = f[2];
			float4 *o = tri4 + 3 * (size_t)(base + t);
			o[0] = make_float4(ax, ay, az, __uint_as_float(1u));
			o[1] = make_float4(ax - f[3], ay - f[4], az - f[5], 0.0f);
			o[2] = make_float4(ax - f[6], ay - f[7], az - f[8], 0.0f);
		}
	}
}

}  // namespace rta_hip
