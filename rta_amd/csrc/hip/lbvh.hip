// Karras LBVH build for gfx950: the seven stages of the reference builder
// (bbvh-cuda/lbvh.h:153-211, bbvh-cuda/lbvh-kernels.cu) as hand-written HIP
// kernels.  Results are bit-identical to the reference's semantics; where
// the reference is racy the behaviour chosen here is deterministic and
// documented at the stage body (lbvh_body.hpp).  This file holds the
// single-mesh kernels and entry points; batch.hip runs the same bodies for
// many meshes per launch.
#include "internal.hpp"
#include "lbvh_body.hpp"

#include <cstdio>

namespace rta_hip {

// One block per 256 triangles; its partial scene box goes to
// partials[blockIdx.x].
__global__ __launch_bounds__(kInitBlock) void init_triangles_kernel(
    rta_triangle *__restrict__ scratch, const rta_triangle *__restrict__ src,
    rta_aabb *__restrict__ boxes, rta_float3 *__restrict__ centers,
    rta_aabb *__restrict__ partials, int n, uint32_t *status, uint32_t *flags) {
	// the words that the later stages OR into
	if (blockIdx.x == 0 && threadIdx.x == 0) {
		if (status) *status = 0u;
		if (flags) *flags = 0u;
	}
	init_triangles_block(scratch, src, boxes, centers, partials + blockIdx.x, n, blockIdx.x);
}

__global__ __launch_bounds__(kBoundsBlock) void voxel_bounds_kernel(
    rta_aabb *__restrict__ bounds, const rta_aabb *__restrict__ partials, int np) {
	voxel_bounds_block(bounds, partials, np);
}

__global__ __launch_bounds__(256) void morton_kernel(
    uint32_t *__restrict__ codes, uint32_t *__restrict__ indices,
    const rta_float3 *__restrict__ centers, const rta_aabb *__restrict__ bounds,
    uint32_t *__restrict__ status, int n) {
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n) return;
	const uint32_t code = morton_of(centers, bounds, i);
	codes[i] = code;
	indices[i] = (uint32_t)i;
	if (code == 0u && status) atomicOr(status, (uint32_t)RTA_LBVH_CODE_ZERO);
}

// Stages 2 to 4 (scene box, Morton codes, stable sort) of a mesh of at most
// kSmallSort triangles in one workgroup: the scene box from the partials, K
// codes per thread, then a stable LSD radix sort of (code, index) in LDS by
// four 8-bit digits.  Per digit every wave ranks its keys with ballots (as
// rs_scatter_kernel does), four threads per digit turn the counts over (item,
// wave) -- index order -- into positions, and the keys move through LDS.
//
// What bounds it: latency and the issue rate of one CU.  It replaces eight
// launches (bounds, codes, three sort passes of two kernels).  Whole packed
// builds, with those launches and with this kernel: 1,024 triangles 55 and 37
// us, 2,048 67 and 52, 4,096 72 and 63, 5,120 73 and 71, 6,144 74 and 73;
// larger meshes take the launches (7,168: 76 and 82, 8,192 76 and 84, 12,288
// 81 and 103).  A build that is waited for crosses a little higher, as its
// launches are not hidden: 6,145 triangles 100 and 95 us, 8,192 97 and 98.
constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / kWave;
constexpr int kSmallItems = 6;
constexpr int kSmallSort = kSmallItems * kSmallThreads;

template <int K>
__global__ __launch_bounds__(kSmallThreads) void small_sort_kernel(
    uint32_t *__restrict__ codes, uint32_t *__restrict__ indices,
    const rta_float3 *__restrict__ centers, const rta_aabb *__restrict__ partials, int np,
    uint32_t *__restrict__ status, int n) {
	// Counts are 16 bits, two groups (item, wave) to a word; an odd row length
	// keeps the ranking's writes (one group, many digits) and the scan's
	// reads (thread 4d + q: a quarter of digit d's row) off each other's banks.
	constexpr int kBins = 256, kGroups = K * kSmallWaves, kRow = kGroups / 2 + 1, kPer = kGroups / 8;
	static_assert(kSmallSort / kInitBlock <= kWave, "one partial box per lane");
	__shared__ union {
		uint32_t cnt[kBins * kRow];            // per digit and group: counts, then positions
		uint32_t kv[2][K * kSmallThreads];     // the keys and indices in their new order
	} sm;
	__shared__ uint32_t wave_sums[kSmallWaves];
	const int t = threadIdx.x, lane = __lane_id(), wave = t / kWave;
	const uint64_t lt = (1ull << lane) - 1ull;

	rta_aabb vb{{kBoundsInit, kBoundsInit, kBoundsInit}, {-kBoundsInit, -kBoundsInit, -kBoundsInit}};
	if (lane < np) {
		const rta_aabb p = partials[lane];
		vb.min = {sel_min(vb.min.x, p.min.x), sel_min(vb.min.y, p.min.y), sel_min(vb.min.z, p.min.z)};
		vb.max = {sel_max(vb.max.x, p.max.x), sel_max(vb.max.y, p.max.y), sel_max(vb.max.z, p.max.z)};
	}
	vb.min = {wave_min(vb.min.x), wave_min(vb.min.y), wave_min(vb.min.z)};
	vb.max = {wave_max(vb.max.x), wave_max(vb.max.y), wave_max(vb.max.z)};

	uint32_t key[K], val[K];
	bool zero = false;
#pragma unroll
	for (int it = 0; it < K; ++it) {
		const int i = it * kSmallThreads + t;
		key[it] = 0u;
		val[it] = (uint32_t)i;
		if (i < n) {
			key[it] = morton_code(centers[i], vb);
			zero = zero || key[it] == 0u;
		}
	}
	if (status && __ballot(zero) != 0ull && lane == 0) atomicOr(status, (uint32_t)RTA_LBVH_CODE_ZERO);

#pragma unroll 1
	for (int shift = 0; shift < 32; shift += 8) {
		uint16_t *const cnt16 = reinterpret_cast<uint16_t *>(sm.cnt);
		for (int i = t; i < kBins * kRow; i += kSmallThreads) sm.cnt[i] = 0u;
		__syncthreads();
		uint32_t rank[K];
#pragma unroll
		for (int it = 0; it < K; ++it) {
			const bool valid = it * kSmallThreads + t < n;
			const uint32_t d = (key[it] >> shift) & (kBins - 1);
			uint64_t match = __ballot(valid);
#pragma unroll
			for (int b = 0; b < 8; ++b) {
				const bool bit = (d >> b) & 1u;
				const uint64_t m = __ballot(bit);
				match &= bit ? m : ~m;
			}
			rank[it] = (uint32_t)__popcll(match & lt);
			if (valid && rank[it] == 0u)
				cnt16[d * 2 * kRow + it * kSmallWaves + wave] = (uint16_t)__popcll(match);
		}
		__syncthreads();
		// thread 4d + q: digit d's groups [q * kPer, +kPer)
		{
			uint32_t *const row = sm.cnt + (t >> 2) * kRow + (t & 3) * kPer;
			uint32_t sum = 0;
#pragma unroll
			for (int i = 0; i < kPer; ++i) sum += (row[i] & 0xffffu) + (row[i] >> 16);
			uint32_t x = sum;   // inclusive over the block, digits in order
			for (int off = 1; off < kWave; off <<= 1) {
				const uint32_t y = __shfl_up(x, off);
				if (lane >= off) x += y;
			}
			if (lane == kWave - 1) wave_sums[wave] = x;
			__syncthreads();
			uint32_t at = x - sum;
			for (int w = 0; w < kSmallWaves; ++w) at += w < wave ? wave_sums[w] : 0u;
#pragma unroll
			for (int i = 0; i < kPer; ++i) {
				const uint32_t c = row[i], second = at + (c & 0xffffu);
				row[i] = at | (second << 16);
				at = second + (c >> 16);
			}
		}
		__syncthreads();
#pragma unroll
		for (int it = 0; it < K; ++it)
			rank[it] += cnt16[((key[it] >> shift) & (kBins - 1)) * 2 * kRow + it * kSmallWaves + wave];
		__syncthreads();   // the positions are dead; their LDS now holds the keys
#pragma unroll
		for (int it = 0; it < K; ++it)
			if (it * kSmallThreads + t < n) {
				sm.kv[0][rank[it]] = key[it];
				sm.kv[1][rank[it]] = val[it];
			}
		__syncthreads();
#pragma unroll
		for (int it = 0; it < K; ++it) {
			const int i = it * kSmallThreads + t;
			if (i < n) {
				key[it] = sm.kv[0][i];
				val[it] = sm.kv[1][i];
			}
		}
		__syncthreads();
	}
#pragma unroll
	for (int it = 0; it < K; ++it) {
		const int i = it * kSmallThreads + t;
		if (i < n) {
			codes[i] = key[it];
			indices[i] = val[it];
		}
	}
}

__global__ __launch_bounds__(kKarrasBlock) void karras_kernel(
    rta_node *__restrict__ nodes, uint32_t *__restrict__ parents,
    uint32_t *__restrict__ visit, uint2 *__restrict__ ranges,
    const uint32_t *__restrict__ codes, int n) {
	__shared__ uint32_t window[kKarrasWindow];
	const int base = blockIdx.x * kKarrasBlock;
	const CodeWindow w = stage_codes(window, codes, n, base);
	const int i = base + threadIdx.x;
	if (i >= 2 * n - 1) return;
	karras_node(nodes, parents, visit, ranges, w, n, i);
}

__global__ __launch_bounds__(kChunk) void bottom_up_chunk_kernel(
    rta_node *__restrict__ nodes, const rta_aabb *__restrict__ boxes,
    const uint32_t *__restrict__ codes, const uint32_t *__restrict__ indices,
    uint2 *__restrict__ ranges, uint4 *__restrict__ slots, uint32_t *__restrict__ counts,
    uint32_t *__restrict__ status, int n, PackOut pk) {
	bottom_up_chunk(nodes, boxes, codes, indices, ranges,
	                slots + (size_t)blockIdx.x * kSlots, counts + blockIdx.x, status, n,
	                (int)blockIdx.x, pk);
}

// One block merges the frontier slots of up to kMergeFan chunks of the
// previous level.
__global__ __launch_bounds__(kMergeThreads) void bottom_up_merge_kernel(
    rta_node *__restrict__ nodes, uint2 *__restrict__ ranges,
    const uint4 *__restrict__ in_slots, const uint32_t *__restrict__ in_counts, int n_in,
    uint4 *__restrict__ out_slots, uint32_t *__restrict__ out_counts,
    uint32_t *__restrict__ status, int n, PackOut pk) {
	const int g0 = blockIdx.x * kMergeFan;
	const int ng = min(kMergeFan, n_in - g0);
	bottom_up_merge(nodes, ranges, in_slots + (size_t)g0 * kSlots,
	                in_counts + g0, ng,
	                out_slots ? out_slots + (size_t)blockIdx.x * kSlots : nullptr,
	                out_counts ? out_counts + blockIdx.x : nullptr, status, n, pk);
}

struct BoxesWork {
	uint32_t *visit;     // per inner node (rta_lbvh_build_tree clears them)
	uint2 *ranges;       // per inner node
	uint4 *slots[2];     // frontier entries
	uint32_t *counts[2];
	uint32_t *status;
	size_t total;
};

static BoxesWork carve_boxes(void *base, int n) {
	BoxesWork w{};
	size_t off = 0;
	char *p = reinterpret_cast<char *>(base);
	auto take = [&](size_t bytes) {
		char *r = p ? p + off : nullptr;
		off += (bytes + 255) & ~(size_t)255;
		return r;
	};
	const size_t nb = (size_t)n;
	const size_t chunks = (nb + kChunk - 1) / kChunk;
	w.visit = (uint32_t *)take(nb * 4);
	w.ranges = (uint2 *)take(nb * 8);
	for (int i = 0; i < 2; ++i) {
		w.slots[i] = (uint4 *)take(chunks * kSlots * 16);
		w.counts[i] = (uint32_t *)take(chunks * 4);
	}
	w.status = (uint32_t *)take(4);
	w.total = off;
	return w;
}

__global__ __launch_bounds__(kPermuteBlock) void permute_kernel(
    rta_triangle *__restrict__ out, const rta_triangle *__restrict__ scratch,
    const uint32_t *__restrict__ indices, int n, float4 *__restrict__ tri4) {
	permute_block(out, scratch, indices, n, (int)blockIdx.x, tri4);
}

// --------------------------------------------------------- workspace

static inline size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

struct LbvhWorkspace {
	rta_triangle *scratch;
	rta_aabb *boxes;
	rta_float3 *centers;
	rta_aabb *partials;
	rta_aabb *bounds;
	uint32_t *codes;
	void *boxes_work;
	void *sort_work;
	size_t sort_bytes;
	size_t total;
};

static LbvhWorkspace carve(void *base, int n) {
	LbvhWorkspace w{};
	size_t off = 0;
	char *p = reinterpret_cast<char *>(base);
	auto take = [&](size_t bytes) {
		char *r = p ? p + off : nullptr;
		off += align256(bytes);
		return r;
	};
	const size_t nb = (size_t)n;
	const size_t nparts = (nb + kInitBlock - 1) / kInitBlock;
	w.scratch = (rta_triangle *)take(nb * sizeof(rta_triangle));
	w.boxes = (rta_aabb *)take(nb * sizeof(rta_aabb));
	w.centers = (rta_float3 *)take(nb * sizeof(rta_float3));
	w.partials = (rta_aabb *)take(nparts * sizeof(rta_aabb));
	w.bounds = (rta_aabb *)take(sizeof(rta_aabb));
	w.codes = (uint32_t *)take(nb * 4);
	w.boxes_work = take(carve_boxes(nullptr, n).total);
	size_t sb = 0;
	rta_lbvh_sort_work_bytes(n, &sb);
	w.sort_work = take(sb);
	w.sort_bytes = sb;
	w.total = off;
	return w;
}

}  // namespace rta_hip

using namespace rta_hip;

extern "C" {

int rta_lbvh_init_triangles(rta_triangle *scratch, const rta_triangle *src, rta_aabb *boxes,
                            rta_float3 *centers, rta_aabb *partials, int n, rta_stream s) {
	if (n <= 0) return invalid("rta_lbvh_init_triangles: n must be > 0");
	if (!scratch || !src || !boxes || !centers || !partials)
		return invalid("rta_lbvh_init_triangles: NULL pointer");
	hipLaunchKernelGGL(init_triangles_kernel, dim3(grid_for(n, kInitBlock)), dim3(kInitBlock), 0,
	                   as_stream(s), scratch, src, boxes, centers, partials, n, (uint32_t *)nullptr,
	                   (uint32_t *)nullptr);
	RTA_LAUNCH_CHECK("init_triangles_kernel");
	return RTA_OK;
}

int rta_lbvh_voxel_bounds(rta_aabb *bounds, const rta_aabb *partials, int n, rta_stream s) {
	if (n <= 0) return invalid("rta_lbvh_voxel_bounds: n must be > 0");
	if (!bounds || !partials) return invalid("rta_lbvh_voxel_bounds: NULL pointer");
	const int np = (int)grid_for(n, kInitBlock);
	hipLaunchKernelGGL(voxel_bounds_kernel, dim3(1), dim3(kBoundsBlock), 0, as_stream(s), bounds,
	                   partials, np);
	RTA_LAUNCH_CHECK("voxel_bounds_kernel");
	return RTA_OK;
}

int rta_lbvh_morton_codes(uint32_t *codes, uint32_t *indices, const rta_float3 *centers,
                          const rta_aabb *bounds, uint32_t *status, int n, rta_stream s) {
	if (n <= 0) return invalid("rta_lbvh_morton_codes: n must be > 0");
	if (!codes || !indices || !centers || !bounds)
		return invalid("rta_lbvh_morton_codes: NULL pointer");
	hipLaunchKernelGGL(morton_kernel, dim3(grid_for(n, 256)), dim3(256), 0, as_stream(s), codes,
	                   indices, centers, bounds, status, n);
	RTA_LAUNCH_CHECK("morton_kernel");
	return RTA_OK;
}

int rta_lbvh_boxes_work_bytes(int n, size_t *bytes) {
	if (n <= 0 || !bytes) return invalid("rta_lbvh_boxes_work_bytes: bad arguments");
	*bytes = carve_boxes(nullptr, n).total;
	return RTA_OK;
}

int rta_lbvh_build_tree(rta_node *nodes, uint32_t *parents, void *work, const uint32_t *codes,
                        int n, rta_stream s) {
	if (n <= 0) return invalid("rta_lbvh_build_tree: n must be > 0");
	if (!nodes || !parents || !codes || !work) return invalid("rta_lbvh_build_tree: NULL pointer");
	BoxesWork w = carve_boxes(work, n);
	// the bottom-up stage ORs RTA_LBVH_FRONTIER_OVERFLOW into this word
	const int rc = rta_hip_fill_u32(w.status, 0u, 1, s);
	if (rc != RTA_OK) return rc;
	hipLaunchKernelGGL(karras_kernel, dim3(grid_for(2LL * n - 1, kKarrasBlock)), dim3(kKarrasBlock), 0,
	                   as_stream(s), nodes, parents, w.visit, w.ranges, codes, n);
	RTA_LAUNCH_CHECK("karras_kernel");
	return RTA_OK;
}

}  // extern "C"

// The bottom-up stage, which also emits the hierarchy (every node whole,
// and the inner nodes' ranges); a frontier overflow sets
// RTA_LBVH_FRONTIER_OVERFLOW in *status (the workspace's own word when
// status is null).
static int build_boxes(rta_node *nodes, void *work, const rta_aabb *boxes, const uint32_t *codes,
                       const uint32_t *indices, int n, uint32_t *status, rta_stream s,
                       PackOut pk = PackOut{}) {
	BoxesWork w = carve_boxes(work, n);
	if (!status) {
		status = w.status;
		const int rc = rta_hip_fill_u32(status, 0u, 1, s);
		if (rc != RTA_OK) return rc;
	}
	hipStream_t st = as_stream(s);
	int groups = (int)grid_for(n, kChunk);
	hipLaunchKernelGGL(bottom_up_chunk_kernel, dim3(groups), dim3(kChunk), 0, st, nodes, boxes,
	                   codes, indices, w.ranges, w.slots[0], w.counts[0], status, n, pk);
	RTA_LAUNCH_CHECK("bottom_up_chunk_kernel");
	int in = 0;
	while (groups > 1) {
		const int blocks = (groups + kMergeFan - 1) / kMergeFan;
		hipLaunchKernelGGL(bottom_up_merge_kernel, dim3(blocks), dim3(kMergeThreads), 0, st, nodes,
		                   w.ranges, w.slots[in], w.counts[in], groups,
		                   blocks > 1 ? w.slots[1 - in] : nullptr,
		                   blocks > 1 ? w.counts[1 - in] : nullptr, status, n, pk);
		RTA_LAUNCH_CHECK("bottom_up_merge_kernel");
		groups = blocks;
		in = 1 - in;
	}
	return RTA_OK;
}

extern "C" {

int rta_lbvh_build_boxes(rta_node *nodes, void *work, const rta_aabb *boxes,
                         const uint32_t *codes, const uint32_t *indices,
                         const uint32_t *parents, int n, rta_stream s) {
	if (n <= 0) return invalid("rta_lbvh_build_boxes: n must be > 0");
	(void)parents;   // the climb derives the hierarchy from the codes
	if (!nodes || !boxes || !codes || !indices || !work)
		return invalid("rta_lbvh_build_boxes: NULL pointer");
	return build_boxes(nodes, work, boxes, codes, indices, n, nullptr, s);
}

int rta_lbvh_permute(rta_triangle *out, const rta_triangle *scratch, const uint32_t *indices,
                     int n, rta_stream s) {
	if (n <= 0) return invalid("rta_lbvh_permute: n must be > 0");
	if (!out || !scratch || !indices) return invalid("rta_lbvh_permute: NULL pointer");
	hipLaunchKernelGGL(permute_kernel, dim3(grid_for(n, kPermuteBlock)), dim3(kPermuteBlock), 0,
	                   as_stream(s), out, scratch, indices, n, (float4 *)nullptr);
	RTA_LAUNCH_CHECK("permute_kernel");
	return RTA_OK;
}

int rta_lbvh_workspace_bytes(int n, size_t *bytes) {
	if (n <= 0 || !bytes) return invalid("rta_lbvh_workspace_bytes: bad arguments");
	*bytes = carve(nullptr, n).total;
	return RTA_OK;
}

int rta_lbvh_copy_ranges(uint32_t *ranges, const void *workspace, int n, rta_stream s) {
	if (n <= 0 || !ranges || !workspace) return invalid("rta_lbvh_copy_ranges: bad arguments");
	if (n == 1) return RTA_OK;
	LbvhWorkspace w = carve(const_cast<void *>(workspace), n);
	BoxesWork b = carve_boxes(w.boxes_work, n);
	RTA_HIP_TRY(hipMemcpyAsync(ranges, b.ranges, (size_t)(n - 1) * 8, hipMemcpyDeviceToDevice,
	                           as_stream(s)));
	return RTA_OK;
}

}  // extern "C"

// Stages 2 to 4 of a small mesh (small_sort_kernel).
static int small_sort(uint32_t *indices, const LbvhWorkspace &w, uint32_t *status, int n,
                      hipStream_t st) {
	const int np = (int)grid_for(n, kInitBlock), items = (int)grid_for(n, kSmallThreads);
	auto launch = [&](auto kernel) {
		hipLaunchKernelGGL(kernel, dim3(1), dim3(kSmallThreads), 0, st, w.codes, indices,
		                   (const rta_float3 *)w.centers, (const rta_aabb *)w.partials, np, status, n);
	};
	if (items <= 1) launch(small_sort_kernel<1>);
	else if (items <= 2) launch(small_sort_kernel<2>);
	else if (items <= 4) launch(small_sort_kernel<4>);
	else launch(small_sort_kernel<kSmallItems>);
	RTA_LAUNCH_CHECK("small_sort_kernel");
	return RTA_OK;
}

// The seven stages (lbvh_constructor::buildCUDA, bbvh-cuda/lbvh.h:153-211).
// With pk set, the permutation also writes tri4 and runs before the
// bottom-up pass, which writes the pair records (and clears the leaf-end
// marks that collapses make interior), so the traversal layout needs no
// pass of its own; the times then follow that order.
static int build_impl(const char *name, rta_triangle *tris, int n, rta_node *nodes,
                      uint32_t *indices, void *workspace, size_t workspace_bytes,
                      uint32_t *status, rta_lbvh_times *times, rta_stream s, PackOut pk) {
	const ScopedRange range(name);
	// n = 0 is rejected, as the reference cannot build it (bbvh-cuda/lbvh.h:47)
	if (n <= 0) return invalid((std::string(name) + ": n must be > 0").c_str());
	if (!tris || !nodes || !indices || !workspace)
		return invalid((std::string(name) + ": NULL pointer").c_str());
	LbvhWorkspace w = carve(workspace, n);
	if (workspace_bytes < w.total) {
		set_error(std::string(name) + ": workspace too small");
		return RTA_E_WORKSPACE;
	}
	hipEvent_t ev[8] = {};
	if (times) {
		for (int i = 0; i < 8; ++i) RTA_HIP_TRY(hipEventCreate(&ev[i]));
		RTA_HIP_TRY(hipEventRecord(ev[0], as_stream(s)));
	}
	int rc = RTA_OK;
	auto mark = [&](int k) {
		if (times && rc == RTA_OK) {
			hipError_t e = hipEventRecord(ev[k], as_stream(s));
			if (e != hipSuccess) rc = hip_status(e, "hipEventRecord");
		}
	};
	const bool packed = pk.pairs != nullptr;
	auto permute = [&]() {
		if (rc != RTA_OK) return;
		hipLaunchKernelGGL(permute_kernel, dim3(grid_for(n, kPermuteBlock)), dim3(kPermuteBlock),
		                   0, as_stream(s), tris, w.scratch, indices, n, pk.tri4);
		const hipError_t e = hipGetLastError();
		if (e != hipSuccess) rc = hip_status(e, "permute_kernel");
	};
	hipLaunchKernelGGL(init_triangles_kernel, dim3(grid_for(n, kInitBlock)), dim3(kInitBlock), 0,
	                   as_stream(s), w.scratch, tris, w.boxes, w.centers, w.partials, n, status,
	                   pk.flags);
	{
		const hipError_t e = hipGetLastError();
		if (e != hipSuccess) rc = hip_status(e, "init_triangles_kernel");
	}
	mark(1);
	if (n <= kSmallSort) {
		mark(2);
		mark(3);
		if (rc == RTA_OK) rc = small_sort(indices, w, status, n, as_stream(s));
	} else {
		if (rc == RTA_OK) rc = rta_lbvh_voxel_bounds(w.bounds, w.partials, n, s);
		mark(2);
		// into the sort's second buffers: its three passes end in codes/indices
		uint32_t *keys, *vals;
		radix_alt_buffers(w.sort_work, n, &keys, &vals);
		if (rc == RTA_OK) rc = rta_lbvh_morton_codes(keys, vals, w.centers, w.bounds, status, n, s);
		mark(3);
		if (rc == RTA_OK) rc = radix_sort_codes(w.codes, indices, n, w.sort_work, as_stream(s));
	}
	mark(4);
	// the hierarchy is emitted by the bottom-up stage: no pass of its own
	mark(5);
	if (packed) {
		permute();
		mark(6);
		if (rc == RTA_OK)
			rc = build_boxes(nodes, w.boxes_work, w.boxes, w.codes, indices, n, status, s, pk);
		mark(7);
	} else {
		if (rc == RTA_OK)
			rc = build_boxes(nodes, w.boxes_work, w.boxes, w.codes, indices, n, status, s);
		mark(6);
		permute();
		mark(7);
	}
	if (times) {
		if (rc == RTA_OK) {
			hipError_t e = hipEventSynchronize(ev[7]);
			if (e != hipSuccess) rc = hip_status(e, "hipEventSynchronize");
		}
		if (rc == RTA_OK) {
			float *slots[7] = {&times->init_triangles, &times->voxel_bounds, &times->morton,
			                   &times->sort, &times->tree,
			                   packed ? &times->permute : &times->boxes,
			                   packed ? &times->boxes : &times->permute};
			for (int k = 0; k < 7; ++k) (void)hipEventElapsedTime(slots[k], ev[k], ev[k + 1]);
			(void)hipEventElapsedTime(&times->total, ev[0], ev[7]);
		}
		for (int i = 0; i < 8; ++i) (void)hipEventDestroy(ev[i]);
	}
	return rc;
}

extern "C" {

int rta_lbvh_build(rta_triangle *tris, int n, rta_node *nodes, uint32_t *indices, void *workspace,
                   size_t workspace_bytes, uint32_t *status, rta_lbvh_times *times,
                   rta_stream s) {
	RTA_FAULT_POINT("rta_lbvh_build");
	return build_impl("rta_lbvh_build", tris, n, nodes, indices, workspace, workspace_bytes,
	                  status, times, s, PackOut{});
}

int rta_lbvh_build_packed(rta_triangle *tris, int n, rta_node *nodes, uint32_t *indices,
                          rta_node_pair *pairs, float *tri4, uint32_t *flags, void *workspace,
                          size_t workspace_bytes, uint32_t *status, rta_lbvh_times *times,
                          rta_stream s) {
	RTA_FAULT_POINT("rta_lbvh_build_packed");
	if (!pairs || !tri4 || !flags) return invalid("rta_lbvh_build_packed: NULL layout pointer");
	PackOut pk;
	pk.pairs = pairs;
	pk.tri4 = reinterpret_cast<float4 *>(tri4);
	pk.flags = flags;
	return build_impl("rta_lbvh_build_packed", tris, n, nodes, indices, workspace,
	                  workspace_bytes, status, times, s, pk);
}

}  // extern "C"
