// Stable LSD radix sort of 30-bit Morton codes with a uint32 payload
// (the reference's thrust::sort_by_key, bbvh-cuda/lbvh-kernels.cu:537-555).
//
// Reduce-then-scan by digits of up to 10 bits (three passes for a code), a
// pass in two or three kernels:
//   1. per-tile digit histograms (LDS counters)           hist[tile][digit]
//   2. many tiles only: exclusive scan over tiles per digit, digit totals
//      (with few tiles every block of the third kernel sums the rows itself)
//   3. per-tile stable ranking with wave ballots (match-any over the digit
//      bits, popcount of the lower-lane mask) on counters of each wave's own,
//      then a digit-grouped write of the tile (contiguous runs per digit).
// No kernel waits on another block, so there is no spin loop anywhere.
// A stable sort is unique, so the output equals std::stable_sort by code.
//
// What bounds it: launches and the latency of one tile below a few hundred
// thousand keys, the scattered writes above.  Against four passes of 8-bit
// digits in 256-thread tiles, whole builds: 14,000 triangles 108 -> 81 us,
// 82,000 134 -> 111, 262,144 159 -> 137, 2.3 M 668 -> 645.
#include "internal.hpp"

#include <utility>

namespace rta_hip {

constexpr int kBits = 10;
constexpr int kBins = 1 << kBits;
constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / kWave;
static_assert(kBins == kThreads, "one digit per thread in the scan helpers");

// The digit of an entry: bits [shift, shift + bits) of its key, or of its
// payload.
struct Digit {
	int shift;
	uint32_t mask;
	bool of_val;
	__device__ uint32_t operator()(uint32_t k, uint32_t v) const {
		return ((of_val ? v : k) >> shift) & mask;
	}
};

// exclusive scan of one value per thread over the block
__device__ inline uint32_t block_exclusive_scan(uint32_t v, uint32_t *wave_sums) {
	const int lane = __lane_id();
	const int wv = threadIdx.x / kWave;
	uint32_t x = v;
	for (int off = 1; off < kWave; off <<= 1) {
		const uint32_t y = __shfl_up(x, off);
		if (lane >= off) x += y;
	}
	if (lane == kWave - 1) wave_sums[wv] = x;
	__syncthreads();
	uint32_t before = 0;
	for (int w = 0; w < kWaves; ++w) before += w < wv ? wave_sums[w] : 0u;
	__syncthreads();
	return before + x - v;
}

template <int ITEMS>
__global__ __launch_bounds__(kThreads) void rs_hist_kernel(const uint32_t *__restrict__ keys,
                                                           const uint32_t *__restrict__ vals, int n,
                                                           Digit digit, uint32_t *__restrict__ hist) {
	__shared__ uint32_t h[kBins];
	h[threadIdx.x] = 0;
	__syncthreads();
	const uint32_t *src = digit.of_val ? vals : keys;
	const long long base = (long long)blockIdx.x * (kThreads * ITEMS);
	uint32_t k[ITEMS];
#pragma unroll
	for (int it = 0; it < ITEMS; ++it) {
		const long long idx = base + it * kThreads + threadIdx.x;
		k[it] = idx < n ? src[idx] : 0u;
	}
#pragma unroll
	for (int it = 0; it < ITEMS; ++it)
		if (base + it * kThreads + threadIdx.x < n) atomicAdd(&h[(k[it] >> digit.shift) & digit.mask], 1u);
	__syncthreads();
	hist[(size_t)blockIdx.x * kBins + threadIdx.x] = h[threadIdx.x];
}

// exclusive scan of hist[0..tiles)[digit] in place and the digit's total; a
// block takes kScanDigits digits, and per digit kScanParts threads take
// consecutive shares of the tiles
constexpr int kScanDigits = 16, kScanParts = kThreads / kScanDigits;
__global__ __launch_bounds__(kThreads) void rs_scan_kernel(uint32_t *__restrict__ hist, int tiles,
                                                           uint32_t *__restrict__ totals) {
	__shared__ uint32_t part[kScanParts][kScanDigits];
	const int d = threadIdx.x % kScanDigits, q = threadIdx.x / kScanDigits;
	const int per = (tiles + kScanParts - 1) / kScanParts;
	const int first = min(q * per, tiles), last = min(first + per, tiles);
	uint32_t *col = hist + blockIdx.x * kScanDigits + d;
	uint32_t sum = 0;
#pragma unroll 8
	for (int i = first; i < last; ++i) sum += col[(size_t)i * kBins];
	part[q][d] = sum;
	__syncthreads();
	// one wave per digit turns its kScanParts = 64 sums into prefixes
	{
		const int lane = __lane_id(), dd = threadIdx.x / kWave;
		uint32_t x = part[lane][dd];
		const uint32_t v = x;
		for (int off = 1; off < kWave; off <<= 1) {
			const uint32_t y = __shfl_up(x, off);
			if (lane >= off) x += y;
		}
		part[lane][dd] = x - v;
		if (lane == kWave - 1) totals[blockIdx.x * kScanDigits + dd] = x;
	}
	__syncthreads();
	uint32_t run = part[q][d];
#pragma unroll 8
	for (int i = first; i < last; ++i) {
		const uint32_t c = col[(size_t)i * kBins];
		col[(size_t)i * kBins] = run;
		run += c;
	}
}
static_assert(kScanParts == kWave && kThreads / kWave == kScanDigits, "a wave per digit");

// Tiles are handed to the XCDs in contiguous eighths: neighbouring tiles'
// runs of a digit are neighbours in the output, so one L2 completes their
// lines (4 M triangles: 1,022 -> 1,006 us a build, 2.3 M: 650 -> 645).
__device__ inline int xcd_tile(int tiles) {
	const int per = (tiles + 7) / 8;
	return (int)(blockIdx.x % 8u) * per + (int)(blockIdx.x / 8u);
}

// Per tile: rank every key among the tile's keys of its digit in index
// order (stable), then write the tile's keys grouped by digit so that each
// digit's run is stored contiguously.
//  1. wave w takes the tile's keys [w * 64 * ITEMS, +64 * ITEMS) in order and
//     ranks them with ballots on its own counters: a key's rank is the
//     digit's count so far plus its lower lanes with that digit;
//  2. one thread per digit turns the waves' counts -- the tile's index order
//     -- into exclusive prefixes and the digit's tile total;
//  3. a key's position in the tile is its digit's start in the tile plus
//     its wave's prefix plus its rank; keys and payloads go to LDS there,
//     and the block writes them out in tile order, key j of digit d to
//     digit_base[d] + (j - start of d in the tile).
// SELF: hist holds the tiles' counts, and the block sums the rows before its
// own and all of them; otherwise hist and totals are rs_scan_kernel's.
// keep: the payload's bits that are stored.
template <int ITEMS, bool SELF>
__global__ __launch_bounds__(kThreads) void rs_scatter_kernel(
    const uint32_t *__restrict__ keys_in, const uint32_t *__restrict__ vals_in,
    uint32_t *__restrict__ keys_out, uint32_t *__restrict__ vals_out, int n, Digit digit,
    const uint32_t *__restrict__ hist, const uint32_t *__restrict__ totals, int tiles, uint32_t keep) {
	constexpr int kTile = kThreads * ITEMS;
	__shared__ union {
		uint16_t cnt[kWaves][kBins];  // per wave: counts, then their prefixes
		uint32_t kv[2][kTile];        // the tile's keys and payloads by digit
	} sm;
	__shared__ uint32_t gbase[kBins];        // where digit d of this tile starts in the output
	__shared__ uint32_t lbase[kBins];        // where digit d starts within the tile
	__shared__ uint32_t wave_sums[kWaves];

	const int t = threadIdx.x, lane = __lane_id(), wv = t / kWave;
	const int tile = xcd_tile(tiles);
	if (tile >= tiles) return;
	uint32_t *cnt_words = reinterpret_cast<uint32_t *>(&sm.cnt[0][0]);
#pragma unroll
	for (int i = 0; i < kWaves * kBins / 2 / kThreads; ++i) cnt_words[t + i * kThreads] = 0u;

	const long long tile_base = (long long)tile * kTile;
	const int count = (int)min((long long)kTile, (long long)n - tile_base);
	uint32_t key[ITEMS], val[ITEMS], pos[ITEMS];
#pragma unroll
	for (int it = 0; it < ITEMS; ++it) {
		const int j = (wv * ITEMS + it) * kWave + lane;
		key[it] = j < count ? keys_in[tile_base + j] : 0u;
		val[it] = j < count ? vals_in[tile_base + j] : 0u;
	}
	uint32_t before = 0, total = 0;
	if (SELF) {
#pragma unroll 8
		for (int i = 0; i < tiles; ++i) {
			const uint32_t c = hist[(size_t)i * kBins + t];
			before += i < tile ? c : 0u;
			total += c;
		}
	} else {
		before = hist[(size_t)tile * kBins + t];
		total = totals[t];
	}
	gbase[t] = block_exclusive_scan(total, wave_sums) + before;   // its barriers also end the clearing

	const uint64_t lt = (1ull << lane) - 1ull;
#pragma unroll
	for (int it = 0; it < ITEMS; ++it) {
		const bool valid = (wv * ITEMS + it) * kWave + lane < count;
		const uint32_t d = digit(key[it], val[it]);
		uint64_t match = __ballot(valid);
#pragma unroll
		for (int b = 0; b < kBits; ++b) {
			const bool bit = (d >> b) & 1u;
			const uint64_t m = __ballot(bit);
			match &= bit ? m : ~m;
		}
		const uint32_t rank = (uint32_t)__popcll(match & lt);
		const uint32_t so_far = sm.cnt[wv][d];
		pos[it] = so_far + rank;
		// the wave's own counter: LDS operations of a wave stay in order
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
		if (valid && rank == 0u) sm.cnt[wv][d] = (uint16_t)(so_far + (uint32_t)__popcll(match));
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
	}
	__syncthreads();
	uint32_t run = 0;
#pragma unroll
	for (int w = 0; w < kWaves; ++w) {
		const uint32_t c = sm.cnt[w][t];
		sm.cnt[w][t] = (uint16_t)run;
		run += c;
	}
	lbase[t] = block_exclusive_scan(run, wave_sums);
	__syncthreads();
#pragma unroll
	for (int it = 0; it < ITEMS; ++it) {
		const uint32_t d = digit(key[it], val[it]);
		pos[it] += lbase[d] + sm.cnt[wv][d];
	}
	__syncthreads();  // the counts are dead; their LDS now holds the tile
#pragma unroll
	for (int it = 0; it < ITEMS; ++it) {
		if ((wv * ITEMS + it) * kWave + lane < count) {
			sm.kv[0][pos[it]] = key[it];
			sm.kv[1][pos[it]] = val[it];
		}
	}
	__syncthreads();
#pragma unroll
	for (int it = 0; it < ITEMS; ++it) {
		const int j = t + it * kThreads;
		if (j >= count) continue;
		const uint32_t k = sm.kv[0][j], v = sm.kv[1][j];
		const uint32_t d = digit(k, v);
		const uint32_t o = gbase[d] + ((uint32_t)j - lbase[d]);
		if (o < (uint32_t)n) {  // always true for consistent histograms
			keys_out[o] = k;
			vals_out[o] = v & keep;
		}
	}
}

static inline size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// Keys per thread: small tiles while there are few, so that more CUs share
// the latency of a tile; large ones (longer runs per digit) once they fill
// the machine.  2 / 4 / 8 keys, whole builds: 200,000 triangles 134 / 140 /
// 146 us, 524,288 198 / 197 / 221, 2.3 M 658 / 645 / 664, 4 M 1,050 / 1,006 /
// 1,013.
static int radix_items(int n) { return n <= (1 << 19) ? 2 : 4; }
// Up to this many tiles the scatter's blocks sum the histogram rows
// themselves (a launch saved; the reads grow with the square): 7 tiles 80.6
// against 83.4 us a build, 15 tiles 98.4 / 99.3, 32 tiles 108.1 / 107.4, 64
// tiles 125 / 115.
constexpr int kSelfTiles = 24;

struct RadixWork {
	uint32_t *alt_keys, *alt_vals, *hist, *totals;
	size_t total;
};

static RadixWork carve_radix(void *base, int n) {
	RadixWork w{};
	size_t off = 0;
	char *p = reinterpret_cast<char *>(base);
	auto take = [&](size_t bytes) {
		uint32_t *r = reinterpret_cast<uint32_t *>(p ? p + off : nullptr);
		off += align256(bytes);
		return r;
	};
	// by the smallest tile, so that a larger n never needs less
	constexpr size_t tile = (size_t)kThreads * 2;
	w.alt_keys = take((size_t)n * 4);
	w.alt_vals = take((size_t)n * 4);
	w.hist = take(((size_t)n + tile - 1) / tile * kBins * 4);
	w.totals = take(kBins * 4);
	w.total = off;
	return w;
}

size_t radix_work_bytes(int n) { return carve_radix(nullptr, n).total; }

void radix_alt_buffers(void *work, int n, uint32_t **keys, uint32_t **vals) {
	const RadixWork w = carve_radix(work, n);
	*keys = w.alt_keys;
	*vals = w.alt_vals;
}

template <int ITEMS>
static int radix_pass_items(const uint32_t *kin, const uint32_t *vin, uint32_t *kout, uint32_t *vout,
                            int n, Digit digit, uint32_t keep, const RadixWork &w, hipStream_t st) {
	const int tiles = (int)(((size_t)n + kThreads * ITEMS - 1) / (kThreads * ITEMS));
	hipLaunchKernelGGL((rs_hist_kernel<ITEMS>), dim3(tiles), dim3(kThreads), 0, st, kin, vin, n, digit,
	                   w.hist);
	RTA_LAUNCH_CHECK("rs_hist_kernel");
	if (tiles <= kSelfTiles) {
		hipLaunchKernelGGL((rs_scatter_kernel<ITEMS, true>), dim3((tiles + 7) / 8 * 8), dim3(kThreads), 0, st, kin, vin,
		                   kout, vout, n, digit, w.hist, w.totals, tiles, keep);
	} else {
		hipLaunchKernelGGL(rs_scan_kernel, dim3(kBins / kScanDigits), dim3(kThreads), 0, st, w.hist, tiles,
		                   w.totals);
		RTA_LAUNCH_CHECK("rs_scan_kernel");
		hipLaunchKernelGGL((rs_scatter_kernel<ITEMS, false>), dim3((tiles + 7) / 8 * 8), dim3(kThreads), 0, st, kin, vin,
		                   kout, vout, n, digit, w.hist, w.totals, tiles, keep);
	}
	RTA_LAUNCH_CHECK("rs_scatter_kernel");
	return RTA_OK;
}

int radix_pass(const uint32_t *kin, const uint32_t *vin, uint32_t *kout, uint32_t *vout, int n,
               int shift, int bits, bool of_val, uint32_t keep, void *work, hipStream_t st) {
	const RadixWork w = carve_radix(work, n);
	const Digit digit{shift, (1u << bits) - 1u, of_val};
	if (radix_items(n) == 2) return radix_pass_items<2>(kin, vin, kout, vout, n, digit, keep, w, st);
	return radix_pass_items<4>(kin, vin, kout, vout, n, digit, keep, w, st);
}

int radix_sort_codes(uint32_t *keys, uint32_t *vals, int n, void *work, hipStream_t st) {
	const RadixWork w = carve_radix(work, n);
	int rc = RTA_OK;
	uint32_t *kin = w.alt_keys, *vin = w.alt_vals, *kout = keys, *vout = vals;
	for (int shift = 0; shift < 30 && rc == RTA_OK; shift += kBits) {
		rc = radix_pass(kin, vin, kout, vout, n, shift, kBits, false, ~0u, work, st);
		std::swap(kin, kout);
		std::swap(vin, vout);
	}
	return rc;
}

}  // namespace rta_hip

using namespace rta_hip;

extern "C" {

int rta_lbvh_sort_work_bytes(int n, size_t *bytes) {
	if (n <= 0 || !bytes) return invalid("rta_lbvh_sort_work_bytes: bad arguments");
	*bytes = radix_work_bytes(n);
	return RTA_OK;
}

int rta_lbvh_sort(uint32_t *codes, uint32_t *indices, int n, void *work, size_t work_bytes,
                  rta_stream s) {
	if (n <= 0) return invalid("rta_lbvh_sort: n must be > 0");
	if (!codes || !indices || !work) return invalid("rta_lbvh_sort: NULL pointer");
	if (work_bytes < radix_work_bytes(n)) {
		set_error("rta_lbvh_sort: work buffer too small");
		return RTA_E_WORKSPACE;
	}
	// four passes over all 32 bits: an even number leaves the result in
	// codes/indices
	uint32_t *ak, *av;
	radix_alt_buffers(work, n, &ak, &av);
	for (int shift = 0; shift < 32; shift += 16) {
		int rc = radix_pass(codes, indices, ak, av, n, shift, 8, false, ~0u, work, as_stream(s));
		if (rc == RTA_OK)
			rc = radix_pass(ak, av, codes, indices, n, shift + 8, 8, false, ~0u, work, as_stream(s));
		if (rc != RTA_OK) return rc;
	}
	return RTA_OK;
}

}  // extern "C"
