/*
 * Signal delivery on the GPU: a batch of signal work items becomes one launch of 64-bit
 * device-scope atomic adds on the counters in HBM.
 *
 * The reference updates each counter from a CPU worker thread through GDRCopy -- a PCIe
 * read and a PCIe write per slot (apply_signal_work, src/rdma/gin/nccl_ofi_gin.cpp:
 * 1193-1256) -- and therefore folds a batch by slot first to save round trips
 * (apply_and_complete, :1425-1479).  Here a workgroup whose items crowd on few lines of counters
 * folds them in an LDS table keyed by the counter's address and adds each sum once; the others
 * add item by item.  Additions are commutative, so every counter ends at the value that N single
 * adds leave.
 *
 * What bounds it: adds to one 64-byte line of counters follow each other at 12 ns, whatever
 * their XCD, so a batch on few counters is a queue at the memory (262,144 items on one counter
 * 3148 us, on 64 counters 311 us, on 262,144 counters 14 us, items in HBM); items in pinned host
 * memory come over the host link (32 B each, 8 MiB in 155 us at 54 GB/s).
 */
#include "common.hpp"
#include "ofi_amd_hotpath.h"

namespace {

constexpr uint32_t kMaxRegions = 16;
constexpr uint32_t kMaxApplyPost = 65536; /* items one workgroup applies in front of a flush read */
constexpr uint32_t kProbes = 4;           /* entries of the fold an item looks at */

struct regions_t {
	uint64_t base[kMaxRegions];
	uint64_t size[kMaxRegions];
	uint64_t *counters[kMaxRegions];
	uint32_t n;
};

/* What a workgroup keeps in LDS: the regions, indexed per lane, and the fold of its items. */
template <uint32_t kSlots> struct fold_t {
	unsigned long long key[kSlots]; /* address of a counter; 0: free */
	unsigned long long sum[kSlots];
	uint32_t used; /* whether anything went into it */
	uint64_t base[kMaxRegions], size[kMaxRegions];
	uint64_t *counters[kMaxRegions];
};

/* Before any item, by the whole workgroup; `fold`: whether items may go into the fold.  The regions (a single
 * one stays in scalar registers) are written by the first four wavefronts, each a quarter of them, from scalars: a
 * lane's own index into the kernel's arguments is a vector load from host memory, a link's round trip of 0.7 us. */
template <uint32_t kSlots>
__device__ __forceinline__ void begin(fold_t<kSlots> &f, const regions_t &regions, bool fold, uint32_t threads)
{
	if (fold) {
		for (uint32_t i = threadIdx.x; i < kSlots; i += threads) {
			f.key[i] = 0;
			f.sum[i] = 0;
		}
		if (threadIdx.x == 0) {
			f.used = 0;
		}
	}
	if (regions.n > 1 && (threadIdx.x & 63u) == 0) {
		const uint32_t wave = threadIdx.x >> 6;
#pragma unroll
		for (uint32_t r = 0; r < kMaxRegions; r++) {
			if (r / 4 == wave && r < regions.n) {
				f.base[r] = regions.base[r];
				f.size[r] = regions.size[r];
				f.counters[r] = regions.counters[r];
			}
		}
	}
	if (fold || regions.n > 1) {
		__syncthreads();
	}
}

/* The counter of a work item, nullptr if it has none.  The window is found by its base; the
 * counter by its address inside the window, which may continue through the regions listed next
 * while each begins where the one before it ends (a window backed by several allocations: the
 * reference looks the segment up by address too, ensure_signal_seg,
 * src/rdma/gin/nccl_ofi_gin.cpp:1038-1122, 1156-1166).  The bases are compared straight through
 * (they sit in scalar registers, the first match wins); only what follows differs from lane to
 * lane and is read from LDS.  A loop that left at the match walked the regions once per
 * distinct base of a wavefront, with a dependent load each: 4096 items a workgroup over 16
 * regions took 24 us. */
template <uint32_t kSlots>
__device__ __forceinline__ uint64_t *slot_of(const fold_t<kSlots> &f, const regions_t &regions, uint64_t base,
					     uint64_t offset)
{
	if (regions.n == 1) {
		const uint64_t size = regions.size[0];
		const bool ok = base == regions.base[0] && (offset & 7u) == 0 && offset <= size && size - offset >= 8;
		return ok ? regions.counters[0] + (offset >> 3) : nullptr;
	}
	uint32_t r = kMaxRegions;
#pragma unroll
	for (int k = (int)kMaxRegions - 1; k >= 0; k--) {
		r = (uint32_t)k < regions.n && base == regions.base[k] ? (uint32_t)k : r;
	}
	if (r == kMaxRegions || (offset & 7u) != 0) {
		return nullptr;
	}
	for (uint64_t off = offset;; r++) {
		const uint64_t size = f.size[r];
		if (off <= size && size - off >= 8) {
			return f.counters[r] + (off >> 3);
		}
		if (off < size || r + 1 >= regions.n || f.base[r + 1] != f.base[r] + size) {
			return nullptr; /* a counter across the end of a segment, or past the window */
		}
		off -= size;
	}
}

/* Relaxed: ordering against the payload is the put-before-signal protocol's business (the reference uses a relaxed
 * fetch_add on its host path for the same reason, :1209). */
__device__ __forceinline__ void add_directly(uint64_t *slot, uint64_t value)
{
	__hip_atomic_fetch_add(slot, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* One item into the fold; past kProbes entries taken by other counters it goes to its own directly. */
template <uint32_t kSlots> __device__ __forceinline__ void add_to_fold(fold_t<kSlots> &f, uint64_t *slot, uint64_t value)
{
	const unsigned long long key = (unsigned long long)reinterpret_cast<uintptr_t>(slot);
	uint32_t h = ((uint32_t)(key >> 3) * 0x9e3779b1u) >> (32 - __builtin_ctz(kSlots));
	for (uint32_t probe = 0; probe < kProbes; probe++) {
		unsigned long long at = __hip_atomic_load(&f.key[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
		if (at == 0) {
			at = atomicCAS(&f.key[h], 0ull, key);
			at = at == 0 ? key : at;
		}
		if (at == key) {
			__hip_atomic_fetch_add(&f.sum[h], (unsigned long long)value, __ATOMIC_RELAXED,
					       __HIP_MEMORY_SCOPE_WORKGROUP);
			return;
		}
		h = (h + 1) & (kSlots - 1);
	}
	add_directly(slot, value);
}

/*
 * Whether the items of a wavefront crowd on few lines of counters: how many of them share a line with lane 0's, 21's
 * or 42's.  The fold costs a workgroup 0.7-1 us (256 items in HBM on 8192 counters: 2.44 us without, 3.18 with),
 * and what it saves is the queue at a line, 12 ns for each of the batch's items on it, of which those lanes are a
 * sample: it pays from about 24576 / n lanes on (crowd_of), a few more than the three themselves at the least.
 */
constexpr uint32_t kMostCrowded = 3 * 64;
__device__ __forceinline__ bool crowded(const uint64_t *slot, uint32_t crowd)
{
	const uint32_t line = (uint32_t)(reinterpret_cast<uintptr_t>(slot) >> 6);
	const uint64_t with_item = __ballot(slot != nullptr);
	uint32_t same = 0;
#pragma unroll
	for (int lane = 0; lane < 63; lane += 21) {
		same += (uint32_t)__popcll(with_item & __ballot(line == (uint32_t)__builtin_amdgcn_readlane((int)line, lane)));
	}
	return same >= crowd;
}
static uint32_t crowd_of(uint32_t n)
{
	return n < 4096u ? 24576u / n : 6u;
}

/* The item of every lane that has one, by a whole wavefront; `folds` becomes and stays true with the first crowd. */
template <uint32_t kSlots>
__device__ __forceinline__ void add_items(fold_t<kSlots> &f, const regions_t &regions, uint64_t base, uint64_t offset,
					  uint64_t value, bool live, uint32_t crowd, bool &folds,
					  uint32_t *__restrict__ rejected)
{
	uint64_t *slot = nullptr;
	if (live) {
		slot = slot_of(f, regions, base, offset);
		if (slot == nullptr && rejected) {
			atomicAdd(rejected, 1u);
		}
	}
	if (!folds && crowded(slot, crowd)) {
		folds = true;
		f.used = 1;
	}
	if (slot != nullptr) {
		if (folds) {
			add_to_fold(f, slot, value);
		} else {
			add_directly(slot, value);
		}
	}
}

/* Behind the last item, by the whole workgroup: the sums onto the counters.  `folds`: this wavefront's. */
template <uint32_t kSlots> __device__ __forceinline__ void end(fold_t<kSlots> &f, bool folds, uint32_t threads)
{
	__syncthreads();
	if (!folds && f.used == 0) {
		return;
	}
	for (uint32_t i = threadIdx.x; i < kSlots; i += threads) {
		if (f.key[i] != 0) {
			add_directly(reinterpret_cast<uint64_t *>(f.key[i]), (uint64_t)f.sum[i]);
		}
	}
}

template <uint32_t kThreads, uint32_t kItems, uint32_t kSlots>
__global__ __launch_bounds__(kThreads) void gin_signal_apply_kernel(
	const ofi_amd_gin_signal_work_t *__restrict__ work, uint32_t n, regions_t regions, uint32_t crowd,
	uint32_t *__restrict__ rejected)
{
	__shared__ __align__(16) fold_t<kSlots> f;
	uint64_t base[kItems], offset[kItems], value[kItems];
	const uint32_t first = blockIdx.x * (kThreads * kItems) + threadIdx.x;
#pragma unroll
	for (uint32_t k = 0; k < kItems; k++) { /* every item of a thread in flight at once */
		const ofi_amd_gin_signal_work_t *w = work + min(first + k * kThreads, n - 1u);
		base[k] = w->base;
		offset[k] = w->offset;
		value[k] = w->value;
	}
	const bool may_fold = crowd <= kMostCrowded;
	begin(f, regions, may_fold, kThreads);
	bool folds = crowd == 0;
	if (folds) {
		f.used = 1;
	}
#pragma unroll
	for (uint32_t k = 0; k < kItems; k++) {
		add_items(f, regions, base[k], offset[k], value[k], first + k * kThreads < n, crowd, folds, rejected);
	}
	if (may_fold) {
		end(f, folds, kThreads);
	}
}

/* The adds of a batch and the flush read behind them in one launch of one workgroup: every
 * thread's adds have been performed at the memory before the workgroup meets, and only then is
 * the flush buffer read back into the host's slots -- what two launches order by the kernel
 * boundary between them.
 * Bound by the trips for the items, 256 at a time, which is why the next ones are asked for before the last ones
 * are added.  In us, items in host memory, every item added by itself / every item folded / as it is:
 *   1 item                         4.5 / 5.3 / 4.4
 *   256 items, 8192 counters       4.9 / 6.0 / 4.9
 *   1024 items, 8192 counters      12.5 / 15.0 / 9.2
 *   4096 items, 1 counter          95 / 31 / 24
 *   65536 items, 64 counters       870 / 441 / 330 */
constexpr uint32_t kPostThreads = 256, kPostSlots = 1024;
__global__ __launch_bounds__(kPostThreads) void gin_signal_apply_post_kernel(
	const ofi_amd_gin_signal_work_t *__restrict__ work, uint32_t n, regions_t regions, uint32_t crowd,
	uint32_t *__restrict__ rejected, const uint64_t *__restrict__ flush_buf, uint64_t *__restrict__ slots,
	uint32_t num_rails)
{
	__shared__ __align__(16) fold_t<kPostSlots> f;
	if (n != 0) {
		uint64_t base, offset, value;
		auto load = [&](uint32_t at) {
			const ofi_amd_gin_signal_work_t *w = work + min(at + threadIdx.x, n - 1u);
			base = w->base;
			offset = w->offset;
			value = w->value;
		};
		load(0); /* on its way while the fold is prepared */
		const bool may_fold = crowd <= kMostCrowded;
		bool folds = false;
		begin(f, regions, may_fold, kPostThreads);
		for (uint32_t at = 0; at < n; at += kPostThreads) {
			const uint64_t b = base, o = offset, v = value;
			if (at + kPostThreads < n) {
				load(at + kPostThreads);
			}
			add_items(f, regions, b, o, v, at + threadIdx.x < n, crowd, folds, rejected);
		}
		if (may_fold) {
			end(f, folds, kPostThreads);
		}
	}
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
	__syncthreads();
	if (threadIdx.x < 64u) {
		ofi_amd::flush_post_lanes(flush_buf, slots, num_rails, threadIdx.x);
	}
}

} // namespace

using namespace ofi_amd;

static int pack_regions(const ofi_amd_gin_signal_region_t *regions, uint32_t n_regions, regions_t *r)
{
	if (!regions || n_regions == 0 || n_regions > kMaxRegions) {
		return -EINVAL;
	}
	r->n = n_regions;
	for (uint32_t i = 0; i < kMaxRegions; i++) {
		const bool live = i < n_regions;
		if (live && (!regions[i].d_counters || (reinterpret_cast<uintptr_t>(regions[i].d_counters) & 7u))) {
			return -EINVAL;
		}
		r->base[i] = live ? regions[i].base : 0;
		r->size[i] = live ? regions[i].size : 0;
		r->counters[i] = live ? static_cast<uint64_t *>(regions[i].d_counters) : nullptr;
	}
	return 0;
}

extern "C" int ofi_amd_gin_signal_apply(const ofi_amd_gin_signal_work_t *d_work, uint32_t n,
					const ofi_amd_gin_signal_region_t *regions, uint32_t n_regions,
					uint32_t *d_rejected, void *stream)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (n == 0) {
		return 0;
	}
	regions_t r;
	if (!d_work || pack_regions(regions, n_regions, &r) != 0) {
		return -EINVAL;
	}
	/* Items per workgroup.  More items fold further, fewer spread the lookups over more CUs; times
	 * in us with a launch per item before the fold / with 256, 512, 1024 x 2, 1024 x 4 items.
	 *   1000 items in host memory, 1 counter           15.3 / 4.0  4.4  5.0  6.0
	 *   1000 items in host memory, 8192 counters        5.6 / 4.5  4.9  5.9  6.8
	 *   16384 items in host memory, 64 counters        24.8 / 16.8 14.3 13.1 13.4
	 *   16384 items in host memory, 8192 counters      15.3 / 13.9 13.8 16.3 20.2
	 *   262144 items in HBM, 64 counters                311 / 166  90   25.9 16.5
	 *   262144 items in HBM, 8192 counters             16.8 / 16.0 15.8 16.5 18.0
	 *   262144 items in HBM, 262144 counters           14.3 / 14.6 14.6 16.5 18.0
	 * so 256 up to 4096 items, then 512, and 2048 or 4096 for long batches on few counters (one to 64 items or more).
	 * Batches up to 32768 items are not told apart by their counters, which costs the fourth line's 1.2 us.
	 * Long batches in host memory take the large workgroups too: the link is read faster from 64 CUs than
	 * from all of them (262144 items over 8192 counters 187 / 188 187 179 160).  The times are of workgroups
	 * that all fold; since only crowded ones do (crowd_of), 1000 items in host memory on 8192 counters take
	 * 3.8 instead of 4.6, 16384 in HBM 3.4 instead of 3.9, 1000 in HBM on one counter 3.1 instead of 2.9. */
	uint64_t counters = 0;
	for (uint32_t i = 0; i < n_regions; i++) {
		counters += r.size[i] / 8;
	}
	const bool large = n > 32768u && (counters <= n / 64u || in_host_memory(d_work));
	auto launch = [&](auto kernel, uint32_t threads, uint32_t items) {
		ofi_amd::launch_kernel(kernel, dim3((n - 1u) / (threads * items) + 1u), dim3(threads), 0, as_stream(stream),
				       d_work, n, r, large ? 0u : crowd_of(n), d_rejected);
	};
	if (n <= 4096u) {
		launch(gin_signal_apply_kernel<256, 1, 512>, 256, 1);
	} else if (!large) {
		launch(gin_signal_apply_kernel<512, 1, 1024>, 512, 1);
	} else if (n <= 131072u) {
		launch(gin_signal_apply_kernel<1024, 2, 4096>, 1024, 2);
	} else {
		launch(gin_signal_apply_kernel<1024, 4, 4096>, 1024, 4);
	}
	OFI_AMD_HIP_TRY(hipGetLastError());
	return 0;
}

extern "C" int ofi_amd_gin_signal_apply_post(const ofi_amd_gin_signal_work_t *d_work, uint32_t n,
					     const ofi_amd_gin_signal_region_t *regions, uint32_t n_regions,
					     uint32_t *d_rejected, const void *d_flush_buf, void *slots_dev,
					     uint32_t num_rails, void *stream)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (!d_flush_buf || !slots_dev || num_rails < 1 || num_rails > OFI_AMD_MAX_NUM_RAILS ||
	    (reinterpret_cast<uintptr_t>(d_flush_buf) & 7u) || (reinterpret_cast<uintptr_t>(slots_dev) & 7u)) {
		return -EINVAL;
	}
	if (n > kMaxApplyPost) {
		return -E2BIG;
	}
	regions_t r = {};
	if (n != 0 && (!d_work || pack_regions(regions, n_regions, &r) != 0)) {
		return -EINVAL;
	}
	ofi_amd::launch_kernel(gin_signal_apply_post_kernel, dim3(1), dim3(kPostThreads), 0, as_stream(stream), d_work, n, r,
			       n != 0 ? crowd_of(n) : 0u, d_rejected, static_cast<const uint64_t *>(d_flush_buf), static_cast<uint64_t *>(slots_dev),
			       num_rails);
	OFI_AMD_HIP_TRY(hipGetLastError());
	return 0;
}
