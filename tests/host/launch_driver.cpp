/*
 * The launches of libofi_amd_hotpath.so with a stand-in for the HIP runtime: this program defines the runtime
 * functions the library calls, so the library's host code runs without a GPU and every launch is seen with its
 * grid and its arguments.  argv[1] names the part to run.
 */
#include <cerrno>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include "ofi_amd_hotpath.h"

/* the tests' own way into the library (csrc/common.hpp) */
extern "C" int ofi_amd_sched_batch_looks(ofi_amd_sched_state_t *, const uint64_t *, uint64_t, uint64_t, uint32_t *,
					 ofi_amd_xfer_info_t *, void *, uint32_t looks);

#define CHECK(cond)                                                                  \
	do {                                                                         \
		if (!(cond)) {                                                       \
			std::printf("%s:%d: %s\n", __FILE__, __LINE__, #cond);       \
			std::exit(1);                                                \
		}                                                                    \
	} while (0)

namespace {

struct launch_t {
	std::string kernel; /* demangled, with its template arguments */
	dim3 grid, block;
	size_t shared;
	void **args;
	hipStream_t stream;
	template <typename T> T arg(int i) const { return *static_cast<T *>(args[i]); }
};

std::map<const void *, std::string> &kernels()
{
	static std::map<const void *, std::string> m;
	return m;
}

std::function<void(const launch_t &)> on_launch = [](const launch_t &) {};
hipError_t last_error = hipSuccess;
int device = 0;
hipError_t copy_answer = hipSuccess, sync_answer = hipSuccess;
hipError_t capture_answer = hipSuccess;
hipStreamCaptureStatus capture_status = hipStreamCaptureStatusNone;
struct config_t {
	dim3 grid, block;
	size_t shared;
	hipStream_t stream;
} pushed;

} // namespace

extern "C" {

/* nothing but malloc behind them */
hipError_t hipMalloc(void **p, size_t n) { return (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t)
{
	return copy_answer == hipSuccess ? hipMemcpy(d, s, n, k) : copy_answer;
}
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = device; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDriverGetVersion(int *v) { *v = 1; return hipSuccess; }
hipError_t hipRuntimeGetVersion(int *v) { *v = 1; return hipSuccess; }
hipError_t hipGetLastError()
{
	const hipError_t e = last_error;
	last_error = hipSuccess;
	return e;
}
hipError_t hipStreamSynchronize(hipStream_t) { return sync_answer; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = reinterpret_cast<hipStream_t>(0x70); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *)
{
	static uint32_t array[1u << 18];
	*p = array;
	return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *status)
{
	*status = capture_status;
	return capture_answer;
}

void **__hipRegisterFatBinary(const void *) { static void *module; return &module; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
	int status = 0;
	char *plain = abi::__cxa_demangle(name, nullptr, nullptr, &status);
	kernels()[host] = plain ? plain : name;
	std::free(plain);
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream)
{
	pushed = { grid, block, shared, stream };
	return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream)
{
	*grid = pushed.grid, *block = pushed.block, *shared = pushed.shared, *stream = pushed.stream;
	return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t shared, hipStream_t stream)
{
	/* what HIP supports: fewer than 2^32 work-items along each dimension */
	if ((uint64_t)grid.x * block.x >> 32 || (uint64_t)grid.y * block.y >> 32 || (uint64_t)grid.z * block.z >> 32) {
		return last_error = hipErrorInvalidConfiguration;
	}
	on_launch({ kernels()[f], grid, block, shared, args, stream });
	return hipSuccess;
}

} /* extern "C" */

namespace {

/*
 * The arrival words of small striping batches.  The stand-in counts as the kernel does: every tile adds one to
 * the batch's word, whoever makes it the number of tiles sets it to zero and moves the counters on, and
 * the word named beside it is cleared.  A batch that finds a count in its word moves the
 * counters on too early, or not at all.
 */
struct arrivals_t {
	std::vector<uint32_t *> words; /* of the batches so far */
	int spoiled = 0, two_launch = 0;
	void operator()(const launch_t &l)
	{
		two_launch += l.kernel.find("stripe_count_kernel") != std::string::npos;
		if (l.kernel.find("stripe_emit_kernel<((anonymous namespace)::stripe_form)0") == std::string::npos) {
			if (l.kernel.find("stripe_scratch_kernel") != std::string::npos) {
				std::memset(l.arg<uint32_t *>(0), 0, 4ull * l.grid.x * l.block.x);
			}
			return;
		}
		uint32_t *word = l.arg<uint32_t *>(6), *ahead = l.arg<uint32_t *>(7);
		const uint32_t tiles = l.grid.x;
		if (tiles == 1) {
			return;
		}
		spoiled += *word != 0;
		*ahead = 0;
		for (uint32_t t = 0; t < tiles; t++) {
			*word = *word + 1 == tiles ? 0 : *word + 1;
		}
		words.push_back(word);
	}
};

int striping()
{
	using batch_t = int (*)(ofi_amd_sched_state_t *, const uint64_t *, uint64_t, uint64_t, uint32_t *, ofi_amd_xfer_info_t *,
				void *);
	ofi_amd_sched_state_t state = {};
	uint64_t sizes[1] = {};
	uint32_t num[1];
	ofi_amd_xfer_info_t xfers[4];
	void *stream = reinterpret_cast<void *>(0x40);
	for (const batch_t batch : { &ofi_amd_sched_batch, &ofi_amd_sched_batch_noalloc }) {
		arrivals_t seen;
		on_launch = std::ref(seen);
		auto small = [&](uint64_t n) { CHECK(batch(&state, sizes, n, 128, num, xfers, stream) == 0); };
		/* no two of 512 batches in a row count in one word, and each finds its own at zero */
		for (int i = 0; i < 5000; i++) {
			small(257 + (i * 97) % 9728); /* up to 9984, the most in one launch */
		}
		CHECK(seen.words.size() == 5000 && seen.spoiled == 0 && seen.two_launch == 0);
		for (size_t i = 0; i + 512 <= seen.words.size(); i++) {
			CHECK(std::set<uint32_t *>(&seen.words[i], &seen.words[i] + 512).size() == 512);
		}
		/* a count left in every word, by whatever went wrong: the batches after it soon find zero again */
		for (uint32_t *w : std::set<uint32_t *>(seen.words.begin(), seen.words.end())) {
			*w = 4;
		}
		for (int i = 0; i < 512; i++) {
			small(1000);
		}
		seen.spoiled = 0;
		for (int i = 0; i < 5000; i++) {
			small(1000);
		}
		CHECK(seen.spoiled == 0);
		/* one message more has totals to publish, in one launch too */
		int once = 0;
		on_launch = [&](const launch_t &l) { once += l.kernel.find("stripe_once_kernel") != std::string::npos ? 1 : 100; };
		small(9985);
		CHECK(once == 1);
		on_launch = std::ref(seen);
		/* a captured batch comes back to the scratch it was captured with: it counts in no word */
		const size_t before = seen.words.size();
		capture_status = hipStreamCaptureStatusActive;
		small(257);
		small(6144);
		small(9984);
		capture_status = hipStreamCaptureStatusNone;
		capture_answer = hipErrorStreamCaptureImplicit;
		small(1000);
		capture_answer = hipSuccess;
		CHECK(seen.words.size() == before && seen.two_launch == 4);
		/* nor does it take a number from the batches that publish totals */
		std::vector<uint64_t> numbers;
		on_launch = [&](const launch_t &l) {
			if (l.kernel.find("stripe_once_kernel") != std::string::npos) {
				numbers.push_back(l.arg<uint64_t>(6));
			}
		};
		small(30001);
		capture_status = hipStreamCaptureStatusActive;
		small(30001);
		capture_status = hipStreamCaptureStatusNone;
		small(262144);
		CHECK(numbers.size() == 2 && numbers[1] == numbers[0] + 1);
		on_launch = std::ref(seen);
		small(256); /* one tile */
		CHECK(seen.words.size() == before && seen.two_launch == 4);
	}
	/* no tile looks for longer than those of an ordinary batch, however it is called */
	std::vector<uint32_t> looks;
	on_launch = [&](const launch_t &l) {
		if (l.kernel.find("stripe_once_kernel") != std::string::npos) {
			looks.push_back(l.arg<uint32_t>(7));
		}
	};
	CHECK(ofi_amd_sched_batch(&state, sizes, 30001, 128, num, xfers, stream) == 0);
	for (const uint32_t asked : { 0u, 1u, ~0u }) {
		CHECK(ofi_amd_sched_batch_looks(&state, sizes, 30001, 128, num, xfers, stream, asked) == 0);
	}
	CHECK(looks.size() == 4 && looks[0] <= 2048 && looks[1] == 0 && looks[2] == 1 && looks[3] == looks[0]);
	CHECK(ofi_amd_sched_stream_release(stream) == 0);
	return 0;
}

/*
 * The scratch of a batch belongs to one stream: hipStreamPerThread is another stream in each thread, the null stream on
 * each GPU, whatever their handles say; other handles are one stream whichever thread calls.
 */
int streams()
{
	ofi_amd_sched_state_t state = {};
	uint64_t sizes[1] = {};
	uint32_t num[1];
	ofi_amd_xfer_info_t xfers[4];
	/* the tile totals of a batch in the two-launch form */
	auto scratch_on = [&](void *stream) {
		uint32_t *totals = nullptr;
		on_launch = [&](const launch_t &l) {
			if (l.kernel.find("stripe_count_kernel") != std::string::npos) {
				totals = l.arg<uint32_t *>(4);
			}
		};
		CHECK(ofi_amd_sched_batch(&state, sizes, 300000, 128, num, xfers, stream) == 0 && totals);
		return totals;
	};
	auto in_another_thread = [&](void *stream) {
		uint32_t *totals = nullptr;
		std::thread([&] { totals = scratch_on(stream); }).join();
		return totals;
	};
	void *const made = reinterpret_cast<void *>(0x40), *const per_thread = hipStreamPerThread;
	CHECK(scratch_on(made) == in_another_thread(made));
	CHECK(scratch_on(nullptr) == in_another_thread(nullptr));
	uint32_t *const mine = scratch_on(per_thread), *const null0 = scratch_on(nullptr);
	CHECK(mine == scratch_on(per_thread) && mine != scratch_on(made) && mine != null0);
	uint32_t *const other = in_another_thread(per_thread), *const third = in_another_thread(per_thread);
	CHECK(other != mine && third != mine && third != other);
	device = 1;
	CHECK(scratch_on(nullptr) != null0 && scratch_on(per_thread) != mine);
	device = 0;
	CHECK(scratch_on(nullptr) == null0 && scratch_on(per_thread) == mine);
	/* a thread hands its own back */
	std::thread([&] {
		scratch_on(per_thread);
		CHECK(ofi_amd_sched_stream_release(per_thread) == 0);
	}).join();
	CHECK(scratch_on(per_thread) == mine && ofi_amd_sched_stream_release(per_thread) == 0);
	/* New scratch is cleared as far as a batch reads what it has not written: 1024 words that batches count in, eight copies
	 * of 512 published words of 64 bits and the one behind them, whichever batch and stream state come first */
	for (const hipStreamCaptureStatus status : { hipStreamCaptureStatusNone, hipStreamCaptureStatusActive }) {
		uint64_t cleared = 0, launches = 0;
		on_launch = [&](const launch_t &l) {
			if (l.kernel.find("stripe_scratch_kernel") != std::string::npos) {
				CHECK(launches == 0);
				cleared += (uint64_t)l.grid.x * l.block.x;
			}
			launches++;
		};
		capture_status = status;
		CHECK(ofi_amd_sched_batch(&state, sizes, 30001, 128, num, xfers, reinterpret_cast<void *>(0x48)) == 0);
		capture_status = hipStreamCaptureStatusNone;
		CHECK(cleared >= 1024 + 2 * (8 * 512 + 1) && ofi_amd_sched_stream_release(reinterpret_cast<void *>(0x48)) == 0);
	}
	return 0;
}

/*
 * Copy tables by pieces of 8 KiB: every table up to 2^31 - 1 pieces is launched, within the limits of a launch,
 * every entry in one launch and with a wavefront for each of its pieces; larger ones are refused with nothing launched.
 */
int pieces()
{
	struct map_t {
		uint32_t per, run_blocks, wave_stride, block_stride;
	};
	uint64_t *const src = reinterpret_cast<uint64_t *>(0x1000000), *const dst = reinterpret_cast<uint64_t *>(0x80000000000);
	uint32_t *const len = reinterpret_cast<uint32_t *>(0x70000000000);
	const uint32_t mib = 1u << 20;
	struct table_t {
		uint32_t n, max_len;
		int rc;
	};
	const table_t tables[] = {
		{ 1, 0, 0 }, { 1, 8192, 0 }, { 1, ~0u, 0 }, { 127, ~0u, 0 }, { 128, ~0u, 0 }, { 4095, ~0u, 0 },
		/* a launch group with one write of 128 MiB: 2^26 pieces */
		{ 4096, 128 * mib, 0 }, { 4095, 128 * mib, 0 }, { 4096, 64 * mib, 0 }, { 8192, 64 * mib - 8192, 0 },
		{ (1u << 24) - 1, 8192, 0 }, { 1u << 24, 8192, 0 }, { (1u << 26) - 1024, 8192, 0 }, { (1u << 26) - 1023, 8192, 0 },
		{ 1u << 26, 8192, 0 }, { 1u << 30, 8192, 0 }, { 1u << 20, 129 * 8192, 0 }, { 1u << 17, 129 * 8192, 0 },
		{ 1u << 21, 8 * 8192, 0 }, { 130055, 129 * 8192, 0 }, { 4096, ~0u, -E2BIG }, { 1u << 20, ~0u, -E2BIG },
	};
	for (const table_t &t : tables) {
		uint64_t covered = 0, launches = 0;
		on_launch = [&](const launch_t &l) {
			const uint32_t n = l.arg<uint32_t>(3);
			const map_t map = l.arg<map_t>(4);
			CHECK(l.arg<uint64_t *>(0) == src + covered && l.arg<uint64_t *>(1) == dst + covered &&
			      l.arg<uint32_t *>(2) == len + covered && l.arg<uint32_t>(5) == t.max_len);
			CHECK((uint64_t)map.per * 8192 >= t.max_len && l.block.x == 256 && l.grid.y * l.grid.z == 1);
			/* whole runs for each of the 8 XCDs, their pieces numbered without a gap, enough of them */
			CHECK(l.grid.x % (8 * map.run_blocks) == 0 && (uint64_t)l.grid.x * 4 >= (uint64_t)n * map.per);
			CHECK((map.wave_stride == 1 && map.block_stride == 4) ||
			      (map.wave_stride == map.run_blocks && map.block_stride == 1));
			covered += n;
			launches++;
		};
		const int rc = ofi_amd_copy_table_pieces(src, dst, len, t.n, t.max_len, nullptr);
		if (rc != t.rc || covered != (rc == 0 ? t.n : 0)) {
			std::printf("n %u max_len %u: %d, %llu of the entries in %llu launches\n", t.n, t.max_len, rc,
				    (unsigned long long)covered, (unsigned long long)launches);
			return 1;
		}
	}
	return 0;
}

/*
 * The bytes of a bounce batch's source are the range its offsets lie in, a pool as a rule, and say nothing about how long
 * the buffers are: beyond what the L2s hold the launch is the same whatever they are.  A batch without flush words has a
 * kernel of its own, which does none of their work.
 */
int bounce()
{
	uint8_t *const src = reinterpret_cast<uint8_t *>(0x1000000), *const arena = reinterpret_cast<uint8_t *>(0x80000000000);
	uint64_t *const off = reinterpret_cast<uint64_t *>(0x70000000000);
	uint32_t *const len = reinterpret_cast<uint32_t *>(0x71000000000), *const words = reinterpret_cast<uint32_t *>(0x72000000000);
	std::set<std::string> with[2];
	for (uint32_t *flush : { words, static_cast<uint32_t *>(nullptr) }) {
		for (uint32_t n : { 8001u, 20000u, 65536u, 200000u }) {
			std::string kernel;
			dim3 block;
			size_t shared = 0;
			for (uint64_t mib : { 33ull, 64ull, 101ull, 130ull, 256ull, 512ull, 1024ull, 1ull << 16 }) {
				int launches = 0;
				on_launch = [&](const launch_t &l) {
					if (kernel.empty()) {
						kernel = l.kernel, block = l.block, shared = l.shared;
					}
					CHECK(l.kernel == kernel && l.block.x == block.x && l.shared == shared);
					CHECK((uint64_t)l.grid.x * l.block.x >= 64ull * n && l.arg<uint64_t>(1) == mib << 20);
					with[flush != nullptr].insert(l.kernel);
					launches++;
				};
				CHECK(ofi_amd_bounce_scatter(src, mib << 20, arena, 1ull << 40, off, off, len, n, flush, nullptr) == 0);
				CHECK(launches == 1);
			}
		}
	}
	for (const std::string &kernel : with[0]) {
		CHECK(with[1].count(kernel) == 0);
	}
	/* however short the buffers of a small source are, the lines of so many do not stay in the L2s */
	auto kernel_of = [&](uint32_t n, uint64_t mib) {
		std::string kernel;
		on_launch = [&](const launch_t &l) { kernel = l.kernel; };
		CHECK(ofi_amd_bounce_scatter(src, mib << 20, arena, 1ull << 40, off, off, len, n, words, nullptr) == 0);
		return kernel;
	};
	CHECK(kernel_of(100000, 16) != kernel_of(100000, 33) && kernel_of(1000000, 16) == kernel_of(1000000, 33));
	return 0;
}

/* The tiles of a region grid follow its axes: on short ones too, most lanes have a point. */
int tiles()
{
	const int32_t colls[] = { 4, 2 }, algos[] = { 1 };
	const uint32_t ppn[] = { 8, 2, 1 };
	const int32_t platforms[] = { 0, 1, 2, 3 };
	const uint32_t shapes[][2] = { { 1, 20000 }, { 2, 20000 }, { 3, 20000 }, { 5, 20000 }, { 20000, 1 }, { 20000, 2 }, { 20000, 3 },
				       { 20000, 5 }, { 1, 90000 }, { 90000, 1 }, { 560, 38 }, { 2000, 17 }, { 17, 2000 } };
	for (const auto &shape : shapes) {
		std::vector<uint64_t> sizes(shape[0]), nodes(shape[1]);
		for (size_t i = 0; i < sizes.size(); i++) {
			sizes[i] = 1000 * i;
		}
		for (size_t i = 0; i < nodes.size(); i++) {
			nodes[i] = i + 1;
		}
		ofi_amd_tuner_plan_t *plan = nullptr;
		CHECK(ofi_amd_tuner_plan_create(colls, 2, sizes.data(), shape[0], nodes.data(), shape[1], ppn, 3, algos, 1, &plan) == 0);
		uint64_t lanes = 0;
		on_launch = [&](const launch_t &l) { lanes += (uint64_t)l.grid.x * l.grid.y * l.block.x; };
		alignas(4) int8_t choice[4];
		CHECK(ofi_amd_tuner_region_grid(plan, platforms, 4, choice, nullptr) == 0);
		const uint64_t points = 4 * ofi_amd_tuner_plan_points(plan);
		CHECK(lanes >= points);
		if (lanes > points * 2) {
			std::printf("%u sizes x %u node counts: %llu lanes for %llu points\n", shape[0], shape[1],
				    (unsigned long long)lanes, (unsigned long long)points);
			return 1;
		}
		CHECK(ofi_amd_tuner_plan_destroy(plan) == 0);
	}
	return 0;
}

/*
 * Workgroups of 1024 threads are for large cost grids most of whose points are only written: never where more than half of
 * the points are modelled, AllReduce's on a platform with a model.  Where all are, fewer workgroups a CU pay later, too.
 */
int model()
{
	std::vector<uint64_t> sizes(140), nodes(11);
	for (size_t i = 0; i < sizes.size(); i++) {
		sizes[i] = 1000 * i;
	}
	for (size_t i = 0; i < nodes.size(); i++) {
		nodes[i] = 1ull << i;
	}
	const uint32_t ppn[] = { 1, 2, 4, 8 };
	const int32_t algos[] = { 1, 0, 6 };
	struct grid_t {
		std::vector<int32_t> colls;
		int32_t platforms[2];
		bool large;
	};
	const grid_t grids[] = { { { 4 }, { 0, 1 }, false },	 { { 4, 2, 3 }, { 0, 1 }, true }, { { 4, 4, 2 }, { 0, 1 }, false },
				 { { 4, 2 }, { 0, 1 }, true },	 { { 4 }, { 0, 2 }, true },	  { { 4 }, { 2, 3 }, true },
				 { { 4, 4, 2 }, { 0, 2 }, true } };
	for (const grid_t &grid : grids) {
		ofi_amd_tuner_plan_t *plan = nullptr;
		CHECK(ofi_amd_tuner_plan_create(grid.colls.data(), (uint32_t)grid.colls.size(), sizes.data(), 140, nodes.data(), 11,
						ppn, 4, algos, 3, &plan) == 0);
		const uint64_t cells = ofi_amd_tuner_plan_cells(plan);
		for (uint64_t mb : { 1, 40, 60, 120, 180, 500, 2000 }) {
			std::vector<ofi_amd_tuner_variant_t> v((size_t)(mb * 1000000 / (16 * cells)) * 2 + 2);
			for (size_t i = 0; i < v.size(); i++) {
				v[i] = { grid.platforms[i % 2], 1, 8, 3 };
			}
			double cost[1];
			alignas(2) int8_t choice[2];
			int launches = 0;
			on_launch = [&](const launch_t &l) {
				const bool large = grid.large && mb >= 180;
				CHECK(l.block.x == (large ? 1024 : 256) && l.grid.y == v.size());
				CHECK((uint64_t)l.grid.x * l.block.x >= ofi_amd_tuner_plan_points(plan));
				CHECK(l.shared >= 36u * l.block.x && l.shared <= 65536);
				CHECK(large || (l.shared > 9216) == (mb >= (grid.colls.size() == 1 && grid.platforms[1] == 1 ? 120 : 60)));
				launches++;
			};
			CHECK(ofi_amd_tuner_model_grid(plan, v.data(), (uint32_t)v.size(), cost, choice, nullptr) == 0);
			CHECK(ofi_amd_tuner_model_grid(plan, v.data(), (uint32_t)v.size(), cost, nullptr, nullptr) == 0);
			CHECK(launches == 2);
		}
		CHECK(ofi_amd_tuner_plan_destroy(plan) == 0);
	}
	return 0;
}

/* A list of variants or platforms that did not reach the GPU is sent again by the next call with the same list. */
int uploads()
{
	const int32_t colls[] = { 4 }, algos[] = { 1 };
	const uint64_t sizes[] = { 1 << 20 }, nodes[] = { 4 };
	const uint32_t ppn[] = { 8 };
	ofi_amd_tuner_plan_t *plan = nullptr;
	CHECK(ofi_amd_tuner_plan_create(colls, 1, sizes, 1, nodes, 1, ppn, 1, algos, 1, &plan) == 0);
	double cost[3];
	int8_t choice[4];
	ofi_amd_tuner_variant_t v = { 0, 1, 8, 3 };
	int launches = 0;
	on_launch = [&](const launch_t &l) {
		CHECK(std::memcmp(l.arg<void *>(1), &v, sizeof(v)) == 0); /* what the kernel reads */
		launches++;
	};
	auto grid = [&] { return ofi_amd_tuner_model_grid(plan, &v, 1, cost, choice, nullptr); };
	CHECK(grid() == 0 && launches == 1);
	for (hipError_t *answer : { &copy_answer, &sync_answer }) {
		v.pipe_ops++;
		*answer = hipErrorUnknown;
		CHECK(grid() == -EIO && launches == 1);
		*answer = hipSuccess;
		CHECK(grid() == 0);
		launches = 1;
	}
	CHECK(ofi_amd_tuner_plan_destroy(plan) == 0);
	return 0;
}

} // namespace

int main(int argc, char **argv)
{
	const std::map<std::string, int (*)()> parts = { { "striping", striping }, { "streams", streams }, { "pieces", pieces },
							       { "bounce", bounce }, { "model", model }, { "tiles", tiles }, { "uploads", uploads } };
	CHECK(argc == 2 && parts.count(argv[1]) && ofi_amd_gpu_init() == 0);
	const int rc = parts.at(argv[1])();
	std::printf("%s: %s\n", argv[1], rc == 0 ? "ok" : "failed");
	return rc;
}
