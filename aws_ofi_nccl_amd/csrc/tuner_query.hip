/*
 * Point queries of the tuner: a list of independent questions (region decision, model
 * decision, chunk size) answered by one launch, one wavefront per question.  The tuner
 * plugin's per-collective entry points are served from here through a cache
 * (tuner_plugin.cpp); irregular batch callers can use it directly.
 */
#include <cstring>
#include <mutex>

#include "common.hpp"
#include "tuner_device.hpp"

using namespace ofi_amd_tuner;

namespace {

/* device form of one question: the public fields, the polygon set that answers for its shape, and
 * log2 coordinates from host libm */
struct dev_query_t {
	ofi_amd_tuner_query_t q;
	region_set_t set;
	double log2_bytes;
	double log2_ranks;
	double log2_nodes;
};
constexpr uint32_t kMostPerLaunch = 1u << 24; /* wavefronts; a launch holds below 2^32 threads */
constexpr uint32_t kQueryWords = sizeof(dev_query_t) / 8;
static_assert(sizeof(dev_query_t) == 96, "the kernel picks the fields out of twelve 8-byte words");

/* word k of the question, held by lane k, as a value of the whole wavefront */
__device__ __forceinline__ uint64_t query_word(uint64_t words, int k)
{
	const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)words, k);
	const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(words >> 32), k);
	return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ double query_double(double v, int k)
{
	return __longlong_as_double((long long)query_word((uint64_t)__double_as_longlong(v), k));
}

/*
 * region_get_coll_info_internal_v3, :2070-2157, for one question put by a whole wavefront: lane e works
 * on edge e of the polygon set, and the wave's ballots give every polygon's on-edge and crossing bits at
 * once.  The first polygon that holds the point (inside or on an edge) wins; polygons whose (algo,
 * proto) bit is clear in the mask are passed over: for v3 those are the cells NCCL marked -1 or that lie
 * beyond numAlgo / numProto (:2109-2114); for v2 PAT and, without NVLS support, NVLS tree (:2023-2030).
 */
__device__ __forceinline__ void region_choose_wave(const int4 *__restrict__ polys, const double4_t *__restrict__ boxes,
						   const edge_t *__restrict__ edges, pt_t far_point, const dev_query_t &d,
						   uint32_t lane, int &algorithm, int &protocol, int &nchannels)
{
	if (d.set.polys == 0 || d.q.num_nodes <= 2) {
		return;
	}
	const double eps = 1e-10;
	const pt_t p = { d.log2_bytes, d.log2_ranks };
	const uint32_t my_poly = d.set.first_poly + min(lane, (uint32_t)d.set.polys - 1u);
	const int4 pw = polys[my_poly];
	const double4_t box = boxes[my_poly];
	const edge_t e = edges[d.set.first_edge + min(lane, (uint32_t)d.set.edges - 1u)];
	const bool mine = lane < d.set.edges;
	const edge_sides_t s = edge_sides(p, vsub(far_point, p), e.a, e.b);
	const double side_f = vcross(vsub(far_point, e.a), vsub(e.b, e.a));
	bool crosses = mine && crossing(s, side_f), touches = mine && fabs(s.side_p) <= touch_reach(e.a, e.b);
	if (mine && !crossing_certain(s, side_f)) {
		crosses = intersects(p, far_point, e.a, e.b, eps);
	}
	if (touches) {
		touches = touches_edge(p, e.a, e.b, s, eps);
	}
	const uint64_t cross_lanes = __ballot(crosses), touch_lanes = __ballot(touches);
	for (int i = 0; i < (int)d.set.polys; i++) {
		const int a = __builtin_amdgcn_readlane(pw.x, i), pr = __builtin_amdgcn_readlane(pw.y, i);
		if (!allowed(d.q.allowed_mask, a, pr)) {
			continue;
		}
		const uint64_t of_poly = edge_lanes(__builtin_amdgcn_readlane(pw.z, i) - (int)d.set.first_edge,
						    __builtin_amdgcn_readlane(pw.w, i));
		const double bounds[4] = { query_double(box.x, i), query_double(box.y, i), query_double(box.z, i),
					   query_double(box.w, i) };
		if ((touch_lanes & of_poly) != 0 || ((__popcll(cross_lanes & of_poly) & 1) && in_bounds(p, bounds, 0.0))) {
			algorithm = a;
			protocol = pr;
			nchannels = region_channels(d.q.platform, d.q.nbytes, d.q.num_ranks, d.q.num_nodes, a, pr);
			return;
		}
	}
}

/*
 * One wavefront per question.  The launch is latency and nothing else, so what counts is the
 * number of dependent trips to memory: the question comes over the host link as one load
 * instruction (a word per lane), a region set's edges lie in the lanes and every polygon's verdict
 * comes out of the same pass over them, the cells of the model are evaluated side by side, one per
 * lane.  With a thread per question each lane walked the polygons by itself through global memory,
 * a trip for the polygon, its bounds and every four edges: 30.6 us for 259 questions, now
 * 5.6.
 */
__global__ __launch_bounds__(64) void tuner_query_kernel(const int4 *__restrict__ polys,
							 const double4_t *__restrict__ boxes,
							 const edge_t *__restrict__ edges, pt_t far_point,
							 const uint64_t *__restrict__ queries, uint32_t call,
							 uint64_t *__restrict__ answers)
{
	const uint32_t i = blockIdx.x, lane = threadIdx.x;
	const uint64_t words = queries[(uint64_t)i * kQueryWords + min(lane, kQueryWords - 1u)];
	dev_query_t d;
	uint64_t w[kQueryWords];
#pragma unroll
	for (uint32_t k = 0; k < kQueryWords; k++) {
		w[k] = query_word(words, (int)k);
	}
	__builtin_memcpy(&d, w, sizeof(d));
	const ofi_amd_tuner_query_t &q = d.q;
	int algo = -1, proto = -1, nch = -1;
	uint64_t chunk = 0;
	switch (q.kind) { /* wave-uniform */
	case 0:
		region_choose_wave(polys, boxes, edges, far_point, d, lane, algo, proto, nch);
		break;
	case 1: {
		/* lane algo * 3 + proto holds that cell's cost; the decision reads the cells it looks at */
		const int cell = (int)min(lane, (uint32_t)(NUM_ALGOS * NUM_PROTOS - 1));
		const float cost = model_cost(q.platform, q.coll, cell / NUM_PROTOS, cell % NUM_PROTOS, q.pipe_ops, q.nbytes,
					      q.num_ranks, q.num_nodes, d.log2_nodes, q.num_channels, q.net_comp_overhead);
		model_choose_with(
			q.platform, q.coll, q.nbytes, q.num_ranks, q.num_nodes, q.allowed_mask,
			[&](int a, int pr) -> float {
				return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cost), a * NUM_PROTOS + pr));
			},
			algo, proto);
		break;
	}
	case 2:
		chunk = region_chunk_size(q.platform, q.coll, q.nbytes, q.algo, q.proto, q.num_ranks,
					  q.num_nodes);
		break;
	default:
		break;
	}
	if (lane == 0) {
		/* The two words of an ofi_amd_tuner_answer_t, each with the call's number in its upper half -- the
		 * padding, and the half that a chunk size (1 MiB at most) leaves -- so that the host sees by
		 * each word on its own that it is this call's. */
		const uint32_t low = (uint32_t)(uint8_t)(int8_t)algo | ((uint32_t)(uint8_t)(int8_t)proto << 8) |
				     ((uint32_t)(uint16_t)(int16_t)nch << 16);
		__hip_atomic_store(&answers[2 * i], (uint64_t)call << 32 | low, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
		__hip_atomic_store(&answers[2 * i + 1], (uint64_t)call << 32 | (uint32_t)chunk, __ATOMIC_RELAXED,
				   __HIP_MEMORY_SCOPE_SYSTEM);
	}
}

/* Pinned staging for questions and answers plus a private stream, grown on demand. */
struct staging_t {
	std::mutex lock;
	dev_query_t *q = nullptr; /* pinned host, device-visible */
	uint64_t *a = nullptr;    /* pinned host, device-visible: two words an answer */
	void *dq = nullptr, *da = nullptr; /* their device addresses */
	uint32_t cap = 0;
	uint32_t call = 0;        /* number of the last call, never 0: what its answers carry */
	hipStream_t stream = nullptr;
};
/* one per GPU: a stream and pinned staging belong to the device that was current when they
 * were made, and a process may drive several */
constexpr int kMaxDevices = 64;
staging_t g_stages[kMaxDevices];

staging_t *stage_of_current_device()
{
	int dev = -1;
	if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
		(void)hipGetLastError();
		return nullptr;
	}
	return &g_stages[dev];
}

} // namespace

using namespace ofi_amd;

/* stream and staging for `want` questions; the caller holds g_stage.lock */
static int ensure_staging(staging_t &g_stage, uint32_t want)
{
	if (!g_stage.stream) {
		OFI_AMD_HIP_TRY(hipStreamCreateWithFlags(&g_stage.stream, hipStreamNonBlocking));
	}
	if (want > g_stage.cap) {
		want = want < 256 ? 256 : want;
		void *q = nullptr, *a = nullptr;
		OFI_AMD_HIP_TRY(hipHostMalloc(&q, sizeof(dev_query_t) * want, hipHostMallocMapped));
		void *dq = nullptr, *da = nullptr;
		hipError_t e = hipHostMalloc(&a, sizeof(ofi_amd_tuner_answer_t) * want, hipHostMallocMapped);
		if (e == hipSuccess) e = hipHostGetDevicePointer(&dq, q, 0);
		if (e == hipSuccess) e = hipHostGetDevicePointer(&da, a, 0);
		/* the last launch may not have retired, though its answers have been read */
		if (e == hipSuccess) e = hipStreamSynchronize(g_stage.stream);
		if (e != hipSuccess) {
			(void)hipGetLastError();
			(void)hipHostFree(q);
			if (a) (void)hipHostFree(a);
			return errno_of(e);
		}
		std::memset(a, 0, sizeof(ofi_amd_tuner_answer_t) * want);
		if (g_stage.q) (void)hipHostFree(g_stage.q);
		if (g_stage.a) (void)hipHostFree(g_stage.a);
		g_stage.q = static_cast<dev_query_t *>(q);
		g_stage.a = static_cast<uint64_t *>(a);
		g_stage.dq = dq;
		g_stage.da = da;
		g_stage.cap = want;
	}
	return 0;
}

extern "C" int ofi_amd_tuner_query_prepare(uint32_t capacity)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	region_tables_t tables;
	rc = device_region_tables(&tables);
	if (rc != 0) {
		return rc;
	}
	staging_t *stage = stage_of_current_device();
	if (!stage) {
		return -ENODEV;
	}
	std::lock_guard<std::mutex> g(stage->lock);
	return ensure_staging(*stage, capacity);
}

/* log2((double)v) as the host's libm gives it; a power of two's is its exponent */
static double log2_count(uint64_t v)
{
	return (v & (v - 1)) == 0 ? (double)__builtin_ctzll(v) : std::log2((double)v);
}

/*
 * Takes the answers as they arrive instead of waiting for the launch to retire, which the host hears of
 * 5 us later (16 questions: 11.4 us for the call instead of 16.7, 259: 16.5 instead of 21.1; from 600 on,
 * where the host's own work per question is what counts, it is the same).  A launch that has retired without
 * all of its answers has failed: the stream is asked now and then, so the wait ends with the launch in any
 * case.
 */
static int collect_answers(const staging_t &stage, uint32_t n, uint32_t call, ofi_amd_tuner_answer_t *answers)
{
	constexpr uint32_t kAskEvery = 4096; /* polls of one answer, some 50 us */
	bool retired = false;
	/* the last answer first: when it is there most of the others are, and lines still being written are
	 * not fetched over and over */
	for (uint32_t i = n; i-- > 0;) {
		uint64_t word[2];
		for (uint32_t k = 2; k-- > 0;) {
			for (uint32_t polls = 0;; polls++) {
				word[k] = __atomic_load_n(&stage.a[2ull * i + k], __ATOMIC_ACQUIRE);
				if ((uint32_t)(word[k] >> 32) == call) {
					break;
				}
				if (retired) {
					return -EIO;
				}
				if (polls % kAskEvery == kAskEvery - 1) {
					const hipError_t e = hipStreamQuery(stage.stream);
					if (e != hipSuccess && e != hipErrorNotReady) {
						(void)hipGetLastError();
						return errno_of(e);
					}
					retired = e == hipSuccess; /* one more look */
				}
				__builtin_ia32_pause();
			}
		}
		ofi_amd_tuner_answer_t &a = answers[i];
		const uint32_t low = (uint32_t)word[0];
		a.algo = (int8_t)low;
		a.proto = (int8_t)(low >> 8);
		a.nchannels = (int16_t)(low >> 16);
		a.pad = 0;
		a.chunk_size = (uint32_t)word[1];
	}
	return 0;
}

extern "C" int ofi_amd_tuner_query(const ofi_amd_tuner_query_t *queries, uint32_t n,
				   ofi_amd_tuner_answer_t *answers)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (n == 0) {
		return 0;
	}
	if (!queries || !answers) {
		return -EINVAL;
	}
	for (uint32_t i = 0; i < n; i++) {
		const ofi_amd_tuner_query_t &q = queries[i];
		if (q.platform < 0 || q.platform >= kNumPlatforms || q.kind < 0 || q.kind > 2 ||
		    q.num_nodes == 0 || q.num_ranks == 0 || q.coll < 0) {
			return -EINVAL;
		}
		if (q.kind == 2 && (q.algo < 0 || q.algo >= NUM_ALGOS || q.proto < 0 || q.proto >= NUM_PROTOS)) {
			return -EINVAL;
		}
	}
	region_tables_t tables;
	rc = device_region_tables(&tables);
	if (rc != 0) {
		return rc;
	}

	staging_t *stage = stage_of_current_device();
	if (!stage) {
		return -ENODEV;
	}
	staging_t &g_stage = *stage;
	std::lock_guard<std::mutex> g(g_stage.lock);
	rc = ensure_staging(g_stage, n);
	if (rc != 0) {
		return rc;
	}
	if (++g_stage.call == 0) { /* the numbers start over: none of the old ones may be left in an answer */
		std::memset(g_stage.a, 0, sizeof(ofi_amd_tuner_answer_t) * g_stage.cap);
		g_stage.call = 1;
	}
	const uint32_t call = g_stage.call;
	for (uint32_t i = 0; i < n; i++) {
		dev_query_t &d = g_stage.q[i];
		d.q = queries[i];
		d.set = region_set(tables, d.q.platform, d.q.coll, d.q.num_ranks, d.q.num_nodes);
		d.log2_bytes = log2_coord((double)queries[i].nbytes);
		d.log2_ranks = log2_count(queries[i].num_ranks);
		d.log2_nodes = log2_count(queries[i].num_nodes);
	}
	for (uint32_t at = 0; at < n; at += kMostPerLaunch) {
		hipLaunchKernelGGL(tuner_query_kernel, dim3(n - at < kMostPerLaunch ? n - at : kMostPerLaunch), dim3(64), 0,
				   g_stage.stream, reinterpret_cast<const int4 *>(tables.poly),
				   reinterpret_cast<const double4_t *>(tables.bbox), tables.edges, tables.far_point,
				   static_cast<const uint64_t *>(g_stage.dq) + (uint64_t)at * kQueryWords, call,
				   static_cast<uint64_t *>(g_stage.da) + 2ull * at);
	}
	OFI_AMD_HIP_TRY(hipGetLastError());
	return collect_answers(g_stage, n, call, answers);
}
