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
							 const uint64_t *__restrict__ queries,
							 ofi_amd_tuner_answer_t *__restrict__ answers)
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
	ofi_amd_tuner_answer_t a;
	a.algo = (int8_t)algo;
	a.proto = (int8_t)proto;
	a.nchannels = (int16_t)nch;
	a.pad = 0;
	a.chunk_size = chunk;
	if (lane == 0) {
		answers[i] = a;
	}
}

/* Pinned staging for questions and answers plus a private stream, grown on demand. */
struct staging_t {
	std::mutex lock;
	dev_query_t *q = nullptr;           /* pinned host, device-visible */
	ofi_amd_tuner_answer_t *a = nullptr; /* pinned host, device-visible */
	uint32_t cap = 0;
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
		if (hipHostMalloc(&a, sizeof(ofi_amd_tuner_answer_t) * want, hipHostMallocMapped) != hipSuccess) {
			(void)hipGetLastError();
			(void)hipHostFree(q);
			return -ENOMEM;
		}
		if (g_stage.q) (void)hipHostFree(g_stage.q);
		if (g_stage.a) (void)hipHostFree(g_stage.a);
		g_stage.q = static_cast<dev_query_t *>(q);
		g_stage.a = static_cast<ofi_amd_tuner_answer_t *>(a);
		g_stage.cap = want;
	}
	return 0;
}

using namespace ofi_amd;

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
	for (uint32_t i = 0; i < n; i++) {
		dev_query_t &d = g_stage.q[i];
		d.q = queries[i];
		d.set = region_set(tables, d.q.platform, d.q.coll, d.q.num_ranks, d.q.num_nodes);
		d.log2_bytes = log2_coord((double)queries[i].nbytes);
		d.log2_ranks = log2_coord((double)queries[i].num_ranks);
		d.log2_nodes = std::log2((double)queries[i].num_nodes);
	}
	void *dq = nullptr, *da = nullptr;
	OFI_AMD_HIP_TRY(hipHostGetDevicePointer(&dq, g_stage.q, 0));
	OFI_AMD_HIP_TRY(hipHostGetDevicePointer(&da, g_stage.a, 0));
	for (uint32_t at = 0; at < n; at += kMostPerLaunch) {
		hipLaunchKernelGGL(tuner_query_kernel, dim3(n - at < kMostPerLaunch ? n - at : kMostPerLaunch), dim3(64), 0,
				   g_stage.stream, reinterpret_cast<const int4 *>(tables.poly),
				   reinterpret_cast<const double4_t *>(tables.bbox), tables.edges, tables.far_point,
				   static_cast<const uint64_t *>(dq) + (uint64_t)at * kQueryWords,
				   static_cast<ofi_amd_tuner_answer_t *>(da) + at);
	}
	OFI_AMD_HIP_TRY(hipGetLastError());
	OFI_AMD_HIP_TRY(hipStreamSynchronize(g_stage.stream));
	std::memcpy(answers, g_stage.a, sizeof(ofi_amd_tuner_answer_t) * n);
	return 0;
}
