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

/* Device form of one question, a cache line: what its kind looks at, with the polygon set that answers for its shape
 * and the log2 coordinates from host libm */
struct dev_query_t {
	uint8_t kind, platform, algo, proto;
	uint32_t allowed_mask;
	int32_t coll;
	int32_t net_comp_overhead;
	uint64_t nbytes, num_ranks, num_nodes;
	union {
		region_set_t set;                   /* region decisions */
		struct {
			int32_t pipe_ops, num_channels; /* model decisions */
		} model;
	};
	union {
		double log2_bytes; /* region decisions */
		double log2_nodes; /* model decisions */
	};
	double log2_ranks;
};
constexpr uint32_t kMostPerLaunch = 1u << 24; /* wavefronts; a launch holds below 2^32 threads */
constexpr uint32_t kQueryWords = sizeof(dev_query_t) / 8;
static_assert(sizeof(dev_query_t) == 64, "the kernel picks the fields out of the eight 8-byte words of a line");
constexpr uint32_t kQueryWaves = 8; /* questions of a workgroup: their answers are a cache line */

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
	if (d.set.polys == 0 || d.num_nodes <= 2) {
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
		if (!allowed(d.allowed_mask, a, pr)) {
			continue;
		}
		const uint64_t of_poly = edge_lanes(__builtin_amdgcn_readlane(pw.z, i) - (int)d.set.first_edge,
						    __builtin_amdgcn_readlane(pw.w, i));
		const double bounds[4] = { query_double(box.x, i), query_double(box.y, i), query_double(box.z, i),
					   query_double(box.w, i) };
		if ((touch_lanes & of_poly) != 0 || ((__popcll(cross_lanes & of_poly) & 1) && in_bounds(p, bounds, 0.0))) {
			algorithm = a;
			protocol = pr;
			nchannels = region_channels(d.platform, d.nbytes, d.num_ranks, d.num_nodes, a, pr);
			return;
		}
	}
}

/*
 * One wavefront per question.  The launch is latency, so what counts is the
 * number of dependent trips to memory: the question comes over the host link as one load
 * instruction (a word per lane, one line), a region set's edges lie in the lanes and every polygon's verdict
 * comes out of the same pass over them, the cells of the model are evaluated side by side, one per
 * lane.  With a thread per question each lane walked the polygons by itself through global memory,
 * a trip for the polygon, its bounds and every four edges: the kernel took 30.6 us for 259 questions,
 * and takes 5.7.  From some hundred questions on it is the answers that bound it: the link takes a write of 8 bytes as
 * slowly as one of 64, so the eight answers of a workgroup, 8 bytes each, meet in LDS and leave as a line
 * (the call for 1200 questions, with two writes of 8 bytes each and questions of a line and a half 37.6 us, now 18.6;
 * for 259 questions 15.7 and 13.0; in workgroups of one question 23.1 and 13.0).
 * The structure comes first, so that no argument is preloaded: here that is no gain (259 questions 13.1 us, preloaded 13.3; 16
 * 10.65 and 10.8).
 */
__global__ __launch_bounds__(64 * kQueryWaves) void tuner_query_kernel(pt_t far_point, const int4 *__restrict__ polys,
								       const double4_t *__restrict__ boxes,
								       const edge_t *__restrict__ edges,
								       const uint64_t *__restrict__ queries, uint32_t n,
								       uint32_t call, uint64_t *__restrict__ answers)
{
	__shared__ uint32_t found[kQueryWaves];
	const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const uint32_t first = blockIdx.x * kQueryWaves, i = first + wave;
	if (i < n) {
		const uint64_t words = queries[(uint64_t)i * kQueryWords + (lane & (kQueryWords - 1u))];
		dev_query_t q;
		uint64_t w[kQueryWords];
#pragma unroll
		for (uint32_t k = 0; k < kQueryWords; k++) {
			w[k] = query_word(words, (int)k);
		}
		__builtin_memcpy(&q, w, sizeof(q));
		int algo = -1, proto = -1, nch = -1;
		uint32_t chunk = 0;
		switch (q.kind) { /* wave-uniform */
		case 0:
			region_choose_wave(polys, boxes, edges, far_point, q, lane, algo, proto, nch);
			break;
		case 1: {
			/* lane algo * 3 + proto holds that cell's cost; the decision reads the cells it looks at */
			const int cell = (int)min(lane, (uint32_t)(NUM_ALGOS * NUM_PROTOS - 1));
			const float cost = model_cost(q.platform, q.coll, cell / NUM_PROTOS, cell % NUM_PROTOS, q.model.pipe_ops,
						      q.nbytes, q.num_ranks, q.num_nodes, q.log2_nodes, q.model.num_channels,
						      q.net_comp_overhead);
			model_choose_with(
				q.platform, q.coll, q.nbytes, q.num_ranks, q.num_nodes, q.allowed_mask,
				[&](int a, int pr) -> float {
					return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cost), a * NUM_PROTOS + pr));
				},
				algo, proto);
			break;
		}
		default:
			chunk = (uint32_t)region_chunk_size(q.platform, q.coll, q.nbytes, q.algo, q.proto, q.num_ranks,
							    q.num_nodes); /* 1 MiB at most */
			break;
		}
		if (lane == 0) {
			found[wave] = q.kind == 2 ? chunk
						  : (uint32_t)(uint8_t)(int8_t)algo | ((uint32_t)(uint8_t)(int8_t)proto << 8) |
							    ((uint32_t)(uint16_t)(int16_t)nch << 16);
		}
	}
	__syncthreads();
	if (threadIdx.x < kQueryWaves && first + threadIdx.x < n) {
		/* with the call's number in its upper half the host sees by each word on its own that it is this call's */
		__hip_atomic_store(&answers[first + threadIdx.x], (uint64_t)call << 32 | found[threadIdx.x], __ATOMIC_RELAXED,
				   __HIP_MEMORY_SCOPE_SYSTEM);
	}
}

/* Pinned staging for questions and answers plus a private stream, grown on demand. */
struct staging_t {
	std::mutex lock;
	dev_query_t *q = nullptr; /* pinned host, device-visible */
	uint64_t *a = nullptr;    /* pinned host, device-visible: a word an answer */
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
		hipError_t e = hipHostMalloc(&a, sizeof(uint64_t) * want, hipHostMallocMapped);
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
		std::memset(a, 0, sizeof(uint64_t) * want);
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
 * 5 us later (16 questions: 11.4 us for the call instead of 16.7).  A launch that has retired without
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
		uint64_t word;
		for (uint32_t polls = 0;; polls++) {
			word = __atomic_load_n(&stage.a[i], __ATOMIC_ACQUIRE);
			if ((uint32_t)(word >> 32) == call) {
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
		const bool chunk = stage.q[i].kind == 2; /* the caller's questions may lie where the answers go */
		const uint32_t low = (uint32_t)word, decision = chunk ? ~0u : low;
		ofi_amd_tuner_answer_t &a = answers[i];
		a.algo = (int8_t)decision;
		a.proto = (int8_t)(decision >> 8);
		a.nchannels = (int16_t)(decision >> 16);
		a.pad = 0;
		a.chunk_size = chunk ? low : 0;
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
		std::memset(g_stage.a, 0, sizeof(uint64_t) * g_stage.cap);
		g_stage.call = 1;
	}
	const uint32_t call = g_stage.call;
	for (uint32_t i = 0; i < n; i++) {
		const ofi_amd_tuner_query_t &q = queries[i];
		dev_query_t &d = g_stage.q[i];
		d.kind = (uint8_t)q.kind;
		d.platform = (uint8_t)q.platform;
		d.algo = (uint8_t)q.algo;
		d.proto = (uint8_t)q.proto;
		d.allowed_mask = q.allowed_mask;
		d.coll = q.coll;
		d.net_comp_overhead = q.net_comp_overhead;
		d.nbytes = q.nbytes;
		d.num_ranks = q.num_ranks;
		d.num_nodes = q.num_nodes;
		if (q.kind == 0) {
			d.set = region_set(tables, q.platform, q.coll, q.num_ranks, q.num_nodes);
			d.log2_bytes = log2_coord((double)q.nbytes);
			d.log2_ranks = log2_count(q.num_ranks);
		} else {
			d.model.pipe_ops = q.pipe_ops;
			d.model.num_channels = q.num_channels;
			d.log2_nodes = q.kind == 1 ? log2_count(q.num_nodes) : 0;
			d.log2_ranks = 0;
		}
	}
	for (uint32_t at = 0; at < n; at += kMostPerLaunch) {
		const uint32_t here = n - at < kMostPerLaunch ? n - at : kMostPerLaunch;
		const uint32_t waves = here < kQueryWaves ? here : kQueryWaves;
		ofi_amd::launch_kernel(tuner_query_kernel, dim3((here + kQueryWaves - 1) / kQueryWaves), dim3(64 * waves), 0,
				       g_stage.stream, tables.far_point, reinterpret_cast<const int4 *>(tables.poly),
				       reinterpret_cast<const double4_t *>(tables.bbox), tables.edges,
				       static_cast<const uint64_t *>(g_stage.dq) + (uint64_t)at * kQueryWords, here, call,
				       static_cast<uint64_t *>(g_stage.da) + at);
	}
	OFI_AMD_HIP_TRY(hipGetLastError());
	return collect_answers(g_stage, n, call, answers);
}
