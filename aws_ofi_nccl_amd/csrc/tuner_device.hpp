/*
 * Device functions of the tuner shared by the grid kernels (tuner_grid.hip) and the
 * point-query kernel (tuner_query.hip).
 *
 * Model: nccl_ofi_tuner_compute_cost and model_get_coll_info_internal_v3 / _v2,
 * src/tuner/nccl_ofi_model.cpp:13-309.  The reference computes in fp32 with two
 * double sub-expressions (log2 of the node count) and never fuses a multiply with
 * an add; every rounding step is kept (explicit round-to-nearest intrinsics, files
 * built with contraction off) and log2(nodes) arrives precomputed by the host's
 * libm, so costs match bit for bit.
 *
 * Regions: region_get_coll_info_internal_v3 / _v2, src/tuner/nccl_ofi_regions.cpp:
 * 1995-2157, with is_inside_region (:159-221) and the channel / chunk heuristics
 * (:1883-1971, :2159-2306).  Polygons and query coordinates arrive log2-transformed
 * from the host.  The reference's `long double` intermediates (:91, :50-56) are
 * 80-bit on x86-64 and plain double here; that can only move a point that lies
 * within ~1e-16 of the 1e-10 on-edge threshold.
 */
#ifndef OFI_AMD_TUNER_DEVICE_HPP_
#define OFI_AMD_TUNER_DEVICE_HPP_

#include <cmath>
#include <cstdint>

#include <hip/hip_runtime.h>

#include "ofi_amd_hotpath.h"

namespace ofi_amd_tuner {

/* nccl/tuner.h:14-41 */
enum { FUNC_ALLGATHER = 2, FUNC_REDUCESCATTER = 3, FUNC_ALLREDUCE = 4, NUM_FUNCS = 5 };
enum { ALGO_TREE = 0, ALGO_RING = 1, ALGO_COLLNET_DIRECT = 2, ALGO_COLLNET_CHAIN = 3,
       ALGO_NVLS = 4, ALGO_NVLS_TREE = 5, ALGO_PAT = 6, NUM_ALGOS = 7 };
enum { PROTO_LL = 0, PROTO_LL128 = 1, PROTO_SIMPLE = 2, NUM_PROTOS = 3 };

constexpr int kNumPlatforms = 4;
constexpr int kNumShapes = 3; /* ranks == 8*nodes, 2*nodes, nodes */
constexpr uint32_t kAllAllowed = (1u << (NUM_ALGOS * NUM_PROTOS)) - 1;

__host__ __device__ inline bool allowed(uint32_t mask, int algo, int proto)
{
	return (mask >> (algo * NUM_PROTOS + proto)) & 1u;
}

struct model_params_t {
	float net_lat;
	float internode_bw;
	float intranode_bw;
	int num_rails;
};

/* src/tuner/nccl_ofi_model.cpp:13-44; the bandwidths are double constant
 * expressions narrowed to float once, as there. */
__device__ __forceinline__ model_params_t model_params(int platform)
{
	if (platform == OFI_AMD_PLATFORM_P5EN) {
		return model_params_t{ 18.0f, (float)(25.0 * 1024 * 1024 * 1024 * 1e-6),
				       (float)(20.0 * 1024 * 1024 * 1024 * 1e-6), 2 };
	}
	return model_params_t{ 20.0f, (float)(12.5 * 1024 * 1024 * 1024 * 1e-6),
			       (float)(20.0 * 1024 * 1024 * 1024 * 1e-6), 4 };
}

/* nccl_nvlink_lat, the same table for both modelled platforms (:19-27, :34-42) */
__device__ __forceinline__ float nvlink_lat(int algo, int proto)
{
	switch (algo * NUM_PROTOS + proto) {
	case ALGO_TREE * 3 + PROTO_LL: return .6f;
	case ALGO_TREE * 3 + PROTO_LL128: return 1.25f;
	case ALGO_TREE * 3 + PROTO_SIMPLE: return 28.f;
	case ALGO_RING * 3 + PROTO_LL: return .6f;
	case ALGO_RING * 3 + PROTO_LL128: return 1.9f;
	case ALGO_RING * 3 + PROTO_SIMPLE: return 3.4f;
	case ALGO_COLLNET_DIRECT * 3 + PROTO_SIMPLE: return 3.7f;
	case ALGO_COLLNET_CHAIN * 3 + PROTO_SIMPLE: return 2.8f;
	case ALGO_NVLS * 3 + PROTO_SIMPLE: return 23.f;
	case ALGO_NVLS_TREE * 3 + PROTO_SIMPLE: return 23.f;
	default: return 0.f;
	}
}

__host__ __device__ inline bool platform_has_model(int platform)
{
	return platform == OFI_AMD_PLATFORM_P5_P5E || platform == OFI_AMD_PLATFORM_P5EN;
}

/* nccl_ofi_tuner_compute_cost, src/tuner/nccl_ofi_model.cpp:46-122 */
__device__ inline float model_cost(int platform, int coll, int algo, int proto, int pipe_ops,
				   uint64_t size, uint64_t num_ranks, uint64_t num_nodes,
				   double log2_nodes, int num_channels, int net_comp_overhead)
{
	if (coll != FUNC_ALLREDUCE) {
		return -1.0f;
	}
	const model_params_t params = model_params(platform);
	const float net_lat = (proto == PROTO_SIMPLE)
				      ? __fadd_rn(params.net_lat, (float)net_comp_overhead)
				      : params.net_lat;
	const float p2p_lat = nvlink_lat(algo, proto);
	float latency, bw;

	switch (algo) {
	case ALGO_RING: {
		int num_steps = (int)(2 * (num_ranks - 1));
		int num_internode_steps = (int)(2 * num_nodes);
		latency = __fadd_rn(__fmul_rn((float)num_internode_steps, net_lat),
				    __fmul_rn((float)(num_steps - num_internode_steps), p2p_lat));
		bw = __fmul_rn(__fmul_rn(params.internode_bw, (float)params.num_rails),
			       (float)num_channels);
		break;
	}
	case ALGO_NVLS_TREE: {
		double t = __dadd_rn((double)p2p_lat, __dmul_rn(log2_nodes, (double)net_lat));
		latency = (float)__dmul_rn(2.0, t);
		float half = __fdiv_rn(__fmul_rn(params.internode_bw, (float)params.num_rails), 2.0f);
		bw = __fmul_rn(half < params.intranode_bw ? half : params.intranode_bw,
			       (float)num_channels);
		break;
	}
	case ALGO_TREE: {
		float a = __fmul_rn((float)(2 * ((num_ranks / num_nodes) - 1)), p2p_lat);
		double b = __dmul_rn(__dmul_rn(2.0, log2_nodes), (double)net_lat);
		latency = (float)__dadd_rn((double)a, b);
		bw = __fdiv_rn(__fmul_rn(__fmul_rn(params.internode_bw, (float)params.num_rails),
					 (float)num_channels),
			       2.0f);
		break;
	}
	default:
		return -1.0f;
	}

	if (proto == PROTO_LL) {
		bw = (float)__dmul_rn((double)bw, 0.5);
	} else if (proto == PROTO_LL128) {
		bw = (float)__dmul_rn((double)bw, 0.9375);
	}
	return __fadd_rn(__fmul_rn(latency, (float)pipe_ops), __fdiv_rn((float)size, bw));
}

/* The three protocols of one algorithm at once: cell for cell the operations of model_cost above,
 * in the same order, with what the three cells share worked out once (the step counts and their
 * conversions, the base bandwidth, the rank quotient and the log term).  size_f = (float)size,
 * ranks_over_nodes = num_ranks / num_nodes (a grid knows it without dividing). */
__device__ inline void model_cost_protos(int platform, int coll, int algo, int pipe_ops, float size_f,
					 uint64_t num_ranks, uint64_t num_nodes, uint64_t ranks_over_nodes,
					 double log2_nodes, int num_channels, int net_comp_overhead,
					 float out[NUM_PROTOS])
{
	out[PROTO_LL] = out[PROTO_LL128] = out[PROTO_SIMPLE] = -1.0f;
	if (coll != FUNC_ALLREDUCE || (algo != ALGO_RING && algo != ALGO_TREE && algo != ALGO_NVLS_TREE)) {
		return;
	}
	const model_params_t params = model_params(platform);
	const float net_lat_of[NUM_PROTOS] = { params.net_lat, params.net_lat,
					       __fadd_rn(params.net_lat, (float)net_comp_overhead) };
	const float rails_bw = __fmul_rn(params.internode_bw, (float)params.num_rails);
	float latency[NUM_PROTOS], bw;
	if (algo == ALGO_RING) {
		const int num_steps = (int)(2 * (num_ranks - 1));
		const int num_internode_steps = (int)(2 * num_nodes);
		const float inter = (float)num_internode_steps, rest = (float)(num_steps - num_internode_steps);
#pragma unroll
		for (int proto = 0; proto < NUM_PROTOS; proto++) {
			latency[proto] = __fadd_rn(__fmul_rn(inter, net_lat_of[proto]),
						   __fmul_rn(rest, nvlink_lat(ALGO_RING, proto)));
		}
		bw = __fmul_rn(rails_bw, (float)num_channels);
	} else if (algo == ALGO_NVLS_TREE) {
#pragma unroll
		for (int proto = 0; proto < NUM_PROTOS; proto++) {
			const double t = __dadd_rn((double)nvlink_lat(ALGO_NVLS_TREE, proto),
						   __dmul_rn(log2_nodes, (double)net_lat_of[proto]));
			latency[proto] = (float)__dmul_rn(2.0, t);
		}
		const float half = __fdiv_rn(rails_bw, 2.0f);
		bw = __fmul_rn(half < params.intranode_bw ? half : params.intranode_bw, (float)num_channels);
	} else {
		const float hops = (float)(2 * (ranks_over_nodes - 1));
		const double log_term = __dmul_rn(2.0, log2_nodes);
#pragma unroll
		for (int proto = 0; proto < NUM_PROTOS; proto++) {
			const float a = __fmul_rn(hops, nvlink_lat(ALGO_TREE, proto));
			const double b = __dmul_rn(log_term, (double)net_lat_of[proto]);
			latency[proto] = (float)__dadd_rn((double)a, b);
		}
		bw = __fdiv_rn(__fmul_rn(rails_bw, (float)num_channels), 2.0f);
	}
	const float bw_of[NUM_PROTOS] = { (float)__dmul_rn((double)bw, 0.5), (float)__dmul_rn((double)bw, 0.9375), bw };
	const float pipe = (float)pipe_ops;
#pragma unroll
	for (int proto = 0; proto < NUM_PROTOS; proto++) {
		out[proto] = __fadd_rn(__fmul_rn(latency[proto], pipe), __fdiv_rn(size_f, bw_of[proto]));
	}
}

/* model_get_coll_info_internal_v3 (:154-234); with the NVLS-tree bit of `mask`
 * clear it is _v2 with nvlsSupport == 0 (:236-309).  The model never looks at
 * NCCL's cost table, so no other bit of the mask matters here.  cost_of(algo, proto) is the
 * cell's cost, negative when not modelled. */
template <typename F>
__device__ __forceinline__ void model_choose_with(int platform, int coll, uint64_t size, uint64_t ranks,
						  uint64_t nodes, uint32_t mask, F cost_of, int &chosen_algo,
						  int &chosen_proto)
{
	chosen_algo = -1;
	chosen_proto = -1;
	if (!platform_has_model(platform) || nodes <= 2) { /* :178 */
		return;
	}
	const bool nvls = allowed(mask, ALGO_NVLS_TREE, PROTO_SIMPLE);
	if (platform == OFI_AMD_PLATFORM_P5_P5E && coll == FUNC_ALLREDUCE && nodes == 16 &&
	    ranks == 128 && nvls && size > 3ULL * 1024 * 1024 * 1024 &&
	    size <= 5ULL * 1024 * 1024 * 1024) { /* :183-192 */
		chosen_algo = ALGO_NVLS_TREE;
		chosen_proto = PROTO_SIMPLE;
		return;
	}
	float lowest = 3.402823466e+38f; /* FLT_MAX */
	for (int algo = 0; algo < NUM_ALGOS; algo++) {
		if (algo == ALGO_COLLNET_DIRECT || algo == ALGO_COLLNET_CHAIN || algo == ALGO_NVLS) {
			continue;
		}
		if (algo == ALGO_NVLS_TREE && !nvls) {
			continue;
		}
		for (int proto = 0; proto < NUM_PROTOS; proto++) {
			if (algo == ALGO_NVLS_TREE && proto != PROTO_SIMPLE) {
				continue;
			}
			float c = cost_of(algo, proto);
			if (c < 0) {
				continue;
			}
			if (c < lowest) {
				chosen_algo = algo;
				chosen_proto = proto;
				lowest = c;
			}
		}
	}
}

__device__ inline void model_choose(int platform, int coll, uint64_t size, uint64_t ranks,
				    uint64_t nodes, double log2_nodes, int pipe_ops, int num_channels,
				    int net_comp_overhead, uint32_t mask, int &chosen_algo,
				    int &chosen_proto)
{
	model_choose_with(
		platform, coll, size, ranks, nodes, mask,
		[&](int algo, int proto) -> float {
			return model_cost(platform, coll, algo, proto, pipe_ops, size, ranks, nodes, log2_nodes,
					  num_channels, net_comp_overhead);
		},
		chosen_algo, chosen_proto);
}

/* ------------------------------------------------------------------ regions */

struct pt_t {
	double x, y;
};

typedef double double4_t __attribute__((ext_vector_type(4)));

/* one edge of a polygon, from the vertex before it (the last one for a polygon's first) to vertex `b` */
struct edge_t {
	pt_t a, b;
};

/* The polygons of one (platform, shape, collective): consecutive in `poly`, their edges -- at most 64 --
 * consecutive in `edges`.  polys == 0: no regions. */
struct region_set_t {
	uint16_t first_poly, polys, first_edge, edges;
};

struct region_tables_t {
	region_set_t set[kNumPlatforms][kNumShapes][NUM_FUNCS];
	const int32_t *poly; /* per polygon {algo, proto, first_edge, num_edges} */
	const edge_t *edges; /* log2 space */
	const double *bbox;  /* per polygon {min_x, max_x, min_y, max_y} as is_inside_region finds them */
	pt_t far_point;      /* log2 of (2*max size, 2*max ranks) */
};

__device__ __forceinline__ pt_t vsub(pt_t a, pt_t b) { return pt_t{ a.x - b.x, a.y - b.y }; }
__device__ __forceinline__ double vdot(pt_t a, pt_t b) { return a.x * b.x + a.y * b.y; }
__device__ __forceinline__ double vcross(pt_t a, pt_t b) { return a.x * b.y - a.y * b.x; }

/* ... where only the sign counts, and only when it is certain */
__device__ __forceinline__ double vcross_sign(pt_t a, pt_t b) { return __builtin_fma(a.x, b.y, -(a.y * b.x)); }

/* intersect, src/tuner/nccl_ofi_regions.cpp:77-109 */
__device__ inline int intersect(pt_t x0, pt_t x1, pt_t y0, pt_t y1, double eps, pt_t *sect)
{
	pt_t dx = vsub(x1, x0);
	pt_t dy = vsub(y1, y0);
	double d = vcross(dy, dx);
	if (fabs(d) < eps) {
		return 0;
	}
	double a = (vcross(x0, dx) - vcross(y0, dx)) / d;
	if (sect) {
		sect->x = y0.x + a * dy.x;
		sect->y = y0.y + a * dy.y;
	}
	if (a < -eps || a > 1 + eps) {
		return -1;
	}
	if (a < eps || a > 1 - eps) {
		return 0;
	}
	a = (vcross(x0, dy) - vcross(y0, dy)) / d;
	if (a < 0 || a > 1) {
		return -1;
	}
	return 1;
}

/* distance, :125-142 */
__device__ inline double seg_distance(pt_t x, pt_t y0, pt_t y1, double eps)
{
	pt_t dy = vsub(y1, y0);
	pt_t x1, s = { 0, 0 };
	x1.x = x.x + dy.y;
	x1.y = x.y - dy.x;
	int r = intersect(x, x1, y0, y1, eps, &s);
	if (r == -1) {
		return HUGE_VAL;
	}
	s = vsub(s, x);
	return sqrt(vdot(s, s));
}

/*
 * Certain-answer forms of the two per-edge tests, from the signs of cross products: no division, no
 * square root, no branch.  With P the point, F the far end of its ray and A, B the edge's ends,
 *
 *   side_a, side_b = (A - P) x (F - P), (B - P) x (F - P)     which side of the ray's line A and B lie on
 *   side_p, side_f = (P - A) x (B - A), (F - A) x (B - A)     which side of the edge's line P and F lie on
 *
 * `intersect`'s quotients are a = side_a / (side_a - side_b) and b = side_p / (side_p - side_f).
 * Coordinates are logarithms to base 2 of 64-bit numbers, so a cross product is below 2e4 and is
 * computed to 1e-11: with |side_a| and |side_b| above kSure = 1e-4, a is outside [0, 1] by 5e-9 when the
 * signs agree and inside (eps, 1 - eps) by as much when they differ (eps is 1e-10), and the same holds
 * for b.  What is not certain goes through the exact code above, so results are the exact code's.
 */
constexpr double kSure = 1e-4;

struct edge_sides_t {
	double side_a, side_b, side_p;
};

__device__ __forceinline__ edge_sides_t edge_sides(pt_t p, pt_t ray, pt_t a, pt_t b)
{
	const pt_t pa = vsub(a, p), pb = vsub(b, p);
	return edge_sides_t{ vcross(pa, ray), vcross(pb, ray), vcross(pb, pa) };
}

/* n / d < t as the exact code's rounded quotient compares, d > 0; `sure` is cleared when n and t * d are too
 * close to tell without dividing (their rounding errors and the quotient's are below 4e-16 of either) */
__device__ __forceinline__ bool quotient_below(double n, double d, double t, bool &sure)
{
	const double gap = n - t * d;
	sure &= fabs(gap) > 1e-15 * (fabs(n) + d);
	return gap < 0;
}

/* intersect(x0, x1, y0, y1, eps, nullptr) == 1.  Grid points sit on the lines of many edges (rank counts that
 * are powers of two), where the quotients are 0 or 1 to the last bit and the signs are not certain; comparing
 * products instead of quotients answers those too, and the two divisions are left for what is within
 * rounding of a threshold. */
__device__ __forceinline__ bool intersects(pt_t x0, pt_t x1, pt_t y0, pt_t y1, double eps)
{
	const pt_t dx = vsub(x1, x0), dy = vsub(y1, y0);
	const double d = vcross(dy, dx), n = vcross(x0, dx) - vcross(y0, dx), m = vcross(x0, dy) - vcross(y0, dy);
	if (fabs(d) < eps) {
		return false;
	}
	const double s = d < 0 ? -1.0 : 1.0, D = fabs(d);
	bool sure = true;
	/* eps <= a <= 1 - eps and 0 <= b <= 1 (what lies beyond -eps or 1 + eps lies beyond these too; a
	 * quotient's sign is exact) */
	const bool inside = !quotient_below(s * n, D, eps, sure) && quotient_below(s * n, D, 1 - eps, sure) &&
			    s * m >= 0 && quotient_below(s * m, D, 1.0, sure);
	return sure ? inside : intersect(x0, x1, y0, y1, eps, nullptr) == 1;
}

/* `crossing` is intersect(p, far, a, b, eps, nullptr) == 1 wherever `crossing_certain` */
__device__ __forceinline__ bool crossing_certain(const edge_sides_t &s, double side_f)
{
	const bool apart = (s.side_a > 0) != (s.side_b > 0);
	return fmin(fabs(s.side_a), fabs(s.side_b)) > kSure &&
	       (!apart || fmin(fabs(s.side_p), fabs(side_f)) > kSure);
}
__device__ __forceinline__ bool crossing(const edge_sides_t &s, double side_f)
{
	return (s.side_a > 0) != (s.side_b > 0) && (s.side_p > 0) != (side_f > 0);
}

/* Whether seg_distance(p, a, b, eps) < eps.  |side_p| is the
 * distance to the edge's line times the edge's length, `along` the foot point's place on the edge times the
 * length squared.  Distances come out to 1e-11 here and to 1e-13 in the exact code (edges are at least
 * kMinEdge long), so a distance beyond 2 eps, or a foot point beyond an end by 1e-6 of the length, is a no.
 * With the foot point as far inside the ends, a point on the side the exact code's perpendicular does not lead
 * to the edge from is a no however close it is (its second quotient is below 0: `m` has that quotient's sign
 * by the same operations), and one on the line or on the other side within half an eps is a yes.  What is
 * left goes through the exact code, as does an edge of length 0 (some polygons list their first vertex
 * again). */
constexpr double kMinEdge = 0.04;
__device__ __forceinline__ bool touches_edge(pt_t p, pt_t a, pt_t b, const edge_sides_t &s, double eps)
{
	const pt_t d = vsub(b, a);
	const double along = vdot(vsub(p, a), d), len2 = vdot(d, d), ends = 1e-6 * len2;
	const double far2 = s.side_p * s.side_p, eps2 = eps * eps * len2;
	const double m = vcross(p, d) - vcross(a, d);
	const bool within = along > ends && along < len2 - ends;
	const bool no = far2 > 4.0 * eps2 || along < -ends || along > len2 + ends || (within && m > 0);
	const bool yes = within && m <= 0 && far2 < 0.25 * eps2;
	return yes || (!no && seg_distance(p, a, b, eps) < eps);
}

/* A point with |side_p| beyond this is farther than kSure from the edge's line: touches_edge is false */
__device__ __forceinline__ double touch_reach(pt_t a, pt_t b)
{
	return kSure * (fabs(b.x - a.x) + fabs(b.y - a.y));
}

/* The bounds is_inside_region computes (:177-196): selections only, so the host can do it
 * once per polygon with the same result.  The y bounds start from vertex 1 as in the reference
 * (:177-178). */
__host__ __device__ inline void region_bounds(const pt_t *v, int n, double out[4])
{
	double min_x = v[0].x, max_x = v[0].x, min_y = v[1].y, max_y = v[1].y;
	for (int i = 0; i < n; i++) {
		if (v[i].x > max_x) max_x = v[i].x;
		if (v[i].x < min_x) min_x = v[i].x;
		if (v[i].y > max_y) max_y = v[i].y;
		if (v[i].y < min_y) min_y = v[i].y;
	}
	out[0] = min_x;
	out[1] = max_x;
	out[2] = min_y;
	out[3] = max_y;
}

/* The edges of polygon i of a set as bits of a wavefront's lanes (edge e of the set is lane e's) */
__device__ __forceinline__ uint64_t edge_lanes(int first_edge, int count)
{
	return (count >= 64 ? ~0ull : (1ull << count) - 1ull) << first_edge;
}

/* is_inside_region's bounding-box test (:159-221) */
__device__ __forceinline__ bool in_bounds(pt_t p, const double *b, double margin)
{
	return !(p.x < b[0] - margin || p.x > b[1] + margin || p.y < b[2] - margin || p.y > b[3] + margin);
}

/*
 * calculateChunkSizeTreeLL128, :1883-1938 (constants: include/internal/tuner/nccl_defaults.h), for the
 * three channel counts its caller tries.  The chunk only ever takes the values kChunkLadder -- it starts
 * at 640 threads x 120 elements x 8 bytes x 15/16 and is halved while the message has too few chunks for
 * the tree's depth -- so every division is by a constant, the ladder's quotients do not wait for each
 * other, and the payload of a rung (whole 1920-byte grains, 480 elements to 2048 bytes) is a
 * constant too.  Messages are at most 32 MiB here.
 */
constexpr uint32_t kChunkLadder[6] = { 576000, 288000, 144000, 72000, 36000, 18000 };
constexpr uint64_t chunk_payload(uint32_t chunk)
{
	const uint32_t grain = 32 * 8 / 16 * 15 * 8; /* 1920 bytes */
	const uint32_t nelem = chunk / grain * (grain / 4);
	return (uint64_t)((nelem + 479) / 480) * 256 * 8;
}

template <uint32_t CHANNELS>
__device__ __forceinline__ uint64_t chunk_tree_ll128(uint32_t message_size, int log2_nnodes)
{
	const int ppn = 8;
	const double nSteps = 1 + log2_nnodes + 0.1 * ppn;
	const double deep = nSteps * 64 / ppn, shallow = nSteps * 16 / ppn;
	int rung = 0;
#pragma unroll
	for (int k = 0; k < 3; k++) { /* while chunk > 131072 */
		rung += rung == k && (double)(message_size / (CHANNELS * kChunkLadder[k])) < deep;
	}
#pragma unroll
	for (int k = 0; k < 5; k++) { /* while chunk > 32768 */
		rung += rung == k && (double)(message_size / (CHANNELS * kChunkLadder[k])) < shallow;
	}
	uint64_t payload = chunk_payload(kChunkLadder[0]);
#pragma unroll
	for (int k = 1; k < 6; k++) {
		payload = rung == k ? chunk_payload(kChunkLadder[k]) : payload;
	}
	return payload;
}

__device__ __forceinline__ int log2i_nodes(uint64_t nodes)
{
	const int x = (int)nodes; /* log2i(int), include/internal/tuner/nccl_defaults.h:92-104 */
	return x <= 0 ? -1 : 31 - __clz(x);
}

/* Which polygon set answers for (platform, collective, ranks per node): shape selection as in
 * the per-platform init functions (:302,:485,:675,:768,:878,...).  The host looks it up: kernels get
 * the set. */
inline region_set_t region_set(const region_tables_t &t, int platform, int coll, uint64_t ranks, uint64_t nodes)
{
	int shape = -1;
	if (ranks == 8 * nodes) shape = 0;
	else if (ranks == 2 * nodes && platform == OFI_AMD_PLATFORM_P5_P5E) shape = 1;
	else if (ranks == nodes) shape = 2;
	if (platform < 0 || platform >= kNumPlatforms || shape < 0 || coll < 0 || coll >= NUM_FUNCS) {
		return region_set_t{};
	}
	return t.set[platform][shape][coll];
}

/* The nChannels override of the chosen region (:2135-2153), -1 when there is none; only P6 has any. */
__host__ __device__ inline bool platform_sets_channels(int platform) { return platform == OFI_AMD_PLATFORM_P6; }
__device__ __forceinline__ int region_channels(int platform, uint64_t size, uint64_t ranks, uint64_t nodes,
						int algorithm, int protocol)
{
	int nchannels = -1;
	if (platform == OFI_AMD_PLATFORM_P6 && size >= 4 * 1024 * 1024 && size <= 32 * 1024 * 1024 &&
	    algorithm == ALGO_TREE && protocol == PROTO_LL128 && nodes * 8 == ranks) { /* :2140-2146 */
		const int log2_nnodes = log2i_nodes(nodes);
		/* calculateBestNChannelTree, :1955-1971: the largest payload, the most channels when they tie */
		const uint32_t bytes = (uint32_t)size;
		const uint64_t with16 = chunk_tree_ll128<16>(bytes, log2_nnodes), with24 = chunk_tree_ll128<24>(bytes, log2_nnodes),
			       with32 = chunk_tree_ll128<32>(bytes, log2_nnodes);
		const int best = with32 >= with24 && with32 >= with16 ? 32 : (with24 >= with16 ? 24 : 16);
		nchannels = best;
	}
	if (platform == OFI_AMD_PLATFORM_P6 && size <= 32 * 1024 * 1024 && algorithm == ALGO_PAT &&
	    protocol == PROTO_SIMPLE && nodes == ranks) {
		/* calculateBestNChannelPat, :1943-1953 */
		nchannels = 0;
		if (size <= nodes * 65536) nchannels = 1;
		else if (size <= nodes * 65536 * 2) nchannels = 2;
	}
	return nchannels;
}

/* region_get_chunk_size_internal, :2276-2306, with chunkSizeTuningTreeLL128P5en
 * (:2211-2274) and chunkSizeTuningAllGatherPatSimpleP5en (:2159-2209).
 * Returns 0 when the tuner leaves the chunk size alone. */
__device__ inline uint64_t region_chunk_size(int platform, int coll, uint64_t nbytes, int algo, int proto,
					     uint64_t ranks, uint64_t nodes)
{
	if (nodes != ranks || platform != OFI_AMD_PLATFORM_P5EN) {
		return 0;
	}
	if (coll == FUNC_ALLREDUCE && algo == ALGO_TREE && proto == PROTO_LL128) {
		const uint64_t nsteps = (uint64_t)(1 + log2i_nodes(nodes));
		uint64_t tuned = 288000;
		if (nbytes / tuned < 2 * nsteps * nsteps) tuned /= 2;
		if (nbytes / tuned < (uint64_t)(1.5 * (double)nsteps)) tuned /= 2;
		while (nbytes / tuned < nsteps + 1 && tuned > 18000) tuned /= 2;
		return tuned;
	}
	if (coll == FUNC_ALLGATHER && algo == ALGO_PAT && proto == PROTO_SIMPLE) {
		const uint64_t sat = nodes >= 16 ? 524288 : 1048576;
		const uint64_t T1 = nodes >= 16 ? 32 : (nodes < 8 ? nodes : 8) + 1;
		const uint64_t T2 = nodes < 16 ? nodes : 16;
		const uint64_t T3 = nodes < 8 ? nodes : 8;
		uint64_t tuned = sat;
		while (nbytes / tuned < T1 && tuned > sat / 2) tuned /= 2;
		while (nbytes / tuned < T2 && tuned > 65536) tuned /= 2;
		while (nbytes / tuned < T3 && tuned > 32768) tuned /= 2;
		return tuned;
	}
	return 0;
}

/* Host side (tuner_grid.hip): the process-wide device copy of the polygon tables and
 * transform_log2 (include/tuner/nccl_ofi_tuner_region.h:87-109) of one coordinate. */
int device_region_tables(region_tables_t *out);
double log2_coord(double v);

} // namespace ofi_amd_tuner

#endif
