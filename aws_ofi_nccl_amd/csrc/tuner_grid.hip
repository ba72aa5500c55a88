/*
 * Batched tuner evaluation for gfx950: the cost model and the region lookup over a
 * whole grid of (collective, size, nodes, ranks/node) points in one call.  The
 * arithmetic lives in tuner_device.hpp; this file holds the grid kernels, the plan
 * object and the host-side construction of the log2-space polygon tables
 * (extend_region + set_regions, src/tuner/nccl_ofi_regions.cpp:224-289).
 *
 * Nothing here is matrix-shaped: one thread per decision point, which also evaluates the
 * point's cost cells (staged in LDS, written out as contiguous runs).
 */
#include <algorithm>
#include <cstring>
#include <mutex>
#include <new>
#include <vector>

#include "common.hpp"
#include "tuner_device.hpp"
#include "region_tables.inc"

using namespace ofi_amd_tuner;

namespace {

/* Quotients of numbers below 2^31 by a number fixed at plan time: with 2^(l-1) < d <= 2^l and m = ceil(2^(31+l) / d),
 * x / d = x * m >> (31 + l), because m * d exceeds 2^(31+l) by less than d <= 2^l */
struct divisor_t {
	uint32_t d, m, l;
};
divisor_t divisor(uint32_t d)
{
	const uint32_t l = d <= 1 ? 0 : 32 - (uint32_t)__builtin_clz(d - 1);
	return { d, (uint32_t)(((1ull << (31 + l)) + d - 1) / d), l };
}
__device__ __forceinline__ uint32_t quotient(uint32_t x, const divisor_t &by)
{
	return __umulhi(x << 1, by.m) >> by.l;
}

struct grid_dims_t {
	uint32_t n_colls, n_sizes, n_nodes, n_ppn, n_algos;
	divisor_t by_ppn, by_nodes, by_coll; /* by_coll: the points of a collective */
	const int32_t *colls;
	const uint64_t *sizes;
	const uint64_t *nodes;
	const uint32_t *ppn;
	const int32_t *algos;
	const double *log2_nodes; /* log2((double)nodes[i]) from the host's libm */
	const double *log2_sizes; /* per size index: transform_log2 of the byte count */
	const double *log2_ranks; /* per (node, ppn): transform_log2 of the rank count */
};

/* tiles of the region grid: 2^shift_n node counts x 2^shift_s sizes, a wavefront each */
struct tiling_t {
	uint32_t shift_n, shift_s, tiles_n, tiles_s;
	const double2 *size_span; /* per tile row: smallest and largest log2_sizes */
	const double2 *rank_span; /* per (tile column, ppn): smallest and largest log2_ranks */
};

/* Model workgroups have 256 threads and, from 48 MiB of costs on (68 where every point is modelled: 64 MB 13.0 us with
 * eight and 14.3 with five, 76 MB 16.0 and 16.1, 82 MB 17.4 and 16.8), claim enough LDS that five of them share a CU instead
 * of eight: the fewer and longer the runs under way, the better they suit the memory.  From 150 MiB on, 1024 threads write
 * longer runs still, but they also evaluate the model all at once and then write all at once, so that they are
 * the slower way where more than half of the points are modelled.  Times in us with eight and with five of 256, and with 1024
 * threads, by the share of modelled points:
 *           a third              half                 two thirds           all
 *    45 MB   8.6 / 8.9 / 10.0     8.7 / 9.7 / 10.3     9.2 / 10.1 / 10.5   10.4 / 11.2 / 13.1
 *    60 MB  12.5 / 12.0 / 12.0   12.3 / 12.4 / 13.0   13.5 / 12.0 / 13.5   13.2 / 13.9 / 15.1
 *    85 MB  16.4 / 15.9 / 16.6   16.2 / 16.6 / 17.4   17.0 / 16.7 / 17.8   18.6 / 17.6 / 19.6
 *   120 MB  23.0 / 22.6 / 22.8   23.0 / 23.0 / 23.9   23.8 / 23.2 / 24.3   24.8 / 23.2 / 25.3
 *   180 MB  34.9 / 34.5 / 33.6   34.8 / 35.2 / 34.9   35.4 / 34.6 / 35.1   34.8 / 32.3 / 34.3
 *   250 MB  47.9 / 47.4 / 46.2   48.4 / 48.0 / 48.1   48.3 / 47.8 / 48.0   47.5 / 43.2 / 45.9
 *   480 MB  91.6 / 91.2 / 88.0   94.2 / 93.4 / 90.5   90.8 / 90.5 / 91.3   90.5 / 79.3 / 84.2 */
constexpr uint32_t kModelThreads = 256, kModelThreadsLarge = 1024;
constexpr uint64_t kModelFewerBytes = 48ull << 20, kModelFewerBytesAll = 68ull << 20, kModelLargeBytes = 150ull << 20;
/* LDS is handed out in units of 1280 bytes, 128 of them to a CU: with column_of this is 22 units, five times and not six */
constexpr size_t kModelFewerLds = 27000;
constexpr size_t kLdsUnit = 1280, kLdsUnits = 128;
static_assert(kLdsUnits / ((kModelFewerLds + kLdsUnit - 1) / kLdsUnit) == 5 &&
	      kLdsUnits / ((kModelFewerLds + NUM_ALGOS * sizeof(int32_t) + kLdsUnit - 1) / kLdsUnit) == 5, "workgroups to a CU");
constexpr size_t kModelLds = 64 * 1024; /* at most, for the larger ones */

/* `cells` doubles at `out`, cell(k) each, by a workgroup: two to a lane and store, 1 KiB per wavefront
 * instruction, where the address allows it */
template <uint32_t kThreads, typename F> __device__ __forceinline__ void write_cells(double *__restrict__ out, uint32_t cells, F cell)
{
	if ((reinterpret_cast<uintptr_t>(out) & 15u) == 0) {
		typedef double double2_t __attribute__((ext_vector_type(2)));
		double2_t *to = reinterpret_cast<double2_t *>(out);
		for (uint32_t k = threadIdx.x; k < cells / 2; k += kThreads) {
			const double2_t v = { cell(2 * k), cell(2 * k + 1) };
			__builtin_nontemporal_store(v, &to[k]);
		}
		if ((cells & 1u) && threadIdx.x == 0) {
			out[cells - 1] = cell(cells - 1);
		}
	} else {
		for (uint32_t k = threadIdx.x; k < cells; k += kThreads) {
			__builtin_nontemporal_store(cell(k), &out[k]);
		}
	}
}

__device__ __forceinline__ void write_choice(int8_t *__restrict__ choice, uint64_t point, int algo, int proto)
{
	const uint64_t at = point * 2u;
	if ((reinterpret_cast<uintptr_t>(choice) & 1u) == 0) {
		*reinterpret_cast<uint16_t *>(choice + at) =
			(uint16_t)((uint8_t)(int8_t)algo | ((uint32_t)(uint8_t)(int8_t)proto << 8));
	} else {
		choice[at + 0] = (int8_t)algo;
		choice[at + 1] = (int8_t)proto;
	}
}

/*
 * One thread per decision point; blockIdx.y is the variant.  The thread evaluates the
 * n_algos x 3 cost cells of its point -- contiguous in the output -- and its decision.  Cells
 * are staged in LDS, as the floats they are, so that the workgroup writes its points' doubles as one
 * contiguous run (a lane-per-point store would touch 64 cache lines per instruction).
 * Bound by that write, which goes at 5.4 TB/s from 60 MB on, and below by its own instructions: a workgroup without a
 * modelled point (two collectives in three, and platforms without a model) writes its -1s and is done, indices are
 * taken apart by multiplications, and floats make half the LDS traffic of doubles.  140 sizes x 11 node counts: 30 grids
 * 9.9 -> 8.0 us, 64 grids 16.5 -> 16.3.
 */
template <bool COST, bool CHOICE, uint32_t kThreads = kModelThreads>
__global__ __launch_bounds__(kThreads) void model_grid_kernel(double *__restrict__ cost,
							 const ofi_amd_tuner_variant_t *__restrict__ variants,
							 int8_t *__restrict__ choice, uint32_t points_per_variant, grid_dims_t g)
{
	extern __shared__ float stage[]; /* [kThreads][cells per point] when COST */
	__shared__ int32_t column_of[NUM_ALGOS]; /* the plan's column of an algorithm, -1: none */
	const uint32_t cpp = g.n_algos * NUM_PROTOS;
	const uint32_t first = blockIdx.x * kThreads, valid = min(kThreads, points_per_variant - first);
	const uint32_t p = first + threadIdx.x;
	const ofi_amd_tuner_variant_t v = variants[blockIdx.y];
	const bool live = threadIdx.x < valid;
	const uint64_t variant_at = (uint64_t)blockIdx.y * points_per_variant;
	double *out = COST ? cost + (variant_at + first) * cpp : nullptr;

	bool modelled = false; /* any point of the workgroup */
	if (platform_has_model(v.platform)) {
		const uint32_t last_coll = quotient(first + valid - 1u, g.by_coll);
		for (uint32_t c = quotient(first, g.by_coll); c <= last_coll; c++) {
			modelled |= g.colls[c] == FUNC_ALLREDUCE;
		}
	}
	if (!modelled) {
		if (COST) {
			write_cells<kThreads>(out, valid * cpp, [](uint32_t) { return -1.0; });
		}
		if (CHOICE && live) {
			write_choice(choice, variant_at + p, -1, -1);
		}
		return;
	}
	if (COST && CHOICE) {
		if (threadIdx.x < NUM_ALGOS) {
			int32_t col = -1;
			for (uint32_t ai = g.n_algos; ai-- > 0;) {
				col = g.algos[ai] == (int32_t)threadIdx.x ? (int32_t)ai : col;
			}
			column_of[threadIdx.x] = col;
		}
		__syncthreads();
	}
	if (live) {
		const uint32_t ci = quotient(p, g.by_coll), of_coll = p - ci * g.by_coll.d;
		const uint32_t row = quotient(of_coll, g.by_ppn), pi = of_coll - row * g.n_ppn;
		const uint32_t si = quotient(row, g.by_nodes), ni = row - si * g.n_nodes;
		const uint64_t nodes = g.nodes[ni];
		const uint64_t per_node = g.ppn[pi];
		const uint64_t ranks = nodes * per_node;
		if (COST) {
			const float size_f = (float)g.sizes[si];
			const int coll = g.colls[ci];
			const double log2_nodes = g.log2_nodes[ni];
			for (uint32_t ai = 0; ai < g.n_algos; ai++) {
				float c[NUM_PROTOS];
				/* ranks = nodes * per_node, so ranks / nodes is per_node */
				model_cost_protos(v.platform, coll, g.algos[ai], v.pipe_ops, size_f, ranks, nodes, per_node,
						  log2_nodes, v.num_channels, v.net_comp_overhead, c);
#pragma unroll
				for (uint32_t proto = 0; proto < NUM_PROTOS; proto++) {
					stage[threadIdx.x * cpp + ai * NUM_PROTOS + proto] = c[proto];
				}
			}
		}
		if (CHOICE) {
			int algo, proto;
			if (COST) {
				/* the cells the decision looks at have just been worked out: it reads this thread's
				 * row of the stage instead of evaluating the model again, and goes to the model
				 * only for an algorithm the plan has no column for */
				const float *cells = &stage[threadIdx.x * cpp];
				model_choose_with(
					v.platform, g.colls[ci], g.sizes[si], ranks, nodes, kAllAllowed,
					[&](int a, int pr) -> float {
						const int32_t col = column_of[a];
						if (col >= 0) {
							return cells[col * NUM_PROTOS + pr];
						}
						return model_cost(v.platform, g.colls[ci], a, pr, v.pipe_ops, g.sizes[si], ranks,
								  nodes, g.log2_nodes[ni], v.num_channels, v.net_comp_overhead);
					},
					algo, proto);
			} else {
				model_choose(v.platform, g.colls[ci], g.sizes[si], ranks, nodes, g.log2_nodes[ni], v.pipe_ops,
					     v.num_channels, v.net_comp_overhead, kAllAllowed, algo, proto);
			}
			write_choice(choice, variant_at + p, algo, proto);
		}
	}
	if (COST) {
		__syncthreads();
		write_cells<kThreads>(out, valid * cpp, [&](uint32_t k) { return (double)stage[k]; });
	}
}

constexpr int kMaxSetEdges = 64; /* of one (platform, shape, collective) set: one per lane */
/* Wavefronts per workgroup of the region kernel: two in launches of more than kPairedTiles tiles, whose workgroups
 * take as long to hand out as to work off (560 sizes x 38 node counts of four platforms 9.3 -> 8.9 us, 280 x 38 7.65
 * -> 7.5; four wavefronts 9.3 and 7.7), one in smaller ones, where two gain nothing. */
constexpr uint32_t kMostRegionWaves = 2;
constexpr uint64_t kPairedTiles = 6000;
constexpr uint64_t kMostRuns = 65535; /* of one launch: gridDim.y */
constexpr uint32_t kXcds = 8;         /* workgroup w of a launch runs on XCD w mod 8, each with its own L2 */
static_assert(kMaxSetEdges <= 64, "one lane per edge of a set");

/* One (platform entry, collective, ranks per node) of a region grid: where its points go and which
 * polygons answer for it (region_set, looked up by the host: ranks = nodes * ppn, so the shape is a
 * function of ppn). */
struct region_run_t {
	uint32_t entry, ci, pi, ppn;
	uint32_t first_poly, first_edge;
	uint32_t counts;   /* edges << 16 | polygons; 0: no regions.  Whole words: they come through the scalar cache */
	int32_t platform;
};

/* What a whole tile knows about one edge of its polygon set: which of the sides of edge_sides are the same, and
 * certainly so, for every point of it, on which side its centre is, and whether a point of it may lie on the edge */
struct tile_edge_t {
	bool a_sure, b_sure, p_sure;
	bool a_pos, b_pos, p_pos;
	bool near;
};

/*
 * Edge e against the tile of points with centre `mid` and half extents `half`.  The sides of edge_sides are
 * affine in the point, so over the tile each stays within a reach, worked out from the extents, of its value at
 * the centre: when all of that is beyond kTileSure on one side, every point's certain answer is the same.  The
 * ends of most edges lie outside the narrow fan of rays between a tile and the far point.
 */
constexpr double kTileSure = 1e-3; /* > kSure */
__device__ __forceinline__ tile_edge_t tile_edge(const edge_t &e, pt_t mid, pt_t half, pt_t far)
{
	const pt_t d = vsub(e.b, e.a), fa = vsub(e.a, far), fb = vsub(e.b, far), fm = vsub(mid, far);
	auto reach = [half](pt_t v) { return __builtin_fma(half.x, fabs(v.y), half.y * fabs(v.x)); };
	const double sa = vcross_sign(fm, fa), sb = vcross_sign(fm, fb), sp = vcross_sign(vsub(mid, e.a), d), rp = reach(d);
	tile_edge_t r;
	r.a_sure = fabs(sa) > reach(fa) + kTileSure, r.a_pos = sa > 0;
	r.b_sure = fabs(sb) > reach(fb) + kTileSure, r.b_pos = sb > 0;
	r.p_sure = fabs(sp) > rp + kTileSure, r.p_pos = sp > 0;
	/* with the whole tile on one side of the edge's line, and not close to it, no point is near */
	bool near = fabs(sp) <= rp + kTileSure * (1.0 + fabs(d.x) + fabs(d.y));
	near &= fmin(e.a.x, e.b.x) <= mid.x + half.x + kTileSure; /* &= : no branches between the comparisons */
	near &= fmax(e.a.x, e.b.x) >= mid.x - half.x - kTileSure;
	near &= fmin(e.a.y, e.b.y) <= mid.y + half.y + kTileSure;
	near &= fmax(e.a.y, e.b.y) >= mid.y - half.y - kTileSure;
	r.near = near;
	return r;
}

__device__ __forceinline__ uint64_t lane_word(uint64_t v, int lane)
{
	const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
	const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane);
	return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ double lane_value(double v, int lane)
{
	return __longlong_as_double((long long)lane_word((uint64_t)__double_as_longlong(v), lane));
}

/* all lanes when m is not 0, else none */
__device__ __forceinline__ uint64_t every(uint64_t m)
{
	return m != 0 ? ~0ull : 0ull;
}

/*
 * One thread per point.  A wavefront works on a tile of neighbouring sizes and node
 * counts of one (collective, ranks per node) pair, because the polygon set depends on that pair
 * alone.  The launch is bound by arithmetic (chains of fp64 operations), so a wavefront first
 * works out, one edge per lane, what its whole tile has in common about each edge of the set
 * (tile_edge); the points then only look at what they differ about, read out of the lanes that hold it: the
 * vertices in the fan of rays from the tile to the far point, one side each, and the edges whose line runs
 * through the tile, three sides each.  More than half of a sweep's tiles lie apart from every polygon, the mean
 * tile has 0.1 such vertices and 0.5 such edges, but those along a border that points at the far point have up
 * to 14 and 19, and the launch lasts as long as they do, which is why their turns count instructions: 1.02 M points
 * of four platforms (560 sizes, 38 node counts) take 8.9-9.7 us by where the sizes lie, 10.9 with three sides of
 * every edge with an end in the fan and the tile's four corners against each edge, 40-42 with every edge for every
 * point and quotients; 4.6 without any polygon, the launch and the handing out of 16,896 wavefronts
 * (kMostRegionWaves).  Measured and slower: the sides a tile knows left out one by one (branches on scalars: 12.4),
 * two points a lane and half the wavefronts (11.6: the longest tile counts), two edges a turn.  A grid of few points
 * is the time of such a tile alone, and takes smaller ones (pick_tiling).
 *
 * In the output the ranks-per-node index runs fastest, so a wavefront's records lie 4 x
 * n_ppn bytes apart and the records between them belong to the same tile's other
 * ranks-per-node values, i.e. to other workgroups.  Those workgroups are given numbers that
 * are equal mod 8: they run on the same XCD, their partial writes to a cache line meet in that
 * XCD's L2 and leave it as one line (64 grids of 140 sizes x 11 node counts: 7.1 MB written for 4.7 MB of
 * records, the rest lines that tiles side by side share; with the workgroups of a tile on different XCDs every
 * L2 wrote its quarter of each line, 18.9 MB).
 */
__global__ __launch_bounds__(64 * kMostRegionWaves) void region_choice_kernel(
	const region_run_t *__restrict__ runs, const int32_t *__restrict__ polys, const double *__restrict__ bboxes,
	const edge_t *__restrict__ edges, int8_t *__restrict__ choice, uint32_t points_per_platform, pt_t far_point, tiling_t t,
	grid_dims_t g)
{
	/* blockIdx.y names a run, blockIdx.x = 8 * group + x the tiles 8 * group .. 8 * group + 7 of it, of
	 * which XCD x takes one (workgroups are dealt to the XCDs in launch order, and gridDim.x is a
	 * multiple of 8); a second wavefront takes its tile from the other half of the groups.  The host lists the
	 * runs by falling cost (edges of the pair's set): the long workgroups start first and the short ones fill
	 * the end of the launch. */
	const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const region_run_t run = runs[blockIdx.y];
	/* The arguments that are not in registers yet lie on four lines of memory: all are asked for at once, along with the run,
	 * and not each when its turn comes (us, 1 platform of 120 x 12 4.7 -> 4.4, 4 of 280 x 30 7.5 -> 7.1, 4 of 560 x 44 8.9 ->
	 * 8.6; model grids lose by the same, 32 of 140 x 11 8.4 -> 8.8: their workgroups then write all at once). */
	__asm__ volatile("" : : "s"(far_point.x), "s"(far_point.y), "s"(t.size_span), "s"(t.rank_span), "s"(g.nodes), "s"(g.log2_sizes),
			 "s"(g.log2_ranks), "s"(run.first_poly), "s"(run.pi));
	/* which of a group's eight tiles an XCD takes rotates with the platform entry: the tiles
	 * differ in cost (size range), and an XCD that kept the same ones for every
	 * entry would keep the same share of the long ones */
	const uint32_t group = (blockIdx.x + wave * gridDim.x) / kXcds;
	const uint32_t tile = group * kXcds + (blockIdx.x + run.entry) % kXcds;
	if (tile >= t.tiles_n * t.tiles_s) {
		return; /* padding of the last group */
	}
	const uint32_t n_polys = run.counts & 0xffffu, n_edges = run.counts >> 16;
	const uint32_t ts = tile / t.tiles_n, tn = tile - ts * t.tiles_n;
	const uint32_t tile_points = 1u << (t.shift_n + t.shift_s), point = min(lane, tile_points - 1u);
	const uint32_t at_n = (tn << t.shift_n) + (point & ((1u << t.shift_n) - 1u));
	const uint32_t at_s = (ts << t.shift_s) + (point >> t.shift_n);
	const bool live = lane < tile_points && at_n < g.n_nodes && at_s < g.n_sizes;
	/* lanes beyond the tile's points and the axes' ends stand on the last point there is */
	const uint32_t ni = min(at_n, g.n_nodes - 1u), si = min(at_s, g.n_sizes - 1u);

	int algorithm = -1, protocol = -1, nchannels = -1;
	if (n_polys > 0) {
		/* everything the wavefront needs is asked for at once: its edge and, in the first lanes, a
		 * polygon's words and bounds; the loop below reads them out of the lanes */
		const uint32_t my_poly = run.first_poly + min(lane, n_polys - 1u);
		const int4 pw = reinterpret_cast<const int4 *>(polys)[my_poly];
		const double4_t box = reinterpret_cast<const double4_t *>(bboxes)[my_poly];
		/* lane e's edge; lanes beyond the set's edges take its last one and are masked out below */
		const edge_t mine = edges[run.first_edge + min(lane, n_edges - 1u)];
		const uint64_t nodes = g.nodes[ni];
		const pt_t at = { g.log2_sizes[si], g.log2_ranks[ni * g.n_ppn + run.pi] };
		const double2 sx = t.size_span[ts], sy = t.rank_span[tn * g.n_ppn + run.pi];

		/* The reference looks for a point on an edge first (result 0) and rejects by bounding
		 * box second (result -1).  A point more than 1e-6 outside the box cannot be within
		 * 1e-10 of an edge -- edges lie inside the box, and the foot of the perpendicular may
		 * leave the segment by at most eps times its length -- so for a tile of such points the second
		 * answer is known without looking at the edges. */
		const double margin = 1e-6;
		const uint64_t apart_polys = __ballot(sx.x > box.y + margin) | __ballot(sx.y < box.x - margin) |
					     __ballot(sy.x > box.w + margin) | __ballot(sy.y < box.z - margin);
		const uint64_t whole_polys = __ballot(sx.x >= box.x) & __ballot(sx.y <= box.y) & __ballot(sy.x >= box.z) &
					     __ballot(sy.y <= box.w);
		uint64_t todo = edge_lanes(0, (int)n_polys) & ~apart_polys;
		uint64_t open = __ballot(live) & __ballot(nodes > 2); /* the points still without a region */

		const double eps = 1e-10;
		const double mine_f = vcross(vsub(far_point, mine.a), vsub(mine.b, mine.a));
		const uint64_t mine_lanes = edge_lanes(pw.z - (int)run.first_edge, pw.w); /* of this lane's polygon */
		const pt_t mid = { 0.5 * (sx.x + sx.y), 0.5 * (sy.x + sy.y) }, half = { 0.5 * (sx.y - sx.x), 0.5 * (sy.y - sy.x) };
		const tile_edge_t te = tile_edge(mine, mid, half, far_point);
		/* points with a |side_p| up to this may lie on the edge */
		const double mine_reach = te.near ? touch_reach(mine.a, mine.b) : -1.0;
		/* From here on conditions are masks of lanes in scalar registers -- lanes standing for edges, polygons
		 * or points -- and the logic between them is scalar: no branch over lanes but the rare ones. */
		const uint64_t all = edge_lanes(0, (int)n_edges);
		const uint64_t a_sure = __ballot(te.a_sure), b_sure = __ballot(te.b_sure);
		const uint64_t a_pos = __ballot(te.a_pos), ends_apart = a_pos ^ __ballot(te.b_pos);
		const uint64_t f_pos = __ballot(mine_f > 0), f_sure = __ballot(fabs(mine_f) > kSure);
		/* Edges between whose line's sides every point and the far point certainly lie, or certainly do not: a ray
		 * crosses the former (`between`) when their ends lie apart, the latter never.  For the points to look
		 * at are left the ends in the fan of rays of edges between, and the edges whose line runs through the tile. */
		const uint64_t near = __ballot(te.near), line_sure = __ballot(te.p_sure) & f_sure & ~near;
		const uint64_t between = all & line_sure & (__ballot(te.p_pos) ^ f_pos);
		const uint64_t through = all & (near | ~(line_sure | (a_sure & b_sure & ~ends_apart)));
		for (; todo != 0 && open != 0; todo &= todo - 1) {
			const int i = __builtin_ctzll(todo);
			const uint64_t of_poly = lane_word(mine_lanes, i);
			/* The rays' crossings with the edges between, counted by vertex: an edge counts its first vertex when
			 * that lies on the positive side of the ray, and its second likewise, so that a vertex (bit e: the
			 * first of edge e) counts for the edges that meet in it, for neither when both are between. */
			const uint64_t c = between & of_poly;
			const uint64_t c_before = ((c << 1) & of_poly) | (((c >> (63 - __builtin_clzll(of_poly))) & 1u) << __builtin_ctzll(of_poly));
			const uint64_t counts = c ^ c_before;
			uint64_t odd = every((uint64_t)(__popcll(counts & a_sure & a_pos) & 1)); /* points with an odd number of crossings */
			uint64_t vertices = (c | c_before) & ~a_sure;
			uint64_t left = through & of_poly;
			if ((odd | vertices | left) == 0) {
				continue;
			}
			uint64_t in_box = open;
			if (!((whole_polys >> i) & 1u)) {
				in_box &= __ballot(at.x >= lane_value(box.x, i)) & __ballot(at.x <= lane_value(box.y, i)) &
					  __ballot(at.y >= lane_value(box.z, i)) & __ballot(at.y <= lane_value(box.w, i));
			}
			left &= near | every(in_box);
			if (in_box == 0 && left == 0) {
				continue; /* of the points still open none is in the box or on an edge */
			}
			const pt_t ray = vsub(far_point, at);
			uint64_t close = 0, touching = 0; /* close: a vertex may lie on the ray */
			for (; vertices != 0; vertices &= vertices - 1) {
				const int e = __builtin_ctzll(vertices);
				const pt_t a = { lane_value(mine.a.x, e), lane_value(mine.a.y, e) };
				const double side = vcross_sign(vsub(a, at), ray);
				close |= __ballot(fabs(side) <= kSure);
				odd ^= __ballot(side > 0) & every((counts >> e) & 1u);
			}
			close &= in_box;
			if (close != 0) {
				/* for these points the exact code on the edges between that have an end in the fan */
				uint64_t exact = every((uint64_t)(__popcll(c & a_sure & b_sure & ends_apart) & 1));
				for (uint64_t ask = c & ~(a_sure & b_sure); ask != 0; ask &= ask - 1) {
					const int e = __builtin_ctzll(ask);
					const pt_t a = { lane_value(mine.a.x, e), lane_value(mine.a.y, e) };
					const pt_t b = { lane_value(mine.b.x, e), lane_value(mine.b.y, e) };
					bool crosses = false;
					if ((close >> lane) & 1u) {
						crosses = intersects(at, far_point, a, b, eps);
					}
					exact ^= __ballot(crosses);
				}
				odd = (odd & ~close) | (exact & close);
			}
			/* where the far point is close to the line of an edge, the exact code, too */
			const uint64_t f_close = every(left & ~f_sure);
			for (; left != 0; left &= left - 1) {
				const int e = __builtin_ctzll(left);
				const pt_t a = { lane_value(mine.a.x, e), lane_value(mine.a.y, e) };
				const pt_t b = { lane_value(mine.b.x, e), lane_value(mine.b.y, e) };
				const pt_t pa = vsub(a, at), pb = vsub(b, at);
				const edge_sides_t s = { vcross_sign(pa, ray), vcross_sign(pb, ray), vcross_sign(pb, pa) };
				const uint64_t apart = __ballot(s.side_a > 0) ^ __ballot(s.side_b > 0);
				const uint64_t unsure = in_box & (__ballot(fabs(s.side_a) <= kSure) | __ballot(fabs(s.side_b) <= kSure) |
								  (apart & (__ballot(fabs(s.side_p) <= kSure) | f_close)));
				odd ^= apart & (__ballot(s.side_p > 0) ^ every((f_pos >> e) & 1u)) & ~unsure;
				const uint64_t reached = open & __ballot(fabs(s.side_p) <= lane_value(mine_reach, e));
				if ((unsure | reached) != 0) {
					bool crosses = false, t = false;
					if ((unsure >> lane) & 1u) {
						crosses = intersects(at, far_point, a, b, eps);
					}
					if ((reached >> lane) & 1u) {
						t = touches_edge(at, a, b, s, eps);
					}
					odd ^= __ballot(crosses);
					touching |= __ballot(t);
				}
			}
			const uint64_t hit = open & (touching | (odd & in_box));
			const int a = __builtin_amdgcn_readlane(pw.x, i), pr = __builtin_amdgcn_readlane(pw.y, i);
			algorithm = (hit >> lane) & 1u ? a : algorithm;
			protocol = (hit >> lane) & 1u ? pr : protocol;
			open &= ~hit;
		}
		if (algorithm >= 0 && platform_sets_channels(run.platform)) {
			nchannels = region_channels(run.platform, g.sizes[si], nodes * run.ppn, nodes, algorithm, protocol);
		}
	}
	if (!live) {
		return;
	}
	const uint32_t p = ((run.ci * g.n_sizes + si) * g.n_nodes + ni) * g.n_ppn + run.pi; /* output order */
	const uint64_t idx = (uint64_t)run.entry * points_per_platform + p;
	/* {int8 algorithm, int8 protocol, int16 nchannels} as one 4-byte store */
	reinterpret_cast<uint32_t *>(choice)[idx] = ((uint32_t)(uint8_t)(int8_t)algorithm) |
						     ((uint32_t)(uint8_t)(int8_t)protocol << 8) |
						     ((uint32_t)(uint16_t)(int16_t)nchannels << 16);
}

/* ---- host side: building the log2-space polygon tables ---- */

constexpr double kTunerMaxRanks = 1024.0 * 1024;               /* nccl_ofi_tuner_region.h:69 */
constexpr double kTunerMaxSize = 100.0 * 1024 * 1024 * 1024;   /* :74 */

/* transform_log2, include/tuner/nccl_ofi_tuner_region.h:87-109 */
pt_t to_log2(pt_t p)
{
	return pt_t{ log2_coord(p.x), log2_coord(p.y) };
}

/* extend_region, src/tuner/nccl_ofi_regions.cpp:254-289 */
pt_t extend(pt_t a, pt_t b, pt_t z)
{
	a = to_log2(a);
	b = to_log2(b);
	z = to_log2(z);
	pt_t ret;
	if (a.x == b.x) {
		ret = pt_t{ a.x, z.y };
	} else if (a.y == b.y) {
		ret = pt_t{ z.x, a.y };
	} else {
		double m = (a.y - b.y) / (a.x - b.x);
		double c = b.y - m * b.x;
		double projected_zy = m * z.x + c;
		if (projected_zy < z.y) {
			ret = pt_t{ z.x, projected_zy };
		} else {
			ret = pt_t{ (z.y - c) / m, z.y };
		}
	}
	return pt_t{ std::pow(2.0, ret.x), std::pow(2.0, ret.y) };
}

template <typename T>
int upload(const std::vector<T> &host, T **dev)
{
	*dev = nullptr;
	if (host.empty()) {
		return 0;
	}
	OFI_AMD_HIP_TRY(hipMalloc((void **)dev, host.size() * sizeof(T)));
	OFI_AMD_HIP_TRY(hipMemcpy(*dev, host.data(), host.size() * sizeof(T), hipMemcpyHostToDevice));
	return 0;
}

/* puts v's elements behind what `to` holds, on a 16-byte boundary; where they begin */
template <typename T>
size_t append(std::vector<uint8_t> &to, const std::vector<T> &v)
{
	const size_t at = (to.size() + 15) / 16 * 16;
	to.resize(at + v.size() * sizeof(T));
	std::memcpy(to.data() + at, v.data(), v.size() * sizeof(T));
	return at;
}

/* log2 of the node counts per tile of 64 points: of 4, 8 and 16 the one that leaves the fewest lanes idle at the
 * end of the axis, 8 x 8 when they tie (a square tile has the narrowest fan of rays) */
uint32_t pick_tile_shift(uint32_t n_nodes)
{
	uint32_t best = 3;
	for (const uint32_t shift : { 2u, 4u }) {
		const uint32_t padded = (n_nodes + (1u << shift) - 1) >> shift << shift;
		const uint32_t padded_best = (n_nodes + (1u << best) - 1) >> best << best;
		best = padded < padded_best ? shift : best;
	}
	return best;
}

uint32_t log2_ceil(uint32_t v)
{
	return v <= 1 ? 0 : 32 - (uint32_t)__builtin_clz(v - 1);
}

/*
 * Tilings a plan keeps, by falling size: 64, 16 (4 x 4), 8 (2 node counts x 4 sizes) and 4 points (2 x 2) to a
 * tile.  The points of a smaller tile differ about fewer edges, so its wavefront is done sooner, at the price of
 * more wavefronts, each of which costs 0.2 ns of dispatch and works out its edges' sides anew.
 * On an axis shorter than the tile, what is left over of the two largest goes to the other axis: one size and
 * 200,000 node counts of four platforms take 46 us in tiles of 64 node counts, 270 in squares with 7 of 8 lanes
 * idle, 3 sizes and 20,000 node counts 42 and 81.  The smallest tiles stay short there, which is what they are for (35
 * sizes at one node count: 4.1 us in pairs of points, 5.4 in fours).
 */
constexpr int kTilings = 4;
void tile_shifts(uint32_t n_sizes, uint32_t n_nodes, uint32_t shift_n[kTilings], uint32_t shift_s[kTilings])
{
	shift_n[0] = pick_tile_shift(n_nodes);
	shift_s[0] = 6 - shift_n[0];
	shift_n[1] = shift_s[1] = 2;
	shift_n[2] = 1, shift_s[2] = 2;
	shift_n[3] = shift_s[3] = 1;
	for (int i = 0; i < 2; i++) {
		const uint32_t most_n = log2_ceil(n_nodes), most_s = log2_ceil(n_sizes), both = shift_n[i] + shift_s[i];
		if (most_s < shift_s[i]) {
			shift_s[i] = most_s, shift_n[i] = both - most_s;
		} else if (most_n < shift_n[i]) {
			shift_n[i] = most_n, shift_s[i] = both - most_n;
		}
	}
}

/*
 * The smallest tiles that make at most kMostTiles: beyond, handing out the wavefronts costs more than their shorter
 * turns save.  Times in us with tiles of 64 / 16 / 8 / 4 points and, in brackets, the tiles these make (3
 * collectives, 4 values of ranks per node):
 *   35 sizes, 11 node counts, 4 platforms      14.9 / 8.8 / 7.5 / 6.1   [ 480, 1296, 2592, 5184]
 *   70 sizes, 11 node counts, 2 platforms      13.7 / 6.8 / 5.8 / 4.9   [ 432, 1296, 2592, 5040]
 *   140 sizes, 27 node counts, 1 platform       7.0 / 5.6 / 5.1 / 4.9   [ 840, 2940, 5880, 11760]
 *   35 sizes, 38 node counts, 4 platforms      10.8 / 7.2 / 7.3 / 7.1   [1200, 4320, 8208, 16416]
 *   140 sizes, 11 node counts, 4 platforms      9.8 / 7.1 / 6.4 / 7.5   [1728, 5040, 10080, 20160]
 *   160 sizes, 27 node counts, 3 platforms      7.4 / 6.6 / 7.6 / 12    [2880, 10080, 20160, 40320]
 *   140 sizes, 38 node counts, 4 platforms      7.6 / 8.1 / 10.1 / 18   [4320, 16800, 31920, 63840]
 * Two sizes far apart, whose tiles see every edge of a set, want fewer: 2000 node counts, 1 and 4 platforms 9.4 and 11.7
 * (3000 tiles of 16, 3024 of 64), 11.2 and 16.3 with four times as many.
 */
constexpr uint64_t kMostTiles = 10500;
uint64_t tiling_tiles(const tiling_t &t)
{
	return (uint64_t)t.tiles_n * t.tiles_s;
}

const tiling_t &pick_tiling(const tiling_t tilings[kTilings], uint64_t n_runs)
{
	int i = kTilings - 1;
	while (i > 0 && n_runs * tiling_tiles(tilings[i]) > kMostTiles) {
		i--;
	}
	return tilings[i];
}

/* smallest and largest of v[k * stride + at], k in [from, to) */
double2 span_of(const double *v, uint32_t from, uint32_t to, uint32_t stride, uint32_t at)
{
	double2 span = { v[(size_t)from * stride + at], v[(size_t)from * stride + at] };
	for (uint32_t k = from + 1; k < to; k++) {
		span.x = std::min(span.x, v[(size_t)k * stride + at]);
		span.y = std::max(span.y, v[(size_t)k * stride + at]);
	}
	return span;
}

int build_region_tables(region_tables_t *t)
{
	std::vector<int32_t> poly;
	std::vector<edge_t> edges;
	std::vector<double> bounds;
	std::memset(t->set, 0, sizeof(t->set));
	const pt_t z = { kTunerMaxSize, kTunerMaxRanks };
	for (int s = 0; s < OFI_REGION_NUM_SETS; s++) {
		const int *set = ofi_region_sets[s];
		const int shape = set[1] == 8 ? 0 : (set[1] == 2 ? 1 : 2);
		pt_t ext[8];
		if (set[6] > 8) {
			return -EINVAL;
		}
		for (int e = 0; e < set[6]; e++) {
			const double *r = ofi_region_exts[set[5] + e];
			ext[e] = extend(pt_t{ r[0], r[1] }, pt_t{ r[2], r[3] }, z);
		}
		const size_t first_poly = poly.size() / 4, first_edge = edges.size();
		for (int q = 0; q < set[4]; q++) {
			const int *pd = ofi_region_polys[set[3] + q];
			if (pd[3] < 2) {
				return -EINVAL;
			}
			poly.push_back(pd[0]);
			poly.push_back(pd[1]);
			poly.push_back((int32_t)edges.size());
			poly.push_back(pd[3]);
			std::vector<pt_t> verts;
			for (int v = 0; v < pd[3]; v++) {
				const int *kind = ofi_region_vert_kind[pd[2] + v];
				const double *xy = ofi_region_vert_xy[pd[2] + v];
				pt_t pt;
				pt.x = kind[0] == 0 ? xy[0]
						    : (((kind[0] - 1) & 1) == 0 ? ext[(kind[0] - 1) / 2].x
										: ext[(kind[0] - 1) / 2].y);
				pt.y = kind[1] == 0 ? xy[1]
						    : (((kind[1] - 1) & 1) == 0 ? ext[(kind[1] - 1) / 2].x
										: ext[(kind[1] - 1) / 2].y);
				verts.push_back(to_log2(pt)); /* set_regions, :236-247 */
			}
			double b[4];
			region_bounds(verts.data(), pd[3], b);
			bounds.insert(bounds.end(), b, b + 4);
			for (int k = 0; k < pd[3]; k++) {
				const edge_t e = { verts[k == 0 ? pd[3] - 1 : k - 1], verts[k] };
				const double length = std::hypot(e.b.x - e.a.x, e.b.y - e.a.y);
				if (length != 0 && length < kMinEdge) {
					return -EINVAL; /* the certain-answer tests rely on it */
				}
				edges.push_back(e);
			}
		}
		if (edges.size() - first_edge > (size_t)kMaxSetEdges || edges.size() > 65535 || set[4] > kMaxSetEdges) {
			return -EINVAL; /* the kernels keep one edge (and one polygon) of a set per lane */
		}
		t->set[set[0]][shape][set[2]] = region_set_t{ (uint16_t)first_poly, (uint16_t)set[4], (uint16_t)first_edge,
							      (uint16_t)(edges.size() - first_edge) };
	}
	t->far_point = to_log2(pt_t{ 2.0 * kTunerMaxSize, 2.0 * kTunerMaxRanks });
	int32_t *d_poly = nullptr;
	edge_t *d_edges = nullptr;
	double *d_bounds = nullptr;
	int rc = upload(poly, &d_poly);
	if (rc == 0) {
		rc = upload(edges, &d_edges);
	}
	if (rc == 0) {
		rc = upload(bounds, &d_bounds);
	}
	if (rc != 0) {
		(void)hipFree(d_poly);
		(void)hipFree(d_edges);
		return rc;
	}
	t->poly = d_poly;
	t->edges = d_edges;
	t->bbox = d_bounds;
	return 0;
}

} // namespace

namespace ofi_amd_tuner {

double log2_coord(double v)
{
	if (v == 0) {
		v = 1e-6; /* "for 0, set to a small positive number for log2()" */
	}
	return std::log2(v);
}

/* Built once per process (about 13 KiB of device memory, never freed).  A failed build is
 * not remembered: the next caller tries again. */
int device_region_tables(region_tables_t *out)
{
	/* one copy of the tables per GPU, uploaded to whichever is current on first use there */
	constexpr int kMaxDevices = 64;
	static std::mutex lock;
	static region_tables_t tables[kMaxDevices];
	static bool built[kMaxDevices];
	int dev = -1;
	if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
		(void)hipGetLastError();
		return -ENODEV;
	}
	std::lock_guard<std::mutex> g(lock);
	if (!built[dev]) {
		const int status = build_region_tables(&tables[dev]);
		if (status != 0) {
			return status;
		}
		built[dev] = true;
	}
	*out = tables[dev];
	return 0;
}

} // namespace ofi_amd_tuner

struct ofi_amd_tuner_plan {
	grid_dims_t g;
	region_tables_t t;
	tiling_t tilings[kTilings];
	uint64_t points;
	uint64_t cells;
	void *d_axes; /* owned: what g's and the tilings' pointers point into */
	/* per-call staging (device): the variants, and the runs of the platform list */
	ofi_amd_tuner_variant_t *d_variants;
	region_run_t *d_runs;
	uint32_t variants_cap;
	uint64_t runs_cap;
	/* what they currently hold, so that an unchanged list is not uploaded again */
	std::vector<ofi_amd_tuner_variant_t> h_variants;
	std::vector<int32_t> h_platforms;
	std::vector<int32_t> h_colls;
	std::vector<uint32_t> h_ppn;
};

using namespace ofi_amd;

extern "C" {

int ofi_amd_tuner_plan_destroy(ofi_amd_tuner_plan_t *plan)
{
	if (!plan) {
		return -EINVAL;
	}
	(void)hipFree(plan->d_axes);
	(void)hipFree(plan->d_variants);
	(void)hipFree(plan->d_runs);
	delete plan;
	return 0;
}

int ofi_amd_tuner_plan_create(const int32_t *colls, uint32_t n_colls, const uint64_t *sizes,
			      uint32_t n_sizes, const uint64_t *nodes, uint32_t n_nodes,
			      const uint32_t *ppn, uint32_t n_ppn, const int32_t *algos,
			      uint32_t n_algos, ofi_amd_tuner_plan_t **out)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (!colls || !sizes || !nodes || !ppn || !algos || !out || n_colls == 0 || n_sizes == 0 ||
	    n_nodes == 0 || n_ppn == 0 || n_algos == 0) {
		return -EINVAL;
	}
	for (uint32_t i = 0; i < n_colls; i++) {
		if (colls[i] < 0 || colls[i] >= NUM_FUNCS) {
			return -EINVAL;
		}
	}
	for (uint32_t i = 0; i < n_algos; i++) {
		if (algos[i] < 0 || algos[i] >= NUM_ALGOS) {
			return -EINVAL;
		}
	}
	for (uint32_t i = 0; i < n_nodes; i++) {
		if (nodes[i] == 0 || nodes[i] > (1u << 30)) {
			return -EINVAL;
		}
	}
	for (uint32_t i = 0; i < n_ppn; i++) {
		if (ppn[i] == 0) {
			return -EINVAL;
		}
	}

	auto *plan = new (std::nothrow) ofi_amd_tuner_plan();
	/* value-initialised: every pointer and capacity starts at zero */
	if (!plan) {
		return -ENOMEM;
	}
	rc = device_region_tables(&plan->t);
	if (rc != 0) {
		delete plan;
		return rc;
	}

	/* query coordinates, through the host's libm */
	std::vector<double> log2_nodes(n_nodes), log2_sizes(n_sizes), log2_ranks((size_t)n_nodes * n_ppn);
	for (uint32_t i = 0; i < n_nodes; i++) {
		log2_nodes[i] = std::log2((double)nodes[i]);
		for (uint32_t j = 0; j < n_ppn; j++) {
			log2_ranks[(size_t)i * n_ppn + j] = log2_coord((double)(nodes[i] * ppn[j]));
		}
	}
	for (uint32_t i = 0; i < n_sizes; i++) {
		log2_sizes[i] = log2_coord((double)sizes[i]);
	}

	/* one allocation and one copy for all of it */
	grid_dims_t &g = plan->g;
	std::vector<uint8_t> axes;
	/* the tilings of the region grid and the span of coordinates of each tile */
	size_t at_spans[kTilings], at_rank_spans[kTilings];
	uint32_t shift_n[kTilings], shift_s[kTilings];
	tile_shifts(n_sizes, n_nodes, shift_n, shift_s);
	for (int i = 0; i < kTilings; i++) {
		const uint32_t per_col = 1u << shift_n[i], per_row = 1u << shift_s[i];
		tiling_t &t = plan->tilings[i];
		t = { shift_n[i], shift_s[i], (n_nodes + per_col - 1) >> shift_n[i], (n_sizes + per_row - 1) >> shift_s[i],
		      nullptr, nullptr };
		std::vector<double2> size_span(t.tiles_s), rank_span((size_t)t.tiles_n * n_ppn);
		for (uint32_t k = 0; k < t.tiles_s; k++) {
			size_span[k] = span_of(log2_sizes.data(), k * per_row, std::min(n_sizes, (k + 1) * per_row), 1, 0);
		}
		for (uint32_t k = 0; k < t.tiles_n; k++) {
			for (uint32_t j = 0; j < n_ppn; j++) {
				rank_span[(size_t)k * n_ppn + j] =
					span_of(log2_ranks.data(), k * per_col, std::min(n_nodes, (k + 1) * per_col), n_ppn, j);
			}
		}
		at_spans[i] = append(axes, size_span);
		at_rank_spans[i] = append(axes, rank_span);
	}
	const size_t at_sizes = append(axes, std::vector<uint64_t>(sizes, sizes + n_sizes));
	const size_t at_nodes = append(axes, std::vector<uint64_t>(nodes, nodes + n_nodes));
	const size_t at_log2_nodes = append(axes, log2_nodes), at_log2_sizes = append(axes, log2_sizes);
	const size_t at_log2_ranks = append(axes, log2_ranks);
	const size_t at_colls = append(axes, std::vector<int32_t>(colls, colls + n_colls));
	const size_t at_algos = append(axes, std::vector<int32_t>(algos, algos + n_algos));
	const size_t at_ppn = append(axes, std::vector<uint32_t>(ppn, ppn + n_ppn));
	uint8_t *d_axes = nullptr;
	rc = upload(axes, &d_axes);
	plan->d_axes = d_axes;
	if (rc != 0) {
		ofi_amd_tuner_plan_destroy(plan);
		return rc;
	}

	try {
		plan->h_colls.assign(colls, colls + n_colls);
		plan->h_ppn.assign(ppn, ppn + n_ppn);
	} catch (...) {
		ofi_amd_tuner_plan_destroy(plan);
		return -ENOMEM;
	}
	g.n_colls = n_colls;
	g.n_sizes = n_sizes;
	g.n_nodes = n_nodes;
	g.n_ppn = n_ppn;
	g.n_algos = n_algos;
	g.by_ppn = divisor(n_ppn);
	g.by_nodes = divisor(n_nodes);
	g.by_coll = divisor((uint32_t)std::min<uint64_t>((uint64_t)n_sizes * n_nodes * n_ppn, 1u << 31));
	g.colls = reinterpret_cast<const int32_t *>(d_axes + at_colls);
	g.sizes = reinterpret_cast<const uint64_t *>(d_axes + at_sizes);
	g.nodes = reinterpret_cast<const uint64_t *>(d_axes + at_nodes);
	g.ppn = reinterpret_cast<const uint32_t *>(d_axes + at_ppn);
	g.algos = reinterpret_cast<const int32_t *>(d_axes + at_algos);
	g.log2_nodes = reinterpret_cast<const double *>(d_axes + at_log2_nodes);
	g.log2_sizes = reinterpret_cast<const double *>(d_axes + at_log2_sizes);
	g.log2_ranks = reinterpret_cast<const double *>(d_axes + at_log2_ranks);
	for (int i = 0; i < kTilings; i++) {
		plan->tilings[i].size_span = reinterpret_cast<const double2 *>(d_axes + at_spans[i]);
		plan->tilings[i].rank_span = reinterpret_cast<const double2 *>(d_axes + at_rank_spans[i]);
	}
	plan->points = (uint64_t)n_colls * n_sizes * n_nodes * n_ppn;
	plan->cells = plan->points * n_algos * NUM_PROTOS;
	*out = plan;
	return 0;
}

uint64_t ofi_amd_tuner_plan_points(const ofi_amd_tuner_plan_t *plan)
{
	return plan ? plan->points : 0;
}

uint64_t ofi_amd_tuner_plan_cells(const ofi_amd_tuner_plan_t *plan)
{
	return plan ? plan->cells : 0;
}

int ofi_amd_tuner_model_grid(ofi_amd_tuner_plan_t *plan, const ofi_amd_tuner_variant_t *variants,
			     uint32_t n_variants, double *d_cost, int8_t *d_choice, void *stream)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (!plan || !variants || n_variants == 0) {
		return -EINVAL;
	}
	for (uint32_t i = 0; i < n_variants; i++) {
		if (variants[i].platform < 0 || variants[i].platform >= kNumPlatforms) {
			return -EINVAL;
		}
	}
	hipStream_t s = as_stream(stream);
	if (n_variants > plan->variants_cap) {
		OFI_AMD_HIP_TRY(hipStreamSynchronize(s));
		(void)hipFree(plan->d_variants);
		plan->d_variants = nullptr;
		plan->variants_cap = 0;
		plan->h_variants.clear();
		OFI_AMD_HIP_TRY(hipMalloc((void **)&plan->d_variants, sizeof(*variants) * n_variants));
		plan->variants_cap = n_variants;
	}
	/* the variants travel to the device only when they differ from the last call's */
	try {
		if (plan->h_variants.size() != n_variants ||
		    std::memcmp(plan->h_variants.data(), variants, sizeof(*variants) * n_variants) != 0) {
			plan->h_variants.clear(); /* stays empty if the upload fails: the next call uploads again */
			OFI_AMD_HIP_TRY(hipMemcpyAsync(plan->d_variants, variants, sizeof(*variants) * n_variants,
						       hipMemcpyHostToDevice, s));
			/* the source is the caller's pageable memory: wait until it has been read */
			OFI_AMD_HIP_TRY(hipStreamSynchronize(s));
			plan->h_variants.assign(variants, variants + n_variants);
		}
	} catch (...) {
		plan->h_variants.clear();
		return -ENOMEM;
	}
	if (plan->points > (1ull << 31) || plan->cells * n_variants > (1ull << 38) || n_variants > 65535) {
		return -EINVAL;
	}
	const uint32_t points = (uint32_t)plan->points;
	const size_t row = (size_t)plan->g.n_algos * NUM_PROTOS * sizeof(float); /* of the stage */
	const uint64_t bytes = d_cost ? plan->cells * n_variants * sizeof(double) : 0;
	/* modelled points: AllReduce's, of the platforms that have a model */
	uint64_t reduces = 0, with_model = 0;
	for (int32_t coll : plan->h_colls) {
		reduces += coll == FUNC_ALLREDUCE;
	}
	for (uint32_t i = 0; i < n_variants; i++) {
		with_model += platform_has_model(variants[i].platform);
	}
	const uint64_t modelled = reduces * with_model, all = plan->h_colls.size() * (uint64_t)n_variants; /* in collectives */
	const bool large = bytes > kModelLargeBytes && 2 * modelled <= all && row * kModelThreadsLarge <= kModelLds;
	const uint32_t threads = large ? kModelThreadsLarge : kModelThreads;
	const bool fewer = !large && bytes > (modelled == all ? kModelFewerBytesAll : kModelFewerBytes);
	const size_t lds = std::max(row * threads, fewer ? kModelFewerLds : 0);
	auto launch = [&](auto kernel) {
		ofi_amd::launch_kernel(kernel, dim3((points + threads - 1) / threads, n_variants), dim3(threads), d_cost ? lds : 0, s,
				       d_cost, plan->d_variants, d_choice, points, plan->g);
	};
	if (d_cost && d_choice) {
		large ? launch(model_grid_kernel<true, true, kModelThreadsLarge>) : launch(model_grid_kernel<true, true>);
	} else if (d_cost) {
		large ? launch(model_grid_kernel<true, false, kModelThreadsLarge>) : launch(model_grid_kernel<true, false>);
	} else if (d_choice) {
		launch(model_grid_kernel<false, true>);
	}
	OFI_AMD_HIP_TRY(hipGetLastError());
	return 0;
}

int ofi_amd_tuner_region_grid(ofi_amd_tuner_plan_t *plan, const int32_t *platforms,
			      uint32_t n_platforms, int8_t *d_choice, void *stream)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (!plan || !platforms || n_platforms == 0 || !d_choice || (reinterpret_cast<uintptr_t>(d_choice) & 3u) != 0) {
		return -EINVAL;
	}
	for (uint32_t i = 0; i < n_platforms; i++) {
		if (platforms[i] < 0 || platforms[i] >= kNumPlatforms) {
			return -EINVAL;
		}
	}
	if (plan->points > (1ull << 31) || n_platforms > 65535) {
		return -EINVAL;
	}
	const uint32_t points = (uint32_t)plan->points;
	const uint64_t n_runs = (uint64_t)n_platforms * plan->g.n_colls * plan->g.n_ppn;
	const tiling_t &tiling = pick_tiling(plan->tilings, n_runs);
	const uint64_t groups = (tiling_tiles(tiling) + kXcds - 1) / kXcds;
	const uint64_t blocks = groups * n_runs * kXcds;
	if (blocks == 0 || blocks > 0x7fffffffull) {
		return -EINVAL;
	}

	hipStream_t s = as_stream(stream);
	if (n_runs > plan->runs_cap) {
		OFI_AMD_HIP_TRY(hipStreamSynchronize(s));
		(void)hipFree(plan->d_runs);
		plan->d_runs = nullptr;
		plan->runs_cap = 0;
		plan->h_platforms.clear();
		OFI_AMD_HIP_TRY(hipMalloc((void **)&plan->d_runs, sizeof(region_run_t) * n_runs));
		plan->runs_cap = n_runs;
	}
	try {
		if (plan->h_platforms.size() != n_platforms ||
		    std::memcmp(plan->h_platforms.data(), platforms, sizeof(int32_t) * n_platforms) != 0) {
			plan->h_platforms.clear(); /* stays empty if an upload fails: the next call uploads again */
			std::vector<region_run_t> runs;
			runs.reserve(n_runs);
			for (uint32_t pi = 0; pi < plan->g.n_ppn; pi++) {
				for (uint32_t ci = 0; ci < plan->g.n_colls; ci++) {
					for (uint32_t e = 0; e < n_platforms; e++) {
						region_run_t run = {};
						run.entry = e;
						run.ci = ci;
						run.pi = pi;
						run.ppn = plan->h_ppn[pi];
						run.platform = platforms[e];
						const region_set_t set = region_set(plan->t, run.platform, plan->h_colls[ci], run.ppn, 1);
						run.first_poly = set.first_poly;
						run.first_edge = set.first_edge;
						run.counts = (uint32_t)set.edges << 16 | set.polys;
						runs.push_back(run);
					}
				}
			}
			std::stable_sort(runs.begin(), runs.end(),
					 [](const region_run_t &a, const region_run_t &b) { return a.counts > b.counts; });
			OFI_AMD_HIP_TRY(hipMemcpyAsync(plan->d_runs, runs.data(), sizeof(region_run_t) * runs.size(),
						       hipMemcpyHostToDevice, s));
			OFI_AMD_HIP_TRY(hipStreamSynchronize(s));
			plan->h_platforms.assign(platforms, platforms + n_platforms);
		}
	} catch (...) {
		plan->h_platforms.clear();
		return -ENOMEM;
	}
	const uint32_t waves = n_runs * tiling_tiles(tiling) > kPairedTiles ? kMostRegionWaves : 1;
	const uint32_t grid_x = (uint32_t)((groups + waves - 1) / waves * kXcds);
	for (uint64_t at = 0; at < n_runs; at += kMostRuns) {
		const uint32_t here = (uint32_t)(n_runs - at < kMostRuns ? n_runs - at : kMostRuns);
		ofi_amd::launch_kernel(region_choice_kernel, dim3(grid_x, here), dim3(64 * waves), 0, s, plan->d_runs + at,
				       plan->t.poly, plan->t.bbox, plan->t.edges, d_choice, points, plan->t.far_point, tiling, plan->g);
	}
	OFI_AMD_HIP_TRY(hipGetLastError());
	return 0;
}

} /* extern "C" */
