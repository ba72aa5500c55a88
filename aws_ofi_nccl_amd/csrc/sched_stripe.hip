/*
 * Batched rail striping (threshold scheduler) for gfx950.
 *
 * The reference schedules one message per call on a stateful object: messages
 * below max_small_msg_size take one rail from rr_small_counter, larger ones take
 * get_num_stripes(size) consecutive rails starting at rr_counter; both counters
 * advance modulo num_rails (src/nccl_ofi_scheduler.cpp:47-133).  For a batch in
 * index order that is two exclusive prefix sums:
 *
 *   small_rail_i = (rr_small + #{j < i : size_j <  max_small}) mod R
 *   start_rail_i = (rr      + sum{j < i : size_j >= max_small} n_j) mod R
 *
 * Four forms, by the size of the batch:
 *   up to kDirectBatch messages, one launch: every workgroup adds up the messages before
 *   its tile by itself, from their sizes (at most 78 KiB out of the L2);
 *   up to kOnceBatch, one launch whose workgroups publish the totals of their tiles and add up those
 *   of the tiles before them (stripe_once_kernel);
 *   up to kSmallBatch, two launches: stripe_count_kernel leaves each tile's totals of
 *   (small count, stripe count), reduced mod R (only the residues matter), and
 *   stripe_emit_kernel, whose workgroups add up the totals of the tiles before them (at most
 *   48 KiB), builds the 96-byte stripe rows in LDS and writes them out as coalesced 16-byte
 *   stores;
 *   beyond, the same two launches with larger tiles, and a level of totals above the tiles', for
 *   every kPart messages.
 * Beyond one tile a batch that is being captured into a graph takes the two launches (launch_batch says why).
 * The count launch snapshots the two counters of *state as the batch's seed, the workgroup of the
 * last tile writes the new ones back; in the one-launch form the workgroup that reads them last does.
 *
 * HBM traffic per message: 8 B read twice (once in the one-launch form) + 4 B + 96 B written.
 */
#include <algorithm>
#include <atomic>
#include <map>
#include <mutex>
#include <tuple>

#include "common.hpp"
#include "ofi_amd_hotpath.h"
#include "sched_once.hpp"

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
namespace once = ofi_amd_once;

/* One-launch form: tiles of 256 messages up to two of them, of 512 beyond, whose twice as many threads share the look
 * at everything before the tile (in us, tiles of 256 / 512 / 1024: 3000 messages 4.7 / 4.3 / 5.1, 6144 5.9 / 4.9 / 5.4).
 * The line was drawn where that look costs nearly what a second launch does: 7000 messages 5.2 against 7.6 us in two launches, 9900
 * 5.7 and 7.7, 12,000 6.2 and 7.6.  The form with published totals, 4.4 us at 9985, is the faster one from some thousands
 * on. */
constexpr uint32_t kDirectTile = 256, kDirectTileLarge = 512;
constexpr uint64_t kDirectBatch = 9984;
static_assert(4 * kDirectBatch < 65536 - 8, "packed sums of a whole batch: up to 4 stripes a message, and the seed");
/* Two-launch form: tiles of 512 messages, counted by 256 threads and written by 512 (21.5 us per 1,000,000
 * messages, 39.0 per 2,000,000; 256 threads twice 21.6 and 40.2, 128 threads four times 23.9 and 43.5). */
constexpr uint32_t kTile = 512;
constexpr uint32_t kCountThreads = 256;
constexpr uint64_t kSmallBatch = 6ull << 20;
/* Beyond: tiles of 1024 messages, a workgroup of 1024 threads each, one to a CU (its rows fill 96 KiB of
 * LDS).  Once the output is larger than the last-level cache the rate of a write-only launch depends on how
 * narrow the front is on which the chip writes: 1.5 GB in pieces of 24 KiB from six workgroups a CU
 * goes at 5.4 TB/s, in 48 KiB pieces from one workgroup a CU at 6.8.  16,000,000 messages take 276 us
 * like this, 314 with four passes of 256 messages, six workgroups a CU; 5,000,000 take 99.7 and, in
 * tiles of 512, 95.0, 7,000,000 take 130.8 and 132.6: the line lies between. */
constexpr uint32_t kBigTile = 1024;
constexpr uint32_t kBlockTiles = 4; /* tiles that share a block total: a workgroup of the count kernel */
/* ... in parts of 2^24 messages, chained through *state.  The sizes of a part, 128 MiB, are still in the
 * last-level cache when the emit launch reads them again; in one part, 60,000,000 messages took
 * 1294 us, in parts 1056. */
constexpr uint64_t kPart = 1ull << 24;
constexpr uint32_t kMaxTiles = (uint32_t)(kPart / kBigTile), kMaxBlocks = kMaxTiles / kBlockTiles;
static_assert(kSmallBatch / kTile <= kMaxTiles && kMaxBlocks <= 4 * kBigTile && kMaxTiles <= 1u << 14,
	      "room for every tile, one 16-byte load a thread, sums of residues below 2^16");
constexpr uint64_t kMaxBatch = 1ull << 28;

struct params_t {
	uint64_t max_small;
	uint64_t stripes[3];    /* 1, 2 and 3 times the minimum stripe size, at most 2^64 - 1 */
	uint64_t align;
	int32_t align_shift;    /* log2 when a power of two, else -1 */
	uint32_t num_rails;
	uint32_t stripe_counts; /* get_num_stripes for this rail count, 4 bits per requested count 1..4 */
	uint32_t mod_magic;     /* 65536 / num_rails + 1, see mod_rails */
};

/* NCCL_OFI_DIV_CEIL, include/nccl_ofi_math.h:23-26 */
__device__ __forceinline__ uint64_t div_ceil_by(uint64_t x, uint64_t d, int32_t shift)
{
	return x == 0 ? 0 : 1 + (shift >= 0 ? ((x - 1) >> shift) : ((x - 1) / d));
}

/* get_num_stripes, src/nccl_ofi_scheduler.cpp:47-64: the request, capped to the rail count,
 * goes down to the largest count >= 2 that divides the rail count and stays as it is when there
 * is none (3 rails: 2 stays 2).  At most 4 rails, so the loop is a 16-entry table, and the request --
 * the size divided by the minimum stripe, rounded up -- needs three comparisons and no division: a
 * division per message made the count kernels 15 KB of code and a third of their time. */
constexpr uint64_t kStripeCounts = 0x4221332122211111ull; /* 16 bits per rail count, 4 per request */

__device__ __forceinline__ uint32_t num_stripes(uint64_t size, const params_t &p)
{
	uint32_t n = (size > p.stripes[0]) + (size > p.stripes[1]) + (size > p.stripes[2]);
	n = n < p.num_rails ? n : p.num_rails - 1u;
	return (p.stripe_counts >> (4u * n)) & 7u;
}

/* x mod num_rails for x < 16384, by multiply and shift (checked exhaustively for 1..4 rails) */
__device__ __forceinline__ uint32_t mod_rails(uint32_t x, const params_t &p)
{
	return x - p.num_rails * ((x * p.mod_magic) >> 16);
}

__device__ __forceinline__ int32_t log2_if_pow2_dev(uint64_t v)
{
	return (v != 0 && (v & (v - 1)) == 0) ? (int32_t)(__ffsll((unsigned long long)v) - 1) : -1;
}

/* Thresholds come from the device-resident state.  False when the state is unusable (rails outside
 * 1..4, zero stripe size). */
__device__ __forceinline__ bool load_params(const ofi_amd_sched_state_t *st, uint64_t align,
					    params_t &p)
{
	p.max_small = st->max_small_msg_size;
	const uint64_t m = st->min_stripe_size;
	p.stripes[0] = m;
	p.stripes[1] = m > ~0ull / 2 ? ~0ull : 2 * m;
	p.stripes[2] = m > ~0ull / 3 ? ~0ull : 3 * m;
	p.align = align;
	p.align_shift = log2_if_pow2_dev(align);
	p.num_rails = (uint32_t)st->num_rails;
	p.stripe_counts = (uint32_t)(kStripeCounts >> (16u * ((p.num_rails - 1u) & 3u))) & 0xffffu;
	p.mod_magic = 65536u / (p.num_rails ? p.num_rails : 1u) + 1u;
	return st->num_rails >= 1 && st->num_rails <= OFI_AMD_MAX_NUM_RAILS && m != 0;
}

/* packed (small count << 16 | stripe count) contribution of one message */
__device__ __forceinline__ uint32_t contribution(uint64_t size, const params_t &p, uint32_t &n_out)
{
	const bool small = size < p.max_small;
	n_out = small ? 1u : num_stripes(size, p);
	return small ? 1u << 16 : n_out;
}

/* Inclusive sum over the 64 lanes with lane-to-lane moves inside the vector unit: shifts by 1,
 * 2, 4 and 8 lanes within each row of 16 (a lane shifted in from outside the row reads 0), then
 * lane 15 of rows 0 and 2 added to rows 1 and 3, then lane 31 added to rows 2 and 3. */
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v)
{
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false); /* row_shr:1 */
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false); /* row_shr:2 */
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false); /* row_shr:4 */
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false); /* row_shr:8 */
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false); /* row_bcast:15 */
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false); /* row_bcast:31 */
	return v;
}

/* residues mod R of a packed pair whose halves are the true sums */
__device__ __forceinline__ uint32_t residues(uint32_t packed, uint32_t num_rails)
{
	return (((packed >> 16) % num_rails) << 16) | ((packed & 0xffffu) % num_rails);
}

__device__ __forceinline__ uint32_t wave_sum_of(uint32_t v)
{
	v = wave_inclusive_scan(v);
	return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

/* The batch's seed: *state's counters as they are before the emit launch's last workgroup moves them on */
__device__ __forceinline__ uint32_t batch_seed(const ofi_amd_sched_state_t *state, uint32_t num_rails)
{
	return ((state->rr_small_counter % num_rails) << 16) | (state->rr_counter % num_rails);
}

/* Totals of one tile of kTile messages per workgroup */
__global__ __launch_bounds__(kCountThreads) void stripe_count_kernel(
	const uint64_t *__restrict__ sizes, uint32_t n, const ofi_amd_sched_state_t *__restrict__ state,
	uint64_t align, uint32_t *__restrict__ tile_totals, uint32_t *__restrict__ seed0,
	uint32_t *__restrict__ err)
{
	constexpr uint32_t kPer = kTile / kCountThreads;
	__shared__ uint32_t wave_sum[kCountThreads / 64];
	/* the tile's sizes are requested before anything waits for the state, so a workgroup pays
	 * one memory latency, not two */
	const uint32_t base = blockIdx.x * kTile;
	uint64_t size_of[kPer];
#pragma unroll
	for (uint32_t j = 0; j < kPer; j++) {
		size_of[j] = sizes[min(base + j * kCountThreads + threadIdx.x, n - 1u)];
	}
	params_t p;
	const bool usable = load_params(state, align, p);
	uint32_t acc = 0;
#pragma unroll
	for (uint32_t j = 0; j < kPer; j++) {
		uint32_t k;
		const uint32_t c = contribution(size_of[j], p, k);
		acc += base + j * kCountThreads + threadIdx.x < n ? c : 0u;
	}
	__asm__ volatile("" : "+v"(acc)); /* the sizes are not asked for behind the test of the state only */
	if (!usable) {
		if (blockIdx.x == 0 && threadIdx.x == 0) {
			atomicOr(err, ofi_amd::ASYNC_ERR_SCHED_STATE);
		}
		return;
	}
	if (blockIdx.x == 0 && threadIdx.x == 0) {
		*seed0 = batch_seed(state, p.num_rails);
	}
	acc = wave_sum_of(acc);
	if ((threadIdx.x & 63u) == 0) {
		wave_sum[threadIdx.x >> 6] = acc;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		tile_totals[blockIdx.x] = residues(wave_sum[0] + wave_sum[1] + wave_sum[2] + wave_sum[3], p.num_rails);
	}
}

/* The same for the large form: a wavefront per tile of kBigTile messages, every load of it in flight at
 * once, and the sum of the workgroup's tiles beside them. */
__global__ __launch_bounds__(64 * kBlockTiles) void stripe_count_big_kernel(
	const uint64_t *__restrict__ sizes, uint32_t n, const ofi_amd_sched_state_t *__restrict__ state,
	uint64_t align, uint32_t *__restrict__ tile_totals, uint32_t *__restrict__ block_totals,
	uint32_t *__restrict__ seed0, uint32_t *__restrict__ err)
{
	constexpr uint32_t kPer = kBigTile / 64;
	__shared__ uint32_t wave_total[kBlockTiles];
	const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const uint32_t tile = blockIdx.x * kBlockTiles + wave;
	const uint64_t base = (uint64_t)tile * kBigTile;
	uint64_t size_of[kPer];
#pragma unroll
	for (uint32_t j = 0; j < kPer; j++) {
		size_of[j] = sizes[min((uint32_t)base + j * 64u + lane, n - 1u)];
	}
	params_t p;
	const bool usable = load_params(state, align, p);
	uint32_t acc = 0;
#pragma unroll
	for (uint32_t j = 0; j < kPer; j++) {
		uint32_t k;
		const uint32_t c = contribution(size_of[j], p, k);
		acc += base + j * 64u + lane < n ? c : 0u;
	}
	__asm__ volatile("" : "+v"(acc)); /* the sizes are not asked for behind the test of the state only */
	if (!usable) {
		if (blockIdx.x == 0 && threadIdx.x == 0) {
			atomicOr(err, ofi_amd::ASYNC_ERR_SCHED_STATE);
		}
		return;
	}
	if (blockIdx.x == 0 && threadIdx.x == 0) {
		*seed0 = batch_seed(state, p.num_rails);
	}
	acc = residues(wave_sum_of(acc), p.num_rails);
	if (lane == 0) {
		wave_total[wave] = acc;
		if (base < n) {
			tile_totals[tile] = acc;
		}
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		uint32_t t = 0;
#pragma unroll
		for (uint32_t w = 0; w < kBlockTiles; w++) {
			t += wave_total[w];
		}
		block_totals[blockIdx.x] = residues(t, p.num_rails);
	}
}

/*
 * The rows of a tile, by its workgroup: this thread's message with its contribution c, its k stripes and what the messages
 * before it in the tile add up to.  BY_WAVE: `rows` has room for half of them.
 */
template <bool BY_WAVE, uint32_t THREADS>
__device__ __forceinline__ void write_rows(uint64_t size, bool live, uint32_t c, uint32_t k, uint32_t excl, uint32_t carry_small,
					   uint32_t carry_big, const params_t &p, uint32_t n, uint32_t base, u32x4 *rows,
					   uint32_t *__restrict__ num_xfers, u32x4 *__restrict__ xfers)
{
	const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, R = p.num_rails;
	/* set_schedule_by_threshold, src/nccl_ofi_scheduler.cpp:77-133 */
	const bool small = (c >> 16) != 0;
	uint32_t rail = mod_rails(small ? carry_small + (excl >> 16) : carry_big + (excl & 0xffffu), p);
	uint64_t max_stripe = size;
	if (!small) {
		/* (size - 1) / k: k is 1, 2 or 4 unless there are three rails */
		uint64_t whole = size == 0 ? 0 : (size - 1) >> (k >> 1);
		if (R == 3) {
			whole = k == 3 ? (size == 0 ? 0 : (size - 1) / 3) : whole;
		}
		const uint64_t per = size == 0 ? 0 : 1 + whole;
		max_stripe = div_ceil_by(per, p.align, p.align_shift) * p.align;
	}
	/* k stripes of max_stripe cover the message, so `left` is 0 from stripe k on and the
	 * length of an unused entry comes out as 0 by itself; lanes past the end have k = 0 */
	uint64_t left = size, offset = 0;
	uint64_t f[12]; /* 4 x {rail word, offset, msg_size} */
#pragma unroll
	for (uint32_t s = 0; s < 4; s++) {
		const bool used = s < k;
		const uint64_t stripe = left < max_stripe ? left : max_stripe;
		f[3 * s + 0] = used ? rail : 0; /* rail_id in the low 16 bits, padding zero */
		f[3 * s + 1] = used ? offset : 0;
		f[3 * s + 2] = stripe;
		offset += stripe;
		left -= stripe;
		rail = rail + 1 == R ? 0 : rail + 1;
	}
	auto stage_row = [&](u32x4 *row) {
#pragma unroll
		for (uint32_t q = 0; q < 6; q++) {
			u32x4 v;
			v.x = (uint32_t)f[2 * q];
			v.y = (uint32_t)(f[2 * q] >> 32);
			v.z = (uint32_t)f[2 * q + 1];
			v.w = (uint32_t)(f[2 * q + 1] >> 32);
			row[q] = v;
		}
	};
	if (live) {
		num_xfers[base + threadIdx.x] = k;
	}
	const uint32_t valid = (n - base) < THREADS ? (n - base) : THREADS;
	u32x4 *out = xfers + (uint64_t)base * 6;
	if (BY_WAVE) {
		/* A wavefront writes its rows by itself, the first and then the second half of its lanes', out of 3 KiB of LDS.  So
		 * four workgroups share a CU, all the wavefronts it has room for, where three did with every row in LDS, and none
		 * waits for another wavefront's rows (us, rows of a workgroup / of a wavefront / of half a one: 400,000 messages 12.7 /
		 * 12.4 / 11.4, 1,000,000 21.7 / 21.1 / 21.2, 2,000,000 39.3 / 38.5 / 37.6, 6,000,000 113.2 / 111.7 / 110.6). */
		u32x4 *const stage = &rows[wave * (32u * 6u)];
#pragma unroll
		for (uint32_t half = 0; half < 2; half++) {
			if (lane / 32u == half) {
				stage_row(&stage[lane % 32u * 6u]);
			}
			__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
			__builtin_amdgcn_wave_barrier();
#pragma unroll
			for (uint32_t q = 0; q < 3; q++) {
				const uint32_t v = q * 64u + lane, at = (wave * 64u + half * 32u) * 6u + v;
				if (at < valid * 6) {
					__builtin_nontemporal_store(stage[v], &out[at]);
				}
			}
			__builtin_amdgcn_wave_barrier(); /* the rows of one half have been read before the other's are written */
		}
	} else {
		/* The rows of the workgroup together: the small batches gain nothing by the other way, and the large ones lose
		 * the narrow front on which the chip writes (16,000,000 messages 270 and 311 us). */
		stage_row(&rows[threadIdx.x * 6]);
		__syncthreads();
		for (uint32_t v = threadIdx.x; v < valid * 6; v += THREADS) {
			__builtin_nontemporal_store(rows[v], &out[v]);
		}
	}
}

/* Where a tile's seed comes from: the sizes before it (DIRECT), the totals of the tiles before it (TILES), or
 * the totals of the blocks of tiles before its block and of the tiles before it in its block (BLOCKS) */
enum stripe_form { DIRECT, TILES, BLOCKS };

template <stripe_form FORM, uint32_t THREADS>
__global__ __launch_bounds__(THREADS) void stripe_emit_kernel(
	const uint64_t *__restrict__ sizes, uint32_t n, ofi_amd_sched_state_t *__restrict__ state,
	uint64_t align, const uint32_t *__restrict__ totals, const uint32_t *__restrict__ block_totals,
	uint32_t *__restrict__ seed0, uint32_t *__restrict__ arrival_ahead, uint32_t num_tiles,
	uint32_t *__restrict__ num_xfers, u32x4 *__restrict__ xfers, uint32_t *__restrict__ err)
{
	constexpr uint32_t kWaves = THREADS / 64;
	/* rows of 96 bytes = 6 x 16 B each, of all threads or of half a wavefront's lanes at a time */
	__shared__ u32x4 rows[FORM == TILES ? THREADS * 3 : THREADS * 6];
	__shared__ uint32_t wave_sum[kWaves], seed_sum[kWaves];
	const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
	const uint32_t tile = blockIdx.x, base = tile * THREADS, i = base + threadIdx.x;
	const bool live = i < n;
	/* Everything a tile reads is asked for before it waits for anything: its sizes, what is before it, the state and the
	 * seed.  What is beyond an end is read inside it and masked out, rather than left out by a branch. */
	const uint64_t size_read = __builtin_nontemporal_load(&sizes[min(i, n - 1u)]);
	/* DIRECT: the first messages before the tile, requested along with its own (8 at a time: 6144 messages 4.93 us,
	 * 12 or 16 at a time 4.9-5.0, 5000 4.73, 4.80 and 4.92) */
	constexpr uint32_t kAhead = THREADS == kDirectTile ? 1 : 8;
	uint64_t before[kAhead];
	auto look_ahead = [&](uint32_t i0) {
#pragma unroll
		for (uint32_t j = 0; j < kAhead; j++) {
			const uint32_t at = i0 + j * THREADS + threadIdx.x;
			before[j] = at < base ? sizes[at] : 0;
		}
	};
	/* TILES: the first words of the totals.  BLOCKS: at most kMaxBlocks words, one 16-byte load a thread, and those of the
	 * block's own tiles */
	const uint32_t blocks = tile / kBlockTiles;
	u32x4 block_words;
	uint32_t total = 0;
	if (FORM == DIRECT) {
		look_ahead(0);
	}
	if (FORM == TILES) {
		total = totals[min(threadIdx.x, tile)];
	}
	if (FORM == BLOCKS) {
		static_assert(FORM != BLOCKS || THREADS * 4 == kMaxBlocks, "a load a thread is within the block totals");
		block_words = *reinterpret_cast<const u32x4 *>(block_totals + threadIdx.x * 4u);
		total = totals[blocks * kBlockTiles + threadIdx.x % kBlockTiles];
	}
	const uint32_t seed = FORM == DIRECT ? 0u : *seed0;
	params_t p;
	const bool usable = load_params(state, align, p);
	const uint32_t R = p.num_rails;
	/* sums of residues: packed halves, below 2^14 words of at most 3 each */
	uint32_t acc = 0;
	if (FORM == TILES) {
		/* A word a thread and turn: the later a tile, the later its workgroup starts to write, and
		 * the launch is faster for it (1,000,000 messages: 21.6 us; with four 16-byte loads in
		 * flight, so that all start at once, 22.8). */
		acc = threadIdx.x < tile ? total : 0u;
		for (uint32_t t = threadIdx.x + THREADS; t < tile; t += THREADS) {
			acc += totals[t];
		}
	}
	if (FORM == BLOCKS) {
		const uint32_t at = threadIdx.x * 4u;
		acc = (at < blocks ? block_words.x : 0u) + (at + 1 < blocks ? block_words.y : 0u) + (at + 2 < blocks ? block_words.z : 0u) +
		      (at + 3 < blocks ? block_words.w : 0u) + (threadIdx.x < tile % kBlockTiles ? total : 0u);
	}
	if (FORM == DIRECT) {
		for (uint32_t i0 = 0; i0 < base;) {
#pragma unroll
			for (uint32_t j = 0; j < kAhead; j++) {
				uint32_t k;
				const uint32_t c = contribution(before[j], p, k);
				acc += i0 + j * THREADS + threadIdx.x < base ? c : 0u;
			}
			i0 += THREADS * kAhead;
			if (i0 < base) {
				look_ahead(i0);
			}
		}
	}
	const uint64_t size = live ? size_read : 0;
	/* in hand from here on: the compiler would move their loads behind the test of the state */
	__asm__ volatile("" : "+v"(acc) : "v"(size), "s"(seed));
	if (!usable) {
		if (FORM == DIRECT && tile == 0 && threadIdx.x == 0) {
			atomicOr(err, ofi_amd::ASYNC_ERR_SCHED_STATE);
		}
		return;
	}
	acc = wave_sum_of(acc);
	uint32_t k = 0;
	const uint32_t c = live ? contribution(size, p, k) : 0;
	const uint32_t inc = wave_inclusive_scan(c);
	if (lane == 0) {
		/* the one reader of the counters in a workgroup of the one-launch form: behind the barrier they have been read */
		seed_sum[wave] = acc + (FORM == DIRECT && wave == 0 ? batch_seed(state, R) : 0u);
	}
	if (lane == 63) {
		wave_sum[wave] = inc;
	}
	uint32_t before_tile = seed, off = 0, tot = 0;
	__syncthreads();
#pragma unroll
	for (uint32_t w = 0; w < kWaves; w++) {
		const uint32_t ws = wave_sum[w];
		off += (w < wave) ? ws : 0;
		tot += ws;
		before_tile += seed_sum[w];
	}
	const uint32_t carry_small = (before_tile >> 16) % R, carry_big = (before_tile & 0xffffu) % R;
	const uint32_t after_small = mod_rails(carry_small + (tot >> 16), p);
	const uint32_t after_big = mod_rails(carry_big + (tot & 0xffffu), p);
	/* Every workgroup reads the counters, so they may only be moved on when all have: each adds itself to the
	 * batch's arrival word (low half), the last tile's with the carries behind it (high half), as soon as it has
	 * read them, and whoever is last puts them in place and leaves the word at zero.  The answer is there when the
	 * rows are written (behind the rows the add took 0.25 us of the launch).
	 * A later batch's word is cleared on the way, whatever is in it (kArrivalWords). */
	uint32_t arrived = 0;
	if (FORM == DIRECT && num_tiles > 1 && threadIdx.x == 0) {
		if (tile == 0) {
			__hip_atomic_store(arrival_ahead, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		}
		const uint32_t mine = 1u + (tile == num_tiles - 1 ? (after_small << 16) | (after_big << 20) : 0u);
		arrived = mine + __hip_atomic_fetch_add(seed0, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	}
	write_rows<FORM == TILES, THREADS>(size, live, c, k, off + inc - c, carry_small, carry_big, p, n, base, rows, num_xfers, xfers);

	if (threadIdx.x != 0) {
		return;
	}
	if (FORM == DIRECT && num_tiles > 1) {
		if ((arrived & 0xffffu) == num_tiles) {
			__hip_atomic_store(seed0, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			state->rr_small_counter = (arrived >> 16) & 3u;
			state->rr_counter = (arrived >> 20) & 3u;
		}
	} else if (tile == num_tiles - 1) {
		/* the carries after the last tile are the counters the next batch starts from;
		 * nobody reads them any more in this launch (the seed was snapshotted) */
		state->rr_small_counter = after_small;
		state->rr_counter = after_big;
	}
}

/*
 * The one-launch form for batches whose sizes are too many for every tile to look through: a tile counts its own messages,
 * publishes the total in a word and adds up the words of the tiles before it, one a thread.  So it waits for other
 * workgroups.  They have been handed out before it as a rule, but on eight XCDs, of which one may be busy with another stream's
 * kernel; every wait has an end, and none is needed for the result (sched_once.hpp has the words and the rules):
 * - After `looks` looks a tile that still misses words adds up the messages before it by itself, from their sizes.
 * - The counters are moved on only when every tile has read them or finds the seed in tile 0's word.  A last tile that
 *   has given up leaves that to tile 0 if tile 0 has not published yet.  Both it and the tiles on their own go by the first
 *   copy of the word: another one may be there before it.
 * A word carries the batch's number, no other batch's on this scratch, so that nothing has to be cleared, and only ever grows.
 * Words are read past the L2s, and up to 512 workgroups ask for the same few lines at once: eight copies, of which a tile
 * reads one, are faster than one (150,000 messages 7.2 and 8.1 us, 300,000 9.2 and 10.3).
 * Us in two launches / in this one, in a row (two launches of this length are also more than some hosts queue in that time):
 *     9985 messages    6.3-6.6 / 4.4
 *    10,300            5.9-7.4 / 4.5
 *    30,000            6.0-7.2 / 4.8
 *   100,000            6.7-7.2 / 6.0
 *   150,000            7.9     / 7.0
 *   262,144            9.0     / 8.5
 * Beyond 262,144 (a word a thread) workgroups would start while others write, and the words take longer than the second
 * launch: 600,000 messages 15.1 / 17.5, 1,000,000 21.7 / 28.9 (23.2 in tiles of 1024 to 2048 messages).
 */
constexpr uint32_t kOnceTile = 512, kOnceCopies = 8;
constexpr uint64_t kOnceBatch = (uint64_t)kOnceTile * kOnceTile;
static_assert(kDirectBatch >= kOnceTile, "tile 0 and the last one are two");
constexpr uint32_t kOnceLooks = 2048; /* some 2 ms */
constexpr uint32_t kMissing = ~0u;
__device__ __forceinline__ uint64_t look(const uint64_t *word)
{
	return __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint64_t raise(uint64_t *word, uint64_t to)
{
	return __hip_atomic_fetch_max(word, to, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* published: [kOnceCopies][kOnceTile] words, and behind them the one in which tile 0 and the last tile meet */
__global__ __launch_bounds__(kOnceTile) void stripe_once_kernel(
	const uint64_t *__restrict__ sizes, uint32_t n, uint32_t num_tiles, ofi_amd_sched_state_t *__restrict__ state, uint64_t align,
	uint64_t *published, uint64_t number, uint32_t max_looks, uint32_t *__restrict__ num_xfers, u32x4 *__restrict__ xfers,
	uint32_t *__restrict__ err)
{
	constexpr uint32_t kWaves = kOnceTile / 64;
	__shared__ u32x4 rows[kOnceTile * 3];
	__shared__ uint32_t wave_sum[kWaves], seed_sum[kWaves];
	const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
	const uint32_t tile = blockIdx.x, base = tile * kOnceTile, i = base + threadIdx.x;
	const bool live = i < n;
	const uint64_t size_read = __builtin_nontemporal_load(&sizes[min(i, n - 1u)]);
	params_t p;
	const bool usable = load_params(state, align, p);
	const uint32_t small_counter = state->rr_small_counter, counter = state->rr_counter;
	const uint64_t size = live ? size_read : 0;
	__asm__ volatile("" : : "v"(size), "s"(small_counter), "s"(counter)); /* as in the emit kernel */
	if (!usable) {
		if (tile == 0 && threadIdx.x == 0) {
			atomicOr(err, ofi_amd::ASYNC_ERR_SCHED_STATE);
		}
		return;
	}
	const uint32_t R = p.num_rails, seed_read = (small_counter % R) << 16 | (counter % R);
	uint32_t k = 0;
	const uint32_t c = live ? contribution(size, p, k) : 0;
	const uint32_t inc = wave_inclusive_scan(c);
	if (lane == 63) {
		wave_sum[wave] = inc;
	}
	__syncthreads();
	uint32_t off = 0, tot = 0;
#pragma unroll
	for (uint32_t w = 0; w < kWaves; w++) {
		const uint32_t ws = wave_sum[w];
		off += (w < wave) ? ws : 0;
		tot += ws;
	}
	uint64_t before = 0;
	if (threadIdx.x < kOnceCopies) {
		before = raise(&published[threadIdx.x * kOnceTile + tile],
			       once::published_word(number, tile == 0 ? seed_read : 0u, residues(tot, R)));
	}

	const uint64_t *const words = published + tile % kOnceCopies * kOnceTile;
	uint32_t acc = tile == 0 && wave == 0 ? seed_read : 0u;
	if (wave * 64u < tile) {
		acc = kMissing;
		for (uint32_t looks = 0; looks < max_looks; looks++) {
			const uint64_t word = threadIdx.x < tile ? look(&words[threadIdx.x]) : once::published_word(number, 0, 0);
			if (__ballot(!once::is_published(word, number)) == 0) {
				acc = wave_sum_of(once::seed_and_total(word));
				break;
			}
			__builtin_amdgcn_s_sleep(1);
		}
	}
	if (lane == 0) {
		seed_sum[wave] = acc;
	}
	__syncthreads();
	uint32_t before_tile = 0;
	bool missing = false;
#pragma unroll
	for (uint32_t w = 0; w < kWaves; w++) {
		missing |= seed_sum[w] == kMissing;
		before_tile += seed_sum[w];
	}
	if (missing) { /* the same in the whole workgroup */
		const uint32_t seed = once::seed_by_itself(look(&published[0]), number, seed_read);
		uint32_t smalls = 0, stripes = 0;
		for (uint32_t at = threadIdx.x; at < base; at += kOnceTile) {
			uint32_t unused;
			const uint32_t each = contribution(sizes[at], p, unused);
			smalls += each >> 16;
			stripes += each & 0xffffu;
		}
		__syncthreads(); /* seed_sum has been read */
		acc = wave_sum_of((smalls % R) << 16 | (stripes % R));
		if (lane == 0) {
			seed_sum[wave] = acc;
		}
		__syncthreads();
		before_tile = seed;
#pragma unroll
		for (uint32_t w = 0; w < kWaves; w++) {
			before_tile += seed_sum[w];
		}
	}
	const uint32_t carry_small = (before_tile >> 16) % R, carry_big = (before_tile & 0xffffu) % R;
	write_rows<true, kOnceTile>(size, live, c, k, off + inc - c, carry_small, carry_big, p, n, base, rows, num_xfers, xfers);

	if (threadIdx.x != 0) {
		return;
	}
	uint64_t *const meet = &published[kOnceCopies * kOnceTile];
	bool stores = false;
	uint32_t counters = 0;
	if (tile == 0) {
		__asm__ volatile("" : : "v"(before) : "memory"); /* it has been answered: the word is there before the one below */
		const uint64_t found = raise(meet, once::first_tile_word(number));
		stores = once::first_tile_stores(found, number);
		counters = once::counters_left(found);
	} else if (tile == num_tiles - 1) {
		counters = mod_rails(carry_small + (tot >> 16), p) << 16 | mod_rails(carry_big + (tot & 0xffffu), p);
		stores = !missing || once::last_tile_stores(raise(meet, once::last_tile_word(number, counters)), number);
	}
	if (stores) {
		state->rr_small_counter = counters >> 16;
		state->rr_counter = counters & 0xffffu;
	}
}

/* Scratch of the batches of one stream: launches on one stream are ordered, so they can share; launches on
 * different streams may overlap and must not.  Layout in 32-bit words: the arrival words of the one-launch
 * form; the seed word of the others, on a 128-byte line of its own; then the block totals; then the
 * tile totals.
 *
 * A batch of the one-launch form takes the next arrival word round the ring, finds it at zero and leaves it at
 * zero, and clears the word half a ring ahead.  So batches that overlap on one scratch, against the rule, do not
 * count in each other's word, and a word that such a mistake (more than half a ring apart) or a launch
 * that never ran to its end has left with a count is at zero again when its turn comes: the damage
 * does not outlast the ring.  With one word for all batches a leftover count spoiled the counters of every
 * later small batch. */
constexpr uint32_t kArrivalWords = 1024;
constexpr uint32_t kSeedWord = kArrivalWords, kBlockWords = kSeedWord + 32;
constexpr uint32_t kTileWords = kBlockWords + kMaxBlocks;
constexpr uint32_t kOnceWords = kTileWords + kMaxTiles; /* words of 64 bits */
constexpr uint32_t kMeetWord = kOnceWords + 2 * kOnceCopies * kOnceTile;
constexpr uint32_t kScratchWords = kMeetWord + 32;
static_assert(kScratchWords == 29760, "116 KiB, as the header says; the graph tests leave memory of this size dirty");
constexpr uint32_t kClearThreads = 256;
static_assert((kArrivalWords & (kArrivalWords - 1)) == 0 && kBlockWords % 32 == 0 && kOnceWords % 32 == 0,
	      "a ring; block totals and published words on a line");
struct scratch_t {
	uint32_t *words = nullptr;
	std::atomic<uint32_t> turn{ 0 };    /* of the next batch that counts arrivals */
	std::atomic<uint64_t> published{ 0 }; /* batches that published totals: the last one's number */
};
/* The stream behind a handle: a created stream has its own, but the null stream's stands for another
 * stream on each GPU, and hipStreamPerThread for another one in each thread besides. */
using stream_key_t = std::tuple<void *, int, uint64_t>;
int key_of_stream(void *stream, stream_key_t *key)
{
	static std::atomic<uint64_t> threads{ 0 };
	static thread_local const uint64_t this_thread = ++threads;
	int dev = -1;
	if (stream == nullptr || stream == hipStreamLegacy || stream == hipStreamPerThread) {
		OFI_AMD_HIP_TRY(hipGetDevice(&dev));
	}
	*key = { stream, dev, stream == hipStreamPerThread ? this_thread : 0 };
	return 0;
}
std::mutex g_ws_lock;
std::map<stream_key_t, scratch_t> g_ws_by_stream;

/* The arrival words, the published ones and the one behind them; the others are written before they are read */
constexpr uint32_t kClearWords = kArrivalWords + kScratchWords - kOnceWords;
constexpr uint32_t kClearBlocks = (kClearWords + kClearThreads - 1) / kClearThreads;
__global__ __launch_bounds__(kClearThreads) void stripe_scratch_kernel(uint32_t *__restrict__ words)
{
	const uint32_t at = blockIdx.x * kClearThreads + threadIdx.x;
	if (at < kClearWords) {
		words[at < kArrivalWords ? at : kOnceWords + (at - kArrivalWords)] = 0;
	}
}

/* also where the runtime cannot say: the null stream while another one is captured */
bool being_captured(hipStream_t s)
{
	hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
	if (hipStreamIsCapturing(s, &capture) != hipSuccess) {
		(void)hipGetLastError();
		return true;
	}
	return capture != hipStreamCaptureStatusNone;
}

/* Scratch for stream s with its arrival words at zero before anything queued on s from here on.  A stream that is
 * being captured would only record the clearing launch, and batches called before the first replay would count
 * from whatever the memory held: there it runs on a stream of its own and is waited for. */
int new_scratch(hipStream_t s, uint32_t **out)
{
	uint32_t *words = nullptr;
	OFI_AMD_HIP_TRY(hipMalloc((void **)&words, sizeof(uint32_t) * kScratchWords));
	hipError_t e = hipSuccess;
	if (!being_captured(s)) {
		ofi_amd::launch_kernel(stripe_scratch_kernel, dim3(kClearBlocks), dim3(kClearThreads), 0, s, words);
		e = hipGetLastError();
	} else {
		hipStream_t own = nullptr;
		e = hipStreamCreateWithFlags(&own, hipStreamNonBlocking);
		if (e == hipSuccess) {
			ofi_amd::launch_kernel(stripe_scratch_kernel, dim3(kClearBlocks), dim3(kClearThreads), 0, own,
					       words);
			e = hipGetLastError();
			const hipError_t waited = hipStreamSynchronize(own);
			e = e == hipSuccess ? waited : e;
			(void)hipStreamDestroy(own);
		}
	}
	if (e != hipSuccess) {
		(void)hipGetLastError();
		(void)hipFree(words);
		return ofi_amd::errno_of(e);
	}
	*out = words;
	return 0;
}

/*
 * The same scratch for callers that may not allocate: one array per GPU, part of the loaded
 * code object (which starts at zero), held until the process ends.  In host code the
 * array's name is only a handle for hipGetSymbolAddress; kernels get the address it returns.
 */
constexpr uint64_t kNoAllocMaxBatch = 1ull << 26; /* what the entry point promises; the scratch would do for any batch */
static __device__ __align__(256) __attribute__((used)) uint32_t scratch[kScratchWords];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_lock;
scratch_t g_scratch[kMaxDevices]; /* words: device address of `scratch` on each GPU, once looked up */

/* The current GPU's copy of `scratch` as ofi_amd_gpu_init() has recorded it; no runtime call that
 * could allocate.  -ENXIO when its address has not been looked up. */
int cached_scratch_of_current_device(scratch_t **out)
{
	int dev = -1;
	OFI_AMD_HIP_TRY(hipGetDevice(&dev));
	if (dev < 0 || dev >= kMaxDevices) {
		return -ENODEV;
	}
	std::lock_guard<std::mutex> g(g_scratch_lock);
	if (!g_scratch[dev].words) {
		return -ENXIO;
	}
	*out = &g_scratch[dev];
	return 0;
}

/* Device address of the current GPU's copy of `scratch` (each GPU has its own), looked up on
 * first use: set-up only. */
int look_up_scratch_of_current_device()
{
	int dev = -1;
	OFI_AMD_HIP_TRY(hipGetDevice(&dev));
	if (dev < 0 || dev >= kMaxDevices) {
		return -ENODEV;
	}
	std::lock_guard<std::mutex> g(g_scratch_lock);
	if (!g_scratch[dev].words) {
		void *p = nullptr;
		OFI_AMD_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
		if (!p) {
			return -EIO;
		}
		g_scratch[dev].words = static_cast<uint32_t *>(p);
	}
	return 0;
}

uint32_t tiles_of(uint64_t n, uint32_t tile)
{
	return (uint32_t)((n + tile - 1) / tile);
}

/* A batch that is being captured goes the two-launch way from its second tile on, all of whose scratch is
 * written before it is read: a replay would come back to the arrival word or the batch number it was captured with, and its
 * stream's other batches may meanwhile be anywhere round the ring. */
void launch_batch(hipStream_t s, const uint64_t *d_sizes, uint64_t total, ofi_amd_sched_state_t *d_state, uint64_t align,
		  scratch_t &scratch, uint32_t *d_num_xfers, u32x4 *d_xfers, uint32_t *err, uint32_t looks = kOnceLooks)
{
	uint32_t *words = scratch.words;
	uint32_t *seed0 = words + kSeedWord, *blocks = words + kBlockWords, *totals = words + kTileWords;
	if (total <= kDirectTile || (total <= kDirectBatch && !being_captured(s))) {
		const bool large = total > 2 * kDirectTile;
		const uint32_t n = (uint32_t)total, tiles = tiles_of(n, large ? kDirectTileLarge : kDirectTile);
		const uint32_t turn = tiles > 1 ? scratch.turn.fetch_add(1, std::memory_order_relaxed) : 0u;
		auto launch = [&](auto kernel, uint32_t threads) {
			ofi_amd::launch_kernel(kernel, dim3(tiles), dim3(threads), 0, s, d_sizes, n, d_state, align, nullptr, nullptr,
					       words + turn % kArrivalWords, words + (turn + kArrivalWords / 2) % kArrivalWords, tiles,
					       d_num_xfers, d_xfers, err);
		};
		if (large) {
			launch(stripe_emit_kernel<DIRECT, kDirectTileLarge>, kDirectTileLarge);
		} else {
			launch(stripe_emit_kernel<DIRECT, kDirectTile>, kDirectTile);
		}
		return;
	}
	if (total > kDirectBatch && total <= kOnceBatch && !being_captured(s)) {
		const uint32_t n = (uint32_t)total, tiles = tiles_of(n, kOnceTile);
		const uint64_t number = scratch.published.fetch_add(1, std::memory_order_relaxed) + 1;
		ofi_amd::launch_kernel(stripe_once_kernel, dim3(tiles), dim3(kOnceTile), 0, s, d_sizes, n, tiles, d_state, align,
				       reinterpret_cast<uint64_t *>(words + kOnceWords), number, looks, d_num_xfers, d_xfers, err);
		return;
	}
	if (total <= kSmallBatch) {
		const uint32_t n = (uint32_t)total, tiles = tiles_of(n, kTile);
		ofi_amd::launch_kernel(stripe_count_kernel, dim3(tiles), dim3(kCountThreads), 0, s, d_sizes, n, d_state, align, totals,
				       seed0, err);
		ofi_amd::launch_kernel((stripe_emit_kernel<TILES, kTile>), dim3(tiles), dim3(kTile), 0, s, d_sizes, n, d_state, align,
				       totals, nullptr, seed0, nullptr, tiles, d_num_xfers, d_xfers, err);
		return;
	}
	for (uint64_t at = 0; at < total; at += kPart) {
		const uint32_t n = (uint32_t)(total - at < kPart ? total - at : kPart), tiles = tiles_of(n, kBigTile);
		ofi_amd::launch_kernel(stripe_count_big_kernel, dim3(tiles_of(tiles, kBlockTiles)), dim3(64 * kBlockTiles), 0, s,
				       d_sizes + at, n, d_state, align, totals, blocks, seed0, err);
		ofi_amd::launch_kernel((stripe_emit_kernel<BLOCKS, kBigTile>), dim3(tiles), dim3(kBigTile), 0, s, d_sizes + at, n,
				       d_state, align, totals, blocks, seed0, nullptr, tiles, d_num_xfers + at, d_xfers + 6 * at, err);
	}
}

/* A batch on a stream's scratch; looks: at most so many does a tile take at the words of the others. */
int batch_on_stream(ofi_amd_sched_state_t *d_state, const uint64_t *d_sizes, uint64_t n, uint64_t align, uint32_t *d_num_xfers,
		    ofi_amd_xfer_info_t *d_xfers, void *stream, uint32_t looks)
{
	int rc = ofi_amd::require_device();
	if (rc != 0) {
		return rc;
	}
	if (!d_state || align == 0 || n > kMaxBatch) {
		return -EINVAL;
	}
	if (n == 0) {
		return 0;
	}
	if (!d_sizes || !d_num_xfers || !d_xfers) {
		return -EINVAL;
	}

	uint32_t *err = ofi_amd::async_error_word();
	if (!err) {
		return -ENOMEM;
	}

	hipStream_t s = ofi_amd::as_stream(stream);
	stream_key_t key;
	rc = key_of_stream(stream, &key);
	if (rc != 0) {
		return rc;
	}
	try {
		/* held until the launches are queued: two threads submitting to one stream share its
		 * scratch, and their count/emit pairs must not interleave */
		std::lock_guard<std::mutex> g(g_ws_lock);
		scratch_t &scratch = g_ws_by_stream[key];
		if (!scratch.words) {
			rc = new_scratch(s, &scratch.words);
			if (rc != 0) {
				return rc;
			}
		}
		launch_batch(s, d_sizes, n, d_state, align, scratch, d_num_xfers, reinterpret_cast<u32x4 *>(d_xfers), err, looks);
	} catch (...) {
		return -ENOMEM;
	}
	OFI_AMD_HIP_TRY(hipGetLastError());
	return 0;
}

} // namespace

namespace ofi_amd {

int sched_noalloc_setup()
{
	int count = 0, before = -1;
	OFI_AMD_HIP_TRY(hipGetDeviceCount(&count));
	OFI_AMD_HIP_TRY(hipGetDevice(&before));
	int rc = 0;
	for (int dev = 0; dev < count && dev < kMaxDevices && rc == 0; dev++) {
		if (hipSetDevice(dev) != hipSuccess) {
			rc = -ENODEV;
			break;
		}
		rc = look_up_scratch_of_current_device();
	}
	(void)hipSetDevice(before);
	return rc;
}

} // namespace ofi_amd

using namespace ofi_amd;

extern "C" {

int ofi_amd_sched_batch(ofi_amd_sched_state_t *d_state, const uint64_t *d_sizes, uint64_t n,
			uint64_t align, uint32_t *d_num_xfers, ofi_amd_xfer_info_t *d_xfers,
			void *stream)
{
	return batch_on_stream(d_state, d_sizes, n, align, d_num_xfers, d_xfers, stream, kOnceLooks);
}

int ofi_amd_sched_batch_looks(ofi_amd_sched_state_t *d_state, const uint64_t *d_sizes, uint64_t n,
			      uint64_t align, uint32_t *d_num_xfers, ofi_amd_xfer_info_t *d_xfers,
			      void *stream, uint32_t looks)
{
	return batch_on_stream(d_state, d_sizes, n, align, d_num_xfers, d_xfers, stream, std::min(looks, kOnceLooks));
}

int ofi_amd_sched_stream_release(void *stream)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	stream_key_t key;
	rc = key_of_stream(stream, &key);
	if (rc != 0) {
		return rc;
	}
	uint32_t *words = nullptr;
	{
		std::lock_guard<std::mutex> g(g_ws_lock);
		auto it = g_ws_by_stream.find(key);
		if (it == g_ws_by_stream.end()) {
			return 0; /* nothing was ever allocated for it */
		}
		words = it->second.words;
		g_ws_by_stream.erase(it);
	}
	/* launches queued on the stream may still read the scratch */
	OFI_AMD_HIP_TRY(hipStreamSynchronize(as_stream(stream)));
	(void)hipFree(words);
	return 0;
}

int ofi_amd_sched_batch_noalloc(ofi_amd_sched_state_t *d_state, const uint64_t *d_sizes, uint64_t n,
				uint64_t align, uint32_t *d_num_xfers, ofi_amd_xfer_info_t *d_xfers,
				void *stream)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (!d_state || align == 0) {
		return -EINVAL;
	}
	if (n > kNoAllocMaxBatch) {
		return -E2BIG;
	}
	if (n == 0) {
		return 0;
	}
	if (!d_sizes || !d_num_xfers || !d_xfers) {
		return -EINVAL;
	}
	uint32_t *err = async_error_word_if_ready();
	if (!err) {
		return -ENXIO; /* ofi_amd_gpu_init() allocates it; this call must not */
	}
	scratch_t *scratch = nullptr;
	/* -ENXIO: ofi_amd_gpu_init() looks the address up; this call must not */
	rc = cached_scratch_of_current_device(&scratch);
	if (rc != 0) {
		return rc;
	}
	launch_batch(as_stream(stream), d_sizes, n, d_state, align, *scratch, d_num_xfers,
		     reinterpret_cast<u32x4 *>(d_xfers), err);
	OFI_AMD_HIP_TRY(hipGetLastError());
	return 0;
}

} /* extern "C" */
