/*
 * Batched bounce / eager copy and read-back flush for gfx950.
 *
 * The reference copies every eager payload with its own loop-back fi_read from
 * the bounce buffer into the receive buffer
 * (rdma_eager_copy_req::post, src/nccl_ofi_rdma.cpp:2729-2776) and forces
 * visibility with a small read-back (rdma_flush_req::post, :2664-2713).  Here
 * one launch moves a whole batch.
 *
 * Work mapping: one 64-lane wavefront per buffer.  Destinations are 64-byte
 * aligned, so every lane stores whole 16-byte words.  A wavefront covers up to
 * 8 KiB (the eager limit) per trip as rows of 1 KiB: all loads of a trip are
 * issued before its first store, so the whole buffer is in flight at once
 * whatever its length.  The table entry of the buffer is wave-uniform and is
 * read through the scalar cache.
 *
 * Every trip is straight-line code.  The number of rows a buffer needs is
 * wave-uniform, so the body is picked by a scalar switch over 1..8 rows, the
 * lanes past the end of the (possibly partial) last row are clamped to the last
 * valid word instead of being predicated: they copy that word again, the same
 * bytes to the same place, and likewise for the sub-16-byte tail.
 * Loads and stores share one in-order counter (vmcnt) on this ISA; with
 * per-load predication the compiler cannot count across the branches and falls
 * back to waiting for *everything* before each store, which serialises the
 * stores of a wave (measured: 5.2 TB/s against 7.1 TB/s for the same traffic).
 *
 * The packed source can start at any byte.  16-byte loads from a 4-byte-aligned
 * address run at full rate on gfx950, loads from an odd byte address do not
 * (measured: about 15 % slower), so a source that is not 4-byte aligned is read
 * as aligned dwords -- four plus the one that follows -- and each output dword
 * is cut out of two neighbours with v_alignbyte_b32.  The fifth dword is the
 * next lane's first, so it travels between lanes (one wave-wide DPP shift per
 * row; lane 63 takes lane 0 of the next row) rather than through a second load
 * instruction over the same cache lines; only the last row of a trip, whose
 * lanes may be clamped, loads it (94.4 -> 91.8 us on the configured batch: the
 * texture-address unit is busy 74 % of the kernel's time).  That dword always
 * contains at least one byte of the buffer, so nothing beyond the dword that
 * holds the last source byte is read.  The rows cover whole 64-byte units of the
 * destination; what is left of the buffer (up to 63 bytes) goes out as single
 * bytes, one per lane, so that nothing outside [dst, dst+len) is written and the
 * last, partial unit is written by one instruction.
 *
 * Flush: behind its stores (they are write-through to the L2 of the XCD) the wave,
 * or one of its workgroup for all of them, re-reads the first 4 bytes
 * of the destination through that L2 and writes them to d_flush[i].  No wider
 * fence is used: on a multi-XCD part a device-scope release per buffer would
 * write back the whole L2 each time; device-wide visibility of the copied
 * bytes comes with the end of the kernel, as for any other kernel output.
 */
#include <cstring>
#include <new>

#include <immintrin.h>
#include <sys/mman.h>
#include <unistd.h>

#include "common.hpp"
#include "ofi_amd_hotpath.h"

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
/* 16 bytes at a 4-byte-aligned address */
struct __attribute__((packed, aligned(4))) dword_aligned_u32x4 {
	u32x4 v;
};

/* Buffers (= wavefronts) per workgroup and consecutive ones that share an XCD, swept over
 * thousands of launches in a row on 65,536 buffers.  Bounce copy: 8 wavefronts per workgroup with
 * runs of 32 buffers per XCD was the fastest (91.1 us per launch, every wavefront reading its own
 * word back; 4 wavefronts: 91.8, 2: 92.5, 16: 92.6; runs of 64 buffers 91.7).  The eager copy, whose sources are rx buffers in
 * arrival order, prefers single-wavefront workgroups while every wavefront reads its own bytes back (runs of 32: 97.8 us, 4
 * wavefronts 98.4, 8: 101.6, 16: 108.6), four where a workgroup reads them back together (eager_copy_kernel), and the table copy
 * single ones (1: 419.9 us per GiB, 4: 439.5, 8: 430.3). */
constexpr int kBounceWaves = 8;
constexpr uint32_t kBounceRun = 32;
constexpr int kEagerWaves = 4; /* of TOGETHER */
constexpr int kTableWaves = 1;
constexpr uint32_t kXcds = 8;
constexpr uint32_t kRows = 8;              /* rows of 64 x 16 bytes per trip: 8 KiB per wave */
constexpr uint32_t kTripVec = kRows * 64u; /* 16-byte words per trip */

__device__ __forceinline__ u32x4 load16_dword_aligned(const uint8_t *p)
{
	return reinterpret_cast<const dword_aligned_u32x4 *>(p)->v;
}

/*
 * Every access to a destination carries the same cache policy, the streaming one, but for the first rows of batches
 * that fit the L2s (kKeepBytes): the 16-byte stores of the rows, the single head and tail bytes and the
 * read-back of the flush.  With the rows streaming and the tail bytes and the read-back as ordinary
 * accesses, the same batch launched over and over on the same buffers slowed down by 6 % within 2,000 launches (91 ->
 * 97 us; fewer and fewer of those ordinary lines leave the L2 between launches, and a read
 * sweep of 16 MiB of other memory brought the first rate back); with one policy the rate does
 * not move (91 us from the first launch to the 20,000th; 84.7 since workgroups read their words back together).
 */
__device__ __forceinline__ void store_byte_streaming(uint8_t *p, uint8_t v)
{
	__builtin_nontemporal_store(v, p);
}

/*
 * One trip: R rows from s (4-byte aligned; the data starts `shift` bytes in) to d (16-byte
 * aligned).  nvec = 16-byte words left, 64*(R-1) < nvec <= 64*R unless FULL, where all R rows
 * are complete.  SHIFTED = false: shift is 0 and the source words are used as they are.  KEEP: the
 * first row is stored by ordinary stores, for the read-back that follows (kKeepBytes).
 */
template <int R, bool SHIFTED, bool FULL, bool KEEP>
__device__ __forceinline__ void copy_rows(const uint8_t *__restrict__ s, uint8_t *__restrict__ d,
					  uint32_t nvec, uint32_t shift, uint32_t lane)
{
	u32x4 v[R];
	uint32_t x[R];
#pragma unroll
	for (int k = 0; k < R; k++) {
		uint32_t j = (uint32_t)k * 64u + lane;
		if (!FULL && k == R - 1) {
			j = min(j, nvec - 1u); /* lanes past the end re-read the last word */
		}
		const uint8_t *p = s + ((uint64_t)j << 4);
		v[k] = load16_dword_aligned(p);
		if (SHIFTED && k == R - 1) {
			x[k] = *reinterpret_cast<const uint32_t *>(p + 16);
		}
	}
	if (SHIFTED) {
		/* The dword that follows a lane's 16 bytes is the first dword of the next lane's: it
		 * comes over from the neighbour (one wave-wide DPP shift; lane 63 takes lane 0 of the
		 * next row) instead of through a second load instruction over the same cache lines.
		 * Only the last row, whose lanes may be clamped, loads it. */
#pragma unroll
		for (int k = 0; k < R - 1; k++) {
			const uint32_t from_next = (uint32_t)__builtin_amdgcn_update_dpp(
				0, (int)v[k].x, 0x130 /* wave_shl:1 */, 0xf, 0xf, false);
			const uint32_t wrap = (uint32_t)__builtin_amdgcn_readfirstlane((int)v[k + 1].x);
			x[k] = lane == 63u ? wrap : from_next;
		}
	}
#pragma unroll
	for (int k = 0; k < R; k++) {
		uint32_t j = (uint32_t)k * 64u + lane;
		if (!FULL && k == R - 1) {
			j = min(j, nvec - 1u); /* ... and re-write it: same bytes, same place */
		}
		u32x4 o = v[k];
		if (SHIFTED) {
			o.x = __builtin_amdgcn_alignbyte(v[k].y, v[k].x, shift);
			o.y = __builtin_amdgcn_alignbyte(v[k].z, v[k].y, shift);
			o.z = __builtin_amdgcn_alignbyte(v[k].w, v[k].z, shift);
			o.w = __builtin_amdgcn_alignbyte(x[k], v[k].w, shift);
		}
		u32x4 *to = reinterpret_cast<u32x4 *>(d + ((uint64_t)j << 4));
		if (KEEP && k == 0) {
			*to = o;
		} else {
			__builtin_nontemporal_store(o, to);
		}
	}
}

template <bool SHIFTED, bool KEEP>
__device__ __forceinline__ void copy_words(const uint8_t *__restrict__ s, uint8_t *__restrict__ d,
					   uint32_t nvec, uint32_t shift, uint32_t lane)
{
	auto part = [&](uint32_t n) { /* at most a trip */
		switch ((n + 63u) >> 6) { /* wave-uniform */
		case 1: copy_rows<1, SHIFTED, false, KEEP>(s, d, n, shift, lane); break;
		case 2: copy_rows<2, SHIFTED, false, KEEP>(s, d, n, shift, lane); break;
		case 3: copy_rows<3, SHIFTED, false, KEEP>(s, d, n, shift, lane); break;
		case 4: copy_rows<4, SHIFTED, false, KEEP>(s, d, n, shift, lane); break;
		case 5: copy_rows<5, SHIFTED, false, KEEP>(s, d, n, shift, lane); break;
		case 6: copy_rows<6, SHIFTED, false, KEEP>(s, d, n, shift, lane); break;
		case 7: copy_rows<7, SHIFTED, false, KEEP>(s, d, n, shift, lane); break;
		case 8: copy_rows<8, SHIFTED, false, KEEP>(s, d, n, shift, lane); break;
		default: break; /* n == 0 */
		}
	};
	auto whole = [&] {
		copy_rows<kRows, SHIFTED, true, false>(s, d, kTripVec, shift, lane);
		s += (uint64_t)kTripVec << 4;
		d += (uint64_t)kTripVec << 4;
		nvec -= kTripVec;
	};
	if constexpr (KEEP) {
		/* the trip that is less than whole is the first, so that one row of a buffer is kept however long it
		 * is (12,000 eager buffers of up to 16 KiB with a row of every trip kept 50.4 us, streamed 43.5) */
		const uint32_t n = nvec != 0 ? (nvec - 1u) % kTripVec + 1u : 0u;
		part(n);
		s += (uint64_t)n << 4;
		d += (uint64_t)n << 4;
		nvec -= n;
		while (nvec != 0) {
			whole();
		}
	} else {
		while (nvec > kTripVec) { /* buffers beyond 8 KiB: whole trips first */
			whole();
		}
		part(nvec);
	}
}

/* bytes, at least one, from s to a 64-byte-aligned d; KEEP: the line at d is left to ordinary stores */
template <bool KEEP>
__device__ __forceinline__ void copy_to_aligned(const uint8_t *__restrict__ s, uint8_t *__restrict__ d, uint32_t bytes,
						uint32_t lane)
{
	/* whole 64-byte units as 16-byte words, the rest (up to 63 bytes) singly, one per
	 * lane: the last, partial unit of memory is then written by one instruction rather
	 * than by the end of a row and by the tail.  Tail bytes first, so their latency
	 * overlaps the body; unpredicated (lanes without a tail byte re-copy the buffer's
	 * last byte) to stay branch-free */
	const uint32_t nvec = (bytes >> 6) << 2;
	const uint32_t tail_at = min((nvec << 4) + lane, bytes - 1u);
	const uint8_t tail_byte = s[tail_at];

	const uint32_t shift = (uint32_t)(reinterpret_cast<uintptr_t>(s) & 3u);
	if (shift == 0) {
		copy_words<false, KEEP>(s, d, nvec, 0, lane);
	} else {
		copy_words<true, KEEP>(s - shift, d, nvec, shift, lane);
	}
	if (KEEP && nvec == 0) { /* no row: the tail's line is the one read back */
		d[tail_at] = tail_byte;
	} else {
		store_byte_streaming(d + tail_at, tail_byte);
	}
}

/* The flush words: no output for them, each buffer's read back by its own wavefront (kept rows), or a workgroup's
 * together (streamed ones, or kept ones). */
enum read_back_t { NO_READ_BACK, BY_ITSELF, TOGETHER, KEPT_TOGETHER };
constexpr bool keeps_rows(read_back_t back)
{
	return back == BY_ITSELF || back == KEPT_TOGETHER;
}
constexpr bool by_workgroup(read_back_t back)
{
	return back == TOGETHER || back == KEPT_TOGETHER;
}

/*
 * TOGETHER: one wavefront reads the words of its workgroup's eight buffers back, in one instruction, behind a barrier,
 * and the other seven are done: a read of a line that has just been streamed takes longer than the copy of a short
 * buffer.  Each by itself and together, on other buffers at every launch / on the same ones over and over, us:
 *   65,536 of up to 8 KiB                116.4 / 88.0  117.0 / 83.1
 *   20,000 of up to 4 KiB                 17.0 / 16.5   16.1 / 15.6
 *   65,536 of up to 1000 B out of a pool  25.7 / 25.4   24.3 / 24.0
 *   65,536 of up to 60 B out of a pool    18.8 / 15.5   19.2 / 16.3
 *   1,000,000 of up to 60 B out of a pool 222 / 219     229 / 221
 * (Counting the wavefronts in an LDS word, for the last one to read back without a barrier, needs a barrier in front of
 * the copies all the same: no faster for long buffers, the last two lines 20.3 / 17.6 and 232 / 229.)
 * KEPT_TOGETHER: the words are found in the L2, but eight of them still leave in one write, to host memory as a rule.  Each by
 * itself and together, rows kept, other buffers at every launch / the same ones, us:
 *   7000 of up to 8 KiB, packed           15.9 / 10.3   16.0 / 10.4   (4000: 11.0 / 6.2  11.2 / 6.4)
 *   8100 of up to 8 KiB, packed           18.1 / 11.4   18.3 / 11.5   (of up to 100 and 1000 B alike)
 *   10,000 of up to 6600 B                18.5 / 11.9   18.6 / 11.9
 *   12,000 of up to 5500 B                19.2 / 12.1   18.7 / 12.1   (kKeepByItself lies between)
 *   16,000 of up to 4 KiB                 18.8 / 12.0   18.5 / 11.8
 *   32,000 of up to 2000 B                22.0 / 13.8   19.9 / 13.1
 *   65,536 of up to 1000 B                28.9 / 18.1   27.7 / 17.9
 *   200,000 of up to 100 B                47.3 / 46.7   44.7 / 44.2
 *   450,000 of up to 60 B                 95.7 / 82.2   91.3 / 80.0
 * NO_READ_BACK is a kernel of its own because one that claims LDS starts later: 65,536 of up to 60 B 11.2 us with
 * the claim, 9.8 without.
 */
template <read_back_t BACK>
__global__ __launch_bounds__(64 * kBounceWaves) void bounce_scatter_kernel(
	const uint8_t *__restrict__ src, uint64_t src_bytes, const uint64_t *__restrict__ src_off,
	const uint64_t *__restrict__ dst_off, const uint32_t *__restrict__ len, uint32_t n, uint8_t *__restrict__ arena,
	uint64_t arena_bytes, uint32_t *__restrict__ flush, uint32_t *__restrict__ err)
{
	constexpr uint32_t kGroup = kBounceRun / kBounceWaves;
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	/* Workgroups are dealt round-robin to the 8 XCDs, each with its own L2.  Runs of kBounceRun
	 * consecutive buffers go to one XCD, so that neighbouring buffers
	 * -- which share a cache line of the packed source at their boundary -- mostly meet in
	 * the same L2, while every XCD still sees an even sample of the whole batch whatever
	 * order the lengths come in. */
	const uint32_t xcd = blockIdx.x % kXcds;
	const uint32_t turn = blockIdx.x / kXcds;
	const uint32_t wg = ((turn / kGroup) * kXcds + xcd) * kGroup + turn % kGroup;
	const uint32_t first = wg * kBounceWaves, buf = first + wave;
	if (!by_workgroup(BACK) && buf >= n) {
		return;
	}

	uint8_t *d = nullptr; /* until there is something to read back */
	if (!by_workgroup(BACK) || buf < n) { /* all of a workgroup come to the barrier */
		const uint64_t doff = dst_off[buf];
		const uint32_t bytes = len[buf];
		const uint64_t soff = src_off[buf];
		/* precondition check: skip (and report) instead of reading or writing out of range; the
		 * read-back takes four bytes at the destination whatever the length */
		const uint64_t need = (BACK != NO_READ_BACK && bytes < 4u) ? 4u : bytes;
		if ((doff & 63u) != 0 || doff > arena_bytes || need > arena_bytes - doff || soff > src_bytes ||
		    bytes > src_bytes - soff) {
			if (lane == 0) {
				atomicOr(err, ofi_amd::ASYNC_ERR_BOUNCE_RANGE);
			}
			if (!by_workgroup(BACK)) {
				return;
			}
		} else {
			const uint8_t *s = src + soff;
			d = arena + doff;
			if (bytes != 0) {
				copy_to_aligned<keeps_rows(BACK)>(s, d, bytes, lane);
			}
		}
	}

	if constexpr (by_workgroup(BACK)) {
		__shared__ uint8_t *back[kBounceWaves]; /* nullptr: none */
		if (lane == 0) {
			back[wave] = d;
		}
		__syncthreads(); /* the copies, too, are in front of it */
		if (threadIdx.x < kBounceWaves && back[lane] != nullptr) {
			const uint32_t *word = reinterpret_cast<const uint32_t *>(back[lane]);
			flush[first + lane] = BACK == TOGETHER ? __builtin_nontemporal_load(word) : *word;
		}
	} else if constexpr (BACK == BY_ITSELF) {
		__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
		if (lane == 0) {
			flush[buf] = *reinterpret_cast<const uint32_t *>(d);
		}
	}
}

/*
 * bytes from s to d, neither aligned: the bytes in front of the first 64-byte boundary of the
 * destination go out singly, one per lane; from there on it is the aligned-destination copy
 * above, with whatever source alignment that leaves.  Stopping at the first 16-byte boundary
 * would do for the 16-byte stores, but then every 1 KiB row of a trip begins and ends inside a
 * 64-byte unit of memory that the neighbouring row completes with a second, partial write
 * (measured on 65,536 buffers: 99.7 us with rows on 16-byte boundaries, 95.7 us on 64- or
 * 128-byte ones).  Wave-collective.
 */
template <bool KEEP = false>
__device__ __forceinline__ void copy_any(const uint8_t *__restrict__ s, uint8_t *__restrict__ d,
					 uint32_t bytes, uint32_t lane)
{
	if (bytes == 0) {
		return;
	}
	const uint32_t head = min(bytes, (64u - (uint32_t)(reinterpret_cast<uintptr_t>(d) & 63u)) & 63u);
	/* lanes without a head byte re-copy byte 0: same value, same place */
	const uint32_t head_at = min(lane, max(head, 1u) - 1u);
	const uint8_t head_byte = s[head_at];
	const uint32_t rem = bytes - head;
	if (rem != 0) {
		const uint8_t *s2 = s + head;
		uint8_t *d2 = d + head;
		const uint32_t nvec = (rem >> 6) << 2; /* as in the bounce copy */
		const uint32_t tail_at = min((nvec << 4) + lane, rem - 1u);
		const uint8_t tail_byte = s2[tail_at];
		const uint32_t shift = (uint32_t)(reinterpret_cast<uintptr_t>(s2) & 3u);
		if (shift == 0) {
			copy_words<false, KEEP>(s2, d2, nvec, 0, lane);
		} else {
			copy_words<true, KEEP>(s2 - shift, d2, nvec, shift, lane);
		}
		store_byte_streaming(d2 + tail_at, tail_byte);
	}
	if (KEEP) {
		d[head_at] = head_byte;
	} else {
		store_byte_streaming(d + head_at, head_byte);
	}
}

/* The first min(4, bytes) destination bytes, little-endian: a quad of lanes reads one byte
 * each in one instruction (the destination has no alignment to read a word from),
 * then the four are combined inside the quad. */
__device__ __forceinline__ uint32_t quad_word(uint32_t byte, uint32_t at)
{
	uint32_t word = byte << (8u * at);
	word |= __shfl_xor(word, 1, 64);
	word |= __shfl_xor(word, 2, 64);
	return word;
}

/*
 * The same copy for eager arrivals as they sit in rx buffers: an 8-byte header, then the
 * payload, which goes to a receive buffer at any alignment, truncated to that buffer's
 * length (rdma_eager_copy_req::post, src/nccl_ofi_rdma.cpp:2729-2776).
 *
 * TOGETHER as in the bounce copy: one wavefront reads the bytes of its workgroup's four buffers back behind a barrier.  Each by
 * itself in workgroups of one and together in workgroups of four, on other buffers at every launch / on the same ones, us:
 *   65,536 of up to 8 KiB    120.7 / 95.5  121.0 / 95.8  (two wavefronts 120.9 / 96.4, eight 121.8 / 99.1;
 *                                                         runs of 32: 121.0 / 97.2)
 *   20,000 of up to 8 KiB     38.2 / 32.7   38.3 / 32.0
 *   65,536 of up to 4000 B    66.3 / 51.1   66.1 / 48.7
 *   65,536 of up to 500 B     27.7 / 26.9   24.7 / 23.5  (two wavefronts 27.4 / 26.3, eight 25.3 / 24.0; no read-back 17.1)
 *   20,000 of up to 500 B     11.7 /  8.9   10.5 /  8.5
 */
constexpr int eager_waves(read_back_t back)
{
	return back == TOGETHER ? kEagerWaves : 1;
}
constexpr uint32_t eager_run(read_back_t back)
{
	return back == TOGETHER ? 64 : 32;
}
template <read_back_t BACK>
__global__ __launch_bounds__(64 * eager_waves(BACK)) void eager_copy_kernel(
	const uint8_t *__restrict__ rx_base, const uint64_t *__restrict__ rx_off,
	const uint32_t *__restrict__ recv_len, uint8_t *__restrict__ dst_base,
	const uint64_t *__restrict__ dst_off, const uint32_t *__restrict__ dst_len, uint32_t n,
	uint32_t *__restrict__ copied, uint32_t *__restrict__ flush)
{
	constexpr int WAVES = eager_waves(BACK);
	constexpr uint32_t kGroup = eager_run(BACK) / WAVES;
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const uint32_t xcd = blockIdx.x % kXcds;
	const uint32_t turn = blockIdx.x / kXcds;
	const uint32_t wg = ((turn / kGroup) * kXcds + xcd) * kGroup + turn % kGroup;
	const uint32_t first = wg * WAVES, buf = first + wave;
	if (BACK != TOGETHER && buf >= n) {
		return;
	}
	uint8_t *d = nullptr;
	uint32_t bytes = 0;
	if (BACK != TOGETHER || buf < n) {
		const uint64_t from = rx_off[buf], to = dst_off[buf];
		const uint32_t received = recv_len[buf], room = dst_len[buf];
		/* all of the entry is in hand from here on: the compiler would ask for the source only once the length is known (us, other
		 * buffers at every launch: 2000 of up to 8 KiB 5.9 -> 5.6, 65,536 of up to 4000 B 67.9 -> 66.4, of up to 500 B 28.5 -> 27.6) */
		__asm__ volatile("" : : "s"(from), "s"(to), "s"(received), "s"(room), "s"(copied), "s"(flush));
		const uint8_t *s = rx_base + from + 8u; /* skip nccl_ofi_eager_msg_header_t */
		d = dst_base + to;
		bytes = min(received, room);
		if (copied != nullptr && lane == 0) {
			copied[buf] = bytes;
		}

		copy_any<BACK == BY_ITSELF>(s, d, bytes, lane);
	}

	if constexpr (BACK == TOGETHER) {
		__shared__ uint8_t *back[WAVES];
		__shared__ uint32_t count[WAVES];
		if (lane == 0) {
			back[wave] = d;
			count[wave] = min(bytes, 4u);
		}
		__syncthreads(); /* the copies, too, are in front of it */
		if (threadIdx.x < WAVES * 4) {
			const uint32_t of = lane >> 2, at = lane & 3u;
			uint32_t byte = 0;
			if (at < count[of]) {
				byte = __builtin_nontemporal_load(back[of] + at);
			}
			const uint32_t word = quad_word(byte, at);
			if (at == 0 && first + of < n) {
				flush[first + of] = word;
			}
		}
	} else if constexpr (BACK == BY_ITSELF) {
		__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
		uint32_t byte = 0;
		if (lane < min(bytes, 4u)) {
			byte = d[lane];
		}
		const uint32_t word = quad_word(byte, lane & 3u);
		if (lane == 0) {
			flush[buf] = word;
		}
	}
}

/*
 * The same for rx buffers in host memory, which the link bounds.  It reads 8 KiB each for thousands of wavefronts at 46 GB/s
 * and for some tens to hundreds at 54, so wavefronts with more than kTurnBytes take turns, one of a workgroup's four at a time, and the
 * others, whose copies are a few trips and no more, do not.  Neighbours are dealt to the XCDs by fours here: by runs of 32 a few
 * hundred buffers load them unevenly, and nothing that neighbours share in host memory stays in an L2.  (Eight to a workgroup:
 * short buffers 0.8 us slower, their pages are looked up CU by CU.  256 wavefronts with a loop over buffers: long ones as
 * fast, 600 of up to 500 B 8.2.)  By the kernel above / in fours without turns / with turns, us:
 *     64 of up to 8 KiB   8.6 / 7.9 / 10.1        300 of up to 4000 B   16.1 / 15.0 / 14.5
 *    150                 16.6 / 14.8 / 14.6      2048                   96.5 / 97 / 83
 *    300                 30.7 / 27.6 / 26.3       300 of up to 500 B     5.1 / 5.2 / 5.2
 *   1000                 96 / 96 / 80             600                    7.3 / 7.4 / 7.4
 *   2048                183 / 183 / 162          2048                   18.0 / 18.1 / 18.1
 * Asking the runtime where the buffers lie takes the host 0.1 us, so that small batches are left to the kernel above.
 */
constexpr uint32_t kHostWaves = 4, kTurnBytes = 1024, kHostBatch = 128;
template <bool READ_BACK>
__global__ __launch_bounds__(64 * kHostWaves) void eager_copy_host_kernel(
	const uint8_t *__restrict__ rx_base, const uint64_t *__restrict__ rx_off,
	const uint32_t *__restrict__ recv_len, uint8_t *__restrict__ dst_base,
	const uint64_t *__restrict__ dst_off, const uint32_t *__restrict__ dst_len, uint32_t n,
	uint32_t *__restrict__ copied, uint32_t *__restrict__ flush)
{
	const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const uint32_t buf = blockIdx.x * kHostWaves + wave;
	const uint32_t at = min(buf, n - 1u);
	const uint64_t from = rx_off[at], to = dst_off[at];
	const uint32_t received = recv_len[at], room = dst_len[at];
	__asm__ volatile("" : : "s"(from), "s"(to), "s"(received), "s"(room), "s"(copied), "s"(flush)); /* as above */
	const uint8_t *s = rx_base + from + 8u;
	uint8_t *d = dst_base + to;
	const uint32_t bytes = buf < n ? min(received, room) : 0u;
	if (copied != nullptr && buf < n && lane == 0) {
		copied[buf] = bytes;
	}
	auto read_back = [&] {
		if (READ_BACK && buf < n) {
			__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
			uint32_t byte = 0;
			if (lane < min(bytes, 4u)) {
				byte = d[lane];
			}
			const uint32_t word = quad_word(byte, lane & 3u);
			if (lane == 0) {
				flush[buf] = word;
			}
		}
	};
	/* kHostWaves - 1 barriers in every wavefront, in front of the copy as many as its turn */
	const bool waits = bytes > kTurnBytes;
	if (waits) {
		for (uint32_t t = 0; t < wave; t++) {
			__builtin_amdgcn_s_barrier();
		}
	}
	copy_any<READ_BACK>(s, d, bytes, lane); /* its loads have come when its stores leave */
	if (!waits) {
		read_back();
	}
	for (uint32_t t = waits ? wave + 1u : 1u; t < kHostWaves; t++) {
		__builtin_amdgcn_s_barrier();
	}
	if (waits) {
		read_back();
	}
}

/* One wavefront per (source address, destination address, length) entry. */
__global__ __launch_bounds__(64 * kTableWaves) void copy_table_kernel(const uint64_t *__restrict__ src_addr,
							     const uint64_t *__restrict__ dst_addr,
							     const uint32_t *__restrict__ len, uint32_t n)
{
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const uint32_t i = blockIdx.x * kTableWaves + wave;
	if (i >= n) {
		return;
	}
	copy_any(reinterpret_cast<const uint8_t *>(src_addr[i]), reinterpret_cast<uint8_t *>(dst_addr[i]), len[i],
		 lane);
}

/*
 * The same table with one wavefront per 8 KiB piece of an entry instead of per entry: entry e has
 * the `per` piece numbers from e * per on, and a wavefront whose piece lies beyond its entry's
 * length leaves at once.  Consecutive wavefronts then sweep long entries densely, 8 KiB each,
 * instead of each streaming through its own entry (1 GiB copied 8 KiB per wavefront: 5.65 TB/s read
 * + written, 256 KiB per wavefront: 5.17), and the XCDs take runs of about 128 consecutive pieces (1 MiB)
 * in turn (5.82 TB/s; runs of 4 or 16: 5.5-5.7).
 *
 * A table of mixed lengths consists mostly of pieces that do not exist (lengths log-uniform in
 * 8 B..1 MiB: 11 of an entry's 128 pieces do), and how those that do are dealt out counts:
 * - Workgroups are handed out at about 4.5 a nanosecond, whatever they hold: 262,144 wavefronts that
 *   leave at once take 56 us singly and 15 us by fours.  244 entries of 8 B..64 MiB: 538 us
 *   singly, 435 us by fours.  By fours a dense copy is as fast as singly; by eights a sparse one is slower
 *   (2048 entries of 8 B..1 MiB 84 us against 76).
 * - Workgroups are dealt to the XCDs, and inside one to the shader engines, in turn.  With a power of two of
 *   pieces to an entry the first, always present pieces of all entries fall to the same few of them.  So
 *   `per` is odd, or an odd number of runs, each of an odd number of workgroups, and the four
 *   wavefronts of a workgroup take pieces a quarter of a run apart (copy_pieces_map says from when
 *   on).  442 entries of 64 KiB..4 MiB: 204 -> 180 us; 16,384 of 8 B..64 KiB: 59 -> 48 us; 10,088
 *   of 8 B..512 KiB 200 -> 183 us.
 * - The table may lie in host memory, a link's round trip away.  Its three words are asked for together,
 *   not the addresses once the length is known (7 entries of 4-8 KiB: 5.6 -> 4.1 us).
 * All told, tables in host memory, other buffers at every launch: 2048 entries of 8 B..1 MiB 78 -> 72 us (5.2 of
 * the 5.4 TB/s read + written of one plain copy of those bytes), 16,384 of 8 B..64 KiB 69 -> 48 us.
 */
constexpr uint32_t kPieceBytes = kRows * 1024u;
constexpr uint32_t kPieceWaves = 4;
constexpr uint32_t kRunPieces = 128;
struct piece_map_t {
	uint32_t per;         /* piece numbers of an entry: at least those of the longest one */
	uint32_t run_blocks;  /* workgroups of a run */
	uint32_t wave_stride; /* piece numbers between two wavefronts of a workgroup, and ... */
	uint32_t block_stride; /* ... between two workgroups of a run */
};
__global__ __launch_bounds__(64 * kPieceWaves) void copy_table_pieces_kernel(const uint64_t *__restrict__ src_addr,
									     const uint64_t *__restrict__ dst_addr,
									     const uint32_t *__restrict__ len, uint32_t n,
									     piece_map_t map, uint32_t max_len,
									     uint32_t *__restrict__ err)
{
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const uint32_t xcd = blockIdx.x % kXcds, turn = blockIdx.x / kXcds;
	const uint32_t run = turn / map.run_blocks, block = turn - run * map.run_blocks;
	const uint32_t g = (run * kXcds + xcd) * map.run_blocks * kPieceWaves + wave * map.wave_stride +
			   block * map.block_stride;
	const uint32_t e = g / map.per, piece = g - e * map.per;
	if (e >= n) {
		return;
	}
	const uint32_t stated = len[e];
	const uint64_t src = src_addr[e], dst = dst_addr[e];
	/* all three are in hand from here on: the compiler would move the addresses behind the test of the length */
	__asm__ volatile("" : : "s"(stated), "s"(src), "s"(dst));
	if (piece == 0 && stated > max_len && lane == 0) {
		atomicOr(err, ofi_amd::ASYNC_ERR_COPY_LENGTH); /* longer than the caller said: the rest stays uncopied */
	}
	const uint32_t bytes = min(stated, max_len);
	const uint64_t off = (uint64_t)piece * kPieceBytes;
	if (off >= bytes) {
		return;
	}
	/* Pieces meet on 64-byte boundaries of the destination, so that only an entry's first and last have single bytes to copy,
	 * the last up to 63 more than a piece, which is still one trip.  Those between are straight-line code of whole rows (us,
	 * before and now, other buffers at every launch / the same ones: 2048 entries of 8 B..1 MiB 75.7 / 67.4 -> 72.2 / 64.6, 400 of
	 * them 17.4 / 18.0 -> 16.6 / 17.5, 3000 of 32-64 KiB 60.7 / 46.1 -> 60.1 / 45.8, 1000 of 128 KiB-8 MiB 788 -> 783; 16 of 32-64 MiB
	 * 294.5 -> 294.1, from odd addresses 294.0 -> 295.4).  Non-temporal loads in them are 2-4 % faster beyond a GiB, but
	 * shorter tables, which the launch cannot tell by their longest entry, lose: 400 entries 19, 3000 on the same buffers 54. */
	const uint32_t skew = (uint32_t)dst & 63u;
	const uint64_t from = piece == 0 ? 0 : off - skew;
	const bool last = bytes - off <= kPieceBytes;
	const uint8_t *s = reinterpret_cast<const uint8_t *>(src + from);
	uint8_t *d = reinterpret_cast<uint8_t *>(dst + from);
	if (piece != 0 && !last) {
		const uint32_t shift = (uint32_t)(reinterpret_cast<uintptr_t>(s) & 3u);
		if (shift == 0) {
			copy_rows<kRows, false, true, false>(s, d, kTripVec, 0, lane);
		} else {
			copy_rows<kRows, true, true, false>(s - shift, d, kTripVec, shift, lane);
		}
	} else {
		copy_any(s, d, last ? (uint32_t)(bytes - from) : kPieceBytes - skew, lane);
	}
}

__global__ __launch_bounds__(256) void flush_read_kernel(const uint8_t *__restrict__ arena,
							 const uint64_t *__restrict__ dst_off,
							 uint32_t n, uint32_t *__restrict__ flush)
{
	const uint32_t i = blockIdx.x * 256u + threadIdx.x;
	if (i < n) {
		flush[i] = __hip_atomic_load(reinterpret_cast<const uint32_t *>(arena + dst_off[i]),
					     __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
	}
}

__global__ __launch_bounds__(64) void flush_fill_kernel(uint64_t *__restrict__ flush_buf, uint64_t sentinel)
{
	if (threadIdx.x < 8) {
		flush_buf[threadIdx.x] = sentinel;
	}
}

__global__ __launch_bounds__(64) void flush_post_kernel(const uint64_t *__restrict__ flush_buf,
							uint64_t *__restrict__ slots, uint32_t num_rails)
{
	ofi_amd::flush_post_lanes(flush_buf, slots, num_rails, threadIdx.x);
}

/*
 * How the pieces of a table are dealt out, by the pieces of its longest entry (`pieces`: of all entries
 * if they were all that long).  Few pieces: neighbours in a workgroup, whose table words then share cache lines
 * (5818 entries of up to 4 pieces 11.0 us, a quarter of a run apart 13.8).  1024 and more: an entry has
 * a run for every XCD and spreads by itself (64 entries of 16-32 MiB 578 us, padded 582).
 * Between the two as the kernel's comment says.  Tables of more than kMostPadded pieces go without the padding,
 * which is less than as much again, so that a launch always stays below what it can number.
 */
constexpr uint32_t kFewPieces = 8, kManyPieces = 1024;
constexpr uint64_t kMostPadded = 1ull << 24;
/* The pieces of one launch, in whole rounds over the XCDs: 2^32 work-items are one too many for a launch. */
constexpr uint64_t kMostPieces = (1ull << 26) - kXcds * kRunPieces;
static_assert(kMostPieces * 64 < 1ull << 32 && 2 * kMostPadded + kXcds * 2 * kRunPieces <= kMostPieces,
	      "a launch, padded or not");
piece_map_t copy_pieces_map(uint32_t per, uint64_t pieces)
{
	piece_map_t m = { per, kRunPieces / kPieceWaves, 1, kPieceWaves };
	if (per < kFewPieces || per >= kManyPieces || pieces > kMostPadded) {
		return m;
	}
	if (per <= kRunPieces) {
		m.per = per | 1u;
	} else {
		const uint32_t runs = ((per + kRunPieces - 1) / kRunPieces) | 1u;
		m.run_blocks = ((per + runs * kPieceWaves - 1) / (runs * kPieceWaves)) | 1u;
		m.per = runs * m.run_blocks * kPieceWaves;
	}
	m.wave_stride = m.run_blocks;
	m.block_stride = 1;
	return m;
}

} // namespace

/* A registered region: on a large-BAR system the whole of device memory is mapped into the
 * process at its device address, so the CPU mapping that GDRCopy creates by pinning and
 * mmap-ing (gdrcopy_RegHandle::mapped_ptr, include/nccl_ofi_gdrcopy.h:54-74) is the device
 * pointer itself. */
struct ofi_amd_devcopy_region {
	uint8_t *base;   /* device address (= CPU-visible mapping where cpu_mapped) */
	size_t size;
	bool cpu_mapped; /* the CPU can store to and load from `base`: large BAR and the range is in the
			  * process's address space; otherwise every copy goes through the copy engine */
};

/* CPU stores into the mapping are write-combined: 0.2-0.4 us for anything up to a page and
 * about 20 GB/s up to 1 MiB, against 11-14 us for the smallest hipMemcpy; from 16 MiB on the
 * copy engine is faster.  CPU loads from it are uncached round trips over PCIe: 2.5 us per
 * 64 bytes, so only a read of a few words beats the 12 us of a hipMemcpy. */
constexpr size_t kCpuStoreMax = 2u << 20;
constexpr size_t kCpuLoadMax = 256;

/*
 * Batches that fit the L2s (8 x 4 MiB) with room to spare keep the first row of every buffer in them instead of
 * streaming it (a buffer without a row, its tail): the read-back behind it then finds its line there.  The bytes of a
 * bounce batch are at most the source's where that is packed; where it is a pool that the batch takes a part of, and in an
 * eager batch, the number of buffers, which are mostly up to 8 KiB, has to do.  However short the buffers are, each keeps a
 * line, and from some hundred thousand on these no longer fit (kKeepLines).  Times in us on other buffers at
 * every launch / on the same ones, streamed (bounce: read back together) and then kept:
 *   6000 bounce buffers of up to 8 KiB     10.9 / 10.2   9.7 / 9.2
 *   8000 of up to 8 KiB                    13.7 / 12.2  13.1 / 12.0  (out of a pool 13.6 / 12.2  13.8 / 12.3)
 *   10,000 of up to 8 KiB                  16.5 / 15.3  18.0 / 15.4
 *   16,000 of up to 4 KiB                  13.6 / 12.6  12.8 / 12.0
 *   60,000 of up to 1000 B                 22.8 / 22.2  18.5 / 17.9
 *   65,536 of up to 60 B                   17.5 / 15.9  17.0 / 14.8  (its tail streamed: 18.9 / 14.9)
 *   200,000 of up to 100 B                   62 / 55      48 / 48
 *   450,000 of up to 60 B                   113 / 105     85 / 85
 *   500,000 of up to 60 B                   123 / 117    113 / 93    (flush words in HBM 104 / 98  110 / 90)
 *   700,000 of up to 60 B                   163 / 162    174 / 128
 *   8000 eager buffers of up to 8 KiB      14.9 / 13.7  14.1 / 12.2
 *   9000 of up to 8 KiB                    16.2 / 15.4  16.3 / 13.5
 *   12,000 of up to 8 KiB                  20.0 / 19.9  21.6 / 17.7
 *   16,000 of up to 8 KiB                  27.5 / 26.0  32.2 / 23.0
 */
constexpr uint64_t kKeepBytes = 32ull << 20;
constexpr uint32_t kKeepBounce = 8000, kKeepByItself = 11000, kKeepLines = 450000, kKeepEager = 9000;
/*
 * Fewer wavefronts a CU for large batches of long buffers -- reads and writes take turns at the memory, and the fewer
 * buffers are open the longer the turns are -- were measured and are not used: 65,536 of up to 8 KiB 110.9 us with 32
 * wavefronts, 109.0 with 24 and 107.2 with 20 (held by the LDS a workgroup claims) on other buffers at every launch, but
 * 81.1, 84.1 and 86.5 on the same ones over and over, and short buffers starve (65,536 of up to 1000 B 25.2 / 31.2 /
 * 34.8).  The host has no lengths to choose by: src_bytes is the range the batch's offsets lie in, a pool as a rule.
 */

using namespace ofi_amd;

extern "C" {

int ofi_amd_bounce_scatter(const void *d_src, uint64_t src_bytes, void *d_arena, uint64_t arena_bytes,
			   const uint64_t *d_src_off, const uint64_t *d_dst_off,
			   const uint32_t *d_len, uint32_t n, uint32_t *d_flush, void *stream)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (n == 0) {
		return 0;
	}
	if (!d_src || !d_arena || !d_src_off || !d_dst_off || !d_len || n > (1u << 30)) {
		return -EINVAL;
	}
	uint32_t *err = async_error_word();
	if (!err) {
		return -ENOMEM;
	}
	const uint32_t runs = (n + kXcds * kBounceRun - 1) / (kXcds * kBounceRun); /* whole rounds over the XCDs */
	auto launch = [&](auto kernel) {
		ofi_amd::launch_kernel(kernel, dim3(runs * kXcds * (kBounceRun / kBounceWaves)), dim3(64 * kBounceWaves), 0,
				       as_stream(stream), static_cast<const uint8_t *>(d_src), src_bytes, d_src_off, d_dst_off, d_len, n,
				       static_cast<uint8_t *>(d_arena), arena_bytes, d_flush, err);
	};
	if (!d_flush) {
		launch(bounce_scatter_kernel<NO_READ_BACK>);
	} else if (n <= kKeepBounce || (n <= kKeepByItself && src_bytes <= kKeepBytes)) {
		launch(bounce_scatter_kernel<BY_ITSELF>);
	} else if (n <= kKeepLines && src_bytes <= kKeepBytes) {
		launch(bounce_scatter_kernel<KEPT_TOGETHER>);
	} else {
		launch(bounce_scatter_kernel<TOGETHER>);
	}
	OFI_AMD_HIP_TRY(hipGetLastError());
	return 0;
}

int ofi_amd_eager_copy_batch(const void *rx_base, const uint64_t *d_rx_off, const uint32_t *d_recv_len,
			     void *dst_base, const uint64_t *d_dst_off, const uint32_t *d_dst_len,
			     uint32_t n, uint32_t *d_copied, uint32_t *d_flush, void *stream)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (n == 0) {
		return 0;
	}
	if (!rx_base || !d_rx_off || !d_recv_len || !d_dst_off || !d_dst_len || n > (1u << 30)) {
		return -EINVAL;
	}
	auto launch = [&](auto kernel, read_back_t back) {
		const uint32_t round = kXcds * eager_run(back), waves = (uint32_t)eager_waves(back); /* whole rounds over the XCDs */
		ofi_amd::launch_kernel(kernel, dim3((n + round - 1) / round * (round / waves)), dim3(64 * waves), 0, as_stream(stream),
				       static_cast<const uint8_t *>(rx_base), d_rx_off, d_recv_len, static_cast<uint8_t *>(dst_base),
				       d_dst_off, d_dst_len, n, d_copied, d_flush);
	};
	if (n >= kHostBatch && in_host_memory(rx_base)) {
		auto launch_host = [&](auto kernel) {
			ofi_amd::launch_kernel(kernel, dim3((n + kHostWaves - 1) / kHostWaves), dim3(64 * kHostWaves), 0, as_stream(stream),
					       static_cast<const uint8_t *>(rx_base), d_rx_off, d_recv_len,
					       static_cast<uint8_t *>(dst_base), d_dst_off, d_dst_len, n, d_copied, d_flush);
		};
		d_flush ? launch_host(eager_copy_host_kernel<true>) : launch_host(eager_copy_host_kernel<false>);
	} else if (!d_flush) {
		launch(eager_copy_kernel<NO_READ_BACK>, NO_READ_BACK);
	} else if (n <= kKeepEager) {
		launch(eager_copy_kernel<BY_ITSELF>, BY_ITSELF);
	} else {
		launch(eager_copy_kernel<TOGETHER>, TOGETHER);
	}
	OFI_AMD_HIP_TRY(hipGetLastError());
	return 0;
}

int ofi_amd_copy_table(const uint64_t *d_src_addr, const uint64_t *d_dst_addr, const uint32_t *d_len,
		       uint32_t n, void *stream)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (n == 0) {
		return 0;
	}
	if (!d_src_addr || !d_dst_addr || !d_len || n > (1u << 30)) {
		return -EINVAL;
	}
	ofi_amd::launch_kernel(copy_table_kernel, dim3((n + kTableWaves - 1) / kTableWaves), dim3(64 * kTableWaves), 0,
			       as_stream(stream), d_src_addr, d_dst_addr, d_len, n);
	OFI_AMD_HIP_TRY(hipGetLastError());
	return 0;
}

int ofi_amd_copy_table_pieces(const uint64_t *d_src_addr, const uint64_t *d_dst_addr, const uint32_t *d_len,
			      uint32_t n, uint32_t max_len, void *stream)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (n == 0) {
		return 0;
	}
	if (!d_src_addr || !d_dst_addr || !d_len || n > (1u << 30)) {
		return -EINVAL;
	}
	const uint64_t pieces_per_entry = max_len == 0 ? 1 : ((uint64_t)max_len + kPieceBytes - 1) / kPieceBytes;
	const uint64_t least = (uint64_t)kXcds * kRunPieces;
	if (((uint64_t)n * pieces_per_entry + least - 1) / least * least > 0x7fffffffull) {
		return -E2BIG; /* split the table */
	}
	uint32_t *err = async_error_word();
	if (!err) {
		return -ENOMEM;
	}
	/* a launch for every kMostPieces pieces: at least 127 entries each, however long */
	const uint32_t part = (uint32_t)(kMostPieces / pieces_per_entry);
	for (uint32_t at = 0; at < n; at += part) {
		const uint32_t here = n - at < part ? n - at : part;
		const piece_map_t map = copy_pieces_map((uint32_t)pieces_per_entry, here * pieces_per_entry);
		const uint64_t round = (uint64_t)kXcds * map.run_blocks * kPieceWaves; /* whole rounds over the XCDs */
		const uint64_t blocks = ((uint64_t)here * map.per + round - 1) / round * (kXcds * map.run_blocks);
		ofi_amd::launch_kernel(copy_table_pieces_kernel, dim3((uint32_t)blocks), dim3(64 * kPieceWaves), 0,
				       as_stream(stream), d_src_addr + at, d_dst_addr + at, d_len + at, here, map, max_len, err);
	}
	OFI_AMD_HIP_TRY(hipGetLastError());
	return 0;
}

int ofi_amd_flush_read(const void *d_arena, const uint64_t *d_dst_off, uint32_t n,
		       uint32_t *d_flush, void *stream)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (n == 0) {
		return 0;
	}
	if (!d_arena || !d_dst_off || !d_flush) {
		return -EINVAL;
	}
	ofi_amd::launch_kernel(flush_read_kernel, dim3((n + 255u) / 256u), dim3(256), 0,
			       as_stream(stream), static_cast<const uint8_t *>(d_arena), d_dst_off, n,
			       d_flush);
	OFI_AMD_HIP_TRY(hipGetLastError());
	return 0;
}

int ofi_amd_flush_buffer_fill(void *d_flush_buf, uint64_t sentinel, void *stream)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (!d_flush_buf || (reinterpret_cast<uintptr_t>(d_flush_buf) & 7u)) {
		return -EINVAL;
	}
	ofi_amd::launch_kernel(flush_fill_kernel, dim3(1), dim3(64), 0, as_stream(stream),
			       static_cast<uint64_t *>(d_flush_buf), sentinel);
	OFI_AMD_HIP_TRY(hipGetLastError());
	return 0;
}

int ofi_amd_flush_post(const void *d_flush_buf, void *slots_dev, uint32_t num_rails, void *stream)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (!d_flush_buf || !slots_dev || num_rails < 1 || num_rails > OFI_AMD_MAX_NUM_RAILS ||
	    (reinterpret_cast<uintptr_t>(d_flush_buf) & 7u) || (reinterpret_cast<uintptr_t>(slots_dev) & 7u)) {
		return -EINVAL;
	}
	ofi_amd::launch_kernel(flush_post_kernel, dim3(1), dim3(64), 0, as_stream(stream),
			       static_cast<const uint64_t *>(d_flush_buf), static_cast<uint64_t *>(slots_dev),
			       num_rails);
	OFI_AMD_HIP_TRY(hipGetLastError());
	return 0;
}

/* ofi_amd_flush_test, the host side of the flush, lives with the other host-only wire code
 * (wire_codec.cpp). */

/* ---- nccl_ofi_device_copy (include/nccl_ofi_device_copy.h:14-69) ---- */

int ofi_amd_devcopy_register(void *device_ptr, size_t size, ofi_amd_devcopy_region_t **out)
{
	int rc = require_device();
	if (rc != 0) {
		return rc;
	}
	if (!device_ptr || size == 0 || !out) {
		return -EINVAL;
	}
	hipPointerAttribute_t attr;
	if (hipPointerGetAttributes(&attr, device_ptr) != hipSuccess) {
		(void)hipGetLastError();
		return -EINVAL;
	}
	if (attr.type != hipMemoryTypeDevice) {
		return -EINVAL;
	}
	/* The CPU reaches device memory only where the whole of it sits behind the PCIe BAR, and
	 * then only allocations that the runtime has mapped into the process at their device
	 * address (hipMalloc memory is; an imported or virtual-memory allocation need not be):
	 * the first and the last page of the range are asked of the kernel.  Without either,
	 * the region still registers and its copies take the copy engine at every size, as the
	 * interface promises nothing about the path. */
	int large_bar = 0;
	if (hipDeviceGetAttribute(&large_bar, hipDeviceAttributeIsLargeBar, attr.device) != hipSuccess) {
		(void)hipGetLastError();
		large_bar = 0;
	}
	bool mapped = large_bar != 0;
	if (mapped) {
		const long page = sysconf(_SC_PAGESIZE);
		const uintptr_t first = reinterpret_cast<uintptr_t>(device_ptr) & ~(uintptr_t)(page - 1);
		const uintptr_t last = (reinterpret_cast<uintptr_t>(device_ptr) + size - 1) & ~(uintptr_t)(page - 1);
		unsigned char vec = 0;
		mapped = mincore(reinterpret_cast<void *>(first), (size_t)page, &vec) == 0 &&
			 mincore(reinterpret_cast<void *>(last), (size_t)page, &vec) == 0;
	}
	auto *h = new (std::nothrow) ofi_amd_devcopy_region;
	if (!h) {
		return -ENOMEM;
	}
	h->base = static_cast<uint8_t *>(device_ptr);
	h->size = size;
	h->cpu_mapped = mapped;
	*out = h;
	return 0;
}

int ofi_amd_devcopy_to_device(const void *host_ptr, ofi_amd_devcopy_region_t *h, size_t offset,
			      size_t size)
{
	if (!h || !host_ptr || offset > h->size || size > h->size - offset) {
		return -EINVAL;
	}
	if (h->cpu_mapped && size <= kCpuStoreMax) {
		/* gdr_copy_to_mapping: CPU stores through the mapping, then drain the
		 * write-combining buffers so that the bytes are on their way before the caller
		 * rings any doorbell */
		std::memcpy(h->base + offset, host_ptr, size);
		_mm_sfence();
		return 0;
	}
	OFI_AMD_HIP_TRY(hipMemcpy(h->base + offset, host_ptr, size, hipMemcpyHostToDevice));
	return 0;
}

int ofi_amd_devcopy_from_device(ofi_amd_devcopy_region_t *h, size_t offset, void *host_ptr,
				size_t size)
{
	if (!h || !host_ptr || offset > h->size || size > h->size - offset) {
		return -EINVAL;
	}
	if (h->cpu_mapped && size <= kCpuLoadMax) {
		/* gdr_copy_from_mapping: CPU loads through the mapping */
		std::memcpy(host_ptr, h->base + offset, size);
		_mm_lfence();
		return 0;
	}
	OFI_AMD_HIP_TRY(hipMemcpy(host_ptr, h->base + offset, size, hipMemcpyDeviceToHost));
	return 0;
}

int ofi_amd_devcopy_cpu_mapped(const ofi_amd_devcopy_region_t *h)
{
	return h ? (h->cpu_mapped ? 1 : 0) : -EINVAL;
}

int ofi_amd_devcopy_forced_pcie_copy(void)
{
	return 0;
}

int ofi_amd_devcopy_deregister(ofi_amd_devcopy_region_t *h)
{
	if (!h) {
		return -EINVAL;
	}
	delete h;
	return 0;
}

} /* extern "C" */
