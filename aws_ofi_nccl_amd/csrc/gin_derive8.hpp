/*
 * iputSignal's derivation (gin_derive.hpp) for up to eight descriptors of a communicator at once, a descriptor per 64-bit
 * lane of the AVX-512 registers, for the proxy's drain loop (gin_proxy.cpp) on CPUs that have them.
 *
 * A descriptor by itself costs some 250 instructions and two branches on its size (12.5 ns on a Zen 5 core, all told); eight
 * together cost 5.5 ns each, 6.6 where a region's words are gathered lane by lane.  What goes from one descriptor to the next --
 * the scheduler's two counters, the pinned rail with the length of its run, the sequence number -- is a prefix over the lanes.
 */
#ifndef OFI_AMD_GIN_DERIVE8_HPP_
#define OFI_AMD_GIN_DERIVE8_HPP_

#include <cstddef>

#include <immintrin.h>

#include "gin_derive.hpp"

namespace ofi_amd_gin {

constexpr uint32_t kLanes = 8;
constexpr uint64_t kFoldKeys[kLanes] = {
	0x9E3779B97F4A7C15ull, 0xBF58476D1CE4E5B9ull, 0x94D049BB133111EBull, 0xD6E8FEB86659FD93ull,
	0xCA5A826395121157ull, 0x2545F4914F6CDD1Dull, 0xA0761D6478BD642Full, 0xE7037ED1A0B428DBull,
};

#define OFI_AMD_WIDE __attribute__((target("avx512f,avx512bw,avx512cd,avx512dq,avx512vl")))

inline bool cpu_has_wide()
{
	return __builtin_cpu_supports("avx512f") && __builtin_cpu_supports("avx512bw") && __builtin_cpu_supports("avx512cd") &&
	       __builtin_cpu_supports("avx512dq") && __builtin_cpu_supports("avx512vl");
}

/* rows and columns of eight registers of eight words change places */
OFI_AMD_WIDE __attribute__((always_inline)) inline void transpose8(__m512i r[kLanes])
{
	__m512i t[kLanes], u[kLanes];
	for (uint32_t k = 0; k < kLanes; k += 2) {
		t[k] = _mm512_unpacklo_epi64(r[k], r[k + 1]);
		t[k + 1] = _mm512_unpackhi_epi64(r[k], r[k + 1]);
	}
	for (uint32_t k = 0; k < 2; k++) { /* u[j]: 128-bit blocks of rows 0..3, u[j + 4]: of rows 4..7 */
		u[k] = _mm512_shuffle_i64x2(t[k], t[k + 2], 0x88);
		u[k + 2] = _mm512_shuffle_i64x2(t[k], t[k + 2], 0xdd);
		u[k + 4] = _mm512_shuffle_i64x2(t[k + 4], t[k + 6], 0x88);
		u[k + 6] = _mm512_shuffle_i64x2(t[k + 4], t[k + 6], 0xdd);
	}
	for (uint32_t k = 0; k < 4; k++) {
		r[k] = _mm512_shuffle_i64x2(u[k], u[k + 4], 0x88);
		r[k + 4] = _mm512_shuffle_i64x2(u[k], u[k + 4], 0xdd);
	}
}

/* sums over the lanes before each */
OFI_AMD_WIDE __attribute__((always_inline)) inline __m512i sum_before(__m512i v)
{
	const __m512i zero = _mm512_setzero_si512();
	v = _mm512_add_epi64(v, _mm512_alignr_epi64(v, zero, 7));
	v = _mm512_add_epi64(v, _mm512_alignr_epi64(v, zero, 6));
	v = _mm512_add_epi64(v, _mm512_alignr_epi64(v, zero, 4));
	return _mm512_alignr_epi64(v, zero, 7);
}

struct derived8_t {
	uint32_t signals, writes;
	alignas(64) uint64_t folds[kLanes]; /* the checksum's sum over each descriptor's words */
};

/*
 * derive<true> for the `count` descriptors from d on, one to eight, where derive_fast_path holds: the records at out, the
 * communicator moved on.  False, with nothing changed, where one of them is not an ordinary put (no payload, a get, an operation
 * or a handle that is none) or the window is far enough gone for an ACK to be asked for: those are derived one by one.
 */
OFI_AMD_WIDE __attribute__((noinline)) inline bool derive8(ofi_amd_gin_comm_t *c, const ofi_amd_gin_mr_t *mrs, uint32_t n_mrs,
							    const ofi_amd_gin_desc_t *d, uint32_t count, ofi_amd_gin_wire_t *out,
							    derived8_t *sums)
{
	static_assert(sizeof(*d) == 64 && sizeof(*out) == 28 * 8 && sizeof(*mrs) == 7 * 8, "words of a descriptor, a record, a region");
	const uint32_t head = c->tx_head;
	if (cursor_delta(head, c->tx_tail) + count > kAckReqThreshold || c->pinned_rail_run >= kReqsPerDoorbell) {
		return false;
	}
	const __mmask8 live = (__mmask8)((1u << count) - 1u);
	const __m512i zero = _mm512_setzero_si512(), one = _mm512_set1_epi64(1);
	const __m512i lane = _mm512_set_epi64(7, 6, 5, 4, 3, 2, 1, 0);
	const __m512i low32 = _mm512_set1_epi64(0xffffffffll), low16 = _mm512_set1_epi64(0xffff);

	__m512i w[kLanes];
	for (uint32_t k = 0; k < kLanes; k++) {
		w[k] = k < count ? _mm512_loadu_si512(&d[k]) : zero;
	}
	transpose8(w);
	const __m512i src_off = w[0], dst_off = w[1], size = w[2], sig_off = w[3], sig_value = w[4];
	const __m512i sop = _mm512_srli_epi64(w[5], 32), opt = _mm512_and_si512(w[6], low32);
	const __m512i src_mr = _mm512_and_si512(w[7], low16), dst_mr = _mm512_and_si512(_mm512_srli_epi64(w[7], 16), low16);
	const __m512i sig_mr = _mm512_and_si512(_mm512_srli_epi64(w[7], 32), low16), kind = _mm512_srli_epi64(w[7], 48);

	const __m512i mr_count = _mm512_set1_epi64(n_mrs);
	const __mmask8 signal = _mm512_mask_test_epi64_mask(live, sop, sop);
	const __mmask8 handle = _mm512_mask_cmpneq_epu64_mask(signal, sig_mr, low16); /* of the signal's own */
	__mmask8 bad = _mm512_cmpge_epu64_mask(src_mr, mr_count) | _mm512_cmpge_epu64_mask(dst_mr, mr_count);
	bad |= _mm512_testn_epi64_mask(size, size) | _mm512_cmpgt_epu64_mask(sop, _mm512_set1_epi64(kSignalAdd));
	bad |= _mm512_cmpeq_epu64_mask(kind, _mm512_set1_epi64(OFI_AMD_GIN_KIND_GET));
	bad |= _mm512_mask_cmpge_epu64_mask(handle, sig_mr, mr_count);
	if ((bad & live) != 0) {
		return false;
	}

	/* the checksum's words */
	__m512i fold = zero;
	for (uint32_t k = 0; k < kLanes; k++) {
		fold = _mm512_add_epi64(fold, _mm512_mullo_epi64(_mm512_add_epi64(w[k], _mm512_set1_epi64(k + 1)),
								 _mm512_set1_epi64((long long)kFoldKeys[k])));
	}
	_mm512_store_si512(sums->folds, fold);

	/* the schedule */
	const uint32_t R = (uint32_t)c->sched.num_rails;
	const __m512i rail_mask = _mm512_set1_epi64(R - 1u);
	const __m512i last = _mm512_sub_epi64(size, one); /* size - 1 */
	const __mmask8 small = _mm512_mask_cmplt_epu64_mask(live, size, _mm512_set1_epi64((long long)c->sched.max_small_msg_size));
	const __m512i over = _mm512_srl_epi64(last, _mm_cvtsi32_si128(__builtin_ctzll(c->sched.min_stripe_size))); /* stripes wanted - 1 */
	const __mmask8 big = live & (__mmask8)~small;
	const __mmask8 two = R >= 2 ? _mm512_mask_cmpge_epu64_mask(big, over, one) : (__mmask8)0;
	const __mmask8 four = R >= 4 ? _mm512_mask_cmpge_epu64_mask(big, over, _mm512_set1_epi64(3)) : (__mmask8)0;
	__m512i n = _mm512_maskz_mov_epi64(live, one); /* stripes */
	n = _mm512_mask_mov_epi64(n, two, _mm512_set1_epi64(2));
	n = _mm512_mask_mov_epi64(n, four, _mm512_set1_epi64(4));
	/* what the messages before each have moved the counters on by: the small ones' in the upper half */
	const __m512i step = _mm512_mask_slli_epi64(n, small, n, 32), moved = sum_before(step);
	const __m512i counter = _mm512_mask_mov_epi64(
		_mm512_add_epi64(moved, _mm512_set1_epi64(c->sched.rr_counter)), small,
		_mm512_add_epi64(_mm512_srli_epi64(moved, 32), _mm512_set1_epi64(c->sched.rr_small_counter)));
	const __m512i first = _mm512_and_si512(counter, rail_mask);
	const uint64_t all_moved = (uint64_t)_mm512_reduce_add_epi64(step);

	/* A deferred doorbell pins the rail of the next descriptor.  `defers`: one stripe, asked to be aggregated, unless it is the
	 * last of a run of kReqsPerDoorbell, which within eight descriptors only the run that comes in can reach. */
	const __mmask8 single = live & (__mmask8)~two;
	uint32_t defers = _mm512_mask_test_epi64_mask(single, opt, _mm512_set1_epi64(kOptAggregate));
	const uint32_t run_in = c->pinned_rail_run;
	const uint32_t room = run_in < kReqsPerDoorbell - 1 ? kReqsPerDoorbell - 1 - run_in : 0; /* of the run that comes in */
	if (room < kLanes && (defers & ((1u << room) - 1u)) == (1u << room) - 1u) {
		defers &= ~(1u << room);
	}
	const int32_t pin_in = c->pinned_rail_id;
	const uint32_t pins = defers << 1 | (pin_in >= 0 ? 1u : 0u); /* a pin is open when the descriptor comes */
	/* the pin's rail is that of the last descriptor before that came without one, or the pin's that comes in */
	const __m512i before = _mm512_sub_epi64(_mm512_sllv_epi64(one, lane), one);
	const __m512i unpinned = _mm512_andnot_si512(_mm512_set1_epi64(pins), before);
	const __m512i from = _mm512_sub_epi64(_mm512_set1_epi64(63), _mm512_lzcnt_epi64(unpinned));
	const __m512i pin = _mm512_mask_permutexvar_epi64(_mm512_set1_epi64(pin_in), _mm512_test_epi64_mask(unpinned, unpinned), from, first);
	/* a striped one rings every rail it touches, so it is made to touch the pin */
	const __m512i apart = _mm512_and_si512(_mm512_sub_epi64(pin, first), rail_mask);
	const __m512i rail0 = _mm512_mask_mov_epi64(first, _mm512_mask_cmpge_epu64_mask((__mmask8)pins, apart, n), pin);

	/* records, word by word */
	const __m512i seq = _mm512_and_si512(_mm512_add_epi64(_mm512_set1_epi64(head), lane), _mm512_set1_epi64(kImmSeqMask));
	const __m512i nseg = _mm512_mask_add_epi64(n, signal, n, one);
	const __m512i imm = _mm512_or_si512(
		_mm512_or_si512(_mm512_slli_epi64(nseg, kImmSegCntShift), _mm512_slli_epi64(seq, kImmSeqShift)),
		_mm512_set1_epi64((uint32_t)(c->comm_id << kImmCommShift)));
	const __m512i halves = _mm512_maskz_set1_epi64(signal, 1);
	const __m512i deferred = _mm512_maskz_set1_epi64((__mmask8)defers, 1);

	/* The regions' words: mostly all of a group's descriptors go from one region to one other, and a gather is eight loads */
	const char *const base = reinterpret_cast<const char *>(mrs);
	const __m512i src_at = _mm512_sub_epi64(_mm512_slli_epi64(src_mr, 3), src_mr); /* words of a region: 7 */
	const __m512i dst_at = _mm512_sub_epi64(_mm512_slli_epi64(dst_mr, 3), dst_mr);
	const char *const keys = base + offsetof(ofi_amd_gin_mr_t, key);
	const __m512i regions = _mm512_and_si512(w[7], low32); /* both handles */
	const bool alike = _mm512_mask_cmpneq_epu64_mask(live, regions, _mm512_broadcastq_epi64(_mm512_castsi512_si128(regions))) == 0;
	__m512i src_base, dest_base, dest_keys = zero;
	if (alike) {
		/* the handles that were checked, not what the slot says by now */
		const uint32_t pair = (uint32_t)_mm512_cvtsi512_si32(regions);
		const ofi_amd_gin_mr_t &to = mrs[pair >> 16];
		src_base = _mm512_set1_epi64((long long)mrs[pair & 0xffffu].local_base);
		dest_base = _mm512_set1_epi64((long long)to.remote_address_offset);
		dest_keys = _mm512_castsi256_si512(_mm256_loadu_si256(reinterpret_cast<const __m256i *>(to.key)));
	} else {
		src_base = _mm512_mask_i64gather_epi64(zero, live, src_at, base + offsetof(ofi_amd_gin_mr_t, local_base), 8);
		dest_base = _mm512_mask_i64gather_epi64(zero, live, dst_at, base + offsetof(ofi_amd_gin_mr_t, remote_address_offset), 8);
	}
	const __m512i src = _mm512_add_epi64(src_off, src_base), dest = _mm512_add_epi64(dst_off, dest_base);
	auto key_of = [&](__mmask8 used, __m512i rail) OFI_AMD_WIDE __attribute__((always_inline)) {
		return alike ? _mm512_maskz_permutexvar_epi64(used, rail, dest_keys)
			     : _mm512_mask_i64gather_epi64(zero, used, _mm512_add_epi64(dst_at, rail), keys, 8);
	};

	__m512i a[kLanes], b[kLanes], e[kLanes];
	a[0] = _mm512_or_si512(seq, _mm512_slli_epi64(nseg, 32));
	a[1] = _mm512_or_si512(_mm512_and_si512(imm, low32), _mm512_slli_epi64(n, 32));
	a[2] = _mm512_or_si512(halves, _mm512_maskz_slli_epi64(signal, rail0, 32));
	a[3] = _mm512_maskz_mov_epi64(signal, deferred);
	/* every stripe but the last has the full length; a single one has the message's, aligned or not */
	const __m512i per = _mm512_add_epi64(one, _mm512_srlv_epi64(last, _mm512_srli_epi64(n, 1)));
	__m512i stripe = _mm512_and_si512(_mm512_add_epi64(per, _mm512_set1_epi64(kStripeAlign - 1)),
					  _mm512_set1_epi64(-(long long)kStripeAlign));
	stripe = _mm512_mask_mov_epi64(stripe, single, size);
	a[4] = src;
	a[5] = _mm512_min_epu64(size, stripe);
	a[6] = dest;
	a[7] = key_of(live, rail0);
	/* the first write has a signal behind it, or a doorbell to come */
	b[0] = _mm512_or_si512(rail0, _mm512_slli_epi64(_mm512_or_si512(halves, deferred), 32));
	transpose8(a);
	if (two == 0) {
		for (uint32_t k = 0; k < kLanes; k++) {
			if (k < count) {
				char *to = reinterpret_cast<char *>(&out[k]);
				_mm512_storeu_si512(to, a[k]);
				_mm512_storeu_si512(to + 64, zero);
				_mm512_storeu_si512(to + 128, zero);
			}
		}
		alignas(64) uint64_t rail_words[kLanes];
		_mm512_store_si512(rail_words, b[0]);
		for (uint32_t k = 0; k < count; k++) {
			std::memcpy(reinterpret_cast<char *>(&out[k]) + 64, &rail_words[k], 8);
		}
	} else {
		__m512i offset = zero;
		for (uint32_t k = 1; k < OFI_AMD_MAX_NUM_RAILS; k++) {
			const __mmask8 used = k == 1 ? two : four;
			offset = _mm512_add_epi64(offset, stripe);
			const __m512i rail = _mm512_and_si512(_mm512_add_epi64(first, _mm512_set1_epi64(k)), rail_mask);
			const __m512i rest = _mm512_maskz_sub_epi64(_mm512_cmpgt_epu64_mask(size, offset), size, offset);
			__m512i x[5];
			x[0] = _mm512_maskz_add_epi64(used, src, offset);
			x[1] = _mm512_maskz_min_epu64(used, rest, stripe);
			x[2] = _mm512_maskz_add_epi64(used, dest, offset);
			x[3] = key_of(used, rail);
			x[4] = _mm512_maskz_mov_epi64(used, rail);
			for (uint32_t q = 0; q < 5; q++) {
				const uint32_t at = 1 + (k - 1) * 5 + q; /* word of b, then of e */
				(at < kLanes ? b[at] : e[at - kLanes]) = x[q];
			}
		}
		transpose8(b);
		transpose8(e);
		for (uint32_t k = 0; k < kLanes; k++) {
			if (k < count) {
				char *to = reinterpret_cast<char *>(&out[k]);
				_mm512_storeu_si512(to, a[k]);
				_mm512_storeu_si512(to + 64, b[k]);
				_mm512_storeu_si512(to + 128, e[k]);
			}
		}
	}
	if (signal == 0) {
		for (uint32_t k = 0; k < count; k++) {
			_mm256_storeu_si256(reinterpret_cast<__m256i *>(out[k].meta), _mm256_setzero_si256());
		}
	} else {
		alignas(64) uint64_t m[4][kLanes];
		const __m512i header = _mm512_or_si512(_mm512_or_si512(_mm512_set1_epi64((c->comm_id & 0x3ffu) << 2), _mm512_slli_epi64(seq, 12)),
						       _mm512_slli_epi64(_mm512_and_si512(nseg, _mm512_set1_epi64(0xf)), 25));
		const __m512i sig_at = _mm512_sub_epi64(_mm512_slli_epi64(sig_mr, 3), sig_mr);
		_mm512_store_si512(m[0], _mm512_maskz_mov_epi64(signal, header));
		_mm512_store_si512(m[1], _mm512_mask_i64gather_epi64(zero, handle, sig_at,
								     base + offsetof(ofi_amd_gin_mr_t, remote_address), 8));
		_mm512_store_si512(m[2], _mm512_maskz_mov_epi64(signal, sig_off));
		_mm512_store_si512(m[3], _mm512_maskz_mov_epi64(
						 signal, _mm512_mask_mov_epi64(sig_value, _mm512_cmpeq_epu64_mask(sop, one), one)));
		for (uint32_t k = 0; k < count; k++) {
			for (uint32_t q = 0; q < 4; q++) {
				out[k].meta[q] = m[q][k];
			}
		}
	}

	/* the communicator behind the last of them */
	c->sched.rr_small_counter = (c->sched.rr_small_counter + (uint32_t)(all_moved >> 32)) & (R - 1u);
	c->sched.rr_counter = (c->sched.rr_counter + (uint32_t)all_moved) & (R - 1u);
	c->tx_head = (head + count) & kCursorMask;
	if ((defers >> (count - 1)) & 1u) {
		alignas(64) uint64_t rails[kLanes];
		_mm512_store_si512(rails, rail0);
		c->pinned_rail_id = (int32_t)rails[count - 1];
		const uint32_t deferred_in_a_row = (uint32_t)__builtin_clz(~(defers << (32 - count)));
		c->pinned_rail_run = deferred_in_a_row == count ? run_in + count : deferred_in_a_row;
	} else {
		c->pinned_rail_id = -1;
		c->pinned_rail_run = 0;
	}
	sums->signals = (uint32_t)__builtin_popcount(signal);
	sums->writes = count + (uint32_t)__builtin_popcount(two) + 2u * (uint32_t)__builtin_popcount(four);
	return true;
}

} // namespace ofi_amd_gin

#endif
