/*
 * Host side of the GIN descriptor path: ring push/pop with the slot protocol of
 * include/nccl_ofi_mpsc_ring.h:56-163 and the proxy loop that drains all rings and
 * hands each descriptor to the wire derivation of gin_wire.cpp.
 */
#include <algorithm>
#include <cerrno>
#include <chrono>
#include <thread>
#include <vector>
#include <cstring>

#include <emmintrin.h>

#include "gin_derive8.hpp"
#include "gin_rings.hpp"

namespace {

inline uint64_t rotl64(uint64_t x, int k) { return (x << k) | (x >> (64 - k)); }

inline uint64_t fold_sum(uint64_t h, uint64_t x) { return (rotl64(h, 5) ^ x) * 0x100000001B3ull; }

/* Order-sensitive fold of n 64-bit words into a running per-context hash. */
inline uint64_t fold_words(uint64_t h, const uint64_t *w, int n)
{
	uint64_t x = 0;
	for (int k = 0; k < n; k++) {
		x += (w[k] + (uint64_t)(k + 1)) * ofi_amd_gin::kFoldKeys[k & 7];
	}
	return fold_sum(h, x);
}

/* n records past the caches, in order; both 16-byte aligned */
inline void stream_records(ofi_amd_gin_wire_t *to, const ofi_amd_gin_wire_t *from, uint32_t n)
{
	static_assert(sizeof(ofi_amd_gin_wire_t) % 32 == 0, "whole pairs of 16-byte words");
	const __m128i *s = reinterpret_cast<const __m128i *>(from);
	__m128i *d = reinterpret_cast<__m128i *>(to);
	for (uint32_t k = 0; k < n * (sizeof(ofi_amd_gin_wire_t) / 16); k += 2) {
		const __m128i a = _mm_load_si128(s + k), b = _mm_load_si128(s + k + 1);
		_mm_stream_si128(d + k, a);
		_mm_stream_si128(d + k + 1, b);
	}
}

/* ... by whole lines of `to`, but for its ends */
OFI_AMD_WIDE inline void stream_records_wide(ofi_amd_gin_wire_t *to, const ofi_amd_gin_wire_t *from, uint32_t n)
{
	const char *s = reinterpret_cast<const char *>(from);
	char *d = reinterpret_cast<char *>(to), *const end = d + n * sizeof(*to);
	auto words = [&](char *until) {
		for (; d < until; d += 16, s += 16) {
			_mm_stream_si128(reinterpret_cast<__m128i *>(d), _mm_load_si128(reinterpret_cast<const __m128i *>(s)));
		}
	};
	words(std::min(end, d + ((64 - (reinterpret_cast<uintptr_t>(d) & 63)) & 63)));
	for (; end - d >= 64; d += 64, s += 64) {
		_mm512_stream_si512(reinterpret_cast<__m512i *>(d), _mm512_loadu_si512(s));
	}
	words(end);
}

constexpr uint32_t kGroup = 16;  /* descriptors looked at and handed on together */
constexpr uint32_t kStaged = 64; /* records of a thread's own array, 14 KiB */
constexpr uint64_t kCachedRecords = 20000; /* 4.5 MB */

struct burst_t {
	uint32_t done; /* descriptors derived */
	int rc;        /* 0, or why the next one could not be */
};

/*
 * Derives up to `limit` published descriptors of one ring, from position `start` on, to the records at `out`, or round
 * `staged` when there is no `out`.  What bounds it is the core: some 250 instructions a descriptor one by one, two of their
 * branches by its size, and the descriptor's line, which comes from memory.  WIDE: eight at a time (derive8), and one by one
 * only the groups that it hands back; one thread, no output array 12.5 -> 5.5 ns a descriptor.  The communicator lives in a
 * copy: one by one its address goes nowhere, so that its fields are registers or stack words, not loads and stores
 * through a pointer that may alias the records, and the derivation is inlined (four threads, no output array: 16.8 -> 14.4 ns).
 * STREAM: records are made in `staged`, which stays in the first-level cache, and leave by groups past the caches: an
 * ordinary store fetches every line of the array first, from memory or from whichever core read it last.  256,000
 * records (57 MB) on four threads, descriptors produced ahead: ordinary 1.3-1.6 ms one by one, streamed 1.03, WIDE 0.61
 * (the stores alone take four threads 0.36); 32,000 (7 MB) that another thread reads between the calls 461 -> 175 us one by one.
 */
template <bool STREAM, bool WIDE>
burst_t derive_burst(const uint32_t *seq, const ofi_amd_gin_desc_t *rec, uint32_t mask, uint32_t start, uint32_t limit,
		     ofi_amd_gin_comm_t *comm, const ofi_amd_gin_mr_t *mrs, uint32_t n_mrs, ofi_amd_gin_wire_t *out,
		     ofi_amd_gin_wire_t *staged, bool fold_wires, uint64_t *hash, ofi_amd_gin_proxy_stats_t *st)
{
	ofi_amd_gin_comm_t c = *comm;
	uint32_t tail = 0, pending = 0;
	/* What an ACK changes is taken up with every group and given back only where the derivation changed it: the thread
	 * that receives ACKs may apply one meanwhile (ofi_amd_gin_apply_ack), also while there is nothing to derive. */
	auto take_acks = [&] {
		c.tx_tail = tail = __atomic_load_n(&comm->tx_tail, __ATOMIC_RELAXED);
		c.has_pending_ack_request = pending = __atomic_load_n(&comm->has_pending_ack_request, __ATOMIC_RELAXED);
	};
	auto give_back = [&] {
		comm->sched = c.sched;
		comm->tx_head = c.tx_head;
		comm->consecutive_puts_without_ack = c.consecutive_puts_without_ack;
		comm->last_ack_requested_seq = c.last_ack_requested_seq;
		comm->pinned_rail_id = c.pinned_rail_id;
		comm->pinned_rail_run = c.pinned_rail_run;
		comm->next_rail_id = c.next_rail_id;
		if (c.tx_tail != tail) {
			__atomic_store_n(&comm->tx_tail, c.tx_tail, __ATOMIC_RELAXED);
		}
		if (c.has_pending_ack_request != pending) {
			__atomic_store_n(&comm->has_pending_ack_request, c.has_pending_ack_request, __ATOMIC_RELAXED);
		}
	};
	uint64_t h = *hash, signals = 0, writes = 0;
	burst_t b = { 0, 0 };
	while (b.done < limit && b.rc == 0) {
		const uint32_t most = limit - b.done < kGroup ? limit - b.done : kGroup;
		uint32_t ready = 0;
		while (ready < most && __atomic_load_n(&seq[(start + b.done + ready) & mask], __ATOMIC_ACQUIRE) ==
					       start + b.done + ready + 1) {
			ready++;
		}
		if (ready == 0) {
			break;
		}
		take_acks();
		uint32_t k = 0, singly = 0; /* singly: those before it are derived one by one */
		while (k < ready) {
			const uint32_t at = start + b.done + k;
			const ofi_amd_gin_desc_t *d = &rec[at & mask];
			if (WIDE && k >= singly) {
				/* up to the ring's end */
				const uint32_t m = std::min({ ready - k, ofi_amd_gin::kLanes, mask + 1 - (at & mask) });
				for (uint32_t j = 0; j < m; j++) {
					__builtin_prefetch(&rec[(at + kGroup + j) & mask]);
				}
				ofi_amd_gin_wire_t *wires = STREAM || !out ? &staged[k] : &out[b.done + k];
				ofi_amd_gin::derived8_t sums;
				if (ofi_amd_gin::derive8(&c, mrs, n_mrs, d, m, wires, &sums)) {
					__asm__ volatile("" : : "r"(wires) : "memory"); /* as below */
					for (uint32_t j = 0; j < m; j++) {
						h = fold_sum(h, sums.folds[j]);
					}
					signals += sums.signals;
					writes += sums.writes;
					k += m;
					continue;
				}
				singly = k + m;
			}
			__builtin_prefetch(&rec[(at + kGroup) & mask]);
			/* the slot is handed back only after this burst, so the record is read in place */
			ofi_amd_gin_wire_t *wire = STREAM ? &staged[k] : (out ? &out[b.done + k] : &staged[at % kStaged]);
			h = fold_words(h, reinterpret_cast<const uint64_t *>(d), 8);
			signals += d->signal_op != 0;
			if (__builtin_expect(d->kind != OFI_AMD_GIN_KIND_GET, 1)) {
				b.rc = ofi_amd_gin::derive<true>(&c, mrs, n_mrs, d, wire);
			} else {
				comm->sched = c.sched; /* all that a get changes */
				b.rc = ofi_amd_gin_iget(comm, mrs, n_mrs, d, wire);
				c.sched = comm->sched;
			}
			if (b.rc != 0) {
				break;
			}
			/* the record is complete in memory here, whoever reads it next: the compiler may
			 * not keep it in registers or drop stores to fields this loop does not read */
			__asm__ volatile("" : : "r"(wire) : "memory");
			writes += wire->num_writes;
			if (fold_wires) {
				h = fold_words(h, reinterpret_cast<const uint64_t *>(wire), (int)(sizeof(*wire) / 8));
			}
			k++;
		}
		give_back();
		if (STREAM) {
			/* the record of a descriptor that failed, which is all zero, too */
			(WIDE ? stream_records_wide : stream_records)(out + b.done, staged, k + (b.rc != 0));
		}
		b.done += k;
		if (ready < most) {
			break;
		}
	}
	*hash = h;
	st->signals += signals;
	st->writes += writes;
	return b;
}

} // namespace

extern "C" {

/* nccl_ofi_mpsc_ring::push, include/nccl_ofi_mpsc_ring.h:79-118 */
int ofi_amd_gin_ring_push(ofi_amd_gin_rings_t *r, uint32_t context, const ofi_amd_gin_desc_t *desc)
{
	if (!r || context >= r->n_contexts || !desc) {
		return -EINVAL;
	}
	const uint32_t mask = r->capacity - 1;
	uint32_t *enq = &r->enqueue_pos[context * 16];
	uint32_t *seq = r->sequences + (size_t)context * r->capacity;
	ofi_amd_gin_desc_t *rec = r->records + (size_t)context * r->capacity;

	uint32_t pos = __atomic_load_n(enq, __ATOMIC_RELAXED);
	for (;;) {
		const uint32_t s = __atomic_load_n(&seq[pos & mask], __ATOMIC_ACQUIRE);
		const int32_t diff = (int32_t)s - (int32_t)pos;
		if (diff == 0) {
			if (__atomic_compare_exchange_n(enq, &pos, pos + 1, true, __ATOMIC_RELAXED,
							__ATOMIC_RELAXED)) {
				break;
			}
		} else if (diff < 0) {
			return 0; /* full */
		} else {
			pos = __atomic_load_n(enq, __ATOMIC_RELAXED);
		}
	}
	rec[pos & mask] = *desc;
	__atomic_store_n(&seq[pos & mask], pos + 1, __ATOMIC_RELEASE);
	return 1;
}

/* nccl_ofi_mpsc_ring::pop, :124-144 */
int ofi_amd_gin_ring_pop(ofi_amd_gin_rings_t *r, uint32_t context, ofi_amd_gin_desc_t *desc)
{
	if (!r || context >= r->n_contexts || !desc) {
		return -EINVAL;
	}
	const uint32_t mask = r->capacity - 1;
	uint32_t *seq = r->sequences + (size_t)context * r->capacity;
	const uint32_t pos = r->dequeue_pos[context];
	if (__atomic_load_n(&seq[pos & mask], __ATOMIC_ACQUIRE) != pos + 1) {
		return 0;
	}
	*desc = r->records[(size_t)context * r->capacity + (pos & mask)];
	r->dequeue_pos[context] = pos + 1;
	__atomic_store_n(&seq[pos & mask], pos + r->capacity, __ATOMIC_RELEASE);
	return 1;
}

/*
 * A call has one thread more for every so many descriptors, up to the number asked for: starting threads takes some 20 us.  Us
 * for a call that may have four, with one for every 2000 / for every 3000, descriptors produced ahead, without an output
 * array and with one:
 *    2400 descriptors   35 and 35 (two threads)    17 and 19 (one)
 *    4800               40 and 41 (three)          36 and 38 (two)
 *    8000               55 and 57 (four)           52 and 57 (three)
 *   12,800              63 and 74 (four)           63 and 74 (four)
 * Derived one by one, 2000 are worth a thread: 6000 on all four 38 and 54, 4000 on three 40 and 44, on four 42 and 38.
 */
static constexpr uint64_t kOpsPerThread = 3000, kOpsPerThreadSingly = 2000;

/* One proxy thread's share: contexts [c_begin, c_end). */
static int drain_contexts(ofi_amd_gin_rings_t *r, uint32_t c_begin, uint32_t c_end,
			  uint64_t ops_per_context, int mode, ofi_amd_gin_desc_t *out_desc,
			  ofi_amd_gin_comm_t *comms, const ofi_amd_gin_mr_t *mrs, uint32_t n_mrs,
			  ofi_amd_gin_wire_t *out_wire, bool alone, uint32_t timeout_ms,
			  ofi_amd_gin_proxy_stats_t *stats)
{
	using clock = std::chrono::steady_clock;
	const uint32_t nctx = c_end - c_begin, cap = r->capacity, mask = cap - 1;
	const uint32_t burst = cap / 2 < 1024 ? cap / 2 : 1024;

	uint64_t *done = new (std::nothrow) uint64_t[nctx]();
	uint64_t *hash = new (std::nothrow) uint64_t[nctx];
	if (!done || !hash) {
		delete[] done;
		delete[] hash;
		return -ENOMEM;
	}
	for (uint32_t k = 0; k < nctx; k++) {
		hash[k] = 0x9E3779B97F4A7C15ull ^ (c_begin + k);
	}
	/* without an output array the records go round this one (it stays in the core's cache), where a post step would
	 * pick them up */
	alignas(64) ofi_amd_gin_wire_t staged[kStaged];
	/* A thread that is the only one of its call stores through the caches while they hold the records: 2.9 MB of them WIDE 84-100
	 * us, streamed 94, 3.6 MB 108-118 and 126, 5.4 MB 203-217 and 183-193, 14 MB 607 and 440; one by one at every size 13.4 ns a
	 * descriptor, streamed 14.6.  (The line fetches that streaming saves cost most when another core has read the array
	 * since, 30-50 ns against 15, which is not known here.) */
	const bool wide = mode == 2 && ofi_amd_gin::cpu_has_wide();
	const bool fits = !wide || ops_per_context <= kCachedRecords / nctx;
	const bool stream = out_wire && !(alone && fits) && (reinterpret_cast<uintptr_t>(out_wire) & 15u) == 0;

	ofi_amd_gin_proxy_stats_t st;
	std::memset(&st, 0, sizeof(st));
	uint64_t remaining = (uint64_t)nctx * ops_per_context;
	int rc = 0;
	const auto t0 = clock::now();
	auto last_progress = t0;
	uint32_t idle_rounds = 0;

	while (remaining > 0) {
		bool progressed = false;
		for (uint32_t k = 0; k < nctx; k++) {
			if (done[k] >= ops_per_context) {
				continue;
			}
			const uint32_t c = c_begin + k;
			uint32_t *seq = r->sequences + (size_t)c * cap;
			const ofi_amd_gin_desc_t *rec = r->records + (size_t)c * cap;
			const uint32_t start = r->dequeue_pos[c];
			uint32_t pos = start;
			const uint64_t want = ops_per_context - done[k], first = (uint64_t)c * ops_per_context + done[k];
			const uint32_t limit = want < burst ? (uint32_t)want : burst;
			uint64_t h = hash[k];

			/* whether the fast form applies is constant over the burst: the derivation keeps the counters below
			 * the rail count */
			if (mode >= 2 && ofi_amd_gin::derive_fast_path(&comms[c])) {
				const burst_t b = (wide ? (stream ? derive_burst<true, true> : derive_burst<false, true>)
							: (stream ? derive_burst<true, false> : derive_burst<false, false>))(
					seq, rec, mask, start, limit, &comms[c], mrs, n_mrs, out_wire ? out_wire + first : nullptr, staged,
					mode == 3, &h, &st);
				pos = start + b.done;
				rc = b.rc;
			} else {
				while (pos - start < limit &&
				       __atomic_load_n(&seq[pos & mask], __ATOMIC_ACQUIRE) == pos + 1) {
					const ofi_amd_gin_desc_t *d = &rec[pos & mask];
					h = fold_words(h, reinterpret_cast<const uint64_t *>(d), 8);
					st.signals += d->signal_op != 0;
					if (mode == 1) {
						out_desc[first + (pos - start)] = *d;
					} else if (mode >= 2) {
						ofi_amd_gin_wire_t *wire = out_wire ? &out_wire[first + (pos - start)] : &staged[pos % kStaged];
						rc = ofi_amd_gin_derive(&comms[c], mrs, n_mrs, d, wire);
						if (rc != 0) {
							break;
						}
						st.writes += wire->num_writes;
						if (mode == 3) {
							h = fold_words(h, reinterpret_cast<const uint64_t *>(wire),
								       (int)(sizeof(*wire) / 8));
						}
					}
					pos++;
				}
			}
			if (pos != start) {
				/* hand the slots back in position order (pop, :139-143) */
				for (uint32_t p = start; p != pos; p++) {
					__atomic_store_n(&seq[p & mask], p + cap, __ATOMIC_RELEASE);
				}
				r->dequeue_pos[c] = pos;
				done[k] += pos - start;
				remaining -= pos - start;
				st.descriptors += pos - start;
				hash[k] = h;
				progressed = true;
			} else {
				st.empty_polls++;
			}
			if (rc != 0) {
				break;
			}
		}
		if (rc != 0) {
			break;
		}
		if (progressed) {
			idle_rounds = 0;
			last_progress = clock::now();
		} else if (++idle_rounds >= 64) {
			idle_rounds = 0;
			const auto now = clock::now();
			if (std::chrono::duration_cast<std::chrono::milliseconds>(now - last_progress).count() >
			    (long long)timeout_ms) {
				rc = -ETIMEDOUT;
				break;
			}
		}
	}
	if (stream) {
		_mm_sfence(); /* the streamed records before whatever tells others that they are there */
	}
	st.seconds = std::chrono::duration<double>(clock::now() - t0).count();
	for (uint32_t k = 0; k < nctx; k++) {
		st.checksum += hash[k];
	}
	*stats = st;
	delete[] done;
	delete[] hash;
	return rc;
}

int ofi_amd_gin_proxy_drain_mt(ofi_amd_gin_rings_t *r, uint64_t ops_per_context, int mode,
			       ofi_amd_gin_desc_t *out_desc, ofi_amd_gin_comm_t *comms,
			       const ofi_amd_gin_mr_t *mrs, uint32_t n_mrs, ofi_amd_gin_wire_t *out_wire,
			       uint32_t timeout_ms, uint32_t n_threads, ofi_amd_gin_proxy_stats_t *stats)
{
	if (!r || mode < 0 || mode > 3 || (mode == 1 && !out_desc) ||
	    (mode >= 2 && (!comms || !mrs || n_mrs == 0)) ||
	    n_threads < 1 || n_threads > 64) {
		return -EINVAL;
	}
	const uint32_t nctx = r->n_contexts;
	uint32_t workers = n_threads < nctx ? n_threads : nctx;
	const uint64_t per_thread = mode == 2 && ofi_amd_gin::cpu_has_wide() ? kOpsPerThread : kOpsPerThreadSingly;
	if (ops_per_context < per_thread) { /* each context is not worth a thread by itself */
		const uint64_t worth = nctx * ops_per_context / per_thread + 1;
		workers = worth < workers ? (uint32_t)worth : workers;
	}
	std::vector<ofi_amd_gin_proxy_stats_t> part(workers);
	std::vector<int> rcs(workers, 0);
	const auto t0 = std::chrono::steady_clock::now();
	auto share = [&](uint32_t w) {
		/* contiguous ranges of contexts, sizes differing by at most one */
		const uint32_t lo = (uint32_t)((uint64_t)nctx * w / workers);
		const uint32_t hi = (uint32_t)((uint64_t)nctx * (w + 1) / workers);
		rcs[w] = drain_contexts(r, lo, hi, ops_per_context, mode, out_desc, comms, mrs, n_mrs, out_wire,
					workers == 1, timeout_ms, &part[w]);
	};
	try {
		std::vector<std::thread> threads;
		for (uint32_t w = 1; w < workers; w++) {
			threads.emplace_back(share, w);
		}
		share(0); /* the calling thread is a proxy thread too */
		for (auto &t : threads) {
			t.join();
		}
	} catch (...) {
		return -ENOMEM;
	}
	ofi_amd_gin_proxy_stats_t st;
	std::memset(&st, 0, sizeof(st));
	int rc = 0;
	for (uint32_t w = 0; w < workers; w++) {
		st.descriptors += part[w].descriptors;
		st.signals += part[w].signals;
		st.writes += part[w].writes;
		st.checksum += part[w].checksum;
		st.empty_polls += part[w].empty_polls;
		if (rcs[w] != 0 && rc == 0) {
			rc = rcs[w];
		}
	}
	st.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
	if (stats) {
		*stats = st;
	}
	return rc;
}

int ofi_amd_gin_proxy_drain(ofi_amd_gin_rings_t *r, uint64_t ops_per_context, int mode,
			    ofi_amd_gin_desc_t *out_desc, ofi_amd_gin_comm_t *comms,
			    const ofi_amd_gin_mr_t *mrs, uint32_t n_mrs, ofi_amd_gin_wire_t *out_wire,
			    uint32_t timeout_ms, ofi_amd_gin_proxy_stats_t *stats)
{
	return ofi_amd_gin_proxy_drain_mt(r, ops_per_context, mode, out_desc, comms, mrs, n_mrs, out_wire,
					  timeout_ms, 1, stats);
}

} /* extern "C" */
