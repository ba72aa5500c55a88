/*
 * derive8 (gin_derive8.hpp) against derive<true>, one descriptor after another: groups of one to eight descriptors of a
 * communicator, records, communicator, checksum words and counts alike, or nothing changed where derive8 hands them back.
 * Then the drain that uses it (mode 2) against the one that does not (mode 3, which folds every record into its checksum).
 */
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "gin_derive8.hpp"
#include "gin_rings.hpp"

using namespace ofi_amd_gin;

static std::mt19937_64 rng(20240607);
static uint64_t below(uint64_t n) { return rng() % n; }

static uint64_t fold(const ofi_amd_gin_desc_t *d)
{
	uint64_t w[8], x = 0;
	std::memcpy(w, d, sizeof(w));
	for (int k = 0; k < 8; k++) {
		x += (w[k] + (uint64_t)(k + 1)) * kFoldKeys[k];
	}
	return x;
}

/* rings of 256 slots whose positions begin in front of a lap's end, of 2^32 or anywhere, filled with `ops` descriptors each */
struct rings_t : ofi_amd_gin_rings {
	std::vector<ofi_amd_gin_desc_t> rec;
	std::vector<uint32_t> seq, deq;
	rings_t(const std::vector<ofi_amd_gin_desc_t> &stream, uint32_t contexts, uint32_t ops, uint32_t start)
	    : ofi_amd_gin_rings{}, rec(contexts * 256), seq(contexts * 256), deq(contexts, start)
	{
		n_contexts = contexts, capacity = 256, records = rec.data(), sequences = seq.data(), dequeue_pos = deq.data();
		for (uint32_t c = 0; c < contexts; c++) {
			for (uint32_t k = 0; k < 256; k++) {
				const uint32_t at = start + k;
				seq[c * 256 + (at & 255)] = k < ops ? at + 1 : at;
				if (k < ops) {
					rec[c * 256 + (at & 255)] = stream[c * ops + k];
				}
			}
		}
	}
};

static bool drains()
{
	ofi_amd_gin_mr_t mrs[3];
	for (auto &mr : mrs) {
		mr.local_base = rng(), mr.remote_address = rng(), mr.remote_address_offset = rng();
		for (auto &key : mr.key) {
			key = rng();
		}
	}
	for (int round = 0; round < 400; round++) {
		/* every twentieth or so with more records than a thread by itself keeps in its caches */
		const uint32_t contexts = round % 20 == 0 ? 90 : 1 + (uint32_t)below(5), ops = round % 20 == 0 ? 250 : 1 + (uint32_t)below(256);
		const uint32_t threads = 1 + (uint32_t)below(3), offset = (uint32_t)below(9) * 8; /* of the records in their array */
		const uint32_t start = below(3) == 0 ? (uint32_t)rng() : below(2) ? 0u - 1u - (uint32_t)below(200) : 250;
		const bool faulty = below(4) == 0, regions_alike = below(2);
		std::vector<ofi_amd_gin_desc_t> stream(contexts * ops);
		for (auto &x : stream) {
			std::memset(&x, 0, sizeof(x));
			x.src_off = rng(), x.dst_off = rng(), x.signal_off = rng(), x.signal_value = rng();
			x.size = below(30) == 0 ? 0 : 1 + below(1u << (3 + below(18)));
			x.opt_flags = (uint32_t)below(2);
			x.src_mr = regions_alike ? 0 : (uint16_t)below(3), x.dst_mr = regions_alike ? 1 : (uint16_t)below(3);
			x.sig_mr = 0xffff, x.kind = below(40) == 0 ? OFI_AMD_GIN_KIND_GET : OFI_AMD_GIN_KIND_PUT;
			if (x.kind == OFI_AMD_GIN_KIND_PUT && below(20) == 0) {
				x.signal_op = 1 + (uint32_t)below(2), x.sig_mr = 2, x.kind = OFI_AMD_GIN_KIND_PUT_SIGNAL;
			}
		}
		if (faulty) {
			ofi_amd_gin_desc_t &wrong = stream[below(stream.size())];
			wrong.src_mr = 3, wrong.size = 1 + below(1000); /* without a payload nobody looks at the handle */
		}
		std::vector<ofi_amd_gin_comm_t> comms[2];
		/* a line more on either side, which has to stay as it is */
		std::vector<unsigned char> wires[2];
		ofi_amd_gin_proxy_stats_t st[2];
		int rc[2];
		for (int run = 0; run < 2; run++) {
			rings_t r(stream, contexts, ops, start);
			for (uint32_t c = 0; c < contexts; c++) {
				comms[run].emplace_back();
				ofi_amd_gin_comm_init(&comms[run].back(), c, 4, 131072, 64, 1);
				/* half of them come to where ACKs are asked for */
				comms[run].back().tx_head = 3900, comms[run].back().tx_tail = round % 2 ? 3900 : 0;
			}
			wires[run].assign(stream.size() * sizeof(ofi_amd_gin_wire_t) + 256, 0xee);
			unsigned char *at = wires[run].data() + 64;
			at += (64 - (reinterpret_cast<uintptr_t>(at) & 63)) & 63;
			std::memset(&st[run], 0, sizeof(st[run]));
			rc[run] = ofi_amd_gin_proxy_drain_mt(&r, ops, run == 0 ? 2 : 3, nullptr, comms[run].data(), mrs, 3,
							      reinterpret_cast<ofi_amd_gin_wire_t *>(at + offset), 10, threads, &st[run]);
			if (rc[run] == 0) {
				for (uint32_t c = 0; c < contexts; c++) {
					for (uint32_t k = 0; k < 256; k++) {
						const uint32_t pos = start + k;
						if (r.seq[c * 256 + (pos & 255)] != (k < ops ? pos + 256 : pos) || r.deq[c] != start + ops) {
							std::printf("round %d: slot %u of context %u is not the producer's\n", round, k, c);
							return false;
						}
					}
				}
			}
			/* where the array began */
			std::memmove(wires[run].data(), at - 64, wires[run].size() - 128);
			wires[run].resize(wires[run].size() - 128);
		}
		bool same = rc[0] == rc[1] && rc[0] == (faulty ? -EINVAL : 0);
		same &= comms[0].size() == comms[1].size() && (threads > 1 && faulty ? true :
			(wires[0] == wires[1] && st[0].descriptors == st[1].descriptors && st[0].writes == st[1].writes &&
			 std::memcmp(comms[0].data(), comms[1].data(), comms[0].size() * sizeof(comms[0][0])) == 0));
		if (!same) {
			std::printf("round %d: %u contexts of %u, %u threads, start %u, offset %u: the drains differ (%d %d)\n", round, contexts, ops,
				    threads, start, offset, rc[0], rc[1]);
			return false;
		}
		if (!faulty) {
			rings_t r(stream, contexts, ops, start);
			ofi_amd_gin_proxy_stats_t plain;
			ofi_amd_gin_proxy_drain_mt(&r, ops, 0, nullptr, nullptr, nullptr, 0, nullptr, 10, 1, &plain);
			if (plain.checksum != st[0].checksum || plain.signals != st[0].signals) {
				std::printf("round %d: checksum or signals differ from the plain drain's\n", round);
				return false;
			}
		}
	}
	return true;
}

int main()
{
	if (!cpu_has_wide()) {
		std::printf("skip\n");
		return 0;
	}
	const uint32_t n_mrs = 5;
	ofi_amd_gin_mr_t mrs[n_mrs];
	for (auto &mr : mrs) {
		mr.local_base = rng(), mr.remote_address = rng(), mr.remote_address_offset = rng();
		for (auto &key : mr.key) {
			key = rng();
		}
	}
	const uint64_t edges[] = { 1, 2, 63, 64, 65, 127, 128, 129, 131072, 131073, 262144, 262145, 393216, 393217, 1ull << 32,
				   (1ull << 63) + 1, ~0ull - 128, ~0ull - 127, ~0ull - 1, ~0ull };
	uint64_t together = 0, handed_back = 0, longest_run = 0;
	for (int stream = 0; stream < 6000; stream++) {
		const uint32_t rails = 1u << below(3), ack_model = (uint32_t)below(2);
		ofi_amd_gin_comm_t c = {};
		c.sched.num_rails = (int32_t)rails;
		c.sched.min_stripe_size = 1ull << (below(4) == 0 ? below(64) : 17);
		c.sched.max_small_msg_size = below(3) == 0 ? below(1 << 20) : below(2) * 64;
		c.sched.rr_small_counter = (uint32_t)below(rails), c.sched.rr_counter = (uint32_t)below(rails);
		c.comm_id = (uint32_t)(below(4) == 0 ? rng() : below(1024)), c.num_rails = rails, c.ack_model = ack_model;
		c.tx_head = (uint32_t)below(1u << 14);
		c.tx_tail = (c.tx_head - (uint32_t)(below(3) == 0 ? below(4096) : 4040 + below(60))) & kCursorMask;
		if (below(2) == 0) {
			c.tx_tail = c.tx_head;
		}
		c.pinned_rail_id = below(2) ? -1 : (int32_t)below(rails);
		c.pinned_rail_run = (uint32_t)(below(8) == 0 ? below(40) : below(16));
		c.next_rail_id = (uint32_t)below(rails);
		const uint64_t aggregates = below(4), signals = below(3), odd = below(8) == 0 ? 3 : 400, sizes = below(3);
		for (int group = 0; group < 40; group++) {
			ofi_amd_gin_desc_t d[8];
			const uint32_t n = below(2) ? 8 : 1 + (uint32_t)below(8);
			for (auto &x : d) {
				std::memset(&x, 0, sizeof(x));
				x.src_off = rng(), x.dst_off = rng(), x.signal_off = rng(), x.signal_value = rng();
				x.size = sizes == 0 ? edges[below(sizeof(edges) / 8)] : sizes == 1 ? 1 + below(1u << (3 + below(18))) : rng() >> below(64);
				x.size += x.size == 0;
				x.rank = (uint32_t)rng(), x.context = (uint32_t)rng();
				x.opt_flags = (uint32_t)rng() & ~1u;
				x.opt_flags |= aggregates == 0 ? 0 : aggregates == 1 ? 1 : aggregates == 2 ? (uint32_t)below(2) : (uint32_t)(below(12) != 0);
				x.src_mr = (uint16_t)below(n_mrs), x.dst_mr = (uint16_t)below(n_mrs), x.sig_mr = 0xffff, x.kind = OFI_AMD_GIN_KIND_PUT;
				if (signals == 2 || (signals == 1 && below(9) == 0)) {
					x.signal_op = 1 + (uint32_t)below(2), x.kind = OFI_AMD_GIN_KIND_PUT_SIGNAL;
					x.sig_mr = below(4) == 0 ? 0xffff : (uint16_t)below(n_mrs);
				}
				if (below(odd) == 0) {
					switch (below(6)) {
					case 0: x.size = 0; break;
					case 1: x.src_mr = (uint16_t)(n_mrs + below(3)); break;
					case 2: x.dst_mr = (uint16_t)(n_mrs + below(3)); break;
					case 3: x.signal_op = 3 + (uint32_t)below(3); break;
					case 4: x.signal_op = 1, x.sig_mr = n_mrs; break;
					default: x.sig_mr = n_mrs; break; /* of no signal: nobody looks */
					}
				}
			}
			if (!derive_fast_path(&c)) {
				std::printf("not a fast path\n");
				return 1;
			}
			ofi_amd_gin_comm_t one = c, eight = c;
			ofi_amd_gin_wire_t want[8], got[8];
			std::memset(want, 0xee, sizeof(want));
			std::memset(got, 0xee, sizeof(got));
			derived8_t sums;
			const bool did = derive8(&eight, mrs, n_mrs, d, n, got, &sums);
			uint32_t k = 0, seen_signals = 0, writes = 0, acks = 0;
			for (; k < n; k++) {
				if (derive<true>(&one, mrs, n_mrs, &d[k], &want[k]) != 0) {
					break;
				}
				seen_signals += d[k].signal_op != 0, writes += want[k].num_writes, acks += want[k].ack_req;
				longest_run = one.pinned_rail_run > longest_run ? one.pinned_rail_run : longest_run;
			}
			bool same;
			if (did) {
				together++;
				same = k == n && acks == 0 && std::memcmp(want, got, sizeof(want)) == 0 && std::memcmp(&one, &eight, sizeof(one)) == 0 &&
				       sums.signals == seen_signals && sums.writes == writes;
				for (uint32_t j = 0; j < n; j++) {
					same &= sums.folds[j] == fold(&d[j]);
				}
			} else {
				handed_back++;
				same = std::memcmp(&eight, &c, sizeof(c)) == 0 && (unsigned char)got[0].seq == 0xee;
			}
			if (!same) {
				std::printf("stream %d group %d of %u: derive8 %s\n", stream, group, n, did ? "differs" : "left something behind");
				return 1;
			}
			c = one;
			if (k < n) { /* the window is full, or a descriptor is wrong */
				c.tx_tail = c.tx_head;
			}
		}
	}
	if (!drains()) {
		return 1;
	}
	std::printf("ok: %llu groups together, %llu handed back, runs up to %llu\n", (unsigned long long)together,
		    (unsigned long long)handed_back, (unsigned long long)longest_run);
	return together > 100000 && handed_back > 1000 && longest_run >= 15 ? 0 : 1;
}
