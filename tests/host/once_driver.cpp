/*
 * The tiles of a striping batch in one launch as far as the scheduler's counters go (csrc/sched_once.hpp), in every order in
 * which their loads, stores and atomics can come: tile 0, a tile behind it and the last one, each of which may wait for the
 * others' words or give up at any time, so also the last one done before tile 0 has begun.  Whatever the order, the counters are
 * stored once and rightly, and every tile finds the seed that the batch began with.
 */
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "sched_once.hpp"

namespace once = ofi_amd_once;

namespace {

enum rule_t {
	AS_IT_IS,
	NOT_HANDED_OVER, /* a last tile that has given up, and finds no word of tile 0, leaves the counters alone */
	NOT_MET,         /* ... and stores them all the same */
	MET_FIRST,       /* tile 0 meets the last one before its word is published */
	rules
};

struct world_t {
	uint32_t counter[2], old[2];      /* small, other; a load may still see the old one */
	uint64_t first, copy, behind, meet; /* tile 0's word and another copy of it, the tile behind it, the word in which they meet */
	int pc[3];                        /* of tile 0, the tile behind it, the last one */
	uint32_t read[3][2], seed[3], next;
	uint64_t found;
	bool stores, alone;
	int stored;
};

struct batch_t {
	uint64_t number;
	uint32_t rails, seed, total[3];
	rule_t rule;
	bool copy_first; /* of tile 0's word */
	long orders, wrong;

	uint32_t mod(uint32_t pair) const { return ((pair >> 16) % rails) << 16 | (pair & 0xffffu) % rails; }
	uint32_t sum(uint32_t a, uint32_t b) const { return mod(a + b); }

	void raise(uint64_t &word, uint64_t to) { word = word > to ? word : to; }

	void go(const world_t &w)
	{
		bool any = false;
		for (int tile = 0; tile < 3; tile++) {
			const int pc = w.pc[tile];
			if (pc < 2) { /* the counters, one after the other, perhaps as they were */
				for (int stale = 0; stale < 1 + (w.counter[pc] != w.old[pc]); stale++) {
					world_t v = w;
					v.read[tile][pc] = stale ? w.old[pc] : w.counter[pc];
					v.pc[tile]++;
					go(v);
				}
				any = true;
				continue;
			}
			const uint32_t counters = w.read[tile][0] << 16 | w.read[tile][1];
			world_t v = w;
			v.pc[tile]++;
			if (tile == 0) {
				int step = pc - 2;
				if (rule == MET_FIRST) {
					const int order[] = { 2, 0, 1, 3, 4 };
					step = step < 5 ? order[step] : step;
				}
				if (step < 2) {
					raise((step == 0) == copy_first ? v.copy : v.first, once::published_word(number, counters, total[0]));
				} else if (step == 2) {
					v.seed[0] = counters;
					v.found = w.meet;
					raise(v.meet, once::first_tile_word(number));
				} else if (step < 5 && once::first_tile_stores(w.found, number)) {
					const uint32_t to = once::counters_left(w.found);
					v.counter[step - 3] = step == 3 ? to >> 16 : to & 0xffffu;
					v.stored++;
				} else {
					continue;
				}
				go(v);
				any = true;
			} else if (tile == 1) {
				if (pc == 2) {
					v.behind = once::published_word(number, 0, total[1]);
					go(v);
				} else if (pc == 3) {
					if (once::is_published(w.copy, number)) {
						v.seed[1] = once::of_four_bits((uint32_t)w.copy >> 4 & 15u);
						go(v);
					}
					v.seed[1] = once::seed_by_itself(w.first, number, counters);
					go(v);
				} else {
					continue;
				}
				any = true;
			} else {
				const uint32_t own = total[2];
				if (pc == 2) {
					if (once::is_published(w.copy, number) && once::is_published(w.behind, number)) {
						const uint32_t before = mod(once::seed_and_total(w.copy) + once::seed_and_total(w.behind));
						v.seed[2] = once::of_four_bits((uint32_t)w.copy >> 4 & 15u);
						v.next = sum(before, own);
						v.stores = true;
						go(v);
					}
					v.seed[2] = once::seed_by_itself(w.first, number, counters);
					v.next = sum(sum(sum(v.seed[2], total[0]), total[1]), own);
					v.alone = true;
					v.stores = false;
					go(v);
				} else if (pc == 3 && w.alone) {
					if (rule == NOT_HANDED_OVER) {
						v.stores = w.first >> 8 >= number;
					} else {
						v.stores = rule == NOT_MET || once::last_tile_stores(w.meet, number);
						raise(v.meet, once::last_tile_word(number, w.next));
					}
					go(v);
				} else if (pc < 6 && (w.stores || pc == 3)) {
					if (pc > 3) {
						v.counter[pc - 4] = pc == 4 ? w.next >> 16 : w.next & 0xffffu;
						v.stored++;
					}
					go(v);
				} else {
					continue;
				}
				any = true;
			}
		}
		if (!any) {
			const uint32_t next = sum(sum(sum(seed, total[0]), total[1]), total[2]);
			orders++;
			wrong += w.stored != 2 || w.counter[0] != next >> 16 || w.counter[1] != (next & 0xffffu) || w.seed[0] != seed ||
				 w.seed[1] != seed || w.seed[2] != seed;
		}
	}
};

} // namespace

int main()
{
	std::srand(1);
	long orders[rules] = {}, wrong[rules] = {};
	for (uint32_t rule = 0; rule < rules; rule++) {
		for (int k = 0; k < (rule == AS_IT_IS ? 24 : 6); k++) {
			batch_t b = {};
			b.rule = (rule_t)rule;
			b.rails = 1 + (uint32_t)k % 4;
			b.number = k < 4 ? 1 : (1ull << 40) + (uint32_t)std::rand();
			b.copy_first = k & 4;
			auto pair = [&] { return b.mod((uint32_t)(std::rand() % 4) << 16 | (uint32_t)(std::rand() % 4)); };
			b.seed = pair();
			for (uint32_t &t : b.total) {
				t = pair();
			}
			world_t w = {};
			w.counter[0] = w.old[0] = b.seed >> 16;
			w.counter[1] = w.old[1] = b.seed & 0xffffu;
			/* what the batch before has left, or the one that cleared the scratch */
			for (uint64_t *word : { &w.first, &w.copy, &w.behind, &w.meet }) {
				*word = b.number == 1 ? 0 : (b.number - 1) << 8 | (uint32_t)(std::rand() & 255);
			}
			b.go(w);
			orders[rule] += b.orders;
			wrong[rule] += b.wrong;
		}
		std::printf("rule %u: %ld orders, %ld wrong\n", rule, orders[rule], wrong[rule]);
	}
	bool ok = wrong[AS_IT_IS] == 0;
	for (uint32_t rule = 1; rule < rules; rule++) {
		ok &= wrong[rule] != 0; /* the model sees what is wrong with the others */
	}
	std::printf(ok ? "ok\n" : "failed\n");
	return ok ? 0 : 1;
}
