/*
 * The words in which the tiles of a striping batch in one launch (stripe_once_kernel, sched_stripe.hip) tell each other what
 * they know, and who of them moves the scheduler's counters on.  Plain functions of the words' values: the kernel
 * puts them between its loads and atomics, and a model on the CPU between its own, in every order.
 *
 * - Every word carries its batch's number, which no other batch on the scratch has, and only ever grows.
 * - A tile reads the counters before it publishes its total.  Tile 0's word also says what the counters were (the seed).
 * - A tile that waits in vain for the words before it reads the counters first and the first copy of tile 0's word second.  If
 *   the word is there, the seed is the word's, for the counters may have been moved on; if not, they have not been.
 * - The last tile moves the counters on by itself when it has seen the words of all the others: they have read them.  When
 *   it has waited in vain, it meets tile 0 in a word of their own: tile 0 says there that the first copy of its word is
 *   published, the last tile what the counters are to be, and whoever comes second stores them.  Neither waits.
 */
#ifndef OFI_AMD_SCHED_ONCE_HPP_
#define OFI_AMD_SCHED_ONCE_HPP_

#include <cstdint>

namespace ofi_amd_once {

/* a pair of residues or counters, as the packed sums have them, in four bits, and back */
constexpr uint32_t four_bits(uint32_t pair)
{
	return (pair >> 16) << 2 | (pair & 3u);
}
constexpr uint32_t of_four_bits(uint32_t bits)
{
	return (bits >> 2 & 3u) << 16 | (bits & 3u);
}

/* a tile's word; seed: tile 0's, of the others 0 */
constexpr uint64_t published_word(uint64_t number, uint32_t seed, uint32_t total)
{
	return number << 8 | four_bits(seed) << 4 | four_bits(total);
}
constexpr bool is_published(uint64_t word, uint64_t number)
{
	return word >> 8 == number;
}
/* what a published word adds to the sum over the tiles before */
constexpr uint32_t seed_and_total(uint64_t word)
{
	return of_four_bits((uint32_t)word & 15u) + of_four_bits((uint32_t)word >> 4 & 15u);
}
/* the seed of a tile that has waited in vain: `counters` as it has read them before the first copy of tile 0's word */
constexpr uint32_t seed_by_itself(uint64_t first_word, uint64_t number, uint32_t counters)
{
	return is_published(first_word, number) ? of_four_bits((uint32_t)first_word >> 4 & 15u) : counters;
}

/* What tile 0 and the last tile put into the word in which they meet (the larger one stays), and what each makes of what it
 * has found there.  A larger number is another batch's, which has overlapped with this one against the rule. */
constexpr uint64_t first_tile_word(uint64_t number)
{
	return number << 8;
}
constexpr uint64_t last_tile_word(uint64_t number, uint32_t counters)
{
	return number << 8 | four_bits(counters);
}
constexpr bool first_tile_stores(uint64_t found, uint64_t number)
{
	return found >> 8 == number;
}
constexpr uint32_t counters_left(uint64_t found)
{
	return of_four_bits((uint32_t)found & 15u);
}
constexpr bool last_tile_stores(uint64_t found, uint64_t number)
{
	return found >> 8 >= number;
}

} // namespace ofi_amd_once

#endif
