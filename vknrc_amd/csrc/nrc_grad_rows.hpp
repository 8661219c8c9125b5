// nrc_grad_rows.hpp -- one gradient row a workgroup or two: the rule, host code alone.
#pragma once

#include <cstdint>

namespace nrc {

// A cache's rows in a gradient launch, and the 64-record chunks of one.
struct GradRows {
	uint32_t rows, chunks;
};

// The end of a launch whose workgroups, each of `per_group` rows of one cache, go in order to
// whichever CU is free first and take base + per_chunk x chunks there.  CUs that are free at the
// same time are one level, and a cache splits one level at most, so there are at most n + 1.
template <uint32_t MAX> inline uint32_t grad_launch_end(const GradRows *items, uint32_t n, uint32_t cus, uint32_t per_group,
                                                        uint32_t base, uint32_t per_chunk) {
	struct Level {
		uint32_t free_at, cus;
	} level[MAX + 2] = {{0u, cus}}; // earliest first
	uint32_t levels = 1, end = 0;
	for (uint32_t i = 0; i < n && i < MAX; ++i) {
		uint32_t groups = (items[i].rows + per_group - 1) / per_group;
		while (groups > 0) {
			const uint32_t take = groups < level[0].cus ? groups : level[0].cus;
			const uint32_t done = level[0].free_at + base + per_chunk * items[i].chunks;
			groups -= take;
			end = done > end ? done : end;
			if (take == level[0].cus) {
				--levels;
				for (uint32_t j = 0; j < levels; ++j) level[j] = level[j + 1];
			} else {
				level[0].cus -= take;
			}
			uint32_t at = 0;
			while (at < levels && level[at].free_at < done) ++at;
			if (at < levels && level[at].free_at == done) {
				level[at].cus += take;
				continue;
			}
			for (uint32_t j = levels; j > at; --j) level[j] = level[j - 1];
			level[at] = Level{done, take};
			++levels;
		}
	}
	return end;
}

// Whether the rows of a launch with multi-chunk rows run two a workgroup (fused_grad_dual_kernel)
// rather than one (fused_grad_small_kernel); either gives the same bits.  A CU holds one workgroup
// of either kind.  A row of c chunks takes 7.2 + 4.4 c us, a pair of them 8.6 + 7.2 c (c = 1..16, one
// cache kind, up to 256 rows): in units of 0.88 us 8 + 5 c and 10 + 8 c, which the launch is dealt
// with.  Pairs must win by a tenth, since full rounds of them, which store the sums of up to 512
// rows at once, take up to 6 us more.  So with rows of one length, pairs run where they save a
// round in three: 320 and 384 rows of 8 chunks 84 -> 68 and 69 us, 384 of 2 chunks 31.5 -> 26.2;
// not up to one row a CU, nor for 560 to 640 rows (three rounds against two: of 2 chunks 47 us
// single, 50 in pairs).  Where lengths differ, the longest rows set the end and a pair of them ends
// later: 256 rows of one chunk and 32 of eight, 53.6 us as single rows and 65.9 as pairs; 16 rows
// of 16 chunks and 768 of 2, 77.5 and 123.0.  Of 113 launches measured both ways the rule takes the
// slower kind by more than 3 % four times (6 % at most), and never pairs that are slower than the
// single rows.
template <uint32_t MAX> inline bool grad_rows_in_pairs(const GradRows *items, uint32_t n, uint32_t cus) {
	uint32_t rows = 0;
	for (uint32_t i = 0; i < n; ++i) rows += items[i].rows;
	if (rows <= cus) return false; // one round of single rows
	const uint32_t single = grad_launch_end<MAX>(items, n, cus, 1u, 8u, 5u);
	const uint32_t pairs = grad_launch_end<MAX>(items, n, cus, 2u, 10u, 8u);
	return 10u * pairs < 9u * single;
}

} // namespace nrc
