// nrc_deal.hpp -- when an inference deals its tiles by the device count: the rule, host code alone.
#pragma once

#include <cstdint>

namespace nrc {

// Dealt by the maximum, a count below it leaves the last workgroups without work; dealt by the
// count, every wave has some.  The count is dealt where it is at most `all` (if it is above `split`)
// or at most `some` (if it is not), in tiles; every other count is dealt by the maximum.
struct DealLimits {
	uint32_t split, all, some;
};

constexpr DealLimits kDealByMaximum{0u, 0u, 0u}, kDealByCount{0u, ~0u, ~0u};

// One FP16 inference of `tiles` 64-record tiles on `waves` waves, `per_cu` of each SIMD.  Dealt by
// the maximum a wave has up to c = ceil(tiles / waves) tiles, and a SIMD per_cu c, or (per_cu - 1) c if
// the count leaves every CU a workgroup without work.  Dealt by the count a SIMD has up to
// per_cu ceil(count / waves), or one tile if there are no more tiles than SIMDs.  The count is dealt
// where that is less, or within an eighth of the waves of it: elsewhere the deal by the maximum is as
// even, and its waves, each of which reads 42 KB of weights first, are fewer.  Two workgroups a CU,
// dealt by the maximum and by the count: 700,001 of 921,600 queries 36.1 and 33.0 us, 118,000 of
// 196,608 11.1 and 9.2, 65,536 of 262,144 8.7 and 8.1; but 187,000 of 196,608 11.4 and 13.1, 482,000
// of 524,288 21.2 and 22.4, 131,072 of 262,144 8.8 and 9.4.
constexpr DealLimits infer_deal_limits(uint32_t tiles, uint32_t waves, uint32_t per_cu) {
	const uint32_t c = (tiles + waves - 1) / waves;
	if (c < 2) return kDealByMaximum;
	const uint32_t slack = waves / 8, spread = waves / per_cu, left = (per_cu - 1) * c;
	const uint32_t some = left > 0 ? (left - 1) / per_cu * waves + slack : 0u;
	return DealLimits{(uint32_t)((uint64_t)tiles * (per_cu - 1) / per_cu), (c - 1) * waves + slack, some > spread ? some : spread};
}

} // namespace nrc
