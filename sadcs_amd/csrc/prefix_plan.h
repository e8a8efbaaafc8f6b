/*
 * prefix_plan.h - Arithmetic of the prefix sort (prefix.h) that needs no device.
 */
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace sadcs {

// Of a window of 128 bits of packed codes, `bits` a character: the bits that hold the `remaining`
// characters up to the text's end. The product is formed of fewer than 128 characters: over a whole
// text's it passes 2^32 (613,566,757 characters of 7 bits) and cut the keys there to a few bits.
constexpr uint32_t heldBits(uint32_t remaining, int bits) {
    const uint32_t held = (remaining < 128u ? remaining : 128u) * static_cast<uint32_t>(bits);
    return held < 128u ? held : 128u;
}

// ---- ties ---------------------------------------------------------------------------------------

constexpr uint32_t kTieGroupMax = 24;  // rows of a group compared in LDS

// Of the 32 rows whose tie bits are `own` (bit r: row r ties with the row before; `next`: the 32 rows
// after), the part of the count of rows in groups of more than kTieGroupMax: a group of g such rows has
// g - 24 rows with 24 tied ones after them, the first of which is the group's head.
constexpr uint32_t largeTieRows(uint32_t own, uint32_t next) {
    static_assert(kTieGroupMax == 24, "runs of 16 + 8 bits");
    const uint64_t after = (static_cast<uint64_t>(next) << 32 | own) >> 1;
    const uint64_t two = after & after >> 1, four = two & two >> 2, eight = four & four >> 4;
    const uint32_t rows = static_cast<uint32_t>(eight & eight >> 8 & eight >> 16);
    return static_cast<uint32_t>(__builtin_popcount(rows)) + kTieGroupMax * static_cast<uint32_t>(__builtin_popcount(rows & ~own));
}

// What a sample says of the rows that tie, before any row is sorted: the share of all rows, and how many
// a group has, as if all groups were of one size.
struct TieEstimate {
    double share;
    double groupRows;
};

// Of `sampled` keys, drawn at `density` a row, `repeated` equal another one and `runs` two others or more.
// A row of a group of g meets x others of its group with the probability of a Poisson variable of mean
// m = density * (g - 1): 1 - e^-m of them at least one, and of those 1 - m / (e^m - 1) two or more. Beyond
// 12 that is all but one in 13,000, too few to tell sizes apart: larger groups count as of 12 / density rows.
inline TieEstimate estimateTies(double sampled, double repeated, double runs, double density) {
    if (repeated <= 0 || sampled <= 0) {
        return {0, 1};
    }
    const double ratio = runs / repeated;
    double low = 0, high = 12;
    for (int i = 0; i < 40; i++) {
        const double m = (low + high) / 2;
        (1 - m / std::expm1(m) < ratio ? low : high) = m;
    }
    const double m = std::max(low, density);  // two rows at least
    return {std::min(1.0, repeated / sampled / -std::expm1(-m)), 1 + m / density};
}

}  // namespace sadcs
