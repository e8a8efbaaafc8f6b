/*
 * prefix_plan.h - Arithmetic of the prefix sort (prefix.h) that needs no device.
 */
#pragma once

#include <cstdint>

namespace sadcs {

// Of a window of 128 bits of packed codes, `bits` a character: the bits that hold the `remaining`
// characters up to the text's end. The product is formed of fewer than 128 characters: over a whole
// text's it passes 2^32 (613,566,757 characters of 7 bits) and cut the keys there to a few bits.
constexpr uint32_t heldBits(uint32_t remaining, int bits) {
    const uint32_t held = (remaining < 128u ? remaining : 128u) * static_cast<uint32_t>(bits);
    return held < 128u ? held : 128u;
}

}  // namespace sadcs
