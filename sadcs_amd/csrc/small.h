/*
 * small.h - Texts of at most kSmallMax bytes: the whole construction in one workgroup's LDS.
 *
 * A small text does not fill the chip, and the phases (ranking, classes, merge) cost it about a
 * hundred launches of a few microseconds each. Here one workgroup builds one text's suffix array
 * and BWT, and a batch of small texts is one launch with a workgroup per text:
 *  - The text's bytes get dense codes 1..sigma (0: past the end) and are packed into a bit stream,
 *    most significant bit first, so any run of its bits compares as the text does.
 *  - The suffixes are sorted by their first 8 * passes stream bits with a stable LSD radix sort
 *    whose digits come straight from the stream (no key array).
 *  - Suffixes still sharing a rank are split by prefix doubling: the order by the rank h further on
 *    is the current order with every position moved back by h (positions past the last h first),
 *    so a round only sorts that order by the suffixes' own ranks, two digit passes. A round ends
 *    the loop when every rank is its own.
 * Suffix indices and ranks are 16-bit, so a text of n bytes needs about 7.2 n bytes of LDS.
 *
 * What bounds it: the barriers and LDS round trips of one workgroup's digit passes, and for a host
 * call the call's own launch and wait. Measured (host calls, SA + BWT, phases against this): 4099
 * bytes of protein 507 to 74 us; 512 documents of 200 B to 16 KiB in one batch 10.9 to 2.4 ms.
 */
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include "dev_common.h"

namespace sadcs {

// The largest text whose arrays fit the LDS of a CU beside the counters: 16384 bytes take 127 KB of
// 160. Alone at that size, from host memory, against a byte more by the prefix sort: protein-like 0.14 and
// 0.24 ms, DNA-like 0.44 and 0.53, periodic 0.45 and 0.66, but Markov 0.57 and 0.33; what a text is like is
// not known here, and a batch of such texts has a workgroup for each (4096 of Markov text 2.4 ms, by the tile
// merge 6.9).
constexpr uint32_t kSmallMax = 16384;
constexpr int kSmallBins = 256;

// LDS of a workgroup of `threads` for texts of up to `capacity` bytes (a multiple of 64).
inline size_t smallSharedBytes(uint32_t capacity, int threads) {
    return (9 * static_cast<size_t>(capacity) / 32 + 6) * sizeof(uint32_t) + 3 * static_cast<size_t>(capacity) * sizeof(uint16_t) +
           static_cast<size_t>(threads / kWave) * kSmallBins * sizeof(uint16_t);
}

template <int kThreads, int kItems>
struct SmallSorter {
    static constexpr int kWaves = kThreads / kWave;
    uint16_t* counts;      // [kWaves][kSmallBins]
    uint32_t* waveSums;    // [kSmallBins / kWave]

    // Stable sort of source(0..total) (kept entries only, `total` up to kItems * kThreads) by digit:
    // source(k, value, digit) gives entry k's value and digit and whether it is kept (asked
    // twice). The kept values go to dst in order. Every thread calls it; it begins and ends with a barrier.
    template <class Source>
    __device__ __forceinline__ void pass(uint32_t total, uint16_t* dst, Source source) const {
        const uint32_t wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
        __syncthreads();
        for (uint32_t x = threadIdx.x; x < kWaves * kSmallBins / 2; x += kThreads) {
            reinterpret_cast<uint32_t*>(counts)[x] = 0;
        }
        __syncthreads();
        const uint32_t rows = (total + kThreads - 1) / kThreads;  // 64-entry rows per wave
        const uint32_t first = wave * rows * kWave + lane;
        uint16_t* mine = counts + wave * kSmallBins;
        uint32_t ranks[kItems / 2];  // two 16-bit ranks each
#pragma unroll
        for (int j = 0; j < kItems; j++) {
            if (static_cast<uint32_t>(j) < rows) {
                const uint32_t k = first + j * kWave;
                uint32_t v = 0, d = 0;
                const bool valid = k < total && source(k, v, d);
                const uint64_t peers = matchDigit<8>(d, valid);
                const uint32_t before = valid ? mine[d] : 0;
                const uint32_t rank = before + countBelow(peers);
                ranks[j / 2] = (j & 1) ? ranks[j / 2] | rank << 16 : rank;
                if (valid && lane == static_cast<uint32_t>(__builtin_ctzll(peers))) {
                    mine[d] = static_cast<uint16_t>(before + __builtin_popcountll(peers));
                }
            }
        }
        __syncthreads();
        // Thread d: the waves' prefixes of digit d, then the digits' starts.
        uint32_t sum = 0;
        if (threadIdx.x < kSmallBins) {
            for (int w = 0; w < kWaves; w++) {
                const uint32_t c = counts[w * kSmallBins + threadIdx.x];
                counts[w * kSmallBins + threadIdx.x] = static_cast<uint16_t>(sum);
                sum += c;
            }
            const uint32_t inclusive = waveInclusive<OpSum>(sum);
            if (lane == kWave - 1) {
                waveSums[wave] = inclusive;
            }
            sum = inclusive - sum;
        }
        __syncthreads();
        if (threadIdx.x < kSmallBins) {
            for (uint32_t w = 0; w < wave; w++) {
                sum += waveSums[w];
            }
            for (int w = 0; w < kWaves; w++) {
                counts[w * kSmallBins + threadIdx.x] += static_cast<uint16_t>(sum);
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kItems; j++) {
            if (static_cast<uint32_t>(j) < rows) {
                const uint32_t k = first + j * kWave;
                uint32_t v = 0, d = 0;
                if (k < total && source(k, v, d)) {
                    dst[mine[d] + (ranks[j / 2] >> (16 * (j & 1)) & 0xFFFFu)] = static_cast<uint16_t>(v);
                }
            }
        }
        __syncthreads();
    }
};

// One workgroup per text. Text s is bytes [segments[s].start, .end) of `text`; its outputs start
// at row segments[s].rowBase of sa (positions in the text) and bwt, either of which may be null;
// firstRows[s] is the row of its suffix 0, rounds[s] its doubling rounds: a word a text, since both lie in
// host memory, where a maximum over the texts was one compare-and-swap after another across the bus
// (1.18 us a text: 16,000 texts of 1 KiB on the device 18.9 ms, 1.35 without). `capacity` is a
// multiple of 64 at least as long as every text. kItems * kThreads >= 2 * capacity (a doubling round
// walks up to twice the text).
template <int kThreads, int kItems>
__global__ __launch_bounds__(kThreads) void smallTextsKernel(const uint8_t* __restrict__ text, const Segment* __restrict__ segments, uint32_t capacity, uint32_t* __restrict__ sa, uint8_t* __restrict__ bwt, uint32_t* __restrict__ firstRows, uint32_t* __restrict__ rounds) {
    using Sorter = SmallSorter<kThreads, kItems>;
    constexpr int kWaves = kThreads / kWave;
    constexpr int kHalf = kItems / 2;  // 64-entry rows per wave of one walk of the text
    extern __shared__ __align__(16) unsigned char shared[];
    uint32_t* stream = reinterpret_cast<uint32_t*>(shared);
    uint16_t* saA = reinterpret_cast<uint16_t*>(stream + 9 * capacity / 32 + 6);
    uint16_t* saB = saA + capacity;
    uint16_t* rank = saB + capacity;
    __shared__ uint32_t waveSums[kSmallBins / kWave];
    __shared__ uint16_t code[kSmallBins];
    __shared__ uint8_t byteOf[kSmallBins + 1];
    __shared__ uint8_t present[kSmallBins];
    __shared__ uint32_t waveLast[kWaves], waveHeads[kWaves];
    __shared__ uint32_t firstRow;
    const Sorter sorter{rank + capacity, waveSums};

    const uint32_t tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
    const Segment segment = segments[blockIdx.x];
    const uint32_t n = min(segment.end - segment.start, capacity);
    const uint8_t* bytes = text + segment.start;
    uint8_t* raw = reinterpret_cast<uint8_t*>(saB);  // the bytes, until the stream holds them

    // Dense codes.
    for (uint32_t x = tid; x < kSmallBins; x += kThreads) {
        present[x] = 0;
    }
    __syncthreads();
    for (uint32_t i = tid; i < n; i += kThreads) {
        const uint8_t b = bytes[i];
        raw[i] = b;
        present[b] = 1;
    }
    __syncthreads();
    uint32_t below = 0;
    bool mineOccurs = false;
    if (tid < kSmallBins) {
        mineOccurs = present[tid] != 0;
        const uint64_t mask = ballot(mineOccurs);
        below = countBelow(mask);
        if (lane == 0) {
            waveSums[wave] = static_cast<uint32_t>(__builtin_popcountll(mask));
        }
    }
    __syncthreads();
    uint32_t sigma = 0;
    for (uint32_t w = 0; w < kSmallBins / kWave; w++) {
        below += w < wave ? waveSums[w] : 0;
        sigma += waveSums[w];
    }
    if (tid < kSmallBins && mineOccurs) {
        code[tid] = static_cast<uint16_t>(below + 1);
        byteOf[below + 1] = static_cast<uint8_t>(tid);
    }
    __syncthreads();

    // The stream: word w holds stream bits [32w, 32w + 32), bit 0 first from the top.
    const uint32_t bits = 32 - __clz(max(sigma, 1u));
    const uint32_t words = (n * bits + 31) / 32 + 4;  // zeros past the end: code 0
    for (uint32_t w = tid; w < words; w += kThreads) {
        uint32_t value = 0;
        for (uint32_t i = 32 * w / bits; i < n && i * bits < 32 * w + 32; i++) {
            const int shift = static_cast<int>(32 * w + 32) - static_cast<int>((i + 1) * bits);
            const uint32_t c = code[raw[i]];
            value |= shift >= 0 ? c << shift : c >> -shift;
        }
        stream[w] = value;
    }
    auto bitsAt = [&](uint32_t at) -> uint32_t {  // 32 stream bits from bit `at`
        const uint32_t w = at >> 5;
        return static_cast<uint32_t>(((static_cast<uint64_t>(stream[w]) << 32 | stream[w + 1]) << (at & 31)) >> 32);
    };

    // The first sort. 48 bits separate the suffixes of most texts of this size (16 characters of
    // DNA); shorter texts need fewer.
    const uint32_t passes = n > 2048 ? 6 : n > 256 ? 5 : 4;
    uint16_t* cur = saA;
    uint16_t* other = saB;
    for (uint32_t k = passes; k-- > 0;) {
        const bool firstPass = k + 1 == passes;
        const uint16_t* from = cur;
        sorter.pass(n, other, [&](uint32_t e, uint32_t& value, uint32_t& digit) {
            value = firstPass ? e : from[e];
            digit = bitsAt(value * bits + 8 * k) >> 24;
            return true;
        });
        uint16_t* t = cur;
        cur = other;
        other = t;
    }

    // Ranks: entry k's is the index of the first entry it ties with (the last head at or before
    // k). equalsPrevious(i, j) tells whether adjacent suffixes i and j still tie; it may read the
    // ranks that this replaces. Returns the number of heads.
    const uint32_t rows = (n + kThreads - 1) / kThreads;
    const uint32_t first = wave * rows * kWave + lane;
    auto assignRanks = [&](auto equalsPrevious) -> uint32_t {
        uint64_t heads[kHalf];
        uint32_t last = 0, count = 0;
#pragma unroll
        for (int j = 0; j < kHalf; j++) {
            if (static_cast<uint32_t>(j) < rows) {
                const uint32_t k = first + j * kWave;
                const bool head = k < n && (k == 0 || !equalsPrevious(cur[k], cur[k - 1]));
                heads[j] = ballot(head);
                count += static_cast<uint32_t>(__builtin_popcountll(heads[j]));
                if (heads[j]) {
                    last = first - lane + j * kWave + 63 - static_cast<uint32_t>(__builtin_clzll(heads[j]));
                }
            }
        }
        if (lane == 0) {
            waveLast[wave] = last;  // heads ascend along the waves, so 0 (no head) never wins the max below
            waveHeads[wave] = count;
        }
        __syncthreads();
        uint32_t carry = 0, total = 0;
        for (uint32_t w = 0; w < kWaves; w++) {
            carry = w < wave ? max(carry, waveLast[w]) : carry;
            total += waveHeads[w];
        }
#pragma unroll
        for (int j = 0; j < kHalf; j++) {
            if (static_cast<uint32_t>(j) < rows) {
                const uint32_t base = first - lane + j * kWave;
                const uint64_t upTo = heads[j] & (~uint64_t(0) >> (63 - lane));
                const uint32_t id = upTo ? base + 63 - static_cast<uint32_t>(__builtin_clzll(upTo)) : carry;
                if (base + lane < n) {
                    rank[cur[base + lane]] = static_cast<uint16_t>(id);
                }
                if (heads[j]) {
                    carry = base + 63 - static_cast<uint32_t>(__builtin_clzll(heads[j]));
                }
            }
        }
        __syncthreads();
        return total;
    };

    const uint32_t lowBits = 8 * passes - 32;  // of the second word compared: 0, 8 or 16
    uint32_t heads = assignRanks([&](uint32_t i, uint32_t j) {
        return bitsAt(i * bits) == bitsAt(j * bits) &&
               (lowBits == 0 || (bitsAt(i * bits + 32) ^ bitsAt(j * bits + 32)) >> (32 - lowBits) == 0);
    });

    // Prefix doubling: tied suffixes share h characters.
    uint32_t h = 8 * passes / bits, doublings = 0;
    while (heads < n && h < n) {
        const uint16_t* order = cur;
        // Entry e of the order by the rank h further on: the last h suffixes, then the others.
        auto moved = [&](uint32_t e, uint32_t& value) {
            value = e < h ? n - h + e : static_cast<uint32_t>(order[e - h]) - h;
            return e < h || order[e - h] >= h;
        };
        sorter.pass(n + h, other, [&](uint32_t e, uint32_t& value, uint32_t& digit) {
            const bool kept = moved(e, value);
            digit = kept ? rank[value] & 255u : 0u;
            return kept;
        });
        uint16_t* sorted = other;
        if (n > 256) {
            const uint16_t* from = other;
            sorted = cur;
            sorter.pass(n, sorted, [&](uint32_t e, uint32_t& value, uint32_t& digit) {
                value = from[e];
                digit = rank[value] >> 8;
                return true;
            });
        }
        other = sorted == cur ? other : cur;
        cur = sorted;
        auto second = [&](uint32_t i) -> uint32_t { return i + h < n ? rank[i + h] + 1u : 0u; };
        heads = assignRanks([&](uint32_t i, uint32_t j) { return rank[i] == rank[j] && second(i) == second(j); });
        h *= 2;
        doublings++;
    }

    for (uint32_t k = tid; k < n; k += kThreads) {
        const uint32_t p = cur[k];
        if (p == 0) {
            firstRow = k;
        }
        if (sa) {
            sa[segment.rowBase + k] = p;
        }
    }
    __syncthreads();
    const uint32_t firstAt = firstRow;
    if (tid == 0) {
        firstRows[blockIdx.x] = firstAt;
        rounds[blockIdx.x] = doublings;
    }
    if (bwt) {
        auto byteAt = [&](uint32_t i) -> uint8_t { return byteOf[bitsAt(i * bits) >> (32 - bits)]; };
        // Byte 0 is the text's last; the row of suffix 0 has none.
        for (uint32_t k = tid; k < n; k += kThreads) {
            const uint32_t p = cur[k];
            if (p != 0) {
                bwt[segment.rowBase + (k < firstAt ? k + 1 : k)] = byteAt(p - 1);
            }
        }
        if (tid == 0) {
            bwt[segment.rowBase] = byteAt(n - 1);
        }
    }
}

}  // namespace sadcs
