/*
 * prefix.h - The prefix-sort path: every suffix sorted by its first characters in two bucket
 * passes and one LDS sort, and only the suffixes that still tie compared by the sample's ranks.
 *
 * The tile merge (merge.h) reads one random 128-byte line per suffix and compares it three times,
 * whatever the text. Most suffixes of most texts differ within the 8 to 24 characters that fit a
 * 56-bit key, and a key read from the text in position order costs no random access at all:
 *  1. Splitters: the keys of a sample of positions, sorted; every kOversample-th one (kCoarseOversample
 *     of a short text) bounds a leaf of about kLeafTarget suffixes, so leaves are even whatever the
 *     text's distribution.
 *  2. The records (key, position) are scattered into buckets straight from the text, the buckets
 *     into leaves, each time staged in LDS in bucket order so that a bucket's records leave in
 *     runs. Where memory does not hold every record, a round takes the buckets that fit and the
 *     text is read again for the next.
 *  3. One workgroup sorts a leaf in LDS and writes its rows of the suffix array, the BWT bytes (the
 *     character before a suffix rides in its key's low byte) and a tie bit for every row whose
 *     key equals the row's before.
 *  4. The sample suffixes are read off the rows in order; their ties are split further (rank.h),
 *     which gives every sample suffix its rank.
 *  5. Rows that tie are put in order by the difference cover's comparison. Groups of up to
 *     kTieGroupMax rows are compared in LDS; larger ones (runs, high-copy repeats) go through the
 *     tile merge as class lists of their own.
 * Texts too many of whose suffixes tie keep the tile merge alone, by what the sample shows of them: near-
 * copies in large numbers, long runs, and ties whose lists the memory planned for the call does not hold.
 *
 * Measured against the tile merge (SA + BWT on the device): 1 GiB of Markov text 100.1 to 58.7 ms,
 * 256 MiB of DNA-like text 31.8 to 18.6 ms (cover 128: 87.2 to 18.6), 16 MiB of uniform ACGT at
 * cover 128 4.06 to 0.95 ms, 1024 texts of 1 KiB to 4 MiB in one batch 62.5 to 40.1 ms.
 */
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include "dev_common.h"
#include "merge.h"
#include "prefix_plan.h"
#include "prim.h"
#include "rank.h"

namespace sadcs {

constexpr int kPrefixThreads = 512;
constexpr int kPrefixItems = 8;
constexpr uint32_t kPrefixBlock = kPrefixThreads * kPrefixItems;  // positions or records placed at once
constexpr int kPrefixKeyBits = 56;       // of a record's 64: the low byte is the character before
constexpr int kPrefixMaxChars = 24;      // characters of a key (one thread's window is 8 + 23 of them)
constexpr uint32_t kPrefixMaxBuckets = 2048;       // first-level buckets
constexpr uint32_t kPrefixMaxRoundBuckets = 512;   // of them in one round (their tables share the LDS with the records)
constexpr uint32_t kPrefixMaxBins = 512;           // leaves of a bucket
// Records of a leaf on average, the most its workgroup sorts in LDS, and sampled keys per leaf: a
// leaf's size spreads by a sixth around its average, and one of twice that without equal keys is
// about one in 200,000. Leaves of 1024 in 27 KB, five workgroups a CU, sort 1 GiB in 12.3 ms;
// 1536 in 40 KB 14.2, 1536 in 53 KB 18.4. Beyond 2^30 rows the most leaves there are hold up to 2048.
constexpr uint32_t kLeafTarget = 1024;
constexpr uint32_t kLeafCapacity = 2048;
constexpr uint32_t kOversample = 32;
// Up to about 2.3 million rows: leaves of 512 to 1536 on average (about 512 of them while that
// holds: every CU has leaves to sort, and a small one sorts sooner), of up to 4096, 16 keys a leaf.
constexpr uint32_t kSmallLeaf = 512;
constexpr uint32_t kCoarseLeaf = 1536;
constexpr uint32_t kCoarseOversample = 16;
constexpr uint64_t kLeafTieShare = 16;             // at most 1 / this of the sample in groups of half a leaf
// The most of the rows, as the sample has it, in groups beyond kTieGroupMax, of long texts (from kLongTies
// rows on) and of shorter ones, whose time is more in launches. Such a row costs 0.34 ns as a class list
// entry; the tile merge of the whole text costs 0.04 ns a row more than the other steps here. Protein-like
// text with near-copies of a piece, prefix sort and tile merge: 48 MiB, 0.1 of it 6.1 and 7.3 ms, 0.2 8.3
// and 7.9, 0.5 15.0 and 9.6; 0.7 MB, 0.2 of it 0.86 and 0.95 ms, 0.4 1.11 and 1.10.
constexpr double kLargeTieShare = 0.125, kLargeTieShareShort = 0.5;
constexpr uint64_t kLongTies = uint64_t(1) << 23;

// A suffix on its way to its row: its key (the character before it in the low byte) and position, 12
// bytes together, so that a run of records is one run of memory: keys and positions apart wrote a
// third more lines.
struct PrefixRecord {
    uint32_t low, high, position;
};

__device__ __forceinline__ PrefixRecord packRecord(uint64_t key, uint32_t position) {
    return PrefixRecord{static_cast<uint32_t>(key), static_cast<uint32_t>(key >> 32), position};
}

__device__ __forceinline__ uint64_t keyOf(const PrefixRecord& r) {
    return static_cast<uint64_t>(r.high) << 32 | r.low;
}

__device__ __forceinline__ uint64_t keyPart(uint64_t key) {
    return key & ~uint64_t(0xFF);
}

// How a position's key is built: the text's index (a batch), then `chars` codes of `charBits` bits
// from the top down, zeros past the text's end. A batch's texts may pack their own codes.
struct PrefixText {
    const uint64_t* words;       // the text, padded with zero words
    uint32_t span;
    int segmentBits;
    int charBits, chars;
    bool wide;                   // all 256 bytes occur: the code is the byte plus one
    const uint8_t* textCodes;    // a batch's own codes (256 per text), or null
    const uint8_t* textShape;    // their width and characters per key (2 per text)
};

// The key of position p (its low byte 0); `code` is the common code table.
template <class Texts>
__device__ __forceinline__ uint64_t prefixKey(const PrefixText& pt, const Texts& texts, const uint8_t* code, uint32_t p) {
    const uint32_t segment = texts.segmentOf(p);
    const uint32_t end = texts.endOf(p);
    const uint8_t* table = code;
    int bits = pt.charBits, chars = pt.chars;
    if (Texts::kBatch && pt.textCodes) {
        table = pt.textCodes + static_cast<size_t>(segment) * 256;
        bits = pt.textShape[2 * segment];
        chars = pt.textShape[2 * segment + 1];
    }
    const uint32_t remaining = p < end ? end - p : 0;
    uint64_t key = 0;
    for (int c0 = 0; c0 < chars; c0 += 8) {
        uint64_t w = static_cast<uint32_t>(c0) < remaining ? load8(pt.words, p + c0) : 0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t byte = static_cast<uint32_t>(w >> 56);
            w <<= 8;
            const uint32_t ch = static_cast<uint32_t>(c0 + j) < remaining ? (pt.wide ? byte + 1 : table[byte]) : 0u;
            key = c0 + j < chars ? (key << bits) | ch : key;
        }
    }
    key <<= 64 - pt.segmentBits - chars * bits;
    return Texts::kBatch && pt.segmentBits ? key | static_cast<uint64_t>(segment) << (64 - pt.segmentBits) : key;
}

// A text's alphabet in LDS for prefixKey.
__device__ __forceinline__ void loadCodes(const CodeTable& codes, uint8_t* code) {
    for (uint32_t x = threadIdx.x; x < 256; x += blockDim.x) {
        code[x] = codes.code[x];
    }
    __syncthreads();
}

// ---- splitters ------------------------------------------------------------------------------------

// Key i of the sample: a position drawn from the i-th of `count` equal parts of the span. Positions
// between a batch's texts give ~0, which sorts last and is left out. places[i] = 0, for countSampleKernel.
template <class Texts>
__global__ __launch_bounds__(256) void samplePrefixesKernel(PrefixText pt, Texts texts, CodeTable codes, uint32_t count, uint64_t* __restrict__ keys, uint32_t* __restrict__ places) {
    __shared__ uint8_t code[256];
    loadCodes(codes, code);
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) {
        return;
    }
    places[i] = 0;
    const uint64_t lo = static_cast<uint64_t>(pt.span) * i / count, hi = static_cast<uint64_t>(pt.span) * (i + 1) / count;
    uint32_t h = i * 0x9E3779B9u;
    h ^= h >> 15;
    h *= 0x85EBCA6Bu;
    h ^= h >> 13;
    const uint32_t p = static_cast<uint32_t>(lo + (hi > lo ? h % (hi - lo) : 0));
    keys[i] = p < texts.endOf(p) ? prefixKey(pt, texts, code, p) : ~uint64_t(0);
}

// A sample of up to kSampleCountMax keys is sorted by counting: a key's place is the number of keys
// before it in (key, index) order, 64 keys a wave against a part of the others each, whose keys the
// wave reads through scalar loads. Three launches, where the radix sort of so few takes thirty: at
// 8192 keys 15 against 110 us; at 32768 the comparisons alone would take 80.
constexpr uint32_t kSampleCountMax = 24576;
constexpr uint32_t kSampleParts = 16;

__global__ __launch_bounds__(256) void countSampleKernel(const uint64_t* __restrict__ keys, uint32_t count, uint32_t* __restrict__ places) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) / kWave);
    const uint32_t groups = (count + kWave - 1) / kWave;
    if (wave >= groups * kSampleParts) {
        return;
    }
    const uint32_t part = wave / groups;
    const uint32_t i = wave % groups * kWave + threadIdx.x % kWave;
    const uint64_t own = keys[min(i, count - 1)];
    const uint32_t first = static_cast<uint32_t>(static_cast<uint64_t>(count) * part / kSampleParts);
    const uint32_t last = static_cast<uint32_t>(static_cast<uint64_t>(count) * (part + 1) / kSampleParts);
    // Keys before the wave's own 64 count when equal, those after do not.
    const uint32_t group = wave % groups * kWave, groupEnd = group + kWave;
    uint32_t smaller = 0;
#pragma unroll 8
    for (uint32_t j = first; j < min(last, group); j++) {
        smaller += keys[j] <= own ? 1 : 0;
    }
    for (uint32_t j = max(first, group); j < min(last, groupEnd); j++) {
        const uint64_t other = keys[j];
        smaller += other < own || (other == own && j < i) ? 1 : 0;
    }
#pragma unroll 8
    for (uint32_t j = max(first, groupEnd); j < last; j++) {
        smaller += keys[j] < own ? 1 : 0;
    }
    if (i < count && smaller) {
        atomicAdd(&places[i], smaller);
    }
}

__global__ __launch_bounds__(256) void placeSampleKernel(const uint64_t* __restrict__ keys, const uint32_t* __restrict__ places, uint32_t count, uint64_t* __restrict__ sorted) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) {
        sorted[min(places[i], count - 1)] = keys[i];
    }
}

// splitters[x] (x in [0, leaves - 1)) = the sorted sample's key at (x + 1) / leaves of its valid
// part. seen counts sampled keys: [0] equal to the one kCoarseOversample places on (a group of that key holds
// about half a leaf of rows or more), [1] equal to another, [2] to two others or more.
__global__ __launch_bounds__(256) void pickSplittersKernel(const uint64_t* __restrict__ sorted, uint32_t count, uint32_t leaves, uint64_t* __restrict__ splitters, uint32_t* __restrict__ seen) {
    uint32_t lo = 0, hi = count;  // the valid keys come before the ~0 ones
    while (lo < hi) {
        const uint32_t mid = (lo + hi) / 2;
        if (sorted[mid] != ~uint64_t(0)) {
            lo = mid + 1;
        } else {
            hi = mid;
        }
    }
    __shared__ uint32_t all[3];
    if (threadIdx.x < 3) {
        all[threadIdx.x] = 0;
    }
    __syncthreads();
    uint32_t counts[3] = {};
    for (uint32_t x = blockIdx.x * blockDim.x + threadIdx.x; x < max(count, leaves); x += gridDim.x * blockDim.x) {
        if (x + 1 < leaves) {
            splitters[x] = lo > 0 ? sorted[static_cast<uint64_t>(lo) * (x + 1) / leaves] : ~uint64_t(0);
        }
        if (x < lo) {
            const uint64_t own = sorted[x], far = sorted[min(x + kCoarseOversample, lo - 1)];
            const uint64_t after = sorted[min(x + 1, lo - 1)], after2 = sorted[min(x + 2, lo - 1)];
            const uint64_t before = sorted[max(x, 1u) - 1], before2 = sorted[max(x, 2u) - 2];
            const bool a1 = x + 1 < lo && after == own, b1 = x > 0 && before == own;
            counts[0] += x + kCoarseOversample < lo && far == own ? 1 : 0;
            counts[1] += (a1 | b1) ? 1 : 0;
            counts[2] += ((a1 & b1) | (x + 2 < lo && after2 == own) | (x > 1 && before2 == own)) ? 1 : 0;
        }
    }
#pragma unroll
    for (int k = 0; k < 3; k++) {
        for (int offset = kWave / 2; offset > 0; offset /= 2) {
            counts[k] += __shfl_xor(counts[k], offset);
        }
        if (threadIdx.x % kWave == 0 && counts[k]) {
            atomicAdd(&all[k], counts[k]);
        }
    }
    __syncthreads();
    if (threadIdx.x < 3 && all[threadIdx.x]) {
        atomicAdd(&seen[threadIdx.x], all[threadIdx.x]);
    }
}

// ---- keys of a block of positions -----------------------------------------------------------------

// LDS of blockKeys: every thread's eight codes, packed, and three more for the last threads' windows;
// and the code tables: the common one, or one per 256 positions (a batch's texts start on such
// boundaries).
template <bool kBatch>
struct BlockCodes {
    static constexpr uint32_t kTables = kBatch ? kPrefixBlock / 256 + 1 : 1;
    uint64_t packed[kPrefixThreads + 4];
    alignas(16) uint8_t table[kTables][256];
    uint32_t tableText[kTables];  // a batch: the text whose codes a table holds
};

template <class Texts>
__device__ __forceinline__ void initBlockCodes(const PrefixText& pt, const CodeTable& common, BlockCodes<Texts::kBatch>& s) {
    for (uint32_t x = threadIdx.x; x < BlockCodes<Texts::kBatch>::kTables * 256; x += kPrefixThreads) {
        s.table[x / 256][x % 256] = common.code[x % 256];
    }
    if (threadIdx.x < BlockCodes<Texts::kBatch>::kTables) {
        s.tableText[threadIdx.x] = ~0u;
    }
    __syncthreads();
}

// A thread's text of a block, read ahead of its use: its eight bytes, the eight of the block after
// (threads 0 to 2) and the byte before (a wave's first lane; the others have it from their neighbour).
struct BlockText {
    uint64_t own, halo;
    uint32_t before;
};

__device__ __forceinline__ BlockText readBlock(const PrefixText& pt, uint64_t base) {
    const uint32_t t = threadIdx.x;
    const uint64_t p0 = base + t * 8, h = base + kPrefixBlock + t * 8;
    BlockText b;
    b.own = p0 < pt.span ? pt.words[p0 >> 3] : 0;
    b.halo = t < 3 && h < pt.span ? pt.words[h >> 3] : 0;
    b.before = t % kWave == 0 && p0 > 0 && p0 < pt.span ? reinterpret_cast<const uint8_t*>(pt.words)[p0 - 1] : 0;
    return b;
}

// The records' keys of positions base + 8 * thread .. + 7 (base a multiple of kPrefixBlock), with the
// character before in the low byte; returns how many of the eight are positions of a text. Every
// thread calls it; the caller synchronises before the next call.
//
// A thread packs its eight codes and takes its neighbours' until it holds the eight windows of `chars`
// characters (at most 31 characters, or 16 of 6 to 8 bits: 128 bits); a key is then a shift and a mask.
template <class Texts>
__device__ __forceinline__ uint32_t blockKeys(const PrefixText& pt, const Texts& texts, BlockCodes<Texts::kBatch>& s, uint32_t base, const BlockText& text, uint64_t (&key)[kPrefixItems]) {
    const uint32_t t = threadIdx.x;
    if constexpr (Texts::kBatch) {
        if (pt.textCodes) {
            // A wave per table: the codes of the text at that 256-position block, if not there yet.
            const uint32_t lane = t % kWave;
            for (uint32_t b = t / kWave; b < BlockCodes<true>::kTables; b += kPrefixThreads / kWave) {
                const uint32_t p = base + b * 256;
                const uint32_t owner = p < pt.span ? texts.segmentOf(p) : ~0u;
                if (owner != ~0u && owner != s.tableText[b]) {
                    reinterpret_cast<uint32_t*>(s.table[b])[lane] = reinterpret_cast<const uint32_t*>(pt.textCodes + static_cast<size_t>(owner) * 256)[lane];
                    if (lane == 0) {
                        s.tableText[b] = owner;
                    }
                }
            }
            __syncthreads();
        }
    }
    const uint32_t p0 = base + t * 8;
    const bool inside = p0 < pt.span && p0 >= base;
    const uint32_t segment = inside ? texts.segmentOf(p0) : 0;
    const uint32_t end = inside ? min(texts.endOf(p0), pt.span) : 0;
    const uint32_t remaining = p0 < end ? end - p0 : 0;
    int bits = pt.charBits, chars = pt.chars;
    auto shape = [&](uint32_t of, int& b, int& c) {
        if (Texts::kBatch && pt.textCodes) {
            b = pt.textShape[2 * of];
            c = pt.textShape[2 * of + 1];
        }
    };
    if (remaining) {
        shape(segment, bits, chars);
    }
    // Eight codes (wide codes: the bytes themselves), the first at the top; 0 from `valid` on.
    auto pack = [&](uint64_t bytes, uint32_t at, uint32_t valid, int b) {
        if (pt.wide) {
            return __builtin_bswap64(bytes);
        }
        const uint8_t* table = s.table[Texts::kBatch ? at / 256 : 0];
        uint64_t packed = 0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t byte = static_cast<uint32_t>(bytes >> (8 * j)) & 255u;
            const uint32_t ch = static_cast<uint32_t>(j) < valid ? table[byte] : 0u;
            packed = (packed << b) | ch;
        }
        return packed;
    };
    const uint64_t own = pack(text.own, t * 8, remaining, bits);
    s.packed[t] = own;
    if (t < 3) {
        const uint32_t q = base + kPrefixBlock + t * 8;
        const bool in = q < pt.span && q >= base;
        const uint32_t qEnd = in ? min(texts.endOf(q), pt.span) : 0;
        int qBits = pt.charBits, qChars = pt.chars;
        if (q < qEnd) {
            shape(texts.segmentOf(q), qBits, qChars);
        }
        s.packed[kPrefixThreads + t] = pack(text.halo, kPrefixBlock + t * 8, q < qEnd ? qEnd - q : 0, qBits);
    }
    __syncthreads();

    // The window, left-aligned in 128 bits.
    unsigned __int128 window;
    if (pt.wide) {
        window = 0;
        const uint64_t next = s.packed[t + 1];
#pragma unroll
        for (uint32_t k = 0; k < 14; k++) {  // 6 characters a key at most
            const uint32_t byte = static_cast<uint32_t>((k < 8 ? own >> (56 - 8 * k) : next >> (120 - 8 * k))) & 255u;
            window = window << 9 | (k < remaining ? byte + 1 : 0u);
        }
        window <<= 2;
    } else {
        // Two groups of eight hold the windows of codes of 6 to 8 bits, three of 4 and 5, four of fewer.
        const int groups = bits >= 6 ? 2 : bits >= 4 ? 3 : 4;
        // A group past the text's end may be another text's, packed at another width: it counts as 0.
        auto group = [&](uint32_t g) -> uint64_t { return !Texts::kBatch || remaining > 8 * g ? s.packed[t + g] : 0; };
        window = static_cast<unsigned __int128>(own) << (8 * bits) | group(1);
        if (groups > 2) {
            window = window << (8 * bits) | group(2);
        }
        if (groups > 3) {
            window = window << (8 * bits) | group(3);
        }
        window <<= 128 - 8 * bits * groups;
    }
    uint64_t high = static_cast<uint64_t>(window >> 64), low = static_cast<uint64_t>(window);
    if constexpr (Texts::kBatch) {
        // Codes of the next text are not this one's.
        const uint32_t held = heldBits(remaining, bits);
        high &= held >= 64 ? ~uint64_t(0) : ~(~uint64_t(0) >> held);
        low &= held >= 128 ? ~uint64_t(0) : held <= 64 ? 0 : ~(~uint64_t(0) >> (held - 64));
    }
    const uint64_t mask = ~uint64_t(0) << (64 - chars * bits);
    const uint64_t top = Texts::kBatch && pt.segmentBits ? static_cast<uint64_t>(segment) << (64 - pt.segmentBits) : 0;
    uint32_t previous = waveShiftUp(static_cast<uint32_t>(text.own >> 56));
    previous = t % kWave == 0 ? text.before : previous;
    if (Texts::kBatch || p0 == 0) {
        previous = remaining && p0 > (Texts::kBatch ? texts.startOf(p0) : 0u) ? previous : 0u;
    }
#pragma unroll
    for (int j = 0; j < kPrefixItems; j++) {
        const uint64_t at = j == 0 ? high : high << (j * bits) | low >> (64 - j * bits);
        uint64_t k = at & mask;
        if constexpr (Texts::kBatch) {
            k = k >> pt.segmentBits | top;
        }
        key[j] = k | (j == 0 ? previous : static_cast<uint32_t>(text.own >> (8 * (j - 1))) & 255u);
    }
    return min(remaining, 8u);
}

// ---- buckets --------------------------------------------------------------------------------------

// The number of splitters at or below key. The splitters are a binary tree in level order (root at 1,
// children of i at 2i and 2i + 1): the nodes of a level are neighbours, where halving steps through
// a sorted table read addresses a power of two apart, all in the same LDS banks (82% of the cycles
// of countBucketsKernel were such conflicts). `steps` levels; the leaves past the last splitter are
// ~0, which no key part reaches.
__device__ __forceinline__ uint32_t bucketOf(const uint64_t* tree, int steps, uint64_t key) {
    uint32_t node = 1;
    for (int s = 0; s < steps; s++) {
        node = 2 * node + (tree[node] <= key ? 1 : 0);
    }
    return node - (1u << steps);
}

inline int log2Ceil(uint32_t x) {
    int s = 0;
    while ((1u << s) < x) {
        s++;
    }
    return s;
}

// The tree of `count` splitters (every stride-th from `from`), 2^steps entries.
__device__ __forceinline__ void loadSplitters(const uint64_t* __restrict__ from, uint32_t count, uint32_t stride, int steps, uint64_t* tree) {
    for (uint32_t x = threadIdx.x + 1; x < (1u << steps); x += kPrefixThreads) {
        const int level = 31 - __builtin_clz(x);
        const uint32_t sorted = ((2 * (x - (1u << level)) + 1) << (steps - 1 - level)) - 1;
        tree[x] = sorted < count ? from[static_cast<uint64_t>(sorted) * stride] : ~uint64_t(0);
    }
}

// counts[b * tiles + tile] = positions of the tile (tileBlocks blocks) whose key is in bucket b. Bucket
// b's first splitter is leaf splitter b * bins - 1 (bins leaves per bucket).
template <class Texts>
__global__ __launch_bounds__(kPrefixThreads) void countBucketsKernel(PrefixText pt, Texts texts, CodeTable codes, const uint64_t* __restrict__ splitters, uint32_t buckets, uint32_t bins, int steps, uint32_t tileBlocks, uint32_t tiles, uint32_t* __restrict__ counts) {
    __shared__ BlockCodes<Texts::kBatch> s;
    __shared__ uint64_t split[kPrefixMaxBuckets];
    __shared__ uint32_t histogram[kPrefixMaxBuckets];
    initBlockCodes<Texts>(pt, codes, s);
    loadSplitters(splitters + bins - 1, buckets - 1, bins, steps, split);
    for (uint32_t x = threadIdx.x; x < buckets; x += kPrefixThreads) {
        histogram[x] = 0;
    }
    __syncthreads();
    const uint32_t tile = xcdTile(blockIdx.x, tiles);
    BlockText text = readBlock(pt, static_cast<uint64_t>(tile) * tileBlocks * kPrefixBlock);
    for (uint32_t b = 0; b < tileBlocks; b++) {
        const uint64_t base = (static_cast<uint64_t>(tile) * tileBlocks + b) * kPrefixBlock;
        if (base >= pt.span) {
            break;
        }
        const BlockText current = text;
        text = readBlock(pt, base + kPrefixBlock);
        uint64_t key[kPrefixItems];
        const uint32_t valid = blockKeys(pt, texts, s, static_cast<uint32_t>(base), current, key);
#pragma unroll
        for (int j = 0; j < kPrefixItems; j++) {
            if (static_cast<uint32_t>(j) < valid) {
                atomicAdd(&histogram[bucketOf(split, steps, keyPart(key[j]))], 1u);
            }
        }
        __syncthreads();
    }
    for (uint32_t x = threadIdx.x; x < buckets; x += kPrefixThreads) {
        counts[static_cast<uint64_t>(x) * tiles + tile] = histogram[x];
    }
}

// out[b] = the first row of bucket b (b = buckets: all rows), and after them the sample's kSeenWords
// counts: what the host reads to plan the rounds.
constexpr uint32_t kSeenWords = 3;

__global__ void bucketRowsKernel(const uint32_t* __restrict__ offsets, uint32_t tiles, uint32_t buckets, uint32_t allRows, const uint32_t* __restrict__ seen, uint32_t* __restrict__ out) {
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < buckets) {
        out[b] = offsets[static_cast<uint64_t>(b) * tiles];
    } else if (b == buckets) {
        out[b] = allRows;
    } else if (b <= buckets + kSeenWords) {
        out[b] = seen[b - buckets - 1];
    }
}

// LDS of placeBlock for up to kPrefixMaxBins bins (one per thread).
struct PlaceStage {
    uint64_t key[kPrefixBlock];
    uint32_t position[kPrefixBlock];
    uint16_t bin[kPrefixBlock];
    uint64_t split[kPrefixMaxBins];
    uint32_t histogram[kPrefixMaxBins];  // zero between calls
    uint32_t start[kPrefixMaxBins];      // a bin's first place in the block
    uint32_t delta[kPrefixMaxBins];      // output index of a bin's records less their place
    uint32_t waveSums[kPrefixThreads / kWave];
};

// Scatters a block's records (`valid` bits of the thread's eight) to their bins, staged in LDS in bin
// order so that each bin's records are written in a run; thread t holds bin t's next output index in
// `cursor`. Order within a bin is not kept. The stage's records are read until the caller's next
// barrier (placeBlock's own first one will do).
__device__ __forceinline__ void placeBlock(PlaceStage& s, const uint64_t (&key)[kPrefixItems], const uint32_t (&position)[kPrefixItems], uint32_t valid, uint32_t bins, int steps, uint32_t& cursor, PrefixRecord* __restrict__ out, uint32_t limit) {
    static_assert(kPrefixMaxBins == kPrefixThreads, "a bin per thread");
    const uint32_t t = threadIdx.x, wave = t / kWave, lane = t % kWave;
    uint32_t place[kPrefixItems];  // bin, rank in the bin (below 4096)
#pragma unroll
    for (int j = 0; j < kPrefixItems; j++) {
        if ((valid >> j) & 1) {
            const uint32_t bin = bucketOf(s.split, steps, keyPart(key[j]));
            place[j] = bin << 16 | atomicAdd(&s.histogram[bin], 1u);
        }
    }
    __syncthreads();
    const uint32_t mine = t < bins ? s.histogram[t] : 0;
    const uint32_t inclusive = waveInclusive<OpSum>(mine);
    if (lane == kWave - 1) {
        s.waveSums[wave] = inclusive;
    }
    __syncthreads();
    uint32_t start = inclusive - mine, total = 0;
    for (uint32_t w = 0; w < kPrefixThreads / kWave; w++) {
        start += w < wave ? s.waveSums[w] : 0;
        total += s.waveSums[w];
    }
    if (t < bins) {
        s.start[t] = start;
        s.delta[t] = cursor - start;
        s.histogram[t] = 0;
        cursor += mine;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPrefixItems; j++) {
        if ((valid >> j) & 1) {
            const uint32_t bin = place[j] >> 16;
            const uint32_t at = s.start[bin] + (place[j] & 0xFFFFu);
            s.key[at] = key[j];
            s.position[at] = position[j];
            s.bin[at] = static_cast<uint16_t>(bin);
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPrefixItems; j++) {
        const uint32_t x = j * kPrefixThreads + t;
        if (x < total) {
            const uint32_t target = s.delta[s.bin[x]] + x;
            if (target < limit) {
                out[target] = packRecord(s.key[x], s.position[x]);
            }
        }
    }
}

// A round's records from the text: positions whose key lies in buckets [firstBucket, firstBucket +
// buckets), at (offsets[bucket * tiles + tile] - rowBase) onwards. The selected records of several
// blocks collect in LDS until another block's might not fit, and are then placed together.
template <class Texts>
__global__ __launch_bounds__(kPrefixThreads, 4) void scatterBucketsKernel(PrefixText pt, Texts texts, CodeTable codes, const uint64_t* __restrict__ splitters, uint32_t allBuckets, uint32_t firstBucket, uint32_t buckets, uint32_t bins, int steps, uint32_t tileBlocks, uint32_t tiles, const uint32_t* __restrict__ offsets, uint32_t rowBase, uint32_t limit, PrefixRecord* __restrict__ out) {
    extern __shared__ __align__(16) unsigned char shared[];
    PlaceStage& stage = *reinterpret_cast<PlaceStage*>(shared);
    BlockCodes<Texts::kBatch>& s = *reinterpret_cast<BlockCodes<Texts::kBatch>*>(shared + (sizeof(PlaceStage) + 15) / 16 * 16);
    __shared__ uint32_t waveCount[kPrefixThreads / kWave];
    const uint32_t t = threadIdx.x, wave = t / kWave, lane = t % kWave;
    const uint32_t tile = xcdTile(blockIdx.x, tiles);
    initBlockCodes<Texts>(pt, codes, s);
    loadSplitters(splitters + static_cast<uint64_t>(firstBucket + 1) * bins - 1, buckets - 1, bins, steps, stage.split);
    stage.histogram[t] = 0;
    uint32_t cursor = t < buckets ? offsets[static_cast<uint64_t>(firstBucket + t) * tiles + tile] - rowBase : 0;
    const uint64_t low = firstBucket > 0 ? splitters[static_cast<uint64_t>(firstBucket) * bins - 1] : 0;
    const bool bounded = firstBucket + buckets < allBuckets;
    const uint64_t high = bounded ? splitters[static_cast<uint64_t>(firstBucket + buckets) * bins - 1] : 0;
    __syncthreads();

    uint32_t fill = 0;  // records waiting in the stage
    auto flush = [&]() {
        uint64_t k[kPrefixItems];
        uint32_t p[kPrefixItems];
        uint32_t valid = 0;
#pragma unroll
        for (int j = 0; j < kPrefixItems; j++) {
            const uint32_t x = j * kPrefixThreads + t;
            k[j] = stage.key[x];
            p[j] = stage.position[x];
            valid |= x < fill ? 1u << j : 0u;
        }
        placeBlock(stage, k, p, valid, buckets, steps, cursor, out, limit);
        fill = 0;
        __syncthreads();
    };
    const uint64_t firstBase = static_cast<uint64_t>(tile) * tileBlocks * kPrefixBlock;
    BlockText text = readBlock(pt, firstBase);
    for (uint32_t b = 0; b <= tileBlocks; b++) {
        const uint64_t base = firstBase + static_cast<uint64_t>(b) * kPrefixBlock;
        if (b == tileBlocks || base >= pt.span) {
            break;
        }
        uint64_t key[kPrefixItems];
        const BlockText current = text;
        text = readBlock(pt, base + kPrefixBlock);
        const uint32_t count = blockKeys(pt, texts, s, static_cast<uint32_t>(base), current, key);
        uint32_t selected = 0;
#pragma unroll
        for (int j = 0; j < kPrefixItems; j++) {
            const uint64_t k = keyPart(key[j]);
            if (static_cast<uint32_t>(j) < count && k >= low && (!bounded || k < high)) {
                selected |= 1u << j;
            }
        }
        const uint32_t own = __builtin_popcount(selected);
        const uint32_t inclusive = waveInclusive<OpSum>(own);
        if (lane == kWave - 1) {
            waveCount[wave] = inclusive;
        }
        __syncthreads();
        uint32_t at = inclusive - own, total = 0;
        for (uint32_t w = 0; w < kPrefixThreads / kWave; w++) {
            at += w < wave ? waveCount[w] : 0;
            total += waveCount[w];
        }
        if (fill + total > kPrefixBlock) {
            flush();
        }
        at += fill;
#pragma unroll
        for (int j = 0; j < kPrefixItems; j++) {
            if ((selected >> j) & 1) {
                stage.key[at] = key[j];
                stage.position[at] = static_cast<uint32_t>(base) + t * 8 + j;
                at++;
            }
        }
        fill += total;
        __syncthreads();
    }
    if (fill > 0) {
        flush();
    }
}

template <class Texts>
constexpr size_t scatterSharedBytes() {
    return (sizeof(PlaceStage) + 15) / 16 * 16 + sizeof(BlockCodes<Texts::kBatch>);
}

// A round's buckets for the second level: starts[b] (round-relative first record; b = buckets: the
// total) and tilesBefore[b] (second-level tiles of tileRecords records of the buckets before; every
// bucket has at least one). One workgroup.
__global__ __launch_bounds__(kPrefixMaxRoundBuckets) void bucketTilesKernel(const uint32_t* __restrict__ offsets, uint32_t tiles, uint32_t allBuckets, uint32_t firstBucket, uint32_t buckets, uint32_t rowBase, uint32_t allRows, uint32_t tileRecords, uint32_t* __restrict__ starts, uint32_t* __restrict__ tilesBefore) {
    __shared__ uint32_t waveSums[kPrefixMaxRoundBuckets / kWave];
    const uint32_t b = threadIdx.x, wave = b / kWave, lane = b % kWave;
    auto startOf = [&](uint32_t x) {
        return (firstBucket + x < allBuckets ? offsets[static_cast<uint64_t>(firstBucket + x) * tiles] : allRows) - rowBase;
    };
    uint32_t own = 0;
    if (b < buckets) {
        const uint32_t s0 = startOf(b), s1 = startOf(b + 1);
        starts[b] = s0;
        own = max(1u, (s1 - s0 + tileRecords - 1) / tileRecords);
        if (b + 1 == buckets) {
            starts[buckets] = s1;
        }
    }
    const uint32_t inclusive = waveInclusive<OpSum>(own);
    if (lane == kWave - 1) {
        waveSums[wave] = inclusive;
    }
    __syncthreads();
    uint32_t prefix = inclusive - own;
    for (uint32_t w = 0; w < wave; w++) {
        prefix += waveSums[w];
    }
    if (b < buckets) {
        tilesBefore[b] = prefix;
        if (b + 1 == buckets) {
            tilesBefore[buckets] = prefix + own;
        }
    }
}

// The bucket of second-level tile `tile`: the last with tilesBefore <= tile.
__device__ __forceinline__ uint32_t bucketOfTile(const uint32_t* __restrict__ tilesBefore, uint32_t buckets, uint32_t tile) {
    uint32_t lo = 0, hi = buckets;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (tilesBefore[mid] <= tile) {
            lo = mid;
        } else {
            hi = mid;
        }
    }
    return lo;
}

// Second level. A tile's counts lie at tilesBefore[bucket] * bins + bin * (tiles of the bucket) + (tile
// in the bucket), so one exclusive sum gives every (bucket, bin, tile) its place in the round.
__global__ __launch_bounds__(kPrefixThreads) void countBinsKernel(const PrefixRecord* __restrict__ records, const uint64_t* __restrict__ splitters, const uint32_t* __restrict__ starts, const uint32_t* __restrict__ tilesBefore, uint32_t firstBucket, uint32_t buckets, uint32_t bins, int steps, uint32_t tileRecords, uint32_t* __restrict__ counts) {
    __shared__ uint64_t split[kPrefixMaxBins];
    __shared__ uint32_t histogram[kPrefixMaxBins];
    const uint32_t tile = xcdTile(blockIdx.x, gridDim.x);
    if (tile >= tilesBefore[buckets]) {
        return;
    }
    const uint32_t bucket = bucketOfTile(tilesBefore, buckets, tile);
    const uint32_t before = tilesBefore[bucket], tilesHere = tilesBefore[bucket + 1] - before;
    loadSplitters(splitters + static_cast<uint64_t>(firstBucket + bucket) * bins, bins - 1, 1, steps, split);
    for (uint32_t x = threadIdx.x; x < bins; x += kPrefixThreads) {
        histogram[x] = 0;
    }
    __syncthreads();
    const uint32_t first = starts[bucket] + (tile - before) * tileRecords;
    const uint32_t last = min(starts[bucket + 1], first + tileRecords);
    for (uint32_t x0 = first + threadIdx.x; x0 < last; x0 += kPrefixBlock) {
        uint64_t key[kPrefixItems];
#pragma unroll
        for (int j = 0; j < kPrefixItems; j++) {
            key[j] = keyOf(records[min(x0 + j * kPrefixThreads, last - 1)]);
        }
#pragma unroll
        for (int j = 0; j < kPrefixItems; j++) {
            if (x0 + j * kPrefixThreads < last) {
                atomicAdd(&histogram[bucketOf(split, steps, keyPart(key[j]))], 1u);
            }
        }
    }
    __syncthreads();
    for (uint32_t x = threadIdx.x; x < bins; x += kPrefixThreads) {
        counts[static_cast<uint64_t>(before) * bins + static_cast<uint64_t>(x) * tilesHere + (tile - before)] = histogram[x];
    }
}

__global__ __launch_bounds__(kPrefixThreads, 4) void scatterBinsKernel(const PrefixRecord* __restrict__ records, const uint64_t* __restrict__ splitters, const uint32_t* __restrict__ starts, const uint32_t* __restrict__ tilesBefore, uint32_t firstBucket, uint32_t buckets, uint32_t bins, int steps, uint32_t tileRecords, const uint32_t* __restrict__ offsets, uint32_t limit, PrefixRecord* __restrict__ out) {
    extern __shared__ __align__(16) unsigned char shared[];
    PlaceStage& stage = *reinterpret_cast<PlaceStage*>(shared);
    const uint32_t tile = xcdTile(blockIdx.x, gridDim.x);
    if (tile >= tilesBefore[buckets]) {
        return;
    }
    const uint32_t bucket = bucketOfTile(tilesBefore, buckets, tile);
    const uint32_t before = tilesBefore[bucket], tilesHere = tilesBefore[bucket + 1] - before;
    const uint32_t first = starts[bucket] + (tile - before) * tileRecords;
    const uint32_t last = min(starts[bucket + 1], first + tileRecords);
    const uint32_t t = threadIdx.x;
    // A block's records are loaded while the block before is placed.
    PrefixRecord next[kPrefixItems];
    auto load = [&](uint32_t block) {
#pragma unroll
        for (int j = 0; j < kPrefixItems; j++) {
            next[j] = records[min(block + j * kPrefixThreads + t, last - 1)];
        }
    };
    if (first < last) {
        load(first);
    }
    loadSplitters(splitters + static_cast<uint64_t>(firstBucket + bucket) * bins, bins - 1, 1, steps, stage.split);
    stage.histogram[t] = 0;
    uint32_t cursor = t < bins ? offsets[static_cast<uint64_t>(before) * bins + static_cast<uint64_t>(t) * tilesHere + (tile - before)] : 0;
    __syncthreads();
    for (uint32_t block = first; block < last; block += kPrefixBlock) {
        uint64_t key[kPrefixItems];
        uint32_t position[kPrefixItems];
        uint32_t valid = 0;
#pragma unroll
        for (int j = 0; j < kPrefixItems; j++) {
            key[j] = keyOf(next[j]);
            position[j] = next[j].position;
            valid |= block + j * kPrefixThreads + t < last ? 1u << j : 0u;
        }
        if (block + kPrefixBlock < last) {
            load(block + kPrefixBlock);
        }
        placeBlock(stage, key, position, valid, bins, steps, cursor, out, limit);
    }
}

// leafStart[x] of a group of buckets: the first record of leaf x in it (x = leaves: the total).
__global__ __launch_bounds__(256) void leafStartsKernel(const uint32_t* __restrict__ starts, const uint32_t* __restrict__ tilesBefore, const uint32_t* __restrict__ offsets, uint32_t buckets, uint32_t bins, uint32_t* __restrict__ leafStart) {
    const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x > buckets * bins) {
        return;
    }
    if (x == buckets * bins) {
        leafStart[x] = starts[buckets] - starts[0];
    } else {
        const uint32_t b = x / bins, before = tilesBefore[b], tilesHere = tilesBefore[b + 1] - before;
        leafStart[x] = offsets[static_cast<uint64_t>(before) * bins + static_cast<uint64_t>(x % bins) * tilesHere];
    }
}

// ---- leaves ---------------------------------------------------------------------------------------

// Where rows go. bwt may be null. ties: bit r mod 32 of word r / 32 is set when row r's key equals
// row r - 1's. firstRows[s]: the row (in text s) of its suffix 0, or of the head of the group it ties
// in: other rows' BWT bytes move up by one exactly when they come before it.
struct RowOut {
    uint32_t* sa;
    uint8_t* bwt;
    uint32_t* ties;
    uint32_t* firstRows;
    const uint64_t* startKeys;  // the key of every text's suffix 0
    const Segment* segments;
    int segmentBits;
};

// Row `row` (of all texts) holds `position`, whose record is `key`; tied: its key equals the row's
// before. The BWT bytes of a group of tied rows wait in the group's places,
// in the order of its positions (those of a text's suffix 0's own group: nowhere, they are read again).
__device__ __forceinline__ void emitRow(const RowOut& out, uint32_t row, uint64_t key, uint32_t position, bool tied) {
    out.sa[row] = position;
    if (out.bwt) {
        const uint32_t segment = out.segmentBits ? static_cast<uint32_t>(key >> (64 - out.segmentBits)) : 0;
        const uint64_t start = out.startKeys[segment];
        const uint64_t k = keyPart(key);
        if (k == start) {
            if (!tied) {
                out.firstRows[segment] = row - out.segments[segment].rowBase;
            }
        } else {
            out.bwt[k < start ? row + 1 : row] = static_cast<uint8_t>(key);
        }
    }
}

// The tie bits of a wave's 64 rows from row `row` (lane 0's).
__device__ __forceinline__ void emitTies(uint32_t* __restrict__ ties, uint32_t row, uint64_t mask) {
    if (mask != 0 && laneId() < 3) {
        const uint32_t shift = row & 31, lane = laneId();
        // Word `lane` of the mask moved up by `shift`.
        const uint32_t word = lane == 0 ? static_cast<uint32_t>(mask << shift)
                            : lane == 1 ? static_cast<uint32_t>((mask << shift) >> 32)
                                        : static_cast<uint32_t>(shift ? mask >> (64 - shift) : 0);
        if (word) {
            atomicOr(&ties[(row >> 5) + lane], word);
        }
    }
}

// Before the rows are written: no ties, the texts' start keys, and with a BWT byte 0 of every text,
// T[end - 1].
template <class Texts>
__global__ __launch_bounds__(256) void initRowsKernel(PrefixText pt, Texts texts, CodeTable codes, const Segment* __restrict__ segments, uint32_t count, uint64_t* __restrict__ startKeys, uint32_t* __restrict__ ties, uint32_t tieWords, uint8_t* __restrict__ bwt) {
    __shared__ uint8_t code[256];
    loadCodes(codes, code);
    const uint32_t first = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
    for (uint32_t w = first; w < tieWords; w += stride) {
        ties[w] = 0;
    }
    for (uint32_t s = first; s < count; s += stride) {
        startKeys[s] = prefixKey(pt, texts, code, segments[s].start);
        if (bwt) {
            bwt[segments[s].rowBase] = reinterpret_cast<const uint8_t*>(pt.words)[segments[s].end - 1];
        }
    }
}

// Leaves too large for their workgroup's LDS: their first row and length, in no order.
struct BigLeaves {
    uint32_t* count;    // [0] leaves, [1] records
    uint2* list;        // kBigLeavesMax
};
constexpr uint32_t kBigLeavesMax = 4096;

constexpr int kLeafThreads = 256;
constexpr int kLeafWaves = kLeafThreads / kWave;
constexpr int kLeafLane = 8;                             // records a lane sorts in registers
constexpr uint32_t kLeafChunk = kWave * kLeafLane;       // records a wave sorts in registers
constexpr int kLeafIndexBits = 12;                       // of a record's index in its leaf
constexpr uint32_t kLeafIndexMask = (1u << kLeafIndexBits) - 1;
constexpr uint32_t kLeafLastValues = 16;                  // of a key's last four bits

// One phase of the bitonic sort of a wave's kLeafChunk values, element lane * kLeafLane + r in v[r]:
// merges sorted runs of kRun / 2 (alternately ascending and descending) into runs of kRun.
template <int kRun, int kStride>
__device__ __forceinline__ void bitonicStages(uint64_t (&v)[kLeafLane], uint32_t lane) {
    if constexpr (kStride >= kLeafLane) {
        // Across lanes: the lower lane of a pair keeps the smaller value in an ascending run.
        constexpr int kLanes = kStride / kLeafLane;
        const bool keepSmaller = ((lane & kLanes) == 0) == ((lane & (kRun / kLeafLane)) == 0);
#pragma unroll
        for (int r = 0; r < kLeafLane; r++) {
            const uint64_t other = laneXor64<kLanes>(v[r]);
            v[r] = (v[r] < other) == keepSmaller ? v[r] : other;
        }
    } else {
#pragma unroll
        for (int r = 0; r < kLeafLane; r++) {
            if ((r & kStride) == 0) {
                const bool ascending = kRun >= kLeafLane ? (lane & (kRun / kLeafLane)) == 0 : (r & kRun) == 0;
                const uint64_t x = v[r], y = v[r + kStride];
                const bool keep = (x < y) == ascending;
                v[r] = keep ? x : y;
                v[r + kStride] = keep ? y : x;
            }
        }
    }
    if constexpr (kStride > 1) {
        bitonicStages<kRun, kStride / 2>(v, lane);
    }
}

template <int kRun>
__device__ __forceinline__ void bitonicSort(uint64_t (&v)[kLeafLane], uint32_t lane) {
    if constexpr (kRun > 2) {
        bitonicSort<kRun / 2>(v, lane);
    }
    bitonicStages<kRun, kRun / 2>(v, lane);
}

__device__ __forceinline__ uint32_t lastBits(uint64_t key) {
    return (static_cast<uint32_t>(key) >> 8) & (kLeafLastValues - 1);
}

// Where value e of a leaf lies in LDS: a lane's eight values are written one after another, and
// unswizzled eight-value strides would fall into four of the banks.
__device__ __forceinline__ uint32_t leafSlot(uint32_t e) {
    return e ^ ((e >> 3) & 7u);
}

// Outputs [t * kPer, t * kPer + kPer) of merging the runs of `run` values pairwise (`total` values).
template <int kPer>
__device__ __forceinline__ void mergeLeafRuns(uint64_t* values, uint32_t total, uint32_t run) {
    const uint32_t o = threadIdx.x * kPer;
    uint64_t merged[kPer];
    if (o < total) {
        const uint32_t base = o / (2 * run) * (2 * run);
        const uint32_t lengthA = min(run, total - base), lengthB = min(run, total - base - lengthA);
        const uint32_t startB = base + lengthA;
        const uint32_t d = o - base;
        uint32_t lo = d > lengthB ? d - lengthB : 0, hi = min(d, lengthA);
        while (lo < hi) {
            const uint32_t mid = (lo + hi) / 2;
            const bool less = values[leafSlot(base + mid)] < values[leafSlot(startB + d - 1 - mid)];
            lo = less ? mid + 1 : lo;
            hi = less ? hi : mid;
        }
        uint32_t ia = lo, ib = d - lo;
        uint64_t a = ia < lengthA ? values[leafSlot(base + ia)] : ~uint64_t(0);
        uint64_t b = ib < lengthB ? values[leafSlot(startB + ib)] : ~uint64_t(0);
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const bool takeA = a < b;
            merged[k] = takeA ? a : b;
            ia += takeA ? 1 : 0;
            ib += takeA ? 0 : 1;
            const uint32_t next = takeA ? base + ia : startB + ib;
            const bool inside = takeA ? ia < lengthA : ib < lengthB;
            const uint64_t v = inside ? values[leafSlot(min(next, total - 1))] : ~uint64_t(0);
            a = takeA ? v : a;
            b = takeA ? b : v;
        }
    }
    __syncthreads();
    if (o < total) {
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            values[leafSlot(o + k)] = merged[k];
        }
    }
    __syncthreads();
}

// One workgroup per leaf of a group of buckets: records [leafStart[leaf], leafStart[leaf + 1]) less
// leafBase, sorted by key in LDS and written to those rows past rowBase. A leaf's keys share their
// upper bits, so the others and a record's index in the leaf fit one 64-bit value: a wave sorts 512
// of them in registers (bitonic), and the sorted runs merge in LDS. Against LSD digit passes over
// the records that is half the instructions, which is what bounds this kernel.
template <uint32_t kCapacity>
__global__ __launch_bounds__(kLeafThreads) void sortLeavesKernel(const PrefixRecord* __restrict__ records, const uint32_t* __restrict__ leafStart, uint32_t leafBase, uint32_t rowBase, RowOut out, BigLeaves big) {
    static_assert(kCapacity <= 1u << kLeafIndexBits, "an index per record");
    constexpr int kPasses = kCapacity / (kLeafChunk * kLeafWaves);  // chunks of a wave
    __shared__ uint64_t values[kCapacity];
    __shared__ uint32_t position[kCapacity];
    __shared__ uint8_t before[kCapacity];
    __shared__ uint32_t differLow, differHigh;
    __shared__ uint32_t lastStart[kLeafLastValues], lastNext[kLeafLastValues];  // truncated leaves

    const uint32_t t = threadIdx.x, wave = t / kWave, lane = t % kWave;
    const uint32_t first = leafStart[blockIdx.x] - leafBase;
    const uint32_t size = leafStart[blockIdx.x + 1] - leafBase - first;
    if (size == 0) {
        return;
    }
    if (size > kCapacity) {
        if (t == 0) {
            const uint32_t at = atomicAdd(&big.count[0], 1u);
            atomicAdd(&big.count[1], size);
            if (at < kBigLeavesMax) {
                big.list[at] = uint2{rowBase + first, size};
            }
        }
        // Its positions wait in its rows, in any order.
        for (uint32_t x = t; x < size; x += kLeafThreads) {
            out.sa[rowBase + first + x] = records[first + x].position;
        }
        return;
    }
    if (t == 0) {
        differLow = 0;
        differHigh = 0;
    }
    if (t < kLeafLastValues) {
        lastNext[t] = 0;
    }
    const uint32_t chunks = (size + kLeafChunk - 1) / kLeafChunk;
    records += first;
    const uint64_t reference = keyOf(records[0]);
    uint64_t key[kPasses][kLeafLane];
    uint64_t differ = 0;
#pragma unroll
    for (int c = 0; c < kPasses; c++) {
        const uint32_t chunk = wave + c * kLeafWaves;
        if (chunk < chunks) {
#pragma unroll
            for (int r = 0; r < kLeafLane; r++) {
                const uint32_t x = min(chunk * kLeafChunk + r * kWave + lane, size - 1);
                const PrefixRecord record = records[x];
                key[c][r] = keyOf(record);
                position[x] = record.position;
            }
#pragma unroll
            for (int r = 0; r < kLeafLane; r++) {
                before[min(chunk * kLeafChunk + r * kWave + lane, size - 1)] = static_cast<uint8_t>(key[c][r]);
                differ |= key[c][r] ^ reference;
            }
        }
    }
    uint32_t low = static_cast<uint32_t>(differ) & ~0xFFu, high = static_cast<uint32_t>(differ >> 32);
    for (int offset = kWave / 2; offset > 0; offset /= 2) {
        low |= __shfl_xor(low, offset);
        high |= __shfl_xor(high, offset);
    }
    __syncthreads();
    if (lane == 0 && (low | high)) {
        atomicOr(&differLow, low);
        atomicOr(&differHigh, high);
    }
    __syncthreads();
    const uint64_t differing = static_cast<uint64_t>(differHigh) << 32 | differLow;
    // The bits all keys share at the top; 4 or more leave room for the index. With fewer, the last
    // four key bits are left out of the values: the records are numbered in the order of those bits,
    // so that the index orders them.
    const int shared = differing ? min(__builtin_clzll(differing), 63) : 63;
    const bool truncated = shared < kLeafIndexBits - 8;
    if (truncated) {
#pragma unroll
        for (int c = 0; c < kPasses; c++) {
#pragma unroll
            for (int r = 0; r < kLeafLane; r++) {
                if ((wave + c * kLeafWaves) * kLeafChunk + r * kWave + lane < size) {
                    atomicAdd(&lastNext[lastBits(key[c][r])], 1u);
                }
            }
        }
        __syncthreads();
        if (t == 0) {
            uint32_t before16 = 0;
            for (uint32_t d = 0; d < kLeafLastValues; d++) {
                const uint32_t count = lastNext[d];
                lastStart[d] = before16;
                lastNext[d] = before16;
                before16 += count;
            }
        }
        __syncthreads();
    }

#pragma unroll
    for (int c = 0; c < kPasses; c++) {
        const uint32_t chunk = wave + c * kLeafWaves;
        if (chunk < chunks) {
            uint64_t v[kLeafLane];
#pragma unroll
            for (int r = 0; r < kLeafLane; r++) {
                uint32_t x = chunk * kLeafChunk + r * kWave + lane;
                if (truncated && x < size) {
                    const uint32_t from = x;
                    x = atomicAdd(&lastNext[lastBits(key[c][r])], 1u);
                    position[x] = records[from].position;
                    before[x] = static_cast<uint8_t>(key[c][r]);
                }
                v[r] = x < size ? ((keyPart(key[c][r]) << shared) & ~static_cast<uint64_t>(kLeafIndexMask)) | x : ~uint64_t(0);
            }
            if (differing) {
                bitonicSort<kLeafChunk>(v, lane);
#pragma unroll
                for (int r = 0; r < kLeafLane; r++) {
                    values[leafSlot(chunk * kLeafChunk + lane * kLeafLane + r)] = v[r];
                }
            } else {
#pragma unroll
                for (int r = 0; r < kLeafLane; r++) {
                    values[leafSlot(chunk * kLeafChunk + r * kWave + lane)] = v[r];
                }
            }
        }
    }
    __syncthreads();
    if (differing) {
        for (uint32_t run = kLeafChunk; run < chunks * kLeafChunk; run *= 2) {
            if (kPasses == 1 || chunks <= kLeafWaves) {
                mergeLeafRuns<kLeafLane>(values, chunks * kLeafChunk, run);
            } else {
                mergeLeafRuns<kLeafLane * kPasses>(values, chunks * kLeafChunk, run);
            }
        }
    }

    const uint64_t top = differing ? (shared ? reference & ~(~uint64_t(0) >> shared) : 0) : keyPart(reference);
    for (uint32_t x = t; x - lane < size; x += kLeafThreads) {
        const bool valid = x < size;
        const uint64_t v = values[leafSlot(min(x, size - 1))];
        const uint32_t index = static_cast<uint32_t>(v) & kLeafIndexMask;
        const uint64_t previous = values[leafSlot(x > 0 && valid ? x - 1 : 0)];
        bool tied = valid && x > 0 && previous >> kLeafIndexBits == v >> kLeafIndexBits;
        uint64_t key = differing ? top | (v & ~static_cast<uint64_t>(kLeafIndexMask)) >> shared : top;
        if (truncated) {
            uint32_t last = 0;
#pragma unroll
            for (uint32_t step = kLeafLastValues / 2; step > 0; step /= 2) {
                last += lastStart[last + step] <= index ? step : 0;
            }
            key |= static_cast<uint64_t>(last) << 8;
            tied = tied && (previous & kLeafIndexMask) >= lastStart[last];
        }
        if (valid) {
            emitRow(out, rowBase + first + x, key | before[index], position[index], tied);
        }
        emitTies(out.ties, rowBase + first + x - lane, ballot(tied));
    }
}

// ---- large leaves ---------------------------------------------------------------------------------

// The large leaves' records, leaf after leaf (list sorted by row; before[x] = records of leaves before
// x): their keys again from the text, their positions from the rows.
__device__ __forceinline__ uint32_t bigLeafOf(const uint32_t* __restrict__ before, uint32_t leaves, uint32_t k) {
    return bucketOfTile(before, leaves, k);
}

template <class Texts>
__global__ __launch_bounds__(256) void bigLeafKeysKernel(PrefixText pt, Texts texts, CodeTable codes, const uint2* __restrict__ list, const uint32_t* __restrict__ before, uint32_t leaves, uint32_t total, const uint32_t* __restrict__ sa, uint64_t* __restrict__ keys, uint32_t* __restrict__ positions) {
    __shared__ uint8_t code[256];
    loadCodes(codes, code);
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= total) {
        return;
    }
    const uint32_t leaf = bigLeafOf(before, leaves, k);
    const uint32_t p = min(sa[list[leaf].x + (k - before[leaf])], pt.span - 1);
    const uint32_t previous = p > texts.startOf(p) ? reinterpret_cast<const uint8_t*>(pt.words)[p - 1] : 0u;
    keys[k] = prefixKey(pt, texts, code, p) | previous;
    positions[k] = p;
}

// The sorted records back to the leaves' rows.
__global__ __launch_bounds__(256) void bigLeafRowsKernel(const uint64_t* __restrict__ keys, const uint32_t* __restrict__ positions, const uint2* __restrict__ list, const uint32_t* __restrict__ before, uint32_t leaves, uint32_t total, RowOut out) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= total) {
        return;
    }
    const uint32_t leaf = bigLeafOf(before, leaves, k);
    const uint32_t row = list[leaf].x + (k - before[leaf]);
    const uint64_t key = keys[k];
    const bool tied = k > 0 && keyPart(keys[k - 1]) == keyPart(key);
    emitRow(out, row, key, positions[k], tied);
    if (tied) {
        atomicOr(&out.ties[row >> 5], 1u << (row & 31));
    }
}

// ---- the sample, read off the rows ----------------------------------------------------------------

// Fields: sample rows before (sum), the last row that does not tie with the one before (max).
using SampleVec = Vec<2, 0x2u>;
constexpr int kSampleItems = 16;

template <int V>
__device__ __forceinline__ bool isSamplePosition(uint32_t p) {
    static_assert(V == 32, "a 32-bit mask");
    return (coverMask<V>() >> (p & (V - 1))) & 1u;
}

template <int V>
struct SampleProducer {
    const uint32_t* sa;
    const uint32_t* ties;
    __device__ SampleVec operator()(uint32_t row) const {
        const uint32_t p = sa[row];
        const uint32_t tied = (ties[row >> 5] >> (row & 31)) & 1u;
        SampleVec r;
        r.v[0] = isSamplePosition<V>(p) ? 1 : 0;
        r.v[1] = tied ? 0 : row;
        return r;
    }
};

// Sample row k of the order: its compact index and the row its group starts at.
template <int V>
struct SampleConsumer {
    const uint32_t* sa;
    uint32_t* index;
    uint32_t* group;
    uint32_t limit;
    struct Prepared {
        uint32_t p;
    };
    __device__ Prepared prepare(uint32_t row) const {
        return Prepared{sa[row]};
    }
    __device__ void complete(Prepared&) const {}
    __device__ void operator()(uint32_t, const Prepared& p, const SampleVec& item, const SampleVec& exclusive, bool valid) const {
        if (valid && item.v[0] && exclusive.v[0] < limit) {
            index[exclusive.v[0]] = packPosition<V>(p.p);
            group[exclusive.v[0]] = max(exclusive.v[1], item.v[1]);
        }
    }
};

// Fields: the last group's first entry (max), unresolved before (sum), unresolved groups before (sum).
using GroupVec = Vec<3, 0x1u>;

struct GroupProducer {
    const uint32_t* group;
    uint32_t count;
    __device__ GroupVec operator()(uint32_t k) const {
        const uint32_t own = group[k], previous = group[k > 0 ? k - 1 : 0], next = group[k + 1 < count ? k + 1 : k];
        const bool head = (k == 0) | (previous != own);
        const bool resolved = head & ((k + 1 == count) | (next != own));
        GroupVec r;
        r.v[0] = head ? k : 0;
        r.v[1] = resolved ? 0 : 1;
        r.v[2] = (!resolved && head) ? 1 : 0;
        return r;
    }
};

// The unresolved entries go to the list of the ranking passes, with their rank so far; the resolved
// ones stay in `index`, whose other entries become ~0, for scatterSortedRanksKernel.
struct GroupConsumer {
    uint32_t* index;
    uint32_t* ranks;
    uint32_t* nextT;
    uint32_t* nextOrdinal;
    uint32_t* nextGroupIds;
    struct Prepared {
        uint32_t t;
    };
    __device__ Prepared prepare(uint32_t k) const {
        return Prepared{index[k]};
    }
    __device__ void complete(Prepared&) const {}
    __device__ void operator()(uint32_t k, const Prepared& p, const GroupVec& item, const GroupVec& exclusive, bool valid) const {
        if (valid && item.v[1]) {
            const uint32_t id = max(exclusive.v[0], item.v[0]);
            ranks[p.t] = id;
            nextT[exclusive.v[1]] = p.t;
            nextOrdinal[exclusive.v[1]] = exclusive.v[2] + item.v[2] - 1;
            if (item.v[2]) {
                nextGroupIds[exclusive.v[2]] = id;
            }
            index[k] = ~0u;
        }
    }
};

// ranks[index[k]] = k for the entries in [first, last): a window of the rank array small enough for
// the memory-side cache (as scatterResolvedRanksKernel).
__global__ __launch_bounds__(256) void scatterSortedRanksKernel(const uint32_t* __restrict__ index, uint32_t count, uint32_t first, uint32_t last, uint32_t* __restrict__ ranks) {
    constexpr uint32_t kItems = 16;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t i0 = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i0 < count; i0 += stride * kItems) {
        uint32_t t[kItems];
#pragma unroll
        for (uint32_t k = 0; k < kItems; k++) {
            const uint64_t i = i0 + k * stride;
            t[k] = i < count ? index[i] : ~0u;
        }
#pragma unroll
        for (uint32_t k = 0; k < kItems; k++) {
            if (t[k] >= first && t[k] < last) {
                ranks[t[k]] = static_cast<uint32_t>(i0 + k * stride);
            }
        }
    }
}

// ---- ties -----------------------------------------------------------------------------------------

// Rows that tie with a neighbour, in order: bit r of the result for row 32 * word + r.
__device__ __forceinline__ uint32_t tiedRows(uint32_t own, uint32_t next) {
    return own | (own >> 1) | (next << 31);
}

struct TieProducer {
    const uint32_t* ties;  // one zero word past the end
    __device__ Vec<1, 0u> operator()(uint32_t w) const {
        Vec<1, 0u> r;
        r.v[0] = __builtin_popcount(tiedRows(ties[w], ties[w + 1]));
        return r;
    }
};

// Fields: rows that tie with a neighbour, rows of groups beyond kTieGroupMax.
struct TieCountProducer {
    const uint32_t* ties;
    __device__ Vec<2, 0u> operator()(uint32_t w) const {
        const uint32_t own = ties[w], next = ties[w + 1];
        Vec<2, 0u> r;
        r.v[0] = __builtin_popcount(tiedRows(own, next));
        r.v[1] = largeTieRows(own, next);
        return r;
    }
};

constexpr uint32_t kTieHead = 0x80000000u;

// rows[slot] = the row, kTieHead set on the first row of its group.
struct TieConsumer {
    const uint32_t* ties;
    uint32_t* rows;
    struct Prepared {
        uint32_t own, next;
    };
    __device__ Prepared prepare(uint32_t w) const {
        return Prepared{ties[w], ties[w + 1]};
    }
    __device__ void complete(Prepared&) const {}
    __device__ void operator()(uint32_t w, const Prepared& p, const Vec<1, 0u>&, const Vec<1, 0u>& exclusive, bool valid) const {
        if (valid) {
            uint32_t slot = exclusive.v[0];
            for (uint32_t m = tiedRows(p.own, p.next); m; m &= m - 1) {
                const uint32_t r = __builtin_ctz(m);
                rows[slot++] = (w * 32 + r) | ((p.own >> r) & 1u ? 0u : kTieHead);
            }
        }
    }
};

constexpr uint32_t kTieTile = 256;
constexpr uint32_t kTieRecords = kTieTile + kTieGroupMax;

constexpr int kTieRounds = (kTieRecords + kTieTile - 1) / kTieTile;  // list entries of a thread
using RankQuad = uint32_t __attribute__((ext_vector_type(4), aligned(4)));

// Groups of up to kTieGroupMax rows whose first row is in the workgroup's part of the list: every
// member's place is the number of members smaller than it. Members of larger groups are flagged.
//
// Two suffixes i and j compare at the smallest offset k with i + k and j + k both sampled: the
// characters before it, then the ranks there. Bound by the random lines this reads, so a member reads
// the one rank of a pair (the window of seven in a larger group), and its text only if some k of its
// group lies past the `shared` characters of the group's key; the comparisons are between copies in LDS.
template <class Texts>
__global__ __launch_bounds__(kTieTile) void tieGroupsKernel(MergeCtx c, Texts texts, uint32_t shared, const uint32_t* __restrict__ rows, uint32_t count, RowOut out, uint8_t* __restrict__ large, uint32_t* __restrict__ largeCount) {
    constexpr int kRanks = CoverSet<32>::kSize;
    __shared__ uint32_t listed[kTieGroupMax + kTieRecords + 1];  // rows from kTieGroupMax before the tile
    __shared__ uint32_t position[kTieRecords];
    __shared__ uint32_t ranks[kRanks][kTieRecords];  // the window's, or the pair's in ranks[0]
    __shared__ uint64_t words[4][kTieRecords];       // characters from shared & ~7 on
    const uint32_t tile0 = blockIdx.x * kTieTile;
    for (uint32_t x = threadIdx.x; x < kTieGroupMax + kTieRecords + 1; x += kTieTile) {
        const int64_t j = static_cast<int64_t>(tile0) + x - kTieGroupMax;
        const uint32_t row = j >= 0 && j < count ? rows[j] : kTieHead;
        listed[x] = row;
        if (x >= kTieGroupMax && x < kTieGroupMax + kTieRecords && j < count) {
            const uint32_t p = out.sa[row & ~kTieHead];
            position[x - kTieGroupMax] = p < c.n ? p : 0;
        }
    }
    __syncthreads();
    const uint32_t inList = min(kTieRecords, count - tile0);  // entries of the tile and after it
    const uint32_t firstChar = shared & ~7u;
    auto offsetOf = [](uint32_t i, uint32_t j) -> uint32_t {
        return __builtin_ctz(windowOf32(coverMask<32>(), i) & windowOf32(coverMask<32>(), j));
    };
    uint32_t head[kTieRounds], size[kTieRounds];  // of the entry's group, size 0 if it is not handled here
    uint32_t flagged = 0;
#pragma unroll
    for (int round = 0; round < kTieRounds; round++) {
        const uint32_t x = threadIdx.x + round * kTieTile;
        head[round] = 0;
        size[round] = 0;
        if (x >= inList) {
            continue;
        }
        uint32_t back = 0;
        while (back <= kTieGroupMax && !(listed[x + kTieGroupMax - back] & kTieHead)) {
            back++;
        }
        // back < kTieGroupMax: the head is listed[x + kTieGroupMax - back]. Past the list's ends every
        // entry is a head.
        uint32_t length = kTieGroupMax + 1;
        if (back < kTieGroupMax) {
            const uint32_t first = x + kTieGroupMax - back;
            length = back + 1;
            while (length <= kTieGroupMax && first + length < kTieGroupMax + kTieRecords + 1 && !(listed[first + length] & kTieHead)) {
                length++;
            }
        }
        if (x < kTieTile) {
            const bool isLarge = length > kTieGroupMax;
            large[tile0 + x] = isLarge ? 1 : 0;
            flagged += isLarge ? 1 : 0;
        }
        // Handled here: small, the head in the tile.
        if (length > kTieGroupMax || back > x || x - back >= kTieTile) {
            continue;
        }
        head[round] = x - back;
        size[round] = length;
        const uint32_t p = position[x];
        uint32_t furthest = 0;
        for (uint32_t y = x - back; y < x - back + length; y++) {
            furthest = y != x ? max(furthest, offsetOf(p, position[y])) : furthest;
        }
        if (length == 2) {
            ranks[0][x] = p + furthest < texts.endOf(p) ? c.ranks[packPosition<32>(p + furthest)] : 0;
        } else {
            const uint32_t* window = c.ranks + (p / 32) * kRanks + coverBelow<32>(p & 31);
            const RankQuad a = *reinterpret_cast<const RankQuad*>(window), b = *reinterpret_cast<const RankQuad*>(window + 3);
            ranks[0][x] = a.x;
            ranks[1][x] = a.y;
            ranks[2][x] = a.z;
            ranks[3][x] = a.w;
            ranks[4][x] = b.y;
            ranks[5][x] = b.z;
            ranks[6][x] = b.w;
        }
        if (furthest > shared) {
            const uint32_t at = p + firstChar, shift = (at & 7) * 8;
            uint64_t low = c.text[at >> 3];
#pragma unroll
            for (uint32_t w = 0; w < 4; w++) {
                if (firstChar + 8 * w < 32) {
                    const uint64_t high = c.text[(at >> 3) + w + 1];
                    words[w][x] = __builtin_bswap64(shift ? (low >> shift) | (high << (64 - shift)) : low);
                    low = high;
                }
            }
        }
    }
    __syncthreads();
    uint32_t target[kTieRounds], byteAt[kTieRounds];
    uint8_t byte[kTieRounds];
#pragma unroll
    for (int round = 0; round < kTieRounds; round++) {
        const uint32_t x = threadIdx.x + round * kTieTile;
        if (size[round] == 0) {
            continue;
        }
        const uint32_t p = position[x], end = texts.endOf(p), start = texts.startOf(p);
        const uint32_t headRow = listed[head[round] + kTieGroupMax] & ~kTieHead;
        uint32_t smaller = 0;
        bool startHere = p == start, afterStart = false;
        for (uint32_t y = head[round]; y < head[round] + size[round]; y++) {
            if (y == x) {
                continue;
            }
            const uint32_t q = position[y];
            const uint32_t k = offsetOf(p, q);
            const uint32_t last = max(p, q);
            const uint32_t common = min(k, end - last);
            bool less = q > p, decided = false;  // one a prefix of the other: the shorter is smaller
            if (common > shared) {
#pragma unroll
                for (uint32_t w = 0; w < 4; w++) {
                    const uint32_t from = firstChar + 8 * w;
                    if (from < common && !decided) {
                        const uint64_t mask = prefixMask(common - from);
                        const uint64_t own = words[w][x] & mask, other = words[w][y] & mask;
                        decided = own != other;
                        less = decided ? other < own : less;
                    }
                }
            }
            if (!decided && last + k < end) {
                const uint32_t before = (1u << k) - 1;
                const uint32_t ownSlot = size[round] == 2 ? 0 : __builtin_popcount(windowOf32(coverMask<32>(), p) & before);
                const uint32_t otherSlot = size[round] == 2 ? 0 : __builtin_popcount(windowOf32(coverMask<32>(), q) & before);
                less = ranks[otherSlot][y] < ranks[ownSlot][x];
            }
            smaller += less ? 1 : 0;
            if (q == start) {
                startHere = true;
                afterStart = less;
            }
        }
        target[round] = headRow + smaller;
        if (out.bwt) {
            const uint32_t segment = texts.segmentOf(p);
            if (!startHere) {
                // The group's bytes are in its own places, one further on before the text's first row.
                const uint32_t shift = headRow - out.segments[segment].rowBase < out.firstRows[segment] ? 1 : 0;
                byte[round] = out.bwt[headRow + (x - head[round]) + shift];
                byteAt[round] = headRow + smaller + shift;
            } else {
                byte[round] = p != start ? reinterpret_cast<const uint8_t*>(c.text)[p - 1] : 0;
                byteAt[round] = headRow + smaller + (afterStart ? 0 : 1);
            }
        }
    }
    const uint64_t any = ballot(flagged != 0);
    if (any != 0) {
        for (int offset = kWave / 2; offset > 0; offset /= 2) {
            flagged += __shfl_xor(flagged, offset);
        }
        if (threadIdx.x % kWave == 0) {
            atomicAdd(largeCount, flagged);
        }
    }
    // Every byte of the tile's groups is read before any is written.
    __syncthreads();
#pragma unroll
    for (int round = 0; round < kTieRounds; round++) {
        if (size[round]) {
            const uint32_t p = position[threadIdx.x + round * kTieTile];
            out.sa[target[round]] = p;
            if (out.bwt) {
                if (p == texts.startOf(p)) {
                    const uint32_t segment = texts.segmentOf(p);
                    out.firstRows[segment] = target[round] - out.segments[segment].rowBase;
                } else {
                    out.bwt[byteAt[round]] = byte[round];
                }
            }
        }
    }
}

// ---- large tie groups -----------------------------------------------------------------------------

// Fields: flagged entries before, flagged heads before.
using LargeVec = Vec<2, 0u>;
constexpr int kLargeItems = 8;

struct LargeProducer {
    const uint8_t* flags;
    const uint32_t* rows;
    __device__ LargeVec operator()(uint32_t j) const {
        LargeVec r;
        r.v[0] = flags[j];
        r.v[1] = r.v[0] && (rows[j] & kTieHead) ? 1 : 0;
        return r;
    }
};

// Large group entries in order: their row, position and sort key: class, group, rank of the next
// sample suffix plus one (0: that suffix is empty). A group shares at least kClasses - 1 characters,
// so within one class its suffixes are in the order of those ranks.
template <int V, class Texts>
struct LargeConsumer {
    const uint32_t* rows;
    const uint32_t* sa;
    const uint32_t* ranks;
    Texts texts;
    uint32_t span;
    int groupBits, rankBits;
    uint32_t* largeRow;
    uint64_t* keys;
    uint32_t* positions;
    struct Prepared {};
    __device__ Prepared prepare(uint32_t) const {
        return {};
    }
    __device__ void complete(Prepared&) const {}
    __device__ void operator()(uint32_t j, const Prepared&, const LargeVec& item, const LargeVec& exclusive, bool valid) const {
        if (valid && item.v[0]) {
            const uint32_t m = exclusive.v[0];
            const uint32_t row = rows[j] & ~kTieHead;
            const uint32_t p = min(sa[row], span - 1);
            const uint32_t d = classOf<V>(p);
            const uint32_t q = p + d;
            const uint64_t rank = q < texts.endOf(p) ? static_cast<uint64_t>(ranks[packPosition<V>(q)]) + 1 : 0;
            const uint64_t group = exclusive.v[1] + item.v[1] - 1;
            largeRow[m] = row;
            positions[m] = p;
            keys[m] = ((static_cast<uint64_t>(d) << groupBits | group) << rankBits) | rank;
        }
    }
};

// classStart[d] (d <= classes) = entries of the sorted keys of classes below d.
__global__ void classStartsKernel(const uint64_t* __restrict__ keys, uint32_t count, int shift, uint32_t classes, uint32_t* __restrict__ classStart) {
    const uint32_t d = threadIdx.x;
    if (d <= classes) {
        uint32_t lo = 0, hi = count;
        while (lo < hi) {
            const uint32_t mid = (lo + hi) / 2;
            if ((keys[mid] >> shift) < d) {
                lo = mid + 1;
            } else {
                hi = mid;
            }
        }
        classStart[d] = lo;
    }
}

// The merged large groups back to their rows: entry m of the merged order is positions[order[m]].
template <class Texts>
__global__ __launch_bounds__(256) void largeRowsKernel(MergeCtx c, Texts texts, const uint32_t* __restrict__ largeRow, const uint32_t* __restrict__ positions, const uint32_t* __restrict__ order, uint32_t count, RowOut out) {
    const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < count) {
        const uint32_t p = positions[min(order[m], count - 1)];
        const uint32_t row = largeRow[m];
        out.sa[row] = p;
        if (p == texts.startOf(p)) {
            const uint32_t segment = texts.segmentOf(p);
            out.firstRows[segment] = row - out.segments[segment].rowBase;
        }
    }
}

// Their BWT bytes, once every text's first row is known.
template <class Texts>
__global__ __launch_bounds__(256) void largeBytesKernel(MergeCtx c, Texts texts, const uint32_t* __restrict__ largeRow, uint32_t count, RowOut out) {
    const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < count) {
        const uint32_t row = largeRow[m];
        const uint32_t p = out.sa[row];
        const uint32_t segment = texts.segmentOf(p);
        if (p != texts.startOf(p)) {
            const uint32_t local = row - out.segments[segment].rowBase;
            out.bwt[local < out.firstRows[segment] ? row + 1 : row] = reinterpret_cast<const uint8_t*>(c.text)[p - 1];
        }
    }
}

// A batch's rows hold positions of all texts; the outputs are positions in each text. A workgroup's
// rows are consecutive, mostly of one text: it searches the row's text once and steps from there (a
// lookup by position reads two tables at random for every row: 2.9 against 1.1 ms for 515M rows).
constexpr int kLocalItems = 16;

__global__ __launch_bounds__(256) void localRowsKernel(const Segment* __restrict__ segments, uint32_t texts, uint32_t* __restrict__ sa, uint32_t count) {
    const uint64_t first = static_cast<uint64_t>(blockIdx.x) * 256 * kLocalItems;
    uint32_t lo = 0, hi = texts;  // the last text with rowBase <= first
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (segments[mid].rowBase <= first) {
            lo = mid;
        } else {
            hi = mid;
        }
    }
    uint32_t text = lo;
    Segment segment = segments[text];
#pragma unroll
    for (int j = 0; j < kLocalItems; j++) {
        const uint64_t row = first + j * 256 + threadIdx.x;
        if (row < count) {
            while (row >= segment.rowBase + static_cast<uint64_t>(segment.end - segment.start)) {
                segment = segments[++text];
            }
            sa[row] -= segment.start;
        }
    }
}

}  // namespace sadcs
