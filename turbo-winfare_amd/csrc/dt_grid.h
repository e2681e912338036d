// Grid sizes of kernels that walk a count of items. Host code only, without HIP.
#pragma once

#include <algorithm>
#include <cstdint>

namespace tdt {

// A launch may hold at most 2^32 - 1 threads in one dimension, and the largest table the library
// accepts (16,777,216 x 8192) has 2^32 weight items of 16 bytes and 2^31 scale words: a part of a
// grid is capped, and its workgroups step over what is left.
constexpr uint64_t kMaxPartThreads = 1ull << 30;

inline uint32_t part_blocks(uint64_t items, uint32_t threads) {
    return static_cast<uint32_t>(std::min<uint64_t>((items + threads - 1u) / threads, kMaxPartThreads / threads));
}

}  // namespace tdt
