// Bit layout of the byte-code matches of k_fv_rows (select.hip), apart from HIP so that the host can
// check it.
#pragma once

#include <cstdint>

namespace tdt {

// A hit word holds the matches of eight code words of four elements: bit 8 e + 7 - w for element e of
// its word w. The bits of those whose word, counted from `first` on, is one of the `words` that the
// thread's part of the row fills; the words after them hold code 0, the code of the largest logits.
constexpr uint32_t filled_hits(uint32_t first, uint32_t words) {
    const uint32_t n = words <= first ? 0u : words - first >= 8u ? 8u : words - first;
    return ((0xFF00u >> n) & 0xFFu) * 0x01010101u;
}

}  // namespace tdt
