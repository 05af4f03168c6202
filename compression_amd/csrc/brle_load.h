// Which loads a thread of the byte RLE encoder may take.  Plain C++, so that
// the rule is checked on the host at the lengths that no test can allocate.
#pragma once

#include <stdint.h>

namespace mdz {

constexpr uint32_t kBrlePer = 32;               // bytes per thread and window

// Whether the whole dwords around the thread's bytes [w0 + at, w0 + at +
// kBrlePer) of a chunk of len bytes, which starts skew bytes past a dword,
// and the dword after them lie inside the chunk.  The window starts at
// w0 < len, and w0 + at fits 32 bits; that plus the bytes does not where a
// chunk ends just below 4 GiB, so the chunk's rest is compared instead.
constexpr bool brle_whole_dwords(uint32_t w0, uint32_t at, uint32_t len, uint32_t skew) {
    return len - w0 >= at + kBrlePer + 4 && w0 + at >= skew;
}

}  // namespace mdz
