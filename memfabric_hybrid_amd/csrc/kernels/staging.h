// What the CPU and the kernels of staging.hip agree on.  Plain C++.
#ifndef MF_STAGING_H
#define MF_STAGING_H

#include <stdint.h>

namespace mf {

constexpr uint32_t kStreamChunkBytes = 64u << 10;      // a slot; a chunk ends in it
constexpr uint32_t kStreamLine = 128;                  // a chunk lies in its slot as far behind a multiple of this as it does in HBM
constexpr uint32_t kStreamWordBytes = 64;              // a word per slot and side, on a line of its own
constexpr uint32_t kStreamMostMillis = 4000;           // of the kernel's wait: its ticks are 32 bits at up to 1 GHz

struct StreamChunk {
    uint64_t at;        // in HBM
    uint32_t len;       // 1 to kStreamChunkBytes - at % kStreamLine
    uint32_t reserved;
};
static_assert(sizeof(StreamChunk) == 16, "");

}  // namespace mf

#endif  // MF_STAGING_H
