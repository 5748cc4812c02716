// Stores that are written through to memory, HBM or the host's: they have reached it when vmcnt says so.
#ifndef MF_THROUGH_H
#define MF_THROUGH_H

#include <stdint.h>

namespace mf {
namespace {

// 16 bytes.  A store of more than 64 bits reads its data late, and a vector instruction may write those registers only two wait states later; the compiler sees to that
// for stores of its own only.
template <class Vector>
__device__ __forceinline__ void StoreThrough16(uint64_t at, Vector v)
{
    static_assert(sizeof(Vector) == 16, "");
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1 nt\n\ts_nop 1" : : "v"(at), "v"(v) : "memory");
}

__device__ __forceinline__ void StoreThrough1(uint64_t at, uint32_t byte)
{
    asm volatile("global_store_byte %0, %1, off sc0 sc1 nt" : : "v"(at), "v"(byte) : "memory");
}

}  // namespace
}  // namespace mf

#endif  // MF_THROUGH_H
