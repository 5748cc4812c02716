// Launching a kernel whose call is short, so that the host's side of the launch is what counts.
//
// What a launch costs there depends on its arguments.  Steady, us (the host settles after some thousand launches): 2.6 with up to
// 112 bytes of them, 3.4 from 120 bytes on, whatever the size; 3.9 with thirteen arguments of which seven are pointers, 2.7 with the
// same as integers: the runtime looks pointers up.  A kernel that asks for its grid's or its workgroups' size (gridDim,
// blockDim, __syncthreads_or) has 256 bytes of arguments more, so such kernels are told.
#ifndef MF_LAUNCH_H
#define MF_LAUNCH_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <tuple>

namespace mf {
namespace {

// A buffer as such kernels get it, and what they make of it.
inline uint64_t At(const volatile void *buffer)
{
    return reinterpret_cast<uint64_t>(buffer);
}

template <typename T>
__device__ __forceinline__ T *Buffer(uint64_t address)
{
    return (T *)reinterpret_cast<__attribute__((address_space(1))) T *>(address);
}

// What <<<>>> does without the launch configuration that it pushes and pops around the same call (0.15 us).  `args` are converted to the types
// of the kernel's parameters.
template <typename... Params, typename... Args>
inline int Launch(void (*kernel)(Params...), uint32_t grid, uint32_t block, uint32_t ldsBytes, hipStream_t stream, Args... args)
{
    std::tuple<Params...> values(static_cast<Params>(args)...);
    return std::apply(
        [&](auto &...value) {
            void *at[] = {const_cast<void *>(static_cast<const volatile void *>(&value))...};
            return static_cast<int>(
                hipLaunchKernel(reinterpret_cast<const void *>(kernel), dim3(grid), dim3(block), at, ldsBytes, stream));
        },
        values);
}

}  // namespace
}  // namespace mf

#endif  // MF_LAUNCH_H
