// How kernels are launched.
#pragma once
#include <hip/hip_runtime.h>

#include <utility>

namespace mrb {

// The launch with its arguments by address. (The <<<>>> form first leaves the grid in a place of the runtime's own, calls a stub that
// fetches it from there, and only then comes to this call: 2.33 to 2.45 us of host time a launch with 24 to 1000 bytes of arguments, this
// way 2.17 to 2.31.)
template <typename... P>
void launch_by_address(const void* kernel, dim3 grid, dim3 block, size_t lds, hipStream_t s, const P&... args) {
    void* at[sizeof...(P) + 1] = {const_cast<void*>(static_cast<const void*>(&args))..., nullptr};
    (void)hipLaunchKernel(kernel, grid, block, at, lds, s);  // (what it returns, hipGetLastError() says)
}

// kernel<<<grid, block, lds, s>>>(args...). An argument of the parameter's own type is passed from where it lies, others are converted.
template <typename... P, typename... A>
void launch_kernel(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, A&&... args) {
    static_assert(sizeof...(P) == sizeof...(A), "an argument for each parameter");
    launch_by_address(reinterpret_cast<const void*>(kernel), grid, block, lds, s, static_cast<const P&>(args)...);
}

}  // namespace mrb
