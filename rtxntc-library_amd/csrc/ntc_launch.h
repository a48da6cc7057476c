// ntc_launch.h - kernel launches of the calls whose time is the launch.
#ifndef NTC_LAUNCH_H
#define NTC_LAUNCH_H
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <atomic>
#include <stdint.h>

namespace ntc_hip_dev {

// Launches KERNEL(args...) on the current device.  The kernel's function is looked up once per device: the runtime does so
// at every launch by the host symbol otherwise (3.0 us of host time for a launch with 136 bytes of arguments, 2.7 this
// way).  Arguments should fit 128 bytes: from there to 256 a launch costs another 0.3 us.  So a kernel should not use
// gridDim or blockDim either, which lie in 256 bytes of arguments that the compiler adds.
template <class> struct KernelParameters;
template <class... T> struct KernelParameters<void (*)(T...)> {
    template <auto KERNEL>
    static hipError_t launch(dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream, hipEvent_t done, T... args)
    {
        constexpr int kDevices = 64;
        static std::atomic<hipFunction_t> functions[kDevices];
        int device = 0;
        if (hipError_t const e = hipGetDevice(&device); e != hipSuccess) return e;
        bool const kept = unsigned(device) < unsigned(kDevices);
        hipFunction_t function = kept ? functions[device].load(std::memory_order_acquire) : nullptr;
        if (!function) {
            if (hipError_t const e = hipGetFuncBySymbol(&function, reinterpret_cast<void const*>(KERNEL)); e != hipSuccess) return e;
            if (kept) functions[device].store(function, std::memory_order_release);
        }
        void* pointers[] = { const_cast<void*>(static_cast<void const*>(&args))... };
        if (done) {                                          // (takes threads, not workgroups)
            if (uint64_t(grid.x) * block.x > 0xffffffffu || uint64_t(grid.y) * block.y > 0xffffffffu) return hipErrorInvalidConfiguration;
            return hipExtModuleLaunchKernel(function, grid.x * block.x, grid.y * block.y, grid.z * block.z, block.x, block.y, block.z, ldsBytes, stream, pointers, nullptr, nullptr, done);
        }
        return hipModuleLaunchKernel(function, grid.x, grid.y, grid.z, block.x, block.y, block.z, unsigned(ldsBytes), stream, pointers, nullptr);
    }
};
template <auto KERNEL, class... ARGS>
inline hipError_t launch_kernel(dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream, ARGS const&... args)
{
    return KernelParameters<decltype(KERNEL)>::template launch<KERNEL>(grid, block, ldsBytes, stream, nullptr, args...);
}
// The same with an event that completes with the launch itself: no packet of its own, as a recorded event is.
template <auto KERNEL, class... ARGS>
inline hipError_t launch_kernel_with_event(dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream, hipEvent_t done, ARGS const&... args)
{
    return KernelParameters<decltype(KERNEL)>::template launch<KERNEL>(grid, block, ldsBytes, stream, done, args...);
}

} // namespace ntc_hip_dev
#endif
