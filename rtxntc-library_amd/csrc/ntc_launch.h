// ntc_launch.h - kernel launches of the calls whose time is the launch.
#ifndef NTC_LAUNCH_H
#define NTC_LAUNCH_H
#include <hip/hip_runtime.h>
#include <atomic>

namespace ntc_hip_dev {

// Launches KERNEL(args...) on the current device.  The kernel's function is looked up once per device: the runtime does so
// at every launch by the host symbol otherwise (3.0 us of host time for a launch with 136 bytes of arguments, 2.7 this
// way).  Arguments should fit 128 bytes: from there to 256 a launch costs another 0.3 us.  So a kernel should not use
// gridDim or blockDim either, which lie in 256 bytes of arguments that the compiler adds.
template <class> struct KernelParameters;
template <class... T> struct KernelParameters<void (*)(T...)> {
    template <auto KERNEL>
    static hipError_t launch(dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream, T... args)
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
        return hipModuleLaunchKernel(function, grid.x, grid.y, grid.z, block.x, block.y, block.z, unsigned(ldsBytes), stream, pointers, nullptr);
    }
};
template <auto KERNEL, class... ARGS>
inline hipError_t launch_kernel(dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream, ARGS const&... args)
{
    return KernelParameters<decltype(KERNEL)>::template launch<KERNEL>(grid, block, ldsBytes, stream, args...);
}

} // namespace ntc_hip_dev
#endif
